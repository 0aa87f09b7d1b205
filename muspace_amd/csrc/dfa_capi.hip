// C-ABI entry points of deformable aggregation (declared in include/muspace_dfa.h).
//
// Replaces the reference's four TVM-FFI exports
// deformable_aggregation_{forward,backward}_{opt,base}
// (/root/reference/csrc/deformable_aggregation/deformable_aggregation_musa.mu:683-751),
// keeping their argument order (feature maps, spatial_shape, scale_start_index,
// sampling_location, weights, outputs) and their accumulate semantics: the
// forward adds into `output` and the backward adds into `grad_mc_ms_feat`
// (callers zero them, as the reference's autograd function does), while the
// location and weight gradients are written. "opt" takes the wavefront-per-
// anchor row kernels when the channel layout allows it; "base" always takes
// the generic kernels.
#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <type_traits>

#include "../../include/muspace_dfa.h"
#include "capi_errors.hpp"
#include "dfa_kernels.hpp"

namespace {

using capi::check_launch;
using capi::fail;
using capi::ok;

struct DfaArgs {
  int64_t batch, cams, feat, embeds, scales, anchors, pts, groups;
};

int validate(const char *fn, const DfaArgs &a, dfa::Dims &d) {
  if (a.batch < 0 || a.cams < 0 || a.feat < 0 || a.embeds <= 0 || a.scales < 0 ||
      a.anchors < 0 || a.pts < 0) {
    return fail(MUSPACE_EINVAL,
                "%s: invalid dims batch=%lld num_cams=%lld num_feat=%lld num_embeds=%lld "
                "num_scale=%lld num_anchors=%lld num_pts=%lld",
                fn, (long long)a.batch, (long long)a.cams, (long long)a.feat,
                (long long)a.embeds, (long long)a.scales, (long long)a.anchors,
                (long long)a.pts);
  }
  if (a.groups <= 0 || a.groups > dfa::kMaxGroups) {
    return fail(MUSPACE_EINVAL, "%s: num_groups must be in [1, %d], got %lld", fn,
                dfa::kMaxGroups, (long long)a.groups);
  }
  if (a.embeds % a.groups != 0) {
    return fail(MUSPACE_EINVAL, "%s: num_embeds %lld must be divisible by num_groups %lld", fn,
                (long long)a.embeds, (long long)a.groups);
  }
  if (a.cams * a.scales > dfa::kMaxViews) {
    return fail(MUSPACE_EINVAL, "%s: num_cams * num_scale must be at most %d, got %lld", fn,
                dfa::kMaxViews, (long long)(a.cams * a.scales));
  }
  if (a.batch * a.anchors > INT_MAX || a.feat > INT_MAX || a.embeds > INT_MAX ||
      a.pts * a.cams > INT_MAX / 2) {
    return fail(MUSPACE_ERANGE, "%s: dims exceed the kernels' 32-bit indexing", fn);
  }
  d.batch = static_cast<int>(a.batch);
  d.cams = static_cast<int>(a.cams);
  d.feat = static_cast<int>(a.feat);
  d.embeds = static_cast<int>(a.embeds);
  d.scales = static_cast<int>(a.scales);
  d.anchors = static_cast<int>(a.anchors);
  d.pts = static_cast<int>(a.pts);
  d.groups = static_cast<int>(a.groups);
  return ok();
}

int generic_blocks(int64_t work) {
  int64_t b = (work + dfa::kBlock - 1) / dfa::kBlock;
  if (b > 65536) b = 65536;
  if (b < 1) b = 1;
  return static_cast<int>(b);
}

// Channel slots per lane of the row kernels (C = 64 * NT), or 0 when the
// layout needs the generic kernels: C a multiple of 64 up to 256, each group
// a power-of-two run of lanes or a whole number of 64-channel slots, and the
// features addressable with 32-bit byte offsets.
int row_slots(const dfa::Dims &d) {
  const int C = d.embeds;
  if (C % dfa::kWave != 0 || C / dfa::kWave > 4) return 0;
  const int cpg = C / d.groups;
  const bool pow2 = (cpg & (cpg - 1)) == 0;
  if (!(cpg % dfa::kWave == 0 || (cpg < dfa::kWave && pow2))) return 0;
  const uint64_t bytes = static_cast<uint64_t>(d.batch) * d.feat * C * 4u;
  if (bytes + 64 > dfa::kOobOffset) return 0;
  return C / dfa::kWave;
}

// Channel slice of dfa_backward_coarse (0: every map is left to the row
// kernel's atomics), with its accumulator budget in cells and the bound on
// contributions per sum (2^pair_log2 >= anchors * pts). The host does not see
// the map sizes (device tensors), so it sizes the slice for the maps below the
// finest of a pyramid that halves each scale, about a quarter of a camera's
// rows: the widest slice whose accumulators hold that many cells. The kernels
// choose the maps that fit on the device. The kernel reads grad_output in
// 16-byte pieces and locations in 8-byte pieces, so it needs pointers aligned
// to those.
int coarse_slice(const dfa::Dims &d, const float *loc, const float *grad_out, int &budget,
                 int &pair_log2) {
  const int64_t pairs = static_cast<int64_t>(d.anchors) * d.pts;
  if (d.scales == 0 || d.cams == 0 || pairs > (int64_t{1} << 20) ||
      reinterpret_cast<uintptr_t>(grad_out) % 16 != 0 || reinterpret_cast<uintptr_t>(loc) % 8 != 0) {
    return 0;
  }
  pair_log2 = 0;
  while ((int64_t{1} << pair_log2) < pairs) ++pair_log2;
  const int cpg = d.embeds / d.groups;
  const int64_t want = static_cast<int64_t>(d.feat) / d.cams / 4;
  for (int cs : {16, 8, 4}) {
    if (cpg % cs != 0) continue;
    budget = dfa::kCoarseLdsBytes / (8 * cs);
    if (budget >= want || cs == 4) return cs;
  }
  return 0;
}

template <int CS>
void launch_coarse(const int32_t *shape, const int32_t *start, const float *loc,
                   const float *weights, const float *grad_out, float *grad_feat,
                   const dfa::Dims &d, int budget, int pair_log2, hipStream_t st) {
  const size_t lds = static_cast<size_t>(budget) * CS * sizeof(unsigned long long);
  (void)hipFuncSetAttribute(reinterpret_cast<const void *>(dfa::dfa_backward_coarse<CS>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
  // a workgroup takes up to four slices of one weight group
  const int per_group = d.embeds / d.groups / CS;
  int ns = 4;
  while (per_group % ns != 0) --ns;
  const int blocks = d.batch * d.cams * (d.embeds / (CS * ns));
  dfa::dfa_backward_coarse<CS><<<blocks, dfa::kCoarseBlock, lds, st>>>(
      shape, start, loc, weights, grad_out, grad_feat, d, budget, pair_log2, ns);
}

// Wavefronts per row of dfa_forward_rows (a power of two up to 16). Few rows give
// each of the 1024 SIMDs few wavefronts with long serial pair walks, so a row's
// pairs are shared, until there are about 8192 wavefronts: from there on each one's
// own cost (maps, locations, its part of the sum) grows the total. At 4, 8 and 16,
// 78 pairs a row: 300 rows of 256 channels 17.1, 14.6 and 15.0 us (64 channels: 11.4,
// 8.8, 8.7); 900 rows 29.4, 28.4, 28.6 (15.6, 13.3, 15.3); 1800 rows of 64 channels
// 20.3, 20.6 and 24.9, of 128 27.5, 26.4 and 28.9. Long rows of 192 and 256 channels
// hold enough work for 8: 1800 rows 53.5 us at 4, 50.6 at 8; 7200 rows 184 and 179;
// but 1970 rows of 18 pairs 10.6 and 12.2. From 16384 rows on two wavefronts, from
// 32768 one (24000 rows of 64 channels: 160 us at 2, 166 at 4).
int forward_parts(const dfa::Dims &d) {
  const int rows = d.batch * d.anchors;
  if (rows >= 8192 * 4) return 1;
  if (rows >= 8192 * 2) return 2;
  int parts = 4;
  while (parts < 16 && rows <= 8192 / (2 * parts)) parts *= 2;
  if (parts == 4 && d.embeds >= 192 && d.pts * d.cams >= 64) parts = 8;
  return parts;
}

int forward_impl(const char *fn, bool optimized, const float *feat, const int32_t *shape,
                 const int32_t *start, const float *loc, const float *weights, float *out,
                 const DfaArgs &a, void *stream) {
  dfa::Dims d;
  if (int rc = validate(fn, a, d)) return rc;
  if (static_cast<int64_t>(d.batch) * d.anchors == 0) return ok();
  if (!out || ((!feat || !shape || !start || !loc || !weights) && d.pts * d.cams > 0)) {
    return fail(MUSPACE_EINVAL, "%s: null tensor pointer", fn);
  }
  if (d.pts * d.cams == 0 || d.scales == 0) return ok();  // nothing is added
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nt = optimized ? row_slots(d) : 0;
  const int rows = d.batch * d.anchors;
  const int parts = forward_parts(d);
  const int block = parts * dfa::kWave > dfa::kBlock ? parts * dfa::kWave : dfa::kBlock;
  const int per_block = block / dfa::kWave;
  const int blocks = (rows * parts + per_block - 1) / per_block;
  const size_t lds = parts > 1 ? static_cast<size_t>(per_block) * d.embeds * sizeof(float) : 0;
  const uint32_t bytes = static_cast<uint32_t>(static_cast<uint64_t>(d.batch) * d.feat *
                                               d.embeds * 4u);
  switch (nt) {
    case 1:
      dfa::dfa_forward_rows<1><<<blocks, block, lds, st>>>(feat, bytes, shape, start, loc,
                                                               weights, out, d, parts);
      break;
    case 2:
      dfa::dfa_forward_rows<2><<<blocks, block, lds, st>>>(feat, bytes, shape, start, loc,
                                                               weights, out, d, parts);
      break;
    case 3:
      dfa::dfa_forward_rows<3><<<blocks, block, lds, st>>>(feat, bytes, shape, start, loc,
                                                               weights, out, d, parts);
      break;
    case 4:
      dfa::dfa_forward_rows<4><<<blocks, block, lds, st>>>(feat, bytes, shape, start, loc,
                                                               weights, out, d, parts);
      break;
    default:
      dfa::dfa_forward_generic<<<generic_blocks(static_cast<int64_t>(rows) * d.embeds),
                                 dfa::kBlock, 0, st>>>(feat, shape, start, loc, weights, out, d);
      break;
  }
  return check_launch(fn);
}

uint32_t feature_bytes(const dfa::Dims &d) {
  return static_cast<uint32_t>(static_cast<uint64_t>(d.batch) * d.feat * d.embeds * 4u);
}

// Location and weight gradients by the row kernels; feature gradients with
// device atomics too (kFeat), but for the maps that dfa_backward_coarse took
// within `budget`.
template <bool kFeat>
void launch_backward_rows(int nt, const float *feat, const int32_t *shape, const int32_t *start,
                          const float *loc, const float *weights, const float *grad_out,
                          float *grad_feat, float *grad_loc, float *grad_weights,
                          const dfa::Dims &d, int budget, hipStream_t st) {
  const int rows = d.batch * d.anchors;
  // wavefronts per row, as in the forward (SparseDrive's 7,200 rows: 205, 195,
  // 205 and 236 us at 2, 4, 8 and 16; each part walks the row's locations)
  const int parts = rows >= 8192 * 4 ? 1 : rows >= 8192 * 2 ? 2 : 4;
  const int per_block = dfa::kBlock / dfa::kWave;
  const int blocks = (rows * parts + per_block - 1) / per_block;
  auto go = [&](auto slots) {
    dfa::dfa_backward_rows<decltype(slots)::value, kFeat><<<blocks, dfa::kBlock, 0, st>>>(
        feat, feature_bytes(d), shape, start, loc, weights, grad_out, grad_feat, grad_loc,
        grad_weights, d, budget, parts);
  };
  switch (nt) {
    case 1: go(std::integral_constant<int, 1>()); break;
    case 2: go(std::integral_constant<int, 2>()); break;
    case 3: go(std::integral_constant<int, 3>()); break;
    default: go(std::integral_constant<int, 4>()); break;
  }
}

void launch_backward_generic(const float *feat, const int32_t *shape, const int32_t *start,
                             const float *loc, const float *weights, const float *grad_out,
                             float *grad_feat, float *grad_loc, float *grad_weights,
                             const dfa::Dims &d, hipStream_t st) {
  const int64_t pairs = static_cast<int64_t>(d.batch) * d.anchors * d.pts * d.cams;
  dfa::dfa_backward_generic<<<generic_blocks(pairs), dfa::kBlock, 0, st>>>(
      feat, shape, start, loc, weights, grad_out, grad_feat, grad_loc, grad_weights, d);
}

// Feature gradients added to grad_feat without scratch: the small maps in LDS,
// the others with the row kernels' atomics.
int backward_impl(const char *fn, bool optimized, const float *feat, const int32_t *shape,
                  const int32_t *start, const float *loc, const float *weights,
                  const float *grad_out, float *grad_feat, float *grad_loc, float *grad_weights,
                  const DfaArgs &a, void *stream) {
  dfa::Dims d;
  if (int rc = validate(fn, a, d)) return rc;
  if (static_cast<int64_t>(d.batch) * d.anchors * d.pts * d.cams == 0) return ok();
  if (!feat || !shape || !start || !loc || !grad_out || !grad_feat || !grad_loc ||
      (!weights && d.scales > 0) || (!grad_weights && d.scales > 0)) {
    return fail(MUSPACE_EINVAL, "%s: null tensor pointer", fn);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nt = optimized ? row_slots(d) : 0;
  if (nt == 0) {
    launch_backward_generic(feat, shape, start, loc, weights, grad_out, grad_feat, grad_loc,
                            grad_weights, d, st);
    return check_launch(fn);
  }
  // the small maps' feature gradients summed in LDS first (they only add)
  int budget = 0, pair_log2 = 0;
  switch (coarse_slice(d, loc, grad_out, budget, pair_log2)) {
    case 16:
      launch_coarse<16>(shape, start, loc, weights, grad_out, grad_feat, d, budget, pair_log2,
                        st);
      break;
    case 8:
      launch_coarse<8>(shape, start, loc, weights, grad_out, grad_feat, d, budget, pair_log2, st);
      break;
    case 4:
      launch_coarse<4>(shape, start, loc, weights, grad_out, grad_feat, d, budget, pair_log2, st);
      break;
    default:
      budget = 0;
      break;
  }
  launch_backward_rows<true>(nt, feat, shape, start, loc, weights, grad_out, grad_feat, grad_loc,
                             grad_weights, d, budget, st);
  return check_launch(fn);
}

// Scratch of the owner sums (deformable_aggregation_backward_ws).
struct OwnerWorkspace {
  size_t list, list_n, cursor, rows, contrib, bytes;
};

// False where the shape has no row kernel, or its contributions would pass
// 32-bit offsets or 8 GiB: the gradients then come from the atomic kernels.
bool plan_owner(const dfa::Dims &d, OwnerWorkspace &w) {
  if (row_slots(d) == 0 || d.feat == 0) return false;
  const uint64_t pairs = static_cast<uint64_t>(d.anchors) * d.pts;
  const uint64_t cams = static_cast<uint64_t>(d.batch) * d.cams;
  const uint64_t per_entry = pairs * d.cams * d.scales;  // Contribution::index
  // dfa_sum_rows addresses an entry's weights and grad_out with 32-bit offsets
  if (per_entry * d.groups * 4 > INT_MAX ||
      static_cast<uint64_t>(d.anchors) * d.embeds * 4 > INT_MAX) {
    return false;
  }
  const uint64_t most = 4u * per_entry * d.batch;
  if (most > INT_MAX || cams * pairs > INT_MAX) return false;
  size_t off = 0;
  auto take = [&off](uint64_t bytes) {
    const size_t at = off;
    off += (bytes + 255) & ~uint64_t{255};
    return at;
  };
  w.list = take(cams * pairs * sizeof(float4));
  w.list_n = take(cams * sizeof(uint32_t));
  w.cursor = take(sizeof(uint32_t));
  w.rows = take(static_cast<uint64_t>(d.batch) * d.feat * sizeof(uint2));
  w.contrib = take(most * sizeof(dfa::Contribution));
  w.bytes = off;
  return off <= (size_t{8} << 30);
}

// Feature rows of a workgroup in dfa_list_rows and dfa_sum_rows: powers of two,
// sum_rows the smaller, so that a workgroup of the sums stays inside a range of
// the list.
//
// A range's workgroup walks its cameras' active pairs alone, so few feature rows
// are cut into shorter ranges, to occupy more CUs. Backward call at ranges of
// 2048, 512, 256 and 128 rows: 4.7 k rows (2 x 4 cameras of 21 x 22 and 11 x 11)
// 52, 42, 42 and 40 us; 60 k rows (2 x 2 cameras, SparseDrive's maps, 12220 pairs)
// 89, 83, 83 and 85 us; 718 k rows (SparseDrive's batch) 485, 495, 513 and 551 us.
//
// A workgroup of the sums takes rows for about 96 contributions, were every pair
// active, on average: 16 rows of small maps under many points hold thousands, and
// the chip then waits for a few long workgroups. At 16, 8, 4, 2 and 1 rows: 2 k
// rows that take 150 (one camera, 21 x 72 to 3 x 9, 9603 pairs) 136, 92, 65, 51 and
// 44 us; 26 k rows that take 54 (6 x 3 cameras, 30 x 37 to 8 x 10, 6588 pairs) 93,
// 83, 79, 81 and 93 us; SparseDrive's batch (12.5) 513, 533, 608, 731 and 986 us.
// Past 16384 workgroups the chip is full, and more rows share a row table's load.
struct OwnerSplit {
  int range_rows, sum_rows;
};

OwnerSplit split_owner(const dfa::Dims &d) {
  const int64_t rows = static_cast<int64_t>(d.batch) * d.feat;
  const int64_t most =  // contributions to an entry's rows
      int64_t{4} * d.anchors * d.pts * d.cams * d.scales;
  OwnerSplit o{dfa::kRangeRows, 1};
  while (o.range_rows > 256 && rows < int64_t{64} * o.range_rows) o.range_rows /= 2;
  while (o.sum_rows < dfa::kSumRows &&
         (2 * o.sum_rows * most <= int64_t{96} * d.feat || rows > int64_t{16384} * o.sum_rows)) {
    o.sum_rows *= 2;
  }
  return o;
}

// Whether the sums by owner beat the atomics. They list and sum at a cost per
// feature row and per active pair of a camera; the atomics pay per contribution,
// and where maps are small, for adds that meet in one row. Measured as the backward
// call with atomics over the call with owner sums (some 600 shapes of 1 to 8 entries, 1
// to 6 cameras, 250 to 240000 pairs, most with 18.6% of the pairs active):
// - 128 channels and more, two scales and more, up to 32768 rows a camera: 1.1 to 6
//   (geometric mean 2.0). 64 channels: 0.7 to 2.7 (1.1).
// - One scale: 0.4 to 2.8 (1.03): every camera's pairs are listed for a fourth of
//   the adds.
// - Larger maps (200 x 200 with 100 x 100, 400 x 400): few adds meet. 0.65 to 0.9 for
//   one and two (entry, camera) pairs, whose list one workgroup writes each; from
//   four on 0.84 to 0.96 at 1300 pairs a camera, 1.2 to 2.3 from 11700. 64 channels
//   0.3 to 0.8.
bool owner_is_faster(const dfa::Dims &d) {
  if (d.scales < 2 || d.cams == 0) return false;
  const int64_t rows = d.feat / d.cams;
  const int64_t pairs = static_cast<int64_t>(d.anchors) * d.pts;
  return rows <= 32768 ||
         (d.embeds >= 128 && static_cast<int64_t>(d.batch) * d.cams >= 4 &&
          2 * pairs * d.scales >= rows);
}

// The backward with grad_feat overwritten: feature gradients by owner sums
// when `workspace` holds them.
int backward_ws_impl(const char *fn, const float *feat, const int32_t *shape,
                     const int32_t *start, const float *loc, const float *weights,
                     const float *grad_out, float *grad_feat, float *grad_loc,
                     float *grad_weights, const DfaArgs &a, void *workspace,
                     size_t workspace_bytes, void *stream) {
  dfa::Dims d;
  if (int rc = validate(fn, a, d)) return rc;
  const int64_t n_feat = static_cast<int64_t>(d.batch) * d.feat * d.embeds;
  const bool sampled = static_cast<int64_t>(d.batch) * d.anchors * d.pts * d.cams > 0;
  if ((n_feat > 0 && !grad_feat) ||
      (sampled && (!feat || !shape || !start || !loc || !grad_out || !grad_loc ||
                   (!weights && d.scales > 0) || (!grad_weights && d.scales > 0)))) {
    return fail(MUSPACE_EINVAL, "%s: null tensor pointer", fn);
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  OwnerWorkspace w;
  // the kernels read and write the workspace in pieces of up to 16 bytes
  const bool aligned = reinterpret_cast<uintptr_t>(workspace) % 256 == 0;
  if (!sampled || !plan_owner(d, w) || !workspace || workspace_bytes < w.bytes || !aligned) {
    if (n_feat > 0) {
      const int64_t blocks = (n_feat / 4 + dfa::kBlock) / dfa::kBlock;
      dfa::dfa_zero<<<static_cast<int>(blocks < (1 << 22) ? blocks : 1 << 22), dfa::kBlock, 0,
                      st>>>(grad_feat, n_feat);
    }
    if (!sampled) return check_launch(fn);
    return backward_impl(fn, true, feat, shape, start, loc, weights, grad_out, grad_feat,
                         grad_loc, grad_weights, a, stream);
  }
  unsigned char *ws = static_cast<unsigned char *>(workspace);
  float4 *list = reinterpret_cast<float4 *>(ws + w.list);
  uint32_t *list_n = reinterpret_cast<uint32_t *>(ws + w.list_n);
  uint32_t *cursor = reinterpret_cast<uint32_t *>(ws + w.cursor);
  uint2 *rows = reinterpret_cast<uint2 *>(ws + w.rows);
  dfa::Contribution *contrib = reinterpret_cast<dfa::Contribution *>(ws + w.contrib);
  const int nt = row_slots(d);
  dfa::dfa_list_active<<<d.batch * d.cams, dfa::kListBlock, 0, st>>>(loc, list, list_n, cursor, d);
  const OwnerSplit split = split_owner(d);
  const int ranges = (d.feat + split.range_rows - 1) / split.range_rows;
  dfa::dfa_list_rows<<<d.batch * ranges, dfa::kRangeBlock, 0, st>>>(
      shape, start, list, list_n, cursor, rows, contrib, d, ranges, split.range_rows);
  launch_backward_rows<false>(nt, feat, shape, start, loc, weights, grad_out, nullptr, grad_loc,
                              grad_weights, d, 0, st);
  const int per_entry = (d.feat + split.sum_rows - 1) / split.sum_rows;
  auto sum = [&](auto slots) {
    dfa::dfa_sum_rows<decltype(slots)::value><<<d.batch * per_entry, dfa::kBlock, 0, st>>>(
        weights, grad_out, rows, contrib, grad_feat, d, per_entry, split.sum_rows);
  };
  switch (nt) {
    case 1: sum(std::integral_constant<int, 1>()); break;
    case 2: sum(std::integral_constant<int, 2>()); break;
    case 3: sum(std::integral_constant<int, 3>()); break;
    default: sum(std::integral_constant<int, 4>()); break;
  }
  return check_launch(fn);
}

}  // namespace

extern "C" {

int deformable_aggregation_forward_opt(const float *mc_ms_feat, const int32_t *spatial_shape,
                                       const int32_t *scale_start_index,
                                       const float *sampling_location, const float *weights,
                                       float *output, int64_t batch, int64_t num_cams,
                                       int64_t num_feat, int64_t num_embeds, int64_t num_scale,
                                       int64_t num_anchors, int64_t num_pts, int64_t num_groups,
                                       void *stream) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  return forward_impl("deformable_aggregation_forward_opt", true, mc_ms_feat, spatial_shape,
                      scale_start_index, sampling_location, weights, output, a, stream);
}

int deformable_aggregation_forward_base(const float *mc_ms_feat, const int32_t *spatial_shape,
                                        const int32_t *scale_start_index,
                                        const float *sampling_location, const float *weights,
                                        float *output, int64_t batch, int64_t num_cams,
                                        int64_t num_feat, int64_t num_embeds, int64_t num_scale,
                                        int64_t num_anchors, int64_t num_pts, int64_t num_groups,
                                        void *stream) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  return forward_impl("deformable_aggregation_forward_base", false, mc_ms_feat, spatial_shape,
                      scale_start_index, sampling_location, weights, output, a, stream);
}

int deformable_aggregation_backward_opt(
    const float *mc_ms_feat, const int32_t *spatial_shape, const int32_t *scale_start_index,
    const float *sampling_location, const float *weights, const float *grad_output,
    float *grad_mc_ms_feat, float *grad_sampling_location, float *grad_weights, int64_t batch,
    int64_t num_cams, int64_t num_feat, int64_t num_embeds, int64_t num_scale,
    int64_t num_anchors, int64_t num_pts, int64_t num_groups, void *stream) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  return backward_impl("deformable_aggregation_backward_opt", true, mc_ms_feat, spatial_shape,
                       scale_start_index, sampling_location, weights, grad_output,
                       grad_mc_ms_feat, grad_sampling_location, grad_weights, a, stream);
}

size_t deformable_aggregation_backward_workspace_size(int64_t batch, int64_t num_cams,
                                                      int64_t num_feat, int64_t num_embeds,
                                                      int64_t num_scale, int64_t num_anchors,
                                                      int64_t num_pts, int64_t num_groups) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  dfa::Dims d;
  OwnerWorkspace w;
  if (validate("deformable_aggregation_backward_workspace_size", a, d) != 0) return 0;
  if (static_cast<int64_t>(d.batch) * d.anchors * d.pts * d.cams == 0) return 0;
  return plan_owner(d, w) ? w.bytes : 0;
}

int deformable_aggregation_backward_prefers_workspace(int64_t batch, int64_t num_cams,
                                                      int64_t num_feat, int64_t num_embeds,
                                                      int64_t num_scale, int64_t num_anchors,
                                                      int64_t num_pts, int64_t num_groups) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  dfa::Dims d;
  OwnerWorkspace w;
  if (validate("deformable_aggregation_backward_prefers_workspace", a, d) != 0) return 0;
  if (static_cast<int64_t>(d.batch) * d.anchors * d.pts * d.cams == 0) return 0;
  return plan_owner(d, w) && owner_is_faster(d) ? 1 : 0;
}

int deformable_aggregation_backward_ws(
    const float *mc_ms_feat, const int32_t *spatial_shape, const int32_t *scale_start_index,
    const float *sampling_location, const float *weights, const float *grad_output,
    float *grad_mc_ms_feat, float *grad_sampling_location, float *grad_weights, int64_t batch,
    int64_t num_cams, int64_t num_feat, int64_t num_embeds, int64_t num_scale,
    int64_t num_anchors, int64_t num_pts, int64_t num_groups, void *workspace,
    size_t workspace_bytes, void *stream) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  return backward_ws_impl("deformable_aggregation_backward_ws", mc_ms_feat, spatial_shape,
                          scale_start_index, sampling_location, weights, grad_output,
                          grad_mc_ms_feat, grad_sampling_location, grad_weights, a, workspace,
                          workspace_bytes, stream);
}

int deformable_aggregation_backward_base(
    const float *mc_ms_feat, const int32_t *spatial_shape, const int32_t *scale_start_index,
    const float *sampling_location, const float *weights, const float *grad_output,
    float *grad_mc_ms_feat, float *grad_sampling_location, float *grad_weights, int64_t batch,
    int64_t num_cams, int64_t num_feat, int64_t num_embeds, int64_t num_scale,
    int64_t num_anchors, int64_t num_pts, int64_t num_groups, void *stream) {
  const DfaArgs a{batch, num_cams, num_feat, num_embeds, num_scale, num_anchors, num_pts,
                  num_groups};
  return backward_impl("deformable_aggregation_backward_base", false, mc_ms_feat, spatial_shape,
                       scale_start_index, sampling_location, weights, grad_output,
                       grad_mc_ms_feat, grad_sampling_location, grad_weights, a, stream);
}

}  // extern "C"
