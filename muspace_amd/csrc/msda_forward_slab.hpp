// MSDA forward with a slab's coarse levels in LDS (gfx950).
//
// The forward row kernel gathers every corner row from L2 and runs at the
// rate L2 serves 128-byte lines (msda_kernels.hpp). Every level takes the same
// number of samples, however few cells it has, so the small levels of a
// pyramid take as many gathers as the large ones: at the BEVFormer SCA shape
// the two smallest of four levels are 6% of the cells and half of the samples.
// Here a workgroup works on one (b, m) slab, copies the rows of the levels
// that fit (a suffix of the levels: the coarsest ones) into LDS once, and
// gathers those from there, so L2 serves only the fine levels.
//
// A stage must then be all-LDS or all-L2 for a wavefront, so a unit's samples
// are walked in order by one lane group (the row kernel spreads them over
// several): the NG = 64/KQ lane groups of a wavefront take NG consecutive
// queries, a pass computes the taps of NS samples of each, one per lane, and a
// stage gathers and sums NH of them. No sums over lane groups are left.
//
// Measured against the row kernel, the kernel alone over and over with its value
// warm in the caches (8 heads x 32 channels; the LDS levels' share of the samples in
// brackets): the SCA shape (6 x 10000 queries, 4
// levels x 8 points) fp32 [1/4] 365 -> 325 us, bf16 [1/2] 313 -> 227 us; twice
// the batch, 15000 queries, bf16 860 -> 697 us; the encoder shape (2 x 22223, 4
// levels x 4 points) fp32 [1/4] 145 -> 99 us, fp16 [1/2] 105 -> 78 us; 3 x 10007
// queries on three levels, fp16 [2/3] 73 -> 52 us; one 200 x 200 level (no LDS
// level; 4 wavefronts a workgroup) fp32 106 -> 83 us, bf16 93 -> 72 us. In a program's
// calls, with other inputs and other kernels between, it takes 246 us at the bf16 SCA
// shape, 746 at twice the batch, 117 at the encoder and 105 on the one level. What is
// left is the fine levels' gathers from L2 (46 M lines in 325 us at the SCA
// shape in fp32), and in bf16 the decode and multiply-adds (about 137 us of VALU
// there). On the way: geometry loads marked non-temporal cost 4-30% (a pass
// reads a part of each line); persistent workgroups walking slabs were slower
// (405 us at the SCA shape: workgroups drift, and the dispatcher's order
// balances them).
#pragma once

#include "msda_kernels.hpp"

namespace msda {

// Shape of the slab kernel per value type and channels, for workgroups of W
// wavefronts (8, or 4 and two workgroups a CU). TS: stages per pass.
template <typename VT, int C, int W>
struct SlabCfg {
  static constexpr int kBlock = W * kWave;
  static constexpr int CPL = RowTraits<VT>::kCpl;
  static constexpr int KQ = C / CPL, NG = kWave / KQ;
  static constexpr int NS = KQ < 8 ? KQ : 8;    // samples of a unit per pass
  static constexpr int TS = NS >= 8 ? 2 : 1;    // stages per pass
  static constexpr int NH = NS / TS;            // samples per stage
  static constexpr int TW = NG * (NS + 1);      // tap table entries per wavefront (one pads a group)
  static constexpr int kRowBytes = C * static_cast<int>(sizeof(VT));
  // tap tables (by pass parity), then the LDS rows, the first of them zero
  static constexpr int kTapBytes = 2 * W * TW * 32;
  static constexpr int kValueBytes = 160 * 1024 / (8 / W) - 4096 - kTapBytes;
  static constexpr int kCells = kValueBytes / kRowBytes - 1;
  static constexpr size_t kLds = kTapBytes + static_cast<size_t>(kCells + 1) * kRowBytes;
};

// A slab's queries are cut into chunks of chunk_q, one workgroup each.
struct SlabPlan {
  int chunk_q;
};

// N consecutive geometry elements, loaded by the widest instructions.
template <typename GT, int N>
__device__ __forceinline__ void load_run(const GT *p, float (&o)[N]) {
  typedef GT Run __attribute__((ext_vector_type(N), aligned(sizeof(GT))));
  const Run r = *reinterpret_cast<const Run *>(p);
#pragma unroll
  for (int i = 0; i < N; ++i) o[i] = r[i];
}
template <typename GT, int N>
__device__ __forceinline__ void load_run16(const GT *p, float (&o)[N]) {
  typedef uint16_t Run __attribute__((ext_vector_type(N), aligned(2)));
  const Run r = *reinterpret_cast<const Run *>(p);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    GT v;
    const uint16_t bits = r[i];
    __builtin_memcpy(&v, &bits, 2);
    o[i] = to_float(v);
  }
}

// EP: consecutive samples of a unit per lane and geometry load (1: any L*P; 2 or
// 4: L*P a multiple of it). A block is NS * EP samples of each of the
// wavefront's units: lane tj of a unit holds samples tj * EP .. of it, and pass e
// takes the e-th of every lane.
//
// Out: DenseRows, or CameraSlots, whose logical blocks are cut into one segment
// per camera (CameraSlots::segment), each camera's valid rows being its slabs'
// queries.
template <typename VT, typename GT, int C, int W, int EP, typename Out>
__global__ void __launch_bounds__(W * kWave, kRowWavesPerSimd)
    msda_forward_slab(const VT *__restrict__ value, uint32_t value_bytes,
                      const int64_t *__restrict__ shapes, const int64_t *__restrict__ starts,
                      const GT *__restrict__ loc, const GT *__restrict__ attn, Out all,
                      Shape s, SlabPlan plan) {
  using Cfg = SlabCfg<VT, C, W>;
  constexpr int CPL = Cfg::CPL, KQ = Cfg::KQ, NG = Cfg::NG, NS = Cfg::NS, TS = Cfg::TS,
                NH = Cfg::NH, TW = Cfg::TW, RB = Cfg::kRowBytes;
  constexpr int VB = static_cast<int>(sizeof(VT));
  static_assert(NG * NS <= kWave && NS % TS == 0, "one tap per lane");
  extern __shared__ __align__(16) unsigned char slab_dyn[];
  __shared__ Level lv[kMaxLevels];
  __shared__ int lds_cell[kMaxLevels + 1];  // first LDS row of each level; [levels]: first LDS level
  u32x4 *tap_off = reinterpret_cast<u32x4 *>(slab_dyn);
  float4 *tap_w = reinterpret_cast<float4 *>(tap_off + 2 * W * TW);
  unsigned char *rows = slab_dyn + Cfg::kTapBytes;  // row 0 is zero
  stage_levels(lv, shapes, starts, s);

  int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const Out out = all.segment(lb, s);  // narrows s.queries to the camera's rows
  const int chunks = (s.queries + plan.chunk_q - 1) / plan.chunk_q;
  const int bm = lb / chunks, ch = lb % chunks;
  const int b = bm / s.heads, m = bm % s.heads;
  const int q0 = ch * plan.chunk_q, q1 = min(s.queries, q0 + plan.chunk_q);
  // geometry row of query 0 (query q: q * heads further) and first value row
  int row0;
  size_t cell0;
  out.locate(b, 0, m, s, row0, cell0);
  const int MC = s.heads * C;
  const uint32_t row_bytes = static_cast<uint32_t>(MC * VB);
  const uint32_t slab = static_cast<uint32_t>((cell0 * MC + m * C) * VB);
  const __amdgpu_buffer_rsrc_t vr = make_rsrc(value, value_bytes);

  if (threadIdx.x == 0) {
    int first = s.levels, at = 1;
    while (first > 0 && at + lv[first - 1].h * lv[first - 1].w <= Cfg::kCells + 1) {
      --first;
      lds_cell[first] = at;
      at += lv[first].h * lv[first].w;
    }
    lds_cell[s.levels] = first;
  }
  __syncthreads();
  const int first_lds = __builtin_amdgcn_readfirstlane(lds_cell[s.levels]);
  const int global_samples = first_lds * s.points;  // samples [0, this) come from L2
  for (int i = threadIdx.x; i < KQ; i += Cfg::kBlock) {
    reinterpret_cast<u32x4 *>(rows)[i] = u32x4{0u, 0u, 0u, 0u};
  }
  for (int l = first_lds; l < s.levels; ++l) {
    const int n = lv[l].h * lv[l].w * KQ;
    const uint32_t src = slab + static_cast<uint32_t>(lv[l].start) * row_bytes;
    u32x4 *dst = reinterpret_cast<u32x4 *>(rows + lds_cell[l] * RB);
    constexpr int U = 8;
    for (int i0 = threadIdx.x; i0 < n; i0 += U * Cfg::kBlock) {
      u32x4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(i0 + u * Cfg::kBlock, n - 1);
        v[u] = buffer_load16(vr, src + static_cast<uint32_t>(i / KQ) * row_bytes +
                                     static_cast<uint32_t>(i % KQ) * 16u);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + u * Cfg::kBlock;
        if (i < n) dst[i] = v[u];
      }
    }
  }
  __syncthreads();

  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int grp = lane / KQ, k = lane % KQ;
  const int tg = min(lane / NS, NG - 1), tj = lane % NS;  // this lane's taps: unit tg
  const int my_entry = wave * TW + tg * (NS + 1) + tj;
  const int grp_entry = wave * TW + grp * (NS + 1);
  const int nblk = (s.lp + NS * EP - 1) / (NS * EP);  // blocks per unit
  const int iters = (q1 - q0 + W * NG - 1) / (W * NG);
  const int total = iters * nblk;

  // geometry of this lane's EP samples of a block
  struct Geometry {
    float xy[2 * EP], a[EP];
    int smp;  // the first sample
    bool ok;  // in the chunk and below L*P
  };
  int gb = 0, gq = q0 + wave * NG + tg;  // the next block to load, and its query
  auto load_geometry = [&]() __attribute__((always_inline)) {
    Geometry g;
    const int smp = gb * NS * EP + tj * EP;
    const bool ok = gq < q1 && lane < NG * NS && smp < s.lp;
    g.smp = smp;
    g.ok = ok;
    const size_t o =
        static_cast<size_t>(row0 + (ok ? gq : 0) * s.heads) * s.lp + (ok ? smp : 0);
    if constexpr (sizeof(GT) == 4) {
      load_run<GT>(loc + 2 * o, g.xy);
      if constexpr (EP == 1) {
        g.a[0] = attn[o];
      } else {
        load_run<GT>(attn + o, g.a);
      }
    } else {
      load_run16<GT>(loc + 2 * o, g.xy);
      if constexpr (EP == 1) {
        g.a[0] = to_float(attn[o]);
      } else {
        load_run16<GT>(attn + o, g.a);
      }
    }
    if (++gb == nblk) {
      gb = 0;
      gq += W * NG;
    }
    return g;
  };
  // this lane's tap of its e-th sample into table `par`
  auto tap = [&](const Geometry &g, int e, int par) __attribute__((always_inline)) {
    const bool ok = g.ok;
    // a unit past the chunk keeps its sample's place: consume picks LDS or L2 by it
    const int smp = min(g.smp + e, s.lp - 1);
    const int l = level_of_sample(smp, s);
    const Level L = lv[l];
    const Tap t = make_tap(g.xy[2 * e], g.xy[2 * e + 1], L, ok);
    const float ai = ok ? g.a[e] : 0.0f;
    const bool lds = smp >= global_samples;
    const uint32_t unit = lds ? static_cast<uint32_t>(RB) : row_bytes;
    const uint32_t base = lds ? static_cast<uint32_t>(lds_cell[l] * RB)
                              : slab + static_cast<uint32_t>(L.start) * row_bytes;
    const uint32_t none = lds ? 0u : kOobOffset;
    const uint32_t c00 = base + static_cast<uint32_t>(t.cell00) * unit;
    const uint32_t c10 = c00 + static_cast<uint32_t>(L.w) * unit;
    if (lane < NG * NS) {
      u32x4 off;
      off.x = t.y0ok && t.x0ok ? c00 : none;
      off.y = t.y0ok && t.x1ok ? c00 + unit : none;
      off.z = t.y1ok && t.x0ok ? c10 : none;
      off.w = t.y1ok && t.x1ok ? c10 + unit : none;
      tap_off[par * W * TW + my_entry] = off;
      tap_w[par * W * TW + my_entry] =
          make_float4(ai * (t.wy0 * t.wx0), ai * (t.wy0 * t.wx1), ai * (t.wy1 * t.wx0),
                      ai * (t.wy1 * t.wx1));
    }
  };
  // Samples of stage h of pass (block bk of its unit, e): sample index of the
  // stage's j-th; uniform, so what a sample gathers from is a scalar branch.
  // A sample past L*P is skipped; a unit past the chunk has zero weights and
  // reads zeros: the zero row of the LDS, or past the value buffer's end.
  auto sample_of = [&](int bk, int e, int h, int j) {
    return bk * NS * EP + (h * NH + j) * EP + e;
  };
  const uint32_t ch16 = static_cast<uint32_t>(k * 16);
  const int l2_samples = min(global_samples, s.lp);
  auto gather = [&](const u32x4 &off, u32x4 (&r)[4]) __attribute__((always_inline)) {
    r[0] = buffer_load16(vr, off.x + ch16);
    r[1] = buffer_load16(vr, off.y + ch16);
    r[2] = buffer_load16(vr, off.z + ch16);
    r[3] = buffer_load16(vr, off.w + ch16);
  };
  auto issue = [&](int bk, int e, int h, int par, u32x4 (&raw)[NH][4]) __attribute__((always_inline)) {
    const int at = par * W * TW + grp_entry + h * NH;
    if (sample_of(bk, e, h, NH - 1) < l2_samples) {  // the whole stage
#pragma unroll
      for (int j = 0; j < NH; ++j) gather(tap_off[at + j], raw[j]);
    } else if (sample_of(bk, e, h, 0) < l2_samples) {  // a part of it
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        if (sample_of(bk, e, h, j) < l2_samples) gather(tap_off[at + j], raw[j]);
      }
    }
  };
  // float32 sums a unit in four chains (by pass parity and stage), as long as
  // those of the row kernel's lane groups; one chain of a unit's 32 samples
  // raised the error against 64 bits from 8.4e-8 to 1.2e-7. In 16 bits the
  // result's own rounding is 2e-4 and more: with two chains the error against 64
  // bits agrees in five digits at 256 samples a unit (fp16 2.0795e-4, bf16
  // 1.6583e-3).
  constexpr int kChains = std::is_same<VT, float>::value ? 2 * TS : 1;
  float acc[kChains][CPL];
#pragma unroll
  for (int i = 0; i < kChains; ++i) {
#pragma unroll
    for (int c = 0; c < CPL; ++c) acc[i][c] = 0.0f;
  }
  auto add = [&](const u32x4 (&r)[4], const float4 &w, float (&sum)[CPL])
      __attribute__((always_inline)) {
    float v0[CPL], v1[CPL], v2[CPL], v3[CPL];
    decode16(VT(), r[0], v0);
    decode16(VT(), r[1], v1);
    decode16(VT(), r[2], v2);
    decode16(VT(), r[3], v3);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      sum[c] += w.x * v0[c] + w.y * v1[c] + w.z * v2[c] + w.w * v3[c];
    }
  };
  const unsigned char *mine = rows + ch16;
  auto add_lds = [&](int at, float (&sum)[CPL]) __attribute__((always_inline)) {
    const u32x4 off = tap_off[at];
    u32x4 r[4];
    r[0] = *reinterpret_cast<const u32x4 *>(mine + off.x);
    r[1] = *reinterpret_cast<const u32x4 *>(mine + off.y);
    r[2] = *reinterpret_cast<const u32x4 *>(mine + off.z);
    r[3] = *reinterpret_cast<const u32x4 *>(mine + off.w);
    add(r, tap_w[at], sum);
  };
  auto consume = [&](int bk, int e, int h, int par, const u32x4 (&raw)[NH][4]) __attribute__((always_inline)) {
    const int at = par * W * TW + grp_entry + h * NH;
    const int lo = sample_of(bk, e, h, 0), hi = sample_of(bk, e, h, NH - 1);
    float(&sum)[CPL] = acc[kChains > 1 ? par * TS + h : 0];
    if (hi < l2_samples) {
#pragma unroll
      for (int j = 0; j < NH; ++j) add(raw[j], tap_w[at + j], sum);
    } else if (lo >= l2_samples && hi < s.lp) {
#pragma unroll
      for (int j = 0; j < NH; ++j) add_lds(at + j, sum);
    } else {
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        const int smp = sample_of(bk, e, h, j);
        if (smp < l2_samples) {
          add(raw[j], tap_w[at + j], sum);
        } else if (smp < s.lp) {
          add_lds(at + j, sum);
        }
      }
    }
  };
  int oq = q0 + wave * NG + grp;  // the unit being summed
  // its epilogue's data (CameraSlots: BEV query and count), the next unit's
  // query ahead of it
  typename Out::Ticket tk, tk_next;
  auto fetch_index = [&](typename Out::Ticket &t, int q) __attribute__((always_inline)) {
    out.fetch_index(t, min(q, s.queries - 1));
  };
  fetch_index(tk, oq);
  out.fetch_count(tk, b, s);
  fetch_index(tk_next, oq + W * NG);
  auto store_unit = [&]() __attribute__((always_inline)) {
    float sum[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      sum[c] = acc[0][c];
      if constexpr (kChains == 4) {
        sum[c] = (acc[0][c] + acc[1][c]) + (acc[2][c] + acc[3][c]);
      } else if constexpr (kChains == 2) {
        sum[c] = acc[0][c] + acc[1][c];
      }
    }
    if (oq < q1) out.template put<C, CPL>(b, oq, m, k, sum, tk, s);
#pragma unroll
    for (int i = 0; i < kChains; ++i) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) acc[i][c] = 0.0f;
    }
    oq += W * NG;
    tk = tk_next;
    out.fetch_count(tk, b, s);
    fetch_index(tk_next, oq + W * NG);
  };

  // Software pipeline over passes: while a pass's gathers are consumed, those of
  // its second stage or of the next pass are in flight, and the geometry of the
  // block after next is being loaded.
  u32x4 raw0[NH][4], raw1[NH][4];
  Geometry cur = load_geometry();
  Geometry nxt = load_geometry();
  tap(cur, 0, 0);
  issue(0, 0, 0, 0, raw0);
  int bk = 0;
  // pass e of block bk in table and (TS == 1) raw set `par`; then pass e2 of
  // block bk2 with geometry g2 is set up
  auto pass = [&](auto par_c, int e, const Geometry &g2, int bk2, int e2, auto &&between) __attribute__((always_inline)) {
    constexpr int par = decltype(par_c)::value;
    if constexpr (TS == 2) {
      issue(bk, e, 1, par, raw1);
      consume(bk, e, 0, par, raw0);
      tap(g2, e2, par ^ 1);
      issue(bk2, e2, 0, par ^ 1, raw0);
      between();
      consume(bk, e, 1, par, raw1);
    } else {
      tap(g2, e2, par ^ 1);
      if constexpr (par == 0) {
        issue(bk2, e2, 0, 1, raw1);
        between();
        consume(bk, e, 0, 0, raw0);
      } else {
        issue(bk2, e2, 0, 0, raw0);
        between();
        consume(bk, e, 0, 1, raw1);
      }
    }
  };
  auto nothing = [] {};
  auto advance = [&]() __attribute__((always_inline)) {
    cur = nxt;
    nxt = load_geometry();
  };
  std::integral_constant<int, 0> even;
  std::integral_constant<int, 1> odd;
  auto next_block = [&] { return bk + 1 == nblk ? 0 : bk + 1; };
  auto end_block = [&]() __attribute__((always_inline)) {
    if (bk + 1 == nblk) store_unit();
    bk = next_block();
  };
  if constexpr (EP == 1) {
    for (int i = 0; i < total; i += 2) {  // past the last block: nothing is stored
      pass(even, 0, nxt, next_block(), 0, advance);
      end_block();
      pass(odd, 0, nxt, next_block(), 0, advance);
      end_block();
    }
  } else {
    for (int i = 0; i < total; ++i) {
#pragma unroll
      for (int e = 0; e < EP; e += 2) {
        pass(even, e, cur, bk, e + 1, nothing);
        if (e + 2 < EP) {
          pass(odd, e + 1, cur, bk, e + 2, nothing);
        } else {
          pass(odd, e + 1, nxt, next_block(), 0, advance);
        }
      }
      end_block();
    }
  }
}

}  // namespace msda
