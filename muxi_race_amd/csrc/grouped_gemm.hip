// Grouped expert GEMMs for gfx950: Stage 1 (gate/up + SiLU*up) and Stage 2
// (down projection * routing weight) on fp16 MFMA (v_mfma_f32_32x32x16_f16),
// int8 MFMA (v_mfma_i32_32x32x32_i8) or fp8 MFMA (v_mfma_f32_32x32x64_f8f6f4,
// OCP e4m3).
//
// Reference algorithm: 初审材料/源代码/submission.py Stage1 family (:136-247,
// :1391-1635) and Stage2 family (:655-795, :1132-1378); base form
// xpuoj_data/submission.py:31-129 and :253-331.  The tiling here is this
// build's own.  One workgroup per item:
//   - narrow items of at most 32 token rows (4 waves, two workgroups per CU)
//     for decode-sized batches;
//   - wide items of up to 288 token rows (8 waves) otherwise: an expert's rows
//     are split evenly over as few items as hold them (moe_common.h Item).
// K advances 128 bytes per step through rings of XOR-swizzled LDS tiles filled
// by direct global->LDS loads (global_load_lds_dwordx4), so the loads of later
// steps stay in flight behind the MFMAs of the current one, with one barrier
// per step.
#include "launch.h"
#include "moe_common.h"

#include <type_traits>

namespace moe {

// out[0..3] += v (two packed fp16 atomic adds; no return value)
__device__ __forceinline__ void atomic_add_f16x4(_Float16* out, f16x4 v) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  typedef __attribute__((address_space(1))) h2 GlobalH2;
  GlobalH2* p = (GlobalH2*)(uintptr_t)out;
  __builtin_amdgcn_global_atomic_fadd_v2f16(p, h2{v[0], v[1]});
  __builtin_amdgcn_global_atomic_fadd_v2f16(p + 1, h2{v[2], v[3]});
#else
  (void)out;
  (void)v;
#endif
}

// Runs f(std::integral_constant<int, NB>) with NB = min(live, MAX), live >= 0:
// the K loops are instantiated per count of live 32-row token blocks.
template <int MAX, typename F>
__device__ __forceinline__ void with_live(int live, F&& f) {
  if constexpr (MAX == 0) {
    f(std::integral_constant<int, 0>{});
  } else {
    if (live >= MAX) f(std::integral_constant<int, MAX>{});
    else with_live<MAX - 1>(live, f);
  }
}

constexpr int kLdsBytes = 160 * 1024;  // LDS of a CU

// The E8M0 scale bytes of one h row for 16 K steps (fp8 Stage 2), held in four
// registers and shifted right one byte per step: the MFMA reads byte 0.
template <bool F8>
struct ScaleBytes {
  uint32_t w[4];
  __device__ __forceinline__ void load(const uint8_t* row, int ks) {
    if constexpr (F8) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(row + ks);
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = v[i];
      // a use right here: the wait for this load sits beside it, not at the
      // MFMAs, where it would drain the ring every step
      asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
    }
  }
  __device__ __forceinline__ int byte0() const { return F8 ? (int)w[0] : 0; }
  __device__ __forceinline__ void next() {
    if constexpr (F8) {
#pragma unroll
      for (int i = 0; i < 3; ++i) w[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], 8);
      w[3] >>= 8;
    }
  }
};

// Stage 2's output tile (BN features wide) is assembled in LDS and stored as
// whole row segments, 16 bytes per lane.  In LDS, 16-byte chunk c of tile row
// r sits at chunk slot c ^ (r & 15): the 16 rows one 8-byte write instruction
// covers per half-wave land on 16 different slots, and a row's chunks, read 16
// at a time, on 16 different slots.
template <int BN>
__device__ __forceinline__ char* out_chunk(char* smem, int r, int c) {
  static_assert(BN % 128 == 0, "at least 16 chunks per row");
  return smem + r * (2 * BN) + 16 * (c ^ (r & 15));
}
template <int BN>
__device__ __forceinline__ void stage_out(char* smem, int r, int n, f16x4 v) {
  *reinterpret_cast<f16x4*>(out_chunk<BN>(smem, r, n >> 3) + 2 * (n & 7)) = v;
}
// Rows [0, rows) of the assembled tile to output rows first + r, columns n0 on.
template <int BN, int NW, bool FUSED>
__device__ __forceinline__ void store_rows(const Stage2Params& p, char* smem, int rows, int row0, int64_t first,
                                           int n0) {
  constexpr int kShift = BN == 256 ? 5 : 4;  // 16-byte chunks per row: BN / 8
  static_assert(BN == 8 << kShift, "");
  _Float16* o = reinterpret_cast<_Float16*>(p.out);
  for (int idx = threadIdx.x; idx < rows << kShift; idx += 64 * NW) {
    const int r = idx >> kShift, c = idx & ((1 << kShift) - 1);
    const u32x4 v = *reinterpret_cast<const u32x4*>(out_chunk<BN>(smem, r, c));
    if constexpr (FUSED && MOE_S2_SCATTER) {
      _Float16* dst = o + (int64_t)(p.sorted_ids[row0 + r] / p.topk) * p.H + n0 + 8 * c;
      atomic_add_f16x4(dst, __builtin_bit_cast(f16x4, u32x2{v[0], v[1]}));
      atomic_add_f16x4(dst + 4, __builtin_bit_cast(f16x4, u32x2{v[2], v[3]}));
    } else {
      *reinterpret_cast<u32x4*>(o + (first + r) * p.H + n0 + 8 * c) = v;
    }
  }
}

// Stage 1 (fp16, int8) for 32-row tiles with narrow gate / up tiles (BN = 64 or
// 32 features each): two or four times the items of the 128-wide tiles, for
// shapes with few items per CU (decode), where the last round of workgroups
// would otherwise stream on a fraction of the CUs.  Each of the 4 waves owns
// one 32 x 32 accumulator: gate (waves 0, 1) or up (waves 2, 3), and
//   BN = 64: features 32 * (w & 1) of the tile, all 4 K sub-steps of a step;
//   BN = 32: all 32 features, K sub-steps 2 * (w & 1) and 2 * (w & 1) + 1,
//            the two halves summed in the epilogue.
// The other accumulators reach the wave writing h through LDS (int8: as exact
// int32 sums, so h has the bits that the 128-wide tiles give).
// int8 ran the 128-wide tiles here until this kernel took it: one workgroup
// per CU, weights under the default cache policy, and at one token (6 experts,
// I 2048) 96 items on 256 CUs.  64 experts, H 7168, I 2048, top-6: 24 tokens
// 291 -> 254 us (5.8 -> 6.6 TB/s of weights), 129 tokens 321 -> 294, 1 token
// 54 -> 41.  fp8 keeps 128-wide items (it scales h per 128 columns) and gains
// from the non-temporal weights alone: 24 tokens 290 -> 268 us.
template <int BN, int S, int QT>
__global__ __launch_bounds__(256) void stage1_narrow_kernel(Stage1Params p) {
  constexpr int BM = 32, NW = 4;
  constexpr bool I8 = QT == kQI8;
  static_assert(QT != kQF8, "fp8 quantises h per 128-column tile: items must span 128 columns");
  using Acc = typename std::conditional<I8, i32x16, f32x16>::type;
  using Elem = typename std::conditional<I8, int, float>::type;
  static_assert(BN == 64 || BN == 32, "narrow tiles are 64 or 32 features wide");
  constexpr bool KSPLIT = BN == 32;
  constexpr int ROWS = BM + 2 * BN;  // stage rows: tokens, gate rows, up rows
  using LD = DmaTile<ROWS, NW>;
  constexpr int STAGE = ROWS * kRowBytes;
  static_assert(S >= 2 && S * STAGE <= kLdsBytes, "LDS ring exceeds the 160 KiB of a CU");
  static_assert(S * STAGE >= 4 * 16 * 64 * 4, "the epilogue exchange reuses the ring");
  __shared__ __attribute__((aligned(16))) char smem[S * STAGE];

  const int nt = (int)(p.I / BN);
  Work w;
  if (!schedule(blockIdx.x, p.gpo, p.E, BM, BN, nt, p.host_blocks, w)) return;
  const int e = w.e;
  const int row0 = w.row0;
  const int n0 = w.n0;
  int actual = p.gs[e] - (row0 - p.gpo[e]);
  actual = actual < 0 ? 0 : (actual > BM ? BM : actual);
  if (actual == 0) return;

  const int64_t kbytes = p.H * (I8 ? 1 : 2);
  const int nk = (int)(kbytes / kRowBytes);
  const bool sh = p.e_shared >= 0 && e == p.e_shared;  // the shared expert's own tensors, same row stride
  const char* gexp = sh ? p.wg_shared : p.wg + (int64_t)e * p.w_es;
  const char* uexp = sh ? p.wu_shared : p.wu + (int64_t)e * p.w_es;
  LD ld;
#pragma unroll
  for (int i = 0; i < LD::NI; ++i) {
    const int r = LD::row_of(i);
    const char* src;
    if (r < BM) {
      const int pid = r < actual ? p.sorted_ids[row0 + r] : 0;
      src = p.x + (int64_t)(pid / p.topk) * kbytes;
    } else if (r < BM + BN) {
      src = gexp + (int64_t)(n0 + r - BM) * p.w_ld;
    } else {
      src = uexp + (int64_t)(n0 + r - BM - BN) * p.w_ld;
    }
    ld.set(i, src);
  }

  const int wave = threadIdx.x >> 6;
  const int mat = wave >> 1;  // 0: gate, 1: up
  const int half = wave & 1;  // feature half (BN = 64) or K half (BN = 32)
  const int wr0 = BM + mat * BN + (KSPLIT ? 0 : 32 * half);
  constexpr int SUB = KSPLIT ? 2 : 4;    // K sub-steps per wave per step
  const int s0 = KSPLIT ? 2 * half : 0;  // first of them
  Acc acc = Acc{};
  // int8: the dequantisation scales of this lane's token row and features,
  // loaded before the K loop so that their latency hides behind it
  const int l = lane_id();
  const int fbase = KSPLIT ? 0 : 32 * half;  // the wave's first feature in the tile
  float sx = 0.0f;
  f32x4 sgv[4], suv[4];
  if constexpr (I8) {
    const int pid = p.sorted_ids[row0 + (l & 31)];
    sx = p.x_scale[(l & 31) < actual ? pid / p.topk : 0];
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const int64_t n = (int64_t)e * p.I + n0 + fbase + 8 * rg + 4 * (l >> 5);
      sgv[rg] = *reinterpret_cast<const f32x4*>(p.sg + n);
      suv[rg] = *reinterpret_cast<const f32x4*>(p.su + n);
    }
  }
  auto k_loop = [&](auto stream_c) {
    constexpr bool STREAM = decltype(stream_c)::value;
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
      if (s < nk) ld.template issue<STREAM, BM>(smem + s * STAGE, s);
    int cur = 0;
    for (int ks = 0; ks < nk; ++ks) {
      wait_stages<LD::NI, S - 2>(nk - 1 - ks);
      barrier_no_fence();
      if (ks + S - 1 < nk) ld.template issue<STREAM, BM>(smem + (cur == 0 ? S - 1 : cur - 1) * STAGE, ks + S - 1);
      const char* st = smem + cur * STAGE;
      cur = cur + 1 == S ? 0 : cur + 1;
      u32x4 xf[2], wf[2];
      xf[0] = frag(st, 0, s0);
      wf[0] = frag(st, wr0, s0);
#pragma unroll
      for (int s = 0; s < SUB; ++s) {
        const int b = s & 1;
        if (s + 1 < SUB) {
          xf[b ^ 1] = frag(st, 0, s0 + s + 1);
          wf[b ^ 1] = frag(st, wr0, s0 + s + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
        acc = mma(wf[b], xf[b], acc);
      }
    }
  };
  // weight rows no other item reads are streamed
  if (w.shared) k_loop(std::false_type{});
  else k_loop(std::true_type{});
  __syncthreads();  // every wave is done with the ring before LDS is reused

  // Accumulator register r of lane l holds the same (token, feature) in every
  // wave that covers the same features, so the hand-over is by (r, l):
  // slot(w, r) for the waves other than the one writing h.
  Elem* xs = reinterpret_cast<Elem*>(smem);
  auto slot = [&](int wv, int r) -> Elem& { return xs[(wv * 16 + r) * 64 + l]; };
  const bool writer = KSPLIT ? wave == 0 : mat == 0;
  if (!writer) {
#pragma unroll
    for (int r = 0; r < 16; ++r) slot(wave, r) = acc[r];
  }
  __syncthreads();
  if (writer) {
    const int m = l & 31;
    if (m < actual) {
      _Float16* hrow = reinterpret_cast<_Float16*>(p.h) + (int64_t)(row0 + m) * p.h_ld;
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int n = n0 + fbase + 8 * rg + 4 * (l >> 5);
        f16x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = 4 * rg + q;
          Elem g, u;
          if constexpr (KSPLIT) {  // waves: 0 gate k0, 1 gate k1, 2 up k0, 3 up k1
            g = acc[r] + slot(1, r);
            u = slot(2, r) + slot(3, r);
          } else {                 // waves: 0/1 gate halves, 2/3 up halves
            g = acc[r];
            u = slot(2 + half, r);
          }
          if constexpr (I8) v[q] = (_Float16)silu_mul(((float)g * sx) * sgv[rg][q], ((float)u * sx) * suv[rg][q]);
          else v[q] = (_Float16)silu_mul(g, u);
        }
        *reinterpret_cast<f16x4*>(hrow + n) = v;
      }
    }
  }
}

// Stage 1 (fp8) for 32-row tiles: 128 gate + 128 up features per item, because
// h takes one scale per 128 columns.  4 waves of 32 gate + 32 up features.  One
// workgroup fits a CU, so nothing else runs beside a wave that issues its nine
// loads of a step: half of them go before each half step's MFMAs (8 tokens, 16
// experts top-2, H 4096, I 2048: 29.0 -> 27.0 us with the policy known at compile time).
template <int S>
__global__ __launch_bounds__(256) void stage1_f8_kernel(Stage1Params p) {
  constexpr int BM = 32, NW = 4;
  constexpr int ROWS = BM + 2 * kBN;  // stage rows: tokens, gate rows, up rows
  using LD = DmaTile<ROWS, NW>;
  constexpr int STAGE = ROWS * kRowBytes;
  static_assert(S >= 2 && S * STAGE <= kLdsBytes, "LDS ring exceeds the CU's LDS");
  __shared__ __attribute__((aligned(16))) char smem[S * STAGE];

  Work w;
  if (!schedule(blockIdx.x, p.gpo, p.E, BM, kBN, (int)(p.I / kBN), p.host_blocks, w)) return;
  const int e = w.e, row0 = w.row0, n0 = w.n0;
  int actual = p.gs[e] - (row0 - p.gpo[e]);
  actual = actual < 0 ? 0 : (actual > BM ? BM : actual);
  if (actual == 0) return;

  const int nk = (int)(p.H / kRowBytes);
  const char* gexp = p.wg + (int64_t)e * p.w_es;
  const char* uexp = p.wu + (int64_t)e * p.w_es;
  LD ld;
#pragma unroll
  for (int i = 0; i < LD::NI; ++i) {
    const int r = LD::row_of(i);
    const char* src;
    if (r < BM) {
      const int pid = r < actual ? p.sorted_ids[row0 + r] : 0;
      src = p.x + (int64_t)(pid / p.topk) * p.H;
    } else if (r < BM + kBN) {
      src = gexp + (int64_t)(n0 + r - BM) * p.w_ld;
    } else {
      src = uexp + (int64_t)(n0 + r - BM - kBN) * p.w_ld;
    }
    ld.set(i, src);
  }
  // dequantisation scales of this lane's token row and features, loaded before
  // the K loop so that their latency hides behind it
  const int l = lane_id(), wn = threadIdx.x >> 6;
  const int pid = p.sorted_ids[row0 + (l & 31)];
  const float sx = p.x_scale[(l & 31) < actual ? pid / p.topk : 0];
  f32x4 sgv[4], suv[4];
#pragma unroll
  for (int rg = 0; rg < 4; ++rg) {
    const int64_t n = (int64_t)e * p.I + n0 + 32 * wn + 8 * rg + 4 * (l >> 5);
    sgv[rg] = *reinterpret_cast<const f32x4*>(p.sg + n);
    suv[rg] = *reinterpret_cast<const f32x4*>(p.su + n);
  }
  f32x16 ag = f32x16{}, au = f32x16{};
  const FragLane fl;
  auto k_loop = [&](auto stream_c) {
    constexpr bool STREAM = decltype(stream_c)::value;
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
      if (s < nk) ld.template issue<STREAM, BM>(smem + s * STAGE, s);
    int cur = 0;
    for (int ks = 0; ks < nk; ++ks) {
      wait_stages<LD::NI, S - 2>(nk - 1 - ks);
      barrier_no_fence();
      const bool more = ks + S - 1 < nk;
      char* next = smem + (cur == 0 ? S - 1 : cur - 1) * STAGE;
      const char* st = smem + cur * STAGE;
      cur = cur + 1 == S ? 0 : cur + 1;
      const uint32_t xb = row_base(st, 0), gb = row_base(st, BM + 32 * wn), ub = row_base(st, BM + kBN + 32 * wn);
      auto half = [&](auto j_c) {
        constexpr int j = decltype(j_c)::value;
        u32x4 xf[2], gf[2], uf[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          xf[q] = frag_at(xb, fl.off[2 * j + q]);
          gf[q] = frag_at(gb, fl.off[2 * j + q]);
          uf[q] = frag_at(ub, fl.off[2 * j + q]);
        }
        if (more) ld.template issue<STREAM, BM, j, 2>(next, ks + S - 1);
        __builtin_amdgcn_sched_barrier(0);
        ag = mma8(gf[0], gf[1], xf[0], xf[1], ag);
        au = mma8(uf[0], uf[1], xf[0], xf[1], au);
      };
      half(std::integral_constant<int, 0>{});
      half(std::integral_constant<int, 1>{});
    }
  };
  if (w.shared || !p.stream) k_loop(std::false_type{});
  else k_loop(std::true_type{});
  __syncthreads();  // every wave is done with the ring before LDS is reused

  // h = silu(g) * u, quantised per row over the item's 128 columns, which are
  // spread over the lane pair (l, l^32) and the 4 waves
  float* red = reinterpret_cast<float*>(smem);  // [NW][BM]
  const bool valid = (l & 31) < actual;
  float hv[16], amax = 0.0f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float x = valid ? sx : 0.0f;
    hv[r] = silu_mul((ag[r] * x) * sgv[r >> 2][r & 3], (au[r] * x) * suv[r >> 2][r & 3]);
    amax = fmaxf(amax, fabsf(hv[r]));
  }
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  if (l < 32) red[wn * BM + l] = amax;
  __syncthreads();
  amax = 0.0f;
#pragma unroll
  for (int j = 0; j < NW; ++j) amax = fmaxf(amax, red[j * BM + (l & 31)]);
  const int sb = pow2_scale_e8m0(amax);
  const float inv = amax > 0.0f ? scale_from_e8m0(254 - sb) : 0.0f;
  if (valid) {
    const int64_t row = row0 + (l & 31);
    uint8_t* hrow = reinterpret_cast<uint8_t*>(p.h) + row * p.h_ld;
#pragma unroll
    for (int rg = 0; rg < 4; ++rg)
      *reinterpret_cast<uint32_t*>(hrow + n0 + 32 * wn + 8 * rg + 4 * (l >> 5)) =
          quant_code4<true>(hv[4 * rg], hv[4 * rg + 1], hv[4 * rg + 2], hv[4 * rg + 3], inv);
    if (wn == 0 && l < 32) p.h_scale[row * p.hs_pitch + n0 / kBN] = (uint8_t)sb;
  }
}

// Stage 2 for 32-row tiles, 128 features per item: 4 waves of 32 features.
template <int S, int QT>
__global__ __launch_bounds__(256) void stage2_narrow_kernel(Stage2Params p) {
  constexpr bool I8 = QT == kQI8, F8 = QT == kQF8;
  using Acc = typename std::conditional<I8, i32x16, f32x16>::type;
  constexpr int BM = 32, NW = 4, BN = kBN;
  constexpr int ROWS = BM + BN;
  using LD = DmaTile<ROWS, NW>;
  constexpr int STAGE = ROWS * kRowBytes;
  static_assert(S >= 2 && S * STAGE <= kLdsBytes, "LDS ring exceeds the CU's LDS");
  __shared__ __attribute__((aligned(16))) char smem[S * STAGE];

  Work w;
  if (!schedule(blockIdx.x, p.gpo, p.E, BM, BN, (int)(p.H / BN), p.host_blocks, w)) return;
  const int e = w.e, row0 = w.row0, n0 = w.n0;
  const int gpo_e = p.gpo[e], go_e = p.go[e];
  int actual = p.gs[e] - (row0 - gpo_e);
  actual = actual < 0 ? 0 : (actual > BM ? BM : actual);
  if (actual == 0) return;

  const int nk = (int)(p.I * (QT == kQF16 ? 2 : 1) / kRowBytes);
  const char* dexp = p.e_shared >= 0 && e == p.e_shared ? p.wd_shared : p.wd + (int64_t)e * p.wd_es;
  LD ld;
#pragma unroll
  for (int i = 0; i < LD::NI; ++i) {
    const int r = LD::row_of(i);
    // token rows past the expert's count read the item's first row
    ld.set(i, r < BM ? p.a + (int64_t)(row0 + (r < actual ? r : 0)) * p.a_ld : dexp + (int64_t)(n0 + r - BM) * p.wd_ld);
  }
  const int wn = threadIdx.x >> 6, l = lane_id();
  const FragLane fl;
  const int m = l & 31;
  const bool valid = m < actual;
  const int pid = p.sorted_ids[row0 + m];  // row0 + m lies inside the padded block
  const int64_t first = (int64_t)go_e + (row0 - gpo_e);  // unpadded expert-sorted row of token row 0
  const float wr = reinterpret_cast<const float*>(p.routed)[valid ? pid : 0];
  if (valid && n0 == 0 && wn == 0 && l < 32) p.pos[pid] = (int32_t)(first + m);
  float sh = 1.0f;
  if constexpr (I8) sh = p.a_scale[row0 + (valid ? m : 0)];
  const uint8_t* sp = F8 ? p.a_scale8 + (int64_t)(row0 + (valid ? m : 0)) * p.as_pitch : nullptr;
  ScaleBytes<F8> sc;
  sc.load(sp, 0);
  Acc acc = Acc{};

  auto k_loop = [&](auto stream_c) {
    constexpr bool STREAM = decltype(stream_c)::value;
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
      if (s < nk) ld.template issue<STREAM, BM>(smem + s * STAGE, s);
    int cur = 0;
    for (int ks = 0; ks < nk; ++ks) {
      wait_stages<LD::NI, S - 2>(nk - 1 - ks);
      barrier_no_fence();
      if (ks + S - 1 < nk) ld.template issue<STREAM, BM>(smem + (cur == 0 ? S - 1 : cur - 1) * STAGE, ks + S - 1);
      const char* st = smem + cur * STAGE;
      cur = cur + 1 == S ? 0 : cur + 1;
      const uint32_t xb = row_base(st, 0), wb = row_base(st, BM + 32 * wn);
      u32x4 xf[2], wf[2];
      auto load_frags = [&](int buf, int q) {
        xf[buf] = frag_at(xb, fl.off[q]);
        wf[buf] = frag_at(wb, fl.off[q]);
      };
      load_frags(0, 0);
      if constexpr (F8) {
        if (ks > 0 && (ks & 15) == 0) sc.load(sp, ks);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          if (j > 0) load_frags(0, 2 * j);
          load_frags(1, 2 * j + 1);
          acc = mma8_scale_b(wf[0], wf[1], xf[0], xf[1], acc, sc.byte0());
        }
        sc.next();
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (q < 3) load_frags((q & 1) ^ 1, q + 1);
          __builtin_amdgcn_sched_barrier(0);
          acc = mma(wf[q & 1], xf[q & 1], acc);
        }
      }
    }
  };
  if (w.shared) k_loop(std::false_type{});
  else k_loop(std::true_type{});

  // The accumulators hold 4-feature runs of one token row; the tile is first
  // assembled in LDS and then stored as whole row segments (see store_rows).
  __syncthreads();
#pragma unroll
  for (int rg = 0; rg < 4; ++rg) {
    const int nl = 32 * wn + 8 * rg + 4 * (l >> 5);
    f32x4 sd = {1.0f, 1.0f, 1.0f, 1.0f};
    if constexpr (QT != kQF16) sd = *reinterpret_cast<const f32x4*>(p.sd + (int64_t)e * p.H + n0 + nl);
    f16x4 v;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float y = (float)acc[4 * rg + q];
      if constexpr (I8) y = y * sh;             // int8: ((acc * s_h[row]) * s_d[n]) * w
      if constexpr (QT != kQF16) y = y * sd[q];
      v[q] = (_Float16)(y * wr);
    }
    if (valid) stage_out<BN>(smem, m, nl, v);
  }
  __syncthreads();
  store_rows<BN, NW, true>(p, smem, actual, row0, first, n0);
}

// ---------------------------------------------------------------------------
// Wide items: 8 waves, up to 128 (kLowRows) or 256 (kWideRows) token rows, or
// 256 and up to 32 absorbed ones (fp16), against WR weight rows.
//
// Ring.  Token rows and weight rows have slots of their own, as many as fit:
// DT + 1 of TS bytes and DW + 1 of WS.  After step j's barrier the token rows
// of step j + DT and the weight rows of step j + DW are issued, the weight rows
// one instruction per K sub-step, so that no wave waits behind a long run of
// its own loads before its MFMAs.
//   256 weight rows: DT = 1 and DW = 3 (128 token rows) or 2 (256): the weight
//     rows (HBM misses) are two or three steps ahead, the token rows (L2 hits,
//     issued in one burst) one.  128 x 256 with DT = DW = 2 measured level.
//   ... with absorbed rows: DT = DW = 1, weights first, in one burst.
//   128 weight rows: DT = 2, DW = 3.  The steps are short: with DT = 1 a 256-row
//     item of reference case 1's Stage 2 took 1.45 us a step, with 2 1.05.
// Loads retire in order, so a step's rows are in LDS once at most the loads
// issued after them are outstanding; their number is exact but for an item's
// last steps, which wait for everything.
// What this bought over rings of whole stages (three of 48 KiB for 128 x 256
// items, two of 64 KiB for 256 x 256), dsv3's weights with every expert at 256
// rows, fp16: Stage 1 2087 -> 1970 us, Stage 2 1180 -> 1084; at 64 rows Stage 2
// 1420 -> 1264; mixtral's shape at 512 rows 964 -> 936 and 477 -> 448.
// In these loops the MFMAs are not the bound: with them (and the LDS reads)
// taken out of the whole-stage kernels, dsv3 at 4096 tokens gained 4% and
// int8 at 2048 tokens 9%; mixtral's step took the same 3500 cycles but at 2.38
// instead of 1.80 GHz.
//
// Token rows past the item's routed ones are not loaded beyond the last
// 64-row group that holds one; rows in that group read the item's first row.
// Their results are never stored.
// ---------------------------------------------------------------------------
template <int TR_, int WR_, bool ABS_>
struct Ring {
  static constexpr int TR = TR_, WR = WR_;
  static constexpr bool ABS = ABS_;
  static constexpr int TS = (TR + (ABS ? kAbsorbRows : 0)) * kRowBytes;
  static constexpr int WS = WR * kRowBytes;
  static constexpr int DT = WR == 256 ? 1 : 2;
  static constexpr int kFit = (kLdsBytes - (DT + 1) * TS) / WS;  // weight slots
  static constexpr int SW = kFit < 4 ? kFit : 4;
  static constexpr int DW = SW - 1;
  static constexpr int NIT = TR / 64, NIW = WR / 64;  // load instructions per wave and step
  static constexpr int BYTES = (DT + 1) * TS + SW * WS;
  static_assert(DT <= DW && BYTES <= kLdsBytes, "LDS ring exceeds the CU's LDS");
  static constexpr bool kBurst = DW == 1;          // one stage in flight: everything at once, weights first
  static constexpr bool kSpreadT = DT == DW && !kBurst;  // token loads are spread over the step too

  const char* t[NIT];   // this lane's 16 bytes of its token rows, K step 0
  const char* w[NIW];   // ... of its weight rows
  const char* a;        // ... of its absorbed row (waves 0-3 when there are any)
  int nt;               // token instructions with a routed row
  bool adma;            // this wave loads absorbed rows

  // slot row of instruction i: 8 rows per wave instruction
  __device__ __forceinline__ static int row_of(int i) { return 8 * (8 * i + wave_id()) + (lane_id() >> 3); }
  __device__ __forceinline__ static char* tslot(char* smem, int i) { return smem + i * TS; }
  __device__ __forceinline__ static char* wslot(char* smem, int i) { return smem + (DT + 1) * TS + i * WS; }

  // token instructions [i0, i1) (absorbed rows ride with the first)
  __device__ __forceinline__ void issue_t(char* slot, int k, int i0, int i1) const {
#pragma unroll
    for (int i = 0; i < NIT; ++i)
      if (i >= i0 && i < i1 && i < nt) dma_to_lds<16>(t[i] + (size_t)k * kRowBytes, slot + 1024 * (8 * i + wave_id()));
    if constexpr (ABS)
      if (i0 == 0 && adma) dma_to_lds<16>(a + (size_t)k * kRowBytes, slot + TR * kRowBytes + 1024 * wave_id());
  }
  // weight instructions [i0, i1); STREAM: non-temporal
  template <bool STREAM>
  __device__ __forceinline__ void issue_w(char* slot, int k, int i0, int i1) const {
#pragma unroll
    for (int i = 0; i < NIW; ++i)
      if (i >= i0 && i < i1)
        dma_to_lds<16, STREAM ? kPolicyWeights : kPolicyDefault>(w[i] + (size_t)k * kRowBytes,
                                                                slot + 1024 * (8 * i + wave_id()));
  }
  // Waits until step ks's rows are in LDS, full: the loads of every later step
  // that the loop has room for have been issued.
  __device__ __forceinline__ void wait(bool full) const {
    constexpr int kLater = (DT - 1 + (DT < DW ? 1 : 0)) * NIW;  // weight instructions issued after step ks's rows
    if (!full || kBurst) {
      wait_vmcnt<0>();
    } else if constexpr (DT == 1) {
      wait_vmcnt<kLater>();
    } else {  // and the token instructions of one step, nt (+ 1): a scalar choice
      wait_tokens<kLater, NIT + (ABS ? 1 : 0)>(nt + (ABS && adma ? 1 : 0));
    }
  }
  template <int W, int T>
  __device__ __forceinline__ static void wait_tokens(int n) {
    if constexpr (T == 0) {
      wait_vmcnt<W>();
    } else {
      if (n >= T) wait_vmcnt<W + T>();
      else wait_tokens<W, T - 1>(n);
    }
  }
};

// Wave placement: WM = TR / 64 waves along the tokens, each owning two 32-row
// blocks, and the rest along the weight rows.  Waves w and w + 4 share a SIMD.
// A wave owns blocks wm and wm + WM, so that an item of 192 rows gives every
// SIMD three of them per weight column, where two neighbouring blocks per wave
// gave two SIMDs four and two SIMDs two (64 experts, H 7168, I 2048: fp8 at 2048
// tokens 731 -> 715 us, int8 at 1000 tokens 554 -> 542).  Items with absorbed
// rows have all blocks full and keep neighbouring ones (measured 0.7% faster).
template <class R>
struct WaveGrid {
  static constexpr int WM = R::TR / 64, WN = 8 / WM;
  static constexpr int kStep = R::ABS ? 32 : 32 * WM;  // rows between a wave's two blocks
  int wm, wn;
  __device__ __forceinline__ WaveGrid() {
    const int wave = threadIdx.x >> 6;
    wm = wave / WN;
    wn = wave % WN;
  }
  __device__ __forceinline__ int x0() const { return (R::ABS ? 64 : 32) * wm; }  // first row of the first block
  // this wave's blocks that hold one of the first n rows
  __device__ __forceinline__ int live(int n) const {
    const int rows = n - x0();
    return rows <= 0 ? 0 : (rows <= kStep ? 1 : 2);
  }
};

// The K loop of one wave: acc[j][b] += weight block j x token block b for its
// NB live token blocks (instantiated per count, chosen outside the loop: a
// branch inside would move the accumulators out of AGPRs every step;
// padding-only blocks get no LDS reads and no MFMAs, and every variant issues
// the same loads and barriers).  Weight blocks [0, NWB / 2) are the 32-row
// blocks of the weight slot from row w0 on, the others those from w1 on.  A:
// also aa += the weight block at row wa x the absorbed rows.  SCB (fp8 Stage
// 2): token rows scaled by their E8M0 bytes at sp[b], one per step.
template <int QT, bool SCB, class R, bool STREAM, int NWB, int NB, bool A, class Acc>
__device__ __forceinline__ void wide_k_loop(const R& ring, int nk, char* smem, int x0, int w0, int w1, int wa,
                                            const FragLane& fl, Acc (&acc)[NWB][2], f32x16& aa,
                                            const uint8_t* const (&sp)[2]) {
  constexpr bool F8 = QT == kQF8;
  constexpr int DT = R::DT, DW = R::DW, SW = R::SW, NIW = R::NIW;
  constexpr bool kWork = NB > 0 || A;
  constexpr int kBlock = WaveGrid<R>::kStep * kRowBytes;  // LDS bytes between the wave's token blocks
  constexpr int kHalf = NWB > 1 ? NWB / 2 : 1;
  ScaleBytes<SCB> sc[2];
#pragma unroll
  for (int b = 0; b < NB; ++b) sc[b].load(sp[b], 0);
  // what iterations -DW .. -1 of the loop below would issue
#pragma unroll
  for (int j = -DW; j < 0; ++j) {
    if (R::kBurst) ring.template issue_w<STREAM>(R::wslot(smem, 0), 0, 0, NIW);
    if (j + DT >= 0 && j + DT < nk) ring.issue_t(R::tslot(smem, j + DT), j + DT, 0, R::NIT);
    if (!R::kBurst && j + DW < nk) ring.template issue_w<STREAM>(R::wslot(smem, j + DW), j + DW, 0, NIW);
  }
  int ct = 0, cw = 0;  // slots of step ks
  for (int ks = 0; ks < nk; ++ks) {
    ring.wait(ks + DW - 1 < nk);
    barrier_no_fence();
    const bool pt = ks + DT < nk, pw = ks + DW < nk;
    char* td = R::tslot(smem, ct == 0 ? DT : ct - 1);
    char* wd = R::wslot(smem, cw == 0 ? SW - 1 : cw - 1);
    const char* ts = R::tslot(smem, ct);
    const char* wsl = R::wslot(smem, cw);
    ct = ct == DT ? 0 : ct + 1;
    cw = cw + 1 == SW ? 0 : cw + 1;
    constexpr bool kSpread = !R::kBurst && kWork, kSpreadT = R::kSpreadT && kWork;
    if (R::kBurst && pw) ring.template issue_w<STREAM>(wd, ks + DW, 0, NIW);
    if (!kSpreadT && pt) ring.issue_t(td, ks + DT, 0, R::NIT);
    if (!R::kBurst && !kSpread && pw) ring.template issue_w<STREAM>(wd, ks + DW, 0, NIW);
    if constexpr (kWork) {
      // Fragments double-buffered across the 4 K sub-steps: the LDS reads of
      // sub-step s+1 are in flight while the MFMAs of sub-step s run.
      u32x4 xf[2][NB > 0 ? NB : 1], wf[2][NWB], xa[2], wfa[2];
      const uint32_t xb = row_base(ts, x0), b0 = row_base(wsl, w0), b1 = row_base(wsl, w1);
      const uint32_t xab = A ? row_base(ts, R::TR) : 0, wab = A ? row_base(wsl, wa) : 0;
      auto load_frags = [&](int buf, int s) {
#pragma unroll
        for (int b = 0; b < NB; ++b) xf[buf][b] = frag_at(xb + kBlock * b, fl.off[s]);
        if constexpr (NB > 0) {
#pragma unroll
          for (int j = 0; j < NWB; ++j)
            wf[buf][j] = frag_at(j < kHalf ? b0 + 4096 * j : b1 + 4096 * (j - kHalf), fl.off[s]);
        }
        if constexpr (A) {
          xa[buf] = frag_at(xab, fl.off[s]);
          wfa[buf] = frag_at(wab, fl.off[s]);
        }
      };
      if constexpr (F8) {
        if constexpr (SCB) {
          if (ks > 0 && (ks & 15) == 0) {
#pragma unroll
            for (int b = 0; b < NB; ++b) sc[b].load(sp[b], ks);
          }
        }
        // one MFMA per 64-byte half step, on the fragments of two sub-steps; the
        // weight blocks in two groups, so that one group's fragments are live
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int b = 0; b < NB; ++b) xf[q][b] = frag_at(xb + kBlock * b, fl.off[2 * h + q]);
          if (kSpreadT && pt) ring.issue_t(td, ks + DT, h * R::NIT / 2, (h + 1) * R::NIT / 2);
          if (kSpread && pw) ring.template issue_w<STREAM>(wd, ks + DW, h * NIW / 2, (h + 1) * NIW / 2);
#pragma unroll
          for (int j0 = 0; j0 < NWB; j0 += kHalf) {
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
              for (int j = 0; j < kHalf; ++j) wf[q][j] = frag_at((j0 ? b1 : b0) + 4096 * j, fl.off[2 * h + q]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < kHalf; ++j)
#pragma unroll
              for (int b = 0; b < NB; ++b) {
                Acc& c = acc[j0 + j][b];
                if constexpr (SCB) c = mma8_scale_b(wf[0][j], wf[1][j], xf[0][b], xf[1][b], c, sc[b].byte0());
                else c = mma8(wf[0][j], wf[1][j], xf[0][b], xf[1][b], c);
              }
          }
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) sc[b].next();
      } else {
        load_frags(0, 0);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int fb = s & 1;
          if (s < 3) load_frags(fb ^ 1, s + 1);
          if (kSpreadT && pt) ring.issue_t(td, ks + DT, s, s + 1);
          if (kSpread && pw && s < NIW) ring.template issue_w<STREAM>(wd, ks + DW, s, s + 1);
          __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of the MFMAs
#pragma unroll
          for (int j = 0; j < NWB; ++j)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[j][b] = mma(wf[fb][j], xf[fb][b], acc[j][b]);
          if constexpr (A) aa = mma(wfa[fb], xa[fb], aa);
        }
      }
    }
  }
}

// Stage 1 item: TR token rows (and absorbed ones) x 128 gate + 128 up rows.
template <int QT, bool GATHER, int TR, bool ABS, bool STREAM>
__device__ __forceinline__ void stage1_item(const Stage1Params& p, const Item& it, char* smem) {
  constexpr bool I8 = QT != kQF16, F8 = QT == kQF8;  // 8-bit operands with row scales
  using R = Ring<TR, 2 * kBN, ABS>;
  using G = WaveGrid<R>;
  using Acc = typename std::conditional<I8 && !F8, i32x16, f32x16>::type;
  constexpr int WTN = kBN / G::WN;  // gate (and up) features per wave
  constexpr int NBN = WTN / 32;     // gate (and up) blocks per wave
  static_assert(!ABS || NBN == 2, "absorbed rows: four weight blocks per wave column");
  const int e = it.e, row0 = it.row0, n0 = it.n0;
  const int actual = it.actual < TR ? it.actual : TR;
  const int nar = ABS ? it.actual - actual : 0;  // absorbed rows

  const int64_t kbytes = p.H * (I8 ? 1 : 2);
  const int nk = (int)(kbytes / kRowBytes);
  // this expert's [I, H] gate / up weights, experts w_es and rows w_ld bytes
  // apart (the shared expert's own tensors, same row stride)
  const bool sh = p.e_shared >= 0 && e == p.e_shared;
  const char* gexp = sh ? p.wg_shared : p.wg + (int64_t)e * p.w_es;
  const char* uexp = sh ? p.wu_shared : p.wu + (int64_t)e * p.w_es;
  auto token_row = [&](int row) { return p.x + (int64_t)(GATHER ? p.sorted_ids[row] / p.topk : row) * kbytes; };
  R ring;
  ring.nt = (actual + 63) / 64;
#pragma unroll
  for (int i = 0; i < R::NIT; ++i) {
    const int r = R::row_of(i);
    ring.t[i] = DmaTile<64, 8>::at(r, token_row(row0 + (r < actual ? r : 0)));
  }
#pragma unroll
  for (int i = 0; i < R::NIW; ++i) {
    const int r = R::row_of(i);
    ring.w[i] = DmaTile<64, 8>::at(r, r < kBN ? gexp + (int64_t)(n0 + r) * p.w_ld : uexp + (int64_t)(n0 + r - kBN) * p.w_ld);
  }
  // absorbed rows: waves 0-3 each load 8 of them (past nar: the item's first row)
  ring.adma = ABS && wave_id() < 4;
  if constexpr (ABS) {
    const int r = R::row_of(0);
    ring.a = DmaTile<64, 8>::at(r, token_row(row0 + (r < nar ? TR + r : 0)));
  }

  const G g;
  const int xr0 = g.x0();               // slot row of this wave's first token row
  const int gr0 = WTN * g.wn;           // ... first gate row; up rows follow the kBN gate rows
  const FragLane fl;
  const int l = lane_id();

  // 8-bit: the dequantisation scales of this lane's token rows and output
  // features, loaded before the K loop so that their latency hides behind it
  // (rows without a token read token 0's scale and are never stored).  The
  // feature scales stay in registers only for wave tiles of up to two 32x32
  // blocks; larger tiles load them in the epilogue (registers would spill).
  constexpr bool kHoistFeat = NBN == 1;
  const float* sgrow = I8 ? p.sg + (int64_t)e * p.I : nullptr;
  const float* surow = I8 ? p.su + (int64_t)e * p.I : nullptr;
  float sxv[2];
  f32x4 sgv[NBN][4], suv[NBN][4];
  if constexpr (I8) {
    int pid[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int m = xr0 + G::kStep * b + (l & 31);
      pid[b] = p.sorted_ids[row0 + (m < actual ? m : 0)];
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) sxv[b] = p.x_scale[pid[b] / p.topk];
    if constexpr (kHoistFeat) {
#pragma unroll
      for (int a = 0; a < NBN; ++a)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int n = n0 + gr0 + 32 * a + 8 * rg + 4 * (l >> 5);
          sgv[a][rg] = *reinterpret_cast<const f32x4*>(sgrow + n);
          suv[a][rg] = *reinterpret_cast<const f32x4*>(surow + n);
        }
    }
  }
  // acc[a]: gate block a, acc[NBN + a]: up block a
  Acc acc[2 * NBN][2];
#pragma unroll
  for (int a = 0; a < 2 * NBN; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = Acc{};
  // absorbed rows x one weight block of this wave: gate blocks 0, 1 for wm =
  // 0, 1, up blocks 0, 1 for wm = 2, 3
  f32x16 aa = {};
  const bool agate = g.wm < 2;
  const int aj = g.wm & 1;
  const int awr0 = (agate ? gr0 : kBN + gr0) + 32 * aj;
  const uint8_t* const no_scale[2] = {nullptr, nullptr};
  with_live<2>(g.live(actual), [&](auto nb_c) {
    wide_k_loop<QT, false, R, STREAM, 2 * NBN, decltype(nb_c)::value, ABS>(ring, nk, smem, xr0, gr0, kBN + gr0, awr0, fl,
                                                                          acc, aa, no_scale);
  });
  __syncthreads();  // every wave is done with the ring before LDS is reused

  if constexpr (!F8) {
    // h = silu(g) * u -> fp16, valid rows only (submission.py:1532-1542).
    // int8: g and u dequantised first, (acc * s_x[token]) * s_w[e, n]; the
    // intermediate is quantised per row afterwards (quant_rows_kernel), so
    // Stage 2 accumulates in int32 over the whole of K.
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int m = xr0 + G::kStep * b + (l & 31);
      if (m < actual) {
        _Float16* hrow = reinterpret_cast<_Float16*>(p.h) + (int64_t)(row0 + m) * p.h_ld;
#pragma unroll
        for (int a = 0; a < NBN; ++a)
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            const int n = n0 + gr0 + 32 * a + 8 * rg + 4 * (l >> 5);
            f16x4 v;
            if constexpr (I8) {
              f32x4 gs, us;
              if constexpr (kHoistFeat) {
                gs = sgv[a][rg];
                us = suv[a][rg];
              } else {
                gs = *reinterpret_cast<const f32x4*>(sgrow + n);
                us = *reinterpret_cast<const f32x4*>(surow + n);
              }
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const float gv = ((float)acc[a][b][4 * rg + q] * sxv[b]) * gs[q];
                const float uv = ((float)acc[NBN + a][b][4 * rg + q] * sxv[b]) * us[q];
                v[q] = (_Float16)silu_mul(gv, uv);
              }
            } else {
#pragma unroll
              for (int q = 0; q < 4; ++q) v[q] = (_Float16)silu_mul(acc[a][b][4 * rg + q], acc[NBN + a][b][4 * rg + q]);
            }
            *reinterpret_cast<f16x4*>(hrow + n) = v;
          }
      }
    }
    if constexpr (ABS) {
      // absorbed rows: each up wave hands its block through LDS to the gate
      // wave of the same features (same wn and block), which writes h
      float* red = reinterpret_cast<float*>(smem);  // [wn * NBN + j][16][64]; the ring is free
      const int aslot = g.wn * NBN + aj;
      if (!agate) {
#pragma unroll
        for (int q = 0; q < 16; ++q) red[(aslot * 16 + q) * 64 + l] = aa[q];
      }
      __syncthreads();
      const int m = l & 31;
      if (agate && m < nar) {
        _Float16* hrow = reinterpret_cast<_Float16*>(p.h) + (int64_t)(row0 + TR + m) * p.h_ld;
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          const int n = n0 + gr0 + 32 * aj + 8 * rg + 4 * (l >> 5);
          f16x4 v;
#pragma unroll
          for (int q = 0; q < 4; ++q)
            v[q] = (_Float16)silu_mul(aa[4 * rg + q], red[(aslot * 16 + 4 * rg + q) * 64 + l]);
          *reinterpret_cast<f16x4*>(hrow + n) = v;
        }
      }
    }
  } else {
    // fp8: dequantise (acc * s_x[token]) * s_w[e, n], h = silu(g) * u, then quantise
    // h per (row, this 128-column tile) to e4m3: amax over the tile's columns,
    // which are spread over the lane pair (l, l^32) and the WN waves.
    float* red = reinterpret_cast<float*>(smem);  // [WN][TR]; loop ended with a barrier
    float hv[2][NBN][16];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int m = xr0 + G::kStep * b + (l & 31);
      const float sx = m < actual ? sxv[b] : 0.0f;
      float amax = 0.0f;
#pragma unroll
      for (int a = 0; a < NBN; ++a)
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          f32x4 gs, us;
          if constexpr (kHoistFeat) {
            gs = sgv[a][rg];
            us = suv[a][rg];
          } else {
            const int n = n0 + gr0 + 32 * a + 8 * rg + 4 * (l >> 5);
            gs = *reinterpret_cast<const f32x4*>(sgrow + n);
            us = *reinterpret_cast<const f32x4*>(surow + n);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float gv = ((float)acc[a][b][4 * rg + q] * sx) * gs[q];
            const float uv = ((float)acc[NBN + a][b][4 * rg + q] * sx) * us[q];
            const float h = silu_mul(gv, uv);
            hv[b][a][4 * rg + q] = h;
            amax = fmaxf(amax, fabsf(h));
          }
        }
      amax = fmaxf(amax, __shfl_xor(amax, 32));
      if (l < 32) red[g.wn * TR + xr0 + G::kStep * b + l] = amax;
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int m = xr0 + G::kStep * b + (l & 31);
      float amax = 0.0f;
#pragma unroll
      for (int j = 0; j < G::WN; ++j) amax = fmaxf(amax, red[j * TR + m]);
      // The power-of-two scale 2^j (amax <= 448 * 2^j), which Stage 2's f8
      // MFMA applies itself; dividing by it is exact.
      const int sb = pow2_scale_e8m0(amax);
      const float inv = amax > 0.0f ? scale_from_e8m0(254 - sb) : 0.0f;  // 2^-j (sb = 0: 2^127, the exact inverse of 2^-127)
      if (m < actual) {
        const int64_t row = row0 + m;
        uint8_t* hrow = reinterpret_cast<uint8_t*>(p.h) + row * p.h_ld;
#pragma unroll
        for (int a = 0; a < NBN; ++a)
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            const int n = n0 + gr0 + 32 * a + 8 * rg + 4 * (l >> 5);
            *reinterpret_cast<uint32_t*>(hrow + n) =
                quant_code4<true>(hv[b][a][4 * rg], hv[b][a][4 * rg + 1], hv[b][a][4 * rg + 2], hv[b][a][4 * rg + 3], inv);
          }
        if (g.wn == 0 && l < 32) p.h_scale[row * p.hs_pitch + n0 / kBN] = (uint8_t)sb;
      }
    }
  }
}

template <int QT, bool GATHER>
__global__ __launch_bounds__(512) void stage1_wide_kernel(Stage1Params p) {
  __shared__ __attribute__((aligned(16))) char smem[kLdsBytes];
  const int nt = (int)(p.I / kBN);
  auto run = [&](const Item& it) {
    if (it.actual <= 0) return;  // no token: Stage 2 writes the rows as 0
    if (it.actual <= kLowRows) {
      if (it.shared || !p.stream) stage1_item<QT, GATHER, kLowRows, false, false>(p, it, smem);
      else stage1_item<QT, GATHER, kLowRows, false, true>(p, it, smem);
    } else if (QT != kQF16 || it.actual <= kWideRows) {
      if (it.shared || !p.stream) stage1_item<QT, GATHER, kWideRows, false, false>(p, it, smem);
      else stage1_item<QT, GATHER, kWideRows, false, true>(p, it, smem);
    } else if constexpr (QT == kQF16) {
      if (it.shared || !p.stream) stage1_item<QT, GATHER, kWideRows, true, false>(p, it, smem);
      else stage1_item<QT, GATHER, kWideRows, true, true>(p, it, smem);
    }
  };
  Item it;
  if constexpr (GATHER) {
    if (item_fused(blockIdx.x, p.istart, p.xb, p.gs, p.gpo, p.E, kBN, nt, p.rows_cap, it)) run(it);
  } else {
    if (item_bx(blockIdx.x, p.gidx, p.host_blocks, p.E, kBN, nt, p.gs, p.gpo, p.hmax, gridDim.x, smem, it)) run(it);
  }
}

// Stage 2 item: TR token rows (and absorbed ones) x BN features.
template <int QT, bool FUSED, int BN, int TR, bool ABS, bool STREAM>
__device__ __forceinline__ void stage2_item(const Stage2Params& p, const Item& it, char* smem) {
  constexpr bool I8 = QT == kQI8, F8 = QT == kQF8;
  using R = Ring<TR, BN, ABS>;
  using G = WaveGrid<R>;
  // int8: exact int32 accumulation over the whole of K (the intermediate has
  // one scale per row, applied in the epilogue); fp16 / fp8: fp32
  using Acc = typename std::conditional<I8, i32x16, f32x16>::type;
  constexpr int WTN = BN / G::WN;
  constexpr int NWB = WTN / 32;
  const int e = it.e, row0 = it.row0, n0 = it.n0;
  const int actual = it.actual < TR ? it.actual : TR;
  const int nar = ABS ? it.actual - actual : 0;  // absorbed rows
  const int gpo_e = p.gpo[e], go_e = p.go[e];

  const int nk = (int)(p.I * (QT == kQF16 ? 2 : 1) / kRowBytes);
  // this expert's [H, I] down weights, experts wd_es and rows wd_ld bytes
  // apart (the shared expert's own tensor, same row stride); intermediate rows
  // a_ld bytes apart
  const char* dexp = p.e_shared >= 0 && e == p.e_shared ? p.wd_shared : p.wd + (int64_t)e * p.wd_es;
  R ring;
  ring.nt = (actual + 63) / 64;
#pragma unroll
  for (int i = 0; i < R::NIT; ++i) {
    const int r = R::row_of(i);
    ring.t[i] = DmaTile<64, 8>::at(r, p.a + (int64_t)(row0 + (r < actual ? r : 0)) * p.a_ld);
  }
#pragma unroll
  for (int i = 0; i < R::NIW; ++i) {
    const int r = R::row_of(i);
    ring.w[i] = DmaTile<64, 8>::at(r, dexp + (int64_t)(n0 + r) * p.wd_ld);
  }
  ring.adma = ABS && wave_id() < 4;
  if constexpr (ABS) {
    const int r = R::row_of(0);
    ring.a = DmaTile<64, 8>::at(r, p.a + (int64_t)(row0 + (r < nar ? TR + r : 0)) * p.a_ld);
  }

  const G g;
  const int l = lane_id();
  const int xr0 = g.x0();      // slot row of this wave's first token row
  const int wr0 = WTN * g.wn;  // ... of its first weight row
  const FragLane fl;

  // Routing weight (and 8-bit row scale) of each of this lane's token rows,
  // loaded before the K loop so that their latency hides behind it.  Loads are
  // unconditional; rows without a token take the item's first row's values and
  // are never stored.
  // Fused: the pair's output row is its unpadded position in the expert-sorted
  // order, so an item writes one contiguous run of rows; the combine finds it
  // through pos[pair], written here once per row.  Pre-routed: the row itself,
  // its routing weight at the raw-order index (problem_detail.json:50 note 2),
  // clamped to the buffer as submission.py:1286-1288 does.
  const int64_t first = FUSED ? (int64_t)go_e + (row0 - gpo_e) : (int64_t)row0;
  auto weight_of = [&](int m, bool valid) -> float {
    if constexpr (FUSED) {
      const int pid = p.sorted_ids[row0 + (valid ? m : 0)];
      if (valid && n0 == 0 && l < 32) p.pos[pid] = (int32_t)(first + m);
      return reinterpret_cast<const float*>(p.routed)[pid];
    } else {
      int64_t ridx = (int64_t)go_e + (row0 - gpo_e) + m;
      ridx = ridx >= p.V ? p.V - 1 : ridx;
      ridx = ridx < 0 ? 0 : ridx;
      if (!valid || p.V <= 0) return 0.0f;
      return p.routed_f16 ? (float)reinterpret_cast<const _Float16*>(p.routed)[ridx]
                          : reinterpret_cast<const float*>(p.routed)[ridx];
    }
  };
  float wr[2], shv[2];
  const uint8_t* sp[2] = {nullptr, nullptr};
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int m = xr0 + G::kStep * b + (l & 31);
    const int mc = m < actual ? m : 0;
    wr[b] = weight_of(m, m < actual);
    if constexpr (I8) shv[b] = p.a_scale[row0 + mc];
    if constexpr (F8) sp[b] = p.a_scale8 + (int64_t)(row0 + mc) * p.as_pitch;
  }
  Acc acc[NWB][2];
#pragma unroll
  for (int a = 0; a < NWB; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) acc[a][b] = Acc{};
  // absorbed rows x weight block wm of this wave's NWB (lane l: absorbed row l % 32)
  f32x16 aa = {};
  const bool awave = ABS && g.wm < NWB;
  const int awr0 = wr0 + 32 * (awave ? g.wm : 0);
  float awr = 0.0f;
  if constexpr (ABS) {
    if (awave) awr = weight_of(TR + (l & 31), (l & 31) < nar);
  }
  auto loop = [&](auto nb_c, auto abs_c) {
    wide_k_loop<QT, F8, R, STREAM, NWB, decltype(nb_c)::value, decltype(abs_c)::value>(
        ring, nk, smem, xr0, wr0, wr0 + 32 * (NWB > 1 ? NWB / 2 : 1), awr0, fl, acc, aa, sp);
  };
  if constexpr (ABS && NWB >= 4) {  // every wave has a block for them, and all 256 rows are routed
    loop(std::integral_constant<int, 2>{}, std::true_type{});
  } else if constexpr (ABS) {
    if (awave) loop(std::integral_constant<int, 2>{}, std::true_type{});
    else loop(std::integral_constant<int, 2>{}, std::false_type{});
  } else {
    with_live<2>(g.live(actual), [&](auto nb_c) { loop(nb_c, std::false_type{}); });
  }

  __syncthreads();  // every wave is done with the ring
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int m = xr0 + G::kStep * b + (l & 31);
    if (m >= actual) continue;
#pragma unroll
    for (int a = 0; a < NWB; ++a)
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int nl = wr0 + 32 * a + 8 * rg + 4 * (l >> 5);  // feature within the tile
        f32x4 sd = {1.0f, 1.0f, 1.0f, 1.0f};
        if constexpr (QT != kQF16) sd = *reinterpret_cast<const f32x4*>(p.sd + (int64_t)e * p.H + n0 + nl);
        f16x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float y = (float)acc[a][b][4 * rg + q];
          if constexpr (I8) y = y * shv[b];  // int8: ((acc * s_h[row]) * s_d[n]) * w
          if constexpr (QT != kQF16) y = y * sd[q];
          v[q] = (_Float16)(y * wr[b]);
        }
        stage_out<BN>(smem, m, nl, v);
      }
  }
  __syncthreads();
  store_rows<BN, 8, FUSED>(p, smem, actual, row0, first, n0);
  if constexpr (ABS) {  // absorbed rows: stored directly
    _Float16* o = reinterpret_cast<_Float16*>(p.out);
    const int m = l & 31;
    if (awave && m < nar) {
      const int64_t orow = FUSED && MOE_S2_SCATTER ? (int64_t)(p.sorted_ids[row0 + TR + m] / p.topk) : first + TR + m;
#pragma unroll
      for (int rg = 0; rg < 4; ++rg) {
        const int n = n0 + awr0 + 8 * rg + 4 * (l >> 5);
        f16x4 v;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = (_Float16)(aa[4 * rg + q] * awr);
        if constexpr (FUSED && MOE_S2_SCATTER) atomic_add_f16x4(o + orow * p.H + n, v);
        else *reinterpret_cast<f16x4*>(o + orow * p.H + n) = v;
      }
    }
  }
}

// BN_: features per item; 0: the plan's (fused).  The kernel that holds both runs
// 256-feature items 0.7% slower than its own does (8 experts of H 4096, I 14336,
// 4096 tokens top-2: the call 2862 -> 2882 us, the same instructions per K step).
template <int QT, bool FUSED, int BN_>
__global__ __launch_bounds__(512) void stage2_wide_kernel(Stage2Params p) {
  __shared__ __attribute__((aligned(16))) char smem[kLdsBytes];
  const int bn = BN_ ? BN_ : *p.bn_plan;
  const int nt = (int)(p.H / bn);
  auto run_bn = [&](const Item& it, auto bn_c) {
    constexpr int BN = decltype(bn_c)::value;
    if (it.actual <= kLowRows) {
      if (it.shared || !p.stream) stage2_item<QT, FUSED, BN, kLowRows, false, false>(p, it, smem);
      else stage2_item<QT, FUSED, BN, kLowRows, false, true>(p, it, smem);
    } else if (QT != kQF16 || it.actual <= kWideRows) {
      if (it.shared || !p.stream) stage2_item<QT, FUSED, BN, kWideRows, false, false>(p, it, smem);
      else stage2_item<QT, FUSED, BN, kWideRows, false, true>(p, it, smem);
    } else if constexpr (QT == kQF16) {
      if (it.shared || !p.stream) stage2_item<QT, FUSED, BN, kWideRows, true, false>(p, it, smem);
      else stage2_item<QT, FUSED, BN, kWideRows, true, true>(p, it, smem);
    }
  };
  auto run = [&](const Item& it) {
    if (it.actual <= 0) return;
    if constexpr (BN_ != 0) {
      run_bn(it, std::integral_constant<int, BN_>{});
    } else {
      if (bn == 256) run_bn(it, std::integral_constant<int, 256>{});
      else run_bn(it, std::integral_constant<int, 128>{});
    }
  };
  Item it;
  if constexpr (FUSED) {
    if (item_fused(blockIdx.x, p.istart, p.xb, p.gs, p.gpo, p.E, bn, nt, p.rows_cap, it)) run(it);
  } else {
    if (!item_bx(blockIdx.x, p.gidx, p.host_blocks, p.E, bn, nt, p.gs, p.gpo, p.hmax, gridDim.x, smem, it)) return;
    // Rows owned by no valid token are written as 0 (problem_detail.json:50 note 4).
    _Float16* o = reinterpret_cast<_Float16*>(p.out);
    const int rows = it.zero_end - (it.row0 + it.actual);
    const int shift = bn == 256 ? 5 : 4;  // 16-byte chunks per row
    for (int idx = threadIdx.x; idx < rows << shift; idx += 512) {
      const int r = it.row0 + it.actual + (idx >> shift), c = idx & ((1 << shift) - 1);
      *reinterpret_cast<u32x4*>(o + (int64_t)r * p.H + it.n0 + 8 * c) = u32x4{0, 0, 0, 0};
    }
    run(it);
  }
}

// Ring depths of the narrow kernels: the stages in flight are what keeps
// enough bytes outstanding to stream weights at HBM rate, with two workgroups
// per CU (one for fp8 Stage 1).  Compile-time tunables (-D...) with the
// measured defaults.
#ifndef MOE_S1N_BN
#define MOE_S1N_BN 32  // gate / up tile width of fp16 and int8 (64 or 32)
#endif
#ifndef MOE_S1N_STAGES
#define MOE_S1N_STAGES 6
#endif
#ifndef MOE_S1N_STAGES_F8
#define MOE_S1N_STAGES_F8 4
#endif
#ifndef MOE_S2N_STAGES
#define MOE_S2N_STAGES 4
#endif

template <int QT>
static hipError_t go1_narrow(const Stage1Params& p, int64_t max_blocks, hipStream_t s) {
  if constexpr (QT == kQF8) {
    const int64_t grid = schedule_grid(max_blocks, p.I / kBN);
    hipLaunchKernelGGL((stage1_f8_kernel<MOE_S1N_STAGES_F8>), dim3((unsigned)grid), dim3(256), 0, s, p);
  } else {
    const int64_t grid = schedule_grid(max_blocks, p.I / MOE_S1N_BN);
    hipLaunchKernelGGL((stage1_narrow_kernel<MOE_S1N_BN, MOE_S1N_STAGES, QT>), dim3((unsigned)grid), dim3(256), 0, s, p);
  }
  return hipGetLastError();
}
static int64_t wide_grid(bool fused, int64_t max_blocks, int64_t nt, int hmax) {
  // pre-routed, where item_bx may cut by cost: an eighth more than an equal cut needs, so that a cut by cost
  // fits.  H 7168, I 2048, 64 experts, 9000 rows 1523 -> 1420 us; the surplus workgroups cost even
  // groupings 1-4% (376 -> 390, 632 -> 639, 1233 -> 1241 us).
  return fused ? kNumXcd * max_blocks : schedule_grid(max_blocks + (hmax > kLowRows ? (max_blocks + 7) / 8 : 0), nt);
}
template <int QT>
static hipError_t go1(const Stage1Params& p, bool gather, int64_t max_blocks, hipStream_t s) {
  const dim3 grid((unsigned)wide_grid(gather, max_blocks, p.I / kBN, p.hmax));
  if (gather) hipLaunchKernelGGL((stage1_wide_kernel<QT, true>), grid, dim3(512), 0, s, p);
  else if constexpr (QT == kQF16) hipLaunchKernelGGL((stage1_wide_kernel<QT, false>), grid, dim3(512), 0, s, p);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}
template <int QT>
static hipError_t go2(const Stage2Params& p, bool fused, int64_t max_blocks, hipStream_t s) {
  const dim3 grid((unsigned)wide_grid(fused, max_blocks, p.H / (p.bn ? p.bn : kBN), p.hmax));
#define MOE_S2W(FUSED, BN) hipLaunchKernelGGL((stage2_wide_kernel<QT, FUSED, BN>), grid, dim3(512), 0, s, p)
  if (fused) {
    if (p.bn == 256) MOE_S2W(true, 256);
    else if (p.bn == 128) MOE_S2W(true, 128);
    else MOE_S2W(true, 0);
  } else if constexpr (QT == kQF16) {
    if (p.bn == 256) MOE_S2W(false, 256);
    else MOE_S2W(false, 128);
  } else {
    return hipErrorInvalidValue;
  }
#undef MOE_S2W
  return hipGetLastError();
}

hipError_t launch_stage1(const Stage1Params& params, bool narrow, int qt, bool gather, int64_t max_blocks, hipStream_t s) {
  Stage1Params p = params;
  p.host_blocks = (int)max_blocks;
  if (p.w_ld == 0) p.w_ld = p.H * (qt != kQF16 ? 1 : 2);
  if (p.w_es == 0) p.w_es = p.I * p.w_ld;
  if (p.h_ld == 0) p.h_ld = p.I;
  if (max_blocks <= 0) return hipSuccess;
  if (narrow) {
    if (!gather) return hipErrorInvalidValue;
    return qt == kQF8 ? go1_narrow<kQF8>(p, max_blocks, s)
                      : (qt == kQI8 ? go1_narrow<kQI8>(p, max_blocks, s) : go1_narrow<kQF16>(p, max_blocks, s));
  }
  return qt == kQF8 ? go1<kQF8>(p, gather, max_blocks, s)
                    : (qt == kQI8 ? go1<kQI8>(p, gather, max_blocks, s) : go1<kQF16>(p, gather, max_blocks, s));
}

hipError_t launch_stage2(const Stage2Params& params, bool narrow, int qt, bool fused,
                         int64_t max_blocks, hipStream_t s) {
  Stage2Params p = params;
  p.host_blocks = (int)max_blocks;
  if (p.a_ld == 0) p.a_ld = p.I * (qt != kQF16 ? 1 : 2);
  if (p.wd_ld == 0) p.wd_ld = p.I * (qt != kQF16 ? 1 : 2);
  if (p.wd_es == 0) p.wd_es = p.H * p.wd_ld;
  if (max_blocks <= 0) return hipSuccess;
  if (narrow) {
    if (!fused) return hipErrorInvalidValue;
    const dim3 grid((unsigned)schedule_grid(max_blocks, p.H / kBN));
    if (qt == kQI8) hipLaunchKernelGGL((stage2_narrow_kernel<MOE_S2N_STAGES, kQI8>), grid, dim3(256), 0, s, p);
    else if (qt == kQF8) hipLaunchKernelGGL((stage2_narrow_kernel<MOE_S2N_STAGES, kQF8>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((stage2_narrow_kernel<MOE_S2N_STAGES, kQF16>), grid, dim3(256), 0, s, p);
    return hipGetLastError();
  }
  if ((!fused || p.bn) && p.bn != 128 && (p.bn != 256 || p.H % 256)) return hipErrorInvalidValue;
  return qt == kQF8 ? go2<kQF8>(p, fused, max_blocks, s)
                    : (qt == kQI8 ? go2<kQI8>(p, fused, max_blocks, s) : go2<kQF16>(p, fused, max_blocks, s));
}

}  // namespace moe
