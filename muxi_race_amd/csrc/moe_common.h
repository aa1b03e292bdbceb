// Shared device-side building blocks for the gfx950 fused-MoE kernels.
//
// Tile geometry.  Every GEMM operand tile is a stack of rows that are
// contiguous along K in global memory (token rows of x / the intermediate,
// output-feature rows of the expert weights).  One K step moves 128 bytes of
// each row (64 fp16 or 128 int8 elements) = eight 16-byte chunks.  In LDS a
// row occupies 128 bytes and chunk c of row r sits at chunk slot
// c ^ swz(r), so the 32 rows read by one MFMA fragment load spread over the
// banks.  One MFMA K sub-step consumes two chunks per row (lanes 0-31 the
// first, lanes 32-63 the second), i.e. 16 fp16 or 32 int8 per row.
//
// MFMA roles.  D[n][m] = sum_k W[n][k] * X[m][k]: the weight tile is the A
// operand (32 output features per MFMA block) and the token tile the B
// operand (32 tokens).  In the 32x32 accumulator lane l holds token
// m = l % 32 and features n = 8*(r/4) + 4*(l/32) + r%4 for register r, so each
// lane owns runs of 4 consecutive output features of one token row: the
// epilogues store 8-byte (fp16) or 4-byte (int8) vectors.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace moe {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kRowBytes = 128;     // bytes of one tile row per K step
constexpr int kBN = 128;           // output-feature tile (N) of every GEMM
constexpr int kNumXcd = 8;         // MI355X: 8 XCDs, workgroups dealt round-robin
constexpr float kLog2e = 1.44269504088896341f;

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// LDS byte offset of 16-byte chunk c of tile row r.  gfx950 serves a
// ds_read_b128 16 lanes at a time across 64 four-byte banks: a fragment read
// (16 consecutive rows, one chunk) is conflict-free when the 16 (row parity,
// chunk slot) pairs are distinct, i.e. when the slot is c ^ f(r) with f taking
// 8 distinct values over the even rows and over the odd rows of any 16-row
// group.  f(r) = (r >> 1) & 7 does that (f(r) = r & 7 puts rows r and r + 8 on
// the same banks: a 2-way conflict on every read, measured).
__device__ __forceinline__ int swz(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int lds_swz(int r, int c) {
  return (r << 7) | (((c ^ swz(r)) & 7) << 4);
}

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }

// s_waitcnt vmcnt(N) with the other counters left alone (gfx9 encoding:
// vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt_hi[15:14]).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Pipelines issue Q loads per wave per stage, in stage order, and vector-memory
// loads retire in order: waiting until at most Q*min(ahead, N) loads are
// outstanding completes every stage but the last min(ahead, N) issued.
template <int Q, int N>
__device__ __forceinline__ void wait_stages(int ahead) {
  if constexpr (N <= 0) {
    wait_vmcnt<0>();
  } else {
    if (ahead >= N) wait_vmcnt<Q * N>();
    else wait_stages<Q, N - 1>(ahead);
  }
}

// Workgroup barrier without a memory fence.  __syncthreads() would first wait
// for every outstanding vector-memory operation (vmcnt(0)), which includes the
// direct-to-LDS loads of the stages still in flight; the pipelines below wait
// for exactly the stage they consume (wait_vmcnt) and then use this barrier.
// The empty asm statements keep the compiler from moving memory accesses
// across it.
__device__ __forceinline__ void barrier_no_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

#define MOE_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

// Cache policy of weight loads that no other tile repeats.  A weight tile read
// by exactly one item is loaded non-temporal (the gfx950 `nt` bit,
// cache-policy immediate 2): decode went from 0.575 to 0.533 ms with it (a
// load-only copy of the 96-row decode ring streamed 6.15 -> 7.12 TB/s at rows
// 14 KiB apart, 5.45 -> 6.14 TB/s at 4 KiB).  Weight tiles that sibling items
// of an expert re-read from L2, and token / intermediate rows, keep the
// default policy (non-temporal there measured slower: fewer L2 hits).
// 0 turns streaming off.
#ifndef MOE_W_POLICY
#define MOE_W_POLICY 2
#endif
constexpr int kPolicyDefault = 0;
constexpr int kPolicyWeights = MOE_W_POLICY;

// global_load_lds_dword[x4]: per-lane global address -> LDS at m0 + 4|16 * lane,
// cache policy POLICY.  The host compilation pass only needs kernel
// signatures (for the launch stubs); the builtin is kept out of that pass,
// where clang's deferred diagnostic for it otherwise stops the remaining
// kernel stubs from being emitted.
template <int BYTES, int POLICY = kPolicyDefault>
__device__ __forceinline__ void dma_to_lds(const void* g, void* lds) {
  static_assert(BYTES == 4 || BYTES == 16, "dword or dwordx4");
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (BYTES == 16)
    __builtin_amdgcn_global_load_lds(g, MOE_LDS_PTR(lds), 16, 0, POLICY);
  else
    __builtin_amdgcn_global_load_lds(g, MOE_LDS_PTR(lds), 4, 0, POLICY);
#else
  (void)g;
  (void)lds;
#endif
}

// Direct global -> LDS loader (global_load_lds_dwordx4) for a tile of ROWS rows
// x 128 bytes, issued by the NW waves of a workgroup.  One wave instruction
// writes 1 KiB of LDS = 8 consecutive tile rows, lane l landing at byte 16*l:
// row r = r0 + l/8, chunk slot l%8.  With the swizzle above that slot holds
// logical chunk (l%8) ^ swz(r), so lane l loads that chunk of its row; the 8
// lanes of a row still cover its 128 contiguous bytes.  Wave w issues the
// instructions for row groups NW*i + w.
template <int ROWS, int NW>
struct DmaTile {
  static constexpr int NI = ROWS / (8 * NW);  // instructions per wave per K step
  static_assert(NI >= 1 && ROWS == 8 * NW * NI, "tile rows must be a multiple of 8 * waves");
  const char* src[NI];

  __device__ __forceinline__ static int row_of(int i) { return 8 * (NW * i + wave_id()) + (lane_id() >> 3); }
  // This lane's 16 bytes of a tile row r at rowp (K step 0).
  __device__ __forceinline__ static const char* at(int r, const char* rowp) {
    return rowp + ((((lane_id() & 7) ^ swz(r)) & 7) << 4);
  }
  // rowp: address of K-step 0 of tile row row_of(i).
  __device__ __forceinline__ void set(int i, const char* rowp) { src[i] = at(row_of(i), rowp); }
  // STREAM: tile rows from FROM on under the streaming weight policy.  Both are
  // known at compile time: chosen at run time, the policy costs two branches per
  // instruction, which one wave per SIMD does not hide (Stage 2 of 32-row tiles at
  // one token, 8 experts top-2, H 4096, I 14336: fp8 52.0 -> 44.5 us, int8 50.1 ->
  // 41.6; int8 Stage 1 at 24 tokens, 64 experts top-6, H 7168, I 2048: 249 -> 246).
  // PART of PARTS: that share of the instructions.
  template <bool STREAM = false, int FROM = 0, int PART = 0, int PARTS = 1>
  __device__ __forceinline__ void issue(char* lds, int ks) const {
    static_assert(FROM % (8 * NW) == 0, "an instruction's rows have one policy");
    const int w = wave_id();
#pragma unroll
    for (int i = PART * NI / PARTS; i < (PART + 1) * NI / PARTS; ++i) {
      const char* g = src[i] + (size_t)ks * kRowBytes;
      char* d = lds + 1024 * (NW * i + w);
      if (STREAM && 8 * NW * i >= FROM) dma_to_lds<16, kPolicyWeights>(g, d);
      else dma_to_lds<16>(g, d);
    }
  }
};

// MFMA fragment of the 32 tile rows starting at `row0`, K sub-step s (0..3).
__device__ __forceinline__ u32x4 frag(const char* lds, int row0, int s) {
  const int l = lane_id();
  return *reinterpret_cast<const u32x4*>(lds + lds_swz(row0 + (l & 31), 2 * s + (l >> 5)));
}

// The same reads by 32-bit LDS address, for the K loops.  A fragment's first
// tile row is a multiple of 32 there, so its row swizzle depends on the lane
// alone (swz(r0 + (l & 31)) = swz(l & 31)) and its address splits into a
// wave-uniform row base, lds + 128 * r0, and a per-lane offset for each K
// sub-step.  With the base taken through readfirstlane (a scalar register,
// recomputed per ring stage) and the four lane offsets held once, the
// compiler keeps one VGPR per sub-step instead of hoisting one address per
// fragment and sub-step out of the K loop.
struct FragLane {
  uint32_t off[4];
  __device__ __forceinline__ FragLane() {
    const int l = lane_id();
#pragma unroll
    for (int s = 0; s < 4; ++s) off[s] = (uint32_t)lds_swz(l & 31, 2 * s + (l >> 5));
  }
};
__device__ __forceinline__ uint32_t row_base(const char* lds, int row0) {
  const uint32_t a = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)lds;
  return __builtin_amdgcn_readfirstlane(a + ((uint32_t)row0 << 7));
}
__device__ __forceinline__ u32x4 frag_at(uint32_t base, uint32_t lane_off) {
  typedef __attribute__((address_space(3))) const u32x4 LdsVec;
  return *(LdsVec*)(uintptr_t)(base + lane_off);
}

__device__ __forceinline__ f32x16 mma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                               __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}
__device__ __forceinline__ i32x16 mma(u32x4 a, u32x4 b, i32x16 c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, a),
                                              __builtin_bit_cast(i32x4, b), c, 0, 0, 0);
}

// fp8 (OCP e4m3) x fp8 over 64 K elements: the lane supplies 32 bytes, the
// fragments of two consecutive 32-byte K sub-steps (frag(.., s) and
// frag(.., s + 1)).  Which K index each byte takes does not matter as long as
// both operands come from the same LDS layout through the same fragment loads.
__device__ __forceinline__ f32x16 mma8(u32x4 a0, u32x4 a1, u32x4 b0, u32x4 b1, f32x16 c) {
  const i32x8 a = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
  const i32x8 b = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
  // format 0 (fp8 e4m3) for both operands, no block scaling
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// As mma8, with the B operand's rows scaled by 2^(sb - 127) (E8M0 byte sb):
// lane l gives the scale of B row l % 32 -- lanes l and l + 32 each cover one
// 32-element K block of that row, and the callers pass the same scale for
// both, since a row's scale is constant over the 64 K elements.
__device__ __forceinline__ f32x16 mma8_scale_b(u32x4 a0, u32x4 a1, u32x4 b0, u32x4 b1, f32x16 c, int sb) {
  const i32x8 a = {(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3], (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
  const i32x8 b = {(int)b0[0], (int)b0[1], (int)b0[2], (int)b0[3], (int)b1[0], (int)b1[1], (int)b1[2], (int)b1[3]};
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 127, 0, sb);
}

// Power-of-two scale for an fp8 block of maximum |value| amax > 0: 2^j with
// the smallest j such that amax <= 448 * 2^j (so amax / 2^j lies in (224,
// 448] and dividing by it is exact), j >= -127.  Returned as its E8M0 byte
// j + 127; scale_from_e8m0 gives the float (2^-127 as a denormal).
__device__ __forceinline__ int pow2_scale_e8m0(float amax) {
  const uint32_t u = __float_as_uint(amax);
  const int e = (int)((u >> 23) & 0xFF) - 127;                  // amax = m * 2^e, m in [1, 2)
  int j = e - 8 + ((u & 0x7FFFFFu) > 0x600000u ? 1 : 0);       // 448 = 1.75 * 2^8
  return j < -127 ? 0 : j + 127;
}
__device__ __forceinline__ float scale_from_e8m0(int b) {
  return b == 0 ? __uint_as_float(0x00400000u) : __uint_as_float((uint32_t)b << 23);
}

// silu(g) * u = u * g / (1 + 2^(-g*log2e)) in fp32 (v_exp_f32 + v_rcp_f32).
__device__ __forceinline__ float silu_mul(float g, float u) {
  const float sig = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * kLog2e));
  return u * (g * sig);
}

// q = clamp(trunc(x*inv +- 0.5), +-127): the product and the +-0.5 are two
// separately rounded fp32 operations (never one fused multiply-add), so the
// result is bit-identical to the same two IEEE operations on the CPU.
__device__ __forceinline__ int quant_i8(float x, float inv) {
#pragma clang fp contract(off)
  const float v = x * inv;
  float t = v + (v >= 0.0f ? 0.5f : -0.5f);
  int q = (int)t;  // truncates toward zero
  q = q > 127 ? 127 : q;
  q = q < -127 ? -127 : q;
  return q;
}

// OCP fp8 e4m3 code of v, round to nearest even, saturating at +-448 (the
// callers scale so that |v| <= 448): the gfx950 conversion instruction
// (v_cvt_pk_fp8_f32, two codes per instruction) on v clamped to [-448, 448].
// Its codes equal a bit-level restatement of the format -- the fp32 mantissa
// rounded to 3 bits with the carry running into the rebiased exponent, and
// below 2^-6 the round-to-even multiple of 2^-9 -- for every float of
// magnitude <= 448 (checked exhaustively by the fp8 GPU tests).
__device__ __forceinline__ float f8_clamp(float v) { return __builtin_amdgcn_fmed3f(v, -448.0f, 448.0f); }
__device__ __forceinline__ uint32_t f8_e4m3(float v) {
  const float c = f8_clamp(v);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(c, c, 0, false) & 0xffu;
}
// codes of a, b, c, d in bytes 0..3
__device__ __forceinline__ uint32_t f8_e4m3x4(float a, float b, float c, float d) {
  const int lo = __builtin_amdgcn_cvt_pk_fp8_f32(f8_clamp(a), f8_clamp(b), 0, false);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(f8_clamp(c), f8_clamp(d), lo, true);
}

// Largest code magnitude of the 8-bit formats: int8 (symmetric) and fp8 e4m3.
template <bool F8> constexpr float qmax() { return F8 ? 448.0f : 127.0f; }

// 8-bit codes (int8 round-half-away or fp8 e4m3) of x[0..3] * inv packed
// into bytes 0..3.
template <bool F8>
__device__ __forceinline__ uint32_t quant_code4(float x0, float x1, float x2, float x3, float inv) {
#pragma clang fp contract(off)
  if constexpr (F8) {
    return f8_e4m3x4(x0 * inv, x1 * inv, x2 * inv, x3 * inv);
  } else {
    return ((uint32_t)quant_i8(x0, inv) & 0xffu) | (((uint32_t)quant_i8(x1, inv) & 0xffu) << 8) |
           (((uint32_t)quant_i8(x2, inv) & 0xffu) << 16) | (((uint32_t)quant_i8(x3, inv) & 0xffu) << 24);
  }
}

// Inclusive prefix sum over the wave's 64 lanes: Hillis-Steele inside each
// 16-lane row with DPP row shifts (lanes shifted in from outside the row read
// 0), then each row adds the totals of the rows before it (read from lanes 15,
// 31, 47).  Integer adds, so the order of the terms does not matter.
__device__ __forceinline__ int wave_inclusive_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);  // row_shr:8
  const int r0 = __builtin_amdgcn_readlane(v, 15), r1 = __builtin_amdgcn_readlane(v, 31),
            r2 = __builtin_amdgcn_readlane(v, 47);
  const int row = lane_id() >> 4;
  return v + (row > 0 ? r0 : 0) + (row > 1 ? r1 : 0) + (row > 2 ? r2 : 0);
}

// ---------------------------------------------------------------------------
// Work schedules.  Items are numbered expert-major and the item range is cut
// into 8 contiguous chunks, one per XCD (workgroup g runs on XCD g % 8 and is
// that XCD's (g / 8)-th workgroup), so the items sharing a weight tile or a
// token tile run close together on one XCD and re-read it from that XCD's L2.
// ---------------------------------------------------------------------------

// The number of workgroup g's item among `total`, or -1 (surplus workgroup).
__device__ __forceinline__ int xcd_item(int g, int total) {
  const int per = (total + kNumXcd - 1) / kNumXcd;
  const int slot = g / kNumXcd;
  const int v = (g % kNumXcd) * per + slot;
  return slot < per && v < total ? v : -1;
}

// 32-row items: one per BM-row block of an expert and output-feature tile of
// width BN, an expert's items ordered by tile.  M blocks of expert e are
// [gpo[e]/BM, gpo[e+1]/BM); `host_blocks` is the number of BM-row blocks the
// caller's buffers hold: expert blocks beyond it are never scheduled, so
// inconsistent metadata cannot move an access out of the buffers.
struct Work {
  int e;        // expert
  int row0;     // first row of the block (in the expert-sorted row space)
  int n0;       // first output feature of the tile
  bool shared;  // other items of this launch read the same weight rows
};

__device__ __forceinline__ bool schedule(int g, const int32_t* __restrict__ gpo, int E, int BM, int BN,
                                         int nt, int host_blocks, Work& w) {
  int blocks = gpo[E] / BM;
  blocks = blocks < host_blocks ? blocks : host_blocks;
  const int v = xcd_item(g, blocks * nt);
  if (v < 0) return false;
  // e = (number of experts whose first item is <= v) - 1, found with ballots.
  const int l = lane_id();
  int cnt = 0;
  for (int base = 0; base < E; base += 64) {
    const int e = base + l;
    int le = 0;
    if (e < E) le = (gpo[e] / BM) * nt <= v;
    cnt += __popcll(__ballot(le));
  }
  const int e = cnt - 1;
  if (e < 0) return false;  // only with inconsistent metadata (gpo[0] > 0)
  const int b0 = gpo[e] / BM;
  const int nb = gpo[e + 1] / BM - b0;
  if (nb <= 0) return false;
  const int local = v - b0 * nt;
  const int t = local / nb;  // N tile
  w.e = e;
  w.shared = nb > 1;
  w.row0 = (b0 + local % nb) * BM;
  w.n0 = t * BN;
  return w.row0 / BM < host_blocks && t < nt;
}

// Wide items (more than 32 rows per expert).  An expert of n routed rows runs
// c = ceil(n / hmax) items per N tile, of rows_of(n, c) rows each, n / c rounded
// up to a multiple of 32; the last one takes what is left, at least one row (385
// rows with hmax 128: 128, 128, 128, 1).  Dealing the 32-row blocks out evenly
// instead (128, 96, 96, 65) was slower, since waves and token loads work in
// 64-row steps and three short pieces then cost what full ones do: H 7168, I
// 2048, 32 experts of 11 rows but 5 of 300 (128, 128, 44 -> 128, 96, 76) 611 ->
// 638 us, 64 of 20 but 10 of 300 1180 -> 1203.
// All items span the whole N tile; item v of expert e is
// N tile (v - first) / c, row piece (v - first) % c, so the c items reading one
// weight tile are adjacent.  hmax is kTallRows at most where the tiles take
// absorbed rows (kAbsorbRows), kWideRows otherwise; shorter where that ends a
// launch of few rounds earlier (fused: launch.h ItemPlan; run_kernel: capi.hip).
constexpr int kLowRows = 128, kWideRows = 256;
constexpr int kAbsorbRows = 32;  // rows past kWideRows that an item takes along
constexpr int kTallRows = kWideRows + kAbsorbRows;

__host__ __device__ inline int items_of(int n, int hmax) { return (n + hmax - 1) / hmax; }
__device__ __forceinline__ int rows_of(int n, int c) { return (n + 32 * c - 1) / (32 * c) * 32; }

// The heights that a plan chooses from: the tallest, 256, 224, .., 128.
constexpr int kPlanHeights = 6;
__device__ __forceinline__ int plan_height(int j, int tall) { return j == 0 ? tall : kWideRows - 32 * (j - 1); }
static_assert(kWideRows - 32 * (kPlanHeights - 2) == kLowRows, "the shortest is the one the host's bounds assume");

struct Item {
  int e;         // expert, or -1 (rows owned by no expert)
  int row0;      // first row
  int actual;    // routed rows of this piece (<= hmax): which tile runs the item
  int n0;        // first output feature of the tile
  int zero_end;  // pre-routed, the expert's last piece: rows [row0 + actual, zero_end) have no token
  bool shared;   // other items of this launch read the same weight rows
};

// Fused launches: istart[e] = items per N tile of the experts below e, and XCD x
// runs the items [xb[x], xb[x + 1]) (both written by align); e's rows are
// [gpo[e], gpo[e] + gs[e]).  rows_cap: rows the caller's buffers hold.
__device__ __forceinline__ bool item_fused(int g, const int32_t* __restrict__ istart, const int32_t* __restrict__ xb,
                                           const int32_t* __restrict__ gs, const int32_t* __restrict__ gpo, int E,
                                           int BN, int nt, int rows_cap, Item& it) {
  const int v = xb[g % kNumXcd] + g / kNumXcd;
  if (v >= xb[g % kNumXcd + 1]) return false;
  const int l = lane_id();
  int cnt = 0;
  for (int base = 0; base < E; base += 64) {
    const int e = base + l;
    cnt += __popcll(__ballot(e < E && istart[e < E ? e : 0] * nt <= v));
  }
  const int e = cnt - 1;  // an empty expert starts where the next one does, so e has items
  const int i0 = istart[e], c = istart[e + 1] - i0;
  if (c <= 0) return false;
  const int n = gs[e], r = rows_of(n, c);
  const int local = v - i0 * nt;
  const int t = local / c, i = local % c;
  it.e = e;
  it.row0 = gpo[e] + i * r;
  it.actual = n - i * r < r ? n - i * r : r;
  it.n0 = t * BN;
  it.zero_end = 0;
  it.shared = c > 1;
  return it.actual > 0 && it.row0 + it.actual <= rows_cap;
}

// XCD shares of a launch's items, for one lane: the first item of XCD x
// (x = 8: the end) and the cost of the items before it.  `weighted`: the items
// are cut where the cost is an eighth each; otherwise into equal numbers.  An
// item of r rows costs kItemCost + r: at 256 experts of H 7168, I 2048 a Stage 1
// step took 1.28 us at 32 rows, 1.42 at 128, 1.64 at 160 and 2.2 at 256.  The
// experts below e cost K(e) = kItemCost * ist[e] + gof[e] per N tile.
constexpr int kItemCost = 256;
struct XcdCut {
  int item;
  double cost;
};
__device__ __forceinline__ XcdCut xcd_cut(int x, bool weighted, const int* ist, const int* gof, int E, int nt) {
  const int total = ist[E] * nt;
  auto K = [&](int e) { return (double)kItemCost * ist[e] + (double)gof[e]; };
  const double all = K(E) * nt;
  XcdCut r;
  const int per = (total + kNumXcd - 1) / kNumXcd;
  r.item = x * per < total ? x * per : total;
  r.cost = all * x / kNumXcd;
  if (x == kNumXcd || (!weighted && r.item == total)) return XcdCut{total, all};
  // the last expert that starts at or before the cut
  int lo = 0, hi = E;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (weighted ? K(mid) * nt <= r.cost : ist[mid] * nt <= r.item) lo = mid;
    else hi = mid;
  }
  const int c = ist[lo + 1] - ist[lo];
  const double ce = K(lo + 1) - K(lo);  // of its c pieces
  if (weighted) {
    const int in = c > 0 ? (int)((r.cost - K(lo) * nt) * c / ce) : 0;
    r.item = ist[lo] * nt + (in < c * nt ? in : c * nt);
  } else {
    r.cost = K(lo) * nt + (c > 0 ? (r.item - ist[lo] * nt) * ce / c : 0.0);
  }
  return r;
}
// Both cuts of a launch's items on 18 lanes of a wave -- lanes 0..8 of them equal
// numbers, 9..17 equal cost; up to three launches at once, one per 18 lanes --
// and the better one: the one whose slowest XCD needs less time, an XCD running
// its items kCusPerXcd at a time.  Equal cost pays where experts differ and
// there are many rounds; with two rounds of like items it would leave some XCD a
// third.  slots: workgroups an XCD has in the launch, which a cut has to fit in.
constexpr int kCusPerXcd = 32;
struct XcdPick {
  int item;       // first item of XCD (lane % 18) % 9
  bool weighted;  // the cut by cost is the better one
  float slow;     // its slowest XCD's time, in rows of cost; INFINITY: neither fits
};
// From the cuts themselves, one per lane.
__device__ __forceinline__ XcdPick xcd_better(XcdCut cut, bool active, int slots) {
  const int l = lane_id(), q = l % 18, base = l - q, x = q % 9;
  const int items = __shfl_down(cut.item, 1) - cut.item;
  const float cost = __shfl_down((float)cut.cost, 1) - (float)cut.cost;
  float t = 0.0f;
  if (active && x < 8 && items > 0) t = (float)((items + kCusPerXcd - 1) / kCusPerXcd) * cost / (float)items;
  float equal = 0.0f, weighted = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    equal = fmaxf(equal, __shfl(t, base + j));
    weighted = fmaxf(weighted, __shfl(t, base + 9 + j));
  }
  const uint64_t over = __ballot(active && x < 8 && items > slots) >> base;
  if (over & 0x1ff) equal = INFINITY;
  if (over & 0x3fe00) weighted = INFINITY;
  return XcdPick{cut.item, weighted < equal, fminf(weighted, equal)};
}
__device__ __forceinline__ XcdPick xcd_pick(const int* ist, const int* gof, int E, int nt, bool active, int slots) {
  const int q = lane_id() % 18;
  XcdCut cut = {0, 0.0};
  if (active) cut = xcd_cut(q % 9, q >= 9, ist, gof, E, nt);
  return xcd_better(cut, active, slots);
}

// An upper bound on an XCD's items with either cut, for `pieces` items per N tile
// and `rows` routed rows in all.
inline int64_t xcd_items_bound(int64_t pieces, int64_t rows, int64_t nt) {
  return (pieces * kItemCost + rows) * nt / (kNumXcd * kItemCost) + 2;
}

// Pre-routed launches (the reference operator): block b of 128 rows belongs to
// expert gidx[b] (problem_detail.json:50 note 5; submission.py:1444), and the
// launch covers blocks [0, nblk) with nblk = min(gidx entries, blocks of the
// row buffers), as submission.py:2115 launches group_idx_for_bx.numel()
// blocks.  The maximal run [s, end) of consecutive blocks with one gidx value
// is treated as one expert: its first n = clamp(gs[e] - (128 s - gpo[e]), 0,
// 128 (end - s)) rows are routed (the per-block rule of each of its blocks),
// and the rest have no token.  A run without tokens still has one item per N
// tile, which writes its rows as 0.  A gidx value outside [0, E) gives e = -1
// (rows owned by no expert).
//
// The items below a run are counted here, by the workgroup's 512 threads, M
// neighbouring blocks each (1 up to 512 blocks, else kScanBlocks): block j of a
// run counts the pieces that its rows add, items_of(min(n, 128 (j + 1))) -
// items_of(min(n, 128 j)), which sums to the run's.  (Numbering by blocks
// instead, with the surplus items ending at once, left the XCDs unequal work: 22
// experts of 155 rows and 10 of 112, H 7168, I 2048, Stage 1 551 us.)  This runs
// before every item's first load, so it makes two dependent round trips to
// memory -- block to expert, expert to its rows -- and finds the rest in LDS.
// A pass covers kThreads * M blocks; only launches of more than 4096 make two.
//
// Launches of up to 512 blocks with an expert of more than kCutRows rows, in
// items of more than kLowRows, cut their items over the XCDs as the fused ones
// do (xcd_better): the thread whose block holds a cut writes it.  Others cut
// into equal numbers: like items gain nothing by the comparison, 1 us before each
// item (22 experts of 155 rows and 10 of 112: 602 us without it, 619 with), and
// short ones differ little (32 experts of 11 rows but 5 of 300: 633 us cut by
// cost, 604 into equal numbers).
constexpr int kScanBlocks = 8;
constexpr int kCutRows = 192;
struct RunScan {
  int last[8], pieces[8], rows[8];     // per wave: its last run's first block, pieces and rows it adds
  int tall[8];                         // ... whether a run has more than kCutRows rows
  int run[8], below[8], val[8], left[8];  // per wave: the last run at or before the item
  int cut_item[2][8];                  // [equal numbers, equal cost][XCD]
  float cut_cost[2][8];
  uint32_t firsts[16 * kScanBlocks];   // bit b: block b starts a run
};

template <int M>
__device__ __forceinline__ bool item_runs(int g, const int32_t* __restrict__ gidx, int nblk, int E, int BN, int nt,
                                          const int32_t* __restrict__ gs, const int32_t* __restrict__ gpo, int hmax,
                                          int grid, char* smem, Item& it) {
  constexpr int BM = 128, kThreads = 512, kPass = kThreads * M;
  RunScan* sh = reinterpret_cast<RunScan*>(smem);
  const int l = lane_id(), w = wave_id(), tid = threadIdx.x;
  const bool one_pass = nblk <= kPass;

  // this thread's blocks of a pass
  int below[M], rbelow[M], pcs[M], rws[M], val[M], left[M];
  uint32_t first = 0;
  int carry_s = 0, carry_p = 0, carry_r = 0;  // of the passes before
  auto pass = [&](int base) {
    const int b0 = base + tid * M;
    int gs_e[M], gpo_e[M];
#pragma unroll
    for (int j = 0; j < M; ++j) val[j] = gidx[b0 + j < nblk ? b0 + j : nblk - 1];
    int prev = gidx[b0 > 0 ? (b0 <= nblk ? b0 - 1 : nblk - 1) : 0];
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int ec = val[j] >= 0 && val[j] < E ? val[j] : 0;
      gs_e[j] = gs[ec];
      gpo_e[j] = gpo[ec];
    }
    first = 0;
    int last = -1;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      if (b0 + j < nblk && (b0 + j == 0 || val[j] != prev)) {
        first |= 1u << j;
        last = b0 + j;
      }
      prev = val[j];
    }
    const uint64_t m = __ballot(first != 0);
    const int wave_last = __builtin_amdgcn_readlane(last, m ? 63 - __builtin_clzll(m) : 0);  // -1 if there is none
    if (l == 0) sh->last[w] = wave_last;
    if (one_pass) {
      if constexpr (M == 1) {
        if (l == 0) reinterpret_cast<uint64_t*>(sh->firsts)[w] = m;
      } else {
        reinterpret_cast<uint8_t*>(sh->firsts)[tid] = (uint8_t)first;
      }
    }
    const uint64_t lower = m & ((1ull << l) - 1);
    const int from_wave = __shfl(last, lower ? 63 - __builtin_clzll(lower) : 0);
    __syncthreads();
    int s = carry_s;
    for (int v = 0; v < w; ++v) s = sh->last[v] >= 0 ? sh->last[v] : s;
    if (lower) s = from_wave;
    int c = 0, r = 0;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      const int b = b0 + j;
      s = first >> j & 1 ? b : s;
      const bool owned = val[j] >= 0 && val[j] < E;
      const int64_t lft = owned ? (int64_t)gs_e[j] - ((int64_t)s * BM - gpo_e[j]) : 0;
      const int64_t lo = (int64_t)(b - s) * BM, hi = lo + BM;
      left[j] = (int)(lft < 0 ? 0 : (lft > 0x7fffffff ? 0x7fffffff : lft));
      pcs[j] = rws[j] = 0;
      if (b < nblk) {
        if (lft > 0) {
          const int upto_hi = (int)(lft < hi ? lft : hi), upto_lo = (int)(lft < lo ? lft : lo);
          pcs[j] = items_of(upto_hi, hmax) - items_of(upto_lo, hmax);
          rws[j] = upto_hi - upto_lo;
        } else {
          pcs[j] = first >> j & 1;
        }
      }
      c += pcs[j];
      r += rws[j];
    }
    const int inc = wave_inclusive_scan(c), incr = wave_inclusive_scan(r);
    const int tall = __ballot(left[0] > kCutRows && b0 < nblk) != 0;  // (M == 1 asks)
    if (l == 63) {
      sh->pieces[w] = inc;
      sh->rows[w] = incr;
      sh->tall[w] = tall;
    }
    __syncthreads();
    int p = carry_p + inc - c, q = carry_r + incr - r;
    for (int v = 0; v < 8; ++v) {
      if (v < w) {
        p += sh->pieces[v];
        q += sh->rows[v];
      }
      carry_p += sh->pieces[v];
      carry_r += sh->rows[v];
      carry_s = sh->last[v] >= 0 ? sh->last[v] : carry_s;
    }
#pragma unroll
    for (int j = 0; j < M; ++j) {
      below[j] = p;
      rbelow[j] = q;
      p += pcs[j];
      q += rws[j];
    }
    if (!one_pass) __syncthreads();  // the next pass writes the same memory
  };
  for (int base = 0; base < nblk; base += kPass) pass(base);
  const int total = carry_p * nt;

  int v;
  bool cut_by_cost = false;
  if (M == 1 && one_pass && hmax > kLowRows)
    for (int u = 0; u < 8; ++u) cut_by_cost = cut_by_cost || sh->tall[u];
  if (M == 1 && cut_by_cost) {
    const int64_t all = ((int64_t)kItemCost * carry_p + carry_r) * nt;
    const int per = (total + kNumXcd - 1) / kNumXcd;
#pragma unroll
    for (int j = 0; j < M; ++j) {
      if (pcs[j] + rws[j] == 0) continue;
      const int i0 = below[j] * nt, i1 = i0 + pcs[j] * nt;
      const int64_t k0 = ((int64_t)kItemCost * below[j] + rbelow[j]) * nt, k1 = k0 + ((int64_t)kItemCost * pcs[j] + rws[j]) * nt;
      for (int x = 1; x < 8; ++x) {
        const int64_t pos = all * x / 8;
        if (k0 <= pos && pos < k1) {
          const int in = (int)((float)(pos - k0) / (float)(k1 - k0) * (float)(i1 - i0));
          sh->cut_item[1][x] = i0 + (in < i1 - i0 ? in : i1 - i0);
          sh->cut_cost[1][x] = (float)pos;
        }
        if (i0 <= x * per && x * per < i1)
          sh->cut_cost[0][x] = (float)k0 + (float)(x * per - i0) / (float)(i1 - i0) * (float)(k1 - k0);
      }
    }
    __syncthreads();
    const int q = l % 18, x = q % 9;
    XcdCut cut = {0, 0.0};
    if (x > 0) {
      const bool weighted = q >= 9, inner = x < 8 && (weighted || x * per < total);
      cut.item = inner ? (weighted ? sh->cut_item[1][x] : x * per) : total;
      cut.cost = inner ? sh->cut_cost[weighted][x] : (double)all;
    }
    const XcdPick pick = xcd_better(cut, l < 18, grid / kNumXcd);
    const int at = (pick.weighted ? 9 : 0) + g % kNumXcd;
    v = __shfl(cut.item, at) + g / kNumXcd;
    const int end = __shfl(cut.item, at + 1);
    // (lanes 18.. hold another group's choice)
    v = __builtin_amdgcn_readfirstlane(v);
    if (v >= __builtin_amdgcn_readfirstlane(end)) return false;
  } else {
    v = xcd_item(g, total);
    if (v < 0) return false;
  }

  // the last run whose first item is <= v: block s, items below it ps
  int s = -1, ps = 0, rval = 0, rleft = 0;
  auto find = [&](int base) {
#pragma unroll
    for (int j = 0; j < M; ++j)
      if ((first >> j & 1) && below[j] * nt <= v) {
        s = base + tid * M + j;
        ps = below[j];
        rval = val[j];
        rleft = left[j];
      }
  };
  if (one_pass) {
    find(0);
  } else {
    carry_s = carry_p = carry_r = 0;
    for (int base = 0; base < nblk; base += kPass) {
      pass(base);
      find(base);
    }
  }
  int most = s;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const int other = __shfl_xor(most, o);
    most = other > most ? other : most;
  }
  if (l == 0 && most < 0) sh->run[w] = -1;
  if (most >= 0 && s == most) {
    sh->run[w] = s;
    sh->below[w] = ps;
    sh->val[w] = rval;
    sh->left[w] = rleft;
  }
  __syncthreads();
  int at = 0;
  for (int u = 1; u < 8; ++u) at = sh->run[u] > sh->run[at] ? u : at;
  s = __builtin_amdgcn_readfirstlane(sh->run[at]);
  ps = __builtin_amdgcn_readfirstlane(sh->below[at]);
  rval = __builtin_amdgcn_readfirstlane(sh->val[at]);
  rleft = __builtin_amdgcn_readfirstlane(sh->left[at]);
  // run end: the next run's first block (or nblk)
  int end = -1;
  if (one_pass) {
    for (int w0 = (s + 1) / 32; end < 0; w0 += 64) {
      const int i = w0 + l;
      uint32_t bits = i * 32 < nblk ? sh->firsts[i] : 0;
      if (i == (s + 1) / 32) bits &= ~0u << ((s + 1) % 32);
      const uint64_t m = __ballot(bits != 0);
      if (m) {
        const int lane = __ffsll((unsigned long long)m) - 1;
        end = (w0 + lane) * 32 + __ffs(__builtin_amdgcn_readlane((int)bits, lane)) - 1;
      } else if ((w0 + 64) * 32 >= nblk) {
        end = nblk;
      }
    }
  } else {
    for (int base = s + 1; end < 0; base += 64) {
      const int b = base + l;
      const uint64_t m = __ballot(b >= nblk || gidx[b < nblk ? b : nblk - 1] != rval);
      if (m) end = base + (__ffsll((unsigned long long)m) - 1);
    }
  }
  __syncthreads();  // the caller reuses smem
  it.e = rval >= 0 && rval < E ? rval : -1;
  const int64_t cap = (int64_t)(end - s) * BM;
  const int n = it.e < 0 ? 0 : (int)(rleft > cap ? cap : rleft);
  const int c = n > 0 ? items_of(n, hmax) : 1;
  const int local = v - ps * nt;
  const int t = local / c, i = local % c;
  const int r = n > 0 ? rows_of(n, c) : 0;
  it.row0 = s * BM + i * r;
  it.actual = n - i * r < r ? n - i * r : r;
  it.n0 = t * BN;
  it.zero_end = i == c - 1 ? end * BM : 0;
  it.shared = c > 1;
  return t < nt;
}
__device__ __forceinline__ bool item_bx(int g, const int32_t* __restrict__ gidx, int nblk, int E, int BN, int nt,
                                        const int32_t* __restrict__ gs, const int32_t* __restrict__ gpo, int hmax,
                                        int grid, char* smem, Item& it) {
  return nblk <= 512 ? item_runs<1>(g, gidx, nblk, E, BN, nt, gs, gpo, hmax, grid, smem, it)
                     : item_runs<kScanBlocks>(g, gidx, nblk, E, BN, nt, gs, gpo, hmax, grid, smem, it);
}

// Workgroups of a launch of `blocks` blocks (or row pieces) x `ntiles` items.
inline int64_t schedule_grid(int64_t blocks, int64_t ntiles) {
  const int64_t total = blocks * ntiles;
  const int64_t per = (total + kNumXcd - 1) / kNumXcd;
  return per * kNumXcd;
}

}  // namespace moe
