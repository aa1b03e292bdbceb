// Internal launcher interface between the C ABI (capi.hip) and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

// Fused Stage 2 scatter-reduce (1): each weighted pair row is added straight
// into its token's fp16 output row with packed fp16 atomics (the output is
// zeroed first, and no combine runs), instead of (0, the default) a per-pair
// row that the deterministic combine sums in choice order.  Off by default:
// device-scope atomics on MI355X run far below plain stores.  A/B in one run
// (2 x 2 interleaved): dsv3's step 5.26 -> 5.61 ms (Stage 2 1.855 -> 2.321 ms
// against the combine's 0.090), mixtral 1.543 -> 1.583, w8a8 int8 0.890 ->
// 1.178, fp8 0.833 -> 1.124, decode level (0.501 -> 0.499).  And the order of
// the additions, so the fp16 rounding of the sum, varies from call to call.
#ifndef MOE_S2_SCATTER
#define MOE_S2_SCATTER 0
#endif

namespace moe {

// Operand formats of the expert GEMMs: fp16, or 8-bit codes with fp32 row
// scales -- int8 (i8 MFMA, int32 accumulation) or OCP fp8 e4m3 (f8 MFMA, fp32
// accumulation).
enum QuantType : int { kQF16 = 0, kQI8 = 1, kQF8 = 2 };

// The wide items of a fused launch (moe_common.h Item) are planned by align from
// the routed rows themselves: the height of each stage's tallest item, and how
// many features Stage 2's take.  A launch of few rounds ends when its slowest
// CU does, which depends on how the counts fall: 16 experts of H 4096, I 2048 at
// 1500 tokens top-2 with Zipf popularity ran Stage 1 in 217 us in items of up to
// 288 rows, 182 in 128 and 168 in 192, and 138, 142 and 128 (224 rows) on an even
// routing.  `out`, int32: [E+1] items per N tile below each expert for Stage 1,
// [E+1] for Stage 2, the 9 XCD bounds of each, Stage 2's features per item.
struct ItemPlan {
  int32_t* out = nullptr;  // null: no plan
  int tall = 0;            // rows of the tallest item
  int nt1 = 0, nt2 = 0;    // N tiles of Stage 1, and of Stage 2 at 128 features
  bool any1 = false, any2 = false;  // may take shorter items (moe_common.h plan_height)
  int bn2 = 0;             // Stage 2's features per item: 128, 256 or either (0)
  int slots1 = 0, slots2 = 0;  // workgroups of each stage's launch per XCD: what a choice has to fit in

  static constexpr int64_t ints(int64_t E) { return 2 * E + 21; }
  static constexpr int64_t istart2(int64_t E) { return E + 1; }
  static constexpr int64_t xb1(int64_t E) { return 2 * E + 2; }
  static constexpr int64_t xb2(int64_t E) { return 2 * E + 11; }
  static constexpr int64_t bn(int64_t E) { return 2 * E + 20; }
};

// Stage 1: h = silu(X Wg^T) * (X Wu^T) for the rows of every M block.
struct Stage1Params {
  const char* x;            // fp16 [rows, H] (direct) / fp16|int8 [T, H] (gather)
  const char* wg;           // [E, I, H]
  const char* wu;           // [E, I, H]
  char* h;                  // fp16 [padded rows, I] (fp16 and int8 operands) | fp8 [padded rows, I]
  uint8_t* h_scale;         // fp8 only: E8M0 bytes [padded rows][hs_pitch], one per 128 columns
  int64_t hs_pitch;         // fp8 only: bytes between rows of h_scale, a multiple of 16
  const float* x_scale;     // 8-bit only: [T]
  const float* sg;          // 8-bit only: [E, I]
  const float* su;          // 8-bit only: [E, I]
  const int32_t* gs;        // [E]
  const int32_t* gpo;       // [E+1]
  const int32_t* sorted_ids;  // gather only: [padded rows], sentinel = T*topk
  const int32_t* gidx;      // direct only: block -> expert ([host_blocks] entries)
  const char* wg_shared;    // weights of expert e_shared ([I, H]) when e_shared >= 0
  const char* wu_shared;
  int e_shared = -1;        // always-on shared expert's index, or -1
  int64_t w_ld = 0;         // bytes between rows of wg / wu / the shared ones (0: H elements)
  int64_t w_es = 0;         // bytes between experts of wg / wu (0: I rows)
  int64_t h_ld = 0;         // elements between rows of h (0: I)
  int topk;
  int E;
  int64_t H;
  int64_t I;
  int host_blocks;          // narrow: 32-row blocks the row buffers hold; direct: blocks of
                            // the launch (gidx entries, clamped); set by the launcher
  const int32_t* istart = nullptr;  // wide, gather: [E+1] items per N tile below each expert
  const int32_t* xb = nullptr;      // wide, gather: [9] first item of each XCD
  int rows_cap = 0;         // wide, gather: rows the buffers hold
  int hmax = 0;             // wide, direct: most rows of an item (moe_common.h Item)
  bool stream = true;       // wide, and fp8 of 32-row tiles: weights that no other item reads non-temporal
};

// Stage 2: y = h Wd^T, scaled by the routing weight of each row.
struct Stage2Params {
  const char* a;            // fp16|int8|fp8 [padded rows, I]
  const float* a_scale;     // int8: [padded rows] (per row)
  const uint8_t* a_scale8;  // fp8: E8M0 bytes [padded rows][as_pitch], one per 128 columns
  int64_t as_pitch;         // fp8: bytes between rows of a_scale8, a multiple of 16
  const char* wd;           // [E, H, I]
  const float* sd;          // 8-bit only: [E, H]
  char* out;                // pre-routed: fp16 [P, H]; fused: fp16 [T*topk, H], row = the pair's
                            // unpadded expert-sorted position go[e] + (row - gpo[e])
  int32_t* pos;             // fused only: pos[pair] = that row (written by the first N tile's items)
  const void* routed;       // pre-routed: [V] raw order (fp32|fp16); fused: fp32 [T*topk]
  int routed_f16;
  const int32_t* gs;
  const int32_t* go;
  const int32_t* gpo;
  const int32_t* sorted_ids;  // fused only
  const int32_t* gidx;      // pre-routed only: block -> expert ([host_blocks] entries)
  const char* wd_shared;    // down weights of expert e_shared ([H, I]) when e_shared >= 0
  int e_shared = -1;        // always-on shared expert's index, or -1
  int64_t a_ld = 0;         // bytes between rows of a (0: I elements)
  int64_t wd_ld = 0;        // bytes between rows of wd / wd_shared (0: I elements)
  int64_t wd_es = 0;        // bytes between experts of wd (0: H rows)
  int E;
  int64_t H;
  int64_t I;
  int64_t V;                // pre-routed: entries of `routed` (raw index is clamped to V-1)
  int host_blocks;          // as Stage 1's
  const int32_t* istart = nullptr;
  const int32_t* xb = nullptr;
  const int32_t* bn_plan = nullptr;  // wide, fused: features of an item, 128 or 256 (the plan's)
  int bn = 0;               // wide: features of an item, 128 or 256; fused, 0: either, as bn_plan says
  int rows_cap = 0;
  int hmax = 0;
  bool stream = true;       // wide: as Stage 1's
  int topk = 0;             // fused, built with MOE_S2_SCATTER: choices per token; `out` is then
                            // fp16 [T, H] (zeroed first) and each pair row is added to its token's
                            // row with packed fp16 atomics
};

// Zeroes n bytes (n a multiple of 16, p 16-byte aligned) with vector stores:
// a kernel, not hipMemsetAsync, so that it can be captured in a graph.
hipError_t launch_zero(void* p, int64_t n, hipStream_t stream);

// qt: a QuantType.  narrow: 32-row items over rows padded to 32 (gather / fused
// only); otherwise wide items.  max_blocks: narrow, 32-row blocks of the launch
// at most; wide, the plan's slots (gather / fused) or 128-row blocks (pre-routed).
hipError_t launch_stage1(const Stage1Params& p, bool narrow, int qt, bool gather,
                         int64_t max_blocks, hipStream_t stream);
hipError_t launch_stage2(const Stage2Params& p, bool narrow, int qt, bool fused,
                         int64_t max_blocks, hipStream_t stream);

// With e_shared >= 0 every token also gets the shared expert as choice k
// (id e_shared, weight 1): ids / w rows hold k + 1 entries.
hipError_t launch_route_topk(const float* logits, const float* bias, int T, int E, int k,
                             int32_t* ids, float* w, hipStream_t stream, int e_shared = -1);
// `whist` (int32 [align_groups(P) * E], may be null) lets a large P be aligned
// by align_groups(P) workgroups in two launches instead of one workgroup.
constexpr int kAlignPairsPerGroup = 2048;
constexpr int kAlignMaxGroups = 64;
// (below 4 groups' worth of pairs the second launch costs more than it saves)
inline int align_groups(int P) {
  const int g = (P + kAlignPairsPerGroup - 1) / kAlignPairsPerGroup;
  return g < 4 ? 1 : (g > kAlignMaxGroups ? kAlignMaxGroups : g);
}
// pairs per workgroup: a multiple of 64 * nw covering P in `groups` workgroups
inline int align_pairs_per_group(int P, int groups, int nw) {
  const int per = (P + groups - 1) / groups;
  return (per + 64 * nw - 1) / (64 * nw) * (64 * nw);
}
// e_off: pairs are bucketed by id - e_off; ids outside [e_off, e_off + E)
// are dropped (an expert shard of a wider routing).  With `plan.out` the wide
// items' plan is written there (moe_common.h ItemPlan).
hipError_t launch_align(const int32_t* ids, int P, int E, int BM, int32_t* sorted_ids,
                        int32_t* block_expert, int32_t* gs, int32_t* go, int32_t* gpo,
                        int32_t* whist, hipStream_t stream, int e_off = 0, const ItemPlan& plan = ItemPlan{});
// launch_route_topk and launch_align in one launch, for small batches (see
// route_align_kernel); false, with nothing launched, for others.
bool launch_route_align(const float* logits, const float* bias, int T, int E_route, int k, int32_t* ids, float* w,
                        int e_shared, int E, int BM, int32_t* sorted_ids, int32_t* block_expert, int32_t* gs,
                        int32_t* go, int32_t* gpo, hipStream_t stream, int e_off, const ItemPlan& plan, hipError_t* err);
// Router GEMM (x . w_router^T, K split in router_splits parts) + routing of
// the summed partials; `part` holds router_partial_floats fp32, `logits`
// (fp32 [T, E]) may be null.
int router_splits(int64_t T, int64_t H, int64_t E);
int64_t router_partial_floats(int64_t T, int64_t H, int64_t E);
hipError_t launch_router(const void* x, const void* w_router, const float* bias, int T, int64_t H, int E,
                         int k, int32_t* ids, float* w, float* logits, float* part, hipStream_t stream,
                         int e_shared = -1);
// ids (may be null): sum only pairs whose expert is in [e_lo, e_lo + e_n).
// y_pair row of pair t*k + j: pos[t*k + j].
hipError_t launch_combine(const void* y_pair, const int32_t* pos, int64_t T, int64_t H, int k, void* out,
                          hipStream_t stream, const int32_t* ids = nullptr, int e_lo = 0, int e_n = 0);
// Routing (as launch_route_topk, no shared expert) and the per-token 8-bit
// quantisation of x [T, H] (as launch_quant_rows) in one launch.
hipError_t launch_route_quant(const float* logits, const float* bias, int T, int E, int k, int32_t* ids,
                              float* w, const void* x, int64_t H, void* xq, float* sx, int qt,
                              hipStream_t stream);
// Per-row 8-bit quantisation of an fp16 [R, K] matrix to the format qt
// (kQI8 or kQF8): codes into q, amax / qmax into scale.  With `ids` set only
// rows r < *used_rows (a device value) with ids[r] < sentinel are quantised
// (the int8 intermediate: rows in the expert-sorted space).
hipError_t launch_quant_rows(const void* w, int64_t R, int64_t K, void* q, float* scale, int qt,
                             hipStream_t stream, const int32_t* ids = nullptr, int32_t sentinel = 0,
                             const int32_t* used_rows = nullptr);

}  // namespace moe
