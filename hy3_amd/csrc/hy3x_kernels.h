// hy3x_kernels.h -- kernel declarations shared by the translation units.
#pragma once
#include "hy3x_common.h"

namespace hy3x {

__global__ void k_router_logits(const float *x, const float *xadd, const float *norm_w,
                                const float *router,
                                const float *bias, int has_bias, float *logits, float *sig,
                                float *score, __half *s16, float *s32, __half *s16m,
                                __half *ssum, unsigned long long *trace, const float *r_in);
__global__ void k_rmsnorm(const float *x, const float *xadd, const float *norm_w, __half *s16,
                          float *s32,
                          __half *s16m, __half *ssum, int T, uint32_t *bits, int wt,
                          const float *r_in);
// Router GEMM shapes by token count, X(up to T, MT, ME, TG, KC, R): a thread of
// k_router_gemm<MT, ME, TG, 8, KC, R> holds MT x ME (token, expert) outputs of one
// chain, a block of 64 TG threads MT TG tokens x 8 ME experts; K is walked in chunks
// of KC floats with R chunks in flight. Every block walks all of K at a pace set by
// LDS latency and its barriers, so up to 1344 tokens the shape is the smallest tile
// whose blocks fit the 256 CUs once (the boundaries: 240 to 256 blocks); eight waves
// hide more of the latency than four where the tile's fetch splits that finely.
// Router stage (RMSNorm + GEMM + top-K) on MI355X, us, the shape taken before (4 x 8
// up to 64 tokens, 8 x 16 to 256, 16 x 24 to 1536, 32 x 32 in four waves to 2560, as
// below above) in brackets:
//   4 x 8    T = 40: 20.4 [22.0]           8 x 8    T = 64: 22.9 [28.2], 75: 23.2 [28.5]
//   8 x 16   T = 160: 26.8 [29.2]          16 x 16  T = 201: 33.2 [36.1], 320: 35.2 [42.0]
//   16 x 24  T = 512: 43.7 (16 x 16: 53.3) 16 x 32  T = 600: 44.7 [60.2]
//   32 x 32  T = 1000: 60.6 [66.9], 1344: 64.6 [86.9] (KC 64, R 4: 73.5 at 1000); with KC
//            64, R 4: T = 2048: 96.9 [112.5] (KC 128: 99.1), 2560: 108.8 [121.0]
//   32 x 48  T = 4096: 164 (64 x 32: 197, 64 x 48 in eight waves: 186)
#define HY3X_ROUTER_SHAPES(X)                                                                  \
  X(40, 1, 1, 4, 256, 2)                                                                       \
  X(80, 1, 1, 8, 256, 2)                                                                       \
  X(168, 2, 2, 4, 256, 2)                                                                      \
  X(336, 2, 2, 8, 128, 2)                                                                      \
  X(512, 4, 3, 4, 128, 1)                                                                      \
  X(672, 2, 4, 8, 128, 2)                                                                      \
  X(1344, 4, 4, 8, 128, 2)                                                                     \
  X(2560, 4, 4, 8, 64, 4)                                                                      \
  X(INT32_MAX, 8, 6, 4, 64, 4)
template <int MT, int ME, int TG, int EG, int KC, int R>
__global__ __launch_bounds__(8 * TG * EG) void k_router_gemm(const float *s32, const float *router,
                                                             int T, float *logits);
#define HY3X_ROUTER_EXTERN(TMAX, MT, ME, TG, KC, R)                                             \
  extern template __global__ void k_router_gemm<MT, ME, TG, 8, KC, R>(const float *, const float *, \
                                                                      int, float *);
HY3X_ROUTER_SHAPES(HY3X_ROUTER_EXTERN)
#undef HY3X_ROUTER_EXTERN
__global__ void k_topk(const float *logits, const float *bias, int has_bias, int K, float scale,
                       int T, int32_t *ids, float *wpre, float *wout, uint32_t *bits, int wt,
                       uint8_t *ranks);
__global__ void k_dispatch_list(const uint8_t *ranks, int T, int K, int NT, const uint32_t *bits,
                                int wt, int32_t *list, int4 *tiles,
                                int32_t *n_tiles, int max_tiles, int NT2, int4 *tiles2,
                                int32_t *n_tiles2, int32_t *counts_out,
                                unsigned long long *stats);
// Up to this many tokens the router runs as one wave per (expert, token)
// (k_router_logits; above as RMSNorm + LDS-tiled GEMM + per-token top-K), and one
// block routes every token and makes the dispatch lists (k_route_small), in one
// launch where top-K, staging and dispatch were three: 2 / 3 / 4 / 8 tokens 73.4 /
// 99.5 / 108.0 / 155.9 -> 64.4 / 90.0 / 98.3 / 145.9 us per forward. It ends where
// one wave per token no longer fits one block; above, s is staged in k_rmsnorm and
// the dispatch alone takes about 4 us. tiles2: the down GEMM's list, of at most NT2
// tokens per tile (0: none).
constexpr int ROUTE_SMALL_T = 8;
__global__ void k_route_small(const float *logits, const float *bias, int has_bias, int K,
                              float scale, int T, int NT, int32_t *ids, float *wpre, float *wout,
                              int32_t *list, int4 *tiles, int32_t *n_tiles, int max_tiles,
                              int NT2, int4 *tiles2, int32_t *n_tiles2, int32_t *counts_out,
                              unsigned long long *stats);
template <int NT>
__global__ void k_gateup_gemv(const uint8_t *wq, const __half *s16, const int32_t *list,
                              const int4 *tiles, const int32_t *n_tiles, int T, int K,
                              __half *h16);
template <int NT>
__global__ void k_down_gemv(const uint8_t *wq, const __half *h16, const int32_t *list,
                            const int4 *tiles, const int32_t *n_tiles, float *out);
__global__ void k_gateup_decode(const uint8_t *wq, const __half *s16, const float *sig,
                                const float *score, int K, float scale, int32_t *ids,
                                float *wpre, float *wout, unsigned long long *stats,
                                __half *h16, unsigned long long *trace);
__global__ void k_route_decode(const float *x, const float *xadd, const float *norm_w,
                               const float *router,
                               const float *bias, int has_bias, int K, float *logits,
                               float *sig, float *score, __half *s16, float *s32,
                               const uint8_t *wq, const uint8_t *wsh, __half *h16,
                               unsigned long long *trace, const float *r_in);
__global__ void k_down_decode(const uint8_t *wq, const __half *h16, const int32_t *ids,
                              const float *w, int K, float *x, const float *xadd,
                              const uint8_t *wsh,
                              unsigned long long *trace);
__global__ void k_stream_read(const uint4 *p, int64_t n16, uint32_t *sink);
__global__ void k_repack_q8x128(const uint8_t *src, uint8_t *dst, int64_t n_super);
__global__ void k_synth_q8_0(uint8_t *dst, int64_t nblocks, uint64_t key, const float *src);
__global__ void k_combine(float *x, const float *xadd, const float *out, const float *w, int T,
                          int K);

extern template __global__ void k_gateup_gemv<1>(const uint8_t *, const __half *, const int32_t *,
                                                 const int4 *, const int32_t *, int, int,
                                                 __half *);
extern template __global__ void k_gateup_gemv<4>(const uint8_t *, const __half *, const int32_t *,
                                                 const int4 *, const int32_t *, int, int,
                                                 __half *);
extern template __global__ void k_down_gemv<1>(const uint8_t *, const __half *, const int32_t *,
                                               const int4 *, const int32_t *, float *);
extern template __global__ void k_down_gemv<4>(const uint8_t *, const __half *, const int32_t *,
                                               const int4 *, const int32_t *, float *);

// Tiles of grid margin for the kernels that deal whole tiles round-robin to
// the XCDs (xcd_tile_rr, hy3x_mfma_ops.h).
constexpr int XCD_TILE_RR_MARGIN = 7;
// The MFMA grouped GEMMs in three shapes (hy3x_mfma.hip, compiled once per
// shape). A work tile has ROWS_GU = 16 WAVES RGU gate/up rows (per matrix) or
// twice as many down rows and up to TOKENS tokens; each wave takes 16 RGU
// gate/up rows or 32 RGU down rows:
//   tiny:   8 tokens, 4 waves -- three workgroups per CU (46 KB of LDS); gate/up
//           of a few tokens;
//   narrow: 32 tokens, 4 waves -- two workgroups per CU; the shape for few
//           tokens per expert;
//   wide:   64 tokens, 8 waves -- one workgroup per CU, half the per-token
//           dequantisation work; the shape for long prefills.
#define HY3X_DECLARE_MFMA(NS, TOK, WV, RGU_)                                                  \
  namespace NS {                                                                            \
  constexpr int TOKENS = TOK, WAVES = WV, RGU = RGU_, ROWS_GU = 16 * WV * RGU_;             \
  template <bool GATEUP>                                                                    \
  __global__ __launch_bounds__(64 * WV) void k_moe_mfma(                                    \
      const uint8_t *wq, const uint8_t *wsh, const __half *act, const __half *act_sum,      \
      const int32_t *list, const int4 *tiles, const int32_t *n_tiles, int T, int K,         \
      __half *h16m, float *out);                                                            \
  extern template __global__ void k_moe_mfma<true>(                                         \
      const uint8_t *, const uint8_t *, const __half *, const __half *, const int32_t *,    \
      const int4 *, const int32_t *, int, int, __half *, float *);                          \
  extern template __global__ void k_moe_mfma<false>(                                        \
      const uint8_t *, const uint8_t *, const __half *, const __half *, const int32_t *,    \
      const int4 *, const int32_t *, int, int, __half *, float *);                          \
  }
HY3X_DECLARE_MFMA(mfma_tiny, 8, 4, 1)
HY3X_DECLARE_MFMA(mfma_narrow, 32, 4, 1)
HY3X_DECLARE_MFMA(mfma_wide, 64, 8, 1)
#undef HY3X_DECLARE_MFMA
// 128-token tiles for experts holding many tokens (hy3x_mfma_big.hip): the
// MFMA tiles' arithmetic, each wave's dequantised
// weights reused over up to eight 16-token column groups.
constexpr int BIG_TOKENS = 128, BIG_WAVES = 8;
namespace mfma_big {
template <bool GATEUP>
__global__ __launch_bounds__(64 * BIG_WAVES) void k_moe_big(
    const uint8_t *wq, const uint8_t *wsh, const __half *act, const __half *act_sum,
    const int32_t *list, const int4 *tiles, const int32_t *n_tiles, int T, int K, __half *h16m,
    float *out);
extern template __global__ void k_moe_big<true>(const uint8_t *, const uint8_t *, const __half *,
                                                const __half *,
                                                const int32_t *, const int4 *, const int32_t *,
                                                int, int, __half *, float *);
extern template __global__ void k_moe_big<false>(const uint8_t *, const uint8_t *,
                                                 const __half *, const __half *,
                                                 const int32_t *, const int4 *, const int32_t *,
                                                 int, int, __half *, float *);
}  // namespace mfma_big
// The down GEMM for few tokens per expert (hy3x_mfma_few.hip): work tiles of
// 16 FEW_WAVES rows and up to FEW_TOKENS tokens (up to FEW_ROWS: their h rows
// whole in LDS).
constexpr int FEW_TOKENS = 32, FEW_ROWS = 4, FEW_WAVES = 4;
__global__ void k_down_few(const uint8_t *wq, const uint8_t *wsh, const __half *act,
                           const __half *act_sum, const int32_t *list, const int4 *tiles,
                           const int32_t *n_tiles, int T, float *out);
__global__ void k_hsums(const __half *h16m, __half *hsum);

__global__ void k_synth_q4k(uint8_t *dst, int64_t nblocks, uint64_t seed, uint32_t layer,
                            const float *src);

}  // namespace hy3x
