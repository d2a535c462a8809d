// hy3x_mfma_few.hip -- the grouped down GEMM for few tokens per expert: a wave's
// whole weight rows in registers.
//
// With few tokens per expert the down GEMM is bound by how the weights stream:
// the narrow MFMA tiles (hy3x_mfma.hip) walk 128-row tiles column by column, 144
// bytes of each row at a time with one or two columns in flight, and their six
// columns hardly outlast the start of the pipeline. A down row is only 864 bytes,
// so here a wave takes 16 rows and requests all of them at once, straight into
// its registers (72 VGPRs per lane; every 128-byte line is requested once and
// used whole). A workgroup is four such waves, four workgroups per CU.
//
// A work tile has up to FEW_TOKENS = 32 tokens, two MFMA row groups, so an expert with
// n tokens has its rows read and dequantised ceil(n / 32) times. Up to FEW_ROWS = 4
// tokens the tokens' h rows are staged in LDS whole and the reduction has no barrier;
// above, whole rows would leave no room for four workgroups, and they are staged a
// column at a time. Down launch where every token chooses the same eight experts, at
// 16 / 24 / 32 / 48 tokens: narrow tiles 14.9 / 16.4 / 17.0 / 21.3 us, here 15.1 / 17.3 /
// 17.8 / 21.4; with tiles of up to 16 tokens 14.7 / 18.6 / 18.9 / 22.8; of up to 4 about
// 1.5 to 2.6 times the narrow tiles'. (All of up to 8, rows whole: evenly spread 42 and
// 65 us at 8 and 16.) With a Q8 shared expert there 17.8 and 20.8 us at 32 and 40, here
// 20.3 and 21.6 (tiles of 16: 20.6 and 25.8): a Q8 row does not fit the registers.
//
// Down launch, weights from HBM, evenly spread over the experts, narrow tiles and
// here: 3 tokens 24.8 and 19.6 us, 8: 47.5 and 38.0, 16: 72.2 and 57.6, 32: 93.3 and
// 79.3, 48: 105.7 and 96.5. Measured beside it: the columns one, two or three at a
// time through a register ring slower than the narrow tiles at 8 tokens, two or
// eight waves per workgroup 2-8 % slower, three column pairs of a Q8 row in flight
// instead of two spill.
//
// The arithmetic per element is the MFMA tiles': the same operands, k order and
// sequence of operations on every accumulator (hy3x_mfma.hip's header), so a
// token's result is the same bits. Lane l holds weight row l % 16 of the wave's
// and, of each half of a block, the 16 qs bytes of piece l / 16. The LDS row
// strides spread the rows over the banks; MFMA rows past the tile's tokens are
// zero or repeat others, and are never stored.
#include "hy3x_mfma_ops.h"
#include "hy3x_q8.h"

namespace hy3x {

constexpr int FW_NKB = F / QK;                 // Q4_K columns of a down row (6)
constexpr int FW_XC = F * 2 / 16;              // 16-byte chunks of an h row (192)
constexpr int FW_SC = F / 32 * 8 / 16;         // and of its sums (24)
constexpr int FW_XROW = FW_XC + 4, FW_SROW = FW_SC + 4;  // LDS row strides, whole rows
constexpr int FW_CXC = FW_XC / FW_NKB, FW_CSC = FW_SC / FW_NKB;  // chunks of one column (32, 4)
constexpr int FW_CXROW = FW_CXC + 1, FW_CSROW = FW_CSC + 1;      // LDS row strides, one column
constexpr int FW_COL = 16 * (FW_CXROW + FW_CSROW);  // one column of a row group in LDS
constexpr int FW_GROUPS = FEW_TOKENS / 16;          // MFMA row groups of a tile
constexpr int FW_THREADS = 64 * FEW_WAVES;
constexpr int FW_LDS = 2 * FW_GROUPS * FW_COL;
static_assert(FW_GROUPS == 2 && FEW_ROWS <= 16 && (FEW_ROWS & (FEW_ROWS - 1)) == 0, "row groups");
static_assert(FEW_ROWS * (FW_XROW + FW_SROW) <= FW_LDS, "whole rows");

// A lane's part of its whole down row in Q4_K.
struct FewRow {
  u4_t hdr[FW_NKB], q[FW_NKB][2];
  __device__ __forceinline__ void request(const uint8_t *wrow, int g) {
#pragma unroll
    for (int kb = 0; kb < FW_NKB; kb++) {
      const u4_t *p = reinterpret_cast<const u4_t *>(wrow + (size_t)kb * QB);
      hdr[kb] = p[0];
      q[kb][0] = p[1 + g];
      q[kb][1] = p[5 + g];
    }
  }
  // column kb of NG row groups, each dequantised weight used for all of them: xc its
  // 32 chunks of this lane's MFMA row and sc the lane's sums, xs and ss from one
  // group's to the next's
  template <int NG>
  __device__ __forceinline__ void column(int kb, const u4_t *xc, int xs, const u4_t *sc, int ss,
                                         int g, f4_t (&acc)[NG]) const {
    const uint32_t sel = bytes_sel(g >> 1), msel = bytes_sel(g & 1);
    const int gch = 8 * (g >> 1) + 2 * (g & 1);
    const Scales6 s6 = unpack_scales(hdr[kb]);
    f4_t dblk[NG];
#pragma unroll
    for (int r = 0; r < NG; r++) dblk[r] = (f4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int piece = 0; piece < 2; piece++) {
      const PairScale ps = pair_scale(s6.sc[piece], sel);
      h8_t wf[4];  // [2h + u]
      dequant_run(q[kb][piece].xy, ps, wf[0], wf[2]);
      dequant_run(q[kb][piece].zw, ps, wf[1], wf[3]);
#pragma unroll
      for (int hu = 0; hu < 4; hu++)
#pragma unroll
        for (int r = 0; r < NG; r++)
          dblk[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(h8_t,
                                 xc[r * xs + 16 * piece + 4 * (hu >> 1) + (hu & 1) + gch]),
              wf[hu], dblk[r], 0, 0, 0);
    }
    const h8_t mo = mins_operand(hdr[kb].x, (g >> 1) ? s6.mn[1] : s6.mn[0], msel);
    const float d = fp16_quirk(hdr[kb].x & 0xffffu);
#pragma unroll
    for (int r = 0; r < NG; r++) {
      acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, sc[r * ss]), mo,
                                                      acc[r], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) acc[r][i] = __builtin_fmaf(d, dblk[r][i], acc[r][i]);
    }
  }
};

// A lane's part of one 144-byte column (128 of K) of a down row in Q8.
struct FewQ8 {
  f4_t dsc;
  u2_t q[4];
  __device__ __forceinline__ void request(const uint8_t *p, int g) {
    dsc = *reinterpret_cast<const f4_t *>(p);
#pragma unroll
    for (int b = 0; b < 4; b++) q[b] = *reinterpret_cast<const u2_t *>(p + 16 + 32 * b + 8 * g);
  }
  // xc: the column's 16 chunks of this lane's MFMA row, xs from one group's to the next's
  template <int NG>
  __device__ __forceinline__ void column(const u4_t *xc, int xs, int g, f4_t (&acc)[NG]) const {
    const f4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const h8_t wf = q8_run(q[b]);
#pragma unroll
      for (int r = 0; r < NG; r++) {
        const f4_t pr = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            __builtin_bit_cast(h8_t, xc[r * xs + 4 * b + g]), wf, zero4, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[r][i] = __builtin_fmaf(dsc[b], pr[i], acc[r][i]);
      }
    }
  }
};

// acc of row group r: lane holds D[token 16 r + 4g + i][its row].
__device__ __forceinline__ void few_store(const f4_t &acc, int r, const int32_t *slots, int n,
                                          int g, int row, float *out) {
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (16 * r + 4 * g + i < n) out[(size_t)slots[16 * r + 4 * g + i] * D + row] = acc[i];
}

// A tile of more than FEW_ROWS tokens, in NG row groups: its rows would not fit LDS
// whole beside three other workgroups, so they are staged a column at a time (two
// buffers, a third column in registers), 16 threads per token of a group; tokens past
// the tile's repeat its last. The weights are requested after those and stay whole in
// registers.
template <bool Q8, int NG>
__device__ __forceinline__ void few_tile_columns(const uint8_t *wrow, const __half *act,
                                                 const __half *act_sum, const int32_t *slots,
                                                 int n, int row, float *out, u4_t *lds) {
  constexpr int COL = NG * FW_COL, XG = 16 * FW_CXROW, SG = 16 * FW_CSROW;
  const int tid = threadIdx.x, lr = tid & 15, g = (tid >> 4) & 3;
  // the thread's chunks c and c + 16 of token t of every group, and part cs of the sums
  // of token ts (four lanes hold the same, or two of either group)
  const int t = tid >> 4, c = tid & 15, cs = c & (FW_CSC - 1), ts = t + 16 * ((c >> 2) % NG);
  static_assert(FW_THREADS == 16 * 16 && FW_CXC == 32 && FW_CSC == 4 && NG <= 2, "staging split");
  struct Col {
    u4_t x[NG][2], s;
  };
  const char *ab = reinterpret_cast<const char *>(act);
  const char *sb = reinterpret_cast<const char *>(act_sum);
  uint32_t xo[NG];
#pragma unroll
  for (int r = 0; r < NG; r++)
    xo[r] = (uint32_t)(slots[min(16 * r + t, n - 1)] * (F * 2) + 16 * c);
  const uint32_t so = (uint32_t)(slots[min(ts, n - 1)] * (F / 32 * 8) + 16 * cs);
  auto request = [&](int kb) {
    Col o;
#pragma unroll
    for (int r = 0; r < NG; r++) {
      o.x[r][0] = *reinterpret_cast<const u4_t *>(ab + (xo[r] + kb * (16 * FW_CXC)));
      o.x[r][1] = *reinterpret_cast<const u4_t *>(ab + (xo[r] + kb * (16 * FW_CXC) + 256));
    }
    if (!Q8) o.s = *reinterpret_cast<const u4_t *>(sb + (so + kb * (16 * FW_CSC)));
    return o;
  };
  auto stage = [&](int kb, const Col &o) {
    u4_t *b = lds + (kb & 1) * COL;
#pragma unroll
    for (int r = 0; r < NG; r++) {
      b[r * XG + t * FW_CXROW + c] = o.x[r][0];
      b[r * XG + t * FW_CXROW + c + 16] = o.x[r][1];
    }
    if (!Q8) b[NG * XG + ts * FW_CSROW + cs] = o.s;
  };
  const Col c0 = request(0), c1 = request(1);
  Col next;
  auto stage_first = [&] {
    __builtin_amdgcn_sched_barrier(0);
    stage(0, c0);
    stage(1, c1);
    __syncthreads();
  };
  f4_t acc[NG];
#pragma unroll
  for (int r = 0; r < NG; r++) acc[r] = (f4_t){0.f, 0.f, 0.f, 0.f};
  if constexpr (Q8) {
    // After column kb: once every wave has read its buffer, kb + 2 goes there (read
    // after the barrier of kb + 1). The last two columns stage one more, which nothing
    // reads.
    next = request(2);
    constexpr int QD = 2;  // column pairs (256 of K) in flight
    static_assert(FW_NKB % QD == 0, "whole rounds of the ring");
    FewQ8 w[QD][2];
    auto request_w = [&](int kb, FewQ8 (&o)[2]) {
#pragma unroll
      for (int j = 0; j < 2; j++) o[j].request(wrow + (size_t)(2 * kb + j) * QB, g);
    };
#pragma unroll
    for (int i = 0; i < QD; i++) request_w(i, w[i]);
    stage_first();
#pragma unroll 1
    for (int k0 = 0; k0 < FW_NKB; k0 += QD)
#pragma unroll
      for (int i = 0; i < QD; i++) {
        const int kb = k0 + i;
        const u4_t *xc = lds + (kb & 1) * COL + lr * FW_CXROW;
#pragma unroll
        for (int j = 0; j < 2; j++) w[i][j].column(xc + 16 * j, XG, g, acc);
        request_w(min(kb + QD, FW_NKB - 1), w[i]);
        __syncthreads();
        stage(kb, next);
        next = request(min(kb + 3, FW_NKB - 1));
      }
  } else {
    FewRow w;
    w.request(wrow, g);
    stage_first();
#pragma unroll
    for (int kb = 0; kb < FW_NKB; kb++) {
      const u4_t *b = lds + (kb & 1) * COL;
      w.column(kb, b + lr * FW_CXROW, XG, b + NG * XG + lr * FW_CSROW + g, SG, g, acc);
      // column kb + 1 goes to the buffer that every wave had read at the last barrier;
      // kb + 2 is requested as late as that, when column kb's weights have made room
      if (kb >= 1 && kb + 1 < FW_NKB) stage(kb + 1, next);
      if (kb + 1 < FW_NKB) __syncthreads();
      if (kb + 2 < FW_NKB) next = request(kb + 2);
    }
  }
#pragma unroll
  for (int r = 0; r < NG; r++) few_store(acc[r], r, slots, n, g, row, out);
}

// A tile of at most FEW_ROWS tokens: its rows in LDS whole, one barrier.
template <bool Q8>
__device__ __forceinline__ void few_tile_rows(const uint8_t *wrow, const __half *act,
                                              const __half *act_sum, const int32_t *slots, int n,
                                              int row, float *out, u4_t *lds) {
  const int tid = threadIdx.x, lr = tid & 15, g = (tid >> 4) & 3;
  u4_t *x_l = lds, *s_l = lds + FEW_ROWS * FW_XROW;
  // staging: 64 threads per token. Every row is written (zeros past the tile's
  // tokens): loads used only under a condition would be moved behind it, and so
  // behind the weights.
  constexpr int TT = FW_THREADS / FEW_ROWS, XL = FW_XC / TT;
  static_assert(XL * TT == FW_XC && FW_SC <= TT, "staging split");
  const int t = tid / TT, c0 = tid % TT;
  u4_t xv[XL], sv = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int u = 0; u < XL; u++) xv[u] = (u4_t){0u, 0u, 0u, 0u};
  if (t < n) {
    const int slot = slots[t];
    const char *xs = reinterpret_cast<const char *>(act);
    const char *ss = reinterpret_cast<const char *>(act_sum);
#pragma unroll
    for (int u = 0; u < XL; u++)
      xv[u] = *reinterpret_cast<const u4_t *>(xs + (uint32_t)(slot * (F * 2) + 16 * (c0 + TT * u)));
    sv = *reinterpret_cast<const u4_t *>(
        ss + (uint32_t)(slot * (F / 32 * 8) + 16 * min(c0, FW_SC - 1)));
  }
  auto stage = [&] {
#pragma unroll
    for (int u = 0; u < XL; u++) x_l[t * FW_XROW + c0 + TT * u] = xv[u];
    s_l[t * FW_SROW + min(c0, FW_SC - 1)] = sv;
    __syncthreads();
  };
  const u4_t *xr = x_l + (lr & (FEW_ROWS - 1)) * FW_XROW;
  const u4_t *sr = s_l + (lr & (FEW_ROWS - 1)) * FW_SROW;
  f4_t acc[1] = {{0.f, 0.f, 0.f, 0.f}};
  if constexpr (Q8) {  // 128 of K per 144-byte column
    stage();
#pragma unroll 4
    for (int kb = 0; kb < F / Q8K; kb++) {
      FewQ8 w8;
      w8.request(wrow + (size_t)kb * QB, g);
      w8.column(xr + 16 * kb, 0, g, acc);
    }
  } else {
    // the rows were requested before the weights (loads complete in the order they
    // were issued): they are staged while the weights arrive, and column kb is
    // computed when it is there
    FewRow w;
    w.request(wrow, g);
    __builtin_amdgcn_sched_barrier(0);
    stage();
#pragma unroll
    for (int kb = 0; kb < FW_NKB; kb++)
      w.column(kb, xr + FW_CXC * kb, 0, sr + FW_CSC * kb + g, 0, g, acc);
  }
  few_store(acc[0], 0, slots, n, g, row, out);
}

__global__ __launch_bounds__(FW_THREADS, 4) void k_down_few(
    const uint8_t *__restrict__ wq, const uint8_t *__restrict__ wsh,
    const __half *__restrict__ act, const __half *__restrict__ act_sum,
    const int32_t *__restrict__ list, const int4 *__restrict__ tiles,
    const int32_t *__restrict__ n_tiles, int T, float *__restrict__ out) {
  constexpr int TROWS = 16 * FEW_WAVES, NRT = D / TROWS;
  __shared__ __attribute__((aligned(16))) u4_t lds[FW_LDS];
  const int nreal = *n_tiles * NRT;
  if ((int)blockIdx.x >= nreal) return;
  const int w = xcd_remap(blockIdx.x, nreal, (T + FEW_TOKENS - 1) / FEW_TOKENS * NRT);
  const int4 td = tiles[w / NRT];
  const int e = td.x, n = td.z;
  const int tid = threadIdx.x, lr = tid & 15;
  const bool q8 = wsh != nullptr && e == E;
  const int row = w % NRT * TROWS + 16 * (tid >> 6) + lr;
  const uint8_t *wrow = q8 ? wsh + 2 * Q8_MAT_BYTES + (size_t)row * (F / Q8K) * QB
                           : wq + (size_t)e * EXPERT_BYTES + 2 * MAT_BYTES +
                                 (size_t)row * FW_NKB * QB;
  const int32_t *slots = list + td.y;
  if (n <= FEW_ROWS) {
    if (q8)
      few_tile_rows<true>(wrow, act, act_sum, slots, n, row, out, lds);
    else
      few_tile_rows<false>(wrow, act, act_sum, slots, n, row, out, lds);
  } else if (n <= 16) {
    if (q8)
      few_tile_columns<true, 1>(wrow, act, act_sum, slots, n, row, out, lds);
    else
      few_tile_columns<false, 1>(wrow, act, act_sum, slots, n, row, out, lds);
  } else if (q8) {
    few_tile_columns<true, 2>(wrow, act, act_sum, slots, n, row, out, lds);
  } else {
    few_tile_columns<false, 2>(wrow, act, act_sum, slots, n, row, out, lds);
  }
}

}  // namespace hy3x
