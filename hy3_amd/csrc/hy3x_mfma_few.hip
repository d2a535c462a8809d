// hy3x_mfma_few.hip -- the grouped down GEMM for few tokens per expert: a wave's
// whole weight rows in registers, no barrier in the reduction.
//
// With few tokens per expert the down GEMM is bound by how the weights stream:
// the narrow MFMA tiles (hy3x_mfma.hip) walk 128-row tiles column by column, 144
// bytes of each row at a time with one or two columns in flight, and their six
// columns hardly outlast the start of the pipeline. A down row is only 864 bytes,
// so here a wave takes 16 rows and requests all of them at once, straight into
// its registers (72 VGPRs per lane; every 128-byte line is requested once and
// used whole). A workgroup is four such waves, four workgroups per CU.
//
// A work tile has up to FEW_TOKENS = 16 tokens, one MFMA row group, so an expert
// with n tokens has its rows read and dequantised ceil(n / 16) times. Up to
// FEW_ROWS = 4 tokens the tokens' h rows are staged in LDS whole and the reduction
// has no barrier; above, whole rows would leave no room for four workgroups, and
// they are staged a column at a time. (All tiles of up to 4 tokens: every token on
// the same eight experts 25.1 / 42.7 / 59.0 us at 16 / 32 / 48 tokens, 16.6 / 20.6 /
// 26.0 now, the narrow tiles 16.3 / 19.0 / 22.2; all of up to 8, rows whole: evenly
// spread 42 and 65 us at 8 and 16.)
//
// Down launch, weights from HBM, evenly spread over the experts, narrow tiles and
// here: 3 tokens 27.3 and 22.7 us, 8: 48.5 and 39.7, 16: 71.6 and 58.4, 32: 94.5 and
// 81.9, 48: 107.6 and 97.1. Measured beside it: the columns one, two or three at a
// time through a register ring slower than the narrow tiles at 8 tokens, two or
// eight waves per workgroup 2-8 % slower.
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
constexpr int FW_COL = FEW_TOKENS * (FW_CXROW + FW_CSROW);       // one column of a tile in LDS
constexpr int FW_THREADS = 64 * FEW_WAVES;
constexpr int FW_LDS = FEW_ROWS * (FW_XROW + FW_SROW) > 2 * FW_COL
                           ? FEW_ROWS * (FW_XROW + FW_SROW) : 2 * FW_COL;
static_assert(FEW_TOKENS == 16 && (FEW_ROWS & (FEW_ROWS - 1)) == 0, "one MFMA row group");

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
  // column kb: xc its 32 chunks of this lane's MFMA row, sv the lane's sums
  __device__ __forceinline__ f4_t column(int kb, const u4_t *xc, u4_t sv, int g, f4_t acc) const {
    const uint32_t sel = bytes_sel(g >> 1), msel = bytes_sel(g & 1);
    const int gch = 8 * (g >> 1) + 2 * (g & 1);
    const Scales6 s6 = unpack_scales(hdr[kb]);
    f4_t dblk = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int piece = 0; piece < 2; piece++) {
      const PairScale ps = pair_scale(s6.sc[piece], sel);
      h8_t wf[4];  // [2h + u]
      dequant_run(q[kb][piece].xy, ps, wf[0], wf[2]);
      dequant_run(q[kb][piece].zw, ps, wf[1], wf[3]);
#pragma unroll
      for (int hu = 0; hu < 4; hu++)
        dblk = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            __builtin_bit_cast(h8_t, xc[16 * piece + 4 * (hu >> 1) + (hu & 1) + gch]), wf[hu],
            dblk, 0, 0, 0);
    }
    const h8_t mo = mins_operand(hdr[kb].x, (g >> 1) ? s6.mn[1] : s6.mn[0], msel);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, sv), mo, acc, 0, 0, 0);
    const float d = fp16_quirk(hdr[kb].x & 0xffffu);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(d, dblk[i], acc[i]);
    return acc;
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
  // xc: the column's 16 chunks of this lane's MFMA row
  __device__ __forceinline__ f4_t column(const u4_t *xc, int g, f4_t acc) const {
    const f4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const f4_t pr = __builtin_amdgcn_mfma_f32_16x16x32_f16(
          __builtin_bit_cast(h8_t, xc[4 * b + g]), q8_run(q[b]), zero4, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(dsc[b], pr[i], acc[i]);
    }
    return acc;
  }
};

// A tile of more than FEW_ROWS tokens: its rows would not fit LDS whole beside
// three other workgroups, so they are staged a column at a time (two buffers, a
// third column in registers), 16 threads per token; tokens past the tile's repeat
// its last. The weights are requested after those and stay whole in registers.
template <bool Q8>
__device__ __forceinline__ f4_t few_tile_columns(const uint8_t *wrow, const __half *act,
                                                 const __half *act_sum, const int32_t *slots,
                                                 int n, u4_t *lds) {
  const int tid = threadIdx.x, lr = tid & 15, g = (tid >> 4) & 3;
  const int t = tid >> 4, c = tid & 15, cs = c & (FW_CSC - 1);
  static_assert(FW_THREADS == 16 * FEW_TOKENS && FW_CXC == 32 && FW_CSC == 4, "staging split");
  struct Col {
    u4_t x[2], s;
  };
  const int slot = slots[min(t, n - 1)];
  const char *xs = reinterpret_cast<const char *>(act) + (uint32_t)(slot * (F * 2) + 16 * c);
  const char *ss =
      reinterpret_cast<const char *>(act_sum) + (uint32_t)(slot * (F / 32 * 8) + 16 * cs);
  auto request = [&](int kb) {
    Col o;
    o.x[0] = *reinterpret_cast<const u4_t *>(xs + kb * (16 * FW_CXC));
    o.x[1] = *reinterpret_cast<const u4_t *>(xs + kb * (16 * FW_CXC) + 256);
    if (!Q8) o.s = *reinterpret_cast<const u4_t *>(ss + kb * (16 * FW_CSC));
    return o;
  };
  auto stage = [&](int kb, const Col &o) {
    u4_t *b = lds + (kb & 1) * FW_COL;
    b[t * FW_CXROW + c] = o.x[0];
    b[t * FW_CXROW + c + 16] = o.x[1];
    if (!Q8) b[FEW_TOKENS * FW_CXROW + t * FW_CSROW + cs] = o.s;  // four lanes, the same value
  };
  const Col c0 = request(0), c1 = request(1);
  Col next = request(2);
  auto stage_first = [&] {
    __builtin_amdgcn_sched_barrier(0);
    stage(0, c0);
    stage(1, c1);
    __syncthreads();
  };
  f4_t acc = {0.f, 0.f, 0.f, 0.f};
  // After column kb: once every wave has read its buffer, kb + 2 goes there (read after
  // the barrier of kb + 1). The last two columns stage one more, which nothing reads.
  if constexpr (Q8) {
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
        const u4_t *xc = lds + (kb & 1) * FW_COL + lr * FW_CXROW;
#pragma unroll
        for (int j = 0; j < 2; j++) acc = w[i][j].column(xc + 16 * j, g, acc);
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
      const u4_t *b = lds + (kb & 1) * FW_COL;
      acc = w.column(kb, b + lr * FW_CXROW, b[FEW_TOKENS * FW_CXROW + lr * FW_CSROW + g], g, acc);
      if (kb + 1 < FW_NKB) __syncthreads();
      if (kb + 2 < FW_NKB) stage(kb, next);
      if (kb + 3 < FW_NKB) next = request(kb + 3);
    }
  }
  return acc;
}

// A tile of at most FEW_ROWS tokens: its rows in LDS whole, one barrier.
template <bool Q8>
__device__ __forceinline__ f4_t few_tile_rows(const uint8_t *wrow, const __half *act,
                                              const __half *act_sum, const int32_t *slots, int n,
                                              u4_t *lds) {
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
  f4_t acc = {0.f, 0.f, 0.f, 0.f};
  if constexpr (Q8) {  // 128 of K per 144-byte column
    stage();
#pragma unroll 4
    for (int kb = 0; kb < F / Q8K; kb++) {
      FewQ8 w8;
      w8.request(wrow + (size_t)kb * QB, g);
      acc = w8.column(xr + 16 * kb, g, acc);
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
      acc = w.column(kb, xr + FW_CXC * kb, sr[FW_CSC * kb + g], g, acc);
  }
  return acc;
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
  const int tid = threadIdx.x, lr = tid & 15, g = (tid >> 4) & 3;
  const bool q8 = wsh != nullptr && e == E;
  const int row = w % NRT * TROWS + 16 * (tid >> 6) + lr;
  const uint8_t *wrow = q8 ? wsh + 2 * Q8_MAT_BYTES + (size_t)row * (F / Q8K) * QB
                           : wq + (size_t)e * EXPERT_BYTES + 2 * MAT_BYTES +
                                 (size_t)row * FW_NKB * QB;
  const int32_t *slots = list + td.y;
  f4_t acc;
  if (n <= FEW_ROWS)
    acc = q8 ? few_tile_rows<true>(wrow, act, act_sum, slots, n, lds)
             : few_tile_rows<false>(wrow, act, act_sum, slots, n, lds);
  else
    acc = q8 ? few_tile_columns<true>(wrow, act, act_sum, slots, n, lds)
             : few_tile_columns<false>(wrow, act, act_sum, slots, n, lds);
  // lane holds D[token 4g + i][its row]
#pragma unroll
  for (int i = 0; i < 4; i++)
    if (4 * g + i < n) out[(size_t)slots[4 * g + i] * D + row] = acc[i];
}

}  // namespace hy3x
