// hy3x_mfma_few.hip -- the grouped down GEMM for few tokens per expert: a wave's
// whole weight rows in registers, no barrier in the reduction.
//
// With few tokens per expert the down GEMM is bound by how the weights stream:
// the narrow MFMA tiles (hy3x_mfma.hip) walk 128-row tiles column by column, 144
// bytes of each row at a time with one or two columns in flight, and their six
// columns hardly outlast the start of the pipeline. A down row is only 864 bytes,
// so here a wave takes 16 rows and requests all of them at once, straight into
// its registers (72 VGPRs per lane; every 128-byte line is requested once and
// used whole). A work tile has up to FEW_TOKENS tokens, a workgroup is four such
// waves, four workgroups per CU. Down launch at 3 / 8 / 16 / 32 tokens: 23.2 /
// 43.7 / 71.1 / 91.0 us with the narrow tiles, 18.4 / 37.2 / 57.7 / 81.0 here (4.8
// TB/s at 16 and 32). Measured beside it: the columns one, two or three at a time
// through a register ring 41-50 us at 8 tokens (of 39 then), two or eight waves
// per workgroup 2-8 % slower, tiles of 8 tokens 42 and 65 us at 8 and 16.
//
// The arithmetic per element is the MFMA tiles': the same operands, k order and
// sequence of operations on every accumulator (hy3x_mfma.hip's header), so a
// token's result is the same bits. Lane l holds weight row l % 16 of the wave's
// and, of each half of a block, the 16 qs bytes of piece l / 16. The tile's h rows
// and their sub-block sums are staged in LDS whole, at a row stride that spreads
// the rows over the banks; MFMA rows past the tile's tokens are zero or repeat
// others, and are never stored.
#include "hy3x_mfma_ops.h"
#include "hy3x_q8.h"

namespace hy3x {

constexpr int FW_NKB = F / QK;                 // Q4_K columns of a down row (6)
constexpr int FW_XC = F * 2 / 16;              // 16-byte chunks of an h row (192)
constexpr int FW_SC = F / 32 * 8 / 16;         // and of its sums (24)
constexpr int FW_XROW = FW_XC + 4, FW_SROW = FW_SC + 4;  // LDS row strides
constexpr int FW_THREADS = 64 * FEW_WAVES;
static_assert(FEW_TOKENS <= 16 && (FEW_TOKENS & (FEW_TOKENS - 1)) == 0, "one MFMA row group");

__global__ __launch_bounds__(FW_THREADS, 4) void k_down_few(
    const uint8_t *__restrict__ wq, const uint8_t *__restrict__ wsh,
    const __half *__restrict__ act, const __half *__restrict__ act_sum,
    const int32_t *__restrict__ list, const int4 *__restrict__ tiles,
    const int32_t *__restrict__ n_tiles, int T, float *__restrict__ out) {
  constexpr int TROWS = 16 * FEW_WAVES, NRT = D / TROWS;
  __shared__ __attribute__((aligned(16))) u4_t x_l[FEW_TOKENS * FW_XROW];
  __shared__ __attribute__((aligned(16))) u4_t s_l[FEW_TOKENS * FW_SROW];
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
  // staging: 32 threads per token. Every row is written (zeros past the tile's
  // tokens): loads used only under a condition would be moved behind it, and so
  // behind the weights.
  constexpr int TT = FW_THREADS / FEW_TOKENS, XL = FW_XC / TT;
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
  const u4_t *xr = x_l + (lr & (FEW_TOKENS - 1)) * FW_XROW;
  const u4_t *sr = s_l + (lr & (FEW_TOKENS - 1)) * FW_SROW;
  const f4_t zero4 = {0.f, 0.f, 0.f, 0.f};
  f4_t acc = zero4;
  // lane holds D[token 4g + i][its row]
  auto store = [&] {
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (4 * g + i < n) out[(size_t)slots[4 * g + i] * D + row] = acc[i];
  };
  if (q8) {  // the shared expert in Q8: 128 of K per 144-byte column
    stage();
#pragma unroll 4
    for (int kb = 0; kb < F / Q8K; kb++) {
      const uint8_t *p = wrow + (size_t)kb * QB;
      const f4_t dsc = *reinterpret_cast<const f4_t *>(p);
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const h8_t wf = q8_run(*reinterpret_cast<const u2_t *>(p + 16 + 32 * b + 8 * g));
        const f4_t pr = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            __builtin_bit_cast(h8_t, xr[16 * kb + 4 * b + g]), wf, zero4, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(dsc[b], pr[i], acc[i]);
      }
    }
    store();
    return;
  }
  // the rows were requested before the weights (loads complete in the order they
  // were issued): they are staged while the weights arrive, and column kb is
  // computed when it is there
  u4_t hdr[FW_NKB], q[FW_NKB][2];
#pragma unroll
  for (int kb = 0; kb < FW_NKB; kb++) {
    const u4_t *p = reinterpret_cast<const u4_t *>(wrow + (size_t)kb * QB);
    hdr[kb] = p[0];
    q[kb][0] = p[1 + g];
    q[kb][1] = p[5 + g];
  }
  __builtin_amdgcn_sched_barrier(0);
  stage();
  const uint32_t sel = bytes_sel(g >> 1), msel = bytes_sel(g & 1);
  const int gch = 8 * (g >> 1) + 2 * (g & 1);
#pragma unroll
  for (int kb = 0; kb < FW_NKB; kb++) {
    const Scales6 s6 = unpack_scales(hdr[kb]);
    f4_t dblk = zero4;
#pragma unroll
    for (int piece = 0; piece < 2; piece++) {
      const PairScale ps = pair_scale(s6.sc[piece], sel);
      h8_t wf[4];  // [2h + u]
      dequant_run(q[kb][piece].xy, ps, wf[0], wf[2]);
      dequant_run(q[kb][piece].zw, ps, wf[1], wf[3]);
#pragma unroll
      for (int hu = 0; hu < 4; hu++)
        dblk = __builtin_amdgcn_mfma_f32_16x16x32_f16(
            __builtin_bit_cast(h8_t, xr[32 * kb + 16 * piece + 4 * (hu >> 1) + (hu & 1) + gch]),
            wf[hu], dblk, 0, 0, 0);
    }
    const h8_t mo = mins_operand(hdr[kb].x, (g >> 1) ? s6.mn[1] : s6.mn[0], msel);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, sr[4 * kb + g]), mo, acc,
                                                 0, 0, 0);
    const float d = fp16_quirk(hdr[kb].x & 0xffffu);
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = __builtin_fmaf(d, dblk[i], acc[i]);
  }
  store();
}

}  // namespace hy3x
