// The backward's products with an operand that the reference holds in fp32 (MI355X, gfx950):
//   grad_W = grad_q^T . x_q   with x_q fp32 (an fp32 input: the self-attention's o projection),
//   grad_x = grad_q . w_q     with w_q fp32 (an fp32 weight),        hif8_linear.py:97,104.
// grad_q is bf16.  The fp32 operand is decode(code) / scale with one scale for the whole tensor, and
// decode(code), an HiF8 value of at most 4 significant bits, is exact in bf16: so the product runs on
// the decode-free MFMA kernel (hif8_gemm_w16_dev.h) with the raw HiF8 values as the operand -- every
// product exact in fp32, as the fp32 product would round it -- and the sums are divided by the scale
// once, in the epilogue.  Against the fp32 FMA kernel (hif8_gemm_f32.hip) that drops the rounding of
// each quotient and most of the rounding of the sums (relative error against float64 over 4100 tokens
// 9e-8, 1.2e-6 before).  It is bound by the MFMA rate like the kernel it instantiates: the 1.3B o
// projection's weight gradient over 32760 tokens (36 tiles in 7 k ranges) takes 0.16 ms, of which the
// partials' sum 26 us, against 8.57 ms in the fp32 FMA kernel (18 TFLOP/s).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hif8_gemm_w16_dev.h"

namespace hif8 {
namespace w16 {

// The split tiles' outputs: like k_split_reduce, with the sums divided by the state's scale and an fp32
// or bf16 output.  The reads of a workgroup's 8 x splits partials are 1 KB per wave and instruction.
__global__ __launch_bounds__(kThreads) void k_split_reduce_scaled(const float *__restrict__ part, int splits,
                                                                  int full_tiles, int tiles_m, int tiles_n, int group_m,
                                                                  int M, int N, const State *__restrict__ st, int f32,
                                                                  uint16_t *__restrict__ Y)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r = lane & 15u, g = lane >> 4;
    int m0, n0;
    const uint32_t tile = blockIdx.x >> 3;
    const int i = int(blockIdx.x & 7u);
    tile_origin(full_tiles + int(tile), tiles_m, tiles_n, group_m, m0, n0);
    const uint32_t wm = (wave & 1u) * 128u, wn = (wave >> 1) * 128u;
    const f32x4 *P = (const f32x4 *)part + size_t(tile) * size_t(splits) * 16384u + wave * 4096u + lane;
    const Divisor d(st ? st->scale : 1.0f);
    const int n = n0 + int(wn) + i * 16 + int(4u * g);
    if (n >= N) return;
    for (int j = 0; j < 8; ++j) {
        const int m = m0 + int(wm) + j * 16 + int(r);
        if (m >= M) continue;
        f32x4 a = P[(i * 8 + j) * 64];
        for (int sp = 1; sp < splits; ++sp) {
            const f32x4 q = P[size_t(sp) * 16384u + (i * 8 + j) * 64];
            a[0] = a[0] + q[0];
            a[1] = a[1] + q[1];
            a[2] = a[2] + q[2];
            a[3] = a[3] + q[3];
        }
        store_scaled(Y, f32 != 0, size_t(m) * size_t(N) + size_t(n), a, d);
    }
}

// y[M, N] = a . b^T / scale with both operands row-major over k, or (tr) k-major.  The shapes are
// those of the kernel (checked by the callers).
static int launch_scaled(const uint16_t *a, const uint16_t *b, const State *st, void *y, int out_dtype, int64_t M,
                         int64_t N, int64_t K, void *workspace, int64_t workspace_bytes, bool tr,
                         hif8_stream_t stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int tiles_m = int((M + kTile - 1) / kTile), tiles_n = int((N + kTile - 1) / kTile);
    const int64_t tiles = int64_t(tiles_m) * tiles_n;
    const int group_m = tiles_n >= 32 ? kGroupWide : kGroupNarrow;
    const int f32 = out_dtype == kF32 ? 1 : 0;
    SplitPlan sp{int(tiles), 0, 1};
    if (workspace) {
        sp = plan_ksplit(tiles, K);
        if (sp.splits > 1 && workspace_bytes < sp.bytes()) return HIF8_ERR_ARG;
        if ((uintptr_t)workspace & 15u) return HIF8_ERR_ALIGN;
    }
    Groups g{};
    g.n = 1;
    g.tile_end[0] = tiles_n;
    g.cols[0] = int(N);
    g.y[0] = (uint16_t *)y;
    if (sp.full > 0 && tr)
        hipLaunchKernelGGL((k_linear_w16<3, true>), dim3(unsigned(sp.full)), dim3(kThreads), 0, s, a, b, g,
                           (const uint16_t *)nullptr, int(M), int(N), int(K), tiles_m, tiles_n, group_m, (State *)st, 0,
                           f32, (float *)nullptr);
    else if (sp.full > 0)
        hipLaunchKernelGGL((k_linear_w16<3, false>), dim3(unsigned(sp.full)), dim3(kThreads), 0, s, a, b, g,
                           (const uint16_t *)nullptr, int(M), int(N), int(K), tiles_m, tiles_n, group_m, (State *)st, 0,
                           f32, (float *)nullptr);
    if (hipGetLastError() != hipSuccess) return HIF8_ERR_HIP;
    if (sp.splits > 1) {
        const int rc = launch_w16_partials(a, b, M, N, K, sp, (float *)workspace, tr, stream);
        if (rc != HIF8_OK) return rc;
        hipLaunchKernelGGL(k_split_reduce_scaled, dim3(unsigned(sp.tail) * 8u), dim3(kThreads), 0, s,
                           (const float *)workspace, sp.splits, sp.full, tiles_m, tiles_n, group_m, int(M), int(N), st,
                           f32, (uint16_t *)y);
        if (hipGetLastError() != hipSuccess) return HIF8_ERR_HIP;
    }
    return HIF8_OK;
}

}  // namespace w16
}  // namespace hif8

using namespace hif8;

extern "C" int hif8_linear_wgrad_scaled(const uint16_t *g, const uint16_t *x, const void *x_state, void *dw,
                                        int out_dtype, int64_t tokens, int64_t n_out, int64_t k_in, void *workspace,
                                        int64_t workspace_bytes, hif8_stream_t stream)
{
    if (!g || !x || !x_state || !dw) return HIF8_ERR_ARG;
    if (tokens <= 0 || n_out <= 0 || k_in <= 0) return HIF8_ERR_ARG;
    if (out_dtype != HIF8_DTYPE_BF16 && out_dtype != HIF8_DTYPE_F32) return HIF8_ERR_ARG;
    if (n_out % 8 != 0 || k_in % 8 != 0) return HIF8_ERR_SHAPE;
    if (n_out >= (int64_t(1) << 31) || k_in >= (int64_t(1) << 31) || tokens >= (int64_t(1) << 22)) return HIF8_ERR_SHAPE;
    // 32-bit offsets, the k-rows of the last k-step past the tokens included (as hif8_linear_wgrad)
    if ((tokens + 128) * n_out * 2 >= (int64_t(1) << 32) || (tokens + 128) * k_in * 2 >= (int64_t(1) << 32))
        return HIF8_ERR_SHAPE;
    if (((uintptr_t)g | (uintptr_t)x | (uintptr_t)dw) & 15u) return HIF8_ERR_ALIGN;
    if (((n_out + w16::kTile - 1) / w16::kTile) * ((k_in + w16::kTile - 1) / w16::kTile) >= (int64_t(1) << 31))
        return HIF8_ERR_SHAPE;
    return w16::launch_scaled(g, x, (const State *)x_state, dw, out_dtype, n_out, k_in, tokens, workspace,
                              workspace_bytes, true, stream);
}

extern "C" int hif8_linear_fwd_scaled(const uint16_t *a, const uint16_t *w, const void *w_state, void *y, int out_dtype,
                                      int64_t M, int64_t N, int64_t K, void *workspace, int64_t workspace_bytes,
                                      hif8_stream_t stream)
{
    if (!a || !w || !y) return HIF8_ERR_ARG;
    if (M <= 0 || N <= 0 || K <= 0) return HIF8_ERR_ARG;
    if (out_dtype != HIF8_DTYPE_BF16 && out_dtype != HIF8_DTYPE_F32) return HIF8_ERR_ARG;
    if (M >= (int64_t(1) << 31) || N >= (int64_t(1) << 31) || K >= (int64_t(1) << 22)) return HIF8_ERR_SHAPE;
    if (K % w16::kBK != 0 || N % 8 != 0) return HIF8_ERR_SHAPE;
    if (((uintptr_t)a | (uintptr_t)w | (uintptr_t)y) & 15u) return HIF8_ERR_ALIGN;
    if (((M + w16::kTile - 1) / w16::kTile) * ((N + w16::kTile - 1) / w16::kTile) >= (int64_t(1) << 31))
        return HIF8_ERR_SHAPE;
    return w16::launch_scaled(a, w, (const State *)w_state, y, out_dtype, M, N, K, workspace, workspace_bytes, false,
                              stream);
}
