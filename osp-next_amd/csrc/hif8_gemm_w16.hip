// Decode-free twin of the fused HiF8 GEMM for MI355X (gfx950):
//   Y[M,N] = X_q[M,K] . W_q[N,K]^T + bias[N]
// with W_q already dequantised to bf16 (hif8_decode of the packed codes, once per call).  The
// fused kernel (hif8_gemm_dtl.hip) decodes every weight element once per 256-row tile of X:
// at M = 75600 that is 296 decodes per element, about a tenth of its cycles and of its energy
// at the board's power limit.  Decoding W once into a workspace and streaming bf16 W costs one
// pass over the codes and twice the weight bytes through L2; for a few thousand rows and more
// it is the faster route.  The products are the same v_mfma_f32_16x16x32_bf16 on the same
// operand values, in the same k order, so the two kernels agree bit for bit.
//
// Design (shared with k_linear_dtl except for W, the wave quadrants and the LDS ring):
//   - One workgroup per 256 x 256 output tile, 4 waves; wave w owns the 128 x 128 quadrant of
//     rows 128 (w & 1) .. +127 and output features 128 (w >> 1) .. +127: 8 x 8 tiles of
//     v_mfma_f32_16x16x32_bf16.  At the board's power limit the 16x16x32 form sustains about
//     13 % more bf16 throughput than 32x32x16 on the same operand data (it moves fewer
//     accumulator bytes per flop).  (k_linear_dtl gives each wave 64 features for all 256
//     rows because a wave decodes the W rows it uses.)
//   - X and W (bf16) go global -> LDS with buffer_load ... lds.  LDS is a ring of five 32 KB
//     operand stages (one operand, 256 rows x 64 k each; 160 KB): k-step j's X and W take
//     stages 2j and 2j + 1.  Each k-step has one barrier (in its second phase); the X loads of
//     k-step j + 2 are issued in the first phase of k-step j and the W loads right after the
//     barrier, so they have three and two phases to land.  With two 64 KB stages (128 KB) the
//     last loads of a k-step had less than one phase, and the loop waited for the misses of
//     every panel that L2 does not hold.
//   - The main loop is the fixed schedule in hif8_gemm_schedule_w16.inc (gen_gemm_schedule.py).
//   - Epilogue: bias, RNE to bf16, staged through LDS into whole 512-byte row stores, non-temporal
//     (the output is not read again here; it should not displace operand panels from L2); the
//     GELU-statistic variant and grouped outputs as in k_linear_dtl.
//   - Tile order: groups of group_m m-tiles, n-tiles outer within a group.  Workgroups go to the
//     8 XCDs round robin, so each XCD runs (group_m / 8) m-tiles x (256 / group_m) n-tiles of
//     every 256 consecutive tiles and its L2 fetches that many X and W panels.  Measured on the
//     14B shapes (ms, groups of 16 / 32 / 64 m-tiles): FFN up 7.37 / 7.22 / 7.17, FFN down
//     (N = 5120) 7.22 / 7.19 / 7.30, o 2.74 / 2.74 / 2.71; 128 was 10 % slower on FFN up.
//   - Token-major operands (TR, the weight gradient grad_q^T x_q on the tensors as they lie):
//     the same loop with k-major LDS stages and fragments built by transposing reads
//     (ds_read_b64_tr_b16), the same products in the same order.
//   - Split tail: for a grid of a few waves whose last one would leave most CUs idle, the tail
//     tiles are computed over k ranges into fp32 partials (EPI 2) that k_split_reduce adds in a
//     fixed order.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hif8_gemm_w16_dev.h"

namespace hif8 {
namespace w16 {

// The split tiles' outputs: workgroup b sums the splits fp32 partials of tile full_tiles + b / 8,
// MFMA tile row i = b % 8 of each wave quadrant, in split order (a fixed order: the result does
// not depend on timing), adds the bias, rounds to bf16 and stores the in-range outputs.  One lane
// per 4 consecutive outputs of a row; 8 workgroups per tile so that the reads fill the chip.
__global__ __launch_bounds__(kThreads) void k_split_reduce(const float *__restrict__ part, int splits, int full_tiles,
                                                            int tiles_m, int tiles_n, int group_m, int M, int N,
                                                            const uint16_t *__restrict__ bias, uint16_t *__restrict__ Y)
{
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t r = lane & 15u, g = lane >> 4;
    int m0, n0;
    const uint32_t tile = blockIdx.x >> 3;
    const int i = int(blockIdx.x & 7u);
    tile_origin(full_tiles + int(tile), tiles_m, tiles_n, group_m, m0, n0);
    const uint32_t wm = (wave & 1u) * 128u, wn = (wave >> 1) * 128u;
    const f32x4 *P = (const f32x4 *)part + size_t(tile) * size_t(splits) * 16384u + wave * 4096u + lane;
    {
        const int n = n0 + int(wn) + i * 16 + int(4u * g);
        if (n >= N) return;
        float b0 = 0.f, b1 = 0.f, b2 = 0.f, b3 = 0.f;
        if (bias) {
            const uint2 bb = *(const uint2 *)(bias + n);
            b0 = __builtin_bit_cast(float, bb.x << 16);
            b1 = __builtin_bit_cast(float, bb.x & 0xFFFF0000u);
            b2 = __builtin_bit_cast(float, bb.y << 16);
            b3 = __builtin_bit_cast(float, bb.y & 0xFFFF0000u);
        }
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
            uint2 v;
            v.x = f2bf_pk(a[0] + b0, a[1] + b1);
            v.y = f2bf_pk(a[2] + b2, a[3] + b3);
            *(uint2 *)(Y + size_t(m) * size_t(N) + n) = v;
        }
    }
}

}  // namespace w16

static int cu_count()
{
    static int cus[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    if (cus[dev] == 0) {
        int c = 0;
        if (hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || c <= 0) c = 256;
        cus[dev] = c;
    }
    return cus[dev];
}

// Split of the last, partial wave of tiles (one workgroup per CU): for grids of fewer than 8
// waves whose tail (tiles % CUs) fills at most half the CUs, each tail tile runs as `splits`
// workgroups over consecutive k ranges (at least 8 k-steps each), so the last wave takes about
// 1/splits of a tile's time.  Measured on MI355X: the 14B FFN-up wgrad (1080 tiles, 4.2 waves)
// 8.08-8.19 -> 7.22-7.26 ms; its dgrad (5920 tiles, 23.1 waves) 7.35 ms either way -- after
// many waves the CUs' tile boundaries have drifted apart and the tail tiles start as CUs free up.
static SplitPlan plan_split(int64_t tiles, int64_t K)
{
    const int cus = cu_count();
    const int tail = int(tiles % cus);
    const int64_t nk = (K + w16::kBK - 1) / w16::kBK;
    SplitPlan p{int(tiles), 0, 1};
    if (tiles < cus || tiles >= 8 * int64_t(cus) || tail == 0 || tail > cus / 2) return p;
    int sp = cus / tail;
    if (sp > 8) sp = 8;
    while (sp > 1 && nk < 8 * int64_t(sp)) --sp;
    if (sp < 2) return p;
    return SplitPlan{int(tiles) - tail, tail, sp};
}

// The weight gradients' grids are small -- 36 tiles over 32760 tokens for the 1.3B q/k/v/o, 400 over
// 75600 for the 14B's -- so besides plan_split's tails, every grid of under 8 waves is split where the
// estimate below says that it saves a fifth of the tail's time: a workgroup takes about 1.33 us per
// k-step and 10 us around them, the CUs run waves of one workgroup each, and a partial's write and
// read cost 0.1 us of the chip.  (Where it said an eighth, 400 tiles over 17199 tokens, the split
// measured 1 % slower.)  At least 8 k-steps per range, at most 3 waves of partials (192 MB on 256
// CUs).  Whole -> split, MI355X: 1.3B q/k/v/o weight gradient over 32760 tokens 512 -> 149 us, 14B
// q/k/v/o over 75600 tokens 3.10 -> 2.86 ms, 1024 x 1024 over 4096 tokens 71 -> 50 us.
SplitPlan plan_ksplit(int64_t tiles, int64_t K)
{
    SplitPlan best = plan_split(tiles, K);
    const int64_t cus = cu_count(), nk = (K + w16::kBK - 1) / w16::kBK;
    const int64_t tail = tiles % cus;
    if (best.splits > 1 || tiles >= 8 * cus || tail == 0) return best;
    auto wave_us = [](int64_t ksteps) { return 10.0 + 1.33 * double(ksteps); };
    double least = 0.8 * wave_us(nk);   // of the tail as one wave of whole tiles
    for (int64_t sp = 2; sp <= 32 && nk >= 8 * sp && tail * sp <= 3 * cus; ++sp) {
        const int64_t per = (nk + sp - 1) / sp;
        if ((nk + per - 1) / per != sp) continue;   // every range holds k-steps
        const double us = double((tail * sp + cus - 1) / cus) * wave_us(per) + 5.0 + double(tail * sp) * 0.1;
        if (us < least) {
            least = us;
            best = SplitPlan{int(tiles - tail), int(tail), int(sp)};
        }
    }
    return best;
}

int launch_w16_partials(const uint16_t *x, const uint16_t *w_q, int64_t M, int64_t N, int64_t K, const SplitPlan &sp,
                        float *part, bool tr, hif8_stream_t stream)
{
    hipStream_t s = (hipStream_t)stream;
    const int tiles_m = int((M + w16::kTile - 1) / w16::kTile);
    const int tiles_n = int((N + w16::kTile - 1) / w16::kTile);
    const int group_m = tiles_n >= 32 ? w16::kGroupWide : w16::kGroupNarrow;
    Groups g{};
    g.n = 1;
    g.tile_end[0] = tiles_n;
    g.cols[0] = int(N);
    if (tr)
        hipLaunchKernelGGL((w16::k_linear_w16<2, true>), dim3(unsigned(sp.tail * sp.splits)), dim3(w16::kThreads), 0, s,
                           x, w_q, g, (const uint16_t *)nullptr, int(M), int(N), int(K), tiles_m, tiles_n, group_m,
                           (State *)nullptr, sp.full, sp.splits, part);
    else
        hipLaunchKernelGGL(w16::k_linear_w16<2>, dim3(unsigned(sp.tail * sp.splits)), dim3(w16::kThreads), 0, s, x, w_q,
                           g, (const uint16_t *)nullptr, int(M), int(N), int(K), tiles_m, tiles_n, group_m,
                           (State *)nullptr, sp.full, sp.splits, part);
    return hipGetLastError() == hipSuccess ? HIF8_OK : HIF8_ERR_HIP;
}

// Shapes: K % 64 == 0, N % 8 == 0, 16-byte aligned X, W_q and Y, 8-byte aligned bias (checked
// by the caller).  M, N < 2^31, K < 2^22.  y_st != NULL selects the GELU-statistic epilogue and the
// settle kernel (scale for y_smax).  part != NULL (one output group, no y_st) splits the tail as
// plan says, with part holding plan->bytes() bytes.  tr: x and w_q are k-major (one output group,
// no y_st).
static int launch_w16(const uint16_t *x, const uint16_t *w_q, const Groups &g, const uint16_t *bias, int64_t M,
                      int64_t N, int64_t K, hif8_stream_t stream, State *y_st, float y_smax, float *part = nullptr,
                      bool tr = false, const SplitPlan *plan = nullptr)
{
    hipStream_t s = (hipStream_t)stream;
    if (K >= (int64_t(1) << 22)) return HIF8_ERR_SHAPE;
    const int tiles_m = int((M + w16::kTile - 1) / w16::kTile);
    const int tiles_n = int((N + w16::kTile - 1) / w16::kTile);
    const int64_t tiles = int64_t(tiles_m) * tiles_n;
    const int group_m = tiles_n >= 32 ? w16::kGroupWide : w16::kGroupNarrow;
    if (tiles >= (int64_t(1) << 31)) return HIF8_ERR_SHAPE;
    SplitPlan sp{int(tiles), 0, 1};
    if (tr && (y_st || g.n != 1)) return HIF8_ERR_ARG;
    if (part) {
        if (y_st || g.n != 1 || !plan) return HIF8_ERR_ARG;
        sp = *plan;
    }
    if (y_st)
        hipLaunchKernelGGL(w16::k_linear_w16<1>, dim3(unsigned(sp.full)), dim3(w16::kThreads), 0, s, x, w_q, g, bias,
                           int(M), int(N), int(K), tiles_m, tiles_n, group_m, y_st, 0, 1, (float *)nullptr);
    else if (sp.full > 0 && tr)
        hipLaunchKernelGGL((w16::k_linear_w16<0, true>), dim3(unsigned(sp.full)), dim3(w16::kThreads), 0, s, x, w_q, g,
                           bias, int(M), int(N), int(K), tiles_m, tiles_n, group_m, (State *)nullptr, 0, 1,
                           (float *)nullptr);
    else if (sp.full > 0)
        hipLaunchKernelGGL(w16::k_linear_w16<0>, dim3(unsigned(sp.full)), dim3(w16::kThreads), 0, s, x, w_q, g, bias,
                           int(M), int(N), int(K), tiles_m, tiles_n, group_m, (State *)nullptr, 0, 1,
                           (float *)nullptr);
    if (hipGetLastError() != hipSuccess) return HIF8_ERR_HIP;
    if (sp.splits > 1) {
        // after the whole tiles on the stream: they fill whole waves, so the split workgroups
        // start as the last of them end
        const int rc = launch_w16_partials(x, w_q, M, N, K, sp, part, tr, stream);
        if (rc != HIF8_OK) return rc;
        hipLaunchKernelGGL(w16::k_split_reduce, dim3(unsigned(sp.tail) * 8u), dim3(w16::kThreads), 0, s, part, sp.splits,
                           sp.full, tiles_m, tiles_n, group_m, int(M), int(N), bias, g.y[0]);
        if (hipGetLastError() != hipSuccess) return HIF8_ERR_HIP;
    }
    return y_st ? launch_gelu_stat_settle(y_st, y_smax, stream) : HIF8_OK;
}

int launch_linear_w16(const uint16_t *x, const uint16_t *w_q, const uint16_t *bias, uint16_t *y, int64_t M,
                      int64_t N, int64_t K, hif8_stream_t stream, State *y_st, float y_smax)
{
    Groups g{};
    g.n = 1;
    g.tile_end[0] = int((N + w16::kTile - 1) / w16::kTile);
    g.cols[0] = int(N);
    g.y[0] = y;
    return launch_w16(x, w_q, g, bias, M, N, K, stream, y_st, y_smax);
}

int launch_linear_w16_groups(const uint16_t *x, const uint16_t *w_q, const Groups &g, const uint16_t *bias,
                             int64_t M, int64_t N, int64_t K, hif8_stream_t stream)
{
    return launch_w16(x, w_q, g, bias, M, N, K, stream, nullptr, 0.0f);
}

}  // namespace hif8

using namespace hif8;

static int check_w16(const void *a, const void *w_q, const uint16_t *bias, const void *y, int64_t M, int64_t N,
                     int64_t K)
{
    if (!a || !w_q || !y) return HIF8_ERR_ARG;
    if (M <= 0 || N <= 0 || K <= 0) return HIF8_ERR_ARG;
    if (M >= (int64_t(1) << 31) || N >= (int64_t(1) << 31) || K >= (int64_t(1) << 22)) return HIF8_ERR_SHAPE;
    if (K % w16::kBK != 0 || N % 8 != 0) return HIF8_ERR_SHAPE;
    if (((uintptr_t)a | (uintptr_t)w_q | (uintptr_t)y) & 15u) return HIF8_ERR_ALIGN;
    if (bias && ((uintptr_t)bias & 7u)) return HIF8_ERR_ALIGN;
    const int64_t tiles = ((M + w16::kTile - 1) / w16::kTile) * ((N + w16::kTile - 1) / w16::kTile);
    if (tiles >= (int64_t(1) << 31)) return HIF8_ERR_SHAPE;
    return HIF8_OK;
}

extern "C" int hif8_linear_fwd_wq(const uint16_t *a, const uint16_t *w_q, const uint16_t *bias, uint16_t *y,
                                  int64_t M, int64_t N, int64_t K, hif8_stream_t stream)
{
    const int rc = check_w16(a, w_q, bias, y, M, N, K);
    return rc != HIF8_OK ? rc : launch_linear_w16(a, w_q, bias, y, M, N, K, stream, nullptr, 0.0f);
}

extern "C" int64_t hif8_linear_split_workspace_bytes(int64_t M, int64_t N, int64_t K)
{
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const int64_t tiles = ((M + w16::kTile - 1) / w16::kTile) * ((N + w16::kTile - 1) / w16::kTile);
    return plan_split(tiles, K).bytes();
}

extern "C" int64_t hif8_linear_ksplit_workspace_bytes(int64_t M, int64_t N, int64_t K)
{
    if (M <= 0 || N <= 0 || K <= 0) return 0;
    const int64_t tiles = ((M + w16::kTile - 1) / w16::kTile) * ((N + w16::kTile - 1) / w16::kTile);
    return plan_ksplit(tiles, K).bytes();
}

// The split plan of a call with a workspace: plan_ksplit's where wide, else plan_split's (the entry point
// says which, never the workspace's size: the sums' order depends on it); part NULL where nothing is split.
static int split_part(void *workspace, int64_t workspace_bytes, int64_t M, int64_t N, int64_t K, bool wide,
                      float **part, SplitPlan *plan)
{
    *part = nullptr;
    if (!workspace) return HIF8_OK;
    const int64_t tiles = ((M + w16::kTile - 1) / w16::kTile) * ((N + w16::kTile - 1) / w16::kTile);
    *plan = wide ? plan_ksplit(tiles, K) : plan_split(tiles, K);
    if (plan->splits < 2) return HIF8_OK;
    if (workspace_bytes < plan->bytes()) return HIF8_ERR_ARG;
    if ((uintptr_t)workspace & 15u) return HIF8_ERR_ALIGN;
    *part = (float *)workspace;
    return HIF8_OK;
}

static int fwd_wq_split(const uint16_t *a, const uint16_t *w_q, const uint16_t *bias, uint16_t *y, int64_t M, int64_t N,
                        int64_t K, void *workspace, int64_t workspace_bytes, bool wide, hif8_stream_t stream)
{
    int rc = check_w16(a, w_q, bias, y, M, N, K);
    if (rc != HIF8_OK) return rc;
    float *part = nullptr;
    SplitPlan plan{};
    rc = split_part(workspace, workspace_bytes, M, N, K, wide, &part, &plan);
    if (rc != HIF8_OK) return rc;
    Groups g{};
    g.n = 1;
    g.tile_end[0] = int((N + w16::kTile - 1) / w16::kTile);
    g.cols[0] = int(N);
    g.y[0] = y;
    return launch_w16(a, w_q, g, bias, M, N, K, stream, nullptr, 0.0f, part, false, &plan);
}

extern "C" int hif8_linear_fwd_wq_split(const uint16_t *a, const uint16_t *w_q, const uint16_t *bias, uint16_t *y,
                                        int64_t M, int64_t N, int64_t K, void *workspace, int64_t workspace_bytes,
                                        hif8_stream_t stream)
{
    return fwd_wq_split(a, w_q, bias, y, M, N, K, workspace, workspace_bytes, false, stream);
}

extern "C" int hif8_linear_fwd_wq_ksplit(const uint16_t *a, const uint16_t *w_q, const uint16_t *bias, uint16_t *y,
                                         int64_t M, int64_t N, int64_t K, void *workspace, int64_t workspace_bytes,
                                         hif8_stream_t stream)
{
    return fwd_wq_split(a, w_q, bias, y, M, N, K, workspace, workspace_bytes, true, stream);
}

static int wgrad(const uint16_t *g, const uint16_t *x, uint16_t *dw, int64_t tokens, int64_t n_out, int64_t k_in,
                 void *workspace, int64_t workspace_bytes, bool wide, hif8_stream_t stream)
{
    if (!g || !x || !dw) return HIF8_ERR_ARG;
    if (tokens <= 0 || n_out <= 0 || k_in <= 0) return HIF8_ERR_ARG;
    if (n_out % 8 != 0 || k_in % 8 != 0) return HIF8_ERR_SHAPE;
    if (n_out >= (int64_t(1) << 31) || k_in >= (int64_t(1) << 31) || tokens >= (int64_t(1) << 31)) return HIF8_ERR_SHAPE;
    // the k-major buffers address g and x with 32-bit offsets, including the k-rows of the last
    // k-step past the tokens (which must fall past the buffers' ranges, not wrap into them)
    if ((tokens + 128) * n_out * 2 >= (int64_t(1) << 32) || (tokens + 128) * k_in * 2 >= (int64_t(1) << 32))
        return HIF8_ERR_SHAPE;
    if (((uintptr_t)g | (uintptr_t)x | (uintptr_t)dw) & 15u) return HIF8_ERR_ALIGN;
    const int64_t tiles = ((n_out + w16::kTile - 1) / w16::kTile) * ((k_in + w16::kTile - 1) / w16::kTile);
    if (tiles >= (int64_t(1) << 31)) return HIF8_ERR_SHAPE;
    float *part = nullptr;
    SplitPlan plan{};
    const int rc = split_part(workspace, workspace_bytes, n_out, k_in, tokens, wide, &part, &plan);
    if (rc != HIF8_OK) return rc;
    Groups gr{};
    gr.n = 1;
    gr.tile_end[0] = int((k_in + w16::kTile - 1) / w16::kTile);
    gr.cols[0] = int(k_in);
    gr.y[0] = dw;
    return launch_w16(g, x, gr, nullptr, n_out, k_in, tokens, stream, nullptr, 0.0f, part, true, &plan);
}

extern "C" int hif8_linear_wgrad(const uint16_t *g, const uint16_t *x, uint16_t *dw, int64_t tokens, int64_t n_out,
                                 int64_t k_in, void *workspace, int64_t workspace_bytes, hif8_stream_t stream)
{
    return wgrad(g, x, dw, tokens, n_out, k_in, workspace, workspace_bytes, false, stream);
}

extern "C" int hif8_linear_wgrad_ksplit(const uint16_t *g, const uint16_t *x, uint16_t *dw, int64_t tokens,
                                        int64_t n_out, int64_t k_in, void *workspace, int64_t workspace_bytes,
                                        hif8_stream_t stream)
{
    return wgrad(g, x, dw, tokens, n_out, k_in, workspace, workspace_bytes, true, stream);
}

extern "C" int hif8_linear_fwd_wq_gelu_stat(const uint16_t *a, const uint16_t *w_q, const uint16_t *bias,
                                            uint16_t *y, int64_t M, int64_t N, int64_t K, float scale_max,
                                            void *y_state, hif8_stream_t stream)
{
    if (!y_state) return HIF8_ERR_ARG;
    const int rc = check_w16(a, w_q, bias, y, M, N, K);
    return rc != HIF8_OK ? rc : launch_linear_w16(a, w_q, bias, y, M, N, K, stream, (State *)y_state, scale_max);
}

extern "C" int hif8_linear_fwd_wq_grouped(const uint16_t *a, const uint16_t *w_q, const uint16_t *bias,
                                          uint16_t *const *ys, const int64_t *ns, int groups, int64_t M, int64_t K,
                                          hif8_stream_t stream)
{
    if (!ys || !ns || groups < 1) return HIF8_ERR_ARG;
    if (groups > kMaxGroups) return HIF8_ERR_SHAPE;
    Groups g{};
    g.n = groups;
    int64_t N = 0;
    for (int i = 0; i < groups; ++i) {
        if (!ys[i] || ns[i] <= 0) return HIF8_ERR_ARG;
        if (ns[i] % 8 != 0 || (i + 1 < groups && ns[i] % w16::kTile != 0)) return HIF8_ERR_SHAPE;
        if ((uintptr_t)ys[i] & 15u) return HIF8_ERR_ALIGN;
        N += ns[i];
        if (N >= (int64_t(1) << 31)) return HIF8_ERR_SHAPE;
        g.tile_end[i] = int((N + w16::kTile - 1) / w16::kTile);
        g.cols[i] = int(ns[i]);
        g.y[i] = ys[i];
    }
    const int rc = check_w16(a, w_q, bias, ys[0], M, N, K);
    return rc != HIF8_OK ? rc : launch_linear_w16_groups(a, w_q, g, bias, M, N, K, stream);
}
