// Fused HiF8 dequant-GEMM on small output tiles for MI355X (gfx950), for calls of few rows or features,
// whose 256 x 256 tiles (hif8_gemm_dtl.hip) would leave most CUs idle:
//   Y[M,N] = X_q[M,K] . W_q[N,K]^T + bias[N]
// with the same operands, the same v_mfma_f32_16x16x32_bf16 products in the same k order and the same
// rounding of acc + bias, so the outputs equal that kernel's bit for bit.
//
// What bounds such a call is the time of one tile's walk along K (all tiles run at once, one workgroup
// per CU), so the tile is as small as keeps every CU at one tile (launch_linear_small has the rule), and
// a k-step's latency chain -- barrier, code read, table lookup, pack, MFMA -- is spread over more work:
//   - 32 x 32 .. 128 x 64 tiles take 2 or 4 64-k stages per barrier and issue all of their LDS reads
//     and lookups before the MFMAs (32 x 32, per 64 k: 0.36 us with one stage per barrier, 0.20 with
//     four);
//   - the 128 x 128 tile is pipelined over half-stages: while one's MFMAs run, the next one's codes are
//     looked up and its X fragments read, MFMAs, LDS reads and VALU interleaved by scheduling groups
//     (per 64 k: 0.80 us as the compiler orders it, 0.55 so).
// X and the W codes go global -> LDS with buffer_load ... lds in a ring of S steps.  The decode table
// has a dword per (code, lane), 64 KB: a lookup's lanes hit 64 banks and its address is one v_perm (with
// 2-byte entries, 32 KB, every lookup conflicts: 1.3-1.6 times the time on the tiles up to 64 x 64).
// Whole linear GEMM, 256 x 256 tiles -> this kernel: 64 x 1536 -> 1536 31.4 -> 8.3 us; 100 x 8960 -> 1536
// 141 -> 31; 512 x 1536 -> 1536 32 -> 12; 512 x 5120 -> 5120 92 -> 51 (530 TFLOP/s).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hif8_internal.h"
#include "hif8_gelu_dev.h"
#include "hif8_state_dev.h"

namespace hif8 {
namespace small {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kBK = 64;

#define ASMV asm volatile

template <int N> __device__ __forceinline__ void wait_vm() { ASMV("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }
// every LDS access of the wave done, then the workgroup barrier
__device__ __forceinline__ void barrier() { ASMV("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// 64 lanes x 16 B from the buffer (voffset per lane) into LDS at m0v + lane * 16
__device__ __forceinline__ void dtl_load(uint32_t m0v, uint32_t voff, const u32x4 &rs)
{
    ASMV("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(m0v), "v"(voff), "s"(rs) : "memory", "m0");
}
__device__ __forceinline__ f32x4 mfma(const u32x4 &a, const u32x4 &b, const f32x4 &c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
}
__device__ __forceinline__ uint32_t f2bf_pk(float lo, float hi)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

constexpr int kWaves = 4, kThreads = kWaves * 64;
constexpr uint32_t kLut = 256 * 64 * 4;   // decode table: dword (code, lane) at code * 256 + lane * 4

// Tile and wave layout: WM x WN waves of MT x NT MFMA tiles (16 rows x 16 features each), KS 64-k
// sub-steps per barrier, a ring of S steps; PIPE: the loop pipelined over half-steps.
template <int WM_, int WN_, int MT_, int NT_, int KS_, int S_, bool PIPE_> struct Cfg {
    static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_, KS = KS_, S = S_;
    static constexpr bool PIPE = PIPE_;
    static constexpr int TM = WM * MT * 16, TN = WN * NT * 16;
    static constexpr uint32_t XB = TM * 128, WB = TN * 64;          // one sub-step's X and W codes
    static constexpr uint32_t SUB = XB + WB, STEP = SUB * KS;
    // 1-KB loads of a sub-step, and per wave (where there are fewer than waves, some are repeated)
    static constexpr int XN = TM / 8, WNI = TN / 16, XI = XN > kWaves ? XN / kWaves : 1,
                         WI = WNI > kWaves ? WNI / kWaves : 1;
    static constexpr int LOADS = (XI + WI) * KS;
    static constexpr uint32_t ROW = TN * 2 + 16;                    // padded LDS row of the output tile
    static constexpr uint32_t RING = S * STEP;
    static constexpr uint32_t OUT = TM * ROW;
    static constexpr uint32_t LDS = kLut + (RING > OUT ? RING : OUT);
    static_assert(WM * WN == kWaves && S >= (PIPE ? 3 : 2) && KS >= 1 && !(PIPE && KS > 1) && LDS <= 163840, "tile");
};

// EPI 1: the GELU statistic of the outputs; 2: fp32 outputs, the sums themselves.
template <class C, int EPI>
__global__ __launch_bounds__(kThreads) void k_linear_small(const uint16_t *__restrict__ X, const uint8_t *__restrict__ Wc,
                                                           const Groups G, const uint16_t *__restrict__ bias, int M,
                                                           int N, int K, int tiles_m, int tiles_n, int group_m,
                                                           State *__restrict__ y_st)
{
    __shared__ __attribute__((aligned(1024))) uint8_t smem[C::LDS];
    const uint32_t lds0 = uint32_t(uintptr_t(smem));
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15u, g = lane >> 4;

    // consecutive tiles of the order on one XCD; the order: groups of group_m m-tiles, n-tiles outer
    int L;
    {
        const int nwg = gridDim.x, w = blockIdx.x;
        const int per = nwg >> 3, rem = nwg & 7, xcd = w & 7, slot = w >> 3;
        L = xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
    }
    const int grp = L / (group_m * tiles_n);
    const int first_m = grp * group_m;
    const int gm = (tiles_m - first_m) < group_m ? (tiles_m - first_m) : group_m;
    const int within = L - grp * group_m * tiles_n;
    const int m0 = (first_m + within % gm) * C::TM;
    const int n0 = (within / gm) * C::TN;
    int gi = 0;
    while (gi + 1 < G.n && n0 / 256 >= G.tile_end[gi]) ++gi;
    const State *__restrict__ w_st = G.st[gi];
    uint16_t *__restrict__ Y = G.y[gi];
    const int col0 = gi == 0 ? 0 : G.tile_end[gi - 1] * 256;
    const int ycols = G.cols[gi];

    u32x4 rx, rw;
    {
        const uint64_t xa = uint64_t(X) + uint64_t(m0) * uint64_t(K) * 2u;
        const uint32_t xrows = uint32_t(M - m0 < C::TM ? M - m0 : C::TM);
        rx = u32x4{uint32_t(xa), uint32_t(xa >> 32), xrows * uint32_t(K) * 2u, 0x00020000u};
        const uint64_t wa = uint64_t(Wc) + uint64_t(n0) * uint64_t(K);
        const uint32_t wrows = uint32_t(N - n0 < C::TN ? N - n0 : C::TN);
        rw = u32x4{uint32_t(wa), uint32_t(wa >> 32), wrows * uint32_t(K), 0x00020000u};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            rx[i] = __builtin_amdgcn_readfirstlane(rx[i]);
            rw[i] = __builtin_amdgcn_readfirstlane(rw[i]);
        }
    }
    const uint32_t wm = (wave % C::WM) * (C::MT * 16), wn = (wave / C::WM) * (C::NT * 16);

    // bias words of this lane's features, requested ahead of the operand loads
    uint2 bw[C::NT];
#pragma unroll
    for (int i = 0; i < C::NT; ++i) {
        const int n = n0 + int(wn + uint32_t(i * 16) + 4u * g);
        bw[i] = (bias && n < N) ? *(const uint2 *)(bias + n) : uint2{0u, 0u};
    }
    // decode table words: thread t's 16-byte pieces t, t + 256, .. hold 4 lanes' copies of one code
    constexpr int kLutIt = int(kLut / 16 / kThreads);
    uint32_t lutv[kLutIt];
#pragma unroll
    for (int it = 0; it < kLutIt; ++it) lutv[it] = w_st->lut_bf16[(uint32_t(it) * kThreads + tid) >> 4];

    // source offsets of k-step 0 (the LDS chunk swizzles are undone here, as in the 256 x 256 kernel)
    uint32_t xoff[C::XI], woff[C::WI];
#pragma unroll
    for (int i = 0; i < C::XI; ++i) {
        const uint32_t it = (wave * C::XI + uint32_t(i)) % C::XN, row = it * 8u + (lane >> 3);
        xoff[i] = row * uint32_t(K) * 2u + ((lane & 7u) ^ (lane >> 3) ^ (it & 1u)) * 16u;
    }
#pragma unroll
    for (int i = 0; i < C::WI; ++i) {
        const uint32_t it = (wave * C::WI + uint32_t(i)) % C::WNI, row = it * 16u + (lane >> 2);
        woff[i] = row * uint32_t(K) + ((lane & 3u) ^ ((lane >> 4) & 3u)) * 16u;
    }
    const int nk = K / kBK;
    // the loads of step st into ring slot `slot`; k past the end reads nothing (zeros, which add nothing)
    auto issue = [&](int st, uint32_t slot) {
#pragma unroll
        for (int ks = 0; ks < C::KS; ++ks) {
            const int k = st * C::KS + ks;
            u32x4 ex = rx, ew = rw;
            ex[2] = k < nk ? rx[2] : 0u;
            ew[2] = k < nk ? rw[2] : 0u;
            const uint32_t base = lds0 + kLut + slot * C::STEP + uint32_t(ks) * C::SUB;
#pragma unroll
            for (int i = 0; i < C::XI; ++i)
                dtl_load(__builtin_amdgcn_readfirstlane(base + ((wave * C::XI + uint32_t(i)) % C::XN) * 1024u),
                         xoff[i] + uint32_t(k) * 128u, ex);
#pragma unroll
            for (int i = 0; i < C::WI; ++i)
                dtl_load(__builtin_amdgcn_readfirstlane(base + C::XB + ((wave * C::WI + uint32_t(i)) % C::WNI) * 1024u),
                         woff[i] + uint32_t(k) * 64u, ew);
        }
    };
#pragma unroll
    for (int st = 0; st < C::S - 1; ++st) issue(st, uint32_t(st));
#pragma unroll
    for (int it = 0; it < kLutIt; ++it) {
        const uint32_t v = lutv[it];
        *(u32x4 *)(smem + (uint32_t(it) * kThreads + tid) * 16u) = u32x4{v, v, v, v};
    }

    // fragment bases inside a sub-step (see hif8_gemm_dtl.hip for the swizzles)
    const uint32_t fr = (r & 7u) ^ ((r >> 3) & 1u), gr = (r >> 2) & 3u;
    uint32_t xb[2], wb[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        xb[p] = kLut + (wm + r) * 128u + (((4u * p + g) ^ fr) << 4);
        wb[p] = kLut + C::XB + (wn + r) * 64u + (((2u * p + (g >> 1)) ^ gr) << 4) + 8u * (g & 1u);
    }
    const uint32_t lane_lut = lane * 4u;
    f32x4 acc[C::NT][C::MT];
#pragma unroll
    for (int i = 0; i < C::NT; ++i)
#pragma unroll
        for (int j = 0; j < C::MT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    struct Set {
        u32x4 A[C::NT], B[C::MT];
    } set[2];
    struct Codes {
        u32x2 w[C::NT];
    } cd[2];
    auto rd_codes = [&](Codes &c, uint32_t stage, int p) {
#pragma unroll
        for (int i = 0; i < C::NT; ++i) c.w[i] = *(const u32x2 *)(smem + stage + wb[p] + i * 1024);
    };
    auto rd_x = [&](Set &s, uint32_t stage, int p) {
#pragma unroll
        for (int j = 0; j < C::MT; ++j) s.B[j] = *(const u32x4 *)(smem + stage + xb[p] + j * 2048);
    };
    // the looked-up bf16 of the codes in cd
    uint32_t T[C::NT][8];
    auto lookup = [&](const Codes &c) {
#pragma unroll
        for (int i = 0; i < C::NT; ++i)
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t w = c.w[i][u >> 2];
                const uint32_t at = __builtin_amdgcn_perm(w, lane_lut, 0x0C0C0400u + (uint32_t(u & 3) << 8));
                T[i][u] = *(const uint16_t *)(smem + at);
            }
    };
    auto pack = [&](Set &s) {
#pragma unroll
        for (int i = 0; i < C::NT; ++i)
#pragma unroll
            for (int d = 0; d < 4; ++d) s.A[i][d] = __builtin_amdgcn_perm(T[i][2 * d + 1], T[i][2 * d], 0x05040100u);
    };
    auto mm = [&](const Set &s) {
#pragma unroll
        for (int i = 0; i < C::NT; ++i)
#pragma unroll
            for (int j = 0; j < C::MT; ++j) acc[i][j] = mfma(s.A[i], s.B[j], acc[i][j]);
    };
    if constexpr (C::PIPE) {
        // the first half-step's operands; the second half's codes stay in cd[0]
        wait_vm<(C::S - 2) * C::LOADS>();
        barrier();
        rd_codes(cd[1], 0, 0);
        rd_codes(cd[0], 0, 1);
        lookup(cd[1]);
        rd_x(set[0], 0, 0);
        pack(set[0]);
        // Phase p of k-step k multiplies what the phase before it read, looks the next phase's codes up
        // and reads its X fragments and the codes after those: k-step k + 1's stage must have landed at
        // k-step k's barrier, and nothing reads k - 1's any more.
        uint32_t slot = 0;
        for (int k = 0; k < nk; ++k) {
            wait_vm<(C::S - 3) * C::LOADS>();
            barrier();
            issue(k + C::S - 1, slot == 0 ? uint32_t(C::S - 1) : slot - 1);
            const uint32_t cur = slot * C::STEP;
            slot = slot + 1 == C::S ? 0u : slot + 1;
            const uint32_t nxt = slot * C::STEP;
            rd_codes(cd[1], nxt, 0);
            lookup(cd[0]);
            rd_x(set[1], cur, 1);
            mm(set[0]);
            pack(set[1]);
            rd_codes(cd[0], nxt, 1);
            lookup(cd[1]);
            rd_x(set[0], nxt, 0);
            mm(set[1]);
            pack(set[0]);
            // one MFMA, kD LDS reads and two VALU in turn
            constexpr int kMf = 2 * C::NT * C::MT, kDs = 2 * (C::NT * 9 + C::MT), kD = (kDs + kMf - 1) / kMf;
#pragma unroll
            for (int i = 0; i < kMf; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, kD, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
        }
    } else {
        const int steps = (nk + C::KS - 1) / C::KS;
        uint32_t slot = 0;
        for (int st = 0; st < steps; ++st) {
            wait_vm<(C::S - 2) * C::LOADS>();
            barrier();
            issue(st + C::S - 1, slot == 0 ? uint32_t(C::S - 1) : slot - 1);
            const uint32_t cur = slot * C::STEP;
            Set ss[2 * C::KS];
            Codes cc[2 * C::KS];
#pragma unroll
            for (int q = 0; q < 2 * C::KS; ++q) rd_codes(cc[q], cur + (q >> 1) * C::SUB, q & 1);
#pragma unroll
            for (int q = 0; q < 2 * C::KS; ++q) rd_x(ss[q], cur + (q >> 1) * C::SUB, q & 1);
#pragma unroll
            for (int q = 0; q < 2 * C::KS; ++q) {
                lookup(cc[q]);
                pack(ss[q]);
            }
#pragma unroll
            for (int q = 0; q < 2 * C::KS; ++q) mm(ss[q]);
            slot = slot + 1 == C::S ? 0u : slot + 1;
        }
    }
    wait_vm<0>();   // no load may still target LDS when it is reused or released
    barrier();

    // Epilogue: acc[i][j] lane (r, g), element e is output n = wn + 16 i + 4 g + e, m = wm + 16 j + r
    if constexpr (EPI == 2) {
        // through VGPRs: stored straight from the accumulators' registers, those took part of the loop's
        // fragments along and the 128 x 128 tile's loop ran 1.5 times its time
        float *Yf = (float *)Y;
#pragma unroll
        for (int i = 0; i < C::NT; ++i) {
            const int n = n0 + int(wn + uint32_t(i * 16) + 4u * g);
#pragma unroll
            for (int j = 0; j < C::MT; ++j) {
                const int m = m0 + int(wm + uint32_t(j * 16) + r);
                f32x4 v = acc[i][j];
                ASMV("" : "+v"(v));
                if (m < M && n < N) *(f32x4 *)(Yf + size_t(m) * size_t(N) + size_t(n)) = v;
            }
        }
        return;
    }
    uint8_t *so = smem + kLut;
#pragma unroll
    for (int i = 0; i < C::NT; ++i) {
        const uint32_t nl = wn + uint32_t(i * 16) + 4u * g;
        const float b0 = __builtin_bit_cast(float, bw[i].x << 16), b1 = __builtin_bit_cast(float, bw[i].x & 0xFFFF0000u);
        const float b2 = __builtin_bit_cast(float, bw[i].y << 16), b3 = __builtin_bit_cast(float, bw[i].y & 0xFFFF0000u);
#pragma unroll
        for (int j = 0; j < C::MT; ++j) {
            const f32x4 &a = acc[i][j];
            *(uint2 *)(so + (wm + uint32_t(j * 16) + r) * C::ROW + nl * 2u) =
                uint2{f2bf_pk(a[0] + b0, a[1] + b1), f2bf_pk(a[2] + b2, a[3] + b3)};
        }
    }
    barrier();
    uint32_t smax_i = 0, smax_u = 0;
    constexpr uint32_t CPR = C::TN / 8, RPW = 64 / CPR;      // 16-byte chunks per row, rows per instruction
    const uint32_t ch = lane % CPR;
    const int n = n0 + int(ch * 8u);
#pragma unroll
    for (uint32_t row = wave * RPW; row < C::TM; row += kWaves * RPW) {
        const uint32_t ml = row + lane / CPR;
        const u32x4 v = *(const u32x4 *)(so + ml * C::ROW + ch * 16u);
        const int m = m0 + int(ml);
        if (m < M && n - col0 < ycols) {
            *(u32x4 *)(Y + size_t(m) * size_t(ycols) + (n - col0)) = v;
            if (EPI == 1) {
                gelu_stat_pk(smax_i, smax_u, v[0], v[1]);
                gelu_stat_pk(smax_i, smax_u, v[2], v[3]);
            }
        }
    }
    if (EPI == 1) {
        uint32_t ystat = gelu_stat_final(smax_i, smax_u);
        for (int o = 32; o > 0; o >>= 1) ystat = max(ystat, (uint32_t)__shfl_xor((int)ystat, o, 64));
        // one atomic per workgroup: atomics on the state's word take turns, and small tiles make many
        // (1000 x 1024 -> 4096, 256 workgroups: 30 us with one per wave, 21 so)
        uint32_t *wmax = (uint32_t *)smem;   // the decode table is done with
        if (lane == 0) wmax[wave] = ystat;
        barrier();
        if (tid == 0) fold_gelu_stat(y_st, max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3])));
    }
}

template <class C>
static int launch(const uint16_t *x, const uint8_t *w, const Groups &g, const uint16_t *bias, int64_t M, int64_t N,
                  int64_t K, State *y_st, bool f32, hipStream_t s)
{
    const int tiles_m = int((M + C::TM - 1) / C::TM), tiles_n = int((N + C::TN - 1) / C::TN);
    const int group_m = tiles_m < 8 ? tiles_m : 8;
    const dim3 grid(unsigned(tiles_m) * unsigned(tiles_n));
    if (y_st)
        hipLaunchKernelGGL((k_linear_small<C, 1>), grid, dim3(kThreads), 0, s, x, w, g, bias, int(M), int(N), int(K),
                           tiles_m, tiles_n, group_m, y_st);
    else if (f32)
        hipLaunchKernelGGL((k_linear_small<C, 2>), grid, dim3(kThreads), 0, s, x, w, g, bias, int(M), int(N), int(K),
                           tiles_m, tiles_n, group_m, (State *)nullptr);
    else
        hipLaunchKernelGGL((k_linear_small<C, 0>), grid, dim3(kThreads), 0, s, x, w, g, bias, int(M), int(N), int(K),
                           tiles_m, tiles_n, group_m, (State *)nullptr);
    return hipGetLastError() == hipSuccess ? HIF8_OK : HIF8_ERR_HIP;
}

typedef Cfg<2, 2, 1, 1, 4, 2, false> T32;        // 32 x 32, 112 KB
typedef Cfg<1, 4, 4, 1, 4, 2, false> T64;        // 64 x 64, 160 KB
typedef Cfg<1, 4, 8, 1, 2, 2, false> T128x64;    // 128 x 64, 144 KB
typedef Cfg<1, 4, 8, 2, 1, 4, true> T128;        // 128 x 128, 160 KB

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

}  // namespace small

// The tile of a call: each kernel's estimated time is its waves of one workgroup per CU times the time
// of one tile, a + b us per 64 k, from GEMMs of 24, 80 and 140 64-k steps in one wave (MI355X, us):
// 32 x 32 8.3 / 19 / 31, 64 x 64 11.6 / 30 / 48, 128 x 64 15.7 / 43.5 / 72, 128 x 128 18.7 / 50 / 81,
// 256 x 256 31 / 90 / 145.  The small tiles are taken where the best of them saves a tenth: on 256 CUs up
// to 384 rows into 8960 features, 768 into 5120, 2688 into 1536 (every tile of one wave still fits).
// Over 16-8000 rows of nine weights no call was more than 2 % slower than on the 256 x 256 kernel; at
// the upper edges 2688 x 1536 -> 1536 took 21 us against 32, 384 x 1536 -> 8960 21 against 31.
int small_linear_tile(int64_t M, int64_t N, int64_t K)
{
    using namespace small;
    const int64_t cus = cu_count(), nk = (K + kBK - 1) / kBK;
    static const struct {
        int tm, tn;
        double a, b;
    } t[5] = {{256, 256, 7.0, 1.0}, {32, 32, 3.5, 0.20}, {64, 64, 4.0, 0.32}, {128, 64, 4.0, 0.49}, {128, 128, 5.5, 0.55}};
    int best = 0;
    double least = 0;
    for (int i = 0; i < 5; ++i) {
        const int64_t tiles = ((M + t[i].tm - 1) / t[i].tm) * ((N + t[i].tn - 1) / t[i].tn);
        const double us = double((tiles + cus - 1) / cus) * (t[i].a + t[i].b * double(nk)) * (i == 0 ? 0.9 : 1.0);
        if (i == 0 || us < least) {
            least = us;
            best = i;
        }
    }
    return best;
}

int launch_linear_small(int tile, const uint16_t *x, const uint8_t *w_codes, const Groups &g, const uint16_t *bias,
                        int64_t M, int64_t N, int64_t K, State *y_st, bool f32, hif8_stream_t stream)
{
    using namespace small;
    hipStream_t s = (hipStream_t)stream;
    switch (tile) {
    case 1: return launch<T32>(x, w_codes, g, bias, M, N, K, y_st, f32, s);
    case 2: return launch<T64>(x, w_codes, g, bias, M, N, K, y_st, f32, s);
    case 3: return launch<T128x64>(x, w_codes, g, bias, M, N, K, y_st, f32, s);
    default: return launch<T128>(x, w_codes, g, bias, M, N, K, y_st, f32, s);
    }
}

}  // namespace hif8
