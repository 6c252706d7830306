// Fused HiF8 dequant-GEMM for MI355X (gfx950), bf16 activations:
//   Y[M,N] = X_q[M,K] . W_q[N,K]^T + bias[N]
// the F.linear(x_q, w_q, bias) of ospnext/modules/hif8_linear.py:86 with W held as
// packed 8-bit HiF8 codes and W_q[n,k] = rnd_bf16(decode(code[n,k]) / scale_w), the
// reference's dequantised weight (ospnext/quant_cy_npu/base/QFuncs/hif8.py qdq).
//
// Design
//   - One workgroup per 256 (m) x 256 (n) output tile, 4 waves (one per SIMD); wave w owns
//     the 64 output features n0 + 64w .. +63 for all 256 rows: 4 x 16 tiles of
//     v_mfma_f32_16x16x32_bf16 (256 fp32 accumulators per lane, all in AGPRs).  At the board's
//     power limit the 16x16x32 form sustains more bf16 throughput than 32x32x16 on the same
//     data, and the decode-free twin (hif8_gemm_w16.hip) issues the same products in the same
//     order, so the two routes give equal outputs.
//   - X (bf16, 32 KB per 64-k step) and the W codes (16 KB per step) go from global memory
//     straight into LDS (buffer_load_dwordx4 ... lds): no VGPR staging, no LDS store
//     instructions.  Two stages (the decode table takes the rest of LDS); a stage's 12 loads
//     per wave are all issued in the phase that frees it, two phases before it is read (half
//     of them had one phase before: 1-1.5 % slower).  Rows past M or N read as zero through
//     the buffer range.
//   - Each wave decodes only its own W rows: a code becomes the bf16 operand through a
//     64 KB LDS table holding one copy per lane (entry (code, lane) at code*256 + lane*4),
//     so the 64 lanes of a lookup hit 64 different banks whatever the codes are.
//   - The main loop is a fixed instruction schedule (hif8_gemm_schedule.inc, generated by
//     gen_gemm_schedule.py): every LDS read, lookup, address computation and operand pack
//     is an ordered inline-asm instruction placed between MFMAs, with explicit waits.
//     Register values produced by asm loads are passed through empty asm statements after
//     the covering wait, so that the compiler cannot touch them earlier.
//   - Epilogue: bias in fp32, RNE to bf16, the 256 x 256 tile is staged through LDS and
//     written as full 512-byte rows with non-temporal stores (the output is not read again
//     here; it should not displace operand panels from L2).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hif8_internal.h"
#include "hif8_gelu_dev.h"
#include "hif8_state_dev.h"

namespace hif8 {
namespace dtl {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 256;
constexpr int kBK = 64;
constexpr int kThreads = 256;
constexpr int kGroupM = 32;  // m-tiles per group in the tile order

// LDS map (bytes).  Every LDS access in the main loop uses these absolute addresses;
// the kernel's only LDS object is the 160 KB array, which therefore starts at 0.
constexpr uint32_t kX0 = 0;        // X stage s at s * 32K: 256 rows x 128 B, 16-B chunks swizzled
constexpr uint32_t kW0 = 65536;    // W stage s at 64K + s * 16K: 256 rows x 64 B, 16-B chunks swizzled
constexpr uint32_t kLut = 98304;   // 256 codes x 64 lanes x 4 B
constexpr uint32_t kLds = 163840;
constexpr uint32_t kOutRow = 528;  // epilogue: padded LDS row of the 256-wide output tile

#define ASMV asm volatile

template <int OFF> __device__ __forceinline__ void ldsb128(u32x4 &d, uint32_t a)
{
    ASMV("ds_read_b128 %0, %1 offset:%2" : "=v"(d) : "v"(a), "i"(OFF));
}
// table lookup: the address is 64K + code*256 + lane*4, the table starts at 96K
__device__ __forceinline__ void lut16(uint32_t &d, uint32_t a)
{
    ASMV("ds_read_u16 %0, %1 offset:32768" : "=v"(d) : "v"(a));
}
template <int OFF> __device__ __forceinline__ void ldsb64(u32x2 &d, uint32_t a)
{
    ASMV("ds_read_b64 %0, %1 offset:%2" : "=v"(d) : "v"(a), "i"(OFF));
}
__device__ __forceinline__ void mfma(f32x4 &c, const u32x4 &a, const u32x4 &b)
{
    ASMV("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
template <int N> __device__ __forceinline__ void wait_lgkm() { ASMV("s_waitcnt lgkmcnt(%0)" ::"i"(N)); }
template <int N> __device__ __forceinline__ void wait_vm() { ASMV("s_waitcnt vmcnt(%0)" ::"i"(N)); }
__device__ __forceinline__ void barrier() { ASMV("s_barrier" ::: "memory"); }
// 64 lanes x 16 B from the buffer (voffset per lane) into LDS at m0v + lane*16
__device__ __forceinline__ void dtl_load(uint32_t m0v, uint32_t voff, const u32x4 &rs)
{
    ASMV("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(m0v), "v"(voff), "s"(rs) : "memory", "m0");
}
__device__ __forceinline__ void vperm(uint32_t &d, uint32_t s0, uint32_t s1, uint32_t sel)
{
    ASMV("v_perm_b32 %0, %1, %2, %3" : "=v"(d) : "v"(s0), "v"(s1), "s"(sel));
}
__device__ __forceinline__ void tie(u32x4 &a) { ASMV("" : "+v"(a)); }
__device__ __forceinline__ void tie(u32x2 &a) { ASMV("" : "+v"(a)); }
__device__ __forceinline__ void tie8(uint32_t *t)
{
    ASMV("" : "+v"(t[0]), "+v"(t[1]), "+v"(t[2]), "+v"(t[3]), "+v"(t[4]), "+v"(t[5]), "+v"(t[6]), "+v"(t[7]));
}

__device__ __forceinline__ uint32_t f2bf_pk(float lo, float hi)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Per-wave loop state.  Fragment sets alternate between phases: set 0 is consumed in
// phase 0 and filled in phase 1, set 1 the other way round.
struct Ctx {
    u32x4 B[2][16];       // [set][j]     X fragments (m-tile j)
    uint32_t T[2][4][8];  // [set][i][u]  looked-up bf16 of code u of W fragment (n-tile i)
    uint32_t A[2][4][4];  // [set][i][d]  packed W fragments
    u32x2 cd[4];          // W codes of the next phase, per n-tile (8 per lane)
    uint32_t xb[2];       // X fragment read base [k-half p]
    uint32_t wb[2];       // W code read base [p]
    uint32_t lane4;       // 64K | lane*4: byte 0 and 2 of every table address
    uint32_t sel[4];      // v_perm selectors: code byte k -> table address
    uint32_t selpk;       // v_perm selector: two bf16 -> one operand dword
    uint32_t ad[4];       // table addresses, computed one gap ahead of their reads
    f32x4 acc[4][16];
    u32x4 rx, rw, ex, ew;  // buffer resources: X, W, and the effective X / W (word 2, the size, 0 past the end)
    int nk_eff;
    uint32_t xoff[8], woff[4];  // DTL source offsets of the next k-step to load
    uint32_t wave;
};

template <int I> __device__ __forceinline__ void adv(Ctx &c)
{
    if (I < 8) ASMV("v_add_u32 %0, 0x80, %0" : "+v"(c.xoff[I]));
    else ASMV("v_add_u32 %0, 64, %0" : "+v"(c.woff[I - 8]));
}
__device__ __forceinline__ void advance_all(Ctx &c)
{
    adv<0>(c); adv<1>(c); adv<2>(c); adv<3>(c); adv<4>(c); adv<5>(c);
    adv<6>(c); adv<7>(c); adv<8>(c); adv<9>(c); adv<10>(c); adv<11>(c);
}

// A load into LDS at m0 + OFF + lane*16 from the buffer at voffset + OFF, with m0 as the previous
// dtl_load left it.  The instruction offset enters both addresses and the buffer's range check
// (a probe kernel on the GPU: lanes whose voffset + OFF passed the range read zero).
template <int OFF> __device__ __forceinline__ void dtl_load_off(uint32_t voff, const u32x4 &rs)
{
    ASMV("buffer_load_dwordx4 %0, %1, 0 offen offset:%2 lds" ::"v"(voff), "s"(rs), "i"(OFF) : "memory");
}
// DTL item I of a k-step into stage S: items 0..7 are X (8 x 1 KB per wave), 8..11 W (4 x 1 KB).
// Items go in groups of four (X 0..3, X 4..7, W 8..11) that share one m0 write: item 4q + u
// lands u KB after the group's base through the instruction offset, and its source offset holds
// u KB less (so the sum is the item's own).  Items are issued in order and the main loop writes
// m0 nowhere else, so a group's later items find its m0 (the schedule test checks the ISA).
template <int S, int I> __device__ __forceinline__ void issue_dtl(Ctx &c)
{
    constexpr int q = I % 4;
    if (I < 8) {
        if (q == 0) {
            const uint32_t m0v = __builtin_amdgcn_readfirstlane(kX0 + S * 32768u + (c.wave * 8u + I) * 1024u);
            dtl_load(m0v, c.xoff[I], c.ex);
        } else dtl_load_off<q * 1024>(c.xoff[I], c.ex);
    } else {
        if (q == 0) {
            const uint32_t m0v = __builtin_amdgcn_readfirstlane(kW0 + S * 16384u + (c.wave * 4u) * 1024u);
            dtl_load(m0v, c.woff[0], c.ew);
        } else dtl_load_off<q * 1024>(c.woff[q], c.ew);
    }
}
template <int S> __device__ __forceinline__ void issue_all(Ctx &c)
{
    issue_dtl<S, 0>(c); issue_dtl<S, 1>(c); issue_dtl<S, 2>(c); issue_dtl<S, 3>(c);
    issue_dtl<S, 4>(c); issue_dtl<S, 5>(c); issue_dtl<S, 6>(c); issue_dtl<S, 7>(c);
    issue_dtl<S, 8>(c); issue_dtl<S, 9>(c); issue_dtl<S, 10>(c); issue_dtl<S, 11>(c);
}

// the 8 codes of n-tile I (16 rows x 64 B of the stage per n-tile)
template <int NS, int NP, int I> __device__ __forceinline__ void rd_code(Ctx &c)
{
    ldsb64<NS * 16384 + I * 1024>(c.cd[I], c.wb[NP]);
}
template <int NS, int NP, int NXT, int J> __device__ __forceinline__ void rd_x(Ctx &c)
{
    ldsb128<NS * 32768 + J * 2048>(c.B[NXT][J], c.xb[NP]);
}
// address of lookup LL (0..31: n-tile i = LL/8, code u) into slot R
template <int R, int LL> __device__ __forceinline__ void lka(Ctx &c)
{
    constexpr int i = LL / 8, u = LL % 8;
    vperm(c.ad[R], c.cd[i][u / 4], c.lane4, c.sel[u % 4]);
}
template <int NXT, int R, int LL> __device__ __forceinline__ void lkr(Ctx &c)
{
    constexpr int i = LL / 8, u = LL % 8;
    lut16(c.T[NXT][i][u], c.ad[R]);
}
// operand dword D of fragment F: codes 2D (low half) and 2D+1 (high half)
template <int SET, int F, int D> __device__ __forceinline__ void pk(Ctx &c)
{
    vperm(c.A[SET][F][D], c.T[SET][F][2 * D + 1], c.T[SET][F][2 * D], c.selpk);
}
// MFMA MI of a phase: 2 x 2 blocks of (n-tile i, m-tile j), (0,0) (1,0) (1,1) (0,1) (0,2) ..
// along j for n-tiles 0 and 1, then back along j for n-tiles 2 and 3, so that each operand feeds
// two MFMAs in a row (at the board's power limit 1.9-2.9 % faster than n-tile-major order on the
// 14B shapes, A/B of builds on one box).  Every accumulator receives its products in k order, as
// in the decode-free kernel, so the two routes still agree bit for bit.
template <int CUR, int MI> __device__ __forceinline__ void mm(Ctx &c)
{
    constexpr int h = MI / 32, q = (MI % 32) / 4, r = MI % 4, bj = h ? 7 - q : q;
    constexpr int i = 2 * h + ((r == 1 || r == 2) ? 1 : 0), j = 2 * bj + (h ? (r >= 2 ? 0 : 1) : (r >= 2 ? 1 : 0));
    const uint32_t *a = c.A[CUR][i];
    mfma(c.acc[i][j], u32x4{a[0], a[1], a[2], a[3]}, c.B[CUR][j]);
}
// after the wait covering the previous phase: the X fragments and the lookups of set SET
template <int SET> __device__ __forceinline__ void tie_set(Ctx &c)
{
#pragma unroll
    for (int j = 0; j < 16; ++j) tie(c.B[SET][j]);
    tie8(c.T[SET][2]);
    tie8(c.T[SET][3]);
}
// after the wait covering this phase's code reads
__device__ __forceinline__ void tie_cd(Ctx &c)
{
    tie(c.cd[0]);
    tie(c.cd[1]);
    tie(c.cd[2]);
    tie(c.cd[3]);
}

#include "hif8_gemm_schedule.inc"

// EPI 0: y = rnd(acc + bias).  EPI 1 (the up-projection of nn.Sequential(linear, GELU, linear)):
// the same y, and the GELU statistic of y (its max, or a non-finite flag) folded into y_st's
// accumulator; the settle kernel launched after it writes amax|GELU(y)| and its scale when max y
// settles them, so that the down-projection's quantisation, which applies GELU, needs no amax
// pass of its own (hif8_gelu_dev.h).
// EPI 0 with f32: y = acc in fp32, no bias (the gradient of an fp32 input, which would otherwise be
// rounded to bf16 and widened by a pass of its own), one output group.
// The output features are G.n groups (G.n = 1 for one linear): the tile's group supplies its
// decode table and its output buffer.
template <int EPI>
__global__ __launch_bounds__(kThreads, 1) void k_linear_dtl(const uint16_t *__restrict__ X, const uint8_t *__restrict__ Wc,
                                                            const Groups G, const uint16_t *__restrict__ bias,
                                                            int M, int N, int K, int tiles_m, int tiles_n,
                                                            State *__restrict__ y_st, int f32)
{
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kLds];
    ASMV("; lds base %0" ::"v"(uint32_t(uintptr_t(smem))) : "memory");
    Ctx c;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15u, g = lane >> 4;

    // tile order: groups of kGroupM m-tiles, n-tiles outer within a group.  Workgroups are
    // dealt round-robin to the 8 XCDs, so the 32 running on one XCD cover 4 m-tiles x 8
    // n-tiles (12 panels through its L2; groups of 16 made it 2 x 16 = 18 panels, 1.5 % slower
    // on the 14B FFN-up shape, and groups of 64 0.5 % slower).
    const int t = blockIdx.x;
    const int group = t / (kGroupM * tiles_n);
    const int first_m = group * kGroupM;
    const int gm = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
    const int within = t - group * kGroupM * tiles_n;
    const int m0 = (first_m + within % gm) * kTile;
    const int n0 = (within / gm) * kTile;
    int gi = 0;
    while (gi + 1 < G.n && n0 / kTile >= G.tile_end[gi]) ++gi;
    const State *__restrict__ w_st = G.st[gi];
    uint16_t *__restrict__ Y = G.y[gi];
    const int col0 = gi == 0 ? 0 : G.tile_end[gi - 1] * kTile;   // first feature of the group
    const int ycols = G.cols[gi];

    {
        const uint64_t xa = uint64_t(X) + uint64_t(m0) * uint64_t(K) * 2u;
        const uint32_t xrows = uint32_t(M - m0 < kTile ? M - m0 : kTile);
        c.rx = u32x4{uint32_t(xa), uint32_t(xa >> 32), xrows * uint32_t(K) * 2u, 0x00020000u};
        const uint64_t wa = uint64_t(Wc) + uint64_t(n0) * uint64_t(K);
        const uint32_t wrows = uint32_t(N - n0 < kTile ? N - n0 : kTile);
        c.rw = u32x4{uint32_t(wa), uint32_t(wa >> 32), wrows * uint32_t(K), 0x00020000u};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            c.rx[i] = __builtin_amdgcn_readfirstlane(c.rx[i]);
            c.rw[i] = __builtin_amdgcn_readfirstlane(c.rw[i]);
        }
    }
    // DTL source offsets of k-step 0.  LDS 16-B slot s of a stage is written by lane s%64 of
    // load s/64; its source chunk is the slot's chunk un-swizzled (the XOR is an involution).
    // Each offset holds (item % 4) KB less: the load's instruction offset adds it back.  Item i
    // starts at row 8i (X, 2K bytes a row) or 16i (W, K bytes), so for K >= 64 no offset is
    // negative.
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t row = (c.wave * 8u + i) * 8u + (lane >> 3);
        const uint32_t ch = (lane & 7u) ^ (lane >> 3) ^ uint32_t(i & 1);
        c.xoff[i] = row * uint32_t(K) * 2u + ch * 16u - uint32_t(i % 4) * 1024u;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t row = (c.wave * 4u + i) * 16u + (lane >> 2);
        const uint32_t ch = (lane & 3u) ^ ((lane >> 4) & 3u);
        c.woff[i] = row * uint32_t(K) + ch * 16u - uint32_t(i) * 1024u;
    }
    // Fragment read bases.  Lane (r, g) = (lane & 15, lane >> 4) holds k = 32p + 8g .. +7 of
    // phase p for row r of its 16-row tile, for both operands (the order hif8_gemm_w16.hip
    // uses).  X row m, 16-B chunk k/8 sits at m*128 + ((chunk ^ f(m)) << 4), f(m) = (m & 7) ^
    // ((m >> 3) & 1): any 16 consecutive rows of one chunk hit distinct banks.  W code row n
    // (64 B per k-step), 16-B chunk k/16 sits at n*64 + ((chunk ^ s(n)) << 4), s(n) =
    // (n >> 2) & 3; a lane reads its 8 codes (k = 32p + 8g ..) as one 8-byte load, and the 32
    // lanes of g = 0, 1 (or 2, 3) cover the 32 8-byte bank slots of 256 bytes.
    const uint32_t fr = (r & 7u) ^ ((r >> 3) & 1u);
#pragma unroll
    for (int p = 0; p < 2; ++p) c.xb[p] = kX0 + r * 128u + (((4u * p + g) ^ fr) << 4);
    const uint32_t gr = (r >> 2) & 3u;
#pragma unroll
    for (int p = 0; p < 2; ++p)
        c.wb[p] = kW0 + (c.wave * 64u + r) * 64u + (((2u * p + (g >> 1)) ^ gr) << 4) + 8u * (g & 1u);
    c.lane4 = 0x00010000u | (lane * 4u);
#pragma unroll
    for (int k = 0; k < 4; ++k) c.sel[k] = __builtin_amdgcn_readfirstlane(0x03020400u | (uint32_t(4 + k) << 8));
    c.selpk = __builtin_amdgcn_readfirstlane(0x05040100u);
#pragma unroll
    for (int k = 0; k < 4; ++k) c.ad[k] = c.lane4;

    const int nk = K / kBK;
    const int odd = nk & 1;  // an odd k-step count gets a zero k-step in front
    c.nk_eff = nk + odd;
    c.ex = c.rx;
    c.ew = c.rw;
    {
        // decode table: dword (code*64 + lane) = W_q(code)
        uint8_t *lt = smem + kLut;
#pragma unroll
        for (int it = 0; it < 16; ++it) {
            const uint32_t q = uint32_t(it) * 256u + tid;
            const uint32_t v = w_st->lut_bf16[q >> 4];
            *(u32x4 *)(lt + q * 16u) = u32x4{v, v, v, v};
        }
        if (odd) {
#pragma unroll
            for (int it = 0; it < 8; ++it) *(u32x4 *)(smem + kX0 + (uint32_t(it) * 256u + tid) * 16u) = u32x4{0, 0, 0, 0};
#pragma unroll
            for (int it = 0; it < 4; ++it) *(u32x4 *)(smem + kW0 + (uint32_t(it) * 256u + tid) * 16u) = u32x4{0, 0, 0, 0};
        }
    }
    // The bias words of this lane's output features (4 per MFMA tile row i), loaded ahead of the
    // operand loads: they land during the main loop (in-order completion puts them before every
    // operand wait), where in the epilogue each was a global load waited for on its own.
    uint2 bw[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n0 + int(c.wave * 64u + uint32_t(i * 16) + 4u * g);
        bw[i] = (bias && n < N) ? *(const uint2 *)(bias + n) : uint2{0u, 0u};
    }
    wait_lgkm<0>();
    if (!odd) {
        issue_all<0>(c);
        advance_all(c);
    }
    c.ex[2] = c.nk_eff > 1 ? c.rx[2] : 0u;
    c.ew[2] = c.nk_eff > 1 ? c.rw[2] : 0u;
    // k-step 1 into stage 1; the first phase 0 advances the offsets to k-step 2
    static_assert(kLoadsPhase1 == 12, "every load of a k-step is issued by phase 1");
    issue_all<1>(c);
    wait_vm<12>();
    barrier();
    // reads for phase (0, 0) from stage 0 into set 0: codes, X fragments, all 32 lookups, and
    // n-tiles 0 and 1's operands (phase 0 packs n-tiles 2 and 3 itself)
    rd_code<0, 0, 0>(c); rd_code<0, 0, 1>(c); rd_code<0, 0, 2>(c); rd_code<0, 0, 3>(c);
    wait_lgkm<0>();
    tie_cd(c);
    rd_x<0, 0, 0, 0>(c); rd_x<0, 0, 0, 1>(c); rd_x<0, 0, 0, 2>(c); rd_x<0, 0, 0, 3>(c);
    rd_x<0, 0, 0, 4>(c); rd_x<0, 0, 0, 5>(c); rd_x<0, 0, 0, 6>(c); rd_x<0, 0, 0, 7>(c);
    rd_x<0, 0, 0, 8>(c); rd_x<0, 0, 0, 9>(c); rd_x<0, 0, 0, 10>(c); rd_x<0, 0, 0, 11>(c);
    rd_x<0, 0, 0, 12>(c); rd_x<0, 0, 0, 13>(c); rd_x<0, 0, 0, 14>(c); rd_x<0, 0, 0, 15>(c);
#define HIF8_LK(LL) lka<0, LL>(c); lkr<0, 0, LL>(c);
    HIF8_LK(0) HIF8_LK(1) HIF8_LK(2) HIF8_LK(3) HIF8_LK(4) HIF8_LK(5) HIF8_LK(6) HIF8_LK(7)
    HIF8_LK(8) HIF8_LK(9) HIF8_LK(10) HIF8_LK(11) HIF8_LK(12) HIF8_LK(13) HIF8_LK(14) HIF8_LK(15)
    HIF8_LK(16) HIF8_LK(17) HIF8_LK(18) HIF8_LK(19) HIF8_LK(20) HIF8_LK(21) HIF8_LK(22) HIF8_LK(23)
    HIF8_LK(24) HIF8_LK(25) HIF8_LK(26) HIF8_LK(27) HIF8_LK(28) HIF8_LK(29) HIF8_LK(30) HIF8_LK(31)
#undef HIF8_LK
    wait_lgkm<0>();
    tie8(c.T[0][0]);
    pk<0, 0, 0>(c); pk<0, 0, 1>(c); pk<0, 0, 2>(c); pk<0, 0, 3>(c);
    tie8(c.T[0][1]);
    pk<0, 1, 0>(c); pk<0, 1, 1>(c); pk<0, 1, 2>(c); pk<0, 1, 3>(c);

#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) c.acc[i][j] = f32x4{};
    // Two k-steps per iteration (stage 0 then stage 1).  The loads of k-step kt+2 use the
    // resources with size 0 past the end: they read nothing and nothing consumes them.
    for (int kt = 0; kt < c.nk_eff; kt += 2) {
        phase0<0>(c);
        c.ex[2] = kt + 2 < c.nk_eff ? c.rx[2] : 0u;
        c.ew[2] = kt + 2 < c.nk_eff ? c.rw[2] : 0u;
        phase1<0>(c);
        phase0<1>(c);
        c.ex[2] = kt + 3 < c.nk_eff ? c.rx[2] : 0u;
        c.ew[2] = kt + 3 < c.nk_eff ? c.rw[2] : 0u;
        phase1<1>(c);
    }
    // no load may still target LDS when it is reused or released
    wait_vm<0>();
    wait_lgkm<0>();
    // the last MFMAs' results must be complete before the accumulators are read
    ASMV("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 16; ++j) ASMV("" : "+a"(c.acc[i][j]));

    if (EPI == 0 && f32) {
        // straight from the accumulators: 4 consecutive features, 16 bytes, per lane.  (Either way out ties
        // each accumulator to its AGPRs where it uses it: without that all of them were copied to VGPRs
        // ahead of the branch and spilled.)
        float *Yf = (float *)Y;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + int(c.wave * 64u + uint32_t(i * 16) + 4u * g);
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const int m = m0 + j * 16 + int(r);
                ASMV("" : "+a"(c.acc[i][j]));
                if (m < M && n < N) *(f32x4 *)(Yf + size_t(m) * size_t(N) + size_t(n)) = c.acc[i][j];
            }
        }
        return;
    }
    // Epilogue.  acc[i][j] lane (r, g), element e: D[n][m] with n = 64w + 16i + 4g + e,
    // m = 16j + r.  Rows go to LDS (padded), then each wave stores 2 rows x 512 B per instruction.
    __syncthreads();
    {
        const uint32_t wl = c.wave * 64u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            {
                const uint32_t nl = wl + uint32_t(i * 16) + 4u * g;
                const uint2 bb = bw[i];
                const float b0 = __builtin_bit_cast(float, bb.x << 16);
                const float b1 = __builtin_bit_cast(float, bb.x & 0xFFFF0000u);
                const float b2 = __builtin_bit_cast(float, bb.y << 16);
                const float b3 = __builtin_bit_cast(float, bb.y & 0xFFFF0000u);
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    ASMV("" : "+a"(c.acc[i][j]));
                    const f32x4 &a = c.acc[i][j];
                    uint2 v;
                    v.x = f2bf_pk(a[0] + b0, a[1] + b1);
                    v.y = f2bf_pk(a[2] + b2, a[3] + b3);
                    *(uint2 *)(smem + (uint32_t(j * 16) + r) * kOutRow + nl * 2u) = v;
                }
            }
        }
    }
    __syncthreads();
    // EPI 1: packed running maxima of the in-range outputs this lane stores (the GELU statistic)
    uint32_t smax_i = 0, smax_u = 0;
    {
        const uint32_t colb = (lane & 31u) * 16u, h = lane >> 5;
        const int n = n0 + int(colb / 2u);
#pragma unroll
        for (int blk = 0; blk < 4; ++blk) {
            u32x4 v[8];
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const uint32_t row = c.wave * 64u + uint32_t(blk * 8 + it) * 2u + h;
                v[it] = *(const u32x4 *)(smem + row * kOutRow + colb);
            }
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int m = m0 + int(c.wave * 64u + uint32_t(blk * 8 + it) * 2u + h);
                if (m < M && n - col0 < ycols) {
                    __builtin_nontemporal_store(v[it], (u32x4 *)(Y + size_t(m) * size_t(ycols) + (n - col0)));
                    if (EPI == 1) {
                        gelu_stat_pk(smax_i, smax_u, v[it][0], v[it][1]);
                        gelu_stat_pk(smax_i, smax_u, v[it][2], v[it][3]);
                    }
                }
            }
        }
    }
    if (EPI == 1) {
        uint32_t ystat = gelu_stat_final(smax_i, smax_u);
        for (int o = 32; o > 0; o >>= 1) ystat = max(ystat, (uint32_t)__shfl_xor((int)ystat, o, 64));
        if (lane == 0) fold_gelu_stat(y_st, ystat);
    }
}

}  // namespace dtl

// Shapes: K % 64 == 0, N % 8 == 0, 16-byte aligned X, W codes and Y, 8-byte aligned bias
// (checked by the caller).  M, N < 2^31, K < 2^22.  y_st != NULL selects the GELU-statistic
// epilogue and the settle kernel (scale for y_smax).  f32: fp32 outputs (one group, no bias, no y_st).
static int launch(const uint16_t *x, const uint8_t *w_codes, const Groups &g, const uint16_t *bias, int64_t M,
                  int64_t N, int64_t K, hif8_stream_t stream, State *y_st, float y_smax, bool f32 = false)
{
    hipStream_t s = (hipStream_t)stream;
    if (K >= (int64_t(1) << 22)) return HIF8_ERR_SHAPE;
    const int tiles_m = int((M + dtl::kTile - 1) / dtl::kTile);
    const int tiles_n = int((N + dtl::kTile - 1) / dtl::kTile);
    const int64_t tiles = int64_t(tiles_m) * tiles_n;
    if (tiles >= (int64_t(1) << 31)) return HIF8_ERR_SHAPE;
    if (const int tile = small_linear_tile(M, N, K)) {
        const int rc = launch_linear_small(tile, x, w_codes, g, bias, M, N, K, y_st, f32, stream);
        if (rc != HIF8_OK) return rc;
        return y_st ? launch_gelu_stat_settle(y_st, y_smax, stream) : HIF8_OK;
    }
    if (y_st)
        hipLaunchKernelGGL(dtl::k_linear_dtl<1>, dim3(unsigned(tiles)), dim3(dtl::kThreads), 0, s, x, w_codes, g, bias,
                           int(M), int(N), int(K), tiles_m, tiles_n, y_st, 0);
    else
        hipLaunchKernelGGL(dtl::k_linear_dtl<0>, dim3(unsigned(tiles)), dim3(dtl::kThreads), 0, s, x, w_codes, g, bias,
                           int(M), int(N), int(K), tiles_m, tiles_n, (State *)nullptr, f32 ? 1 : 0);
    if (hipGetLastError() != hipSuccess) return HIF8_ERR_HIP;
    return y_st ? launch_gelu_stat_settle(y_st, y_smax, stream) : HIF8_OK;
}

int launch_linear_dtl(const uint16_t *x, const uint8_t *w_codes, const State *w_st, const uint16_t *bias, uint16_t *y,
                      int64_t M, int64_t N, int64_t K, hif8_stream_t stream, State *y_st, float y_smax)
{
    Groups g{};
    g.n = 1;
    g.tile_end[0] = int((N + dtl::kTile - 1) / dtl::kTile);
    g.cols[0] = int(N);
    g.st[0] = w_st;
    g.y[0] = y;
    return launch(x, w_codes, g, bias, M, N, K, stream, y_st, y_smax);
}

int launch_linear_dtl_f32(const uint16_t *x, const uint8_t *w_codes, const State *w_st, float *y, int64_t M, int64_t N,
                          int64_t K, hif8_stream_t stream)
{
    Groups g{};
    g.n = 1;
    g.tile_end[0] = int((N + dtl::kTile - 1) / dtl::kTile);
    g.cols[0] = int(N);
    g.st[0] = w_st;
    g.y[0] = (uint16_t *)y;
    return launch(x, w_codes, g, nullptr, M, N, K, stream, nullptr, 0.0f, true);
}

int launch_linear_dtl_groups(const uint16_t *x, const uint8_t *w_codes, const Groups &g, const uint16_t *bias,
                             int64_t M, int64_t N, int64_t K, hif8_stream_t stream)
{
    return launch(x, w_codes, g, bias, M, N, K, stream, nullptr, 0.0f);
}

}  // namespace hif8
