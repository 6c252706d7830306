// The kernel of the decode-free GEMM (hif8_gemm_w16.hip has its design), shared by the translation
// units that instantiate it: hif8_gemm_w16.hip (bf16 outputs, split partials) and
// hif8_gemm_scaled.hip (a scaled fp32 or bf16 output).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hif8_internal.h"
#include "hif8_gelu_dev.h"
#include "hif8_state_dev.h"

namespace hif8 {
namespace w16 {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 256;
constexpr int kBK = 64;
constexpr int kThreads = 256;
// m-tiles per group of the tile order: wide output (>= 32 n-tiles) / narrow output
constexpr int kGroupWide = 64;
constexpr int kGroupNarrow = 32;

// LDS map (bytes): operand stage s (0..4) at s * 32K, 256 rows x 128 B (64 k) with the 16-B
// chunks of row m XOR-swizzled by f(m) = (m & 7) ^ ((m >> 3) & 1): the 32 rows of a fragment
// read hit distinct banks.  The epilogue reuses the first 132 KB.
constexpr uint32_t kSlot = 32768;
constexpr uint32_t kSlots = 5;
constexpr uint32_t kOutRow = 528;  // epilogue: padded LDS row of the 256-wide output tile
constexpr uint32_t kLds = kSlots * kSlot;
static_assert(kLds >= 256 * kOutRow, "the epilogue staging fits in the ring");

#define ASMV asm volatile

template <int OFF> __device__ __forceinline__ void ldsb128(u32x4 &d, uint32_t a)
{
    ASMV("ds_read_b128 %0, %1 offset:%2" : "=v"(d) : "v"(a), "i"(OFF));
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
__device__ __forceinline__ void tie(u32x4 &a) { ASMV("" : "+v"(a)); }

__device__ __forceinline__ uint32_t f2bf_pk(float lo, float hi)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

// Per-wave loop state.  Fragment sets alternate between phases: set 0 is consumed in the even
// phase (first 32 k of a k-step) and filled in the odd one, set 1 the other way round.
// TR: the operands are k-major (token-major) in memory and in LDS, read with transposing loads
// (the K-major layout below).
template <bool TR> struct Ctx {
    u32x4 B[2][8];    // [set][j]  X fragments (m-tile j)
    u32x4 A[2][8];    // [set][i]  W fragments (n-tile i)
    uint32_t xb[2], wb[2];  // fragment read bases in stage 0: [phase p]; TR: [parity of the tile]
    uint32_t xr, wr;        // the same in the stages read this phase (TR: even tiles)
    uint32_t xr1, wr1;      // TR: odd tiles
    uint32_t xstep, wstep;  // TR: source bytes per k-step of X and W (uniform)
    f32x4 acc[8][8];
    u32x4 rx, rw, ex, ew;  // buffer resources: X, W, and the effective ones (size 0 past the end)
    uint32_t xoff[8], woff[8];  // DTL source offsets of the next X and W stage to load
    uint32_t xs, ws, ls;  // LDS offsets of the X and W stages read and of the stage loaded this phase
    uint32_t wave;
};

// K-major stage (TR): 64 k-rows x 256 columns of one operand in 128-byte blocks of 4 k-rows x
// 16 columns (the width of an MFMA tile); block (q, P) -- k-rows 4q .. 4q + 3, columns
// 16P .. 16P + 15 -- at (16 q + (P ^ ((q >> 1) & 1))) * 128, k-row 4q + e at +32 e.  A
// ds_read_b64_tr_b16 gives lane l of each 16-lane group element j of the 4 loaded by lane
// 4 j + (l % 16) / 4 of the group, at position (l % 4): with lane 4 j + u of group g loading
// columns 4u .. 4u + 3 of k-row 8 g + j (+ 4 for the second read), lane (r, g) receives k-rows
// 8 g .. 8 g + 7 of column r -- the operand layout of v_mfma_f32_16x16x32_bf16.  The XOR puts
// the k-rows 8 g + 0..3 of groups g and g + 1, read in the same cycle, in opposite halves of the
// 64 banks; within a block the 4 k-rows cover 32 distinct banks.  A DTL item (1 KB) is the 8
// blocks of one 4-k-row group and one half of the columns.

__device__ __forceinline__ uint32_t ring(uint32_t off, uint32_t n) { return off + n * kSlot >= kLds ? off + n * kSlot - kLds : off + n * kSlot; }
// before the reads of phase P: the even phase reads the second half of its own k-step, the odd
// phase the first half of the next one, whose stages are two further along the ring
template <int P, bool TR> __device__ __forceinline__ void read_bases(Ctx<TR> &c)
{
    if (P == 1) {
        c.xs = ring(c.xs, 2);
        c.ws = ring(c.ws, 2);
    }
    constexpr int p = 1 - P;
    if (TR) {
        // k-rows 32 p .. of the stage: 8 blocks of 4 k-rows further
        c.xr = c.xb[0] + c.xs + uint32_t(p) * 16384u;
        c.xr1 = c.xb[1] + c.xs + uint32_t(p) * 16384u;
        c.wr = c.wb[0] + c.ws + uint32_t(p) * 16384u;
        c.wr1 = c.wb[1] + c.ws + uint32_t(p) * 16384u;
    } else {
        c.xr = c.xb[p] + c.xs;
        c.wr = c.wb[p] + c.ws;
    }
}
template <bool TR> __device__ __forceinline__ void rotate(Ctx<TR> &c) { c.ls = ring(c.ls, 1); }
// a k-step further in the source: 64 k (128 bytes) along a row, or 64 k-rows (TR)
template <int I, bool TR> __device__ __forceinline__ void adv(Ctx<TR> &c)
{
    if (TR) {
        if (I < 8) ASMV("v_add_u32 %0, %1, %0" : "+v"(c.xoff[I]) : "s"(c.xstep));
        else ASMV("v_add_u32 %0, %1, %0" : "+v"(c.woff[I - 8]) : "s"(c.wstep));
    } else {
        if (I < 8) ASMV("v_add_u32 %0, 0x80, %0" : "+v"(c.xoff[I]));
        else ASMV("v_add_u32 %0, 0x80, %0" : "+v"(c.woff[I - 8]));
    }
}

// DTL item i of the X (OP 0) or W (OP 1) stage at the current source offsets, into the stage at
// `stage`: 1 KB at (8 wave + i) KB, rows (8 wave + i) * 8 .. + 7 x 128 B, or (TR) one half of the
// columns of 4 k-rows.
template <int OP, bool TR> __device__ __forceinline__ void issue_dtl(Ctx<TR> &c, uint32_t stage, int i)
{
    const uint32_t m0v = __builtin_amdgcn_readfirstlane(stage + (c.wave * 8u + uint32_t(i)) * 1024u);
    if (OP == 0) dtl_load(m0v, c.xoff[i], c.ex);
    else dtl_load(m0v, c.woff[i], c.ew);
}
template <int OP, bool TR> __device__ __forceinline__ void issue_dtl(Ctx<TR> &c, int i) { issue_dtl<OP>(c, c.ls, i); }

// two transposing reads (TR): k-rows 8 g + 0..3 and 8 g + 4..7 of a 16-column tile
template <int OFF> __device__ __forceinline__ void ldstr(u32x4 &d, uint32_t a)
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 lo, hi;
    ASMV("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(a), "i"(OFF));
    ASMV("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(a), "i"(OFF + 2048));
    d = u32x4{lo.x, lo.y, hi.x, hi.y};
}
// one of the two transposing reads of a fragment (TR): H = 0 its k-rows 8 g + 0..3, H = 1 the
// next four, into the fragment's low or high half
template <int OFF, int H> __device__ __forceinline__ void ldstr_half(u32x4 &d, uint32_t a)
{
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    u32x2 v;
    ASMV("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(a), "i"(OFF + H * 2048));
    if (H == 0) d = u32x4{v.x, v.y, d.z, d.w};
    else d = u32x4{d.x, d.y, v.x, v.y};
}
template <int NXT, int J, int H, bool TR> __device__ __forceinline__ void rd_x_half(Ctx<TR> &c)
{
    ldstr_half<(J & ~1) * 128, H>(c.B[NXT][J], (J & 1) ? c.xr1 : c.xr);
}
template <int NXT, int I, int H, bool TR> __device__ __forceinline__ void rd_w_half(Ctx<TR> &c)
{
    ldstr_half<(I & ~1) * 128, H>(c.A[NXT][I], (I & 1) ? c.wr1 : c.wr);
}
// fragment reads: 16 rows x 128 B per m- or n-tile, or (TR) a 16-column block column
template <int NXT, int J, bool TR> __device__ __forceinline__ void rd_x(Ctx<TR> &c)
{
    if (TR) ldstr<(J & ~1) * 128>(c.B[NXT][J], (J & 1) ? c.xr1 : c.xr);
    else ldsb128<J * 2048>(c.B[NXT][J], c.xr);
}
template <int NXT, int I, bool TR> __device__ __forceinline__ void rd_w(Ctx<TR> &c)
{
    if (TR) ldstr<(I & ~1) * 128>(c.A[NXT][I], (I & 1) ? c.wr1 : c.wr);
    else ldsb128<I * 2048>(c.A[NXT][I], c.wr);
}
// Issue order of a phase's 64 MFMAs over the 8 x 8 tiles (i: W fragment, j: X fragment): 2 x 2
// blocks, (2bi, 2bj), (2bi + 1, 2bj), (2bi + 1, 2bj + 1), (2bi, 2bj + 1), the blocks in a snake
// along j.  Each fragment register pair feeds two MFMAs in a row before the next one switches in,
// and at the board's power limit that cost less: against the row order (A fixed for 8 MFMAs, B
// changing every MFMA) 1.3-2.6 % on the 14B shapes; a plain snake 0.3-1.7 %, 4 x 4 blocks 0.4-1.7 %,
// 2 x 4 or 4 x 2 blocks 1.0-1.4 %, a Hilbert curve 0.9-2.4 % (A/B of builds on one box).  Every
// accumulator still receives its products in k order, so the outputs do not change.
constexpr int blk2_order(int m)
{
    const int q = m / 4, r = m % 4, bi = q / 4, bj = (q / 4) % 2 ? 3 - q % 4 : q % 4;
    return 8 * (2 * bi + ((r == 1 || r == 2) ? 1 : 0)) + 2 * bj + (r >= 2 ? 1 : 0);
}
template <int CUR, int MI, bool TR> __device__ __forceinline__ void mm(Ctx<TR> &c)
{
    constexpr int i = blk2_order(MI) / 8, j = blk2_order(MI) % 8;
    mfma(c.acc[i][j], c.A[CUR][i], c.B[CUR][j]);
}
// after the wait covering the fragments of set SET
template <int SET, bool TR> __device__ __forceinline__ void tie_set(Ctx<TR> &c)
{
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        tie(c.B[SET][j]);
        tie(c.A[SET][j]);
    }
}

#include "hif8_gemm_schedule_w16.inc"

// a / s for a scale s >= 0, Inf or NaN: the product with the rounded reciprocal, corrected by its exact
// remainder (two fma), the IEEE quotient wherever that is a normal number.  Below 2^-126, where the
// reciprocal may overflow (an fp32 tensor with an amax above scale_max * 2^126), a and s are both taken
// 2^64 times: a sum that overflows so has an infinite quotient.  Where the quotient is not finite the
// correction would turn an infinity into NaN; an infinite s leaves none (the quotient is 0).
struct Divisor {
    float up, s, r;
    __device__ explicit Divisor(float scale) : up(scale < 0x1p-126f ? 0x1p64f : 1.0f), s(scale * up), r(1.0f / s)
    {
        if (s == __builtin_inff()) s = 0.0f;
    }
    __device__ __forceinline__ float operator()(float a) const
    {
        a *= up;
        const float q = a * r;
        const float c = __builtin_fmaf(__builtin_fmaf(-q, s, a), r, q);
        return __builtin_fabsf(q) < __builtin_inff() ? c : q;
    }
};
__device__ __forceinline__ void store_scaled(void *y, bool f32, size_t at, const f32x4 &a, const Divisor &d)
{
    const f32x4 v = f32x4{d(a[0]), d(a[1]), d(a[2]), d(a[3])};
    if (f32) *(f32x4 *)((float *)y + at) = v;
    else *(uint2 *)((uint16_t *)y + at) = uint2{f2bf_pk(v[0], v[1]), f2bf_pk(v[2], v[3])};
}

// Tile t of the order: groups of group_m m-tiles, n-tiles outer within a group.
__device__ __forceinline__ void tile_origin(int t, int tiles_m, int tiles_n, int group_m, int &m0, int &n0)
{
    const int group = t / (group_m * tiles_n);
    const int first_m = group * group_m;
    const int gm = (tiles_m - first_m) < group_m ? (tiles_m - first_m) : group_m;
    const int within = t - group * group_m * tiles_n;
    m0 = (first_m + within % gm) * kTile;
    n0 = (within / gm) * kTile;
}

// EPI 0: y = rnd(acc + bias).  EPI 1: the same y, and the GELU statistic of y (its max, or a
// non-finite flag) folded into y_st's accumulator; the settle kernel launched after it turns that
// into amax|GELU(y)| and its scale when max y settles it (hif8_gelu_dev.h).  The output features
// are G.n groups, each with its output buffer.
// EPI 2, split tiles: each workgroup computes one of `splits` k ranges (consecutive k-steps) of one
// tile from tile0 on and writes its fp32 sums to part (256 KB per workgroup, in the accumulators'
// lane order) for k_split_reduce.  (A separate instantiation: in the same kernel as the bf16
// epilogue, the register allocator moved all accumulators to VGPRs ahead of the branch and
// spilled.)
// EPI 3: y = acc / scale, no bias, with the scale of the state y_st (1 without one): one of the operands holds the
// raw HiF8 values of codes instead of their quotients by the scale.  y is fp32 when splits != 0, else
// bf16.
// TR: X and Wq are k-major, X^T [K][M] and Wq^T [K][N] (contiguous rows of M and N elements):
// the weight gradient's grad_q [tokens][out] and x_q [tokens][in] as they are, K = tokens.  Rows
// past K read as zero through the buffers' ranges; columns past M or N read other data, which
// only reaches outputs that are not stored.
template <int EPI, bool TR = false>
__global__ __launch_bounds__(kThreads, 1) void k_linear_w16(const uint16_t *__restrict__ X, const uint16_t *__restrict__ Wq,
                                                            const Groups G, const uint16_t *__restrict__ bias,
                                                            int M, int N, int K, int tiles_m, int tiles_n,
                                                            int group_m, State *__restrict__ y_st, int tile0,
                                                            int splits, float *__restrict__ part)
{
    __shared__ __attribute__((aligned(1024))) uint8_t smem[kLds];
    ASMV("; lds base %0" ::"v"(uint32_t(uintptr_t(smem))) : "memory");
    Ctx<TR> c;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    c.wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15u, g = lane >> 4;

    int t = blockIdx.x;
    int nk = TR ? (K + kBK - 1) / kBK : K / kBK, kb = 0;
    uint32_t part_at = 0;
    if (EPI == 2) {
        // range-major order over the XCDs (workgroup b runs on XCD b % 8): an XCD's workgroups share
        // one or two k ranges, so its L2 fetches each operand slice once for all of its tiles
        const int nwg = int(gridDim.x), tail = nwg / splits, xcd = t & 7, in_xcd = nwg >> 3, more = nwg & 7;
        const int at = xcd * in_xcd + (xcd < more ? xcd : more) + (t >> 3);
        const int range = at / tail, tile = at - range * tail;
        t = tile0 + tile;
        part_at = uint32_t(tile) * uint32_t(splits) + uint32_t(range);
        const int per = (nk + splits - 1) / splits;
        kb = range * per;
        nk = (nk - kb < per ? nk - kb : per);
    }
    int m0, n0;
    tile_origin(t, tiles_m, tiles_n, group_m, m0, n0);
    int gi = 0;
    while (gi + 1 < G.n && n0 / kTile >= G.tile_end[gi]) ++gi;
    uint16_t *__restrict__ Y = G.y[gi];
    const int col0 = gi == 0 ? 0 : G.tile_end[gi - 1] * kTile;
    const int ycols = G.cols[gi];

    if (!TR) {
        // the buffers start at k-step kb of row 0; rows past M or N lie past the range
        const uint32_t kofs = uint32_t(kb) * uint32_t(kBK) * 2u;
        const uint64_t xa = uint64_t(X) + uint64_t(m0) * uint64_t(K) * 2u + kofs;
        const uint32_t xrows = uint32_t(M - m0 < kTile ? M - m0 : kTile);
        c.rx = u32x4{uint32_t(xa), uint32_t(xa >> 32), xrows * uint32_t(K) * 2u - kofs, 0x00020000u};
        const uint64_t wa = uint64_t(Wq) + uint64_t(n0) * uint64_t(K) * 2u + kofs;
        const uint32_t wrows = uint32_t(N - n0 < kTile ? N - n0 : kTile);
        c.rw = u32x4{uint32_t(wa), uint32_t(wa >> 32), wrows * uint32_t(K) * 2u - kofs, 0x00020000u};
    } else {
        // the buffers start at column m0 (n0) of k-row 64 kb and end with the matrix: k-rows past
        // K lie past the range (the caller keeps K * M * 2 and K * N * 2 below 2^32)
        const uint64_t xofs = uint64_t(kb) * uint64_t(kBK) * uint64_t(M) * 2u + uint64_t(m0) * 2u;
        const uint64_t xa = uint64_t(X) + xofs;
        c.rx = u32x4{uint32_t(xa), uint32_t(xa >> 32), uint32_t(uint64_t(K) * uint64_t(M) * 2u - xofs), 0x00020000u};
        const uint64_t wofs = uint64_t(kb) * uint64_t(kBK) * uint64_t(N) * 2u + uint64_t(n0) * 2u;
        const uint64_t wa = uint64_t(Wq) + wofs;
        c.rw = u32x4{uint32_t(wa), uint32_t(wa >> 32), uint32_t(uint64_t(K) * uint64_t(N) * 2u - wofs), 0x00020000u};
        c.xstep = __builtin_amdgcn_readfirstlane(uint32_t(kBK) * uint32_t(M) * 2u);
        c.wstep = __builtin_amdgcn_readfirstlane(uint32_t(kBK) * uint32_t(N) * 2u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        c.rx[i] = __builtin_amdgcn_readfirstlane(c.rx[i]);
        c.rw[i] = __builtin_amdgcn_readfirstlane(c.rw[i]);
    }
    const uint32_t wm = (c.wave & 1u) * 128u, wn = (c.wave >> 1) * 128u;
    if (!TR) {
        // DTL source offsets of k-step 0.  LDS 16-B slot s of a stage is written by lane s%64 of
        // load s/64; its source chunk is the slot's chunk un-swizzled (the XOR is an involution).
        // X and W rows share the layout.
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t row = (c.wave * 8u + i) * 8u + (lane >> 3);
            const uint32_t ch = (lane & 7u) ^ (lane >> 3) ^ uint32_t(i & 1);
            c.xoff[i] = row * uint32_t(K) * 2u + ch * 16u;
            c.woff[i] = c.xoff[i];
        }
        // Fragment read bases.  Lane (r, g) = (lane & 15, lane >> 4) holds k = 32p + 8g .. +7 of
        // phase p for row r of its 16-row tile, for both operands: chunk 4p + g of rows wm + 16j + r
        // (X) and wn + 16i + r (W); f(row) = f(r).
        const uint32_t fr = (r & 7u) ^ ((r >> 3) & 1u);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t ch = ((4u * p + g) ^ fr) << 4;
            c.xb[p] = (wm + r) * 128u + ch;
            c.wb[p] = (wn + r) * 128u + ch;
        }
    } else {
        // DTL item it = 8 wave + i: 4-k-row group q = it / 2, column half it % 2; lane s writes
        // block P' = 8 (it % 2) + s / 8, k-row e = (s % 8) / 2, bytes 16 (s % 2) .. of its 32; the
        // source is column block P = P' ^ ((q >> 1) & 1) of k-row 4 q + e.
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t it = c.wave * 8u + uint32_t(i), q = it >> 1;
            const uint32_t pb = ((it & 1u) * 8u + (lane >> 3)) ^ ((q >> 1) & 1u);
            const uint32_t krow = 4u * q + ((lane & 7u) >> 1);
            const uint32_t col = pb * 32u + (lane & 1u) * 16u;
            c.xoff[i] = krow * uint32_t(M) * 2u + col;
            c.woff[i] = krow * uint32_t(N) * 2u + col;
        }
        // Fragment read bases: lane (L, g) = (lane & 15, lane >> 4) reads k-rows 8 g + L / 4 (and
        // + 4) of the stage, columns 4 (L % 4) .. of a 16-column block: block group q = 2 g (+ 1),
        // XOR bit s = g & 1.  Even tiles J sit at J * 128 + s * 128, odd ones at (J - 1) * 128 +
        // 128 - s * 128 from the quadrant's first block (wm / 16 or wn / 16).
        const uint32_t sx = g & 1u;
        const uint32_t common = g * 4096u + (r >> 2) * 32u + (r & 3u) * 8u;
        c.xb[0] = common + (wm / 16u) * 128u + sx * 128u;
        c.xb[1] = common + (wm / 16u) * 128u + 128u - sx * 128u;
        c.wb[0] = common + (wn / 16u) * 128u + sx * 128u;
        c.wb[1] = common + (wn / 16u) * 128u + 128u - sx * 128u;
    }

    // The bias words of this lane's output features (4 per MFMA tile row i), loaded ahead of the
    // operand loads: they land during the main loop (in-order completion puts them before every
    // operand wait), where in the epilogue each was a global load waited for on its own.
    uint2 bw[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int n = n0 + int(wn + uint32_t(i * 16) + 4u * (lane >> 4));
        bw[i] = (bias && n < N) ? *(const uint2 *)(bias + n) : uint2{0u, 0u};
    }

    // Prologue: X and W of k-steps 0 and 1 into stages 0..3; wait for k-step 0.
    c.ex = c.rx;
    c.ew = c.rw;
#pragma unroll
    for (int i = 0; i < 8; ++i) issue_dtl<0>(c, 0u, i);
#pragma unroll
    for (int i = 0; i < 8; ++i) issue_dtl<1>(c, kSlot, i);
    c.ex[2] = nk > 1 ? c.rx[2] : 0u;
    c.ew[2] = nk > 1 ? c.rw[2] : 0u;
    adv<0>(c); adv<1>(c); adv<2>(c); adv<3>(c); adv<4>(c); adv<5>(c); adv<6>(c); adv<7>(c);
    adv<8>(c); adv<9>(c); adv<10>(c); adv<11>(c); adv<12>(c); adv<13>(c); adv<14>(c); adv<15>(c);
#pragma unroll
    for (int i = 0; i < 8; ++i) issue_dtl<0>(c, 2u * kSlot, i);
#pragma unroll
    for (int i = 0; i < 8; ++i) issue_dtl<1>(c, 3u * kSlot, i);
    adv<0>(c); adv<1>(c); adv<2>(c); adv<3>(c); adv<4>(c); adv<5>(c); adv<6>(c); adv<7>(c);
    adv<8>(c); adv<9>(c); adv<10>(c); adv<11>(c); adv<12>(c); adv<13>(c); adv<14>(c); adv<15>(c);
    wait_vm<16>();
    barrier();
    // reads for the first phase (k-step 0, first half) into set 0
    c.xs = 0;
    c.ws = kSlot;
    c.xr = c.xb[0];
    c.wr = c.wb[0] + kSlot;
    c.xr1 = c.xb[1];  // TR: the odd tiles' bases
    c.wr1 = c.wb[1] + kSlot;
    rd_w<0, 0>(c); rd_x<0, 0>(c); rd_x<0, 1>(c); rd_x<0, 2>(c); rd_x<0, 3>(c);
    rd_x<0, 4>(c); rd_x<0, 5>(c); rd_x<0, 6>(c); rd_x<0, 7>(c);
    rd_w<0, 1>(c); rd_w<0, 2>(c); rd_w<0, 3>(c); rd_w<0, 4>(c); rd_w<0, 5>(c); rd_w<0, 6>(c); rd_w<0, 7>(c);
    c.ls = 4u * kSlot;  // the first phase loads X of k-step 2
    read_bases<0>(c);

#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) c.acc[i][j] = f32x4{};
    // One k-step per iteration.  The loads of k-step kk + 2 use the resources with size 0 past
    // the end: they read nothing and nothing consumes them.
    for (int kk = 0; kk < nk; ++kk) {
        c.ex[2] = kk + 2 < nk ? c.rx[2] : 0u;
        c.ew[2] = kk + 2 < nk ? c.rw[2] : 0u;
        if (TR) {
            phase0_tr(c);
            phase1_tr(c);
        } else {
            phase0(c);
            phase1(c);
        }
    }
    // no load may still target LDS when it is reused or released
    wait_vm<0>();
    wait_lgkm<0>();
    // the last MFMAs' results must be complete before the accumulators are read
    ASMV("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) ASMV("" : "+a"(c.acc[i][j]));

    if (EPI == 2) {
        // a k range of a split tile: the fp32 sums, 1 KB per store instruction
        f32x4 *P = (f32x4 *)part + size_t(part_at) * 16384u + c.wave * 4096u + lane;
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) P[(i * 8 + j) * 64] = c.acc[i][j];
        return;
    }
    if (EPI == 3) {
        // straight from the accumulators: 4 consecutive features per lane, 16 (fp32) or 8 bytes
        const Divisor d(y_st ? y_st->scale : 1.0f);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int n = n0 + int(wn) + i * 16 + int(4u * g);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int m = m0 + int(wm) + j * 16 + int(r);
                if (m < M && n < N) store_scaled(Y, splits != 0, size_t(m) * size_t(N) + size_t(n), c.acc[i][j], d);
            }
        }
        return;
    }

    // Epilogue.  acc[i][j] lane (r, g), element e: D[n][m] with n = wn + 16i + 4g + e,
    // m = wm + 16j + r.  Rows go to LDS (padded), then each wave stores 2 rows x 512 B per
    // instruction.
    __syncthreads();
    {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            {
                const uint32_t nl = wn + uint32_t(i * 16) + 4u * g;
                const uint2 bb = bw[i];
                const float b0 = __builtin_bit_cast(float, bb.x << 16);
                const float b1 = __builtin_bit_cast(float, bb.x & 0xFFFF0000u);
                const float b2 = __builtin_bit_cast(float, bb.y << 16);
                const float b3 = __builtin_bit_cast(float, bb.y & 0xFFFF0000u);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const f32x4 &a = c.acc[i][j];
                    uint2 v;
                    v.x = f2bf_pk(a[0] + b0, a[1] + b1);
                    v.y = f2bf_pk(a[2] + b2, a[3] + b3);
                    *(uint2 *)(smem + (wm + uint32_t(j * 16) + r) * kOutRow + nl * 2u) = v;
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

}  // namespace w16
}  // namespace hif8
