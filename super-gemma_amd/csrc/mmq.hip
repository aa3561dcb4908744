// Prefill int8 MMQ GEMM for gfx950: Y[m×n] = Xq[m×k] · W[n×k]^T with the
// per-32-block rescale of the reference's gemm_q4_0_i8 family
// (crates/sg-gpu/shaders/gemm_q4_0_i8.wgsl:153-393; FFN-down variant
// gemm_q4_0_i8_bb_pfd.wgsl): for every block b,
//     Y[m,n] += (d_a[m,b] * d_w[n,b]) * f32( sum_j xq[m,32b+j] * (wq[n,32b+j]-8) )
// where the i32 block dot is exact and the scale product of two f16 values
// is exact in f32.
//
// Design:
//  * One v_mfma_i32_32x32x32_i8 is exactly one Q4_0 block (K = 32) of a
//    32×32 output tile: lane (r, h) = (lane%32, lane/32) feeds 16 K-bytes
//    [16h, 16h+16) of row/column r.  For the weights that half is the low
//    (h = 0) or high (h = 1) nibbles of the block's 16 qs bytes, so the
//    logical K order of q4_0.rs:31-42 falls out with no shuffle.
//  * Workgroup = 4 waves (2×2), tile 128×128, each wave 64×64 = 2×2 MFMA
//    tiles.  A K-stage is 4 blocks (128 K): activations (int8) and weights
//    (unpacked once per workgroup to int8 16·(q-8) by the loading thread) go to
//    LDS, rows padded to 144 B so the 16-byte fragment reads of 8 lanes hit
//    32 distinct banks.  Double-buffered: stage s+1's global loads are in
//    flight while stage s computes; one barrier per stage.
//  * Rescale: the scale products d_a·d_w of a 32×32 tile come from the
//    matrix cores too — one v_mfma_f32_32x32x8_f16 whose only non-zero K
//    term is (d_a[row], d_w[col]) gives the exact outer product (f16·f16 is
//    exact in f32) in the accumulator layout of the int8 MFMA (the K=8 form
//    costs the matrix cores less than the K=16 one: config 2 571 -> 620-627
//    TOP/s, M = 4096 750 -> 786, with half the operand registers).  The VALU is
//    left with one cvt and one FMA per output element and block, and that —
//    not the MFMA — bounds the kernel: a wave64 VALU op holds its SIMD for 4
//    cycles, and counters put VALU issue at 88% of the cycles (M = 4096,
//    K = 5376, N = 21504).  Every other VALU op of the loop therefore costs
//    its share: with uniform pointers advanced by the scalar unit, one-op
//    unpacks and the scale words moved up instead of selected, a stage takes
//    632 VALU ops against 683 (512 of them cvt + FMA, 32 MFMA issues):
//    1215-1221 -> 1146-1149 us there; K = 21504, M = 2048, split 4 666 -> 643;
//    K = 5376, M = 512 172 -> 170.
//  * Ragged tiles read clamped rows and run the same loop (they had a
//    bounds-checked one: 1500 tokens through six layers of the released
//    geometry 15.3 -> 14.15 ms, M = 37, N = 8192 86 -> 81 us).
//  * Tile order is XCD-aware: consecutive workgroup ids land on different
//    XCDs (each with its own L2), so ids are remapped so that every XCD
//    walks a contiguous range of N-tiles with all their M-tiles, and a
//    weight strip is fetched from HBM once per XCD; with many M-tiles the
//    XCD takes them 8 at a time across its N-tiles.
//  * Split-K (slices of the block range, factor 1/2/4/8) writes fp32
//    partial tiles; a second kernel sums them in fixed order s = 0..S-1.
#include "sgq_internal.h"

namespace sgq {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int BM = 128, BN = 128, KB = 4;   // tile rows, cols, blocks per stage
constexpr int ROWB = KB * 32 + 16;          // padded LDS row bytes (144)
constexpr int kMWG = 256;
#ifndef SGQ_MMQ_WG_PER_CU
#define SGQ_MMQ_WG_PER_CU 2
#endif

struct Stage {
    int8_t a[BM * ROWB];      // activations, [row][k]
    int8_t b[BN * ROWB];      // weights 16·(q-8), [col][k]
    uint2 da[BM];             // activation scales (f16 bits), [row], 4 blocks
    uint2 dw[BN];             // weight scales (f16 bits), [col], 4 blocks
    uint2 zero[34];           // [0] and [32] zero: the scale words of lanes 32..63 (ld_scales)
};

// Nibbles as int8 16·(q-8): the nibble moved to the byte's high half with its
// top bit flipped, one three-input logic op (plus a shift for the low
// nibbles) per 4 weights against 3-4 for q-8 itself.  The factor 16 is taken
// off the finished sums, exactly: a block dot stays below 2^20, and the sums
// (scales are f16) far inside fp32's exponent range.
constexpr float kUnscale = 1.0f / 16.0f;
__device__ __forceinline__ uint32_t unpack_lo(uint32_t q) {
    return ((q << 4) & 0xF0F0F0F0u) ^ 0x80808080u;
}
__device__ __forceinline__ uint32_t unpack_hi(uint32_t q) {
    return (q & 0xF0F0F0F0u) ^ 0x80808080u;
}

struct Prefetch {
    v4i a[4];          // 64 activation bytes: row = tid/2, k-half = tid%2 (native
                       // vectors: HIP's uint4 is a struct, copied through scratch)
    uint32_t w[9];     // two Q4_0 blocks (36 bytes): col = tid/2, blocks 2*(tid%2)+{0,1}
    uint2 da;          // threads < 128: 4 block scales of row tid
};

// A tile's three sources: uniform pointers (scalar registers, advanced by
// the scalar unit) plus a 32-bit offset per thread that stays fixed, so a
// stage's loads cost the VALU nothing.  Rows past m and columns past n
// (ragged tiles) read the last row / column instead, and their results are
// not stored: odd sizes run the same loop as whole tiles.
typedef const __attribute__((address_space(1))) char *gptr;
template <typename O>         // uint32_t; uint64_t from kWideK on (128 rows' offsets)
struct TileSrc {
    gptr a, w, d;             // tile row 0 / column 0 / row 0, at the stage's first block
    O oa, ow, od, od2;        // byte offsets: row t/2, byte 64·(t%2) / column t/2, block
                              // 2·(t%2) / row t, blocks 0-1 and 2-3
};
constexpr uint32_t kWideK = 1u << 25;

template <typename O>
__device__ __forceinline__ TileSrc<O> tile_src(const int8_t *__restrict__ xq,
                                            const uint16_t *__restrict__ xs,
                                            const uint8_t *__restrict__ W, int m, int n, int k,
                                            int nb, int m0, int n0) {
    const uint32_t t = threadIdx.x, pair = nb < KB ? 0 : t & 1;  // nb = 2: both read blocks 0-1
    TileSrc<O> s;
    s.a = (gptr)(xq + (size_t)m0 * k);
    s.w = (gptr)(W + (size_t)n0 * nb * 18);
    s.d = (gptr)(xs + (size_t)m0 * nb);
    s.oa = (O)min((int)t >> 1, m - 1 - m0) * (O)k + pair * 64;
    s.ow = ((O)min((int)t >> 1, n - 1 - n0) * (O)nb + 2 * pair) * 18;
    s.od = (O)min((int)t & (BM - 1), m - 1 - m0) * (O)nb * 2;
    s.od2 = s.od + (nb < KB ? 0 : 4);
    return s;
}

typedef uint32_t u32a2 __attribute__((aligned(2)));  // xs is 2-byte aligned
template <typename O>
__device__ __forceinline__ void load_stage(Prefetch &pf, const TileSrc<O> &src, int b0) {
    gptr a = src.a + (size_t)b0 * 32, w = src.w + (size_t)b0 * 18, d = src.d + (size_t)b0 * 2;
    // Base in scalar registers, 32-bit offset in a vector register: the loads'
    // own addressing form (the offsets are made opaque here, or the compiler
    // widens them once outside the loop and adds 64-bit vectors per stage).
    O oa = src.oa, ow = src.ow, od = src.od, od2 = src.od2;
    asm volatile("" : "+s"(a), "+s"(w), "+s"(d), "+v"(oa), "+v"(ow), "+v"(od), "+v"(od2));
#pragma unroll
    for (int i = 0; i < 4; i++)
        pf.a[i] = *(const __attribute__((address_space(1))) v4i *)(a + oa + 16 * i);
    // plain loads: a weight strip serves every M-tile of its column group
    // (from L2); with the nontemporal hint config 2 ran at 526-530 against
    // 573-579 TOP/s and M = 4096 at 676 against 758-763
#pragma unroll
    for (int j = 0; j < 9; j++)
        pf.w[j] = *(const __attribute__((address_space(1))) uint32_t *)(w + ow + 4 * j);
    if (threadIdx.x < BM)
        pf.da = make_uint2(*(const __attribute__((address_space(1))) u32a2 *)(d + od),
                           *(const __attribute__((address_space(1))) u32a2 *)(d + od2));
}

// Zero scales for the dead block pair of a K end with two blocks: their
// products then add exact zeros (the dots are finite).
__device__ __forceinline__ void kill_pair(Prefetch &pf, int dead) {
    if ((int)(threadIdx.x & 1) == dead) pf.w[0] = pf.w[4] = 0u;
    if (dead)
        pf.da.y = 0u;
    else
        pf.da.x = 0u;
}

__device__ __forceinline__ void store_stage(const Prefetch &pf, Stage &S) {
    const int t = threadIdx.x;
    {
        const int row = t >> 1, half = t & 1;
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<v4i *>(&S.a[row * ROWB + half * 64 + i * 16]) = pf.a[i];
    }
    {
        const int col = t >> 1, pair = t & 1;
        // Block A: d in low half of w0, qs bytes = w0.hi .. w4.lo
        uint32_t qa[4], qb[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            qa[j] = __builtin_amdgcn_alignbyte(pf.w[j + 1], pf.w[j], 2);
            qb[j] = pf.w[5 + j];
        }
        int8_t *dst = &S.b[col * ROWB + pair * 64];
        uint4 lo, hi;
        lo = make_uint4(unpack_lo(qa[0]), unpack_lo(qa[1]), unpack_lo(qa[2]), unpack_lo(qa[3]));
        hi = make_uint4(unpack_hi(qa[0]), unpack_hi(qa[1]), unpack_hi(qa[2]), unpack_hi(qa[3]));
        *reinterpret_cast<uint4 *>(dst) = lo;
        *reinterpret_cast<uint4 *>(dst + 16) = hi;
        lo = make_uint4(unpack_lo(qb[0]), unpack_lo(qb[1]), unpack_lo(qb[2]), unpack_lo(qb[3]));
        hi = make_uint4(unpack_hi(qb[0]), unpack_hi(qb[1]), unpack_hi(qb[2]), unpack_hi(qb[3]));
        *reinterpret_cast<uint4 *>(dst + 32) = lo;
        *reinterpret_cast<uint4 *>(dst + 48) = hi;
        // the two blocks' scales: low half of word 0, high half of word 4
        reinterpret_cast<uint32_t *>(&S.dw[col])[pair] =
            (pf.w[0] & 0xffffu) | (pf.w[4] & 0xffff0000u);
    }
    if (t < BM) S.da[t] = pf.da;
}

// Tile of the jl-th workgroup slot of XCD x (workgroup b runs on XCD b % 8,
// jl = b / 8; tiles % 8 == 0, else x = 0 and jl = b).  XCD-aware order:
// every XCD walks a contiguous range of the tiles.
constexpr int kXcds = 8, kGroupM = 8;
__device__ __forceinline__ void mmq_tile(int x, int jl, int mt, int nt, int *tm, int *tn) {
    const int tiles = mt * nt;
    if (nt % kXcds == 0 && mt % kGroupM == 0) {
        // XCD x owns N-tiles [x·nt/8, (x+1)·nt/8) with every M-tile, walked in
        // groups of 8 M-tiles across all its N-tiles: the XCD's resident
        // tiles (64) then share 8 activation panels and 8 weight strips in
        // its L2 instead of all M-tiles' panels and 2 strips (M = 4096: 646
        // -> 656 TOP/s, the 4096-token prefill +1.3-2%; 16 M-tiles per group
        // measured as the plain order)
        const int ntx = nt / kXcds, gs = kGroupM * ntx;
        const int g = jl / gs, r = jl % gs;
        *tm = g * kGroupM + r % kGroupM;
        *tn = x * ntx + r / kGroupM;
    } else if (tiles % kXcds == 0 && mt % kGroupM == 0) {
        // N-tiles not a multiple of 8: the same grouped order over the whole
        // grid, each XCD a contiguous eighth of it (the down projection at
        // M = 4096, K = 21504: 614-627 -> 634-642 TOP/s)
        const int j = x * (tiles / kXcds) + jl, gs = kGroupM * nt;
        const int g = j / gs, r = j % gs;
        *tm = g * kGroupM + r % kGroupM;
        *tn = r / kGroupM;
    } else {
        const int id = tiles % kXcds == 0 ? x * (tiles / kXcds) + jl : jl;
        *tn = id / mt, *tm = id % mt;
    }
}

// Tail split (split = 1 only): when the tiles are more than whole rounds of
// the resident workgroups, each XCD computes its first tail_fx tiles whole
// and splits each of its remaining tiles over K into tail_st parts, one
// workgroup each, so the last round is full; the parts go to tailp as
// 128×128 fp32 tiles (slot = x·(tiles/8 − tail_fx) + tail tile, part) and
// mmq_tail_reduce_kernel sums them in part order.
struct TailSplit {
    int fx, st;    // whole tiles per XCD, parts per tail tile (0: off)
    float *part;
};

// HOUT: the output is f16 (uint16_t bits, each sum rounded to nearest even:
// the reference's y binding, gemm_q4_0_i8.wgsl:63); else fp32.  TAIL: the
// tail split is built in (a separate kernel, so the others keep their code).
template <bool HOUT, bool TAIL = false, typename O = uint32_t>
__global__ __launch_bounds__(kMWG, SGQ_MMQ_WG_PER_CU) void mmq_kernel(const uint8_t *__restrict__ W,
                                                      const int8_t *__restrict__ xq,
                                                      const uint16_t *__restrict__ xs,
                                                      void *__restrict__ out_, int m, int n,
                                                      int k, int mt, int nt, int split,
                                                      TailSplit ts) {
    extern __shared__ __align__(16) uint8_t smem[];
    Stage *stages = reinterpret_cast<Stage *>(smem);

    // XCD-aware tile order (see header).
    const int tiles = mt * nt;
    const bool by_xcd = tiles % kXcds == 0;
    const int x = by_xcd ? (int)(blockIdx.x % kXcds) : 0;
    int jl = by_xcd ? (int)(blockIdx.x / kXcds) : (int)blockIdx.x;
    int z = blockIdx.y;
    int tail_slot = -1;
    if (TAIL && jl >= ts.fx) {
        const int k2 = jl - ts.fx, lx = tiles / kXcds - ts.fx;
        jl = ts.fx + k2 / ts.st;
        z = k2 % ts.st;
        split = ts.st;
        tail_slot = x * lx + k2 / ts.st;
    }
    int tm, tn;
    mmq_tile(x, jl, mt, nt, &tm, &tn);
    const int m0 = tm * BM, n0 = tn * BN;

    const int nb = k / 32;
    const int b_beg = (int)((long)nb * z / split) & ~(KB - 1);
    const int b_end = z + 1 == split ? nb : ((int)((long)nb * (z + 1) / split) & ~(KB - 1));
    const int n_stages = (b_end - b_beg + KB - 1) / KB;

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int r = lane & 31, h = lane >> 5;

    float acc[2][2][16];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[a][b][i] = 0.f;

    // register prefetch one stage ahead: stage s+1's global loads are in
    // flight while stage s computes (four blocks of MFMAs and rescales),
    // then go to the other LDS buffer
    Prefetch pf;
    const TileSrc<O> src = tile_src<O>(xq, xs, W, m, n, k, nb, m0, n0);
    // A range that ends with two blocks (nb is even, the split bounds are
    // multiples of KB): its last stage starts two blocks early, with the scales
    // of the pair it has seen zeroed, so its loads stay in the rows; a K of 64
    // has one stage whose second pair is dead.
    const bool short_end = (b_end - b_beg) % KB != 0;
    const int dead = nb < KB ? 1 : 0;
    auto load = [&](int s) {
        const int b0 = b_beg + s * KB;
        load_stage(pf, src, b0 + KB <= b_end || dead ? b0 : b_end - KB);
    };
    auto store = [&](int s) {
        if (short_end && s + 1 == n_stages) kill_pair(pf, dead);
        store_stage(pf, stages[s & 1]);
    };
    if (threadIdx.x < 4) stages[threadIdx.x >> 1].zero[32 * (threadIdx.x & 1)] = make_uint2(0u, 0u);
    if (n_stages > 0) {
        load(0);
        store(0);
    }
    __syncthreads();

    // LDS operands of one block: int8 fragments of the wave's two row and
    // two column tiles
    struct Ops {
        v4i af[2], bf[2];
    };
    // the f16 scale bits of the wave's two row and two column tiles for the
    // stage's four blocks (two per word), read once per stage; zero in the
    // lanes (h = 1) whose K terms of the scale MFMA are zero: they read the
    // stage's zero words
    uint32_t sa[2], sa2[2], sb[2], sb2[2];  // blocks 0-1, blocks 2-3
    const uint32_t ga = (uint32_t)(h ? offsetof(Stage, zero) : offsetof(Stage, da) + (wm * 64 + r) * 8);
    const uint32_t gb = (uint32_t)(h ? offsetof(Stage, zero) : offsetof(Stage, dw) + (wn * 64 + r) * 8);
    auto ld_scales = [&](const Stage &S) {
        const uint8_t *sp = reinterpret_cast<const uint8_t *>(&S);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const uint2 a = *reinterpret_cast<const uint2 *>(sp + ga + i * 256);
            const uint2 b = *reinterpret_cast<const uint2 *>(sp + gb + i * 256);
            sa[i] = a.x, sa2[i] = a.y, sb[i] = b.x, sb2[i] = b.y;
        }
    };
    const uint32_t fa = (uint32_t)((wm * 64 + r) * ROWB + h * 16);
    const uint32_t fb = (uint32_t)(offsetof(Stage, b) + (wn * 64 + r) * ROWB + h * 16);
    auto ld_ops = [&](const Stage &S, int blk, Ops &o) {
        const uint8_t *sp = reinterpret_cast<const uint8_t *>(&S) + blk * 32;
#pragma unroll
        for (int i = 0; i < 2; i++) {
            o.af[i] = *reinterpret_cast<const v4i *>(sp + fa + i * 32 * ROWB);
            o.bf[i] = *reinterpret_cast<const v4i *>(sp + fb + i * 32 * ROWB);
        }
    };
    // Scale operands: lane (r, h = 0) holds K term 0 = d of its row (A) /
    // column (B); every other K term is zero.  Kept across blocks, so only
    // the first word of each is rewritten per block (the zero words stay in
    // their registers).
    v2i asv[2] = {}, bsv[2] = {};
    // One block on the wave's 2×2 tiles.  Tile t's MFMAs are issued before
    // tile t-1's rescale, so the matrix cores work while the VALU converts.
    // wa / wb: the scale words of the block pair (blocks 2p, 2p + 1), hi =
    // the pair's second block
    auto block = [&](const Ops &o, const uint32_t (&wa)[2], const uint32_t (&wb)[2], bool hi) {
        h4 as[2], bs[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            asv[i][0] = (int)(hi ? wa[i] >> 16 : wa[i] & 0xffffu);
            bsv[i][0] = (int)(hi ? wb[i] >> 16 : wb[i] & 0xffffu);
            as[i] = __builtin_bit_cast(h4, asv[i]);
            bs[i] = __builtin_bit_cast(h4, bsv[i]);
        }
        v16i d[2];
        f32x16 sc[2];
        const v16i zero = {};
        const f32x16 fzero = {};
#pragma unroll
        for (int t = 0; t <= 4; t++) {
            if (t < 4) {
                const int i = t >> 1, j = t & 1;
                d[t & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(o.af[i], o.bf[j], zero, 0, 0, 0);
                sc[t & 1] = __builtin_amdgcn_mfma_f32_32x32x8f16(as[i], bs[j], fzero, 0, 0, 0);
            }
            if (t > 0) {
                const int u = t - 1, i = u >> 1, j = u & 1;
#pragma unroll
                for (int q = 0; q < 16; q++)
                    acc[i][j][q] = __builtin_fmaf((float)d[u & 1][q], sc[u & 1][q], acc[i][j][q]);
            }
        }
    };
    auto step = [&](int s) {
        if (s + 1 < n_stages) load(s + 1);
        const Stage &S = stages[s & 1];
        // the next block's LDS operands load while this block computes
        // (two blocks per iteration, so both operand sets keep fixed registers)
        Ops o0, o1;
        ld_ops(S, 0, o0);
        ld_scales(S);
#pragma unroll 1
        for (int bp = 0; bp < KB; bp += 2) {
            ld_ops(S, bp + 1, o1);
            asm volatile("" ::: "memory");  // keeps the reads above the block's MFMAs
            uint32_t wa[2], wb[2];
#pragma unroll
            for (int i = 0; i < 2; i++) {
                wa[i] = sa[i], sa[i] = sa2[i];  // the next pair's word moves up
                wb[i] = sb[i], sb[i] = sb2[i];
            }
            block(o0, wa, wb, false);
            ld_ops(S, min(bp + 2, KB - 1), o0);
            asm volatile("" ::: "memory");
            block(o1, wa, wb, true);
        }
        if (s + 1 < n_stages) store(s + 1);
        __syncthreads();
    };
    for (int s = 0; s < n_stages; s++) step(s);

    float *dst = static_cast<float *>(out_) + (size_t)z * m * n;
    uint16_t *dsth = static_cast<uint16_t *>(out_);
    if (TAIL && tail_slot >= 0) {  // a K-part of a tail tile: tile-local rows of 128
        float *tp = ts.part + ((size_t)tail_slot * ts.st + z) * (BM * BN);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int q = 0; q < 16; q++)
                    tp[(wm * 64 + i * 32 + 8 * (q / 4) + 4 * h + (q % 4)) * BN + wn * 64 + j * 32 +
                       r] = acc[i][j][q] * kUnscale;
        return;
    }
    auto put = [&](bool whole) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int col = n0 + wn * 64 + j * 32 + r;
                if (!whole && col >= n) continue;
#pragma unroll
                for (int q = 0; q < 16; q++) {
                    const int row = m0 + wm * 64 + i * 32 + 8 * (q / 4) + 4 * h + (q % 4);
                    if (whole || row < m) {
                        const float v = acc[i][j][q] * kUnscale;
                        if (HOUT)
                            dsth[(size_t)row * n + col] = f32_to_f16_bits(v);
                        else
                            dst[(size_t)row * n + col] = v;
                    }
                }
            }
    };
    if (m0 + BM <= m && n0 + BN <= n)
        put(true);
    else
        put(false);
}

__global__ void splitk_reduce_kernel(const float4 *__restrict__ part, float4 *__restrict__ y,
                                     uint64_t n4, int split) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4;
         i += (uint64_t)gridDim.x * blockDim.x) {
        float4 a = part[i];
        for (int s = 1; s < split; s++) {
            const float4 b = part[(uint64_t)s * n4 + i];
            a.x += b.x;
            a.y += b.y;
            a.z += b.z;
            a.w += b.w;
        }
        y[i] = a;
    }
}

// y of the tail tiles: the tail_st parts summed in part order (float4 per
// thread, one 128×128 tile per 16 workgroups of 256 threads).
__global__ __launch_bounds__(256) void mmq_tail_reduce_kernel(TailSplit ts, float *__restrict__ y,
                                                              int n, int mt, int nt) {
    const int tiles = mt * nt, lx = tiles / kXcds - ts.fx;
    const int slot = blockIdx.x / 16;  // tail tile
    const int e = (blockIdx.x % 16) * 256 + threadIdx.x;  // float4 within the tile
    const int x = slot / lx, jl = ts.fx + slot % lx;
    int tm, tn;
    mmq_tile(x, jl, mt, nt, &tm, &tn);
    const float4 *p = reinterpret_cast<const float4 *>(ts.part + (size_t)slot * ts.st * (BM * BN));
    float4 a = p[e];
    for (int zz = 1; zz < ts.st; zz++) {
        const float4 b = p[(size_t)zz * (BM * BN / 4) + e];
        a.x += b.x;
        a.y += b.y;
        a.z += b.z;
        a.w += b.w;
    }
    const int row = e / (BN / 4), c4 = e % (BN / 4);  // whole tiles only
    *reinterpret_cast<float4 *>(y + (size_t)(tm * BM + row) * n + tn * BN + 4 * c4) = a;
}

// Few rows (m <= 32·TM): one workgroup per 32 columns computes all rows, its W
// waves each a contiguous range of K, so that even a narrow matrix has waves
// on every CU and its weights stream once; the waves' sums meet in LDS, in
// wave order.  A step is 4 blocks: each wave loads its 32 columns' 72 bytes
// and its rows' 128 bytes with consecutive lanes on consecutive addresses
// (a lane per row instead touched 32 cache lines per load, and that bounded
// the kernel), one step ahead in registers, and turns them into MFMA operands
// through an LDS tile of its own (no barriers in the loop).  Two steps ahead
// measured slower (M = 37, N = 8192, K = 5376 16.9 -> 17.3 us; M = 64, N =
// 21504 38.6 -> 45.3): once the first load is in, the rescale's VALU ops on
// whole 32-row tiles are the time.
template <int TM, int W, bool HOUT>
__global__ __launch_bounds__(W * 64, 2) void mmq_skinny_kernel(
    const uint8_t *__restrict__ W_, const int8_t *__restrict__ xq, const uint16_t *__restrict__ xs,
    void *__restrict__ out_, int m, int n, int k) {
    constexpr int kABytes = TM * 32 * 128, kBWords = 32 * 18;
    constexpr int kWaveBytes = kABytes + kBWords * 4;
    constexpr int kRedBytes = TM * 16 * 64 * 4;
    __shared__ __align__(16) uint8_t lds[W * (kWaveBytes > kRedBytes ? kWaveBytes : kRedBytes)];
    const int nb = k / 32, ns = (nb + KB - 1) / KB;  // nb is even
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int n0 = blockIdx.x * 32;
    const int s0 = (int)((long)ns * wave / W), s1 = (int)((long)ns * (wave + 1) / W);
    uint8_t *la = lds + wave * kWaveBytes;
    uint32_t *lb = reinterpret_cast<uint32_t *>(la + kABytes);

    // load offsets from the step's first block; a K of 64 (one step with one
    // live pair) reads the live bytes again in place of the dead ones
    const int live_blocks = min(nb, KB);
    uint32_t ob[9], oa[4 * TM], od[TM];
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int d = i * 64 + lane, col = d / 18, e = min(d % 18, live_blocks * 9 / 2 - 1);
        ob[i] = (uint32_t)min(col, n - 1 - n0) * (uint32_t)nb * 18 + 4 * e;
    }
#pragma unroll
    for (int i = 0; i < 4 * TM; i++)
        oa[i] = (uint32_t)min(8 * i + (lane >> 3), m - 1) * (uint32_t)k +
                16 * min(lane & 7, 2 * live_blocks - 1);
#pragma unroll
    for (int i = 0; i < TM; i++) od[i] = (uint32_t)min(32 * i + r, m - 1) * (uint32_t)nb * 2;
    const uint32_t od2 = nb < KB ? 0 : 4;
    // LDS: activation chunk c (16 bytes) of row x at slot c ^ (x % 8), so the
    // operand reads of 8 lanes fall on distinct banks; weights as loaded
    uint8_t *wa = la + ((lane & ~7) + ((lane & 7) ^ (lane >> 3))) * 16;
    const uint8_t *ra = la + r * 128;
    const uint32_t rx = (uint32_t)(h ^ (r & 7)) * 16;
    const uint32_t *rb = lb + r * 18;

    v4i ga[4 * TM];
    uint32_t gb[9];
    uint2 gs[TM];
    // a K end with two blocks: the last step starts two blocks early and the
    // pair it repeats has zero scales (K of 64: the second pair)
    const bool short_end = nb % KB != 0;
    const int dead = nb < KB ? 1 : 0;
    auto load = [&](int st) {
        const int b0 = short_end && !dead && st + 1 == ns ? nb - KB : st * KB;
        gptr a = (gptr)xq + (size_t)b0 * 32, d = (gptr)xs + (size_t)b0 * 2;
        gptr w = (gptr)W_ + ((size_t)n0 * nb + b0) * 18;
        asm volatile("" : "+s"(a), "+s"(w), "+s"(d));
#pragma unroll
        for (int i = 0; i < 9; i++) {
            uint32_t o = ob[i];
            asm volatile("" : "+v"(o));
            gb[i] = *(const __attribute__((address_space(1))) uint32_t *)(w + o);
        }
#pragma unroll
        for (int i = 0; i < 4 * TM; i++) {
            uint32_t o = oa[i];
            asm volatile("" : "+v"(o));
            ga[i] = *(const __attribute__((address_space(1))) v4i *)(a + o);
        }
#pragma unroll
        for (int i = 0; i < TM; i++) {
            uint32_t o = od[i];
            asm volatile("" : "+v"(o));
            gs[i] = make_uint2(*(const __attribute__((address_space(1))) u32a2 *)(d + o),
                               *(const __attribute__((address_space(1))) u32a2 *)(d + o + od2));
        }
    };
    f32x16 acc[TM];
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int q = 0; q < 16; q++) acc[i][q] = 0.f;
    const uint32_t sh = h ? 0 : 4;           // this half's nibbles to the bytes' high halves
    const uint32_t live = h ? 0u : 0xffffu;  // the scale MFMA's one live K term (h = 0)
    if (s0 < s1) load(s0);
#pragma unroll 1
    for (int st = s0; st < s1; st++) {
        const bool cut = short_end && st + 1 == ns;
#pragma unroll
        for (int i = 0; i < 4 * TM; i++) *reinterpret_cast<v4i *>(wa + i * 1024) = ga[i];
#pragma unroll
        for (int i = 0; i < 9; i++) lb[i * 64 + lane] = gb[i];
        // the wave's other lanes read these: ordered for the compiler (LDS
        // operations of one wave complete in order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        uint32_t sa[TM][2];
#pragma unroll
        for (int i = 0; i < TM; i++) {
            sa[i][0] = cut && !dead ? 0u : gs[i].x;
            sa[i][1] = cut && dead ? 0u : gs[i].y;
        }
        if (st + 1 < s1) load(st + 1);
#pragma unroll
        for (int p = 0; p < 2; p++) {
            uint32_t w[9];
#pragma unroll
            for (int e = 0; e < 9; e++) w[e] = rb[9 * p + e];
            const uint32_t lw = cut && p == dead ? 0u : live;
#pragma unroll
            for (int blk = 0; blk < 2; blk++) {
                v4i bf;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint32_t q = blk ? w[5 + e] : __builtin_amdgcn_alignbyte(w[e + 1], w[e], 2);
                    bf[e] = (int)(((q << sh) & 0xF0F0F0F0u) ^ 0x80808080u);
                }
                const h4 bs = __builtin_bit_cast(h4, v2i{(int)((blk ? w[4] >> 16 : w[0]) & lw), 0});
#pragma unroll
                for (int i = 0; i < TM; i++) {
                    const v4i af = *reinterpret_cast<const v4i *>(
                        ra + i * 4096 + (rx ^ (32u * (2 * p + blk))));
                    const h4 as = __builtin_bit_cast(
                        h4, v2i{(int)((blk ? sa[i][p] >> 16 : sa[i][p]) & live), 0});
                    const v16i d = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, v16i{}, 0, 0, 0);
                    const f32x16 sc = __builtin_amdgcn_mfma_f32_32x32x8f16(as, bs, f32x16{}, 0, 0, 0);
#pragma unroll
                    for (int q = 0; q < 16; q++)
                        acc[i][q] = __builtin_fmaf((float)d[q], sc[q], acc[i][q]);
                }
            }
        }
        // this step's reads before the next step's stores
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();  // every wave is done with its tile
    float(*red)[TM * 16 * 64] = reinterpret_cast<float(*)[TM * 16 * 64]>(lds);
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int q = 0; q < 16; q++) red[wave][(i * 16 + q) * 64 + lane] = acc[i][q];
    __syncthreads();
    // element e of the workgroup's rows: (row tile, q, lane)
    for (int e = threadIdx.x; e < TM * 1024; e += W * 64) {
        float v = red[0][e];
#pragma unroll
        for (int z = 1; z < W; z++) v += red[z][e];
        v *= kUnscale;
        const int l = e & 63, q = (e >> 6) & 15, i = e >> 10;
        const int row = 32 * i + 8 * (q / 4) + 4 * (l >> 5) + (q % 4), col = n0 + (l & 31);
        if (row < m && col < n) {
            if (HOUT)
                static_cast<uint16_t *>(out_)[(size_t)row * n + col] = f32_to_f16_bits(v);
            else
                static_cast<float *>(out_)[(size_t)row * n + col] = v;
        }
    }
}

}  // namespace

namespace {
template <int TM, int W, bool HOUT>
void skinny_launch(hipStream_t st, const void *w, const int8_t *xq, const uint16_t *xs, void *y,
                   uint32_t m, uint32_t n, uint32_t k) {
    hipLaunchKernelGGL((mmq_skinny_kernel<TM, W, HOUT>), dim3((n + 31) / 32), dim3(W * 64), 0, st,
                       static_cast<const uint8_t *>(w), xq, xs, y, (int)m, (int)n, (int)k);
}

// The few-rows kernel against the tiles, whose launch of one round costs the
// same for 1 row as for 128 (81 us at K = 5376; 310 at K = 21504, or 69 split
// over K 8 ways).  us at N = 21504, K = 5376 / N = 5376, K = 21504, tiles at
// split 1 81 / 310: M = 1 21 / 26, 37 35 / 43, 64 38 / 48, 100 77 / 87.  Its
// time grows with n by 1.0 / 1.8 / 3.6 us per 1000 columns (M <= 32 / 64 /
// 128, K = 5376) where the tiles' stays until their round of 65536 columns is
// full, hence the limits on n; above 64 rows a caller's split over K is the
// faster of the two.  Above 96 rows 16384 columns are one round of the few-rows
// workgroups, and the second costs more than the tiles' (128 rows, N = 21504,
// tiles / few rows: K = 512 12.3 / 16.4, 21504 312 / 375; N = 16384 12.2 / 11.6,
// 312 / 175).  A K of a few blocks leaves most of the waves that cut it idle (K =
// 64, N = 21504: 65 rows 6.7 / 9.4, 128 rows 7.5 / 13.0; from K = 512 on it pays).
bool skinny(uint32_t m, uint32_t n, uint32_t k, uint32_t split_k) {
    if (m <= 32) return true;
    if (k < 256 && n > 8192) return false;
    if (m <= 64) return n <= 43008;
    return m <= 128 && n <= (m <= 96 ? 21504 : 16384) && split_k == 1;
}

template <bool HOUT>
int gemm_t(hipStream_t st, const void *w, const int8_t *xq, const uint16_t *xs, void *y,
           uint32_t m, uint32_t n, uint32_t k, uint32_t split_k, float *partials) {
    SGQ_CHECK(k % 64 == 0 && k > 0, "gemm_q4_0_q8: k=%u must be a positive multiple of 64", k);
    SGQ_CHECK(m > 0 && n > 0, "gemm_q4_0_q8: empty shape");
    SGQ_CHECK(split_k == 1 || split_k == 2 || split_k == 4 || split_k == 8,
              "gemm_q4_0_q8: split_k=%u not in {1,2,4,8}", split_k);
    SGQ_CHECK(split_k == 1 || partials != nullptr, "gemm_q4_0_q8: split_k>1 needs partials");
    SGQ_CHECK(!HOUT || split_k == 1, "gemm_q4_0_q8: f16 output is not built with split-K");
    SGQ_CHECK(k % 16 == 0 && ((uintptr_t)xq & 15) == 0, "gemm_q4_0_q8: xq must be 16-byte aligned");
    SGQ_CHECK(((uintptr_t)w & 3) == 0, "gemm_q4_0_q8: weights must be 4-byte aligned");
    SGQ_CHECK((uint64_t)m * n < (1ull << 31) * 4, "gemm_q4_0_q8: output too large");
    SGQ_CHECK(split_k == 1 || (m * (uint64_t)n) % 4 == 0, "gemm_q4_0_q8: m*n must be a multiple of 4 for split-K");
    if (k < kWideK && skinny(m, n, k, split_k)) {
        // W: 8 waves cut a column tile's K finer (N = 5376, K = 21504, M = 37:
        // 43 against 69 us); with two tiles or more per CU, 4 leave smaller
        // workgroups to even out over the CUs (N = 21504, M = 37: 35 against 45)
        const bool w4 = n >= 16384;
        const int tm = (int)(m + 31) / 32;
#define SGQ_SKINNY(TM)                                                          \
    (w4 ? skinny_launch<TM, 4, HOUT>(st, w, xq, xs, y, m, n, k)                  \
        : skinny_launch<TM, 8, HOUT>(st, w, xq, xs, y, m, n, k))
        if (tm == 1)
            SGQ_SKINNY(1);
        else if (tm == 2)
            SGQ_SKINNY(2);
        else if (tm == 3)
            SGQ_SKINNY(3);
        else
            SGQ_SKINNY(4);
#undef SGQ_SKINNY
        SGQ_HIP(hipGetLastError());
        return SGQ_OK;
    }
    static bool attr = false;
    const size_t lds = 2 * sizeof(Stage);
    if (!attr) {
        SGQ_HIP(hipFuncSetAttribute((const void *)mmq_kernel<HOUT>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        SGQ_HIP(hipFuncSetAttribute((const void *)mmq_kernel<HOUT, false, uint64_t>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        SGQ_HIP(hipFuncSetAttribute((const void *)mmq_kernel<false, true>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        attr = true;
    }
    const int mt = (int)((m + BM - 1) / BM), nt = (int)((n + BN - 1) / BN);
    void *dst = split_k == 1 ? y : static_cast<void *>(partials);
    // Tail split: fp32 output in whole column tiles, split_k = 1 and a
    // partials buffer (m·n floats suffice when m is whole tiles; the parts are
    // at most one round of tiles)
    TailSplit ts{0, 0, partials};
    const int tiles = mt * nt, slots_x = device_info().cus * SGQ_MMQ_WG_PER_CU / kXcds;
    // (only below two whole rounds: at M = 4096, N = 21504, with a tail of
    // half a round split in 2, the launch measured 1.3% slower)
    if (m % BM == 0 && n % BN == 0 && k < kWideK && !HOUT && split_k == 1 && partials != nullptr && tiles % kXcds == 0 &&
        slots_x > 0 && tiles / kXcds > slots_x && tiles / kXcds < 2 * slots_x) {
        const int tx = tiles / kXcds, fx = tx / slots_x * slots_x, lx = tx - fx;
        const int parts = lx > 0 ? std::min(4, slots_x / lx) : 0;
        if (parts >= 2 && (int)(k / 32) / parts >= 4 * KB) ts.fx = fx, ts.st = parts;
    }
    const int grid_x = ts.st ? kXcds * (ts.fx + (tiles / kXcds - ts.fx) * ts.st) : tiles;
    if (ts.st)
        hipLaunchKernelGGL((mmq_kernel<false, true>), dim3(grid_x, split_k), dim3(kMWG), lds, st,
                           static_cast<const uint8_t *>(w), xq, xs, dst, (int)m, (int)n, (int)k, mt,
                           nt, (int)split_k, ts);
    else if (k >= kWideK)
        hipLaunchKernelGGL((mmq_kernel<HOUT, false, uint64_t>), dim3(grid_x, split_k), dim3(kMWG),
                           lds, st, static_cast<const uint8_t *>(w), xq, xs, dst, (int)m, (int)n,
                           (int)k, mt, nt, (int)split_k, ts);
    else
        hipLaunchKernelGGL((mmq_kernel<HOUT>), dim3(grid_x, split_k), dim3(kMWG), lds, st,
                           static_cast<const uint8_t *>(w), xq, xs, dst, (int)m, (int)n, (int)k, mt,
                           nt, (int)split_k, ts);
    SGQ_HIP(hipGetLastError());
    if (ts.st) {
        const int tail_tiles = kXcds * (tiles / kXcds - ts.fx);
        hipLaunchKernelGGL(mmq_tail_reduce_kernel, dim3(tail_tiles * 16), dim3(256), 0, st, ts,
                           static_cast<float *>(y), (int)n, mt, nt);
        SGQ_HIP(hipGetLastError());
    }
    if (split_k > 1) {
        const uint64_t n4 = (uint64_t)m * n / 4;
        uint64_t g = (n4 + 255) / 256;
        if (g > (uint64_t)device_info().cus * 8) g = (uint64_t)device_info().cus * 8;
        hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)g), dim3(256), 0, st,
                           reinterpret_cast<const float4 *>(partials),
                           static_cast<float4 *>(y), n4, (int)split_k);
        SGQ_HIP(hipGetLastError());
    }
    return SGQ_OK;
}

}  // namespace

int launch_gemm_q4_0_q8(hipStream_t st, const void *w, const int8_t *xq, const uint16_t *xs,
                        float *y, uint32_t m, uint32_t n, uint32_t k, uint32_t split_k,
                        float *partials) {
    return gemm_t<false>(st, w, xq, xs, y, m, n, k, split_k, partials);
}
int launch_gemm_q4_0_q8(hipStream_t st, const void *w, const int8_t *xq, const uint16_t *xs,
                        uint16_t *y, uint32_t m, uint32_t n, uint32_t k) {
    return gemm_t<true>(st, w, xq, xs, y, m, n, k, 1, nullptr);
}

}  // namespace sgq
