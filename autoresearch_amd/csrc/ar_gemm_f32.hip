// ar_gemm_f32.hip -- the fp32 products (linear_fwd, linear_bwd_dx,
// linear_bwd_dw of ops.mojo:110-203, 870-950, 953-1033 and the fp32 Muon
// products, optimizer.mojo:288-336) on the bf16 matrix cores, at fp32 accuracy.
//
// Each operand value is split exactly into three bf16 terms (ar_split.hpp) and
// the product is the sum of the six terms down to 2^-18 of the leading one,
// accumulated in fp32: hi hi in one accumulator, the smaller terms in another.
// Six v_mfma_f32_32x32x16_bf16 do 16 k-values in 192 cycles where eight
// v_mfma_f32_32x32x2_f32 take 512, and round the sum once instead of eight
// times: norm-wise error against fp64 1.3e-7 at 512^3 (N(0, 1) operands) where
// the fp32 instruction gave 4.1e-7.
//
// The split is exact for zero and for magnitudes from 2^-110 to 3.39e38; what
// lies outside is formed on the fp32 matrix cores (fp32_block), per block:
//   * an infinity or NaN, or a finite value that bf16 rounds to infinity, makes
//     every output it touches non-finite, which the block sees;
//   * a value below 2^-110 (7.7e-34) loses up to 2^-134 (half of bf16's least
//     magnitude), so a sum of R products moves by at most R 2^-134 (max|a| +
//     max|b|).  With both maxima at 2^24 or less and R at 2^25 or less that is
//     2^-24 of any output of 2^-60 or more.  A block with a smaller output that
//     no row of zeros explains, or with a larger operand, looks for such values
//     and is formed again where it holds one.
// Muon meets them: the momentum of a row without gradient decays into the
// subnormals and stays there.  One step of a 2048 x 512 matrix with 2 % of rows
// at 1e-36 takes 291 us where an ordinary one takes 214 (484 with a second pass
// of unstaged scalar loads by one wave group, wherever such a row is staged).
//
// Layout of a product (GEMM space): C[m, n] (+)= sum_r A(m, r) B(n, r), each
// operand K-major (r contiguous) or MN-major (m / n contiguous).
#include "ar_internal.hpp"
#include "ar_split.hpp"

#include <math.h>

#include <type_traits>

namespace ar {
namespace {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
// 4-byte aligned 16-byte vector: odd row strides load with the same instruction
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Block tile BM x BN of NWM x NWN waves, times KG groups of waves that share
// the reduction: group g takes KS of the 16-deep k-steps of every staged
// k-tile (BK = 16 KS KG), and the groups' sums are added through LDS at the
// end.  Two LDS stages.
template <int BM_, int BN_, int NWM_, int NWN_, int KG_, int KS_>
struct X3Tile {
    static constexpr int BM = BM_, BN = BN_, NWM = NWM_, NWN = NWN_, KG = KG_, KS = KS_;
    static constexpr int THREADS = 64 * NWM * NWN * KG, BK = 16 * KS * KG;
    static constexpr int WM = BM / NWM, WN = BN / NWN, TM = WM / 32, TN = WN / 32;
    static constexpr int PA = BM * BK * 2, PB = BN * BK * 2;  // bytes of one plane
    static constexpr int STAGE = 3 * (PA + PB);
    static constexpr int RED = KG > 1 ? KG * BM * BN * 4 : 0;
    static constexpr int LDS = 2 * STAGE > RED ? 2 * STAGE : RED;
};

struct X3Args {
    float* C;
    const float *A, *B;
    int64_t M, N, K;
    int64_t lda, ldb, ldc;
    int64_t kps;
    int splits;        // reduction per split (a multiple of BK), split count
    float* partial;    // splits > 1: fp32 partials [batch][split][M][N]
    const float* aux;  // C = alpha acc + beta aux (null: C = acc); may be C itself
    float alpha, beta;
    int64_t sA, sB, sC;  // batch strides
    int batch;
};

// Chunk swizzle of a staged MN-major tile [k][ROWS]: the four k-rows one
// transpose read touches (64 bytes of each) fall into different quarters of the banks.
template <int ROWS>
__device__ __forceinline__ int mnswz(int k) {
    return ROWS >= 128 ? 4 * (k & 3) : ROWS == 64 ? 4 * ((k >> 1) & 1) : 0;
}

// v[0..7] = v[s..7], then whatever was there (s < 8): a conditional move per
// value and bit of s.
__device__ __forceinline__ void shift8(float (&v)[8], int s) {
    const float a0 = v[0], a1 = v[1], a2 = v[2], a3 = v[3], a4 = v[4], a5 = v[5], a6 = v[6], a7 = v[7];
    const bool p = s & 4, q = s & 2, r = s & 1;
    const float b0 = p ? a4 : a0, b1 = p ? a5 : a1, b2 = p ? a6 : a2, b3 = p ? a7 : a3;
    const float c0 = q ? b2 : b0, c1 = q ? b3 : b1, c2 = q ? a4 : b2, c3 = q ? a5 : b3, c4 = q ? a6 : a4,
                c5 = q ? a7 : a5;
    v[0] = r ? c1 : c0;
    v[1] = r ? c2 : c1;
    v[2] = r ? c3 : c2;
    v[3] = r ? c4 : c3;
    v[4] = r ? c5 : c4;
    v[5] = r ? a6 : c5;
    v[6] = r ? a7 : a6;
}

// One operand's staging: thread items of 8 values (8 consecutive k of a row,
// or 8 consecutive rows of a k), loaded a k-tile ahead with two 16-byte loads
// (4-byte alignment is enough for them) from a wave-uniform base plus a
// per-lane offset fixed for the whole kernel, then split and written.  Rows
// past the extent repeat valid ones; their outputs are not stored.
// EDGE adds sizes that are no multiple of 8:
//   an item that would pass the end of an MN-major operand's rows (SHIFT) or of
//   the reduction (the last, partial k-tile) loads the last 8 values before it
//   and write() shifts them down; the A operand's values past the reduction's
//   end are zeroed, which zeroes their products.  MN-major extents, and the
//   reduction where an operand is K-major, are at least 8.
template <bool KMAJ, int ROWS, int BK, int THREADS, bool EDGE>
struct X3Load {
    static constexpr int ITEMS = ROWS * BK / 8, NP = ITEMS / THREADS;
    static_assert(ITEMS % THREADS == 0 && NP >= 1, "whole items per thread");
    static constexpr int U = BK / 8, PLANE = ROWS * BK * 2, C8 = ROWS / 8;
    using Off = std::conditional_t<EDGE, int64_t, unsigned>;
    float v[NP][8];
    Off off[NP];  // byte offset of each item from the block's first value of a k-tile
    float mx[KMAJ ? NP : 8];  // largest magnitude seen of each stored row this thread stages
    const float* base;
    int64_t ld;
    int rows;  // valid rows of this block

    __device__ __forceinline__ static int item(int p) { return p * THREADS + (int)threadIdx.x; }
    // item p's first k-value within the tile
    __device__ __forceinline__ static int item_k(int p) { return KMAJ ? (item(p) % U) * 8 : item(p) / C8; }
    __device__ __forceinline__ void init(const float* g, int64_t ld_, int64_t row0, int64_t extent, int64_t kbeg) {
        ld = ld_;
        rows = extent - row0 < ROWS ? (int)(extent - row0) : ROWS;
        base = g + (KMAJ ? row0 * ld + kbeg : kbeg * ld + row0);
        static_assert(KMAJ || THREADS % C8 == 0, "a thread's items hold the same rows");
#pragma unroll
        for (float& m : mx) m = 0.f;
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            if constexpr (KMAJ) {
                int r = item(p) / U;
                r = r < rows ? r : rows - 1;
                off[p] = (Off)((Off)r * (Off)ld + (Off)item_k(p)) * 4;
            } else {
                int r = (item(p) % C8) * 8;
                r = r + 8 <= rows ? r : rows - 8;  // (EDGE: may be below 0, still inside the stored row)
                off[p] = (Off)((Off)item_k(p) * (Off)ld + (Off)r) * 4;
            }
        }
    }
    __device__ __forceinline__ bool large() const {
        float m = 0.f;
#pragma unroll
        for (const float x : mx) m = fmaxf(m, x);
        return m > 0x1p24f;
    }
    // folds mx into the block's largest magnitude of each row (bit patterns)
    __device__ __forceinline__ void row_max(unsigned* most) const {
#pragma unroll
        for (int i = 0; i < (KMAJ ? NP : 8); ++i)
            atomicMax(most + (KMAJ ? item(i) / U : (item(0) % C8) * 8 + i), __float_as_uint(mx[i]));
    }
    // the ragged end of the rows lies in this block
    __device__ __forceinline__ bool ragged() const { return !KMAJ && (rows & 7) != 0; }
    // How far past the reduction's end item p reaches (left: k-values from the
    // tile's first to the end).
    __device__ __forceinline__ static int over_k(int p, int left) {
        const int o = item_k(p) + (KMAJ ? 8 : 1) - left;
        return o > 0 ? o : 0;
    }
    // k0: first k-value of the tile, relative to the split's first
    template <bool TAIL>
    __device__ __forceinline__ void load(int64_t k0, int left) {
        const char* const s = reinterpret_cast<const char*>(base + (KMAJ ? k0 : k0 * ld));
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const char* q = s + off[p];
            if constexpr (TAIL) q -= (KMAJ ? (int64_t)over_k(p, left) : over_k(p, left) * ld) * 4;
            const f32x4u a = *reinterpret_cast<const f32x4u*>(q), b = *reinterpret_cast<const f32x4u*>(q + 16);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                v[p][e] = a[e];
                v[p][4 + e] = b[e];
            }
        }
    }
    __device__ __forceinline__ void zero_past(int left) {
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (item_k(p) + (KMAJ ? e : 0) >= left) v[p][e] = 0.f;
    }
    // undo the moves of SHIFT blocks and of a TAIL load (8 and more: nothing valid left)
    template <bool SHIFT, bool TAIL>
    __device__ __forceinline__ void unshift(int left) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            if constexpr (KMAJ && TAIL) shift8(v[p], over_k(p, left) & 7);
            if constexpr (!KMAJ && SHIFT) {
                const int s = (item(p) % C8) * 8 + 8 - rows;
                shift8(v[p], s > 0 ? s & 7 : 0);
            }
        }
    }
    __device__ __forceinline__ void write(unsigned char* st) {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            const int it = item(p);
            int o;
            if constexpr (KMAJ) {
                o = kslot<U>(it / U, it % U) * 16;
            } else {
                const int k = it / C8, c = it % C8;
                o = (k * ROWS + ((c ^ mnswz<ROWS>(k)) << 3)) * 2;
            }
            bf16x8 hi, mid, lo;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const float x0 = v[p][e], x1 = v[p][e + 1];
                if constexpr (KMAJ) {
                    mx[p] = fmaxf(fmaxf(fabsf(x0), fabsf(x1)), mx[p]);
                } else {
                    mx[e] = fmaxf(mx[e], fabsf(x0));
                    mx[e + 1] = fmaxf(mx[e + 1], fabsf(x1));
                }
                split2(x0, x1, e, hi, mid, lo);
            }
            *reinterpret_cast<bf16x8*>(st + o) = hi;
            *reinterpret_cast<bf16x8*>(st + PLANE + o) = mid;
            *reinterpret_cast<bf16x8*>(st + 2 * PLANE + o) = lo;
        }
    }
};

// MFMA fragment: 32 rows from r0, the 16 k-values from 16 ks (lane: row
// r0 + lane % 32, k 8 (lane / 32) + 0..7).
template <bool KMAJ, int ROWS, int BK>
__device__ __forceinline__ bf16x8 x3frag(const unsigned char* plane, int r0, int ks, int lane) {
    if constexpr (KMAJ) {
        return *reinterpret_cast<const bf16x8*>(plane + kslot<BK / 8>(r0 + (lane & 31), 2 * ks + (lane >> 5)) * 16);
    } else {
        // two transpose reads: inside each 16-lane group, lane 4 k + q supplies
        // the address of k-row k, columns 4 q .. 4 q + 3, and lane i receives
        // k-rows 0..3 of column i
        const bf16* t = reinterpret_cast<const bf16*>(plane);
        const int g = lane >> 4, src = lane & 15;
        const int k = 16 * ks + 8 * (g >> 1) + (src >> 2);
        const int col = r0 + 16 * (g & 1) + 4 * (src & 3);
        const int co = (((col >> 3) ^ mnswz<ROWS>(k)) << 3) + (col & 7);  // k and k + 4 share the swizzle
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t + k * ROWS + co));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t + (k + 4) * ROWS + co));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
}

__device__ __forceinline__ int acc_row(int v, int lane) { return (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3); }

constexpr unsigned kTinyBits = 0x08800000u;  // 2^-110

// Whether the block's part of an operand (rows x [kbeg, kend)) holds a value
// below 2^-110 that is not zero.
template <bool KMAJ, int ROWS, int THREADS>
__device__ __forceinline__ bool holds_tiny(const float* g, int64_t ld, int64_t row0, int64_t extent, int64_t kbeg,
                                           int64_t kend) {
    constexpr int W = KMAJ || ROWS >= kWave ? kWave : ROWS;  // lanes along what is contiguous
    const int64_t rows = extent - row0 < ROWS ? extent - row0 : ROWS;
    const int64_t outer = KMAJ ? rows : kend - kbeg, inner = KMAJ ? kend - kbeg : rows;
    const float* const s = g + (KMAJ ? row0 * ld + kbeg : kbeg * ld + row0);
    const int tid = threadIdx.x;
    unsigned least = ~0u;
    auto see = [&](float x) __attribute__((always_inline)) {
        const unsigned u = __float_as_uint(x) * 2u - 1u;  // zero of either sign wraps to the top
        least = u < least ? u : least;
    };
#pragma unroll 4
    for (int64_t o = tid / W; o < outer; o += THREADS / W) {
        const float* const q = s + o * ld;
        if constexpr (KMAJ) {
#pragma unroll 8
            for (int64_t i = tid % W; i < inner; i += W) see(q[i]);
        } else {
#pragma unroll
            for (int i = tid % W; i < ROWS; i += W)
                if (i < inner) see(q[i]);
        }
    }
    return least < kTinyBits * 2u - 1u;
}

// Eight values of an operand fragment of fp32_block: row r, k-values k .. k + 7
// (TAIL: those at or past kend are zero).
template <bool KMAJ, bool TAIL>
__device__ __forceinline__ void x8(float (&v)[8], const float* g, int64_t ld, int64_t r, int64_t k, int64_t kend) {
    if constexpr (KMAJ && !TAIL) {
        const f32x4u a = *reinterpret_cast<const f32x4u*>(g + r * ld + k), b = *reinterpret_cast<const f32x4u*>(g + r * ld + k + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int64_t kk = TAIL && k + e >= kend ? kend - 1 : k + e;
            const float x = KMAJ ? g[r * ld + kk] : g[kk * ld + r];
            v[e] = TAIL && k + e >= kend ? 0.f : x;
        }
    }
}

// A wave's block on the fp32 matrix cores, straight from memory: every kg-th of
// KG 16-deep k-steps, each loaded while the one before is multiplied.  Lane half
// h holds k-values 8 h .. 8 h + 7 of a step; instruction e takes value e of both.
template <bool AK, bool BKM, int TM, int TN, int KG>
__device__ __forceinline__ void fp32_block(f32x16 (&acc)[TM][TN], const float* A, const float* B, int64_t lda,
                                           int64_t ldb, int64_t M, int64_t N, int64_t row0, int64_t col0, int64_t kbeg,
                                           int64_t kend, int kg) {
    const int lane = threadIdx.x % kWave, h8 = (lane >> 5) * 8;
    int64_t ra[TM], rb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        ra[i] = row0 + i * 32 + (lane & 31);
        ra[i] = ra[i] < M ? ra[i] : M - 1;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        rb[j] = col0 + j * 32 + (lane & 31);
        rb[j] = rb[j] < N ? rb[j] : N - 1;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
    float a[TM][8], b[TN][8];
    auto load = [&](auto tail_, int64_t k) __attribute__((always_inline)) {
        constexpr bool TAIL = decltype(tail_)::value;
#pragma unroll
        for (int i = 0; i < TM; ++i) x8<AK, TAIL>(a[i], A, lda, ra[i], k + h8, kend);
#pragma unroll
        for (int j = 0; j < TN; ++j) x8<BKM, TAIL>(b[j], B, ldb, rb[j], k + h8, kend);
    };
    auto mul = [&](const float (&x)[TM][8], const float (&y)[TN][8]) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x[i][e], y[j][e], acc[i][j], 0, 0, 0);
    };
    const int64_t whole = (kend - kbeg) / 16, last = kbeg + whole * 16;
    if (kg < whole) {
        load(std::false_type{}, kbeg + kg * 16);
#pragma unroll 1
        for (int64_t s = kg; s < whole; s += KG) {
            float x[TM][8], y[TN][8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
#pragma unroll
                for (int i = 0; i < TM; ++i) x[i][e] = a[i][e];
#pragma unroll
                for (int j = 0; j < TN; ++j) y[j][e] = b[j][e];
            }
            load(std::false_type{}, kbeg + (s + KG < whole ? s + KG : s) * 16);
            mul(x, y);
        }
    }
    if (last < kend && whole % KG == kg) {
        load(std::true_type{}, last);
        mul(a, b);
    }
}

template <bool AK, bool BKM, typename TL, bool EDGE>
__global__ __launch_bounds__(TL::THREADS, 2) void gemm_x3_k(X3Args p) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    constexpr int BM = TL::BM, BN = TL::BN, BK = TL::BK, TM = TL::TM, TN = TL::TN;
    using LA = X3Load<AK, BM, BK, TL::THREADS, EDGE>;
    using LB = X3Load<BKM, BN, BK, TL::THREADS, EDGE>;

    // block -> (batch, split, tile): each XCD (8, dispatched round-robin) owns a
    // contiguous run of row-major tiles, so an A panel stays in one L2
    const int tiles_n = (int)((p.N + BN - 1) / BN), tiles_mn = (int)((p.M + BM - 1) / BM) * tiles_n;
    int id = blockIdx.x;
    const int total = (int)gridDim.x;
    if (total % 8 == 0) id = (id % 8) * (total / 8) + id / 8;
    const int bt = id / (tiles_mn * p.splits);
    id -= bt * tiles_mn * p.splits;
    const int z = id / tiles_mn, t = id - z * tiles_mn;
    int64_t m0 = (int64_t)(t / tiles_n) * BM, n0 = (int64_t)(t % tiles_n) * BN;
    // EDGE: the last block of a ragged extent starts early enough to be whole
    // (where the extent allows it), and stores only its own rows / columns
    int mskip = 0, nskip = 0;
    if constexpr (EDGE) {
        if (!AK && p.M >= BM && m0 + BM > p.M) {
            mskip = (int)(m0 + BM - p.M);
            m0 -= mskip;
        }
        if (!BKM && p.N >= BN && n0 + BN > p.N) {
            nskip = (int)(n0 + BN - p.N);
            n0 -= nskip;
        }
    }
    const float* const A = p.A + bt * p.sA;
    const float* const B = p.B + bt * p.sB;
    const int64_t kbeg = z * p.kps, kend = kbeg + p.kps < p.K ? kbeg + p.kps : p.K;

    const int lane = threadIdx.x % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int kg = wave / (TL::NWM * TL::NWN), wq = wave % (TL::NWM * TL::NWN);
    const int wrow = (wq / TL::NWN) * TL::WM, wcol = (wq % TL::NWN) * TL::WN;

    LA la;
    LB lb;
    // the hi hi products, and the five smaller terms on their own: the large
    // sum is then rounded once per 16 k-values instead of six times
    f32x16 acc[TM][TN], low[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = low[i][j][v] = 0.f;

    auto frags = [&](const unsigned char* st, int s, bf16x8 (&fa)[TM][3], bf16x8 (&fb)[TN][3])
                     __attribute__((always_inline)) {
        const int ks = kg * TL::KS + s;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
            for (int i = 0; i < TM; ++i) fa[i][q] = x3frag<AK, BM, BK>(st + q * TL::PA, wrow + i * 32, ks, lane);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[j][q] = x3frag<BKM, BN, BK>(st + 3 * TL::PA + q * TL::PB, wcol + j * 32, ks, lane);
        }
    };
    auto compute = [&](const unsigned char* st) __attribute__((always_inline)) {
        constexpr int PQ[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
        for (int s = 0; s < TL::KS; ++s) {
            bf16x8 fa[TM][3], fb[TN][3];
            frags(st, s, fa, fb);
            __builtin_amdgcn_sched_barrier(0);  // all reads before the products: no spills
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        f32x16& c = q < 5 ? low[i][j] : acc[i][j];
                        c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][PQ[q][0]], fb[j][PQ[q][1]], c, 0, 0, 0);
                    }
        }
    };

    // this wave's block: rows / columns left, and the first element
    struct Block {
        int64_t ldc, mleft, nleft;
        int mlow, nlow;  // first own row / column
        float* C;
        const float* aux;
        __device__ __forceinline__ bool own(int row, int col) const {
            return row < mleft && col < nleft && (!EDGE || (row >= mlow && col >= nlow));
        }
        __device__ __forceinline__ bool whole() const {
            return mleft >= TL::WM && nleft >= TL::WN && (!EDGE || (mlow <= 0 && nlow <= 0));
        }
    };
    auto block = [&]() __attribute__((always_inline)) {
        const bool part = p.splits > 1;
        const int64_t ldc = part ? p.N : p.ldc, c0 = (m0 + wrow) * ldc + n0 + wcol;
        return Block{ldc, p.M - m0 - wrow, p.N - n0 - wcol, mskip - wrow, nskip - wcol,
                     (part ? p.partial + ((int64_t)bt * p.splits + z) * p.M * p.N : p.C + bt * p.sC) + c0,
                     part || !p.aux ? nullptr : p.aux + bt * p.sC + c0};
    };
    // D: the epilogue operand is on its way while the product forms
    constexpr bool EARLY = TL::KG == 1 && TM * TN == 1;
    f32x16 old;
    if constexpr (EARLY) {
        const Block b = block();
        if (b.aux && b.whole()) {
#pragma unroll
            for (int v = 0; v < 16; ++v) old[v] = b.aux[acc_row(v, lane) * b.ldc + (lane & 31)];
        } else if (b.aux) {
#pragma unroll
            for (int v = 0; v < 16; ++v)
                old[v] = b.own(acc_row(v, lane), lane & 31) ? b.aux[acc_row(v, lane) * b.ldc + (lane & 31)] : 0.f;
        }
    }

    la.init(A, p.lda, m0, p.M, kbeg);
    lb.init(B, p.ldb, n0, p.N, kbeg);
    const int64_t klen = kend - kbeg;
    // n whole k-tiles: tile t is computed from LDS stage t % 2, then tile t + 1
    // (in registers since the tile before) is converted into the other stage and
    // tile t + 2 loaded.  (Past the last tile the loads repeat it.)
    auto tiles = [&](auto shift_, int64_t n) __attribute__((always_inline)) {
        constexpr bool SHIFT = decltype(shift_)::value;
        auto load = [&](int64_t t) __attribute__((always_inline)) {
            const int64_t k0 = (t < n ? t : n - 1) * BK;
            la.template load<false>(k0, BK);
            lb.template load<false>(k0, BK);
        };
        auto write = [&](unsigned char* st) __attribute__((always_inline)) {
            la.template unshift<SHIFT, false>(BK);
            lb.template unshift<SHIFT, false>(BK);
            la.write(st);
            lb.write(st + 3 * TL::PA);
        };
        load(0);
        write(smem_raw);
        load(1);
        __syncthreads();
        int cur = 0;
        for (int64_t t = 0; t < n; ++t, cur ^= 1) {
            compute(smem_raw + cur * TL::STAGE);
            if (t + 1 < n) write(smem_raw + (cur ^ 1) * TL::STAGE);
            load(t + 2);
            __syncthreads();
        }
    };
    if constexpr (!EDGE) {
        tiles(std::false_type{}, klen / BK);
    } else {
        const int64_t n = klen / BK, whole = n * BK;
        if (n > 0) {
            if (la.ragged() || lb.ragged()) tiles(std::true_type{}, n);
            else tiles(std::false_type{}, n);
        }
        if (whole < klen) {
            const int left = (int)(klen - whole);
            la.template load<true>(whole, left);
            lb.template load<true>(whole, left);
            la.template unshift<true, true>(left);
            lb.template unshift<true, true>(left);
            la.zero_past(left);
            la.write(smem_raw);
            lb.write(smem_raw + 3 * TL::PA);
            __syncthreads();
            compute(smem_raw);
            __syncthreads();
        }
    }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] += low[i][j][v];
    const Block blk = block();
    const int64_t ldc = blk.ldc;
    float* const C = blk.C;
    const float* const aux = blk.aux;
    auto own = [&](int row, int col) __attribute__((always_inline)) { return blk.own(row, col); };

    // Where groups share the reduction, each leaves its sums in LDS and then
    // adds, in group order, 1 / KG of the block: values of 32 x 32 sub-block
    // s / 16, row group s % 16.
    constexpr int NV = TM * TN * 16, PER = NV / TL::KG;
    static_assert(NV % TL::KG == 0, "whole values per group");
    float x[TL::KG > 1 ? PER : 1];
    auto merge = [&]() __attribute__((always_inline)) {
        if constexpr (TL::KG > 1) {
            float* const red = reinterpret_cast<float*>(smem_raw) + wq * TL::WM * TL::WN + lane;
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) red[kg * BM * BN + ((i * TN + j) * 16 + v) * kWave] = acc[i][j][v];
            __syncthreads();
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                x[u] = red[(kg * PER + u) * kWave];
#pragma unroll
                for (int g = 1; g < TL::KG; ++g) x[u] += red[g * BM * BN + (kg * PER + u) * kWave];
            }
        }
    };
    // f(value, row, column within the wave's block) of this thread's outputs
    auto each = [&](auto f) __attribute__((always_inline)) {
        if constexpr (TL::KG > 1) {
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const int s = kg * PER + u, ij = s / 16;
                f(x[u], (ij / TN) * 32 + acc_row(s % 16, lane), (ij % TN) * 32 + (lane & 31));
            }
        } else {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) f(acc[i][j][v], i * 32 + acc_row(v, lane), j * 32 + (lane & 31));
        }
    };
    [[maybe_unused]] auto store = [&]() __attribute__((always_inline)) {
        // every epilogue operand is read before the first store (C may be aux)
        if (aux) {
            float y[PER];
            int n = 0;
            each([&](float, int row, int col) __attribute__((always_inline)) {
                y[n++] = own(row, col) ? aux[row * ldc + col] : 0.f;
            });
#pragma unroll
            for (int u = 0; u < PER; ++u) x[u] = p.alpha * x[u] + p.beta * y[u];
        }
        each([&](float v, int row, int col) __attribute__((always_inline)) {
            if (own(row, col)) C[row * ldc + col] = v;
        });
    };
    auto any = [](bool b) __attribute__((always_inline)) { return __builtin_amdgcn_readfirstlane(__syncthreads_or(b)) != 0; };

    // An output that is not finite or small, or a large operand; and whether that
    // is a value outside the split's range.
    bool inf = false, odd = false;
    auto odd_block = [&]() __attribute__((always_inline)) {
        odd = la.large() || lb.large();
        each([&](float v, int, int) __attribute__((always_inline)) {
            inf |= !(fabsf(v) <= 3.402823466e38f);
            odd |= fabsf(v) < 0x1p-60f;
        });
        return any(inf || odd);
    };
    auto outside = [&]() __attribute__((always_inline)) {
        if (any(inf)) return true;
        unsigned* const most = reinterpret_cast<unsigned*>(smem_raw);  // rows of A, then of B
        for (int i = threadIdx.x; i < BM + BN; i += TL::THREADS) most[i] = 0;
        __syncthreads();
        la.row_max(most);
        lb.row_max(most + BM);
        __syncthreads();
        odd = la.large() || lb.large();
        bool tiny = false;
        each([&](float v, int row, int col) __attribute__((always_inline)) {
            const unsigned a = most[wrow + row], b = most[BM + wcol + col];
            odd |= fabsf(v) < 0x1p-60f && a != 0 && b != 0;
            tiny |= a - 1u < kTinyBits - 1u || b - 1u < kTinyBits - 1u;
        });
        if (!any(odd)) return false;
        if (any(tiny)) return true;
        return any(holds_tiny<AK, BM, TL::THREADS>(A, p.lda, m0, p.M, kbeg, kend) ||
                   holds_tiny<BKM, BN, TL::THREADS>(B, p.ldb, n0, p.N, kbeg, kend));
    };
    auto redo = [&]() __attribute__((always_inline)) {
        fp32_block<AK, BKM, TM, TN, TL::KG>(acc, A, B, p.lda, p.ldb, p.M, p.N, m0 + wrow, n0 + wcol, kbeg, kend, kg);
    };

    if constexpr (TL::KG > 1) {
        // Small products: the code they seldom run stays behind their end (in front
        // of the stores it took a 2048 x 512 x 512 product from 11.4 to 12.5 us).
        merge();
        if (!odd_block()) {
            store();
            return;
        }
        if (outside()) {
            redo();
            merge();
        }
        store();
        return;
    }
#pragma unroll 1
    for (int pass = 0;; ++pass) {
        if (pass == 1) redo();
        if (pass == 1 || !odd_block() || !outside()) break;
    }
    // as store() does it, written out: through the lambda the 256 x 128 tile
    // spills 8 to 21 registers (8192 x 2048 x 512 NT 95 -> 100 us)
    if (aux) {
        if constexpr (EARLY) {
            low[0][0] = old;
        } else {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const int row = i * 32 + acc_row(v, lane), col = j * 32 + (lane & 31);
                        low[i][j][v] = own(row, col) ? aux[row * ldc + col] : 0.f;
                    }
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = p.alpha * acc[i][j][v] + p.beta * low[i][j][v];
    }
    if (EARLY && blk.whole()) {
#pragma unroll
        for (int v = 0; v < 16; ++v) C[acc_row(v, lane) * ldc + (lane & 31)] = acc[0][0][v];
        return;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = i * 32 + acc_row(v, lane), col = j * 32 + (lane & 31);
                if (own(row, col)) C[row * ldc + col] = acc[i][j][v];
            }
}

// Block tiles.  T and S keep small products parallel (their waves share the
// reduction, so a block's chain of k-tiles is 1/8 or 1/2 as long); M and L move fewer operand bytes and convert each value for more MFMAs.
using X3T = X3Tile<32, 32, 1, 1, 8, 1>;     // 8 waves, one 32 x 32 each, every 8th k-step
using X3S = X3Tile<64, 64, 2, 2, 2, 2>;     // 2 x 4 waves of 32 x 32
using X3M = X3Tile<128, 128, 4, 2, 1, 2>;   // 8 waves of 32 x 64
using X3L = X3Tile<256, 128, 4, 2, 1, 2>;   // 8 waves of 64 x 64
using X3D = X3Tile<64, 64, 2, 2, 1, 2>;     // 4 waves of 32 x 32: short reductions (x3_plan)

// Time of a launch in us: c0 + rounds (e + c2 k), k = the reduction in whole
// k-tiles / 512, rounds of 256 blocks (one per CU), fitted to products timed on
// one box (us; NT, the other layouts within 8 %):
//                        T     S     M     L
//    512 x  512 x  512   7.1  11.3  23.6  38.7
//   2048 x  512 x  512  24.2  13.1  24.8  39.3
//   2048 x 2048 x  512  86.8  44.5  28.4  42.2
//  65536 x 2048 x  512  2781  1376   852   743 (185 TF/s)
//   4096 x 4096 x 4096  1587  1027   749   655 (210 TF/s)
// Converting inside the products (scheduling barriers per product group, loads
// two k-tiles ahead) was slower (M 852 -> 962, L 743 -> 798): the compiler's own
// order, which converts after the last product, leaves the overlap to the
// other wave of the SIMD.
struct X3Cost {
    int bm, bn, bk;
    double c0, e, c2;
};
constexpr int kX3Tiles = 4, kX3D = 4;
constexpr X3Cost kX3Cost[kX3Tiles] = {{32, 32, 128, 1.6, 2.7, 2.9}, {64, 64, 64, 2.5, 3.3, 7.3},
                               {128, 128, 32, 2.0, 3.2, 22.9}, {256, 128, 32, 2.0, 6.0, 39.9}};

struct X3Plan {
    int tile;
    int64_t splits;
};

// The cheapest tile and split of the reduction (a power of two, at most
// max_splits; each split at least two k-tiles).  A split costs its partials'
// way to memory and back at ~4 TB/s and the launch that adds them.
//
// A product of a short reduction that fills the chip is bound by its output's
// way to memory, and there by how many blocks a CU keeps: D's four (one LDS
// stage each) against the others' one (us, against L or M where it was chosen):
//   8192 x 4096, C += :    R 16 86 -> 62   R 32 80 -> 51   R 64 88 -> 67   R 96 97 -> 81
//   8192 x 4096, NT:       R 16 44 -> 38   R 32 42 -> 37   R 48 54 -> 50   (64: 51 -> 55)
//   1024 x 512, C += / NT: R 16 9.9 -> 5.3 / 7.0 -> 4.4    512 x 512: 5.6 -> 5.1 / 4.8 -> 4.3
// With B MN-major and nothing to add, D and L are even.  Below 48 blocks T's
// shared reduction leaves more of the chip at work.
X3Plan x3_plan(bool nt, int64_t M, int64_t N, int64_t K, int64_t batch, int64_t max_splits, bool aux) {
    if (K <= (aux ? 96 : nt ? 48 : 0) && cdiv(M, X3D::BM) * cdiv(N, X3D::BN) * batch >= 48) return X3Plan{kX3D, 1};
    X3Plan best{0, 1};
    double least = 1e30;
    for (int t = 0; t < kX3Tiles; ++t) {
        const X3Cost& c = kX3Cost[t];
        const double tiles = (double)cdiv(M, c.bm) * cdiv(N, c.bn) * batch;
        for (int64_t s = 1; s <= max_splits && (s == 1 || K / s >= 2 * c.bk); s *= 2) {
            const double rounds = ceil(tiles * s / 256.0), k = cdiv(cdiv(K, s), c.bk) * c.bk / 512.0;
            double us = c.c0 + rounds * (c.e + c.c2 * k);
            if (s > 1) us += 4.0 + (double)s * batch * M * N * 8.0 / 4e6;
            if (us < least) {
                least = us;
                best = X3Plan{t, s};
            }
        }
    }
    return best;
}

template <bool AK, bool BKM, typename TL, bool EDGE>
int32_t x3_launch_e(hipStream_t st, const X3Args& p, const char* nm) {
    if (TL::LDS > 65536) {
        static bool attr_set = false;
        if (!attr_set && hipFuncSetAttribute((const void*)gemm_x3_k<AK, BKM, TL, EDGE>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, TL::LDS) != hipSuccess)
            return set_error(AR_EHIP, "%s: cannot set the LDS size", nm);
        attr_set = true;
    }
    const int64_t grid = cdiv(p.M, TL::BM) * cdiv(p.N, TL::BN) * p.splits * p.batch;
    // a reduction of less than two k-tiles uses one stage only
    const int lds = p.K >= 2 * TL::BK ? TL::LDS : TL::STAGE > TL::RED ? TL::STAGE : TL::RED;
    gemm_x3_k<AK, BKM, TL, EDGE><<<(unsigned)grid, TL::THREADS, lds, st>>>(p);
    return check_launch(nm);
}

template <bool AK, bool BKM, typename TL>
int32_t x3_launch(hipStream_t st, const X3Args& p, const char* nm) {
    const bool far = p.lda >= (1 << 22) || p.ldb >= (1 << 22);  // the plain form's item offsets are 32-bit
    const bool edge = far || p.K % TL::BK != 0 || (!AK && p.M % 8 != 0) || (!BKM && p.N % 8 != 0);
    return edge ? x3_launch_e<AK, BKM, TL, true>(st, p, nm) : x3_launch_e<AK, BKM, TL, false>(st, p, nm);
}

}  // namespace

int32_t gemm_x3(hipStream_t st, bool ak, bool bk, float* C, const float* A, const float* B, int64_t M, int64_t N,
                int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t max_splits, float* partial,
                const float* aux, float alpha, float beta, int64_t batch, int64_t sA, int64_t sB, int64_t sC,
                int64_t* splits, const char* nm) {
    // the 8-value loads need 8 values of every stored row (and of the reduction,
    // where an operand is K-major)
    if (!(M > 0 && N > 0 && K > 0 && (ak || M >= 8) && (bk || N >= 8) && (!(ak || bk) || K >= 8)))
        return set_error(AR_EINVAL, "%s: extent below 8", nm);
    const X3Plan plan = x3_plan(ak && bk, M, N, K, batch, partial ? max_splits : 1, aux != nullptr);
    X3Args p{C, A, B, M, N, K, lda, ldb, ldc, 0, 1, partial, aux, alpha, beta, sA, sB, sC, (int)batch};
    const int64_t bkk = plan.tile == kX3D ? X3D::BK : kX3Cost[plan.tile].bk;
    p.kps = cdiv(cdiv(K, plan.splits), bkk) * bkk;
    p.splits = (int)cdiv(K, p.kps);
    if (splits) *splits = p.splits;
#define AR_X3(AKv, BKv)                                             \
    switch (plan.tile) {                                            \
        case 0: return x3_launch<AKv, BKv, X3T>(st, p, nm);         \
        case 1: return x3_launch<AKv, BKv, X3S>(st, p, nm);         \
        case 2: return x3_launch<AKv, BKv, X3M>(st, p, nm);         \
        case kX3D: return x3_launch<AKv, BKv, X3D>(st, p, nm);      \
        default: return x3_launch<AKv, BKv, X3L>(st, p, nm);        \
    }
    if (ak && bk) AR_X3(true, true)
    if (ak) AR_X3(true, false)
    if (bk) AR_X3(false, true)
    AR_X3(false, false)
#undef AR_X3
}

}  // namespace ar
