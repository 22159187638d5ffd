// ar_attn_f32.hip -- fp32 flash attention forward and backward for the
// reference's flash_attn_fwd (ops.mojo:244-323), flash_attn_bwd_dq
// (ops.mojo:349-411) and flash_attn_bwd_dkv (ops.mojo:414-480), on the bf16
// matrix cores at fp32 accuracy (three-term splits, ar_split.hpp).
//
// Layout: q, k, v, O, dO are [B, T, H, hd] (token-major, heads interleaved:
// row stride H*hd), LSE and D are [B, T, H].  Key kp is visible from query qp
// iff kp <= qp and (window <= 0 or kp >= qp - window).
//
// Work decomposition: a workgroup owns 32 rows of one (b, h) -- queries for
// fwd / dQ, keys for dK / dV -- and its four waves walk the 32-row tiles of the
// other side, wave kg every fourth tile; at the end the four partial results
// are merged through LDS (the forward's with their softmax maxima).  Short
// sequences thus still fill the chip: at B 4, T 512, H 4 there are 256
// workgroups with two or three tiles per wave, where 128-row workgroups that
// walk all tiles in order were 64 with a chain of six.
//
// MFMA mapping.  The owned rows are the MFMA columns: the forward computes
// S^T = K Q^T, where lane l holds query l % 32 and 16 keys, so softmax
// statistics are per-lane values (two lanes share a query) and P (or dS) feeds
// the next product (O^T += V^T P^T) straight from the accumulators: lane half
// g holds rows {16 s + 4 g + 0..3, 16 s + 8 + 4 g + 0..3} for k-step s, and the
// other operand is read in that row order.
//
// Operands.  The owned rows (Q; Q and dO; K and V) are split once per
// workgroup into bf16 planes in LDS.  The streamed rows go straight from memory
// to registers, where each wave splits its own fragments: a row fragment is two
// 16-byte loads, a transposed one eight 4-byte loads of 32 consecutive columns.
// Nothing is staged and there is no barrier in the tile loop.
//
// The small terms of a product have their own accumulator, added to the large
// one per tile.
//
// Magnitudes.  The split is exact for zero and from 2^-110 to 3.39e38; below, a
// value loses up to 2^-134, and a block where that could show is formed on the
// fp32 matrix cores (EX):
//   * an own row with such a value;
//   * a result that is not finite (infinities, NaN, what bf16 rounds to infinity);
//   * a result below kSmall, or a magnitude above kBig among the own rows, the
//     streamed rows that form S and the dS, if the streamed rows hold a value
//     below 2^-110.
// Otherwise what is lost is below fp32's own rounding.  hd 2^-134 kBig = 2^-109
// of a score or of dP changes no exponential and moves a result by 2^-109 kBig
// per unit of P, the T 2^-134 kBig of small dS less; O and dV, formed from P
// 2^24 (so P keeps every bit above 2^-126), by 2^-134 per unit of P.  Against
// 2^-24 kSmall that leaves T up to 2^17.
//
// dK/dV are accumulated by key ownership and dQ by query ownership (no
// atomics: deterministic).
#include "ar_internal.hpp"
#include "ar_split.hpp"

namespace ar {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kTiny = 0x1p-110f, kBig = 0x1p18f, kSmall = 0x1p-48f, kScaleP = 0x1p24f;
constexpr int kRows = 32, kWaves = 4, kThreads = kWaves * kWave;  // own rows and waves of a workgroup

__device__ __forceinline__ int acc_row(int v, int lane) { return (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3); }

// 2^x with the hardware's v_exp_f32 (1 ulp): results below 2^-126
// (probabilities that change no fp32 sum they enter) flush to zero, and
// 2^-inf = 0.
__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// An MFMA operand fragment of 8 values per lane: split planes, or (EX) the
// values themselves.
template <bool EX> struct Frag;
template <> struct Frag<false> {
    bf16x8 p[3];
    __device__ __forceinline__ explicit Frag(const float (&x)[8]) {
#pragma unroll
        for (int e = 0; e < 8; e += 2) split2(x[e], x[e + 1], e, p[0], p[1], p[2]);
    }
    __device__ __forceinline__ Frag(const unsigned char* planes, int plane_bytes, int off) {
#pragma unroll
        for (int i = 0; i < 3; ++i) p[i] = *reinterpret_cast<const bf16x8*>(planes + i * plane_bytes + off);
    }
};
template <> struct Frag<true> {
    float x[8];
    __device__ __forceinline__ explicit Frag(const float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = v[e];
    }
};

// c + low (+)= a b over 16 k-values.  The fp32 instruction takes one k-value
// per lane half: step e multiplies value e of both halves.
__device__ __forceinline__ void dot16(f32x16& c, f32x16& low, const Frag<false>& a, const Frag<false>& b) {
    constexpr int PQ[5][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
#pragma unroll
    for (int q = 0; q < 5; ++q) low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[PQ[q][0]], b.p[PQ[q][1]], low, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.p[0], b.p[0], c, 0, 0, 0);
}
__device__ __forceinline__ void dot16(f32x16& c, f32x16&, const Frag<true>& a, const Frag<true>& b) {
#pragma unroll
    for (int e = 0; e < 8; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x[e], b.x[e], c, 0, 0, 0);
}
__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int e = 0; e < 16; ++e) z[e] = 0.f;
    return z;
}

// One (b, h) of an operand: rows of HD values, rs apart, with the lane's byte
// offsets into a tile (row fragments: row lane % 32, columns 8 (lane / 32)..;
// transposed ones: row 4 (lane / 32), column lane % 32).
struct Src {
    const float* base;
    int64_t rs;
    unsigned roff, coff;
    __device__ __forceinline__ Src(const float* p, int64_t rs_, int lane)
        : base(p), rs(rs_), roff((unsigned)((lane & 31) * (int)rs_ + (lane >> 5) * 8) * 4u),
          coff((unsigned)((lane >> 5) * 4 * (int)rs_ + (lane & 31)) * 4u) {}
};
__device__ __forceinline__ void ld8(float (&x)[8], const float* s) {
    const float4 a = *reinterpret_cast<const float4*>(s), b = *reinterpret_cast<const float4*>(s + 4);
    x[0] = a.x; x[1] = a.y; x[2] = a.z; x[3] = a.w;
    x[4] = b.x; x[5] = b.y; x[6] = b.z; x[7] = b.w;
}
// Values of a row fragment of the tile at row0: columns 16 ks + 8 (lane / 32) +
// 0..7.  The split products read whole tiles inside the sequence: a
// wave-uniform address plus the lane's offset; EX clamps each row to it.
template <bool EX>
__device__ __forceinline__ void row_vals(float (&x)[8], const Src& t, int row0, int T, int ks, int lane) {
    if constexpr (EX) {
        const int row = row0 + (lane & 31);
        ld8(x, t.base + (int64_t)(row < T ? row : T - 1) * t.rs + ks * 16 + (lane >> 5) * 8);
    } else {
        ld8(x, reinterpret_cast<const float*>(reinterpret_cast<const char*>(t.base + (int64_t)row0 * t.rs + ks * 16) + t.roff));
    }
}
// Values of a transposed fragment: column 32 dt + lane % 32, the 8 rows of
// k-step s in the accumulators' order.
template <bool EX>
__device__ __forceinline__ void col_vals(float (&x)[8], const Src& t, int row0, int T, int dt, int s, int lane) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int r = row0 + 16 * s + (e & 3) + (e >> 2) * 8;
        if constexpr (EX) {
            const int row = r + 4 * (lane >> 5);
            x[e] = t.base[(int64_t)(row < T ? row : T - 1) * t.rs + dt * 32 + (lane & 31)];
        } else {
            x[e] = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(t.base + (int64_t)r * t.rs + dt * 32) + t.coff);
        }
    }
}
__device__ __forceinline__ void acc_vals(float (&x)[8], const f32x16& a, int s, float f) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = a[8 * s + e] * f;
}

// What a thread has met: its least magnitude that is not zero and its largest.
struct Range {
    unsigned least = ~0u;  // twice the bits, less one: zero of either sign wraps to the top
    float most = 0.f;
    __device__ __forceinline__ void see(float x) {
        const unsigned u = __float_as_uint(x) * 2u - 1u;
        least = u < least ? u : least;
        most = fmaxf(most, fabsf(x));
    }
    __device__ __forceinline__ bool tiny() const { return least < __float_as_uint(kTiny) * 2u - 1u; }
    __device__ __forceinline__ bool big() const { return most > kBig; }
};
// Whether rows [r0, r1) hold a value below kTiny that is not zero, asked by the whole workgroup.
template <int HD>
__device__ __forceinline__ bool rows_tiny(const Src& t, int r0, int r1) {
    Range f;
#pragma unroll 2
    for (int r = r0 + (int)threadIdx.x / (HD / 8); r < r1; r += kThreads / (HD / 8)) {
        float x[8];
        ld8(x, t.base + (int64_t)r * t.rs + threadIdx.x % (HD / 8) * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) f.see(x[e]);
    }
    return f.tiny();
}

// Split planes of the own rows of an operand in LDS (K-major units, kslot
// order), written by the whole workgroup.
template <int HD>
__device__ __forceinline__ void own_planes(unsigned char* planes, const Src& t, int row0, int T, Range& seen) {
    constexpr int U = HD / 8, PB = kRows * HD * 2;
    for (int it = threadIdx.x; it < kRows * U; it += kThreads) {
        const int r = it / U, c = it % U, row = row0 + r;
        float x[8];
        ld8(x, t.base + (int64_t)(row < T ? row : T - 1) * t.rs + c * 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) seen.see(x[e]);
        const Frag<false> f(x);
        const int o = kslot<U>(r, c) * 16;
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(planes + i * PB + o) = f.p[i];
    }
}

// The own rows as MFMA columns: row row0 + lane % 32 of src, or its split planes.
struct Own {
    const unsigned char* planes;
    int row0;
};
template <bool EX, int HD>
__device__ __forceinline__ Frag<EX> own_frag(const Own& w, const Src& t, int T, int ks, int lane) {
    if constexpr (EX) {
        float x[8];
        row_vals<true>(x, t, w.row0, T, ks, lane);
        return Frag<true>(x);
    } else {
        return Frag<false>(w.planes, kRows * HD * 2, kslot<HD / 8>(lane & 31, 2 * ks + (lane >> 5)) * 16);
    }
}

// c[cols] += X^T . (f B) for the 32-row tile of X at row0 (columns dt 32..) and
// the 32 x 32 block b (accumulator layout): the small terms of the tile are
// summed apart.
template <bool EX, int HD>
__device__ __forceinline__ void add_tile(f32x16 (&c)[HD / 32], const Src& t, int row0, int T, const f32x16& b, float f, int lane) {
    float x[8];
    acc_vals(x, b, 0, f);
    const Frag<EX> b0(x);
    acc_vals(x, b, 1, f);
    const Frag<EX> b1(x);
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt) {
        f32x16 low = zero16();
        col_vals<EX>(x, t, row0, T, dt, 0, lane);
        dot16(c[dt], low, Frag<EX>(x), b0);
        col_vals<EX>(x, t, row0, T, dt, 1, lane);
        dot16(c[dt], low, Frag<EX>(x), b1);
        if constexpr (!EX) {
#pragma unroll
            for (int e = 0; e < 16; ++e) c[dt][e] += low[e];
        }
    }
}

// The 32 x 32 block of (streamed rows at row0) . (own rows)^T.  most: the largest
// streamed magnitude so far (null: not asked for).
template <bool EX, int HD>
__device__ __forceinline__ f32x16 row_products(const Src& t, int row0, int T, const Own& w, const Src& own, int lane,
                                               float* most = nullptr) {
    f32x16 c = zero16(), low = zero16();
#pragma unroll
    for (int ks = 0; ks < HD / 16; ++ks) {
        float x[8];
        row_vals<EX>(x, t, row0, T, ks, lane);
        if (!EX && most) {
#pragma unroll
            for (int e = 0; e < 8; e += 2) *most = fmaxf(fmaxf(fabsf(x[e]), fabsf(x[e + 1])), *most);
        }
        dot16(c, low, Frag<EX>(x), own_frag<EX, HD>(w, own, T, ks, lane));
        // two k-steps' loads in flight: with all HD / 16 hoisted dQ spills at hd
        // 128 and every kernel was slower (B16 T2048: fwd 552 -> 530 us, dQ 896 -> 842)
        if (ks & 1) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!EX) {
#pragma unroll
        for (int e = 0; e < 16; ++e) c[e] += low[e];
    }
    return c;
}

// Block id -> (head, row block): one head's blocks on one XCD (workgroups are
// dispatched round-robin over 8), the heaviest row blocks first.
__device__ __forceinline__ void block_of(int nblk, int heads, bool last_first, int& bh, int& blk) {
    int id = blockIdx.x;
    if (heads % 8 == 0) {
        const int x = id % 8, w = id / 8;
        bh = x + 8 * (w / nblk);
        blk = w % nblk;
    } else {
        bh = id / nblk;
        blk = id % nblk;
    }
    if (last_first) blk = nblk - 1 - blk;
}

template <int HD> constexpr int ld_out() { return HD + 4; }

// acc (transposed: rows d, column = the wave's row l % 32), times f, into the
// wave's 32 x HD region.
template <int HD>
__device__ __forceinline__ void put_block(float* reg, const f32x16 (&acc)[HD / 32], float f, int lane) {
    float* row = reg + (lane & 31) * ld_out<HD>() + (lane >> 5) * 4;
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<float4*>(row + dt * 32 + g * 8) =
                make_float4(acc[dt][g * 4] * f, acc[dt][g * 4 + 1] * f, acc[dt][g * 4 + 2] * f, acc[dt][g * 4 + 3] * f);
}

// Sums the regions of each row over the first ng waves (those that had a tile),
// in order, times scale_row[row]; y holds this thread's float4s.  inf, small:
// whether one of a valid row is not finite / below kSmall.
template <int HD>
__device__ __forceinline__ void sum_blocks(float4 (&y)[HD / 32], const float* regs, const float* scale_row,
                                           int valid, int ng, bool& inf, bool& small) {
    constexpr int RB = kRows * ld_out<HD>();
#pragma unroll
    for (int n = 0; n < HD / 32; ++n) {
        const int i = (n * kThreads + (int)threadIdx.x) * 4, r = i / HD, d = i % HD;
        const float* s = regs + r * ld_out<HD>() + d;
        float4 t = *reinterpret_cast<const float4*>(s);
#pragma unroll
        for (int g = 1; g < kWaves; ++g) {
            if (g >= ng) break;
            const float4 u = *reinterpret_cast<const float4*>(s + g * RB);
            t = make_float4(t.x + u.x, t.y + u.y, t.z + u.z, t.w + u.w);
        }
        const float f = scale_row ? scale_row[r] : 1.0f;
        t = make_float4(t.x * f, t.y * f, t.z * f, t.w * f);
        y[n] = t;
        const bool fine = (t.x - t.x) + (t.y - t.y) + (t.z - t.z) + (t.w - t.w) == 0.f;
        inf |= r < valid && !fine;
        small |= r < valid && fminf(fminf(fabsf(t.x), fabsf(t.y)), fminf(fabsf(t.z), fabsf(t.w))) < kSmall;
    }
}
template <int HD>
__device__ __forceinline__ void store_blocks(float* out, int64_t rs, const float4 (&y)[HD / 32], int valid) {
#pragma unroll
    for (int n = 0; n < HD / 32; ++n) {
        const int i = (n * kThreads + (int)threadIdx.x) * 4, r = i / HD, d = i % HD;
        if (r < valid) *reinterpret_cast<float4*>(out + (int64_t)r * rs + d) = y[n];
    }
}

// The planes of NP operands, or the waves' regions; then two values
// of every wave and row (m and l; LSE and D), and a row of scales.
constexpr int kStatLds = (2 * kWaves + 1) * kRows * 4;
template <int HD, int NP>
constexpr size_t attn_lds() {
    const size_t planes = (size_t)NP * 3 * kRows * HD * 2, regs = (size_t)kWaves * kRows * ld_out<HD>() * 4;
    return (planes > regs ? planes : regs) + kStatLds;
}

// First row of tile t as it is read: split products take whole tiles, so a
// sequence's last, partial tile starts early (the rows it shares with the tile
// before are masked: row >= 32 t).
template <bool EX>
__device__ __forceinline__ int tile_row(int t, int T) {
    return EX || t * 32 + 32 <= T ? t * 32 : T - 32;
}

// The tiles that the rows from r0 see: keys of queries, queries of keys.
struct Tiles {
    int first, last;
    __device__ __forceinline__ int waves() const { return last - first + 1 < kWaves ? last - first + 1 : kWaves; }
};
__device__ __forceinline__ Tiles key_tiles(int r0, int T, int window) {
    return {window > 0 && r0 > window ? (r0 - window) / 32 : 0, (r0 + 31 < T ? r0 + 31 : T - 1) / 32};
}
__device__ __forceinline__ Tiles query_tiles(int r0, int T, int window) {
    return {r0 / 32, (window > 0 && r0 + 31 + window < T ? r0 + 31 + window : T - 1) / 32};
}

// ============================ forward ============================
template <bool EX, int HD>
__device__ __forceinline__ void fwd_tiles(f32x16 (&o)[HD / 32], float& m, float& l, const Own& w, const Src& q,
                                          const Src& k, const Src& v, int T, int window, float scale_log2, int kg,
                                          int lane) {
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt) o[dt] = zero16();
    m = -INFINITY;
    l = 0.f;
    const int qw = w.row0, my_q = qw + (lane & 31);
    if (qw >= T) return;
    const Tiles tiles = key_tiles(qw, T, window);
#pragma unroll 1
    for (int kt = tiles.first + kg; kt <= tiles.last; kt += kWaves) {
        const int k0 = tile_row<EX>(kt, T);
        f32x16 s = row_products<EX, HD>(k, k0, T, w, q, lane);
        float mt = -INFINITY;
        const bool full = kt * 32 + 31 <= qw && (window <= 0 || kt * 32 >= qw + 31 - window);  // no masked pair
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int key = k0 + acc_row(e, lane);
            const bool ok = full || (key >= kt * 32 && key <= my_q && key < T && (window <= 0 || key >= my_q - window));
            s[e] = ok ? s[e] * scale_log2 : -INFINITY;
            mt = fmaxf(mt, s[e]);
        }
        mt = fmaxf(mt, __shfl_xor(mt, 32, kWave));
        const float m_new = fmaxf(m, mt);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = exp2_hw(m - m_use);
        float rsum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[e] = exp2_hw(s[e] - m_use);
            rsum += s[e];
        }
        rsum += __shfl_xor(rsum, 32, kWave);
        l = l * alpha + rsum;
        if (__ballot(m_new != m)) {
#pragma unroll
            for (int dt = 0; dt < HD / 32; ++dt)
#pragma unroll
                for (int e = 0; e < 16; ++e) o[dt][e] *= alpha;
        }
        m = m_new;
        add_tile<EX, HD>(o, v, k0, T, s, EX ? 1.f : kScaleP, lane);
    }
}

template <int HD>
__global__ __launch_bounds__(kThreads, HD == 128 ? 2 : HD == 64 ? 3 : 4) void attn_fwd_k(float* out, float* lse, const float* qp, const float* kp,
                                                     const float* vp, int T, int H, int nblk, int heads, int window,
                                                     float scale_log2) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr size_t kMain = attn_lds<HD, 1>() - kStatLds;
    float* const regs = reinterpret_cast<float*>(smem);
    float* const ml = reinterpret_cast<float*>(smem + kMain);  // m, l per wave and row, then 1 / l per row
    float* const inv = ml + 2 * kWaves * kRows;
    const int lane = threadIdx.x % kWave, kg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int bh, blk;
    block_of(nblk, heads, true, bh, blk);
    const int b = bh / H, h = bh % H, q0 = blk * kRows;
    const int64_t rs = (int64_t)H * HD, off = (int64_t)b * T * rs + (int64_t)h * HD;
    const Src q(qp + off, rs, lane), k(kp + off, rs, lane), v(vp + off, rs, lane);
    const Own w{smem, q0};
    const Tiles seen = key_tiles(q0, T, window);
    const int ng = seen.waves();
    const int valid = T - q0 < kRows ? T - q0 : kRows, my_q = w.row0 + lane;

    Range mine;
    own_planes<HD>(smem, q, q0, T, mine);
    __syncthreads();
    f32x16 o[HD / 32];
    float m, l;
    if (T >= 32) fwd_tiles<false, HD>(o, m, l, w, q, k, v, T, window, scale_log2, kg, lane);
    float4 y[HD / 32];
    float my_lse = 0.f;
#pragma unroll 1
    for (int pass = T >= 32 ? 0 : 1;; ++pass) {
        if (pass == 1) fwd_tiles<true, HD>(o, m, l, w, q, k, v, T, window, scale_log2, kg, lane);
        __syncthreads();  // the planes / the first pass's regions are done with
        if (lane < 32) {
            ml[(kg * 2) * 32 + lane] = m;
            ml[(kg * 2 + 1) * 32 + lane] = l;
        }
        __syncthreads();
        float mt = -INFINITY, lt = 0.f;
#pragma unroll
        for (int g = 0; g < kWaves; ++g) mt = fmaxf(mt, ml[g * 64 + (lane & 31)]);
        const float m_use = mt == -INFINITY ? 0.f : mt;
#pragma unroll
        for (int g = 0; g < kWaves; ++g) {
            const int i = g * 64 + (lane & 31);
            lt += ml[i + 32] * exp2_hw(ml[i] - m_use);
        }
        if (kg < ng) put_block<HD>(regs + kg * kRows * ld_out<HD>(), o, exp2_hw(m - m_use), lane);
        if (kg == 0 && lane < 32) {
            inv[lane] = lt > 0.f ? (pass == 0 ? 1.0f / kScaleP : 1.0f) / lt : 0.f;
            my_lse = lt > 0.f ? (mt + log2f(lt)) * kLn2 : -INFINITY;
        }
        __syncthreads();
        bool redo = mine.tiny() || (kg == 0 && lane < 32 && my_q < T && !(fabsf(my_lse) <= 3.402823466e38f));
        bool look = mine.big();
        sum_blocks<HD>(y, regs, inv, valid, ng, redo, look);
        if (pass == 1 || !__syncthreads_or(redo || look)) break;
        const int r0 = seen.first * 32, r1 = q0 + valid;
        if (!__syncthreads_or(redo) && !__syncthreads_or(rows_tiny<HD>(k, r0, r1) || rows_tiny<HD>(v, r0, r1))) break;
    }
    store_blocks<HD>(out + off + (int64_t)q0 * rs, rs, y, valid);
    if (kg == 0 && lane < 32 && my_q < T) lse[((int64_t)b * T + my_q) * H + h] = my_lse;
}

// ============================ backward: dQ ============================
template <bool EX, int HD>
__device__ __forceinline__ void dq_tiles(f32x16 (&acc)[HD / 32], const Own& w, const Src& q, const Src& k, const Src& v,
                                         const Src& dout, int T, int window, float scale_log2, float lse2, float dd,
                                         float& most, int kg, int lane) {
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt) acc[dt] = zero16();
    const int qw = w.row0, my_q = qw + (lane & 31);
    if (qw >= T) return;
    const Own wd{w.planes + 3 * kRows * HD * 2, w.row0};  // Q planes, then dO planes
    const Tiles tiles = key_tiles(qw, T, window);
#pragma unroll 1
    for (int kt = tiles.first + kg; kt <= tiles.last; kt += kWaves) {
        const int k0 = tile_row<EX>(kt, T);
        const f32x16 s = row_products<EX, HD>(k, k0, T, w, q, lane, &most);
        f32x16 ds = row_products<EX, HD>(v, k0, T, wd, dout, lane);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int key = k0 + acc_row(e, lane);
            const bool ok = key >= kt * 32 && key <= my_q && key < T && my_q < T && (window <= 0 || key >= my_q - window);
            const float p = ok ? exp2_hw(s[e] * scale_log2 - lse2) : 0.f;
            ds[e] = p * (ds[e] - dd);
            if (!EX) most = fmaxf(most, fabsf(ds[e]));
        }
        add_tile<EX, HD>(acc, k, k0, T, ds, 1.f, lane);
    }
}

template <int HD>
__global__ __launch_bounds__(kThreads, HD == 128 ? 2 : HD == 64 ? 3 : 4) void attn_dq_k(float* dq, const float* qp, const float* kp, const float* vp,
                                                    const float* dop, const float* lse, const float* dbuf, int T, int H,
                                                    int nblk, int heads, int window, float scale_log2, float scale) {
    extern __shared__ __align__(16) unsigned char smem[];
    float* const regs = reinterpret_cast<float*>(smem);
    const int lane = threadIdx.x % kWave, kg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int bh, blk;
    block_of(nblk, heads, true, bh, blk);
    const int b = bh / H, h = bh % H, q0 = blk * kRows;
    const int64_t rs = (int64_t)H * HD, off = (int64_t)b * T * rs + (int64_t)h * HD;
    const Src q(qp + off, rs, lane), k(kp + off, rs, lane), v(vp + off, rs, lane), dout(dop + off, rs, lane);
    const Own w{smem, q0};
    const Tiles seen = key_tiles(q0, T, window);
    const int ng = seen.waves();
    const int valid = T - q0 < kRows ? T - q0 : kRows, my_q = w.row0 + (lane & 31);
    const int64_t bth = ((int64_t)b * T + (my_q < T ? my_q : 0)) * H + h;
    const float lse2 = lse[bth] * kLog2e, dd = dbuf[bth];

    Range mine;
    own_planes<HD>(smem, q, q0, T, mine);
    own_planes<HD>(smem + 3 * kRows * HD * 2, dout, q0, T, mine);
    __syncthreads();
    f32x16 acc[HD / 32];
    float most = 0.f;
    if (T >= 32) dq_tiles<false, HD>(acc, w, q, k, v, dout, T, window, scale_log2, lse2, dd, most, kg, lane);
    float4 y[HD / 32];
#pragma unroll 1
    for (int pass = T >= 32 ? 0 : 1;; ++pass) {
        if (pass == 1) dq_tiles<true, HD>(acc, w, q, k, v, dout, T, window, scale_log2, lse2, dd, most, kg, lane);
        __syncthreads();
        if (kg < ng) put_block<HD>(regs + kg * kRows * ld_out<HD>(), acc, scale, lane);
        __syncthreads();
        bool redo = mine.tiny(), look = mine.big() || most > kBig;
        sum_blocks<HD>(y, regs, nullptr, valid, ng, redo, look);
        if (pass == 1 || !__syncthreads_or(redo || look)) break;
        const int r0 = seen.first * 32, r1 = q0 + valid;
        if (!__syncthreads_or(redo) && !__syncthreads_or(rows_tiny<HD>(k, r0, r1) || rows_tiny<HD>(v, r0, r1))) break;
    }
    store_blocks<HD>(dq + off + (int64_t)q0 * rs, rs, y, valid);
}

// ============================ backward: dK, dV ============================
template <bool EX, int HD>
__device__ __forceinline__ void dkv_tiles(f32x16 (&dka)[HD / 32], f32x16 (&dva)[HD / 32], const Own& w, const Src& q,
                                          const Src& k, const Src& v, const Src& dout, const float* lse,
                                          const float* dbuf, float* stat, int H, int T, int window,
                                          float scale_log2, float& most, int kg, int lane) {
#pragma unroll
    for (int dt = 0; dt < HD / 32; ++dt) dka[dt] = dva[dt] = zero16();
    const int kw = w.row0, my_k = kw + (lane & 31);
    if (kw >= T) return;
    const Own wv{w.planes + 3 * kRows * HD * 2, w.row0};  // K planes, then V planes
    const Tiles tiles = query_tiles(kw, T, window);
#pragma unroll 1
    for (int qt = tiles.first + kg; qt <= tiles.last; qt += kWaves) {
        const int q0 = tile_row<EX>(qt, T);
        // LSE and D of the tile's queries, a row per lane, on their way before the
        // product that needs them, then from LDS.  (Loaded by the masked
        // exponentials they were a chain of 16 trips to memory and 16 addresses in
        // registers: B64 T128 H8 hd128 155 -> 109 us, hd64 60 -> 50.)
        const int qr = q0 + (lane & 31);
        const int64_t at = (int64_t)(!EX || qr < T ? qr : T - 1) * H;
        if (lane < 32) {
            stat[lane] = lse[at] * kLog2e;
            stat[32 + lane] = dbuf[at];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        f32x16 p = row_products<EX, HD>(q, q0, T, w, k, lane, &most);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int qi = q0 + acc_row(e, lane);
            const bool ok = qi >= qt * 32 && my_k <= qi && qi < T && my_k < T && (window <= 0 || my_k >= qi - window);
            const float x = exp2_hw(p[e] * scale_log2 - stat[acc_row(e, lane)]);
            p[e] = ok ? x : 0.f;
        }
        add_tile<EX, HD>(dva, dout, q0, T, p, EX ? 1.f : kScaleP, lane);
        f32x16 ds = row_products<EX, HD>(dout, q0, T, wv, v, lane);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            ds[e] = p[e] * (ds[e] - stat[32 + acc_row(e, lane)]);
            if (!EX) most = fmaxf(most, fabsf(ds[e]));
        }
        add_tile<EX, HD>(dka, q, q0, T, ds, 1.f, lane);
    }
}

// OCC: workgroups per CU the registers allow.  At hd 128 one per CU (all of
// both accumulators, both fragments and their loads in registers) is faster
// while each CU has no more than one (B4 T512 H4 window 256: 35 against 38 us,
// B1 T2048 H4: 160 against 207), two with 32 spilled registers beyond that
// (B24 T64 H8: 26 against 32, B16 T2048 H4: 1061 against 1480).
template <int HD, int OCC>
__global__ __launch_bounds__(kThreads, OCC) void attn_dkv_k(float* dk, float* dv, const float* qp, const float* kp,
                                                     const float* vp, const float* dop, const float* lse,
                                                     const float* dbuf, int T, int H, int nblk, int heads, int window,
                                                     float scale_log2, float scale) {
    extern __shared__ __align__(16) unsigned char smem[];
    float* const regs = reinterpret_cast<float*>(smem);
    const int lane = threadIdx.x % kWave, kg = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    int bh, blk;
    block_of(nblk, heads, false, bh, blk);
    const int b = bh / H, h = bh % H, k0 = blk * kRows;
    const int64_t rs = (int64_t)H * HD, off = (int64_t)b * T * rs + (int64_t)h * HD;
    const Src q(qp + off, rs, lane), k(kp + off, rs, lane), v(vp + off, rs, lane), dout(dop + off, rs, lane);
    const Own w{smem, k0};
    const Tiles seen = query_tiles(k0, T, window);
    const int ng = seen.waves();
    const int valid = T - k0 < kRows ? T - k0 : kRows;
    const float* const lb = lse + (int64_t)b * T * H + h;
    const float* const db = dbuf + (int64_t)b * T * H + h;
    float* const stat = reinterpret_cast<float*>(smem + attn_lds<HD, 2>() - kStatLds) + kg * 2 * kRows;

    Range mine;
    own_planes<HD>(smem, k, k0, T, mine);
    own_planes<HD>(smem + 3 * kRows * HD * 2, v, k0, T, mine);
    __syncthreads();
    f32x16 dka[HD / 32], dva[HD / 32];
    float most = 0.f;
    if (T >= 32) dkv_tiles<false, HD>(dka, dva, w, q, k, v, dout, lb, db, stat, H, T, window, scale_log2, most, kg, lane);
    float4 yk[HD / 32], yv[HD / 32];
#pragma unroll 1
    for (int pass = T >= 32 ? 0 : 1;; ++pass) {
        if (pass == 1)
            dkv_tiles<true, HD>(dka, dva, w, q, k, v, dout, lb, db, stat, H, T, window, scale_log2, most, kg, lane);
        __syncthreads();
        if (kg < ng) put_block<HD>(regs + kg * kRows * ld_out<HD>(), dka, scale, lane);
        __syncthreads();
        bool redo = mine.tiny(), look = mine.big() || most > kBig;
        sum_blocks<HD>(yk, regs, nullptr, valid, ng, redo, look);
        __syncthreads();
        if (kg < ng) put_block<HD>(regs + kg * kRows * ld_out<HD>(), dva, pass == 0 ? 1.0f / kScaleP : 1.0f, lane);
        __syncthreads();
        sum_blocks<HD>(yv, regs, nullptr, valid, ng, redo, look);
        if (pass == 1 || !__syncthreads_or(redo || look)) break;
        const int r1 = seen.last * 32 + 32 < T ? seen.last * 32 + 32 : T;
        if (!__syncthreads_or(redo) && !__syncthreads_or(rows_tiny<HD>(q, k0, r1) || rows_tiny<HD>(dout, k0, r1))) break;
    }
    store_blocks<HD>(dk + off + (int64_t)k0 * rs, rs, yk, valid);
    store_blocks<HD>(dv + off + (int64_t)k0 * rs, rs, yv, valid);
}

template <typename K>
int32_t attn_attr(K* kern, size_t lds) {
    if (lds > 65536 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return set_error(AR_EHIP, "flash attention: cannot set the LDS size");
    return AR_OK;
}

template <int HD>
int32_t attn_launch(hipStream_t st, AttnOp op, float* o1, float* o2, const float* q, const float* k, const float* v,
                    const float* dout, const float* lse, const float* dbuf, int B, int T, int H, int window, float sc) {
    const float scale = sc > 0.f ? sc : 1.0f / sqrtf((float)HD), scale_log2 = scale * kLog2e;
    const int nblk = (int)cdiv(T, kRows), heads = B * H;
    const unsigned grid = (unsigned)nblk * (unsigned)heads;
    if (op == AttnOp::FWD) {
        constexpr size_t lds = attn_lds<HD, 1>();
        static const int32_t ok = attn_attr(attn_fwd_k<HD>, lds);
        if (ok) return ok;
        attn_fwd_k<HD><<<grid, kThreads, lds, st>>>(o1, o2, q, k, v, T, H, nblk, heads, window, scale_log2);
        return check_launch("flash_attn_fwd");
    }
    constexpr size_t lds = attn_lds<HD, 2>();
    if (op == AttnOp::DQ) {
        static const int32_t ok = attn_attr(attn_dq_k<HD>, lds);
        if (ok) return ok;
        attn_dq_k<HD><<<grid, kThreads, lds, st>>>(o1, q, k, v, dout, lse, dbuf, T, H, nblk, heads, window,
                                                      scale_log2, scale);
        return check_launch("flash_attn_bwd_dq");
    }
#define AR_DKV(OCC)                                                                                                  \
    do {                                                                                                             \
        static const int32_t ok = attn_attr(attn_dkv_k<HD, OCC>, lds);                                       \
        if (ok) return ok;                                                                                           \
        attn_dkv_k<HD, OCC><<<grid, kThreads, lds, st>>>(o1, o2, q, k, v, dout, lse, dbuf, T, H, nblk, heads, window, \
                                                            scale_log2, scale);                                      \
    } while (0)
    if constexpr (HD == 128) {
        if (grid <= 256) AR_DKV(1);
        else AR_DKV(2);
    } else {
        AR_DKV(HD == 64 ? 2 : 3);
    }
#undef AR_DKV
    return check_launch("flash_attn_bwd_dkv");
}

}  // namespace

int32_t attn_f32(hipStream_t st, AttnOp op, float* o1, float* o2, const float* q, const float* k, const float* v,
                 const float* dout, const float* lse, const float* dbuf, int64_t B, int64_t T, int64_t H, int64_t HD,
                 int64_t window, float scale) {
    if (HD > 128) return set_error(AR_EUNSUPPORTED, "flash attention: head_dim %lld > 128", (long long)HD);
    if (B <= 0 || T <= 0 || H <= 0) return B == 0 || T == 0 ? AR_OK : set_error(AR_EINVAL, "flash attention: bad shape");
    if (B * H > 65535 || T > (1 << 30)) return set_error(AR_EINVAL, "flash attention: shape too large");
    const int w = window > T ? (int)T : (int)window;  // a window >= T is full causal
#define AR_AT(HDv) attn_launch<HDv>(st, op, o1, o2, q, k, v, dout, lse, dbuf, (int)B, (int)T, (int)H, w, scale)
    switch (HD) {
        case 32: return AR_AT(32);
        case 64: return AR_AT(64);
        case 128: return AR_AT(128);
        default: return set_error(AR_EUNSUPPORTED, "flash attention: head_dim %lld not in {32, 64, 128}", (long long)HD);
    }
#undef AR_AT
}

}  // namespace ar
