// Whole-matrix DCT-II / DCT-III (orthonormal) in two passes over memory: the
// 1-D transforms of all rows, then those of all columns, a workgroup holding
// 2 PC neighbouring lines (rows or columns) in LDS.
//
// 1-D transform of length N by Makhoul's reordering (J. Makhoul, "A fast
// cosine transform in one and two dimensions", IEEE Trans. ASSP 28(1),
// 1980), two real lines packed into one complex sequence, so that N may be
// odd:
//   forward  v[m] = x[2m], v[N-1-m] = x[2m+1]; Z = DFT_N(v1 + i v2);
//            V1[k] = (Z[k] + conj Z[N-k]) / 2, V2[k] = (Z[k] - conj Z[N-k]) / 2i;
//            X[k] = s_k Re(w_4N^-k V[k]), X[N-k] = -s_{N-k} Im(w_4N^-k V[k])
//   inverse  H[0] = s_0 c[0], H[k] = s_k w_4N^k (c[k] - i c[N-k]) / 2;
//            Z = H1 + i H2; v1 + i v2 = unnormalised inverse DFT_N(Z)
// with w_n = e^(2 pi i / n), s_0 = sqrt(1/N), s_k = sqrt(2/N).  The DFT runs
// in LDS as a Stockham autosort FFT in f32 (radix 16, 8, 4, 2, 3, 5, 7, then
// other primes up to 127 as direct sums), twiddles rounded from double.
//
// The row pass writes its result in panels [h / G][w][G] of G rows, its own
// 2 PC or those of two or four workgroups of one XCD (panel_share): the
// column pass, whose lines are 2 PC columns, reads 2 PC G neighbouring values
// at a time.  The column pass writes the row-major result, 2 PC elements of
// a row at a time; workgroups of neighbouring columns are placed on one XCD
// so that its L2 joins their writes into whole lines.  Where a workgroup
// holds two columns only (more than 8192 rows), it writes them as panels and
// untangle_kernel makes rows of them through LDS tiles (through_panels).
//
// What bounds it: each pass reads and writes the matrix once (4096 x 4096 to
// bf16: 64 + 64 + 64 + 32 MB, 36 us at the device copy's 6.3 TB/s); a pass
// takes 42-43 us there, its workgroups' loads, ~1,100 VALU instructions per
// wave and stores one after the other (VALU ~40 % busy).  Against the row
// transforms and transposes of dct_fft.hip (four passes over f32 matrices):
// 4096 x 4096 87 against 141 us, 14336 x 4096 forward 432 against 638 us; and
// against the dense products, which shapes below 1024 and sides with other
// primes took: 576 x 576 18 against 105 us, 3000 x 1280 44 against 330 us --
// so every shape this file supports takes it.
//
// The reference's whole-matrix transforms switch to an FFT above 4096
// (haagenti-cuda/src/dct_gpu.rs:1081,1381-1412, via cufft_ffi.rs:423-506);
// its CPU path is the same Makhoul construction (haagenti-core/src/
// dct.rs:154-259).
#include "hh_internal.hpp"

namespace hh {
namespace {

constexpr uint32_t kMaxPoints = 16384;  // complex points per workgroup: 128 KiB of LDS and its padding
constexpr uint32_t kPerThread = 16;     // of them per thread (1024 threads of at most 128 registers)
constexpr uint32_t kMaxLds = 160u * 1024u;
constexpr uint32_t kMaxPrime = 127;
constexpr uint32_t kMaxFrags = 16;
constexpr uint32_t kQB = 8;             // output pairs per wave task of a prime pass
constexpr uint32_t kMaxTasks = 2;       // wave tasks of a prime pass held in registers
constexpr uint32_t kFewButterflies = 64;  // below them a prime pass has a thread per output pair
constexpr uint32_t kFewPairs = 4;         // of them per thread, at most (63 butterflies, 63 pairs)

enum : int { kSrcRows = 0, kSrcPanels = 1, kSrcFrags = 2 };
enum : int { kDstPanels = 3 };          // else the dtype of a row-major result
// prime passes of a kernel: none, of at least kFewButterflies butterflies, any
// (each its own kernel: the last one's registers cost the others up to 5 %)
enum : int { kPrimesNone = 0, kPrimesMany = 1, kPrimesAny = 2 };

struct Lines {
    const float *in;
    void *out;
    // twiddles (lines_tables_kernel): per pass q (radix R_q, p_q the product
    // of the earlier radices) w_N^(j k N / (p_q R_q)) at [off_q + (j - 1)
    // p_q + k]; s_1 / 2 w_4N^k for k <= N / 2; the r-th roots of unity of
    // each prime pass in order
    const float2 *ptab, *w4, *rt;
    uint32_t N;       // line length
    uint32_t lines;   // number of lines
    uint32_t gsh;     // log2 of the panels' height G (kSrcPanels)
    uint32_t ipitch;  // points from a panel to the next (kSrcPanels)
    uint32_t opitch;  // the same of the output (kDstPanels)
    uint32_t pcs;     // log2 of the pairs of lines per workgroup
    uint32_t psh;     // LDS: point x at slot x + (x >> psh)
    uint32_t per_xcd; // workgroups per XCD (0: not placed)
    uint32_t msh;     // kDstPanels: log2 of the workgroups that fill a panel
    uint32_t nr;
    uint64_t radix[2]; // a byte each, in order (kept in scalar registers)
    // kSrcFrags: fragment f's bitmap (bit row N + n), values and per-row set
    // bit counts
    uint32_t nfrag, coef_f32;
    const uint8_t *bitmap[kMaxFrags];
    const uint8_t *coef[kMaxFrags];
    const uint32_t *counts[kMaxFrags];
    uint32_t ncoef[kMaxFrags];
};

struct Untangle {
    const float *in;
    void *out;
    uint32_t N, lines, pcs;
};

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
    return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
// i^S a for S = +1 (INV) or -1
template <bool INV>
__device__ __forceinline__ float2 rot90(float2 a) {
    return INV ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}
// a (c + i s) for INV, a (c - i s) otherwise
template <bool INV>
__device__ __forceinline__ float2 rot(float2 a, float c, float s) {
    return cmul(a, make_float2(c, INV ? s : -s));
}

// In-register DFT of length R with e^(+-2 pi i / R) (+ for INV).
template <int R, bool INV>
struct Dft;

template <bool INV>
struct Dft<2, INV> {
    __device__ __forceinline__ static void run(float2 *x) {
        const float2 a = x[0], b = x[1];
        x[0] = cadd(a, b);
        x[1] = csub(a, b);
    }
};

template <bool INV>
__device__ __forceinline__ void dft4(float2 &a, float2 &b, float2 &c, float2 &d) {
    const float2 t0 = cadd(a, c), t1 = csub(a, c);
    const float2 t2 = cadd(b, d), t3 = rot90<INV>(csub(b, d));
    a = cadd(t0, t2);
    c = csub(t0, t2);
    b = cadd(t1, t3);
    d = csub(t1, t3);
}

template <bool INV>
struct Dft<4, INV> {
    __device__ __forceinline__ static void run(float2 *x) { dft4<INV>(x[0], x[1], x[2], x[3]); }
};

template <bool INV>
struct Dft<8, INV> {
    __device__ __forceinline__ static void run(float2 *x) {
        float2 e[4] = {x[0], x[2], x[4], x[6]};
        float2 o[4] = {x[1], x[3], x[5], x[7]};
        Dft<4, INV>::run(e);
        Dft<4, INV>::run(o);
        constexpr float h = 7.071067812e-01f;  // 1 / sqrt(2)
        o[1] = INV ? make_float2(h * (o[1].x - o[1].y), h * (o[1].x + o[1].y))
                   : make_float2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
        o[2] = rot90<INV>(o[2]);
        o[3] = INV ? make_float2(-h * (o[3].x + o[3].y), h * (o[3].x - o[3].y))
                   : make_float2(h * (o[3].y - o[3].x), -h * (o[3].x + o[3].y));
#pragma unroll
        for (int q = 0; q < 4; q++) {
            x[q] = cadd(e[q], o[q]);
            x[q + 4] = csub(e[q], o[q]);
        }
    }
};

template <bool INV>
struct Dft<16, INV> {
    __device__ __forceinline__ static void run(float2 *x) {
        // columns b of x[4 a + b] over a, the twiddles w_16^(b q), rows over b
#pragma unroll
        for (int b = 0; b < 4; b++) dft4<INV>(x[b], x[4 + b], x[8 + b], x[12 + b]);
        constexpr float h = 7.071067812e-01f, c = 9.238795325e-01f, s = 3.826834324e-01f;
        // x[4 q + b] holds frequency q of column b
        x[5] = rot<INV>(x[5], c, s);
        x[6] = rot<INV>(x[6], h, h);
        x[7] = rot<INV>(x[7], s, c);
        x[9] = rot<INV>(x[9], h, h);
        x[10] = rot90<INV>(x[10]);
        x[11] = rot<INV>(x[11], -h, h);
        x[13] = rot<INV>(x[13], s, c);
        x[14] = rot<INV>(x[14], -h, h);
        x[15] = rot<INV>(x[15], -c, -s);
#pragma unroll
        for (int q = 0; q < 4; q++) dft4<INV>(x[4 * q], x[4 * q + 1], x[4 * q + 2], x[4 * q + 3]);
        // frequency q + 4 t sits at 4 q + t: transpose the 4 x 4
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
            for (int t = q + 1; t < 4; t++) {
                const float2 u = x[4 * q + t];
                x[4 * q + t] = x[4 * t + q];
                x[4 * t + q] = u;
            }
    }
};

template <bool INV>
struct Dft<3, INV> {
    __device__ __forceinline__ static void run(float2 *x) {
        constexpr float s3 = 8.660254038e-01f;  // sin(2 pi / 3)
        const float2 t = cadd(x[1], x[2]);
        const float2 u = rot90<INV>(csub(x[1], x[2]));
        const float2 m = make_float2(x[0].x - 0.5f * t.x, x[0].y - 0.5f * t.y);
        x[0] = cadd(x[0], t);
        x[1] = make_float2(m.x + s3 * u.x, m.y + s3 * u.y);
        x[2] = make_float2(m.x - s3 * u.x, m.y - s3 * u.y);
    }
};

// odd R: y_q = x_0 + sum_m a_m cos(2 pi m q / R) +- i sum_m b_m sin(2 pi m q / R)
// over m = 1 .. (R-1)/2 with a_m = x_m + x_{R-m}, b_m = x_m - x_{R-m}
template <int R, bool INV>
__device__ __forceinline__ void dft_odd(float2 *x, const float *c, const float *sn) {
    constexpr int H = (R - 1) / 2;
    float2 a[H], b[H];
#pragma unroll
    for (int m = 1; m <= H; m++) {
        a[m - 1] = cadd(x[m], x[R - m]);
        b[m - 1] = rot90<INV>(csub(x[m], x[R - m]));
    }
    const float2 x0 = x[0];
#pragma unroll
    for (int m = 0; m < H; m++) x[0] = cadd(x[0], a[m]);
#pragma unroll
    for (int q = 1; q <= H; q++) {
        float2 re = x0, im = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int m = 1; m <= H; m++) {
            const int j = (m * q) % R;  // cos / sin of 2 pi j / R, j in [1, R)
            const float cj = j <= H ? c[j - 1] : c[R - j - 1];
            const float sj = j <= H ? sn[j - 1] : -sn[R - j - 1];
            re = make_float2(re.x + cj * a[m - 1].x, re.y + cj * a[m - 1].y);
            im = make_float2(im.x + sj * b[m - 1].x, im.y + sj * b[m - 1].y);
        }
        x[q] = cadd(re, im);
        x[R - q] = csub(re, im);
    }
}

template <bool INV>
struct Dft<5, INV> {
    __device__ __forceinline__ static void run(float2 *x) {
        constexpr float c[2] = {3.090169944e-01f, -8.090169944e-01f};
        constexpr float sn[2] = {9.510565163e-01f, 5.877852523e-01f};
        dft_odd<5, INV>(x, c, sn);
    }
};

template <bool INV>
struct Dft<7, INV> {
    __device__ __forceinline__ static void run(float2 *x) {
        constexpr float c[3] = {6.234898019e-01f, -2.225209340e-01f, -9.009688679e-01f};
        constexpr float sn[3] = {7.818314825e-01f, 9.749279122e-01f, 4.338837391e-01f};
        dft_odd<7, INV>(x, c, sn);
    }
};

// base + so, so uniform, kept in scalar registers: an access at it plus a
// 32-bit lane offset then takes no address arithmetic per lane (the empty
// asm keeps the compiler from adding the lane offset first)
typedef __attribute__((address_space(1))) uint8_t glb8;
__device__ __forceinline__ glb8 *global(const void *p) { return (glb8 *)(uintptr_t)p; }
__device__ __forceinline__ glb8 *scalar_ptr(const void *base, int64_t bytes) {
    glb8 *b = global(base) + bytes;
    __asm__("" : "+s"(b));
    return b;
}
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <class V>
__device__ __forceinline__ V ld_s(const void *base, int64_t bytes, uint32_t lane_bytes) {
    return *(__attribute__((address_space(1))) const V *)(scalar_ptr(base, bytes) + (size_t)lane_bytes);
}
template <class I, class V>
__device__ __forceinline__ void st_s(glb8 *b, I lane_bytes, V v) {
    *(__attribute__((address_space(1))) V *)(b + (size_t)lane_bytes) = v;
}
// Neighbouring elements v of a row (kDstPanels: a pair) to o[at]: vec as one
// store, else each in its own, the second one only if it is there.
template <int DST, class I>
__device__ __forceinline__ void store_pair(glb8 *o, I at, bool vec, bool second, float2 v) {
    const I x = at * (DST == kDstPanels ? 8 : DST == HH_F32 ? 4 : 2);
    if constexpr (DST == kDstPanels) {
        st_s(o, x, f32x2{v.x, v.y});
    } else if constexpr (DST == HH_F32) {
        if (vec) {
            st_s(o, x, f32x2{v.x, v.y});
        } else {
            st_s(o, x, v.x);
            if (second) st_s(o, x + 4u, v.y);
        }
    } else {
        uint32_t b;
        if constexpr (DST == HH_BF16) {
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            b = __builtin_bit_cast(uint32_t, bf16x2{(__bf16)v.x, (__bf16)v.y});
        } else {
            b = f32_to_f16_bits(v.x) | (f32_to_f16_bits(v.y) << 16);
        }
        if (vec) {
            st_s(o, x, b);
        } else {
            st_s(o, x, (uint16_t)b);
            if (second) st_s(o, x + 2u, (uint16_t)(b >> 16));
        }
    }
}
// t[so + idx], so uniform
__device__ __forceinline__ float2 tab_at(const float2 *t, uint32_t so, uint32_t idx) {
    const f32x2 v = ld_s<f32x2>(t, 8ll * so, 8u * idx);
    return make_float2(v.x, v.y);
}
// x mod p for x < 2^22: (x + 1/2) / p lies at least 1/(2p) from an integer,
// more than the float product's error
__device__ __forceinline__ uint32_t mod_p(uint32_t x, uint32_t p, float invp) {
    return x - (uint32_t)(((float)x + 0.5f) * invp) * p;
}
// x / p for a multiple x of p, as above
__device__ __forceinline__ uint32_t mod_div(uint32_t x, uint32_t p, float invp) {
    return (uint32_t)(((float)x + 0.5f) * invp);
}
// LDS slot of point x of pair pr
__device__ __forceinline__ uint32_t slot(const Lines &A, uint32_t x, uint32_t pr) {
    return ((x + (x >> A.psh)) << A.pcs) + pr;
}
// the line element at point t of the reordered sequence
__device__ __forceinline__ uint32_t element_of(uint32_t t, uint32_t N) { return 2 * t < N ? 2 * t : 2 * N - 1 - 2 * t; }

// Makes a pass's index base unknown to the compiler, which otherwise hoists
// every radix's addresses out of the loop over the passes and spills.
__device__ __forceinline__ void keep_here(uint32_t &T, uint32_t &tid, uint32_t &nb) {
    __asm__("" : "+s"(T), "+v"(tid), "+s"(nb));
}

// One Stockham pass of radix R, p = the product of the earlier radices:
// butterfly i (of N / R, times the pairs) takes points i + j N/R, multiplies
// point j by w_N^(+-j k N/(p R)) with k = i mod p, transforms, and writes
// output j to (i - k) R + k + j p.  All inputs are read before the barrier,
// so the pass runs in place.  With LDF a first pass takes its points from
// ld(i, pair, x), with STF a last one (p = N / R, i = k) gives its outputs to
// st(i, pair, x), in place of the LDS.
// The slots step linearly in j: without padding always; with psh = 4 (N a
// multiple of 256, first radix 16) N/R and, past the first pass, p are
// multiples of 16, and the first pass's outputs stay inside 16 points.
template <int R, bool INV, bool LDF, bool STF, class LD, class ST>
__device__ __forceinline__ void fft_pass(float2 *buf, const Lines &A, uint32_t p, const float2 *__restrict__ ptab,
                                         LD ld, ST st) {
    constexpr int MAXB = ((int)kPerThread + R - 1) / R;
    // the twiddles are loaded with the pass's inputs, before the barrier,
    // where the registers allow; the first pass (p = 1) has none
    constexpr bool kPre = MAXB * (R - 1) <= 16;
    uint32_t T = blockDim.x, tid = threadIdx.x, nb = A.N / R;
    keep_here(T, tid, nb);
    const uint32_t nbt = nb << A.pcs, pm = (1u << A.pcs) - 1u;
    const bool tw = !LDF && p > 1;
    const float invp = 1.0f / (float)p;
    float2 x[MAXB][R];
    float2 w[kPre ? MAXB : 1][R - 1];
    const uint32_t rstep = (nb + (nb >> A.psh)) << A.pcs;
#pragma unroll
    for (int b = 0; b < MAXB; b++) {
        const uint32_t g = tid + b * T;
        if (g < nbt) {
            const uint32_t i = g >> A.pcs, pr = g & pm;
            if constexpr (LDF) {
                ld(i, pr, x[b]);
            } else {
                const uint32_t s = slot(A, i, pr);
#pragma unroll
                for (int j = 0; j < R; j++) x[b][j] = buf[s + j * rstep];
            }
            if (kPre && tw) {
                const uint32_t k = mod_p(i, p, invp);
#pragma unroll
                for (int j = 1; j < R; j++) w[kPre ? b : 0][j - 1] = tab_at(ptab, (j - 1) * p, k);
            }
        }
    }
    if constexpr (!LDF && !STF) __syncthreads();
    const uint32_t wstep = (p + (p >> A.psh)) << A.pcs;
#pragma unroll
    for (int b = 0; b < MAXB; b++) {
        const uint32_t g = tid + b * T;
        if (g < nbt) {
            const uint32_t i = g >> A.pcs, pr = g & pm;
            const uint32_t k = LDF ? 0u : mod_p(i, p, invp);
            if (tw) {
#pragma unroll
                for (int j = 1; j < R; j++) {
                    float2 t = kPre ? w[kPre ? b : 0][j - 1] : tab_at(ptab, (j - 1) * p, k);
                    if (!INV) t.y = -t.y;
                    x[b][j] = cmul(x[b][j], t);
                }
            }
            Dft<R, INV>::run(x[b]);
            const uint32_t base = (i - k) * R + k;
            if constexpr (STF) {
                st(i, pr, x[b]);
            } else {
                const uint32_t s = slot(A, base, pr);
#pragma unroll
                for (int j = 0; j < R; j++) buf[s + j * wstep] = x[b][j];
            }
        }
    }
    if constexpr (!STF) __syncthreads();
}

// A pass of prime radix r > 7 as direct sums (y_q and y_{r-q} share their
// products, see dft_odd): a_m and b_m are formed in place, then each wave
// task sums kQB outputs q for 64 butterflies, the roots of unity scalar.
// With fewer butterflies most of those lanes would idle through 63 steps one
// after the other: there every output pair (q, butterfly) has a thread.  127 x
// 127 85 -> 13 us (the dense products 41), 381^2 107 -> 16 (79), 1016^2 152 ->
// 35 (163).
template <bool INV, int PR>
__device__ __forceinline__ void prime_pass(float2 *buf, const Lines &A, uint32_t r, uint32_t p,
                                           const float2 *__restrict__ ptab, const float2 *__restrict__ rt) {
    uint32_t T = blockDim.x, tid = threadIdx.x, nb = A.N / r;
    keep_here(T, tid, nb);
    const uint32_t lane = tid & 63u, nbt = nb << A.pcs, pm = (1u << A.pcs) - 1u, H = (r - 1u) / 2u;
    const float invp = 1.0f / (float)p;
    const uint32_t rstep = (nb + (nb >> A.psh)) << A.pcs, wstep = (p + (p >> A.psh)) << A.pcs;
    // a_m and b_m of butterfly g
    auto pair_up = [&](uint32_t m, uint32_t g) {
        const uint32_t i = g >> A.pcs, s = slot(A, i, g & pm);
        float2 a = buf[s + m * rstep], b = buf[s + (r - m) * rstep];
        if (p > 1) {
            const uint32_t k = mod_p(i, p, invp);
            float2 ta = tab_at(ptab, 0, (m - 1) * p + k), tb = tab_at(ptab, 0, (r - m - 1) * p + k);
            if (!INV) {
                ta.y = -ta.y;
                tb.y = -tb.y;
            }
            a = cmul(a, ta);
            b = cmul(b, tb);
        }
        buf[s + m * rstep] = cadd(a, b);
        buf[s + (r - m) * rstep] = rot90<INV>(csub(a, b));
    };
    if (PR == kPrimesAny && nbt < kFewButterflies) {
        // a thread per output pair (q, butterfly) instead: the sums over m
        // are the chain that counts
        const uint32_t all = H * nbt;
        const float invn = 1.0f / (float)nbt;
        for (uint32_t e = tid; e < all; e += T) {
            const uint32_t g = mod_p(e, nbt, invn);
            pair_up(mod_div(e - g, nbt, invn) + 1u, g);
        }
        __syncthreads();
        float2 re[kFewPairs], im[kFewPairs], y0[kFewPairs];
#pragma unroll
        for (uint32_t t = 0; t < kFewPairs; t++) {
            const uint32_t e = tid + t * T;
            if (e >= all) continue;
            const uint32_t g = mod_p(e, nbt, invn), q = mod_div(e - g, nbt, invn) + 1u;
            const uint32_t s = slot(A, g >> A.pcs, g & pm);
            re[t] = y0[t] = buf[s];
            im[t] = make_float2(0.0f, 0.0f);
            uint32_t idx = 0;
#pragma unroll 4
            for (uint32_t m = 1; m <= H; m++) {
                const float2 a = buf[s + m * rstep], b = buf[s + (r - m) * rstep];
                idx += q;
                idx = idx >= r ? idx - r : idx;
                const float2 cs = rt[idx];
                y0[t] = cadd(y0[t], a);
                re[t] = make_float2(__builtin_fmaf(cs.x, a.x, re[t].x), __builtin_fmaf(cs.x, a.y, re[t].y));
                im[t] = make_float2(__builtin_fmaf(cs.y, b.x, im[t].x), __builtin_fmaf(cs.y, b.y, im[t].y));
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t t = 0; t < kFewPairs; t++) {
            const uint32_t e = tid + t * T;
            if (e >= all) continue;
            const uint32_t g = mod_p(e, nbt, invn), q = mod_div(e - g, nbt, invn) + 1u;
            const uint32_t i = g >> A.pcs, k = mod_p(i, p, invp), s = slot(A, (i - k) * r + k, g & pm);
            if (q == 1) buf[s] = y0[t];
            buf[s + q * wstep] = cadd(re[t], im[t]);
            buf[s + (r - q) * wstep] = csub(re[t], im[t]);
        }
        __syncthreads();
        return;
    }
    for (uint32_t m = 1; m <= H; m++)
        for (uint32_t g = tid; g < nbt; g += T) pair_up(m, g);
    __syncthreads();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = T >> 6;
    const uint32_t wb = (nbt + 63u) / 64u, nq = (H + kQB - 1u) / kQB;
    float2 re[kMaxTasks][kQB], im[kMaxTasks][kQB], y0[kMaxTasks];
#pragma unroll
    for (uint32_t t = 0; t < kMaxTasks; t++) {
        const uint32_t task = wave + t * nw;
        if (task >= wb * nq) continue;
        const uint32_t qb = task / wb, g = (task - qb * wb) * 64u + lane;
        const uint32_t gc = g < nbt ? g : nbt - 1u;
        const uint32_t s = slot(A, gc >> A.pcs, gc & pm);
        const float2 x0 = buf[s];
        y0[t] = x0;
        uint32_t idx[kQB];
#pragma unroll
        for (uint32_t q = 0; q < kQB; q++) {
            re[t][q] = x0;
            im[t][q] = make_float2(0.0f, 0.0f);
            idx[q] = 0;
        }
        for (uint32_t m = 1; m <= H; m++) {
            const float2 a = buf[s + m * rstep], b = buf[s + (r - m) * rstep];
            y0[t] = cadd(y0[t], a);
#pragma unroll
            for (uint32_t q = 0; q < kQB; q++) {
                // (m (qb kQB + q + 1)) mod r; past H the outputs are not used
                idx[q] += qb * kQB + q + 1u;
                idx[q] = idx[q] >= r ? idx[q] - r : idx[q];
                const float2 cs = rt[idx[q]];
                re[t][q] = make_float2(__builtin_fmaf(cs.x, a.x, re[t][q].x), __builtin_fmaf(cs.x, a.y, re[t][q].y));
                im[t][q] = make_float2(__builtin_fmaf(cs.y, b.x, im[t][q].x), __builtin_fmaf(cs.y, b.y, im[t][q].y));
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t t = 0; t < kMaxTasks; t++) {
        const uint32_t task = wave + t * nw;
        if (task >= wb * nq) continue;
        const uint32_t qb = task / wb, g = (task - qb * wb) * 64u + lane;
        if (g >= nbt) continue;
        const uint32_t i = g >> A.pcs, k = mod_p(i, p, invp);
        const uint32_t s = slot(A, (i - k) * r + k, g & pm);
        if (qb == 0) buf[s] = y0[t];
#pragma unroll
        for (uint32_t q = 0; q < kQB; q++) {
            const uint32_t o = qb * kQB + q + 1u;
            if (o <= H) {
                buf[s + o * wstep] = cadd(re[t][q], im[t][q]);
                buf[s + (r - o) * wstep] = csub(re[t][q], im[t][q]);
            }
        }
    }
    __syncthreads();
}

// 32 bits of the bitmap from bit `b` on (bits past the bitmap's bytes read as
// whatever its last dword holds; no dword without bitmap bytes is read).
__device__ __forceinline__ uint32_t bits32(const uint8_t *bm, uint32_t nbytes, uint64_t b) {
    const uint32_t mis = (uint32_t)((uintptr_t)bm & 3u);
    const uint32_t *base = reinterpret_cast<const uint32_t *>(bm - mis);
    const uint32_t last = (mis + nbytes - 1u) >> 2;
    const uint64_t q = b + 8u * mis;
    const uint32_t d = (uint32_t)(q >> 5), sh = (uint32_t)q & 31u;
    const uint32_t lo = base[d < last ? d : last];
    const uint32_t hi = base[d + 1u < last ? d + 1u : last];
    return __builtin_amdgcn_alignbit(hi, lo, sh);
}

// Set bits per row of each fragment's bitmap (rows of w bits, one after the
// other): one wave per row, fragment blockIdx.y.
struct RowCounts {
    const uint8_t *bitmap[kMaxFrags];
    uint32_t *counts[kMaxFrags];
    uint32_t rows, w, nbytes;
};
__global__ __launch_bounds__(256) void row_counts_kernel(RowCounts P) {
    const uint32_t row = blockIdx.x * 4u + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (row >= P.rows) return;
    const uint8_t *bm = P.bitmap[blockIdx.y];
    const uint64_t b0 = (uint64_t)row * P.w;
    uint32_t c = 0;
    for (uint32_t n = 32u * lane; n < P.w; n += 2048u) {
        uint32_t v = bits32(bm, P.nbytes, b0 + n);
        if (P.w - n < 32u) v &= (1u << (P.w - n)) - 1u;
        c += (uint32_t)__popc(v);
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) c += __shfl_xor(c, d);
    if (lane == 0) P.counts[blockIdx.y][row] = c;
}

// One pass: the transforms of 2 PC lines per workgroup.
template <bool INV, int SRC, int DST, int PR>
__global__ __launch_bounds__(1024) void lines_kernel(Lines A) {
    extern __shared__ float2 buf[];
    const uint32_t N = A.N, T = blockDim.x, tid = threadIdx.x;
    const uint32_t pm = (1u << A.pcs) - 1u;
    uint32_t grp = blockIdx.x;
    if (A.per_xcd) {
        // workgroups go round the 8 XCDs: give each XCD neighbouring columns
        grp = (grp & 7u) * A.per_xcd + (grp >> 3);
        if (grp >= ((A.lines + 2u * pm + 1u) >> (A.pcs + 1u))) return;
    }
    const uint32_t line0 = grp << (A.pcs + 1u);
    const float s1 = sqrtf(2.0f / (float)N), s0 = sqrtf(1.0f / (float)N);

    // Lines l and l + 1 of a thread's pair: the column pass of an inverse
    // reads its columns where the row pass left them, at their points: pair m
    // (elements 2 m and 2 m + 1) at points m and w - 1 - m.  A line past the
    // last is read as the last and not written.
    const uint32_t G = 1u << A.gsh;
    auto line_off = [&](uint32_t pr, uint32_t &second) -> uint32_t {  // in elements, of n = 0
        uint32_t l = line0 + 2u * pr;
        const uint32_t lm = A.lines - 1u;
        if constexpr (SRC == kSrcRows) {
            l = l < lm ? l : lm;
            second = l < lm ? N : 0u;
            return l * N;
        } else if constexpr (INV) {
            l = (l < lm ? l : lm) >> 1;
            second = (lm - 2u * l) << A.gsh;
            return l << A.gsh;
        } else {
            l = l < lm ? l : lm;
            second = l < lm ? G : 0u;
            return l << A.gsh;
        }
    };
    // offset of element n in its line; linear in steps of multiples of G
    auto elem_off = [&](uint32_t n) -> uint32_t {
        if constexpr (SRC == kSrcRows)
            return n;
        else
            return (((n >> A.gsh) * A.ipitch) << A.gsh) + (n & (G - 1u));
    };
    // input element at scalar offset so + lane offset vo (elements; a matrix
    // has fewer than 2^29)
    auto in_at = [&](int32_t so, uint32_t vo) -> float {
        return ld_s<float>(A.in, 4ll * so, 4u * vo);
    };
    // Elements n of a pair of lines to the output at scalar offset so + lane
    // offset vo, in units of a line element (kDstPanels: a pair)
    const bool vec = ((A.lines | (uint32_t)((uintptr_t)A.out >> (DST == HH_F32 ? 2 : 1))) & 1u) == 0;
    auto put2 = [&](int32_t so, uint32_t vo, uint32_t l, float2 v) {
        constexpr int kUnit = DST == kDstPanels ? 8 : DST == HH_F32 ? 4 : 2;
        store_pair<DST>(scalar_ptr(A.out, (int64_t)so * kUnit), vo, vec, l + 1u < A.lines, v);
    };
    // the output's steps: elements of a line, and where pair pr's lines are
    const uint32_t osh = A.pcs + A.msh, part = (grp & ((1u << A.msh) - 1u)) << A.pcs;
    const uint32_t ostep = DST == kDstPanels ? 1u << osh : A.lines;
    const int32_t obase = (int32_t)(DST == kDstPanels ? (((grp >> A.msh) * A.opitch) << osh) + part : line0);
    auto opair = [&](uint32_t pr) -> uint32_t { return DST == kDstPanels ? pr : 2u * pr; };

    // (k, N - k) pairs, k = 0 with N / 2; a thread's are istep apart (a
    // multiple of 16, so LDS slots and panel offsets step linearly)
    const uint32_t nk = (N + 1u) / 2u, i0 = tid >> A.pcs, pr0 = tid & pm, istep = T >> A.pcs;
    const uint32_t sstep = (istep + (istep >> A.psh)) << A.pcs;
    constexpr uint32_t kTasks = kPerThread / 2u;  // of them a thread, at most
    constexpr uint32_t CH = 4;  // inverse: of them loaded together (4096^2 bf16 86 us; eight: 88)
    if constexpr (INV) {
        auto other = [&](uint32_t k) { return k == 0 ? N / 2u : N - k; };
        // Z[k] = s_1/2 w^k ((c1[k] + c2[N-k]) + i (c2[k] - c1[N-k])), w^(N-k) = i conj w^k,
        // from elements k (u) and N - k (v) of the pair of lines, into slots sk and sn
        auto emit = [&](uint32_t k, uint32_t sk, uint32_t sn, float2 w, float2 u, float2 v) {
            if (k == 0) {
                buf[sk] = make_float2(s0 * u.x, s0 * u.y);
                if ((N & 1u) == 0)
                    buf[slot(A, N / 2u, pr0)] = cmul(tab_at(A.w4, N / 2u, 0), make_float2(v.x + v.y, v.y - v.x));
            } else {
                buf[sk] = cmul(w, make_float2(u.x + v.y, u.y - v.x));
                buf[sn] = cmul(make_float2(w.y, w.x), make_float2(v.x + u.y, v.y - u.x));
            }
        };
        // (the mirrored slot of k = 0, N, is only stepped from)
        const uint32_t sk0 = slot(A, i0, pr0), sn0 = slot(A, N - i0, pr0);
        if constexpr (SRC == kSrcFrags) {
            // per fragment: this workgroup's bitmap rows and the rank of each
            // dword's first bit, after the FFT points
            const uint32_t nwd = (N + 31u) / 32u, C = 2u << A.pcs;
            uint32_t *wd = reinterpret_cast<uint32_t *>(buf + slot(A, N - 1u, pm) + 1u);
            uint32_t *wp = wd + C * nwd;
            uint32_t *sm = wp + C * nwd;  // 16 words
            const uint32_t lane = tid & 63u, wave = tid >> 6, nwv = T >> 6;
            const uint32_t nbytes = (uint32_t)(((uint64_t)A.lines * N + 7u) / 8u);
            for (uint32_t f = 0; f < A.nfrag; f++) {
                // set bits of all earlier rows, four of them to a load (one:
                // 16384 rows of 256 91 us in all)
                const uint32_t *cnt = A.counts[f];
                const uint4 *cnt4 = reinterpret_cast<const uint4 *>(cnt);
                uint32_t sum = tid < (line0 & 3u) ? cnt[(line0 & ~3u) + tid] : 0u;
#pragma unroll 4
                for (uint32_t i = tid; i < line0 / 4u; i += T) {
                    const uint4 v = cnt4[i];
                    sum += v.x + v.y + v.z + v.w;
                }
#pragma unroll
                for (int d = 32; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
                if (lane == 0) sm[wave] = sum;
                __syncthreads();
                uint32_t before = 0;
                for (uint32_t i = 0; i < nwv; i++) before += sm[i];
                for (uint32_t l = wave; l < C; l += nwv) {
                    if (line0 + l >= A.lines) {
                        for (uint32_t j = lane; j < nwd; j += 64u) wd[l * nwd + j] = 0u;
                        continue;
                    }
                    uint32_t run = before;
                    for (uint32_t i = 0; i < l; i++) run += cnt[line0 + i];
                    const uint64_t b0 = (uint64_t)(line0 + l) * N;
                    for (uint32_t j0 = 0; j0 < nwd; j0 += 64u) {
                        const uint32_t j = j0 + lane;
                        uint32_t x = 0;
                        if (j < nwd) {
                            x = bits32(A.bitmap[f], nbytes, b0 + 32u * j);
                            if (N - 32u * j < 32u) x &= (1u << (N - 32u * j)) - 1u;
                        }
                        const uint32_t c = (uint32_t)__popc(x);
                        uint32_t incl = c;
#pragma unroll
                        for (int d = 1; d < 64; d <<= 1) {
                            const uint32_t t = __shfl_up(incl, d);
                            if (lane >= (uint32_t)d) incl += t;
                        }
                        if (j < nwd) {
                            wd[l * nwd + j] = x;
                            wp[l * nwd + j] = run + incl - c;
                        }
                        run += __shfl(incl, 63);
                    }
                }
                __syncthreads();
                const uint32_t nc = A.ncoef[f];
                const uint8_t *cb = A.coef[f];
                const bool f32c = A.coef_f32 != 0, aligned = ((uintptr_t)cb & (f32c ? 3u : 1u)) == 0;
                // value number of element n of line l, or ~0
                auto rank = [&](uint32_t l, uint32_t n) -> uint32_t {
                    const uint32_t x = wd[l * nwd + (n >> 5)], bit = n & 31u;
                    const uint32_t rk = wp[l * nwd + (n >> 5)] + (uint32_t)__popc(x & ((1u << bit) - 1u));
                    return ((x >> bit) & 1u) && rk < nc ? rk : ~0u;
                };
                // bits of value rk (value 0 where there is none, not used)
                auto value = [&](uint32_t rk) -> uint32_t {
                    rk = rk == ~0u ? 0u : rk;
                    if (f32c) {
                        if (aligned) return reinterpret_cast<const uint32_t *>(cb)[rk];
                        const uint8_t *q = cb + 4ull * rk;
                        return (uint32_t)q[0] | ((uint32_t)q[1] << 8) | ((uint32_t)q[2] << 16) | ((uint32_t)q[3] << 24);
                    }
                    if (aligned) return reinterpret_cast<const uint16_t *>(cb)[rk];
                    const uint8_t *q = cb + 2ull * rk;
                    return (uint32_t)q[0] | ((uint32_t)q[1] << 8);
                };
                auto pick = [&](uint32_t rk, uint32_t bits, float old) -> float {
                    return rk == ~0u ? old : f32c ? __uint_as_float(bits) : f16_bits_to_f32(bits);
                };
                // the elements so far are kept in the slots of their points
                // until the last fragment
                const bool first = f == 0, last = f + 1u == A.nfrag;
                const uint32_t l = 2u * pr0;
                for (uint32_t c0 = 0; c0 * istep < nk; c0 += CH) {
                    uint32_t rk[CH][4], x[CH][4];
#pragma unroll
                    for (uint32_t c = 0; c < CH; c++) {
                        const uint32_t k = i0 + (c0 + c) * istep;
                        if (k < nk) {
                            const uint32_t o = other(k);
                            rk[c][0] = rank(l, k);
                            rk[c][1] = rank(l + 1u, k);
                            rk[c][2] = rank(l, o);
                            rk[c][3] = rank(l + 1u, o);
                            if (nc > 0) {
#pragma unroll
                                for (int e = 0; e < 4; e++) x[c][e] = value(rk[c][e]);
                            }
                        }
                    }
#pragma unroll
                    for (uint32_t c = 0; c < CH; c++) {
                        const uint32_t k = i0 + (c0 + c) * istep;
                        if (k < nk) {
                            const uint32_t sk = sk0 + (c0 + c) * sstep, sn = sn0 - (c0 + c) * sstep;
                            const uint32_t so = k == 0 ? slot(A, N / 2u, pr0) : sn;
                            float2 u = make_float2(0.0f, 0.0f), v = u;
                            if (!first) {
                                u = buf[sk];
                                v = buf[so];
                            }
                            u = make_float2(pick(rk[c][0], x[c][0], u.x), pick(rk[c][1], x[c][1], u.y));
                            v = make_float2(pick(rk[c][2], x[c][2], v.x), pick(rk[c][3], x[c][3], v.y));
                            if (last) {
                                emit(k, sk, sn, tab_at(A.w4, (c0 + c) * istep, i0), u, v);
                            } else {
                                buf[so] = v;
                                buf[sk] = u;
                            }
                        }
                    }
                }
                __syncthreads();  // the next fragment rewrites wd, wp and sm
            }
        } else {
            uint32_t second;
            const uint32_t lo = line_off(pr0, second);
            const uint32_t vk = lo + elem_off(i0), vn = lo + elem_off(N - i0);
            const uint32_t vh = lo + elem_off(N / 2u);
            const int32_t step = (int32_t)elem_off(istep);
            for (uint32_t c0 = 0; c0 * istep < nk; c0 += CH) {
                float2 u[CH], v[CH], w[CH];
#pragma unroll
                for (uint32_t c = 0; c < CH; c++) {
                    if (i0 + (c0 + c) * istep < nk) {
                        const int32_t so = (int32_t)(c0 + c) * step;
                        u[c] = make_float2(in_at(so, vk), in_at(so, vk + second));
                        if (c == 0 && c0 == 0 && i0 == 0)
                            v[c] = make_float2(in_at(0, vh), in_at(0, vh + second));
                        else
                            v[c] = make_float2(in_at(-so, vn), in_at(-so, vn + second));
                        w[c] = tab_at(A.w4, (c0 + c) * istep, i0);
                    }
                }
#pragma unroll
                for (uint32_t c = 0; c < CH; c++) {
                    const uint32_t k = i0 + (c0 + c) * istep;
                    if (k < nk) emit(k, sk0 + (c0 + c) * sstep, sn0 - (c0 + c) * sstep, w[c], u[c], v[c]);
                }
            }
            __syncthreads();
        }
    }
    // the first pass's points i + j N/16 of the forward transform: elements
    // 2 i + 2 j N/16 for j < 8, 2 N - 1 - 2 i - 2 j N/16 above
    auto load16 = [&](uint32_t i, uint32_t pr, float2 (&x)[16]) {
        uint32_t second;
        const uint32_t lo = line_off(pr, second), nb = N / 16u;
        if (SRC == kSrcRows || ((2u * nb) & (G - 1u)) == 0) {
            const uint32_t ve = lo + elem_off(2u * i), vo = lo + elem_off(2u * (nb - 1u - i) + 1u);
            const int32_t step = (int32_t)elem_off(2u * nb);
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) {
                const int32_t so = (int32_t)(j < 8 ? j : 15u - j) * step;
                const uint32_t vv = j < 8 ? ve : vo;
                x[j] = make_float2(in_at(so, vv), in_at(so, vv + second));
            }
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) {
                const uint32_t vv = lo + elem_off(element_of(i + j * nb, N));
                x[j] = make_float2(in_at(0, vv), in_at(0, vv + second));
            }
        }
    };
    // the last pass's points i + j N/16 of the inverse: panels hold them at
    // their points, a matrix at their elements (as above)
    auto store16 = [&](uint32_t i, uint32_t pr, const float2 (&x)[16]) {
        const uint32_t l = line0 + 2u * pr, nb = N / 16u;
        if constexpr (DST == kDstPanels) {
            const uint32_t vv = i * ostep + pr;
#pragma unroll
            for (uint32_t j = 0; j < 16; j++) put2(obase + (int32_t)(j * nb * ostep), vv, l, x[j]);
        } else {
            if (l >= A.lines) return;
            const uint32_t ve = 2u * i * ostep + 2u * pr, vo = 2u * (nb - 1u - i) * ostep + 2u * pr;
#pragma unroll
            for (uint32_t j = 0; j < 16; j++)
                put2(obase + (int32_t)((j < 8 ? 2u * j * nb : 2u * (15u - j) * nb + 1u) * ostep), j < 8 ? ve : vo, l,
                     x[j]);
        }
    };
    // forward: a first pass of radix 16 reads its points from memory;
    // inverse: a last one writes its points there; else through LDS
    auto radix = [&](uint32_t j) -> uint32_t { return (uint32_t)(A.radix[j >> 3] >> (8u * (j & 7u))) & 0xffu; };
    uint32_t q = 0, p = 1, poff = 0, roff = 0, nq = A.nr;
    if constexpr (!INV) {
        if (nq > 0 && radix(0) == 16) {
            fft_pass<16, INV, true, false>(buf, A, 1u, A.ptab, load16, store16);
            q = 1;
            p = 16;
            poff = 15;
        } else {
            uint32_t second;
            const uint32_t lo = line_off(pr0, second);
            for (uint32_t t = i0; t < N; t += istep) {
                const uint32_t vv = lo + elem_off(element_of(t, N));
                buf[slot(A, t, pr0)] = make_float2(in_at(0, vv), in_at(0, vv + second));
            }
            __syncthreads();
        }
    }
    const bool direct = INV && nq > 0 && radix(nq - 1u) == 16;
    if (direct) nq--;
    for (; q < nq; q++) {
        const uint32_t r = radix(q);
        const float2 *pt = A.ptab + poff;
        switch (r) {
            case 16: fft_pass<16, INV, false, false>(buf, A, p, pt, load16, store16); break;
            case 8: fft_pass<8, INV, false, false>(buf, A, p, pt, load16, store16); break;
            case 4: fft_pass<4, INV, false, false>(buf, A, p, pt, load16, store16); break;
            case 2: fft_pass<2, INV, false, false>(buf, A, p, pt, load16, store16); break;
            case 3: fft_pass<3, INV, false, false>(buf, A, p, pt, load16, store16); break;
            case 5: fft_pass<5, INV, false, false>(buf, A, p, pt, load16, store16); break;
            case 7: fft_pass<7, INV, false, false>(buf, A, p, pt, load16, store16); break;
            default:
                if constexpr (PR != kPrimesNone) prime_pass<INV, PR>(buf, A, r, p, pt, A.rt + roff);
                roff += r;
                break;
        }
        poff += p * (r - 1u);
        p *= r;
    }
    if constexpr (INV) {
        if (direct) {
            fft_pass<16, INV, false, true>(buf, A, p, A.ptab + poff, load16, store16);
        } else {
            const uint32_t l = line0 + 2u * pr0;
            if (DST == kDstPanels || l < A.lines)
                for (uint32_t t = i0; t < N; t += istep)
                    put2(obase, (DST == kDstPanels ? t : element_of(t, N)) * ostep + opair(pr0), l,
                         buf[slot(A, t, pr0)]);
        }
    }
    if constexpr (!INV) {
        // V1 = ((a + c), (b - d)) / 2, V2 = ((b + d), (c - a)) / 2 from Z[k] = (a, b),
        // Z[N-k] = (c, d); X[k] = s Re(conj(w) V), X[N-k] = -s Im(conj(w) V)
        const uint32_t l = line0 + 2u * pr0;
        if (DST != kDstPanels && l >= A.lines) return;
        const uint32_t sk0 = slot(A, i0, pr0), sn0 = slot(A, N - i0, pr0);
        const uint32_t vk = i0 * ostep + opair(pr0), vn = (N - i0) * ostep + opair(pr0);
        float2 w[kTasks];
#pragma unroll
        for (uint32_t c = 0; c < kTasks; c++)
            if (i0 + c * istep < nk) w[c] = tab_at(A.w4, c * istep, i0);
#pragma unroll
        for (uint32_t c = 0; c < kTasks; c++) {
            if (i0 + c * istep >= nk) continue;
            const float2 zk = buf[sk0 + c * sstep];
            const int32_t so = (int32_t)(c * istep * ostep);
            if (c == 0 && i0 == 0) {
                put2(obase, vk, l, make_float2(s0 * zk.x, s0 * zk.y));
                if ((N & 1u) == 0) {
                    const float2 zh = buf[slot(A, N / 2u, pr0)];
                    const float h = s1 * 7.071067812e-01f;
                    put2(obase, N / 2u * ostep + opair(pr0), l, make_float2(h * zh.x, h * zh.y));
                }
            } else {
                const float2 zn = buf[sn0 - c * sstep];
                const float r1 = zk.x + zn.x, i1 = zk.y - zn.y, r2 = zk.y + zn.y, i2 = zn.x - zk.x;
                put2(obase + so, vk, l, make_float2(__builtin_fmaf(w[c].x, r1, w[c].y * i1),
                                                    __builtin_fmaf(w[c].x, r2, w[c].y * i2)));
                put2(obase - so, vn, l, make_float2(__builtin_fmaf(w[c].y, r1, -(w[c].x * i1)),
                                                    __builtin_fmaf(w[c].y, r2, -(w[c].x * i2))));
            }
        }
    }
}

// The columns' panels (groups of 2 << pcs columns, N points each) to the
// row-major result: 64 points of 64 columns per workgroup through LDS, rows
// of 256 or 128 bytes out.  Bound by memory: 14336 x 4096 f32 85 us, 5.5 TB/s
// (the device copy reaches 6.3).
constexpr uint32_t kTileSide = 64, kTileStride = kTileSide + 2;  // even: pairs of columns stay aligned
template <bool INV, int DST>
__global__ __launch_bounds__(256) void untangle_kernel(Untangle U) {
    __shared__ __attribute__((aligned(8))) float tile[kTileSide * kTileStride];
    const uint32_t tid = threadIdx.x, t0 = blockIdx.x * kTileSide, c0 = blockIdx.y * kTileSide;
    const uint32_t pm = (1u << U.pcs) - 1u, pairs = (U.lines + 1u) >> 1;
    constexpr uint32_t kLoads = kTileSide * kTileSide / 2u / 256u;
    f32x2 v[kLoads];
    // 64 points of a group's pairs are contiguous (past the last: the last)
    auto at = [&](uint32_t j, uint32_t &t, uint32_t &pr) {
        const uint32_t e = tid + j * 256u, x = e & ((kTileSide << U.pcs) - 1u);
        pr = ((e >> (6u + U.pcs)) << U.pcs) + (x & pm);
        t = x >> U.pcs;
    };
#pragma unroll
    for (uint32_t j = 0; j < kLoads; j++) {
        uint32_t t, pr;
        at(j, t, pr);
        const uint32_t pair = c0 / 2u + pr < pairs ? c0 / 2u + pr : pairs - 1u, n = t0 + t < U.N ? t0 + t : U.N - 1u;
        v[j] = *(const f32x2 *)(U.in + 2ull * ((((uint64_t)(pair >> U.pcs) * U.N + n) << U.pcs) + (pair & pm)));
    }
#pragma unroll
    for (uint32_t j = 0; j < kLoads; j++) {
        uint32_t t, pr;
        at(j, t, pr);
        *reinterpret_cast<f32x2 *>(&tile[t * kTileStride + 2u * pr]) = v[j];
    }
    __syncthreads();
    const uint32_t c = (tid & 31u) * 2u, l = c0 + c;
    if (l >= U.lines) return;
    const bool vec = ((U.lines | (uint32_t)((uintptr_t)U.out >> (DST == HH_F32 ? 2 : 1))) & 1u) == 0;
#pragma unroll
    for (uint32_t j = 0; j < kTileSide / 8u; j++) {
        const uint32_t t = (tid >> 5) + j * 8u;
        if (t0 + t >= U.N) break;
        const f32x2 r = *reinterpret_cast<const f32x2 *>(&tile[t * kTileStride + c]);
        const uint64_t o = (uint64_t)(INV ? element_of(t0 + t, U.N) : t0 + t) * U.lines + l;
        store_pair<DST>(global(U.out), o, vec, l + 1u < U.lines, make_float2(r.x, r.y));
    }
}

struct LinePlan {
    uint32_t N = 0, nr = 0, psh = 31, roots = 0;
    uint8_t r[16] = {};
};
constexpr uint32_t tab_w4(uint32_t N) { return N; }  // after the pass tables (N - 1 entries, one pad)
constexpr uint32_t tab_rt(uint32_t N) { return N + N / 2u + 1u; }
uint32_t tab_len(const LinePlan &P) { return tab_rt(P.N) + P.roots; }

// Radices of N: a 16 first where there are two or more, then 8, 4 or 2, the
// odd primes, and the other 16s last (the first and the last pass of radix
// 16 read and write memory themselves; with padded LDS slots, N a multiple
// of 256, every pass's p is then 1 or a multiple of 16); false when N is out
// of range or has a prime factor above kMaxPrime.
bool make_line_plan(uint32_t N, LinePlan &P) {
    if (N == 0 || N > kMaxPoints) return false;
    P = LinePlan();
    P.N = N;
    uint32_t n = N, n16 = 0;
    while (n % 16 == 0) n16++, n /= 16;
    if (n16 > 1) P.r[P.nr++] = 16, n16--;
    for (uint32_t f : {8u, 4u, 2u})
        if (n % f == 0) {
            P.r[P.nr++] = (uint8_t)f, n /= f;
            break;
        }
    for (uint32_t f = 3; f <= kMaxPrime; f += 2)
        while (n % f == 0) {
            if (P.nr == 12) return false;
            P.r[P.nr++] = (uint8_t)f, n /= f;
            if (f > 7) P.roots += f;
        }
    if (n != 1) return false;
    while (n16 > 0) P.r[P.nr++] = 16, n16--;
    P.psh = N % 256u == 0 ? 4u : 31u;
    return true;
}

// How a pass splits its lines over workgroups: pairs of lines each (log2),
// threads.
struct Split {
    uint32_t pcs, threads, lds;
    int primes;
};
uint32_t lds_points(uint32_t N, uint32_t psh, uint32_t pcs) { return (N + (psh == 4u ? N / 16u : 0u)) << pcs; }

bool make_split(const LinePlan &P, uint32_t lines, bool frags, uint32_t want_groups, Split &S) {
    uint32_t pcs = 0;
    while (pcs < 3 && (P.N << (pcs + 1)) <= kMaxPoints) pcs++;
    // fewer lines per workgroup until there is one for every CU
    while (pcs > 0 && (lines + (2u << pcs) - 1u) / (2u << pcs) < want_groups) pcs--;
    // and where workgroups that have a CU each would leave a last round of up
    // to three tenths: 5120 x 1536 to bf16 73 -> 64 us (70 on rows and
    // transposes, which took it before), 5120 x 1280 65 -> 54 (63), 2560^2 60
    // -> 44; at half a round 1536 x 6144 loses 2 %, and so do single pairs (8192
    // x 1280 5 %), whose pieces of a row are 8 bytes
    const uint32_t parts = (lines + (2u << pcs) - 1u) / (2u << pcs);
    if (pcs > 1 && lds_points(P.N, P.psh, pcs) * 8u > kMaxLds / 2u && parts > want_groups &&
        10u * parts < 13u * want_groups)
        pcs--;
    const uint32_t pts = P.N << pcs;
    // (threads per pair of lines a multiple of 16, see lines_kernel)
    const uint32_t unit = pcs == 3 ? 128u : 64u;
    uint32_t T = ((pts + kPerThread - 1u) / kPerThread + unit - 1u) / unit * unit;
    S.primes = kPrimesNone;
    for (uint32_t q = 0; q < P.nr; q++) {
        const uint32_t r = P.r[q];
        if (r <= 8 || r == 16) continue;
        const uint32_t nbt = (P.N / r) << pcs, H = (r - 1u) / 2u;
        const uint32_t tasks = (nbt + 63u) / 64u * ((H + kQB - 1u) / kQB);
        const uint32_t few = nbt * H < 1024u ? nbt * H : 1024u;
        const int kind = nbt < kFewButterflies ? kPrimesAny : kPrimesMany;
        S.primes = S.primes < kind ? kind : S.primes;
        const uint32_t need = nbt < kFewButterflies ? few : (tasks + kMaxTasks - 1u) / kMaxTasks * 64u;
        T = T < need ? (need + unit - 1u) / unit * unit : T;
    }
    // More waves than the FFT's radix-16 butterflies need, up to one per 64
    // pairs of points, as long as all workgroups run at once (16 waves to a
    // CU): a small pass is the latency of its loads and stores.  Four times as
    // many: 1024 x 512 inverse to f32 18.0 -> 13.5 us (17.7 on rows and
    // transposes, which took it before), 3072 x 192 20.9 -> 16.1 (20.2), 5120
    // x 64 19.6 -> 16.7 (18.9); twice: 14.9, 17.3, 17.1.
    const uint32_t c = 2u << pcs, groups = (lines + c - 1u) / c;
    const uint32_t per_cu = (groups + want_groups - 1u) / want_groups, fill = (pts / 2u + 63u) / 64u;
    uint32_t waves = 4u * T / 64u < fill ? 4u * T / 64u : fill;
    if (frags) {
        // Placing a fragment's values is a chain of loads, scans and barriers:
        // a wave a line for the bitmap words, up to four.  1024 x 512 (a wave
        // of four lines before) 33 -> 22 us, with eight fragments 117 -> 43
        // (28 and 92 on rows and transposes); 2048^2 43 -> 39, 123 -> 91.
        // Past all running at once they wait for each other: 1536^2 with 16
        // waves 42 us, with 8 34, 16384 x 64 with 16 62, with 4 42; but where
        // the LDS holds one workgroup it gets all 16 (2304^2 with eight
        // fragments 254 -> 192, rows and transposes 249), and two and a half
        // to a CU on average have 8 (2560^2 237 -> 183, 205; with 16 196).
        const uint32_t held = kMaxLds / (lds_points(P.N, P.psh, pcs) * 8u + c * ((P.N + 31u) / 32u) * 8u + 64u);
        uint32_t at_once = per_cu < held ? per_cu : held > 0 ? held : 1u;
        at_once = at_once == 3u ? 2u : at_once;
        waves = fill < c ? c : fill < 4u * c ? fill : 4u * c;
        waves = waves < 16u / at_once ? waves : 16u / at_once;
    } else {
        waves = waves < 16u / per_cu ? waves : 16u / per_cu;
    }
    T = T < 64u * waves ? 64u * waves / unit * unit : T;
    if (T > 1024u) return false;
    S.pcs = pcs;
    S.threads = T;
    S.lds = lds_points(P.N, P.psh, pcs) * 8u;
    if (frags) S.lds += (2u << pcs) * ((P.N + 31u) / 32u) * 8u + 64u;
    return S.lds <= kMaxLds;
}

struct LineTabArgs {
    uint32_t N, nr, roots;
    uint8_t r[16];
};
__global__ __launch_bounds__(256) void lines_tables_kernel(float2 *__restrict__ tab, LineTabArgs P) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, N = P.N;
    if (i >= tab_rt(N) + P.roots) return;
    double s = 0.0, c = 1.0;
    if (i < N) {
        uint32_t p = 1, off = 0;
        for (uint32_t q = 0; q < P.nr; q++) {
            const uint32_t R = P.r[q], n = p * (R - 1u);
            if (i < off + n) {
                const uint32_t j = (i - off) / p + 1u, k = (i - off) % p;
                sincospi(2.0 * (double)(j * k) / (double)(p * R), &s, &c);
                break;
            }
            off += n;
            p *= R;
        }
    } else if (i < tab_rt(N)) {
        sincospi((double)(i - N) / (2.0 * (double)N), &s, &c);
        const double h = 0.5 * sqrt(2.0 / (double)N);
        s *= h;
        c *= h;
    } else {
        uint32_t o = i - tab_rt(N);
        for (uint32_t q = 0; q < P.nr; q++) {
            if (P.r[q] <= 8 || P.r[q] == 16) continue;
            if (o < P.r[q]) {
                sincospi(2.0 * (double)o / (double)P.r[q], &s, &c);
                break;
            }
            o -= P.r[q];
        }
    }
    tab[i] = make_float2((float)c, (float)s);
}

// The context's twiddle tables for length N (kLineTabs kept, the least
// recently used replaced).
int32_t tables_for(hh_context *ctx, const LinePlan &P, hipStream_t s, const float2 **out) {
    hh_context::FftTables *v = &ctx->line_tab[0];
    for (hh_context::FftTables &t : ctx->line_tab) {
        if (t.tab && t.n == P.N) {
            t.stamp = ++ctx->dct_stamp;
            *out = reinterpret_cast<const float2 *>(t.tab);
            return HH_OK;
        }
        if (v->tab && (!t.tab || t.stamp < v->stamp)) v = &t;
    }
    if (v->tab) {
        // the stream may still read the old table: wait before freeing
        hipError_t e = hipStreamSynchronize(s);
        if (e == hipSuccess) e = hipFree(v->tab);
        v->tab = nullptr;
        v->n = 0;
        if (e != hipSuccess) return from_hip(e);
    }
    const uint32_t n = tab_len(P);
    hipError_t e = hipMalloc(&v->tab, (size_t)n * sizeof(float2));
    if (e != hipSuccess) {
        v->tab = nullptr;
        return from_hip(e);
    }
    LineTabArgs TP;
    TP.N = P.N;
    TP.nr = P.nr;
    TP.roots = P.roots;
    for (int q = 0; q < 16; q++) TP.r[q] = P.r[q];
    hipLaunchKernelGGL(lines_tables_kernel, dim3((n + 255) / 256), dim3(256), 0, s,
                       reinterpret_cast<float2 *>(v->tab), TP);
    e = hipGetLastError();
    if (e != hipSuccess) return from_hip(e);
    v->n = P.N;  // found from here on
    v->stamp = ++ctx->dct_stamp;
    *out = reinterpret_cast<const float2 *>(v->tab);
    return HH_OK;
}

void fill(Lines &A, const LinePlan &P, const Split &S, uint32_t lines, const float2 *tab) {
    A.ptab = tab;
    A.w4 = tab + tab_w4(P.N);
    A.rt = tab + tab_rt(P.N);
    A.N = P.N;
    A.lines = lines;
    A.gsh = 0;
    A.pcs = S.pcs;
    A.psh = P.psh;
    A.per_xcd = 0;
    A.msh = 0;
    A.ipitch = lines;
    A.opitch = P.N;
    A.nr = P.nr;
    A.radix[0] = A.radix[1] = 0;
    for (uint32_t q = 0; q < P.nr; q++) A.radix[q >> 3] |= (uint64_t)P.r[q] << (8u * (q & 7u));
    A.nfrag = 0;
    A.coef_f32 = 0;
}

template <bool INV, int SRC, int DST, int PR>
hipError_t launch_lines_pr(const Lines &A, const Split &S, uint32_t grid, hipStream_t s) {
    hipError_t e = hipFuncSetAttribute((const void *)lines_kernel<INV, SRC, DST, PR>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)S.lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((lines_kernel<INV, SRC, DST, PR>), dim3(grid), dim3(S.threads), S.lds, s, A);
    return hipGetLastError();
}
template <bool INV, int SRC, int DST>
hipError_t launch_lines(const Lines &A, const Split &S, uint32_t grid, hipStream_t s) {
    switch (S.primes) {
        case kPrimesNone: return launch_lines_pr<INV, SRC, DST, kPrimesNone>(A, S, grid, s);
        case kPrimesMany: return launch_lines_pr<INV, SRC, DST, kPrimesMany>(A, S, grid, s);
        default: return launch_lines_pr<INV, SRC, DST, kPrimesAny>(A, S, grid, s);
    }
}

// Whether the columns go to the result by way of panels of their own and
// untangle_kernel.  A workgroup of two columns (more than 8192 rows) writes 8
// or 4 bytes of a row: 14336 x 4096 forward 394 us for that pass, against 184
// to panels (241 before panel_share) and 85 for the tiles; inverse, whole, 489 -> 450 (bf16 437 -> 424).
// Four columns gain nothing (8192 x 4096 232 -> 265), nor do lengths with a
// prime pass, whose workgroups don't write all at once (11008 x 4096 bf16 498
// -> 523).
bool through_panels(const LinePlan &Ph) { return Ph.N > kMaxPoints / 2u && Ph.roots == 0; }

// log2 of the row workgroups that share a panel.  A column workgroup reads
// pieces of 2 PC columns x G rows; below a line of memory (128 bytes) two
// share: 4096 x 14336 bf16 375 -> 353 us, 8192^2 459 -> 437 (four: 378, 479).
// Before untangle_kernel 256 bytes pay, four at most: 14336 x 4096 485 -> 458
// (two) -> 445 us, 12288 x 3072 334 -> 301 -> 293; eight no more.  Not for
// f32 results whose rows are a multiple of 32 KiB apart: pieces of 64 bytes
// are faster beside the columns' stores, 8192^2 546 -> 518 us (518 on rows and
// transposes, which took it before), 7168 x 8192 434 -> 418, 4608 x 8192 320
// -> 291, 4096 x 16384 443 -> 424 (others lose: 8064^2
// 525 -> 546, 7168^2 354 -> 379; with a prime pass, 7936 x 8192, 541 -> 559;
// pieces of 32 bytes, 5120 x 16384, 616 -> 642).
uint32_t panel_share(bool inverse, int32_t dtype, const LinePlan &Pw, const LinePlan &Ph, const Split &Sw,
                     const Split &Sh) {
    const bool through = through_panels(Ph);
    const uint32_t piece = 4u + Sw.pcs + Sh.pcs, want = through ? 8u : 7u, most = through ? 2u : 1u;
    if (inverse && dtype == HH_F32 && piece == 6u && Pw.N % 8192u == 0 && Ph.roots == 0) return 0u;
    return piece >= want ? 0u : want - piece < most ? want - piece : most;
}

// The f32 panels of the rows (whole panels) and those of the columns.
struct Panels {
    uint32_t msh;      // panel_share
    uint32_t pitch;    // points from a panel of the rows to the next
    size_t rows, all;  // floats
};
Panels panels_for(bool inverse, int32_t dtype, const LinePlan &Pw, const LinePlan &Ph, const Split &Sw,
                  const Split &Sh) {
    Panels P;
    P.msh = panel_share(inverse, dtype, Pw, Ph, Sw, Sh);
    const uint32_t g = 2u << (Sw.pcs + P.msh), gc = 2u << Sh.pcs;
    // Large forward transforms leave two points between the panels of the rows:
    // a column reads one piece of each, of all of which the addresses would
    // otherwise differ by a multiple of the line length.  8192^2 575 -> 535 us
    // (552 on rows and transposes, which took it before), 4096 x 16384 492 ->
    // 437, 4096 x 11008 497 -> 478, 6144 x 4096 157 -> 155 (four, eight and
    // twelve points: 546, 534, 532; 448, 461, 448; 472, 477, 476; 159, 158,
    // 158).  Below 2^23 elements the panels stay in the caches (1024 x 4096
    // 29.5 -> 30.4); inverse transforms read two pieces and lose (4096 x 8192
    // 196 -> 202 with eight), as do columns in panels of their own (16384^2).
    P.pitch = Pw.N + (!inverse && !through_panels(Ph) && (uint64_t)Ph.N * Pw.N >= (1u << 23) ? 2u : 0u);
    P.rows = (size_t)((Ph.N + g - 1u) / g * g) * P.pitch;
    P.all = P.rows + (through_panels(Ph) ? (size_t)((Pw.N + gc - 1u) / gc * gc) * Ph.N : 0u);
    return P;
}

// Both passes of an h x w transform: rows (from d_in, or the fragments in F)
// to panels in d_mid, columns to d_out, where they don't lie a line of memory
// side by side by way of panels and tiles.
int32_t two_passes(hh_context *ctx, bool inverse, const float *d_in, const Lines *F, float *d_mid, const LinePlan &Pw,
                   const LinePlan &Ph, const Split &Sw, const Split &Sh, const Panels &M, int32_t dtype, void *d_out,
                   hipStream_t s) {
    const float2 *tw, *th;
    int32_t rc = tables_for(ctx, Pw, s, &tw);
    if (rc == HH_OK) rc = tables_for(ctx, Ph, s, &th);
    if (rc != HH_OK) return rc;
    const uint32_t h = Ph.N, w = Pw.N;
    Lines A;
    if (F) A = *F;
    const uint32_t nfrag = F ? F->nfrag : 0, cf = F ? F->coef_f32 : 0;
    fill(A, Pw, Sw, h, tw);
    A.nfrag = nfrag;
    A.coef_f32 = cf;
    A.in = d_in;
    A.out = d_mid;
    uint32_t ga = (h + (2u << Sw.pcs) - 1u) >> (Sw.pcs + 1u);
    A.msh = M.msh;
    A.opitch = M.pitch;
    if (A.msh) {
        A.per_xcd = (((ga + 7u) / 8u - 1u) | ((1u << A.msh) - 1u)) + 1u;
        ga = 8u * A.per_xcd;
    }
    hipError_t e = F         ? launch_lines<true, kSrcFrags, kDstPanels>(A, Sw, ga, s)
                   : inverse ? launch_lines<true, kSrcRows, kDstPanels>(A, Sw, ga, s)
                             : launch_lines<false, kSrcRows, kDstPanels>(A, Sw, ga, s);
    if (e != hipSuccess) return from_hip(e);
    Lines B;
    fill(B, Ph, Sh, w, th);
    B.in = d_mid;
    B.out = d_out;
    B.gsh = Sw.pcs + A.msh + 1u;
    B.ipitch = M.pitch;
    const uint32_t gb = (w + (2u << Sh.pcs) - 1u) >> (Sh.pcs + 1u);
    B.per_xcd = (gb + 7u) / 8u;
    const uint32_t grid = 8u * B.per_xcd;
    if (!through_panels(Ph)) {
        if (!inverse)
            e = launch_lines<false, kSrcPanels, HH_F32>(B, Sh, grid, s);
        else if (dtype == HH_BF16)
            e = launch_lines<true, kSrcPanels, HH_BF16>(B, Sh, grid, s);
        else if (dtype == HH_F16)
            e = launch_lines<true, kSrcPanels, HH_F16>(B, Sh, grid, s);
        else
            e = launch_lines<true, kSrcPanels, HH_F32>(B, Sh, grid, s);
        return from_hip(e);
    }
    float *cols = d_mid + M.rows;
    B.out = cols;
    e = inverse ? launch_lines<true, kSrcPanels, kDstPanels>(B, Sh, grid, s)
                : launch_lines<false, kSrcPanels, kDstPanels>(B, Sh, grid, s);
    if (e != hipSuccess) return from_hip(e);
    const Untangle U{cols, d_out, h, w, Sh.pcs};
    const dim3 tiles((h + kTileSide - 1u) / kTileSide, (w + kTileSide - 1u) / kTileSide);
    if (!inverse)
        hipLaunchKernelGGL((untangle_kernel<false, HH_F32>), tiles, dim3(256), 0, s, U);
    else if (dtype == HH_BF16)
        hipLaunchKernelGGL((untangle_kernel<true, HH_BF16>), tiles, dim3(256), 0, s, U);
    else if (dtype == HH_F16)
        hipLaunchKernelGGL((untangle_kernel<true, HH_F16>), tiles, dim3(256), 0, s, U);
    else
        hipLaunchKernelGGL((untangle_kernel<true, HH_F32>), tiles, dim3(256), 0, s, U);
    return from_hip(hipGetLastError());
}

bool make_plans(const hh_context *ctx, uint32_t h, uint32_t w, bool frags, LinePlan &Pw, LinePlan &Ph, Split &Sw,
                Split &Sh) {
    const uint32_t want = ctx->num_cus > 0 ? (uint32_t)ctx->num_cus : 256u;
    return make_line_plan(w, Pw) && make_line_plan(h, Ph) && make_split(Pw, h, frags, want, Sw) &&
           make_split(Ph, w, false, want, Sh);
}

int32_t mid_scratch(hh_context *ctx, size_t bytes, hipStream_t s, uint8_t **out) {
    if (ctx->fft_bytes < bytes) {
        if (ctx->d_fft) {
            hipError_t e = hipStreamSynchronize(s);
            if (e == hipSuccess) e = hipFree(ctx->d_fft);
            ctx->d_fft = nullptr;
            ctx->fft_bytes = 0;
            if (e != hipSuccess) return from_hip(e);
        }
        hipError_t e = hipMalloc(&ctx->d_fft, bytes);
        if (e != hipSuccess) {
            ctx->d_fft = nullptr;
            return from_hip(e);
        }
        ctx->fft_bytes = bytes;
    }
    *out = reinterpret_cast<uint8_t *>(ctx->d_fft);
    return HH_OK;
}

}  // namespace

bool lines_supported(const hh_context *ctx, uint32_t h, uint32_t w, bool frags) {
    LinePlan Pw, Ph;
    Split Sw, Sh;
    return make_plans(ctx, h, w, frags, Pw, Ph, Sw, Sh);
}

int32_t dct2d_lines(hh_context *ctx, bool inverse, const float *d_in, uint32_t h, uint32_t w, int32_t out_dtype,
                    void *d_out, hipStream_t s) {
    LinePlan Pw, Ph;
    Split Sw, Sh;
    if (!make_plans(ctx, h, w, false, Pw, Ph, Sw, Sh)) return HH_ERR_UNSUPPORTED;
    const Panels M = panels_for(inverse, out_dtype, Pw, Ph, Sw, Sh);
    uint8_t *mid;
    int32_t rc = mid_scratch(ctx, M.all * sizeof(float), s, &mid);
    if (rc != HH_OK) return rc;
    return two_passes(ctx, inverse, d_in, nullptr, reinterpret_cast<float *>(mid), Pw, Ph, Sw, Sh, M, out_dtype, d_out,
                      s);
}

int32_t hct3_decode_lines(hh_context *ctx, const Hct3Frag *frags, uint32_t nfrags, bool coef_f32, uint32_t h,
                          uint32_t w, int32_t dtype, void *d_out, hipStream_t s) {
    LinePlan Pw, Ph;
    Split Sw, Sh;
    if (nfrags == 0 || nfrags > kMaxFrags || !make_plans(ctx, h, w, true, Pw, Ph, Sw, Sh)) return HH_ERR_UNSUPPORTED;
    const Panels M = panels_for(true, dtype, Pw, Ph, Sw, Sh);
    const size_t mid_bytes = (M.all * sizeof(float) + 255u) & ~(size_t)255u;
    uint8_t *mid;
    const uint32_t pitch = (h + 3u) & ~3u;  // each fragment's counts 16-byte aligned
    int32_t rc = mid_scratch(ctx, mid_bytes + (size_t)nfrags * pitch * 4u, s, &mid);
    if (rc != HH_OK) return rc;
    Lines F;
    RowCounts C;
    F.nfrag = nfrags;
    F.coef_f32 = coef_f32 ? 1u : 0u;
    C.rows = h;
    C.w = w;
    C.nbytes = (uint32_t)(((uint64_t)h * w + 7u) / 8u);
    for (uint32_t f = 0; f < nfrags; f++) {
        uint32_t *cnt = reinterpret_cast<uint32_t *>(mid + mid_bytes) + (size_t)f * pitch;
        C.bitmap[f] = F.bitmap[f] = frags[f].bitmap;
        C.counts[f] = cnt;
        F.counts[f] = cnt;
        F.coef[f] = frags[f].coef;
        F.ncoef[f] = frags[f].ncoef;
    }
    hipLaunchKernelGGL(row_counts_kernel, dim3((h + 3u) / 4u, nfrags), dim3(256), 0, s, C);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return from_hip(e);
    return two_passes(ctx, true, nullptr, &F, reinterpret_cast<float *>(mid), Pw, Ph, Sw, Sh, M, dtype, d_out, s);
}

void release_line_tables(hh_context *ctx) {
    for (hh_context::FftTables &t : ctx->line_tab) {
        if (t.tab) (void)hipFree(t.tab);
        t.tab = nullptr;
        t.n = 0;
    }
}

}  // namespace hh
