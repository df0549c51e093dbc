// Register-blocked power-of-two FFT for gfx950.
//
// A length n = 2^LOGN transform is factored n = N_0 N_1 ... N_{m-1} with
// N_s = 16 for the leading stages and one trailing 2/4/8 stage (E = 16; E = 4
// and E = 8 elements per thread work alike, with N_s = E). Each thread owns
// E elements; a stage is a batch of in-register DFTs of size N_s, and
// the only LDS traffic is one exchange between consecutive stages.
//
// Position of an element: pos = sum_j d_j S_j with S_j = prod_{i>j} N_i. The
// group of stage s (the N_s elements one small DFT combines) is every digit
// but digit s: pos = high*N_s*S_s + v*S_s + low, g = high*S_s + low; thread
// th handles groups g = th*G_s + q, G_s = E/N_s.
//
// Forward: natural-order input, output in digit-reversed order: the value at
// pos is X[k], k = sum_j d_j P_j with P_j = prod_{i<j} N_i. Inverse: consumes
// the digit-reversed order and returns natural order. Forward stage m-1 and
// inverse stage m-1 share their grouping, so a spectral multiply between them
// needs no exchange.
//
// FP64: stage s of the forward is the DFT over digit s of inputs times w^v, v
// the digit and w = W_n^{S_s k'}, k' the part of k known so far (sum_{j<s} d_j
// P_j); stage s of the inverse, s = m-1 .. 0, takes conj(w)^v, w = W_{N_s
// S_s}^{low}. Both directions meet their twiddles on the inputs of a DFT, where
// they cost no operation of their own (dft_tw).
// FP32: the forward multiplies the outputs of stage s < m-1 by
// W_{N_s S_s}^{v*low}, the inverse its inputs by the conjugates.
#pragma once

#include "common.hpp"

#include <type_traits>

namespace aspher {
namespace rb {

// cos(pi j / 16), j = 0..8
__device__ constexpr double kCos16[9] = {
    1.0,
    0.98078528040323044912618223613423903697,
    0.92387953251128675612818318939678828683,
    0.83146961230254523707878837761790575673,
    0.70710678118654752440084436210484903928,
    0.55557023301960222474283081394853287438,
    0.38268343236508977172845998403039886676,
    0.19509032201612826784828486847702224093,
    0.0};

__device__ __forceinline__ constexpr double cospi16(int j) {
    j = ((j % 32) + 32) % 32;
    if (j > 16) j = 32 - j;
    return (j <= 8) ? kCos16[j] : -kCos16[16 - j];
}
__device__ __forceinline__ constexpr double sinpi16(int j) { return cospi16(j - 8); }

template <typename T, bool INV>
__device__ __forceinline__ cx<T> rot90(cx<T> a) {
    return INV ? cx<T>{-a.im, a.re} : cx<T>{a.im, -a.re};
}

// a * W_32^j (forward: exp(-2 pi i j/32); inverse: conjugate). j must fold
// to a constant after unrolling.
template <typename T, bool INV>
__device__ __forceinline__ cx<T> w32(cx<T> a, int j) {
    j = ((j % 32) + 32) % 32;
    if (j == 0) return a;
    if (j == 8) return rot90<T, INV>(a);
    if (j == 16) return cx<T>{-a.re, -a.im};
    if (j == 24) return rot90<T, !INV>(a);
    const T c = static_cast<T>(cospi16(j)), s = static_cast<T>(sinpi16(j));
    return INV ? cx<T>{a.re * c - a.im * s, a.re * s + a.im * c}
               : cx<T>{a.re * c + a.im * s, a.im * c - a.re * s};
}

template <typename T, bool INV>
__device__ __forceinline__ void dft2(cx<T>* a) {
    const cx<T> t = a[0];
    a[0] = t + a[1];
    a[1] = t - a[1];
}

template <typename T, bool INV>
__device__ __forceinline__ void dft4(cx<T>* a) {
    const cx<T> s0 = a[0] + a[2], d0 = a[0] - a[2];
    const cx<T> s1 = a[1] + a[3], d1 = rot90<T, INV>(a[1] - a[3]);
    a[0] = s0 + s1;
    a[2] = s0 - s1;
    a[1] = d0 + d1;
    a[3] = d0 - d1;
}

template <typename T, bool INV>
__device__ __forceinline__ void dft8(cx<T>* a) {
    cx<T> e[4] = {a[0], a[2], a[4], a[6]};
    cx<T> o[4] = {a[1], a[3], a[5], a[7]};
    dft4<T, INV>(e);
    dft4<T, INV>(o);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const cx<T> t = w32<T, INV>(o[k], 4 * k);
        a[k] = e[k] + t;
        a[k + 4] = e[k] - t;
    }
}

// 16-point DFT as 4 x 4 (decimation in frequency), natural order in and out.
template <typename T, bool INV>
__device__ __forceinline__ void dft16(cx<T>* a) {
    cx<T> b[16];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        cx<T> t[4] = {a[n2], a[4 + n2], a[8 + n2], a[12 + n2]};
        dft4<T, INV>(t);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) b[4 * k1 + n2] = w32<T, INV>(t[k1], 2 * k1 * n2);
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        cx<T> t[4] = {b[4 * k1], b[4 * k1 + 1], b[4 * k1 + 2], b[4 * k1 + 3]};
        dft4<T, INV>(t);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) a[k1 + 4 * k2] = t[k2];
    }
}

// dft16 with a[8..15] == 0 (the zero-padded half of a free-space
// transform): the first 4-point pass sees two zero inputs.
template <typename T, bool INV>
__device__ __forceinline__ void dft16_zin(cx<T>* a) {
    cx<T> b[16];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        const cx<T> x0 = a[n2], x1 = a[4 + n2];
        const cx<T> r1 = rot90<T, INV>(x1);
        const cx<T> t[4] = {x0 + x1, x0 + r1, x0 - x1, x0 - r1};
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) b[4 * k1 + n2] = w32<T, INV>(t[k1], 2 * k1 * n2);
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        cx<T> t[4] = {b[4 * k1], b[4 * k1 + 1], b[4 * k1 + 2], b[4 * k1 + 3]};
        dft4<T, INV>(t);
#pragma unroll
        for (int k2 = 0; k2 < 4; ++k2) a[k1 + 4 * k2] = t[k2];
    }
}

// dft16 computing only the outputs a[0..7] (the half of a free-space
// transform that is kept); a[8..15] are left unspecified.
template <typename T, bool INV>
__device__ __forceinline__ void dft16_hout(cx<T>* a) {
    cx<T> b[16];
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) {
        cx<T> t[4] = {a[n2], a[4 + n2], a[8 + n2], a[12 + n2]};
        dft4<T, INV>(t);
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) b[4 * k1 + n2] = w32<T, INV>(t[k1], 2 * k1 * n2);
    }
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        const cx<T> s0 = b[4 * k1] + b[4 * k1 + 2], d0 = b[4 * k1] - b[4 * k1 + 2];
        const cx<T> s1 = b[4 * k1 + 1] + b[4 * k1 + 3];
        const cx<T> d1 = rot90<T, INV>(b[4 * k1 + 1] - b[4 * k1 + 3]);
        a[k1] = s0 + s1;
        a[k1 + 4] = d0 + d1;
    }
}

// The same for radix 4 and 8: a[R/2 ..] == 0, resp. only a[0 .. R/2) wanted.
template <typename T, int R, bool INV>
__device__ __forceinline__ void dft_zin(cx<T>* a) {
    static_assert(R == 4 || R == 8 || R == 16, "pruned radices");
    if constexpr (R == 4) {
        const cx<T> x0 = a[0], x1 = a[1], r1 = rot90<T, INV>(x1);
        a[0] = x0 + x1;
        a[1] = x0 + r1;
        a[2] = x0 - x1;
        a[3] = x0 - r1;
    } else if constexpr (R == 8) {
        // even inputs a0, a2 and odd inputs a1, a3 of a radix-8 transform
        cx<T> e[4] = {a[0], a[2], {T(0), T(0)}, {T(0), T(0)}};
        cx<T> o[4] = {a[1], a[3], {T(0), T(0)}, {T(0), T(0)}};
        dft_zin<T, 4, INV>(e);
        dft_zin<T, 4, INV>(o);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const cx<T> t = w32<T, INV>(o[k], 4 * k);
            a[k] = e[k] + t;
            a[k + 4] = e[k] - t;
        }
    } else {
        dft16_zin<T, INV>(a);
    }
}
template <typename T, int R, bool INV>
__device__ __forceinline__ void dft_hout(cx<T>* a) {
    static_assert(R == 4 || R == 8 || R == 16, "pruned radices");
    if constexpr (R == 4) {
        const cx<T> s0 = a[0] + a[2], d0 = a[0] - a[2];
        const cx<T> s1 = a[1] + a[3], d1 = rot90<T, INV>(a[1] - a[3]);
        a[0] = s0 + s1;
        a[1] = d0 + d1;
    } else if constexpr (R == 8) {
        cx<T> e[4] = {a[0], a[2], a[4], a[6]};
        cx<T> o[4] = {a[1], a[3], a[5], a[7]};
        dft4<T, INV>(e);
        dft4<T, INV>(o);
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = e[k] + w32<T, INV>(o[k], 4 * k);
    } else {
        dft16_hout<T, INV>(a);
    }
}

template <typename T, int R, bool INV>
__device__ __forceinline__ void dft(cx<T>* a) {
    if constexpr (R == 1) {
    } else if constexpr (R == 2) dft2<T, INV>(a);
    else if constexpr (R == 4) dft4<T, INV>(a);
    else if constexpr (R == 8) dft8<T, INV>(a);
    else dft16<T, INV>(a);
}

// LE: log2 of the elements per thread, which is also the largest radix.
// ILV: the transforms of a workgroup interleave across its lanes (columns);
// else each takes consecutive lanes (rows).
template <int LOGN_, int LE_ = 4, bool ILV_ = true>
struct Shape {
    static constexpr int LOGN = LOGN_, LE = LE_;
    static constexpr bool ILV = ILV_;
    static_assert(LE >= 2 && LE <= 4 && LOGN >= LE && LOGN <= 13,
                  "register-blocked sizes up to 8192, 4 to 16 elements per thread");
    static constexpr int n = 1 << LOGN;
    static constexpr int E = 1 << LE;            // elements per thread
    static constexpr int A = LOGN / LE;
    static constexpr int RL = LOGN % LE;
    static constexpr int m = A + (RL ? 1 : 0);
    static constexpr int threads = n / E;
    static __host__ __device__ constexpr int N(int s) { return s < A ? E : (1 << RL); }
    static __host__ __device__ constexpr int S(int s) {
        int p = 1;
        for (int j = s + 1; j < m; ++j) p *= N(j);
        return p;
    }
    static __host__ __device__ constexpr int P(int s) {
        int p = 1;
        for (int j = 0; j < s; ++j) p *= N(j);
        return p;
    }
    static __host__ __device__ constexpr int G(int s) { return E / N(s); }
    // position of element v of group g in stage s
    static __host__ __device__ constexpr int pos(int s, int g, int v) {
        const int Ss = S(s), Ns = N(s);
        return (g / Ss) * Ns * Ss + v * Ss + (g % Ss);
    }
    // frequency index of a digit-reversed position
    static __host__ __device__ constexpr int kidx(int p) {
        int k = 0;
#pragma unroll
        for (int j = 0; j < m; ++j) k += ((p / S(j)) % N(j)) * P(j);
        return k;
    }
};

// LDS index with a skew of one element every 16. The exchanges read and
// write with lane strides of 1, 16 and 32 elements; with this skew those
// strides map 16 lanes of 8-byte elements (and 8 lanes of 16-byte elements)
// to distinct banks (a skew of one per 32 left two-way conflicts on the
// stride-32 exchanges).
__device__ __forceinline__ int lds_ix(int p) { return p + (p >> 4); }
__host__ __device__ constexpr int lds_len(int n) { return n + (n >> 4) + 1; }

// Element -> slot layouts of LDS buffers. The LDS serves a wave's 4- and
// 8-byte accesses in two halves of 32 lanes, whose slots are conflict-free
// when they differ mod 32, and its 16-byte accesses in four quarters of 16
// lanes, conflict-free when they differ mod 16 (measured: a 2-way conflict
// costs two cycles per access in the first case, four in the second).
// Skew16 (one slot of skew per 16 elements) keeps stride-16 and
// stride-32-pair patterns apart but folds the two ends of a 32-element run
// onto one bank; Skew32x2 (two slots per 32) keeps runs of 32 and the
// stride-32 pairs apart. Both fit in lds_len(n) slots.
struct Skew16 {
    static __host__ __device__ constexpr int ix(int p) { return p + (p >> 4); }
};
struct Skew32x2 {
    static __host__ __device__ constexpr int ix(int p) { return p + 2 * (p >> 5); }
};

// FP32: twiddles W^{v*idx}, v = 0..N-1, applied to a group from one FP64 table
// read w = tw[idx] (tw[t] = exp(-2 pi i t/len)).
// Radix 16: w, w^2, w^4, w^8 by FP64 squaring, rounded once to FP32; the
// other powers are FP32 products of at most three of those (<= 4 roundings,
// ~2.5e-7 relative, the accuracy of an FP32 twiddle table). Smaller radices:
// a running FP64 product, rounded once (FP64 data: every power from the table). One table read per group measured faster than reading every power
// (the table reads, not the arithmetic, bound the stage).
// FP32 twiddle powers of one radix-16 group (f[v] = W^{v idx}, f[0]
// unused), formed by a forward stage and reused, conjugated, by the same
// stage of the inverse, which would otherwise form the powers of the
// conjugated table value again (the same values in exact arithmetic; the
// compiled sequences differ in FMA contraction, so results move at the
// FP32 rounding level: 1.1e-7 relative on a 4096^2 free-space matvec).
struct TwKeep {
    cx<float> f[16];
};

// KEEP: 0 = form the powers; 1 = form them and keep them in *keep
// (forward); 2 = apply the conjugates of *keep (inverse, same group)
template <typename T, int NS, bool INV, int KEEP = 0>
__device__ __forceinline__ void twiddle_group(cx<T>* a, const cx<double>* __restrict__ tw,
                                              int idx, int /*tmask*/, TwKeep* keep = nullptr) {
    if (idx == 0) return;
    if constexpr (KEEP == 2) {
        static_assert(std::is_same_v<T, float> && NS == 16, "kept powers: FP32 radix 16");
#pragma unroll
        for (int v = 1; v < 16; ++v) a[v] = a[v] * cx<float>{keep->f[v].re, -keep->f[v].im};
    } else if constexpr (NS == 16) {
        cx<double> w = tw[idx];
        if (INV) w.im = -w.im;
        const cx<double> w2 = w * w, w4 = w2 * w2, w8 = w4 * w4;
        auto f32 = [](cx<double> z) { return cx<float>{(float)z.re, (float)z.im}; };
        cx<float> f[16];
        f[1] = f32(w);
        f[2] = f32(w2);
        f[4] = f32(w4);
        f[8] = f32(w8);
        f[3] = f[2] * f[1];
        f[5] = f[4] * f[1];
        f[6] = f[4] * f[2];
        f[7] = f[4] * f[3];
#pragma unroll
        for (int v = 9; v < 16; ++v) f[v] = f[8] * f[v - 8];
        if constexpr (KEEP == 1) {
#pragma unroll
            for (int v = 1; v < 16; ++v) keep->f[v] = f[v];
        }
#pragma unroll
        for (int v = 1; v < 16; ++v) a[v] = a[v] * f[v];
    } else {
        static_assert(KEEP == 0, "kept powers: FP32 radix 16");
        cx<double> w = tw[idx];
        if (INV) w.im = -w.im;
        cx<double> wv = w;
#pragma unroll
        for (int v = 1; v < NS; ++v) {
            if constexpr (sizeof(T) == 8) {
                wv = tw[v * idx];
                if (INV) wv.im = -wv.im;
            } else if (v > 1) wv = wv * w;
            a[v] = a[v] * cx<T>{static_cast<T>(wv.re), static_cast<T>(wv.im)};
        }
    }
}

// exp(-2 pi i v/32), v = 0..15: the twiddles of a radix-16 stage of stride 2
// (followed by a radix-2 stage), whose groups take either these or ones.
constexpr double kW32re[16] = {
    1.0, 0.98078528040323044913, 0.92387953251128675613, 0.83146961230254523708,
    0.7071067811865475244, 0.55557023301960222474, 0.38268343236508977173,
    0.19509032201612826785, 0.0, -0.19509032201612826785, -0.38268343236508977173,
    -0.55557023301960222474, -0.7071067811865475244, -0.83146961230254523708,
    -0.92387953251128675613, -0.98078528040323044913};
constexpr double kW32im[16] = {
    0.0, -0.19509032201612826785, -0.38268343236508977173, -0.55557023301960222474,
    -0.7071067811865475244, -0.83146961230254523708, -0.92387953251128675613,
    -0.98078528040323044913, -1.0, -0.98078528040323044913, -0.92387953251128675613,
    -0.83146961230254523708, -0.7071067811865475244, -0.55557023301960222474,
    -0.38268343236508977173, -0.19509032201612826785};

template <typename T, bool INV>
__device__ __forceinline__ void twiddle_w32(cx<T>* a, int low) {
    if (low == 0) return;
#pragma unroll
    for (int v = 1; v < 16; ++v) {
        const cx<T> w = {static_cast<T>(kW32re[v]),
                         static_cast<T>(INV ? -kW32im[v] : kW32im[v])};
        a[v] = a[v] * w;
    }
}

// FP32: stage s of the forward (INV=false, DFT then twiddle) or inverse
// (INV=true, twiddle then DFT) transform on the registers of thread th. PR (stage 0
// only, where every thread holds one group of 16 at positions v*S_0 + th):
// 1 = inputs v >= 8 are zero, 2 = only outputs v < 8 are needed.
// KS: the stage whose FP32 twiddle powers the forward keeps in *keep and
// the inverse reuses (-1: none; see keep_stage)
template <typename T, typename Sh, int s, bool INV, int PR = 0, int KS = -1>
__device__ __forceinline__ void stage(cx<T>* r, int th, const cx<double>* __restrict__ tw,
                                      int twmul, TwKeep* keep = nullptr) {
    constexpr int Ns = Sh::N(s), Ss = Sh::S(s), Gs = Sh::G(s);
    constexpr int tstep = Sh::n / (Ns * Ss);     // table stride of W_{Ns Ss}
    constexpr int KP = (s == KS) ? (INV ? 2 : 1) : 0;
    static_assert(PR == 0 || (s == 0 && Gs == 1), "pruned stage 0 only");
    static_assert(KP == 0 || (Ns == 16 && Gs == 1 && Ss > 2 && s < Sh::m - 1),
                  "kept powers: a twiddled radix-16 stage with one group per thread");
#pragma unroll
    for (int q = 0; q < Gs; ++q) {
        cx<T>* a = r + q * Ns;
        const int low = (th * Gs + q) % Ss;
        // stride 2: the group's twiddles are W32^v (low = 1) or ones,
        // constants rather than table reads and products
        constexpr bool W32 = (Ns == 16 && Ss == 2);
        if constexpr (INV) {
            if constexpr (s < Sh::m - 1) {
                if constexpr (W32) twiddle_w32<T, true>(a, low);
                else twiddle_group<T, Ns, true, KP>(a, tw, low * tstep * twmul,
                                                    Sh::n * twmul - 1, keep);
            }
            if constexpr (PR == 2) dft_hout<T, Ns, true>(a);
            else dft<T, Ns, true>(a);
        } else {
            if constexpr (PR == 1) dft_zin<T, Ns, false>(a);
            else dft<T, Ns, false>(a);
            if constexpr (s < Sh::m - 1) {
                if constexpr (W32) twiddle_w32<T, false>(a, low);
                else twiddle_group<T, Ns, false, KP>(a, tw, low * tstep * twmul,
                                                     Sh::n * twmul - 1, keep);
            }
        }
    }
}

// The stage whose twiddle powers a forward-then-inverse kernel can keep:
// stage 1 where it is a generic twiddled radix-16 stage (n >= 1024).
template <typename Sh>
__host__ __device__ constexpr int keep_stage() {
    return (Sh::m >= 3 && Sh::N(1) == 16 && Sh::G(1) == 1 && Sh::S(1) > 2) ? 1 : -1;
}

// FP64: the powers of a stage's twiddle w that its butterflies take: level l of
// the radix-2 network of a DFT of R inputs multiplies by w^{R >> (l+1)} times
// W_{2^(l+1)}^rev, rev < 2^l; rev >= 2^(l-1) is a quarter turn of another one.
// One table read per group, the other powers by squaring.
template <int R, bool INV>
struct TwPowers {
    cx<double> f[R / 2];
    __device__ __forceinline__ explicit TwPowers(cx<double> w) {
        if (INV) w.im = -w.im;
#pragma unroll
        for (int half = R / 4; half >= 1; half >>= 1) {
#pragma unroll
            for (int j = 0; j < half; ++j) f[half + j] = w32<double, INV>(w, (8 / half) * j);
            w = w * w;
        }
        f[0] = w;
    }
    // factor of level l, block rev
    __device__ __forceinline__ cx<double> at(int l, int rev) const {
        if (l == 0) return f[0];
        const int half = 1 << (l - 1);
        return rev < half ? f[half + rev] : rot90<double, INV>(f[half + rev - half]);
    }
};

__host__ __device__ constexpr int bitrev(int x, int bits) {
    int y = 0;
    for (int i = 0; i < bits; ++i) y |= ((x >> i) & 1) << (bits - 1 - i);
    return y;
}

// a[k] = sum_v a[v] w^v W_R^{vk}: radix-2 butterflies a +- wb of six fused
// multiply-adds, u = a + wb and 2a - u (DIRECT, 4-element threads, whose stages are
// many and short: a - wb, one rounding less for two operations more), so neither the twiddles nor the
// rotations inside the DFT are operations of their own: 192 + 28 for R = 16,
// where a 4 x 4 DFT, 15 powers and the products by them take 160 + 56 + 60.
// HOUT: only a[0 .. R/2) is wanted.
// Measured, kernels of a response, twiddled DFTs -> these: free space 2048^2
// 94.0 -> 91.7 us, 4096^2 451 -> 440, 1024^2 39.7 -> 37.1; torus 2048^2 54.4 ->
// 51.1, 4096^2 198 -> 190.
// FP64 only. There its error (torus response, relative, against 80-bit sums) is
// no larger than that of 16-element threads with running powers: 64^2 5.8e-16
// -> 4.4e-16, 512^2 7.9e-16 -> 5.8e-16, 2048^2 1.02e-15 -> 0.96e-15 (free space
// 64^2 2.8e-16 -> 2.7e-16, 128^2 2.03e-16 -> 2.10e-16). In FP32,
// whose powers have one to four roundings, the two more roundings per element
// and level raise the error of a response by 20% (64^2 8.4e-8 -> 1.0e-7, 512^2
// 1.04e-7 -> 1.31e-7).
template <int R, bool INV, bool HOUT, bool DIRECT>
__device__ __forceinline__ void dft_tw(cx<double>* a, const TwPowers<R, INV>& w) {
    constexpr int LR = R == 16 ? 4 : R == 8 ? 3 : R == 4 ? 2 : 1;
    static_assert(R == 1 << LR, "radix 2, 4, 8 or 16");
    cx<double> x[R];
#pragma unroll
    for (int v = 0; v < R; ++v) x[v] = a[v];
#pragma unroll
    for (int l = 0; l < LR; ++l) {
        const int half = R >> (l + 1);
#pragma unroll
        for (int j = 0; j < (1 << l); ++j) {
            const cx<double> f = w.at(l, bitrev(j, l));
#pragma unroll
            for (int i = 0; i < half; ++i) {
                cx<double>&p = x[2 * half * j + i], &q = x[2 * half * j + i + half];
                const cx<double> u = {fma(-f.im, q.im, fma(f.re, q.re, p.re)),
                                      fma(f.im, q.re, fma(f.re, q.im, p.im))};
                if (!HOUT || l + 1 < LR) {
                    if constexpr (DIRECT)
                        q = {fma(f.im, q.im, fma(-f.re, q.re, p.re)),
                             fma(-f.im, q.re, fma(-f.re, q.im, p.im))};
                    else q = {fma(2.0, p.re, -u.re), fma(2.0, p.im, -u.im)};
                }
                p = u;
            }
        }
    }
#pragma unroll
    for (int k = 0; k < (HOUT ? R / 2 : R); ++k) a[k] = x[bitrev(k, LR)];
}

// FP64: the twiddle w of thread th's (first) group in stage s: forward s > 0,
// inverse s < m-1. tw[t] = exp(-2 pi i t/(n*twmul)).
template <typename Sh, int s, bool INV>
__device__ __forceinline__ cx<double> stage_twiddle(int th, const cx<double>* __restrict__ tw,
                                                    int twmul) {
    if constexpr (INV ? s + 1 >= Sh::m : s == 0) {
        return {1.0, 0.0};
    } else if constexpr (INV) {
        return tw[(th % Sh::S(s)) * (Sh::n / (Sh::N(s) * Sh::S(s))) * twmul];
    } else {
        int block = th * Sh::G(s) / Sh::S(s), k = 0;
#pragma unroll
        for (int j = s - 1; j >= 0; --j) {
            k += (block % Sh::N(j)) * Sh::P(j);
            block /= Sh::N(j);
        }
        return tw[k * Sh::S(s) * twmul];
    }
}

// FP64: stage s of the forward or inverse transform, with the thread's twiddle
// w. PR as in `stage`.
template <typename Sh, int s, bool INV, int PR>
__device__ __forceinline__ void stage_fused(cx<double>* r, cx<double> w,
                                            const cx<double>* __restrict__ tw, int twmul) {
    constexpr int Ns = Sh::N(s), Gs = Sh::G(s);
    constexpr bool plain = INV ? s + 1 == Sh::m : s == 0;
    static_assert(PR == 0 || (s == 0 && Gs == 1), "pruned stage 0 only");
    static_assert(PR != 1 || plain, "a pruned input is not twiddled");
#pragma unroll
    for (int q = 0; q < Gs; ++q) {
        cx<double>* a = r + q * Ns;
        if constexpr (!plain) {
            // the groups of a last stage below radix E are neighbours in
            // digit m-2 of the position: w of group q is w W_n^{P q}, a
            // constant for radix 2 (W_{2E}^q), else a uniform read
            cx<double> wq = w;
            if constexpr (Gs > 1 && Ns == 2) wq = w32<double, false>(w, (16 / Sh::E) * q);
            else if (q > 0) wq = w * tw[Sh::P(s > 0 ? s - 1 : 0) * q * twmul];
            dft_tw<Ns, INV, PR == 2, Sh::E == 4>(a, TwPowers<Ns, INV>(wq));
        } else if constexpr (PR == 1) {
            dft_zin<double, Ns, INV>(a);
        } else if constexpr (PR == 2) {
            dft_hout<double, Ns, INV>(a);
        } else {
            dft<double, Ns, INV>(a);
        }
    }
}

// Transforms whose twiddles are fused into the butterflies: FP64, except those of a
// 32-point plan (rows of 16, columns of 32), most of whose twiddles are 1 and cost
// no rounding as factors (torus 32^2: fused 4.1e-16 off, factors from the table
// 2.8e-16, 16-element threads 2.7e-16; 10 us a response either way).
template <typename T, typename Sh>
constexpr bool kFused = sizeof(T) == 8 && Sh::LOGN > 5 - (Sh::ILV ? 0 : 1);

// No-op hook of the exchanges.
struct NoHook {
    __device__ __forceinline__ void operator()() const {}
};

// Positions of the registers of thread th in stage s's grouping, as
// base(th) + off(q, v) = Shape::pos(s, th*G + q, v): a radix-16 stage holds
// one group (off = v*S), the last stage of a radix below 16 holds G groups
// of stride 1 (base = 16 th, off = q*N + v). The skew does not carry
// between the two parts (for Skew16, base mod 16 plus off mod 16 stays below
// 16 in both cases; for Skew32x2, the same mod 32 on the exchanges it is
// used for), so Lay::ix(base + off) = Lay::ix(base) + Lay::ix(off): one
// address per thread and compile-time offsets.
template <typename Sh, int s, typename Lay = Skew16>
struct Grouping {
    static constexpr int N = Sh::N(s), S = Sh::S(s), G = Sh::G(s);
    static_assert(G == 1 || S == 1, "only the last stage holds several groups");
    static __device__ __forceinline__ int base(int th) {
        if constexpr (G == 1) return (th / S) * N * S + th % S;
        else return Sh::E * th;
    }
    static constexpr int off(int q, int v) {
        const int o = G == 1 ? v * S : q * N + v;
        return Lay::ix(o);
    }
};

// Layout of the exchange between stages e and e + 1 (both directions). For
// transforms with whole waves per transform (n >= 1024) every exchange but
// the last takes Skew32x2: its groupings are runs of 32 (or two runs of 16)
// on one side and runs or stride-32 pairs on the other, which Skew16
// conflicts on and Skew32x2 does not, for 4-, 8- and 16-byte elements
// alike; the last exchange's stride-16 side needs Skew16. Both stay linear in the same way as above:
// ix(base + off) = ix(base) + ix(off) for every base and offset used, so
// addressing stays one address per thread plus compile-time offsets.
template <typename Sh, int e>
using ExLayout =
    std::conditional_t<(Sh::LE == 4 && Sh::LOGN >= 10 && e + 2 < Sh::m), Skew32x2, Skew16>;

// Whether the exchange between groupings sa and sb stays inside groups of
// `lanes` consecutive threads: each group's positions are the same set in
// both groupings, so no element crosses to another group. `lanes` is the
// fewest threads of one transform a wave can hold. Columns: 64 / W with W up
// to 512 / threads transforms per workgroup (a column workgroup interleaves
// its W columns across threads), 64 when one transform fills the wave. Rows:
// 64, or the whole transform where a wave holds several.
template <typename Sh, int sa, int sb>
constexpr bool wave_local() {
    constexpr int T = Sh::threads;
    constexpr int Wmax = T >= 512 ? 1 : 512 / T;
    constexpr int lanes = !Sh::ILV ? (T < 64 ? T : 64) : 64 / Wmax;
    if (lanes < 1 || (Sh::ILV && T < 64)) return false;
    auto pos = [](int s, int g, int v) {
        return (g / Sh::S(s)) * Sh::N(s) * Sh::S(s) + v * Sh::S(s) + (g % Sh::S(s));
    };
    for (int g0 = 0; g0 < T; g0 += lanes) {
        int lo[2] = {1 << 30, 1 << 30}, hi[2] = {-1, -1};
        const int st[2] = {sa, sb};
        for (int k = 0; k < 2; ++k)
            for (int th = g0; th < g0 + lanes; ++th)
                for (int q = 0; q < Sh::G(st[k]); ++q)
                    for (int v = 0; v < Sh::N(st[k]); ++v) {
                        const int p = pos(st[k], th * Sh::G(st[k]) + q, v);
                        lo[k] = p < lo[k] ? p : lo[k];
                        hi[k] = p > hi[k] ? p : hi[k];
                    }
        // E distinct positions per thread: equal bounds spanning exactly
        // E * lanes positions mean equal sets
        if (lo[0] != lo[1] || hi[0] != hi[1] || hi[0] - lo[0] + 1 != Sh::E * lanes) return false;
    }
    return true;
}

// Order a wave's LDS writes before its later LDS reads: the LDS executes one
// wave's accesses in issue order, so this only keeps the compiler from
// moving the reads above the writes (no instruction is emitted).
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exchanges of FP32 data that stay inside every wave are ordered by
// wave_order instead of workgroup barriers.
template <typename Sh, int sa, int sb>
__device__ __forceinline__ void exchange_sync() {
    if constexpr (wave_local<Sh, sa, sb>()) wave_order();
    else __syncthreads();
}

// Regroup registers from stage sa's grouping to stage sb's through LDS.
// `hook` runs between the LDS writes and the barrier, where the registers
// of the data are free: a caller issues global loads there (the kernel
// spectrum of the column pass) so that their latency overlaps the barrier,
// the LDS reads and the next stage.
template <typename T, typename Sh, int sa, int sb, typename Hook = NoHook>
__device__ __forceinline__ void exchange(cx<T>* r, cx<T>* lds, int th,
                                         const Hook& hook = Hook{}) {
    using Lay = ExLayout<Sh, (sa < sb ? sa : sb)>;
    using A = Grouping<Sh, sa, Lay>;
    using B = Grouping<Sh, sb, Lay>;
    exchange_sync<Sh, sa, sb>();
    cx<T>* wa = lds + Lay::ix(A::base(th));
#pragma unroll
    for (int q = 0; q < A::G; ++q)
#pragma unroll
        for (int v = 0; v < A::N; ++v) wa[A::off(q, v)] = r[q * A::N + v];
    hook();
    exchange_sync<Sh, sa, sb>();
    const cx<T>* rbp = lds + Lay::ix(B::base(th));
#pragma unroll
    for (int q = 0; q < B::G; ++q)
#pragma unroll
        for (int v = 0; v < B::N; ++v) r[q * B::N + v] = rbp[B::off(q, v)];
}

// The same regrouping through a real (T) LDS buffer of half the size: real
// parts first, then imaginary parts (four barriers instead of two). The
// second write reads only the imaginary parts, which the first read left
// untouched. Half the LDS per transform lets more workgroups be resident.
template <typename T, typename Sh, int sa, int sb, typename Hook = NoHook>
__device__ __forceinline__ void exchange(cx<T>* r, T* lds, int th,
                                         const Hook& hook = Hook{}) {
    using Lay = ExLayout<Sh, (sa < sb ? sa : sb)>;
    using A = Grouping<Sh, sa, Lay>;
    using B = Grouping<Sh, sb, Lay>;
    T* wa = lds + Lay::ix(A::base(th));
    const T* rbp = lds + Lay::ix(B::base(th));
    exchange_sync<Sh, sa, sb>();
#pragma unroll
    for (int q = 0; q < A::G; ++q)
#pragma unroll
        for (int v = 0; v < A::N; ++v) wa[A::off(q, v)] = r[q * A::N + v].re;
    hook();
    exchange_sync<Sh, sa, sb>();
#pragma unroll
    for (int q = 0; q < B::G; ++q)
#pragma unroll
        for (int v = 0; v < B::N; ++v) r[q * B::N + v].re = rbp[B::off(q, v)];
    exchange_sync<Sh, sa, sb>();
#pragma unroll
    for (int q = 0; q < A::G; ++q)
#pragma unroll
        for (int v = 0; v < A::N; ++v) wa[A::off(q, v)] = r[q * A::N + v].im;
    exchange_sync<Sh, sa, sb>();
#pragma unroll
    for (int q = 0; q < B::G; ++q)
#pragma unroll
        for (int v = 0; v < B::N; ++v) r[q * B::N + v].im = rbp[B::off(q, v)];
}

// LDS element type L: cx<T> (one pass per exchange) or T (split passes). An
// FP64 stage's twiddle is read ahead of the exchange before it (and of the
// loads its hook issues: loads return in order).
template <typename T, typename Sh, int s, bool ZIN, typename Hook, typename L, int KS>
__device__ __forceinline__ void forward_from(cx<T>* r, L* lds, int th, cx<double> w,
                                             const cx<double>* __restrict__ tw, int twmul,
                                             const Hook& hook, TwKeep* keep) {
    constexpr int PR = (s == 0 && ZIN) ? 1 : 0;
    if constexpr (kFused<T, Sh>) stage_fused<Sh, s, false, PR>(r, w, tw, twmul);
    else stage<T, Sh, s, false, PR, KS>(r, th, tw, twmul, keep);
    if constexpr (s + 1 < Sh::m) {
        if constexpr (kFused<T, Sh>) w = stage_twiddle<Sh, s + 1, false>(th, tw, twmul);
        if constexpr (s + 2 == Sh::m) exchange<T, Sh, s, s + 1>(r, lds, th, hook);
        else exchange<T, Sh, s, s + 1>(r, lds, th);
        forward_from<T, Sh, s + 1, ZIN, Hook, L, KS>(r, lds, th, w, tw, twmul, hook, keep);
    } else if constexpr (s == 0) {
        hook();   // single-stage transform: no exchange to hide the loads in
    }
}

template <typename T, typename Sh, int s, bool HOUT, typename L, int KS>
__device__ __forceinline__ void inverse_from(cx<T>* r, L* lds, int th, cx<double> w,
                                             const cx<double>* __restrict__ tw, int twmul,
                                             TwKeep* keep) {
    constexpr int PR = (s == 0 && HOUT) ? 2 : 0;
    if constexpr (kFused<T, Sh>) stage_fused<Sh, s, true, PR>(r, w, tw, twmul);
    else stage<T, Sh, s, true, PR, KS>(r, th, tw, twmul, keep);
    if constexpr (s > 0) {
        if constexpr (kFused<T, Sh>) w = stage_twiddle<Sh, s - 1, true>(th, tw, twmul);
        exchange<T, Sh, s, s - 1>(r, lds, th);
        inverse_from<T, Sh, s - 1, HOUT, L, KS>(r, lds, th, w, tw, twmul, keep);
    }
}

// forward: registers in stage-0 grouping (natural order) -> stage m-1
// grouping (digit-reversed); inverse: the reverse. ZIN: the upper half of
// the input (positions >= n/2, i.e. v >= 8 of stage 0) is zero; HOUT: only
// the lower half of the output is used.
// `hook` runs once, inside the last exchange (see `exchange`). KS >= 0 (FP32):
// the forward keeps stage KS's twiddle powers in *keep, and an inverse of the
// same thread with the same KS reuses them.
template <typename T, typename Sh, bool ZIN = false, typename Hook = NoHook, typename L = cx<T>,
          int KS = -1>
__device__ __forceinline__ void forward(cx<T>* r, L* lds, int th,
                                        const cx<double>* __restrict__ tw, int twmul,
                                        const Hook& hook = Hook{}, TwKeep* keep = nullptr) {
    forward_from<T, Sh, 0, ZIN, Hook, L, KS>(r, lds, th, {1.0, 0.0}, tw, twmul, hook, keep);
}
template <typename T, typename Sh, bool HOUT = false, typename L = cx<T>, int KS = -1>
__device__ __forceinline__ void inverse(cx<T>* r, L* lds, int th,
                                        const cx<double>* __restrict__ tw, int twmul,
                                        TwKeep* keep = nullptr) {
    inverse_from<T, Sh, Sh::m - 1, HOUT, L, KS>(r, lds, th, {1.0, 0.0}, tw, twmul, keep);
}

} // namespace rb
} // namespace aspher
