// Mixed-radix FFT in LDS for every transform length that is not a power of
// two (and the powers of two below the register-blocked range).
//
// A length whose prime factors are at most 13 is factored L = r_0 ... r_{m-1}
// into radices of 2 .. 16 (kWide), each an in-register DFT. Stage s combines the
// elements at pos = high*r_s*S_s + v*S_s + low, v < r_s, S_s = r_{s+1}...r_{m-1};
// group g = high*S_s + low. Forward (decimation in frequency): DFT over v,
// then multiply by W_{r_s S_s}^{v low}; every group is read and written by one
// thread at the same positions, so a stage is one LDS round trip and one
// barrier, in place. The output is digit-reversed: position sum_j d_j S_j
// holds frequency sum_j d_j P_j, P_j = r_0...r_{j-1}. Inverse (decimation in
// time): stages m-1 .. 0, conjugate twiddle before each DFT, natural output.
// The last forward and the first inverse stage share their groups, so a
// convolution multiplies by its symbol in registers between them.
//
// Prime factors from 17 to 97 (FP32: 67) are direct passes (prime_pass), placed
// last, where they take no twiddles. They read one LDS buffer and write another.
//
// Any other length runs as a chirp convolution (Bluestein 1970): with
// c_j = exp(-pi i j^2/L), X_k = c_k sum_j (x_j c_j) conj(c_{k-j}), a cyclic
// convolution of a smooth length >= 2L - 1 on the same stages; its result is
// in natural order. The inverse is the same with c and the convolution's
// spectrum conjugated.
//
// The radices are run-time values: a transform is a list of passes walked by
// the whole workgroup, each pass one branch into the code of its radix.
#pragma once

#include "fft_rb.hpp"

namespace aspher {
namespace mr {

constexpr int kMaxStages = 8;

// One pass over the groups of a stage.
struct Pass {
    int r, S;          // radix, stride of its digit
    float invS;        // 1/S, for the group's (high, low) split
    int step;          // LDS slots between the elements of a group
    int twstep;        // W_{rS}^low = tw[low * twstep], tw of length Lc
    int fwd, inv;      // forward DFT (then twiddle); (twiddle then) inverse DFT
    int from_mem, to_mem;   // column passes: first stage from, last to memory
    // prime passes: r/Lc; multiply the outputs by the symbol; multiply them by
    // the twiddles of the next inverse stage, of radix nr and stride nS (0: none)
    float invG;
    int sym, nr, nS, ntwstep;
    float ninvS;
};

struct Program {
    int n = 0;
    Pass p[2 * kMaxStages];
};

// cos(2 pi j/P), sin(2 pi j/P), j = 1 .. P/2
template <int P> struct Roots;
template <> struct Roots<3> {
    static constexpr double c[1] = {-0.5};
    static constexpr double s[1] = {0.8660254037844386};
};
template <> struct Roots<5> {
    static constexpr double c[2] = {0.30901699437494745, -0.8090169943749475};
    static constexpr double s[2] = {0.9510565162951535, 0.5877852522924731};
};
template <> struct Roots<7> {
    static constexpr double c[3] = {0.6234898018587335, -0.2225209339563144,
        -0.9009688679024191};
    static constexpr double s[3] = {0.7818314824680298, 0.9749279121818236,
        0.4338837391175581};
};
template <> struct Roots<9> {
    static constexpr double c[4] = {0.766044443118978, 0.17364817766693036, -0.5,
        -0.9396926207859084};
    static constexpr double s[4] = {0.6427876096865394, 0.984807753012208,
        0.8660254037844386, 0.3420201433256687};
};
template <> struct Roots<11> {
    static constexpr double c[5] = {0.8412535328311812, 0.41541501300188644,
        -0.14231483827328514, -0.6548607339452851, -0.9594929736144974};
    static constexpr double s[5] = {0.5406408174555976, 0.9096319953545183,
        0.9898214418809327, 0.7557495743542583, 0.28173255684142967};
};
template <> struct Roots<13> {
    static constexpr double c[6] = {0.8854560256532099, 0.5680647467311558,
        0.12053668025532305, -0.3546048870425356, -0.7485107481711011, -0.970941817426052};
    static constexpr double s[6] = {0.46472317204376856, 0.8229838658936564,
        0.992708874098054, 0.9350162426854148, 0.6631226582407952, 0.23931566428755777};
};

// cos and sin of 2 pi j/P for any j that folds to a constant
template <int P>
__host__ __device__ __forceinline__ constexpr double root_c(int j) {
    j = ((j % P) + P) % P;
    if (j == 0) return 1.0;
    return Roots<P>::c[(j <= P / 2 ? j : P - j) - 1];
}
template <int P>
__host__ __device__ __forceinline__ constexpr double root_s(int j) {
    j = ((j % P) + P) % P;
    if (j == 0) return 0.0;
    return j <= P / 2 ? Roots<P>::s[j - 1] : -Roots<P>::s[P - j - 1];
}

// the j < P/2 for which the cosine of 2 pi k (j+1)/P is the lowest
template <int P>
__host__ __device__ __forceinline__ constexpr int near_half(int k) {
    int at = 0;
    for (int j = 1; j < P / 2; ++j)
        if (root_c<P>(k * (j + 1)) < root_c<P>(k * (at + 1))) at = j;
    return at;
}

// a0 + sum_j cos(2 pi k (j+1)/P) t_j, t_j a sum of two inputs. ZERO: exactly 0
// where all inputs are equal. The mean of a field lies far above its other
// frequencies, and what the rounded cosines leave of it is the same in every row,
// so the columns add it up: with the plain sum a torus response of a field with
// a mean was 2.2e-15 off at 243^2 in FP64, now 4.7e-16. The cosines sum to -1/2:
// one t, that of the lowest cosine, takes the weight -1/2 and the others come as
// differences from it (of 9 points, without the third t, whose weight is -1/2 by
// itself).
template <int P, bool ZERO, typename A>
__device__ __forceinline__ A cosines(A a0, const A* t, int k) {
    const int ref = near_half<P>(k);
    A c = a0;
    if constexpr (!ZERO) {
#pragma unroll
        for (int j = 0; j < P / 2; ++j) c += static_cast<A>(root_c<P>(k * (j + 1))) * t[j];
    } else if (P == 9 && k == 3) {
        c = (a0 + t[2]) - A(0.5) * (t[0] + t[1] + t[3]);
    } else {
        c -= A(0.5) * t[P == 9 ? 2 : ref];
#pragma unroll
        for (int j = 0; j < P / 2; ++j)
            if (j != ref && !(P == 9 && j == 2))
                c += static_cast<A>(root_c<P>(k * (j + 1))) * (t[j] - t[ref]);
    }
    return c;
}

// Odd P: the pairs a_j + a_{P-j} carry the cosines, a_j - a_{P-j} the
// sines; the two real components are formed one after the other, so only
// half of the outputs' operands are live at a time. 9 points as well: 3 x 3 with
// twiddles between take as many operations and are 1.3 times as far off.
// FP32 values are summed in FP64, whose multiply-adds issue as often as the
// scalar FP32 ones, and rounded once: sums in FP32 left the responses of
// 3^a 5^b 11^c sides 1.1 to 1.3 times as far off as direct DFTs with one rounded
// table (243^2: 2.4e-7 against 2.1e-7, relative, of a partial contact's
// pressure), these 0.5 to 0.9 times (1.6e-7). The conversions cost a response of
// 1215^2 7 us of 62, and a chirp of 1009^2 12 of 66 (chirps of prime factors
// below 200 need them: 1660^2 1.2e-6 -> 5.8e-7, direct sums 6.8e-7).
template <typename T, int P, bool INV>
__device__ __forceinline__ void dft_odd(cx<T>* a) {
    using A = std::conditional_t<(P > 3), double, T>;
    constexpr int H = P / 2;
    A tr[H], ti[H], ur[H], ui[H];
    cx<A> s0 = {(A)a[0].re, (A)a[0].im};
    const cx<A> a0 = s0;
#pragma unroll
    for (int j = 0; j < H; ++j) {
        const cx<T> x = a[j + 1], y = a[P - 1 - j];
        tr[j] = (A)x.re + (A)y.re;
        ti[j] = (A)x.im + (A)y.im;
        ur[j] = (A)x.re - (A)y.re;
        ui[j] = (A)x.im - (A)y.im;
        s0.re += tr[j];
        s0.im += ti[j];
    }
    a[0] = {static_cast<T>(s0.re), static_cast<T>(s0.im)};
    // X_k = sum cos t -+ i sum sin u, X_{P-k} = the conjugate combination
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        A c = cosines<P, sizeof(A) == sizeof(T)>(a0.re, tr, k), s = A(0);
#pragma unroll
        for (int j = 0; j < H; ++j)
            s += static_cast<A>(root_s<P>(k * (j + 1))) * ui[j];
        a[k].re = static_cast<T>(INV ? c - s : c + s);
        a[P - k].re = static_cast<T>(INV ? c + s : c - s);
    }
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        A c = cosines<P, sizeof(A) == sizeof(T)>(a0.im, ti, k), s = A(0);
#pragma unroll
        for (int j = 0; j < H; ++j)
            s += static_cast<A>(root_s<P>(k * (j + 1))) * ur[j];
        a[k].im = static_cast<T>(INV ? c + s : c - s);
        a[P - k].im = static_cast<T>(INV ? c - s : c + s);
    }
}

template <typename T, int R, bool INV> __device__ __forceinline__ void dft(cx<T>* a);

// R = A*B with A, B coprime: index maps instead of twiddles (Good 1958;
// input n = B i + A j mod R, output k with k = ka mod A, k = kb mod B).
template <typename T, int A, int B, bool INV>
__device__ __forceinline__ void dft_coprime(cx<T>* a) {
    constexpr int R = A * B;
    cx<T> t[R];
#pragma unroll
    for (int j = 0; j < B; ++j) {
        cx<T> x[A];
#pragma unroll
        for (int i = 0; i < A; ++i) x[i] = a[(B * i + A * j) % R];
        dft<T, A, INV>(x);
#pragma unroll
        for (int i = 0; i < A; ++i) t[i * B + j] = x[i];
    }
#pragma unroll
    for (int i = 0; i < A; ++i) {
        dft<T, B, INV>(t + i * B);
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k % A == i) a[k] = t[i * B + k % B];
    }
}

template <typename T, int R, bool INV>
__device__ __forceinline__ void dft(cx<T>* a) {
    if constexpr (R == 1) {
    } else if constexpr (R == 2 || R == 4 || R == 8 || R == 16) rb::dft<T, R, INV>(a);
    else if constexpr (R == 6) dft_coprime<T, 3, 2, INV>(a);
    else if constexpr (R == 10) dft_coprime<T, 5, 2, INV>(a);
    else if constexpr (R == 12) dft_coprime<T, 3, 4, INV>(a);
    else if constexpr (R == 15) dft_coprime<T, 3, 5, INV>(a);
    else dft_odd<T, R, INV>(a);
}

// a[v] *= W^{v i}, v < R, or its conjugate, W^t = tw[t].
// FP64: every power from the table, four at a time (all at once they spill, 78 us
// a response of 1000^2; four at a time 73.8, the powers 1, 2, 4, 8 and products of
// them 72.1). The products are 1.04 to 1.06 times as far off in a response, a
// running product of one table value 1.6 times in a transform.
// FP32: those products in FP64, rounded once.
template <typename T, int R, bool CONJ>
__device__ __forceinline__ void twiddle(cx<T>* a, const cx<double>* __restrict__ tw, int i) {
    constexpr int B = sizeof(T) == 8 ? 4 : 16;
    cx<double> p[16];
#pragma unroll
    for (int v0 = 1; v0 < R; v0 += B) {
#pragma unroll
        for (int v = v0; v < v0 + B && v < R; ++v)
            if (sizeof(T) == 8 || (v & (v - 1)) == 0) p[v] = tw[v * i];
#pragma unroll
        for (int v = v0; v < v0 + B && v < R; ++v) {
            const int top = v >= 8 ? 8 : v >= 4 ? 4 : v >= 2 ? 2 : 1;
            if (sizeof(T) == 4 && v != top) p[v] = p[top] * p[v - top];
            a[v] = a[v] * cx<T>{static_cast<T>(p[v].re),
                                static_cast<T>(CONJ ? -p[v].im : p[v].im)};
        }
        // the next four wait for these
        if (v0 + B < R) asm volatile("" : "+v"(i), "+v"(a[v0].re), "+v"(a[v0 + B - 1].re));
    }
}

// q = g / S for 0 <= g < 2^15, S >= 1, from the rounded reciprocal: (g + 0.5)/S
// is at least 0.5/S away from an integer, far above the float rounding
__host__ __device__ __forceinline__ int div_by(int g, float invS) {
    return (int)(((float)g + 0.5f) * invS);
}

// LDS slot of a position: `pad` slots of skew after every C positions, C one
// of the stage strides. Every stage's stride is then a multiple of C or its
// groups lie within one run of C, so the slots of a group are a base plus
// v times a constant of the stage (Pass::step): one address per element,
// formed by one addition. C and pad are chosen on the host for the fewest
// bank conflicts.
struct Layout {
    int pad = 0;
    float invC = 1.0f;
    __host__ __device__ __forceinline__ int slot(int p) const {
        return p + pad * div_by(p, invC);
    }
};

// Where a column pass reads its first stage and writes its last: column c of
// a panel of 1 << lq columns in memory (a uniform base and 32-bit offsets);
// rows from rows_in on are zero, from rows_out on not wanted.
template <typename T>
struct Column {
    cx<T>* panel = nullptr;
    int lq = 0, c = 0, rows_in = 0, rows_out = 0;
    __device__ __forceinline__ unsigned at(int row) const {
        return ((unsigned)row << lq) + (unsigned)c;
    }
};

// A pass of radix R over one transform of length Lc in `buf`, by threads th,
// th + T, ... `sym` multiplies the R values of group g between the forward
// and the inverse DFT of a combined pass (last stage: positions g*R + v).
template <typename T, int R, bool COL, typename Sym>
__device__ __forceinline__ void run_pass(const Pass& ps, cx<T>* buf, const Layout& lay, int Lc,
                                         int th, int T_, const cx<double>* __restrict__ tw,
                                         const Column<T>& col, const Sym& sym) {
    const int G = Lc / R;
    const int S = ps.S, step = ps.step;
    for (int g = th; g < G; g += T_) {
        const int hi = div_by(g, ps.invS), low = g - hi * S;
        const int base = hi * R * S + low;
        cx<T> a[R];
        if (COL && ps.from_mem) {
#pragma unroll
            for (int v = 0; v < R; ++v) {
                const int row = base + v * S;
                a[v] = row < col.rows_in ? col.panel[col.at(row)]
                                         : cx<T>{T(0), T(0)};
            }
            // keeps the compiler from merging this branch's loads with the
            // other's into loads through one generic pointer
            asm volatile("");
        } else {
            const cx<T>* src = buf + lay.slot(base);
#pragma unroll
            for (int v = 0; v < R; ++v) a[v] = src[v * step];
        }
        if (ps.fwd) {
            dft<T, R, false>(a);
            if (S > 1) {
                // read here, not ahead of the DFT: four more FP64 values live
                // over it spill
                int i = low * ps.twstep;
                asm volatile("" : "+v"(i));
                twiddle<T, R, false>(a, tw, i);
            }
            if (ps.inv) {
                sym.template apply<R>(a, g);
                dft<T, R, true>(a);
            }
        } else {
            if (S > 1) {
                twiddle<T, R, true>(a, tw, low * ps.twstep);
            }
            dft<T, R, true>(a);
        }
        if (COL && ps.to_mem) {
#pragma unroll
            for (int v = 0; v < R; ++v) {
                const int row = base + v * S;
                if (row < col.rows_out) col.panel[col.at(row)] = a[v];
            }
            asm volatile("");
        } else {
            // the slot is recomputed, not kept live over the DFT
            int at = base;
            asm volatile("" : "+v"(at));
            cx<T>* dst = buf + lay.slot(at);
#pragma unroll
            for (int v = 0; v < R; ++v) dst[v * step] = a[v];
        }
    }
}

// A pass of prime radix P = ps.r > 13, from src to dst: a thread forms four outputs
// of a group, k, k + K and their mirrors P - k, P - k - K, from the sums and
// differences of the inputs j and P - j and the P-th roots of the twiddle table, in
// FP64. Neighbouring threads take the same k of neighbouring groups, so they read
// the same roots.
// Bound by the latency of its P/2 steps of two values and two roots each. A chirp
// convolution takes fewer from about P = 40 on, but four transforms of more than
// twice the length, and its responses were further off than those of direct sums:
// FP32 torus 340^2 (P = 17) 4.6e-7 against 2.7e-7, now 1.8e-7; FP64 510^2 1.2e-15
// against 5.4e-16, now 5.0e-16. In FP32 a chirp is as good from P = 71 on, in FP64
// from P = 101 on (790^2, P = 79: 1.6e-15 against 9.4e-16). Per response, chirp ->
// direct: FP32 340^2 33 -> 30 us, 1020^2 53 -> 47, 1220^2 (P = 61) 77 -> 106; FP64
// 340^2 38 -> 30, 1020^2 77 -> 57, 1220^2 135 -> 109, 970^2 (P = 97) 74 -> 74.
template <typename T, bool COL, typename Sym>
__device__ __forceinline__ void prime_pass(const Pass& ps, const cx<T>* src, cx<T>* dst,
                                           const Layout& lay, int Lc, int th, int T_,
                                           const cx<double>* __restrict__ tw,
                                           const Column<T>& col, const Sym& sym) {
    const int P = ps.r, S = ps.S, step = ps.step, G = Lc / P, H = P / 2, K = H / 2 + 1;
    for (int e = th; e < G * K; e += T_) {
        const int k = div_by(e, ps.invG), g = e - k * G;
        const int hi = div_by(g, ps.invS), low = g - hi * S;
        const int base = hi * P * S + low, at = lay.slot(base), i = low * ps.twstep;
        auto input = [&](int j) -> cx<double> {
            cx<T> z;
            if (COL && ps.from_mem) {
                const int row = base + j * S;
                z = row < col.rows_in ? col.panel[col.at(row)] : cx<T>{T(0), T(0)};
                asm volatile("");
            } else {
                z = src[at + j * step];
            }
            return {(double)z.re, (double)z.im};
        };
        // outputs k, k + K and their mirrors: sums with the cosines and sines
        cx<double> c[2], s[2] = {{0.0, 0.0}, {0.0, 0.0}};
        c[0] = c[1] = input(0);
        int t[2] = {0, 0};   // j k mod P
#pragma unroll 2
        for (int j = 1; j <= H; ++j) {
            const cx<double> x = input(j), y = input(P - j);
            const cx<double> a = x + y, b = x - y;
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                t[q] += k + q * K;
                if (t[q] >= P) t[q] -= P;
                const cx<double> w = tw[t[q] * G];
                c[q].re += w.re * a.re;
                c[q].im += w.re * a.im;
                s[q].re += w.im * b.im;
                s[q].im += w.im * b.re;
            }
        }
        auto output = [&](int v, cx<double> X) {
            if (ps.fwd && S > 1) X = X * tw[v * i];
            const int p = base + v * S;
            if (ps.nS) {
                const int q = div_by(p, ps.ninvS);
                X = X * conjg(tw[q % ps.nr * (p - q * ps.nS) * ps.ntwstep]);
            }
            cx<T> z = {static_cast<T>(X.re), static_cast<T>(X.im)};
            if (ps.sym) z = sym.value(z, p);
            if (COL && ps.to_mem) {
                if (p < col.rows_out) col.panel[col.at(p)] = z;
                asm volatile("");
            } else {
                dst[at + v * step] = z;
            }
        };
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int v = k + q * K;
            if (v > H) continue;
            if (ps.inv) s[q] = {-s[q].re, -s[q].im};
            output(v, cx<double>{c[q].re - s[q].re, c[q].im + s[q].im});
            if (v > 0) output(P - v, cx<double>{c[q].re + s[q].re, c[q].im - s[q].im});
        }
    }
}

// The largest prime factor of a direct transform.
template <typename T>
constexpr int kMaxPrime = sizeof(T) == 4 ? 67 : 97;

// Radices: 2 .. 10, 11 and 13; in FP32 also 12, 15 and 16, which in FP64 do not
// fit the 128 registers of four waves per SIMD (34 to 93 of them spilled).
template <typename T>
constexpr bool kWide = sizeof(T) == 4;

template <typename T, bool COL, typename Sym>
__device__ __forceinline__ void run_any(const Pass& ps, cx<T>* buf, const Layout& lay, int Lc,
                                        int th, int T_, const cx<double>* __restrict__ tw,
                                        const Column<T>& col, const Sym& sym) {
#define MR_CASE(R) \
    case R: run_pass<T, R, COL>(ps, buf, lay, Lc, th, T_, tw, col, sym); return;
    if constexpr (kWide<T>) {
        switch (ps.r) { MR_CASE(12) MR_CASE(15) MR_CASE(16) default: break; }
    }
    switch (ps.r) {
        MR_CASE(2) MR_CASE(3) MR_CASE(4) MR_CASE(5) MR_CASE(6) MR_CASE(7) MR_CASE(8)
        MR_CASE(9) MR_CASE(10) MR_CASE(11) MR_CASE(13)
        default: break;
    }
#undef MR_CASE
}

} // namespace mr
} // namespace aspher
