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

// Odd P: the pairs a_j + a_{P-j} carry the cosines, a_j - a_{P-j} the
// sines; the two real components are formed one after the other, so only
// half of the outputs' operands are live at a time. 9 points as well: 3 x 3 with
// twiddles between take as many operations and are 1.2 times as far off (FP32
// transform of 1215 = 15*9*9 points 1.25e-7 -> 1.16e-7, relative).
template <typename T, int P, bool INV>
__device__ __forceinline__ void dft_odd(cx<T>* a) {
    constexpr int H = P / 2;
    T tr[H], ti[H], ur[H], ui[H];
    cx<T> s0 = a[0];
    const cx<T> a0 = a[0];
#pragma unroll
    for (int j = 0; j < H; ++j) {
        const cx<T> x = a[j + 1], y = a[P - 1 - j];
        tr[j] = x.re + y.re;
        ti[j] = x.im + y.im;
        ur[j] = x.re - y.re;
        ui[j] = x.im - y.im;
        s0.re += tr[j];
        s0.im += ti[j];
    }
    a[0] = s0;
    // X_k = sum cos t -+ i sum sin u, X_{P-k} = the conjugate combination
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        T c = a0.re, s = T(0);
#pragma unroll
        for (int j = 0; j < H; ++j) {
            c += static_cast<T>(root_c<P>(k * (j + 1))) * tr[j];
            s += static_cast<T>(root_s<P>(k * (j + 1))) * ui[j];
        }
        a[k].re = INV ? c - s : c + s;
        a[P - k].re = INV ? c + s : c - s;
    }
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        T c = a0.im, s = T(0);
#pragma unroll
        for (int j = 0; j < H; ++j) {
            c += static_cast<T>(root_c<P>(k * (j + 1))) * ti[j];
            s += static_cast<T>(root_s<P>(k * (j + 1))) * ur[j];
        }
        a[k].im = INV ? c + s : c - s;
        a[P - k].im = INV ? c - s : c + s;
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

// Twiddles W^{v i}, v < R, of a group: the powers 1, 2, 4, 8 from the table
// (tw[v*i]), the others products of two or three of them, rounded once to
// FP32 where the data are. A running product of one table value was 1.6 times
// as far off in FP64; reading every power costs a gather each.
template <int R>
struct Twiddle {
    cx<double> p[16];
    __device__ __forceinline__ void load(const cx<double>* __restrict__ tw, int i) {
#pragma unroll
        for (int v = 1; v < R; v *= 2) p[v] = tw[v * i];
    }
    // a[v] *= w^v, or its conjugate
    template <bool CONJ, typename T>
    __device__ __forceinline__ void apply(cx<T>* a) {
#pragma unroll
        for (int v = 1; v < R; ++v) {
            const int top = v >= 8 ? 8 : v >= 4 ? 4 : v >= 2 ? 2 : 1;
            if (v != top) p[v] = p[top] * p[v - top];
            const cx<T> w = {static_cast<T>(p[v].re), static_cast<T>(CONJ ? -p[v].im : p[v].im)};
            a[v] = a[v] * w;
        }
    }
};

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
                Twiddle<R> w;
                w.load(tw, i);
                w.template apply<false>(a);
            }
            if (ps.inv) {
                sym.template apply<R>(a, g);
                dft<T, R, true>(a);
            }
        } else {
            if (S > 1) {
                Twiddle<R> w;
                w.load(tw, low * ps.twstep);
                w.template apply<true>(a);
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
