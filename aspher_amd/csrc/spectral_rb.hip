// Power-of-two spectral convolution kernels built on the register-blocked
// FFT (fft_rb.hpp). Data flow of y = inv(s . fwd(x)) on an n x n grid:
//
//   rows_fwd : x rows -> half spectrum, in panels of Q adjacent frequencies
//   cols     : each column -> forward, symbol, inverse -> in place
//   rows_inv : panels -> y rows
//
// The transposition happens in the row passes, which move runs of B rows by Q
// frequencies; a column workgroup moves whole columns (Q of them where it
// holds W = Q). The tiles of one panel run on one XCD (the XCD-aware block
// mapping), so partial lines merge in its L2.
#include "embed.hpp"
#include "fft_rb.hpp"
#include "reduce.hpp"
#include "spectral_rb.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

namespace aspher {

namespace {

// two consecutive reals as one 8- (FP32) or 16-byte (FP64) access
template <typename T>
struct alignas(2 * sizeof(T)) Pair {
    T a, b;
};

__host__ __device__ __forceinline__ bool pair_aligned(const void* p, std::size_t elt) {
    return (reinterpret_cast<std::uintptr_t>(p) % (2 * elt)) == 0;
}

// Slot of natural-order element k in a row pass's LDS row (the
// digit-reversed write and packed-spectrum split of the forward pass, the
// merge and gather of the inverse). The B rows of a workgroup are
// read and written together there, lane t on row t % B at element t / B + c:
// rows take Skew32x2 and start P / B slots apart mod P (row_stride; P = 32
// for 8-byte elements, 16 for 16-byte ones), so the lanes the LDS serves
// together fall in distinct banks.
template <typename T>
__device__ __forceinline__ int row_ix(int k) {
    return rb::Skew32x2::ix(k);
}
template <typename T>
__host__ __device__ inline int row_stride(int L, int B) {
    const int base = rb::lds_len(L);
    constexpr int P = sizeof(cx<T>) >= 16 ? 16 : 32;
    if (B < 2 || B > P) return base;
    return base + ((P / B - base % P) % P + P) % P;
}

// Half spectrum between the passes, in panels of Q = 1 << lq adjacent
// frequencies: value (k, row) at ((k >> lq)*pitch + row)*Q + k % Q.
// A row workgroup's share: thread t holds row bb = (t / Q) % B and the
// frequencies k0 + i TPR, i < L/(2 TPR), k0 < TPR, with their mirrors L - k
// (and L/2, held by k0 = 0). Addresses are a lane's byte offset (below 4 GiB)
// and uniform steps of TPR frequencies (TPR is a multiple of Q).
template <typename T, int L, int TPR>
struct Half {
    int bb, k0;
    unsigned up, down, mid;
    std::ptrdiff_t step;
    template <typename P>
    static __device__ __forceinline__ P* at(P* A, std::ptrdiff_t steps, unsigned lane) {
        using C = std::conditional_t<std::is_const_v<P>, const char, char>;
        return reinterpret_cast<P*>(reinterpret_cast<C*>(A + steps) + lane);
    }
    __device__ __forceinline__ Half(int t, int B, int lq, int pitch, int row0) {
        const int Q = 1 << lq, q = t & (Q - 1), t1 = t >> lq;
        bb = t1 % B;
        k0 = ((t1 / B) << lq) + q;
        const int row = row0 + bb, m0 = L - k0;
        auto bytes = [&](int k) {
            return (unsigned)sizeof(cx<T>) *
                   ((((unsigned)(k >> lq) * (unsigned)pitch + (unsigned)row) << lq) +
                    (unsigned)(k & (Q - 1)));
        };
        up = bytes(k0);
        down = bytes(m0);
        mid = bytes(L / 2);
        step = (std::ptrdiff_t)TPR * pitch;
    }
};

__device__ __forceinline__ int xcd_block(int b, int G) {
    const int q = G >> 3, r = G & 7;
    const int x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

// ── rows: real -> half spectrum ────────────────────────────────────────────
// Z: the row's nonzero reals are x[0 .. L) of n = 2L (zero-padded free-space
// rows), so the upper half of the packed input is never loaded and the first
// radix-16 stage is pruned.
template <typename T, int LOGL, int LE, int IN, bool Z>
__global__ void __launch_bounds__(1024)
k_rb_rows_fwd(const T* __restrict__ x, int x_pitch, int ncols, int nrows,
              cx<T>* __restrict__ AT, int pitchT, int lq, int B,
              const cx<double>* __restrict__ tw,
              const std::uint8_t* __restrict__ mask, const double* __restrict__ scal,
              int gmean_idx, const double* __restrict__ table, int Ns_embed, int remap,
              RbBatch bt) {
    using Sh = rb::Shape<LOGL, LE, false>;
    constexpr int L = Sh::n, n = 2 * L, TPR = Sh::threads, E = Sh::E;
    const int LL = row_stride<T>(L, B);
    extern __shared__ __align__(16) unsigned char smem[];
    {
        const int li = blockIdx.y, gi = bt.first + li;
        if (bt.gate >= 0 && bt.gscal[(std::size_t)gi * bt.sstride + bt.gate] == 0.0) return;
        x += li * bt.x_stride;
        if (mask) mask += li * (bt.m_stride >= 0 ? bt.m_stride : bt.x_stride);
        AT += li * bt.at_stride;
        if (scal) scal += (std::size_t)gi * bt.sstride;
    }
    cx<T>* lds_all = reinterpret_cast<cx<T>*>(smem);
    const int blk = remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int b = threadIdx.x / TPR, th = threadIdx.x - b * TPR;
    const int row = blk * B + b;
    cx<T>* lds = lds_all + b * LL;
    T gmean = T(0);
    if constexpr (IN == 1) gmean = static_cast<T>(scal[gmean_idx]);

    auto load = [&](int col) -> T {
        if (row >= nrows || col >= ncols) return T(0);
        if constexpr (IN >= 2 && IN <= 4) {
            // wrap-around embedding of an offset table:
            // 2 even, 3 even transposed, 4 odd-odd
            const int Ns = Ns_embed;
            const int ady = embed_offset(row, Ns, n), adx = embed_offset(col, Ns, n);
            if (ady < 0 || adx < 0) return T(0);
            if constexpr (IN == 2) {
                return static_cast<T>(table[(size_t)ady * Ns + adx]);
            } else if constexpr (IN == 3) {
                return static_cast<T>(table[(size_t)adx * Ns + ady]);
            } else {
                if (adx == 0 || ady == 0) return T(0);
                const T v = static_cast<T>(table[(size_t)ady * Ns + adx]);
                return ((col < Ns) == (row < Ns)) ? v : T(-v);
            }
        } else {
            const size_t i = (size_t)row * x_pitch + col;
            if constexpr (IN == 1) return mask[i] ? T(x[i] - gmean) : T(0);
            else return x[i];
        }
    };

    cx<T> r[E];
    // plain or masked input on an even pitch and width from a pair-aligned
    // base: both reals of a packed element in one access (and their two
    // mask bytes in one)
    const bool pairs = (IN == 0 || IN == 1) && ((x_pitch | ncols) & 1) == 0 &&
                       pair_aligned(x, sizeof(T)) &&
                       (IN == 0 || (reinterpret_cast<std::uintptr_t>(mask) & 1u) == 0);
    if (pairs) {
#pragma unroll
        for (int v = 0; v < E; ++v) {
            const int p = Sh::pos(0, th, v);
            r[v] = {T(0), T(0)};
            if ((Z && v >= E / 2) || row >= nrows || 2 * p >= ncols) continue;
            const std::size_t i = (size_t)row * x_pitch + 2 * p;
            const Pair<T> q = *reinterpret_cast<const Pair<T>*>(x + i);
            if constexpr (IN == 1) {
                const unsigned mm = *reinterpret_cast<const unsigned short*>(mask + i);
                r[v] = {(mm & 0xffu) ? T(q.a - gmean) : T(0), (mm >> 8) ? T(q.b - gmean) : T(0)};
            } else {
                r[v] = {q.a, q.b};
            }
        }
    } else {
#pragma unroll
        for (int v = 0; v < E; ++v) {
            const int p = Sh::pos(0, th, v);   // packed index j: reals 2j, 2j+1
            if (Z && v >= E / 2) r[v] = {T(0), T(0)};
            else r[v] = {load(2 * p), load(2 * p + 1)};
        }
    }
    // W^k of the split: W^k0, read ahead of the transform, times the uniform
    // W^{i TPR} (scalar loads)
    const Half<T, L, TPR> hs(threadIdx.x, B, lq, pitchT, blk * B);
    const cx<double> w0 = tw[hs.k0];
    rb::forward<T, Sh, Z>(r, lds, th, tw, 2);
    // digit-reversed registers -> natural order in LDS, then split the
    // packed spectrum: X[k] = (Z_k + conj Z_{L-k})/2 - i W^k (Z_k - conj Z_{L-k})/2
    __syncthreads();
    constexpr int Gl = Sh::G(Sh::m - 1), Nl = Sh::N(Sh::m - 1);
#pragma unroll
    for (int q = 0; q < Gl; ++q)
#pragma unroll
        for (int v = 0; v < Nl; ++v)
            lds[row_ix<T>(Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, v)))] = r[q * Nl + v];
    __syncthreads();
    // frequencies k and L - k come from the same two values: X_k = E + W^k O,
    // X_{L-k} = conj(E - W^k O). The Q frequencies of a panel are the fastest
    // lanes, then the B rows, so a store is a run of B*Q values
    const int nb = (nrows - blk * B < B) ? (nrows - blk * B) : B;
    if (hs.bb < nb) {
        const cx<T>* lb = lds_all + hs.bb * LL;
#pragma unroll
        for (int i = 0; i < E / 2; ++i) {
            const int k = hs.k0 + i * TPR;
            const cx<T> Zk = lb[row_ix<T>(k)];
            const cx<T> Zc = conjg(lb[row_ix<T>(k == 0 ? 0 : L - k)]);
            const cx<T> Ev = scale(Zk + Zc, T(0.5));
            const cx<T> D = Zk - Zc;
            const cx<T> O = {D.im * T(0.5), -D.re * T(0.5)};
            const cx<double> wd = i == 0 ? w0 : w0 * tw[i * TPR];
            const cx<T> WO = cx<T>{static_cast<T>(wd.re), static_cast<T>(wd.im)} * O;
            *hs.at(AT, i * hs.step, hs.up) = Ev + WO;
            *hs.at(AT, -i * hs.step, hs.down) = conjg(Ev - WO);
        }
        // W^{L/2} = -i
        if (hs.k0 == 0) *hs.at(AT, 0, hs.mid) = conjg(lb[row_ix<T>(L / 2)]);
    }
}

// NV contiguous values from an address aligned to all of them, as 16-byte
// vector loads
template <int NV>
__device__ __forceinline__ void loadv(const float* __restrict__ p, float* v) {
    const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
    for (int j = 0; j < NV / 4; ++j) {
        const float4 t = q[j];
        v[4 * j] = t.x;
        v[4 * j + 1] = t.y;
        v[4 * j + 2] = t.z;
        v[4 * j + 3] = t.w;
    }
}
template <int NV>
__device__ __forceinline__ void loadv(const double* __restrict__ p, double* v) {
    const double2* q = reinterpret_cast<const double2*>(p);
#pragma unroll
    for (int j = 0; j < NV / 2; ++j) {
        const double2 t = q[j];
        v[2 * j] = t.x;
        v[2 * j + 1] = t.y;
    }
}

// ── columns: forward . symbol . inverse, in place ──────────────────────────
template <typename T, int SYM, int LOGN>
__device__ __forceinline__ T symbol_rb(int kx, int ky, int n, const T* __restrict__ ktab,
                                       int kp, double sc) {
    if constexpr (SYM == 1) {
        const int my = (ky < ((n + 1) >> 1)) ? ky : ky - n;
        const double m2 = (double)kx * kx + (double)my * my;
        return m2 > 0.0 ? static_cast<T>(sc / sqrt(m2)) : T(0);
    } else {
        const int kof = (ky < (n >> 1)) ? ky : ky - n;
        // |k| rounded once to float. Up to n = 4096, kx^2 + kof^2 <= n^2/2 is
        // an exact float and the correctly rounded FP32 root of it is that
        // rounding (checked for every integer below 2^24); beyond, FP64.
        float h;
        if constexpr (LOGN <= 12) h = sqrtf((float)(kx * kx + kof * kof));
        else h = (float)sqrt((double)kx * kx + (double)kof * kof);
        const float w = (kx == 0 && ky == 0) ? 0.0f : (float)sc * h;
        return static_cast<T>(w);
    }
}

// Free-space column passes that exchange through a real (T) LDS buffer: FP64
// from n = 4096 on, where complex values take 70 KiB a column, two resident
// workgroups of 256 threads (n = 4096; 49.8 against 44.5 us), and more than
// half of the LDS at n = 8192 (3.5% slower at 4096^2). FP32 columns exchange
// complex values: their 8-byte exchanges fit two workgroups in LDS anyway, and
// with bank-conflict-free layouts the halved barrier count wins (FP32 column
// pass at 4096^2: 128 -> 122 us against the split exchanges).
template <typename T, int LOGN, int SYM>
constexpr bool kColsSplit = SYM == 0 && sizeof(T) == 8 && LOGN >= 12;

// Waves per SIMD that a column pass's registers are held to. Free space: 128
// VGPRs for two resident 512-thread workgroups, FP32 and FP64 at n = 8192 (no
// bound: 247 against 210 us; 80 VGPRs for a third FP32 workgroup spilled and
// was ~12% slower); three waves in FP64 at n = 4096 (two: 45.8 us, three:
// 44.6, four spill: 53.9). The computed symbols lose by a bound (torus 4096^2
// FP64: 62.9 -> 70.9).
template <typename T, int LOGN, int SYM>
constexpr int kColsWaves = SYM != 0                       ? 1
                           : sizeof(T) == 4 || LOGN >= 13 ? 4
                           : LOGN == 12                   ? 3
                                                          : 1;

template <typename T, int LOGN, int LE, int SYM>
__global__ void __launch_bounds__(512, (kColsWaves<T, LOGN, SYM>))
k_rb_cols(cx<T>* AT, int pitchT, int lq,
          int ncols, int rows_in, int rows_out, int W, const cx<double>* __restrict__ tw,
          const T* __restrict__ ktab, int kp, double sc, T* __restrict__ kout,
          double* __restrict__ part, int remap, RbBatch bt, const int* __restrict__ kmap) {
    using Sh = rb::Shape<LOGN, LE>;
    {
        const int li = blockIdx.y, gi = bt.first + li;
        if (bt.gate >= 0 && bt.gscal[(std::size_t)gi * bt.sstride + bt.gate] == 0.0) return;
        AT += li * bt.at_stride;
    }
    constexpr int n = Sh::n, E = Sh::E;
    constexpr int LL = rb::lds_len(n);
    constexpr int Gl = Sh::G(Sh::m - 1), Nl = Sh::N(Sh::m - 1);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double red[16];
    const int tile0 = remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    // tiles beyond the grid (the host folds a small last round, e.g. the
    // Nyquist column of an (Ns+1)-column half spectrum, into the first
    // blocks) are taken in a second pass; the pass condition is uniform
    for (int tile = tile0; tile * W < ncols; tile += gridDim.x) {
    // the lane's indices are made opaque per pass, so the address arithmetic
    // derived from them is recomputed in the pass rather than kept live
    // across it (which would cost occupancy)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    // columns interleaved across lanes: the values of a panel's columns in one
    // row are adjacent within each load and store instruction
    const int c = tid % W, th = tid / W;
    // kColsSplit: the exchanges pass real and imaginary parts separately
    // through half the LDS
    using LT = std::conditional_t<kColsSplit<T, LOGN, SYM>, T, cx<T>>;
    LT* lds = reinterpret_cast<LT*>(smem) + c * LL;
    const int kx = tile * W + c;
    const bool live = kx < ncols;

    // free-space symbol: rows_in, rows_out <= n/2, so the zero-padded upper
    // half is neither loaded nor transformed forward, nor produced inverse
    constexpr bool ZP = (SYM == 0);
    cx<T> r[E];
    // this thread's rows th + v n/E of the column: a byte offset of its own
    // below 4 GiB and a uniform one per v
    const int kl = live ? kx : 0, Q = 1 << lq;
    const unsigned lane = (unsigned)sizeof(cx<T>) *
                          ((((unsigned)(kl >> lq) * (unsigned)pitchT + (unsigned)th) << lq) +
                           (unsigned)(kl & (Q - 1)));
    auto element = [&](int v) -> cx<T>* {
        char* base = reinterpret_cast<char*>(AT + ((std::size_t)(v * Sh::S(0)) << lq));
        return reinterpret_cast<cx<T>*>(base + lane);
    };
#pragma unroll
    for (int v = 0; v < E; ++v) {
        const int p = Sh::pos(0, th, v);
        if (ZP && v >= E / 2) r[v] = {T(0), T(0)};
        else r[v] = (live && p < rows_in) ? *element(v) : cx<T>{T(0), T(0)};
    }
    // the kernel table in the plan's digit-reversed layout: the E values of
    // this thread are contiguous at kx*kp + E*chunk (Gl*Nl = E); loaded
    // inside the last forward exchange so the HBM latency is hidden
    T kv[E];
    // half-size table: mirror-paired threads share a chunk, the upper one
    // reads it reversed (kmap); without a map, one chunk per thread
    int km = th << 1;
    // FP32 table symbol: the inverse reuses the forward's stage-KS twiddle
    // powers (15 values more per thread, within the bounded columns' 128
    // VGPRs; the computed-symbol passes have no such bound and would lose a
    // resident workgroup)
    constexpr int KS = SYM == 0 && std::is_same_v<T, float> ? rb::keep_stage<Sh>() : -1;
    rb::TwKeep keep;
    if constexpr (SYM == 0) {
        if (kmap) km = kmap[th];
        const T* kr = ktab + (size_t)(live ? kx : 0) * kp + E * (km >> 1);
        auto hook = [&]() { loadv<E>(kr, kv); };
        rb::forward<T, Sh, ZP, decltype(hook), LT, KS>(r, lds, th, tw, 1, hook, &keep);
    } else {
        rb::forward<T, Sh, ZP, rb::NoHook, LT, KS>(r, lds, th, tw, 1, rb::NoHook{}, &keep);
    }

    if constexpr (SYM == 3) {
        // kernel-spectrum build (src/fft_operator.cpp:46-68): realness check
        // over every mode, Re/n^2 stored for ky in [0, n/2] (even in ky)
        const double norm = 1.0 / ((double)n * (double)n);
        double mi = 0.0, mr = 0.0;
#pragma unroll
        for (int q = 0; q < Gl; ++q)
#pragma unroll
            for (int v = 0; v < Nl; ++v) {
                const int ky = Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, v));
                const cx<T> z = r[q * Nl + v];
                if (live) {
                    mi = fmax(mi, fabs((double)z.im));
                    mr = fmax(mr, fabs((double)z.re));
                    if (ky <= (n >> 1)) kout[(size_t)kx * kp + ky] = static_cast<T>(norm * (double)z.re);
                }
            }
        mi = block_reduce<RMAX>(mi, red);
        if (threadIdx.x == 0) part[2 * blockIdx.x] = mi;
        mr = block_reduce<RMAX>(mr, red);
        if (threadIdx.x == 0) part[2 * blockIdx.x + 1] = mr;
        return;
    } else {
        if constexpr (SYM == 0) {
            const bool rev = (km & 1) != 0;
#pragma unroll
            for (int i = 0; i < E; ++i) {
                const T k = rev ? kv[E - 1 - i] : kv[i];
                r[i] = scale(r[i], live ? k : T(0));
            }
        } else {
#pragma unroll
            for (int q = 0; q < Gl; ++q)
#pragma unroll
                for (int v = 0; v < Nl; ++v) {
                    const int ky = Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, v));
                    const T s = live ? symbol_rb<T, SYM, LOGN>(kx, ky, n, ktab, kp, sc) : T(0);
                    r[q * Nl + v] = scale(r[q * Nl + v], s);
                }
        }
        rb::inverse<T, Sh, ZP, LT, KS>(r, lds, th, tw, 1, &keep);
        if (live) {
            // in place, the column's rows [0, rows_out) (every thread's loads
            // of it were consumed before the first exchange barrier)
#pragma unroll
            for (int v = 0; v < (ZP ? E / 2 : E); ++v) {
                const int p = Sh::pos(0, th, v);
                if (p < rows_out) *element(v) = r[v];
            }
        }
    }
    }
}

// ── rows: half spectrum -> real ────────────────────────────────────────────
// H: only the reals y[0 .. L) of n = 2L are wanted (free-space rows), so the
// last radix-16 stage computes half of its outputs.
template <typename T, int LOGL, int LE, int OUT, bool H>
__global__ void __launch_bounds__(1024)
k_rb_rows_inv(const cx<T>* __restrict__ AT, int pitchT, int lq, int nrows, int B,
              const cx<double>* __restrict__ tw, T* __restrict__ y, int y_pitch, int ncols,
              const std::uint8_t* __restrict__ mask, double* __restrict__ part, int remap,
              RbBatch bt, RowEpilogue<T> epi) {
    using Sh = rb::Shape<LOGL, LE, false>;
    {
        const int li = blockIdx.y, gi = bt.first + li;
        if (bt.gate >= 0 && bt.gscal[(std::size_t)gi * bt.sstride + bt.gate] == 0.0) return;
        AT += li * bt.at_stride;
        y += li * bt.y_stride;
        if (mask) mask += li * (bt.m_stride >= 0 ? bt.m_stride : bt.y_stride);
        if (part) part += (std::size_t)gi * bt.pstride;
    }
    constexpr int L = Sh::n, TPR = Sh::threads, E = Sh::E;
    const int LL = row_stride<T>(L, B);
    constexpr int Gl = Sh::G(Sh::m - 1), Nl = Sh::N(Sh::m - 1);
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double red[16];
    cx<T>* lds_all = reinterpret_cast<cx<T>*>(smem);
    const int blk = remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int b = threadIdx.x / TPR, th = threadIdx.x - b * TPR;
    const int row = blk * B + b;
    cx<T>* lds = lds_all + b * LL;
    cx<T> r[E];
    // Z_k = (X_k + conj X_{L-k}) + i (X_k - conj X_{L-k}) W^{-k} and its mirror
    // Z_{L-k} from the same two values (Im of the DC and Nyquist modes is
    // ignored, the c2r convention), in natural order into LDS; every load is
    // issued before the first is waited for
    {
        const Half<T, L, TPR> hs(threadIdx.x, B, lq, pitchT, blk * B);
        const bool in = blk * B + hs.bb < nrows;
        cx<T>* lb = lds_all + hs.bb * LL;
        const cx<T> zero = {T(0), T(0)};
        // (W^k0 before the data: loads return in order)
        const cx<double> w0 = tw[hs.k0];
        cx<T> xk[E / 2], xc[E / 2], xm = zero;
#pragma unroll
        for (int i = 0; i < E / 2; ++i) {
            xk[i] = in ? *hs.at(AT, i * hs.step, hs.up) : zero;
            xc[i] = in ? *hs.at(AT, -i * hs.step, hs.down) : zero;
        }
        if (hs.k0 == 0 && in) xm = *hs.at(AT, 0, hs.mid);
#pragma unroll
        for (int i = 0; i < E / 2; ++i) {
            const int k = hs.k0 + i * TPR;
            if (k == 0) {
                xk[i].im = T(0);
                xc[i].im = T(0);
            }
            const cx<T> Xc = conjg(xc[i]);
            const cx<double> wd = i == 0 ? w0 : w0 * tw[i * TPR];
            const cx<T> S = xk[i] + Xc;
            const cx<T> D = (xk[i] - Xc) * cx<T>{static_cast<T>(wd.re), static_cast<T>(-wd.im)};
            lb[row_ix<T>(k)] = {S.re - D.im, S.im + D.re};
            if (k != 0) lb[row_ix<T>(L - k)] = {S.re + D.im, D.re - S.im};
        }
        if (hs.k0 == 0) lb[row_ix<T>(L / 2)] = scale(conjg(xm), T(2));
    }
    __syncthreads();
    // gathered into the digit-reversed grouping of the inverse: the last digit
    // v of a group's positions is the top digit of k
#pragma unroll
    for (int q = 0; q < Gl; ++q) {
        const int kg = Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, 0));
#pragma unroll
        for (int v = 0; v < Nl; ++v) r[q * Nl + v] = lds[row_ix<T>(kg + v * (L / Nl))];
    }
    // every wave has gathered from the whole row before the transform's
    // first exchange writes (it may be ordered within each wave only)
    __syncthreads();
    rb::inverse<T, Sh, H>(r, lds, th, tw, 2);
    if constexpr (OUT >= 2) {
        // the values and their epilogue operands in aligned pairs (the launcher
        // checks the pitch, the width and the alignment)
        double s0 = 0.0, s1 = 0.0, s2 = __builtin_huge_val();
        if (row < nrows) {
#pragma unroll
            for (int v = 0; v < (H ? E / 2 : E); ++v) {
                const int p = Sh::pos(0, th, v);
                if (2 * p >= ncols) continue;
                const std::size_t i = (size_t)row * y_pitch + 2 * p;
                const T val[2] = {r[v].re, r[v].im};
                *reinterpret_cast<Pair<T>*>(y + i) = Pair<T>{val[0], val[1]};
                const Pair<T> pa = *reinterpret_cast<const Pair<T>*>(epi.a + i);
                const Pair<T> pb = *reinterpret_cast<const Pair<T>*>(epi.b + i);
                const T av[2] = {pa.a, pa.b}, bv[2] = {pb.a, pb.b};
                if constexpr (OUT == 2) {
                    T ov[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        ov[h] = val[h] + av[h];
                        const double d = (double)ov[h];
                        if (d < s2) s2 = d;
                        if (bv[h] > T(0)) {
                            s0 += d;
                            s1 += 1.0;
                        }
                    }
                    *reinterpret_cast<Pair<T>*>(epi.o + i) = Pair<T>{ov[0], ov[1]};
                } else {
                    const unsigned mm = *reinterpret_cast<const unsigned short*>(epi.mask + i);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        if (!((mm >> (8 * h)) & 0xffu)) continue;
                        s0 += (double)val[h];
                        s1 += (double)av[h] * (double)bv[h];
                    }
                }
            }
        }
        double* prow = epi.part + (std::size_t)blockIdx.x * kPartVals;
        s0 = block_reduce<RSUM>(s0, red);
        if (threadIdx.x == 0) prow[0] = s0;
        s1 = block_reduce<RSUM>(s1, red);
        if (threadIdx.x == 0) prow[1] = s1;
        if constexpr (OUT == 2) {
            s2 = block_reduce<RMIN>(s2, red);
            if (threadIdx.x == 0) prow[2] = s2;
        }
        return;
    }
    double acc = 0.0;
    const bool pairs = (OUT == 0 || OUT == 1) && ((y_pitch | ncols) & 1) == 0 &&
                       pair_aligned(y, sizeof(T)) &&
                       (OUT == 0 || (reinterpret_cast<std::uintptr_t>(mask) & 1u) == 0);
    if (row < nrows && pairs) {
        // plain or masked output on an even pitch and width: pair stores
        // (and the two mask bytes in one load)
#pragma unroll
        for (int v = 0; v < (H ? E / 2 : E); ++v) {
            const int p = Sh::pos(0, th, v);
            if (2 * p >= ncols) continue;
            const std::size_t i = (size_t)row * y_pitch + 2 * p;
            T a = r[v].re, b = r[v].im;
            if constexpr (OUT == 1) {
                const unsigned mm = *reinterpret_cast<const unsigned short*>(mask + i);
                if (mm & 0xffu) acc += (double)a;
                else a = T(0);
                if (mm >> 8) acc += (double)b;
                else b = T(0);
            }
            *reinterpret_cast<Pair<T>*>(y + i) = Pair<T>{a, b};
        }
    } else if (row < nrows) {
#pragma unroll
        for (int v = 0; v < (H ? E / 2 : E); ++v) {
            const int p = Sh::pos(0, th, v);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int col = 2 * p + h;
                if (col >= ncols) continue;
                T val = h ? r[v].im : r[v].re;
                const size_t i = (size_t)row * y_pitch + col;
                if constexpr (OUT == 1) {
                    if (mask[i]) acc += (double)val;
                    else val = T(0);
                }
                y[i] = val;
            }
        }
    }
    if constexpr (OUT == 1) {
        acc = block_reduce<RSUM>(acc, red);
        if (threadIdx.x == 0) part[(std::size_t)blockIdx.x * kPartVals] = acc;
    }
}

void allow_lds_rb(const void* fn, std::size_t bytes) {
    static std::mutex mu;
    static std::map<const void*, std::size_t> done;
    if (bytes <= 65536) return;
    std::lock_guard<std::mutex> lk(mu);
    auto it = done.find(fn);
    if (it != done.end() && it->second >= bytes) return;
    ASPHER_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize,
                                   static_cast<int>(bytes)));
    done[fn] = bytes;
}

// a row's threads walk whole panels
void check_panels(int threads, int lq) {
    if (lq < 0 || threads % (1 << lq))
        throw std::invalid_argument("row transform: panels wider than the row's threads");
}

template <typename T, int LOGL, int LE>
void launch_rows_fwd(const RbRowsFwd<T>& a, hipStream_t s) {
    constexpr int L = 1 << LOGL;
    // every operand the mode reads must be present
    const bool ok = a.mode == 0   ? a.x != nullptr
                    : a.mode == 1 ? (a.x && a.mask && a.scal)
                    : a.mode <= 4 ? a.table != nullptr
                                  : false;
    if (!ok) throw std::invalid_argument("row transform: missing operand for its input mode");
    check_panels(L >> LE, a.lq);
    const int block = a.B * (L >> LE);
    const dim3 grid((a.nrows + a.B - 1) / a.B, a.bt.count);
    const std::size_t lds = sizeof(cx<T>) * (std::size_t)a.B * row_stride<T>(L, a.B);
    const void* fn;
#define RF_ARGS a.x, a.x_pitch, a.ncols, a.nrows, a.AT, a.pitchT, a.lq, a.B, a.tw, a.mask, a.scal, \
        a.gmean_idx, a.table, a.Ns_embed, a.remap, a.bt
    if (a.mode == 0 && a.ncols <= L) {
        fn = (const void*)k_rb_rows_fwd<T, LOGL, LE, 0, true>;
        allow_lds_rb(fn, lds);
        k_rb_rows_fwd<T, LOGL, LE, 0, true><<<grid, block, lds, s>>>(RF_ARGS);
    } else if (a.mode == 0) {
        fn = (const void*)k_rb_rows_fwd<T, LOGL, LE, 0, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_fwd<T, LOGL, LE, 0, false><<<grid, block, lds, s>>>(RF_ARGS);
    } else if (a.mode == 1) {
        fn = (const void*)k_rb_rows_fwd<T, LOGL, LE, 1, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_fwd<T, LOGL, LE, 1, false><<<grid, block, lds, s>>>(RF_ARGS);
    } else if (a.mode == 2) {
        fn = (const void*)k_rb_rows_fwd<T, LOGL, LE, 2, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_fwd<T, LOGL, LE, 2, false><<<grid, block, lds, s>>>(RF_ARGS);
    } else if (a.mode == 3) {
        fn = (const void*)k_rb_rows_fwd<T, LOGL, LE, 3, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_fwd<T, LOGL, LE, 3, false><<<grid, block, lds, s>>>(RF_ARGS);
    } else {
        fn = (const void*)k_rb_rows_fwd<T, LOGL, LE, 4, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_fwd<T, LOGL, LE, 4, false><<<grid, block, lds, s>>>(RF_ARGS);
    }
#undef RF_ARGS
    ASPHER_LAUNCH_CHECK();
}

// Concurrent workgroups of a kernel on the device (occupancy x CUs), cached.
int resident_blocks(const void* fn, int block, std::size_t lds) {
    static std::mutex mu;
    static std::map<std::tuple<int, const void*, int, std::size_t>, int> done;
    int dev = 0;
    ASPHER_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    const auto key = std::make_tuple(dev, fn, block, lds);   // per device: CU counts differ
    auto it = done.find(key);
    if (it != done.end()) return it->second;
    int per_cu = 0, cus = 0;
    ASPHER_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, block, lds));
    ASPHER_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int r = std::max(1, per_cu) * std::max(1, cus);
    done[key] = r;
    return r;
}

// Grid of the column pass: when the tiles exceed one round of resident
// workgroups by a small remainder (at most 1/16 of a round), the remainder
// is folded into the first blocks as a second pass instead of a last round
// that would run almost alone.
int cols_grid(int tiles, int resident) {
    if (tiles <= resident) return tiles;
    const int rem = tiles % resident;
    if (rem == 0 || rem > resident / 16) return tiles;
    return tiles - rem;
}

template <typename T, int LOGN, int LE>
void launch_cols(const RbCols<T>& a, hipStream_t s) {
    constexpr int n = 1 << LOGN;
    if (a.W < 1 || (a.W & (a.W - 1)))
        throw std::invalid_argument("column transform: the width is not a power of two");
    const int block = a.W * (n >> LE);
    const int tiles = (a.ncols + a.W - 1) / a.W;
    const std::size_t elt = (a.sym == 0 && kColsSplit<T, LOGN, 0>) ? sizeof(T) : sizeof(cx<T>);
    const std::size_t lds = elt * (std::size_t)a.W * rb::lds_len(n);
    int gx = tiles;
    if (a.sym != 3 && a.bt.count == 1) {
        const void* f = a.sym == 0 ? (const void*)k_rb_cols<T, LOGN, LE, 0>
                        : a.sym == 1 ? (const void*)k_rb_cols<T, LOGN, LE, 1>
                                     : (const void*)k_rb_cols<T, LOGN, LE, 2>;
        allow_lds_rb(f, lds);
        gx = cols_grid(tiles, resident_blocks(f, block, lds));
    }
    const dim3 grid(gx, a.bt.count);
#define RC_ARGS a.AT, a.pitchT, a.lq, a.ncols, a.rows_in, a.rows_out, a.W, a.tw, a.ktab, a.kp, \
        a.sc, a.kout, a.part, a.remap, a.bt, a.kmap
#define RC_CASE(S)                                                     \
    case S: {                                                          \
        const void* fn = (const void*)k_rb_cols<T, LOGN, LE, S>;           \
        allow_lds_rb(fn, lds);                                         \
        k_rb_cols<T, LOGN, LE, S><<<grid, block, lds, s>>>(RC_ARGS);       \
        break;                                                         \
    }
    if (a.sym == 0 && (a.rows_in > n / 2 || a.rows_out > n / 2))
        throw std::invalid_argument("table symbol needs rows_in, rows_out <= n/2");
    if (a.rows_in > a.pitchT || a.rows_out > a.pitchT)
        throw std::invalid_argument("column transform: more rows than the panels hold");
    switch (a.sym) {
        RC_CASE(0)
        RC_CASE(1)
        RC_CASE(2)
        RC_CASE(3)
        default: throw std::invalid_argument("unknown symbol");
    }
#undef RC_CASE
#undef RC_ARGS
    ASPHER_LAUNCH_CHECK();
}

template <typename T, int LOGL, int LE>
void launch_rows_inv(const RbRowsInv<T>& a, hipStream_t s) {
    constexpr int L = 1 << LOGL;
    const RowEpilogue<T>& ep = a.epi;
    const bool ok = a.y && (a.mode == 0   ? true
                            : a.mode == 1 ? (a.mask && a.part)
                            : a.mode == 2 ? (ep.a && ep.b && ep.o && ep.part)
                            : a.mode == 3 ? (ep.a && ep.b && ep.mask && ep.part)
                                          : false);
    if (!ok) throw std::invalid_argument("row transform: missing operand for its output mode");
    check_panels(L >> LE, a.lq);
    const int block = a.B * (L >> LE);
    const dim3 grid((a.nrows + a.B - 1) / a.B, a.bt.count);
    const std::size_t lds = sizeof(cx<T>) * (std::size_t)a.B * row_stride<T>(L, a.B);
#define RI_ARGS a.AT, a.pitchT, a.lq, a.nrows, a.B, a.tw, a.y, a.y_pitch, a.ncols, a.mask, \
        a.part, a.remap, a.bt, a.epi
    if (a.mode == 0 && a.ncols <= L) {
        const void* fn = (const void*)k_rb_rows_inv<T, LOGL, LE, 0, true>;
        allow_lds_rb(fn, lds);
        k_rb_rows_inv<T, LOGL, LE, 0, true><<<grid, block, lds, s>>>(RI_ARGS);
    } else if (a.mode == 0) {
        const void* fn = (const void*)k_rb_rows_inv<T, LOGL, LE, 0, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_inv<T, LOGL, LE, 0, false><<<grid, block, lds, s>>>(RI_ARGS);
    } else if (a.mode >= 2) {
        if constexpr (LE == kSmallLE) {
            if (a.bt.count != 1 || ((a.y_pitch | a.ncols) & 1) ||
                !pair_aligned(a.y, sizeof(T)) || !pair_aligned(ep.a, sizeof(T)) ||
                !pair_aligned(ep.b, sizeof(T)) || !pair_aligned(ep.o, sizeof(T)) ||
                (reinterpret_cast<std::uintptr_t>(ep.mask) & 1u))
                throw std::invalid_argument("row transform: unaligned epilogue operand");
#define RI_EPI(OUT, H)                                                           \
    {                                                                            \
        const void* fn = (const void*)k_rb_rows_inv<T, LOGL, LE, OUT, H>;        \
        allow_lds_rb(fn, lds);                                                   \
        k_rb_rows_inv<T, LOGL, LE, OUT, H><<<grid, block, lds, s>>>(RI_ARGS);    \
    }
            if (a.mode == 2 && a.ncols <= L) RI_EPI(2, true)
            else if (a.mode == 2) RI_EPI(2, false)
            else if (a.ncols <= L) RI_EPI(3, true)
            else RI_EPI(3, false)
#undef RI_EPI
        } else {
            throw std::invalid_argument("row transform: epilogues are for short rows");
        }
    } else {
        const void* fn = (const void*)k_rb_rows_inv<T, LOGL, LE, 1, false>;
        allow_lds_rb(fn, lds);
        k_rb_rows_inv<T, LOGL, LE, 1, false><<<grid, block, lds, s>>>(RI_ARGS);
    }
#undef RI_ARGS
    ASPHER_LAUNCH_CHECK();
}


// ── two-component (tangential) column pass ───────────────────────────────
// One workgroup per column kx: threads [0, TPC) transform the x component
// (plan instance 0), threads [TPC, 2 TPC) the y component (instance 1). After
// the forward transforms both halves swap their spectra through LDS (the two
// components hold the same digit-reversed positions), mix them by the real
// symmetric 2x2 symbol and run their inverse transforms.
template <typename T, int LOGN, int SYM>
__global__ void __launch_bounds__(512)
k_rb_cols2(cx<T>* AT, int pitchT, int lq, std::int64_t at_stride, int ncols, int rows_in,
           int rows_out, const cx<double>* __restrict__ tw, const T* __restrict__ kxx,
           const T* __restrict__ kyy, const T* __restrict__ kxy, int kp, double gamma,
           double norm, int remap) {
    using Sh = rb::Shape<LOGN>;
    constexpr int n = Sh::n, TPC = Sh::threads;
    constexpr int LL = rb::lds_len(n);
    constexpr int Gl = Sh::G(Sh::m - 1), Nl = Sh::N(Sh::m - 1);
    constexpr bool ZP = (SYM == 5);
    extern __shared__ __align__(16) unsigned char smem[];
    const int kx = remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int c = threadIdx.x / TPC, th = threadIdx.x - c * TPC;
    const bool live = kx < ncols;
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem) + c * LL;
    const cx<T>* ldo = reinterpret_cast<cx<T>*>(smem) + (1 - c) * LL;

    cx<T> r[16];
    const int kl = live ? kx : 0;
    cx<T>* col = AT + c * at_stride + (((std::size_t)(kl >> lq) * pitchT) << lq) +
                 (kl & ((1 << lq) - 1));
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int p = Sh::pos(0, th, v);
        if (ZP && v >= 8) r[v] = {T(0), T(0)};
        else r[v] = (live && p < rows_in) ? col[(std::size_t)p << lq] : cx<T>{T(0), T(0)};
    }
    rb::forward<T, Sh, ZP>(r, lds, th, tw, 1);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) lds[rb::lds_ix(16 * th + i)] = r[i];
    __syncthreads();
    cx<T> o[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) o[i] = ldo[rb::lds_ix(16 * th + i)];
    if constexpr (SYM == 5) {
        const std::size_t at = (size_t)(live ? kx : 0) * kp + 16 * th;
        T kd[16], kc[16];
        loadv<16>((c == 0 ? kxx : kyy) + at, kd);
        loadv<16>(kxy + at, kc);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const T a = live ? kd[i] : T(0), b = live ? kc[i] : T(0);
            r[i] = {a * r[i].re + b * o[i].re, a * r[i].im + b * o[i].im};
        }
    } else {
#pragma unroll
        for (int q = 0; q < Gl; ++q)
#pragma unroll
            for (int v = 0; v < Nl; ++v) {
                const int i = q * Nl + v;
                const int ky = Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, v));
                const double fx = (double)kx;
                const double fy = (double)(ky < (n >> 1) ? ky : ky - n);
                const double k2 = fx * fx + fy * fy;
                double wd = 0.0, wc = 0.0;
                if (live && k2 > 0.0) {
                    const double kk = sqrt(k2);
                    const double f = c == 0 ? fx : fy;
                    wd = norm * kk * (1.0 + gamma * f * f / k2);
                    wc = (kx == (n >> 1) || ky == (n >> 1)) ? 0.0
                                                            : norm * kk * gamma * fx * fy / k2;
                }
                const T a = static_cast<T>(wd), b = static_cast<T>(wc);
                r[i] = {a * r[i].re + b * o[i].re, a * r[i].im + b * o[i].im};
            }
    }
    // the other component has read this one's spectrum before the inverse's
    // first exchange overwrites it (that exchange may be ordered within
    // each wave only)
    __syncthreads();
    rb::inverse<T, Sh, ZP>(r, lds, th, tw, 1);
    if (live) {
        // in place: this column's loads were consumed before the barriers
#pragma unroll
        for (int v = 0; v < (ZP ? 8 : 16); ++v) {
            const int p = Sh::pos(0, th, v);
            if (p < rows_out) col[(std::size_t)p << lq] = r[v];
        }
    }
}

template <typename T, int LOGN>
void launch_cols2(const RbCols2<T>& a, hipStream_t s) {
    constexpr int n = 1 << LOGN;
    static_assert(2 * (n / 16) <= 512, "two-component columns up to n = 4096");
    const int block = 2 * (n / 16);
    const int grid = a.ncols;
    const std::size_t lds = sizeof(cx<T>) * 2 * (std::size_t)rb::lds_len(n);
    if (a.sym == 5) {
        if (a.rows_in > n / 2 || a.rows_out > n / 2)
            throw std::invalid_argument("tangential columns need rows <= n/2");
        const void* fn = (const void*)k_rb_cols2<T, LOGN, 5>;
        allow_lds_rb(fn, lds);
        k_rb_cols2<T, LOGN, 5><<<grid, block, lds, s>>>(
            a.AT, a.pitchT, a.lq, a.at_stride, a.ncols, a.rows_in, a.rows_out,
            a.tw, a.kxx, a.kyy, a.kxy, a.kp, a.gamma, a.norm, a.remap);
    } else {
        const void* fn = (const void*)k_rb_cols2<T, LOGN, 6>;
        allow_lds_rb(fn, lds);
        k_rb_cols2<T, LOGN, 6><<<grid, block, lds, s>>>(
            a.AT, a.pitchT, a.lq, a.at_stride, a.ncols, a.rows_in, a.rows_out,
            a.tw, a.kxx, a.kyy, a.kxy, a.kp, a.gamma, a.norm, a.remap);
    }
    ASPHER_LAUNCH_CHECK();
}

// ── free-space kernel spectrum in the column kernel's register order ──────
// kout[kx*n + pos] = K(kx, ky) with ky = kidx(pos) the frequency that the
// forward column transform leaves at digit-reversed position pos, folded by
// evenness to the (n/2+1)-wide unique table kin[kx*kp + min(ky, n-ky)].
template <typename T, int LOGN>
__global__ void __launch_bounds__(256)
k_rb_permute_table(const T* __restrict__ kin, int kp, int nh, T* __restrict__ kout, bool odd) {
    using Sh = rb::Shape<LOGN>;
    constexpr int n = Sh::n;
    const std::int64_t total = (std::int64_t)nh * n;
    for (std::int64_t i = (std::int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (std::int64_t)gridDim.x * blockDim.x) {
        const int kx = (int)(i / n), pos = (int)(i - (std::int64_t)kx * n);
        const int ky = Sh::kidx(pos);
        const int kyp = (ky <= (n >> 1)) ? ky : n - ky;
        const T v = kin[(std::size_t)kx * kp + kyp];
        kout[i] = (odd && ky > (n >> 1)) ? T(-v) : v;
    }
}

template <typename T, int LOGN>
void launch_permute(const T* kin, int kp, int nh, T* kout, hipStream_t s, bool odd) {
    const std::int64_t total = (std::int64_t)nh * (1 << LOGN);
    const int grid = (int)std::min<std::int64_t>((total + 255) / 256, 65536);
    k_rb_permute_table<T, LOGN><<<grid, 256, 0, s>>>(kin, kp, nh, kout, odd);
    ASPHER_LAUNCH_CHECK();
}

template <typename T, int LOGN, int LE>
__global__ void __launch_bounds__(256)
k_rb_permute_table_half(const T* __restrict__ kin, int kp, int nh, const int* __restrict__ kmap,
                        int kph, T* __restrict__ kout) {
    using Sh = rb::Shape<LOGN, LE>;
    constexpr int n = Sh::n, Tn = Sh::threads, E = Sh::E;
    constexpr int Gl = Sh::G(Sh::m - 1), Nl = Sh::N(Sh::m - 1);
    const std::int64_t total = (std::int64_t)nh * n;
    for (std::int64_t i = (std::int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (std::int64_t)gridDim.x * blockDim.x) {
        const int kx = (int)(i / n), e = (int)(i - (std::int64_t)kx * n);
        const int th = e / E, j = e % E;
        const int km = kmap[th];
        if (km & 1) continue;   // this chunk is written by its forward reader
        const int q = j / Nl, v = j - q * Nl;
        const int ky = Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, v));
        const int kyp = (ky <= (n >> 1)) ? ky : n - ky;
        kout[(std::size_t)kx * kph + E * (km >> 1) + j] = kin[(std::size_t)kx * kp + kyp];
    }
}

template <typename T, int LOGN, int LE>
void launch_permute_half(const T* kin, int kp, int nh, const int* kmap, int kph, T* kout,
                         hipStream_t s) {
    const std::int64_t total = (std::int64_t)nh * (1 << LOGN);
    const int grid = (int)std::min<std::int64_t>((total + 255) / 256, 65536);
    k_rb_permute_table_half<T, LOGN, LE><<<grid, 256, 0, s>>>(kin, kp, nh, kmap, kph, kout);
    ASPHER_LAUNCH_CHECK();
}

// ── rough-surface generator: spectrum synthesis + inverse column pass ─────
__device__ __forceinline__ double hash_uniform(unsigned long long seed, unsigned long long idx) {
    // SplitMix64 output number idx of a generator seeded with `seed`
    unsigned long long z = seed + (idx + 1ull) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z = z ^ (z >> 31);
    return (double)(z >> 11) * 0x1.0p-53;
}

template <int LOGN>
__global__ void __launch_bounds__(512)
k_rb_gen_cols(cx<double>* __restrict__ AT, int pitchT, int lq, double hurst, double k_low,
              double k_high, double scale, unsigned long long seed,
              const cx<double>* __restrict__ tw, int W, int remap) {
    using Sh = rb::Shape<LOGN>;
    constexpr int n = Sh::n, TPC = Sh::threads, nh = n / 2 + 1;
    constexpr int LL = rb::lds_len(n);
    constexpr int Gl = Sh::G(Sh::m - 1), Nl = Sh::N(Sh::m - 1);
    extern __shared__ __align__(16) unsigned char smem[];
    const int tile = remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int c = threadIdx.x / TPC, th = threadIdx.x - c * TPC;
    const int kx = tile * W + c;
    const bool live = kx < nh;
    cx<double>* lds = reinterpret_cast<cx<double>*>(smem) + c * LL;
    const double two_pi = 6.283185307179586476925286766559;
    cx<double> r[16];
#pragma unroll
    for (int q = 0; q < Gl; ++q)
#pragma unroll
        for (int v = 0; v < Nl; ++v) {
            const int ky = Sh::kidx(Sh::pos(Sh::m - 1, th * Gl + q, v));
            cx<double> h = {0.0, 0.0};
            if (live) {
                const int mx = kx < n / 2 ? kx : kx - n;   // fftfreq order
                const int my = ky < n / 2 ? ky : ky - n;
                const double mag = sqrt((double)mx * mx + (double)my * my);
                if (mag >= k_low && mag <= k_high && mag > 0.0) {
                    const double A = 0.5 * scale * pow(mag, -(1.0 + hurst));
                    const int kxn = (n - kx) % n, kyn = (n - ky) % n;
                    const double p1 = two_pi * hash_uniform(seed, (unsigned long long)ky * n + kx);
                    const double p2 = two_pi * hash_uniform(seed, (unsigned long long)kyn * n + kxn);
                    double s1, c1, s2, c2;
                    sincos(p1, &s1, &c1);
                    sincos(p2, &s2, &c2);
                    h = {A * (c1 + c2), A * (s1 - s2)};
                }
            }
            r[q * Nl + v] = h;
        }
    rb::inverse<double, Sh>(r, lds, th, tw, 1);
    if (live) {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const int p = Sh::pos(0, th, v);
            AT[(((std::size_t)(kx >> lq) * pitchT + p) << lq) + (kx & ((1 << lq) - 1))] = r[v];
        }
    }
}

template <int LOGN>
void launch_gen(const RbGen& a, hipStream_t s) {
    constexpr int n = 1 << LOGN;
    const int block = a.W * (n / 16);
    const int grid = (n / 2 + 1 + a.W - 1) / a.W;
    const std::size_t lds = sizeof(cx<double>) * (std::size_t)a.W * rb::lds_len(n);
    const void* fn = (const void*)k_rb_gen_cols<LOGN>;
    allow_lds_rb(fn, lds);
    k_rb_gen_cols<LOGN><<<grid, block, lds, s>>>(a.AT, a.pitchT, a.lq, a.hurst, a.k_low, a.k_high,
                                                 a.scale, a.seed, a.tw, a.W, a.remap);
    ASPHER_LAUNCH_CHECK();
}
} // namespace

template <typename T>
void rb_rows_fwd(int logL, const RbRowsFwd<T>& a, hipStream_t s) {
    if (a.le == kSmallLE) {
        switch (logL) {
            case 4: launch_rows_fwd<T, 4, kSmallLE>(a, s); return;
            case 5: launch_rows_fwd<T, 5, kSmallLE>(a, s); return;
            case 6: launch_rows_fwd<T, 6, kSmallLE>(a, s); return;
            case 7: launch_rows_fwd<T, 7, kSmallLE>(a, s); return;
            case 8: launch_rows_fwd<T, 8, kSmallLE>(a, s); return;
            case 9: launch_rows_fwd<T, 9, kSmallLE>(a, s); return;
            default: break;
        }
        throw std::invalid_argument("row transform length out of range");
    }
    switch (logL) {
        case 4: launch_rows_fwd<T, 4, 4>(a, s); break;
        case 5: launch_rows_fwd<T, 5, 4>(a, s); break;
        case 6: launch_rows_fwd<T, 6, 4>(a, s); break;
        case 7: launch_rows_fwd<T, 7, 4>(a, s); break;
        case 8: launch_rows_fwd<T, 8, 4>(a, s); break;
        case 9: launch_rows_fwd<T, 9, 4>(a, s); break;
        case 10: launch_rows_fwd<T, 10, 4>(a, s); break;
        case 11: launch_rows_fwd<T, 11, 4>(a, s); break;
        case 12: launch_rows_fwd<T, 12, 4>(a, s); break;
        case 13: launch_rows_fwd<T, 13, 4>(a, s); break;
        default: throw std::invalid_argument("row transform length out of range");
    }
}

template <typename T>
void rb_cols(int logN, const RbCols<T>& a, hipStream_t s) {
    if (a.le == kSmallLE) {
        switch (logN) {
            case 5: launch_cols<T, 5, kSmallLE>(a, s); return;
            case 6: launch_cols<T, 6, kSmallLE>(a, s); return;
            case 7: launch_cols<T, 7, kSmallLE>(a, s); return;
            case 8: launch_cols<T, 8, kSmallLE>(a, s); return;
            case 9: launch_cols<T, 9, kSmallLE>(a, s); return;
            case 10: launch_cols<T, 10, kSmallLE>(a, s); return;
            default: break;
        }
        throw std::invalid_argument("column transform length out of range");
    }
    switch (logN) {
        case 5: launch_cols<T, 5, 4>(a, s); break;
        case 6: launch_cols<T, 6, 4>(a, s); break;
        case 7: launch_cols<T, 7, 4>(a, s); break;
        case 8: launch_cols<T, 8, 4>(a, s); break;
        case 9: launch_cols<T, 9, 4>(a, s); break;
        case 10: launch_cols<T, 10, 4>(a, s); break;
        case 11: launch_cols<T, 11, 4>(a, s); break;
        case 12: launch_cols<T, 12, 4>(a, s); break;
        case 13: launch_cols<T, 13, 4>(a, s); break;
        default: throw std::invalid_argument("column transform length out of range");
    }
}

template <typename T>
void rb_rows_inv(int logL, const RbRowsInv<T>& a, hipStream_t s) {
    if (a.le == kSmallLE) {
        switch (logL) {
            case 4: launch_rows_inv<T, 4, kSmallLE>(a, s); return;
            case 5: launch_rows_inv<T, 5, kSmallLE>(a, s); return;
            case 6: launch_rows_inv<T, 6, kSmallLE>(a, s); return;
            case 7: launch_rows_inv<T, 7, kSmallLE>(a, s); return;
            case 8: launch_rows_inv<T, 8, kSmallLE>(a, s); return;
            case 9: launch_rows_inv<T, 9, kSmallLE>(a, s); return;
            default: break;
        }
        throw std::invalid_argument("row transform length out of range");
    }
    switch (logL) {
        case 4: launch_rows_inv<T, 4, 4>(a, s); break;
        case 5: launch_rows_inv<T, 5, 4>(a, s); break;
        case 6: launch_rows_inv<T, 6, 4>(a, s); break;
        case 7: launch_rows_inv<T, 7, 4>(a, s); break;
        case 8: launch_rows_inv<T, 8, 4>(a, s); break;
        case 9: launch_rows_inv<T, 9, 4>(a, s); break;
        case 10: launch_rows_inv<T, 10, 4>(a, s); break;
        case 11: launch_rows_inv<T, 11, 4>(a, s); break;
        case 12: launch_rows_inv<T, 12, 4>(a, s); break;
        case 13: launch_rows_inv<T, 13, 4>(a, s); break;
        default: throw std::invalid_argument("row transform length out of range");
    }
}

template <typename T>
void rb_cols2(int logN, const RbCols2<T>& a, hipStream_t s) {
    switch (logN) {
        case 5: launch_cols2<T, 5>(a, s); break;
        case 6: launch_cols2<T, 6>(a, s); break;
        case 7: launch_cols2<T, 7>(a, s); break;
        case 8: launch_cols2<T, 8>(a, s); break;
        case 9: launch_cols2<T, 9>(a, s); break;
        case 10: launch_cols2<T, 10>(a, s); break;
        case 11: launch_cols2<T, 11>(a, s); break;
        case 12: launch_cols2<T, 12>(a, s); break;
        default: throw std::invalid_argument("two-component transform length out of range");
    }
}
template void rb_cols2<float>(int, const RbCols2<float>&, hipStream_t);
template void rb_cols2<double>(int, const RbCols2<double>&, hipStream_t);

void rb_gen_cols(int logN, const RbGen& a, hipStream_t s) {
    switch (logN) {
        case 5: launch_gen<5>(a, s); break;
        case 6: launch_gen<6>(a, s); break;
        case 7: launch_gen<7>(a, s); break;
        case 8: launch_gen<8>(a, s); break;
        case 9: launch_gen<9>(a, s); break;
        case 10: launch_gen<10>(a, s); break;
        case 11: launch_gen<11>(a, s); break;
        case 12: launch_gen<12>(a, s); break;
        case 13: launch_gen<13>(a, s); break;
        default: throw std::invalid_argument("surface size out of range");
    }
}

template <typename T>
void rb_permute_table(int logN, const T* kin, int kp, int nh, T* kout, hipStream_t s,
                      bool odd) {
    switch (logN) {
        case 5: launch_permute<T, 5>(kin, kp, nh, kout, s, odd); break;
        case 6: launch_permute<T, 6>(kin, kp, nh, kout, s, odd); break;
        case 7: launch_permute<T, 7>(kin, kp, nh, kout, s, odd); break;
        case 8: launch_permute<T, 8>(kin, kp, nh, kout, s, odd); break;
        case 9: launch_permute<T, 9>(kin, kp, nh, kout, s, odd); break;
        case 10: launch_permute<T, 10>(kin, kp, nh, kout, s, odd); break;
        case 11: launch_permute<T, 11>(kin, kp, nh, kout, s, odd); break;
        case 12: launch_permute<T, 12>(kin, kp, nh, kout, s, odd); break;
        case 13: launch_permute<T, 13>(kin, kp, nh, kout, s, odd); break;
        default: throw std::invalid_argument("column transform length out of range");
    }
}
template <typename T>
void rb_permute_table_half(int logN, int le, const T* kin, int kp, int nh, const int* kmap,
                           int kph, T* kout, hipStream_t s) {
    if (!kmap) throw std::invalid_argument("permute_table_half: no mirror map");
    if (le == kSmallLE) {
        switch (logN) {
            case 5: launch_permute_half<T, 5, kSmallLE>(kin, kp, nh, kmap, kph, kout, s); return;
            case 6: launch_permute_half<T, 6, kSmallLE>(kin, kp, nh, kmap, kph, kout, s); return;
            case 7: launch_permute_half<T, 7, kSmallLE>(kin, kp, nh, kmap, kph, kout, s); return;
            case 8: launch_permute_half<T, 8, kSmallLE>(kin, kp, nh, kmap, kph, kout, s); return;
            case 9: launch_permute_half<T, 9, kSmallLE>(kin, kp, nh, kmap, kph, kout, s); return;
            case 10: launch_permute_half<T, 10, kSmallLE>(kin, kp, nh, kmap, kph, kout, s); return;
            default: break;
        }
        throw std::invalid_argument("column transform length out of range");
    }
    switch (logN) {
        case 5: launch_permute_half<T, 5, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 6: launch_permute_half<T, 6, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 7: launch_permute_half<T, 7, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 8: launch_permute_half<T, 8, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 9: launch_permute_half<T, 9, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 10: launch_permute_half<T, 10, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 11: launch_permute_half<T, 11, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 12: launch_permute_half<T, 12, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        case 13: launch_permute_half<T, 13, 4>(kin, kp, nh, kmap, kph, kout, s); break;
        default: throw std::invalid_argument("column transform length out of range");
    }
}
template void rb_permute_table_half<float>(int, int, const float*, int, int, const int*, int,
                                           float*, hipStream_t);
template void rb_permute_table_half<double>(int, int, const double*, int, int, const int*, int,
                                            double*, hipStream_t);
template void rb_permute_table<float>(int, const float*, int, int, float*, hipStream_t, bool);
template void rb_permute_table<double>(int, const double*, int, int, double*, hipStream_t,
                                       bool);

template void rb_rows_fwd<float>(int, const RbRowsFwd<float>&, hipStream_t);
template void rb_rows_fwd<double>(int, const RbRowsFwd<double>&, hipStream_t);
template void rb_cols<float>(int, const RbCols<float>&, hipStream_t);
template void rb_cols<double>(int, const RbCols<double>&, hipStream_t);
template void rb_rows_inv<float>(int, const RbRowsInv<float>&, hipStream_t);
template void rb_rows_inv<double>(int, const RbRowsInv<double>&, hipStream_t);

} // namespace aspher
