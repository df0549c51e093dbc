// Spectral convolution kernels for the lengths the register-blocked kernels
// do not cover, on the mixed-radix LDS transforms of fft_mr.hpp. The three
// launches and their fusion are those of spectral_rb.hip:
//
//   rows_fwd : x rows -> half spectrum, panels of Q frequencies
//   cols     : panel -> forward, symbol, inverse -> the same panel
//   rows_inv : panels -> y rows
//
// A row of even length n is packed as n/2 complex values; two rows of odd
// length are packed as the real and imaginary parts of one transform.
//
// What bounds them: the VALU and the LDS round trips of the passes, at the few
// waves per SIMD that one transform's LDS and 128 registers leave; traffic is
// one read and one write of each intermediate. Measured against direct DFTs
// of every prime factor (index arithmetic modulo the length per term, columns
// read with a row's stride): free space 1000^2 FP64 336 -> 74 us a response,
// torus 1215^2 FP32 173 -> 61 us, torus 38^2 FP64 (P = 19) 262 -> 25 us, 501^2
// FP64 (chirp, P = 167) 19200 -> 57 us.
#include "embed.hpp"
#include "reduce.hpp"
#include "spectral_mr.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <map>
#include <mutex>

namespace aspher {

namespace {

__device__ __forceinline__ int xcd_block(int b, int G) {
    const int q = G >> 3, r = G & 7;
    const int x = b & 7;
    return x * q + (x < r ? x : r) + (b >> 3);
}

struct NoSym {
    template <int R, typename T>
    __device__ __forceinline__ void apply(cx<T>*, int) const {}
    template <typename T>
    __device__ __forceinline__ cx<T> value(cx<T> a, int) const { return a; }
};

// chirp spectrum (conjugated for the inverse transform)
template <typename T>
struct ChirpSym {
    const cx<T>* b;
    bool conj;
    template <int R>
    __device__ __forceinline__ void apply(cx<T>* a, int g) const {
#pragma unroll
        for (int v = 0; v < R; ++v) {
            cx<T> w = b[g * R + v];
            if (conj) w.im = -w.im;
            a[v] = a[v] * w;
        }
    }
};

template <typename T>
__device__ __forceinline__ T sym_value(int sym, int kx, int ky, int n, double sc) {
    if (sym == 1) {
        const int my = (ky < ((n + 1) >> 1)) ? ky : ky - n;
        const double m2 = (double)kx * kx + (double)my * my;
        return m2 > 0.0 ? static_cast<T>(sc / sqrt(m2)) : T(0);
    }
    const int kof = (ky < (n >> 1)) ? ky : ky - n;
    const float h = (float)sqrt((double)kx * kx + (double)kof * kof);
    const float w = (kx == 0 && ky == 0) ? 0.0f : (float)sc * h;
    return static_cast<T>(w);
}

// the operator's symbol at the R frequencies of group g of the last stage
template <typename T, int SYM>
struct ColSym {
    const T* row;                  // SYM 0: this column's table, position order
    const unsigned short* kof;
    int kx, n;
    double sc;
    template <int R>
    __device__ __forceinline__ void apply(cx<T>* a, int g) const {
        if constexpr (SYM == 0) {
#pragma unroll
            for (int v = 0; v < R; ++v) a[v] = scale(a[v], row[g * R + v]);
        } else {
            // the last digit of a position is the top digit of its frequency
            const int k0 = kof[g * R], dk = n / R;
#pragma unroll
            for (int v = 0; v < R; ++v)
                a[v] = scale(a[v], sym_value<T>(SYM, kx, k0 + v * dk, n, sc));
        }
    }
    // at one position
    __device__ __forceinline__ cx<T> value(cx<T> a, int p) const {
        if constexpr (SYM == 0) return scale(a, row[p]);
        else return scale(a, sym_value<T>(SYM, kx, kof[p], n, sc));
    }
};

// Runs a program on `buf`; prime passes go back and forth between it and `alt`.
// Returns the buffer that holds the result (the same one for every thread).
template <MrKind KIND, bool COL = false, typename T, typename Sym>
__device__ __forceinline__ cx<T>* run(const MrDev<T>& t, const mr::Program& pr, cx<T>* buf,
                                      cx<T>* alt, int th, int T_, const Sym& sym,
                                      const mr::Column<T>& col = mr::Column<T>{}) {
    for (int i = 0; i < pr.n; ++i) {
        if (KIND == MrKind::prime && pr.p[i].r > 16) {
            if constexpr (KIND == MrKind::prime)
                mr::prime_pass<T, COL>(pr.p[i], buf, alt, t.lay, t.Lc, th, T_, t.tw, col, sym);
            cx<T>* const done = alt;
            alt = buf;
            buf = done;
        } else {
            mr::run_any<T, COL>(pr.p[i], buf, t.lay, t.Lc, th, T_, t.tw, col, sym);
        }
        __syncthreads();
    }
    return buf;
}

// ── rows: real -> half spectrum ────────────────────────────────────────────
template <typename T, int IN, MrKind KIND>
__global__ void __launch_bounds__(512, 4) k_mr_rows_fwd(const MrRows<T> a) {
    constexpr bool BLUE = KIND == MrKind::chirp;
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem);
    const int n = a.n, L = a.t.L, Lc = a.t.Lc;
    const mr::Layout lay = a.t.lay;
    const bool packed = !(n & 1);
    const int LS = mr_stride<T>(a.t.slots, a.B);
    const int blk = a.remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int b = threadIdx.x / a.threads, th = threadIdx.x - b * a.threads;
    const int unit = blk * a.B + b;
    cx<T>* buf = lds + b * LS;
    T gmean = T(0);
    if constexpr (IN == 1) gmean = static_cast<T>(a.scal[a.gmean_idx]);
    auto load = [&](int row, int col) -> T {
        if (row >= a.nrows || col >= a.ncols) return T(0);
        if constexpr (IN == 2) {
            const int Ns = a.Ns_embed;
            const int ady = embed_offset(row, Ns, n), adx = embed_offset(col, Ns, n);
            if (ady < 0 || adx < 0) return T(0);
            return static_cast<T>(a.table[(std::size_t)ady * Ns + adx]);
        } else {
            const std::size_t i = (std::size_t)row * a.row_pitch + col;
            if constexpr (IN == 1) return a.mask[i] ? T(a.x[i] - gmean) : T(0);
            else return a.x[i];
        }
    };
    const int nz = packed ? (a.ncols + 1) >> 1 : a.ncols;   // nonzero inputs
    for (int j = th; j < Lc; j += a.threads) {
        cx<T> z = {T(0), T(0)};
        if (j < nz) {
            if (packed) z = {load(unit, 2 * j), load(unit, 2 * j + 1)};
            else z = {load(2 * unit, j), load(2 * unit + 1, j)};
            if constexpr (BLUE) z = z * a.t.chirp[j];
        }
        buf[lay.slot(j)] = z;
    }
    __syncthreads();
    cx<T>* res;
    if constexpr (BLUE)
        res = run<KIND>(a.t, a.t.conv, buf, buf, th, a.threads, ChirpSym<T>{a.t.bhat, false});
    else res = run<KIND>(a.t, a.t.fwd, buf, buf + a.B * LS, th, a.threads, NoSym{});
    const cx<T>* const out0 = lds + (res - buf);
    auto at = [&](const cx<T>* src, int k) -> cx<T> {
        if constexpr (BLUE) return src[lay.slot(k)] * a.t.chirp[k];
        else return src[lay.slot(a.t.pos[k])];
    };
    // frequencies k and L - k of the packed spectrum give X_k and X_{L-k}
    // (packed) or X_k of both rows of a pair; the Q frequencies of a panel
    // and the B rows are the fastest lanes, so a store is a run of B*Q values
    const int Q = 1 << a.lq;
    const int half = packed ? L >> 1 : (n - 1) >> 1;
    const int total = ((half >> a.lq) + 1) << (a.lq + a.lb);
    for (int e = threadIdx.x; e < total; e += blockDim.x) {
        const int bb = (e >> a.lq) & (a.B - 1);
        const int k = ((e >> (a.lq + a.lb)) << a.lq) + (e & (Q - 1));
        const int u = blk * a.B + bb;
        if (k > half) continue;
        const cx<T>* src = out0 + bb * LS;
        const int kc = (k == 0) ? 0 : L - k;
        const cx<T> Zk = at(src, k), Zc = conjg(at(src, kc));
        const cx<T> E = scale(Zk + Zc, T(0.5));
        const cx<T> D = Zk - Zc;
        const cx<T> O = {D.im * T(0.5), -D.re * T(0.5)};
        if (packed) {
            if (u >= a.nrows) continue;
            const cx<double> wd = a.tw[k];
            const cx<T> WO = cx<T>{static_cast<T>(wd.re), static_cast<T>(wd.im)} * O;
            a.A[((std::size_t)(k >> a.lq) * a.pitch + u) * Q + (k & (Q - 1))] = E + WO;
            const int k2 = L - k;
            if (k2 != k)
                a.A[((std::size_t)(k2 >> a.lq) * a.pitch + u) * Q + (k2 & (Q - 1))] =
                    conjg(E - WO);
        } else {
            cx<T>* out = a.A + ((std::size_t)(k >> a.lq) * a.pitch + 2 * u) * Q + (k & (Q - 1));
            if (2 * u < a.nrows) out[0] = E;
            if (2 * u + 1 < a.nrows) out[Q] = O;
        }
    }
}

// ── columns: forward . symbol . inverse, one panel per workgroup ──────────
template <typename T, int SYM, MrKind KIND>
__global__ void __launch_bounds__(512, 4) k_mr_cols(const MrCols<T> a) {
    constexpr bool BLUE = KIND == MrKind::chirp;
    extern __shared__ __align__(16) unsigned char smem[];
    const int L = a.t.L, Lc = a.t.Lc, Q = 1 << a.lq;
    const mr::Layout lay = a.t.lay;
    const int LS = mr_stride<T>(a.t.slots, Q);
    const int tile = a.remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int c = threadIdx.x & (Q - 1), th = threadIdx.x >> a.lq, T_ = a.threads;
    const int kx = tile * Q + c;
    const bool live = kx < a.ncols;
    cx<T>* buf = reinterpret_cast<cx<T>*>(smem) + c * LS;
    // the direct transforms read their first stage from the panel and write
    // their last one to it; a lane without a column has no rows
    const mr::Column<T> io{a.A + (std::size_t)tile * a.pitch * Q, a.lq, c,
                           live ? a.rows_in : 0, live ? a.rows_out : 0};
    if constexpr (SYM == 3) {
        // kernel-spectrum build (src/fft_operator.cpp:46-68): realness check
        // over every mode, Re/n^2 stored for ky in [0, n/2] (even in ky)
        run<KIND, true>(a.t, a.t.fwd, buf, buf + Q * LS, th, T_, NoSym{}, io);
        const double norm = 1.0 / ((double)L * (double)L);
        double mi = 0.0, mrr = 0.0;
        for (int ky = th; ky < L; ky += T_) {
            if (!live) break;
            const cx<T> z = buf[lay.slot(a.t.pos[ky])];
            mi = fmax(mi, fabs((double)z.im));
            mrr = fmax(mrr, fabs((double)z.re));
            if (ky <= (L >> 1))
                a.kout[(std::size_t)kx * a.kp + ky] = static_cast<T>(norm * (double)z.re);
        }
        double* red = reinterpret_cast<double*>(smem);
        mi = block_reduce<RMAX>(mi, red);
        if (threadIdx.x == 0) a.part[2 * blockIdx.x] = mi;
        mrr = block_reduce<RMAX>(mrr, red);
        if (threadIdx.x == 0) a.part[2 * blockIdx.x + 1] = mrr;
        return;
    } else if constexpr (BLUE) {
        for (int j = th; j < Lc; j += T_)
            buf[lay.slot(j)] = j < io.rows_in ? io.panel[io.at(j)] * a.t.chirp[j]
                                              : cx<T>{T(0), T(0)};
        __syncthreads();
        run<KIND>(a.t, a.t.conv, buf, buf, th, T_, ChirpSym<T>{a.t.bhat, false});
        // X_k = c_k y_k is multiplied by the symbol and by conj(c_k) for the
        // inverse: the chirps cancel
        for (int j = th; j < Lc; j += T_) {
            cx<T> z = {T(0), T(0)};
            if (j < L)
                z = scale(buf[lay.slot(j)], sym_value<T>(SYM, kx, j, L, a.sc));
            buf[lay.slot(j)] = z;
        }
        __syncthreads();
        run<KIND>(a.t, a.t.conv, buf, buf, th, T_, ChirpSym<T>{a.t.bhat, true});
    } else {
        const ColSym<T, SYM> sym{
            SYM == 0 ? a.ktab + (std::size_t)(live ? kx : 0) * a.kp : nullptr, a.t.kof, kx, L,
            a.sc};
        run<KIND, true>(a.t, a.t.conv, buf, buf + Q * LS, th, T_, sym, io);
    }
    if constexpr (BLUE)
        for (int j = th; j < io.rows_out; j += T_)
            io.panel[io.at(j)] = buf[lay.slot(j)] * conjg(a.t.chirp[j]);
}

// ── rows: half spectrum -> real ────────────────────────────────────────────
template <typename T, int OUT, MrKind KIND>
__global__ void __launch_bounds__(512, 4) k_mr_rows_inv(const MrRows<T> a) {
    constexpr bool BLUE = KIND == MrKind::chirp;
    extern __shared__ __align__(16) unsigned char smem[];
    cx<T>* lds = reinterpret_cast<cx<T>*>(smem);
    const int n = a.n, L = a.t.L, Lc = a.t.Lc;
    const mr::Layout lay = a.t.lay;
    const bool packed = !(n & 1);
    const int LS = mr_stride<T>(a.t.slots, a.B);
    const int blk = a.remap ? xcd_block(blockIdx.x, gridDim.x) : blockIdx.x;
    const int b = threadIdx.x / a.threads, th = threadIdx.x - b * a.threads;
    const int unit = blk * a.B + b;
    const int Q = 1 << a.lq;
    auto put = [&](cx<T>* dst, int k, cx<T> z) {
        if constexpr (BLUE) dst[lay.slot(k)] = z * conjg(a.t.chirp[k]);
        else dst[lay.slot(a.t.pos[k])] = z;
    };
    // packed: Z_k = (X_k + conj X_{L-k}) + i (X_k - conj X_{L-k}) W^{-k} and
    // its mirror Z_{L-k} from the same two values; Im of the DC and Nyquist
    // modes is ignored (c2r convention)
    const int half = packed ? L >> 1 : (n - 1) >> 1;
    const int total = ((half >> a.lq) + 1) << (a.lq + a.lb);
    for (int e = threadIdx.x; e < total; e += blockDim.x) {
        const int bb = (e >> a.lq) & (a.B - 1);
        const int k = ((e >> (a.lq + a.lb)) << a.lq) + (e & (Q - 1));
        const int u = blk * a.B + bb;
        if (k > half) continue;
        cx<T>* dst = lds + bb * LS;
        if (packed) {
            const int k2 = L - k;
            cx<T> Xk = {T(0), T(0)}, Xc = {T(0), T(0)};
            if (u < a.nrows) {
                Xk = a.A[((std::size_t)(k >> a.lq) * a.pitch + u) * Q + (k & (Q - 1))];
                Xc = a.A[((std::size_t)(k2 >> a.lq) * a.pitch + u) * Q + (k2 & (Q - 1))];
            }
            if (k == 0) {
                Xk.im = T(0);
                Xc.im = T(0);
            }
            Xc = conjg(Xc);
            const cx<double> wd = a.tw[k];
            const cx<T> S = Xk + Xc;
            const cx<T> D = (Xk - Xc) * cx<T>{static_cast<T>(wd.re), static_cast<T>(-wd.im)};
            put(dst, k, cx<T>{S.re - D.im, S.im + D.re});
            if (k != 0 && k2 != k) put(dst, k2, cx<T>{S.re + D.im, D.re - S.im});
        } else {
            cx<T> Xa = {T(0), T(0)}, Xb = {T(0), T(0)};
            const cx<T>* in = a.A + ((std::size_t)(k >> a.lq) * a.pitch + 2 * u) * Q +
                              (k & (Q - 1));
            if (2 * u < a.nrows) Xa = in[0];
            if (2 * u + 1 < a.nrows) Xb = in[Q];
            if (k == 0) {
                Xa.im = T(0);
                Xb.im = T(0);
            }
            put(dst, k, cx<T>{Xa.re - Xb.im, Xa.im + Xb.re});
            if (k != 0) put(dst, n - k, cx<T>{Xa.re + Xb.im, Xb.re - Xa.im});
        }
    }
    if constexpr (BLUE)
        for (int j = L + th; j < Lc; j += a.threads)
            lds[b * LS + lay.slot(j)] = cx<T>{T(0), T(0)};
    __syncthreads();
    cx<T>* buf = lds + b * LS;
    if constexpr (BLUE)
        buf = run<KIND>(a.t, a.t.conv, buf, buf, th, a.threads, ChirpSym<T>{a.t.bhat, true});
    else buf = run<KIND>(a.t, a.t.inv, buf, buf + a.B * LS, th, a.threads, NoSym{});
    double acc = 0.0;
    auto store = [&](int row, int col, T v) {
        if (row >= a.nrows || col >= a.ncols) return;
        const std::size_t i = (std::size_t)row * a.row_pitch + col;
        if constexpr (OUT == 1) {
            if (a.mask[i]) acc += (double)v;
            else v = T(0);
        }
        a.y[i] = v;
    };
    const int nz = packed ? (a.ncols + 1) >> 1 : a.ncols;
    for (int j = th; j < nz; j += a.threads) {
        cx<T> z = buf[lay.slot(j)];
        if constexpr (BLUE) z = z * conjg(a.t.chirp[j]);
        if (packed) {
            store(unit, 2 * j, z.re);
            store(unit, 2 * j + 1, z.im);
        } else {
            store(2 * unit, j, z.re);
            store(2 * unit + 1, j, z.im);
        }
    }
    if constexpr (OUT == 1) {
        // the transform's LDS is free once every thread is past its reads
        // (block_reduce begins with a barrier)
        double* red = reinterpret_cast<double*>(smem);
        acc = block_reduce<RSUM>(acc, red);
        if (threadIdx.x == 0) a.part[(std::size_t)blockIdx.x * kPartVals] = acc;
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
k_mr_permute(const unsigned short* __restrict__ kof, int n, const T* __restrict__ kin, int kp,
             int nh, T* __restrict__ kout) {
    const std::int64_t total = (std::int64_t)nh * n;
    for (std::int64_t i = (std::int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (std::int64_t)gridDim.x * blockDim.x) {
        const int kx = (int)(i / n), p = (int)(i - (std::int64_t)kx * n);
        const int ky = kof[p];
        kout[i] = kin[(std::size_t)kx * kp + (ky <= (n >> 1) ? ky : n - ky)];
    }
}

void allow_lds_mr(const void* fn, std::size_t bytes) {
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

// ── host: factorisation and tables ─────────────────────────────────────────

constexpr std::size_t kMaxLds = 160 * 1024;
constexpr int kRadix[] = {16, 15, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2};

// fewest passes first, then the smallest sum of radices
bool split(int L, bool wide, int most, int stages, int sum, int& best_stages, int& best_sum,
           std::vector<int>& cur, std::vector<int>& best) {
    if (L == 1) {
        if (stages < best_stages || (stages == best_stages && sum < best_sum)) {
            best_stages = stages;
            best_sum = sum;
            best = cur;
        }
        return true;
    }
    if (stages + 1 > best_stages || stages >= mr::kMaxStages) return false;
    bool any = false;
    for (int r : kRadix) {
        if (r > most || L % r || (!wide && (r == 12 || r > 13))) continue;
        cur.push_back(r);
        any = split(L / r, wide, r, stages + 1, sum + r, best_stages, best_sum, cur, best) || any;
        cur.pop_back();
    }
    return any;
}

// exp(-2 pi i num/den) in long double
std::complex<long double> unit_root(long long num, long long den) {
    const long double two_pi = 6.283185307179586476925286766559005768L;
    num %= den;
    if (num < 0) num += den;
    if (num == 0) return {1.0L, 0.0L};
    if (2 * num == den) return {-1.0L, 0.0L};
    if (4 * num == den) return {0.0L, -1.0L};
    if (4 * num == 3 * den) return {0.0L, 1.0L};
    const long double ang = two_pi * (long double)num / (long double)den;
    return {cosl(ang), -sinl(ang)};
}

int max_prime(bool wide) { return wide ? mr::kMaxPrime<float> : mr::kMaxPrime<double>; }

int largest_prime(int L) {
    int p = 2;
    while (p * p <= L) {
        if (L % p == 0) L /= p;
        else ++p;
    }
    return L;
}

// plain recursive mixed-radix DFT (host, once per length)
void host_fft(std::vector<std::complex<long double>>& x) {
    const int n = (int)x.size();
    if (n == 1) return;
    int r = n;
    for (int p = 2; p * p <= n; ++p)
        if (n % p == 0) {
            r = p;
            break;
        }
    const int m = n / r;
    std::vector<std::vector<std::complex<long double>>> sub(r);
    for (int j = 0; j < r; ++j) {
        sub[j].resize(m);
        for (int i = 0; i < m; ++i) sub[j][i] = x[(std::size_t)i * r + j];
        host_fft(sub[j]);
    }
    std::vector<std::complex<long double>> w(n);
    for (int t = 0; t < n; ++t) w[t] = unit_root(t, n);
    for (int k = 0; k < n; ++k) {
        std::complex<long double> s = 0.0L;
        for (int j = 0; j < r; ++j) s += sub[j][k % m] * w[(long long)j * k % n];
        x[k] = s;
    }
}

// Host tables of one length, kept for the process (built once per length).
struct HostTables {
    int Lc = 0;
    bool blue = false;
    std::vector<int> radix;
    std::vector<cx<double>> tw;
    std::vector<unsigned short> pos, kof;
    std::vector<std::complex<long double>> chirp, bhat;
    // skew of the LDS layout (mr::Layout): pad slots after every C positions
    int C = 1, pad = 0;
};

void choose_skew(HostTables& h, int lanes, int slots_max);

const HostTables& host_tables(int L, bool wide) {
    static std::mutex mu;
    static std::map<std::pair<int, bool>, HostTables> cache;
    std::lock_guard<std::mutex> lk(mu);
    const auto key = std::make_pair(L, wide);
    auto it = cache.find(key);
    if (it != cache.end()) return it->second;
    HostTables h;
    h.blue = largest_prime(L) > max_prime(wide);
    h.Lc = L;
    if (h.blue) {
        // the smooth length of the fewest passes among the next few
        int best = 0, cost = 1 << 30;
        for (int c = 2 * L - 1; c <= 2 * L + L / 8 + 16; ++c) {
            if (!mr_smooth(c) || (std::size_t)c * (wide ? 8 : 16) > kMaxLds) continue;
            const int k = (int)mr_radices(c, wide).size() * c;
            if (k < cost) {
                cost = k;
                best = c;
            }
        }
        h.Lc = best;
    }
    h.radix = mr_radices(h.Lc, wide);
    h.tw.resize(h.Lc);
    for (int t = 0; t < h.Lc; ++t) {
        const auto w = unit_root(t, h.Lc);
        h.tw[t] = {(double)w.real(), (double)w.imag()};
    }
    h.kof.resize(h.Lc);
    h.pos.resize(h.Lc);
    for (int p = 0; p < h.Lc; ++p) {
        int k = 0, P = 1, S = h.Lc, rest = p;
        for (int r : h.radix) {
            S /= r;
            k += (rest / S) * P;
            rest %= S;
            P *= r;
        }
        h.kof[p] = (unsigned short)k;
        h.pos[k] = (unsigned short)p;
    }
    if (h.blue) {
        h.chirp.resize(L);
        for (int j = 0; j < L; ++j) h.chirp[j] = unit_root((long long)j * j % (2LL * L), 2LL * L);
        std::vector<std::complex<long double>> b(h.Lc, 0.0L);
        for (int j = 0; j < L; ++j) {
            b[j] = std::conj(h.chirp[j]) / (long double)h.Lc;
            if (j) b[h.Lc - j] = b[j];
        }
        host_fft(b);
        h.bhat.resize(h.Lc);
        for (int p = 0; p < h.Lc; ++p) h.bhat[p] = b[h.kof[p]];
    }
    const int buffers = h.blue || mr_smooth(L) ? 1 : 2;
    choose_skew(h, wide ? 32 : 16, (int)(kMaxLds / (wide ? 8 : 16)) / buffers);
    return cache.emplace(key, std::move(h)).first->second;
}

// The skew with the fewest bank conflicts, C among the stage strides, counted
// over the accesses of one transform: `lanes` consecutive threads are served
// together and conflict where their slots agree mod `lanes`.
void choose_skew(HostTables& h, int lanes, int slots_max) {
    const int m = (int)h.radix.size(), Lc = h.Lc;
    std::vector<int> S(m + 1, 1);
    for (int j = m - 1; j >= 0; --j) S[j] = S[j + 1] * h.radix[j];   // S[j+1]: stride of j
    double best = 1e30;
    for (int c = 0; c < m; ++c)
        for (int pad = 0; pad <= 3; ++pad) {
            const int C = S[c + 1];
            if (pad == 0 ? c > 0 : C == 1) continue;
            if (Lc + pad * ((Lc - 1) / C) > slots_max) continue;
            auto slot = [&](int p) { return p + pad * (p / C); };
            double cost = 0.0;
            std::vector<int> hit(lanes);
            auto add = [&](auto pos, int count, double weight) {
                double sum = 0.0;
                int rounds = 0;
                for (int g0 = 0; g0 < count && rounds < 64; g0 += lanes, ++rounds) {
                    std::fill(hit.begin(), hit.end(), 0);
                    int worst = 0;
                    for (int l = 0; l < lanes && g0 + l < count; ++l)
                        worst = std::max(worst, ++hit[slot(pos(g0 + l)) % lanes]);
                    sum += worst;
                }
                if (rounds) cost += weight * sum / rounds;
            };
            for (int s = 0; s < m; ++s) {
                const int St = S[s + 1], r = h.radix[s];
                // one element of every group of the stage, and as many passes
                // over the elements either way
                add([&](int g) { return (g / St) * r * St + g % St; }, Lc / r, 2.0);
            }
            // natural-order accesses of a row transform's split
            if (!h.blue) add([&](int k) { return (int)h.pos[k]; }, Lc, 1.0);
            if (cost < best - 1e-9) {
                best = cost;
                h.C = C;
                h.pad = pad;
            }
        }
}

mr::Pass make_pass(const HostTables& h, int stage, bool fwd, bool inv) {
    mr::Pass p{};
    p.r = h.radix[stage];
    p.S = 1;
    for (std::size_t j = stage + 1; j < h.radix.size(); ++j) p.S *= h.radix[j];
    p.invS = 1.0f / (float)p.S;
    p.step = p.S % h.C == 0 ? p.S + h.pad * (p.S / h.C) : p.S;
    p.twstep = h.Lc / (p.r * p.S);
    p.fwd = fwd ? 1 : 0;
    p.inv = inv ? 1 : 0;
    p.invG = (float)p.r / (float)h.Lc;
    return p;
}

// The three programs of a transform. A column's convolution and its forward
// transform take their first stage from memory, the convolution gives its
// last one back there (Column; a chirp transform's passes stay in LDS).
void make_programs(const HostTables& h, mr::Program& fwd, mr::Program& inv, mr::Program& conv) {
    const int m = (int)h.radix.size();
    // a last stage of prime radix ends the forward transform with the symbol and
    // begins the inverse: two passes
    const bool apart = m > 0 && h.radix[m - 1] > 16;
    for (int s = 0; s < m; ++s) {
        fwd.p[fwd.n++] = make_pass(h, s, true, false);
        inv.p[inv.n++] = make_pass(h, m - 1 - s, false, true);
        conv.p[conv.n++] = make_pass(h, s, true, s == m - 1 && !apart);
    }
    if (apart) {
        conv.p[m - 1].sym = 1;
        conv.p[conv.n++] = make_pass(h, m - 1, false, true);
    }
    for (int s = m - 2; s >= 0; --s)
        conv.p[conv.n++] = make_pass(h, s, false, true);
    // an inverse prime pass leaves the twiddles of its inputs to the prime pass
    // before it, which applies each once
    for (mr::Program* pr : {&inv, &conv})
        for (int i = 1; i < pr->n; ++i) {
            const mr::Pass& p = pr->p[i];
            if (p.fwd || p.r <= 16 || p.S == 1) continue;
            mr::Pass& b = pr->p[i - 1];
            b.nr = p.r;
            b.nS = p.S;
            b.ntwstep = p.twstep;
            b.ninvS = p.invS;
        }
    if (m > 0 && !h.blue) {
        fwd.p[0].from_mem = 1;
        conv.p[0].from_mem = 1;
        conv.p[conv.n - 1].to_mem = 1;
    }
}

} // namespace

std::vector<int> mr_radices(int L, bool wide) {
    std::vector<int> cur, best, primes;
    for (int p = 17; p <= max_prime(wide); p += 2)
        while (L % p == 0 && largest_prime(p) == p) {
            primes.push_back(p);
            L /= p;
        }
    int bs = mr::kMaxStages + 1, bsum = 1 << 30;
    if (!split(L, wide, 16, 0, 0, bs, bsum, cur, best)) return {};
    // powers of two first: the strides of the later stages are then odd
    std::stable_sort(best.begin(), best.end(), [](int a, int b) {
        return (a & -a) > (b & -b);
    });
    best.insert(best.end(), primes.begin(), primes.end());
    return best;
}

bool mr_smooth(int L) {
    if (L < 1) return false;
    for (int p : {2, 3, 5, 7, 11, 13})
        while (L % p == 0) L /= p;
    return L == 1;
}

int mr_smooth_side(int at_least) {
    int n = at_least + (at_least & 1);
    while (!mr_smooth(n)) n += 2;
    return n;
}

template <typename T>
MrTransforms<T>::MrTransforms(int L_row, int L_col) : one_(L_row == L_col) {
    std::vector<unsigned char> block;
    // appends a table at a 16-byte boundary, returns its offset
    auto put = [&](const void* p, std::size_t bytes) {
        const std::size_t at = (block.size() + 15) / 16 * 16;
        block.resize(at + bytes);
        std::memcpy(block.data() + at, p, bytes);
        return at;
    };
    std::size_t tw[2], map[2], chirp[2];
    const int count = one_ ? 1 : 2;
    for (int i = 0; i < count; ++i) {
        const int L = i ? L_col : L_row;
        const HostTables& h = host_tables(L, mr::kWide<T>);
        MrDev<T>& d = d_[i];
        d.L = L;
        d.Lc = h.Lc;
        d.kind = h.blue ? MrKind::chirp : mr_smooth(L) ? MrKind::smooth : MrKind::prime;
        d.lay.pad = h.pad;
        d.lay.invC = 1.0f / (float)h.C;
        d.slots = h.Lc + h.pad * ((h.Lc - 1) / h.C);
        make_programs(h, d.fwd, d.inv, d.conv);
        tw[i] = put(h.tw.data(), sizeof(cx<double>) * h.tw.size());
        if (!h.blue) {
            map[i] = put(h.pos.data(), sizeof(unsigned short) * L);
            put(h.kof.data(), sizeof(unsigned short) * L);
        } else {
            std::vector<cx<T>> c(h.chirp.size() + h.bhat.size());
            auto cast = [](std::complex<long double> z) {
                return cx<T>{static_cast<T>(z.real()), static_cast<T>(z.imag())};
            };
            std::transform(h.chirp.begin(), h.chirp.end(), c.begin(), cast);
            std::transform(h.bhat.begin(), h.bhat.end(), c.begin() + L, cast);
            chirp[i] = put(c.data(), sizeof(cx<T>) * c.size());
        }
    }
    bytes_ = block.size();
    block_ = dev_alloc(bytes_);
    ASPHER_HIP(hipMemcpy(block_, block.data(), bytes_, hipMemcpyHostToDevice));
    const unsigned char* base = static_cast<const unsigned char*>(block_);
    for (int i = 0; i < count; ++i) {
        MrDev<T>& d = d_[i];
        d.tw = reinterpret_cast<const cx<double>*>(base + tw[i]);
        if (d.kind != MrKind::chirp) {
            d.pos = reinterpret_cast<const unsigned short*>(base + map[i]);
            d.kof = reinterpret_cast<const unsigned short*>(
                base + (map[i] + sizeof(unsigned short) * d.L + 15) / 16 * 16);
        } else {
            d.chirp = reinterpret_cast<const cx<T>*>(base + chirp[i]);
            d.bhat = d.chirp + d.L;
        }
    }
}

template <typename T>
MrTransforms<T>::~MrTransforms() {
    dev_free(block_, bytes_);
}

// what the threads of a prime pass share (prime_pass: four outputs each)
static int prime_items(int Lc, int r) { return Lc / r * (r / 4 + 1); }

template <typename T>
int mr_threads(const MrDev<T>& t, int count) {
    // between 24 and 4 elements per thread (or one thread for each four outputs of
    // a prime pass, where those are more: at the bound of 4 elements a few items
    // were left for a second turn, 148^2 FP32 62 -> 46 us a call): the fewest turns (a pass takes
    // ceil(groups/threads) turns of about r + 4 units), each of which costs
    // the issue of the workgroup's waves and a latency worth about four
    const int Lc = t.Lc;
    const int most = std::max(1, 512 / count);
    int items = (Lc + 3) / 4;
    for (int i = 0; i < t.fwd.n; ++i)
        if (t.fwd.p[i].r > 16) items = std::max(items, prime_items(Lc, t.fwd.p[i].r));
    const int hi = std::max(1, std::min(most, items));
    const int lo = std::max(1, std::min(hi, (Lc + 23) / 24));
    int best = hi;
    double cost = 1e30;
    for (int th = hi; th >= lo; --th) {
        const int waves = (th * count + 63) / 64;
        double c = 0.0;
        for (int i = 0; i < t.fwd.n; ++i) {
            const int r = t.fwd.p[i].r;
            if (r > 16) c += (double)((prime_items(Lc, r) + th - 1) / th) * (2 * r) * (waves + 4);
            else c += (double)((Lc / r + th - 1) / th) * (r + 4) * (waves + 4);
        }
        if (c < cost) {
            cost = c;
            best = th;
        }
    }
    return best;
}

template class MrTransforms<float>;
template class MrTransforms<double>;
template int mr_threads<float>(const MrDev<float>&, int);
template int mr_threads<double>(const MrDev<double>&, int);

template <typename T>
void mr_rows_fwd(const MrRows<T>& a, hipStream_t s) {
    const bool ok = a.mode == 0   ? a.x != nullptr
                    : a.mode == 1 ? (a.x && a.mask && a.scal)
                    : a.mode == 2 ? a.table != nullptr
                                  : false;
    if (!ok) throw std::invalid_argument("row transform: missing operand for its input mode");
    const int units = (a.n & 1) ? (a.nrows + 1) / 2 : a.nrows;
    const int grid = (units + a.B - 1) / a.B, block = a.B * a.threads;
    const std::size_t lds = mr_lds<T>(a.t, a.B);
#define RF_CASE(IN, BL)                                          \
    {                                                            \
        allow_lds_mr((const void*)k_mr_rows_fwd<T, IN, BL>, lds); \
        k_mr_rows_fwd<T, IN, BL><<<grid, block, lds, s>>>(a);    \
    }
    constexpr MrKind smooth = MrKind::smooth, prime = MrKind::prime, chirp = MrKind::chirp;
    if (a.mode == 2) {
        if (a.t.kind != smooth)
            throw std::logic_error("row transform: the embedding needs a smooth length");
        RF_CASE(2, smooth)
    } else if (a.t.kind == chirp) {
        if (a.mode == 0) RF_CASE(0, chirp)
        else RF_CASE(1, chirp)
    } else if (a.t.kind == prime) {
        if (a.mode == 0) RF_CASE(0, prime)
        else RF_CASE(1, prime)
    } else {
        if (a.mode == 0) RF_CASE(0, smooth)
        else RF_CASE(1, smooth)
    }
#undef RF_CASE
    ASPHER_LAUNCH_CHECK();
}

template <typename T>
void mr_rows_inv(const MrRows<T>& a, hipStream_t s) {
    const bool ok = a.y && (a.mode == 0 ? true : a.mode == 1 ? (a.mask && a.part) : false);
    if (!ok) throw std::invalid_argument("row transform: missing operand for its output mode");
    const int units = (a.n & 1) ? (a.nrows + 1) / 2 : a.nrows;
    const int grid = (units + a.B - 1) / a.B, block = a.B * a.threads;
    const std::size_t lds = mr_lds<T>(a.t, a.B);
#define RI_CASE(OUT, BL)                                          \
    {                                                             \
        allow_lds_mr((const void*)k_mr_rows_inv<T, OUT, BL>, lds); \
        k_mr_rows_inv<T, OUT, BL><<<grid, block, lds, s>>>(a);    \
    }
    if (a.t.kind == MrKind::chirp) {
        if (a.mode == 0) RI_CASE(0, MrKind::chirp)
        else RI_CASE(1, MrKind::chirp)
    } else if (a.t.kind == MrKind::prime) {
        if (a.mode == 0) RI_CASE(0, MrKind::prime)
        else RI_CASE(1, MrKind::prime)
    } else {
        if (a.mode == 0) RI_CASE(0, MrKind::smooth)
        else RI_CASE(1, MrKind::smooth)
    }
#undef RI_CASE
    ASPHER_LAUNCH_CHECK();
}

template <typename T>
void mr_cols(const MrCols<T>& a, hipStream_t s) {
    const int Q = 1 << a.lq;
    const int grid = (a.ncols + Q - 1) / Q, block = Q * a.threads;
    const std::size_t lds = mr_lds<T>(a.t, Q);
    if (a.rows_in > a.t.L || a.rows_out > a.t.L || a.rows_in > a.pitch || a.rows_out > a.pitch)
        throw std::invalid_argument("column transform: more rows than the transform holds");
    if (a.sym == 0 && !a.ktab) throw std::invalid_argument("column transform: no symbol table");
#define RC_CASE(SYM, BL)                                      \
    {                                                         \
        allow_lds_mr((const void*)k_mr_cols<T, SYM, BL>, lds); \
        k_mr_cols<T, SYM, BL><<<grid, block, lds, s>>>(a);    \
    }
    constexpr MrKind smooth = MrKind::smooth, prime = MrKind::prime, chirp = MrKind::chirp;
    if (a.sym == 0 || a.sym == 3) {
        if (a.t.kind != smooth)
            throw std::logic_error("column transform: a table symbol needs a smooth length");
        if (a.sym == 0) RC_CASE(0, smooth)
        else RC_CASE(3, smooth)
    } else if (a.t.kind == chirp) {
        if (a.sym == 1) RC_CASE(1, chirp)
        else RC_CASE(2, chirp)
    } else if (a.t.kind == prime) {
        if (a.sym == 1) RC_CASE(1, prime)
        else RC_CASE(2, prime)
    } else {
        if (a.sym == 1) RC_CASE(1, smooth)
        else RC_CASE(2, smooth)
    }
#undef RC_CASE
    ASPHER_LAUNCH_CHECK();
}

template <typename T>
void mr_permute_table(const MrDev<T>& t, const T* kin, int kp, int nh, T* kout, hipStream_t s) {
    if (t.kind != MrKind::smooth) throw std::logic_error("permute_table: needs a smooth length");
    const std::int64_t total = (std::int64_t)nh * t.L;
    const int grid = (int)std::min<std::int64_t>((total + 255) / 256, 65536);
    k_mr_permute<T><<<grid, 256, 0, s>>>(t.kof, t.L, kin, kp, nh, kout);
    ASPHER_LAUNCH_CHECK();
}

template void mr_rows_fwd<float>(const MrRows<float>&, hipStream_t);
template void mr_rows_fwd<double>(const MrRows<double>&, hipStream_t);
template void mr_rows_inv<float>(const MrRows<float>&, hipStream_t);
template void mr_rows_inv<double>(const MrRows<double>&, hipStream_t);
template void mr_cols<float>(const MrCols<float>&, hipStream_t);
template void mr_cols<double>(const MrCols<double>&, hipStream_t);
template void mr_permute_table<float>(const MrDev<float>&, const float*, int, int, float*,
                                      hipStream_t);
template void mr_permute_table<double>(const MrDev<double>&, const double*, int, int, double*,
                                       hipStream_t);

} // namespace aspher
