// Launch interface of the mixed-radix spectral kernels (fft_mr.hpp).
#pragma once

#include "common.hpp"
#include "fft_mr.hpp"

#include <cstdint>
#include <vector>

namespace aspher {

// How the kernels run a complex transform of length L: in place (prime factors
// up to 13), with direct passes of prime factors up to 67 (FP32) or 97 between two
// buffers (Lc == L), or as a chirp convolution of smooth length Lc >= 2L - 1.
enum class MrKind : int { smooth = 0, prime = 1, chirp = 2 };

template <typename T>
struct MrDev {
    int L = 0, Lc = 0;
    MrKind kind = MrKind::smooth;
    int slots = 0;                           // LDS slots of one transform
    mr::Layout lay;
    const cx<double>* tw = nullptr;          // exp(-2 pi i t/Lc), t < Lc
    const unsigned short* pos = nullptr;     // frequency k -> position (direct)
    const unsigned short* kof = nullptr;     // position -> frequency (direct)
    const cx<T>* chirp = nullptr;            // exp(-pi i j^2/L), j < L
    const cx<T>* bhat = nullptr;             // spectrum of its conjugate, over Lc
    mr::Program fwd, inv, conv;              // conv: forward, symbol, inverse
};

// LDS slots between the transforms when `count` of them share a workgroup:
// they start P / count slots apart mod P (P = 16 slots of 16 bytes or 32 of
// 8, the span the LDS serves at once), so lanes of neighbouring transforms
// fall in distinct banks.
template <typename T>
__host__ __device__ inline int mr_stride(int slots, int count) {
    constexpr int P = sizeof(cx<T>) >= 16 ? 16 : 32;
    if (count < 2 || count > P) return slots;
    return slots + ((P / count - slots % P) % P + P) % P;
}

// LDS buffers of a transform, each of mr_stride(slots, count) per transform of a
// workgroup, all first buffers before all second ones.
__host__ __device__ inline int mr_buffers(MrKind k) { return k == MrKind::prime ? 2 : 1; }
template <typename T>
std::size_t mr_lds(const MrDev<T>& t, int count) {
    return sizeof(cx<T>) * (std::size_t)mr_buffers(t.kind) * count * mr_stride<T>(t.slots, count);
}

// Host side of the transforms of one plan: their factorisations and their
// device tables, laid out in one block and uploaded at once (a plan is made
// for every new operator, and each upload costs it about 20 us).
template <typename T>
class MrTransforms {
public:
    // lengths of the row and the column transform (equal: one transform)
    MrTransforms(int L_row, int L_col);
    ~MrTransforms();
    MrTransforms(const MrTransforms&) = delete;
    MrTransforms& operator=(const MrTransforms&) = delete;
    const MrDev<T>& row() const { return d_[0]; }
    const MrDev<T>& col() const { return d_[one_ ? 0 : 1]; }
    std::size_t bytes() const { return bytes_; }

private:
    MrDev<T> d_[2];
    bool one_ = false;
    void* block_ = nullptr;
    std::size_t bytes_ = 0;
};

// threads of each of `count` transforms of a workgroup, at most 512 together
template <typename T> int mr_threads(const MrDev<T>& t, int count);

// The radices of a length that is transformed directly, with the FP32-only ones or
// without, prime ones above 13 last; empty for L == 1 and any other length.
std::vector<int> mr_radices(int L, bool wide);
bool mr_smooth(int L);
// the smallest even smooth length >= at_least
int mr_smooth_side(int at_least);

// Half spectrum between the passes, in panels of Q = 1 << lq adjacent
// frequencies: value (kx, iy) at ((kx >> lq)*pitch + iy)*Q + kx % Q. A column
// workgroup owns one panel and moves it as one contiguous run; a row
// workgroup of B rows moves runs of B*Q values.
template <typename T>
struct MrRows {
    MrDev<T> t;                  // length n/2 (n even) or n (n odd, row pairs)
    int n = 0, nrows = 0, ncols = 0;
    int B = 1, lb = 0, threads = 64;   // row units per workgroup (B = 1 << lb)
    cx<T>* A = nullptr;
    int pitch = 0, lq = 0;
    const cx<double>* tw = nullptr;    // exp(-2 pi i t/n) of the split (n even)
    int mode = 0;                // in: 0 plain, 1 masked, 2 embedding; out: 0, 1
    const T* x = nullptr;
    T* y = nullptr;
    int row_pitch = 0;
    const std::uint8_t* mask = nullptr;
    const double* scal = nullptr;
    int gmean_idx = 0;
    const double* table = nullptr;
    int Ns_embed = 0;
    double* part = nullptr;
    int remap = 1;
};

template <typename T>
struct MrCols {
    MrDev<T> t;                  // length n
    int ncols = 0, rows_in = 0, rows_out = 0;
    cx<T>* A = nullptr;
    int pitch = 0, lq = 0, threads = 64;
    int sym = 0;                 // 0 table, 1 periodic, 2 precond, 3 build
    const T* ktab = nullptr;     // sym 0: nh rows of n values in position order
    int kp = 0;
    double sc = 0.0;
    T* kout = nullptr;
    double* part = nullptr;
    int remap = 1;
};

template <typename T> void mr_rows_fwd(const MrRows<T>& a, hipStream_t s);
template <typename T> void mr_rows_inv(const MrRows<T>& a, hipStream_t s);
template <typename T> void mr_cols(const MrCols<T>& a, hipStream_t s);
// unique (n/2+1)-wide spectrum -> nh rows of n values in position order
template <typename T>
void mr_permute_table(const MrDev<T>& t, const T* kin, int kp, int nh, T* kout, hipStream_t s);

} // namespace aspher
