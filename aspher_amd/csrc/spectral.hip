// Plans of the spectral convolutions (see spectral.hpp for the pipeline):
// which kernels a transform size takes, its tiling, workspaces and tables.
// Powers of two from 32 to 8192 run on the register-blocked kernels
// (spectral_rb.hip), every other length on the mixed-radix LDS kernels
// (spectral_mr.hip).
#include "spectral.hpp"

#include "spectral_mr.hpp"
#include "spectral_rb.hpp"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>

namespace aspher {

namespace {

int ilog2(int v) {
    int l = 0;
    while ((1 << l) < v) ++l;
    return l;
}

constexpr std::size_t kMaxLds = 160 * 1024;

} // namespace

namespace {
[[noreturn]] void too_large() {
    throw std::invalid_argument("non power-of-two transform length too large for LDS");
}
} // namespace

void check_side(int n) {
    if (!is_pow2(n) && 2 * (std::size_t)(n + 1) * sizeof(cx<double>) > kMaxLds) too_large();
}

int free_space_side(int Ns) {
    check_side(2 * Ns);
    return is_pow2(2 * Ns) || mr_smooth(2 * Ns) ? 2 * Ns : mr_smooth_side(2 * Ns - 1);
}

bool is_pow2(int n) { return n > 0 && (n & (n - 1)) == 0; }

// exp(-2 pi i t/n), t < n: evaluated once per n in long double (n long-double
// sin/cos cost ~1.5 ms at n = 8192, and every operator build creates several
// plans) and kept for the process
const std::vector<cx<double>>& twiddle_host(int n) {
    static std::mutex mu;
    static std::map<int, std::vector<cx<double>>> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(n);
    if (it != cache.end()) return it->second;
    std::vector<cx<double>> h(n);
    const long double two_pi = 6.283185307179586476925286766559005768L;
    for (int t = 0; t < n; ++t) {
        long long a = t, N = n;
        // angle = 2 pi a / N ; use exact symmetries where they apply
        long double ang = two_pi * (long double)a / (long double)N;
        long double c = cosl(ang), s = sinl(ang);
        if (4 * a == N) { c = 0; s = 1; }
        if (2 * a == N) { c = -1; s = 0; }
        if (4 * a == 3 * N) { c = 0; s = -1; }
        if (a == 0) { c = 1; s = 0; }
        h[t] = {static_cast<double>(c), static_cast<double>(-s)};
    }
    return cache.emplace(n, std::move(h)).first->second;
}

Twiddles::Twiddles(int n_) : n(n_) {
    const std::vector<cx<double>>& h = twiddle_host(n);
    dev = static_cast<cx<double>*>(dev_alloc(sizeof(cx<double>) * n));
    ASPHER_HIP(hipMemcpy(dev, h.data(), sizeof(cx<double>) * n, hipMemcpyHostToDevice));
}

Twiddles::~Twiddles() {
    dev_free(dev, sizeof(cx<double>) * n);
}

// Mirror map of the register-blocked column transform of length n = 2^logn
// (host restatement of rb::Shape): for each column thread t, the chunk of the
// half-size symbol table holding its E = 2^le values and whether it reads them
// reversed. Thread t' is t's mirror when it holds the frequencies n - ky of
// t's registers i at registers E - 1 - i; a pair shares one chunk (the lower
// thread reads it forward), every other thread gets a chunk of its own.
// Evaluated once per size for the process.
const std::vector<int>& mirror_map(int logn, int le, int& nchunks) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, std::pair<std::vector<int>, int>> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find({logn, le});
    if (it == cache.end()) {
        const int n = 1 << logn, E = 1 << le, A = logn / le, RL = logn % le;
        const int m = A + (RL ? 1 : 0);
        int N[8], S[8], P[8];
        for (int j = 0; j < m; ++j) N[j] = j < A ? E : (1 << RL);
        for (int j = 0; j < m; ++j) {
            S[j] = 1;
            for (int i = j + 1; i < m; ++i) S[j] *= N[i];
            P[j] = 1;
            for (int i = 0; i < j; ++i) P[j] *= N[i];
        }
        auto pos = [&](int st, int g, int v) {
            return (g / S[st]) * N[st] * S[st] + v * S[st] + g % S[st];
        };
        auto kidx = [&](int p) {
            int k = 0;
            for (int j = 0; j < m; ++j) k += ((p / S[j]) % N[j]) * P[j];
            return k;
        };
        const int Tn = n / E, Nl = N[m - 1], Gl = E / Nl;
        std::vector<int> ky((std::size_t)Tn * E), own_t(n), own_i(n);
        for (int t = 0; t < Tn; ++t)
            for (int q = 0; q < Gl; ++q)
                for (int v = 0; v < Nl; ++v) {
                    const int i = q * Nl + v, k = kidx(pos(m - 1, t * Gl + q, v));
                    ky[(std::size_t)t * E + i] = k;
                    own_t[k] = t;
                    own_i[k] = i;
                }
        std::vector<int> km(Tn, -1);
        int nc = 0;
        for (int t = 0; t < Tn; ++t) {
            if (km[t] >= 0) continue;
            const int tp = own_t[(n - ky[(std::size_t)t * E]) % n];
            bool pair = tp > t && km[tp] < 0;
            for (int i = 0; i < E && pair; ++i) {
                const int k2 = (n - ky[(std::size_t)t * E + i]) % n;
                pair = own_t[k2] == tp && own_i[k2] == E - 1 - i;
            }
            km[t] = nc << 1;
            if (pair) km[tp] = (nc << 1) | 1;
            ++nc;
        }
        it = cache.emplace(std::make_pair(logn, le), std::make_pair(std::move(km), nc)).first;
    }
    nchunks = it->second.second;
    return it->second.first;
}

int column_width(int want, int threads, std::size_t lds) {
    int W = 1;
    while (2 * W <= want && 2 * W * threads <= 512 && 2 * W * lds <= 98304) W *= 2;
    return W;
}

int transform_le(int len, int count, int batch, int longest) {
    return len <= longest && (std::int64_t)len * count * batch <= 600000 ? kSmallLE : 4;
}

template <typename T>
SpectralPlan<T>::SpectralPlan(int n_, int rin, int cin, int rout, int cout,
                              SpectralTuning tune, int batch)
    : n(n_), rows_in(rin), cols_in(cin), rows_out(rout), cols_out(cout), batch_(batch) {
    if (n < 2) throw std::invalid_argument("transform size must be >= 2");
    if (batch < 1) throw std::invalid_argument("batch must be >= 1");
    nh = n / 2 + 1;
    const bool packed = (n % 2 == 0);
    const int Lr = packed ? n / 2 : n;
    logn_ = ilog2(n);
    xcd_remap_ = tune.xcd_remap;
    const std::size_t cs = sizeof(cx<T>);
    rb_ = is_pow2(n) && n >= 32 && n <= 8192;
    if (rb_) {
        // threads per row/column are L/16 resp. n/16; the inverse row pass
        // aims for 256-thread workgroups (more resident ones: 6% faster than
        // 512 at 4096^2 FP32), the column pass for 512, while the LDS of one
        // workgroup stays <= 96 KiB
        const std::size_t rowlds = cs * (std::size_t)(Lr + Lr / 16 + 1);
        const std::size_t collds = cs * (std::size_t)(n + n / 16 + 1);
        row_le_ = transform_le(Lr, std::max(rows_in, rows_out), batch, 512);
        col_le_ = transform_le(n, nh, batch, 1024);
        const int TR = Lr >> row_le_, TC = n >> col_le_;
        int B = tune.row_batch > 0 ? tune.row_batch : std::max(1, 256 / TR);
        while (B > 1 && (B * TR > 512 || B * rowlds > 98304)) --B;
        const int W = column_width(tune.col_width > 0 ? tune.col_width : std::max(1, 512 / TC),
                                   TC, collds);
        if (B * TR > 512 || W * TC > 512 || B * rowlds > kMaxLds ||
            W * collds > kMaxLds)
            throw std::invalid_argument("spectral tiling exceeds the workgroup limits");
        row_batch_ = B;
        col_width_ = W;
        // the forward row pass writes the half spectrum in runs of B rows by
        // one panel: it takes as many rows as 1024 threads and 144 KiB of LDS
        // allow (one resident workgroup), measured faster than two smaller
        // ones; the inverse pass keeps B (more resident workgroups)
        int Bf = tune.row_batch > 0 ? B : std::max(1, 1024 / TR);
        while (tune.row_batch <= 0 && Bf > B && Bf * rowlds > 147456) --Bf;
        row_batch_fwd_ = std::max(Bf, B);
        // small transforms: the batches above would put a whole pass in one
        // or two workgroups (64 rows of a 128-point transform in one
        // 1024-thread group), so they are halved until a pass has 256
        // workgroups (one per CU) or a single row/column each. Measured on
        // the nested 4096^2 solves (levels 64^2 .. 1024^2): mixed with the
        // Fourier engine 0.0904 -> 0.0875 s, with the stencil 0.3455 ->
        // 0.3436 s; targets of 16 and 64 groups gained less. Columns are
        // spread to four groups per CU: at n = 2048, 256 groups of four
        // columns are one round and a last group alone (free space 1024^2
        // FP32 column pass 26.6 us; 512 groups 15.6, 1024 groups 14.4; FP64
        // 22.4 -> 19.9; torus 2048^2 FP32 32.3 -> 20.4, FP64 28.9 -> 25.6).
        {
            const int nr = std::max(rows_in, rows_out);
            auto spread = [](int v, int count, int target) {
                while (v > 1 && (count + v - 1) / v < target) v = (v + 1) / 2;
                return v;
            };
            if (tune.row_batch <= 0) {
                row_batch_ = spread(row_batch_, nr, 256);
                row_batch_fwd_ = std::max(spread(row_batch_fwd_, nr, 256), row_batch_);
            }
            if (tune.col_width <= 0) col_width_ = spread(col_width_, nh, 1024);
        }
        pitchT_ = (std::max(rows_in, rows_out) + 31) / 32 * 32 + 32;
        // Panels as wide as a workgroup's columns, up to 64 bytes of adjacent
        // frequencies. Where a workgroup takes one column, a panel of two is
        // shared by two workgroups: the column pass then moves halves of 32
        // byte runs, the rows store twice the run. At n = 8192 the rows gain
        // more (FP64, free space 4096^2: rows 149 + 163 -> 115 + 135 us,
        // columns 197 -> 210; FP32 237 -> 219 us in all), at n = 4096 less
        // (FP64, free space 2048^2: 98.8 -> 101.3 us; torus 4096^2 equal).
        // Panels of four lose at both (columns 235 us at n = 8192).
        lq_ = 0;
        while ((2 << lq_) <= std::min(col_width_, TR) && (2 << lq_) * (int)cs <= 64) ++lq_;
        if (col_width_ == 1 && n == 8192) lq_ = 1;
        row_batch_inv_ = std::min(row_batch_fwd_, std::max(row_batch_, 2));
        tw64_ = std::make_unique<Twiddles>(n);
        at_stride_ = (std::int64_t)((nh + (1 << lq_) - 1) >> lq_) * ((std::int64_t)pitchT_ << lq_);
        at_bytes_ = cs * (std::size_t)at_stride_ * batch_;
        AT_ = static_cast<cx<T>*>(dev_alloc(at_bytes_));
        const std::vector<int>& km = mirror_map(logn_, col_le_, kmap_chunks_);
        kmap_ = static_cast<int*>(dev_alloc(sizeof(int) * km.size()));
        ASPHER_HIP(hipMemcpy(kmap_, km.data(), sizeof(int) * km.size(), hipMemcpyHostToDevice));
        return;
    }
    if (batch_ != 1)
        throw std::invalid_argument("batched transforms need a power-of-two length in [32, 8192]");
    if (is_pow2(n) && n > 8192)
        throw std::invalid_argument("transform length exceeds the LDS capacity");
    if (!is_pow2(n) && 2 * (std::size_t)n * cs > kMaxLds) too_large();
    mr_ = std::make_unique<MrTransforms<T>>(Lr, n);
    // rows and columns per workgroup: as many as 80 KiB of LDS (two resident
    // workgroups) take, runs of at most 64 bytes of adjacent frequencies, and
    // 256 workgroups (one per CU) or one row or column each
    auto share = [&](const MrDev<T>& t, int count, int most) {
        int lg = 0;
        while ((2 << lg) <= most &&
               mr_lds<T>(t, 2 << lg) <= kMaxLds / 2 &&
               (count + (2 << lg) - 1) / (2 << lg) >= 256)
            ++lg;
        return lg;
    };
    const int units = packed ? std::max(rows_in, rows_out) : (std::max(rows_in, rows_out) + 1) / 2;
    lq_ = share(mr_->col(), nh, (int)(64 / cs));
    lb_ = share(mr_->row(), units, 8);
    col_width_ = 1 << lq_;
    row_batch_ = 1 << lb_;
    // an odd number of 16-row steps, so panels do not start on one channel
    pitchT_ = ((std::max(rows_in, rows_out) + 15) / 16 | 1) * 16;
    // the split of even rows reads the column transform's table, except where
    // that one is of a chirp convolution's length
    if (packed && mr_->col().kind == MrKind::chirp) tw64_ = std::make_unique<Twiddles>(n);
    at_bytes_ = cs * ((std::size_t)(nh + col_width_ - 1) / col_width_) * pitchT_ * col_width_;
    AT_ = static_cast<cx<T>*>(dev_alloc(at_bytes_));
}

template <typename T>
SpectralPlan<T>::~SpectralPlan() {
    dev_free(AT_, at_bytes_);
    if (kmap_) dev_free(kmap_, sizeof(int) * (std::size_t)(n >> col_le_));
}

template <typename T>
std::size_t SpectralPlan<T>::external_ws_bytes() const {
    return rb_ ? sizeof(cx<T>) * (std::size_t)at_stride_ : 0;
}

template <typename T>
std::size_t SpectralPlan<T>::workspace_bytes() const {
    if (!rb_) return at_bytes_ + mr_->bytes();
    return at_bytes_ + sizeof(cx<double>) * n;
}

template <typename T>
void SpectralPlan<T>::generate_surface(double hurst, double k_low, double k_high, double scale,
                                       unsigned long long seed, T* out, hipStream_t s) {
    if constexpr (!std::is_same_v<T, double>) {
        throw std::logic_error("generate_surface: FP64 plans only");
    } else {
        if (!rb_ || rows_in != n || rows_out != n || cols_in != n || cols_out != n)
            throw std::invalid_argument(
                "generate_surface: needs a power-of-two n x n plan, 32 <= n <= 8192");
        RbGen g;
        g.AT = AT_;
        g.pitchT = pitchT_;
        g.lq = lq_;
        g.hurst = hurst;
        g.k_low = k_low;
        g.k_high = k_high;
        g.scale = scale;
        g.seed = seed;
        g.tw = tw64_->dev;
        g.W = col_width_;
        g.remap = xcd_remap_ ? 1 : 0;
        rb_gen_cols(logn_, g, s);
        RbRowsInv<double> r;
        r.AT = AT_;
        r.pitchT = pitchT_;
        r.lq = lq_;
        r.nrows = n;
        r.B = row_batch_inv_;
    r.le = row_le_;
        r.tw = tw64_->dev;
        r.y = out;
        r.y_pitch = n;
        r.ncols = n;
        r.mode = 0;
        r.remap = g.remap;
        rb_rows_inv<double>(ilog2(n / 2), r, s);
    }
}

template <typename T>
void SpectralPlan<T>::permute_table(const T* kunique, int kp, T* kout, hipStream_t s,
                                    bool odd) const {
    if (!rb_) {
        if (odd) throw std::invalid_argument("permute_table: odd tables need a power-of-two plan");
        mr_permute_table<T>(mr_->col(), kunique, kp, nh, kout, s);
        return;
    }
    rb_permute_table<T>(logn_, kunique, kp, nh, kout, s, odd);
}

template <typename T>
void SpectralPlan<T>::permute_table_half(const T* kunique, int kp, T* kout,
                                         hipStream_t s) const {
    if (!rb_) throw std::logic_error("permute_table_half: register-blocked plans only");
    rb_permute_table_half<T>(logn_, col_le_, kunique, kp, nh, kmap_, table_pitch_half(), kout, s);
}

template <typename T>
int SpectralPlan<T>::row_out_blocks() const {
    if (rb_) return (rows_out + row_batch_inv_ - 1) / row_batch_inv_;
    const int units = n % 2 == 0 ? rows_out : (rows_out + 1) / 2;
    return (units + row_batch_ - 1) / row_batch_;
}

template <typename T>
int SpectralPlan<T>::col_blocks() const {
    return (nh + col_width_ - 1) / col_width_;
}

template <typename T>
MrRows<T> SpectralPlan<T>::mr_rows() const {
    MrRows<T> a;
    a.t = mr_->row();
    a.n = n;
    a.B = row_batch_;
    a.lb = lb_;
    a.threads = mr_threads<T>(a.t, 1 << lb_);
    a.A = AT_;
    a.pitch = pitchT_;
    a.lq = lq_;
    a.tw = tw64_ ? tw64_->dev : mr_->col().tw;
    a.remap = xcd_remap_ ? 1 : 0;
    return a;
}

template <typename T>
MrCols<T> SpectralPlan<T>::mr_columns() const {
    MrCols<T> a;
    a.t = mr_->col();
    a.ncols = nh;
    a.A = AT_;
    a.pitch = pitchT_;
    a.lq = lq_;
    a.threads = mr_threads<T>(a.t, 1 << lq_);
    a.remap = xcd_remap_ ? 1 : 0;
    return a;
}

template <typename T>
void SpectralPlan<T>::convolve(const T* x, int x_pitch, T* y, int y_pitch, Symbol sym,
                               const T* ktab, int ktab_pitch, double sym_scale,
                               hipStream_t s, RowIn in_mode, RowOut out_mode,
                               const std::uint8_t* mask, const double* scal,
                               int gmean_idx, double* part, hipEvent_t* ev,
                               const SpecBatch* sb, void* ext_ws,
                               const RowEpilogue<T>* epi) {
    const int out_code = static_cast<int>(out_mode);
    if (out_code >= 2 && (!epi || !epilogues()))
        throw std::invalid_argument("convolve: this plan takes no epilogue");
    if (sym == Symbol::build) throw std::invalid_argument("convolve: build symbol");
    if (sb && (!rb_ || sb->count > batch_ || sb->count < 1))
        throw std::invalid_argument("convolve: batch exceeds the plan");
    if (ext_ws && (!rb_ || sb))
        throw std::invalid_argument("convolve: caller workspace needs a single-instance "
                                    "register-blocked plan");
    if (rb_) {
        // intermediate spectrum: the plan's own, or the caller's workspace
        cx<T>* ws_at = ext_ws ? static_cast<cx<T>*>(ext_ws) : AT_;
        RbBatch bt;
        if (sb) {
            bt.count = sb->count;
            bt.x_stride = sb->x_stride;
            bt.y_stride = sb->y_stride;
            bt.at_stride = at_stride_;
            bt.first = sb->first;
            bt.sstride = sb->sstride;
            bt.pstride = sb->pstride;
            bt.gscal = sb->gscal;
            bt.gate = sb->gate;
        }
        const int Lr = n / 2;
        RbRowsFwd<T> f;
        f.x = x;
        f.x_pitch = x_pitch;
        f.ncols = cols_in;
        f.nrows = rows_in;
        f.AT = ws_at;
        f.pitchT = pitchT_;
        f.lq = lq_;
        f.B = row_batch_fwd_;
    f.le = row_le_;
        f.tw = tw64_->dev;
        f.mode = in_mode == RowIn::masked ? 1 : 0;
        f.mask = mask;
        f.scal = scal;
        f.gmean_idx = gmean_idx;
        f.remap = xcd_remap_ ? 1 : 0;
        f.bt = bt;
        RbCols<T> c;
        c.bt = bt;
        c.AT = ws_at;
        c.pitchT = pitchT_;
        c.lq = lq_;
        c.ncols = nh;
        c.rows_in = rows_in;
        c.rows_out = rows_out;
        c.W = col_width_;
        c.le = col_le_;
        c.tw = f.tw;
        c.sym = static_cast<int>(sym);
        c.ktab = ktab;
        c.kp = ktab_pitch;
        c.kmap = kmap_;
        c.sc = sym_scale;
        c.remap = f.remap;
        RbRowsInv<T> r;
        r.AT = ws_at;
        r.pitchT = pitchT_;
        r.lq = lq_;
        r.nrows = rows_out;
        r.B = row_batch_inv_;
    r.le = row_le_;
        r.tw = f.tw;
        r.y = y;
        r.y_pitch = y_pitch;
        r.ncols = cols_out;
        r.mode = out_code;
        if (epi) r.epi = *epi;
        r.mask = mask;
        r.part = part;
        r.remap = f.remap;
        r.bt = bt;
        if (ev) ASPHER_HIP(hipEventRecord(ev[0], s));
        rb_rows_fwd<T>(ilog2(Lr), f, s);
        if (ev) ASPHER_HIP(hipEventRecord(ev[1], s));
        rb_cols<T>(logn_, c, s);
        if (ev) ASPHER_HIP(hipEventRecord(ev[2], s));
        rb_rows_inv<T>(ilog2(Lr), r, s);
        if (ev) ASPHER_HIP(hipEventRecord(ev[3], s));
        return;
    }
    MrRows<T> f = mr_rows();
    f.nrows = rows_in;
    f.ncols = cols_in;
    f.x = x;
    f.row_pitch = x_pitch;
    f.mode = in_mode == RowIn::masked ? 1 : 0;
    f.mask = mask;
    f.scal = scal;
    f.gmean_idx = gmean_idx;
    MrCols<T> c = mr_columns();
    c.rows_in = rows_in;
    c.rows_out = rows_out;
    c.sym = static_cast<int>(sym);
    c.ktab = ktab;
    c.kp = ktab_pitch;
    c.sc = sym_scale;
    MrRows<T> r = mr_rows();
    r.nrows = rows_out;
    r.ncols = cols_out;
    r.y = y;
    r.row_pitch = y_pitch;
    r.mode = out_mode == RowOut::masked ? 1 : 0;
    r.mask = mask;
    r.part = part;
    if (ev) ASPHER_HIP(hipEventRecord(ev[0], s));
    mr_rows_fwd<T>(f, s);
    if (ev) ASPHER_HIP(hipEventRecord(ev[1], s));
    mr_cols<T>(c, s);
    if (ev) ASPHER_HIP(hipEventRecord(ev[2], s));
    mr_rows_inv<T>(r, s);
    if (ev) ASPHER_HIP(hipEventRecord(ev[3], s));
}

template <typename T>
void SpectralPlan<T>::build_spectrum(const double* table, int Ns, T* kout, double* part,
                                     hipStream_t s, int embed) {
    if (rows_in != n) throw std::invalid_argument("build_spectrum: plan must read all rows");
    if (Ns < 1 || n < 2 * Ns - 1)
        throw std::invalid_argument("build_spectrum: the torus does not hold the embedding");
    if (rb_) {
        RbRowsFwd<T> f;
        f.ncols = n;
        f.nrows = n;
        f.AT = AT_;
        f.pitchT = pitchT_;
        f.lq = lq_;
        f.B = row_batch_fwd_;
    f.le = row_le_;
        f.tw = tw64_->dev;
        f.mode = embed;
        f.table = table;
        f.Ns_embed = Ns;
        f.remap = xcd_remap_ ? 1 : 0;
        RbCols<T> c;
        c.AT = AT_;
        c.pitchT = pitchT_;
        c.lq = lq_;
        c.ncols = nh;
        c.rows_in = n;
        c.rows_out = 0;
        c.W = col_width_;
        c.le = col_le_;
        c.tw = f.tw;
        c.sym = 3;
        c.kp = nh;
        c.kout = kout;
        c.part = part;
        c.remap = f.remap;
        rb_rows_fwd<T>(ilog2(n / 2), f, s);
        rb_cols<T>(logn_, c, s);
        return;
    }
    if (embed != 2) throw std::invalid_argument("build_spectrum: table kinds need a power-of-two plan");
    MrRows<T> f = mr_rows();
    f.nrows = n;
    f.ncols = n;
    f.mode = 2;
    f.table = table;
    f.Ns_embed = Ns;
    MrCols<T> c = mr_columns();
    c.rows_in = n;
    c.sym = static_cast<int>(Symbol::build);
    c.kp = nh;
    c.kout = kout;
    c.part = part;
    mr_rows_fwd<T>(f, s);
    mr_cols<T>(c, s);
}

template <typename T>
void SpectralPlan<T>::convolve2(const T* x, int x_pitch, std::int64_t x_stride, T* y,
                                int y_pitch, std::int64_t y_stride, int sym, const T* kxx,
                                const T* kyy, const T* kxy, int kp, double gamma, double norm,
                                hipStream_t s, RowIn in_mode, RowOut out_mode,
                                const std::uint8_t* mask, const double* scal, int gmean_idx,
                                double* part, std::int64_t pstride) {
    if (!rb_ || batch_ < 2 || n > 4096)
        throw std::invalid_argument("convolve2: needs a power-of-two plan of batch >= 2, n <= 4096");
    RbBatch bt;
    bt.count = 2;
    bt.x_stride = x_stride;
    bt.y_stride = y_stride;
    bt.m_stride = 0;
    bt.at_stride = at_stride_;
    bt.pstride = pstride;
    RbRowsFwd<T> f;
    f.x = x;
    f.x_pitch = x_pitch;
    f.ncols = cols_in;
    f.nrows = rows_in;
    f.AT = AT_;
    f.pitchT = pitchT_;
    f.lq = lq_;
    f.B = row_batch_fwd_;
    f.le = row_le_;
    f.tw = tw64_->dev;
    f.mode = in_mode == RowIn::masked ? 1 : 0;
    f.mask = mask;
    f.scal = scal;
    f.gmean_idx = gmean_idx;
    f.remap = xcd_remap_ ? 1 : 0;
    f.bt = bt;
    RbCols2<T> c;
    c.AT = AT_;
    c.pitchT = pitchT_;
    c.lq = lq_;
    c.at_stride = at_stride_;
    c.ncols = nh;
    c.rows_in = rows_in;
    c.rows_out = rows_out;
    c.tw = f.tw;
    c.sym = sym;
    c.kxx = kxx;
    c.kyy = kyy;
    c.kxy = kxy;
    c.kp = kp;
    c.gamma = gamma;
    c.norm = norm;
    c.remap = f.remap;
    RbRowsInv<T> r;
    r.AT = AT_;
    r.pitchT = pitchT_;
    r.lq = lq_;
    r.nrows = rows_out;
    r.B = row_batch_inv_;
    r.le = row_le_;
    r.tw = f.tw;
    r.y = y;
    r.y_pitch = y_pitch;
    r.ncols = cols_out;
    r.mode = out_mode == RowOut::masked ? 1 : 0;
    r.mask = mask;
    r.part = part;
    r.remap = f.remap;
    r.bt = bt;
    rb_rows_fwd<T>(ilog2(n / 2), f, s);
    rb_cols2<T>(logn_, c, s);
    rb_rows_inv<T>(ilog2(n / 2), r, s);
}

template class SpectralPlan<float>;
template class SpectralPlan<double>;

} // namespace aspher
