// psm_pass.hip -- the splitting step of pseudospectral_mobility (psm.hip has the
// scheme) as passes over lines of the half spectrum, 2D and 3D:
//   k_psm_row KIND 1  c2r of rho, M(rho) and its maximum, f'(rho), r2c   (between steps)
//   k_psm_split       last axis: forward transform of f', mu_hat, and per
//                     axis the gradient's inverse transform
//   k_psm_row KIND 0  per axis c2r, (M - M0) g / N^d, r2c
//   k_psm_join        last axis: forward transforms of the fluxes, their
//                     divergence, the update of rho_hat, its inverse transform
// In 3D the y passes run between the row passes and the last axis.  A step is
// 4 launches in 2D (8 in 3D) where whole transforms with element-wise kernels
// between them take 22 (37): below N = 1024 each launch lasts 4 to 6.5 us
// whatever it does (a kernel start plus one round trip to lines that another
// XCD wrote), so the step's time is mostly its number of launches.  2D N = 512
// FP64 on MI355X: 104 -> 41 us per step (32 steps per call).
// The per-entry operations and their order are those of the element-wise
// kernels (psm_ops.h, psm.hip).
#include "line_fft.h"
#include "psm_ops.h"

namespace chd {

namespace {

template <typename T>
using C2 = typename Complex<T>::type;

// partials a consumer reduces by itself; more are reduced by k_max_final first
constexpr int kMaxParts = 1024;

__global__ __launch_bounds__(256) void k_max_final(const double *__restrict__ parts, int n, double *__restrict__ out) {
    __shared__ double red[256];
    double m = 0.0;
    for(int i = threadIdx.x; i < n; i += 256) m = parts[i] > m ? parts[i] : m;
    red[threadIdx.x] = m;
    __syncthreads();
    for(int s = 128; s > 0; s >>= 1) {
        if(threadIdx.x < s) red[threadIdx.x] = red[threadIdx.x + s] > red[threadIdx.x] ? red[threadIdx.x + s] : red[threadIdx.x];
        __syncthreads();
    }
    if(threadIdx.x == 0) *out = red[0];
}

__device__ __forceinline__ double wave_max(double m) {
#pragma unroll
    for(int d = 32; d > 0; d >>= 1) {
        const double o = __shfl_xor(m, d);
        m = o > m ? o : m;
    }
    return m;
}

// M0 = max(0, the partial maxima), by every wave for itself: load() after the
// line's own loads, value() where M0 is needed, so the partials (written by the
// other XCDs) arrive with the line.  All loads are independent: a loop over them
// waits for each in turn (2D N = 512: 14.7 us for k_psm_join in place of 10.9).
struct M0Reader {
    double m[kMaxParts / 64];
    __device__ __forceinline__ void load(const double *__restrict__ parts, int n) {
        const int lane = threadIdx.x & 63;
#pragma unroll
        for(int i = 0; i < kMaxParts / 64; i++) m[i] = lane + 64 * i < n ? parts[lane + 64 * i] : 0.0;
    }
    __device__ __forceinline__ double value() const {
        double v = 0.0;
#pragma unroll
        for(int i = 0; i < kMaxParts / 64; i++) v = m[i] > v ? m[i] : v;
        return wave_max(v);
    }
};

// the mobility of a cell (ch_device.h's expressions, without a branch) under the
// constant, regularised and linear rules; the density itself under the
// free-energy rule, whose power is left to a pass of its own (psm.hip)
template <typename T>
__device__ __forceinline__ T mobility_or_rho(const Params &p, int rule, T r) {
#pragma clang fp contract(off)
    const T den = rule == CH_MOB_REGULARISED ? r + (T)p.rho_min : (T)p.rho_ref;
    const T M = (T)p.M * r / den;
    return rule == CH_MOB_CONSTANT ? (T)p.M : (rule == CH_MOB_FREE_ENERGY ? r : M);
}

// the three half spectra of the gradient components
template <typename T2>
struct Fields {
    T2 *f[3];
};

// ------------------------------------------------------------------ row passes
// One row pass over blockIdx.y fields.  KIND 0: the flux of field blockIdx.y
// (W = its half spectrum, mob read, M0 from parts).  KIND 1: between two steps
// (mob written, parts[block] = the block's largest mobility; the densities
// instead under the free-energy rule).
template <typename T, int KIND, int MODEL, int LOG2N, int NLR>
__global__ __launch_bounds__((FftGeom<LOG2N, NLR>::NT)) void k_psm_row(
    Fields<C2<T>> Ws, const C2<T> *__restrict__ tw, Params p, int rows, long rs, T *__restrict__ mob, int rule,
    double *__restrict__ parts, int nparts) {
    using T2 = C2<T>;
    using G = FftGeom<LOG2N, NLR>;
    constexpr int n = G::n, N = 2 * n, nl = G::NL, NT = G::NT, Nh = n + 1;
    __shared__ T2 buf[padded(G::E + nl)];
    T2 *__restrict__ W = Ws.f[blockIdx.y];
    LineFFT<T2, LOG2N, nl> fft;
    fft.prefetch(tw, 2);
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int row0 = tile * nl;
    T mv[8];
    M0Reader rd;
    if constexpr(KIND == 0) {
#pragma unroll
        for(int i = 0; i < 8; i++) {
            const int e = threadIdx.x + i * NT;
            const int row = row0 + e / N;
            mv[i] = row < rows ? mob[(size_t)row * N + e % N] : (T)0;
        }
    }
    for(int e = threadIdx.x; e < nl * Nh; e += NT) {
        const int line = e / Nh, k = e % Nh;
        const int row = row0 + line;
        buf[pidx(e)] = (row < rows) ? W[(size_t)row * rs + k] : T2{0, 0};
    }
    if constexpr(KIND == 0) rd.load(parts, nparts);
    __syncthreads();
    double m0 = 0.0;
    if constexpr(KIND == 0) m0 = rd.value();
    T2 z[4];
#pragma unroll
    for(int i = 0; i < 4; i++) {
        const int q = threadIdx.x + i * NT;
        const int line = q / n, k = q % n;
        T2 xk = buf[pidx(line * Nh + k)];
        T2 xnk = buf[pidx(line * Nh + n - k)];
        if(k == 0) { xk.y = 0; xnk.y = 0; }
        const T2 Ev = T2{xk.x + xnk.x, xk.y - xnk.y};
        const T2 Ov = cmul(T2{xk.x - xnk.x, xk.y + xnk.y}, conj_(tw[k]));
        z[i] = T2{Ev.x - Ov.y, Ev.y + Ov.x};
    }
    __syncthreads();
#pragma unroll
    for(int i = 0; i < 4; i++) buf[pidx(threadIdx.x + i * NT)] = z[i];
    __syncthreads();
    fft.template run<true>(buf);
    T *bufT = reinterpret_cast<T *>(buf);
    double mx = 0.0;
#pragma unroll
    for(int i = 0; i < 8; i++) {
        const int e = threadIdx.x + i * NT;
        const int row = row0 + e / N;
        const int a = 2 * pidx(e >> 1) + (e & 1);
        if constexpr(KIND == 0) {
            bufT[a] = psm_flux<T>(bufT[a], mv[i], (T)m0, (T)p.inv_bins);
        }
        else {
            const T r = bufT[a];
            if(row < rows) {
                const T M = mobility_or_rho<T>(p, rule, r);
                mob[(size_t)row * N + e % N] = M;
                mx = (double)M > mx ? (double)M : mx;
                bufT[a] = fprime<T, MODEL>(p, r);
            }
            else {
                bufT[a] = (T)0;
            }
        }
    }
    if constexpr(KIND == 1) {
        // the waves' maxima through the first entries of a buffer of their own
        __shared__ double red[(NT + 63) / 64];
        mx = wave_max(mx);
        if((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
        __syncthreads();
        if(threadIdx.x == 0) {
#pragma unroll
            for(int w = 1; w < (NT + 63) / 64; w++) mx = red[w] > mx ? red[w] : mx;
            parts[tile] = mx;
        }
    }
    else {
        __syncthreads();
    }
    fft.template run<false>(buf);
    for(int e = threadIdx.x; e < nl * Nh; e += NT) {
        const int line = e / Nh, k = e % Nh;
        const int row = row0 + line;
        if(row >= rows) continue;
        const T2 zk = buf[pidx(line * n + (k == n ? 0 : k))];
        const T2 znk = buf[pidx(line * n + (k == 0 ? 0 : n - k))];
        W[(size_t)row * rs + k] = r2c_entry<T>(zk, znk, tw[k]);
    }
}

// the same on one wave per row (N >= 1024), NR rows per block sharing the
// staged twiddle table; KIND 1: parts[row].  The mobility rule is a template
// parameter: a branch between the transforms would keep products and sums from
// being fused where the separate row passes fuse them (other bits).
template <typename T, int KIND, int MODEL, int MOB, int LOG2N, int NR>
__global__ __launch_bounds__(64 * NR) void k_psm_roww(Fields<C2<T>> Ws, const C2<T> *tw, Params p, int rows, long rs,
                                                      T *__restrict__ mob, double *__restrict__ parts, int nparts) {
    using T2 = C2<T>;
    using F = WaveFFT<T2, LOG2N>;
    constexpr int E = F::E, n = F::n;
    __shared__ T2 lds[NR][F::LDS];
    using Stage = TwiddleStage<T2, 2 * n>;
    __shared__ Stage stage;
    const int row = xcd_tile(blockIdx.x, gridDim.x) * NR + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if(row - (int)(threadIdx.x >> 6) >= rows) return;  // the whole block lies past the last row (rows % NR == 0)
    const int lane = threadIdx.x & 63;
    T2 twr[Stage::template per<64 * NR>()];
    stage.template load<64 * NR>(tw, threadIdx.x, twr);
    T2 *w = Ws.f[blockIdx.y] + (size_t)row * rs;
    T2 *mrow = reinterpret_cast<T2 *>(mob + (size_t)row * 2 * n);
    T2 v[E], mv[KIND == 0 ? E : 1];
    M0Reader rd;
    double mx = 0.0;
    c2r_pre<T, E>(w, 1, lane, tw, v);  // before the first barrier: global table
    if constexpr(KIND == 0) {
#pragma unroll
        for(int m = 0; m < E; m++) mv[m] = mrow[lane + 64 * m];
        rd.load(parts, nparts);
    }
    tw = stage.template store<64 * NR>(tw, threadIdx.x, twr);
    T2 *own = lds[threadIdx.x >> 6];
    lds_barrier();  // the staged table; every buffer below is one wave's own
    wave_transform<T2, LOG2N, true, false>(lane, v, own, tw, 2);
    if constexpr(KIND == 0) {
        const T M0 = (T)rd.value(), ib = (T)p.inv_bins;
#pragma unroll
        for(int m = 0; m < E; m++)
            v[m] = T2{psm_flux<T>(v[m].x, mv[m].x, M0, ib), psm_flux<T>(v[m].y, mv[m].y, M0, ib)};
    }
    else {
#pragma unroll
        for(int m = 0; m < E; m++) {
            const T2 M{mobility_or_rho<T>(p, MOB, v[m].x), mobility_or_rho<T>(p, MOB, v[m].y)};
            mrow[lane + 64 * m] = M;
            mx = (double)M.x > mx ? (double)M.x : mx;
            mx = (double)M.y > mx ? (double)M.y : mx;
            v[m] = T2{fprime<T, MODEL>(p, v[m].x), fprime<T, MODEL>(p, v[m].y)};
        }
        mx = wave_max(mx);
    }
    wave_transform<T2, LOG2N, false, false>(lane, v, own, tw, 2);
    r2c_post<T, LOG2N>(v, own, lane, tw, w, 1);
    if(KIND == 1 && lane == 0) parts[row] = mx;
}

// the lines of the last axis: line l, entry j at base + j stride, and its modes
template <int DIMS>
struct LastAxis {
    int ix, mid;
    size_t base;
    long stride;
    __device__ __forceinline__ LastAxis(const Params &p, int l) {
        const int Nh = p.N / 2 + 1;
        ix = l % Nh;
        mid = l / Nh;  // 2D: 0; 3D: the y index
        base = DIMS == 2 ? (size_t)ix : (size_t)mid * Nh + ix;
        stride = DIMS == 2 ? Nh : (long)p.N * Nh;
    }
    __device__ __forceinline__ size_t at(int j) const { return base + (size_t)j * stride; }
    // entry j of line l in a line-major field
    __device__ __forceinline__ size_t own(const Params &p, int l, int j) const { return (size_t)l * p.N + j; }
    __device__ __forceinline__ int iy(int j) const { return DIMS == 2 ? j : mid; }
    __device__ __forceinline__ int iz(int j) const { return DIMS == 2 ? 0 : j; }
};

// f_hat of each line (kept in FH), mu_hat = (f_hat + 2k q^2 rho_hat) deal, and
// per axis d the inverse transform of (i k_d) deal mu_hat
// Blocks of one line keep f_hat, which only these two passes touch, line-major
// (entry j of line l at l N + j), and in 2D rho_hat too from the first step's join
// to the last one's (lm: rho_hat is line-major).  A line's entries in the half
// spectrum lie a row apart, one 128 B line of memory each for 16 B of use, and
// that traffic, not the transforms, bounds both passes (running a line's axes
// beside each other changed nothing; other row strides neither).  2D on MI355X, us
// per step, all fields in the half spectrum's layout -> f_hat -> rho_hat too:
//   N = 256   FP64 31.9 -> 31.2 -> 31.2   FP32 28.6 -> 28.0 -> 28.0
//   N = 512        44.0 -> 41.5 -> 40.8        36.2 -> 33.2 -> 32.2
//   N = 1024       89.2 -> 85.8 -> 80.2        62.1 -> 59.3 -> 53.5
template <typename T, class ENG, int DIMS>
__global__ __launch_bounds__(ENG::NT) void k_psm_split(const C2<T> *__restrict__ W, const C2<T> *__restrict__ RH, bool lm,
                                                       C2<T> *__restrict__ FH, Fields<C2<T>> Gs,
                                                       const C2<T> *__restrict__ table, Params p, int lines) {
#pragma clang fp contract(off)
    using T2 = C2<T>;
    constexpr int E = ENG::E;
    __shared__ typename ENG::Smem sm;
    const int l0 = xcd_tile(blockIdx.x, gridDim.x) * ENG::NL;
    if(l0 >= lines) return;  // grid padded to a multiple of 8 blocks
    ENG eng(sm);
    eng.begin(table);
    const int l = l0 + eng.line();
    const bool on = ENG::NL == 1 || l < lines;
    const LastAxis<DIMS> ax(p, on ? l : l0);
    T2 v[E], mu[E];
#pragma unroll
    for(int i = 0; i < E; i++) v[i] = W[ax.at(eng.in(i))];
#pragma unroll
    for(int i = 0; i < E; i++) {
        const int j = eng.freq(i);
        mu[i] = RH[lm ? ax.own(p, l, j) : ax.at(j)];
    }
    eng.finish(table);
    eng.forward(v);
#pragma unroll
    for(int i = 0; i < E; i++) {
        const int j = eng.freq(i);
        if(on) FH[ENG::NL == 1 ? ax.own(p, l, j) : ax.at(j)] = v[i];
        double k2, deal;
        mode_q2(p, ax.ix, ax.iy(j), ax.iz(j), k2, deal);
        if(!p.use_dealias) deal = 1.0;
        const T d = (T)deal, c = (T)(2.0 * p.k * k2);
        mu[i] = T2{(v[i].x + c * mu[i].x) * d, (v[i].y + c * mu[i].y) * d};
    }
#pragma unroll
    for(int a = 0; a < DIMS; a++) {
#pragma unroll
        for(int i = 0; i < E; i++) {
            const int j = eng.freq(i);
            v[i] = psm_grad_term<T>(p, ax.ix, ax.iy(j), ax.iz(j), a, mu[i]);
        }
        eng.inverse(v);
#pragma unroll
        for(int i = 0; i < E; i++)
            if(on) Gs.f[a][ax.at(eng.in(i))] = v[i];
    }
}

// div_hat of the fluxes' transforms, the update of rho_hat (:290-297) and the
// inverse transform of rho_hat / N^d into W
template <typename T, class ENG, int DIMS>
__global__ __launch_bounds__(ENG::NT) void k_psm_join(Fields<C2<T>> Gs, const C2<T> *__restrict__ FH,
                                                      const C2<T> *RH, bool lm, C2<T> *RO, bool lm_out,
                                                      C2<T> *__restrict__ W,
                                                      const C2<T> *__restrict__ table, Params p, int lines,
                                                      const double *__restrict__ parts, int nparts) {
#pragma clang fp contract(off)
    using T2 = C2<T>;
    constexpr int E = ENG::E;
    __shared__ typename ENG::Smem sm;
    const int l0 = xcd_tile(blockIdx.x, gridDim.x) * ENG::NL;
    if(l0 >= lines) return;
    ENG eng(sm);
    eng.begin(table);
    const int l = l0 + eng.line();
    const bool on = ENG::NL == 1 || l < lines;
    const LastAxis<DIMS> ax(p, on ? l : l0);
    T2 g[DIMS][E], r[E], f[E], dv[E];
#pragma unroll
    for(int a = 0; a < DIMS; a++)
#pragma unroll
        for(int i = 0; i < E; i++) g[a][i] = Gs.f[a][ax.at(eng.in(i))];
#pragma unroll
    for(int i = 0; i < E; i++) {
        const int j = eng.freq(i);
        r[i] = RH[lm ? ax.own(p, l, j) : ax.at(j)];
        f[i] = FH[ENG::NL == 1 ? ax.own(p, l, j) : ax.at(j)];
        dv[i] = T2{0, 0};
    }
    M0Reader rd;
    rd.load(parts, nparts);
    eng.finish(table);
#pragma unroll
    for(int a = 0; a < DIMS; a++) {
        eng.forward(g[a]);
#pragma unroll
        for(int i = 0; i < E; i++) {
            const int j = eng.freq(i);
            dv[i] = psm_div_term<T>(p, ax.ix, ax.iy(j), ax.iz(j), a, g[a][i], dv[i]);
        }
    }
    const double M0 = rd.value();
    const T dt = (T)p.dt, S = (T)p.S, ib = (T)p.inv_bins;
#pragma unroll
    for(int i = 0; i < E; i++) {
        const int j = eng.freq(i);
        double k2, deal;
        mode_q2(p, ax.ix, ax.iy(j), ax.iz(j), k2, deal);
        const double k4 = k2 * k2;
        const T den = (T)(1.0 + p.dt * M0 * (p.S * k2 + 2.0 * p.k * k4)), a = (T)(p.dt * M0 * k2);
        const T re = (r[i].x + dt * dv[i].x - a * (f[i].x - S * r[i].x)) / den;
        const T im = (r[i].y + dt * dv[i].y - a * (f[i].y - S * r[i].y)) / den;
        r[i] = T2{re, im};
        dv[i] = T2{re * ib, im * ib};
    }
    eng.inverse(dv);
#pragma unroll
    for(int i = 0; i < E; i++)
        if(on) {
            const int j = eng.freq(i);
            RO[lm_out ? ax.own(p, l, j) : ax.at(j)] = r[i];
            W[ax.at(eng.in(i))] = dv[i];
        }
}

// ------------------------------------------------------------------ host side
template <typename T, int LOG2N, int DIMS>
struct Chain {
    using T2 = C2<T>;
    static constexpr int N = 1 << LOG2N, Nh = N / 2 + 1, LX = LOG2N - 1;
    const PsmArgs &B;
    hipStream_t s;
    const Params &p;
    int rows, lines;
    const T2 *tw;
    Fields<T2> G;

    Chain(const PsmArgs &b, hipStream_t st) : B(b), s(st), p(b.a.p) {
        rows = DIMS == 2 ? N : N * N;
        lines = DIMS == 2 ? Nh : N * Nh;
        tw = (const T2 *)B.a.twiddles;
        G = Fields<T2>{{(T2 *)B.gh, (T2 *)B.divh, (T2 *)B.muh}};
    }
    static int row_parts(int rows) {
        if constexpr(wave_len<LX>()) return rows;
        else return (rows + row_lines() - 1) / row_lines();
    }
    // rows per block of k_psm_row; 3D from N = 128 four times as many, which keeps its
    // partial maxima within kMaxParts (N = 128: no reduction launch of their own)
    static constexpr int row_lines() { return DIMS == 3 && LX >= 6 && LX < 8 ? 1 << (10 - LX) : PackedLines<LX>::value; }
    template <int KIND, int MODEL>
    void row(Fields<T2> W, int nf, int nparts) {
        T *field = (T *)(KIND == 1 && B.mob_rule == CH_MOB_FREE_ENERGY ? B.a.rho : B.mob);
        if constexpr(wave_len<LX>()) {
            auto go = [&](auto tag) {
                constexpr int NR = 4, MOB = decltype(tag)::value;
                hipLaunchKernelGGL((k_psm_roww<T, KIND, MODEL, MOB, LX, NR>), dim3((rows / NR + 7) / 8 * 8, nf),
                                   dim3(64 * NR), 0, s, W, tw, p, rows, Nh, field, B.max_parts, nparts);
            };
            if constexpr(KIND == 0) go(std::integral_constant<int, CH_MOB_CONSTANT>{});
            else if(B.mob_rule == CH_MOB_CONSTANT) go(std::integral_constant<int, CH_MOB_CONSTANT>{});
            else if(B.mob_rule == CH_MOB_REGULARISED) go(std::integral_constant<int, CH_MOB_REGULARISED>{});
            else if(B.mob_rule == CH_MOB_LINEAR) go(std::integral_constant<int, CH_MOB_LINEAR>{});
            else go(std::integral_constant<int, CH_MOB_FREE_ENERGY>{});
        }
        else {
            constexpr int NL = row_lines();
            hipLaunchKernelGGL((k_psm_row<T, KIND, MODEL, LX, NL>), dim3((rows + NL - 1) / NL, nf),
                               dim3(FftGeom<LX, NL>::NT), 0, s, W, tw, p, rows, Nh, field, B.mob_rule, B.max_parts,
                               nparts);
        }
    }
    // more partial maxima than a consumer reads become one
    int reduce(int nparts) {
        if(nparts <= kMaxParts) return nparts;
        hipLaunchKernelGGL(k_max_final, dim3(1), dim3(256), 0, s, B.max_parts, nparts, B.max_parts);
        return 1;
    }
    hipError_t y_pass(const Fields<T2> &F, int nf, bool inverse) {
        if constexpr(DIMS == 3)
            for(int f = 0; f < nf; f++) {
                const hipError_t e = spec_y_pass(B.a, F.f[f], inverse, s);
                if(e != hipSuccess) return e;
            }
        return hipSuccess;
    }
    hipError_t run(int64_t nsteps) {
        using Eng = Engine<T, LOG2N, DIMS>;
        const Fields<T2> W{{(T2 *)B.a.work, nullptr, nullptr}};
        const int blocks = col_blocks(lines, Eng::NL);
        constexpr bool keep = DIMS == 2 && Eng::NL == 1;
        int nparts = 0;
        hipError_t e = psm_mobility(B, B.max_parts, nparts, s);
        if(e == hipSuccess) e = spec_x_forward(B.a, B.a.rho, B.a.work, true, s);
        if(e == hipSuccess) nparts = reduce(nparts);
        for(int64_t t = 0; t < nsteps && e == hipSuccess; t++) {
            if((e = y_pass(W, 1, false)) != hipSuccess) return e;
            const bool lm = keep && t > 0;  // 2D: the third component's spectrum is free
            const T2 *RH = (const T2 *)(lm ? B.muh : B.a.rho_hat);
            hipLaunchKernelGGL((k_psm_split<T, Eng, DIMS>), dim3(blocks), dim3(Eng::NT), 0, s, W.f[0],
                               RH, lm, (T2 *)B.fh, G, tw, p, lines);
            if((e = y_pass(G, DIMS, true)) != hipSuccess) return e;
            row<0, CH_LANDAU>(G, DIMS, nparts);
            if((e = y_pass(G, DIMS, false)) != hipSuccess) return e;
            const bool lmo = keep && t + 1 < nsteps;
            hipLaunchKernelGGL((k_psm_join<T, Eng, DIMS>), dim3(blocks), dim3(Eng::NT), 0, s, G, (const T2 *)B.fh, RH, lm,
                               lmo ? (T2 *)B.muh : (T2 *)B.a.rho_hat, lmo, W.f[0], tw, p, lines,
                               (const double *)B.max_parts, nparts);
            if((e = y_pass(W, 1, true)) != hipSuccess) return e;
            if(t + 1 < nsteps) {
                if(B.a.model == CH_LANDAU) row<1, CH_LANDAU>(W, 1, 0);
                else row<1, CH_SIMPLE_WERTHEIM>(W, 1, 0);
                if(B.mob_rule == CH_MOB_FREE_ENERGY) {
                    if((e = psm_mobility(B, B.max_parts, nparts, s)) != hipSuccess) return e;
                }
                else {
                    nparts = row_parts(rows);
                }
                nparts = reduce(nparts);
            }
            e = hipGetLastError();
        }
        return e == hipSuccess ? spec_x_inverse(B.a, B.a.work, B.a.rho, s) : e;
    }
};

template <typename T, int DIMS>
hipError_t chain_n(const PsmArgs &B, int64_t nsteps, hipStream_t s) {
    switch(B.a.p.log2N) {
    case 2: return Chain<T, 2, DIMS>(B, s).run(nsteps);
    case 3: return Chain<T, 3, DIMS>(B, s).run(nsteps);
    case 4: return Chain<T, 4, DIMS>(B, s).run(nsteps);
    case 5: return Chain<T, 5, DIMS>(B, s).run(nsteps);
    case 6: return Chain<T, 6, DIMS>(B, s).run(nsteps);
    case 7: return Chain<T, 7, DIMS>(B, s).run(nsteps);
    case 8: return Chain<T, 8, DIMS>(B, s).run(nsteps);
    case 9: return Chain<T, 9, DIMS>(B, s).run(nsteps);
    case 10: return Chain<T, 10, DIMS>(B, s).run(nsteps);
    }
    if constexpr(DIMS == 2 && sizeof(T) == 4) {  // FP64: psm.hip's whole transforms are faster there
        if(B.a.p.log2N == 11) return Chain<T, 11, 2>(B, s).run(nsteps);
        if(B.a.p.log2N == 12) return Chain<T, 12, 2>(B, s).run(nsteps);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t psm_chain(const PsmArgs &B, int64_t nsteps, hipStream_t s) {
    if(B.a.precision == CH_FP64)
        return B.a.p.dims == 2 ? chain_n<double, 2>(B, nsteps, s) : chain_n<double, 3>(B, nsteps, s);
    return B.a.p.dims == 2 ? chain_n<float, 2>(B, nsteps, s) : chain_n<float, 3>(B, nsteps, s);
}

}  // namespace chd
