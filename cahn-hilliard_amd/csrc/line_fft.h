// line_fft.h -- the line transforms shared by the spectral passes: the LDS
// Stockham transform of one block (LineFFT), the one-wave transform's driver
// and its staged twiddle table (wave_fft.h), the packing of real rows, and the
// half-spectrum layout.
#pragma once

#include <type_traits>

#include "ch_internal.h"
#include "wave_fft.h"

namespace chd {

template <typename T2>
__device__ __forceinline__ T2 cmul(T2 a, T2 b) {
    return T2{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T2>
__device__ __forceinline__ T2 cadd(T2 a, T2 b) { return T2{a.x + b.x, a.y + b.y}; }
template <typename T2>
__device__ __forceinline__ T2 csub(T2 a, T2 b) { return T2{a.x - b.x, a.y - b.y}; }
template <typename T2>
__device__ __forceinline__ T2 conj_(T2 a) { return T2{a.x, -a.y}; }

// streaming store of one complex entry (written once, read by the next pass)
template <typename T2>
__device__ __forceinline__ void nt_store(T2 *p, T2 v) {
    using T = decltype(T2{}.x);
    typedef T V2 __attribute__((ext_vector_type(2)));
    V2 w;
    w.x = v.x;
    w.y = v.y;
    __builtin_nontemporal_store(w, reinterpret_cast<V2 *>(p));
}

// LDS index with one pad element every 32: the Stockham writes of the first
// passes (stride 4 elements) then spread over every bank group.
__device__ __forceinline__ constexpr int pidx(int i) { return i + (i >> 5); }
constexpr int padded(int n) { return n + (n >> 5) + 1; }

// Block geometry of a length-2^LOG2N line FFT: E elements, NT = E / 4 threads.
template <int LOG2N, int NLINES>
struct FftGeom {
    static constexpr int n = 1 << LOG2N;
    static constexpr int NL = NLINES;
    static constexpr int E = n * NL;
    static constexpr int NT = E / 4;
    static constexpr bool R2 = (LOG2N & 1) != 0;
    static constexpr int NP4 = LOG2N / 2;  // radix-4 passes
};

// Rows per block of the LDS row passes: as many as one wave takes (NT = 64), so that
// the few rows of a 2D grid reach many CUs (256-thread blocks left N = 256 on 32 of
// them); n <= 4 as 256 threads take.  2D on MI355X, us per step, 256 threads -> 64:
// pseudospectral FP64 N = 64 11.1 -> 9.9, 128 11.8 -> 10.4, 256 12.7 -> 11.2 (FP32 10.4
// -> 9.2, 10.7 -> 9.6, 11.2 -> 10.1); splitting step FP64 27.4 -> 25.2, 29.3 -> 26.3,
// 31.3 -> 28.0; 3D N = 32 to 128 equal.
template <int LOG2N>
struct PackedLines { static constexpr int value = LOG2N >= 8 ? 1 : (1 << ((LOG2N <= 2 ? 10 : 8) - LOG2N)); };

template <typename T2, int LOG2N, int NLINES>
struct LineFFT {
    using G = FftGeom<LOG2N, NLINES>;
    T2 tw[G::NP4 > 0 ? G::NP4 : 1][3];

    // table: W_Ntab^m; twstride = Ntab / n
    __device__ __forceinline__ void prefetch(const T2 *__restrict__ table, int twstride) {
        constexpr int n = G::n, qn = n >> 2;
        const int j = (int)threadIdx.x % (qn > 0 ? qn : 1);
#pragma unroll
        for(int ps = 0; ps < G::NP4; ps++) {
            const int Ns = (G::R2 ? 2 : 1) << (2 * ps);
            const int tscale = (n / (4 * Ns)) * twstride;
            const int jm = j & (Ns - 1);
#pragma unroll
            for(int r = 1; r < 4; r++) tw[ps][r - 1] = table[r * jm * tscale];
        }
    }

    // in-place transform of NL lines stored line-major in buf; INV: e^{+i}
    template <bool INV>
    __device__ __forceinline__ void run(T2 *buf) const {
        constexpr int n = G::n, NT = G::NT;
        const int tid = threadIdx.x;
        if constexpr(G::R2) {
            constexpr int h = n >> 1;
            T2 v0[2], v1[2];
#pragma unroll
            for(int i = 0; i < 2; i++) {
                const int q = tid + i * NT;
                const int line = q / h, j = q % h;
                v0[i] = buf[pidx(line * n + j)];
                v1[i] = buf[pidx(line * n + j + h)];
            }
            __syncthreads();
#pragma unroll
            for(int i = 0; i < 2; i++) {
                const int q = tid + i * NT;
                const int line = q / h, j = q % h;
                buf[pidx(line * n + 2 * j)] = cadd(v0[i], v1[i]);
                buf[pidx(line * n + 2 * j + 1)] = csub(v0[i], v1[i]);
            }
            __syncthreads();
        }
        constexpr int qn = n >> 2;
        const int line = tid / (qn > 0 ? qn : 1), j = tid % (qn > 0 ? qn : 1);
#pragma unroll
        for(int ps = 0; ps < G::NP4; ps++) {
            const int Ns = (G::R2 ? 2 : 1) << (2 * ps);
            const int jm = j & (Ns - 1);
            T2 v[4];
#pragma unroll
            for(int r = 0; r < 4; r++) v[r] = buf[pidx(line * n + j + r * qn)];
#pragma unroll
            for(int r = 1; r < 4; r++) v[r] = cmul(v[r], INV ? conj_(tw[ps][r - 1]) : tw[ps][r - 1]);
            __syncthreads();
            const T2 a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
            const T2 a2 = cadd(v[1], v[3]);
            const T2 d = csub(v[1], v[3]);
            const T2 a3 = INV ? T2{-d.y, d.x} : T2{d.y, -d.x};  // (+-i)(v1 - v3)
            const int o = line * n + (j - jm) * 4 + jm;
            buf[pidx(o)] = cadd(a0, a2);
            buf[pidx(o + Ns)] = cadd(a1, a3);
            buf[pidx(o + 2 * Ns)] = csub(a0, a2);
            buf[pidx(o + 3 * Ns)] = csub(a1, a3);
            __syncthreads();
        }
    }
};

// The first barrier orders the block's earlier LDS accesses (the staged
// twiddle table, another wave's reads of this buffer) before the transform;
// the buffer is the wave's own from there on, so the passes within the
// transform are ordered by wave_lds_sync alone.  BLOCK_FIRST = false: the
// caller has ordered the block's accesses already and the buffer is the
// wave's own, so the first sync is the wave's too.
template <typename T2, int LOG2N, bool INV, bool BLOCK_FIRST = true, int E>
__device__ __forceinline__ void wave_transform(int lane, T2 (&v)[E], T2 *lds, const T2 *tw, int tstride) {
    static_assert(E == WaveFFT<T2, LOG2N>::E, "entries per lane");
    using F = WaveFFT<T2, LOG2N>;
    if constexpr(BLOCK_FIRST) lds_barrier();
    else wave_lds_sync();
    F::template pass1_write<INV>(lane, v, lds);
    wave_lds_sync();
    F::pass_read(lane, v, lds);
    wave_lds_sync();
    F::template pass2_write<INV>(lane, v, lds, tw, tstride);
    wave_lds_sync();
    F::pass_read(lane, v, lds);
    F::template pass3_final<INV>(lane, v, tw, tstride);
}

// The system's twiddle table (N entries, W_N^m) staged in LDS when N <= 1024:
// one wave runs per SIMD at most (a line per wave), so nothing hides a global
// load, and every transform pass after the first barrier would otherwise wait
// on its twiddles.  load() fetches a thread's share of the table into
// registers and store() writes it to LDS: a kernel issues load(), then the
// line's own loads, then store(), so that the two sets of loads are in flight
// together (a store straight after each load would wait out the table's
// latency before the line's loads issue).
template <typename T2, int TN>
struct TwiddleStage {
    static constexpr bool on = TN <= 1024;
    T2 t[on ? TN : 1];
    // entries per thread of NT threads (the register array of load / store)
    template <int NT>
    static constexpr int per() { return on ? TN / NT : 1; }
    template <int NT>
    __device__ __forceinline__ void load(const T2 *__restrict__ tw, int tid, T2 (&r)[per<NT>()]) const {
        if constexpr(on) {
#pragma unroll
            for(int i = 0; i < TN / NT; i++) r[i] = tw[tid + NT * i];
        }
        else {
            (void)tw;
            (void)tid;
            (void)r;
        }
    }
    // the table to read from: the LDS copy, visible after the next barrier
    template <int NT>
    __device__ __forceinline__ const T2 *store(const T2 *tw, int tid, const T2 (&r)[per<NT>()]) {
        if constexpr(on) {
#pragma unroll
            for(int i = 0; i < TN / NT; i++) t[tid + NT * i] = r[i];
            return t;
        }
        else {
            (void)tid;
            (void)r;
            return tw;
        }
    }
};

// entry k of the c2r pre-processing: the packed n-point inverse transform
// input Z_k from X_k and X_{n-k} of a row of n + 1 half-spectrum entries
// (table W_N^m, N = 2 n)
template <typename T2>
__device__ __forceinline__ T2 c2r_entry(const T2 *__restrict__ in, long ks, int k, int n, const T2 *__restrict__ tw) {
    T2 xk = in[(size_t)k * ks];
    T2 xnk = in[(size_t)(n - k) * ks];
    if(k == 0) { xk.y = 0; xnk.y = 0; }
    // E = X_k + conj X_{n-k}; O = (X_k - conj X_{n-k}) conj(W_N^k); Z = E + i O
    const T2 Ev = T2{xk.x + xnk.x, xk.y - xnk.y};
    const T2 Ov = cmul(T2{xk.x - xnk.x, xk.y + xnk.y}, conj_(tw[k]));
    return T2{Ev.x - Ov.y, Ev.y + Ov.x};
}

// entry k of the r2c post-processing: X_k from Z_k and Z_{n-k} and w = W_N^k
template <typename T, typename T2>
__device__ __forceinline__ T2 r2c_entry(T2 zk, T2 znk, T2 w) {
    // E = (Z_k + conj Z_{n-k}) / 2, O = (Z_k - conj Z_{n-k}) / (2i), X_k = E + W_N^k O
    const T2 Ev = T2{(zk.x + znk.x) * (T)0.5, (zk.y - znk.y) * (T)0.5};
    const T2 dd = T2{zk.x - znk.x, zk.y + znk.y};
    const T2 Ov = T2{dd.y * (T)0.5, -dd.x * (T)0.5};
    return cadd(Ev, cmul(w, Ov));
}

// c2r pre-processing of a row of n + 1 half-spectrum entries into the packed
// n-point inverse transform input, in distribution D (k = lane + 64 m)
template <typename T, int E>
__device__ __forceinline__ void c2r_pre(const typename Complex<T>::type *__restrict__ in, long ks, int lane,
                                        const typename Complex<T>::type *__restrict__ tw,
                                        typename Complex<T>::type (&z)[E]) {
    constexpr int n = 64 * E;
#pragma unroll
    for(int m = 0; m < E; m++) z[m] = c2r_entry(in, ks, lane + 64 * m, n, tw);
}

// r2c post-processing: Z (distribution D) -> n + 1 half-spectrum entries;
// NT: streaming stores (the pseudospectral chain's work field)
template <typename T, int LOG2N, bool NT = false, typename T2>
__device__ __forceinline__ void r2c_post(const T2 *z, T2 *lds, int lane, const T2 *__restrict__ tw,
                                         T2 *__restrict__ out, long ks) {
    using F = WaveFFT<T2, LOG2N>;
    constexpr int E = F::E, n = F::n;
    wave_lds_sync();  // one-wave blocks: the buffer is the wave's own
#pragma unroll
    for(int m = 0; m < E; m++) lds[F::pad(lane + 64 * m)] = z[m];
    wave_lds_sync();
    auto emit = [&](int k, T2 zk, T2 znk) {
        if constexpr(NT) nt_store(&out[(size_t)k * ks], r2c_entry<T>(zk, znk, tw[k]));
        else out[(size_t)k * ks] = r2c_entry<T>(zk, znk, tw[k]);
    };
#pragma unroll
    for(int m = 0; m < E; m++) {
        const int k = lane + 64 * m;
        emit(k, z[m], lds[F::pad(k == 0 ? 0 : n - k)]);
    }
    if(lane == 0) emit(n, z[0], z[0]);
}

// lengths the wave kernels take; the others run the LDS ones
template <int LOG2N>
constexpr bool wave_len() { return LOG2N >= 9 && LOG2N <= 11; }

// columns per block of the strided passes: NLC lines of n = N, NT = NLC n / 4
// threads (<= 1024)
template <int LOG2N>
struct ColLines { static constexpr int value = LOG2N >= 11 ? 1 : (LOG2N == 10 ? 2 : (LOG2N >= 8 ? 4 : (1024 >> LOG2N))); };

// ---- line engines (psm_pass.hip, k_cole)
// A block's transform of its lines, entries in registers: entry i of a thread
// is entry in(i) of its line before a forward and after an inverse transform,
// and entry freq(i) after a forward and before an inverse one.  begin() issues
// the loads of the twiddles, finish() (after the line's loads) stages them.

// NLC lines per block in LDS (LineFFT); thread t works on line t % NLC
template <typename T2, int LOG2N, int NLC>
struct LdsEngine {
    using G = FftGeom<LOG2N, NLC>;
    static constexpr int E = 4, NT = G::NT, NL = NLC, n = G::n;
    struct Smem { T2 buf[padded(G::E)]; };
    LineFFT<T2, LOG2N, NLC> fft;
    T2 *buf;
    int lb, j0;
    __device__ __forceinline__ LdsEngine(Smem &sm) : buf(sm.buf), lb(threadIdx.x % NLC), j0(threadIdx.x / NLC) {}
    __device__ __forceinline__ void begin(const T2 *table) { fft.prefetch(table, 1); }
    __device__ __forceinline__ void finish(const T2 *) {}
    __device__ __forceinline__ int line() const { return lb; }
    __device__ __forceinline__ int in(int i) const { return j0 + i * (NT / NLC); }
    __device__ __forceinline__ int freq(int i) const { return in(i); }
    template <bool INV>
    __device__ __forceinline__ void run(T2 (&v)[E]) {
        __syncthreads();  // the previous transform's reads
#pragma unroll
        for(int i = 0; i < E; i++) buf[pidx(lb * n + in(i))] = v[i];
        __syncthreads();
        fft.template run<INV>(buf);
#pragma unroll
        for(int i = 0; i < E; i++) v[i] = buf[pidx(lb * n + in(i))];
    }
    __device__ __forceinline__ void forward(T2 (&v)[E]) { run<false>(v); }
    __device__ __forceinline__ void inverse(T2 (&v)[E]) { run<true>(v); }
};

// two waves per line (the scheme of k_colw2): half-length transforms of the
// even and odd entries joined by one exchange.  N = 512 uses the 256-point
// four-pass transform, so that its 257 lines fill 514 waves.
template <typename T2, int LOG2N>
struct TwoWaveEngine {
    static constexpr int n = 1 << LOG2N, n2 = n / 2, E = n2 / 64, NT = 128, NL = 1;
    using F = std::conditional_t<LOG2N == 9, WaveFFT4<T2>, WaveFFT<T2, LOG2N == 9 ? 9 : LOG2N - 1>>;
    using Stage = TwiddleStage<T2, n>;
    static constexpr int TWR = Stage::on ? n / NT : 1;
    struct Smem {
        T2 lds[2][F::LDS];
        Stage stage;
    };
    Smem &sm;
    const T2 *tw = nullptr;
    T2 *own, *other;
    int lane, h;
    T2 twr[TWR];
    __device__ __forceinline__ TwoWaveEngine(Smem &s) : sm(s) {
        lane = threadIdx.x & 63;
        h = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        own = sm.lds[h];
        other = sm.lds[h ^ 1];
    }
    __device__ __forceinline__ void begin(const T2 *table) { sm.stage.template load<NT>(table, threadIdx.x, twr); }
    __device__ __forceinline__ void finish(const T2 *table) {
        tw = sm.stage.template store<NT>(table, threadIdx.x, twr);  // visible after the next barrier
    }
    __device__ __forceinline__ int line() const { return 0; }
    __device__ __forceinline__ int in(int m) const { return 2 * (lane + 64 * m) + h; }
    __device__ __forceinline__ int freq(int m) const { return lane + 64 * m + h * n2; }
    template <bool INV>
    __device__ __forceinline__ void half(T2 (&v)[E]) {
        if constexpr(LOG2N == 9) {
            lds_barrier();
            F::template run<INV>(lane, v, own, tw, 2);
        }
        else {
            wave_transform<T2, LOG2N - 1, INV>(lane, v, own, tw, 2);
        }
    }
    __device__ __forceinline__ void forward(T2 (&v)[E]) {
        half<false>(v);
#pragma unroll
        for(int m = 0; m < E; m++)
            if(h == 1) v[m] = cmul(v[m], tw[lane + 64 * m]);
        wave_lds_sync();  // the other wave has not read this buffer since the transform's barrier
#pragma unroll
        for(int m = 0; m < E; m++) own[lane + 64 * m] = v[m];
        lds_barrier();
#pragma unroll
        for(int m = 0; m < E; m++) {
            const T2 o = other[lane + 64 * m];
            v[m] = h == 0 ? cadd(v[m], o) : csub(o, v[m]);
        }
    }
    __device__ __forceinline__ void inverse(T2 (&v)[E]) {
        lds_barrier();
#pragma unroll
        for(int m = 0; m < E; m++) own[lane + 64 * m] = v[m];
        lds_barrier();
#pragma unroll
        for(int m = 0; m < E; m++) {
            const T2 o = other[lane + 64 * m];
            if(h == 0) v[m] = cadd(v[m], o);
            else v[m] = cmul(csub(o, v[m]), conj_(tw[lane + 64 * m]));
        }
        half<true>(v);
    }
};

// lines per block of the LDS engine: in 2D few (N / 2 + 1 lines have to reach
// many CUs, 64 threads per block), in 3D as the axis passes (k_col)
template <int LOG2N, int DIMS>
constexpr int engine_lines() {
    return DIMS == 3 ? ColLines<LOG2N>::value : (LOG2N >= 8 ? 1 : (256 >> LOG2N));
}

template <typename T, int LOG2N, int DIMS>
using Engine = std::conditional_t<(LOG2N >= 9 && LOG2N <= 11), TwoWaveEngine<typename Complex<T>::type, (LOG2N >= 9 && LOG2N <= 11) ? LOG2N : 10>,
                                  LdsEngine<typename Complex<T>::type, LOG2N, engine_lines<LOG2N, DIMS>()>>;

// k_col grid: the line groups padded to a multiple of the 8 XCDs
static inline int col_blocks(int lines, int nlc) { return ((lines + nlc - 1) / nlc + 7) / 8 * 8; }

// Half-spectrum layout: (z, y, kx) with kx fastest, FFTW's r2c layout
// (PseudospectralCPU.cpp:90-96), in 1D, 2D and 3D.  (A transposed 2D layout,
// whole contiguous lines for the column pass, measured slower overall on
// MI355X: the column pass gained 5 %, the x passes lost 18 %.)
struct SpecLayout {
    long rs, ks;              // x pass: entry (row, kx) at row * rs + kx * ks
    long yP, yls, ystride;    // y pass: line l at (l / Nh) * yP + (l % Nh) * yls, step ystride
    long zP, zls, zstride;    // z pass (3D)
    bool ycontig;
};

static SpecLayout spec_layout(int dims, int N) {
    const long Nh = N / 2 + 1;
    (void)dims;
    return SpecLayout{Nh, 1, (long)N * Nh, 1, Nh, Nh, 1, (long)N * Nh, false};
}

}  // namespace chd
