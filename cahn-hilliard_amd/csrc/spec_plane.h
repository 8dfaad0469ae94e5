// spec_plane.h -- the y and x passes between two 3D pseudospectral steps, one
// z plane per block.
//
// Between the last-axis passes of two steps the chain takes each plane of W
// through y inverse, x c2r, f', x r2c, y forward.  As separate passes these are
// three launches that each read and write W; here the plane (N (N/2 + 1) complex
// values: 67 KB in FP32 at N = 128, of the 160 KB of LDS) stays in LDS and
// registers, and W is read and written once.
//
// A line of L = R1 R2 points is transformed by R2 threads with R1 entries each
// (entries j + R2 r of thread j) in two register butterflies around one exchange:
//   X_{k + R1 m} = sum_j W_R2^{j m} W_L^{j k} sum_r x_{j + R2 r} W_R1^{r k}.
// The outputs k = j + R2 i, m of thread j are the entries j + R2 (i + (R1/R2) m):
// the distribution of the inputs, so transforms chain without a rearrangement.
// Columns are spread with the lanes along kx, rows with the lanes along y; the
// plane's pitch N/2 + 1 is odd, so both orders reach distinct LDS banks.
#pragma once

#include "line_fft.h"

namespace chd {

template <int L>
struct TwoPass {
    static constexpr int R1 = L >= 128 ? 16 : (L >= 32 ? 8 : 4), R2 = L / R1, I = R1 / R2;
    static_assert(R1 * R2 == L && R1 % R2 == 0, "R1 R2 = L, R2 divides R1");

    // entry (k, j) of the exchange at S[(k R2 + j) lines + line]; tw: W_L^m at tw[m ts]
    template <bool INV, typename T2>
    __device__ __forceinline__ static void run(T2 (&v)[R1], T2 *S, int lines, int line, int j, bool on, const T2 *tw,
                                               int ts) {
        dft<R1, INV>(v);
#pragma unroll
        for(int k = 1; k < R1; k++) {
            const T2 w = tw[j * k * ts];
            v[k] = w_mul(v[k], INV ? T2{w.x, -w.y} : w);
        }
        lds_barrier();  // earlier reads of S
        if(on) {
#pragma unroll
            for(int k = 0; k < R1; k++) S[(k * R2 + j) * lines + line] = v[k];
        }
        lds_barrier();
#pragma unroll
        for(int i = 0; i < I; i++) {
            T2 u[R2];
            if(on) {
#pragma unroll
                for(int q = 0; q < R2; q++) u[q] = S[((j + R2 * i) * R2 + q) * lines + line];
            }
            dft<R2, INV>(u);
#pragma unroll
            for(int m = 0; m < R2; m++) v[i + I * m] = u[m];
        }
    }
};

template <int LOG2N>
struct PlaneGeom {
    static constexpr int N = 1 << LOG2N, n = N / 2, Nh = n + 1;
    using Col = TwoPass<N>;
    using Row = TwoPass<n>;
    static constexpr int TC = Nh * Col::R2, TR = N * Row::R2;  // threads of the column and row passes
    static constexpr int NT = ((TC > TR ? TC : TR) + 63) / 64 * 64;
};

// PLANE_BOTH: between two steps; rho (may be null): the c2r rows are also stored
// there.  PLANE_R2C / PLANE_FPRIME: only x r2c (of f') and y forward, from rho
// (the start of a chain); PLANE_C2R: only y inverse and x c2r, into rho (its end):
// the same operations, so a chain may be split anywhere with the same bits.
enum { PLANE_BOTH = 0, PLANE_R2C = 1, PLANE_FPRIME = 2, PLANE_C2R = 3 };
template <typename T, int MODEL, int LOG2N, int PART>
__global__ __launch_bounds__(PlaneGeom<LOG2N>::NT) void k_ps_plane(const typename Complex<T>::type *in,
                                                                   typename Complex<T>::type *out,
                                                                   const typename Complex<T>::type *__restrict__ table,
                                                                   Params p, T *__restrict__ rho) {
    using T2 = typename Complex<T>::type;
    using G = PlaneGeom<LOG2N>;
    using Col = typename G::Col;
    using Row = typename G::Row;
    constexpr int N = G::N, n = G::n, Nh = G::Nh;
    constexpr bool INVERSE = PART == PLANE_BOTH || PART == PLANE_C2R, FORWARD = PART != PLANE_C2R;
    __shared__ T2 S[N * Nh];
    __shared__ T2 tw[N];
    const int t = threadIdx.x;
    const int z = xcd_tile(blockIdx.x, gridDim.x);
    const size_t plane = (size_t)z * N * Nh;
    const bool con = t < G::TC, ron = t < G::TR;
    const int c = con ? t % Nh : 0, cj = con ? t / Nh : 0;  // column, its thread
    const int y = t % N, rj = ron ? t / N : 0;              // row, its thread
    T2 *row = reinterpret_cast<T2 *>(rho + ((size_t)z * N + y) * N);
    T2 v[Col::R1], u[Row::R1];
    if constexpr(INVERSE) {
#pragma unroll
        for(int r = 0; r < Col::R1; r++) v[r] = in[plane + (cj + Col::R2 * r) * Nh + c];
    }
    else {
#pragma unroll
        for(int r = 0; r < Row::R1; r++) u[r] = row[rj + Row::R2 * r];
    }
    for(int i = t; i < N; i += G::NT) tw[i] = table[i];
    lds_barrier();
    if constexpr(INVERSE) {
        Col::template run<true>(v, S, Nh, c, cj, con, tw, 1);
        lds_barrier();
        if(con) {
#pragma unroll
            for(int r = 0; r < Col::R1; r++) S[(cj + Col::R2 * r) * Nh + c] = v[r];
        }
        lds_barrier();
#pragma unroll
        for(int r = 0; r < Row::R1; r++) u[r] = c2r_entry<T2>(S + y * Nh, 1, rj + Row::R2 * r, n, tw);
        Row::template run<true>(u, S, N, y, rj, ron, tw, 2);
        if((PART == PLANE_C2R || rho) && ron) {
#pragma unroll
            for(int r = 0; r < Row::R1; r++) row[rj + Row::R2 * r] = u[r];
        }
    }
    if constexpr(FORWARD) {
        if constexpr(PART != PLANE_R2C) {
#pragma unroll
            for(int r = 0; r < Row::R1; r++) u[r] = T2{fprime<T, MODEL>(p, u[r].x), fprime<T, MODEL>(p, u[r].y)};
        }
        Row::template run<false>(u, S, N, y, rj, ron, tw, 2);
        lds_barrier();
        if(ron) {
#pragma unroll
            for(int r = 0; r < Row::R1; r++) S[(rj + Row::R2 * r) * N + y] = u[r];
        }
        lds_barrier();
        const T2 z0 = u[0];
#pragma unroll
        for(int r = 0; r < Row::R1; r++) {
            const int k = rj + Row::R2 * r;
            u[r] = r2c_entry<T>(u[r], S[(k == 0 ? 0 : n - k) * N + y], tw[k]);
        }
        lds_barrier();
        if(ron) {
#pragma unroll
            for(int r = 0; r < Row::R1; r++) S[y * Nh + rj + Row::R2 * r] = u[r];
            if(rj == 0) S[y * Nh + n] = r2c_entry<T>(z0, z0, tw[n]);
        }
        lds_barrier();
#pragma unroll
        for(int r = 0; r < Col::R1; r++) v[r] = S[(cj + Col::R2 * r) * Nh + c];
        Col::template run<false>(v, S, Nh, c, cj, con, tw, 1);
        if(con) {
#pragma unroll
            for(int r = 0; r < Col::R1; r++) out[plane + (cj + Col::R2 * r) * Nh + c] = v[r];
        }
    }
}

// whether the plane pass covers the size (3D, N = 32, 64; 128 in FP32).  us per
// step with it and with the separate passes: N = 32 10.9 / 21.1 FP64, 10.1 /
// 19.8 FP32; N = 64 15.6 / 23.8, 12.8 / 20.5; N = 128 29.8 / 39.5 in FP32, but
// 61.7 / 57.0 in FP64, whose 16 entries per column thread spill and whose 135 KB
// leave one block per CU.
template <typename T>
constexpr bool plane_len(int log2N) { return log2N >= 5 && log2N <= (sizeof(T) == 4 ? 7 : 6); }

template <typename T, int MODEL, int LOG2N, int PART>
void launch_plane(typename Complex<T>::type *W, const typename Complex<T>::type *tw, const Params &p, T *rho,
                  hipStream_t s) {
    hipLaunchKernelGGL((k_ps_plane<T, MODEL, LOG2N, PART>), dim3(1 << LOG2N), dim3(PlaneGeom<LOG2N>::NT), 0, s, W, W,
                       tw, p, rho);
}

}  // namespace chd
