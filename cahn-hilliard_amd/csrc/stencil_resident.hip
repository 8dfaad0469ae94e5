// stencil_resident.hip -- many euler / euler_mobility steps per launch on grids
// that one block holds, and on 1D grids of any size.
//
//   2D N = 64                  wave_region's whole mode (stencil_wave.h)
//   1D N <= 1024, 2D N <= 32,  k_resident: the whole periodic grid, one to four
//   3D N <= 16                 cells per thread, psi in registers, neighbours
//                              through LDS, two barriers per step
//   1D N > 1024                the same on tiles of 512 cells with a halo of two
//                              cells per step, up to 32 steps per launch
// On such grids a step is a fraction of a microsecond of work and a launch costs
// two to three, so the time is the number of launches: one per step (2D N < 64,
// 1D, 3D), one per 8 steps (2D N = 64) before.  The per-cell arithmetic is
// ch_device.h's: the same bits as one step per launch.  us per step on MI355X,
// Landau euler in FP64 where nothing else is said, before -> now:
//   1D N = 64      1.64 -> 0.18      2D N = 16  1.92 -> 0.26    3D N = 8   2.63 -> 0.34
//   1D N = 1024    2.29 -> 0.33      2D N = 32  2.65 -> 0.36    3D N = 16  5.09 -> 1.28
//   1D N = 4096    2.18 -> 0.36      2D N = 64  1.07 -> 0.81
//   1D N = 65536   2.22 -> 0.37      2D N = 64, FP32  0.78 -> 0.59
//   1D N = 2^20    4.93 -> 1.26      2D N = 64, Wertheim, free-energy mobility  3.72 -> 3.40
// What is left is one compute unit's: two barriers and LDS trips per step on the
// smallest grids, and at 2D N = 64 its vector instructions (80 per wave and step
// on 16 waves, 0.59 us of the 0.81; 8 x 8 waves 0.813, 16 x 4 waves 0.828).
#include "ch_internal.h"
#include "stencil_wave.h"

namespace chd {

namespace {

// steps of one launch where the whole grid is resident (a few milliseconds)
constexpr int kResidentSteps = 4096;
// steps per launch and threads (region cells) of a 1D tile
constexpr int kTile1D = 512, kTile1DSteps = 32;

// one step's two phases on the block's cells: `at` the cell's LDS place, nm / nq
// its neighbours' places
template <typename T, int DIMS, int MODEL, int MOB, bool EM, int CPT, int CELLS>
struct Resident {
    static constexpr bool VARM = EM && MOB != CH_MOB_CONSTANT;
    struct Smem {
        T P[CELLS], U[CELLS], V[VARM ? CELLS : 1];
    };
    __device__ __forceinline__ static void steps(const Params &p, Smem &sm, T (&psi)[CPT], const int (&at)[CPT],
                                                 const int (&nm)[CPT][DIMS], const int (&nq)[CPT][DIMS], int n) {
        const T Mc = (T)p.M;
#pragma unroll 1
        for(int s = 0; s < n; s++) {
#pragma unroll
            for(int k = 0; k < CPT; k++) sm.P[at[k]] = psi[k];
            lds_barrier();
            T mu[CPT], mob[CPT];
#pragma unroll
            for(int k = 0; k < CPT; k++) {
                T m[DIMS], q[DIMS];
#pragma unroll
                for(int d = 0; d < DIMS; d++) {
                    m[d] = sm.P[nm[k][d]];
                    q[d] = sm.P[nq[k][d]];
                }
                mu[k] = chem_pot<T, DIMS, MODEL>(p, psi[k], m, q);
                sm.U[at[k]] = mu[k];
                if constexpr(VARM) {
                    mob[k] = mobility<T, MOB>(p, psi[k]);
                    sm.V[at[k]] = mob[k];
                }
            }
            lds_barrier();
#pragma unroll
            for(int k = 0; k < CPT; k++) {
                T m[DIMS], q[DIMS], Mm[DIMS], Mq[DIMS];
#pragma unroll
                for(int d = 0; d < DIMS; d++) {
                    m[d] = sm.U[nm[k][d]];
                    q[d] = sm.U[nq[k][d]];
                    if constexpr(VARM) {
                        Mm[d] = sm.V[nm[k][d]];
                        Mq[d] = sm.V[nq[k][d]];
                    }
                    else {
                        Mm[d] = Mc;
                        Mq[d] = Mc;
                    }
                }
                if constexpr(!EM) psi[k] = euler_update<T, DIMS>(p, psi[k], mu[k], m, q);
                else psi[k] = mobility_update<T, DIMS>(p, psi[k], mu[k], m, q, VARM ? mob[k] : Mc, Mm, Mq);
            }
        }
    }
};

// the whole grid of 2^(DIMS log2N) <= NT CPT cells; threads beyond it repeat
// cells (the same values in the same places)
template <typename T, int DIMS, int MODEL, int MOB, bool EM, int NT, int CPT>
__global__ __launch_bounds__(NT) void k_resident(const T *__restrict__ in, T *__restrict__ out, Params p, int steps) {
    using R = Resident<T, DIMS, MODEL, MOB, EM, CPT, NT * CPT>;
    __shared__ typename R::Smem sm;
    const int L = p.log2N, mask = p.mask, all = (1 << (DIMS * L)) - 1;
    T psi[CPT];
    int at[CPT], nm[CPT][DIMS], nq[CPT][DIMS];
#pragma unroll
    for(int k = 0; k < CPT; k++) {
        const int i = (threadIdx.x + NT * k) & all;
        at[k] = i;
#pragma unroll
        for(int d = 0; d < DIMS; d++) {
            const int c = (i >> (d * L)) & mask, rest = i & ~(mask << (d * L));
            nm[k][d] = rest | (((c - 1) & mask) << (d * L));
            nq[k][d] = rest | (((c + 1) & mask) << (d * L));
        }
        psi[k] = in[i];
    }
    R::steps(p, sm, psi, at, nm, nq, steps);
#pragma unroll
    for(int k = 0; k < CPT; k++)
        if((int)threadIdx.x + NT * k <= all) out[at[k]] = psi[k];
}

// 1D tiles: kTile1D cells around an interior of kTile1D - 4 kTile1DSteps
template <typename T, int MODEL, int MOB, bool EM>
__global__ __launch_bounds__(kTile1D) void k_tiles1d(const T *__restrict__ in, T *__restrict__ out, Params p, int steps) {
    constexpr int NT = kTile1D, H = 2 * kTile1DSteps, W = NT - 2 * H;
    using R = Resident<T, 1, MODEL, MOB, EM, 1, NT>;
    __shared__ typename R::Smem sm;
    const int r = threadIdx.x;
    const int64_t x0 = (int64_t)xcd_tile(blockIdx.x, gridDim.x) * W - H;
    const int64_t x = (x0 + r) & p.mask;
    T psi[1] = {in[x]};
    // the outermost cells read themselves: wrong values, two cells further in per step
    const int at[1] = {r}, nm[1][1] = {{r > 0 ? r - 1 : 0}}, nq[1][1] = {{r < NT - 1 ? r + 1 : NT - 1}};
    R::steps(p, sm, psi, at, nm, nq, steps);
    if(r >= H && r < NT - H && x0 + r < p.N) out[x0 + r] = psi[0];
}

template <typename T, int MODEL, int MOB, bool EM>
__global__ __launch_bounds__(1024) void k_whole64(const T *__restrict__ in, T *__restrict__ out, Params p, int steps) {
    using CFG = WaveCfg<1, 4, 16>;
    __shared__ WaveExchange<T, exchange_fields<MOB, EM>(), CFG::NW, CFG::C> ex;
    wave_region<T, MODEL, MOB, EM, 8, CFG, true>(in, out, p, 0, 0, ex, nullptr, nullptr, steps);
}

template <typename T, int MODEL, int MOB, bool EM>
hipError_t multi_t(const Params &p, int steps, const T *in, T *out, hipStream_t s) {
    auto go = [&](auto kernel, int nb, int nt) {
        hipLaunchKernelGGL(kernel, dim3(nb), dim3(nt), 0, s, in, out, p, steps);
        return hipGetLastError();
    };
    if(p.dims == 1) {
        if(p.N <= 64) return go(k_resident<T, 1, MODEL, MOB, EM, 64, 1>, 1, 64);
        if(p.N <= 256) return go(k_resident<T, 1, MODEL, MOB, EM, 256, 1>, 1, 256);
        if(p.N <= 1024) return go(k_resident<T, 1, MODEL, MOB, EM, 1024, 1>, 1, 1024);
        constexpr int W = kTile1D - 4 * kTile1DSteps;
        return go(k_tiles1d<T, MODEL, MOB, EM>, (p.N + W - 1) / W, kTile1D);
    }
    if(p.dims == 2) {
        if(p.N <= 8) return go(k_resident<T, 2, MODEL, MOB, EM, 64, 1>, 1, 64);
        if(p.N == 16) return go(k_resident<T, 2, MODEL, MOB, EM, 256, 1>, 1, 256);
        if(p.N == 32) return go(k_resident<T, 2, MODEL, MOB, EM, 1024, 1>, 1, 1024);
        return go(k_whole64<T, MODEL, MOB, EM>, 1, 1024);
    }
    if(p.N == 4) return go(k_resident<T, 3, MODEL, MOB, EM, 64, 1>, 1, 64);
    if(p.N == 8) return go(k_resident<T, 3, MODEL, MOB, EM, 512, 1>, 1, 512);
    return go(k_resident<T, 3, MODEL, MOB, EM, 1024, 4>, 1, 1024);
}

template <typename T, int MODEL>
hipError_t multi_model(const Params &p, int integrator, int mob, int steps, const void *in, void *out, hipStream_t s) {
    const T *a = (const T *)in;
    T *b = (T *)out;
    if(integrator == CH_EULER) return multi_t<T, MODEL, CH_MOB_CONSTANT, false>(p, steps, a, b, s);
    switch(mob) {
    case CH_MOB_CONSTANT: return multi_t<T, MODEL, CH_MOB_CONSTANT, true>(p, steps, a, b, s);
    case CH_MOB_REGULARISED: return multi_t<T, MODEL, CH_MOB_REGULARISED, true>(p, steps, a, b, s);
    case CH_MOB_LINEAR: return multi_t<T, MODEL, CH_MOB_LINEAR, true>(p, steps, a, b, s);
    case CH_MOB_FREE_ENERGY:
        if constexpr(MODEL == CH_SIMPLE_WERTHEIM) return multi_t<T, MODEL, CH_MOB_FREE_ENERGY, true>(p, steps, a, b, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

int stencil_multi_steps(int dims, int N) {
    if(dims == 1) return N <= 1024 ? kResidentSteps : kTile1DSteps;
    return N <= (dims == 2 ? 64 : 16) ? kResidentSteps : 0;
}

hipError_t stencil_multi(const Params &p, int precision, int integrator, int model, int mob, int steps, const void *in,
                         void *out, hipStream_t s) {
    if(steps < 1 || steps > stencil_multi_steps(p.dims, p.N)) return hipErrorInvalidValue;
    if(precision == CH_FP64) {
        if(model == CH_LANDAU) return multi_model<double, CH_LANDAU>(p, integrator, mob, steps, in, out, s);
        return multi_model<double, CH_SIMPLE_WERTHEIM>(p, integrator, mob, steps, in, out, s);
    }
    if(model == CH_LANDAU) return multi_model<float, CH_LANDAU>(p, integrator, mob, steps, in, out, s);
    return multi_model<float, CH_SIMPLE_WERTHEIM>(p, integrator, mob, steps, in, out, s);
}

}  // namespace chd
