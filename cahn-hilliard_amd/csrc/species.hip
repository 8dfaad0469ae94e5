// species.hip -- multi-species Wertheim models and their integrators.
//
// Models (per cell, on the species vector rho_s, FP64 in both precisions):
//   SalehWertheim   src/models/SalehWertheim.cpp:47-110    3 species, closed-form X
//   RicciWertheim   src/models/RicciWertheim.cpp:43-98     2 species, closed-form X
//   GenericWertheim src/models/GenericWertheim.cpp:184-291 any patch topology:
//       X_p = 1 / (1 + sum_terms rho_s X_q c), Gauss-Seidel sweeps over the
//       patch types in ascending order until a sweep moves no X by 1e-8
//       (at most 10000 sweeps), warm-started from the cell's X of the
//       previous evaluation (X lives in HBM, patch-major, n_patches per cell).
// A species whose density is exactly 0 gets f' = 0 (the reference leaves its
// previous value in a static buffer).  f' takes its logarithms from
// log_series (ch_device.h, within 2 ulp); the free energy keeps the library's.
//
// Integrators over species-major fields rho[s * bins + i]:
//   (generic models of at most 4 species and 4 patch types: small_update_X)
//   euler / euler_mobility: k_sp_mu (mobility from the previous X, X update,
//     f', mu_s = f'_s - 2 k_s lap rho_s) then k_sp_update (rho_s += dt M lap mu_s,
//     or the flux form with M_s per species), in place: 2 launches per step
//     (EulerCPU.cpp:18-36, EulerMobilityCPU.cpp:31-83 over species);
//   pseudospectral: k_sp_fprime, then per species r2c, the update (k_s in the
//     denominator, PseudospectralCPU.cpp:112-136) and c2r; in 2D the columns'
//     transforms and the update are one pass (k_sp_ps_col), else k_sp_ps_update.
#include <algorithm>
#include <cmath>

#include "ch_internal.h"
#include "line_fft.h"

namespace chd {

namespace {

template <typename T>
using C2 = typename Complex<T>::type;

constexpr int kSpBlocks = 2048;

// more than kSpSmall species or patch types, and the free energy: the bare sweeps
__device__ void generic_update_X(const SpModel &m, const double *rhos, double *X) {
#pragma clang fp contract(off)
    for(int iter = 0; iter < 10000; iter++) {
        double max_delta = 0.0;
        for(int u = 0; u < m.n_unique; u++) {
            const int patch = m.unique[u];
            double sum = 0.0;
            for(int t = m.term_start[u]; t < m.term_start[u + 1]; t++) {
                const double rho = rhos[m.t_species[t]];
                if(rho != 0.0) sum += rho * X[m.t_other[t]] * m.t_coeff[t];
            }
            const double new_X = 1.0 / (1.0 + sum);
            const double d = fabs(new_X - X[patch]);
            max_delta = (max_delta < d) ? d : max_delta;
            X[patch] = new_X;
        }
        if(max_delta < 1e-8) return;
    }
}

// ln X of one Saleh bonding site; rf = delta (valence rho + lh rho_linker)
__device__ __forceinline__ double saleh_log_X(const SpSmallModel &m, const double (&rhos)[3], int species) {
#pragma clang fp contract(off)
    const double delta = species == 0 ? m.dAA : m.dBB;
    const double rho_factor = delta * (m.val[species] * rhos[species] + m.lh * rhos[2]);
    const double X = (-1.0 + sqrt(1.0 + 4.0 * rho_factor)) / (2.0 * rho_factor);
    return rho_factor >= 0 ? log_series(X) : 0.0;
}

// generic_update_X's sweeps, on X_p = 1 / (1 + sum_q a_pq X_q)
template <int P, bool SHORT>
__device__ __forceinline__ void small_sweeps(const double (&a)[P][P], double (&X)[P]) {
#pragma clang fp contract(off)
#pragma unroll 1
    for(int iter = 0; iter < 10000; iter++) {
        double max_delta = 0.0;
#pragma unroll
        for(int p = 0; p < P; p++) {
            double sum = 1.0;
#pragma unroll
            for(int q = 0; q < P; q++) sum = __builtin_fma(a[p][q], X[q], sum);
            const double new_X = SHORT ? recip_newton(sum) : 1.0 / sum;
            const double d = fabs(new_X - X[p]);
            max_delta = (max_delta < d) ? d : max_delta;
            X[p] = new_X;
        }
        if(max_delta < 1e-8) return;
    }
}

// generic_update_X for a small model: the same sweeps in the same order with
// a_pq = delta_pq sum_s rho_s n_sq formed once per cell.  A cell needs some 200
// sweeps from X = 1 and a few per time step, each a dependent chain, so the
// chain's length and its branches are what count: P^2 fused terms, the short
// reciprocal and no branch per sweep, where the general form tests and indexes
// every (species, patch) pair (2D N = 256, 3 species, 2 patch types, FP64: see
// k_sp_mu).  Densities that are negative, NaN or huge take the IEEE division.
// Newton steps between the sweeps reach the fixed point in 3 sweeps, but not
// the state at which the reference's rule stops: up to 8e-8 away for slowly
// contracting topologies.
template <int P>
__device__ __forceinline__ void small_update_X(const SpSmallModel &m, const double (&rhos)[kSpSmall], double (&X)[P]) {
#pragma clang fp contract(off)
    double a[P][P];
    bool tame = true;
#pragma unroll
    for(int q = 0; q < P; q++) {
        double n = 0.0;
#pragma unroll
        for(int s = 0; s < kSpSmall; s++)
            if(s < m.S) n += rhos[s] * (double)m.pc[s][q];
#pragma unroll
        for(int p = 0; p < P; p++) {
            a[p][q] = m.dl[p][q] * n;
            tame = tame && a[p][q] >= 0.0 && a[p][q] < 0x1p90;
        }
    }
    if(tame) small_sweeps<P, true>(a, X);
    else small_sweeps<P, false>(a, X);
}

// A model whose species and patch vectors have sizes known at compile time
// keeps them in registers; the others (dyn: more than kSpSmall species or patch
// types, or a patch type that no species carries) index them at run time.  S, P: sizes of the vectors; exact: S is the
// number of species (else it is m.S <= S).
struct SalehModel {
    using M = SpSmallModel;
    static constexpr int model = CH_SALEH_WERTHEIM, S = 3, P = 1;
    static constexpr bool exact = true, dyn = false;
};
struct RicciModel {
    using M = SpSmallModel;
    static constexpr int model = CH_RICCI_WERTHEIM, S = 2, P = 1;
    static constexpr bool exact = true, dyn = false;
};
template <int P_>
struct SmallModel {
    using M = SpSmallModel;
    static constexpr int model = CH_GENERIC_WERTHEIM, S = kSpSmall, P = P_;
    static constexpr bool exact = false, dyn = false;
};
struct LargeModel {
    using M = const SpModel *;
    static constexpr int model = CH_GENERIC_WERTHEIM, S = kSpMaxSpecies, P = kSpMaxPatches;
    static constexpr bool dyn = true;
};
__device__ __forceinline__ const SpSmallModel &model_of(const SpSmallModel &m) { return m; }
__device__ __forceinline__ const SpModel &model_of(const SpModel *const &m) { return *m; }

// f(s) for every species s of the model (unrolled where the sizes are static)
template <class MD, class M, typename F>
__device__ __forceinline__ void each_species(const M &m, F &&f) {
    if constexpr(MD::dyn) {
        for(int s = 0; s < m.S; s++) f(s);
    }
    else {
#pragma unroll
        for(int s = 0; s < MD::S; s++)
            if(MD::exact || s < m.S) f(s);
    }
}
// f(q) for every patch type of a generic model
template <class MD, class M, typename F>
__device__ __forceinline__ void each_patch(const M &m, F &&f) {
    if constexpr(MD::model != CH_GENERIC_WERTHEIM) return;
    else if constexpr(MD::dyn) {
        for(int q = 0; q < m.P; q++) f(q);
    }
    else {
#pragma unroll
        for(int q = 0; q < MD::P; q++) f(q);
    }
}

template <class MD, class M>
__device__ __forceinline__ void update_X(const M &m, const double (&rhos)[MD::S], double (&X)[MD::P]) {
    if constexpr(MD::dyn) generic_update_X(m, rhos, X);
    else if constexpr(MD::model == CH_GENERIC_WERTHEIM) small_update_X<MD::P>(m, rhos, X);
}

// f' of every species at one cell; X (Generic) in/out
template <class MD, class M>
__device__ __forceinline__ void sp_fprime(const M &m, const double (&rhos)[MD::S], double (&X)[MD::P],
                                          double (&out)[MD::S]) {
#pragma clang fp contract(off)
    double rho_tot = 0.;
    each_species<MD>(m, [&](int s) { rho_tot += rhos[s]; });
    if constexpr(MD::model == CH_SALEH_WERTHEIM) {
        const double c0 = saleh_log_X(m, rhos, 0), c1 = saleh_log_X(m, rhos, 1);
        const double bond[3] = {m.val[0] * c0, m.val[1] * c1, m.lh * (c0 + c1)};
#pragma unroll
        for(int s = 0; s < 3; s++) {
            const double ref = log_series(rhos[s]) + 2.0 * m.sB2 * rho_tot + 3.0 * m.sB3 * (rho_tot * rho_tot);
            out[s] = rhos[s] == 0. ? 0.0 : ref + bond[s];
        }
    }
    else if constexpr(MD::model == CH_RICCI_WERTHEIM) {
        const double A = rhos[1] * m.d12, B = rhos[0] * m.d12;
        const double X0 = (-1 + sqrt((1 + 12 * rhos[0] * m.d00))) / (6 * rhos[0] * m.d00);
        const double u = 1 + 2 * A - B;
        const double X1 = (B - 1 - 2 * A + sqrt(u * u + 4 * B)) / (2 * B);
        const double v = B - 2 * A + 1;
        const double X2 = (-B + 2 * A - 1 + sqrt(v * v + 8 * A)) / (4 * A);
        const double bond[2] = {3 * log_series(X0) + log_series(X1), 2 * log_series(X2)};
#pragma unroll
        for(int s = 0; s < 2; s++) {
            const double ref = log_series(rhos[s]) + 2.0 * m.rB2 * rho_tot;
            out[s] = rhos[s] == 0. ? 0.0 : ref + bond[s];
        }
    }
    else {
        update_X<MD>(m, rhos, X);
        double logX[MD::P];
        each_patch<MD>(m, [&](int q) { logX[q] = log_series(X[q]); });
        each_species<MD>(m, [&](int s) {
            double B2c = 0., bond = 0.;
            each_species<MD>(m, [&](int o) { B2c += 2.0 * rhos[o] * m.B2[s][o]; });
            const double ref = log_series(rhos[s]) + B2c;
            each_patch<MD>(m, [&](int q) {
                if(m.pc[s][q] > 0) bond += m.pc[s][q] * logX[q];
            });
            out[s] = rhos[s] == 0. ? 0.0 : ref + bond;
        });
    }
}

// bulk free-energy density at one cell (SalehWertheim.cpp:47-78,
// RicciWertheim.cpp:43-70, GenericWertheim.cpp:210-248; Generic X from 0)
__device__ double sp_bulk(const SpModel &m, double dcf, const double *rhos) {
#pragma clang fp contract(off)
    const int S = m.S;
    double rho = 0.;
    for(int i = 0; i < S; i++) rho += rhos[i];
    double mixing_S = 0., B2c = 0.;
    for(int i = 0; i < S; i++) {
        const double x_i = rhos[i] / rho;
        mixing_S += (x_i > 0) ? x_i * log(x_i) : 0;
        if(m.model == CH_GENERIC_WERTHEIM)
            for(int j = 0; j < S; j++) B2c += rhos[i] * rhos[j] * m.B2[i][j];
    }
    auto term = [](double X) { return log(X) - X / 2.0 + 0.5; };
    if(m.model == CH_SALEH_WERTHEIM) {
        const double f_ref = rho * (log(rho * dcf) - 1.0 + mixing_S + m.sB2 * rho + 0.5 * m.sB3 * (rho * rho));
        double rf = m.dAA * (m.val[0] * rhos[0] + m.lh * rhos[2]);
        const double X1A = (-1.0 + sqrt(1.0 + 4.0 * rf)) / (2.0 * rf);
        const double p1 = term(X1A);
        rf = m.dBB * (m.val[1] * rhos[1] + m.lh * rhos[2]);
        const double X2B = (-1.0 + sqrt(1.0 + 4.0 * rf)) / (2.0 * rf);
        const double p2 = term(X2B);
        return f_ref + (rhos[0] * m.val[0] * p1 + rhos[1] * m.val[1] * p2 + rhos[2] * m.lh * (p1 + p2));
    }
    if(m.model == CH_RICCI_WERTHEIM) {
        const double f_ref = rho * (log(rho * dcf) - 1.0 + mixing_S + m.rB2 * rho);
        const double X0 = (-1 + sqrt((1 + 12 * rhos[0] * m.d00))) / (6 * rhos[0] * m.d00);
        const double A = rhos[1] * m.d12, B = rhos[0] * m.d12;
        const double u = 1 + 2 * A - B, v = B - 2 * A + 1;
        const double X1 = (B - 1 - 2 * A + sqrt(u * u + 4 * B)) / (2 * B);
        const double X2 = (-B + 2 * A - 1 + sqrt(v * v + 8 * A)) / (4 * A);
        double bond = rhos[0] * (3 * (log(X0) - X0 / 2) + log(X1) - X1 / 2 + 2);
        bond += rhos[1] * (2 * log(X2) - X2 + 1);
        return f_ref + bond;
    }
    const double f_ref = rho * (log(rho * dcf) - 1.0 + mixing_S) + B2c;
    double X[kSpMaxPatches];
    for(int q = 0; q < kSpMaxPatches; q++) X[q] = 0.0;
    generic_update_X(m, rhos, X);
    double bond = 0;
    for(int s = 0; s < S; s++) {
        double sf = 0;
        for(int q = 0; q < m.P; q++)
            if(m.pc[s][q] > 0) sf += m.pc[s][q] * term(X[q]);
        bond += rhos[s] * sf;
    }
    return f_ref + bond;
}

// x^n, n >= 1 (patch multiplicities are small): products up to 4, binary powers above
__device__ __forceinline__ double int_power(double x, int n) {
#pragma clang fp contract(off)
    const double x2 = x * x;
    if(n <= 4) return n == 1 ? x : (n == 2 ? x2 : (n == 3 ? x2 * x : x2 * x2));
    double r = 1.0;
    for(;;) {
        if(n & 1) r *= x;
        n >>= 1;
        if(n == 0) return r;
        x *= x;
    }
}

// mobility of species s (RegularisedMobility.h:26-33; GenericWertheim.cpp:276-291)
template <class MD, class M>
__device__ __forceinline__ double sp_mobility(const Params &p, const M &m, int mob, int s, double r,
                                              const double (&X)[MD::P]) {
#pragma clang fp contract(off)
    switch(mob) {
    case CH_MOB_CONSTANT: return p.M;
    case CH_MOB_REGULARISED: return p.M * r / (r + p.rho_min);
    case CH_MOB_LINEAR: return p.M * r / p.rho_ref;
    default: {
        double D = p.M;
        each_patch<MD>(m, [&](int q) {
            if(m.pc[s][q] > 0) D *= int_power(X[q], m.pc[s][q]);
        });
        return r * D;
    }
    }
}

// cell index -> the 2 DIMS neighbour indices (-x, +x, -y, +y, -z, +z)
template <int DIMS>
__device__ __forceinline__ void neighbours(const Params &p, int64_t i, int64_t (&m)[DIMS], int64_t (&q)[DIMS]) {
    const int N = p.N, L = p.log2N, mask = p.mask;
    const int x = (int)(i & mask);
    const int y = DIMS >= 2 ? (int)((i >> L) & mask) : 0;
    const int z = DIMS == 3 ? (int)(i >> (2 * L)) : 0;
    auto idx = [&](int a, int b, int c) { return (int64_t)a + ((int64_t)b << L) + ((int64_t)c << (2 * L)); };
    m[0] = idx((x - 1) & mask, y, z);
    q[0] = idx((x + 1) & mask, y, z);
    if constexpr(DIMS >= 2) {
        m[1] = idx(x, (y - 1) & mask, z);
        q[1] = idx(x, (y + 1) & mask, z);
    }
    if constexpr(DIMS == 3) {
        m[2] = idx(x, y, (z - 1) & mask);
        q[2] = idx(x, y, (z + 1) & mask);
    }
    (void)N;
}

#define SP_CELLS for(int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < bins; i += (int64_t)gridDim.x * 256)

// the densities and X of cell i
template <class MD, class M, typename T>
__device__ __forceinline__ void load_cell(const M &m, const T *__restrict__ rho, const double *__restrict__ Xf,
                                          int64_t i, int64_t bins, double (&rhos)[MD::S], double (&X)[MD::P]) {
    each_species<MD>(m, [&](int s) { rhos[s] = (double)rho[s * bins + i]; });
    each_patch<MD>(m, [&](int q) { X[q] = Xf[q * bins + i]; });
}

// X = 1 (GenericWertheim.cpp:252-254), then the model evaluation of
// CahnHilliard.cpp:226-228 at set-up
template <typename T, class MD>
__global__ __launch_bounds__(256) void k_sp_warm(const T *__restrict__ rho, double *__restrict__ Xf,
                                                 typename MD::M arg, int64_t bins) {
    const auto &m = model_of(arg);
    SP_CELLS {
        double rhos[MD::S], X[MD::P];
        each_species<MD>(m, [&](int s) { rhos[s] = (double)rho[s * bins + i]; });
        each_patch<MD>(m, [&](int q) { X[q] = 1.0; });
        update_X<MD>(m, rhos, X);
        each_patch<MD>(m, [&](int q) { Xf[q * bins + i] = X[q]; });
    }
}

// mu_s = f'_s - 2 k_s lap rho_s (and M_s from the X before this evaluation).
// One cell per thread: at the sizes in use (2D N = 256: one wave per SIMD) the
// model's dependent divisions, roots and logarithms bound it, so the loads are
// all issued first, the species are unrolled to overlap their chains and nothing
// branches on the model's sizes (SmallModel): 7.7 us at 2D N = 256 FP64 with 3
// species, 2 patch types and the free-energy mobility, 16.1 with run-time
// indexed vectors and pow() (k_sp_warm: 41 us, 276).
template <typename T, int DIMS, class MD>
__global__ __launch_bounds__(256) void k_sp_mu(const T *__restrict__ rho, double *__restrict__ Xf, T *__restrict__ mu,
                                               T *__restrict__ mobf, Params p, typename MD::M arg,
                                               int64_t bins, int mob) {
#pragma clang fp contract(off)
    const auto &m = model_of(arg);
    SP_CELLS {
        double rhos[MD::S], X[MD::P], f[MD::S];
        load_cell<MD>(m, rho, Xf, i, bins, rhos, X);
        int64_t nm[DIMS], nq[DIMS];
        neighbours<DIMS>(p, i, nm, nq);
        const T inv_dx2 = (T)p.inv_dx2;
        T lap[MD::S];
        each_species<MD>(m, [&](int s) {
            const T *r = rho + s * bins;
            T a[DIMS], b[DIMS];
#pragma unroll
            for(int d = 0; d < DIMS; d++) {
                a[d] = r[nm[d]];
                b[d] = r[nq[d]];
            }
            lap[s] = laplacian<T, DIMS>((T)rhos[s], a, b, inv_dx2);
        });
        if(mob >= 0)
            each_species<MD>(m, [&](int s) { mobf[s * bins + i] = (T)sp_mobility<MD>(p, m, mob, s, rhos[s], X); });
        sp_fprime<MD>(m, rhos, X, f);
        each_patch<MD>(m, [&](int q) { Xf[q * bins + i] = X[q]; });
        each_species<MD>(m, [&](int s) { mu[s * bins + i] = (T)f[s] - (T)(2 * m.k[s]) * lap[s]; });
    }
}

// rho_s += dt M lap mu_s (euler) or dt div J_s (euler_mobility), in place; one
// species per grid row, so a cell's species run in different blocks
template <typename T, int DIMS, bool EM>
__global__ __launch_bounds__(256) void k_sp_update(T *__restrict__ rho, const T *__restrict__ mu,
                                                   const T *__restrict__ mobf, Params p, int64_t bins) {
#pragma clang fp contract(off)
    const int64_t base = (int64_t)blockIdx.y * bins;
    const T *u = mu + base, *M = mobf + base;
    T *r = rho + base;
    SP_CELLS {
        int64_t nm[DIMS], nq[DIMS];
        neighbours<DIMS>(p, i, nm, nq);
        T a[DIMS], b[DIMS];
#pragma unroll
        for(int d = 0; d < DIMS; d++) {
            a[d] = u[nm[d]];
            b[d] = u[nq[d]];
        }
        if constexpr(!EM) {
            r[i] = euler_update<T, DIMS>(p, r[i], u[i], a, b);
        }
        else {
            T Ma[DIMS], Mb[DIMS];
#pragma unroll
            for(int d = 0; d < DIMS; d++) {
                Ma[d] = M[nm[d]];
                Mb[d] = M[nq[d]];
            }
            r[i] = mobility_update<T, DIMS>(p, r[i], u[i], a, b, M[i], Ma, Mb);
        }
    }
}

// f'_s into out (X updated), the pseudospectral path's model evaluation
template <typename T, class MD>
__global__ __launch_bounds__(256) void k_sp_fprime(const T *__restrict__ rho, double *__restrict__ Xf,
                                                   T *__restrict__ out, typename MD::M arg, int64_t bins) {
    const auto &m = model_of(arg);
    SP_CELLS {
        double rhos[MD::S], X[MD::P], f[MD::S];
        load_cell<MD>(m, rho, Xf, i, bins, rhos, X);
        sp_fprime<MD>(m, rhos, X, f);
        each_patch<MD>(m, [&](int q) { Xf[q * bins + i] = X[q]; });
        each_species<MD>(m, [&](int s) { out[s * bins + i] = (T)f[s]; });
    }
}

// mobility field of every species from rho and the current X
template <typename T>
__global__ __launch_bounds__(256) void k_sp_mob(const T *__restrict__ rho, const double *__restrict__ Xf,
                                                double *__restrict__ out, Params p, const SpModel *__restrict__ mp,
                                                int64_t bins, int mob) {
    const SpModel &m = *mp;
    SP_CELLS {
        double X[kSpMaxPatches];
        for(int q = 0; q < m.P; q++) X[q] = Xf[q * bins + i];
        for(int s = 0; s < m.S; s++)
            out[s * bins + i] = sp_mobility<LargeModel>(p, m, mob, s, (double)rho[s * bins + i], X);
    }
}
#undef SP_CELLS

// the pseudospectral update of one species (PseudospectralCPU.cpp:118-133)
// one spectral entry of the semi-implicit update; k_s in the denominator
template <typename T>
__device__ __forceinline__ void sp_ps_entry(const Params &p, double ks, int ix, int iy, int iz, C2<T> f, C2<T> &r, C2<T> &out) {
#pragma clang fp contract(off)
    double k2, deal;
    mode_q2(p, ix, iy, iz, k2, deal);
    if(p.use_dealias) f = C2<T>{f.x * (T)deal, f.y * (T)deal};
    const double k4 = k2 * k2;
    const T den = (T)(1.0 + p.dt * p.M * (p.S * k2 + 2.0 * ks * k4));
    const T a = (T)(p.dt * p.M * k2), S = (T)p.S, ib = (T)p.inv_bins;
    const T re = (r.x - a * (f.x - S * r.x)) / den;
    const T im = (r.y - a * (f.y - S * r.y)) / den;
    r = C2<T>{re, im};
    out = C2<T>{re * ib, im * ib};
}

template <typename T>
__global__ __launch_bounds__(256) void k_sp_ps_update(C2<T> *__restrict__ rh, C2<T> *__restrict__ fh,
                                                      C2<T> *__restrict__ copy, Params p, int64_t hat, double ks) {
    for(int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < hat; q += (int64_t)gridDim.x * 256) {
        int ix, iy, iz;
        mode_index(p, q, ix, iy, iz);
        C2<T> r = rh[q], o;
        sp_ps_entry<T>(p, ks, ix, iy, iz, fh[q], r, o);
        rh[q] = r;
        copy[q] = o;
    }
}

// 2D up to N = 2048: the column transforms around the update in one pass (the line
// engines of line_fft.h), three launches per species for five, each a start and a
// round trip to what the other XCDs wrote.  Saleh, FP64 on MI355X, us per step, with
// the row passes' smaller blocks (line_fft.h): N = 64 71.0 -> 42.7, 256 82.3 -> 49.2,
// 512 93.8 -> 67.3, 1024 162 -> 108; Generic N = 256 237 -> 66.6 (its sweeps, too).
template <typename T, class ENG>
__global__ __launch_bounds__(ENG::NT) void k_sp_ps_col(const C2<T> *__restrict__ in, C2<T> *__restrict__ out,
                                                       C2<T> *__restrict__ rho_hat, const C2<T> *__restrict__ table, Params p,
                                                       int lines, double ks) {
    constexpr int E = ENG::E, Nh = ENG::n / 2 + 1;
    __shared__ typename ENG::Smem sm;
    const int l0 = xcd_tile(blockIdx.x, gridDim.x) * ENG::NL;
    if(l0 >= lines) return;  // grid padded to a multiple of 8 blocks
    ENG eng(sm);
    eng.begin(table);
    const bool on = ENG::NL == 1 || l0 + eng.line() < lines;
    const int l = on ? l0 + eng.line() : l0;
    C2<T> v[E], rh[E];
#pragma unroll
    for(int i = 0; i < E; i++) v[i] = in[(size_t)eng.in(i) * Nh + l];
#pragma unroll
    for(int i = 0; i < E; i++) rh[i] = rho_hat[(size_t)eng.freq(i) * Nh + l];
    eng.finish(table);
    eng.forward(v);
#pragma unroll
    for(int i = 0; i < E; i++) sp_ps_entry<T>(p, ks, l, eng.freq(i), 0, v[i], rh[i], v[i]);
    eng.inverse(v);
#pragma unroll
    for(int i = 0; i < E; i++)
        if(on) {
            rho_hat[(size_t)eng.freq(i) * Nh + l] = rh[i];
            out[(size_t)eng.in(i) * Nh + l] = v[i];
        }
}

template <typename T, int LOG2N = 2>
static hipError_t sp_ps_col(const SpectralArgs &a, const C2<T> *in, C2<T> *out, C2<T> *rh, double ks, hipStream_t s) {
    if constexpr(LOG2N > 11) return hipErrorInvalidValue;
    else {
        if(a.p.log2N != LOG2N) return sp_ps_col<T, LOG2N + 1>(a, in, out, rh, ks, s);
        using Eng = Engine<T, LOG2N, 2>;
        constexpr int lines = (1 << LOG2N) / 2 + 1;
        hipLaunchKernelGGL((k_sp_ps_col<T, Eng>), dim3(col_blocks(lines, Eng::NL)), dim3(Eng::NT), 0, s, in, out, rh,
                           (const C2<T> *)a.twiddles, a.p, lines, ks);
        return hipGetLastError();
    }
}

// FP64 mass and free energy partials over cells (CahnHilliard.cpp:285-319)
template <typename T, int DIMS>
__global__ __launch_bounds__(256) void k_sp_observables(const T *__restrict__ rho, Params p,
                                                        const SpModel *__restrict__ mp, int64_t bins,
                                                        double *__restrict__ partials) {
#pragma clang fp contract(off)
    const SpModel &m = *mp;
    __shared__ double red[2][256];
    double ms = 0., fe = 0.;
    for(int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < bins; i += (int64_t)gridDim.x * 256) {
        double rhos[kSpMaxSpecies], cell = 0.;
        for(int s = 0; s < m.S; s++) {
            rhos[s] = (double)rho[s * bins + i];
            cell += rhos[s];
        }
        ms += cell;
        int64_t nm[DIMS], nq[DIMS];
        neighbours<DIMS>(p, i, nm, nq);
        double inter = 0.;
        for(int s = 0; s < m.S; s++)
            for(int d = 0; d < DIMS; d++) {
                const double g = ((double)rho[s * bins + nq[d]] - rhos[s]) / p.dx;
                inter += m.k[s] * g * g;
            }
        fe += sp_bulk(m, p.dcf, rhos) + inter;
    }
    red[0][threadIdx.x] = ms;
    red[1][threadIdx.x] = fe;
    __syncthreads();
    for(int k = 128; k > 0; k >>= 1) {
        if(threadIdx.x < k) {
            red[0][threadIdx.x] += red[0][threadIdx.x + k];
            red[1][threadIdx.x] += red[1][threadIdx.x + k];
        }
        __syncthreads();
    }
    if(threadIdx.x == 0) {
        partials[2 * blockIdx.x] = red[0][0];
        partials[2 * blockIdx.x + 1] = red[1][0];
    }
}

template <int DIMS, typename F>
hipError_t by_precision(int precision, F &&f) {
    if(precision == CH_FP64) return f(double{});
    return f(float{});
}

int grid_for(int64_t n) { return (int)std::min<int64_t>(kSpBlocks, (n + 255) / 256); }

bool is_small(const SpModel &m) {
    return m.model != CH_GENERIC_WERTHEIM || (m.S <= kSpSmall && m.P <= kSpSmall && m.n_unique == m.P);
}

SpSmallModel small_model(const SpModel &in) {
    SpSmallModel m{};
    m.model = in.model;
    m.S = in.S;
    m.P = in.P;
    for(int i = 0; i < 3; i++) m.val[i] = in.val[i];
    m.lh = in.lh;
    m.sB2 = in.sB2;
    m.sB3 = in.sB3;
    m.dAA = in.dAA;
    m.dBB = in.dBB;
    m.rB2 = in.rB2;
    m.d00 = in.d00;
    m.d12 = in.d12;
    for(int a = 0; a < kSpSmall; a++) {
        m.k[a] = in.k[a];
        for(int b = 0; b < kSpSmall; b++) {
            m.pc[a][b] = in.pc[a][b];
            m.B2[a][b] = in.B2[a][b];
            m.dl[a][b] = in.delta[a][b];
        }
    }
    return m;
}

// f(model tag, kernel argument): the model form with static sizes where it applies
template <typename F>
hipError_t by_model(const SpArgs &a, F &&f) {
    const SpModel &m = *a.m_host;
    if(!is_small(m)) return f(LargeModel{}, a.m);
    const SpSmallModel sm = small_model(m);
    if(m.model == CH_SALEH_WERTHEIM) return f(SalehModel{}, sm);
    if(m.model == CH_RICCI_WERTHEIM) return f(RicciModel{}, sm);
    switch(m.P) {
    case 1: return f(SmallModel<1>{}, sm);
    case 2: return f(SmallModel<2>{}, sm);
    case 3: return f(SmallModel<3>{}, sm);
    default: return f(SmallModel<4>{}, sm);
    }
}

}  // namespace

void sp_build_model(const ch_species_model &in, SpModel &m) {
    m = SpModel{};
    m.model = in.model;
    m.S = in.n_species;
    for(int s = 0; s < kSpMaxSpecies; s++) m.k[s] = in.k[s];
    for(int i = 0; i < 3; i++) m.val[i] = in.saleh_valence[i];
    m.lh = in.saleh_valence[2] / 2;
    m.sB2 = in.saleh_B2;
    m.sB3 = in.saleh_B3;
    m.dAA = in.saleh_delta_AA;
    m.dBB = in.saleh_delta_BB;
    m.rB2 = in.ricci_B2;
    m.d00 = in.ricci_delta_00;
    m.d12 = in.ricci_delta_12;
    m.P = in.model == CH_GENERIC_WERTHEIM ? in.n_patches : 0;
    for(int s = 0; s < kSpMaxSpecies; s++)
        for(int q = 0; q < kSpMaxPatches; q++) m.pc[s][q] = in.model == CH_GENERIC_WERTHEIM ? in.patch_count[s][q] : 0;
    for(int s = 0; s < kSpMaxSpecies; s++)
        for(int t = 0; t < kSpMaxSpecies; t++) m.B2[s][t] = in.B2[s][t];
    if(in.model != CH_GENERIC_WERTHEIM) return;
    // GenericWertheim.cpp:123-149: unique patch types ascending; per type the
    // terms over species in order and their patch types ascending
    int used[kSpMaxPatches] = {0};
    for(int s = 0; s < m.S; s++)
        for(int q = 0; q < m.P; q++)
            if(m.pc[s][q] > 0) used[q] = 1;
    for(int q = 0; q < m.P; q++)
        for(int o = 0; o < m.P; o++) m.delta[q][o] = used[q] && used[o] && in.delta[q][o] > 0.0 ? in.delta[q][o] : 0.0;
    int nt = 0;
    for(int q = 0; q < m.P; q++) {
        if(!used[q]) continue;
        const int u = m.n_unique++;
        m.unique[u] = q;
        m.term_start[u] = nt;
        for(int s = 0; s < m.S; s++)
            for(int o = 0; o < m.P; o++)
                if(m.pc[s][o] > 0 && in.delta[q][o] > 0.0) {
                    m.t_species[nt] = s;
                    m.t_other[nt] = o;
                    m.t_coeff[nt] = (double)m.pc[s][o] * in.delta[q][o];
                    nt++;
                }
    }
    m.term_start[m.n_unique] = nt;
}

hipError_t sp_warm(const SpArgs &a, hipStream_t s) {
    if(a.m_host->model != CH_GENERIC_WERTHEIM) return hipSuccess;
    return by_precision<1>(a.precision, [&](auto tag) {
        using T = decltype(tag);
        return by_model(a, [&](auto md, const auto &arg) {
            hipLaunchKernelGGL((k_sp_warm<T, decltype(md)>), dim3(grid_for(a.bins)), dim3(256), 0, s, (const T *)a.rho,
                               a.X, arg, a.bins);
            return hipGetLastError();
        });
    });
}

hipError_t sp_step_stencil(const SpArgs &a, int integrator, hipStream_t s) {
    return by_precision<1>(a.precision, [&](auto tag) -> hipError_t {
        using T = decltype(tag);
        const int g = grid_for(a.bins);
        const int mob = integrator == CH_EULER_MOBILITY ? a.mob_rule : -1;
        auto go = [&](auto dims_tag) -> hipError_t {
            constexpr int D = decltype(dims_tag)::value;
            hipError_t e = by_model(a, [&](auto md, const auto &arg) {
                hipLaunchKernelGGL((k_sp_mu<T, D, decltype(md)>), dim3(g), dim3(256), 0, s, (const T *)a.rho, a.X,
                                   (T *)a.mu, (T *)a.mob, a.p, arg, a.bins, mob);
                return hipGetLastError();
            });
            if(e != hipSuccess) return e;
            if(integrator == CH_EULER_MOBILITY)
                hipLaunchKernelGGL((k_sp_update<T, D, true>), dim3(g, a.m_host->S), dim3(256), 0, s, (T *)a.rho,
                                   (const T *)a.mu, (const T *)a.mob, a.p, a.bins);
            else
                hipLaunchKernelGGL((k_sp_update<T, D, false>), dim3(g, a.m_host->S), dim3(256), 0, s, (T *)a.rho,
                                   (const T *)a.mu, (const T *)a.mob, a.p, a.bins);
            return hipGetLastError();
        };
        if(a.p.dims == 1) return go(std::integral_constant<int, 1>{});
        if(a.p.dims == 2) return go(std::integral_constant<int, 2>{});
        return go(std::integral_constant<int, 3>{});
    });
}

hipError_t sp_step_spectral(const SpArgs &a, const SpectralArgs &sa, hipStream_t s) {
    return by_precision<1>(a.precision, [&](auto tag) -> hipError_t {
        using T = decltype(tag);
        const int S = a.m_host->S;
        hipError_t e = by_model(a, [&](auto md, const auto &arg) {
            hipLaunchKernelGGL((k_sp_fprime<T, decltype(md)>), dim3(grid_for(a.bins)), dim3(256), 0, s,
                               (const T *)a.rho, a.X, (T *)a.mu, arg, a.bins);
            return hipGetLastError();
        });
        for(int sp = 0; sp < S && e == hipSuccess; sp++) {
            SpectralArgs b = sa;
            b.rho = (T *)a.rho + sp * a.bins;
            C2<T> *rh = (C2<T> *)a.rho_hat + sp * a.hat;
            if(a.p.dims == 2 && a.p.N <= 2048) {
                e = spec_x_forward(b, (const T *)a.mu + sp * a.bins, a.spec[0], false, s);
                if(e == hipSuccess)
                    e = sp_ps_col<T>(b, (const C2<T> *)a.spec[0], (C2<T> *)a.spec[1], rh, a.m_host->k[sp], s);
                if(e == hipSuccess) e = spec_x_inverse(b, a.spec[1], (T *)a.rho + sp * a.bins, s);
                continue;
            }
            e = spec_r2c(b, (const T *)a.mu + sp * a.bins, a.spec[0], false, s);
            if(e != hipSuccess) break;
            hipLaunchKernelGGL((k_sp_ps_update<T>), dim3(grid_for(a.hat)), dim3(256), 0, s, rh, (C2<T> *)a.spec[0],
                               (C2<T> *)a.spec[1], a.p, a.hat, a.m_host->k[sp]);
            e = hipGetLastError();
            if(e == hipSuccess) e = spec_c2r(b, a.spec[1], (T *)a.rho + sp * a.bins, s);
        }
        return e;
    });
}

hipError_t sp_init_spectral(const SpArgs &a, const SpectralArgs &sa, hipStream_t s) {
    return by_precision<1>(a.precision, [&](auto tag) -> hipError_t {
        using T = decltype(tag);
        hipError_t e = hipSuccess;
        for(int sp = 0; sp < a.m_host->S && e == hipSuccess; sp++)
            e = spec_r2c(sa, (const T *)a.rho + sp * a.bins, (C2<T> *)a.rho_hat + sp * a.hat, false, s);
        return e;
    });
}

hipError_t sp_mobility_field(const SpArgs &a, double *out, hipStream_t s) {
    return by_precision<1>(a.precision, [&](auto tag) {
        using T = decltype(tag);
        hipLaunchKernelGGL((k_sp_mob<T>), dim3(grid_for(a.bins)), dim3(256), 0, s, (const T *)a.rho, a.X, out, a.p, a.m,
                           a.bins, a.mob_rule);
        return hipGetLastError();
    });
}

hipError_t sp_observables(const SpArgs &a, double *partials, int nparts, double *result, hipStream_t s, double *ring,
                          unsigned *count) {
    return by_precision<1>(a.precision, [&](auto tag) -> hipError_t {
        using T = decltype(tag);
        const int nb = (int)std::min<int64_t>(nparts, (a.bins + 255) / 256);
        auto go = [&](auto dims_tag) {
            constexpr int D = decltype(dims_tag)::value;
            hipLaunchKernelGGL((k_sp_observables<T, D>), dim3(nb), dim3(256), 0, s, (const T *)a.rho, a.p, a.m, a.bins,
                               partials);
            return hipGetLastError();
        };
        hipError_t e = a.p.dims == 1 ? go(std::integral_constant<int, 1>{})
                                     : (a.p.dims == 2 ? go(std::integral_constant<int, 2>{})
                                                      : go(std::integral_constant<int, 3>{}));
        if(e != hipSuccess) return e;
        return ring ? finalize_pairs_ring(partials, nb, ring, count, s) : finalize_pairs(partials, nb, result, s);
    });
}

}  // namespace chd
