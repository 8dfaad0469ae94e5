// stencil_march.hip -- the 3D euler / euler_mobility step in one launch, marching
// along z (Params::tile3d 4 and 5).
//
// A block owns TX x TY columns of ZC cells, one thread per column of the region
// with its 2-cell ring.  A thread loads its ZC + 4 values of psi at once, so the
// block waits for memory once; then plane by plane the in-plane neighbours of
// psi and of mu (and M) go through LDS, two buffers each and one barrier per
// plane (mu of plane j and the update of plane j - 1 share a phase), while the
// z neighbours stay in registers.  psi is read and written once, where the
// two-launch step (stencil_split.hip) moves 40 to 56 B per cell at some 4 TB/s,
// and mu is evaluated on (TX + 2)(TY + 2)(ZC + 2) cells per TX TY ZC, 1.5 times
// the cells, where the LDS tile (stencil.h) evaluates 1.76 times and spends its
// time on the index divisions of its loops.  The per-cell arithmetic is
// ch_device.h's: the same bits as both.
//
// us per step on MI355X against the LDS tile (Landau, free-energy mobility) or
// the two-launch step (the other SimpleWertheim systems):
//                                   N = 32     N = 64     N = 128      N = 256
//   Landau euler        FP32   2.8 / 4.8  3.5 / 4.6  8.2 / 13.1  41.8 / 82.4
//                       FP64   3.1 / 5.4  4.0 / 5.3 11.5 / 17.5  62.9 / 118
//   Wertheim, linear M  FP64   4.7 / 7.4  6.6 / 8.5 21.8 / 28.1   126 / 282
//            constant M FP64   4.4 / 6.1  6.1 / 7.0 19.0 / 20.9   107 / 179
//                       FP32   4.0 / 4.8  5.3 / 5.1 14.9 / 13.5   103 / 90
//            free-energy M FP64 4.9 / 7.3 6.9 / 7.3 22.3 / 31.9   128 / 215
// and in FP32, march, LDS tile, two launches (measured side by side):
//   Wertheim, linear M         4.4, 6.6, 6.0   5.8, 6.4, 6.2   15.7, 21.7, 15.6   93.8, 142, 98.7
//            regularised M     4.5, 6.6, 6.0   6.0, 6.4, 6.2   16.3, 22.2, 15.6   98.5, 150, 101
//            free-energy M     4.7, 6.8, 9.9   6.1, 6.7, 9.4   16.6, 23.2, 24.2   101, 160, 169
//            constant M        4.3, 6.2, 5.1   5.5, 6.1, 5.4   15.1, 20.2, 13.4   91.5, 136, 80.3
// FP32 SimpleWertheim with constant mobility moves half the bytes for the same
// FP64 f', so there the launch that evaluates f' once per cell stays ahead from
// N = 64 (march3d_better); with the other rules the march is ahead or level but
// for the regularised one at N = 128 (six runs in both orders).  Chunks of 8 planes
// from N = 128 (16: 8.9 us for Landau FP32, fewer blocks than the CUs hold), 32 x 8 x 4
// at N = 64 and 32 x 8 x 2 at N = 32, where smaller blocks fill more CUs.
#include "adjoint_math.h"
#include "ch_internal.h"

namespace chd {

// cell s of the perimeter of the W x H box whose corner is (o, o)
template <int W, int H>
__device__ __forceinline__ void perimeter(int s, int o, int &lx, int &ly) {
    if(s < 2 * W) {
        lx = o + s % W;
        ly = o + (s < W ? 0 : H - 1);
    }
    else {
        const int r = s - 2 * W;
        lx = o + (r < H - 2 ? 0 : W - 1);
        ly = o + 1 + (r < H - 2 ? r : r - (H - 2));
    }
}

// REC: mu of the old state goes to mu_out, for the reverse step
template <typename T, int MODEL, int MOB, bool EM, int TX, int TY, int ZC, int NT, bool REC>
__global__ __launch_bounds__(NT) void k_march3d(const T *__restrict__ in, T *__restrict__ out, Params p, int tiles_x,
                                                int tiles_y, T *__restrict__ mu_out) {
    constexpr int RX = TX + 4, RY = TY + 4, R = RX * RY;
    constexpr int NI = TX * TY, NU = (TX + 2) * (TY + 2);  // updated cells, mu cells of a plane
    static_assert(R <= NT && NI % 64 == 0, "one thread per cell of the plane, whole waves of updated cells");
    constexpr bool VARM = EM && MOB != CH_MOB_CONSTANT;
    __shared__ T P[2][R + 1], U[2][R + 1], V[VARM ? 2 : 1][VARM ? R + 1 : 1];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, tz = tile / (tiles_x * tiles_y);
    const int lg = p.log2N, mask = p.mask;
    const int s = threadIdx.x;
    // Wertheim: the threads of the updated cells first, then the ring of mu
    // cells, then the ring that only carries psi, so that whole waves skip the
    // FP64 f' (10 of 12 evaluate it); Landau's f' costs less than the scattered
    // ring loads, its threads follow the rows
    constexpr bool PACK = MODEL == CH_SIMPLE_WERTHEIM;
    int lx, ly;
    if(!PACK) {
        lx = s % RX;
        ly = s < R ? s / RX : 0;
    }
    else if(s < NI) {
        lx = 2 + s % TX;
        ly = 2 + s / TX;
    }
    else if(s < NU) perimeter<TX + 2, TY + 2>(s - NI, 1, lx, ly);
    else perimeter<RX, RY>(s < R ? s - NU : 0, 0, lx, ly);
    const int w0 = __builtin_amdgcn_readfirstlane(s & ~63);  // first thread of the wave
    const bool wave_mu = !PACK || w0 < NU;
    const bool upd = PACK ? w0 < NI : lx >= 2 && lx < TX + 2 && ly >= 2 && ly < TY + 2;
    const int t = s < R ? ly * RX + lx : R;  // the cell's place in the plane (R: none)
    // as a centre with its neighbours in range
    const int tc = (PACK ? s < NU : lx >= 1 && lx < RX - 1 && ly >= 1 && ly < RY - 1) ? t : RX + 1;
    const uint32_t x = (uint32_t)(tx * TX + lx - 2) & mask, y = (uint32_t)(ty * TY + ly - 2) & mask;
    const uint32_t at = ((y << lg) + x) * (uint32_t)sizeof(T);  // byte offset in a plane
    const int z0 = tz * ZC - 2;
    auto plane = [&](int j) { return (size_t)((z0 + j) & mask) << (2 * lg); };
    T psi[ZC + 4];
#pragma unroll
    for(int j = 0; j < ZC + 4; j++)
        psi[j] = *reinterpret_cast<const T *>(reinterpret_cast<const char *>(in + plane(j)) + at);
    T um = 0, uc = 0, mc = 0, mm = 0;
    const T Mc = (T)p.M;
    P[1][t] = psi[1];
    lds_barrier();
#pragma unroll
    for(int j = 1; j < ZC + 3; j++) {
        const T *Pj = P[j & 1], *Uj = U[(j - 1) & 1], *Vj = V[VARM ? (j - 1) & 1 : 0];
        T mu = 0, mob = 0;
        if(wave_mu) {
            const T m[3] = {Pj[tc - 1], Pj[tc - RX], psi[j - 1]}, q[3] = {Pj[tc + 1], Pj[tc + RX], psi[j + 1]};
            mu = chem_pot<T, 3, MODEL>(p, psi[j], m, q);
            U[j & 1][t] = mu;
            if constexpr(VARM) {
                mob = mobility<T, MOB>(p, psi[j]);
                V[j & 1][t] = mob;
            }
        }
        if(j < ZC + 2) P[(j + 1) & 1][t] = psi[j + 1];
        if(REC && j >= 2 && j < ZC + 2 && upd)
            *reinterpret_cast<T *>(reinterpret_cast<char *>(mu_out + plane(j)) + at) = mu;
        if(j >= 3 && upd) {
            const T Um[3] = {Uj[t - 1], Uj[t - RX], um}, Uq[3] = {Uj[t + 1], Uj[t + RX], mu};
            T r;
            if constexpr(!EM) {
                r = euler_update<T, 3>(p, psi[j - 1], uc, Um, Uq);
            }
            else if constexpr(!VARM) {
                const T Mm[3] = {Mc, Mc, Mc}, Mq[3] = {Mc, Mc, Mc};
                r = mobility_update<T, 3>(p, psi[j - 1], uc, Um, Uq, Mc, Mm, Mq);
            }
            else {
                const T Mm[3] = {Vj[t - 1], Vj[t - RX], mm}, Mq[3] = {Vj[t + 1], Vj[t + RX], mob};
                r = mobility_update<T, 3>(p, psi[j - 1], uc, Um, Uq, mc, Mm, Mq);
            }
            *reinterpret_cast<T *>(reinterpret_cast<char *>(out + plane(j - 1)) + at) = r;
        }
        if(j < ZC + 2) lds_barrier();
        um = uc;
        uc = mu;
        mm = mc;
        mc = mob;
    }
}

template <typename T, int MODEL, int MOB, bool EM, int TX, int TY, int ZC, int NT, bool REC>
static hipError_t march_cfg(const Params &p, const T *in, T *out, T *mu, hipStream_t s) {
    const int tiles_x = p.N / TX, tiles_y = p.N / TY;
    hipLaunchKernelGGL((k_march3d<T, MODEL, MOB, EM, TX, TY, ZC, NT, REC>), dim3(tiles_x * tiles_y * (p.N / ZC)),
                       dim3(NT), 0, s, in, out, p, tiles_x, tiles_y, mu);
    return hipGetLastError();
}

template <typename T, int MODEL, int MOB, bool EM, bool REC = false>
static hipError_t march_t(const Params &p, const void *in, void *out, hipStream_t s,
                          void *mu = nullptr) {
    const T *a = (const T *)in;
    T *b = (T *)out, *u = (T *)mu;
    if(p.N >= 128) return march_cfg<T, MODEL, MOB, EM, 32, 16, 8, 768, REC>(p, a, b, u, s);
    if(p.N >= 64) return march_cfg<T, MODEL, MOB, EM, 32, 8, 4, 448, REC>(p, a, b, u, s);
    return march_cfg<T, MODEL, MOB, EM, 32, 8, 2, 448, REC>(p, a, b, u, s);
}

template <typename T, int MODEL>
static hipError_t march_model(const Params &p, int integrator, int mob, const void *in, void *out, hipStream_t s) {
    if(integrator == CH_EULER) return march_t<T, MODEL, CH_MOB_CONSTANT, false>(p, in, out, s);
    switch(mob) {
    case CH_MOB_CONSTANT: return march_t<T, MODEL, CH_MOB_CONSTANT, true>(p, in, out, s);
    case CH_MOB_REGULARISED: return march_t<T, MODEL, CH_MOB_REGULARISED, true>(p, in, out, s);
    case CH_MOB_LINEAR: return march_t<T, MODEL, CH_MOB_LINEAR, true>(p, in, out, s);
    case CH_MOB_FREE_ENERGY:
        if constexpr(MODEL == CH_SIMPLE_WERTHEIM) return march_t<T, MODEL, CH_MOB_FREE_ENERGY, true>(p, in, out, s);
    }
    return hipErrorInvalidValue;
}

// ---- the euler_mobility reverse step in one launch, marching the same way:
// nu = D(Mob, lambda) of plane j on the region and its first ring, eta and the
// Laplacian of psi of plane j, and lambda_n of plane j - 1 share a phase.  lambda,
// psi and mu are read once and lambda_n written, the mobilities evaluated again from
// psi (the same function: the same bits; 3 to 14 operations against a third field on
// the tape, N = 128 linear M 54 -> 47 us), where the two-launch form (k_adj_split_nu,
// k_adj_split_upd in stencil_split.hip) also reads the mobilities, writes nu and
// reads lambda and nu again; the cells' arithmetic is the same (adjoint_math.h), so
// lambda has the same bits, and only the order of the FP64 gradient sums differs.
// us per reverse step on MI355X, two launches -> this (linear M; constant M):
//   FP64  N = 32 16.0 -> 6.9; 8.9 -> 6.1   N = 64 12.8 -> 9.8; 11.6 -> 8.8   N = 128 52.6 -> 47.3; 46.2 -> 39.2
//   FP32  N = 32  7.7 -> 5.8; 6.9 -> 5.7   N = 64  8.6 -> 8.7;  8.2 -> 7.9   N = 128 25.7 -> 27.1; 21.7 -> 24.1
// and the recorded step, FP64 linear M, 8.0 -> 5.1, 8.9 -> 7.2, 29.4 -> 24.3.  In FP32 the
// two launches' bytes halve and the FP64 derivatives do not, so from N = 128 on
// they stay (march3d_reverse_better; FP32 record + sweep, us per step, two launches -> this:
// N = 64 linear M 31.5 -> 29.7, constant M 30.8 -> 28.7, N = 128 133 -> 134).  Bound by the FP64 cells and, with one
// block per CU, by the wait for its first loads.  Blocks as the forward's: at N =
// 64 FP64 linear M 32 x 8 x 4 9.7, x 2 10.6, x 8 12.5, 32 x 16 x 4 12.2, 64 x 4 x 8 12.8;
// at N = 128 (linear; constant) 32 x 16 x 8 46; 39, x 4 47; 44, 32 x 8 x 8 51; 38, x 16 40; 43.
template <typename T, int MODEL, int MOB, int TX, int TY, int ZC, int NT>
__global__ __launch_bounds__(NT) void k_adj_march3d(const T *__restrict__ lam, const T *__restrict__ psi,
                                                    const T *__restrict__ mu, T *__restrict__ lam_out, Params p,
                                                    int tiles_x, int tiles_y, double *__restrict__ gacc) {
    constexpr int RX = TX + 4, RY = TY + 4, R = RX * RY;
    constexpr int NI = TX * TY, NU = (TX + 2) * (TY + 2);  // updated cells, nu cells of a plane
    static_assert(R <= NT && NI % 64 == 0, "one thread per cell of the plane, whole waves of updated cells");
    constexpr bool VARM = MOB != CH_MOB_CONSTANT;
    __shared__ T L[2][R + 1], M[VARM ? 2 : 1][VARM ? R + 1 : 1], U[2][R + 1], S[2][R + 1], V[2][R + 1];
    __shared__ double red[kGradSlots][NT / 64];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tx = tile % tiles_x, ty = (tile / tiles_x) % tiles_y, tz = tile / (tiles_x * tiles_y);
    const int lg = p.log2N, mask = p.mask;
    const int s = threadIdx.x;
    int lx, ly;  // updated cells first, then the ring of nu cells, then the outer ring
    if(s < NI) {
        lx = 2 + s % TX;
        ly = 2 + s / TX;
    }
    else if(s < NU) perimeter<TX + 2, TY + 2>(s - NI, 1, lx, ly);
    else perimeter<RX, RY>(s < R ? s - NU : 0, 0, lx, ly);
    const int w0 = __builtin_amdgcn_readfirstlane(s & ~63);
    const bool wave_nu = w0 < NU, upd = w0 < NI;
    const int t = s < R ? ly * RX + lx : R;
    const int tc = s < NU ? t : RX + 1;
    const uint32_t x = (uint32_t)(tx * TX + lx - 2) & mask, y = (uint32_t)(ty * TY + ly - 2) & mask;
    const uint32_t at = ((y << lg) + x) * (uint32_t)sizeof(T);
    const int z0 = tz * ZC - 2;
    auto plane = [&](int j) { return (size_t)((z0 + j) & mask) << (2 * lg); };
    auto load = [&](const T *f, int j) {
        return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(f + plane(j)) + at);
    };
    const T inv_dx2 = (T)p.inv_dx2, Mc = (T)p.M;
    T l[ZC + 4], u[ZC + 4], c[ZC + 4];
#pragma unroll
    for(int j = 0; j < ZC + 4; j++) {
        l[j] = load(lam, j);
        if(VARM || (j > 0 && j < ZC + 3)) c[j] = load(psi, j);
    }
    if(wave_nu) {
#pragma unroll
        for(int j = 1; j < ZC + 3; j++) u[j] = load(mu, j);
    }
    T num = 0, nuc = 0, etac = 0, lpsc = 0;
    double ge = 0, gk = 0, gm = 0, gd = 0;
    L[1][t] = l[1];
    T mm = Mc, mc = Mc;  // mobilities of planes j - 1 and j
    if constexpr(VARM) {
        mm = mobility<T, MOB>(p, c[0]);
        mc = mobility<T, MOB>(p, c[1]);
        M[1][t] = mc;
    }
    lds_barrier();
#pragma unroll
    for(int j = 1; j < ZC + 3; j++) {
        const T *Lj = L[j & 1], *Mj = M[VARM ? j & 1 : 0], *Uj = U[j & 1], *Sj = S[j & 1], *Vp = V[(j - 1) & 1];
        T nu = 0, eta = 0, lps = 0, mq = Mc;
        if constexpr(VARM) mq = mobility<T, MOB>(p, c[j + 1]);
        if(wave_nu) {
            const T lm[3] = {Lj[tc - 1], Lj[tc - RX], l[j - 1]}, lq[3] = {Lj[tc + 1], Lj[tc + RX], l[j + 1]};
            T Mm[3] = {Mc, Mc, Mc}, Mq[3] = {Mc, Mc, Mc};
            if constexpr(VARM) {
                Mm[0] = Mj[tc - 1], Mm[1] = Mj[tc - RX], Mm[2] = mm;
                Mq[0] = Mj[tc + 1], Mq[1] = Mj[tc + RX], Mq[2] = mq;
            }
            nu = adj_nu<T, 3>(l[j], mc, lm, lq, Mm, Mq, inv_dx2);
            V[j & 1][t] = nu;
            if(upd && j >= 2 && j < ZC + 2) {
                const T um[3] = {Uj[t - 1], Uj[t - RX], u[j - 1]}, uq[3] = {Uj[t + 1], Uj[t + RX], u[j + 1]};
                const T cm[3] = {Sj[t - 1], Sj[t - RX], c[j - 1]}, cq[3] = {Sj[t + 1], Sj[t + RX], c[j + 1]};
                eta = adj_eta<T, 3>(u[j], l[j], um, uq, lm, lq, inv_dx2);
                lps = laplacian<T, 3>(c[j], cm, cq, inv_dx2);
            }
            if(j < ZC + 1) {
                U[(j + 1) & 1][t] = u[j + 1];
                S[(j + 1) & 1][t] = c[j + 1];
            }
        }
        if(j < ZC + 2) {
            L[(j + 1) & 1][t] = l[j + 1];
            if constexpr(VARM) M[(j + 1) & 1][t] = mq;
        }
        if(j >= 3 && upd) {
            const T nm[3] = {Vp[t - 1], Vp[t - RX], num}, nq[3] = {Vp[t + 1], Vp[t + RX], nu};
            const T lnu = laplacian<T, 3>(nuc, nm, nq, inv_dx2);
            const double ps = (double)c[j - 1];
            const MobDeriv<MOB> md = mob_deriv<MOB>(p, ps);
            *reinterpret_cast<T *>(reinterpret_cast<char *>(lam_out + plane(j - 1)) + at) =
                adj_em_step<T>(p, l[j - 1], (T)fsecond<MODEL>(p, ps), nuc, lnu, (T)md.drho, etac);
            ge += (double)nuc * ps;
            gk += (double)nuc * (double)lpsc;
            gm += (double)etac * md.hat;
            if constexpr(MODEL == CH_SIMPLE_WERTHEIM)
                gd += (double)nuc * dfprime_ddelta<MODEL>(p, ps) + (double)etac * md.ddelta;
        }
        if(j < ZC + 2) lds_barrier();
        mm = mc;
        mc = mq;
        num = nuc;
        nuc = nu;
        etac = eta;
        lpsc = lps;
    }
    const double gs[kGradSlots] = {ge, gk, gm, gd};
    block_accumulate<NT>(gs, red, gacc + kGradSlots * blockIdx.x);
}

template <typename T, int MODEL, int MOB, int TX, int TY, int ZC, int NT>
static hipError_t adj_march_cfg(const Params &p, const void *const f[3], void *lam_out, double *gacc, hipStream_t s) {
    const int tiles_x = p.N / TX, tiles_y = p.N / TY;
    hipLaunchKernelGGL((k_adj_march3d<T, MODEL, MOB, TX, TY, ZC, NT>), dim3(tiles_x * tiles_y * (p.N / ZC)), dim3(NT), 0,
                       s, (const T *)f[0], (const T *)f[1], (const T *)f[2], (T *)lam_out, p, tiles_x, tiles_y, gacc);
    return hipGetLastError();
}

template <typename T, int MOB>
static hipError_t adj_march_t(const Params &p, const void *const f[3], void *lam_out, double *gacc, hipStream_t s) {
    constexpr int MODEL = CH_SIMPLE_WERTHEIM;
    if(p.N >= 128) return adj_march_cfg<T, MODEL, MOB, 32, 16, 8, 768>(p, f, lam_out, gacc, s);
    if(p.N >= 64) return adj_march_cfg<T, MODEL, MOB, 32, 8, 4, 448>(p, f, lam_out, gacc, s);
    return adj_march_cfg<T, MODEL, MOB, 32, 8, 2, 448>(p, f, lam_out, gacc, s);
}

// one recorded step of a system that adj_march3d sweeps back: psi_{t+1} and mu_t
hipError_t march3d_record(const Params &p, int precision, int mob, const void *in, void *out, void *mu,
                          hipStream_t s) {
    auto go = [&](auto mt) {
        constexpr int MOB = decltype(mt)::value;
        return precision == CH_FP64 ? march_t<double, CH_SIMPLE_WERTHEIM, MOB, true, true>(p, in, out, s, mu)
                                    : march_t<float, CH_SIMPLE_WERTHEIM, MOB, true, true>(p, in, out, s, mu);
    };
    switch(mob) {
    case CH_MOB_CONSTANT: return go(std::integral_constant<int, CH_MOB_CONSTANT>{});
    case CH_MOB_REGULARISED: return go(std::integral_constant<int, CH_MOB_REGULARISED>{});
    case CH_MOB_LINEAR: return go(std::integral_constant<int, CH_MOB_LINEAR>{});
    }
    return hipErrorInvalidValue;
}

// the reverse step: `slot` as march3d_record leaves it, {psi, mu}
hipError_t adj_march3d(const Params &p, int precision, int mob, const void *lam_in, void *lam_out,
                       const void *const slot[2], double *gacc, hipStream_t s) {
    const void *const f[3] = {lam_in, slot[0], slot[1]};
    auto go = [&](auto mt) {
        constexpr int MOB = decltype(mt)::value;
        return precision == CH_FP64 ? adj_march_t<double, MOB>(p, f, lam_out, gacc, s)
                                    : adj_march_t<float, MOB>(p, f, lam_out, gacc, s);
    };
    switch(mob) {
    case CH_MOB_CONSTANT: return go(std::integral_constant<int, CH_MOB_CONSTANT>{});
    case CH_MOB_REGULARISED: return go(std::integral_constant<int, CH_MOB_REGULARISED>{});
    case CH_MOB_LINEAR: return go(std::integral_constant<int, CH_MOB_LINEAR>{});
    }
    return hipErrorInvalidValue;
}

bool march3d_better(const Params &p, int precision, int integrator, int model, int mob) {
    if(p.N < 32) return false;
    const bool constant = integrator == CH_EULER || mob == CH_MOB_CONSTANT;
    return !(precision == CH_FP32 && model == CH_SIMPLE_WERTHEIM && constant && p.N >= 64);
}

bool march3d_reverse_better(const Params &p, int precision) { return precision == CH_FP64 || p.N < 128; }

hipError_t stencil_march3d(const Params &p, int precision, int integrator, int model, int mob, const void *in,
                           void *out, hipStream_t s) {
    if(precision == CH_FP64) {
        if(model == CH_LANDAU) return march_model<double, CH_LANDAU>(p, integrator, mob, in, out, s);
        return march_model<double, CH_SIMPLE_WERTHEIM>(p, integrator, mob, in, out, s);
    }
    if(model == CH_LANDAU) return march_model<float, CH_LANDAU>(p, integrator, mob, in, out, s);
    return march_model<float, CH_SIMPLE_WERTHEIM>(p, integrator, mob, in, out, s);
}

}  // namespace chd
