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
//   Wertheim, linear M  FP64   4.4 / 7.2  6.3 / 8.2 20.6 / 27.7   145 / 284
//            constant M FP64   4.2 / 5.9  5.9 / 6.8 17.9 / 20.4   119 / 188
//                       FP32   4.0 / 4.8  5.3 / 5.1 14.9 / 13.5   103 / 90
//            free-energy M FP64 4.9 / 7.1 6.8 / 7.1 21.3 / 30.5   153 / 248
// FP32 SimpleWertheim with constant mobility moves half the bytes for the same
// FP64 f', so there the launch that evaluates f' once per cell stays ahead from
// N = 64 (march3d_better).  Chunks of 8 planes from N = 128 (16: 8.9 us for
// Landau FP32, fewer blocks than the CUs hold), 32 x 8 x 4 at N = 64 and 32 x 8
// x 2 at N = 32, where smaller blocks fill more CUs.
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

template <typename T, int MODEL, int MOB, bool EM, int TX, int TY, int ZC, int NT>
__global__ __launch_bounds__(NT) void k_march3d(const T *__restrict__ in, T *__restrict__ out, Params p, int tiles_x,
                                                int tiles_y) {
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

template <typename T, int MODEL, int MOB, bool EM, int TX, int TY, int ZC, int NT>
static hipError_t march_cfg(const Params &p, const T *in, T *out, hipStream_t s) {
    const int tiles_x = p.N / TX, tiles_y = p.N / TY;
    hipLaunchKernelGGL((k_march3d<T, MODEL, MOB, EM, TX, TY, ZC, NT>), dim3(tiles_x * tiles_y * (p.N / ZC)), dim3(NT), 0,
                       s, in, out, p, tiles_x, tiles_y);
    return hipGetLastError();
}

template <typename T, int MODEL, int MOB, bool EM>
static hipError_t march_t(const Params &p, const void *in, void *out, hipStream_t s) {
    const T *a = (const T *)in;
    T *b = (T *)out;
    if(p.N >= 128) return march_cfg<T, MODEL, MOB, EM, 32, 16, 8, 768>(p, a, b, s);
    if(p.N >= 64) return march_cfg<T, MODEL, MOB, EM, 32, 8, 4, 448>(p, a, b, s);
    return march_cfg<T, MODEL, MOB, EM, 32, 8, 2, 448>(p, a, b, s);
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

bool march3d_better(const Params &p, int precision, int integrator, int model, int mob) {
    if(p.N < 32) return false;
    const bool constant = integrator == CH_EULER || mob == CH_MOB_CONSTANT;
    return !(precision == CH_FP32 && model == CH_SIMPLE_WERTHEIM && constant && p.N >= 64);
}

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
