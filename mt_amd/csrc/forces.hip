// forces.hip -- streamed-mode kernels: one thread per bead, bead state in
// HBM (float4 SoA, double-buffered), neighbour lists k-major so that a
// wavefront's list loads coalesce.
#include "bead_physics.h"
#include "engine_internal.h"

namespace mte {

// Workgroup size of k_frames; the per-step bead kernels take theirs from the
// engine's tuning (64, 128 or 256).
constexpr int STREAM_BLOCK = 256;

constexpr int FORCE_TILE = 256;   // k_forces_lds: beads per workgroup (the 256-bead tiles of e->tiles)

struct GlobalAcc {
    DevState S;
    const DevTopo &T;
    __device__ __forceinline__ int mon(int j) const { return T.mon_type[j]; }
    __device__ __forceinline__ bool gtp1(int j) const { return T.gtp[j] == 1; }
    __device__ __forceinline__ bool offtub(int j) const { return T.on_tub[j] == 0; }
    __device__ __forceinline__ float4 xyz(int j) const { return S.xyz[j]; }
    __device__ __forceinline__ float4 ang(int j) const { return S.ang[j]; }
    __device__ __forceinline__ float4 fn(int j) const { return S.fn[j]; }
    __device__ __forceinline__ float4 fp1(int j) const { return S.fp1[j]; }
    __device__ __forceinline__ float4 fp2(int j) const { return S.fp2[j]; }
    // as bead_force reads them: the handle is the bead's index
    static constexpr int SCALE = 1;
    __device__ __forceinline__ float4 lat(int j, bool p2nd) const { return (p2nd ? S.fp2 : S.fp1)[j]; }
    __device__ __forceinline__ float3 angles(float4, int j) const { return f3(S.ang[j]); }
    __device__ __forceinline__ int flags(float4, int j) const { return T.flags[j]; }
};

__global__ void __launch_bounds__(STREAM_BLOCK) k_frames(DevState S, int nb, LatOffsets L) {
    const int b = blockIdx.x * STREAM_BLOCK + threadIdx.x;
    if (b >= nb) return;
    const float4 a = S.ang[b];
    float4 n, p1, p2;
    frame_vectors(a.x, a.y, a.z, L, n, p1, p2);
    S.fn[b] = n;
    S.fp1[b] = p1;
    S.fp2[b] = p2;
}

// Force + Euler-Maruyama step.  Reads Sin, writes Sout (both positions and
// rotated offsets), advances the HybridTaus states of mobile beads only
// (src/compute_cuda.cu:949-953) unless noise is injected.
// A second thread per bead, in another wave, draws its normals and sums its LJ
// forces beside its bonds; the sums are added in the order of one thread.  A
// bead's work is a chain of dependent waits, and a thread per bead leaves too
// few waves to cover them (blocks of 256: 100 steps of 3982 beads 752 -> 644
// us, of 45436 beads 870 -> 763; 200 steps of 122646 beads 2256 -> 1974).
template <int BS, bool PERIODIC>
__global__ void __launch_bounds__(2 * BS)
    k_step_plain(ForceK K, DevTopo T, DevState Sin, DevState Sout, uint4 *seeds, const float *noise,
                 LatOffsets L) {
    __shared__ float4 xlj[BS], xrx[BS], xra[BS];
    const bool helper = threadIdx.x >= BS;
    const int q = threadIdx.x - (helper ? BS : 0), b = xcd_block() * BS + q;
    const bool valid = b < T.nb;
    const int flags = valid ? T.flags[b] : FL_FIXED;
    const bool mobile = is_mobile(flags);
    float4 x, a;
    float F[6];
    if (mobile) {
        const AheadLists<1> Ls(T, b, 0, 0);
        const GlobalAcc A{Sin, T};
        x = Sin.xyz[b];
        Own I;
        if (helper) {
            I.r = f3(x);
            if (PERIODIC) set_box(I, T.tbox[T.tid[b]]);
            if (!noise) {
                uint4 s = seeds[b];
                xrx[q] = normals4(s);
                seeds[b] = s;
                s = seeds[b + T.nb];
                xra[q] = normals4(s);
                seeds[b + T.nb] = s;
            }
            if (K.lj_on) {
                const float3 lj = lj_sum<PERIODIC>(K, A, Ls, I);
                xlj[q] = make_float4(lj.x, lj.y, lj.z, 0.f);
            }
        } else {
            a = Sin.ang[b];
            I = make_own(x, a, Sin.fn[b], Sin.fp1[b], Sin.fp2[b], flags);
            if (PERIODIC) set_box(I, T.tbox[T.tid[b]]);
            bond_total(bond_forces<PERIODIC>(K, A, Ls, I), I, F);
        }
    }
    __syncthreads();
    if (!valid || helper) return;
    if (!mobile) {
        Sout.xyz[b] = Sin.xyz[b];
        Sout.ang[b] = Sin.ang[b];
        Sout.fn[b] = Sin.fn[b];
        Sout.fp1[b] = Sin.fp1[b];
        Sout.fp2[b] = Sin.fp2[b];
        return;
    }
    add_lj_walls(K, f3(xlj[q]), K.is_wall ? T.zs[T.tid[b]] : 0.f, f3(x), F);
    float4 rx, ra;
    if (noise) {
        const float *nz = noise + 6 * (size_t)b;
        rx = make_float4(nz[0], nz[1], nz[2], 0.f);
        ra = make_float4(nz[3], nz[4], nz[5], 0.f);
    } else {
        rx = xrx[q];
        ra = xra[q];
    }
    em_update(K, F, rx, ra, x, a);
    float4 n, p1, p2;
    frame_vectors(a.x, a.y, a.z, L, n, p1, p2);
    Sout.xyz[b] = x;
    Sout.ang[b] = a;
    Sout.fn[b] = n;
    Sout.fp1[b] = p1;
    Sout.fp2[b] = p2;
}

// Forces (compute_kernel semantics; extra beads get zero), optionally with
// the TEA random forces.
// The helper thread of k_step_plain again (100 MLP-HI steps of 262426 beads 19.43
// -> 19.32 ms; 50 TEA steps of 3982 beads 1613 -> 1542 us).
template <int BS, bool PERIODIC>
__global__ void __launch_bounds__(2 * BS)
    k_forces(ForceK K, DevTopo T, DevState S, float4 *fxyz, float4 *fang, TeaDraw D) {
    __shared__ float4 xlj[BS];
    const bool helper = threadIdx.x >= BS;
    const int q = threadIdx.x - (helper ? BS : 0), b = xcd_block() * BS + q;
    const bool valid = b < T.nb;
    const int flags = valid ? T.flags[b] : FL_EXTRA;
    const bool extra = (flags & FL_EXTRA) != 0;
    float3 r;
    float F[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (!extra) {
        const AheadLists<1> Ls(T, b, 0, 0);
        const GlobalAcc A{S, T};
        const float4 x = S.xyz[b];
        r = f3(x);
        Own I;
        if (helper) {
            I.r = r;
            if (PERIODIC) set_box(I, T.tbox[T.tid[b]]);
            if (D.R) D.R[b] = tea_draw(D, K.vF, b, false);
            if (K.lj_on) {
                const float3 lj = lj_sum<PERIODIC>(K, A, Ls, I);
                xlj[q] = make_float4(lj.x, lj.y, lj.z, 0.f);
            }
        } else {
            I = make_own(x, S.ang[b], S.fn[b], S.fp1[b], S.fp2[b], flags);
            if (PERIODIC) set_box(I, T.tbox[T.tid[b]]);
            bond_total(bond_forces<PERIODIC>(K, A, Ls, I), I, F);
        }
    } else if (valid && helper && D.R) {
        D.R[b] = tea_draw(D, K.vF, b, true);
    }
    __syncthreads();
    if (!valid || helper) return;
    if (!extra) add_lj_walls(K, f3(xlj[q]), K.is_wall ? T.zs[T.tid[b]] : 0.f, r, F);
    fxyz[b] = make_float4(F[0], F[1], F[2], 0.f);
    fang[b] = make_float4(F[3], F[4], F[5], 0.f);
}

// The same forces with the bead's whole trajectory staged in LDS (positions,
// rotated offsets, angles and flags of every bead), one workgroup per
// 256-bead tile of a trajectory: neighbour data are read from LDS instead of
// gathered from L2 per pair.  For trajectories that fit (forces_lds_bytes).
// Bounded by the staging, five times each bead of a 1040-bead trajectory: its
// tiles go to one XCD, whose L2 then serves all but the first (64 tubes: 12.5
// -> 9.6 us with the update kernel's beads and the pair units in the same
// eighths, tea_build_units).
// HELPED: a second thread per bead, in another wave, draws its random force and
// sums its LJ forces beside its bonds (about one wave per SIMD otherwise, each
// bound by its own waits: 64 tubes of 1040 beads 9.3 -> 8.0 us, 100 steps of 1
// and 8 such tubes 1882 -> 1711 and 2354 -> 2192); the sums are added in the
// same order.
template <bool PERIODIC, bool HELPED>
__global__ void __launch_bounds__(HELPED ? 2 * FORCE_TILE : FORCE_TILE)
    k_forces_lds(ForceK K, DevTopo T, DevState S, const int2 *tiles, int ntiles, float4 *fxyz, float4 *fang, TeaDraw D) {
    extern __shared__ float4 lds[];
    const int tile = xcd_block();   // a trajectory's tiles share one L2
    if (tile >= ntiles) return;
    const int2 tl = tiles[tile];
    const int t = tl.x, base = T.tbase[t], n = T.tsize[t];
    float4 *lx = lds, *ln = lds + n, *l1 = ln + n, *l2 = l1 + n;
    const LdsAcc A(lx, ln, l1, l2);
    const bool helper = HELPED && threadIdx.x >= FORCE_TILE;
    const int q = threadIdx.x - (helper ? FORCE_TILE : 0);
    float4 *xlj = l2 + n + q;   // HELPED: the helper's LJ sum
    const int i = tl.y + q, b = base + min(i, n - 1);
    const AheadLists<LdsAcc::SCALE> Ls(T, b, base, A.origin());
    stage_state(T, S, base, n, lx, ln, l1, l2);
    __syncthreads();
    float F[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const float wall_z = K.is_wall ? T.zs[t] : 0.f;
    Own I;
    bool extra = true;
    if (i < n) {
        const float4 x = lx[i];
        const int flags = __float_as_int(x.w);
        extra = (flags & FL_EXTRA) != 0;
        if (helper) {
            I.r = f3(x);
            if (PERIODIC) set_box(I, T.tbox[t]);
            float3 lj = make_float3(0.f, 0.f, 0.f);
            if (!extra && K.lj_on) lj = lj_sum<PERIODIC>(K, A, Ls, I);
            *xlj = make_float4(lj.x, lj.y, lj.z, 0.f);
        } else if (!extra) {
            const float4 fn = ln[i], f1 = l1[i], f2 = l2[i];
            I = make_own(x, make_float4(fn.w, f1.w, f2.w, 0.f), fn, f1, f2, flags);
            if (PERIODIC) set_box(I, T.tbox[t]);
            if (HELPED) bond_total(bond_forces<PERIODIC>(K, A, Ls, I), I, F);
            else bead_force<PERIODIC>(K, A, Ls, wall_z, I, F);
        }
        if (D.R && (!HELPED || helper)) D.R[b] = tea_draw(D, K.vF, b, extra);
    }
    if (HELPED) __syncthreads();
    if (i >= n || helper) return;
    if (HELPED && !extra) add_lj_walls(K, f3(*xlj), wall_z, I.r, F);
    fxyz[b] = make_float4(F[0], F[1], F[2], 0.f);
    fang[b] = make_float4(F[3], F[4], F[5], 0.f);   // fi, theta, psi
}

// Dynamic LDS of k_forces_lds for trajectories of up to nmax beads, without
// the helpers' sums.
size_t forces_lds_bytes(int nmax) { return (size_t)4 * sizeof(float4) * nmax; }

template <int BS>
__global__ void __launch_bounds__(BS)
    k_energies(mte_params P, DevTopo T, DevState S, double *en) {
    const int b = xcd_bead(BS);
    if (b >= T.nb) return;
    float U[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (!T.extra[b]) {
        Own I = make_own(S.xyz[b], S.ang[b], S.fn[b], S.fp1[b], S.fp2[b], 0);
        set_box(I, T.tbox[T.tid[b]]);
        bead_energy(P, T, GlobalAcc{S, T}, b, I, U);
    }
#pragma unroll
    for (int q = 0; q < 7; q++) en[7 * (size_t)b + q] = (double)U[q];
}

// Per-trajectory FP64 sums of the per-bead energies (OutputAllEnergies,
// src/updater.cpp:3-43), one workgroup per trajectory, fixed reduction order.
__global__ void __launch_bounds__(256) k_traj_sum(DevTopo T, const double *en, double *out) {
    __shared__ double red[7][256];
    const int t = blockIdx.x;
    const int base = T.tbase[t], n = T.tsize[t];
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int i = threadIdx.x; i < n; i += 256)
        for (int q = 0; q < 7; q++) acc[q] += en[7 * (size_t)(base + i) + q];
    for (int q = 0; q < 7; q++) red[q][threadIdx.x] = acc[q];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int q = 0; q < 7; q++) red[q][threadIdx.x] += red[q][threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x < 7) out[7 * t + threadIdx.x] = red[threadIdx.x][0];
}

static inline int grid_for(int n, int bs = STREAM_BLOCK) { return (n + bs - 1) / bs; }

// The updater's tubule classification (mt_length, src/updater.cpp:164-205)
// on the device: a bead is on the tubule when rad_lo < sqrt(x^2 + y^2) <
// rad_hi and cos(theta) > cos_min.  Writes the per-bead flag, optionally
// into the barrier's on_tubule array too, and counts per trajectory.
__global__ void __launch_bounds__(STREAM_BLOCK)
    k_mt_length(DevTopo T, DevState S, float rad_hi, float rad_lo, float cos_min, int apply, int *flags,
                int *counts) {
    const int b = blockIdx.x * STREAM_BLOCK + threadIdx.x;
    if (b >= T.nb) return;
    const float4 x = S.xyz[b];
    const float rad = sqrtf(x.x * x.x + x.y * x.y);
    const int on = (rad < rad_hi && rad > rad_lo && cosf(S.ang[b].y) > cos_min) ? 1 : 0;
    flags[b] = on;
    if (apply) T.on_tub[b] = on;
    if (on) atomicAdd(&counts[T.tid[b]], 1);
}

__global__ void __launch_bounds__(256) k_zero_ints(int *p, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void __launch_bounds__(STREAM_BLOCK) k_pack_flags(DevTopo T) {
    const int b = blockIdx.x * STREAM_BLOCK + threadIdx.x;
    if (b >= T.nb) return;
    T.flags[b] = (uint8_t)((T.mon_type[b] ? FL_MON : 0) | (T.gtp[b] == 1 ? FL_GTP1 : 0) |
                           (T.on_tub[b] == 0 ? FL_OFFTUB : 0) | (T.fixed[b] ? FL_FIXED : 0) | (T.extra[b] ? FL_EXTRA : 0));
}

// After any of the arrays behind the flags has changed: a byte per bead then
// serves every step, where the five arrays are 14 (64 tubes of 1040 beads:
// forces 9.6 -> 9.3 us, update 7.0 -> 6.8; one tube of 312: both in one 7.6 ->
// 7.3).
hipError_t launch_pack_flags(mte_engine *e) {
    hipLaunchKernelGGL(k_pack_flags, dim3(grid_for(e->nb)), dim3(STREAM_BLOCK), 0, e->stream, e->T);
    return hipGetLastError();
}

hipError_t launch_mt_length(mte_engine *e, float rad_hi, float rad_lo, float cos_min, int apply) {
    hipLaunchKernelGGL(k_zero_ints, dim3((e->ntraj + 255) / 256), dim3(256), 0, e->stream, e->mtl_counts, e->ntraj);
    hipLaunchKernelGGL(k_mt_length, dim3(grid_for(e->nb)), dim3(STREAM_BLOCK), 0, e->stream, e->T, e->S[e->cur],
                       rad_hi, rad_lo, cos_min, apply, e->mtl_flags, e->mtl_counts);
    if (apply) {
        const hipError_t s = launch_pack_flags(e);
        if (s != hipSuccess) return s;
    }
    return hipGetLastError();
}

hipError_t launch_frames(mte_engine *e, int buf) {
    hipLaunchKernelGGL(k_frames, dim3(grid_for(e->nb)), dim3(STREAM_BLOCK), 0, e->stream, e->S[buf], e->nb, e->L);
    return hipGetLastError();
}

// Batches with a periodic box take the kernels with the minimum image; there
// an open trajectory's separations are unchanged (side and inverse zero).
template <bool PERIODIC>
static void step_plain(mte_engine *e, const float *noise_step) {
    const int bs = e->tune.stream_block;
    const dim3 grid(grid_xcd(e->nb, bs)), block(2 * bs);
    auto k = bs == 64 ? k_step_plain<64, PERIODIC> : bs == 128 ? k_step_plain<128, PERIODIC> : k_step_plain<256, PERIODIC>;
    hipLaunchKernelGGL(k, grid, block, 0, e->stream, e->K, e->T, e->S[e->cur], e->S[1 - e->cur], e->seeds, noise_step,
                       e->L);
}
hipError_t launch_step_plain(mte_engine *e, const float *noise_step) {
    if (e->periodic) step_plain<true>(e, noise_step);
    else step_plain<false>(e, noise_step);
    e->cur = 1 - e->cur;
    return hipGetLastError();
}

template <bool PERIODIC>
static hipError_t forces_draw(mte_engine *e, TeaDraw D) {
    if (e->tune.forces == MTE_FORCES_LDS && e->forces_lds > 0) {
        const size_t helped_lds = e->forces_lds + sizeof(float4) * FORCE_TILE;
        const bool helped = helped_lds <= (size_t)e->lds_limit;   // up to 2496 beads
        auto k = helped ? k_forces_lds<PERIODIC, true> : k_forces_lds<PERIODIC, false>;
        const size_t lds = helped ? helped_lds : e->forces_lds;
        const hipError_t s = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (s != hipSuccess) return s;
        hipLaunchKernelGGL(k, dim3(grid_xcd(e->ntiles, 1)), dim3(helped ? 2 * FORCE_TILE : FORCE_TILE), lds, e->stream, e->K,
                           e->T, e->S[e->cur], e->tiles, e->ntiles, e->fxyz, e->fang, D);
    } else {
        const int bs = e->tune.stream_block;
        const dim3 grid(grid_xcd(e->nb, bs)), block(2 * bs);
        auto k = bs == 64 ? k_forces<64, PERIODIC> : bs == 128 ? k_forces<128, PERIODIC> : k_forces<256, PERIODIC>;
        hipLaunchKernelGGL(k, grid, block, 0, e->stream, e->K, e->T, e->S[e->cur], e->fxyz, e->fang, D);
    }
    return hipGetLastError();
}
static hipError_t launch_forces_draw(mte_engine *e, TeaDraw D) {
    return e->periodic ? forces_draw<true>(e, D) : forces_draw<false>(e, D);
}

hipError_t launch_forces(mte_engine *e) { return launch_forces_draw(e, TeaDraw{nullptr, nullptr, nullptr}); }

hipError_t launch_forces_tea(mte_engine *e, const float *noise_step) {
    return launch_forces_draw(e, TeaDraw{e->seeds, noise_step, e->tea.R});
}

hipError_t launch_energies(mte_engine *e) {
    const int bs = e->tune.stream_block;
    auto k = bs == 64 ? k_energies<64> : bs == 128 ? k_energies<128> : k_energies<256>;
    hipLaunchKernelGGL(k, dim3(grid_xcd(e->nb, bs)), dim3(bs), 0, e->stream, e->P, e->T, e->S[e->cur], e->en_bead);
    hipLaunchKernelGGL(k_traj_sum, dim3(e->ntraj), dim3(256), 0, e->stream, e->T, e->en_bead, e->en_traj);
    return hipGetLastError();
}

}  // namespace mte
