// bead_physics.h -- per-bead force and energy evaluation, shared by the
// streamed kernels (state in HBM) and the resident kernel (state in LDS).
// An accessor type supplies neighbour data by a handle, a list type the handles.
//
// Restates compute_kernel (src/compute_cuda.cu:32-525) and energy_kernel
// (:676-911) in attachment-point form; see device_common.h.
#pragma once
#include "device_common.h"

namespace mte {

__device__ __forceinline__ float3 scale3(float s, float3 v) { return make_float3(s * v.x, s * v.y, s * v.z); }

// Own-bead quantities needed for the angular gradients.
struct Own {
    float3 r, n, a1, a2, uphi;
    float2 uth;
    float fi, theta, psi;
    float box;   // periodic side of the bead's trajectory (0: open)
    float ibox;  // inv_side(box)
    int flags;   // packed (FL_*)
};
__device__ __forceinline__ void set_box(Own &o, float L) {
    o.box = L;
    o.ibox = inv_side(L);
}

// trig = (sin theta, cos theta, sin psi, cos psi) of the bead.
__device__ __forceinline__ Own make_own_trig(float4 xyz, float4 ang, float4 fn, float4 fp1, float4 fp2, float4 trig,
                                             int flags) {
    Own o;
    o.r = f3(xyz);
    o.n = f3(fn);
    o.a1 = f3(fp1);
    o.a2 = f3(fp2);
    o.fi = ang.x;
    o.theta = ang.y;
    o.psi = ang.z;
    o.uphi = make_float3(trig.w * trig.y, trig.z * trig.y, -trig.x);
    o.uth = make_float2(-trig.z, trig.w);
    o.box = o.ibox = 0.f;
    o.flags = flags;
    return o;
}

__device__ __forceinline__ Own make_own(float4 xyz, float4 ang, float4 fn, float4 fp1, float4 fp2, int flags) {
    float4 trig;
    sincos_fast(ang.y, &trig.x, &trig.y);
    sincos_fast(ang.z, &trig.z, &trig.w);
    return make_own_trig(xyz, ang, fn, fp1, fp2, trig, flags);
}

// Neighbour data by a handle that the list entry gives.  In LDS, four arrays
// hold per bead its position with the packed flags in w, and the rotated
// offsets with the Euler angles in w (n|fi, p1|theta, p2|psi); the handle is
// the LDS address of the bead's position, and n, p1, p2 are the distances of
// the other arrays from that one.
typedef float v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void *)p;
}
__device__ __forceinline__ float4 lds_f4(uint32_t a) {
    const v4f v = *(const __attribute__((address_space(3))) v4f *)(uintptr_t)a;
    return make_float4(v.x, v.y, v.z, v.w);
}
struct LdsAcc {
    uint32_t x, n, p1, p2;   // x: address of the position array
    static constexpr int SCALE = sizeof(float4);
    __device__ __forceinline__ LdsAcc(const float4 *lx, const float4 *ln, const float4 *l1, const float4 *l2)
        : x(lds_addr(lx)), n(in_vgpr(lds_addr(ln) - lds_addr(lx))), p1(in_vgpr(lds_addr(l1) - lds_addr(lx))),
          p2(in_vgpr(lds_addr(l2) - lds_addr(lx))) {}
    __device__ __forceinline__ uint32_t origin() const { return x; }
    __device__ __forceinline__ float4 xyz(uint32_t h) const { return lds_f4(h); }
    __device__ __forceinline__ float4 fn(uint32_t h) const { return lds_f4(h + n); }
    __device__ __forceinline__ float4 lat(uint32_t h, bool p2nd) const { return lds_f4(h + (p2nd ? p2 : p1)); }
    __device__ __forceinline__ float3 angles(float4 fnj, uint32_t h) const {
        return make_float3(fnj.w, lds_f4(h + p1).w, lds_f4(h + p2).w);
    }
    __device__ __forceinline__ int flags(float4 xj, uint32_t) const { return __float_as_int(xj.w); }
};

// Stages beads [0, n) of the trajectory starting at global bead `base` into
// the four LDS arrays (all threads of the workgroup; no barrier).
__device__ __forceinline__ void stage_state(const DevTopo &T, const DevState &S, int base, int n, float4 *lx,
                                            float4 *ln, float4 *l1, float4 *l2) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int b = base + i;
        float4 x = S.xyz[b];
        x.w = __int_as_float(T.flags[b]);
        const float4 a = S.ang[b];
        float4 fn = S.fn[b], f1 = S.fp1[b], f2 = S.fp2[b];
        fn.w = a.x;
        f1.w = a.y;
        f2.w = a.z;
        lx[i] = x;
        ln[i] = fn;
        l1[i] = f1;
        l2[i] = f2;
    }
}

// Neighbour lists held in the k-major global arrays of bead b.  The handle of
// global bead j is origin + SCALE (j - base): its index, or the LDS address of
// its position.
template <int SCALE>
struct GlobalLists {
    const DevTopo &T;
    int b, base;
    uint32_t origin;
    __device__ __forceinline__ int harm() const { return T.harm[b]; }
    __device__ __forceinline__ int nlon() const { return T.lon_n[b]; }
    __device__ __forceinline__ int lon(int k) const { return T.lon[k * T.nb + b]; }
    __device__ __forceinline__ int nlat() const { return T.lat_n[b]; }
    __device__ __forceinline__ int lat(int k) const { return T.lat[k * T.nb + b]; }
    __device__ __forceinline__ uint32_t handle(int j) const { return origin + (uint32_t)((j - base) * SCALE); }
    __device__ __forceinline__ uint32_t ref(int e) const { return handle(ent_j(e)); }
    // The LJ entries in order: four(h0, h1, h2, h3) for each four of them,
    // one(h) for each of the rest.
    template <class Four, class One>
    __device__ __forceinline__ void lj(const Four &four, const One &one) const {
        const int n = T.lj_n[b];
        auto at = [&](int k) { return handle(T.lj[(size_t)k * T.nb + b]); };
        int k = 0;
        for (; k + 4 <= n; k += 4) four(at(k), at(k + 1), at(k + 2), at(k + 3));
        for (; k < n; k++) one(at(k));
    }
};

// The same lists, for one force evaluation: what most beads need (the counts,
// one longitudinal, two lateral and the first LJ entries) is requested at
// once when the lists are made, before the bead's state.  Read where they are
// used, each count and entry is one more trip to memory that nothing overlaps
// (64 tubes of 1040 beads: k_forces_lds 14.6 -> 12.5 us, one tube of 312 beads
// 7.7 -> 5.7, 4 periodic systems of 122646 beads: k_step_plain 11.1 -> 10.1).
// Slots beyond a count hold no entry but exist.
constexpr int LJ_AHEAD = 4;
template <int SCALE>
struct AheadLists {
    const DevTopo &T;
    int b, base;
    uint32_t origin;
    int eh, cl, ct, cj, elon, elat0, elat1, elj[LJ_AHEAD];
    __device__ __forceinline__ AheadLists(const DevTopo &T, int b, int base, uint32_t origin)
        : T(T), b(b), base(base), origin(origin), eh(T.harm[b]), cl(T.lon_n[b]), ct(T.lat_n[b]), cj(T.lj_n[b]),
          elon(T.lon[b]), elat0(T.lat[b]), elat1(T.lat[T.nb + b]) {
#pragma unroll
        for (int u = 0; u < LJ_AHEAD; u++) elj[u] = T.lj[(size_t)min(u, T.max_lj - 1) * T.nb + b];
    }
    __device__ __forceinline__ int harm() const { return eh; }
    __device__ __forceinline__ int nlon() const { return cl; }
    __device__ __forceinline__ int lon(int k) const { return k == 0 ? elon : T.lon[k * T.nb + b]; }
    __device__ __forceinline__ int nlat() const { return ct; }
    __device__ __forceinline__ int lat(int k) const { return k == 0 ? elat0 : k == 1 ? elat1 : T.lat[k * T.nb + b]; }
    __device__ __forceinline__ uint32_t handle(int j) const { return origin + (uint32_t)((j - base) * SCALE); }
    __device__ __forceinline__ uint32_t ref(int e) const { return handle(ent_j(e)); }
    // the next four entries are requested before the current ones' positions
    template <class Four, class One>
    __device__ __forceinline__ void lj(const Four &four, const One &one) const {
        uint32_t h[LJ_AHEAD];
#pragma unroll
        for (int u = 0; u < LJ_AHEAD; u++) h[u] = handle(elj[u]);
        int k = 0;
        for (; k + LJ_AHEAD <= cj; k += LJ_AHEAD) {
            int e[LJ_AHEAD];
#pragma unroll
            for (int u = 0; u < LJ_AHEAD; u++) e[u] = T.lj[(size_t)min(k + LJ_AHEAD + u, cj - 1) * T.nb + b];
            four(h[0], h[1], h[2], h[3]);
#pragma unroll
            for (int u = 0; u < LJ_AHEAD; u++) h[u] = handle(e[u]);
        }
#pragma unroll
        for (int u = 0; u < LJ_AHEAD - 1; u++)
            if (k + u < cj) one(h[u]);
    }
};

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// What a bead's bonds add up to: force, and the moments about the bead of
// its bonds at the axial offset (M, to be crossed with n) and at the lateral
// ones (Tq).  A bond's torque is a x f with a its offset; the three angular
// components are the torque's along u_phi, u_theta, u_psi, taken once.
struct BondSum {
    float3 F, M, Tq;
    float3 bend;   // fi, theta, psi
};
__device__ __forceinline__ float3 cross_add(float3 a, float3 f, float3 t) {
    return make_float3(fmaf(a.y, f.z, fmaf(-a.z, f.y, t.x)), fmaf(a.z, f.x, fmaf(-a.x, f.z, t.y)),
                       fmaf(a.x, f.y, fmaf(-a.y, f.x, t.z)));
}

// Bending torques of a harmonic or longitudinal pair (:156-177, :271-295):
// rm > 0: F += B sin(d - d0); rm < 0: F -= B sin(-d - d0), one form for both
// since sin is odd: B sin(d - s d0), s = rm / 2 = +-1.
__device__ __forceinline__ void bending(const ForceK &K, float rm, float th_h, const Own &I, float3 aj, float3 &bend) {
    const float3 s = sin3(make_float3(fmaf(-rm, K.fi_h, aj.x - I.fi), fmaf(-rm, th_h, aj.y - I.theta),
                                      fmaf(-rm, K.psi_h, aj.z - I.psi)));
    bend.x = fmaf(K.Bfi, s.x, bend.x);
    bend.y = fmaf(K.Bth, s.y, bend.y);
    bend.z = fmaf(K.Bpsi, s.z, bend.z);
}

// |g|^2, above zero (1e-30 nm^2 is below the rounding of any other gap): its
// reciprocal root is finite, and a closed gap's force is 0 times it.
__device__ __forceinline__ float gap2(float3 g) { return fmaf(g.x, g.x, fmaf(g.y, g.y, fmaf(g.z, g.z, 1e-30f))); }

// dU/dr over r of a Morse bond (d = 2 A D, na = -A log2 e) with its barrier.
__device__ __forceinline__ float bond_slope(float d2, float na, float d, bool barrier, float br, float bk, float bc) {
    const float inv = rsq_fast(d2), dr = d2 * inv;
    const float e = exp2_fast(na * dr);
    float s = d * fmaf(-e, e, e);
    if (__any(barrier)) {   // rare: a branch, where the compiler would select
        const float x = dr - br;
        s = barrier ? fmaf(bc * x, exp2_fast(bk * (x * x)), s) : s;
    }
    return s * inv;
}

template <bool PERIODIC>
__device__ __forceinline__ float3 separation(const Own &I, float4 xj) {
    const float3 d = sub3(I.r, f3(xj));
    if (!PERIODIC) return d;
    return min_image_inv(d, I.box, I.ibox);
}

// 1 for r2 < LJ_CUT^2, else 0 (NaN: 0), by a fused product and clamp: below
// the cutoff 2^100 (LJ_CUT^2 - r2) is at least 2^81.  Two 2-cycle operations
// per pair with the product, where comparing and selecting take 4 each.
__device__ __forceinline__ float below_cut(float r2, float nscale, float offset) {
    return __builtin_amdgcn_fmed3f(fmaf(nscale, r2, offset), 0.f, 1.f);
}

// LJ repulsion over the list; the cutoff test scales the force (no branch
// around the accumulation), and runs with and without the regularization cap
// get separate loops (a uniform choice: the cap's reciprocal square root is
// not paid per pair when it is off).
// Without the regularization the sum is to be scaled by K.lj6 (lj_scale).
template <bool PERIODIC, bool REG, class Acc, class Lists>
__device__ __forceinline__ float3 lj_sum_as(const ForceK &K, const Acc &A, const Lists &Ls, const Own &I) {
    const float nscale = in_vgpr(-0x1p100f), offset = in_vgpr(LJ_CUT * LJ_CUT * 0x1p100f);
    float3 f = make_float3(0.f, 0.f, 0.f);
    auto pair = [&](float4 xj) {
        const float3 d = separation<PERIODIC>(I, xj);
        const float r2 = d.x * d.x + d.y * d.y + d.z * d.z;
        const float inv = rcp_fast(r2);
        const float inv2 = inv * inv;
        float s = below_cut(r2, nscale, offset) * (inv2 * inv2);
        // REGULARIZATION (src/compute_cuda.cu:482-486): the pair force s r is
        // capped at gammaR r_mon / dt, i.e. s at that over r (r_mon = 2 nm)
        if (REG) s = fminf(K.lj6 * s, K.lj_cap * rsq_fast(r2));
        f.x = fmaf(s, d.x, f.x);
        f.y = fmaf(s, d.y, f.y);
        f.z = fmaf(s, d.z, f.z);
    };
    // four positions requested before the first is used (one wait for the four
    // gathers rather than one each), then summed in list order
    Ls.lj(
        [&](uint32_t h0, uint32_t h1, uint32_t h2, uint32_t h3) {
            const float4 x0 = A.xyz(h0), x1 = A.xyz(h1), x2 = A.xyz(h2), x3 = A.xyz(h3);
            pair(x0);
            pair(x1);
            pair(x2);
            pair(x3);
        },
        [&](uint32_t h) { pair(A.xyz(h)); });
    return f;
}
template <bool PERIODIC, class Acc, class Lists>
__device__ __forceinline__ float3 lj_sum(const ForceK &K, const Acc &A, const Lists &Ls, const Own &I) {
    return K.lj_reg ? lj_sum_as<PERIODIC, true>(K, A, Ls, I) : lj_sum_as<PERIODIC, false>(K, A, Ls, I);
}
__device__ __forceinline__ float lj_scale(const ForceK &K) { return K.lj_reg ? 1.f : K.lj6; }

// The bonds of a bead.
template <bool PERIODIC, class Acc, class Lists>
__device__ __forceinline__ BondSum bond_forces(const ForceK &K, const Acc &A, const Lists &Ls, const Own &I) {
    BondSum S;
    S.F = S.M = S.Tq = S.bend = make_float3(0.f, 0.f, 0.f);
    const bool gtp = (I.flags & FL_GTP1) != 0, off = K.barrier && (I.flags & FL_OFFTUB) != 0;
    // an axial bond with force slope s over its gap g
    auto axial = [&](float rm, float s, float3 g) {
        const float3 f = scale3(-s, g);
        S.F = make_float3(S.F.x + f.x, S.F.y + f.y, S.F.z + f.z);
        S.M = make_float3(fmaf(rm, f.x, S.M.x), fmaf(rm, f.y, S.M.y), fmaf(rm, f.z, S.M.z));
    };
    auto axial_gap = [&](float rm, float4 xj, float4 nj) {
        const float3 d = separation<PERIODIC>(I, xj);
        return make_float3(fmaf(rm, I.n.x + nj.x, d.x), fmaf(rm, I.n.y + nj.y, d.y), fmaf(rm, I.n.z + nj.z, d.z));
    };
    // harmonic (intra-dimer spring + bending), :70-182
    const int eh = Ls.harm();
    if (eh >= 0) {
        const uint32_t j = Ls.ref(eh);
        const float rm = ent_f(eh) ? RMON : -RMON;
        const float4 xj = A.xyz(j), nj = A.fn(j);
        const float3 g = axial_gap(rm, xj, nj);
        axial(rm, K.C, g);
        if (gap2(g) < ANGLE_CUT * ANGLE_CUT)
            bending(K, rm, gtp ? K.th_gtp_h : K.th_gdp_h, I, A.angles(nj, j), S.bend);
    }
    // longitudinal Morse + barrier + bending, :189-299
    const int nlon = Ls.nlon();
    for (int k = 0; k < nlon; k++) {
        const int e = Ls.lon(k);
        const uint32_t j = Ls.ref(e);
        const float rm = ent_f(e) ? RMON : -RMON;
        const float4 xj = A.xyz(j), nj = A.fn(j);
        const float3 g = axial_gap(rm, xj, nj);
        const float d2 = gap2(g);
        const int fj = A.flags(xj, j);
        axial(rm, bond_slope(d2, K.lon_a, K.lon_d, off && (fj & FL_OFFTUB), K.lonb_r, K.lonb_k, K.lonb_c), g);
        if (d2 < ANGLE_CUT * ANGLE_CUT) {
            const bool gl = (I.r.z > xj.z) ? gtp : (fj & FL_GTP1) != 0;   // theta0 of the bead with larger z
            bending(K, rm, gl ? K.th_gtp_h : K.th_gdp_h, I, A.angles(nj, j), S.bend);
        }
    }
    // lateral Morse + barrier with seam weakening, :304-466
    const int nlat = Ls.nlat();
    for (int k = 0; k < nlat; k++) {
        const int e = Ls.lat(k);
        const uint32_t j = Ls.ref(e);
        const bool sw = ent_f(e) != 0;
        const float3 a = sw ? I.a1 : I.a2;
        const float4 xj = A.xyz(j), bj = A.lat(j, sw);
        const float3 d = separation<PERIODIC>(I, xj);
        const float3 g = make_float3(d.x + (a.x - bj.x), d.y + (a.y - bj.y), d.z + (a.z - bj.z));
        const int fj = A.flags(xj, j);
        // seam bonds (monomer types differ) are weakened by seam_coeff (:447-452)
        const float dl = (fj ^ I.flags) & FL_MON ? K.seam_d : K.lat_d;
        const float s = bond_slope(gap2(g), K.lat_a, dl, off && (fj & FL_OFFTUB), K.latb_r, K.latb_k, K.latb_c);
        const float3 f = scale3(-s, g);
        S.F = make_float3(S.F.x + f.x, S.F.y + f.y, S.F.z + f.z);
        S.Tq = cross_add(a, f, S.Tq);
    }
    return S;
}

// Their force and torque.
__device__ __forceinline__ void bond_total(const BondSum &S, const Own &I, float F[6]) {
    const float3 t = cross_add(I.n, S.M, S.Tq);
    F[0] = S.F.x;
    F[1] = S.F.y;
    F[2] = S.F.z;
    F[3] = fmaf(I.uphi.x, t.x, fmaf(I.uphi.y, t.y, fmaf(I.uphi.z, t.z, S.bend.x)));
    F[4] = fmaf(I.uth.x, t.x, fmaf(I.uth.y, t.y, S.bend.y));
    F[5] = t.z + S.bend.z;
}

// Adds the LJ sum (:470-495) and the walls; wall_z is Parameters.zs of the
// bead's trajectory.
__device__ __forceinline__ void add_lj_walls(const ForceK &K, float3 lj, float wall_z, const float3 r, float F[6]) {
    if (K.lj_on) {
        const float s6 = lj_scale(K);
        F[0] = fmaf(s6, lj.x, F[0]);
        F[1] = fmaf(s6, lj.y, F[1]);
        F[2] = fmaf(s6, lj.z, F[2]);
    }
    // cylindrical and end walls, :497-517
    if (K.is_wall) {
        const float z = r.z, lb = K.wall_left, zt = wall_z + lb;
        if (z < lb) F[2] += K.wall_eps * fabsf(z - lb);
        else if (z > zt) F[2] += -K.wall_eps * fabsf(z - zt);
        const float rad2 = r.x * r.x + r.y * r.y;
        if (rad2 > K.wall_r * K.wall_r) {
            const float rad = sqrtf(rad2);
            const float coeff = -K.wall_eps * (rad - K.wall_r);
            F[0] += r.x / rad * coeff;
            F[1] += r.y / rad * coeff;
        }
    }
}

template <bool PERIODIC, class Acc, class Lists>
__device__ __forceinline__ void bead_force(const ForceK &K, const Acc &A, const Lists &Ls, float wall_z, const Own &I,
                                           float F[6]) {
    bond_total(bond_forces<PERIODIC>(K, A, Ls, I), I, F);
    const float3 lj = K.lj_on ? lj_sum<PERIODIC>(K, A, Ls, I) : make_float3(0.f, 0.f, 0.f);
    add_lj_walls(K, lj, wall_z, I.r, F);
}

// Energies in the energy_kernel convention (:676-911): U_harm, U_long,
// U_lat, U_psi, U_fi, U_teta, U_lj, each halved.
template <class Acc>
__device__ __forceinline__ void bead_energy(const mte_params &P, const DevTopo &T, const Acc &A, int b, const Own &I,
                                            float U[7]) {
#pragma unroll
    for (int q = 0; q < 7; q++) U[q] = 0.f;
    const int nb = T.nb;
    const int h = T.harm[b];
    if (h >= 0) {
        const int j = ent_j(h);
        const float rm = ent_f(h) ? RMON : -RMON;
        const Grad G = gap_grad(min_image_pre(sub3(I.r, f3(A.xyz(j))), I.box, I.ibox), scale3(rm, I.n), scale3(-rm, f3(A.fn(j))), I.uphi, I.uth);
        U[0] += (P.C / 2.f) * G.dr * G.dr;
        if (G.dr < ANGLE_CUT) {
            const float4 aj = A.ang(j);
            const float psiij = I.psi - aj.z, fiij = I.fi - aj.x, thetaji = aj.y - I.theta;
            U[3] += P.B_psi * (1.f - cosf(psiij - P.psi_0));
            U[4] += P.B_fi * (1.f - cosf(fiij - P.fi_0));
            U[5] += P.B_theta * (1.f - cosf(thetaji - (A.gtp1(b) ? P.theta0_gtp : P.theta0_gdp)));
        }
    }
    const int nlon = T.lon_n[b];
    for (int k = 0; k < nlon; k++) {
        const int e = T.lon[k * nb + b];
        const int j = ent_j(e);
        const float rm = ent_f(e) ? RMON : -RMON;
        const float4 xj = A.xyz(j);
        const Grad G = gap_grad(min_image_pre(sub3(I.r, f3(xj)), I.box, I.ibox), scale3(rm, I.n), scale3(-rm, f3(A.fn(j))), I.uphi, I.uth);
        U[1] += morse_en(P.D_long, P.A_long, G.dr);
        if (P.barrier && A.offtub(b) && A.offtub(j))
            U[1] += barr(P.a_barr_long, P.r_barr_long, P.w_barr_long, G.dr);
        if (G.dr < ANGLE_CUT) {
            const float4 aj = A.ang(j);
            const float psiij = I.psi - aj.z, fiij = I.fi - aj.x, thetaij = I.theta - aj.y;
            const int last = (I.r.z > xj.z) ? b : j;
            const float th0 = A.gtp1(last) ? P.theta0_gtp : P.theta0_gdp;
            U[3] += P.B_psi * (1.f - cosf(psiij - P.psi_0));
            U[4] += P.B_fi * (1.f - cosf(fiij - P.fi_0));
            U[5] += P.B_theta * (1.f - cosf(thetaij - th0));
        }
    }
    const int nlat = T.lat_n[b];
    for (int k = 0; k < nlat; k++) {
        const int e = T.lat[k * nb + b];
        const int j = ent_j(e);
        const int sw = ent_f(e);
        const Grad G = gap_grad(min_image_pre(sub3(I.r, f3(A.xyz(j))), I.box, I.ibox), sw ? I.a1 : I.a2, f3(sw ? A.fp2(j) : A.fp1(j)),
                                I.uphi, I.uth);
        if (A.mon(b) != A.mon(j)) U[2] += morse_en(P.D_lat / P.seam_coeff, P.A_lat, G.dr);
        else U[2] += morse_en(P.D_lat, P.A_lat, G.dr);
        if (P.barrier && A.offtub(b) && A.offtub(j))
            U[2] += barr(P.a_barr_lat, P.r_barr_lat, P.w_barr_lat, G.dr);
    }
    if (P.lj_on) {
        const int nlj = T.lj_n[b];
        for (int k = 0; k < nlj; k++) {
            const int j = T.lj[k * nb + b];
            const float3 d = min_image_pre(sub3(I.r, f3(A.xyz(j))), I.box, I.ibox);
            const float dx = d.x, dy = d.y, dz = d.z;
            const float r2 = dx * dx + dy * dy + dz * dz;
            if (sqrtf(r2) < LJ_CUT) {
                const float inv = 1.f / r2;
                U[6] += P.ljscale * P.ljsigma6 * (inv * inv * inv);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 7; q++) U[q] *= 0.5f;
}

// Euler-Maruyama update of one mobile bead, src/compute_cuda.cu:955-961.
__device__ __forceinline__ void em_update(const ForceK &K, const float F[6], float4 rx, float4 ra, float4 &x,
                                          float4 &a) {
    x.x += fmaf(K.dtg, F[0], K.vR * rx.x);
    x.y += fmaf(K.dtg, F[1], K.vR * rx.y);
    x.z += fmaf(K.dtg, F[2], K.vR * rx.z);
    em_angles(K, F[3], F[4], F[5], ra, a);
}

// Random-force draw for TEA steps, fused into the force pass: every bead
// draws sqrt(2 kB T gammaR / dt) xi from its xyz stream
// (integrateTea_prepare, src/bdhitea_kernel.cu:16-36).
struct TeaDraw {
    uint4 *seeds;
    const float *noise;
    float4 *R;   // nullptr: no draw
};

// One bead's share of it.
__device__ __forceinline__ float4 tea_draw(const TeaDraw &D, float var, int b, bool extra) {
    float4 r;
    if (D.noise) {
        const float *nz = D.noise + 6 * (size_t)b;
        r = make_float4(nz[0], nz[1], nz[2], 0.f);
    } else {
        uint4 s = D.seeds[b];
        r = normals4(s);
        D.seeds[b] = s;
    }
    return extra ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(r.x * var, r.y * var, r.z * var, 0.f);
}

}  // namespace mte
