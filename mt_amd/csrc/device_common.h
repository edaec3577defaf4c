// device_common.h -- device-side building blocks shared by the gfx950 kernels.
//
// Bonded geometry is written in attachment-point form: each bonded gap is
// g = (r_i + a_i) - (r_j + b_j) with body-fixed offsets rotated by
// R = Rz(psi) Ry(theta) Rx(phi) (the rotation whose entries the reference
// expands at src/compute_cuda.cu:89-96 and :337-352).  The gradient of
// |g|^2/2 with respect to bead i is g for x, y, z and u_q . (a_i x g) for the
// angles, u_phi = Rz Ry e_x, u_theta = Rz e_y, u_psi = e_z.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/mt_engine.h"

namespace mte {

constexpr float RMON = 2.0f;          // src/mt.h:24
constexpr float LJ_CUT = 6.0f;        // src/mt.h:25
constexpr float ANGLE_CUT = 1.0f;     // src/mt.h:42
constexpr float PAIR_CUT = 2.5f;      // src/mt.h:61
constexpr float KB = 0.0019872041f;   // src/mt.h:40
constexpr int MAXLON = 8;             // src/preparator.cpp:722
constexpr int MAXLAT = 16;            // src/preparator.cpp:721
// Centre distance beyond which no bonded candidate can pass PAIR_CUT:
// |g| >= d - 2*r_mon (axial) and |g| >= d - |p1| - |p2| ~ d - 3.995 (lateral).
constexpr float BOND_PREFILTER = 6.75f;

// Lateral attachment offsets p1, p2 of src/mt.h:44-50, evaluated in double on
// the host and rounded once (p2 = (p1x, -p1y, -p1z)).
struct LatOffsets { float p1x, p1y, p1z, p2x, p2y, p2z; };

// Packed list entries: (global j << 1) | flag, where flag is "R_MON > 0" for
// harmonic/longitudinal entries and "p1/p2 swapped" for lateral entries.
__device__ __forceinline__ int ent_j(int e) { return e >> 1; }
__device__ __forceinline__ int ent_f(int e) { return e & 1; }

// Topology on the device (global bead indices, k-major list slots).
struct DevTopo {
    int nb, ntraj, max_lj;
    const int *tid;       // bead -> trajectory
    const int *tbase;     // trajectory -> first bead
    const int *tsize;     // trajectory -> bead count
    const int *harm;      // packed partner or -1
    const int *harm_raw;  // reference-encoded partner (local), drives pairs_kernel semantics
    int *lon_n, *lon;     // lon[k * nb + b]
    int *lat_n, *lat;
    int *lj_n, *lj;
    const uint8_t *fixed;
    uint8_t *extra;
    const int *mon_type;
    int *gtp, *on_tub;
    uint8_t *flags;       // the five per-bead flags (FL_*), packed by k_pack_flags
    const float *zs;
    const float *tbox;    // trajectory -> periodic box side (0: open boundaries)
    int *overflow;        // set to 1 by a rebuild that ran out of list capacity
    int *frozen;          // steps the resident kernel left undone because `overflow` was set
};

// Per-bead flags: monomer type, GTP state 1, off the tubule, fixed, extra.
constexpr int FL_MON = 1, FL_GTP1 = 2, FL_OFFTUB = 4, FL_FIXED = 8, FL_EXTRA = 16;
__device__ __forceinline__ bool is_mobile(int flags) { return (flags & (FL_FIXED | FL_EXTRA)) == 0; }

// One buffer of bead state: positions, angles and the rotated offsets.
struct DevState {
    float4 *xyz;   // x, y, z, -
    float4 *ang;   // fi, theta, psi, -   (Coord order)
    float4 *fn;    // R e_z
    float4 *fp1;   // R p1
    float4 *fp2;   // R p2
};

__device__ __forceinline__ float3 f3(float4 v) { return make_float3(v.x, v.y, v.z); }

// Minimum-image separation in a cubic periodic box of side L (L == 0: open).
// The reference has no periodic boundaries; the uneven free-dimer batches
// run in one.
__device__ __forceinline__ float3 min_image(float3 d, float L) {
    if (L > 0.f) {
        const float iL = 1.f / L;
        d.x -= L * rintf(d.x * iL);
        d.y -= L * rintf(d.y * iL);
        d.z -= L * rintf(d.z * iL);
    }
    return d;
}
// min_image with 1/L taken outside a loop (iL = 0 on open boundaries, where
// d comes back unchanged): no branch in the loop body
__device__ __forceinline__ float3 min_image_inv(float3 d, float L, float iL) {
    d.x -= L * rintf(d.x * iL);
    d.y -= L * rintf(d.y * iL);
    d.z -= L * rintf(d.z * iL);
    return d;
}
__device__ __forceinline__ float inv_side(float L) { return L > 0.f ? 1.f / L : 0.f; }
// min_image with iL = inv_side(L) taken by the caller (outside its loops):
// the same values, without a division per call
__device__ __forceinline__ float3 min_image_pre(float3 d, float L, float iL) {
    if (L > 0.f) d = min_image_inv(d, L, iL);
    return d;
}
__device__ __forceinline__ float3 sub3(float3 a, float3 b) { return make_float3(a.x - b.x, a.y - b.y, a.z - b.z); }

// Cells per side of a periodic box for cells of side >= `side` searched K
// cells either way (at least 2K + 1, where the stencil spans the whole box).
// Every kernel that reads a cell table must count the cells as the kernel
// that filled it did, but the fast division rounds otherwise where the
// compiler knows `side` (672 nm / 12 nm came to 56 in one kernel and to 55 in
// another): products decide, which round alike everywhere.
__device__ __forceinline__ int cell_dims(float box, float side, int K) {
    int n = (int)floorf(box / side);
    if ((float)n * side > box) n--;
    if ((float)(n + 1) * side <= box) n++;
    return max(2 * K + 1, n);
}

struct CellGeom {
    float cs;      // cell side
    int dims;      // cells per side in a periodic box (0: open)
};
__device__ __forceinline__ CellGeom cell_geom(float box, float side, int K) {
    CellGeom g;
    g.dims = box > 0.f ? cell_dims(box, side, K) : 0;
    g.cs = g.dims > 0 ? box / (float)g.dims : side;
    return g;
}
// A coordinate in cells from the origin (of the box, where it is periodic).
__device__ __forceinline__ float cell_coord(float x, float box, const CellGeom &g) {
    if (g.dims > 0) x -= box * floorf(x / box);
    return x / g.cs;
}

// Bucket hash of a cell, masked to the table's size by the caller.
__device__ __forceinline__ uint32_t cell_hash(int cx, int cy, int cz) {
    return ((uint32_t)cx * 73856093u) ^ ((uint32_t)cy * 19349663u) ^ ((uint32_t)cz * 83492791u);
}
// Periodic cell index: i in [-dims, 2 dims) wrapped into [0, dims) (a
// neighbour stencil never reaches further), without an integer division.
__device__ __forceinline__ int wrap_cell(int i, int dims) { return i < 0 ? i + dims : (i >= dims ? i - dims : i); }

// sin and cos by Cody-Waite reduction modulo pi/2 (two-part pi/2, exact
// with FMA for |x| < 8192) and the single-precision minimax polynomials of
// the Cephes library (S. L. Moshier, sinf.c / cosf.c) on [-pi/4, pi/4];
// about 1 ulp.  The quadrant is the low bits of 2 x / pi + 1.5 2^23, and the
// signs are set by exclusive or (2-cycle operations, where a conversion, a
// comparison or a selection takes 4).
constexpr float SINCOS_MAX = 8192.f;
__device__ __forceinline__ void sincos_reduced(float x, float *s, float *c) {   // |x| < SINCOS_MAX
    const float jm = fmaf(x, 0.63661977236758134f, 12582912.f);
    const uint32_t q = __float_as_uint(jm);
    const float j = jm - 12582912.f;
    float r = fmaf(j, -1.57079637050628662109375f, x);
    r = fmaf(j, 4.37113900018624283e-8f, r);
    const float z = r * r;
    const float sp = fmaf(z * r, fmaf(z, fmaf(z, -1.9515295891e-4f, 8.3321608736e-3f), -1.6666654611e-1f), r);
    const float cp = fmaf(z * z, fmaf(z, fmaf(z, 2.443315711809948e-5f, -1.388731625493765e-3f), 4.166664568298827e-2f),
                          fmaf(-0.5f, z, 1.0f));
    const float ss = (q & 1u) ? cp : sp, cc = (q & 1u) ? sp : cp;
    *s = __uint_as_float(__float_as_uint(ss) ^ ((q << 30) & 0x80000000u));
    *c = __uint_as_float(__float_as_uint(cc) ^ (((q + 1u) << 30) & 0x80000000u));
}
// |x| >= 8192 is first reduced modulo 2*pi in FP64.
__device__ __forceinline__ float reduce_far(float x) {
    const double d = (double)x;
    return (float)(d - 6.283185307179586477 * rint(d * 0.15915494309189533577));
}
__device__ __forceinline__ void sincos_fast(float x, float *s, float *c) {
    if (!(fabsf(x) < SINCOS_MAX)) x = reduce_far(x);
    sincos_reduced(x, s, c);
}
__device__ __forceinline__ float sin_fast(float x) {
    float s, c;
    sincos_fast(x, &s, &c);
    return s;
}
// Three sines of arguments that usually need no reduction (bonded angle
// differences): where all lie in [-pi/4, pi/4], the reduction's identity, only
// the sine polynomials are evaluated, and a wave takes the full path only if
// one of its lanes needs it.
__device__ __forceinline__ float sin_poly(float x) {
    const float z = x * x;
    return fmaf(z * x, fmaf(z, fmaf(z, -1.9515295891e-4f, 8.3321608736e-3f), -1.6666654611e-1f), x);
}
__device__ __forceinline__ float3 sin3(float3 x) {
    if (fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fabsf(x.z)) <= 0.78539816f)
        return make_float3(sin_poly(x.x), sin_poly(x.y), sin_poly(x.z));
    return make_float3(sin_fast(x.x), sin_fast(x.y), sin_fast(x.z));
}
// Keeps a loop constant in a vector register: an FP32 operation with a scalar
// operand issues at half rate (4 cycles per wave, measured, against 2).
__device__ __forceinline__ float in_vgpr(float v) {
    __asm__("" : "+v"(v));
    return v;
}

__device__ __forceinline__ uint32_t in_vgpr(uint32_t v) {
    __asm__("" : "+v"(v));
    return v;
}

__device__ __forceinline__ float rcp_fast(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float rsq_fast(float x) { return __builtin_amdgcn_rsqf(x); }

// A bead's frame: the rotated offsets R e_z, R p1, R p2 and the sines and
// cosines of theta and psi, R = Rz(psi) Ry(theta) Rx(phi).  p2 is p1 with its
// y and z components negated (LatOffsets), so R p1 and R p2 are x c1 +- (y c2
// + z c3) with c1, c2, c3 the columns of R.
struct Frame {
    float3 n, p1, p2;
    float st, ct, sp, cp;
};
__device__ __forceinline__ Frame make_frame(float fi, float theta, float psi, const LatOffsets &L) {
    if (!(fmaxf(fmaxf(fabsf(fi), fabsf(theta)), fabsf(psi)) < SINCOS_MAX)) {
        if (!(fabsf(fi) < SINCOS_MAX)) fi = reduce_far(fi);
        if (!(fabsf(theta) < SINCOS_MAX)) theta = reduce_far(theta);
        if (!(fabsf(psi) < SINCOS_MAX)) psi = reduce_far(psi);
    }
    Frame o;
    float sf, cf;
    sincos_reduced(fi, &sf, &cf);
    sincos_reduced(theta, &o.st, &o.ct);
    sincos_reduced(psi, &o.sp, &o.cp);
    const float a = o.cp * o.st, b = o.sp * o.st;
    o.n = make_float3(fmaf(a, cf, o.sp * sf), fmaf(b, cf, -(o.cp * sf)), o.ct * cf);
    const float3 c2 = make_float3(fmaf(a, sf, -(o.sp * cf)), fmaf(b, sf, o.cp * cf), o.ct * sf);
    const float3 q = make_float3(fmaf(L.p1y, c2.x, L.p1z * o.n.x), fmaf(L.p1y, c2.y, L.p1z * o.n.y),
                                 fmaf(L.p1y, c2.z, L.p1z * o.n.z));
    const float3 c1 = make_float3(o.cp * o.ct, o.sp * o.ct, -o.st);
    o.p1 = make_float3(fmaf(L.p1x, c1.x, q.x), fmaf(L.p1x, c1.y, q.y), fmaf(L.p1x, c1.z, q.z));
    o.p2 = make_float3(fmaf(L.p1x, c1.x, -q.x), fmaf(L.p1x, c1.y, -q.y), fmaf(L.p1x, c1.z, -q.z));
    return o;
}

// Rotated offsets of one bead.
__device__ __forceinline__ void frame_vectors(float fi, float theta, float psi, const LatOffsets &L, float4 &n,
                                              float4 &a1, float4 &a2) {
    const Frame f = make_frame(fi, theta, psi, L);
    n = make_float4(f.n.x, f.n.y, f.n.z, 0.f);
    a1 = make_float4(f.p1.x, f.p1.y, f.p1.z, 0.f);
    a2 = make_float4(f.p2.x, f.p2.y, f.p2.z, 0.f);
}

// Gap g = dij + (a - b), dij = r_i - r_j (minimum image), and the gradient
// of |g|^2/2 with respect to bead i.  grad order: x, y, z, fi, theta, psi.
// uphi = (cp*ct, sp*ct, -st), uth = (-sp, cp, 0).
struct Grad { float g[6]; float dr, inv; };   // inv = 1/dr (0 when dr == 0)

__device__ __forceinline__ Grad gap_grad(float3 dij, float3 a, float3 b, float3 uphi, float2 uth) {
    Grad o;
    const float gx = dij.x + (a.x - b.x);
    const float gy = dij.y + (a.y - b.y);
    const float gz = dij.z + (a.z - b.z);
    const float t0 = a.y * gz - a.z * gy;
    const float t1 = a.z * gx - a.x * gz;
    const float t2 = a.x * gy - a.y * gx;
    o.g[0] = gx; o.g[1] = gy; o.g[2] = gz;
    o.g[3] = uphi.x * t0 + uphi.y * t1 + uphi.z * t2;
    o.g[4] = uth.x * t0 + uth.y * t1;
    o.g[5] = t2;
    const float d2 = gx * gx + gy * gy + gz * gz;
    o.inv = d2 > 0.f ? rsq_fast(d2) : 0.f;
    o.dr = d2 * o.inv;
    return o;
}

// src/compute_cuda.cu:16-30
__device__ __forceinline__ float morse_en(float D, float a, float x) {
    const float e = 1.f - __expf(-a * x);
    return D * e * e - D;
}
__device__ __forceinline__ float barr(float a, float r, float w, float x) {
    return a * __expf(-0.5f * (x - r) * (x - r) * rcp_fast(w * w));
}

// ---------------------------------------------------------------- HybridTaus
// GPU Gems 3, ch. 37 combined Tausworthe + LCG generator with the constants of
// src/HybridTaus.cu:72-82 and src/ht.cuh:8-10.
// One Tausworthe step z -> ((z & m) << S3) ^ (((z << S1) ^ z) >> S2): m clears
// the bits of z that S3 would leave in the low 32 - S2 bits, so the result is
// the high bits of z << S3 above the low ones of the other term, one funnel
// shift of (z >> (32 - S2 - S3), (z << S1) ^ z).  Four operations; two normals'
// draws of a wave take 714 cycles so, 791 with the two parts shifted and
// merged by a bit selection, 936 written out.
template <int S1, int S2, int S3, uint32_t M>
__device__ __forceinline__ uint32_t taus_step(uint32_t z) {
    constexpr int n = 32 - S2;   // bits from the second term
    static_assert(n > S3 && M == ~((1u << (n - S3)) - 1u), "the two terms meet at bit n");
    return __builtin_amdgcn_alignbit(z >> (n - S3), (z << S1) ^ z, S2);
}
// The four states' exclusive or, its low 23 bits as the mantissa of a float
// in [1, 2).
__device__ __forceinline__ float hybrid_taus(uint4 &s) {
    s.x = taus_step<13, 19, 12, 4294967294u>(s.x);
    s.y = taus_step<2, 25, 4, 4294967288u>(s.y);
    s.z = taus_step<3, 11, 17, 4294967280u>(s.z);
    s.w = 1664525u * s.w + 1013904223u;
    const uint32_t x = __builtin_amdgcn_bitop3_b32(s.x, s.y, s.z, 0x96) ^ s.w;   // 0x96: x ^ y ^ z
    // 0xE4: mask ? x : one
    return __uint_as_float(__builtin_amdgcn_bitop3_b32(x, in_vgpr(0x3f800000u), in_vgpr(0x007fffffu), 0xE4));
}
// Uniform in (0, 1): a zero, the only value below 1e-8, becomes 1e-8.
__device__ __forceinline__ float u01(uint4 &s) { return fmaxf(hybrid_taus(s) - 1.0f, 1.0e-8f); }
// Box-Muller radius sqrt(-2 ln u) = sqrt(-2 ln2 log2 u) from the hardware
// log2 and square root (1 ulp each).  u lies in [2^-23, 1) or is 1e-8, so
// both arguments are normal floats and need none of the denormal scaling and
// rounding fix-ups that logf and sqrtf expand to.
__device__ __forceinline__ float bm_radius(float u) {
    return __builtin_amdgcn_sqrtf(-1.38629436111989061883f * __builtin_amdgcn_logf(u));
}
// One draw of four normals (two Box-Muller pairs), advancing the state four
// times as src/HybridTaus.cu:85-98 does.  The angle 2 pi u goes to the
// hardware sine and cosine as it is, in revolutions: no product with 2 pi and
// its inverse and no range reduction.
__device__ __forceinline__ float4 normals4(uint4 &s) {
    float4 o;
    float r = bm_radius(u01(s));
    float u = u01(s);
    o.x = r * __builtin_amdgcn_sinf(u);
    o.y = r * __builtin_amdgcn_cosf(u);
    r = bm_radius(u01(s));
    u = u01(s);
    o.z = r * __builtin_amdgcn_sinf(u);
    o.w = r * __builtin_amdgcn_cosf(u);
    return o;
}

// Bead of this thread in a grid of 8 x nb8 workgroups (grid_xcd).  The
// dispatcher hands workgroup k to XCD k mod 8, so workgroup k takes the
// (k / 8)-th block of the (k mod 8)-th eighth of the beads: each XCD works
// on a contiguous eighth, whose trajectories' state then stays in that
// XCD's L2 while their neighbours are gathered.  The bead a thread computes
// does not change any result.
__device__ __forceinline__ int xcd_block() {
    return ((int)blockIdx.x & 7) * ((int)gridDim.x >> 3) + ((int)blockIdx.x >> 3);
}
__device__ __forceinline__ int xcd_bead(int bs) { return xcd_block() * bs + (int)threadIdx.x; }
// The grid of such a kernel over n items, bs to a workgroup: a multiple of 8.
inline int grid_xcd(int n, int bs) { return 8 * (((n + bs - 1) / bs + 7) / 8); }

// Constants of the force field and the integrator as the kernels use them,
// derived once on the host: per step and bead, quotients of the parameters
// (with the scaling and fix-ups a division expands to) would be taken anew.
struct ForceK {
    float C, Bpsi, Bfi, Bth;                 // spring; bending
    float psi_h, fi_h, th_gtp_h, th_gdp_h;   // bending offsets, halved (times r_mon = 2: exact)
    float lon_a, lon_d, lat_a, lat_d, seam_d;   // -A log2 e; 2 A D (lateral across the seam: over seam_coeff)
    float lonb_r, lonb_k, lonb_c, latb_r, latb_k, latb_c;   // barrier: r; -log2 e / (2 w^2); -a / w^2
    float lj6, lj_cap;                       // 6 scale sigma^6; gammaR r_mon / dt
    float wall_eps, wall_r, wall_left;
    float dtg, dta, dtt, vR, vta, vth;       // integrator: dt / gamma's, noise amplitudes
    float vF;                                // random force of the hydrodynamic steps: sqrt(2 kB T gammaR / dt)
    int barrier, lj_on, lj_reg, is_wall;
};
inline ForceK force_constants(const mte_params &P) {
    constexpr double LOG2E = 1.4426950408889634074;
    ForceK K{};
    K.C = P.C;
    K.Bpsi = P.B_psi, K.Bfi = P.B_fi, K.Bth = P.B_theta;
    K.psi_h = 0.5f * P.psi_0, K.fi_h = 0.5f * P.fi_0, K.th_gtp_h = 0.5f * P.theta0_gtp, K.th_gdp_h = 0.5f * P.theta0_gdp;
    K.lon_a = (float)(-P.A_long * LOG2E), K.lat_a = (float)(-P.A_lat * LOG2E);
    K.lon_d = 2.f * P.A_long * P.D_long, K.lat_d = 2.f * P.A_lat * P.D_lat;
    K.seam_d = (float)(2.0 * P.A_lat * P.D_lat / P.seam_coeff);
    const double wl = (double)P.w_barr_long * P.w_barr_long, wt = (double)P.w_barr_lat * P.w_barr_lat;
    K.lonb_r = P.r_barr_long, K.latb_r = P.r_barr_lat;
    K.lonb_k = (float)(-0.5 * LOG2E / wl), K.latb_k = (float)(-0.5 * LOG2E / wt);
    K.lonb_c = (float)(-P.a_barr_long / wl), K.latb_c = (float)(-P.a_barr_lat / wt);
    K.lj6 = 6.f * (P.ljscale * P.ljsigma6);
    K.lj_cap = P.gammaR * 2.f / P.dt;
    K.wall_eps = P.rep_eps, K.wall_r = P.rep_r, K.wall_left = P.rep_leftborder;
    K.dtg = P.dt / P.gammaR;
    K.dta = P.dt / (P.gammaTheta * P.alpha);
    K.dtt = P.dt / P.gammaTheta;
    K.vR = P.varR;
    K.vta = P.varTheta * sqrtf(P.freeze_temp / P.alpha);
    K.vth = P.varTheta;
    K.vF = sqrtf(2.0f * KB * P.temp * P.gammaR / P.dt);
    K.barrier = P.barrier, K.lj_on = P.lj_on, K.lj_reg = P.lj_regularize, K.is_wall = P.is_wall;
    return K;
}

// Euler-Maruyama update of the angles, src/compute_cuda.cu:958-961.  The
// increment is summed first: one rounding at the angle's own magnitude.
__device__ __forceinline__ void em_angles(const ForceK &K, float ffi, float fth, float fpsi, float4 ra, float4 &a) {
    a.x += fmaf(K.dta, ffi, K.vta * ra.x);    // fi
    a.z += fmaf(K.dta, fpsi, K.vta * ra.y);   // psi
    a.y += fmaf(K.dtt, fth, K.vth * ra.z);    // theta
}
}  // namespace mte
