// tea.hip -- TEA hydrodynamic interactions (Geyer & Winter 2009) on gfx950.
//
// Restates src/bdhitea_kernel.cu:16-213 and the host FP64 normalisation of
// src/bdhitea.cu:57-118, with the normalisation moved on device in FP64:
//   per bead  ci_i = sum_j rowwise (D_hat_ij)^2, eps_i = sum_j sum(D_hat_ij)
//   per traj  eps = sum_i eps_i / (3N(3N-3)), a = (3N-1)eps^2 - (3N-2)eps,
//             beta = (1 - sqrt(1-a))/a  (0.5 when |a| < 1e-7)
//   per bead  C_i = 1/sqrt(1 + beta^2 ci_i),
//             f_i = F_i + C_i.R_i + sum_{j!=i} D_hat_ij (F_j + beta C_i.R_j),
//             r_i += dt/gammaR f_i
// with D_hat_ij = D_ij/D_ii the Rotne-Prager-Yamakawa block, N the count of
// non-extra beads of the trajectory.
//
// The per-step product has three forms (mte_tuning.tea_chunk), the first two
// bound by VALU issue:
//   one-sided  work units of (trajectory, 256-bead i group, j chunk of 64, 128
//              or 256 beads), each block evaluated for i (pair_chunk);
//   symmetric  each block evaluated once for both beads, units of a pair of
//              64-bead chunks against a run of chunks (pair_unit);
//   moments    products of tabulated moments on the matrix cores
//              (k_tea_pairs_mfma).
// Their FP32 partial sums are added in a fixed order by the kernel that ends
// the step (k_tea_finish; k_tea_turn, which also forms the next forces), with
// the self term, and integrated.
#include "bead_physics.h"
#include "engine_internal.h"
#include <type_traits>

namespace mte {

constexpr int TEA_TILE = 256;

struct RpyCoef { float crr, cii; };

// RPY coefficients of D_hat = cii I + crr e e^T at r^2 (rinv = 1/r), both
// branches of src/bdhitea_kernel.cu:38-58 evaluated and selected (no
// divergence); ia = 1/a.
__device__ __forceinline__ RpyCoef rpy_select(float r2, float rinv, float a, float ia) {
    const float u1 = a * rinv, u2 = u1 * u1;
    const float ra = r2 * rinv * ia;
    const bool near = !(ra > 2.f);
    RpyCoef c;
    c.cii = near ? fmaf(-0.28125f, ra, 1.f) : 0.75f * u1 * fmaf(0.66666666666666667f, u2, 1.f);
    c.crr = near ? 0.09375f * ra : 0.75f * u1 * fmaf(-2.f, u2, 1.f);
    return c;
}

// Lane l of the wave receives lane (l + 1) mod 64's value (all lanes active).
__device__ __forceinline__ float wave_rol1(float v) {
    const int x = __float_as_int(v);
    return __int_as_float(__builtin_amdgcn_update_dpp(x, x, 0x134, 0xF, 0xF, false));
}

// How the pair loops take a pair's nearest image: not at all (open), by
// coordinates that are 32-bit integers of box / 2^32, whose difference wraps
// by itself, or in float from nm.  The integers cost 18 issue cycles a pair,
// the float image 30, but their quantum grows with the box, where the float
// difference of two near beads is exact: a tube of 312 beads at the origin
// moves in one step with an error (FP64, of the largest move) of 3-5e-7 by
// either in boxes up to 4096 nm (2^-20 nm, a quarter of the rounding of a
// coordinate there), by the integers with 5e-6 at 1e5 and 4e-5 at 1e6 nm.
enum PairBox { OPEN_BOX, INT_BOX, FLOAT_BOX };
constexpr float INT_BOX_MAX = 4096.f;
// A batch's kernels are made for one of them: open batches, those whose boxes
// are all within INT_BOX_MAX (an open trajectory among them is taken as such),
// and the rest (there a float image with a box of 0 changes nothing).
constexpr PairBox unboxed(PairBox b) { return b == FLOAT_BOX ? FLOAT_BOX : OPEN_BOX; }
static PairBox batch_box(const mte_engine *e) {
    return !e->periodic ? OPEN_BOX : e->box_max <= INT_BOX_MAX ? INT_BOX : FLOAT_BOX;
}

// One coordinate of the pair loops: x itself, or (INT_BOX) its place in the
// periodic box as a 32-bit integer (bit pattern), taken modulo the box in FP64.
template <PairBox BOX>
__device__ __forceinline__ float pair_coord(float x, double ibox) {
    if (BOX != INT_BOX) return x;
    double v = (double)x * ibox;
    v -= rint(v);
    // 1.5 2^52 leaves the rounded integer in the low mantissa word
    return __int_as_float(__double2loint(fma(v, 4294967296.0, 6755399441055744.0)));
}
// Integer places apart, wrapped to the nearest image: the subtraction is
// unsigned, where wrapping is defined (a signed one does not compile in the
// constant expression below).
__host__ __device__ constexpr int wrap_diff(uint32_t a, uint32_t b) { return (int)(a - b); }
static_assert(wrap_diff(0x7fffffffu, 0x80000000u) == -1 && wrap_diff(0x80000000u, 0x7fffffffu) == 1 &&
                  wrap_diff(0u, 0x80000000u) == INT32_MIN && wrap_diff(5u, 7u) == -2,
              "differences across the faces of the box wrap");
// side, iside: the box and its inverse (FLOAT_BOX; both 0 on open boundaries).
template <PairBox BOX>
__device__ __forceinline__ float pair_diff(float a, float b, float side, float iside) {
    if (BOX == INT_BOX) return (float)wrap_diff(__float_as_uint(a), __float_as_uint(b));
    const float d = a - b;
    return BOX == FLOAT_BOX ? d - side * rintf(d * iside) : d;
}

// Epsilon partials and ci of bead i over all j of its trajectory
// (integrateTea_epsilon_unlisted, src/bdhitea_kernel.cu:61-101), with the
// block sums in closed form (|e| = 1):
//   sum of the 9 entries of D_hat      = 3 cii + crr (ex + ey + ez)^2
//   row a sum of squares               = cii^2 + crr (2 cii + crr) e_a^2
// Extra beads enter with weight 0; the j == i slot (d = 0, its distance
// clamped finite) is taken out after the loop, so no branch sits in the pair
// loop.  PERIODIC: some trajectory has a periodic box.
template <bool PERIODIC>
__global__ void __launch_bounds__(TEA_TILE)
    k_tea_eps(mte_params P, DevTopo T, DevState S, const int2 *tiles, float4 *ci, float *eps) {
    __shared__ float4 sx[TEA_TILE];
    const int2 tl = tiles[blockIdx.x];
    const int base = T.tbase[tl.x], n = T.tsize[tl.x];
    const int li = tl.y + threadIdx.x;
    const bool active = li < n;
    const int b = base + li;
    float3 ri = make_float3(0, 0, 0);
    bool skip = true;
    if (active) {
        ri = f3(S.xyz[b]);
        skip = T.extra[b] != 0;
    }
    const float box = T.tbox[tl.x], ibox = inv_side(box);
    const float a = P.tea_a, ia = rcp_fast(P.tea_a);
    float scc = 0.f, sx2 = 0.f, sy2 = 0.f, sz2 = 0.f, sall = 0.f;
    for (int j0 = 0; j0 < n; j0 += TEA_TILE) {
        const int jl = j0 + threadIdx.x;
        if (jl < n) {
            float4 v = S.xyz[base + jl];
            v.w = T.extra[base + jl] ? 0.f : 1.f;
            sx[threadIdx.x] = v;
        }
        __syncthreads();
        const int m = min(TEA_TILE, n - j0);
        if (active && !skip) {
            // not unrolled: measured faster than unrolled by 2 or 4
#pragma unroll 1
            for (int jj = 0; jj < m; jj++) {
                const float4 xj = sx[jj];
                float3 d = sub3(f3(xj), ri);
                if (PERIODIC) d = min_image_inv(d, box, ibox);
                const float wj = xj.w;
                const float r2 = fmaxf(d.x * d.x + d.y * d.y + d.z * d.z, 1e-12f);
                const float rinv = rsq_fast(r2);
                const RpyCoef c = rpy_select(r2, rinv, a, ia);
                const float ex = d.x * rinv, ey = d.y * rinv, ez = d.z * rinv;
                const float cw = wj * c.cii;
                const float k = wj * c.crr * fmaf(2.f, c.cii, c.crr);
                const float se = ex + ey + ez;
                scc = fmaf(cw, c.cii, scc);
                sx2 = fmaf(k, ex * ex, sx2);
                sy2 = fmaf(k, ey * ey, sy2);
                sz2 = fmaf(k, ez * ez, sz2);
                sall += fmaf(wj * c.crr, se * se, 3.f * cw);
            }
        }
        __syncthreads();
    }
    if (active && !skip) {
        // the j == i slot entered as a coincident bead of weight 1 (d = 0):
        // cii^2 into scc and 3 cii into sall, recomputed and taken out
        const float r2 = 1e-12f, rinv = rsq_fast(r2);
        const float cii = rpy_select(r2, rinv, a, ia).cii;
        scc = fmaf(-cii, cii, scc);
        sall = fmaf(-3.f, cii, sall);
    }
    if (active) {
        ci[b] = make_float4(scc + sx2, scc + sy2, scc + sz2, 0.f);
        eps[b] = sall;
    }
}

// Epsilon partials and ci with each pair evaluated once.  The five sums of
// k_tea_eps are even in e (cii^2, crr (2 cii + crr) e_a^2, 3 cii + crr
// (ex + ey + ez)^2), so a pair adds the same terms to both beads.  Work unit:
// (trajectory, group I of WAVES x PER chunks of 64 beads, group J >= I), one
// workgroup of WAVES waves; wave w takes chunks c = WAVES (PER I + h) + w,
// h < PER (one bead of each per lane) against each chunk c_J of group J in
// turn, staged in LDS:
//   c_J > c    both sides, lane l meeting j = (l + s) mod 64 at step s, the
//              j-side sums carried along by a one-lane rotation (wave_rol1);
//              when c_J lies above all of the wave's chunks, the lane's
//              beads meet the same j together and share the rotation,
//   c_J = c    one-sided over the chunk, the j == i term at weight 0,
//   c_J < c    nothing (that pair of chunks is the wave c_J's).
// The waves' j-side sums of a chunk are added in wave order in LDS.  Output
// (deterministic, no atomics): i-side sums of a bead of group H into
// part[0][J][.] for J >= H, j-side sums into part[1][I][.] for I <= H.  A pair
// counts for two non-extra beads (WEIGHTED: some bead of the batch is extra)
// inside the trajectory: the weight, 0 or 1, multiplies 1 / r, of which every
// far term holds a power, and the near terms themselves.
//
// With v = 1 / r^2, u = a / r (far branch) the terms are
//   cii^2   = 9/16 a^2  v A^2            A = 1 + 2/3 a^2 v
//   k e_x^2 = 9/16 a^2  v^2 B E  d_x^2   B = 1 - 2 a^2 v, E = 3 - 2/3 a^2 v
//   3 cii + crr (e_x + e_y + e_z)^2 = 3/4 a  (1 / r) (3 A + B v (d_x + d_y + d_z)^2)
// so the loop sums them without their constant factors and forms no unit
// vector; lengths and minimum images are those of the pair kernel below.
// Bound: VALU issue, 38 operations per pair and 64 lanes in a box, of them 32
// FP32 adds and products, at a clock that falls to 2.2 GHz under them; four or
// two chunks per wave, 4 or 6 waves per SIMD, take the same time.  Measured,
// against unit vectors, per-pair constant factors and float minimum images:
// eight periodic trajectories of 24k-40k beads (4.2e9 pairs) 4.48 -> 3.81 ms,
// 64 x 1040 beads 351 -> 75 us (with the smaller groups, tea_build_eps_units).
// Waves of a workgroup whose waves take `per` chunks.
constexpr int eps_waves(int per) { return per == 1 ? 4 : EPS_GROUP_MAX / 64 / per; }
// What a pair's terms need beside the beads, in loop units.
struct EpsCoef {
    float c1, c2, c3, c4;       // a^2 times 2/3, -2, -2/3, 2
    float near2, ia, r2min;     // (2a)^2 with its margin, 1 / a, the floor of r^2
    float i0, i4;               // 1 / (9/16 a^2), 1 / (3/4 a)
    float side, iside;          // FLOAT_BOX: the box
};

// One pair's five terms: added to the sums t and, unless ONE_SIDE, to t2,
// which takes the next lane's t2 first when SIDES is ROTATE (the j-side
// rotation, done with the first of the lane's beads to meet this j).  WT: the
// pair's weight ww is formed.
enum EpsSides { ONE_SIDE, BOTH_SIDES, ROTATE };
template <PairBox BOX, bool WT, EpsSides SIDES>
__device__ __forceinline__ void eps_pair(const EpsCoef &K, float3 xa, float wa, float4 xj, float (&t)[5],
                                         float (&t2)[5]) {
    const float dx = pair_diff<BOX>(xj.x, xa.x, K.side, K.iside), dy = pair_diff<BOX>(xj.y, xa.y, K.side, K.iside), dz = pair_diff<BOX>(xj.z, xa.z, K.side, K.iside);
    // r2min (1e-12 nm^2) keeps coincident beads finite and is below the
    // rounding of any other r^2
    const float qx = dx * dx, qy = dy * dy, qz = fmaf(dz, dz, K.r2min);
    const float r2 = (qx + qy) + qz;
    const float ww = WT ? wa * xj.w : 1.f;
    float rinv = rsq_fast(r2);
    if (WT) rinv *= ww;
    const float v = rinv * rinv;
    const float A = fmaf(K.c1, v, 1.f), B = fmaf(K.c2, v, 1.f);
    const float Bv = B * v, sd = (dx + dy) + dz;
    float m = v * A, mA = A;                                             // cii^2 = m mA
    float kk = Bv * (v * fmaf(K.c3, v, 3.f));                            // crr (2 cii + crr) / r^2
    float h = rinv, hA = fmaf(Bv, sd * sd, fmaf(K.c4, v, 3.f));          // 3 cii + crr se^2 = h hA
    if (__any(r2 <= K.near2)) {
        __asm__ volatile("");   // a branch: the near form is not evaluated otherwise
        const float rn = rsq_fast(r2), ra = r2 * rn * K.ia;
        const bool nr = !(ra > 2.f);
        const float cii = fmaf(-0.28125f, ra, 1.f), crr = 0.09375f * ra, vn = rn * rn;
        m = nr ? ww * K.i0 * cii : m;
        mA = nr ? cii : mA;
        kk = nr ? ww * K.i0 * crr * fmaf(2.f, cii, crr) * vn : kk;
        h = nr ? ww * K.i4 : h;
        hA = nr ? fmaf(crr * vn, sd * sd, 3.f * cii) : hA;
    }
    t[0] = fmaf(m, mA, t[0]);
    t[1] = fmaf(kk, qx, t[1]);
    t[2] = fmaf(kk, qy, t[2]);
    t[3] = fmaf(kk, qz, t[3]);
    t[4] = fmaf(h, hA, t[4]);
    if (SIDES != ONE_SIDE) {
        constexpr bool ROT = SIDES == ROTATE;
        t2[0] = fmaf(m, mA, ROT ? wave_rol1(t2[0]) : t2[0]);
        t2[1] = fmaf(kk, qx, ROT ? wave_rol1(t2[1]) : t2[1]);
        t2[2] = fmaf(kk, qy, ROT ? wave_rol1(t2[2]) : t2[2]);
        t2[3] = fmaf(kk, qz, ROT ? wave_rol1(t2[3]) : t2[3]);
        t2[4] = fmaf(h, hA, ROT ? wave_rol1(t2[4]) : t2[4]);
    }
}

// The lane's N beads against every j of the staged chunk, both sides.
template <PairBox BOX, bool WT, int N>
__device__ __forceinline__ void eps_sweep(const EpsCoef &K, const float4 *jl, const float3 *xi, const float *wi,
                                          float (*ai)[5], float (&gj)[5]) {
#pragma unroll 1
    for (int s = 0; s < 64; s++) {
        const float4 xj = jl[s];
        eps_pair<BOX, WT, ROTATE>(K, xi[0], wi[0], xj, ai[0], gj);
#pragma unroll
        for (int h = 1; h < N; h++) eps_pair<BOX, WT, BOTH_SIDES>(K, xi[h], wi[h], xj, ai[h], gj);
    }
}

template <PairBox BOX, bool WEIGHTED, int PER>
__device__ __forceinline__ void eps_unit(const mte_params &P, const DevTopo &T, const DevState &S, int4 u, int ngrp,
                                         float *part, float4 *jx, float (*jred)[5][64]) {
    constexpr int WAVES = eps_waves(PER), CHUNKS = WAVES * PER;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), l = threadIdx.x % 64;
    const int base = T.tbase[u.x], n = T.tsize[u.x], nb = T.nb;
    const int nch = (n + 63) / 64;
    const float box = T.tbox[u.x];
    const double ibox = BOX == INT_BOX ? 1.0 / (double)box : 0.0;
    const float sc = BOX == INT_BOX ? box * 0x1p-32f : 1.f;   // nm per loop unit
    const float a = P.tea_a / sc, s2 = a * a, lim = 2.002f * a;
    EpsCoef K;
    K.c1 = in_vgpr(0.66666666666666667f * s2);
    K.c2 = in_vgpr(-2.f * s2);
    K.c3 = in_vgpr(-0.66666666666666667f * s2);
    K.c4 = in_vgpr(2.f * s2);
    K.near2 = in_vgpr(lim * lim);
    K.ia = sc * rcp_fast(P.tea_a);
    K.r2min = in_vgpr(1e-12f / (sc * sc));
    K.i0 = 1.f / (0.5625f * s2);
    K.i4 = 1.f / (0.75f * a);
    K.side = in_vgpr(box);
    K.iside = in_vgpr(inv_side(box));
    // the lane's bead in each of the wave's chunks
    int cI[PER];
    bool vi[PER];
    float3 xi[PER];
    float wi[PER], ai[PER][5];
    auto bead = [&](int li, float &wt) {
        wt = 0.f;
        if (li >= n) return make_float3(0.f, 0.f, 0.f);
        const float3 x = f3(S.xyz[base + li]);
        // a lost position (inf, NaN), which an integer cannot hold, spreads
        // through the bead's weight as it would through r
        const float lost = BOX == INT_BOX ? (x.x - x.x) + (x.y - x.y) + (x.z - x.z) : 0.f;
        wt = (T.extra[base + li] ? 0.f : 1.f) + lost;
        return make_float3(pair_coord<BOX>(x.x, ibox), pair_coord<BOX>(x.y, ibox), pair_coord<BOX>(x.z, ibox));
    };
    bool odd = false;   // a lost bead among the lane's own
#pragma unroll
    for (int h = 0; h < PER; h++) {
        cI[h] = u.y * CHUNKS + w + h * WAVES;
        vi[h] = cI[h] * 64 + l < n;
        xi[h] = bead(cI[h] * 64 + l, wi[h]);
        odd |= !(fabsf(wi[h]) <= 1.f);
#pragma unroll
        for (int k = 0; k < 5; k++) ai[h][k] = 0.f;
    }
    const bool wto = WEIGHTED || __any(odd);
    const int c0 = u.z * CHUNKS, c1 = min(c0 + CHUNKS, nch);
    float wj = 0.f;
    for (int cJ = c0; cJ < c1; cJ++) {
        if (threadIdx.x < 128) {
            const float3 x = bead(cJ * 64 + l, wj);
            jx[threadIdx.x] = make_float4(x.x, x.y, x.z, wj);
        }
        __syncthreads();
        const float4 *jl = jx + l;
        float gj[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
        // step s of a both-sided sweep: lane l meets j = (l + s) mod 64, its
        // gj the sums of that j (rotated in from lane l + 1, which held j at
        // the sweep's step s - 1; sweeps in a row continue the rotation).
        // A chunk below c_J is full; c_J may be the padded last one, and its
        // weights are formed there, or where a bead of it is lost.
        const bool wtj = wto || (cJ + 1) * 64 > n || __any(!(fabsf(jx[l].w) <= 1.f));
        int low = 0;   // the wave's chunks below c_J: the first `low`
#pragma unroll
        for (int h = 0; h < PER; h++) low += cI[h] < nch && cJ > cI[h] ? 1 : 0;
        if (low == PER) {
            if (wtj) eps_sweep<BOX, true, PER>(K, jl, xi, wi, ai, gj);
            else eps_sweep<BOX, false, PER>(K, jl, xi, wi, ai, gj);
        } else if (PER > 1) {
#pragma unroll
            for (int h = 0; h < PER; h++)
                if (h < low) eps_sweep<BOX, true, 1>(K, jl, xi + h, wi + h, ai + h, gj);
        }
#pragma unroll
        for (int h = 0; h < PER; h++)
            if (cI[h] < nch && cJ == cI[h]) {
                // one-sided over the chunk's beads, the bead itself (q == l)
                // at weight 0: what a coincident bead of weight 1 adds, taken
                // out afterwards, outgrows the sums where a is small
                const int jn = min(64, n - cJ * 64);
#pragma unroll 1
                for (int q = 0; q < jn; q++)
                    eps_pair<BOX, true, ONE_SIDE>(K, xi[h], q == l ? 0.f : wi[h], jx[q], ai[h], gj);
            }
        // after a multiple of 64 rotations lane l holds the sums of j =
        // (l + 63) mod 64; with none, gj is zero
#pragma unroll
        for (int k = 0; k < 5; k++) jred[w][k][(l + 63) & 63] = gj[k];
        __syncthreads();
        for (int e = threadIdx.x; e < 5 * 64; e += 64 * WAVES) {
            const int k = e / 64, q = e % 64;
            const int lj = cJ * 64 + q;
            if (lj < n) {
                float sum = 0.f;
                for (int v = 0; v < WAVES; v++) sum += jred[v][k][q];
                part[(((size_t)1 * ngrp + u.y) * 5 + k) * nb + base + lj] = sum * (k < 4 ? 0.5625f * s2 : 0.75f * a);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int h = 0; h < PER; h++)
        if (vi[h]) {
#pragma unroll
            for (int k = 0; k < 5; k++)
                part[(((size_t)0 * ngrp + u.z) * 5 + k) * nb + base + cI[h] * 64 + l] =
                    ai[h][k] * (k < 4 ? 0.5625f * s2 : 0.75f * a);
        }
}

template <PairBox BOX, bool WEIGHTED, int PER>
__global__ void __launch_bounds__(64 * eps_waves(PER))
    k_tea_eps_sym(mte_params P, DevTopo T, DevState S, const int4 *units, int ngrp, float *part) {
    __shared__ float4 jx[2 * 64];              // chunk c_J: x, weight; twice, no wrap
    __shared__ float jred[eps_waves(PER)][5][64];   // j-side sums of each wave
    const int4 u = units[blockIdx.x];
    if (BOX == INT_BOX && T.tbox[u.x] > 0.f) eps_unit<INT_BOX, WEIGHTED, PER>(P, T, S, u, ngrp, part, jx, jred);
    else eps_unit<unboxed(BOX), WEIGHTED, PER>(P, T, S, u, ngrp, part, jx, jred);
}

// Per bead: the group sums of k_tea_eps_sym added in fixed order into ci and
// eps, as k_tea_eps writes them.
__global__ void __launch_bounds__(256)
    k_tea_eps_reduce(DevTopo T, int group, int ngrp, const float *part, float4 *ci, float *eps) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= T.nb) return;
    const int t = T.tid[b], n = T.tsize[t];
    const int h = (b - T.tbase[t]) / group, g = (n + group - 1) / group;
    const int nb = T.nb;
    // each of the five sums in the same order (groups h..g-1 of side 0, then
    // 0..h of side 1), the five advancing together so their loads overlap
    float s[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
    for (int j = h; j < g; j++) {
        float v[5];
#pragma unroll
        for (int k = 0; k < 5; k++) v[k] = part[(((size_t)0 * ngrp + j) * 5 + k) * nb + b];
#pragma unroll
        for (int k = 0; k < 5; k++) s[k] += v[k];
    }
    for (int i = 0; i <= h; i++) {
        float v[5];
#pragma unroll
        for (int k = 0; k < 5; k++) v[k] = part[(((size_t)1 * ngrp + i) * 5 + k) * nb + b];
#pragma unroll
        for (int k = 0; k < 5; k++) s[k] += v[k];
    }
    ci[b] = make_float4(s[0] + s[1], s[0] + s[2], s[0] + s[3], 0.f);
    eps[b] = s[4];
}

// FP64 epsilon / beta per trajectory, one workgroup each; then beta C of its
// beads.
__global__ void __launch_bounds__(256)
    k_tea_beta(mte_params P, DevTopo T, const float *eps, const float4 *ci, float *beta, float4 *bc, double *stats,
               int *status) {
    __shared__ double red[256];
    __shared__ int cnt[256];
    const int t = blockIdx.x;
    const int base = T.tbase[t], n = T.tsize[t];
    double s = 0.0;
    int c = 0;
    for (int i = threadIdx.x; i < n; i += 256) {
        s += (double)eps[base + i];
        c += T.extra[base + i] ? 0 : 1;
    }
    red[threadIdx.x] = s;
    cnt[threadIdx.x] = c;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) {
            red[threadIdx.x] += red[threadIdx.x + k];
            cnt[threadIdx.x] += cnt[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double nn = (double)cnt[0];
        // A trajectory of one bead (the rest extra) has no tensor to average or
        // to check: epsilon 0 and its beta, 0.5, where 0 / 0 would lose the bead.
        const bool alone = cnt[0] < 2;
        double e = alone ? 0.0 : red[0] / (3. * nn * (3. * nn - 3.));
        int fail = 0;
        if (e > 1.0) {
            if (P.tea_capricious) fail = 1;
            e = 1.0;
        }
        if (e > (double)P.tea_epsmax) fail = 1;
        const double a = (3. * nn - 1.) * e * e - (3. * nn - 2.) * e;
        double bt;
        if (fabs(a) < 1e-7) {
            bt = 0.5;
            if (P.tea_capricious && P.tea_a > 0.0f && !alone) fail = 1;
        } else {
            bt = (1. - sqrt(1. - a)) / a;
        }
        beta[t] = (float)bt;
        stats[2 * t] = e;
        stats[2 * t + 1] = (double)(float)bt;
        if (fail) atomicCAS(status, 0, 1 + t);
        red[0] = bt;
    }
    __syncthreads();
    // beta C_i = beta / sqrt(1 + beta^2 ci) (eq. 19), which the steps until
    // the next refresh read
    const float bt = (float)red[0], w = bt * bt;
    for (int i = threadIdx.x; i < n; i += 256) {
        const float4 c = ci[base + i];
        bc[base + i] = make_float4(bt * rsq_fast(1.f + w * c.x), bt * rsq_fast(1.f + w * c.y),
                                   bt * rsq_fast(1.f + w * c.z), 0.f);
    }
}

// Pair sums with each (i, j) RPY block evaluated once for both beads.  Work
// unit: (trajectory, I pair p: the 64-bead chunks 2p and 2p + 1, chunks J of a
// range at or above 2p).  D_hat_ji = D_hat_ij, so a block serves
//   i-side  D_hat_ij (F_j + beta C_i . R_j)  into acc of bead i,
//   j-side  D_hat_ij (F_i + beta C_j . R_i)  into g, carried with j.
// Lane l holds bead l of both I chunks and meets j = (l + s) mod 64 of J at
// step s, so no two lanes meet the same j in a step; after each step g moves
// one lane down (DPP wave_rol:1), so it sits in the lane that meets j next.
//   J > 2p + 1  both I chunks, 64 steps, their j-side sums in one g;
//   J = 2p + 1  chunk 2p against J, and J against itself;
//   J = 2p      the chunk against itself: steps 1 .. 31 meet every pair of it
//               but the opposite ones once, both sides; step 32 meets those
//               from both ends and takes the i-side only.  No bead meets
//               itself.
// Partials (12 bytes per bead, planes of x, y, z): slot p of a j bead holds
// its sum over I pair p, slot ioff + J0 / jrun of an i bead its sum over the
// unit's J range, each written by exactly one unit (k_tea_finish adds them
// in slot order).  Beads past the trajectory's end and extra beads carry
// zero F and R, so their terms vanish.
//
// Lengths in the loop are nm on open boundaries and in large boxes (PairBox).
// In other periodic boxes they are units of box / 2^32 and positions 32-bit
// integers, so a difference wraps to the minimum image by itself: 3
// subtractions and 3 conversions (18 issue cycles) instead of subtract, scale,
// round, fused subtract (30).
// The coefficients are those beyond 2a; a wave with a pair inside 2a (margin
// over the rounding of r / a) selects the near ones in a branch.
//
// SPLIT waves share a unit, each taking its part of the steps, and add their
// sums in wave order (small batches, tea_build_units).
// Bound: VALU issue, 45 operations per pair and 64 lanes: 98 issue cycles open
// and 110 in a box (of them 8 for the reciprocal square root, 4 for the near
// test, 6 for moving g); the constants sit in vector registers because an FP32
// operation with a scalar operand takes 4 cycles and not 2.
// Measured, against the same pairs with float minimum images, near and far
// coefficients selected per pair, scalar constants, one J chunk per unit and
// one slot per chunk: four periodic trajectories of 24k-37k beads 2.20 ->
// 1.71 ms (89% of the issue rate at the 2.07 GHz that the chip holds here) and
// the finish kernel 206 -> 57 us; 64 x 1040 beads 53.5 -> 44.3 us (a third of
// it ramp and tail); one trajectory of 312 beads 18.4 -> 5.8 us.
constexpr int SYM_CHUNK = 64;
// What a pair's evaluation needs beside the beads.
struct PairCoef {
    float k1, k3, k5;       // cii = k1 w + k3 w^3, crr / r^2 = w^3 (k1 + k5 w^2), w = 1 / r in loop units
    float near2, ia, r2min; // (2a)^2 with its margin, 1 / a, the clamp of coincident beads
    float side, iside;      // FLOAT_BOX: the box
};
struct PairBead {
    float3 x, F, R, C;      // position (loop units), force, random force, beta C
};
template <PairBox BOX>
__device__ __forceinline__ PairCoef pair_coef(const mte_params &P, float box) {
    const float sc = BOX == INT_BOX ? box * 0x1p-32f : 1.f;   // nm per loop unit
    const float a = P.tea_a / sc, a1 = fmaxf(P.tea_a, 1e-15f);
    // Coincident beads are taken apart to 1e-6 nm, or to a where that is less:
    // they are near ones (r <= 2a) for every radius, 0 among them, where the
    // far coefficients are infinite or undefined.
    const float am = a1 / sc, lim = 2.002f * am;
    PairCoef K;
    K.k1 = in_vgpr(0.75f * a);
    K.k3 = in_vgpr(0.5f * a * a * a);
    K.k5 = in_vgpr(-1.5f * a * a * a);
    K.near2 = in_vgpr(lim * lim);
    K.ia = sc * rcp_fast(a1);
    K.r2min = fminf(1e-12f / (sc * sc), am * am);
    K.side = in_vgpr(box);
    K.iside = in_vgpr(inv_side(box));
    return K;
}

// Bead b (zeros where it is not valid); extra beads have zero F and R.
template <PairBox BOX>
__device__ __forceinline__ PairBead pair_bead(const float4 *xyz, const float4 *fxyz, const float4 *R, const float4 *bc,
                                              int b, bool valid, double ibox) {
    PairBead v;
    v.x = v.F = v.R = v.C = make_float3(0.f, 0.f, 0.f);
    if (valid) {
        const float3 x = f3(xyz[b]), F = f3(fxyz[b]);
        v.x = make_float3(pair_coord<BOX>(x.x, ibox), pair_coord<BOX>(x.y, ibox), pair_coord<BOX>(x.z, ibox));
        // zero for a finite position; a lost one (inf, NaN), which an
        // integer cannot hold, spreads through F as it would through r
        const float lost = BOX == INT_BOX ? (x.x - x.x) + (x.y - x.y) + (x.z - x.z) : 0.f;
        v.F = make_float3(F.x + lost, F.y + lost, F.z + lost);
        v.R = f3(R[b]);
        v.C = f3(bc[b]);
    }
    return v;
}

// Bead I against the j of (A, B, Cq): i-side into acc, and j-side into g
// (BOTH).
template <PairBox BOX, bool BOTH>
__device__ __forceinline__ void pair_block(const PairCoef &K, const PairBead &I, float4 A, float4 B, float4 Cq,
                                           float3 &acc, float3 &g) {
    const float dx = pair_diff<BOX>(A.x, I.x.x, K.side, K.iside), dy = pair_diff<BOX>(A.y, I.x.y, K.side, K.iside), dz = pair_diff<BOX>(A.z, I.x.z, K.side, K.iside);
    const float r2 = dx * dx + dy * dy + dz * dz;
    const float w = rsq_fast(r2);
    const float w2 = w * w;
    float cii = w * fmaf(K.k3, w2, K.k1);
    float cr = (w * w2) * fmaf(K.k5, w2, K.k1);
    if (__any(r2 <= K.near2)) {
        __asm__ volatile("");   // a branch: the near form is not evaluated otherwise
        const float r2c = fmaxf(r2, K.r2min), wc = rsq_fast(r2c);
        const float ra = r2c * wc * K.ia;
        const bool nr = !(ra > 2.f);
        cii = nr ? fmaf(-0.28125f, ra, 1.f) : cii;
        cr = nr ? 0.09375f * ra * wc * wc : cr;
    }
    // i-side: F_j + beta C_i . R_j
    const float vx = fmaf(I.C.x, B.z, A.w), vy = fmaf(I.C.y, B.w, B.x), vz = fmaf(I.C.z, Cq.x, B.y);
    const float sv = cr * fmaf(dz, vz, fmaf(dy, vy, dx * vx));
    acc.x = fmaf(sv, dx, fmaf(cii, vx, acc.x));
    acc.y = fmaf(sv, dy, fmaf(cii, vy, acc.y));
    acc.z = fmaf(sv, dz, fmaf(cii, vz, acc.z));
    if (BOTH) {
        // j-side: F_i + beta C_j . R_i (e e^T is even in e)
        const float wx = fmaf(Cq.y, I.R.x, I.F.x), wy = fmaf(Cq.z, I.R.y, I.F.y), wz = fmaf(Cq.w, I.R.z, I.F.z);
        const float sw = cr * fmaf(dz, wz, fmaf(dy, wy, dx * wx));
        g.x = fmaf(sw, dx, fmaf(cii, wx, g.x));
        g.y = fmaf(sw, dy, fmaf(cii, wy, g.y));
        g.z = fmaf(sw, dz, fmaf(cii, wz, g.z));
    }
}

__device__ __forceinline__ void rotate(float3 &g) {
    g.x = wave_rol1(g.x);
    g.y = wave_rol1(g.y);
    g.z = wave_rol1(g.z);
}

template <PairBox BOX, int SPLIT>
__device__ __forceinline__ void pair_unit(const mte_params &P, const PairUnit &U, int nb, const float4 *xyz,
                                          const float4 *fxyz, const float4 *R, const float4 *bc, int jrun, int ioff,
                                          float *partial, float4 (*jd)[2 * SYM_CHUNK],
                                          float (*red)[9][SPLIT == 1 ? 1 : SYM_CHUNK]) {
    const int l = threadIdx.x % SYM_CHUNK, k = threadIdx.x / SYM_CHUNK;
    const int base = U.base, n = U.n, pair = U.pair, J0 = U.J0, J1 = U.J0 + U.nJ;
    const double ibox = BOX == INT_BOX ? 1.0 / (double)U.box : 0.0;
    const PairCoef K = pair_coef<BOX>(P, U.box);
    const int c0 = 2 * pair, i0 = c0 * SYM_CHUNK + l;
    PairBead I[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        const int li = i0 + h * SYM_CHUNK;
        I[h] = pair_bead<BOX>(xyz, fxyz, R, bc, base + li, li < n, ibox);
    }
    float3 acc[2] = {make_float3(0.f, 0.f, 0.f), make_float3(0.f, 0.f, 0.f)};
    auto load_j = [&](int J) {
        const int lj = J * SYM_CHUNK + l;
        return pair_bead<BOX>(xyz, fxyz, R, bc, base + lj, lj < n, ibox);
    };
    PairBead next{};
    if (SPLIT == 1) next = load_j(J0);
    for (int J = J0; J < J1; J++) {
        // the chunk's beads, packed and written twice (q and q + 64) so that
        // lane l reads slot l + s at step s with no wrap
        if (SPLIT == 1 || k == 0) {
            if (SPLIT > 1) next = load_j(J);
            const float4 d0 = make_float4(next.x.x, next.x.y, next.x.z, next.F.x),
                         d1 = make_float4(next.F.y, next.F.z, next.R.x, next.R.y),
                         d2 = make_float4(next.R.z, next.C.x, next.C.y, next.C.z);
#pragma unroll
            for (int q = 0; q < 2; q++) {
                jd[0][l + q * SYM_CHUNK] = d0;
                jd[1][l + q * SYM_CHUNK] = d1;
                jd[2][l + q * SYM_CHUNK] = d2;
            }
        }
        __syncthreads();
        if (SPLIT == 1 && J + 1 < J1) next = load_j(J + 1);   // requested ahead of this chunk's steps
        const float4 *j0 = &jd[0][l], *j1 = &jd[1][l], *j2 = &jd[2][l];
        float3 g = make_float3(0.f, 0.f, 0.f);
        // this wave's steps of a full sweep and of a chunk against itself
        constexpr int W = SYM_CHUNK / SPLIT, D = SYM_CHUNK / 2 / SPLIT;
        const int s0 = k * W, s1 = s0 + W;
        if (J > c0 + 1) {
#pragma unroll 1
            for (int s = s0; s < s1; s++) {
                const float4 A = j0[s], B = j1[s], Cq = j2[s];
                pair_block<BOX, true>(K, I[0], A, B, Cq, acc[0], g);
                pair_block<BOX, true>(K, I[1], A, B, Cq, acc[1], g);
                rotate(g);
            }
        } else {
            if (J > c0)
#pragma unroll 1
                for (int s = s0; s < s1; s++) {
                    pair_block<BOX, true>(K, I[0], j0[s], j1[s], j2[s], acc[0], g);
                    rotate(g);
                }
            const int h = J - c0;
            const PairBead &D0 = h ? I[1] : I[0];
            float3 own = make_float3(0.f, 0.f, 0.f), gd = own;
            const int t0 = 1 + k * D, t1 = t0 + D, t2 = min(t1, SYM_CHUNK / 2);
#pragma unroll 1
            for (int s = t0; s < t2; s++) {
                pair_block<BOX, true>(K, D0, j0[s], j1[s], j2[s], own, gd);
                rotate(gd);
            }
            if (t2 < t1) pair_block<BOX, false>(K, D0, j0[t2], j1[t2], j2[t2], own, gd);
            // lane l holds the j-side sums of bead l + t2 of the chunk
            const int src = (l - t2) & (SYM_CHUNK - 1);
            own.x += __shfl(gd.x, src);
            own.y += __shfl(gd.y, src);
            own.z += __shfl(gd.z, src);
#pragma unroll
            for (int q = 0; q < 2; q++)
                if (q == h) {
                    acc[q].x += own.x;
                    acc[q].y += own.y;
                    acc[q].z += own.z;
                }
        }
        const int lj = J * SYM_CHUNK + l;
        float *out = partial + (size_t)3 * pair * nb + base + lj;
        if (SPLIT == 1) {
            if (J > c0 && lj < n) {
                out[0] = g.x;
                out[nb] = g.y;
                out[2 * (size_t)nb] = g.z;
            }
            __syncthreads();   // the chunk's slots are free
        } else {
            // lane l holds the sums of bead l + s1 of J
            const int q = (l + s1) & (SYM_CHUNK - 1);
            red[k][6][q] = g.x;
            red[k][7][q] = g.y;
            red[k][8][q] = g.z;
            __syncthreads();
            if (k < 3 && J > c0 && lj < n) {
                float v = 0.f;
#pragma unroll
                for (int w = 0; w < SPLIT; w++) v += red[w][6 + k][l];
                out[(size_t)k * nb] = v;
            }
            __syncthreads();
        }
    }
    float *out = partial + (size_t)3 * (ioff + J0 / jrun) * nb + base + i0;
    if (SPLIT == 1) {
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (i0 + h * SYM_CHUNK < n) {
                out[h * SYM_CHUNK] = acc[h].x;
                out[(size_t)nb + h * SYM_CHUNK] = acc[h].y;
                out[2 * (size_t)nb + h * SYM_CHUNK] = acc[h].z;
            }
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            red[k][3 * h][l] = acc[h].x;
            red[k][3 * h + 1][l] = acc[h].y;
            red[k][3 * h + 2][l] = acc[h].z;
        }
        __syncthreads();
        for (int c = k; c < 6; c += SPLIT) {
            const int h = c / 3, o = h * SYM_CHUNK;
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < SPLIT; w++) v += red[w][c][l];
            if (i0 + o < n) out[(size_t)(c % 3) * nb + o] = v;
        }
    }
}

template <PairBox BOX, int SPLIT>
__global__ void __launch_bounds__(SYM_CHUNK *SPLIT, 5)
    k_tea_pairs_sym(mte_params P, int nb, const float4 *xyz, const float4 *fxyz, const float4 *R, const float4 *bc,
                    const PairUnit *units, int jrun, int ioff, float *partial) {
    static_assert(SPLIT == 1 || SPLIT >= 3, "three waves add the j-side components");
    __shared__ float4 jd[3][2 * SYM_CHUNK];
    __shared__ float red[SPLIT][9][SPLIT == 1 ? 1 : SYM_CHUNK];
    const PairUnit U = units[blockIdx.x];
    if (BOX == INT_BOX && U.box > 0.f)
        pair_unit<INT_BOX, SPLIT>(P, U, nb, xyz, fxyz, R, bc, jrun, ioff, partial, jd, red);
    else
        pair_unit<unboxed(BOX), SPLIT>(P, U, nb, xyz, fxyz, R, bc, jrun, ioff, partial, jd, red);
}

// Pair sums of one (trajectory, 256-bead i group, j chunk) work unit:
//   partial_i = sum_{j in chunk, j != i, non-extra} D_hat_ij (F_j + beta C_i . R_j)
// The chunk's j data sit in LDS; extra beads enter with zero force and
// noise, so they contribute nothing and need no branch.  Coordinates and
// coefficients are those of k_tea_pairs_sym, so both forms take the same
// image of a pair half a box apart.
// Splitting j into chunks gives ~10 work units per SIMD at 64 x 1040 beads,
// against ~1 per SIMD for one thread per bead over the whole trajectory.
template <PairBox BOX, int CHUNK>
__device__ __forceinline__ void pair_chunk(const mte_params &P, const DevTopo &T, const DevState &S, const float4 *fxyz,
                                           const float4 *R, const float4 *bc, int4 u, float4 *partial,
                                           float4 (*jd)[CHUNK]) {
    const int base = T.tbase[u.x], n = T.tsize[u.x];
    const float box = T.tbox[u.x];
    const double ibox = BOX == INT_BOX ? 1.0 / (double)box : 0.0;
    const PairCoef K = pair_coef<BOX>(P, box);
    const int jn = min(CHUNK, n - u.z);
    for (int q = threadIdx.x; q < jn; q += TEA_TILE) {
        const PairBead v = pair_bead<BOX>(S.xyz, fxyz, R, bc, base + u.z + q, true, ibox);
        jd[0][q] = make_float4(v.x.x, v.x.y, v.x.z, v.F.x);
        jd[1][q] = make_float4(v.F.y, v.F.z, v.R.x, v.R.y);
        jd[2][q] = make_float4(v.R.z, v.C.x, v.C.y, v.C.z);
    }
    __syncthreads();
    const int li = u.y + threadIdx.x;
    if (li >= n) return;
    const int b = base + li;
    float3 acc = make_float3(0.f, 0.f, 0.f);
    if (!T.extra[b]) {
        const PairBead I = pair_bead<BOX>(S.xyz, fxyz, R, bc, b, true, ibox);
        float3 none = acc;
        for (int q = 0; q < jn; q++) pair_block<BOX, false>(K, I, jd[0][q], jd[1][q], jd[2][q], acc, none);
        const int self = li - u.z;   // position of i in this chunk, if any
        if (self >= 0 && self < jn) {
            // The loop took the j == i slot as a coincident bead: d = 0 leaves
            // only its cii (v_i) term, recomputed here from the same operands
            // and taken out again.
            const float cii = fmaf(-0.28125f, K.r2min * rsq_fast(K.r2min) * K.ia, 1.f);
            acc.x = fmaf(-cii, fmaf(I.C.x, I.R.x, I.F.x), acc.x);
            acc.y = fmaf(-cii, fmaf(I.C.y, I.R.y, I.F.y), acc.y);
            acc.z = fmaf(-cii, fmaf(I.C.z, I.R.z, I.F.z), acc.z);
        }
    }
    partial[(size_t)u.w * T.nb + b] = make_float4(acc.x, acc.y, acc.z, 0.f);
}

template <int CHUNK, PairBox BOX>
__global__ void __launch_bounds__(TEA_TILE)
    k_tea_pairs(mte_params P, DevTopo T, DevState S, const float4 *fxyz, const float4 *R, const float4 *bc,
                const int4 *units, float4 *partial) {
    __shared__ float4 jd[3][CHUNK];
    const int4 u = units[blockIdx.x];   // traj, i0, j0, chunk index
    if (BOX == INT_BOX && T.tbox[u.x] > 0.f)
        pair_chunk<INT_BOX, CHUNK>(P, T, S, fxyz, R, bc, u, partial, jd);
    else
        pair_chunk<unboxed(BOX), CHUNK>(P, T, S, fxyz, R, bc, u, partial, jd);
}

// What the update of a bead adds up and moves, k_tea_finish and k_tea_turn.
struct TeaMove {
    const float4 *fxyz, *fang, *R, *ci;
    const float *beta;
    const int *nchunks;
    int jrun, ioff;
    const float4 *partial;
    uint4 *seeds;
};

// Self term and chunk partials in fixed order, of bead b of trajectory t, and
// the bead's state (integrateTea_kernel_unlisted, src/bdhitea_kernel.cu:148-213).
// SYM: the partials of k_tea_pairs_sym (planes of x, y, z; the bead's j-side
// slots, then its i-side slots), else the float4 slots of its trajectory's
// chunks.
template <bool SYM>
__device__ __forceinline__ float3 tea_sum(const DevTopo &T, const DevState &Sin, const TeaMove &M, int b, int t, float4 &x,
                                          float4 &an, float4 &n4, float4 &p1, float4 &p2) {
    const float bt = M.beta[t];
    const float4 cc = M.ci[b], Fi = M.fxyz[b], Ri = M.R[b];
    const float w = bt * bt;
    // C_i = 1/sqrt(1 + beta^2 ci) per row (eq. 19)
    const float cx = rsq_fast(1.f + w * cc.x), cy = rsq_fast(1.f + w * cc.y), cz = rsq_fast(1.f + w * cc.z);
    float fx = fmaf(Ri.x, cx, Fi.x), fy = fmaf(Ri.y, cy, Fi.y), fz = fmaf(Ri.z, cz, Fi.z);
    // the bead's state is requested before the partial sums are added
    x = Sin.xyz[b];
    an = Sin.ang[b];
    n4 = Sin.fn[b];
    p1 = Sin.fp1[b];
    p2 = Sin.fp2[b];
    const size_t nb = T.nb;
    if (SYM) {
        const float *part = reinterpret_cast<const float *>(M.partial) + b;
        const int chunk = (b - T.tbase[t]) / SYM_CHUNK, nch = (T.tsize[t] + SYM_CHUNK - 1) / SYM_CHUNK;
        // the j-side slots, then the i-side ones, eight at a time: 24 loads in
        // flight, then added in order (of a last group, those that exist)
        const int nj = (chunk + 1) / 2, i0 = M.ioff + (chunk & ~1) / M.jrun;
        const int ns = nj + (nch - 1) / M.jrun + 1 - (chunk & ~1) / M.jrun;
        for (int c = 0; c < ns; c += 8) {
            float v[8][3];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int q = min(c + u, ns - 1);
                const float *p = part + 3 * (size_t)(q < nj ? q : i0 + q - nj) * nb;
#pragma unroll
                for (int k = 0; k < 3; k++) v[u][k] = p[k * nb];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) {
                if (c + u < ns) {
                    fx += v[u][0];
                    fy += v[u][1];
                    fz += v[u][2];
                }
            }
        }
    } else {
        const int nc = M.nchunks[t];
        // partials four at a time: four loads in flight, then added in order
        int c = 0;
        for (; c + 4 <= nc; c += 4) {
            float4 pp[4];
#pragma unroll
            for (int u = 0; u < 4; u++) pp[u] = M.partial[(size_t)(c + u) * nb + b];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                fx += pp[u].x;
                fy += pp[u].y;
                fz += pp[u].z;
            }
        }
        for (; c < nc; c++) {
            const float4 pp = M.partial[(size_t)c * nb + b];
            fx += pp.x;
            fy += pp.y;
            fz += pp.z;
        }
    }
    return make_float3(fx, fy, fz);
}
// The angular normals of a bead, and its update by the sum f.
__device__ __forceinline__ float4 tea_angles(const DevTopo &T, const TeaMove &M, const float *noise, int b) {
    if (noise) {
        const float *q = noise + 6 * (size_t)b;
        return make_float4(q[3], q[4], q[5], 0.f);
    }
    uint4 s = M.seeds[b + T.nb];
    const float4 ra = normals4(s);
    M.seeds[b + T.nb] = s;
    return ra;
}
__device__ __forceinline__ void tea_update(const ForceK &K, const TeaMove &M, const LatOffsets &L, int b, int flags,
                                           float3 f, float4 ra, float4 &x, float4 &an, float4 &n4, float4 &p1,
                                           float4 &p2) {
    if (!is_mobile(flags)) return;
    x.x = fmaf(K.dtg, f.x, x.x);
    x.y = fmaf(K.dtg, f.y, x.y);
    x.z = fmaf(K.dtg, f.z, x.z);
    const float4 fa = M.fang[b];
    em_angles(K, fa.x, fa.y, fa.z, ra, an);
    frame_vectors(an.x, an.y, an.z, L, n4, p1, p2);
}
__device__ __forceinline__ void store_bead(const DevState &S, int b, float4 x, float4 an, float4 n4, float4 p1,
                                           float4 p2) {
    S.xyz[b] = x;
    S.ang[b] = an;
    S.fn[b] = n4;
    S.fp1[b] = p1;
    S.fp2[b] = p2;
}

template <bool SYM>
__global__ void __launch_bounds__(TEA_TILE)
    k_tea_finish(ForceK K, DevTopo T, DevState Sin, DevState Sout, TeaMove M, const float *noise, LatOffsets L) {
    const int b = xcd_bead(TEA_TILE);
    if (b >= T.nb) return;
    float4 x, an, n4, p1, p2;
    const float3 f = tea_sum<SYM>(T, Sin, M, b, T.tid[b], x, an, n4, p1, p2);
    tea_update(K, M, L, b, T.flags[b], f, tea_angles(T, M, noise, b), x, an, n4, p1, p2);
    store_bead(Sout, b, x, an, n4, p1, p2);
}

// The end of one step and the forces of the next in one launch, a workgroup
// per trajectory and a thread per bead: each moves its bead and stages it in
// LDS, then the new forces and random forces are formed from there.  Bounded,
// as the two kernels it stands for, by waiting, not by bytes or operations:
// it saves a launch, their second reading of every state and the wait between
// them.  The lists are requested before the bead is moved.
// HELPED: a second thread per bead, in another wave, draws both its normals
// while the sums come in, and sums its LJ forces beside its bonds; the sums
// are added in the same order.
// One tube of 312 beads: 5.7 us of forces and 4.2 of update apart, 7.3 in one,
// 5.9 helped.
constexpr int TURN_THREADS = 640, TURN_HELPED = 512;   // beads at most
template <bool PERIODIC, bool HELPED>
__global__ void __launch_bounds__(HELPED ? 2 * TURN_HELPED : TURN_THREADS)
    k_tea_turn(ForceK K, DevTopo T, DevState Sin, DevState Sout, TeaMove M, const float *noise, TeaDraw D,
               float4 *fxyz, float4 *fang, LatOffsets L) {
    extern __shared__ float4 lds[];
    const int t = xcd_block();   // through the L2 that the pair kernel left its partials in
    if (t >= T.ntraj) return;
    const int base = T.tbase[t], n = T.tsize[t];
    float4 *lx = lds, *ln = lds + n, *l1 = ln + n, *l2 = l1 + n, *xb = l2 + n;   // xb: from the helpers
    const LdsAcc A(lx, ln, l1, l2);
    const float wall_z = K.is_wall ? T.zs[t] : 0.f;
    const int nmain = HELPED ? blockDim.x / 2 : blockDim.x;
    const bool helper = HELPED && (int)threadIdx.x >= nmain;
    const int i = threadIdx.x - (helper ? nmain : 0), b = base + min(i, n - 1);
    const AheadLists<LdsAcc::SCALE> Ls(T, b, base, A.origin());
    const int flags = T.flags[b];
    const bool extra = (flags & FL_EXTRA) != 0;
    float4 x, an, n4, p1, p2, R;   // R: the next random force
    float3 f;
    if (i < n) {
        if (!helper) f = tea_sum<true>(T, Sin, M, b, t, x, an, n4, p1, p2);
        if (helper) xb[i] = tea_angles(T, M, noise, b);
        if (!HELPED || helper) R = tea_draw(D, K.vF, b, extra);
    }
    if (HELPED) __syncthreads();
    if (i < n && !helper) {
        tea_update(K, M, L, b, flags, f, HELPED ? xb[i] : tea_angles(T, M, noise, b), x, an, n4, p1, p2);
        store_bead(Sout, b, x, an, n4, p1, p2);
        x.w = __int_as_float(flags);
        lx[i] = x;
        ln[i] = make_float4(n4.x, n4.y, n4.z, an.x);
        l1[i] = make_float4(p1.x, p1.y, p1.z, an.y);
        l2[i] = make_float4(p2.x, p2.y, p2.z, an.z);
    }
    __syncthreads();
    // written once the bead has been moved: its sum has read the last one
    if (i < n && (!HELPED || helper)) D.R[b] = R;
    float F[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (i < n && !extra) {
        if (helper) {
            Own I;
            I.r = f3(lx[i]);
            if (PERIODIC) set_box(I, T.tbox[t]);
            const float3 lj = K.lj_on ? lj_sum<PERIODIC>(K, A, Ls, I) : make_float3(0.f, 0.f, 0.f);
            xb[i] = make_float4(lj.x, lj.y, lj.z, 0.f);
        } else {
            Own I = make_own(x, an, n4, p1, p2, flags);
            if (PERIODIC) set_box(I, T.tbox[t]);
            if (HELPED) bond_total(bond_forces<PERIODIC>(K, A, Ls, I), I, F);
            else bead_force<PERIODIC>(K, A, Ls, wall_z, I, F);
        }
    }
    if (HELPED) __syncthreads();
    if (i >= n || helper) return;
    if (HELPED && !extra) add_lj_walls(K, f3(xb[i]), wall_z, f3(x), F);
    fxyz[b] = make_float4(F[0], F[1], F[2], 0.f);
    fang[b] = make_float4(F[3], F[4], F[5], 0.f);   // fi, theta, psi
}

// ------------------------------------------------------------------ MFMA
// Pair sums on the matrix cores (open boundaries).  With d = r_i - r_j and
// the far-branch coefficients (r > 2a) of D_hat = cii I + c d d^T,
//   cii = p1 w + p3 w^3,  c = p1 w^3 - 3 p3 w^5,  w = 1/r, p1 = 3a/4, p3 = a^3/2,
// the sum over the j of a tile of D_hat_ij (F_j + C'_i . R_j), C' = beta C,
// splits into two scalar kernels times per-j moments about the tile's centre
// Y (s = r_j - Y, b = r_i - Y, d = b - s):
//   sum_j cii (F_j + C'_i . R_j)                          -> moments F, R
//   sum_j c d (d . F_j)  = b (b . S[F]) - b S[s.F] - S[s F^T] b + S[s (s.F)]
//   sum_j c d_al d_ga R_ga = b_al b_ga S[R_ga] - b_al S[s_ga R_ga]
//                            - b_ga S[s_al R_ga] + S[s_al s_ga R_ga]
// with S[m] = sum_j kernel_ij m_j: 6 moment columns on cii and 37 on c.  The
// moments depend on the source tile alone, so k_tea_moments tabulates them
// once per step (split into bf16 hi + lo, a value being hi + lo to 2^-18 of
// itself), and the pair kernel only evaluates the two kernels per pair and
// contracts them with the tables on v_mfma_f32_16x16x32_bf16 (hi hi, hi lo,
// lo hi, accumulated in FP32).  The kernels are symmetric in (i, j), so each
// pair's values serve both beads: tile I's sums over tile J and tile J's
// over tile I, as k_tea_pairs_sym does with its 3 x 3 blocks.
// Tiles are 64 consecutive beads of the spatial (Morton cell) order that
// k_rebuild_order computes when a state is set, a compact patch (on a
// microtubule at most ~24 nm from its centre); any order gives the same
// sums in exact arithmetic, but the rounding of the expansion grows with
// the tile's radius.  Pairs closer than MF_RNEAR (> 2a, so every product
// pair takes the far branch) are summed exactly on the VALU instead: they
// carry the largest kernel values, and beyond MF_RNEAR the terms of the
// expansion exceed the result by at most (1 + |s| / r)^2.  Trajectories
// above REBUILD_ORDER_MAX beads keep the index order, so the engine does
// not offer this form for them.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
constexpr int MF_TILE = 64;
constexpr int MF_COLS = 64;     // moment columns per bead in the tables: 0-36 on c, 48-53 on cii
constexpr int MF_USED = 43;     // the columns in use, packed (c: 0-36, cii: 37-42)
constexpr int MF_OUT_LD = 68;   // row stride of the LDS result rows (floats)
constexpr float MF_RNEAR = 6.f;

// packed index of moment column c, or -1 for an unused column
__device__ __forceinline__ int mf_packed(int c) { return c < 37 ? c : (c >= 48 && c < 54 ? c - 11 : -1); }

// Moment tables and bead records of one 64-bead tile (one wave; lane = bead
// of the tile): centre Y = mean position of the tile's beads, radius = the
// largest distance of one of them from Y; per bead, with s = r - Y,
//   0-2  s_al (s.F)     3-11 s_al F_be    12 s.F     13-15 F_be
//   16-24 s_al s_ga R_ga  25-33 s_al R_ga  34-36 R_ga             (kernel c)
//   48-50 F   51-53 R                                              (kernel cii)
// Extra beads and slots past the trajectory's end have zero F and R, so all
// their moments vanish.  Tables: mom[tile][hi, lo][column][bead] bf16;
// records rec[tile][position (w = 1 if active), F, R, C'][bead] and
// rbead[tile][bead] (global index, -1 past the end), so that the pair kernel
// reads each tile with coalesced loads that depend on nothing but the unit.
__global__ void __launch_bounds__(MF_TILE)
    k_tea_moments(DevTopo T, DevState S, const float4 *fxyz, const float4 *R, const float4 *ci, const float *beta,
                  const int *order, const int2 *tiles, __bf16 *mom, float4 *ctr, float4 *rec, int *rbead) {
    const int2 tl = tiles[blockIdx.x];   // trajectory, first position
    const int base = T.tbase[tl.x], n = T.tsize[tl.x];
    const int lane = threadIdx.x, p = tl.y + lane;
    const bool in = p < n;
    const int bi = in ? base + order[base + p] : base;
    const float4 x = in ? S.xyz[bi] : make_float4(0.f, 0.f, 0.f, 0.f);
    float sum[4] = {x.x, x.y, x.z, in ? 1.f : 0.f};
#pragma unroll
    for (int m = 1; m < MF_TILE; m <<= 1)
#pragma unroll
        for (int k = 0; k < 4; k++) sum[k] += __shfl_xor(sum[k], m);
    const float cx = sum[0] / sum[3], cy = sum[1] / sum[3], cz = sum[2] / sum[3];
    const bool act = in && !T.extra[bi];
    const float4 F = act ? fxyz[bi] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 Rb = act ? R[bi] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float s[3] = {x.x - cx, x.y - cy, x.z - cz}, Fv[3] = {F.x, F.y, F.z}, Rv[3] = {Rb.x, Rb.y, Rb.z};
    float rad = in ? sqrtf(s[0] * s[0] + s[1] * s[1] + s[2] * s[2]) : 0.f;
#pragma unroll
    for (int m = 1; m < MF_TILE; m <<= 1) rad = fmaxf(rad, __shfl_xor(rad, m));
    const float sF = s[0] * Fv[0] + s[1] * Fv[1] + s[2] * Fv[2];
    float m[MF_COLS];
#pragma unroll
    for (int c = 0; c < MF_COLS; c++) m[c] = 0.f;
#pragma unroll
    for (int al = 0; al < 3; al++) {
        m[al] = s[al] * sF;
        m[13 + al] = Fv[al];
        m[34 + al] = Rv[al];
        m[48 + al] = Fv[al];
        m[51 + al] = Rv[al];
#pragma unroll
        for (int be = 0; be < 3; be++) {
            m[3 + 3 * al + be] = s[al] * Fv[be];
            m[16 + 3 * al + be] = s[al] * s[be] * Rv[be];
            m[25 + 3 * al + be] = s[al] * Rv[be];
        }
    }
    m[12] = sF;
    __bf16 *hi = mom + (size_t)blockIdx.x * 2 * MF_COLS * MF_TILE, *lo = hi + MF_COLS * MF_TILE;
#pragma unroll
    for (int c = 0; c < MF_COLS; c++) {
        const __bf16 h = (__bf16)m[c];
        hi[c * MF_TILE + lane] = h;
        lo[c * MF_TILE + lane] = (__bf16)(m[c] - (float)h);
    }
    float4 C = make_float4(0.f, 0.f, 0.f, 0.f);
    if (act) {
        const float bt = beta[tl.x], w2b = bt * bt;
        const float4 cc = ci[bi];
        C = make_float4(bt * rsq_fast(1.f + w2b * cc.x), bt * rsq_fast(1.f + w2b * cc.y),
                        bt * rsq_fast(1.f + w2b * cc.z), 0.f);
    }
    float4 *rt = rec + (size_t)blockIdx.x * 4 * MF_TILE;
    rt[lane] = in ? make_float4(x.x, x.y, x.z, act ? 1.f : 0.f) : make_float4(1e6f, 1e6f, 1e6f, 0.f);
    rt[MF_TILE + lane] = F;
    rt[2 * MF_TILE + lane] = Rb;
    rt[3 * MF_TILE + lane] = C;
    rbead[(size_t)blockIdx.x * MF_TILE + lane] = in ? bi : -1;
    if (lane == 0) ctr[blockIdx.x] = make_float4(cx, cy, cz, rad);
}

__device__ __forceinline__ void mf_split8(const float v[8], bf16x8_t &hi, bf16x8_t &lo) {
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const __bf16 h = (__bf16)v[q];
        hi[q] = h;
        lo[q] = (__bf16)(v[q] - (float)h);
    }
}

// Sum over one source tile for a target bead from the packed moment sums o
// (MF_USED columns), b = r_target - Y_source and the target's C'.
__device__ __forceinline__ float3 mf_reconstruct(const float *o, const float b[3], const float cp[3]) {
    const float bF = b[0] * o[13] + b[1] * o[14] + b[2] * o[15];
    float f[3];
#pragma unroll
    for (int al = 0; al < 3; al++) {
        // cii (F + C' . R)
        float v = fmaf(cp[al], o[40 + al], o[37 + al]);
        // c d (d . F)
        v += o[al] - (b[0] * o[3 + 3 * al] + b[1] * o[4 + 3 * al] + b[2] * o[5 + 3 * al]) - b[al] * o[12] +
             b[al] * bF;
        // sum_ga C'_ga c d_al d_ga R_ga
#pragma unroll
        for (int ga = 0; ga < 3; ga++)
            v = fmaf(cp[ga],
                     o[16 + 3 * al + ga] - b[ga] * o[25 + 3 * al + ga] - b[al] * o[25 + 4 * ga] +
                         b[al] * b[ga] * o[34 + ga],
                     v);
        f[al] = v;
    }
    return make_float3(f[0], f[1], f[2]);
}

// Pair kernel.  Work unit: (tile I, tile J >= I of the same trajectory,
// partial slots I and J), 256 threads.  Wave w takes the 32 x 32 block
// (i half w / 2, j half w % 2) of the unit's 64 x 64 pairs; lane (g, il)
// evaluates the pairs (i = 16 rb + il, j = 8 g + q) of its block, rb < 2,
// q < 8, which is the A operand layout of two 16 x 32 MFMA tiles (row il,
// k = 8 g + q).  I side: those tiles times tile J's moment tables (16 bytes
// per lane from global memory, requested with the tiles' records before
// anything waits) give the 64 moment sums of each i over the block's 32 j.
// J side: the wave stores its kernel values transposed in LDS (rows j, 8
// consecutive i per 16 bytes, the 16-byte groups XOR-swizzled by row so that
// the four lane groups of a store hit different banks) and reads them back
// as A operands against tile I's tables.  The two halves of each target's
// sums meet in LDS; one thread per target adds them, reconstructs the sum
// over the source tile and writes it to the target's partial slot (I side:
// slot J, J side: slot I), as k_tea_pairs_sym does.  A diagonal unit
// (I == J) sums every ordered pair on the I side alone.  Near pairs
// (r < MF_RNEAR) enter the products as zero and are added exactly per lane,
// on both sides, and reduced across the lanes in fixed order: the result
// does not depend on scheduling.  A unit whose tiles' bounding spheres lie
// more than MF_RNEAR apart holds no near pair and skips those tests.
constexpr int MF_KT_WAVE = 4 * 32 * 32;   // bf16 per wave: kd hi, kd lo, kc hi, kc lo; 32 j x 32 i
struct MfLds {
    float4 rec[2][4][MF_TILE];   // [I, J][position (w: active), F, R, C'][bead]
    int bead[2][MF_TILE];
    float near_i[2][MF_TILE][3];   // exact near-pair sums, I side, per j half
    float near_j[2][MF_TILE][3];   // J side, per i half
    union {
        __bf16 kt[4][MF_KT_WAVE];
        float out[2][2][MF_USED][MF_OUT_LD];   // [side][half][packed column][target]
    } u;
};

__device__ __forceinline__ int mf_kt_index(int type, int jj, int ii) {
    // row jj of 32 i; 16-byte group (8 i) swizzled by (jj / 8) % 4
    return (type * 32 + jj) * 32 + (ii ^ (8 * ((jj >> 3) & 3)));
}

// Kernels of one lane's 16 pairs as MFMA A operands; with NEAR, the pairs
// closer than MF_RNEAR enter as zero and their exact blocks are summed into
// ni (I side, per row block) and nj (J side, per q).
template <bool NEAR>
__device__ __forceinline__ void mf_pairs(const MfLds &L, int ha, int hb, int g, int il, bool diag, float a, float ia,
                                         bf16x8_t (&kA)[2][4], float3 (&ni)[2], float3 (&nj)[8], bool &any_near) {
    const float p1 = 0.75f * a, p3 = 0.5f * a * a * a;
#pragma unroll
    for (int rb = 0; rb < 2; rb++) {
        const int ii = 32 * ha + 16 * rb + il;
        const float4 xi = L.rec[0][0][ii];
        float kd[8], kc[8];
#pragma unroll
        for (int q = 0; q < 8; q++) {
            const int jj = 32 * hb + 8 * g + q;
            const float4 xj = L.rec[1][0][jj];
            const float dx = xi.x - xj.x, dy = xi.y - xj.y, dz = xi.z - xj.z;
            const float r2 = dx * dx + dy * dy + dz * dz;
            const float wv = rsq_fast(NEAR ? fmaxf(r2, 1e-12f) : r2), wv2 = wv * wv, wv3 = wv2 * wv;
            kd[q] = fmaf(p3, wv3, p1 * wv);
            kc[q] = wv3 * fmaf(-3.f * p3, wv2, p1);
            if (NEAR) {
                const bool nearp = r2 < MF_RNEAR * MF_RNEAR;
                kd[q] = nearp ? 0.f : kd[q];
                kc[q] = nearp ? 0.f : kc[q];
                any_near |= nearp;
                if (nearp && xi.w != 0.f && xj.w != 0.f && !(diag && ii == jj)) {
                    // the exact RPY block (both branches), src/bdhitea_kernel.cu:38-58, 104-146
                    const float r2c = fmaxf(r2, 1e-12f), rinv = rsq_fast(r2c);
                    const RpyCoef cf = rpy_select(r2c, rinv, a, ia);
                    const float cr = cf.crr * rinv * rinv;
                    const float4 Ci = L.rec[0][3][ii], Fj = L.rec[1][1][jj], Rj = L.rec[1][2][jj];
                    const float vx = fmaf(Ci.x, Rj.x, Fj.x), vy = fmaf(Ci.y, Rj.y, Fj.y),
                                vz = fmaf(Ci.z, Rj.z, Fj.z);
                    const float sv = cr * (dx * vx + dy * vy + dz * vz);
                    ni[rb].x = fmaf(sv, dx, fmaf(cf.cii, vx, ni[rb].x));
                    ni[rb].y = fmaf(sv, dy, fmaf(cf.cii, vy, ni[rb].y));
                    ni[rb].z = fmaf(sv, dz, fmaf(cf.cii, vz, ni[rb].z));
                    if (!diag) {
                        const float4 Cj = L.rec[1][3][jj], Fi = L.rec[0][1][ii], Ri = L.rec[0][2][ii];
                        const float ux = fmaf(Cj.x, Ri.x, Fi.x), uy = fmaf(Cj.y, Ri.y, Fi.y),
                                    uz = fmaf(Cj.z, Ri.z, Fi.z);
                        const float su = cr * (dx * ux + dy * uy + dz * uz);
                        nj[q].x = fmaf(su, dx, fmaf(cf.cii, ux, nj[q].x));
                        nj[q].y = fmaf(su, dy, fmaf(cf.cii, uy, nj[q].y));
                        nj[q].z = fmaf(su, dz, fmaf(cf.cii, uz, nj[q].z));
                    }
                }
            }
        }
        mf_split8(kd, kA[rb][0], kA[rb][1]);
        mf_split8(kc, kA[rb][2], kA[rb][3]);
    }
}

// kernel x table product of one 16-column tile: hi hi + hi lo + lo hi
__device__ __forceinline__ f32x4_t mf_product(const bf16x8_t &khi, const bf16x8_t &klo, const bf16x8_t &bh,
                                              const bf16x8_t &bl) {
    const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
    f32x4_t s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(khi, bh, zero4, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(khi, bl, s, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(klo, bh, s, 0, 0, 0);
}

__global__ void __launch_bounds__(256)
    k_tea_pairs_mfma(mte_params P, const int4 *units, const __bf16 *mom, const float4 *ctr, const float4 *rec,
                     const int *rbead, int chunk_stride, float4 *partial) {
    __shared__ MfLds L;
    const int4 u = units[blockIdx.x];   // tile I, tile J, slot I, slot J
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, g = lane >> 4, il = lane & 15;
    const int ha = w >> 1, hb = w & 1;   // i half, j half of this wave's block
    const bool diag = u.x == u.y;
    // requests that depend on the unit alone: both tiles' records, this
    // lane's fragments of both tables (16 bytes each), the two centres
    float4 rv[4];
    int rbv = -1;
    const int side0 = tid >> 6, k0 = tid & 63;
    if (tid < 2 * MF_TILE) {
        const float4 *rt = rec + (size_t)(side0 ? u.y : u.x) * 4 * MF_TILE;
#pragma unroll
        for (int c = 0; c < 4; c++) rv[c] = rt[c * MF_TILE + k0];
        rbv = rbead[(size_t)(side0 ? u.y : u.x) * MF_TILE + k0];
    }
    bf16x8_t tb[2][4][2];   // [I side: tile J's table, J side: tile I's table][column tile][hi, lo]
#pragma unroll
    for (int sd = 0; sd < 2; sd++) {
        if (sd == 1 && diag) break;
        const __bf16 *mt = mom + (size_t)(sd ? u.x : u.y) * 2 * MF_COLS * MF_TILE;
        const int kk = 32 * (sd ? ha : hb) + 8 * g;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int col = 16 * t + il;
            tb[sd][t][0] = *reinterpret_cast<const bf16x8_t *>(mt + col * MF_TILE + kk);
            tb[sd][t][1] = *reinterpret_cast<const bf16x8_t *>(mt + (MF_COLS + col) * MF_TILE + kk);
        }
    }
    const float4 YI = ctr[u.x], YJ = ctr[u.y];
    if (tid < 2 * MF_TILE) {
#pragma unroll
        for (int c = 0; c < 4; c++) L.rec[side0][c][k0] = rv[c];
        L.bead[side0][k0] = rbv;
    }
    __syncthreads();
    const float a = P.tea_a, ia = rcp_fast(P.tea_a);
    bf16x8_t kA[2][4];   // [rb][kd hi, kd lo, kc hi, kc lo]
    float3 ni[2] = {make_float3(0.f, 0.f, 0.f), make_float3(0.f, 0.f, 0.f)};
    float3 nj[8];
#pragma unroll
    for (int q = 0; q < 8; q++) nj[q] = make_float3(0.f, 0.f, 0.f);
    bool any_near = false;
    const float gap = sqrtf((YI.x - YJ.x) * (YI.x - YJ.x) + (YI.y - YJ.y) * (YI.y - YJ.y) +
                            (YI.z - YJ.z) * (YI.z - YJ.z)) - YI.w - YJ.w;
    const bool near_unit = diag || !(gap > MF_RNEAR + 0.01f);
    if (near_unit) mf_pairs<true>(L, ha, hb, g, il, diag, a, ia, kA, ni, nj, any_near);
    else mf_pairs<false>(L, ha, hb, g, il, diag, a, ia, kA, ni, nj, any_near);
    // I side: the block's pairs times tile J's tables (k = j of half hb)
    f32x4_t acc[2][4], accj[2][4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int kh = t < 3 ? 2 : 0;   // kernel c for the 48 columns 0-47, cii for 48-63
#pragma unroll
        for (int rb = 0; rb < 2; rb++) acc[rb][t] = mf_product(kA[rb][kh], kA[rb][kh + 1], tb[0][t][0], tb[0][t][1]);
    }
    // J side, first the transposed kernels of this wave's block
    if (!diag) {
        __bf16 *kt = L.u.kt[w];
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int q = 0; q < 8; q++)
#pragma unroll
                for (int ty = 0; ty < 4; ty++) kt[mf_kt_index(ty, 8 * g + q, 16 * rb + il)] = kA[rb][ty][q];
    }
    __syncthreads();
    if (!diag) {
        const __bf16 *kt = L.u.kt[w];
        bf16x8_t kB[2][4];
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int ty = 0; ty < 4; ty++)
                kB[rb][ty] = *reinterpret_cast<const bf16x8_t *>(kt + mf_kt_index(ty, 16 * rb + il, 8 * g));
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int kh = t < 3 ? 2 : 0;
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
                accj[rb][t] = mf_product(kB[rb][kh], kB[rb][kh + 1], tb[1][t][0], tb[1][t][1]);
        }
    }
    // near sums: I side over the four lane groups, J side over the 16 lanes of a row
    if (near_unit && __ballot(any_near) != 0) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int m = 16; m < 64; m <<= 1) {
                ni[rb].x += __shfl_xor(ni[rb].x, m);
                ni[rb].y += __shfl_xor(ni[rb].y, m);
                ni[rb].z += __shfl_xor(ni[rb].z, m);
            }
        if (!diag)
#pragma unroll
            for (int q = 0; q < 8; q++)
#pragma unroll
                for (int m = 1; m < 16; m <<= 1) {
                    nj[q].x += __shfl_xor(nj[q].x, m);
                    nj[q].y += __shfl_xor(nj[q].y, m);
                    nj[q].z += __shfl_xor(nj[q].z, m);
                }
    }
    __syncthreads();   // every wave is done with its kt before out overwrites them
    if (g == 0)
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            float *o = L.near_i[hb][32 * ha + 16 * rb + il];
            o[0] = ni[rb].x;
            o[1] = ni[rb].y;
            o[2] = ni[rb].z;
        }
    if (il == 0 && !diag)
#pragma unroll
        for (int q = 0; q < 8; q++) {
            float *o = L.near_j[ha][32 * hb + 8 * g + q];
            o[0] = nj[q].x;
            o[1] = nj[q].y;
            o[2] = nj[q].z;
        }
    // lane (g, il) holds rows 4 g + r of column il of each 16-column tile
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int pc = mf_packed(16 * t + il);
        if (pc < 0) continue;
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            *reinterpret_cast<f32x4_t *>(&L.u.out[0][hb][pc][32 * ha + 16 * rb + 4 * g]) = acc[rb][t];
            if (!diag) *reinterpret_cast<f32x4_t *>(&L.u.out[1][ha][pc][32 * hb + 16 * rb + 4 * g]) = accj[rb][t];
        }
    }
    __syncthreads();
    if (tid >= 2 * MF_TILE) return;
    const int side = tid >> 6, k = tid & 63;
    if (side == 1 && diag) return;
    const int bi = L.bead[side][k];
    if (bi < 0) return;
    float3 f = make_float3(0.f, 0.f, 0.f);
    const float4 xt = L.rec[side][0][k];
    if (xt.w != 0.f) {
        float o[MF_USED];
#pragma unroll
        for (int c = 0; c < MF_USED; c++) o[c] = L.u.out[side][0][c][k] + L.u.out[side][1][c][k];
        const float4 Y = side ? YI : YJ;
        const float4 cc = L.rec[side][3][k];
        const float b[3] = {xt.x - Y.x, xt.y - Y.y, xt.z - Y.z}, cp[3] = {cc.x, cc.y, cc.z};
        f = mf_reconstruct(o, b, cp);
        const float *n0 = side ? L.near_j[0][k] : L.near_i[0][k], *n1 = side ? L.near_j[1][k] : L.near_i[1][k];
        f.x += n0[0] + n1[0];
        f.y += n0[1] + n1[1];
        f.z += n0[2] + n1[2];
    }
    const int slot = side ? u.z : u.w;
    partial[(size_t)slot * chunk_stride + bi] = make_float4(f.x, f.y, f.z, 0.f);
}

template <PairBox BOX, int PER>
static void launch_eps_box(mte_engine *e) {
    auto kern = e->any_extra ? k_tea_eps_sym<BOX, true, PER> : k_tea_eps_sym<BOX, false, PER>;
    hipLaunchKernelGGL(kern, dim3(e->tea.eps_nunits), dim3(64 * eps_waves(PER)), 0, e->stream, e->P, e->T, e->S[e->cur],
                       e->tea.eps_units, e->tea.eps_ngrp, e->tea.eps_part);
}
template <int PER>
static void launch_eps_per(mte_engine *e) {
    switch (batch_box(e)) {
    case OPEN_BOX: launch_eps_box<OPEN_BOX, PER>(e); break;
    case INT_BOX: launch_eps_box<INT_BOX, PER>(e); break;
    case FLOAT_BOX: launch_eps_box<FLOAT_BOX, PER>(e); break;
    }
}
static void launch_eps_units(mte_engine *e) {
    if (e->tea.eps_group == EPS_GROUP_MIN) launch_eps_per<1>(e);
    else launch_eps_per<EPS_PER>(e);
}
static_assert(EPS_GROUP_MIN == 64 * eps_waves(1), "a group is the workgroup's chunks");

hipError_t launch_tea_eps(mte_engine *e) {
    if (e->tune.tea_eps == MTE_TEA_EPS_ONEPASS) {
        launch_eps_units(e);
        hipLaunchKernelGGL(k_tea_eps_reduce, dim3((e->nb + 255) / 256), dim3(256), 0, e->stream, e->T,
                           e->tea.eps_group, e->tea.eps_ngrp, e->tea.eps_part, e->tea.ci, e->tea.eps);
    } else if (e->periodic)
        hipLaunchKernelGGL(k_tea_eps<true>, dim3(e->ntiles), dim3(TEA_TILE), 0, e->stream, e->P, e->T,
                           e->S[e->cur], e->tiles, e->tea.ci, e->tea.eps);
    else
        hipLaunchKernelGGL(k_tea_eps<false>, dim3(e->ntiles), dim3(TEA_TILE), 0, e->stream, e->P, e->T,
                           e->S[e->cur], e->tiles, e->tea.ci, e->tea.eps);
    hipLaunchKernelGGL(k_tea_beta, dim3(e->ntraj), dim3(256), 0, e->stream, e->P, e->T, e->tea.eps, e->tea.ci,
                       e->tea.beta, e->tea.bc, e->tea.stats, e->tea.status);
    return hipGetLastError();
}

template <int CHUNK>
static void launch_pairs_chunk(mte_engine *e) {
    const PairBox box = batch_box(e);
    auto kern = box == OPEN_BOX ? k_tea_pairs<CHUNK, OPEN_BOX>
                : box == INT_BOX ? k_tea_pairs<CHUNK, INT_BOX> : k_tea_pairs<CHUNK, FLOAT_BOX>;
    hipLaunchKernelGGL(kern, dim3(e->tea.nunits), dim3(TEA_TILE), 0, e->stream, e->P, e->T, e->S[e->cur], e->fxyz,
                       e->tea.R, e->tea.bc, e->tea.units, e->tea.partial);
}

template <int SPLIT>
static void launch_pairs_sym(mte_engine *e) {
    const PairBox box = batch_box(e);
    auto kern = box == OPEN_BOX ? k_tea_pairs_sym<OPEN_BOX, SPLIT>
                : box == INT_BOX ? k_tea_pairs_sym<INT_BOX, SPLIT> : k_tea_pairs_sym<FLOAT_BOX, SPLIT>;
    hipLaunchKernelGGL(kern, dim3(e->tea.nunits), dim3(SYM_CHUNK * SPLIT), 0, e->stream, e->P, e->nb,
                       e->S[e->cur].xyz, e->fxyz, e->tea.R, e->tea.bc, e->tea.pair_units, e->tea.jrun,
                       e->tea.ioff, reinterpret_cast<float *>(e->tea.partial));
}

hipError_t launch_tea_pairs(mte_engine *e) {
    // the kernel's chunk must be the one the work units were built for
    if (e->tea.unit_chunk == MTE_TEA_SYMMETRIC) {
        switch (e->tea.split) {
        case 8: launch_pairs_sym<8>(e); break;
        case 4: launch_pairs_sym<4>(e); break;
        default: launch_pairs_sym<1>(e); break;
        }
        return hipGetLastError();
    }
    if (e->tea.unit_chunk == MTE_TEA_MFMA) {
        if (e->periodic) return hipErrorInvalidValue;   // minimum images are not in the moment form
        hipLaunchKernelGGL(k_tea_moments, dim3(e->tea.ntiles), dim3(MF_TILE), 0, e->stream, e->T, e->S[e->cur],
                           e->fxyz, e->tea.R, e->tea.ci, e->tea.beta, e->rb_order, e->tea.tiles,
                           static_cast<__bf16 *>(e->tea.mom), e->tea.ctr, e->tea.rec, e->tea.rbead);
        hipLaunchKernelGGL(k_tea_pairs_mfma, dim3(e->tea.nunits), dim3(256), 0, e->stream, e->P, e->tea.units,
                           static_cast<const __bf16 *>(e->tea.mom), e->tea.ctr, e->tea.rec, e->tea.rbead, e->nb,
                           e->tea.partial);
        return hipGetLastError();
    }
    switch (e->tea.unit_chunk) {
    case 64: launch_pairs_chunk<64>(e); break;
    case 128: launch_pairs_chunk<128>(e); break;
    case 256: launch_pairs_chunk<256>(e); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

static TeaMove tea_move_args(const mte_engine *e) {
    return TeaMove{e->fxyz, e->fang,    e->tea.R,    e->tea.ci,      e->tea.beta, e->tea.nchunks,
                   e->tea.jrun, e->tea.ioff, e->tea.partial, e->seeds};
}

hipError_t launch_tea_finish(mte_engine *e, const float *noise_step) {
    auto kern = e->tea.unit_chunk == MTE_TEA_SYMMETRIC ? k_tea_finish<true> : k_tea_finish<false>;
    hipLaunchKernelGGL(kern, dim3(grid_xcd(e->nb, TEA_TILE)), dim3(TEA_TILE), 0, e->stream, e->K, e->T, e->S[e->cur],
                       e->S[1 - e->cur], tea_move_args(e), noise_step, e->L);
    e->cur = 1 - e->cur;
    return hipGetLastError();
}

// k_tea_turn serves the symmetric pair kernel's partials, with forces from
// LDS, for trajectories of up to 640 beads: a workgroup's one bead per thread
// then costs less than the launch it saves (per 100 steps, two kernels -> one:
// 1, 8 and 64 tubes of 520 beads 1571 -> 1600, 1621 -> 1560 and 2906 -> 2768
// us, of 624 beads 1591 -> 1589, 1641 -> 1582 and 3194 -> 3058; of 780 beads
// 1631 -> 1760, 1878 -> 2031 and 3863 -> 4013: the two keep more CUs busy).
// Where two threads per bead fit, they do (64 and 1 tubes of 312 beads 1742 ->
// 1623 and 1386 -> 1298).
bool tea_turn_fits(const mte_engine *e) {
    return e->tea.unit_chunk == MTE_TEA_SYMMETRIC && e->tune.forces == MTE_FORCES_LDS && e->forces_lds > 0 &&
           e->nmax <= TURN_THREADS;
}

hipError_t launch_tea_turn(mte_engine *e, const float *noise_step, const float *noise_next) {
    const bool helped = e->nmax <= TURN_HELPED;
    auto kern = helped ? (e->periodic ? k_tea_turn<true, true> : k_tea_turn<false, true>)
                       : (e->periodic ? k_tea_turn<true, false> : k_tea_turn<false, false>);
    const int threads = ((e->nmax + 63) / 64) * 64 * (helped ? 2 : 1);
    const size_t lds = e->forces_lds + (helped ? sizeof(float4) * e->nmax : 0);   // at most 40 KB
    hipLaunchKernelGGL(kern, dim3(grid_xcd(e->ntraj, 1)), dim3(threads), lds, e->stream, e->K, e->T, e->S[e->cur],
                       e->S[1 - e->cur], tea_move_args(e), noise_step, TeaDraw{e->seeds, noise_next, e->tea.R}, e->fxyz,
                       e->fang, e->L);
    e->cur = 1 - e->cur;
    return hipGetLastError();
}

}  // namespace mte
