// resident.hip -- plain Langevin dynamics with each trajectory resident in
// one workgroup's LDS across many steps.
//
// One workgroup owns one trajectory.  LDS holds, per bead, the position and
// the three rotated offsets with the Euler angles packed into their spare
// lanes (64 B), plus the bead's neighbour lists compacted into a uint16 CSR
// (the LDS address of the neighbour's position; bonds: with their flag in bit
// 0) whose places are sized for the full lists, so a distance-filtered list
// and its later refill share one layout.  Each
// thread owns PT beads and keeps their two HybridTaus states in registers.
// A launch runs every step up to the next
// list-rebuild boundary (LJPairsUpdateFreq steps; 100 in the batched
// workload), after the rebuild kernel of lists.hip has refreshed the lists
// when one is due, so HBM sees the state once per launch instead of twice
// per step.  Per step:
//   forces + Euler-Maruyama for own beads, every operand from LDS
//   -> barrier -> own new state to LDS -> barrier.
// The arithmetic is bead_force / em_update, the code the streamed step runs.
//
// What bounds it: the vector operations, about 3 cycles each, of 16 waves on
// four SIMDs (256 tubes of 1040 beads, a workgroup per CU); of a step the LJ
// sums take some 30 %, the normals 20 %, the bonds 27 %, the frames 9 %.  So
// the operations were cut: quotients and halves taken on the host (ForceK),
// torques summed as vectors and projected once, lists with ready LDS
// addresses, LJ lists padded to the groups they are summed in, fewer
// operations per HybridTaus draw, no minimum image in open batches: 713 ->
// 575 us per 100 steps, one tube of 312 beads 435 -> 343 us.
// If a trajectory's lists do not fit the LDS left over, that workgroup reads
// them from the global k-major arrays instead (same results, slower).
#include "bead_physics.h"
#include "engine_internal.h"

namespace mte {

constexpr int RES_MAX_THREADS = 1024;   // one bead per thread
constexpr int RES_MULTI_THREADS = 768;  // several beads per thread: leaves room for more VGPRs
constexpr int RES_MAX_PT = 3;
constexpr int STATE_ARRAYS = 4;         // xyz|flags, n|fi, p1|theta, p2|psi
constexpr int HDR_INTS = 2;             // per bead: list offset, packed counts
constexpr int SCAN_INTS = RES_MAX_THREADS;
constexpr int FLAG_INTS = 2;            // per-step "a bead left its skin" flags, alternating by step parity
// Noise offload (two beads per thread): a second-pass bead owned by a wave
// of the first SIMD (wave % 4 == 0) draws its normals through the thread
// RNG_HELP places further on, which has no second-pass bead of its own; the
// helper draws them one step ahead into LDS (two buffers by step parity).
// The first SIMD carries one more second-pass wave than the others when a
// trajectory is not a multiple of 256 beads; this moves the HybridTaus and
// Box-Muller work of its second-pass beads to an idle SIMD.
constexpr int RNG_HELP = 6 * 64;
constexpr int RNG_SLOTS = 128;          // offloaded beads at most (two waves)
constexpr int RNG_F4 = 2 * RNG_SLOTS * 2;   // float4: [parity][slot][rx, ra]
__device__ __forceinline__ int rng_slot(int t) { return (t / 256) * 64 + (t % 64); }
// Whether thread t's second-pass bead draws through a helper (t + RNG_HELP).
__device__ __forceinline__ bool rng_offloaded(int t, int m2, int nthreads) {
    return (t / 64) % 4 == 0 && t < m2 && t + RNG_HELP < nthreads && t + RNG_HELP >= m2 && rng_slot(t) < RNG_SLOTS;
}
// LJ entries copied to LDS are those within LJ_CUT + 2 SKIN_HALF (+ margin)
// of the bead at the launch's first step; while every bead stays within
// SKIN_HALF of where it was then, no dropped pair can come below LJ_CUT.
constexpr float SKIN_HALF = 0.75f;
constexpr float FILTER_R = LJ_CUT + 2.f * SKIN_HALF + 0.01f;
// Minimum room for list entries per bead when sizing the plan.
constexpr int MIN_ENTRIES_PER_BEAD = 24;
// List entries a thread requests at once when it fills its bead's place.
constexpr int FILL_BATCH = 8;

// Packed counts: bit 0 harmonic present, bits 1-4 longitudinal, 5-9 lateral,
// 10-19 LJ.
__device__ __forceinline__ int pack_counts(int h, int nlon, int nlat, int nlj) {
    return (h ? 1 : 0) | (nlon << 1) | (nlat << 5) | (nlj << 10);
}

// Lists compacted in LDS at ent[off]: the LDS address of the neighbour's
// position (LdsAcc's handle), a bond's flag in bit 0.  Made once per launch
// by threads that keep their bead's state: the harmonic entry itself, and the
// addresses of the others.
template <bool HELD>
struct LdsLists {
    int eh, cnt, elon, elat0, elat1;   // the harmonic entry; HELD: the first longitudinal and two lateral ones
    uint32_t alon, alat, alj;
    __device__ __forceinline__ static int at(uint32_t a, int k) {
        return *(const __attribute__((address_space(3))) uint16_t *)(uintptr_t)(a + 2 * k);
    }
    __device__ __forceinline__ LdsLists(const uint16_t *ent, int off, int c) : cnt(c) {
        const uint32_t a = lds_addr(ent) + 2 * off;
        eh = c & 1 ? at(a, 0) : -1;
        alon = a + 2 * (c & 1);
        alat = alon + 2 * nlon();
        alj = alat + 2 * nlat();
        elon = HELD && nlon() > 0 ? at(alon, 0) : 0;
        elat0 = HELD && nlat() > 0 ? at(alat, 0) : 0;
        elat1 = HELD && nlat() > 1 ? at(alat, 1) : 0;
    }
    __device__ __forceinline__ int harm() const { return eh; }
    __device__ __forceinline__ int nlon() const { return (cnt >> 1) & 15; }
    __device__ __forceinline__ int lon(int k) const { return HELD && k == 0 ? elon : at(alon, k); }
    __device__ __forceinline__ int nlat() const { return (cnt >> 5) & 31; }
    __device__ __forceinline__ int lat(int k) const { return HELD && k == 0 ? elat0 : HELD && k == 1 ? elat1 : at(alat, k); }
    __device__ __forceinline__ uint32_t ref(int e) const { return e & 0xfff0; }
    template <class Four, class One>
    __device__ __forceinline__ void lj(const Four &four, const One &one) const {
        const int n = cnt >> 10;
        int k = 0;
        for (; k + 4 <= n; k += 4) four(at(alj, k), at(alj, k + 1), at(alj, k + 2), at(alj, k + 3));
        for (; k < n; k++) one(at(alj, k));
    }
};

// A bead's state as LDS holds it: position (w: packed flags), rotated offsets
// with the Euler angles in w (n|fi, p1|theta, p2|psi).
struct BeadState {
    float4 x, n, p1, p2;
};
__device__ __forceinline__ BeadState load_state(const LdsAcc &A, int i) {
    const uint32_t h = A.origin() + i * LdsAcc::SCALE;
    return {A.xyz(h), A.fn(h), A.lat(h, false), A.lat(h, true)};
}
// The state at position x with angles a; trig = (sin theta, cos theta, sin
// psi, cos psi).
__device__ __forceinline__ BeadState new_state(float4 x, float4 a, const LatOffsets &L, float4 &trig) {
    const Frame f = make_frame(a.x, a.y, a.z, L);
    trig = make_float4(f.st, f.ct, f.sp, f.cp);
    return {x, make_float4(f.n.x, f.n.y, f.n.z, a.x), make_float4(f.p1.x, f.p1.y, f.p1.z, a.y),
            make_float4(f.p2.x, f.p2.y, f.p2.z, a.z)};
}

// What a thread carries from step to step for each of its beads.
template <int PT>
struct Lanes {
    bool mob[PT];
    int ib[PT];             // local index
    uint4 s0[PT], s1[PT];   // HybridTaus states
    float4 trig[PT];
};

// The step loop over steps [first, nsteps).  FILTERED: the LJ lists in LDS
// hold only the pairs within FILTER_R at step `first`; each mobile bead's
// displacement from its position then is checked every step, and once any
// bead of the trajectory has moved SKIN_HALF or more the loop returns the
// next step, for the caller to restore the full lists before that step's
// force evaluation (dropped pairs contribute exactly zero force until then,
// so the sums are those over the full lists) and go on unfiltered.
// Returns nsteps when every step ran.
//
// A step has two phases, one before each barrier: forces and update from the
// old state in LDS, and the stores of the new one.  With one bead per thread
// the new frame belongs to the first phase, the normals of the next step,
// which need no neighbour, to the second (drawn while the stores drain), and
// the thread keeps its bead's state and list position in registers.  Several
// beads per thread leave no registers for that: state read back from LDS,
// normals drawn where they are used, frames made before they are stored.
template <int PT, bool FILTERED, bool PERIODIC, class Lists, class MakeLists>
__device__ __forceinline__ int run_steps(const ForceK &K0, const DevTopo &T, const LdsAcc &A, int t, float4 *lx,
                                         float4 *ln, float4 *l1, float4 *l2, Lanes<PT> &W, const float *noise,
                                         int first, int nsteps, const LatOffsets &L0, const MakeLists &make_lists,
                                         int *flags, float4 *rbuf, int own_slot, int help_slot) {
    const int base = T.tbase[t], nb = T.nb;
    const float box = PERIODIC ? T.tbox[t] : 0.f, ibox = inv_side(box);
    constexpr bool KEEP = PT == 1;
    ForceK K = K0;
    LatOffsets L = L0;
    if (KEEP) {   // constants used several times a step: 2 cycles an operation, 4 with a scalar operand
        for (float *c : {&K.dtg, &K.vR, &K.fi_h, &K.psi_h, &K.lat_d, &K.seam_d, &L.p1x, &L.p1y, &L.p1z}) *c = in_vgpr(*c);
    }
    const float wall_z = K.is_wall ? T.zs[t] : 0.f;
    float3 xr[PT];
#pragma unroll
    for (int k = 0; k < PT; k++) xr[k] = FILTERED && W.mob[k] ? f3(lx[W.ib[k]]) : make_float3(0.f, 0.f, 0.f);
    BeadState st;     // KEEP: the bead's state
    float4 rx1, ra1;  // and its next normals
    if (KEEP && W.mob[0]) {
        st = load_state(A, W.ib[0]);
        if (!noise) {
            rx1 = normals4(W.s0[0]);
            ra1 = normals4(W.s1[0]);
        }
    }
    const Lists own = make_lists(W.ib[0], base + W.ib[0], KEEP && W.mob[0]);
    for (int s = first; s < nsteps; s++) {
        float4 nx[PT], na[PT];
        bool moved = false;
#pragma unroll
        for (int k = 0; k < PT; k++) {
            if (!W.mob[k]) continue;
            const int i = W.ib[k];
            const int b = base + i;
            const BeadState B = KEEP ? st : load_state(A, i);
            float4 x = B.x, a = make_float4(B.n.w, B.p1.w, B.p2.w, 0.f);
            Own I = make_own_trig(x, a, B.n, B.p1, B.p2, W.trig[k], __float_as_int(x.w));
            if (PERIODIC) I.box = box, I.ibox = ibox;
            float F[6];
            bead_force<PERIODIC>(K, A, KEEP ? own : make_lists(i, b, true), wall_z, I, F);
            float4 rx, ra;
            if (noise) {
                const float *nz = noise + (size_t)s * 6 * nb + 6 * (size_t)b;
                rx = make_float4(nz[0], nz[1], nz[2], 0.f);
                ra = make_float4(nz[3], nz[4], nz[5], 0.f);
            } else if (KEEP) {
                rx = rx1;
                ra = ra1;
            } else if (k == 1 && own_slot >= 0) {   // drawn by the helper (PT == 2)
                rx = rbuf[((s & 1) * RNG_SLOTS + own_slot) * 2];
                ra = rbuf[((s & 1) * RNG_SLOTS + own_slot) * 2 + 1];
            } else {
                rx = normals4(W.s0[k]);
                ra = normals4(W.s1[k]);
            }
            em_update(K, F, rx, ra, x, a);
            if (KEEP) {
                st = new_state(x, a, L, W.trig[k]);   // x.w keeps the packed flags
            } else {
                nx[k] = x;
                na[k] = a;
            }
            if (FILTERED) {
                const float dx = x.x - xr[k].x, dy = x.y - xr[k].y, dz = x.z - xr[k].z;
                moved |= dx * dx + dy * dy + dz * dz >= SKIN_HALF * SKIN_HALF;
            }
        }
        if (PT == 2 && help_slot >= 0 && s + 1 < nsteps) {   // the owner's draws of the next step
            rbuf[(((s + 1) & 1) * RNG_SLOTS + help_slot) * 2] = normals4(W.s0[PT - 1]);
            rbuf[(((s + 1) & 1) * RNG_SLOTS + help_slot) * 2 + 1] = normals4(W.s1[PT - 1]);
        }
        if (FILTERED && moved) flags[s & 1] = 1;
        __syncthreads();
        const bool left = FILTERED && flags[s & 1] != 0;
        if (FILTERED && threadIdx.x == 0) flags[(s + 1) & 1] = 0;   // read at the next step, after its barrier
#pragma unroll
        for (int k = 0; k < PT; k++) {
            if (!W.mob[k]) continue;
            const int i = W.ib[k];
            if (!KEEP) st = new_state(nx[k], na[k], L, W.trig[k]);
            lx[i] = st.x;
            ln[i] = st.n;
            l1[i] = st.p1;
            l2[i] = st.p2;
            if (KEEP && !noise && s + 1 < nsteps && !left) {   // (after leaving, the next call draws them)
                rx1 = normals4(W.s0[0]);
                ra1 = normals4(W.s1[0]);
            }
        }
        __syncthreads();
        if (left) return s + 1;   // uniform: every thread read the same flag
    }
    return nsteps;
}

// The step loop with two waves to each 64 beads: thread t < nmain owns bead
// W.ib[0] as in run_steps<1, ...>, thread t + nmain helps it.  The helper sums
// the bead's LJ forces while the owner sums its bonds, and draws its next
// normals while the owner moves it; both pass through xbuf (per main thread
// the LJ sum and two pairs of normals by step parity).  The sums are added as
// run_steps adds them: the same values.  `drawn`: the helper has drawn the
// normals of step `first` already.
constexpr int XBUF_F4 = 5;
template <bool FILTERED, bool PERIODIC, class Lists, class MakeLists>
__device__ __forceinline__ int run_steps_helped(const ForceK &K0, const DevTopo &T, const LdsAcc &A, int t, float4 *lx,
                                                float4 *ln, float4 *l1, float4 *l2, Lanes<1> &W, const float *noise,
                                                int first, int nsteps, const LatOffsets &L0,
                                                const MakeLists &make_lists, int *flags, float4 *xbuf, int nmain,
                                                bool drawn) {
    const int base = T.tbase[t], nb = T.nb;
    const float box = PERIODIC ? T.tbox[t] : 0.f, ibox = inv_side(box);
    ForceK K = K0;
    LatOffsets L = L0;
    for (float *c : {&K.dtg, &K.vR, &K.fi_h, &K.psi_h, &K.lat_d, &K.seam_d, &L.p1x, &L.p1y, &L.p1z}) *c = in_vgpr(*c);
    const float wall_z = K.is_wall ? T.zs[t] : 0.f;
    const bool helper = (int)threadIdx.x >= nmain;   // uniform in a wave
    const int main_t = threadIdx.x - (helper ? nmain : 0);
    float4 *xlj = xbuf + main_t, *xrx = xbuf + nmain + main_t, *xra = xbuf + 3 * nmain + main_t;   // normals: + parity nmain
    const int i = W.ib[0], b = base + i;
    const bool mob = W.mob[0];
    const Lists own = make_lists(i, b, mob);
    BeadState st{};
    if (mob) st = load_state(A, i);
    const float3 xr = f3(st.x);
    auto draw = [&](int s) {
        xrx[(s & 1) * nmain] = normals4(W.s0[0]);
        xra[(s & 1) * nmain] = normals4(W.s1[0]);
    };
    if (helper && mob && !noise && !drawn) draw(first);
    for (int s = first; s < nsteps; s++) {
        float F[6];
        if (mob) {
            Own I;
            if (helper) {
                if (K.lj_on) {
                    I.r = f3(lds_f4(A.origin() + i * LdsAcc::SCALE));
                    I.box = box, I.ibox = ibox;
                    const float3 f = lj_sum<PERIODIC>(K, A, own, I);
                    *xlj = make_float4(f.x, f.y, f.z, 0.f);
                }
            } else {
                const float4 a = make_float4(st.n.w, st.p1.w, st.p2.w, 0.f);
                I = make_own_trig(st.x, a, st.n, st.p1, st.p2, W.trig[0], __float_as_int(st.x.w));
                if (PERIODIC) I.box = box, I.ibox = ibox;
                bond_total(bond_forces<PERIODIC>(K, A, own, I), I, F);
            }
        }
        __syncthreads();
        if (FILTERED && threadIdx.x == 0) flags[(s + 1) & 1] = 0;   // all have read it (after the last step's end)
        if (mob) {
            if (helper) {
                if (!noise && s + 1 < nsteps) draw(s + 1);
            } else {
                add_lj_walls(K, f3(*xlj), wall_z, f3(st.x), F);
                float4 rx, ra;
                if (noise) {
                    const float *nz = noise + (size_t)s * 6 * nb + 6 * (size_t)b;
                    rx = make_float4(nz[0], nz[1], nz[2], 0.f);
                    ra = make_float4(nz[3], nz[4], nz[5], 0.f);
                } else {
                    rx = xrx[(s & 1) * nmain];
                    ra = xra[(s & 1) * nmain];
                }
                float4 x = st.x, a = make_float4(st.n.w, st.p1.w, st.p2.w, 0.f);
                em_update(K, F, rx, ra, x, a);
                st = new_state(x, a, L, W.trig[0]);   // x.w keeps the packed flags
                lx[i] = st.x;
                ln[i] = st.n;
                l1[i] = st.p1;
                l2[i] = st.p2;
                if (FILTERED) {
                    const float dx = x.x - xr.x, dy = x.y - xr.y, dz = x.z - xr.z;
                    if (dx * dx + dy * dy + dz * dz >= SKIN_HALF * SKIN_HALF) flags[s & 1] = 1;
                }
            }
        }
        __syncthreads();
        // uniform: set before the barrier, and next written after the barrier
        // of the following step or, when this returns, never again
        if (FILTERED && flags[s & 1] != 0) return s + 1;
    }
    return nsteps;
}

template <int PT, int MAXT, bool PERIODIC, bool HELPED = false>
__global__ void __launch_bounds__(MAXT)
    k_resident(ForceK K, float ljpairscutoff, DevTopo T, DevState S, uint4 *seeds, const float *noise, int nsteps, LatOffsets L,
               int stride, int entry_cap, const int *order) {
    extern __shared__ float4 lds[];
    const int overflow = *(volatile const int *)T.overflow;
    float4 *lx = lds, *ln = lds + stride, *l1 = lds + 2 * stride, *l2 = lds + 3 * stride;
    float4 *rbuf = lds + STATE_ARRAYS * stride;
    static_assert(!HELPED || PT == 1, "a helper serves one bead");
    const int nmain = HELPED ? blockDim.x / 2 : blockDim.x;   // threads that own beads
    const bool helper = HELPED && (int)threadIdx.x >= nmain;
    float4 *xbuf = rbuf + RNG_F4;
    int *hoff = reinterpret_cast<int *>(xbuf + (HELPED ? XBUF_F4 * nmain : 0));
    int *hcnt = hoff + stride;
    int *scan = hcnt + stride;
    int *flags = scan + SCAN_INTS;
    uint16_t *ent = reinterpret_cast<uint16_t *>(flags + FLAG_INTS);
    const int t = blockIdx.x;
    const int base = T.tbase[t], n = T.tsize[t];
    const int nb = T.nb;
    if (threadIdx.x == 0) flags[0] = 0;
    stage_state(T, S, base, n, lx, ln, l1, l2);
    Lanes<PT> W;   // this thread's lane slots (order: immobile beads last)
    int lcnt[PT];   // its list counts, packed as in hcnt
    // everything a bead needs is requested at once, of the trajectory's last
    // bead where a slot has none, before its flags tell whether it is mobile
#pragma unroll
    for (int k = 0; k < PT; k++) {
        const int slot = (helper ? threadIdx.x - nmain : threadIdx.x) + k * blockDim.x;
        const int i = order[base + min(slot, n - 1)], b = base + i;
        const int fl = T.flags[b], h = T.harm[b], c0 = T.lon_n[b], c1 = T.lat_n[b], c2 = T.lj_n[b];
        const float4 a = S.ang[b];
        if (!noise) {
            W.s0[k] = seeds[b];
            W.s1[k] = seeds[b + nb];
        }
        W.ib[k] = i;
        W.mob[k] = slot < n && is_mobile(fl);
        lcnt[k] = W.mob[k] ? pack_counts(h >= 0, c0, c1, K.lj_on ? c2 : 0) : 0;
        sincos_fast(a.y, &W.trig[k].x, &W.trig[k].y);
        sincos_fast(a.z, &W.trig[k].z, &W.trig[k].w);
    }
    // A rebuild that ran out of list capacity stops the dynamics: the state
    // and RNG streams stay at that rebuild's step, and the host reports the
    // error with the steps not taken (every thread returns before any
    // barrier).
    if (overflow) {
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(T.frozen, nsteps);
        return;
    }
    // noise offload roles (two beads per thread, drawn noise); the first
    // wave offloads too only when a later second-pass wave of the first SIMD
    // has work (its lanes past the mobile beads hold the immobile ones)
    const int m2 = n - (int)blockDim.x;
    // (flags[0] was cleared before the first barrier; the skin test clears it
    // again before its first use)
    __syncthreads();
    if (PT == 2 && threadIdx.x >= 256 && W.mob[PT - 1]) flags[0] = 1;
    __syncthreads();
    const bool tail_busy = flags[0] != 0;
    auto offloaded = [&](int tt) {
        return PT == 2 && !noise && rng_offloaded(tt, m2, blockDim.x) && (tt >= 256 || tail_busy);
    };
    const int own_slot = offloaded(threadIdx.x) ? rng_slot(threadIdx.x) : -1;
    const int owner = (int)threadIdx.x - RNG_HELP;
    int help_slot = -1, help_b = -1;
    if (owner >= 0 && offloaded(owner)) {
        const int b = base + order[base + owner + blockDim.x];   // the owner's second-pass bead
        if (is_mobile(T.flags[b])) {
            help_slot = rng_slot(owner);
            help_b = b;
            W.s0[PT - 1] = seeds[b];
            W.s1[PT - 1] = seeds[b + nb];
            rbuf[help_slot * 2] = normals4(W.s0[PT - 1]);   // step 0's draws (parity 0)
            rbuf[help_slot * 2 + 1] = normals4(W.s1[PT - 1]);
        }
    }
    __syncthreads();
    const LdsAcc A(lx, ln, l1, l2);
    const float box = PERIODIC ? T.tbox[t] : 0.f, ibox = inv_side(box);
    // LJ entries of bead i kept in LDS: all of them (rf2 == 0), or those
    // within sqrt(rf2) of it now.
    auto lj_keep = [lx, box, ibox](int i, int j, float rf2) {
        if (rf2 == 0.f) return true;
        const float3 d = min_image_pre(sub3(f3(lx[i]), f3(lx[j])), box, ibox);
        return d.x * d.x + d.y * d.y + d.z * d.z < rf2;
    };
    // Offsets of this trajectory's full lists in LDS, for the mobile beads
    // (the only ones whose forces are computed): the per-bead totals go
    // through a block scan into hoff.  Returns the number of entries.  Every
    // later fill writes at these offsets (a filtered list uses a prefix of
    // its bead's place), so the layout is computed once per launch.
    auto handle = [&](int j) { return A.origin() + (uint32_t)((j - base) * LdsAcc::SCALE); };
    auto layout = [&]() {
        for (int i = threadIdx.x; i < n; i += blockDim.x) hoff[i] = 0;   // immobile beads use no lists
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PT; k++) {
            if (!W.mob[k] || helper) continue;
            const int i = W.ib[k], hc = lcnt[k];
            hcnt[i] = hc;
            hoff[i] = (hc & 1) + ((hc >> 1) & 15) + ((hc >> 5) & 31) + (hc >> 10);
        }
        // Chunked exclusive scan: thread t owns beads [t*c, (t+1)*c); a wave
        // scans its lanes' chunk totals by shuffles, the first wave the
        // wave totals.
        const int c = (n + blockDim.x - 1) / blockDim.x;
        __syncthreads();
        int run = 0;
        const int lo = threadIdx.x * c, hi = min(n, lo + c);
        for (int i = lo; i < hi; i++) run += hoff[i];
        const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
        int inc = run;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(inc, d, 64);
            if (lane >= d) inc += v;
        }
        if (lane == 63) scan[wv] = inc;
        __syncthreads();
        if (wv == 0) {
            int w = lane < nw ? scan[lane] : 0;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(w, d, 64);
                if (lane >= d) w += v;
            }
            if (lane < nw) scan[lane] = w;
        }
        __syncthreads();
        const int total = scan[nw - 1];
        int acc = (wv ? scan[wv - 1] : 0) + inc - run;   // exclusive prefix of this chunk
        for (int i = lo; i < hi; i++) {
            const int v = hoff[i];
            hoff[i] = acc;
            acc += v;
        }
        __syncthreads();
        return total;
    };
    // Copy the lists into their places, of the LJ entries only those
    // lj_keep admits; hcnt's LJ field records the number copied.  A bead's
    // entries (harmonic, longitudinal, lateral, LJ: the full counts of the
    // layout) are requested FILL_BATCH at a time, each from its own array.
    // Each thread fills the places of its own mobile beads.
    int nent = 0;   // entries of the full lists (layout)
    auto fill = [&](float rf2) {
#pragma unroll
        for (int kk = 0; kk < PT; kk++) {
            if (!W.mob[kk] || helper) continue;
            const int i = W.ib[kk], b = base + i;
            const int hc = hcnt[i];
            const int h = hc & 1, nlon = (hc >> 1) & 15, nlat = (hc >> 5) & 31;
            const int nbond = h + nlon + nlat;
            const int o0 = hoff[i];
            const int nall = (i + 1 < n ? hoff[i + 1] : nent) - o0;
            int o = o0, nlj = 0;
            int spare[3] = {0, 0, 0}, nspare = 0;   // the last three dropped
            for (int k0 = 0; k0 < nall; k0 += FILL_BATCH) {
                int v[FILL_BATCH];
#pragma unroll
                for (int u = 0; u < FILL_BATCH; u++) {
                    const int k = k0 + u;
                    const int *src = k < h          ? T.harm
                                     : k < h + nlon ? T.lon + (size_t)(k - h) * nb
                                     : k < nbond    ? T.lat + (size_t)(k - h - nlon) * nb
                                                    : T.lj + (size_t)(k - nbond) * nb;
                    v[u] = k < nall ? src[b] : 0;
                }
#pragma unroll
                for (int u = 0; u < FILL_BATCH; u++) {
                    const int k = k0 + u;
                    if (k < nbond) {
                        ent[o++] = (uint16_t)(handle(ent_j(v[u])) | ent_f(v[u]));
                    } else if (k < nall) {
                        if (lj_keep(i, v[u] - base, rf2)) {
                            ent[o++] = (uint16_t)handle(v[u]);
                            nlj++;
                        } else {
                            spare[2] = spare[1];
                            spare[1] = spare[0];
                            spare[0] = v[u];
                            nspare++;
                        }
                    }
                }
            }
            // Dropped entries, which contribute nothing, fill the list up to
            // a multiple of the four that lj_sum takes at once: a remainder
            // runs one entry at a time, for the whole wave.
#pragma unroll
            for (int u = 0; u < 3; u++)
                if ((nlj & 3) != 0 && u < nspare) {
                    ent[o++] = (uint16_t)handle(spare[u]);
                    nlj++;
                }
            hcnt[i] = (hc & 1023) | (nlj << 10);
        }
        __syncthreads();
    };
    // The full lists decide between LDS and global lists; in LDS, the LJ
    // lists are filtered by distance when the list cutoff reaches beyond
    // FILTER_R (the full lists fit, so a refill always fits too).
    nent = layout();
    const bool use_lds = nent <= entry_cap;
    if (use_lds) {
        const bool filter = K.lj_on && ljpairscutoff > FILTER_R;
        fill(filter ? FILTER_R * FILTER_R : 0.f);
        using LL = LdsLists<PT == 1>;
        auto mk = [&](int i, int, bool lists) { return LL(ent, lists ? hoff[i] : 0, lists ? hcnt[i] : 0); };
        int s = 0;
        if (filter) {
            // Cleared once, before the loop that reads them, and not again at
            // the refill, where waves of the helped loop may still be reading
            // the flag that ended it (after that step's last barrier).
            if (threadIdx.x == 0) flags[0] = flags[1] = 0;
            __syncthreads();
            if constexpr (HELPED)
                s = run_steps_helped<true, PERIODIC, LL>(K, T, A, t, lx, ln, l1, l2, W, noise, 0, nsteps, L, mk, flags,
                                                         xbuf, nmain, false);
            else
                s = run_steps<PT, true, PERIODIC, LL>(K, T, A, t, lx, ln, l1, l2, W, noise, 0, nsteps, L, mk, flags, rbuf,
                                                      own_slot, help_slot);
            if (s < nsteps) fill(0.f);   // a bead left its skin: the full lists from step s on
        }
        if (s < nsteps) {
            if constexpr (HELPED)
                run_steps_helped<false, PERIODIC, LL>(K, T, A, t, lx, ln, l1, l2, W, noise, s, nsteps, L, mk, flags, xbuf,
                                                      nmain, s > 0);
            else
                run_steps<PT, false, PERIODIC, LL>(K, T, A, t, lx, ln, l1, l2, W, noise, s, nsteps, L, mk, flags, rbuf,
                                                   own_slot, help_slot);
        }
    } else {
        using Lists = GlobalLists<LdsAcc::SCALE>;
        auto mk = [&](int, int b, bool) { return Lists{T, b, base, A.origin()}; };
        if constexpr (HELPED)
            run_steps_helped<false, PERIODIC, Lists>(K, T, A, t, lx, ln, l1, l2, W, noise, 0, nsteps, L, mk, flags, xbuf,
                                                     nmain, false);
        else
            run_steps<PT, false, PERIODIC, Lists>(K, T, A, t, lx, ln, l1, l2, W, noise, 0, nsteps, L, mk,
                                          flags, rbuf, own_slot, help_slot);
    }
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int b = base + i;
        float4 x = lx[i], fn = ln[i], f1 = l1[i], f2 = l2[i];
        x.w = 0.f;
        S.xyz[b] = x;
        S.ang[b] = make_float4(fn.w, f1.w, f2.w, 0.f);
        fn.w = f1.w = f2.w = 0.f;
        S.fn[b] = fn;
        S.fp1[b] = f1;
        S.fp2[b] = f2;
    }
#pragma unroll
    for (int k = 0; k < PT; k++) {
        if (W.mob[k] && !noise && (!HELPED || helper) && !(k == 1 && own_slot >= 0)) {   // an offloaded bead's state is the helper's
            const int b = base + W.ib[k];
            seeds[b] = W.s0[k];
            seeds[b + nb] = W.s1[k];
        }
    }
    if (help_b >= 0) {
        seeds[help_b] = W.s0[PT - 1];
        seeds[help_b + nb] = W.s1[PT - 1];
    }
}

static size_t fixed_lds_bytes(int nmax) {
    return (size_t)STATE_ARRAYS * sizeof(float4) * nmax + (size_t)RNG_F4 * sizeof(float4) +
           (size_t)HDR_INTS * sizeof(int) * nmax + (size_t)(SCAN_INTS + FLAG_INTS) * sizeof(int);
}

// Launch plan with pt beads per thread (pt = 1 allows up to 1024 threads,
// 2 and 3 up to 768 so the multi-bead kernels keep their registers).  Where
// the mobile beads fill at most half the largest workgroup, every bead gets a
// second thread (run_steps_helped): a wave alone on its SIMD spends 7500
// cycles on a step, most of them waiting, and the idle half of the workgroup
// takes the two longest independent parts of it.  Per 100 steps, through the
// API: 1, 256 and 700 tubes of 312 beads 390 -> 288, 514 -> 422 and 1323 ->
// 1057 us, 1 and 512 tubes of 520 beads (494 mobile) 370 -> 327 and 1079 ->
// 1000, 256 of 910 beads (500 mobile) 431 with two beads per thread, 365.
// From 922 beads on the LDS has no room for the helpers' buffer: one bead per
// thread alone (64 tubes of 1040 beads, 500 mobile: 405 with two, 394).
bool resident_plan_for(const mte_engine *e, int pt, ResidentPlan *plan) {
    *plan = ResidentPlan{};
    if (e->P.tea_on || pt < 1 || pt > RES_MAX_PT) return false;
    int nmax = 0;
    for (int t = 0; t < e->ntraj; t++) nmax = std::max<int>(nmax, (int)(e->off[t + 1] - e->off[t]));
    if (nmax > 4096) return false;   // uint16 list entries (16 x the local index: the position array is at LDS address 0)
    int lds_limit = 0;
    if (hipDeviceGetAttribute(&lds_limit, hipDeviceAttributeMaxSharedMemoryPerBlock, e->device) != hipSuccess)
        return false;
    const int nmain = std::min(((nmax + 63) / 64) * 64, RES_MAX_THREADS / 2);
    auto room = [&](size_t fixed) { return fixed + (size_t)MIN_ENTRIES_PER_BEAD * 2 * nmax <= (size_t)lds_limit; };
    const size_t alone = fixed_lds_bytes(nmax), with_xbuf = alone + (size_t)XBUF_F4 * sizeof(float4) * nmain;
    const bool helped = pt == 1 && e->res_mobile_max <= nmain && room(with_xbuf);
    const size_t fixed = helped ? with_xbuf : alone;
    if (!room(fixed)) return false;
    int threads = (nmax + pt - 1) / pt;
    threads = ((threads + 63) / 64) * 64;
    // One bead per thread also covers a trajectory longer than the largest
    // workgroup when every bead past it is immobile: the lane order puts the
    // mobile beads first, and an immobile bead needs its place in LDS only.
    if (pt == 1 && threads > RES_MAX_THREADS && e->res_mobile_max <= RES_MAX_THREADS) threads = RES_MAX_THREADS;
    // Two beads per thread run on 12 waves when the batch allows: the
    // second-pass beads then leave idle waves on the third SIMD for the
    // noise offload.
    if (pt == 2 && nmax > RES_MULTI_THREADS) threads = RES_MULTI_THREADS;
    if (helped) threads = 2 * nmain;
    if (threads > (pt == 1 ? RES_MAX_THREADS : RES_MULTI_THREADS)) return false;
    plan->threads = threads;
    plan->per_thread = pt;
    plan->helped = helped;
    plan->max_beads = nmax;
    plan->lds_bytes = (size_t)lds_limit & ~(size_t)15;
    plan->entry_cap = (int)std::min<size_t>((plan->lds_bytes - fixed) / 2, 1u << 30);
    return true;
}

// Default plan: the fewest beads per thread the batch allows.
bool resident_fits(const mte_engine *e, ResidentPlan *plan) {
    for (int pt = 1; pt <= RES_MAX_PT; pt++)
        if (resident_plan_for(e, pt, plan)) return true;
    return false;
}

template <int PT, int MAXT, bool PERIODIC, bool HELPED = false>
static hipError_t launch_pt(mte_engine *e, int nsteps, const float *noise) {
    const ResidentPlan &pl = e->rplan;
    hipError_t s = hipFuncSetAttribute((const void *)k_resident<PT, MAXT, PERIODIC, HELPED>,
                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds_bytes);
    if (s != hipSuccess) return s;
    hipLaunchKernelGGL((k_resident<PT, MAXT, PERIODIC, HELPED>), dim3(e->ntraj), dim3(pl.threads), pl.lds_bytes, e->stream, e->K,
                       e->P.ljpairscutoff, e->T, e->S[e->cur], e->seeds, noise, nsteps, e->L, pl.max_beads, pl.entry_cap, e->res_order);
    return hipGetLastError();
}

template <bool PERIODIC>
static hipError_t launch_box(mte_engine *e, int nsteps, const float *noise) {
    switch (e->rplan.per_thread) {
    case 1:
        return e->rplan.helped ? launch_pt<1, RES_MAX_THREADS, PERIODIC, true>(e, nsteps, noise)
                               : launch_pt<1, RES_MAX_THREADS, PERIODIC>(e, nsteps, noise);
    case 2: return launch_pt<2, RES_MULTI_THREADS, PERIODIC>(e, nsteps, noise);
    case 3: return launch_pt<3, RES_MULTI_THREADS, PERIODIC>(e, nsteps, noise);
    default: return hipErrorInvalidValue;
    }
}

// Batches with a periodic box take the kernels with the minimum image; there
// an open trajectory's separations are unchanged (side and inverse zero).
hipError_t launch_resident(mte_engine *e, int nsteps, const float *noise) {
    return e->periodic ? launch_box<true>(e, nsteps, noise) : launch_box<false>(e, nsteps, noise);
}

}  // namespace mte
