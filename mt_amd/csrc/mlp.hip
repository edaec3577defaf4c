// mlp.hip -- the learned hydrodynamic correction (MLP-HI); the reference has
// no counterpart.
//
// Per bead i the engine predicts the local hydrodynamic tensor
//   G_i = sum_{j != i, r_ij < 12 nm} phi(r_ij) D_hat_ij
// (D_hat the RPY block of src/bdhitea_kernel.cu:38-58, phi = 1 up to 8 nm and
// a cosine taper to 0 at 12 nm) from the relative positions of its 32 nearest
// neighbours (96 inputs), with a 96-128-128-128-9 tanh network, and replaces
// TEA's per-step O(N^2) pair sums by it (k_mlp_step), keeping TEA's beta and
// C_i normalisation.  The exact G_i (the same neighbour sum over every
// neighbour within 12 nm) is the training label and the sampled-error judge;
// plain TEA is the fallback.
//
// Kernels: neighbour features and exact labels over the hashed cell tables
// (cs >= 12 nm); inference fused with the integrator on the matrix cores
// (v_mfma_f32_16x16x32_bf16: bf16 weights, activations carried as bf16
// hi + lo pairs, FP32 accumulation; the weight fragments sit in LDS and the
// activations stay in registers from layer to layer); training (forward,
// backward and weight gradients of a sample tile in one kernel, then the
// reduction over tiles with the Adam step) in FP32 on the matrix cores.
#include "engine_internal.h"

#include <mutex>
#include <type_traits>

namespace mte {

constexpr int MLP_BLOCK = MLP_SEARCH_BLOCK;
constexpr int MLP_LANES = 4;   // lanes per bead of the neighbour search
constexpr float MLP_RC = 12.f, MLP_RIN = 8.f;
constexpr float MLP_CELL = 2.f * MLP_RC + 0.02f;   // search cells: the margin is far above the rounding of a
                                                   // bead's place in its cell
// flat parameter offsets
constexpr int OW1 = 0, OB1 = OW1 + MLP_IN * MLP_H, OW2 = OB1 + MLP_H, OB2 = OW2 + MLP_H * MLP_H, OW3 = OB2 + MLP_H,
              OB3 = OW3 + MLP_H * MLP_H, OW4 = OB3 + MLP_H, OB4 = OW4 + MLP_H * MLP_OUT;
static_assert(OB4 + MLP_OUT == MLP_NPARAM, "parameter layout");

__device__ __forceinline__ float taper(float r) {
    if (r <= MLP_RIN) return 1.f;
    if (r >= MLP_RC) return 0.f;
    float s, c;
    sincos_fast(3.14159265358979f * (r - MLP_RIN) / (MLP_RC - MLP_RIN), &s, &c);
    return 0.5f * (1.f + c);
}

// ------------------------------------------------------------ features, labels
constexpr int FEAT_BLK_NN = 8;   // neighbours per block of written features (24 floats: whole
                                 // float4 stores and whole 8-float MFMA operand slices)
static_assert(3 * FEAT_BLK_NN % 8 == 0 && FEAT_BLK_NN % 4 == 0 && FEAT_BLK_NN * MLP_LANES == MLP_NN,
              "feature blocks, one per lane of the bead");
// A bucket's range as [first, end) slots of the bucket-ordered positions.  A
// trajectory's beads hold the slots [base, base + n) of its buckets, so with
// trajectory-local indices of 16 bits (n < 65536) both ends pack into one
// word.
template <typename JT>
struct BucketRange {
    using W = int2;
    __device__ __forceinline__ static W pack(int2 r, int) { return make_int2(r.x, r.x + r.y); }
    __device__ __forceinline__ static W none() { return make_int2(0, 0); }
    __device__ __forceinline__ static int lo(W w, int) { return w.x; }
    __device__ __forceinline__ static int hi(W w, int) { return w.y; }
};
template <>
struct BucketRange<uint16_t> {
    using W = uint32_t;
    __device__ __forceinline__ static W pack(int2 r, int base) {
        const uint32_t s = (uint32_t)(r.x - base);
        return s | ((s + (uint32_t)r.y) << 16);
    }
    __device__ __forceinline__ static W none() { return 0; }
    __device__ __forceinline__ static int lo(W w, int base) { return base + (int)(w & 0xffffu); }
    __device__ __forceinline__ static int hi(W w, int base) { return base + (int)(w >> 16); }
};

// FP64 minimum and maximum of two keys (never NaN: the intrinsics would first
// quiet both operands).
__device__ __forceinline__ double key_min(double a, double b) {
    double r;
    __asm__("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ double key_max(double a, double b) {
    double r;
    __asm__("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// kn into the ascending keys, slots K0 .. K1 - 1 of them: a slot takes the
// middle one of its key, the key below and kn (from the top down).
template <int K0, int K1>
__device__ __forceinline__ void insert_key(double (&key)[MLP_NN], double kn) {
#pragma unroll
    for (int k = K1 - 1; k >= K0; k--) {
        const double low = key_min(key[k], kn);
        key[k] = k > 0 ? key_max(key[k - 1], low) : low;
    }
}
// Index of the key at slot N part + u.
template <int N>
__device__ __forceinline__ int pick_key(const double (&key)[MLP_NN], int part, int u) {
    const int j0 = __double2loint(key[u]), j1 = __double2loint(key[N + u]), j2 = __double2loint(key[2 * N + u]),
              j3 = __double2loint(key[3 * N + u]);
    return part & 2 ? (part & 1 ? j3 : j2) : (part & 1 ? j1 : j0);
}

// A value of the lane that differs in bit 0 (XOR = 1) or bit 1 (XOR = 2) of
// its number, within the four lanes of a bead.
template <int XOR>
__device__ __forceinline__ int quad_swap(int v) {
    return __builtin_amdgcn_mov_dpp(v, XOR == 1 ? 0xB1 : 0x4E, 0xF, 0xF, true);   // quad_perm 1,0,3,2 / 2,3,0,1
}
template <int XOR>
__device__ __forceinline__ double quad_swap(double v) {
    return __hiloint2double(quad_swap<XOR>(__double2hiint(v)), quad_swap<XOR>(__double2loint(v)));
}
// Orders the LDS accesses of a wave's lanes before and after it, for values
// that pass between lanes of one wave: the hardware keeps a wave's LDS accesses
// in order, and this keeps the compiler from moving them.
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// The value of lane L of the bead's four.
template <int L>
__device__ __forceinline__ int quad_lane(int v) {
    return __builtin_amdgcn_mov_dpp(v, L * 0x55, 0xF, 0xF, true);   // quad_perm L,L,L,L
}
template <int XOR>
__device__ __forceinline__ float quad_swap(float v) {
    return __int_as_float(quad_swap<XOR>(__float_as_int(v)));
}

// The first N keys of this lane and of the lane XOR of it, both ascending,
// merged: the N smallest, ascending, in both lanes.  The smaller of key k
// here and key N - 1 - k there are those N and a bitonic sequence.
template <int XOR, int N>
__device__ __forceinline__ void merge_keys(double (&key)[MLP_NN]) {
#pragma unroll
    for (int k = 0; k < N / 2; k++) {
        const double a = key[k], b = key[N - 1 - k];
        const double oa = quad_swap<XOR>(a), ob = quad_swap<XOR>(b);
        key[k] = key_min(a, ob);
        key[N - 1 - k] = key_min(b, oa);
    }
#pragma unroll
    for (int d = N / 2; d > 0; d >>= 1)
#pragma unroll
        for (int k = 0; k < N; k++)
            if ((k & d) == 0) {
                const double a = key[k], b = key[k + d];
                key[k] = key_min(a, b);
                key[k + d] = key_max(a, b);
            }
}

// Neighbour scan over eight cells of the hashed table.  Its cells are at
// least twice the radius wide, so the sphere around a bead reaches at most
// the cell on the nearer side in each direction (in a box of fewer than two
// cells the bead's own cell is the whole side, and the second one the same).
// The eight bucket ranges are loaded up front; a bucket that two of the cells
// hash to is visited once, and the candidates are streamed from the
// bucket-ordered positions.  Every bead within 12 nm lies in one of the
// cells, so visiting their buckets (each once) sees it exactly once, and the
// distance test rejects the beads of other cells sharing a bucket.  A dilute
// bead's candidates are mostly those (the tables hold one bead per two
// buckets): eight wide cells give 7 where 27 cells of the radius gave 13, for
// eight range loads instead of 27; a tube bead's grow from 120 to 160.
// Four lanes share a bead: each loads two of its ranges and visits every
// fourth candidate (of four neighbouring slots, one cache line), then the four
// sorted lists merge.  A tube's waves, few and each bound by its own
// instructions (one wave per SIMD issues at half rate), thus become four times
// as many with a quarter of the visits and insertions.  Keeps
// the 32 nearest (distance, then index) and sums the exact label over every
// neighbour within 12 nm (LABELS: only on check steps and for training data).
// The 32 nearest live in registers as 64-bit keys (the squared distance's
// float bits, which order as integers for non-negative floats, over the
// trajectory-local index), ascending, empty slots at infinity.  Read as
// doubles the keys order the same way (squared distances below 144 keep the
// exponent finite), so a candidate that precedes the last key is inserted
// with one FP64 minimum and one maximum per slot, 8 issue cycles where an
// integer comparison and four selects take 20, and without branches: a
// wave's lanes never wait on one another's shift loops, on a crowded tube
// (60-130 candidates per lane, most of them inserted).
// Measured per step, eight periodic systems of 24k-40k beads: 112 -> 45 us
// (integer keys, 27 cells, one lane per bead: 112; FP64 keys 78; eight cells
// 71; four lanes per bead 61; the dilute waves' own path 45); 8 x 1820 beads of
// tubes alone 61 -> 22 us.  Bound by dependent loads (range, candidates,
// neighbours) at three waves per SIMD: the keys take 64 of 168 registers.
// JT selects the bucket-range packing (16-bit where every
// trajectory has fewer than 65536 beads).
// With fblk, a bead's features are written only up to the 24-float block
// (8 neighbours) holding its last neighbour, and the number of blocks goes
// to fblk: the step's network reads the rest as zeros, so in a dilute box
// (a few neighbours within 12 nm) most of the 384 feature bytes per bead
// never cross HBM.
// Neighbours N part .. N part + N - 1 of a bead's sorted keys as features
// (f: the bead's row; xyz: its trajectory's positions), zeros past the last.
template <int N>
__device__ __forceinline__ void write_features(const float4 *xyz, const double (&key)[MLP_NN], int part, int cnt,
                                               float3 ri, float box, float ibox, float *f) {
    const int k0 = N * part;
    float4 xj[N];
#pragma unroll
    for (int u = 0; u < N; u++) {
        const int j = pick_key<N>(key, part, u);
        xj[u] = k0 + u < cnt ? xyz[j] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float v[3 * N];
#pragma unroll
    for (int u = 0; u < N; u++) {
        float3 d = make_float3(0.f, 0.f, 0.f);
        if (k0 + u < cnt) {
            d = min_image_pre(sub3(f3(xj[u]), ri), box, ibox);
            constexpr float irc = 1.f / MLP_RC;   // features in units of the radius
            d = make_float3(d.x * irc, d.y * irc, d.z * irc);
        }
        v[3 * u] = d.x;
        v[3 * u + 1] = d.y;
        v[3 * u + 2] = d.z;
    }
    float2 *o = reinterpret_cast<float2 *>(f + 3 * k0);
#pragma unroll
    for (int w = 0; w < 3 * N / 2; w++) o[w] = make_float2(v[2 * w], v[2 * w + 1]);
}

template <bool LABELS, typename JT>
__global__ void __launch_bounds__(MLP_BLOCK * MLP_LANES, 3)
    k_mlp_local(mte_params P, DevTopo T, DevState S, CellTables C, const int2 *blocks, float *feat, float *targ,
                uint8_t *fblk) {
    using Range = BucketRange<JT>;
    __shared__ typename Range::W srg[MLP_BLOCK][8];   // the beads' bucket ranges
    const int2 blk = blocks[blockIdx.x];
    const int t = blk.x;
    const int base = T.tbase[t];
    const int lb = threadIdx.x / MLP_LANES, part = threadIdx.x % MLP_LANES;
    const int b = base + blk.y * MLP_BLOCK + lb;
    if (b >= base + T.tsize[t]) return;   // all four lanes of a bead
    double key[MLP_NN];
#pragma unroll
    for (int k = 0; k < MLP_NN; k++) key[k] = __hiloint2double(0x7ff00000, 0);
    const float box = T.tbox[t], ibox = inv_side(box);
    const float3 ri = f3(S.xyz[b]);
    float A[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    int cnt = 0;
    if (!T.extra[b]) {
        const int4 me = C.cell[b];
        const CellGeom geo = cell_geom(box, MLP_CELL, 0);
        const int dims = geo.dims;
        const uint32_t mask = (uint32_t)(C.tsize[t] - 1);
        const int toff = C.toff[t];
        const float ia = 1.f / P.tea_a;
        // the cell on the nearer side: the bead's place from its cell's lower
        // face, in cells (taken modulo the box, so it does not matter where
        // the table kernel's rounding put a bead on a face)
        const float ics = 1.f / geo.cs, fdims = (float)dims, idims = dims > 0 ? 1.f / fdims : 0.f;
        auto nearer = [&](float x, int cell) {
            float u = x * ics - (float)cell;
            u -= fdims * rintf((u - 0.5f) * idims);
            const int n = u < 0.5f ? cell - 1 : cell + 1;
            return dims > 0 ? wrap_cell(n, dims) : n;
        };
        const int nx = nearer(ri.x, me.x), ny = nearer(ri.y, me.y), nz = nearer(ri.z, me.z);
        // this lane's two cells: x and y by its part, own and nearer z; cells
        // are numbered part and part + 4
        const int cx = part & 1 ? nx : me.x, cy = part & 2 ? ny : me.y;
        const int b0 = toff + (int)(cell_hash(cx, cy, me.z) & mask), b1 = toff + (int)(cell_hash(cx, cy, nz) & mask);
        const int2 r0 = C.range[b0], r1 = C.range[b1];
        // a bucket that two cells hash to is visited for the first of them
        bool dup0 = false, dup1 = false;
        auto against = [&](int q, int o0, int o1) {   // the buckets of part q's two cells
            dup0 |= q < part && o0 == b0;
            dup1 |= o0 == b1 || (q < part && o1 == b1);
        };
        against(0, quad_lane<0>(b0), quad_lane<0>(b1));
        against(1, quad_lane<1>(b0), quad_lane<1>(b1));
        against(2, quad_lane<2>(b0), quad_lane<2>(b1));
        against(3, quad_lane<3>(b0), quad_lane<3>(b1));
        const int n0 = dup0 ? 0 : r0.y, n1 = dup1 ? 0 : r1.y;
        // a candidate; SMALL: the lane has at most 8, so its first 8 slots do
        auto visit = [&](auto small, const float4 pj) {
            const int jw = __float_as_int(pj.w);
            const int j = jw & 0x7fffffff;
            const float3 d = min_image_pre(make_float3(pj.x - ri.x, pj.y - ri.y, pj.z - ri.z), box, ibox);
            const float r2 = d.x * d.x + d.y * d.y + d.z * d.z;
            // extra beads, this bead and beads beyond the radius drop out
            if (jw < 0 || j == b || r2 >= MLP_RC * MLP_RC) return;
            if (LABELS) {
                // exact label: phi(r) D_hat(d)
                const float r = sqrtf(r2), rinv = 1.f / r;
                const float ra = r * ia;
                float cii, crr;
                if (ra > 2.f) {
                    const float u = 1.f / ra, u2 = u * u;
                    cii = 0.75f * u * (1.f + (2.f / 3.f) * u2);
                    crr = 0.75f * u * (1.f - 2.f * u2);
                } else {
                    cii = 1.f - 9.f * ra / 32.f;
                    crr = 3.f * ra / 32.f;
                }
                const float w = taper(r);
                const float e[3] = {d.x * rinv, d.y * rinv, d.z * rinv};
#pragma unroll
                for (int x = 0; x < 3; x++)
#pragma unroll
                    for (int y = 0; y < 3; y++) A[3 * x + y] += w * (crr * e[x] * e[y] + (x == y ? cii : 0.f));
            }
            // 32 nearest, ordered by (r2, j)
            const double kn = __hiloint2double(__float_as_int(r2), j - base);
            if (decltype(small)::value) {
                insert_key<0, 8>(key, kn);
                cnt++;
            } else if (kn < key[MLP_NN - 1]) {
                // slots in chunks of 8, a chunk only where some lane of the
                // wave holds a key in it (the rest are empty and stay so)
                const bool u1 = __any(cnt >= 8), u2 = __any(cnt >= 16), u3 = __any(cnt >= 24);
                if (u3) insert_key<24, 32>(key, kn);
                if (u2) insert_key<16, 24>(key, kn);
                if (u1) insert_key<8, 16>(key, kn);
                insert_key<0, 8>(key, kn);
                cnt = min(cnt + 1, MLP_NN);
            }
        };
        constexpr int PF = 4;
        if (!__any(n0 + n1 > 8)) {
            // a dilute wave: each lane visits its own two ranges, the first
            // four candidates requested together (a lane past its last one
            // requests the bead itself)
            const int own = n0 + n1, o1 = r1.x - n0;
            float4 pf[PF];
#pragma unroll
            for (int k0 = 0; k0 < 8; k0 += PF) {
                if (!__any(own > k0)) break;
#pragma unroll
                for (int u = 0; u < PF; u++) {
                    const int k = k0 + u;
                    pf[u] = C.spos[k < n0 ? r0.x + k : k < own ? o1 + k : b];
                }
#pragma unroll
                for (int u = 0; u < PF; u++)
                    if (k0 + u < own) visit(std::true_type{}, pf[u]);
            }
        } else {
            srg[lb][part] = dup0 ? Range::none() : Range::pack(r0, base);
            srg[lb][part + 4] = dup1 ? Range::none() : Range::pack(r1, base);
            wave_order();   // the four lanes are of one wave
            int total = n0 + n1;
            total += quad_swap<1>(total);
            total += quad_swap<2>(total);
            // One flat walk over every fourth of the bead's candidates (buckets
            // in order, each bucket's in slot order), the loads PF candidates
            // ahead of the visits (pf[k % PF] holds candidate k; the cursor q, in
            // range r, is the next one to request).  A lane past its last
            // candidate requests that one again: with no branch around the
            // loads, the wait before a visit leaves the later ones in flight.
            int r = 0, q = Range::lo(srg[lb][0], base), qend = Range::hi(srg[lb][0], base);
            int last = q;
            auto step = [&](int by) {
                q += by;
                while (q >= qend && r < 7) {
                    const int over = q - qend;
                    r++;
                    q = Range::lo(srg[lb][r], base) + over;
                    qend = Range::hi(srg[lb][r], base);
                }
                last = q < qend ? q : last;
            };
            step(part);
            const int mine = (total - part + MLP_LANES - 1) / MLP_LANES;   // candidates of this lane
            if (mine <= 0) last = b;   // none: any slot of the trajectory
            float4 pf[PF];
#pragma unroll
            for (int u = 0; u < PF; u++) {
                pf[u] = C.spos[last];
                step(MLP_LANES);
            }
            for (int k = 0; k < mine; k += PF) {
#pragma unroll
                for (int u = 0; u < PF; u++) {
                    const float4 pj = pf[u];
                    pf[u] = C.spos[last];
                    step(MLP_LANES);
                    if (k + u < mine) visit(std::false_type{}, pj);
                }
            }
        }
        // the four lists into one, which all four lanes hold; the keys of a
        // wave whose beads have at most 8 or 16 neighbours fill that many slots
        const int c1 = cnt + quad_swap<1>(cnt), all = c1 + quad_swap<2>(c1);
        if (!__any(all > 8)) {
            merge_keys<1, 8>(key);
            merge_keys<2, 8>(key);
        } else if (!__any(all > 16)) {
            merge_keys<1, 16>(key);
            merge_keys<2, 16>(key);
        } else {
            merge_keys<1, MLP_NN>(key);
            merge_keys<2, MLP_NN>(key);
        }
        cnt = min(all, MLP_NN);
        if (LABELS)
#pragma unroll
            for (int c = 0; c < 9; c++) {
                A[c] += quad_swap<1>(A[c]);
                A[c] += quad_swap<2>(A[c]);
            }
    }
    if (feat) {
        // each lane a block of eight neighbours (24 floats), their positions
        // requested together
        const int nblk = (cnt + FEAT_BLK_NN - 1) / FEAT_BLK_NN;
        if (fblk && part == 0) fblk[b] = (uint8_t)nblk;
        if (fblk && !__any(nblk > 1)) {
            // a dilute wave's one block, two neighbours per lane
            if (nblk > 0)
                write_features<FEAT_BLK_NN / MLP_LANES>(S.xyz + base, key, part, cnt, ri, box, ibox,
                                                        feat + (size_t)b * MLP_IN);
        } else if (!fblk || part < nblk) {
            write_features<FEAT_BLK_NN>(S.xyz + base, key, part, cnt, ri, box, ibox, feat + (size_t)b * MLP_IN);
        }
    }
    if (LABELS && part == 0) {
#pragma unroll
        for (int q = 0; q < 9; q++) targ[(size_t)b * MLP_OUT + q] = A[q];
    }
}

// ------------------------------------------------------------------ network
// Cholesky factor of the symmetric 3x3 S (row-major); false when a pivot
// falls below 1e-3 (not positive definite enough to use).
__device__ __forceinline__ bool chol3(const float S[9], float Lc[6]) {
    const float l00s = S[0];
    if (!(l00s > 1e-3f)) return false;
    const float l00 = sqrtf(l00s);
    const float l10 = S[3] / l00, l20 = S[6] / l00;
    const float l11s = S[4] - l10 * l10;
    if (!(l11s > 1e-3f)) return false;
    const float l11 = sqrtf(l11s);
    const float l21 = (S[7] - l20 * l10) / l11;
    const float l22s = S[8] - l20 * l20 - l21 * l21;
    if (!(l22s > 1e-3f)) return false;
    Lc[0] = l00; Lc[1] = l10; Lc[2] = l11; Lc[3] = l20; Lc[4] = l21; Lc[5] = sqrtf(l22s);
    return true;
}

// ------------------------------------------------------ inference on MFMA
// Each layer is computed transposed, D^T = W^T X^T, with
// v_mfma_f32_16x16x32_bf16: output neurons are the 16 rows (M), 16 beads the
// columns (N), inputs the reduction (K = 32 per instruction).  Lane l supplies
// A[l%16][8(l/16)+q] and B[8(l/16)+q][l%16] (q = 0..7) and receives
// D[4(l/16)+r][l%16] (r = 0..3).  The outputs of two adjacent 16-neuron
// tiles therefore already sit in B-operand position for the next layer if
// that layer's K index 8g+q is read as neuron 4g+q (q < 4) or 16+4g+(q-4)
// (q >= 4) of the 32-neuron block: the weight image is packed in that order
// and activations never leave registers.  Activations enter as bf16 hi + lo
// pairs (|x - hi - lo| <= 2^-18 |x|), so with bf16 weights the products are
// those of the FP32 network with bf16-rounded weights, accumulated in FP32.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int NET_WAVES = 12;                 // waves per workgroup (3 per SIMD)
constexpr int NET_THREADS = 64 * NET_WAVES;
constexpr int NET_GROUPS = 2;                 // 16-bead column groups per wave iteration
constexpr int NET_TILE = 16 * NET_GROUPS;     // beads per wave iteration
constexpr int MT_H = MLP_H / 16;              // output tiles of a hidden layer
constexpr int KS_IN = MLP_IN / 32, KS_H = MLP_H / 32;
// weight image in 16-byte fragments, [layer][m tile][k step][lane]
constexpr int FR1 = 0, FR2 = FR1 + MT_H * KS_IN * 64, FR3 = FR2 + MT_H * KS_H * 64, FR4 = FR3 + MT_H * KS_H * 64,
              FR_END = FR4 + KS_H * 64;
// FP32 biases after the fragments: b1, b2, b3, then b4 padded to 16
constexpr int BI2 = MLP_H, BI3 = 2 * MLP_H, BI4 = 3 * MLP_H, BI_END = 3 * MLP_H + 16;
constexpr size_t NET_IMG_BYTES = (size_t)FR_END * 16 + (size_t)BI_END * 4;
static_assert(MLP_IN % 32 == 0 && MLP_H % 32 == 0 && MLP_OUT <= 16, "network shape vs MFMA tiles");
static_assert(NET_IMG_BYTES % 16 == 0, "image size");

// Weight image from the bf16-rounded weights (exact bf16 values).
__global__ void __launch_bounds__(256) k_mlp_pack(const float *__restrict__ wi, u32x4 *img) {
    const int id = blockIdx.x * 256 + threadIdx.x;
    if (id < FR_END) {
        const float *W;
        int M, ks, mt, local;
        bool chained = true;
        if (id < FR2) {
            local = id - FR1; W = wi + OW1; M = MLP_H; chained = false;
            mt = (local / 64) / KS_IN; ks = (local / 64) % KS_IN;
        } else if (id < FR3) {
            local = id - FR2; W = wi + OW2; M = MLP_H;
            mt = (local / 64) / KS_H; ks = (local / 64) % KS_H;
        } else if (id < FR4) {
            local = id - FR3; W = wi + OW3; M = MLP_H;
            mt = (local / 64) / KS_H; ks = (local / 64) % KS_H;
        } else {
            local = id - FR4; W = wi + OW4; M = MLP_OUT;
            mt = 0; ks = local / 64;
        }
        const int lane = local % 64, g = lane / 16, m = 16 * mt + lane % 16;
        unsigned int word[4] = {0u, 0u, 0u, 0u};
        for (int q = 0; q < 8; q++) {
            const int k = 32 * ks + (chained ? (q < 4 ? 4 * g + q : 16 + 4 * g + (q - 4)) : 8 * g + q);
            const float v = m < M ? W[k * M + m] : 0.f;
            word[q / 2] |= (__float_as_uint(v) >> 16) << (16 * (q % 2));
        }
        img[id] = u32x4{word[0], word[1], word[2], word[3]};
    } else if (id < FR_END + BI_END) {
        const int j = id - FR_END;
        float v;
        if (j < BI2) v = wi[OB1 + j];
        else if (j < BI3) v = wi[OB2 + j - BI2];
        else if (j < BI4) v = wi[OB3 + j - BI3];
        else v = j - BI4 < MLP_OUT ? wi[OB4 + j - BI4] : 0.f;
        reinterpret_cast<float *>(img + FR_END)[j] = v;
    }
}

__device__ __forceinline__ float tanh_fast(float x) {
    // tanh x = 1 - 2 / (exp(2x) + 1) for either sign: absolute error a few
    // 1e-7; exp(2x) overflows to inf for large x (1) and underflows to 0
    // for large -x (-1)
    const float e = __expf(2.f * x);
    return fmaf(-2.f, rcp_fast(e + 1.f), 1.f);
}

__device__ __forceinline__ void split8(const float v[8], bf16x8 &hi, bf16x8 &lo) {
#pragma unroll
    for (int q = 0; q < 8; q++) {
        const __bf16 h = (__bf16)v[q];
        hi[q] = h;
        lo[q] = (__bf16)(v[q] - (float)h);
    }
}

// One layer over the bead groups: acc[mt][grp] = bias + W^T (hi + lo).
template <int KS, int MT>
__device__ __forceinline__ void net_layer(const u32x4 *frag, const float *bias, const bf16x8 (&hi)[KS][NET_GROUPS],
                                          const bf16x8 (&lo)[KS][NET_GROUPS], f32x4 (&acc)[MT][NET_GROUPS], int lane) {
    const int g = lane >> 4;
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(bias + 16 * mt + 4 * g);
#pragma unroll
        for (int grp = 0; grp < NET_GROUPS; grp++) acc[mt][grp] = b;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const bf16x8 a = __builtin_bit_cast(bf16x8, frag[(mt * KS + ks) * 64 + lane]);
#pragma unroll
            for (int grp = 0; grp < NET_GROUPS; grp++) {
                acc[mt][grp] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, hi[ks][grp], acc[mt][grp], 0, 0, 0);
                acc[mt][grp] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, lo[ks][grp], acc[mt][grp], 0, 0, 0);
            }
        }
    }
}

// The input layer over the k-slices in kuse (bit ks: features 32 ks ..
// 32 ks + 31); a slice outside kuse is zero for every bead of the tile and
// adds nothing.
__device__ __forceinline__ void net_layer_in(const u32x4 *frag, const float *bias,
                                             const bf16x8 (&hi)[KS_IN][NET_GROUPS],
                                             const bf16x8 (&lo)[KS_IN][NET_GROUPS], f32x4 (&acc)[MT_H][NET_GROUPS],
                                             int lane, uint32_t kuse) {
    const int g = lane >> 4;
#pragma unroll
    for (int mt = 0; mt < MT_H; mt++) {
        const f32x4 b = *reinterpret_cast<const f32x4 *>(bias + 16 * mt + 4 * g);
#pragma unroll
        for (int grp = 0; grp < NET_GROUPS; grp++) acc[mt][grp] = b;
    }
#pragma unroll
    for (int ks = 0; ks < KS_IN; ks++) {
        if (!((kuse >> ks) & 1u)) continue;
#pragma unroll
        for (int mt = 0; mt < MT_H; mt++) {
            const bf16x8 a = __builtin_bit_cast(bf16x8, frag[(mt * KS_IN + ks) * 64 + lane]);
#pragma unroll
            for (int grp = 0; grp < NET_GROUPS; grp++) {
                acc[mt][grp] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, hi[ks][grp], acc[mt][grp], 0, 0, 0);
                acc[mt][grp] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, lo[ks][grp], acc[mt][grp], 0, 0, 0);
            }
        }
    }
}

// tanh of a hidden layer, repacked as the next layer's B fragments.
template <int KS>
__device__ __forceinline__ void hidden_to_frags(f32x4 (&acc)[2 * KS][NET_GROUPS], bf16x8 (&hi)[KS][NET_GROUPS],
                                                bf16x8 (&lo)[KS][NET_GROUPS]) {
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
        for (int grp = 0; grp < NET_GROUPS; grp++) {
            float v[8];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                v[r] = tanh_fast(acc[2 * ks][grp][r]);
                v[4 + r] = tanh_fast(acc[2 * ks + 1][grp][r]);
            }
            split8(v, hi[ks][grp], lo[ks][grp]);
        }
}

// The network on beads b0 .. b0+NET_TILE-1 (features of beads >= n read as
// zero); returns in lane t < NET_TILE the 9 outputs of bead b0 + t.
// lim, byte grp: the features of the lane's bead in column group grp past
// that count are zeros and are not read (feat_limits).
__device__ __forceinline__ void net_tile(const u32x4 *frag, const float *bias, const float *__restrict__ feat,
                                         uint32_t lim, int b0, int lane, float y[MLP_OUT]) {
    const int g = lane >> 4, col = lane & 15;
    // The fragments are the same for every tile: keep the compiler from
    // hoisting all of them (368 registers) out of the caller's tile loop.
    __asm__ volatile("" ::: "memory");
    // k-slices of the input with a feature present for some bead of the tile
    int most = 0;
#pragma unroll
    for (int grp = 0; grp < NET_GROUPS; grp++) most = max(most, (int)((lim >> (8 * grp)) & 0xffu));
    uint32_t kuse = 0;
#pragma unroll
    for (int ks = 0; ks < KS_IN; ks++) kuse |= __any(most > 32 * ks) ? 1u << ks : 0u;
    bf16x8 hi1[KS_IN][NET_GROUPS], lo1[KS_IN][NET_GROUPS];
#pragma unroll
    for (int grp = 0; grp < NET_GROUPS; grp++) {
        const int bead = b0 + 16 * grp + col;
#pragma unroll
        for (int ks = 0; ks < KS_IN; ks++) {
            if (!((kuse >> ks) & 1u)) continue;
            float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (32 * ks + 8 * g < (int)((lim >> (8 * grp)) & 0xffu)) {
                const float4 *src = reinterpret_cast<const float4 *>(feat + (size_t)bead * MLP_IN + 32 * ks + 8 * g);
                const float4 u = src[0], w = src[1];
                v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
                v[4] = w.x; v[5] = w.y; v[6] = w.z; v[7] = w.w;
            }
            split8(v, hi1[ks][grp], lo1[ks][grp]);
        }
    }
    f32x4 acc[MT_H][NET_GROUPS];
    net_layer_in(frag + FR1, bias, hi1, lo1, acc, lane, kuse);
    bf16x8 hi[KS_H][NET_GROUPS], lo[KS_H][NET_GROUPS];
    hidden_to_frags<KS_H>(acc, hi, lo);
    net_layer<KS_H, MT_H>(frag + FR2, bias + BI2, hi, lo, acc, lane);
    hidden_to_frags<KS_H>(acc, hi, lo);
    net_layer<KS_H, MT_H>(frag + FR3, bias + BI3, hi, lo, acc, lane);
    hidden_to_frags<KS_H>(acc, hi, lo);
    f32x4 out[1][NET_GROUPS];
    net_layer<KS_H, 1>(frag + FR4, bias + BI4, hi, lo, out, lane);
    // output q of bead 16 grp + c sits in lane 16 (q / 4) + c, element q % 4
    const int grp = (lane >> 4) % NET_GROUPS;
#pragma unroll
    for (int q = 0; q < MLP_OUT; q++) {
        const int src = 16 * (q >> 2) + col;
        float v = 0.f;
#pragma unroll
        for (int gg = 0; gg < NET_GROUPS; gg++) {
            const float vg = __shfl(out[0][gg][q & 3], src);
            v = gg == grp ? vg : v;
        }
        y[q] = v;
    }
}

// Features present for the lane's beads of the tile at b0, one byte per
// column group (net_tile's lim): all 96 without fblk, else fblk's blocks of
// 24; none past the last bead.
__device__ __forceinline__ uint32_t feat_limits(const uint8_t *__restrict__ fblk, int n, int b0, int lane) {
    uint32_t lim = 0;
#pragma unroll
    for (int grp = 0; grp < NET_GROUPS; grp++) {
        const int bead = b0 + 16 * grp + (lane & 15);
        const int l = bead >= n ? 0 : fblk ? 3 * FEAT_BLK_NN * (int)fblk[bead] : MLP_IN;
        lim |= (uint32_t)l << (8 * grp);
    }
    return lim;
}
static_assert(MLP_IN < 256 && NET_GROUPS <= 4, "feature limits packed in bytes");

// Weight image into LDS (dynamic, NET_IMG_BYTES).
__device__ __forceinline__ void load_image(const u32x4 *__restrict__ img, u32x4 *lds) {
    for (int i = threadIdx.x; i < (int)(NET_IMG_BYTES / 16); i += NET_THREADS) lds[i] = img[i];
    __syncthreads();
}

__global__ void __launch_bounds__(NET_THREADS)
    k_mlp_forward(const u32x4 *__restrict__ img, const float *__restrict__ feat, int n, float *out) {
    extern __shared__ u32x4 net_lds[];
    load_image(img, net_lds);
    const float *bias = reinterpret_cast<const float *>(net_lds + FR_END);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int ntiles = (n + NET_TILE - 1) / NET_TILE;
    for (int tile = blockIdx.x * NET_WAVES + wave; tile < ntiles; tile += gridDim.x * NET_WAVES) {
        float y[MLP_OUT];
        net_tile(net_lds, bias, feat, feat_limits(nullptr, n, tile * NET_TILE, lane), tile * NET_TILE, lane, y);
        const int s = tile * NET_TILE + lane;
        if (lane < NET_TILE && s < n)
            for (int q = 0; q < MLP_OUT; q++) out[(size_t)s * MLP_OUT + q] = y[q];
    }
}

struct MlpStepArgs {
    ForceK K;
    DevTopo T;
    DevState Sin, Sout;
    const float4 *fxyz, *fang, *ci;
    const float *beta;
    uint4 *seeds;
    const float *noise;
    float *yout;
    int *nbad;
    LatOffsets L;
};

// MLP-HI integration of bead b from the network outputs y.  With G the
// predicted local HI tensor (symmetrised), TEA's per-trajectory beta and
// per-bead row normalisation C_i (refreshed by the epsilon pass as in TEA):
//   drift  (dt/gammaR) (I + G) F_i               local form of F_i + sum_j D_hat_ij F_j
//   noise  varR L xi,  L L^T = C (I + 2 beta G) C  row sum of TEA's noise covariance
//                                                  (src/bdhitea_kernel.cu:104-213) to first order in beta
// so cluster centre-of-mass diffusion follows TEA's.  A prediction whose
// covariance is not positive definite falls back to C^2 for the bead (counted).
// Noise draws as the plain integrator (mobile beads only).
// What the integrator reads of bead b, requested together after the network
// (before it, 256 registers and 8 waves per CU, or 162 and 12 as here: the
// step of 1,384,000 beads 387 against 354 us).
struct MlpIn {
    float4 x, an, n4, p1, p2, F, fa, cc;
    uint4 s0, s1;
    float bt;
    bool mobile;
};
__device__ __forceinline__ MlpIn mlp_load(const MlpStepArgs &A, int b) {
    MlpIn v;
    const DevTopo &T = A.T;
    v.x = A.Sin.xyz[b];
    v.an = A.Sin.ang[b];
    v.n4 = A.Sin.fn[b];
    v.p1 = A.Sin.fp1[b];
    v.p2 = A.Sin.fp2[b];
    v.F = A.fxyz[b];
    v.fa = A.fang[b];
    v.cc = A.ci[b];
    v.bt = A.beta[T.tid[b]];
    v.mobile = is_mobile(T.flags[b]);
    if (!A.noise) {
        v.s0 = A.seeds[b];
        v.s1 = A.seeds[b + T.nb];
    }
    return v;
}

__device__ __forceinline__ void mlp_integrate(const MlpStepArgs &A, int b, const float y[MLP_OUT], const MlpIn &in) {
    const ForceK &K = A.K;
    const DevTopo &T = A.T;
    float4 x = in.x, an = in.an;
    float4 n4 = in.n4, p1 = in.p1, p2 = in.p2;
    const bool mobile = in.mobile;
    if (mobile) {
        if (A.yout)
            for (int q = 0; q < MLP_OUT; q++) A.yout[(size_t)b * MLP_OUT + q] = y[q];
        float G[9];
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) G[3 * r + c] = 0.5f * (y[3 * r + c] + y[3 * c + r]);
        const float bt = in.bt;
        const float4 cc = in.cc;
        const float Cd[3] = {rsq_fast(1.f + bt * bt * cc.x), rsq_fast(1.f + bt * bt * cc.y),
                             rsq_fast(1.f + bt * bt * cc.z)};
        float Sg[9], Lc[6];
#pragma unroll
        for (int r = 0; r < 3; r++)
#pragma unroll
            for (int c = 0; c < 3; c++) Sg[3 * r + c] = Cd[r] * Cd[c] * ((r == c ? 1.f : 0.f) + 2.f * bt * G[3 * r + c]);
        if (!chol3(Sg, Lc)) {
            atomicAdd(A.nbad, 1);
            Lc[0] = Cd[0]; Lc[1] = 0.f; Lc[2] = Cd[1]; Lc[3] = 0.f; Lc[4] = 0.f; Lc[5] = Cd[2];
        }
        float4 rx, ra;
        if (A.noise) {
            const float *nz = A.noise + 6 * (size_t)b;
            rx = make_float4(nz[0], nz[1], nz[2], 0.f);
            ra = make_float4(nz[3], nz[4], nz[5], 0.f);
        } else {
            uint4 s = in.s0;
            rx = normals4(s);
            A.seeds[b] = s;
            s = in.s1;
            ra = normals4(s);
            A.seeds[b + T.nb] = s;
        }
        const float4 F = in.F;
        const float d0 = F.x + G[0] * F.x + G[1] * F.y + G[2] * F.z;
        const float d1 = F.y + G[3] * F.x + G[4] * F.y + G[5] * F.z;
        const float d2 = F.z + G[6] * F.x + G[7] * F.y + G[8] * F.z;
        const float n0 = Lc[0] * rx.x, n1 = Lc[1] * rx.x + Lc[2] * rx.y, n2 = Lc[3] * rx.x + Lc[4] * rx.y + Lc[5] * rx.z;
        x.x += fmaf(K.dtg, d0, K.vR * n0);
        x.y += fmaf(K.dtg, d1, K.vR * n1);
        x.z += fmaf(K.dtg, d2, K.vR * n2);
        em_angles(K, in.fa.x, in.fa.y, in.fa.z, ra, an);
        frame_vectors(an.x, an.y, an.z, A.L, n4, p1, p2);
    } else if (A.yout) {
        for (int q = 0; q < MLP_OUT; q++) A.yout[(size_t)b * MLP_OUT + q] = 0.f;
    }
    A.Sout.xyz[b] = x;
    A.Sout.ang[b] = an;
    A.Sout.fn[b] = n4;
    A.Sout.fp1[b] = p1;
    A.Sout.fp2[b] = p2;
}

// MLP-HI step: network on the matrix cores, then lanes 0..NET_TILE-1
// integrate the tile's beads.
__global__ void __launch_bounds__(NET_THREADS)
    k_mlp_step(const u32x4 *__restrict__ img, const float *__restrict__ feat, const uint8_t *__restrict__ fblk,
               MlpStepArgs A) {
    extern __shared__ u32x4 net_lds[];
    load_image(img, net_lds);
    const float *bias = reinterpret_cast<const float *>(net_lds + FR_END);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = A.T.nb;
    const int ntiles = (n + NET_TILE - 1) / NET_TILE;
    for (int tile = blockIdx.x * NET_WAVES + wave; tile < ntiles; tile += gridDim.x * NET_WAVES) {
        const uint32_t lim = feat_limits(fblk, n, tile * NET_TILE, lane);
        const int b = tile * NET_TILE + lane;
        const bool integ = lane < NET_TILE && b < n;
        float y[MLP_OUT];
        net_tile(net_lds, bias, feat, lim, tile * NET_TILE, lane, y);
        if (integ) mlp_integrate(A, b, y, mlp_load(A, b));
    }
}

// Per-trajectory squared error and squared label norm of predictions y
// against labels t over mobile beads (sampled-error judge), FP64 sums: each
// of MLP_ERR_PARTS workgroups per trajectory sums every MLP_ERR_PARTS-th
// 256-bead slice into its partial, and k_mlp_error_sum adds the partials in
// order.
__global__ void __launch_bounds__(256)
    k_mlp_error(DevTopo T, const float *y, const float *t, double *part) {
    __shared__ double se[256], sn[256];
    const int tr = blockIdx.x, p = blockIdx.y;
    const int base = T.tbase[tr], n = T.tsize[tr];
    double e = 0, m = 0;
    for (int i = p * 256 + threadIdx.x; i < n; i += 256 * MLP_ERR_PARTS) {
        const int b = base + i;
        if (T.fixed[b] || T.extra[b]) continue;
        for (int q = 0; q < MLP_OUT; q++) {
            const double d = (double)y[(size_t)b * MLP_OUT + q] - (double)t[(size_t)b * MLP_OUT + q];
            e += d * d;
            m += (double)t[(size_t)b * MLP_OUT + q] * (double)t[(size_t)b * MLP_OUT + q];
        }
    }
    se[threadIdx.x] = e;
    sn[threadIdx.x] = m;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (threadIdx.x < k) {
            se[threadIdx.x] += se[threadIdx.x + k];
            sn[threadIdx.x] += sn[threadIdx.x + k];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * ((size_t)tr * MLP_ERR_PARTS + p)] = se[0];
        part[2 * ((size_t)tr * MLP_ERR_PARTS + p) + 1] = sn[0];
    }
}

__global__ void __launch_bounds__(64) k_mlp_error_sum(int ntraj, const double *part, double *out) {
    const int tr = blockIdx.x * 64 + threadIdx.x;
    if (tr >= ntraj) return;
    double e = 0, m = 0;
    for (int p = 0; p < MLP_ERR_PARTS; p++) {
        e += part[2 * ((size_t)tr * MLP_ERR_PARTS + p)];
        m += part[2 * ((size_t)tr * MLP_ERR_PARTS + p) + 1];
    }
    out[2 * tr] = e;
    out[2 * tr + 1] = m;
}

// ----------------------------------------------------------------- training
// Forward, backward and every weight gradient of a sample tile in one kernel,
// in FP32 on the matrix cores (v_mfma_f32_16x16x4_f32: FP32 operands and
// accumulation).  A workgroup of 8 waves takes tiles of 32 samples (one per
// CU and pass at the usual 8192-sample batch) and keeps their activations in
// LDS; wave w owns neurons 16 w .. 16 w + 15 of each hidden layer.
//   forward   D^T = W^T X^T: neurons are the 16 rows, samples the columns.
//             K step r of block q reads inputs 16 q + 4 g + r (g = lane / 16),
//             so four steps take one float4 of a sample's row, and the rows a
//             lane receives (4 g + r of its wave's neurons) are the operand
//             the output layer needs: its K is split over the waves without
//             an exchange, the partial outputs added in wave order.
//   backward  the same with W's rows; dL/d(pre-activation) overwrites the
//             layer's activations (each wave only its own columns, which no
//             other wave reads once that layer's weight gradient is taken).
//   dW        in^T g over the tile's samples; K step st of a 16-sample block
//             takes samples 4 g + st, which with row pitches of 4 mod 64
//             words reads LDS without bank conflicts.  The sums stay in
//             registers over a workgroup's tiles (23 16x16 tiles per wave).
// Each workgroup writes one partial gradient; k_mlp_reduce adds the partials
// in a fixed order (no atomics: training repeats bit for bit) and takes the
// Adam step.
// Bound at 8192 samples by waits: of the 40 us the matrix cores are busy for
// 13 (504 instructions of 32 cycles per wave, two waves per SIMD: 2.27 GFLOP
// at the FP32 matrix rate).  A wave spends 44% of its time on outstanding
// loads (weights from L2 at each layer, LDS operands) and barriers and 42%
// ready to issue, behind matrix instructions; two waves per SIMD, each with
// 104 registers of sums (28 more spill, 15 MB of the 62 written), cover neither.
// Bank conflicts are 3% of the cycles.
// Measured per iteration of 8192 samples: 40 us here and 12 us in the
// reduction; with one thread per sample, per weight and per activation, nine
// launches, atomics and a read-back of the loss, 1290 us.  777 samples (25
// workgroups): 34 + 4 us, before 480 us.
constexpr int TR_TILE = 32, TR_WAVES = MLP_H / 16, TR_THREADS = 64 * TR_WAVES;
constexpr int TR_PX = MLP_IN + 4, TR_PH = MLP_H + 4, TR_PY = 20;   // LDS row pitches
constexpr int TR_OX = 0, TR_OH1 = TR_OX + TR_TILE * TR_PX, TR_OH2 = TR_OH1 + TR_TILE * TR_PH,
              TR_OH3 = TR_OH2 + TR_TILE * TR_PH, TR_OG = TR_OH3 + TR_TILE * TR_PH, TR_OY = TR_OG + TR_TILE * TR_PY,
              TR_END = TR_OY + TR_WAVES * TR_TILE * TR_PY;   // floats
constexpr size_t TR_LDS = sizeof(float) * TR_END;
static_assert(TR_PX % 64 == 36 && TR_PH % 64 == 4 && TR_TILE == 32 && TR_THREADS == 16 * TR_TILE, "training tile");

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 ld4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }
__device__ __forceinline__ void st4(float *p, f32x4 v) { *reinterpret_cast<f32x4 *>(p) = v; }

// Keeps the compiler from requesting the operands of all following steps at
// once (the 104 registers of sums leave no room for them).
__device__ __forceinline__ void tr_fence() { __asm__ volatile("" ::: "memory"); }

// This lane's share of a layer's weights for its wave's 16 rows: column
// 16 w + i of W (forward) or row 16 w + i (backward), K of the reduction.
// `of`: the lane's offset, made opaque once per tile so that the loads take
// a scalar base and it instead of addresses kept in registers over the loop.
template <int K>
__device__ __forceinline__ void tr_wfwd(const float *__restrict__ W, uint32_t of, float (&a)[K / 4]) {
#pragma unroll
    for (int q = 0; q < K / 16; q++)
#pragma unroll
        for (int r = 0; r < 4; r++) a[4 * q + r] = (W + (16 * q + r) * MLP_H)[of];
}
__device__ __forceinline__ void tr_wbwd(const float *__restrict__ W, uint32_t of, float (&a)[MLP_H / 4]) {
#pragma unroll
    for (int q = 0; q < MLP_H / 16; q++) {
        const f32x4 v = ld4(W + 16 * q + of);
#pragma unroll
        for (int r = 0; r < 4; r++) a[4 * q + r] = v[r];
    }
}

// acc[sc] += the wave's 16 rows over K inputs held in LDS rows of `pitch`.
template <int K>
__device__ __forceinline__ void tr_rows(const float (&a)[K / 4], const float *in, int pitch, int g, int i,
                                        f32x4 (&acc)[2]) {
#pragma unroll
    for (int q = 0; q < K / 16; q++) {
        const f32x4 b0 = ld4(in + i * pitch + 16 * q + 4 * g), b1 = ld4(in + (16 + i) * pitch + 16 * q + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            acc[0] = mfma_f32(a[4 * q + r], b0[r], acc[0]);
            acc[1] = mfma_f32(a[4 * q + r], b1[r], acc[1]);
        }
    }
}

// Hidden layer: h = tanh(bias + W^T in), kept in registers and written to out.
template <int K>
__device__ __forceinline__ void tr_hidden(const float (&a)[K / 4], const float *__restrict__ bias, const float *in,
                                          int pitch, float *out, int w, int g, int i, f32x4 (&h)[2]) {
    f32x4 acc[2];
#pragma unroll
    for (int r = 0; r < 4; r++) acc[0][r] = acc[1][r] = bias[16 * w + 4 * g + r];
    tr_rows<K>(a, in, pitch, g, i, acc);
#pragma unroll
    for (int sc = 0; sc < 2; sc++) {
#pragma unroll
        for (int r = 0; r < 4; r++) h[sc][r] = tanhf(acc[sc][r]);
        st4(out + (16 * sc + i) * TR_PH + 16 * w + 4 * g, h[sc]);
    }
}

// One operand of a weight gradient: column 16 c + i of the tile's rows, the
// eight K steps of its 32 samples.
__device__ __forceinline__ void tr_column(const float *m, int pitch, int c, int g, int i, float (&v)[8]) {
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
        for (int st = 0; st < 4; st++) v[4 * b + st] = m[(16 * b + 4 * g + st) * pitch + 16 * c + i];
}
__device__ __forceinline__ f32x4 tr_outer(const float (&a)[8], const float (&b)[8], f32x4 c) {
#pragma unroll
    for (int k = 0; k < 8; k++) c = mfma_f32(a[k], b[k], c);
    return c;
}

// Layer W (its inputs' activations h in `in`, its output gradients in `gout`):
// dW of the wave's 16 input rows, then the gradient at the inputs over the
// wave's columns of `in`.
__device__ __forceinline__ void tr_back(const float (&a)[MLP_H / 4], const float *gout, float *in, int w, int g, int i,
                                        f32x4 (&dw)[MT_H], f32x4 &db) {
    float col[8];
    tr_column(in, TR_PH, w, g, i, col);
#pragma unroll
    for (int mt = 0; mt < MT_H; mt++) {
        float b[8];
        tr_column(gout, TR_PH, mt, g, i, b);
        dw[mt] = tr_outer(col, b, dw[mt]);
        tr_fence();
    }
    wave_order();   // other lanes' columns have been read: the gradients overwrite them
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    tr_rows<MLP_H>(a, gout, TR_PH, g, i, acc);
#pragma unroll
    for (int sc = 0; sc < 2; sc++) {
        float *own = in + (16 * sc + i) * TR_PH + 16 * w + 4 * g;
        const f32x4 h = ld4(own);
#pragma unroll
        for (int r = 0; r < 4; r++) acc[sc][r] *= 1.f - h[r] * h[r];
        st4(own, acc[sc]);
    }
    db += acc[0] + acc[1];
}

__global__ void __launch_bounds__(TR_THREADS)
    k_mlp_train(const float *__restrict__ w, const float *__restrict__ feat, const float *__restrict__ targ, int n,
                float *__restrict__ gpart, double *__restrict__ lpart) {
    extern __shared__ float tr_lds[];
    float *X = tr_lds + TR_OX, *H1 = tr_lds + TR_OH1, *H2 = tr_lds + TR_OH2, *H3 = tr_lds + TR_OH3,
          *G = tr_lds + TR_OG, *Y = tr_lds + TR_OY;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g = lane >> 4, i = lane & 15;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 dw1[MLP_IN / 16], dw2[MT_H], dw3[MT_H], dw4 = zero, db1 = zero, db2 = zero, db3 = zero;
#pragma unroll
    for (int k = 0; k < MLP_IN / 16; k++) dw1[k] = zero;
#pragma unroll
    for (int k = 0; k < MT_H; k++) dw2[k] = dw3[k] = zero;
    float db4 = 0.f;
    double loss = 0.0;
    const float scale = 2.f / ((float)n * (float)MLP_OUT);
    const int ntiles = (n + TR_TILE - 1) / TR_TILE;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int s0 = tile * TR_TILE;
        uint32_t of = 4 * g * MLP_H + 16 * wv + i, ob = (16 * wv + i) * MLP_H + 4 * g;
        __asm__ volatile("" : "+v"(of), "+v"(ob));
        float a1[MLP_IN / 4], a2[MLP_H / 4];
        tr_wfwd<MLP_IN>(w + OW1, of, a1);
        for (int k = tid; k < TR_TILE * MLP_IN / 4; k += TR_THREADS) {
            const int s = k / (MLP_IN / 4), c = k % (MLP_IN / 4);
            st4(X + s * TR_PX + 4 * c, s0 + s < n ? ld4(feat + (size_t)(s0 + s) * MLP_IN + 4 * c) : zero);
        }
        __syncthreads();
        f32x4 h[2], h3[2];
        tr_wfwd<MLP_H>(w + OW2, of, a2);
        tr_hidden<MLP_IN>(a1, w + OB1, X, TR_PX, H1, wv, g, i, h);
        __syncthreads();
        float a3[MLP_H / 4];
        tr_wfwd<MLP_H>(w + OW3, of, a3);
        tr_hidden<MLP_H>(a2, w + OB2, H1, TR_PH, H2, wv, g, i, h);
        __syncthreads();
        // output layer weights in both directions, and layer 3's rows for the way back
        float o4[4], b4[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
            o4[r] = i < MLP_OUT ? w[OW4 + (16 * wv + 4 * g + r) * MLP_OUT + i] : 0.f;
            b4[r] = 4 * g + r < MLP_OUT ? w[OW4 + (16 * wv + i) * MLP_OUT + 4 * g + r] : 0.f;
        }
        float r3[MLP_H / 4];
        tr_wbwd(w + OW3, ob, r3);
        tr_hidden<MLP_H>(a3, w + OB3, H2, TR_PH, H3, wv, g, i, h3);
        // output layer: this wave's 16 inputs, which its lanes hold
#pragma unroll
        for (int sc = 0; sc < 2; sc++) {
            f32x4 y = zero;
#pragma unroll
            for (int r = 0; r < 4; r++) y = mfma_f32(o4[r], h3[sc][r], y);
            st4(Y + (wv * TR_TILE + 16 * sc + i) * TR_PY + 4 * g, y);
        }
        __syncthreads();
        {   // one thread per (sample, output of 16): dL/dy and the squared error
            const int s = tid / 16, o = tid % 16;
            float gy = 0.f;
            if (o < MLP_OUT && s0 + s < n) {
                float y = w[OB4 + o];
#pragma unroll
                for (int v = 0; v < TR_WAVES; v++) y += Y[(v * TR_TILE + s) * TR_PY + o];
                const float d = y - targ[(size_t)(s0 + s) * MLP_OUT + o];
                gy = scale * d;
                loss += (double)d * d;
            }
            G[s * TR_PY + o] = gy;
            db4 += gy;
        }
        __syncthreads();
        float r2[MLP_H / 4];
        tr_wbwd(w + OW2, ob, r2);
        {
            float hc[8], gc[8];
            tr_column(H3, TR_PH, wv, g, i, hc);
            tr_column(G, TR_PY, 0, g, i, gc);
            dw4 = tr_outer(hc, gc, dw4);
            wave_order();   // other lanes' columns have been read: the gradients overwrite them
            f32x4 acc[2] = {zero, zero};
#pragma unroll
            for (int sc = 0; sc < 2; sc++) {
                const f32x4 gy = ld4(G + (16 * sc + i) * TR_PY + 4 * g);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[sc] = mfma_f32(b4[r], gy[r], acc[sc]);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[sc][r] *= 1.f - h3[sc][r] * h3[sc][r];
                st4(H3 + (16 * sc + i) * TR_PH + 16 * wv + 4 * g, acc[sc]);
            }
            db3 += acc[0] + acc[1];
        }
        __syncthreads();
        tr_back(r3, H3, H2, wv, g, i, dw3, db2);
        __syncthreads();
        tr_back(r2, H2, H1, wv, g, i, dw2, db1);
        wave_order();   // the wave's other lanes have written their gradients
        {   // layer 1: the wave's own gradient columns against every input
            float gc[8];
            tr_column(H1, TR_PH, wv, g, i, gc);
#pragma unroll
            for (int kt = 0; kt < MLP_IN / 16; kt++) {
                float xc[8];
                tr_column(X, TR_PX, kt, g, i, xc);
                dw1[kt] = tr_outer(xc, gc, dw1[kt]);
                tr_fence();
            }
        }
        __syncthreads();   // the tile's rows are free
    }
    float *gp = gpart + (size_t)blockIdx.x * MLP_NPARAM;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int k = 16 * wv + 4 * g + r;
#pragma unroll
        for (int kt = 0; kt < MLP_IN / 16; kt++) gp[OW1 + (16 * kt + 4 * g + r) * MLP_H + 16 * wv + i] = dw1[kt][r];
#pragma unroll
        for (int mt = 0; mt < MT_H; mt++) {
            gp[OW2 + k * MLP_H + 16 * mt + i] = dw2[mt][r];
            gp[OW3 + k * MLP_H + 16 * mt + i] = dw3[mt][r];
        }
        if (i < MLP_OUT) gp[OW4 + k * MLP_OUT + i] = dw4[r];
        // bias gradients: over the 16 sample columns of the wave
        float b1 = db1[r], b2 = db2[r], b3 = db3[r];
#pragma unroll
        for (int m = 1; m < 16; m <<= 1) {
            b1 += __shfl_xor(b1, m);
            b2 += __shfl_xor(b2, m);
            b3 += __shfl_xor(b3, m);
        }
        if (i == 0) {
            gp[OB1 + k] = b1;
            gp[OB2 + k] = b2;
            gp[OB3 + k] = b3;
        }
    }
    // output bias and loss: over the workgroup's threads, in a fixed order
    float *rb = tr_lds;
    double *rl = reinterpret_cast<double *>(tr_lds + TR_THREADS);
    rb[tid] = db4;
    rl[tid] = loss;
    __syncthreads();
    for (int k = TR_THREADS / 2; k >= 16; k >>= 1) {
        if (tid < k) {
            rb[tid] += rb[tid + k];
            rl[tid] += rl[tid + k];
        }
        __syncthreads();
    }
    if (tid < MLP_OUT) gp[OB4 + tid] = rb[tid];
    if (tid == 0) {
        double s = 0.0;
        for (int k = 0; k < 16; k++) s += rl[k];
        lpart[blockIdx.x] = s;
    }
}

__device__ __forceinline__ float round_bf16(float v) {
    uint32_t u = __float_as_uint(v);
    u = (u + 0x7FFFu + ((u >> 16) & 1u)) & 0xFFFF0000u;
    return __uint_as_float(u);
}

// Adam step (Kingma & Ba 2015) of the FP32 master weights: moment decay
// rates, step size and the two bias corrections of this step.
struct AdamStep {
    float *w, *m1, *m2, *wi;   // wi: the bf16-rounded copy used by inference
    float lr, b1, b2, eps, c1, c2;
};

// The gradient, the workgroups' partials added in a fixed order (four waves
// take a quarter of them each, sixteen loads in flight per lane), the Adam
// step where w is given, and the mean squared error.  Bound by reading the
// partials (48 MB from 256 workgroups).
constexpr int RED_PARAMS = 64, RED_WAVES = 4;
__global__ void __launch_bounds__(RED_PARAMS * RED_WAVES)
    k_mlp_reduce(const float *__restrict__ gpart, const double *__restrict__ lpart, int nwg, int n, float *grad,
                 double *loss, AdamStep A) {
    __shared__ float part[RED_WAVES][RED_PARAMS];
    const int lane = threadIdx.x % RED_PARAMS, wv = threadIdx.x / RED_PARAMS;
    const int p = blockIdx.x * RED_PARAMS + lane;
    const int per = (nwg + RED_WAVES - 1) / RED_WAVES, k0 = wv * per, k1 = min(nwg, k0 + per);
    float s = 0.f;
    if (p < MLP_NPARAM) {
        const float *q = gpart + (size_t)k0 * MLP_NPARAM + p;
        int k = k0;
        for (; k + 16 <= k1; k += 16, q += (size_t)16 * MLP_NPARAM) {
            float v[16];
#pragma unroll
            for (int u = 0; u < 16; u++) v[u] = q[(size_t)u * MLP_NPARAM];
#pragma unroll
            for (int u = 0; u < 16; u++) s += v[u];
        }
        for (; k < k1; k++, q += MLP_NPARAM) s += *q;
    }
    part[wv][lane] = s;
    __syncthreads();
    if (wv == 0 && p < MLP_NPARAM) {
        const float gi = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
        grad[p] = gi;
        if (A.w) {
            const float a = A.b1 * A.m1[p] + (1.f - A.b1) * gi;
            const float v = A.b2 * A.m2[p] + (1.f - A.b2) * gi * gi;
            A.m1[p] = a;
            A.m2[p] = v;
            const float nw = A.w[p] - A.lr * (a / A.c1) / (sqrtf(v / A.c2) + A.eps);
            A.w[p] = nw;
            A.wi[p] = round_bf16(nw);
        }
    }
    if (blockIdx.x == 0 && wv == 1) {
        double e = 0.0;
        for (int k = lane; k < nwg; k += RED_PARAMS) e += lpart[k];
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) e += __shfl_xor(e, m);
        if (lane == 0) *loss = e / ((double)n * MLP_OUT);
    }
}

__global__ void __launch_bounds__(256) k_mlp_round(const float *w, float *wi, int n) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) wi[i] = round_bf16(w[i]);
}

// ------------------------------------------------------------------ launchers
static inline int blocks(int n, int bs) { return (n + bs - 1) / bs; }

hipError_t launch_mlp_cells(mte_engine *e) { return build_cells(e, MLP_CELL, 0); }

hipError_t launch_mlp_local(mte_engine *e, float *feat, float *targ, bool build_tables, uint8_t *fblk) {
    if (build_tables) {
        const hipError_t s = launch_mlp_cells(e);
        if (s != hipSuccess) return s;
    }
    const dim3 grid(e->mlp.nblocks), block(MLP_BLOCK * MLP_LANES);
    const int2 *bl = e->mlp.blocks;
    const bool narrow = e->nmax < 65536;   // trajectory-local indices and bucket ends fit 16 bits
    if (targ && narrow)
        hipLaunchKernelGGL((k_mlp_local<true, uint16_t>), grid, block, 0, e->stream, e->P, e->T, e->S[e->cur],
                           e->cells, bl, feat, targ, fblk);
    else if (targ)
        hipLaunchKernelGGL((k_mlp_local<true, int>), grid, block, 0, e->stream, e->P, e->T, e->S[e->cur], e->cells,
                           bl, feat, targ, fblk);
    else if (narrow)
        hipLaunchKernelGGL((k_mlp_local<false, uint16_t>), grid, block, 0, e->stream, e->P, e->T, e->S[e->cur],
                           e->cells, bl, feat, targ, fblk);
    else
        hipLaunchKernelGGL((k_mlp_local<false, int>), grid, block, 0, e->stream, e->P, e->T, e->S[e->cur], e->cells,
                           bl, feat, targ, fblk);
    return hipGetLastError();
}

// Workgroups of the inference kernels: one per CU at most (the weight image
// takes most of a CU's LDS), each wave looping over bead tiles.
static int net_blocks(const mte_engine *e, int n) {
    const int need = blocks(blocks(n, NET_TILE), NET_WAVES);
    return std::max(1, std::min(need, e->num_cus));
}

static hipError_t net_lds_attr(const void *k) {
    return hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)NET_IMG_BYTES);
}

hipError_t launch_mlp_forward(mte_engine *e, const float *feat, int n, float *out) {
    hipError_t s = net_lds_attr((const void *)k_mlp_forward);
    if (s != hipSuccess) return s;
    hipLaunchKernelGGL(k_mlp_forward, dim3(net_blocks(e, n)), dim3(NET_THREADS), NET_IMG_BYTES, e->stream,
                       reinterpret_cast<const u32x4 *>(e->mlp.img), feat, n, out);
    return hipGetLastError();
}

hipError_t launch_mlp_step(mte_engine *e, const float *noise_step, float *yout) {
    hipError_t s = net_lds_attr((const void *)k_mlp_step);
    if (s != hipSuccess) return s;
    MlpStepArgs A{e->K, e->T, e->S[e->cur], e->S[1 - e->cur], e->fxyz, e->fang, e->tea.ci, e->tea.beta,
                  e->seeds, noise_step, yout, e->mlp.nbad, e->L};
    hipLaunchKernelGGL(k_mlp_step, dim3(net_blocks(e, e->nb)), dim3(NET_THREADS), NET_IMG_BYTES, e->stream,
                       reinterpret_cast<const u32x4 *>(e->mlp.img), e->mlp.feat, e->mlp.fblk, A);
    e->cur = 1 - e->cur;
    return hipGetLastError();
}

hipError_t launch_mlp_error(mte_engine *e, const float *y, const float *t) {
    hipLaunchKernelGGL(k_mlp_error, dim3(e->ntraj, MLP_ERR_PARTS), dim3(256), 0, e->stream, e->T, y, t,
                       e->mlp.err_part);
    hipLaunchKernelGGL(k_mlp_error_sum, dim3((e->ntraj + 63) / 64), dim3(64), 0, e->stream, e->ntraj,
                       (const double *)e->mlp.err_part, e->mlp.err);
    return hipGetLastError();
}

// Workgroups of k_mlp_train, and so partial gradients, at most.
int mlp_train_groups(const mte_engine *e, int n) {
    return (int)std::min<int64_t>(((int64_t)n + TR_TILE - 1) / TR_TILE, e->num_cus);
}

// Gradient of n samples already on the device into e->mlp.grad and their
// mean squared error into *loss (device); with t > 0 also Adam step t.
hipError_t launch_mlp_grad(mte_engine *e, const float *feat, const float *targ, int n, double *loss, float lr, int t) {
    MlpBuffers &M = e->mlp;
    const hipError_t s = hipFuncSetAttribute((const void *)k_mlp_train, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)TR_LDS);
    if (s != hipSuccess) return s;
    const int nwg = mlp_train_groups(e, n);
    hipLaunchKernelGGL(k_mlp_train, dim3(nwg), dim3(TR_THREADS), TR_LDS, e->stream, M.w, feat, targ, n, M.gpart,
                       M.lpart);
    AdamStep A{};
    if (t > 0) {
        const float b1 = 0.9f, b2 = 0.999f;
        A = AdamStep{M.w, M.m1, M.m2, M.wi, lr, b1, b2, 1e-8f, 1.f - powf(b1, (float)t), 1.f - powf(b2, (float)t)};
    }
    hipLaunchKernelGGL(k_mlp_reduce, dim3(blocks(MLP_NPARAM, RED_PARAMS)), dim3(RED_PARAMS * RED_WAVES), 0, e->stream,
                       (const float *)M.gpart, (const double *)M.lpart, nwg, n, M.grad, loss, A);
    return hipGetLastError();
}

hipError_t launch_mlp_round(mte_engine *e) {
    hipLaunchKernelGGL(k_mlp_round, dim3(blocks(MLP_NPARAM, 256)), dim3(256), 0, e->stream, e->mlp.w, e->mlp.wi,
                       MLP_NPARAM);
    return launch_mlp_pack(e);
}

hipError_t launch_mlp_pack(mte_engine *e) {
    hipLaunchKernelGGL(k_mlp_pack, dim3(blocks(FR_END + BI_END, 256)), dim3(256), 0, e->stream, e->mlp.wi,
                       reinterpret_cast<u32x4 *>(e->mlp.img));
    return hipGetLastError();
}

size_t mlp_image_bytes() { return NET_IMG_BYTES; }

// ------------------------------------------- inference without allocation
// Staging of mte_mlp_forward_noalloc: features (MLP_NOALLOC_ROWS x 96) then
// outputs (MLP_NOALLOC_ROWS x 9), in one fixed device array.  Each GPU the
// library runs on holds its own copy until the process ends.  Host code
// never uses the array's name as an address: the per-device address comes
// from hipGetSymbolAddress below.
static __device__ __align__(256) float scratch[(size_t)MLP_NOALLOC_ROWS * (MLP_IN + MLP_OUT)];

namespace {
std::mutex g_scratch_mu;
float *g_scratch_ptr[MLP_NOALLOC_MAX_DEVICES] = {};
}  // namespace

hipError_t noalloc_scratch_init(int device, float **ptr) {
    *ptr = nullptr;
    if (device < 0 || device >= MLP_NOALLOC_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[device]) {   // once per device, with that device current
        float *p = nullptr;
        const hipError_t s = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(scratch));
        if (s != hipSuccess) return s;
        g_scratch_ptr[device] = p;
    }
    *ptr = g_scratch_ptr[device];
    return hipSuccess;
}

}  // namespace mte
