// cells.hip -- cell-list neighbour search (sort and scan) for list rebuilds
// of large trajectories.
//
// The reference rebuilds its lists by scanning every bead of the trajectory
// for every bead (pairs_kernel, src/compute_cuda.cu:527-674; LJ_kernel,
// :913-940), O(N^2) per trajectory.  Here the rebuild is:
//   1. assign: cell coordinates floor(x / cs) per bead (wrapped in periodic
//      boxes), hashed into a per-trajectory table of 2^k buckets; count;
//   2. ranges: every bucket gets as many consecutive slots as it has beads;
//   3. scatter: beads into bucket order (counting sort), with their
//      positions copied into that order for the searches;
//   4. search: each bead visits the buckets of the 27 neighbouring cells,
//      keeps the beads within the candidate radius, sorts the candidates by
//      index and runs the reference's per-pair tests on them in that order,
//      so the lists come out identical to the all-pairs scan (same entries,
//      same order).
// A hash collision only adds beads that the distance rejects, or that have
// been met already.
#include "engine_internal.h"
#include "rebuild_common.h"

namespace mte {

constexpr int CELL_BLOCK = 64;
constexpr int CAND_CAP = 128;   // candidates per bead within the candidate radius
// A lane's buffer: one more, and lanes in banks of their own (an odd number of words).
template <class JT>
constexpr int CAND_STRIDE = CAND_CAP + (sizeof(JT) == 2 ? 2 : 1);

__device__ __forceinline__ int3 cell_of(float3 r, float box, const CellGeom &g) {
    const float x = cell_coord(r.x, box, g), y = cell_coord(r.y, box, g), z = cell_coord(r.z, box, g);
    if (g.dims > 0) return make_int3(min(g.dims - 1, (int)x), min(g.dims - 1, (int)y), min(g.dims - 1, (int)z));
    return make_int3((int)floorf(x), (int)floorf(y), (int)floorf(z));
}

// The bead's slot within its bucket comes from the atomic that counts it.
// Neighbouring beads of a microtubule share cells: while the first lane left
// has at least ASSIGN_GROUP lanes of its bucket, that group takes one atomic,
// its first lane adding the group's size and its lanes taking consecutive
// slots from the returned count.  Below that a round costs the wave more than
// the atomics it saves, but the two monomers of a free dimer, neighbouring
// lanes, are still joined.  The order of the beads within a bucket is not
// fixed; every user of the tables orders what it finds there by bead index or
// by distance.
constexpr int ASSIGN_GROUP = 8;
__global__ void __launch_bounds__(256)
    k_cell_assign(DevTopo T, DevState S, CellTables C, float side, int K) {
    const int b = xcd_bead(256);
    const bool valid = b < T.nb;
    int bucket = -1;
    if (valid) {
        const int t = T.tid[b];
        const float box = T.tbox[t];
        const CellGeom g = cell_geom(box, side, K);
        const int3 c = cell_of(f3(S.xyz[b]), box, g);
        bucket = C.toff[t] + (int)(cell_hash(c.x, c.y, c.z) & (uint32_t)(C.tsize[t] - 1));
        C.cell[b] = make_int4(c.x, c.y, c.z, bucket);
    }
    for (int t = blockIdx.x * 256 + threadIdx.x; t < T.ntraj; t += 256 * (int)gridDim.x) C.cursor[CELL_CURSOR_STRIDE * t] = T.tbase[t];   // for k_cell_ranges
    const int lane = threadIdx.x & 63;
    uint64_t todo = __ballot(valid), group = valid ? 1ull << lane : 0;
    int leader = lane;
    while (todo) {
        const int l0 = __ffsll((unsigned long long)todo) - 1;
        const int kb = __builtin_amdgcn_readlane(bucket, l0);
        const uint64_t m = __ballot(valid && bucket == kb);
        if (__popcll(m) < ASSIGN_GROUP) break;
        if (valid && bucket == kb) {
            leader = l0;
            group = m;
        }
        todo &= ~m;
    }
    if ((todo >> lane) & 1) {
        const int other = __builtin_amdgcn_update_dpp(0, bucket, 0xB1, 0xf, 0xf, true);   // lane ^ 1
        if (other == bucket && ((todo >> (lane ^ 1)) & 1)) {
            leader = lane & ~1;
            group = 3ull << leader;
        }
    }
    int first = 0;
    if (valid && lane == leader) first = atomicAdd(&C.count[bucket], __popcll(group));
    first = __shfl(first, leader);
    if (valid) C.rank[b] = first + __popcll(group & ((1ull << lane) - 1ull));
}

// Slots of the buckets: each workgroup sums and scans the counts of
// CELL_SCAN_SPAN buckets in LDS and takes that many slots from the cursor of
// their trajectory with one atomic (a span of small tables: one for each),
// so a trajectory's beads hold the slots [tbase, tbase + n).  Which of them a
// span gets depends on the order the workgroups arrive in; no user of the
// tables looks beyond a bucket's range.  (A scan over all buckets, in bucket
// order, took three launches and 17 us for 851968 buckets, this one 6.)  Bounded
// by the bytes, 16 per bucket, and by the cursors: atomics on one cache line
// from all XCDs take about 10 ns each, so a cursor has a line of its own and
// a span is 4096 buckets (1024: 13.5 us).
constexpr int SCAN_T = CELL_SCAN_SPAN / 4;   // four buckets to a thread: whole 16-byte loads and stores
static_assert(CELL_TABLE_MIN % 4 == 0, "the tables, and so the buckets, come in whole fours");
static_assert(CELL_SCAN_SPAN / CELL_TABLE_MIN + 1 <= SCAN_T, "a thread for each table in a span");
__global__ void __launch_bounds__(SCAN_T) k_cell_ranges(CellTables C) {
    __shared__ int wsum[SCAN_T / 64], shift[SCAN_T], first[SCAN_T];   // per table in the span: slot shift, first bucket
    __shared__ int4 before[SCAN_T + 1];                               // beads of the span before each bucket
    const int n = C.total, g0 = blockIdx.x * CELL_SCAN_SPAN, g = g0 + 4 * (int)threadIdx.x;
    const int t0 = C.span_traj[blockIdx.x], nt = C.span_traj[blockIdx.x + 1] - t0 + 1;   // tables that reach into the span
    int4 v = make_int4(0, 0, 0, 0);
    if (g < n) {
        v = *reinterpret_cast<const int4 *>(C.count + g);
        *reinterpret_cast<int4 *>(C.count + g) = make_int4(0, 0, 0, 0);   // ready for the next build's counting atomics
    }
    const int s = v.x + v.y + v.z + v.w;
    // exclusive prefix of the threads' sums: lanes by shuffles, then the waves
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int inc = s;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(inc, d, 64);
        if (lane >= d) inc += u;
    }
    if (lane == 63) wsum[wv] = inc;
    __syncthreads();
    int acc = inc - s;
#pragma unroll
    for (int w = 0; w < SCAN_T / 64; w++) acc += w < wv ? wsum[w] : 0;
    const int4 p = make_int4(acc, acc + v.x, acc + v.x + v.y, acc + v.x + v.y + v.z);
    before[threadIdx.x] = p;
    if (threadIdx.x == SCAN_T - 1) before[SCAN_T].x = acc + s;
    __syncthreads();
    if ((int)threadIdx.x < nt) {
        const int t = t0 + threadIdx.x;
        const int lo = max(0, C.toff[t] - g0), hi = min(CELL_SCAN_SPAN, C.toff[t] + C.tsize[t] - g0);
        const int *bf = reinterpret_cast<const int *>(before);
        if (lo < hi) shift[threadIdx.x] = atomicAdd(&C.cursor[CELL_CURSOR_STRIDE * t], bf[hi] - bf[lo]) - bf[lo];
        first[threadIdx.x] = lo;
    }
    __syncthreads();
    if (g >= n) return;
    int q = 0;   // the table of the thread's four buckets
    while (q + 1 < nt && first[q + 1] <= 4 * (int)threadIdx.x) q++;
    const int sh = shift[q];
    int4 *out = reinterpret_cast<int4 *>(C.range + g);
    out[0] = make_int4(sh + p.x, v.x, sh + p.y, v.y);
    out[1] = make_int4(sh + p.z, v.z, sh + p.w, v.w);
}

__global__ void __launch_bounds__(256) k_cell_scatter(DevTopo T, DevState S, CellTables C) {
    const int b = xcd_bead(256);
    if (b >= T.nb) return;
    const int slot = C.range[C.cell[b].w].x + C.rank[b];
    const float4 x = S.xyz[b];
    C.spos[slot] = make_float4(x.x, x.y, x.z, __int_as_float(b | (T.extra[b] ? (int)0x80000000 : 0)));
}
// Candidates of a bead: the beads of the (2K + 1)^3 cells about it that lie
// within the radius, in ascending index; -1 if there are more than CAND_CAP.
// Bounded by trips to memory: a tube's wave, one of few on its CU, visits 27
// cells of up to a dozen beads.  So the ranges of a plane's cells (K = 2: of a
// row's) are requested together, then four positions at a time, each with its
// bead's index.  A bucket that a hash collision shows twice, or one that holds
// other cells' beads too, needs no cell check: what lies within the radius is
// a candidate (met twice, it stands there twice, side by side once sorted, and
// the caller takes it once).  Up to 32 are sorted in registers.  4 periodic
// systems of 122646 beads: 188 us with three gathers per bead and an insertion
// sort in LDS, 108 with the requests together, 61 with the sort, 53 with each
// XCD on its own eighth of the beads, whose tables then stay in its L2.
template <int K, class JT>
__device__ __forceinline__ int gather_candidates(const DevTopo &T, const DevState &S, const CellTables &C, int b,
                                                 float radius, JT *cand) {
    const int t = T.tid[b], base = T.tbase[t];
    const float box = T.tbox[t], ibox = inv_side(box);
    const CellGeom g = cell_geom(box, radius / K, K);
    const int4 me = C.cell[b];
    const float3 ri = f3(S.xyz[b]);
    const float r2max = radius * radius;
    const uint32_t mask = (uint32_t)(C.tsize[t] - 1);
    const int toff = C.toff[t];
    constexpr int W = 2 * K + 1, ROWS = K == 1 ? W : 1, NC = ROWS * W;   // cells whose ranges are requested together
    int n = 0;
    bool over = false;
    // the n entries of the buffer in ascending order, each once; their number
    auto ordered = [](JT *cand, int n) {
        for (int i = 1; i < n; i++) {
            const JT v = cand[i];
            int k = i;
            for (; k > 0 && cand[k - 1] > v; k--) cand[k] = cand[k - 1];
            cand[k] = v;
        }
        int m = 0;
        for (int i = 0; i < n; i++)
            if (m == 0 || cand[i] != cand[m - 1]) cand[m++] = cand[i];
        return m;
    };
    auto test = [&](float4 pj) {
        const int j = __float_as_int(pj.w) & 0x7fffffff;
        const float3 d = min_image_pre(sub3(ri, f3(pj)), box, ibox);
        if (j == b || d.x * d.x + d.y * d.y + d.z * d.z >= r2max || over) return;
        cand[n++] = (JT)(j - base);
        if (n > CAND_CAP) {   // full: too many, unless some have been met twice
            n = ordered(cand, n);
            over = n > CAND_CAP;
        }
    };
    for (int r0 = 0; r0 < W * W; r0 += ROWS) {
        int2 rg[NC];
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int r = r0 + c / W;
            int cx = me.x + c % W - K, cy = me.y + r % W - K, cz = me.z + r / W - K;
            if (g.dims > 0) {
                cx = wrap_cell(cx, g.dims);
                cy = wrap_cell(cy, g.dims);
                cz = wrap_cell(cz, g.dims);
            }
            rg[c] = C.range[toff + (int)(cell_hash(cx, cy, cz) & mask)];
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
            for (int q = 0; q < rg[c].y; q += 4) {
                float4 p[4];
#pragma unroll
                for (int u = 0; u < 4; u++) p[u] = C.spos[rg[c].x + min(q + u, rg[c].y - 1)];
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (q + u < rg[c].y) test(p[u]);
            }
        }
    }
    if (over) return -1;
    if (n > SORT_W) return ordered(cand, n);
    sort_cands<SORT_W>(cand, 1, n);
    return n;
}

template <int K, class JT>
__global__ void __launch_bounds__(CELL_BLOCK)
    k_rebuild_cells(mte_params P, DevTopo T, DevState S, CellTables C, float radius, int do_lj, int do_bonded) {
    __shared__ JT cand_all[CELL_BLOCK * CAND_STRIDE<JT>];
    const int b = xcd_bead(CELL_BLOCK);
    if (b >= T.nb) return;
    const int t = T.tid[b], base = T.tbase[t];
    RebuildOwn o = rebuild_own(S.xyz[b], S.fn[b], S.fp1[b], S.fp2[b], T.mon_type[b], T.harm_raw[b], b - base, b,
                               base, T.tbox[t]);
    if (!T.extra[b]) {
        JT *cand = cand_all + threadIdx.x * CAND_STRIDE<JT>;
        const int n = gather_candidates<K>(T, S, C, b, radius, cand);
        if (n < 0) {
            o.ovf = 1;
        } else if (n > 0) {
            // the next candidate's data are requested before the current one's tests
            auto bead = [&](int k) { return base + (int)cand[min(k, n - 1)]; };
            int j = bead(0);
            float4 x = S.xyz[j], fn = S.fn[j], f1 = S.fp1[j], f2 = S.fp2[j];
            int mt = T.mon_type[j];
            for (int k = 0; k < n; k++) {
                const int jn = bead(k + 1);
                const float4 xn = S.xyz[jn], fnn = S.fn[jn], f1n = S.fp1[jn], f2n = S.fp2[jn];
                const int mtn = T.mon_type[jn];
                if (k + 1 < n && jn == j) continue;   // met twice: once more in the next turn
                rebuild_pair(T, o, j - base, x, fn, f1, f2, mt, P.ljpairscutoff, do_lj, do_bonded);
                j = jn, x = xn, fn = fnn, f1 = f1n, f2 = f2n, mt = mtn;
            }
        }
    }
    rebuild_finish(T, o, do_lj, do_bonded);
}

float candidate_radius(const mte_params &P) {
    return rebuild_radius(P.ljpairscutoff, P.lj_on != 0, P.is_assembly != 0);   // superset of every list test
}

hipError_t build_cells(mte_engine *e, float side, int K) {
    const CellTables &C = e->cells;
    const int gb = grid_xcd(e->nb, 256);
    // the bucket counts are zero here: set at creation, and cleared by
    // k_cell_ranges once it has read them
    hipLaunchKernelGGL(k_cell_assign, dim3(gb), dim3(256), 0, e->stream, e->T, e->S[e->cur], C, side, K);
    hipLaunchKernelGGL(k_cell_ranges, dim3((C.total + CELL_SCAN_SPAN - 1) / CELL_SCAN_SPAN), dim3(SCAN_T), 0, e->stream, C);
    hipLaunchKernelGGL(k_cell_scatter, dim3(gb), dim3(256), 0, e->stream, e->T, e->S[e->cur], C);
    return hipGetLastError();
}

hipError_t launch_rebuild_cells(mte_engine *e) {
    const int do_lj = e->P.lj_on ? 1 : 0;
    const int do_bonded = e->P.is_assembly ? 1 : 0;
    if (!do_lj && !do_bonded) return hipSuccess;
    const float radius = candidate_radius(e->P);
    const int K = e->tune.cell_stencil == 2 ? 2 : 1;
    hipError_t s = build_cells(e, radius / K, K);
    if (s != hipSuccess) return s;
    // 16-bit candidates where a trajectory's indices fit: half the LDS, twice the waves on a CU
    const bool small = e->nmax <= 65536;
    auto kern = K == 2 ? (small ? k_rebuild_cells<2, uint16_t> : k_rebuild_cells<2, int>)
                       : (small ? k_rebuild_cells<1, uint16_t> : k_rebuild_cells<1, int>);
    hipLaunchKernelGGL(kern, dim3(grid_xcd(e->nb, CELL_BLOCK)), dim3(CELL_BLOCK), 0, e->stream, e->P, e->T,
                       e->S[e->cur], e->cells, radius, do_lj, do_bonded);
    return hipGetLastError();
}

}  // namespace mte
