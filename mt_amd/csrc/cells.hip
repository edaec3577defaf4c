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
//   4. search: each bead visits the 27 neighbouring cells, keeps the beads of
//      exactly those cells within the candidate radius, sorts the candidates
//      by index and runs the reference's per-pair tests on them in that
//      order, so the lists come out identical to the all-pairs scan (same
//      entries, same order).
// A hash collision only adds beads that the exact cell check then rejects.
#include "engine_internal.h"
#include "rebuild_common.h"

namespace mte {

constexpr int CELL_BLOCK = 64;
constexpr int CAND_CAP = 128;   // candidates per bead within the candidate radius

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
    const int b = blockIdx.x * 256 + threadIdx.x;
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
    for (int t = b; t < T.ntraj; t += 256 * (int)gridDim.x) C.cursor[CELL_CURSOR_STRIDE * t] = T.tbase[t];   // for k_cell_ranges
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
// tables looks beyond a bucket's range.  (A scan over all buckets, in bucket order, took three
// launches: 17 us for 2^20 buckets, this one
// 6.)  Bounded by the bytes, 16 per bucket, and by the cursors: atomics on one
// cache line from all XCDs take about 10 ns each, so a cursor has a line of
// its own and a span is 4096 buckets (1024: 13.5 us).
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
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= T.nb) return;
    const int slot = C.range[C.cell[b].w].x + C.rank[b];
    C.sorted[slot] = b;
    const float4 x = S.xyz[b];
    C.spos[slot] = make_float4(x.x, x.y, x.z, __int_as_float(b | (T.extra[b] ? (int)0x80000000 : 0)));
}

// Candidates of bead b: beads of the (2K+1)^3 neighbouring cells (of side
// >= radius / K) within `radius` (minimum image), as local indices in
// ascending order.  Returns the count, or -1 when more than CAND_CAP were
// found.
__device__ int gather_candidates(const DevTopo &T, const DevState &S, const CellTables &C, int b, float radius,
                                 int K, int *cand) {
    const int t = T.tid[b], base = T.tbase[t];
    const float box = T.tbox[t], ibox = inv_side(box);
    const CellGeom g = cell_geom(box, radius / K, K);
    const int4 me = C.cell[b];
    const float3 ri = f3(S.xyz[b]);
    const float r2max = radius * radius;
    const uint32_t mask = (uint32_t)(C.tsize[t] - 1);
    int n = 0;
    for (int dz = -K; dz <= K; dz++)
        for (int dy = -K; dy <= K; dy++)
            for (int dx = -K; dx <= K; dx++) {
                int cx = me.x + dx, cy = me.y + dy, cz = me.z + dz;
                if (g.dims > 0) {
                    cx = wrap_cell(cx, g.dims);
                    cy = wrap_cell(cy, g.dims);
                    cz = wrap_cell(cz, g.dims);
                }
                const int bucket = C.toff[t] + (int)(cell_hash(cx, cy, cz) & mask);
                const int2 rg = C.range[bucket];
                const int s0 = rg.x, s1 = rg.x + rg.y;
                for (int q = s0; q < s1; q++) {
                    const int j = C.sorted[q];
                    if (j == b) continue;
                    const int4 cj = C.cell[j];
                    if (cj.x != cx || cj.y != cy || cj.z != cz) continue;
                    const float3 d = min_image_pre(sub3(ri, f3(S.xyz[j])), box, ibox);
                    if (d.x * d.x + d.y * d.y + d.z * d.z >= r2max) continue;
                    if (n >= CAND_CAP) return -1;
                    // insertion keeps the candidates sorted by index
                    int k = n++;
                    const int lj = j - base;
                    while (k > 0 && cand[k - 1] > lj) {
                        cand[k] = cand[k - 1];
                        k--;
                    }
                    cand[k] = lj;
                }
            }
    return n;
}

__global__ void __launch_bounds__(CELL_BLOCK)
    k_rebuild_cells(mte_params P, DevTopo T, DevState S, CellTables C, float radius, int K, int do_lj,
                    int do_bonded) {
    __shared__ int cand_all[CELL_BLOCK * CAND_CAP];
    const int b = blockIdx.x * CELL_BLOCK + threadIdx.x;
    if (b >= T.nb) return;
    const int t = T.tid[b], base = T.tbase[t];
    RebuildOwn o = rebuild_own(S.xyz[b], S.fn[b], S.fp1[b], S.fp2[b], T.mon_type[b], T.harm_raw[b], b - base, b,
                               base, T.tbox[t]);
    if (!T.extra[b]) {
        int *cand = cand_all + threadIdx.x * CAND_CAP;
        const int n = gather_candidates(T, S, C, b, radius, K, cand);
        if (n < 0) {
            o.ovf = 1;
        } else {
            for (int k = 0; k < n; k++) {
                const int j = base + cand[k];
                rebuild_pair(T, o, cand[k], S.xyz[j], S.fn[j], S.fp1[j], S.fp2[j], T.mon_type[j], P.ljpairscutoff,
                             do_lj, do_bonded);
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
    const int gb = (e->nb + 255) / 256;
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
    hipLaunchKernelGGL(k_rebuild_cells, dim3((e->nb + CELL_BLOCK - 1) / CELL_BLOCK), dim3(CELL_BLOCK), 0, e->stream,
                       e->P, e->T, e->S[e->cur], e->cells, radius, K, do_lj, do_bonded);
    return hipGetLastError();
}

}  // namespace mte
