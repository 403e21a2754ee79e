// gfx950 kernels of the point-vs-SDF contact path.
//
// Batched path:
//   cull_kernel    per group of 256 sorted points: can its box reach a cell where
//                  a point may be active? (the tiles' live-group masks); it also
//                  clears the evaluation's counters.
//   detect_kernel  tiles of Morton-sorted FP32 contact points, taken from one
//                  queue in instance order (or grid-grouped / per-XCD queues).
//                  Streams each tile's live groups (several points per lane, nontemporal
//                  loads), maps every point into the grid's padded cell space
//                  with an FP64 affine map and reads one byte of the grid's cell
//                  classification table (inactive / active / open). Open cells
//                  go through an LDS candidate ring and the exact test; the
//                  active points are appended to the tile's slice of the
//                  active list, with one 64-bit atomic per tile reserving
//                  record slots and work items of the bounded record pool.
//   slow_kernel    the FP64 FD-stencil samples of the few active points whose
//                  stencil leaves their cell.
//   contact_kernel work items of kChunk active points (ItemWalk): builds
//                  the records (sample of phi, grad phi, Hessian) and sums the
//                  wrench (optionally the p6 column) into the item's partial row.
//   jacobian_kernel the same with Km/Dm, one workgroup per item: sums the wrench,
//                  the p6 column and the 3x3 blocks that Km and Dm are made of.
//   vjp_kernel     the adjoint of the same records.
//   reduce_kernel  per-instance sums of the partial rows in a fixed order
//                  (reduce_jacobian_kernel: then Km and Dm from the block sums).
// Plain path (the one-launch-per-instance baseline): plain_kernel, one lane per
// point, inline contact math, FP64 atomics.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <type_traits>
#include "atac_kernels.h"
#include "contact_math.h"
#include "wave_ops.h"

namespace atac {

// Per-lane wrench accumulator: FP64 for both arithmetics (an FP32 term is
// converted exactly and added in FP64: two full-rate instructions, and the
// lane's sum carries no FP32 rounding).
template <typename R>
struct LaneAcc {
    double s;
    __device__ void zero() { s = 0.0; }
    __device__ void add(R v) { s += (double)v; }
    __device__ double value() const { return s; }
};

// ------------------------------------------------------------------ tile assignment
// Tiles are split into nq contiguous queues of balanced point counts (nq is 1,
// or 8 for per-XCD queues). Workgroup b belongs to queue b % nq (with nq = 8 the
// XCD it is dispatched to, with round-robin dispatch over the XCDs, so a queue's
// tiles share that XCD's L2) and takes the
// queue's tiles r, r + m, r + 2m, ... where r = b / nq is its rank among the m
// workgroups of the queue. The assignment is static: no shared counter, and
// every workgroup's tile sequence is known from the start.
struct TileWalk {
    int k, end, step;
    __device__ TileWalk(const QueueDev& Q) {
        const int nq = Q.nq, q = (int)blockIdx.x % nq, r = (int)blockIdx.x / nq;
        step = ((int)gridDim.x - q + nq - 1) / nq;
        k = as_const(Q.begin)[q] + r;
        end = as_const(Q.begin)[q + 1];
    }
};

// ------------------------------------------------------------------ records
template <typename R> struct RecOf;
template <> struct RecOf<float> { using type = Rec32; };
template <> struct RecOf<double> { using type = Rec64; };

__device__ __forceinline__ void store_rec(Rec32* p, const Rec32& r) {
    float4* q = reinterpret_cast<float4*>(p);
    q[0] = make_float4(r.a[0], r.a[1], r.a[2], r.a[3]);
    q[1] = make_float4(r.b[0], r.b[1], r.b[2], r.b[3]);
    q[2] = make_float4(r.c[0], r.c[1], r.c[2], r.c[3]);
}
__device__ __forceinline__ Rec32 load_rec(const Rec32* p) {
    const float4* q = reinterpret_cast<const float4*>(p);
    const float4 a = q[0], b = q[1], c = q[2];
    Rec32 r;
    r.a[0] = a.x; r.a[1] = a.y; r.a[2] = a.z; r.a[3] = a.w;
    r.b[0] = b.x; r.b[1] = b.y; r.b[2] = b.z; r.b[3] = b.w;
    r.c[0] = c.x; r.c[1] = c.y; r.c[2] = c.z; r.c[3] = c.w;
    return r;
}
__device__ __forceinline__ void store_rec(Rec64* p, const Rec64& r) { *p = r; }
__device__ __forceinline__ Rec64 load_rec(const Rec64* p) { return *p; }

// A slow-path FP32 record points at its diagonal Hessian entries in slow_diag.
__device__ __forceinline__ void mark_slow_index(Rec32& r, int slow) { r.c[3] = __int_as_float(slow); }
__device__ __forceinline__ void mark_slow_index(Rec64&, int) {}

// ------------------------------------------------------------------ batched detection
// Points o0 + 64 k + lane, k < PPL, of a step into (x, y, z)[k]: each load
// instruction reads 64 consecutive points (a contiguous 256-byte span), so the
// points a wavefront handles together are neighbours in the Morton order and
// their block-bound reads share cache lines. Points at or past `end` read point 0
// (in bounds; their results are masked by the caller).
template <int PPL, typename P>
__device__ __forceinline__ void load_points(P px, P py, P pz, int o0, int lane, int end, float (&x)[PPL],
                                            float (&y)[PPL], float (&z)[PPL]) {
#pragma unroll
    for (int k = 0; k < PPL; ++k) {
        const int o = o0 + 64 * k + lane;
        const uint32_t oo = (uint32_t)(o < end ? o : 0) * 4u;   // byte offset
        x[k] = nt_load_at<float>(px, oo);
        y[k] = nt_load_at<float>(py, oo);
        z[k] = nt_load_at<float>(pz, oo);
    }
}

// Points of one tile per work item. The tile's live groups are shared among its
// wavefronts by rank (contiguous ranges, so their outputs follow one another in
// point order), and each wavefront streams its groups: a step takes 64 * PPL
// consecutive points of a group, lane l the points 64 k + l (each load and
// table-read instruction covers 64 neighbouring points; the next step's points
// are loaded behind the table reads of the current ones, so a step waits once),
// and only the classification table is read (detect_candidates). The candidates a step finds (settled active or open; a
// few per cent, near the surface) are appended, with their coordinates, to the
// wavefront's LDS ring in ascending order (ballots per point slot k); whenever 64
// are waiting, the next step finishes them one per lane (candidate_locate and
// candidate_finish: cell read and interpolation of the open ones, FD-stencil
// test), overlapped with its own work, instead of every stream step branching
// into that work for a few lanes. The active offsets (bit 15: slow path; tiles
// hold at most 8192 points) go to a per-wave LDS segment, then to the tile's
// slots of the active list, and the tile pushes its work items for the record,
// contact and adjoint passes.
template <int BLOCK, int PPL>
__global__ __launch_bounds__(BLOCK) void detect_kernel(DetectArgs a) {
    constexpr int NW = BLOCK / 64;
    constexpr int CAP = detect_ring_cap(PPL);
    extern __shared__ __align__(16) unsigned char s_lds[];
    __shared__ int s_wcount[NW];
    __shared__ int s_base;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int span = a.wave_span;
    uint16_t* s_queue = reinterpret_cast<uint16_t*>(s_lds);   // [NW][span] active offsets, bit 15 = slow path
    float4* cand = reinterpret_cast<float4*>(s_lds + (size_t)NW * span * 2) + w * CAP;
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    const bool all_active = a.all_active != 0;
    const auto order = as_const(a.q.order);
    const TileWalk walk(a.q);
    for (int kk = walk.k; kk < walk.end; kk += walk.step) {
        const int tile = order[kk];
        const TileDev t = as_const(a.tiles)[tile];
        const InstDev in = as_const(a.inst)[t.inst];
        const GridDev G = as_const(a.grids)[t.grid];
        const auto px = as_global(in.px) + t.begin;
        const auto py = as_global(in.py) + t.begin;
        const auto pz = as_global(in.pz) + t.begin;
        uint16_t* q = s_queue + w * span;
        // the tile's groups that can hold a candidate (all without the mask); this
        // wave takes those of ranks [w m / NW, (w + 1) m / NW), in ascending order,
        // so the waves' output segments follow one another in point order
        const int ng = (t.count + kGroup - 1) / kGroup;
        const uint32_t all_groups = ng >= 32 ? 0xffffffffu : ((1u << ng) - 1u);
        uint32_t mine = a.tile_live ? (as_const(a.tile_live)[tile] & all_groups) : all_groups;
        {
            const int wu = __builtin_amdgcn_readfirstlane(w);
            const int m = __popc(mine), r0 = (wu * m) / NW, r1 = ((wu + 1) * m) / NW;
            for (int r = 0; r < r0; ++r) mine &= mine - 1u;
            uint32_t later = mine;
            for (int r = r0; r < r1; ++r) later &= later - 1u;
            mine &= ~later;
        }
        // candidates wait in a ring of CAP entries: [rd, rd + occ) (mod CAP)
        int wcount = 0, rd = 0, occ = 0, npend = 0;   // wave-uniform
        auto ring = [](int i) { return i >= CAP ? i - CAP : i; };   // i < 2 CAP
        const float cth = (float)in.col_th;
        const ClsConsts kc = cls_consts_vgpr(G, in);
        // A batch: the n <= 64 oldest candidates, one per lane. start() reads
        // them and issues their cell reads; complete() decides them into the
        // output segment. A step starts one at its top, before its own work, and
        // completes it once its own reads are out, so the cell reads' latency
        // overlaps the step. Every step starts one, empty or not, and every lane
        // issues the two reads (lanes without an open candidate read the first
        // cell), so the reads in flight are the same on every path.
        CandRead pend;
        uint32_t ptag = 0;
        const auto cells = ATAC_GLOBAL(G.cells);
        auto start = [&](int n) {
            uint32_t off = 0;
            if (lane < n) {
                const float4 e = cand[ring(rd + lane)];
                ptag = __float_as_uint(e.w);
                off = candidate_locate(G, in, e.x, e.y, e.z, (ptag >> 15) != 0u, pend);
            }
            pend.lo = load_f4_at(cells, off);
            pend.hi = load_f4_at(cells, off + 16u);
            rd = ring(rd + n);
            occ -= n;
            npend = n;
        };
        auto complete = [&]() {
            bool act = false, slow = false;
            if (lane < npend) act = candidate_finish(pend, cth, slow);
            const uint64_t bal = __ballot(act);
            if (act) q[wcount + __popcll(bal & lt_mask)] = (uint16_t)((ptag & 0x7fffu) | (slow ? 0x8000u : 0u));
            wcount += __popcll(bal);
            npend = 0;
        };
        // one step: points (cx, cy, cz) at o0 (valid below we) are tested while
        // the next step's points (at on, valid below wn) load into (nx, ny, nz);
        // the loop alternates the two buffers, so no register copy waits for the
        // loads in flight
        auto step = [&](int o0, int we, int on, int wn, const float (&cx)[PPL], const float (&cy)[PPL],
                        const float (&cz)[PPL], float (&nx)[PPL], float (&ny)[PPL], float (&nz)[PPL]) {
            start(occ >= 64 ? 64 : 0);
            unsigned valid = 0;
#pragma unroll
            for (int k = 0; k < PPL; ++k)
                if (o0 + 64 * k + lane < we) valid |= 1u << k;
            unsigned op;
            const unsigned m = detect_candidates<PPL>(G, in, kc, cx, cy, cz, valid, all_active, op, [] {}, [&]() {
                __builtin_amdgcn_sched_barrier(0);
                load_points<PPL>(px, py, pz, on, lane, wn, nx, ny, nz);
                __builtin_amdgcn_sched_barrier(0);
                complete();   // its cell reads went out before this step's reads
            });
            // appended in point order: point k of every lane (lane order) before point k + 1
            int pos = rd + occ;   // stays < 2 CAP: occ + (this step's candidates) <= CAP
#pragma unroll
            for (int k = 0; k < PPL; ++k) {
                const bool is_c = ((m >> k) & 1u) != 0u;
                const uint64_t bal = __ballot(is_c);
                if (is_c)
                    cand[ring(pos + __popcll(bal & lt_mask))] = make_float4(
                        cx[k], cy[k], cz[k], __uint_as_float((uint32_t)(o0 + 64 * k + lane) | (((op >> k) & 1u) << 15)));
                pos += __popcll(bal);
            }
            occ = pos - rd;
            // the next step takes at most 64 * PPL and starts by taking 64 if it
            // has them: room for it while occ <= 128 (always with one point per
            // lane); beyond (rare), batches finish here
            if constexpr (PPL > 1) {
                while (occ > 128) {
                    start(64);
                    complete();
                }
            }
        };
        // the wave's steps: kGroup / (64 PPL) per group of `mine`, lowest group
        // first; (g, s) is the current one, advance() moves to the next and says
        // whether there is one (a step without a next loads point 0, in bounds)
        if (mine) {
            constexpr int SP = 64 * PPL, NS = kGroup / SP;
            auto gend = [&](int gg) { return min(t.count, (gg + 1) * kGroup); };
            auto advance = [](uint32_t& lv, int& g, int& s) {
                if (++s < NS) return true;
                s = 0;
                lv &= lv - 1u;
                if (!lv) return false;
                g = __builtin_ctz(lv);
                return true;
            };
            uint32_t lv = mine;
            int g = __builtin_ctz(lv), s = 0;
            float x0[PPL], y0[PPL], z0[PPL], x1[PPL], y1[PPL], z1[PPL];
            load_points<PPL>(px, py, pz, g * kGroup, lane, gend(g), x0, y0, z0);
            for (;;) {
                uint32_t lv1 = lv;
                int g1 = g, s1 = s;
                const bool more = advance(lv1, g1, s1);
                step(g * kGroup + s * SP, gend(g), more ? g1 * kGroup + s1 * SP : 0, more ? gend(g1) : 0, x0, y0, z0,
                     x1, y1, z1);
                if (!more) break;
                lv = lv1; g = g1; s = s1;
                const bool more2 = advance(lv1, g1, s1);
                step(g * kGroup + s * SP, gend(g), more2 ? g1 * kGroup + s1 * SP : 0, more2 ? gend(g1) : 0, x1, y1,
                     z1, x0, y0, z0);
                if (!more2) break;
                lv = lv1; g = g1; s = s1;
            }
        }
        while (occ > 0) {
            start(occ < 64 ? occ : 64);
            complete();
        }
        if (lane == 0) s_wcount[w] = wcount;
        __syncthreads();
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < NW; ++k) cnt += s_wcount[k];
        // the tile's records: one range of the pool, reserved by one atomic; a
        // tile that does not fit marks the evaluation as overflowed and writes
        // nothing (its outputs then come out NaN)
        if (tid == 0) {
            int base = -1;
            if (cnt > 0) {
                const int nch = (cnt + kChunk - 1) / kChunk;
                const unsigned long long old = atomicAdd(reinterpret_cast<unsigned long long*>(a.counters + CNT_RECS),
                                                         ((unsigned long long)nch << 32) | (unsigned long long)cnt);
                const int r0 = (int)(uint32_t)old, c0 = (int)(uint32_t)(old >> 32);
                const bool ok = r0 <= a.rec_cap - cnt && c0 <= a.chunk_cap - nch;
                if (ok) {
                    base = r0;
                    a.tile_chunk0[tile] = c0;
                } else {
                    atomicOr(a.counters + CNT_OVERFLOW, 1);
                }
                // the items this tile took: its ranges, or (overflowed) empty ones
                for (int k = 0; k < nch && c0 + k < a.chunk_cap; ++k)
                    a.chunks[c0 + k] = ok ? ChunkDev{t.inst, min(kChunk, cnt - k * kChunk), (int64_t)base + (int64_t)k * kChunk}
                                          : ChunkDev{t.inst, 0, 0};
            }
            s_base = base;
            a.tile_active[tile] = base >= 0 ? cnt : 0;
        }
        __syncthreads();
        const int base = s_base;
        if (base >= 0) {
            // the tile's active offsets, in ascending point order, at its pool range;
            // the contact pass builds their records (the slow pass those of the
            // contacts whose FD stencil leaves the cell; one the slow list has no room for
            // is not marked, so that its record is formed all the same, as if inside its
            // cell: the outputs are NaN, and the passes read no record nobody wrote)
            uint32_t* act = a.act + base;
            const uint32_t tb = (uint32_t)t.begin;
            for (int qi = tid; qi < cnt; qi += BLOCK) {
                int rem = qi, ww = 0;
                while (rem >= s_wcount[ww]) { rem -= s_wcount[ww]; ++ww; }
                const uint32_t e = s_queue[ww * span + rem];
                bool slow = (e >> 15) != 0u;
                if (slow) {
                    const int si = atomicAdd(a.counters + CNT_SLOW, 1);
                    slow = si < a.slow_cap;
                    if (slow) a.slow[si] = SlowDev{(uint32_t)(base + qi), t.inst};
                    else atomicOr(a.counters + CNT_OVERFLOW, 1);
                }
                act[qi] = (tb + (e & 0x7fffu)) | (slow ? kActSlow : 0u);
            }
        }
        __syncthreads();
    }
}

// Wavefront-granular passes take work items in a fixed stride: wavefront g of
// the launch takes items g, g + G, g + 2G, ... (G = wavefronts in the launch),
// the items being near-equal (at most kChunk records). No shared counter is
// touched, and the item index is wave-uniform (readfirstlane), so every branch
// on it is uniform.
__device__ __forceinline__ int wave_id() {
    return (int)blockIdx.x * (int)(blockDim.x >> 6) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}
__device__ __forceinline__ int wave_count() { return (int)gridDim.x * (int)(blockDim.x >> 6); }

// Records of the slow-path contacts (a few per thousand): the 20 FD-stencil
// evaluations of a point run on 20 lanes at once (three points per wavefront),
// and one lane per point combines them and writes the record.
template <bool PREC>
__global__ __launch_bounds__(64) void slow_kernel(SlowArgs a) {
    using Rec = typename RecOf<typename std::conditional<PREC, double, float>::type>::type;
    constexpr int GROUPS = 64 / kStencil;
    __shared__ double s_v[GROUPS][kStencil];
    const int lane = threadIdx.x, grp = lane / kStencil, st = lane % kStencil;
    const int n = min(a.counters[CNT_SLOW], a.slow_cap);
    for (int base = (int)blockIdx.x * GROUPS; base < n; base += (int)gridDim.x * GROUPS) {
        const int i = base + grp;
        const bool mine = grp < GROUPS && i < n;
        SlowDev sd{0u, 0};
        Rec r;
        if (mine) {
            sd = a.slow[i];
            const InstDev& in = a.inst[sd.inst];
            const uint32_t off = a.act[sd.slot] & ~kActSlow;
            r.a[0] = in.px[off]; r.a[1] = in.py[off]; r.a[2] = in.pz[off]; r.a[3] = __uint_as_float(off);
            double x[3], q[3];
            bool accurate;
            body2_point(in, (double)r.a[0], (double)r.a[1], (double)r.a[2], x);
            stencil_point(x, st, q, accurate);
            s_v[grp][st] = query_sdf64(a.grids[in.grid], q[0], q[1], q[2], accurate);
        }
        __syncthreads();
        if (mine && st == 0) {
            double v[kStencil], val, g[3], H[6];
#pragma unroll
            for (int k = 0; k < kStencil; ++k) v[k] = s_v[grp][k];
            stencil_combine(v, val, g, H);
            float* diag = a.slow_diag ? a.slow_diag + 4 * (int64_t)i : nullptr;
            record_slow_fill(a.inst[sd.inst], val, g, H, r, diag);
            mark_slow_index(r, i);
            store_rec(static_cast<Rec*>(a.rec) + sd.slot, r);
        }
        __syncthreads();
    }
}

// Column sums of a wavefront's 64 x N lane values through LDS (s: this wave's
// 64 * N doubles), in a fixed order: lane k < N adds column k as four interleaved
// sums of rows r = 4i + q, combined as (q0 + q1) + (q2 + q3). Returns lane k's
// column sum (0 on lanes >= N). One pass for all N values: no per-value wave
// reduction and no wave-uniform results to hold.
template <int N>
__device__ __forceinline__ double lds_column_sums(double* s, const double (&v)[N]) {
    static_assert(N <= 64, "one column per lane");
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < N; ++k) s[lane * N + k] = v[k];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    double r = 0.0;
    if (lane < N) {
        double q[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
        for (int i = 0; i < 64; i += 4)
#pragma unroll
            for (int j = 0; j < 4; ++j) q[j] += s[(i + j) * N + lane];
        r = (q[0] + q[1]) + (q[2] + q[3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();   // the buffer is free for the wave's next use
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return r;
}

// ------------------------------------------------------------------ batched contact pass
// A lane's active contact `j` of a work item: its record, built from the packed
// cell and stored for the adjoint on the fast path, read back on the slow one.
template <typename Rec>
__device__ __forceinline__ Rec item_record(const GridDev& G, const InstDev& in, uint32_t e, float qx, float qy, float qz,
                                           Rec* rec) {
    if (e & kActSlow) return load_rec(rec);   // written by the slow pass
    Rec r;
    double cc[3], fd[3];
    int idx[3];
    grid_coords(in, qx, qy, qz, cc);
    cell_of_c(G, cc, idx, fd);
    const Corners cr = G.fast ? load_cell(G, idx[0], idx[1], idx[2]) : load_corners(G, idx[0], idx[1], idx[2]);
    r.a[0] = qx; r.a[1] = qy; r.a[2] = qz; r.a[3] = __uint_as_float(e);
    record_fast(G, in, cr, fd, r);
    store_rec(rec, r);
    return r;
}

// Work items of kChunk records: how the contact and adjoint kernels deal them out.
// SPLIT: a workgroup per item, a wavefront per 64 records, whose sums are added in LDS;
// otherwise a wavefront per item, its lanes taking the records 64 apart in turn. With
// few items (about one per tile) the second leaves the SIMDs with one or two wavefronts
// and four dependent steps each; with many, the first only adds sums. 96 FP64 instances
// (244 tiles), an evaluation and its adjoint: 57 us by wavefront, 46 by workgroup; the
// fused pass over 300 instances (1,500 tiles) 76.8 and 75.5.
template <bool SPLIT>
struct ItemWalk {
    static constexpr int U = SPLIT ? 1 : kChunk / 64;   // records per lane
    static __device__ __forceinline__ int begin() { return SPLIT ? (int)blockIdx.x : wave_id(); }
    static __device__ __forceinline__ int step() { return SPLIT ? (int)gridDim.x : wave_count(); }
    static __device__ __forceinline__ int first() { return SPLIT ? (int)(threadIdx.x & ~63u) : 0; }   // of the wavefront's records
    // the item's row from its wavefronts' column sums (lane k: component k)
    template <int NF>
    static __device__ __forceinline__ void store(double (*s_row)[NF], double col, double* dst) {
        const int lane = threadIdx.x & 63;
        if constexpr (SPLIT) {
            if (lane < NF) s_row[threadIdx.x >> 6][lane] = col;
            __syncthreads();
            if (threadIdx.x < NF) {
                const int k = threadIdx.x;
                dst[k] = s_row[0][k] + s_row[1][k] + s_row[2][k] + s_row[3][k];
            }
            __syncthreads();
        } else if (lane < NF) {
            dst[lane] = col;
        }
    }
};

// The wrench (and p6 column) of every record, summed per lane, then over the wave in a
// fixed order into the item's partial row.
template <bool P6, typename R, bool SPLIT>
__global__ __launch_bounds__(256) void contact_kernel(ContactArgs a) {
    using Rec = typename RecOf<R>::type;
    constexpr int NF = P6 ? 24 : 12;
    using Walk = ItemWalk<SPLIT>;
    constexpr int U = Walk::U;
    __shared__ double s_red[4][64 * NF], s_row[4][NF];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int total = min(a.counters[CNT_CHUNKS], a.chunk_cap);
    for (int c = Walk::begin(); c < total; c += Walk::step()) {
        const ChunkDev ch = as_const(a.chunks)[c];
        const InstDev in = as_const(a.inst)[ch.inst];
        const GridDev G = as_const(a.grids)[in.grid];
        const int64_t rec0 = ch.rec0 + Walk::first();
        const int n = ch.n - Walk::first();
        Rec* rec = static_cast<Rec*>(a.rec) + rec0;
        const auto act = as_global(a.act) + rec0;
        const InstR<R> I = make_inst<R>(in);
        LaneAcc<R> acc[NF];
#pragma unroll
        for (int k = 0; k < NF; ++k) acc[k].zero();
        // this lane's active-list entries and points, all loaded first
        uint32_t e[U];
        float qx[U], qy[U], qz[U];
#pragma unroll
        for (int u = 0; u < U; ++u) e[u] = (u * 64 + lane < n) ? act[u * 64 + lane] : kActSlow;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t off = e[u] & ~kActSlow;
            qx[u] = as_global(in.px)[off];
            qy[u] = as_global(in.py)[off];
            qz[u] = as_global(in.pz)[off];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = u * 64 + lane;
            if (j < n) {
                const Rec r = item_record(G, in, e[u], qx[u], qy[u], qz[u], rec + j);
                ContactFwd<R> s;
                record_decode(r, a.slow_diag, in, s);
                R p6[12];
                contact_forward<R>(I, s, P6 ? p6 : nullptr);
#pragma unroll
                for (int k = 0; k < 12; ++k) acc[k].add(s.f[k]);
                if (P6) {
#pragma unroll
                    for (int k = 0; k < 12; ++k) acc[P6 ? 12 + k : 0].add(p6[k]);
                }
            }
        }
        double* dst = a.partial + (int64_t)c * NF;
        double lv[NF];
#pragma unroll
        for (int k = 0; k < NF; ++k) lv[k] = acc[k].value();
        Walk::template store<NF>(s_row, n > 0 ? lds_column_sums<NF>(&s_red[w][0], lv) : 0.0, dst);
    }
}

// ------------------------------------------------------------------ wrench and Jacobian sums
// Work items of kChunk records, one workgroup each, wavefront w taking records
// [64 w, 64 w + 64), one per lane: the wrench, the p6 column and the blocks Km and
// Dm are made of (contact_jac), summed over the item into its partial row
// (kJacRow of its kJvpRow values; poses that are not rotations fill it). Bound by
// instruction issue: about 1,700 instructions per 64 contacts, where 24 tangents per
// contact and their 288 wave sums took about 13,000 (an evaluation of 256 poses x 5,000
// points with Km/Dm: 149 us with these, 57 with the blocks, 47 with what the other
// kernels gained since; this one 31). 64 contacts per wavefront rather than 256: small
// batches have few items and need the waves. RIGID: every instance's poses are
// rotations. Otherwise each item takes the form of its instance (InstDev::rigid), which
// costs the blocks 4 % (FP32) and 25 % (FP64, spilled registers) of an evaluation.
template <typename R, bool RIGID>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void jacobian_kernel(ContactArgs a) {
    using Rec = typename RecOf<R>::type;
    __shared__ double s_col[4][JacColumns::SIZE];
    __shared__ double s_part[4][RIGID ? kJacRowPad : kJvpRowPad];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int total = min(a.counters[CNT_CHUNKS], a.chunk_cap);
    for (int c = (int)blockIdx.x; c < total; c += (int)gridDim.x) {
        const ChunkDev ch = as_const(a.chunks)[c];
        const int n = ch.n - 64 * w;   // this wavefront's records
        const bool rigid = RIGID || as_const(a.inst)[ch.inst].rigid != 0;
        // lanes past the end repeat the last record; their rows are not summed
        const int64_t j = ch.rec0 + 64 * w + min(lane, n - 1);
        const auto forward = [&](const InstDev& in, ContactFwd<R>& s, R p6[12]) {
            const GridDev G = as_const(a.grids)[in.grid];
            const uint32_t e = as_global(a.act)[j], off = e & ~kActSlow;
            const Rec r = item_record(G, in, e, as_global(in.px)[off], as_global(in.py)[off], as_global(in.pz)[off],
                                      static_cast<Rec*>(a.rec) + j);
            record_decode(r, a.slow_diag, in, s);
            contact_forward<R>(make_inst<R>(in), s, p6);
        };
        ContactFwd<R> s;
        R p6[12];
        if (n > 0 && rigid) {
            const InstDev in = as_const(a.inst)[ch.inst];
            forward(in, s, p6);
            put_jac_row<R>(JacColumns{&s_col[w][0], &s_part[w][0], lane, n}, jac_inst(in), s, p6);
        } else if (!RIGID && n > 0) {
            // the record again, behind an opaque pointer: nothing of this rare branch is formed
            // (and kept in registers) ahead of the other
            const InstDev* again = a.inst;
            asm volatile("" : "+s"(again));
            const InstDev in = as_const(again)[ch.inst];
            forward(in, s, p6);
            put_jvp_row<R>(JvpColumns{&s_col[w][0], &s_part[w][0], lane, n}, make_inst<R>(in), s, p6);
        }
        __syncthreads();
        for (int k = (int)threadIdx.x; k < (rigid ? kJacRow : kJvpRow) && ch.n > 0; k += 256) {
            double v = s_part[0][k];
            for (int i = 1; i < 4; ++i)
                if (ch.n > 64 * i) v += s_part[i][k];
            a.partial[(int64_t)c * kJvpRow + k] = v;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ fused wrench and adjoint
// Work items of kChunk records, one wavefront each, for a cotangent known when
// the contacts are evaluated (re-evaluation in a backward pass): each record's
// sample is formed as in contact_kernel (the slow pass's records read), its
// wrench summed as contact_kernel's mode 0 sums it and its adjoint as
// vjp_kernel does, per lane over the records 64 apart in turn, then over the
// lanes: the partial row is fm 12 | kVjpOut. No record is written.
template <typename R, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 3 : 1))) void fused_kernel(ContactArgs a) {
    using Rec = typename RecOf<R>::type;
    using Walk = ItemWalk<SPLIT>;
    __shared__ double s_red[4][64 * kVjpOut], s_row[4][kFmOut], s_vrow[4][kVjpOut];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int total = min(a.counters[CNT_CHUNKS], a.chunk_cap);
    for (int c = Walk::begin(); c < total; c += Walk::step()) {
        const ChunkDev ch = as_const(a.chunks)[c];
        const InstDev in = as_const(a.inst)[ch.inst];
        const GridDev G = as_const(a.grids)[in.grid];
        const int64_t rec0 = ch.rec0 + Walk::first();
        const int n = min(64 * Walk::U, ch.n - Walk::first());
        const Rec* rec = static_cast<const Rec*>(a.rec) + rec0;
        const auto act = as_global(a.act) + rec0;
        const InstR<R> I = make_inst<R>(in);
        R gb[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) gb[k] = (R)a.g_fm[(int64_t)ch.inst * 12 + k];
        LaneAcc<R> acc[kFmOut];
#pragma unroll
        for (int k = 0; k < kFmOut; ++k) acc[k].zero();
        R vacc[kVjpOut];
#pragma unroll
        for (int k = 0; k < kVjpOut; ++k) vacc[k] = (R)0;
        for (int j = lane; j < n; j += 64) {
            const uint32_t e = act[j];
            Rec r;
            if (e & kActSlow) {
                r = load_rec(rec + j);   // written by the slow pass
            } else {
                const uint32_t off = e;
                const float qx = as_global(in.px)[off], qy = as_global(in.py)[off], qz = as_global(in.pz)[off];
                double cc[3], fd[3];
                int idx[3];
                grid_coords(in, qx, qy, qz, cc);
                cell_of_c(G, cc, idx, fd);
                const Corners cr = G.fast ? load_cell(G, idx[0], idx[1], idx[2]) : load_corners(G, idx[0], idx[1], idx[2]);
                r.a[0] = qx; r.a[1] = qy; r.a[2] = qz; r.a[3] = __uint_as_float(e);
                record_fast(G, in, cr, fd, r);
            }
            ContactFwd<R> s;
            record_decode(r, a.slow_diag, in, s);
            contact_forward<R>(I, s, nullptr);
#pragma unroll
            for (int k = 0; k < kFmOut; ++k) acc[k].add(s.f[k]);
            contact_vjp<R, true>(I, s, gb, vacc);
        }
        double* dst = a.partial + (int64_t)c * (kFmOut + kVjpOut);
        double lf[kFmOut];
#pragma unroll
        for (int k = 0; k < kFmOut; ++k) lf[k] = acc[k].value();
        Walk::template store<kFmOut>(s_row, n > 0 ? lds_column_sums<kFmOut>(&s_red[w][0], lf) : 0.0, dst);
        double lv[kVjpOut];
#pragma unroll
        for (int k = 0; k < kVjpOut; ++k) lv[k] = (double)vacc[k];
        double col = n > 0 ? lds_column_sums<kVjpOut>(&s_red[w][0], lv) : 0.0;
        if (lane == 24 || lane == 25) col *= in.kn_chain;   // d/d kn = kn_chain * d/d kn_eff (ForceGeneralSDFContact.cpp:155-156)
        Walk::template store<kVjpOut>(s_vrow, col, dst + kFmOut);
    }
}

// ------------------------------------------------------------------ batched adjoint
// The adjoint of every record of a work item, with d(loss)/d(wrench) of its
// instance, summed into the item's partial row (kVjpOut).
template <typename R, bool SPLIT>
__global__ __launch_bounds__(256) void vjp_kernel(VjpArgs a) {
    using Rec = typename RecOf<R>::type;
    using Walk = ItemWalk<SPLIT>;
    __shared__ double s_red[4][64 * kVjpOut], s_row[4][kVjpOut];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int total = min(a.counters[CNT_CHUNKS], a.chunk_cap);
    for (int c = Walk::begin(); c < total; c += Walk::step()) {
        const ChunkDev ch = as_const(a.chunks)[c];
        if (ch.n == 0) continue;   // its row is not read
        const InstDev in = as_const(a.inst)[ch.inst];
        const int n = min(64 * Walk::U, ch.n - Walk::first());
        const Rec* rec = static_cast<const Rec*>(a.rec) + ch.rec0 + Walk::first();
        const InstR<R> I = make_inst<R>(in);
        R gb[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) gb[k] = (R)a.g_fm[(int64_t)ch.inst * 12 + k];
        R acc[kVjpOut];
#pragma unroll
        for (int k = 0; k < kVjpOut; ++k) acc[k] = (R)0;
        const auto add = [&](const Rec& r) {
            ContactFwd<R> s;
            record_decode(r, a.slow_diag, in, s);
            contact_forward<R>(I, s, nullptr);
            contact_vjp<R, true>(I, s, gb, acc);
        };
        if constexpr (SPLIT) {
            if (lane < n) add(load_rec(rec + lane));
        } else {
            // the next iteration's record is loaded while this one is computed
            Rec cur;
            if (lane < n) cur = load_rec(rec + lane);
            for (int j = lane; j < n; j += 64) {
                Rec nxt = cur;
                if (j + 64 < n) nxt = load_rec(rec + j + 64);
                add(cur);
                cur = nxt;
            }
        }
        double* dst = a.partial + (int64_t)c * kVjpOut;
        double lv[kVjpOut];
#pragma unroll
        for (int k = 0; k < kVjpOut; ++k) lv[k] = (double)acc[k];
        double col = n > 0 ? lds_column_sums<kVjpOut>(&s_red[w][0], lv) : 0.0;
        if (lane == 24 || lane == 25) col *= in.kn_chain;   // d/d kn = kn_chain * d/d kn_eff (ForceGeneralSDFContact.cpp:155-156)
        Walk::template store<kVjpOut>(s_row, col, dst);
    }
}

// ------------------------------------------------------------------ per-instance reduction
// One wavefront per instance. The lanes load the instance's tile entries (active
// count, first work item), 64 tiles at a time, and list the work items' partial rows
// in LDS in tile order, each tile's items in order. Then 64 / W groups of W lanes (W:
// the components, rounded up) take the rows in turn, GROUP of a group's rows read
// together, and the groups' sums are added by halves. The order depends only on the
// tiling: the same result on every run. Every instance's outputs are written (zeros
// when it has no active contact). The chain of dependent reads bounds it: 2,048
// instances of 12,500 points take 4.9 us for 12 components and 6.5 for 26 (one group, the rows
// listed by a scalar cursor: 11.7), 96 of them 3.9 and 4.4 (5.9).
template <int W>
__global__ __launch_bounds__(256) void reduce_kernel(ReduceArgs a) {
    constexpr int G = 64 / W, GROUP = G > 1 ? 8 : 16;
    __shared__ int s_rows[4][64 * 32];   // a tile holds at most 8192 / kChunk items
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int i = (int)blockIdx.x * 4 + w;
    if (a.overflow_out && blockIdx.x == 0 && threadIdx.x == 0) *a.overflow_out = a.counters[CNT_OVERFLOW];
    if (i >= a.n_inst) return;
    const auto in = as_const(a.inst) + i;
    const int tb = in->tile_begin, nt = in->tile_count;
    const auto part = as_global(a.partial);
    int* const rows = s_rows[w];
    // an evaluation whose records did not fit is incomplete: NaN outputs, n_active -1
    const bool ovf = a.counters[CNT_OVERFLOW] != 0;
    const int g = lane / W, comp = lane % W;
    const bool mine = comp < a.nacc;
    double sum = 0.0;
    int nact = 0;
    for (int g0 = 0; g0 < nt; g0 += 64) {
        int cnt = 0, c0 = 0;
        if (g0 + lane < nt) {   // both entries read at once (tile_chunk0 is only meaningful when cnt > 0)
            cnt = a.tile_active[tb + g0 + lane];
            c0 = a.tile_chunk0[tb + g0 + lane];
        }
        nact += cnt;
        const int nch = (cnt + kChunk - 1) / kChunk;
        int pos = nch;
        for (int d = 1; d < min(64, nt - g0); d <<= 1) {
            const int v = __shfl_up(pos, d, 64);
            if (lane >= d) pos += v;
        }
        const int nr = __builtin_amdgcn_readlane(pos, min(64, nt - g0) - 1);
        for (int j = 0; j < nch; ++j) rows[pos - nch + j] = c0 + j;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        for (int j0 = g; j0 < nr; j0 += G * GROUP) {
            int row[GROUP];
            double v[GROUP];
#pragma unroll
            for (int u = 0; u < GROUP; ++u) row[u] = j0 + u * G < nr ? rows[j0 + u * G] : -1;
#pragma unroll
            for (int u = 0; u < GROUP; ++u) v[u] = row[u] >= 0 && mine ? part[(int64_t)row[u] * a.nacc + comp] : 0.0;
#pragma unroll
            for (int u = 0; u < GROUP; ++u) sum += v[u];
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the list is read before the next one
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
#pragma unroll
    for (int d = W; d < 64; d <<= 1) sum += __shfl_xor(sum, d, 64);
    if (ovf) sum = __builtin_nan("");
    if (lane < W && mine) {
        for (int sg = 0; sg < a.nseg; ++sg) {
            const int rel = comp - a.begin[sg];
            if (rel >= 0 && rel < a.width[sg] && a.dst[sg]) a.dst[sg][(int64_t)i * a.width[sg] + rel] = sum;
        }
    }
    if (a.n_active) {
        const int n = (int)wave_sum((double)nact);
        if (lane == 0) a.n_active[i] = ovf ? -1 : n;
    }
    if (a.host_dst) __threadfence_system();   // the stores reach host memory before the launch completes
    if (a.done && lane == 0)
        __hip_atomic_store(a.done + i, a.counters[CNT_CALL], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The per-instance reduction of jacobian_kernel's rows, one workgroup per
// instance: thread k sums component k of the instance's rows, in tile order and
// each tile's items in order (the rows of 64 tiles listed in LDS first, so that
// their reads go out together); the wrench and p6 sums are outputs, and the
// threads form the 288 entries of Km and Dm from the block sums (jac_entry). Rows
// of tangent columns (InstDev::rigid 0) have two components a thread.
template <bool RIGID>
__global__ __launch_bounds__(256) void reduce_jacobian_kernel(ReduceArgs a, int first) {
    constexpr int kRows = 64 * 32;   // a tile holds at most 8192 / kChunk items
    __shared__ int s_rows[kRows];
    __shared__ int s_nrows, s_nact;
    __shared__ double s_sum[RIGID ? kJacRow : kJvpRow], s_m[288], s_R[9], s_t[3];
    const int k = (int)threadIdx.x, i = first + (int)blockIdx.x;
    const bool ovf = a.counters[CNT_OVERFLOW] != 0;
    if (a.overflow_out && i == 0 && k == 0) *a.overflow_out = ovf ? 1 : 0;
    const InstDev in = as_const(a.inst)[i];
    const auto part = as_global(a.partial);
    const bool rigid = RIGID || in.rigid != 0;
    double sum = 0.0, sum2 = 0.0;
    int nact = 0;
    for (int g0 = 0; g0 < in.tile_count; g0 += 64) {
        if (k < 64) {
            int cnt = 0, c0 = 0;
            if (g0 + k < in.tile_count) {   // tile_chunk0 is only meaningful when cnt > 0
                cnt = a.tile_active[in.tile_begin + g0 + k];
                c0 = a.tile_chunk0[in.tile_begin + g0 + k];
            }
            const int nch = (cnt + kChunk - 1) / kChunk;
            int pos = nch;
            for (int d = 1; d < 64; d <<= 1) {
                const int v = __shfl_up(pos, d, 64);
                if (k >= d) pos += v;
            }
            for (int j = 0; j < nch; ++j) s_rows[pos - nch + j] = c0 + j;
            nact += cnt;
            if (k == 63) s_nrows = pos;
        }
        __syncthreads();
        const int nr = s_nrows;
        const auto add_rows = [&](double& to, int comp) {
            int j = 0;
            for (; j + 8 <= nr; j += 8) {
                double v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) v[u] = part[(int64_t)s_rows[j + u] * kJvpRow + comp];
#pragma unroll
                for (int u = 0; u < 8; ++u) to += v[u];
            }
            for (; j < nr; ++j) to += part[(int64_t)s_rows[j] * kJvpRow + comp];
        };
        if (k < kJacRow || !rigid) add_rows(sum, k);
        if (!rigid && k < kJvpRow - 256) add_rows(sum2, k + 256);
        __syncthreads();
    }
    if (k < kJacRow || !rigid) s_sum[k] = ovf ? __builtin_nan("") : sum;
    if (!rigid && k < kJvpRow - 256) s_sum[k + 256] = ovf ? __builtin_nan("") : sum2;
    if (k < 64) {
        nact = (int)wave_sum((double)nact);
        if (k == 0) s_nact = nact;
    }
    if (k == 64) {
        const JacInst J = jac_inst(in);
#pragma unroll
        for (int q = 0; q < 9; ++q) s_R[q] = J.R.a[q];
        s_t[0] = J.t.x; s_t[1] = J.t.y; s_t[2] = J.t.z;
    }
    __syncthreads();
    if (k < 12 && a.dst[0]) a.dst[0][(int64_t)i * 12 + k] = s_sum[k];
    if (k >= 12 && k < 24 && a.dst[1]) a.dst[1][(int64_t)i * 12 + k - 12] = s_sum[k];
    if (k == 0 && a.n_active) a.n_active[i] = ovf ? -1 : s_nact;
    if (a.dst[2] || a.dst[3]) {
        if (rigid)
            for (int e = k; e < 288; e += 256) s_m[e] = jac_element(s_sum + 24, s_sum + 9, s_t, e / 24, e % 24);
        __syncthreads();
        for (int e = k; e < 288; e += 256) {
            const int m = e / 144, row = (e % 144) / 12, col = e % 12;
            double* dst = m ? a.dst[3] : a.dst[2];
            if (dst)
                dst[(int64_t)i * 144 + e % 144] = rigid ? jac_entry(s_m, s_R, row, 12 * m + col) : jvp_entry(s_sum, m, row, col);
        }
    }
    if (a.host_dst) __threadfence_system();   // the stores reach host memory before the launch completes
    if (a.done) {
        __syncthreads();
        if (k == 0) __hip_atomic_store(a.done + i, a.counters[CNT_CALL], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ------------------------------------------------------------------ one workgroup per instance
// The whole evaluation of an instance of at most inst_points(MODE) points by one workgroup
// of 8 wavefronts: detection, the slow-path records, the wrench (p6 column, Km/Dm)
// and the instance's sums, in LDS from step to step. For small batches: the five
// launches of the pipeline above are each a chain of dependent reads, with a drain
// and a launch between them; this is one chain. 64 instances of 500 points: 14 us
// against 30 (wrench), 21 against 33 (Km/Dm); of 2,000 points 18 against 34 and 37
// against 37. What a workgroup's points cost depends on the contacts among them (a
// round of 512 takes 4 us, for Km/Dm some 20), which no rule knows beforehand: of 3,000
// points with 5 % contacts (12 instances) 13.7 us against 25.5, with nothing else 37.6
// against 30.8. So inst_points is small for Km/Dm, and while the GPU is not full the
// wrench of larger instances has a workgroup per tile (MORE), the last of which adds
// the tiles' sums: one of 8,000 points takes 14.6 us with 5 % contacts and 48 with
// nothing else (by one workgroup 16.7 and 84; the pipeline 24 and 31).
// Slow-path contacts: 102 among 2,048 points 14.8 us against 23 in the pipeline, 500 of
// 500 26 against 26, but 2,048 of 2,048 85 against 34 (slow_kernel has the whole GPU;
// with 20 lanes per contact it was 206). One FP32 instance with a tenth, a quarter and
// half of its points slow: of 1,000 14, 19 and 27 us against 22, 24 and 25; of 2,048 18,
// 28 and 48 against 25, 26 and 29; of 8,000 29, 55 and 97 against 27, 31 and 39. So the
// pipeline is the faster one for large faces on a cell plane, which no rule knows either.
// Nothing is reserved with atomics: an instance's records start at its tile's slot
// and its work items at InstDev::chunk0, so a batch needs a record per point. The
// active list, records, work items and tile entries are left as the pipeline leaves
// them, all under the instance's first tile (the slow index of an FP32 record is its
// slot), for the adjoint; the sums run in the pipeline's order, per work item, then the
// items in turn. A host call's instances are read from its pinned copy: an upload of
// its own costs 4 us.
// RIGID: as for jacobian_kernel (MODE 2). MORE (MODE 0): a workgroup per tile.
template <int MODE, typename R, bool RIGID, bool MORE>
__global__ __launch_bounds__(kInstBlock) __attribute__((amdgpu_waves_per_eu(MODE == 2 ? 2 : 4)))
void instance_kernel(InstanceArgs a) {
    using Rec = typename RecOf<R>::type;
    constexpr int NT = kInstBlock, NW = NT / 64, PPL = 4, SP = 64, ITEMS = NW / 4;
    constexpr bool JAC = MODE == 2;
    constexpr int NF = JAC ? (RIGID ? kJacRow : kJvpRow) : MODE == 1 ? 24 : 12;
    constexpr int GROUPS = 64 / kStencil, MANY = 96;
    __shared__ uint16_t s_list[inst_points(MODE)];   // the active offsets in point order, bit 15 = slow path
    __shared__ double s_stencil[NW][GROUPS][kStencil];
    __shared__ double s_val[NW][JAC ? JacColumns::SIZE : 64 * NF];
    // until the contacts: the wavefronts' own active offsets, and the slow ones' places in s_list
    static_assert(sizeof s_val >= 4 * inst_points(MODE), "both lists lie in s_val");
    uint16_t* const s_q = reinterpret_cast<uint16_t*>(s_val);
    uint16_t* const s_slow = s_q + inst_points(MODE);
    __shared__ double s_part[NW][JAC ? (RIGID ? kJacRowPad : kJvpRowPad) : 1];
    __shared__ double s_row[ITEMS][JAC ? 1 : NF];
    __shared__ double s_sum[NF], s_m[JAC ? 288 : 1], s_R[9], s_t[3];
    __shared__ int s_count[NW], s_nslow, s_last;
    const int tid = (int)threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool first = !MORE || (int)blockIdx.x < a.n_inst;   // the instance's first (or only) tile
    const int tile = first ? 0 : as_const(a.more)[(int)blockIdx.x - a.n_inst];
    const int i = first ? (int)blockIdx.x : as_const(a.tiles)[tile].inst;
    const uint64_t lt_mask = (1ull << lane) - 1ull;
    if (tid == 0) s_nslow = 0;
    if (a.src) {
        constexpr int WORDS = sizeof(InstDev) / sizeof(uint4);
        if (tid < WORDS) reinterpret_cast<uint4*>(a.inst + i)[tid] = reinterpret_cast<const uint4*>(a.src + i)[tid];
        __threadfence();
    }
    __syncthreads();
    const InstDev* inst = a.inst;
    asm volatile("" : "+s"(inst));   // its reads stay behind the copy
    // the tile's points: `begin` on, `np` of them
    const auto part = [&](const InstDev& in, int& begin, int& np) {
        begin = first ? 0 : (tile - in.tile_begin) * a.tile_points;
        np = MORE ? min(a.tile_points, (int)in.pt_count - begin) : (int)in.pt_count;
    };
    // detection: wavefront w takes a contiguous range of the steps of 64 points, PPL
    // steps at a time: their point reads, then their table reads, then their cells are
    // out together, so a pass over 2,048 points waits three times
    int wcount = 0, st0;
    {
        const InstDev in = as_const(inst)[i];
        const GridDev G = as_const(a.grids)[in.grid];
        int begin, np;
        part(in, begin, np);
        const int ns = (np + SP - 1) / SP, st1 = (w + 1) * ns / NW;
        st0 = w * ns / NW;
        const auto px = as_global(in.px) + begin, py = as_global(in.py) + begin, pz = as_global(in.pz) + begin;
        const ClsConsts kc = cls_consts_vgpr(G, in);
        const auto cells = ATAC_GLOBAL(G.cells);
        const float cth = (float)in.col_th;
        for (int st = st0; st < st1; st += PPL) {
            const int end = min(np, st1 * SP);
            float x[PPL], y[PPL], z[PPL];
            load_points<PPL>(px, py, pz, st * SP, lane, end, x, y, z);
            unsigned valid = 0, open;
#pragma unroll
            for (int k = 0; k < PPL; ++k)
                if ((st + k) * SP + lane < end) valid |= 1u << k;
            const unsigned cand = detect_candidates<PPL>(G, in, kc, x, y, z, valid, false, open, [] {}, [] {});
            if (!__any(cand != 0u)) continue;
            CandRead r[PPL];
#pragma unroll
            for (int k = 0; k < PPL; ++k) {
                uint32_t off = 0;
                if ((cand >> k) & 1u) off = candidate_locate(G, in, x[k], y[k], z[k], ((open >> k) & 1u) != 0u, r[k]);
                r[k].lo = load_f4_at(cells, off);
                r[k].hi = load_f4_at(cells, off + 16u);
            }
#pragma unroll
            for (int k = 0; k < PPL; ++k) {
                bool act = false, slow = false;
                if ((cand >> k) & 1u) act = candidate_finish(r[k], cth, slow);
                const uint64_t bal = __ballot(act);
                if (act)
                    s_q[st0 * SP + wcount + __popcll(bal & lt_mask)] =
                        (uint16_t)((unsigned)((st + k) * SP + lane) | (slow ? 0x8000u : 0u));
                wcount += __popcll(bal);
            }
        }
    }
    if (lane == 0) s_count[w] = wcount;
    __syncthreads();
    // the record again, behind an opaque pointer: kept from the detection on, its 700
    // bytes would go through register spills
    const InstDev* again = a.inst;
    asm volatile("" : "+s"(again));
    const InstDev in = as_const(again)[i];
    const GridDev G = as_const(a.grids)[in.grid];
    int begin, np;
    part(in, begin, np);
    const auto px = as_global(in.px) + begin, py = as_global(in.py) + begin, pz = as_global(in.pz) + begin;
    // the active list in point order, for the adjoint too, and the slow-path contacts
    int before = 0, cnt = 0;
    for (int k = 0; k < NW; ++k) {
        if (k < w) before += s_count[k];
        cnt += s_count[k];
    }
    const int64_t slot0 = in.tile_count ? as_const(a.tiles)[in.tile_begin].slot + begin : 0;
    for (int k = lane; k < wcount; k += 64) {
        const uint32_t e = s_q[st0 * SP + k];
        const int j = before + k;
        s_list[j] = (uint16_t)e;
        a.act[slot0 + j] = ((uint32_t)begin + (e & 0x7fffu)) | (e >> 15 ? kActSlow : 0u);
        if (e >> 15) s_slow[atomicAdd(&s_nslow, 1)] = (uint16_t)j;
    }
    // work items: kChunk contacts each
    const int items = (cnt + kChunk - 1) / kChunk;
    const int tile_at = first ? in.tile_begin : tile, chunk0 = in.chunk0 + begin / kChunk;
    if (tid == 0 && in.tile_count) {
        a.tile_active[tile_at] = cnt;
        a.tile_chunk0[tile_at] = chunk0;
        if constexpr (!MORE)   // one workgroup for all of the instance's tiles
            for (int t = 1; t < in.tile_count; ++t) a.tile_active[tile_at + t] = 0;
    }
    if (tid < (np + kChunk - 1) / kChunk)
        a.chunks[chunk0 + tid] = tid < items ? ChunkDev{i, min(kChunk, cnt - tid * kChunk), slot0 + tid * kChunk}
                                             : ChunkDev{i, 0, 0};
    if (blockIdx.x == 0 && tid == 0) {
        a.counters[CNT_RECS] = 0;   // counted by the tiles' entries
        a.counters[CNT_CHUNKS] = a.chunk_total;
        a.counters[CNT_SLOW] = 0;
        a.counters[CNT_OVERFLOW] = 0;
    }
    __syncthreads();
    // slow-path records: the 20 stencil evaluations of a contact on 20 lanes, as slow_kernel
    // (2.4 us for 24 contacts); many: a lane per contact, the stencil's positions along the
    // axes formed once (14 us for 512)
    Rec* rec = static_cast<Rec*>(a.rec) + slot0;
    const auto slow_point = [&](int k, Rec& r) {
        const int j = s_slow[k];
        const uint32_t off = s_list[j] & 0x7fffu;
        r.a[0] = px[off]; r.a[1] = py[off]; r.a[2] = pz[off]; r.a[3] = __uint_as_float((uint32_t)begin + off);
        return j;
    };
    const auto diag_of = [&](int j) { return a.slow_diag ? a.slow_diag + 4 * (slot0 + j) : nullptr; };
    const int many = s_nslow > MANY ? s_nslow : 0;
    for (int k = tid; k < many; k += NT) {
        Rec r;
        const int j = slow_point(k, r);
        record_slow(G, in, r, diag_of(j));
        mark_slow_index(r, (int)(slot0 + j));
        store_rec(rec + j, r);
    }
    for (int base = many + w * GROUPS; base < s_nslow; base += NW * GROUPS) {
        const int grp = lane / kStencil, st = lane % kStencil;
        const bool mine = grp < GROUPS && base + grp < s_nslow;
        Rec r;
        int j = 0;
        if (mine) {
            j = slow_point(base + grp, r);
            double x[3], q[3];
            bool accurate;
            body2_point(in, (double)r.a[0], (double)r.a[1], (double)r.a[2], x);
            stencil_point(x, st, q, accurate);
            s_stencil[w][grp][st] = query_sdf64(G, q[0], q[1], q[2], accurate);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (mine && st == 0) {
            double v[kStencil], val, g[3], H[6];
#pragma unroll
            for (int q = 0; q < kStencil; ++q) v[q] = s_stencil[w][grp][q];
            stencil_combine(v, val, g, H);
            record_slow_fill(in, val, g, H, r, diag_of(j));
            mark_slow_index(r, (int)(slot0 + j));
            store_rec(rec + j, r);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    // ITEMS work items at a time, a wavefront per 64 contacts
    const bool rigid = RIGID || in.rigid != 0;
    const int nf = JAC && rigid ? kJacRow : NF;
    double total = 0.0;   // thread k < nf: component k of the instance's sums
    const InstR<R> I = make_inst<R>(in);
    for (int m0 = 0; m0 < items; m0 += ITEMS) {
        const int start = (m0 + (w >> 2)) * kChunk, n = max(0, min(kChunk, cnt - start));
        const int p0 = 64 * (w & 3), nw = n - p0;
        if (nw > 0) {
            const int j = start + p0 + min(lane, nw - 1);   // lanes past the end repeat the last record, not summed
            const uint32_t e = s_list[j], off = e & 0x7fffu;
            ContactFwd<R> s;
            R p6[12];
            const auto forward = [&](const InstDev& in, const InstR<R>& I) {
                const Rec r = item_record(G, in, ((uint32_t)begin + off) | (e >> 15 ? kActSlow : 0u), px[off], py[off], pz[off],
                                          rec + j);
                record_decode(r, a.slow_diag, in, s);
                contact_forward<R>(I, s, MODE >= 1 ? p6 : nullptr);
            };
            if constexpr (JAC) {
                if (RIGID || rigid) {
                    forward(in, I);
                    put_jac_row<R>(JacColumns{&s_val[w][0], &s_part[w][0], lane, nw}, jac_inst(in), s, p6);
                } else {   // a branch of its own, as in jacobian_kernel
                    const InstDev* third = a.inst;
                    asm volatile("" : "+s"(third));
                    const InstDev in3 = as_const(third)[i];
                    const InstR<R> I3 = make_inst<R>(in3);
                    forward(in3, I3);
                    put_jvp_row<R>(JvpColumns{&s_val[w][0], &s_part[w][0], lane, nw}, I3, s, p6);
                }
            } else {
                forward(in, I);
#pragma unroll
                for (int k = 0; k < 12; ++k) s_val[w][lane * NF + k] = (double)s.f[k];
                if constexpr (MODE == 1) {
#pragma unroll
                    for (int k = 0; k < 12; ++k) s_val[w][lane * NF + 12 + k] = (double)p6[k];
                }
            }
        }
        __syncthreads();
        if constexpr (!JAC) {
            if ((w & 3) == 0 && n > 0) {   // a lane's records 64 apart in turn, then the lanes
                double lv[NF];
#pragma unroll
                for (int k = 0; k < NF; ++k) lv[k] = lane < n ? s_val[w][lane * NF + k] : 0.0;
                for (int u = 1; u < 4; ++u)
                    if (64 * u + lane < n) {
#pragma unroll
                        for (int k = 0; k < NF; ++k) lv[k] += s_val[w + u][lane * NF + k];
                    }
                const double col = lds_column_sums<NF>(&s_val[w][0], lv);
                if (lane < NF) s_row[w >> 2][lane] = col;
            }
            __syncthreads();
            if (tid < NF) {
                for (int h = 0; h < ITEMS && m0 + h < items; ++h) total += s_row[h][tid];
            }
        } else if (tid < nf) {
            for (int h = 0; h < ITEMS && m0 + h < items; ++h) {
                const int nh = min(kChunk, cnt - (m0 + h) * kChunk);
                double v = s_part[4 * h][tid];
                for (int u = 1; u < 4; ++u)
                    if (nh > 64 * u) v += s_part[4 * h + u][tid];
                total += v;
            }
        }
        __syncthreads();
    }
    if (tid < nf) s_sum[tid] = total;
    if constexpr (JAC) {
        if (tid == NT - 1) {
            const JacInst J = jac_inst(in);
#pragma unroll
            for (int q = 0; q < 9; ++q) s_R[q] = J.R.a[q];
            s_t[0] = J.t.x; s_t[1] = J.t.y; s_t[2] = J.t.z;
        }
    }
    __syncthreads();
    if constexpr (MORE) {
        if (in.tile_count > 1) {   // the last of the instance's workgroups adds the tiles' sums, in their order
            if (tid < 12)
                __hip_atomic_store(a.tile_sum + 12 * (int64_t)tile_at + tid, s_sum[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (tid == 0)   // one release and acquire for the workgroup: each writes the XCD's L2 back
                s_last = __hip_atomic_fetch_add(a.tiles_done + i, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == in.tile_count - 1;
            __syncthreads();
            if (!s_last) return;
            cnt = 0;
            double sum = 0.0;
            for (int t = in.tile_begin; t < in.tile_begin + in.tile_count; ++t) {
                cnt += __hip_atomic_load(a.tile_active + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (tid < 12) sum += __hip_atomic_load(a.tile_sum + 12 * (int64_t)t + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            if (tid < 12) s_sum[tid] = sum;
            if (tid == 0) __hip_atomic_store(a.tiles_done + i, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
        }
    }
    if (a.overflow_out && i == 0 && tid == 0) *a.overflow_out = 0;
    if (tid < 12 && a.fm) a.fm[(int64_t)i * 12 + tid] = s_sum[tid];
    if (MODE >= 1 && tid >= 12 && tid < 24 && a.p6) a.p6[(int64_t)i * 12 + tid - 12] = s_sum[MODE >= 1 ? tid : 0];
    if (tid == 0 && a.n_active) a.n_active[i] = cnt;
    if constexpr (JAC) {
        if (tid < 288 && rigid) s_m[JAC ? tid : 0] = jac_element(s_sum + 24, s_sum + 9, s_t, tid / 24, tid % 24);
        __syncthreads();
        if (tid < 288) {
            const int m = tid / 144, row = (tid % 144) / 12, col = tid % 12;
            double* dst = m ? a.Dm : a.Km;
            if (dst)
                dst[(int64_t)i * 144 + tid % 144] = rigid ? jac_entry(s_m, s_R, row, 12 * m + col) : jvp_entry(s_sum, m, row, col);
        }
    }
    if (a.host_dst) __threadfence_system();   // the stores reach host memory before the launch completes
    if (a.done) {
        __syncthreads();
        if (tid == 0) __hip_atomic_store(a.done + i, a.call, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// The instances' records from (pinned) host memory to the device: a kernel rather
// than a copy, which starts and ends several microseconds later in a stream.
__global__ __launch_bounds__(256) void upload_kernel(const uint4* src, uint4* dst, int64_t n, const int32_t* call,
                                                     int32_t* counters) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k < n) dst[k] = src[k];
    if (k == 0 && call) counters[CNT_CALL] = *call;
}

__global__ __launch_bounds__(64) void pose_rows_kernel(const double* E1, const double* E2, const double* phi1,
                                                       const double* phi2, const double* kn, const double* kt, double* rows,
                                                       int32_t* done, int32_t call) {
    const int k = (int)threadIdx.x;
    const int64_t i = blockIdx.x;
    if (k < kPoseRow)
        rows[i * kPoseRow + k] = k < 16 ? E1[16 * i + k] : k < 22 ? phi1[6 * i + k - 16] : k < 38 ? E2[16 * i + k - 22]
                               : k < 44 ? phi2[6 * i + k - 38] : k == 44 ? kn[i] : kt[i];
    __threadfence_system();   // one wavefront: every lane's store is out before lane 0's
    if (k == 0) __hip_atomic_store(done + i, call, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A lane per pose: E^T X = M by elimination with row exchanges, in registers. A pose
// with a pivot within 2^-40 of its largest entry (or no number) is reported: a matrix
// without an inverse leaves a rounding (2^-52 of that entry) there as often as a zero.
__global__ __launch_bounds__(64) void pose_gradients_kernel(const double* E1, const double* g1, double* gE1,
                                                            const double* E2, const double* g2, double* gE2,
                                                            int32_t* done, int32_t call, int n) {
    const int64_t t = (int64_t)blockIdx.x * 64 + threadIdx.x, i = t >> 1;
    if (i >= n) return;
    const double* E = (t & 1) ? E2 : E1;
    const double* g = (t & 1) ? g2 : g1;
    double* out = (t & 1) ? gE2 : gE1;
    bool singular = false;
    if (out) {
        double m[4][8];   // [E^T | M]
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                m[r][c] = E[16 * i + 4 * c + r];
                m[r][4 + c] = 0.0;
            }
        const double w0 = 0.5 * g[6 * i], w1 = 0.5 * g[6 * i + 1], w2 = 0.5 * g[6 * i + 2];
        m[0][5] = -w2; m[0][6] = w1;
        m[1][4] = w2;  m[1][6] = -w0;
        m[2][4] = -w1; m[2][5] = w0;
        m[0][7] = g[6 * i + 3]; m[1][7] = g[6 * i + 4]; m[2][7] = g[6 * i + 5];
        double least = 0.0;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) least = fmax(least, fabs(m[r][c]));
        least *= 0x1p-40;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
#pragma unroll
            for (int r = k + 1; r < 4; ++r) {
                const bool swap = fabs(m[r][k]) > fabs(m[k][k]);
#pragma unroll
                for (int c = k; c < 8; ++c) {
                    const double a = m[k][c], b = m[r][c];
                    m[k][c] = swap ? b : a;
                    m[r][c] = swap ? a : b;
                }
            }
            singular = singular || !(fabs(m[k][k]) > least);
#pragma unroll
            for (int r = k + 1; r < 4; ++r) {
                const double f = m[r][k] / m[k][k];
#pragma unroll
                for (int c = k + 1; c < 8; ++c) m[r][c] -= f * m[k][c];
            }
        }
#pragma unroll
        for (int c = 4; c < 8; ++c) {
#pragma unroll
            for (int k = 3; k >= 0; --k) {
                double v = m[k][c];
#pragma unroll
                for (int j = k + 1; j < 4; ++j) v -= m[k][j] * m[j][c];
                m[k][c] = v / m[k][k];
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) out[16 * i + 4 * r + c] = m[r][4 + c];
    }
    __hip_atomic_store(done + t, singular ? -call : call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------------ grid set-up
__global__ void build_cells_kernel(GridDev G, float4* cells) {
    const int64_t ci = G.n[0], cj = G.n[1], ck = G.n[2], nc = ci * cj * ck;
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < nc; c += (int64_t)gridDim.x * blockDim.x)
        pack_cell(G, (int)(c % ci), (int)((c / ci) % cj), (int)(c / (ci * cj)), cells + 2 * c);
}

__global__ void build_cls_kernel(GridDev G, double col_th, uint8_t* cls) {
    const int64_t ne = (int64_t)cls_bytes(G);
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < ne; e += (int64_t)gridDim.x * blockDim.x)
        cls[e] = cls_fill(G, col_th, (uint32_t)e);
}

hipError_t launch_grid_setup(const GridDev& G, float4* cells, hipStream_t st) {
    hipLaunchKernelGGL(build_cells_kernel, dim3(1024), dim3(256), 0, st, G, cells);
    return hipGetLastError();
}

hipError_t launch_cls_setup(const GridDev& G, double col_th, uint8_t* cls, hipStream_t st) {
    hipLaunchKernelGGL(build_cls_kernel, dim3(1024), dim3(256), 0, st, G, col_th, cls);
    return hipGetLastError();
}

// The table's entries: 0 on the lower faces, elsewhere whether block (x-1, y-1, z-1) is open.
__global__ void sat_mark_kernel(GridDev G, const uint8_t* cls, int32_t* sat) {
    const uint32_t dx = sat_dim(G, 0), dy = sat_dim(G, 1), dz = sat_dim(G, 2);
    const int64_t n = (int64_t)dx * dy * dz;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        const uint32_t x = (uint32_t)(e % dx), y = (uint32_t)((e / dx) % dy), z = (uint32_t)(e / ((int64_t)dx * dy));
        sat[e] = (x && y && z && sat_block_open(G, cls, x - 1, y - 1, z - 1)) ? 1 : 0;
    }
}

// Running sums along one axis, one lane per line.
__global__ void sat_scan_kernel(GridDev G, int32_t* sat, int axis) {
    const uint32_t d[3] = {sat_dim(G, 0), sat_dim(G, 1), sat_dim(G, 2)};
    const int a1 = axis == 0 ? 1 : 0, a2 = axis == 2 ? 1 : 2;
    const int64_t lines = (int64_t)d[a1] * d[a2];
    const int64_t stride = axis == 0 ? 1 : (axis == 1 ? (int64_t)d[0] : (int64_t)d[0] * d[1]);
    for (int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; l < lines; l += (int64_t)gridDim.x * blockDim.x) {
        uint32_t c[3];
        c[axis] = 0;
        c[a1] = (uint32_t)(l % d[a1]);
        c[a2] = (uint32_t)(l / d[a1]);
        int32_t* p = sat + sat_index(G, c[0], c[1], c[2]);
        int32_t run = 0;
        for (uint32_t k = 0; k < d[axis]; ++k) {
            run += p[k * stride];
            p[k * stride] = run;
        }
    }
}

hipError_t launch_sat_setup(const GridDev& G, const uint8_t* cls, int32_t* sat, hipStream_t st) {
    hipLaunchKernelGGL(sat_mark_kernel, dim3(512), dim3(256), 0, st, G, cls, sat);
    for (int axis = 0; axis < 3; ++axis) hipLaunchKernelGGL(sat_scan_kernel, dim3(64), dim3(256), 0, st, G, sat, axis);
    return hipGetLastError();
}

// One lane per group, `slots` lanes per tile (so 64 / slots tiles per
// wavefront): the tiles' live-group masks. Block 0 also clears the evaluation's
// counters, which the detection kernel launched after it accumulates into.
__global__ __launch_bounds__(256) void cull_kernel(CullArgs a) {
    if (blockIdx.x == 0 && threadIdx.x < CNT_WORDS) a.counters[threadIdx.x] = 0;
    const int lane = threadIdx.x & 63, S = a.slots;
    const int64_t gi = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int tile = (int)(gi / S), g = (int)(gi % S);
    bool live = false;
    if (tile < a.n_tiles) {
        const TileDev& t = a.tiles[tile];
        const int ng = (t.count + kGroup - 1) / kGroup;
        if (g < ng) {
            live = true;
            const InstDev& in = a.inst[t.inst];
            const GridDev& G = a.grids[t.grid];
            if (G.fast && in.cls && in.csat && in.gbox) {
                const float4* b = reinterpret_cast<const float4*>(in.gbox) + 2 * (t.begin / kGroup + g);
                const float4 l = b[0], h = b[1];
                const float lo[3] = {l.x, l.y, l.z}, hi[3] = {h.x, h.y, h.z};
                live = group_live(G, in, in.csat, lo, hi);
            }
        }
    }
    const uint64_t m = __ballot(live);
    if ((lane & (S - 1)) == 0 && tile < a.n_tiles)
        a.tile_live[tile] = (uint32_t)((m >> lane) & (S >= 32 ? 0xffffffffull : ((1ull << S) - 1ull)));
}

hipError_t launch_cull(const CullArgs& a, hipStream_t st) {
    if (a.n_tiles <= 0) return hipSuccess;
    const int64_t lanes = (int64_t)a.n_tiles * a.slots;
    hipLaunchKernelGGL(cull_kernel, dim3((unsigned)((lanes + 255) / 256)), dim3(256), 0, st, a);
    return hipGetLastError();
}

__global__ void reset_counters_kernel(int32_t* c, int n) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = 0;
}

__global__ void zero_words_kernel(uint32_t* p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = 0u;
}

// ------------------------------------------------------------------ plain per-instance path
template <typename R>
__global__ void plain_kernel(PlainArgs a) {
    const int64_t o = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const InstDev& in = a.inst[a.i];
    if (o >= in.pt_count) return;
    const GridDev G = a.grids[in.grid];
    const float x = in.px[o], y = in.py[o], z = in.pz[o];
    if (!(detect_value(G, in, x, y, z) < 0.0f)) return;
    const InstR<R> I = make_inst<R>(in);
    ContactFwd<R> s;
    contact_sample<R>(G, in, (double)x, (double)y, (double)z, s);
    R p6[12];
    contact_forward<R>(I, s, a.p6 ? p6 : nullptr);
    for (int k = 0; k < 12; ++k) atomicAdd(a.fm + k, (double)s.f[k]);
    if (a.p6)
        for (int k = 0; k < 12; ++k) atomicAdd(a.p6 + k, (double)p6[k]);
    if (a.Km) {
        for (int j = 0; j < 24; ++j) {
            R col[12];
            contact_jvp<R>(I, s, unit_tangent<R>(j), col);
            double* dst = (j < 12) ? a.Km + j : a.Dm + (j - 12);
            for (int r = 0; r < 12; ++r) atomicAdd(dst + 12 * r, (double)col[r]);
        }
    }
    if (a.grad) {
        R gb[12], v[kVjpOut];
        for (int k = 0; k < 12; ++k) gb[k] = (R)a.g_fm[k];
        contact_vjp<R>(I, s, gb, v);
        v[24] *= (R)in.kn_chain;   // d/d kn = kn_chain * d/d kn_eff (ForceGeneralSDFContact.cpp:155-156)
        v[25] *= (R)in.kn_chain;
        for (int k = 0; k < kVjpOut; ++k) atomicAdd(a.grad + k, (double)v[k]);
    }
    atomicAdd(a.n_active, 1);
}

// ------------------------------------------------------------------ per-point API kernels
// BodySDFObj::distance for world points (BodySDFObj.cpp:207-213): x in FP64,
// cell and fraction in FP64, corners and interpolation in FP32.
__global__ void distance_kernel(PointArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const double xw0 = a.xw[3 * i], xw1 = a.xw[3 * i + 1], xw2 = a.xw[3 * i + 2];
    const double q0 = xw0 - a.in.p2[0], q1 = xw1 - a.in.p2[1], q2 = xw2 - a.in.p2[2];
    double x[3];
    for (int r = 0; r < 3; ++r) x[r] = a.in.R2[r] * q0 + a.in.R2[3 + r] * q1 + a.in.R2[6 + r] * q2;
    const GridDev& G = a.grid;
    const bool inside = x[0] >= G.minb[0] && x[0] <= G.maxb[0] && x[1] >= G.minb[1] && x[1] <= G.maxb[1] &&
                        x[2] >= G.minb[2] && x[2] <= G.maxb[2];
    if (!inside) {
        a.out[i] = (double)FLT_MAX + a.in.col_th;
        return;
    }
    int idx[3];
    float f[3];
    int64_t st[3];
    for (int k = 0; k < 3; ++k) {
        const double c = (x[k] - G.minb[k]) / G.d[k];
        int ii = (int)floor(c);
        const double fr = c - ii;
        ii = ii < 0 ? 0 : (ii > G.n[k] - 1 ? G.n[k] - 1 : ii);
        idx[k] = ii;
        f[k] = (float)fr;
    }
    st[0] = idx[0] < G.n[0] - 1 ? 1 : 0;
    st[1] = idx[1] < G.n[1] - 1 ? G.n[0] : 0;
    st[2] = idx[2] < G.n[2] - 1 ? (int64_t)G.n[0] * G.n[1] : 0;
    const float* v = G.v + grid_index(G, idx[0], idx[1], idx[2]);
    const float p = lerpf(v[0], v[st[0]], f[0]), q = lerpf(v[st[1]], v[st[1] + st[0]], f[0]);
    const float r = lerpf(v[st[2]], v[st[2] + st[0]], f[0]), s = lerpf(v[st[2] + st[1]], v[st[2] + st[1] + st[0]], f[0]);
    a.out[i] = (double)lerpf(lerpf(p, q, f[1]), lerpf(r, s, f[1]), f[2]) + a.in.col_th;
}

// BodySDFObj::collision for world points and velocities (BodySDFObj.cpp:239-377):
// values (11 per point) and, with DERIV, the 14 derivative blocks (135 per point)
// in the reference's order, each block row-major. A wavefront takes kCollPoints
// points, two lanes each: both form the point's values and each takes every other
// of the 18 directions. The results wait in LDS (in the arithmetic's type) and
// leave in memory order, 512 bytes per store: written by the lanes themselves,
// each store touched 64 lines 1,080 bytes apart (120,000 points with derivatives:
// 191 -> 51 us a call). Bound by the 1,168 bytes a point writes.
constexpr int kCollPoints = 32, kCollLanes = 64 / kCollPoints;
template <bool DERIV, typename R>
__global__ __launch_bounds__(64) void collision_kernel(PointArgs a) {
    constexpr int NV = 11, ND = 135;
    __shared__ R s_v[kCollPoints * NV];
    __shared__ R s_d[DERIV ? kCollPoints * ND : 1];
    const int lane = (int)threadIdx.x, pt = lane / kCollLanes, half = lane % kCollLanes;
    const int64_t base = (int64_t)blockIdx.x * kCollPoints;
    const int np = (int)min((int64_t)kCollPoints, a.n - base);
    if (pt < np) {
        const int64_t i = base + pt;
        const InstR<R> I = make_inst<R>(a.in);
        ContactFwd<R> s;
        contact_sample<R>(a.grid, a.in, a.xw[3 * i], a.xw[3 * i + 1], a.xw[3 * i + 2], s);
        s.xw1dot = mk3<R>((R)a.xwdot[3 * i], (R)a.xwdot[3 * i + 1], (R)a.xwdot[3 * i + 2]);
        collision_forward<R>(I, s);
        if (half == 0) {
            R* v = s_v + NV * pt;
            v[0] = s.d; v[1] = s.n.x; v[2] = s.n.y; v[3] = s.n.z; v[4] = s.ddot;
            v[5] = s.tdot.x; v[6] = s.tdot.y; v[7] = s.tdot.z; v[8] = s.xi2.x; v[9] = s.xi2.y; v[10] = s.xi2.z;
        }
        if constexpr (DERIV) {
            R* o = s_d + ND * pt;
            // offsets of the blocks in the 135-value record
            enum { DD_DXW = 0, DD_DQ2 = 3, DN_DXW = 9, DN_DQ2 = 18, DDD_DXW = 36, DDD_DXWDOT = 39, DDD_DQ2 = 42, DDD_DPHI2 = 48,
                   DT_DXW = 54, DT_DXWDOT = 63, DT_DQ2 = 72, DT_DPHI2 = 90, DXI_DXW = 108, DXI_DQ2 = 117 };
#pragma unroll 1
            for (int c = half; c < 18; c += kCollLanes) {   // xw 3, xw_dot 3, q2 = [w2; v2] 6, phi2 6
                const int slot = c / 3, ax = c - 3 * slot;
                const v3<R> u = mk3<R>((R)(ax == 0), (R)(ax == 1), (R)(ax == 2)), Z = zero3<R>();
                CollTangent<R> t;
                collision_jvp<R>(I, s, slot == 0 ? u : Z, slot == 1 ? u : Z, slot == 2 ? u : Z, slot == 3 ? u : Z,
                                 slot == 4 ? u : Z, slot == 5 ? u : Z, t);
                const bool xw = slot == 0, xd = slot == 1, q2 = slot == 2 || slot == 3;
                const int col = (xw || xd) ? ax : (q2 ? c - 6 : c - 12), w = (xw || xd) ? 3 : 6;   // column and width of its blocks
                const R dn[3] = {t.dn.x, t.dn.y, t.dn.z}, dt[3] = {t.dtdot.x, t.dtdot.y, t.dtdot.z};
                const R dx[3] = {t.dxi2.x, t.dxi2.y, t.dxi2.z};
                const int od = xw ? DDD_DXW : xd ? DDD_DXWDOT : q2 ? DDD_DQ2 : DDD_DPHI2;
                const int ot = xw ? DT_DXW : xd ? DT_DXWDOT : q2 ? DT_DQ2 : DT_DPHI2;
                o[od + col] = t.dddot;
#pragma unroll
                for (int r = 0; r < 3; ++r) o[ot + w * r + col] = dt[r];
                if (xw || q2) {
                    o[(xw ? DD_DXW : DD_DQ2) + col] = t.dd;
                    const int on = xw ? DN_DXW : DN_DQ2, ox = xw ? DXI_DXW : DXI_DQ2;
#pragma unroll
                    for (int r = 0; r < 3; ++r) { o[on + w * r + col] = dn[r]; o[ox + w * r + col] = dx[r]; }
                }
            }
        }
    }
    __syncthreads();
    for (int k = lane; k < np * NV; k += 64) a.out[base * NV + k] = (double)s_v[k];
    if constexpr (DERIV)
        for (int k = lane; k < np * ND; k += 64) a.out2[base * ND + k] = (double)s_d[k];
}

// Marks every grid value read by the 8-corner stencil of an inside point.
__global__ void touched_kernel(TouchedArgs a) {
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int inst_i = blockIdx.y;
    const InstDev& in = a.inst[inst_i];
    for (int64_t o = gid; o < in.pt_count; o += (int64_t)gridDim.x * blockDim.x) {
        const GridDev G = a.grids[in.grid];
        double cc[3];
        grid_coords(in, in.px[o], in.py[o], in.pz[o], cc);
        const double c0 = cc[0], c1 = cc[1], c2 = cc[2];
        if (!(c0 >= 0.0 && c0 <= in.cmax[0] && c1 >= 0.0 && c1 <= in.cmax[1] && c2 >= 0.0 && c2 <= in.cmax[2])) continue;
        int i = (int)c0, j = (int)c1, k = (int)c2;
        i = i < G.n[0] - 1 ? i : G.n[0] - 1;
        j = j < G.n[1] - 1 ? j : G.n[1] - 1;
        k = k < G.n[2] - 1 ? k : G.n[2] - 1;
        const int ip = i < G.n[0] - 1 ? i + 1 : i, jp = j < G.n[1] - 1 ? j + 1 : j, kp = k < G.n[2] - 1 ? k + 1 : k;
        uint32_t* bits = a.bits + a.bit_offset[in.grid];
        const int ii[2] = {i, ip}, jj[2] = {j, jp}, kk[2] = {k, kp};
        for (int c = 0; c < 8; ++c) {
            const int64_t idx = grid_index(G, ii[c & 1], jj[(c >> 1) & 1], kk[c >> 2]);
            atomicOr(bits + (idx >> 5), 1u << (idx & 31));
        }
    }
}

__global__ void popcount_kernel(const uint32_t* bits, int64_t nwords, unsigned long long* out) {
    unsigned long long c = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nwords; i += (int64_t)gridDim.x * blockDim.x)
        c += __popc(bits[i]);
    atomicAdd(out, c);
}

// ------------------------------------------------------------------ launchers
template <int BLOCK>
static const void* detect_ptr_b(int ppl) {
    return ppl == 1 ? (const void*)&detect_kernel<BLOCK, 1>
         : ppl == 2 ? (const void*)&detect_kernel<BLOCK, 2> : (const void*)&detect_kernel<BLOCK, 4>;
}

const void* detect_kernel_ptr(int block, int ppl) {
    if (ppl != 1 && ppl != 2 && ppl != 4) return nullptr;
    switch (block) {
        case 64: return detect_ptr_b<64>(ppl);
        case 128: return detect_ptr_b<128>(ppl);
        case 256: return detect_ptr_b<256>(ppl);
        case 512: return detect_ptr_b<512>(ppl);
        case 1024: return detect_ptr_b<1024>(ppl);
        default: return nullptr;
    }
}

hipError_t launch_detect(const DetectArgs& a, int block, int ppl, int grid, size_t lds, hipStream_t st) {
    const void* f = detect_kernel_ptr(block, ppl);
    if (!f) return hipErrorInvalidValue;
    DetectArgs args = a;
    void* params[] = {&args};
    return hipLaunchKernel(f, dim3(grid), dim3(block), params, lds, st);
}

hipError_t launch_slow(const SlowArgs& a, bool precise, int grid, hipStream_t st) {
    if (precise) hipLaunchKernelGGL(slow_kernel<true>, dim3(grid), dim3(64), 0, st, a);
    else hipLaunchKernelGGL(slow_kernel<false>, dim3(grid), dim3(64), 0, st, a);
    return hipGetLastError();
}

template <typename R, bool SPLIT>
static const void* contact_ptr_t(int mode, bool rigid) {
    return mode == 0   ? (const void*)&contact_kernel<false, R, SPLIT>
           : mode == 1 ? (const void*)&contact_kernel<true, R, SPLIT>
           : rigid     ? (const void*)&jacobian_kernel<R, true> : (const void*)&jacobian_kernel<R, false>;
}

const void* contact_kernel_ptr(int mode, bool precise, bool split, bool rigid) {
    if (split) return precise ? contact_ptr_t<double, true>(mode, rigid) : contact_ptr_t<float, true>(mode, rigid);
    return precise ? contact_ptr_t<double, false>(mode, rigid) : contact_ptr_t<float, false>(mode, rigid);
}

hipError_t launch_contact(const ContactArgs& a, int mode, bool precise, bool split, bool rigid, int grid, hipStream_t st) {
    ContactArgs args = a;
    void* params[] = {&args};
    return hipLaunchKernel(contact_kernel_ptr(mode, precise, split, rigid), dim3(grid), dim3(256), params, 0, st);
}

hipError_t launch_vjp(const VjpArgs& a, bool precise, bool split, int grid, hipStream_t st) {
    VjpArgs args = a;
    void* params[] = {&args};
    const void* k = split ? (precise ? (const void*)&vjp_kernel<double, true> : (const void*)&vjp_kernel<float, true>)
                          : (precise ? (const void*)&vjp_kernel<double, false> : (const void*)&vjp_kernel<float, false>);
    return hipLaunchKernel(k, dim3(grid), dim3(256), params, 0, st);
}

hipError_t launch_fused(const ContactArgs& a, bool precise, bool split, int grid, hipStream_t st) {
    ContactArgs args = a;
    void* params[] = {&args};
    const void* k = split ? (precise ? (const void*)&fused_kernel<double, true> : (const void*)&fused_kernel<float, true>)
                          : (precise ? (const void*)&fused_kernel<double, false> : (const void*)&fused_kernel<float, false>);
    return hipLaunchKernel(k, dim3(grid), dim3(256), params, 0, st);
}

hipError_t launch_reduce(const ReduceArgs& a, hipStream_t st) {
    if (a.n_inst <= 0) return hipSuccess;
    const dim3 grid((a.n_inst + 3) / 4), block(256);
    if (a.nacc <= 16) hipLaunchKernelGGL(reduce_kernel<16>, grid, block, 0, st, a);
    else if (a.nacc <= 32) hipLaunchKernelGGL(reduce_kernel<32>, grid, block, 0, st, a);
    else hipLaunchKernelGGL(reduce_kernel<64>, grid, block, 0, st, a);
    return hipGetLastError();
}

hipError_t launch_reduce_jacobian(const ReduceArgs& a, bool rigid, hipStream_t st) {
    constexpr int64_t kMost = 1 << 23;   // a launch holds fewer than 2^32 threads
    for (int64_t first = 0; first < a.n_inst; first += kMost) {
        const dim3 grid((unsigned)(a.n_inst - first < kMost ? a.n_inst - first : kMost));
        if (rigid) hipLaunchKernelGGL(reduce_jacobian_kernel<true>, grid, dim3(256), 0, st, a, (int)first);
        else hipLaunchKernelGGL(reduce_jacobian_kernel<false>, grid, dim3(256), 0, st, a, (int)first);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

template <int MODE, bool RIGID, bool MORE>
static void launch_instance_m(const InstanceArgs& a, bool precise, hipStream_t st) {
    const dim3 grid(a.n_inst + (MORE ? a.n_more : 0));
    if (precise) hipLaunchKernelGGL((instance_kernel<MODE, double, RIGID, MORE>), grid, dim3(kInstBlock), 0, st, a);
    else hipLaunchKernelGGL((instance_kernel<MODE, float, RIGID, MORE>), grid, dim3(kInstBlock), 0, st, a);
}

hipError_t launch_instance(const InstanceArgs& a, int mode, bool precise, bool rigid, hipStream_t st) {
    if (a.n_inst <= 0) return hipSuccess;
    if (mode == 0 && a.n_more) launch_instance_m<0, true, true>(a, precise, st);
    else if (mode == 0) launch_instance_m<0, true, false>(a, precise, st);
    else if (mode == 1) launch_instance_m<1, true, false>(a, precise, st);
    else if (rigid) launch_instance_m<2, true, false>(a, precise, st);
    else launch_instance_m<2, false, false>(a, precise, st);
    return hipGetLastError();
}

hipError_t launch_pose_rows(const double* E1, const double* E2, const double* phi1, const double* phi2, const double* kn,
                            const double* kt, double* rows, int32_t* done, int32_t call, int n, hipStream_t st) {
    hipLaunchKernelGGL(pose_rows_kernel, dim3(n), dim3(64), 0, st, E1, E2, phi1, phi2, kn, kt, rows, done, call);
    return hipGetLastError();
}

hipError_t launch_pose_gradients(const double* E1, const double* g1, double* gE1, const double* E2, const double* g2,
                                 double* gE2, int32_t* done, int32_t call, int n, hipStream_t st) {
    hipLaunchKernelGGL(pose_gradients_kernel, dim3((n + 31) / 32), dim3(64), 0, st, E1, g1, gE1, E2, g2, gE2, done, call, n);
    return hipGetLastError();
}

hipError_t launch_upload(const InstDev* src, InstDev* dst, int n, const int32_t* call, int32_t* counters, hipStream_t st) {
    static_assert(sizeof(InstDev) % sizeof(uint4) == 0, "copied 16 bytes at a time");
    if (n <= 0) return hipSuccess;
    const int64_t words = (int64_t)n * (sizeof(InstDev) / sizeof(uint4));
    hipLaunchKernelGGL(upload_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st,
                       reinterpret_cast<const uint4*>(src), reinterpret_cast<uint4*>(dst), words, call, counters);
    return hipGetLastError();
}

hipError_t launch_reset(int32_t* c, int n, hipStream_t st) {
    hipLaunchKernelGGL(reset_counters_kernel, dim3((n + 63) / 64), dim3(64), 0, st, c, n);
    return hipGetLastError();
}

hipError_t launch_zero(void* p, int64_t n_words, hipStream_t st) {
    if (n_words <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((n_words + 255) / 256, 4096);
    hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)blocks), dim3(256), 0, st, (uint32_t*)p, n_words);
    return hipGetLastError();
}

hipError_t launch_plain(const PlainArgs& a, int64_t n_points, bool precise, hipStream_t st) {
    if (n_points <= 0) return hipSuccess;
    const int64_t blocks = (n_points + 255) / 256;
    if (precise) hipLaunchKernelGGL(plain_kernel<double>, dim3((unsigned)blocks), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(plain_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_distance(const PointArgs& a, hipStream_t st) {
    if (a.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(distance_kernel, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, st, a);
    return hipGetLastError();
}

template <bool DERIV>
static void launch_collision_t(const PointArgs& a, bool precise, hipStream_t st) {
    const dim3 grid((unsigned)((a.n + kCollPoints - 1) / kCollPoints));
    if (precise) hipLaunchKernelGGL((collision_kernel<DERIV, double>), grid, dim3(64), 0, st, a);
    else hipLaunchKernelGGL((collision_kernel<DERIV, float>), grid, dim3(64), 0, st, a);
}

hipError_t launch_collision(const PointArgs& a, bool precise, hipStream_t st) {
    if (a.n <= 0) return hipSuccess;
    if (a.out2) launch_collision_t<true>(a, precise, st);
    else launch_collision_t<false>(a, precise, st);
    return hipGetLastError();
}

hipError_t launch_touched(const TouchedArgs& a, int n_inst, hipStream_t st) {
    if (n_inst <= 0) return hipSuccess;
    hipLaunchKernelGGL(touched_kernel, dim3(64, n_inst), dim3(256), 0, st, a);
    return hipGetLastError();
}

hipError_t launch_popcount(const uint32_t* bits, int64_t nwords, unsigned long long* out, hipStream_t st) {
    hipLaunchKernelGGL(popcount_kernel, dim3(256), dim3(256), 0, st, bits, nwords, out);
    return hipGetLastError();
}

}  // namespace atac
