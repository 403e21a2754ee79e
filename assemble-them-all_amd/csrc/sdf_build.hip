// Mesh -> signed distance grid on the GPU: the level-set construction of
// sdfgen::make_level_set3 (simulation/externals/sdfgen/makelevelset3.cpp:163-230),
// node for node the same values.
//
// * Band: one wavefront per triangle; lanes over the nodes of its index box
//   widened by the exact band. A node keeps the smallest (distance, triangle)
//   pair (one 64-bit atomic min on distance bits << 32 | triangle): the
//   sequential loop keeps the first triangle reaching the minimum, the lowest
//   index among equal distances, and so does the min. Crossings of the x-rays
//   through the node lines (j, k) with the triangle are counted with atomics.
// * Fast sweeping: within one of the 16 directional sweeps a node reads only its
//   7 neighbours one step back along the sweep axes. One launch runs a sweep:
//   workgroups march along x over tiles of columns, skewed so that each lane's
//   neighbours are one to three steps behind it (ls_sweep_kernel); every node
//   sees its neighbours' values of this sweep, as in the sequential sweep.
// * Signs: one wavefront per x line, parity of the crossings so far.
// FMA contraction is off in this file: every float operation rounds as written.
#pragma clang fp contract(off)

#include "sdf_build.h"
#include "levelset.h"

namespace atac {

using ls::F3;

__device__ __forceinline__ F3 vertex(const float* x, uint32_t v) {
    return ls::f3(x[3 * (int64_t)v], x[3 * (int64_t)v + 1], x[3 * (int64_t)v + 2]);
}
__device__ __forceinline__ F3 grid_node(const LsArgs& a, int i, int j, int k) {
    return ls::f3((float)i * a.dx + a.o[0], (float)j * a.dy + a.o[1], (float)k * a.dz + a.o[2]);
}
__device__ __forceinline__ int64_t node_id(const LsArgs& a, int i, int j, int k) {
    return i + (int64_t)a.ni * (j + (int64_t)a.nj * k);
}

__global__ __launch_bounds__(256) void ls_band_kernel(LsArgs a) {
    const int lane = (int)threadIdx.x & 63;
    const int64_t nw = (int64_t)gridDim.x * 4;
    for (int64_t t = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); t < a.nf;
         t += nw) {
        const uint32_t p = a.tri[3 * t], q = a.tri[3 * t + 1], r = a.tri[3 * t + 2];
        const F3 xp = vertex(a.x, p), xq = vertex(a.x, q), xr = vertex(a.x, r);
        // grid coordinates in double
        const double fip = ((double)xp.x - (double)a.o[0]) / (double)a.dx;
        const double fjp = ((double)xp.y - (double)a.o[1]) / (double)a.dy;
        const double fkp = ((double)xp.z - (double)a.o[2]) / (double)a.dz;
        const double fiq = ((double)xq.x - (double)a.o[0]) / (double)a.dx;
        const double fjq = ((double)xq.y - (double)a.o[1]) / (double)a.dy;
        const double fkq = ((double)xq.z - (double)a.o[2]) / (double)a.dz;
        const double fir = ((double)xr.x - (double)a.o[0]) / (double)a.dx;
        const double fjr = ((double)xr.y - (double)a.o[1]) / (double)a.dy;
        const double fkr = ((double)xr.z - (double)a.o[2]) / (double)a.dz;
        const double mi = ls::lmin(fip, ls::lmin(fiq, fir)), Mi = ls::lmax(fip, ls::lmax(fiq, fir));
        const double mj = ls::lmin(fjp, ls::lmin(fjq, fjr)), Mj = ls::lmax(fjp, ls::lmax(fjq, fjr));
        const double mk = ls::lmin(fkp, ls::lmin(fkq, fkr)), Mk = ls::lmax(fkp, ls::lmax(fkq, fkr));
        // distances over the index box widened by the band
        const int i0 = ls::lclamp((int)mi - a.band, 0, a.ni - 1), i1 = ls::lclamp((int)Mi + a.band + 1, 0, a.ni - 1);
        const int j0 = ls::lclamp((int)mj - a.band, 0, a.nj - 1), j1 = ls::lclamp((int)Mj + a.band + 1, 0, a.nj - 1);
        const int k0 = ls::lclamp((int)mk - a.band, 0, a.nk - 1), k1 = ls::lclamp((int)Mk + a.band + 1, 0, a.nk - 1);
        const int nI = i1 - i0 + 1, nJ = j1 - j0 + 1;
        const int64_t tot = (int64_t)nI * nJ * (k1 - k0 + 1);
        for (int64_t e = lane; e < tot; e += 64) {
            const int i = i0 + (int)(e % nI), j = j0 + (int)((e / nI) % nJ), k = k0 + (int)(e / ((int64_t)nI * nJ));
            const float d = ls::tri_dist(grid_node(a, i, j, k), xp, xq, xr);
            if (d < a.phi0)
                atomicMin(a.best + node_id(a, i, j, k), ((unsigned long long)__float_as_uint(d) << 32) | (uint32_t)t);
        }
        // crossings of the x-rays through the node lines (j, k) the triangle spans
        const int cj0 = ls::lclamp((int)ceil(mj), 0, a.nj - 1), cj1 = ls::lclamp((int)floor(Mj), 0, a.nj - 1);
        const int ck0 = ls::lclamp((int)ceil(mk), 0, a.nk - 1), ck1 = ls::lclamp((int)floor(Mk), 0, a.nk - 1);
        if (cj0 > cj1 || ck0 > ck1) continue;
        const int nJ2 = cj1 - cj0 + 1;
        const int64_t tot2 = (int64_t)nJ2 * (ck1 - ck0 + 1);
        for (int64_t e = lane; e < tot2; e += 64) {
            const int j = cj0 + (int)(e % nJ2), k = ck0 + (int)(e / nJ2);
            double ba, bb, bc;
            if (!ls::in_triangle_2d((double)j, (double)k, fjp, fkp, fjq, fkq, fjr, fkr, ba, bb, bc)) continue;
            const double fi = ba * fip + bb * fiq + bc * fir;
            const int ii = (int)ceil(fi);   // the crossing lies in (ii - 1, ii]
            if (ii < 0) atomicAdd(a.count + node_id(a, 0, j, k), 1);
            else if (ii < a.ni) atomicAdd(a.count + node_id(a, ii, j, k), 1);
        }
    }
}

// A node's word during the sweeps: its closest triangle + 1 (0: none) and, in the
// last 5 bits, the sweep that found it (0: the band; sweep s: s + 1). Meshes with
// 2^27 triangles or more keep no sweep number.
constexpr int kLsStampShift = 27;
constexpr uint32_t kLsIdMask = (1u << kLsStampShift) - 1u;
__host__ __device__ __forceinline__ bool ls_stamped(int64_t nf) { return nf < (int64_t)kLsIdMask; }

__global__ void ls_unpack_kernel(LsArgs a, int64_t n) {
    const int64_t t0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
    for (int64_t e = t0; e < n; e += step) {
        const unsigned long long b = a.best[e];
        const bool none = b == ~0ull;
        a.phi[e] = none ? a.phi0 : __uint_as_float((uint32_t)(b >> 32));
        a.best[e] = none ? 0ull : (b & 0xffffffffull) + 1ull;   // tag 0
    }
    for (int64_t t = t0; t < a.nf; t += step)
        a.tris[t] = ls::make_tri(vertex(a.x, a.tri[3 * t]), vertex(a.x, a.tri[3 * t + 1]), vertex(a.x, a.tri[3 * t + 2]));
    if (t0 < kLsSync) a.sync[t0] = 0;
}

struct LsSweep {
    int32_t d[3];        // the sweep's direction per axis, +1 or -1
    int32_t index;       // 0 .. 15
    int32_t last[7];     // per neighbour (in the order of the tests): 1 + the last sweep that tested it, -1 if none
    int32_t tiles_j, tiles_k;
    int32_t marked;      // ls_mark_kernel has run: only marked nodes have tests of their own
};

// The state word's upper half: the number (tag) of the sweep that stored it, and the mark.
constexpr uint32_t kLsMark = 0x80000000u;

// Which of a node's neighbours it has tested (bit e): the neighbour's triangle is
// older than the sweep that last compared the two. A node on a face of the grid is
// left out by half of the sweeps, so there nothing counts as tested (`known` 0).
// Branch-free vector arithmetic, here and in ls_tests: with one wavefront per SIMD
// a compare, mask and branch cost several times a vector instruction.
__device__ __forceinline__ uint32_t ls_tested(const LsSweep& s, const uint32_t (&n)[7], uint32_t known) {
    uint32_t t = 0;
#pragma unroll
    for (int e = 0; e < 7; ++e)
        t |= (((n[e] >> kLsStampShift) - (uint32_t)(s.last[e] + 1)) >> 31) << e;   // stamp <= last
    return known ? t : 0u;
}

// The tests left of `todo` (bit per neighbour) when no triangle is tested twice and
// none that a tested neighbour has too, or that is the node's own, or none.
__device__ __forceinline__ uint32_t ls_tests(const uint32_t (&id)[7], uint32_t own, uint32_t todo, uint32_t tested) {
    uint32_t keep[7];
#pragma unroll
    for (int e = 0; e < 7; ++e) keep[e] = min(min(id[e], id[e] ^ own), (todo >> e) & 1u);
#pragma unroll
    for (int e = 1; e < 7; ++e) {
        const uint32_t open = ((tested >> e) & 1u) ^ 1u;
#pragma unroll
        for (int f = 0; f < e; ++f) {
            const uint32_t differ = id[e] ^ id[f];
            keep[e] = min(keep[e], differ);
            keep[f] = min(keep[f], differ | open);
        }
    }
    uint32_t m = 0;
#pragma unroll
    for (int e = 0; e < 7; ++e) m |= keep[e] << e;
    return m;
}

// Marks the nodes that a neighbour's triangle, as it stands before the sweep, would
// bring nearer. The tests of the others come out the same during the sweep (a node's
// distance only shrinks), so there they need testing only against triangles that the
// sweep itself has moved: after the first sweeps that leaves a few nodes in a hundred,
// then in a thousand. All nodes at once: 10 to 50 us for 96 x 96 x 96 nodes.
__global__ __launch_bounds__(256) void ls_mark_kernel(LsArgs a, LsSweep s, int64_t n) {
    const int64_t e0 = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e0 >= n) return;
    const int i = (int)(e0 % a.ni), j = (int)((e0 / a.ni) % a.nj), k = (int)(e0 / ((int64_t)a.ni * a.nj));
    const int x = i - s.d[0], y = j - s.d[1], z = k - s.d[2];
    if (x < 0 || x >= a.ni || y < 0 || y >= a.nj || z < 0 || z >= a.nk) return;   // the face the sweep starts from
    auto word = [&](int p, int q, int r) { return (uint32_t)a.best[node_id(a, p, q, r)]; };
    const uint32_t w[7] = {word(x, j, k), word(i, y, k), word(x, y, k), word(i, j, z), word(x, j, z), word(i, y, z), word(x, y, z)};
    const unsigned long long old = a.best[e0];
    uint32_t id[7];
#pragma unroll
    for (int e = 0; e < 7; ++e) id[e] = w[e] & kLsIdMask;
    const uint32_t known = (i > 0) & (i < a.ni - 1) & (j > 0) & (j < a.nj - 1) & (k > 0) & (k < a.nk - 1);
    const uint32_t tested = ls_tested(s, w, known);
    uint32_t todo = ls_tests(id, (uint32_t)old & kLsIdMask, ~tested & 0x7fu, tested);
    const float p = a.phi[e0];
    const F3 gx = grid_node(a, i, j, k);
    bool nearer = false;
    while (todo && !nearer) {
        uint32_t t = id[6];
#pragma unroll
        for (int e = 5; e >= 0; --e) t = (todo >> e) & 1u ? id[e] : t;
        todo &= todo - 1u;
        nearer = ls::tri_dist_below(gx, a.tris[t - 1u], p) < p;
    }
    const uint32_t hi = (uint32_t)(old >> 32), want = (hi & ~kLsMark) | (nearer ? kLsMark : 0u);
    if (hi != want) a.best[e0] = ((unsigned long long)want << 32) | (uint32_t)old;
}

constexpr int kLsSide = 16;           // a tile's lanes per axis
constexpr int kLsTile = kLsSide - 1;  // its columns per axis
constexpr int kLsLanes = kLsSide * kLsSide;
constexpr int kLsChunk = 4;           // steps whose values are read and written together
constexpr int kLsRing = 2 * kLsChunk;
constexpr int kLsSpins = 1 << 22;     // polls (about 1 us each) before a wait is given up

// One sweep. A workgroup of 4 wavefronts takes a tile of 15 x 15 columns (along x)
// and, on the lanes of its low j and k sides, the neighbouring tiles' columns: lane
// (b, c) holds column sb = 15 J - 1 + b, sc = 15 K - 1 + c in steps from the sweep's
// corner, and at step q stands at node sa = q - b - c - 1 of it. The neighbours a node
// tests are then nodes the lanes (b, c), (b-1, c), (b, c-1), (b-1, c-1) stood at one to
// three steps ago: their words are in LDS, with one barrier per step and no launch
// per plane. The side lanes only pass on what their columns' own tile stores: a node's
// state word carries the sweep's number in its upper half (one 8-byte store, device
// scope), so a reader that finds another number reads again. Tiles are taken in
// ascending order from a counter; a tile waits only for tiles taken before it, which
// are running or done, so every wait ends (kLsSpins bounds it all the same). The layer
// sa = -1 (and columns sb = -1, sc = -1) is the grid's face, which no sweep updates.
//
// What a node tests: a neighbour's triangle is skipped when it is the node's own, or
// another neighbour's already in the list, or tested before (ls_tested), or, on an
// unmarked node (ls_mark_kernel), when this sweep has not moved it. None of these can
// be nearer than the node's distance, so the result is that of testing all seven. A
// wavefront's tests are dealt out over its lanes through LDS (their number varies from
// node to node), and each node takes its distances in the neighbours' order. A chunk
// of steps without marked nodes or moved triangles passes its words on untouched.
//
// Bound by the chain of dependent steps: (ni + nj + nk) nodes per sweep at the least,
// with the waits for the tiles before. Loads and stores therefore wait once per
// kLsChunk steps (the next chunk's values are read, and the last one's written, at its
// start: the memory counter is in order, so a load's wait would wait for the stores
// before it at every step). For about 99^3 nodes and 12,288 triangles: one launch per
// diagonal plane took 10.9 us a plane (4,672 planes, 51.0 ms for the whole build); this
// kernel 1.6 ms in the first sweeps and 0.5 ms in the last (14.8 ms in all). Tiles of
// 7 x 7 columns on one wavefront (no barrier, but twice the tiles to cross) 17.7 ms,
// chunks of 8 steps 16.3 ms, without the marks 17.7 ms.
__global__ __launch_bounds__(kLsLanes) void ls_sweep_kernel(LsArgs a, LsSweep s) {
    __shared__ uint32_t s_word[kLsRing][kLsLanes];    // the last steps' words, this chunk's still to come as loaded
    __shared__ float s_ph[kLsChunk][kLsLanes];
    __shared__ uint2 s_test[4][7 * 64];               // per wavefront: a step's tests, lane | neighbour << 8, triangle
    __shared__ float s_dist[7][kLsLanes];             // and their distances
    __shared__ int s_ticket;
    const int tid = (int)threadIdx.x, b = tid % kLsSide, c = tid / kLsSide, lane = tid & 63, wv = tid >> 6;
    const int A = a.ni - 1, B = a.nj - 1, C = a.nk - 1;
    if (tid == 0) s_ticket = atomicAdd(a.sync + s.index, 1);
    __syncthreads();
    const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    const int J = ticket % s.tiles_j, K = ticket / s.tiles_j;
    const int sb0 = kLsTile * J - 1, sc0 = kLsTile * K - 1, sb = sb0 + b, sc = sc0 + c;
    const bool column = sb < B && sc < C;                       // in the grid
    const bool mine = column && b > 0 && c > 0;                 // updated here
    const bool foreign = column && !mine && sb >= 0 && sc >= 0;   // updated by an earlier tile
    auto x_of = [&](int sa) { return s.d[0] > 0 ? 1 + sa : a.ni - 2 - sa; };
    auto y_of = [&](int t) { return s.d[1] > 0 ? 1 + t : a.nj - 2 - t; };
    auto z_of = [&](int t) { return s.d[2] > 0 ? 1 + t : a.nk - 2 - t; };
    const int j = y_of(sb), k = z_of(sc);
    const int64_t row = column ? node_id(a, 0, j, k) : 0;
    const bool stamped = ls_stamped(a.nf);
    const bool inner_column = stamped && j > 0 && j < a.nj - 1 && k > 0 && k < a.nk - 1;
    const uint32_t id_mask = stamped ? kLsIdMask : 0xffffffffu;
    const uint32_t tag = (uint32_t)s.index + 1u, stamp = stamped ? tag << kLsStampShift : 0u;
    const bool shared = b == kLsTile || c == kLsTile;           // a later tile reads this column
    // the lanes (b-1, c), (b, c-1), (b-1, c-1); lanes without one read themselves and do not use it
    const int t01 = b ? tid - 1 : tid, t10 = c ? tid - kLsSide : tid, t11 = b && c ? tid - kLsSide - 1 : tid;
    auto sync_wave = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto poll = [&](int sa) {
        return __hip_atomic_load(a.best + row + x_of(sa), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto tag_of = [](unsigned long long w) { return (uint32_t)(w >> 32) & ~kLsMark; };
    unsigned long long nw[kLsChunk];   // the next chunk's state words and distances
    float np[kLsChunk];
    auto fetch = [&](int q0) {
#pragma unroll
        for (int u = 0; u < kLsChunk; ++u) {
            const int sa = q0 + u - b - c - 1;
            nw[u] = 0ull;
            np[u] = 0.0f;
            if (column && sa >= -1 && sa < A) {
                if (foreign) {
                    nw[u] = poll(sa);
                } else {
                    nw[u] = a.best[row + x_of(sa)];
                    if (mine) np[u] = a.phi[row + x_of(sa)];
                }
            }
        }
    };
    unsigned changed = 0;              // this chunk's steps that changed the lane's node
    const int steps = A + 1 + 2 * kLsTile;   // sa from -1 on lane (0, 0) to A - 1 on lane (15, 15)
    // a chunk's results, from LDS
    auto store = [&](int q0) {
#pragma unroll
        for (int u = 0; u < kLsChunk; ++u) {
            const int sa = q0 + u - b - c - 1;
            if (mine && sa >= 0 && sa < A) {
                const uint32_t w = s_word[(q0 + u) % kLsRing][tid];
                const bool ch = (changed >> u) & 1u;
                if (ch) a.phi[row + x_of(sa)] = s_ph[u][tid];
                if (shared)
                    __hip_atomic_store(a.best + row + x_of(sa), ((unsigned long long)tag << 32) | w, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                else if (ch) a.best[row + x_of(sa)] = w;
            }
        }
    };
#pragma unroll
    for (int u = 0; u < kLsRing; ++u) s_word[u][tid] = 0u;
    fetch(0);
    bool gave_up = false;
    for (int q0 = 0; q0 < steps; q0 += kLsChunk) {
        // the chunk's values; first those that still lack this sweep's number
        unsigned late = 0;
#pragma unroll
        for (int u = 0; u < kLsChunk; ++u) {
            const int sa = q0 + u - b - c - 1;
            if (foreign && sa >= 0 && sa < A && tag_of(nw[u]) != tag) late |= 1u << u;
        }
        if (q0 > 0) store(q0 - kLsChunk);
        for (int spins = 0; __any(late != 0u && !gave_up);) {
#pragma unroll
            for (int u = 0; u < kLsChunk; ++u)
                if ((late >> u) & 1u) nw[u] = poll(q0 + u - b - c - 1);
#pragma unroll
            for (int u = 0; u < kLsChunk; ++u)
                if (tag_of(nw[u]) == tag) late &= ~(1u << u);
            if (++spins >= kLsSpins) {
                gave_up = true;
                if (lane == 0) atomicOr(a.sync + kLsGaveUp, 1);
            }
        }
        // can anything move? a marked node, or a triangle this sweep has moved, here or
        // among the last steps' words
        unsigned marks = 0;
        uint32_t moved = 0;
#pragma unroll
        for (int u = 0; u < kLsChunk; ++u) {
            const int sa = q0 + u - b - c - 1;
            const uint32_t w = (uint32_t)nw[u];
            if (mine && sa >= 0 && sa < A) {
                if (!s.marked || ((uint32_t)(nw[u] >> 32) & kLsMark)) marks |= 1u << u;
            } else {
                moved |= (w >> kLsStampShift) == tag ? 1u : 0u;
            }
            s_word[(q0 + u) % kLsRing][tid] = w;
            s_ph[u][tid] = np[u];
        }
#pragma unroll
        for (int u = 1; u <= 3; ++u)
            moved |= (s_word[(q0 + kLsRing - u) % kLsRing][tid] >> kLsStampShift) == tag ? 1u : 0u;
        const bool any = __syncthreads_or((marks != 0u) | (moved != 0u) | !stamped) != 0;
        fetch(q0 + kLsChunk);
        changed = 0;
        if (!any) continue;
#pragma unroll 1
        for (int u = 0; u < kLsChunk; ++u) {
            const int q = q0 + u, sa = q - b - c - 1;
            const int r0 = q % kLsRing, r1 = (q + kLsRing - 1) % kLsRing, r2 = (q + kLsRing - 2) % kLsRing,
                      r3 = (q + kLsRing - 3) % kLsRing;
            const uint32_t n4 = s_word[r2][t10], n2 = s_word[r2][t01], n5 = s_word[r2][t11], n6 = s_word[r3][t11];
            uint32_t own = s_word[r0][tid];
            float p = s_ph[u][tid];
            if (u > 0) __syncthreads();   // the last step's words
            // (i-1, j, k), (i, j-1, k), (i-1, j-1, k), (i, j, k-1), (i-1, j, k-1), (i, j-1, k-1), (i-1, j-1, k-1)
            const uint32_t n[7] = {s_word[r1][tid], s_word[r1][t01], n2, s_word[r1][t10], n4, n5, n6};
            // nothing to test unless the node is marked or a neighbour is this sweep's (words
            // that differ from its stamp only below it)
            uint32_t least = n[0] ^ stamp;
#pragma unroll
            for (int e = 1; e < 7; ++e) least = min(least, n[e] ^ stamp);
            const bool live = mine & (sa >= 0) & (sa < A);
            const bool marked = ((marks >> u) & 1u) != 0u;
            if (!__any(live & (marked | (least <= kLsIdMask) | !stamped))) continue;
            const int i = x_of(sa);
            const uint32_t known = inner_column & (i > 0) & (i < a.ni - 1);
            uint32_t id[7], fresh = 0;   // fresh: this sweep's
#pragma unroll
            for (int e = 0; e < 7; ++e) {
                id[e] = n[e] & id_mask;
                fresh |= ((((n[e] ^ stamp) >> kLsStampShift) - 1u) >> 31) << e;
            }
            const uint32_t tested = ls_tested(s, n, known);
            const uint32_t untested = stamped ? (marked ? ~tested : fresh) : ~0u;
            const uint32_t todo = ls_tests(id, own & id_mask, live ? untested & 0x7fu : 0u, tested);
            if (__any(todo != 0u)) {
                // the wavefront's tests in one list, dealt out 64 at a time
                int total = 0;
#pragma unroll
                for (int e = 0; e < 7; ++e) {
                    const bool mark = ((todo >> e) & 1u) != 0u;
                    const uint64_t m = __ballot(mark);
                    if (mark) {
                        const int at = total + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                              __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
                        s_test[wv][at] = make_uint2((uint32_t)tid | ((uint32_t)e << 8), id[e]);
                    }
                    total += __popcll(m);
                }
                sync_wave();
                for (int t = lane; t < total; t += 64) {
                    const uint2 w = s_test[wv][t];
                    const int l = (int)(w.x & 255u), lb = l % kLsSide, lc = l / kLsSide;
                    s_dist[w.x >> 8][l] = ls::tri_dist_below(grid_node(a, x_of(q - lb - lc - 1), y_of(sb0 + lb), z_of(sc0 + lc)),
                                                             a.tris[w.y - 1u], s_ph[u][l]);
                }
                sync_wave();
#pragma unroll
                for (int e = 0; e < 7; ++e) {
                    const float d = s_dist[e][tid];   // stale where nothing was tested
                    const bool nearer = (((todo >> e) & 1u) != 0u) & (d < p);
                    p = nearer ? d : p;
                    own = nearer ? id[e] | stamp : own;
                    changed |= nearer ? 1u << u : 0u;
                }
                sync_wave();
                s_word[r0][tid] = own;
                s_ph[u][tid] = p;
            }
        }
    }
    store((steps - 1) / kLsChunk * kLsChunk);
}

// One wavefront per x line: the parity of the crossings up to each node.
__global__ __launch_bounds__(256) void ls_sign_kernel(LsArgs a) {
    const int lane = (int)threadIdx.x & 63;
    const int64_t lines = (int64_t)a.nj * a.nk, step = (int64_t)gridDim.x * 4;
    for (int64_t line = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); line < lines; line += step) {
        const int64_t row = line * a.ni;
        unsigned odd = 0;
        for (int i0 = 0; i0 < a.ni; i0 += 64) {
            const int i = i0 + lane;
            const uint64_t m = __ballot(i < a.ni && (a.count[row + (i < a.ni ? i : 0)] & 1));
            const unsigned here = odd + (unsigned)__popcll(m & (~0ull >> (63 - lane)));
            if (i < a.ni && (here & 1u)) a.phi[row + i] = -a.phi[row + i];
            odd += (unsigned)__popcll(m);
        }
    }
}

hipError_t ls_build(const LsArgs& a, hipStream_t st) {
    const int64_t n = (int64_t)a.ni * a.nj * a.nk;
    if (a.nf > 0) {
        const int64_t blocks = std::min<int64_t>((a.nf + 3) / 4, 65536);
        hipLaunchKernelGGL(ls_band_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(ls_unpack_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 65536)), dim3(256), 0, st, a, n);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int A = a.ni - 1, B = a.nj - 1, C = a.nk - 1;
    if (A > 0 && B > 0 && C > 0) {
        static const int dirs[8][3] = {{+1, +1, +1}, {-1, -1, -1}, {+1, +1, -1}, {-1, -1, +1},
                                       {+1, -1, +1}, {-1, +1, -1}, {+1, -1, -1}, {-1, +1, +1}};
        // the axes a test steps back along, in the order of the tests
        static const int back[7][3] = {{1, 0, 0}, {0, 1, 0}, {1, 1, 0}, {0, 0, 1}, {1, 0, 1}, {0, 1, 1}, {1, 1, 1}};
        for (int p = 0; p < kLsSweeps; ++p) {
            LsSweep s{};
            for (int x = 0; x < 3; ++x) s.d[x] = dirs[p % 8][x];
            s.index = p;
            for (int t = 0; t < 7; ++t) {
                s.last[t] = -1;
                for (int q = 0; q < p; ++q) {   // the last sweep that stepped back the same way
                    bool same = true;
                    for (int x = 0; x < 3; ++x) same = same && (!back[t][x] || dirs[q % 8][x] == s.d[x]);
                    if (same) s.last[t] = q + 1;
                }
            }
            s.tiles_j = (B + kLsTile - 1) / kLsTile;
            s.tiles_k = (C + kLsTile - 1) / kLsTile;
            // the first two sweeps move nearly every node
            s.marked = ls_stamped(a.nf) && p >= 2;
            if (s.marked) {
                hipLaunchKernelGGL(ls_mark_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, s, n);
                e = hipGetLastError();
                if (e != hipSuccess) return e;
            }
            hipLaunchKernelGGL(ls_sweep_kernel, dim3((unsigned)((int64_t)s.tiles_j * s.tiles_k)), dim3(kLsLanes), 0, st, a, s);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    const int64_t blocks = std::min<int64_t>(((int64_t)a.nj * a.nk + 3) / 4, 65536);
    hipLaunchKernelGGL(ls_sign_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
    return hipGetLastError();
}

}  // namespace atac
