// BVH contact variant: mesh preprocessing on the host, signed-distance and force
// kernels on the GPU (the sampler is bvh.h; the contact math is contact_math.h's,
// with the pseudonormal as gradient and a zero Hessian, BodyBVHObj.cpp:453-566).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <numeric>
#include <utility>
#include "atac.h"
#include "bvh_host.h"
#include "wave_ops.h"

namespace atac {

// ------------------------------------------------------------------ preprocessing
namespace {

struct V3d {
    double x, y, z;
};
V3d vrow(const std::vector<double>& a, int64_t i) { return V3d{a[3 * i], a[3 * i + 1], a[3 * i + 2]}; }
V3d vsub(V3d a, V3d b) { return V3d{a.x - b.x, a.y - b.y, a.z - b.z}; }
V3d vcross(V3d a, V3d b) { return V3d{a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x}; }
double vdot(V3d a, V3d b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
void add_row(std::vector<double>& a, int64_t i, V3d v, double w) {
    a[3 * i] += w * v.x; a[3 * i + 1] += w * v.y; a[3 * i + 2] += w * v.z;
}
void normalize_rows(std::vector<double>& a) {
    for (size_t i = 0; i + 2 < a.size(); i += 3) {
        const double r = std::sqrt(a[i] * a[i] + a[i + 1] * a[i + 1] + a[i + 2] * a[i + 2]);
        if (r > 0.0) { a[i] /= r; a[i + 1] /= r; a[i + 2] /= r; }
    }
}

// Median splits along the longest axis of the centroids, three levels to a node,
// at multiples of the leaf size: every leaf but the last holds kBvhWidth triangles.
struct Builder {
    const MeshHost& m;
    std::vector<double> cen;      // centroids, nf x 3
    std::vector<int32_t> idx;     // faces in leaf order
    std::vector<float4> nodes;
    explicit Builder(const MeshHost& mh) : m(mh) {}

    void box_of(int32_t b, int32_t e, float4& lo, float4& hi) const {
        double l[3] = {INFINITY, INFINITY, INFINITY}, h[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int32_t k = b; k < e; ++k)
            for (int c = 0; c < 3; ++c) {
                const int32_t v = m.F[3 * (int64_t)idx[k] + c];
                for (int a = 0; a < 3; ++a) {
                    l[a] = std::min(l[a], m.V[3 * (int64_t)v + a]);
                    h[a] = std::max(h[a], m.V[3 * (int64_t)v + a]);
                }
            }
        lo = make_float4(f32_down(l[0]), f32_down(l[1]), f32_down(l[2]), 0.0f);
        hi = make_float4(f32_up(h[0]), f32_up(h[1]), f32_up(h[2]), 0.0f);
    }
    static float bits(int v) { float f; std::memcpy(&f, &v, sizeof f); return f; }
    static int32_t leaves(int32_t b, int32_t e) { return (e - b + kBvhWidth - 1) / kBvhWidth; }

    // Faces idx[b, e) into at most 2^levels ranges of whole leaves.
    void split(int32_t b, int32_t e, int levels, std::vector<std::pair<int32_t, int32_t>>& out) {
        const int32_t n = leaves(b, e);
        if (levels == 0 || n <= 1) { out.push_back({b, e}); return; }
        double cl[3] = {INFINITY, INFINITY, INFINITY}, ch[3] = {-INFINITY, -INFINITY, -INFINITY};
        for (int32_t k = b; k < e; ++k)
            for (int a = 0; a < 3; ++a) {
                cl[a] = std::min(cl[a], cen[3 * (int64_t)idx[k] + a]);
                ch[a] = std::max(ch[a], cen[3 * (int64_t)idx[k] + a]);
            }
        int ax = 0;
        for (int a = 1; a < 3; ++a)
            if (ch[a] - cl[a] > ch[ax] - cl[ax]) ax = a;
        const int32_t mid = b + kBvhWidth * (n / 2);
        std::nth_element(idx.begin() + b, idx.begin() + mid, idx.begin() + e, [&](int32_t p, int32_t q) {
            const double cp = cen[3 * (int64_t)p + ax], cq = cen[3 * (int64_t)q + ax];
            return cp < cq || (cp == cq && p < q);
        });
        split(b, mid, levels - 1, out);
        split(mid, e, levels - 1, out);
    }

    // Appends the node over faces idx[b, e) and, behind it, its children; returns its first entry.
    int32_t build(int32_t b, int32_t e) {
        std::vector<std::pair<int32_t, int32_t>> kids;
        split(b, e, 3, kids);
        const int32_t first = (int32_t)(nodes.size() / 2);
        for (int c = 0; c < kBvhWidth; ++c) {
            nodes.push_back(make_float4(INFINITY, INFINITY, INFINITY, bits(kBvhEmpty)));
            nodes.push_back(make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f));
        }
        for (size_t c = 0; c < kids.size(); ++c) {
            const int32_t kb = kids[c].first, ke = kids[c].second;
            float4 lo, hi;
            box_of(kb, ke, lo, hi);
            lo.w = bits(ke - kb <= kBvhWidth ? -(kb / kBvhWidth) - 1 : build(kb, ke));
            nodes[2 * (first + (int32_t)c)] = lo;
            nodes[2 * (first + (int32_t)c) + 1] = hi;
        }
        return first;
    }
};

}  // namespace

std::string mesh_build(const double* V, int64_t nv, const int64_t* F, int64_t nf, MeshHost& m) {
    if (!V || !F || nv < 3 || nf < 1) return "a mesh needs at least 3 vertices and 1 triangle";
    if (nf >= (int64_t)1 << 30 || nv >= (int64_t)1 << 31) return "mesh too large";
    m.V.assign(V, V + 3 * nv);
    for (int64_t i = 0; i < 3 * nv; ++i)
        if (!std::isfinite(V[i])) return "vertex coordinates must be finite";
    m.F.resize(3 * nf);
    for (int64_t i = 0; i < 3 * nf; ++i) {
        if (F[i] < 0 || F[i] >= nv) return "triangle vertex index out of range";
        m.F[i] = (int32_t)F[i];
    }
    for (int a = 0; a < 3; ++a) { m.bmin[a] = INFINITY; m.bmax[a] = -INFINITY; }
    for (int64_t v = 0; v < nv; ++v)
        for (int a = 0; a < 3; ++a) {
            m.bmin[a] = std::min(m.bmin[a], V[3 * v + a]);
            m.bmax[a] = std::max(m.bmax[a], V[3 * v + a]);
        }
    // face normals: (v1 - v0) x (v2 - v0), normalised; a face is degenerate when
    // |ab x ac|^2 <= 1e-20 |ab|^2 |ac|^2 (zero area to rounding), and its normal is zero
    m.FN.assign(3 * nf, 0.0);
    std::vector<char> degenerate(nf, 0);
    for (int64_t f = 0; f < nf; ++f) {
        const V3d a = vrow(m.V, m.F[3 * f]), b = vrow(m.V, m.F[3 * f + 1]), c = vrow(m.V, m.F[3 * f + 2]);
        const V3d ab = vsub(b, a), ac = vsub(c, a), n = vcross(ab, ac);
        degenerate[f] = vdot(n, n) <= 1e-20 * vdot(ab, ab) * vdot(ac, ac);
        if (!degenerate[f]) add_row(m.FN, f, n, 1.0);
    }
    normalize_rows(m.FN);
    // edges: the edge opposite corner c of face f is (F[f][c+1], F[f][c+2]); its
    // normal is the normalised sum of the normals of the faces that hold it
    std::map<std::pair<int32_t, int32_t>, int32_t> edge_id;
    m.FE.resize(3 * nf);
    for (int64_t f = 0; f < nf; ++f)
        for (int c = 0; c < 3; ++c) {
            int32_t u = m.F[3 * f + (c + 1) % 3], w = m.F[3 * f + (c + 2) % 3];
            if (u > w) std::swap(u, w);
            auto it = edge_id.emplace(std::make_pair(u, w), (int32_t)edge_id.size()).first;
            m.FE[3 * f + c] = it->second;
        }
    m.ne = (int64_t)edge_id.size();
    m.EN.assign(3 * m.ne, 0.0);
    for (int64_t f = 0; f < nf; ++f)
        for (int c = 0; c < 3; ++c) add_row(m.EN, m.FE[3 * f + c], vrow(m.FN, f), 1.0);
    normalize_rows(m.EN);
    // vertex normals: face normals weighted by the face's angle at the vertex
    m.VN.assign(3 * nv, 0.0);
    for (int64_t f = 0; f < nf; ++f)
        for (int c = 0; c < 3; ++c) {
            const V3d p = vrow(m.V, m.F[3 * f + c]);
            const V3d u = vsub(vrow(m.V, m.F[3 * f + (c + 1) % 3]), p), w = vsub(vrow(m.V, m.F[3 * f + (c + 2) % 3]), p);
            const double lu = std::sqrt(vdot(u, u)), lw = std::sqrt(vdot(w, w));
            double cs = (lu > 0.0 && lw > 0.0) ? vdot(u, w) / (lu * lw) : 1.0;
            cs = std::min(1.0, std::max(-1.0, cs));
            add_row(m.VN, m.F[3 * f + c], vrow(m.FN, f), std::acos(cs));
        }
    normalize_rows(m.VN);
    // BVH
    Builder B(m);
    B.cen.resize(3 * nf);
    for (int64_t f = 0; f < nf; ++f)
        for (int a = 0; a < 3; ++a)
            B.cen[3 * f + a] = (m.V[3 * (int64_t)m.F[3 * f] + a] + m.V[3 * (int64_t)m.F[3 * f + 1] + a] +
                                m.V[3 * (int64_t)m.F[3 * f + 2] + a]) / 3.0;
    B.idx.resize(nf);
    std::iota(B.idx.begin(), B.idx.end(), 0);
    B.build(0, (int32_t)nf);
    m.nodes = std::move(B.nodes);
    const int64_t nl = (nf + kBvhWidth - 1) / kBvhWidth;
    m.tri.assign(nl * kBvhWidth, kNoTriangle);
    m.tv.assign(nl * kBvhWidth * 9, 0.0);
    for (int64_t k = 0; k < nf; ++k) {
        const int32_t f = B.idx[k];
        m.tri[k] = degenerate[f] ? ~f : f;
        for (int c = 0; c < 3; ++c)
            for (int a = 0; a < 3; ++a)
                m.tv[(k / kBvhWidth) * 9 * kBvhWidth + (3 * c + a) * kBvhWidth + k % kBvhWidth] =
                    m.V[3 * (int64_t)m.F[3 * (int64_t)f + c] + a];
    }
    return "";
}

// ------------------------------------------------------------------ kernels
// Lane values across the 8 lanes of a group (aligned groups of a DPP row): the
// value of lane gl ^ X.
template <int X>
__device__ __forceinline__ uint32_t group_xor(uint32_t v) {
    constexpr int kQuad[4] = {0xE4, 0xB1, 0x4E, 0x1B};   // quad_perm of lane ^ 0 .. 3
    int r = (int)v;
    if constexpr (X & 4) r = dpp_i<0x141>(r);            // row_half_mirror: lane ^ 7
    constexpr int Q = (X & 4) ? (X ^ 7) : X;
    if constexpr (Q != 0) r = dpp_i<kQuad[Q]>(r);
    return (uint32_t)r;
}
__device__ __forceinline__ double group_min(double v) {
    v = fmin(v, dpp_move<0xB1>(v));
    v = fmin(v, dpp_move<0x4E>(v));
    return fmin(v, dpp_move<0x141>(v));
}

// The closest triangle to p, searched by the 8 lanes of a group (all with the same
// p; gl = the lane's place in it): each lane tests one child box of a node, or one
// triangle of a leaf, and keeps the best triangle it has tested; the group's bound
// is the least of them. A node's children whose boxes can hold a closer point go on
// the group's stack (LDS), the nearest on top: an entry is the child's code and its
// key (bvh_key). Boxes as near as the best triangle are visited too: among equal
// distances the smallest face wins, whatever the order. One lane per point is limited
// by its chain of dependent reads (1.08 ms for 60,000 points, 4,224 triangles, under
// one wavefront per SIMD, and a stack in scratch); eight lanes make eight times the
// wavefronts and an eighth of the steps.
__device__ __forceinline__ MeshHit mesh_closest(const MeshDev& M, D3 p, int gl, uint2* stack) {
    MeshHit h;
    h.c = p;
    h.b[0] = h.b[1] = h.b[2] = 0.0;
    double best = INFINITY;
    int code = 0, sp = 0;
    const int shift = (int)(threadIdx.x & 63) & ~7;
    const auto nodes = as_global(M.nodes);
    const auto tri = as_global(M.tri);
    const auto tv = as_global(M.tv);
    // the next entry that can hold a closer point, or none
    auto pop = [&]() {
        while (sp > 0) {
            const uint2 e = stack[--sp];
            if (bvh_key_bound(e.y) <= best) { code = (int)e.x; return true; }
        }
        return false;
    };
    for (bool more = true; more;) {
        while (more && code >= 0) {   // internal nodes, until a leaf is on top
            const float4 lo = nodes[2 * (code + gl)], hi = nodes[2 * (code + gl) + 1];
            const double e = box_dist2(p, lo, hi);
            const bool push = node_w(lo.w) != kBvhEmpty && e <= best;
            const uint32_t key = push ? bvh_key(e, gl) : 0u;
            int rank = 0;   // children on top of this one are nearer, those below it farther
            rank += group_xor<1>(key) > key;
            rank += group_xor<2>(key) > key;
            rank += group_xor<3>(key) > key;
            rank += group_xor<4>(key) > key;
            rank += group_xor<5>(key) > key;
            rank += group_xor<6>(key) > key;
            rank += group_xor<7>(key) > key;
            if (push) stack[sp + rank] = make_uint2((uint32_t)node_w(lo.w), key);
            sp += __popcll((__ballot(push) >> shift) & 0xffull);
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            more = pop();
        }
        if (!more) break;
        const int at = (-code - 1) * kBvhWidth;
        const int t = tri[at + gl];
        if (t != kNoTriangle) {
            const auto v = tv + (int64_t)at * 9 + gl;
            h.test(p, d3(v[0], v[8], v[16]), d3(v[24], v[32], v[40]), d3(v[48], v[56], v[64]), t < 0 ? ~t : t, t < 0);
        }
        best = group_min(h.d2);
        more = pop();
    }
    return h;
}

// Does this lane hold the group's closest triangle (the smallest face among equal
// distances)? Exactly one lane does; lane 0 when no triangle was found.
__device__ __forceinline__ bool mesh_winner(const MeshHit& h, int gl) {
    const double best = group_min(h.d2);
    uint32_t f = h.d2 == best && h.f >= 0 ? (uint32_t)h.f : 0xffffffffu;
    uint32_t m = f;
    m = min(m, group_xor<1>(m));
    m = min(m, group_xor<2>(m));
    m = min(m, group_xor<7>(m));
    return m == 0xffffffffu ? gl == 0 : f == m;
}

constexpr int kBvhStackStride = kBvhStack + 1;   // odd: the groups' stacks start in different banks

__global__ __launch_bounds__(256) void mesh_distance_kernel(MeshQueryArgs a) {
    __shared__ uint2 s_stack[32][kBvhStackStride];
    const int gl = threadIdx.x & 7, g = threadIdx.x >> 3;
    const int64_t i = (int64_t)blockIdx.x * 32 + g;
    if (i >= a.n) return;
    const double q0 = a.xw[3 * i] - a.p2[0], q1 = a.xw[3 * i + 1] - a.p2[1], q2 = a.xw[3 * i + 2] - a.p2[2];
    const D3 x = d3(a.R2[0] * q0 + a.R2[3] * q1 + a.R2[6] * q2, a.R2[1] * q0 + a.R2[4] * q1 + a.R2[7] * q2,
                    a.R2[2] * q0 + a.R2[5] * q1 + a.R2[8] * q2);
    double d = 10.0;   // BodyBVHObj.cpp:326-327: points outside the box keep d = 10, normal 0
    D3 nrm = d3(0.0, 0.0, 0.0);
    int f = -1;
    bool mine = gl == 0;
    if (mesh_box_filter(a.M, x)) {
        const MeshHit h = mesh_closest(a.M, x, gl, &s_stack[g][0]);
        mine = mesh_winner(h, gl);
        if (mine) {
            d = mesh_hit_distance(a.M, x, h, nrm) + a.col_th;
            f = h.f;
        }
    }
    if (!mine) return;
    a.d[i] = d;
    if (a.normal) { a.normal[3 * i] = nrm.x; a.normal[3 * i + 1] = nrm.y; a.normal[3 * i + 2] = nrm.z; }
    if (a.face) a.face[i] = f;
}

// One force object over workgroups of 8 wavefronts, block_points points each,
// kBvhStep at a time: 8 lanes find each point's signed distance; a point inside
// the mesh's box with d = signed distance + col_th < 0 is a contact
// (collision_detection_general_BVH, CollisionDetection.cpp:150-185). The first
// wavefront gathers the step's contacts, in point order, one per lane, and sums
// their wrench, p6 column and Jacobian blocks (FP64, put_jac_row); the steps'
// sums are added in order into the workgroup's partial row, and
// bvh_reduce_kernel adds the rows in a fixed order: the same result on every run.
// Small steps rather than many points per workgroup: a body has a few thousand
// points, and the traversal needs every CU (10,242 points in 6 workgroups of one
// lane per point: 2.46 ms).
// RIGID: the poses are rotations (InstDev::rigid); a kernel of its own, as the tangent
// columns of others would cost this one 63 spilled registers and 8 us.
template <bool RIGID>
__global__ __launch_bounds__(512) void bvh_force_kernel(BvhForceArgs a) {
    __shared__ union {
        uint2 stack[kBvhStep][kBvhStackStride];
        double col[JacColumns::SIZE];
    } s;
    __shared__ double s_part[RIGID ? kJacRowPad : kJvpRowPad];
    __shared__ double s_hit[4][kBvhStep];   // d, normal
    __shared__ int s_idx[kBvhStep], s_m;
    const int tid = (int)threadIdx.x, gl = tid & 7, g = tid >> 3, lane = tid & 63;
    const bool p6on = (a.flags & ATAC_EVAL_P6) != 0u, deriv = (a.flags & ATAC_EVAL_DERIV) != 0u;
    constexpr int NJ = RIGID ? kJacRow : kJvpRow;
    const int nrow = deriv ? NJ : 24;
    const int64_t b0 = (int64_t)blockIdx.x * a.block_points;
    const int64_t b1 = b0 + a.block_points < a.n ? b0 + a.block_points : a.n;
    double acc = 0.0;   // thread k < nrow: component k of the row
    int64_t cnt = 0;
    for (int64_t base = b0; base < b1; base += kBvhStep) {
        const int64_t i = base + g;
        bool mine = gl == 0;
        double d = 1.0;   // no contact
        D3 nrm = d3(0.0, 0.0, 0.0);
        if (i < b1) {
            double x[3];
            body2_point(a.in, a.xi[3 * i], a.xi[3 * i + 1], a.xi[3 * i + 2], x);
            const D3 xb = d3(x[0], x[1], x[2]);
            if (mesh_box_filter(a.M, xb)) {
                const MeshHit h = mesh_closest(a.M, xb, gl, &s.stack[g][0]);
                mine = mesh_winner(h, gl);
                if (mine) d = mesh_hit_distance(a.M, xb, h, nrm) + a.in.col_th;
            }
        }
        if (mine) { s_hit[0][g] = d; s_hit[1][g] = nrm.x; s_hit[2][g] = nrm.y; s_hit[3][g] = nrm.z; }
        __syncthreads();   // the stacks are done with: their room holds the columns
        if (tid < 64) {
            const bool have = s_hit[0][lane] < 0.0;
            const uint64_t bal = __ballot(have);
            const int m = __popcll(bal);
            if (have) s_idx[__popcll(bal & ((1ull << lane) - 1ull))] = lane;
            if (lane == 0) s_m = m;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (m > 0) {
                const int at = s_idx[min(lane, m - 1)];   // lanes past the last repeat it; their rows are not summed
                const int64_t j = base + at;
                ContactFwd<double> c;
                double x[3], p6[12];
                body2_point(a.in, a.xi[3 * j], a.xi[3 * j + 1], a.xi[3 * j + 2], x);
                c.xi1 = mk3<double>(a.xi[3 * j], a.xi[3 * j + 1], a.xi[3 * j + 2]);
                c.x = mk3<double>(x[0], x[1], x[2]);
                c.d = s_hit[0][at];
                c.g = mk3<double>(s_hit[1][at], s_hit[2][at], s_hit[3][at]);
#pragma unroll
                for (int k = 0; k < 6; ++k) c.H[k] = 0.0;
                c.slow = false;
                contact_forward<double>(make_inst<double>(a.in), c, p6);
                if (!p6on) {
#pragma unroll
                    for (int k = 0; k < 12; ++k) p6[k] = 0.0;
                }
                if (deriv && RIGID) put_jac_row<double>(JacColumns{s.col, s_part, lane, m}, jac_inst(a.in), c, p6);
                else if (deriv) put_jvp_row<double>(JvpColumns{s.col, s_part, lane, m}, make_inst<double>(a.in), c, p6);
                else put_wrench_row<double>(WaveColumns<24>{s.col, s_part, lane, m}, c, p6);
            }
        }
        __syncthreads();
        if (s_m > 0) {
            if (tid < nrow) acc += s_part[tid];
            cnt += s_m;
        }
        __syncthreads();
    }
    if (tid < NJ) a.part[(int64_t)blockIdx.x * kJvpRow + tid] = acc;
    if (tid == 0) a.part_cnt[blockIdx.x] = cnt;
}

// The workgroups' partial rows, added six rows apart in order and the six sums in
// order (three of tangent columns); then Km and Dm from the sums (zeros when not
// asked for).
template <bool RIGID>
__global__ __launch_bounds__(1024) void bvh_reduce_kernel(BvhForceArgs a, int nb) {
    constexpr int S = 960;   // threads that add rows; the last wavefront adds the counts
    constexpr int G = RIGID ? 6 : 3, W = S / G, NJ = RIGID ? kJacRow : kJvpRow;
    static_assert(NJ <= W, "G rows at a time");
    __shared__ double s_sum[S], s_m[288], s_R[9], s_t[3];
    __shared__ int64_t s_cnt[64];
    const int tid = (int)threadIdx.x, g = tid / W, k = tid % W;
    if (g < G && k < NJ) {
        double v = 0.0;
        int b = g;
        for (; b + 7 * G < nb; b += 8 * G) {
            double q[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) q[u] = a.part[(int64_t)(b + u * G) * kJvpRow + k];
#pragma unroll
            for (int u = 0; u < 8; ++u) v += q[u];
        }
        for (; b < nb; b += G) v += a.part[(int64_t)b * kJvpRow + k];
        s_sum[tid] = v;
    }
    if (tid >= S) {
        const int l = tid - S;
        int64_t c = 0;
        for (int b = l; b < nb; b += 64) c += a.part_cnt[b];
        s_cnt[l] = c;
        if (l == 0) {
            const JacInst J = jac_inst(a.in);
#pragma unroll
            for (int q = 0; q < 9; ++q) s_R[q] = J.R.a[q];
            s_t[0] = J.t.x; s_t[1] = J.t.y; s_t[2] = J.t.z;
        }
    }
    __syncthreads();
    if (tid < NJ) {
        double v = s_sum[tid];
        for (int q = 1; q < G; ++q) v += s_sum[q * W + tid];
        s_sum[tid] = v;
    }
    __syncthreads();
    if (tid < 24) a.out[tid] = s_sum[tid];
    const bool deriv = (a.flags & ATAC_EVAL_DERIV) != 0u;
    if (RIGID && tid < 288) s_m[tid] = jac_element(s_sum + 24, s_sum + 9, s_t, tid / 24, tid % 24);
    __syncthreads();
    if (tid < 288) {
        const int m = tid / 144, row = (tid % 144) / 12, col = tid % 12;
        a.out[24 + tid] = !deriv ? 0.0 : RIGID ? jac_entry(s_m, s_R, row, 12 * m + col) : jvp_entry(s_sum, m, row, col);
    }
    if (tid == 0 && a.n_active) {
        int64_t c = 0;
        for (int l = 0; l < 64; ++l) c += s_cnt[l];
        *a.n_active = c;
    }
}

hipError_t launch_mesh_distance(MeshQueryArgs a, hipStream_t st) {
    // a launch holds fewer than 2^32 threads, eight per point
    constexpr int64_t kMost = (int64_t)1 << 28;
    for (int64_t left = a.n; left > 0; left -= kMost) {
        a.n = left < kMost ? left : kMost;
        hipLaunchKernelGGL(mesh_distance_kernel, dim3((unsigned)((a.n + 31) / 32)), dim3(256), 0, st, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        a.xw += 3 * a.n;
        a.d += a.n;
        if (a.normal) a.normal += 3 * a.n;
        if (a.face) a.face += a.n;
    }
    return hipSuccess;
}

// ------------------------------------------------------------------ fixed scratch
// The partial rows and contact counts of the force launches of
// atac_bvh_force_noalloc: kBvhMaxBlocks workgroups' rows (kJvpRow doubles
// each), then their counts (one 8-byte word each). One copy per device, held
// until the process ends. Host code never passes `scratch` itself to a kernel
// (on the host it names a stand-in, not device memory): it uses the address
// hipGetSymbolAddress gave for the device, kept in g_scratch_addr.
static __device__ __align__(256) double scratch[kBvhMaxBlocks * (kJvpRow + 1)];

namespace {
constexpr int kScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_addr[kScratchDevices] = {};
}  // namespace

hipError_t bvh_scratch_setup(int device) {
    if (device < 0 || device >= kScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_addr[device]) return hipSuccess;
    int cur = -1;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device) return hipErrorInvalidDevice;   // the lookup needs the device current
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_addr[device] = p;
    return hipSuccess;
}

void* bvh_scratch_address(int device) {
    if (device < 0 || device >= kScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    return g_scratch_addr[device];
}

hipError_t launch_bvh_force(BvhForceArgs a, hipStream_t st) {
    a.block_points = bvh_block_points(a.n);
    const int nb = (int)bvh_force_blocks(a.n);
    if (a.in.rigid) hipLaunchKernelGGL(bvh_force_kernel<true>, dim3(nb), dim3(512), 0, st, a);
    else hipLaunchKernelGGL(bvh_force_kernel<false>, dim3(nb), dim3(512), 0, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (a.in.rigid) hipLaunchKernelGGL(bvh_reduce_kernel<true>, dim3(1), dim3(1024), 0, st, a, nb);
    else hipLaunchKernelGGL(bvh_reduce_kernel<false>, dim3(1), dim3(1024), 0, st, a, nb);
    return hipGetLastError();
}

}  // namespace atac
