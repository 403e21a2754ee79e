// Wavefront primitives of the kernels: DPP moves, sums over the lanes and the
// column sums that collect a contact's wrench and Jacobian blocks. Device code.
#pragma once
#include <hip/hip_runtime.h>
#include <utility>
#include "contact_math.h"

namespace atac {

// ------------------------------------------------------------------ wave primitives
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(dpp_i<CTRL>(__float_as_int(v)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(dpp_i<CTRL>(hi), dpp_i<CTRL>(lo));
}
__device__ __forceinline__ float read_lane(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double read_lane(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l), __builtin_amdgcn_readlane(__double2loint(v), l));
}

// Sum over the 64 lanes of a wavefront; every lane must be active. Within each
// row of 16 lanes: quad_perm [1,0,3,2], quad_perm [2,3,0,1], row_half_mirror,
// row_mirror; the four row totals are then read as scalars. The result is
// wave-uniform and its summation order is fixed.
template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    v += dpp_move<0xB1>(v);
    v += dpp_move<0x4E>(v);
    v += dpp_move<0x141>(v);
    v += dpp_move<0x140>(v);
    return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}

// Values a wavefront sums over its lanes, handed over one at a time (put<k>, in
// order of k): 16 columns wait in LDS (64 rows of 17 doubles: conflict-free writes
// by row and reads by column), then four lanes add each column, 16 rows each, and
// the sums go to `out`. Rows at or past `n` (lanes without a contact) are left
// out. One LDS write and, over four lanes, one read and one add per value and row:
// the butterfly over the lanes it replaces took about 25 VALU instructions.
template <int N>
struct WaveColumns {
    static constexpr int W = 16, STRIDE = 17, SIZE = 64 * STRIDE;
    double* s;     // SIZE doubles of this wavefront (all its lanes take part)
    double* out;   // N rounded up to W
    int lane, n;
    template <int K>
    __device__ __forceinline__ void put(double v) const {
        s[lane * STRIDE + K % W] = v;
        if constexpr (K % W == W - 1 || K == N - 1) flush(out + K / W * W);
    }
    template <int K0, int... I>
    __device__ __forceinline__ void put_all(const double* v, std::integer_sequence<int, I...>) const {
        (put<K0 + I>(v[I]), ...);
    }
    __device__ __forceinline__ void flush(double* to) const {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        const int r0 = lane & 48;
        const double* p = s + r0 * STRIDE + (lane & 15);
        double q[4] = {0.0, 0.0, 0.0, 0.0};
        // every row is read (each lane wrote one); rows past n add nothing
#pragma unroll
        for (int i = 0; i < 16; i += 4)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double v = p[(i + j) * STRIDE];
                q[j] += r0 + i + j < n ? v : 0.0;
            }
        double v = (q[0] + q[1]) + (q[2] + q[3]);
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        if (lane < W) to[lane] = v;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();   // the columns are free for the next round
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
};
using JacColumns = WaveColumns<kJacRow>;
constexpr int kJacRowPad = (kJacRow + JacColumns::W - 1) / JacColumns::W * JacColumns::W;

// A contact's wrench and p6 column into the columns, from its forward state.
template <typename R, int N>
__device__ __forceinline__ void put_wrench_row(const WaveColumns<N>& col, const ContactFwd<R>& s, const R p6[12]) {
    double f[24];
#pragma unroll
    for (int k = 0; k < 12; ++k) { f[k] = (double)s.f[k]; f[12 + k] = (double)p6[k]; }
    col.template put_all<0>(f, std::make_integer_sequence<int, 24>());
}

// The same followed by its Jacobian blocks (kJacRow values).
template <typename R>
__device__ __forceinline__ void put_jac_row(const JacColumns& col, const JacInst& J, const ContactFwd<R>& s, const R p6[12]) {
    put_wrench_row<R>(col, s, p6);
    const double H[6] = {s.H[0], s.H[1], s.H[2], s.H[3], s.H[4], s.H[5]};
    contact_jac(J, mk3<double>(s.xi1.x, s.xi1.y, s.xi1.z), (double)s.d, mk3<double>(s.g.x, s.g.y, s.g.z), H, s.fric, s.stat,
                [&](auto b, const m3<double>& M) {
                    col.put_all<24 + 9 * decltype(b)::value>(M.a, std::make_integer_sequence<int, 9>());
                });
}

// The same with the 24 tangent columns in place of the blocks, for poses that are not
// rotations (kJvpRow values, column by column; `col` hands over one of 12 at a time and
// writes W): the derivative of the wrench with the pose matrices as they are given.
using JvpColumns = WaveColumns<24>;
constexpr int kJvpRowPad = kJvpRow + JvpColumns::W;
template <typename R>
__device__ __forceinline__ void put_jvp_row(const JvpColumns& col, const InstR<R>& I, const ContactFwd<R>& s, const R p6[12]) {
    put_wrench_row<R>(col, s, p6);
    for (int j = 0; j < 24; ++j) {
        R df[12];
        contact_jvp<R>(I, s, unit_tangent<R>(j), df);
        double v[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) v[k] = (double)df[k];
        WaveColumns<12>{col.s, col.out + 24 + 12 * j, col.lane, col.n}.template put_all<0>(v, std::make_integer_sequence<int, 12>());
    }
}

// Km (m = 0) or Dm (m = 1), entry (row, c), from a row summed that way.
__device__ __forceinline__ double jvp_entry(const double* sum, int m, int row, int c) { return sum[24 + 12 * (12 * m + c) + row]; }

}  // namespace atac
