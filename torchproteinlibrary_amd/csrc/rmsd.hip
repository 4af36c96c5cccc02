// Coords2RMSD for MI355X (gfx950): minimal RMSD over rigid rotations and its
// gradient, each direction one kernel launch (the forward two for few large
// structures).  The C ABI is include/tpl_rmsd.h.
//
// The layer follows the reference's method (quaternion eigenproblem of the
// centred correlation matrix; coords2rmsd_interface.cpp:12-49,52-111,
// RMSDKernels.cu:5-39) with everything on the device:
//   forward, one workgroup per structure:
//     1. FP64 moments of the atoms relative to the structure's first atom
//        (sum x, sum y, sum x y^T, sum |x|^2, sum |y|^2), four atoms per
//        thread and pass, summed over the workgroup in two levels through LDS
//        (few large structures: over several workgroups, in two launches);
//     2. lane 0 centres them, builds the symmetric 4x4 matrix F of the
//        centred correlation R (the reference's element layout,
//        coords2rmsd_interface.cpp:153-158), takes its largest eigenpair
//        (rmsd_math.h: Newton on the characteristic quartic, eigenvector from
//        the adjugate; a shifted adjugate for a double root), forms U from the quaternion
//        (same formula, :35-45) and rmsd = sqrt((R2 - 2 |lambda| + 1e-10) / n)
//        (:182);
//   backward, one thread per atom: (x - cx - U^T (y - cy)) * g / (rmsd * n)
//     (Coords2RMSD.py:47-56), zero past num_atoms.
// Shifting by the first atom keeps the raw moments at the size of the
// structure, so centring them afterwards loses no digits to a large offset
// from the origin.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "report.h"
#include "rmsd_flagged.h"
#include "rmsd_math.h"
#include "tpl_rmsd.h"

namespace {

constexpr double kEpsLimit = 1e-10;  // coords2rmsd_interface.cpp:10
constexpr int kThreads = 256;        // forward workgroup: 4 waves
constexpr int kBwdThreads = 256;     // backward: one thread per atom
constexpr int kState = 16;           // doubles per structure: cx[3] cy[3] U[9] rmsd
constexpr int kMoments = 17;         // sx[3] sy[3] sxy[9] sxx syy

// Atoms a0 .. a0+3 of one structure (xyz interleaved) as 12 values: three
// 16-byte loads per 4 floats (six for doubles) when the run is whole, else
// element loads; atoms at or past `lim` read as 0.  The loads need the
// alignment of the values only, so a stride of any size has them: float32, 300
// structures of 3000..6001 atoms at a stride of 6001, forward 20.7 -> 12.3 us
// against 16-byte loads where the structure is 16-byte aligned.
template <typename T>
__device__ __forceinline__ void load4(const T* p, int a0, int lim, T t[12]) {
    typedef uint32_t Vec __attribute__((ext_vector_type(4), aligned(4)));
    if (a0 + 4 <= lim) {
        constexpr int E = 16 / (int)sizeof(T);  // elements per 16-byte load
#pragma unroll
        for (int k = 0; k < 12; k += E) {
            const Vec u = *reinterpret_cast<const Vec*>(p + 3 * (size_t)a0 + k);
            __builtin_memcpy(t + k, &u, 16);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 12; ++k) t[k] = (a0 + k / 3 < lim) ? p[3 * (size_t)a0 + k] : (T)0;
    }
}

__device__ __forceinline__ int clamp_count(int n, int A, const Report& rep, bool report_it) {
    if (n < 0 || n > A) {
        if (report_it) report_bits(rep, TPL_RMSD_STATUS_COUNT);
        return n < 0 ? 0 : A;
    }
    return n;
}

// Sums of the threads' moments over the workgroup, in tot (LDS): every thread's
// 17 partial sums (laid out [moment][thread]), then kParts partial sums per
// moment, then the totals.  A cross-lane butterfly over 17 doubles measured
// 5 us per workgroup, bound by the LDS crossbar at 16 waves per CU; this takes
// plain LDS reads and three barriers.  `low` (nullptr: not wanted) takes what
// the last level rounds off: the levels before it add up few and small terms.
__device__ __forceinline__ void workgroup_sums(const double m[kMoments], double* tot, double* low) {
    constexpr int kParts = kThreads / kMoments;  // 15 threads per moment in the middle level
    __shared__ double s_m[kMoments * kThreads];
    __shared__ double s_p[kMoments * kParts];
    const int tid = threadIdx.x;
#pragma unroll
    for (int e = 0; e < kMoments; ++e) s_m[e * kThreads + tid] = m[e];
    __syncthreads();
    if (tid < kMoments * kParts) {
        const int e = tid / kParts, part = tid - e * kParts;
        double acc = 0.0;
        for (int t = part; t < kThreads; t += kParts) acc += s_m[e * kThreads + t];
        s_p[e * kParts + part] = acc;
    }
    __syncthreads();
    if (tid < kMoments) {
        double acc = 0.0, off = 0.0;
#pragma unroll
        for (int part = 0; part < kParts; ++part) {
            const rmsd_math::Two t = rmsd_math::two_sum(acc, s_p[tid * kParts + part]);
            acc = t.h;
            off += t.l;
        }
        tot[tid] = acc;
        if (low) low[tid] = off;
    }
    __syncthreads();
}

// Thread's moments of atoms first, first + step, .. (runs of four) below n,
// relative to x0 and y0.
template <typename T>
__device__ __forceinline__ void add_moments(const T* xb, const T* yb, int first, int step, int n,
                                            const double x0[3], const double y0[3], double m[kMoments]) {
    for (int a0 = first; a0 < n; a0 += step) {
        T xv[12], yv[12];
        load4(xb, a0, n, xv);
        load4(yb, a0, n, yv);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const bool in = a0 + j < n;
            double dx[3], dy[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                dx[c] = in ? (double)xv[3 * j + c] - x0[c] : 0.0;
                dy[c] = in ? (double)yv[3 * j + c] - y0[c] : 0.0;
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                m[c] += dx[c];
                m[3 + c] += dy[c];
                m[15] += dx[c] * dx[c];
                m[16] += dy[c] * dy[c];
            }
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) m[6 + 3 * r + c] += dx[r] * dy[c];
        }
    }
}
template <typename T>
__device__ __forceinline__ void first_atoms(const T* xb, const T* yb, int n, double x0[3], double y0[3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        x0[c] = n > 0 ? (double)xb[c] : 0.0;
        y0[c] = n > 0 ? (double)yb[c] : 0.0;
    }
}

// One lane: the result of structure b, whose means are x0 + mx and y0 + my.
template <typename T>
__device__ __forceinline__ void store_result(double rmsd, const double U[9], const double x0[3], const double y0[3],
                                             const double mx[3], const double my[3], int b, T* rmsd_out, T* ut_out,
                                             double* state, const Report& rep) {
    rmsd_out[b] = (T)rmsd;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k) ut_out[9 * b + 3 * j + k] = (T)U[3 * k + j];
    if (state) {
        double* s = state + (size_t)b * kState;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s[c] = x0[c] + mx[c];
            s[3 + c] = y0[c] + my[c];
        }
#pragma unroll
        for (int k = 0; k < 9; ++k) s[6 + k] = U[k];
        s[15] = rmsd;
    }
    if (rmsd != rmsd) report_bits(rep, TPL_RMSD_STATUS_NAN);
}

// r2 - 2|lambda| is >= 0 in exact arithmetic; for (nearly) identical
// structures its FP64 rounding (~1e-16 r2) can make it negative, which
// the reference's formula turns into NaN.  Clamped at 0 here; a NaN (from
// NaN coordinates) stays NaN and is reported.
__device__ __forceinline__ double rmsd_of(double dev, double nd) {
    return sqrt(((dev < 0.0 ? 0.0 : dev) + kEpsLimit) / nd);
}

// One lane: the result of structure b from its moments.
template <typename T>
__device__ __forceinline__ void finish(const double m[kMoments], const double x0[3], const double y0[3], int n, int b,
                                       T* rmsd_out, T* ut_out, double* state, const Report& rep) {
    const double nd = (double)n;
    double mx[3], my[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        mx[c] = n > 0 ? m[c] / nd : 0.0;
        my[c] = n > 0 ? m[3 + c] / nd : 0.0;
    }
    // Centred correlation R[r][c] = sum (x - cx)_r (y - cy)_c, and R2.
    double R[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int c = 0; c < 3; ++c) R[3 * r + c] = m[6 + 3 * r + c] - nd * mx[r] * my[c];
    const double r2 = (m[15] - nd * (mx[0] * mx[0] + mx[1] * mx[1] + mx[2] * mx[2])) +
                      (m[16] - nd * (my[0] * my[0] + my[1] * my[1] + my[2] * my[2]));
    double F[16], U[9];
    rmsd_math::f_matrix(R, F);
    const rmsd_math::Eigenpair eig = rmsd_math::max_eigenpair(F, 0.5 * r2);
    rmsd_math::u_from_q(eig, U);
    const double rmsd = rmsd_of(r2 - 2.0 * fabs(eig.lam), nd);
    store_result(rmsd, U, x0, y0, mx, my, b, rmsd_out, ut_out, state, rep);
}

template <typename T>
__global__ void __launch_bounds__(kThreads) rmsd_fwd(const T* __restrict__ x, const T* __restrict__ y,
                                                     const int32_t* __restrict__ num_atoms, T* rmsd_out, T* ut_out,
                                                     double* state, Report rep, int A) {
    __shared__ double s_tot[kMoments];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int n = clamp_count(num_atoms[b], A, rep, tid == 0);
    const T* xb = x + (size_t)b * 3 * A;
    const T* yb = y + (size_t)b * 3 * A;
    double x0[3], y0[3], m[kMoments] = {};
    first_atoms(xb, yb, n, x0, y0);
    add_moments(xb, yb, 4 * tid, 4 * kThreads, n, x0, y0, m);
    workgroup_sums(m, s_tot, nullptr);
    if (tid != 0) return;
#pragma unroll
    for (int e = 0; e < kMoments; ++e) m[e] = s_tot[e];
    finish(m, x0, y0, n, b, rmsd_out, ut_out, state, rep);
}

// Few large structures: S workgroups per structure, whose sums go to part
// [B][kMoments][2][S] with what they round off, and a workgroup per structure that
// adds them up.  One workgroup alone is bound by the latency of its passes (20
// of 1024 atoms at 20000), us, back to back: 8 structures of 20000 atoms, float64,
// 16.4 -> 11.4; one, float32, 15.6 -> 9.6.  The second launch is bound by the
// eigen-solve of one lane and takes most of that.
// In float64 the last levels of the sums, the centring and r2 - 2 lambda keep
// both parts of each number: in another order than one workgroup's the plain
// sums round as much, but not the same way, and r2 is hundreds of times what
// remains of it.  rmsd of 8 structures of 9000..12001 atoms, 16 draws, off by
// (root mean square, relative): one workgroup 1.6e-13, plain split 1.5e-13,
// this 1.2e-14.
template <typename T>
__global__ void __launch_bounds__(kThreads) rmsd_part(const T* __restrict__ x, const T* __restrict__ y,
                                                      const int32_t* __restrict__ num_atoms, double* part, int A,
                                                      int S) {
    __shared__ double s_tot[kMoments], s_low[kMoments];
    const int b = (int)blockIdx.x / S, s = (int)blockIdx.x - b * S, tid = threadIdx.x;
    const int n = clamp_count(num_atoms[b], A, Report{nullptr, nullptr}, false);
    const T* xb = x + (size_t)b * 3 * A;
    const T* yb = y + (size_t)b * 3 * A;
    double x0[3], y0[3], m[kMoments] = {};
    first_atoms(xb, yb, n, x0, y0);
    add_moments(xb, yb, 4 * (s * kThreads + tid), 4 * kThreads * S, n, x0, y0, m);
    workgroup_sums(m, s_tot, s_low);
    if (tid < 2 * kMoments)
        part[((size_t)b * 2 * kMoments + tid) * S + s] = (tid & 1 ? s_low : s_tot)[tid >> 1];
}
__device__ __forceinline__ rmsd_math::Two two_sum_over(rmsd_math::Two v, int width) {
    for (int d = width / 2; d > 0; d >>= 1)
        v = rmsd_math::two_add(v, rmsd_math::Two{__shfl_xor(v.h, d), __shfl_xor(v.l, d)});
    return v;
}
constexpr int kJoin = 16;                                      // threads per moment
constexpr int kJoinThreads = (kMoments * kJoin + 63) / 64 * 64;  // whole waves
template <typename T>
__global__ void __launch_bounds__(kJoinThreads) rmsd_join(const T* __restrict__ x, const T* __restrict__ y,
                                                          const int32_t* __restrict__ num_atoms,
                                                          const double* __restrict__ part, T* rmsd_out, T* ut_out,
                                                          double* state, Report rep, int A, int S) {
    using rmsd_math::Two;
    __shared__ Two s_tot[kMoments], s_r[10];
    const int b = blockIdx.x, lane = threadIdx.x;
    Two v{0.0, 0.0};
    const int e = lane / kJoin;
    if (e < kMoments) {
        const double* p = part + ((size_t)b * kMoments + e) * 2 * S;
        for (int s = lane % kJoin; s < S; s += kJoin) {
            const Two t = rmsd_math::two_sum(v.h, p[s]);
            v = Two{t.h, v.l + (t.l + p[S + s])};
        }
    }
    v = two_sum_over(v, kJoin);
    if (e < kMoments && lane % kJoin == 0) s_tot[e] = v;
    __syncthreads();
    if (lane >= 64) return;
    const int n = clamp_count(num_atoms[b], A, rep, lane == 0);
    const double nd = (double)n;
    double x0[3], y0[3], m[kMoments];
    first_atoms(x + (size_t)b * 3 * A, y + (size_t)b * 3 * A, n, x0, y0);
#pragma unroll
    for (int k = 0; k < kMoments; ++k) m[k] = s_tot[k].h;
    if constexpr (sizeof(T) == 4) {  // the rounding to float is far larger
        if (lane == 0) finish(m, x0, y0, n, b, rmsd_out, ut_out, state, rep);
        return;
    }
    // R by lanes 0-8, |x|^2 and |y|^2 centred by lanes 16-23, each sum less
    // what centring takes off.
    if (lane < 9 || (lane >= 16 && lane < 24)) {
        const int k = lane - 18;
        const int r = lane < 9 ? lane / 3 : k, c = lane < 9 ? 3 + lane % 3 : k;
        v = lane < 9 ? s_tot[6 + lane] : k < 0 ? s_tot[lane - 1] : Two{0.0, 0.0};
        if ((lane < 9 || k >= 0) && n > 0) v = rmsd_math::two_sub(v, rmsd_math::two_mul_div(s_tot[r], s_tot[c], nd));
    } else {
        v = Two{0.0, 0.0};
    }
    if (lane < 9) s_r[lane] = v;
    v = two_sum_over(v, 8);
    if (lane == 16) s_r[9] = v;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // one wave is left
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const Two f = rmsd_math::deviation_factor(s_r, s_r[9], lane < 10 ? lane : 0);
    double R[9], F[16], U[9], mx[3], my[3];
#pragma unroll
    for (int k = 0; k < 9; ++k) R[k] = s_r[k].h;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        mx[c] = n > 0 ? m[c] / nd : 0.0;
        my[c] = n > 0 ? m[3 + c] / nd : 0.0;
    }
    rmsd_math::f_matrix(R, F);
    const rmsd_math::Eigenpair eig = rmsd_math::max_eigenpair(F, 0.5 * s_r[9].h);
    v = two_sum_over(lane < 10 ? rmsd_math::deviation_term(f, eig, lane) : Two{0.0, 0.0}, 16);
    if (lane != 0) return;
    rmsd_math::u_from_q(eig, U);
    store_result(rmsd_of(v.h, nd), U, x0, y0, mx, my, b, rmsd_out, ut_out, state, rep);
}

// One thread per atom slot; the grid covers nblk blocks per structure.
template <typename T>
__global__ void __launch_bounds__(kBwdThreads) rmsd_bwd(T* gx, const T* __restrict__ grad_rmsd,
                                                        const T* __restrict__ x,
                                                        const T* __restrict__ y,
                                                        const int32_t* __restrict__ num_atoms,
                                                        const double* __restrict__ state,
                                                        Report rep, int A, int nblk) {
    const int b = blockIdx.x / nblk;
    const int i = (blockIdx.x - b * nblk) * kBwdThreads + threadIdx.x;
    if (i >= A) return;
    const int n = clamp_count(num_atoms[b], A, rep, false);
    T* g = gx + (size_t)b * 3 * A + 3 * (size_t)i;
    if (i >= n) {
        g[0] = (T)0;
        g[1] = (T)0;
        g[2] = (T)0;
        return;
    }
    const double* s = state + (size_t)b * kState;
    const double scale = (double)grad_rmsd[b] / (s[15] * (double)n);
    const T* xi = x + (size_t)b * 3 * A + 3 * (size_t)i;
    const T* yi = y + (size_t)b * 3 * A + 3 * (size_t)i;
    double dx[3], dy[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        dx[c] = (double)xi[c] - s[c];
        dy[c] = (double)yi[c] - s[3 + c];
    }
    bool bad = false;
#pragma unroll
    for (int c = 0; c < 3; ++c) {  // (U^T dy)_c = sum_k U[k][c] dy_k
        const double uty = s[6 + c] * dy[0] + s[9 + c] * dy[1] + s[12 + c] * dy[2];
        const T v = (T)((dx[c] - uty) * scale);
        bad |= (v != v);
        g[c] = v;
    }
    if (bad) report_bits(rep, TPL_RMSD_STATUS_NAN);
}

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

int check(int dtype, int B, int A) {
    if (dtype != TPL_RMSD_F32 && dtype != TPL_RMSD_F64) return TPL_RMSD_ERR_ARG;
    if (B < 0 || A < 0) return TPL_RMSD_ERR_ARG;
    if ((int64_t)3 * A > INT32_MAX || (int64_t)9 * B > INT32_MAX) return TPL_RMSD_ERR_SIZE;
    return TPL_RMSD_OK;
}

// Workgroups per structure in the split forward, 1 where it does not pay: every
// workgroup has a full pass of 1024 atoms and no more of them run than the GPU
// holds at two per CU.  The second launch costs as much as 8 passes, and 64
// structures fill the GPU by themselves; one launch -> split, float64, us:
// 8 structures of 8192 atoms 10.4 -> 10.8, of 12001 12.7 -> 11.6, 32 of 12001
// 12.9 -> 12.1, 64 of 12001 15.8 -> 16.7.
int split_of(int B, int A) {
    if (B <= 0 || B > 32) return 1;
    const int s = std::min({64, A / (4 * kThreads), 512 / B});
    return s >= 10 ? s : 1;
}

template <typename T>
void launch_forward(const void* input, const void* target, const int32_t* num_atoms, void* rmsd, void* ut,
                    void* state, double* part, const Report& rep, int B, int A, hipStream_t s) {
    const T *x = static_cast<const T*>(input), *y = static_cast<const T*>(target);
    T *r = static_cast<T*>(rmsd), *u = static_cast<T*>(ut);
    double* st = static_cast<double*>(state);
    const int S = split_of(B, A);
    if (S > 1 && part) {
        hipLaunchKernelGGL(rmsd_part<T>, dim3(B * S), dim3(kThreads), 0, s, x, y, num_atoms, part, A, S);
        hipLaunchKernelGGL(rmsd_join<T>, dim3(B), dim3(kJoinThreads), 0, s, x, y, num_atoms, part, r, u, st, rep, A, S);
    } else {
        hipLaunchKernelGGL(rmsd_fwd<T>, dim3(B), dim3(kThreads), 0, s, x, y, num_atoms, r, u, st, rep, A);
    }
}

// The two directions, reporting as `rep` says.
int forward_on(int dtype, const void* input, const void* target, const int32_t* num_atoms, void* rmsd, void* ut,
               void* state, void* workspace, const Report& rep, int batch, int atoms_stride,
               tpl_rmsd_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_RMSD_OK) return rc;
    if (batch == 0) return TPL_RMSD_OK;
    if (!num_atoms || !rmsd || !ut || (atoms_stride > 0 && (!input || !target)))
        return TPL_RMSD_ERR_ARG;
    if (state && (reinterpret_cast<uintptr_t>(state) & 255)) return TPL_RMSD_ERR_ARG;
    (dtype == TPL_RMSD_F32 ? launch_forward<float> : launch_forward<double>)(
        input, target, num_atoms, rmsd, ut, state, static_cast<double*>(workspace), rep, batch, atoms_stride,
        static_cast<hipStream_t>(stream));
    return hipGetLastError() == hipSuccess ? TPL_RMSD_OK : TPL_RMSD_ERR_LAUNCH;
}

int backward_on(int dtype, void* grad_input, const void* grad_rmsd, const void* input,
                      const void* target, const int32_t* num_atoms, const void* state,
                      const Report& rep, int batch, int atoms_stride, tpl_rmsd_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_RMSD_OK) return rc;
    if (batch == 0 || atoms_stride == 0) return TPL_RMSD_OK;
    if (!grad_input || !grad_rmsd || !input || !target || !num_atoms || !state)
        return TPL_RMSD_ERR_ARG;
    if (reinterpret_cast<uintptr_t>(state) & 255) return TPL_RMSD_ERR_ARG;
    const int nblk = (atoms_stride + kBwdThreads - 1) / kBwdThreads;
    if ((int64_t)nblk * batch > INT32_MAX) return TPL_RMSD_ERR_SIZE;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const dim3 grid(nblk * batch);
    if (dtype == TPL_RMSD_F32)
        hipLaunchKernelGGL(rmsd_bwd<float>, grid, dim3(kBwdThreads), 0, s,
                           static_cast<float*>(grad_input), static_cast<const float*>(grad_rmsd),
                           static_cast<const float*>(input), static_cast<const float*>(target),
                           num_atoms, static_cast<const double*>(state), rep, atoms_stride, nblk);
    else
        hipLaunchKernelGGL(rmsd_bwd<double>, grid, dim3(kBwdThreads), 0, s,
                           static_cast<double*>(grad_input), static_cast<const double*>(grad_rmsd),
                           static_cast<const double*>(input), static_cast<const double*>(target),
                           num_atoms, static_cast<const double*>(state), rep, atoms_stride, nblk);
    return hipGetLastError() == hipSuccess ? TPL_RMSD_OK : TPL_RMSD_ERR_LAUNCH;
}

}  // namespace

extern "C" {

const char* tpl_rmsd_strerror(int code) {
    switch (code) {
        case TPL_RMSD_OK: return "ok";
        case TPL_RMSD_ERR_ARG: return "invalid argument (null pointer, negative size or unknown dtype)";
        case TPL_RMSD_ERR_LAUNCH: return "kernel launch failed";
        case TPL_RMSD_ERR_SIZE: return "batch * atoms_stride too large";
        default: return "unknown error code";
    }
}

size_t tpl_rmsd_state_bytes(int batch) {
    return batch <= 0 ? 0 : align256((size_t)batch * kState * sizeof(double));
}

int tpl_rmsd_forward(int dtype, const void* input, const void* target, const int32_t* num_atoms,
                     void* rmsd, void* ut, void* state, uint32_t* status, int batch,
                     int atoms_stride, tpl_rmsd_stream_t stream) {
    return forward_on(dtype, input, target, num_atoms, rmsd, ut, state, nullptr, Report{status, nullptr}, batch,
                      atoms_stride, stream);
}

int tpl_rmsd_backward(int dtype, void* grad_input, const void* grad_rmsd, const void* input,
                      const void* target, const int32_t* num_atoms, const void* state,
                      uint32_t* status, int batch, int atoms_stride, tpl_rmsd_stream_t stream) {
    return backward_on(dtype, grad_input, grad_rmsd, input, target, num_atoms, state, Report{status, nullptr},
                       batch, atoms_stride, stream);
}

size_t tplx_rmsd_workspace_bytes(int batch, int atoms_stride) {
    const int S = split_of(batch, atoms_stride);
    return S > 1 ? (size_t)batch * 2 * kMoments * S * sizeof(double) : 0;
}

int tplx_rmsd_forward(int dtype, const void* input, const void* target, const int32_t* num_atoms, void* rmsd,
                      void* ut, void* state, void* workspace, uint32_t* status, uint32_t* flags, int batch,
                      int atoms_stride, tpl_rmsd_stream_t stream) {
    return forward_on(dtype, input, target, num_atoms, rmsd, ut, state, workspace, Report{status, flags}, batch,
                      atoms_stride, stream);
}

int tplx_rmsd_backward(int dtype, void* grad_input, const void* grad_rmsd, const void* input, const void* target,
                       const int32_t* num_atoms, const void* state, uint32_t* flags, int batch, int atoms_stride,
                       tpl_rmsd_stream_t stream) {
    return backward_on(dtype, grad_input, grad_rmsd, input, target, num_atoms, state, Report{nullptr, flags},
                       batch, atoms_stride, stream);
}

}  // extern "C"
