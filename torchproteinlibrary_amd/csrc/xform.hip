// Coordinate transforms for MI355X (gfx950): translate, rotate and centre
// batches of structures, forward and backward.  The C ABI is
// include/tpl_xform.h.
//
// The reference launches <<<atoms_stride, batch_size>>> grids (one block per
// atom index, one thread per structure: TransformCUDAKernels.cu:14-17,
// 34-36,51-53,71-74,100-107), so neighbouring threads touch addresses
// 12*atoms_stride bytes apart, and its centre is a serial loop in one thread
// per structure (:77-86).  Here every global access is a 16-byte one at
// consecutive addresses across a wave: translation and rotation stage a
// wave's chunk of atoms through LDS, the centre's backward writes 16-byte
// blocks directly; every slot past num_atoms is written 0, and the centre is
// a workgroup sum in FP64 per structure.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "report.h"
#include "tpl_xform.h"
#include "xform_flagged.h"

namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ int clamp_count(int n, int A, const Report& rep, bool report_it) {
    if (n < 0 || n > A) {
        if (report_it) report_bits(rep, TPL_XFORM_STATUS_COUNT);
        return n < 0 ? 0 : A;
    }
    return n;
}

constexpr int kAtoms = 4;  // atoms per 16-byte run in the centre's loads
constexpr int kBlocksPerThread = 3;  // 16-byte blocks per thread in xform_shift

// 16 bytes of global memory, aligned like the values (4 bytes are enough), so
// that structures at a stride of any size have them: float32, 300 structures at a
// stride of 6001 atoms, translation 14.8 -> 7.4 us, centre 7.9 -> 5.7, its
// backward 10.6 -> 6.2 (16-byte accesses to aligned structures alone before).
typedef uint32_t Vec __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ Vec load16(const void* p) { return *static_cast<const Vec*>(p); }
__device__ __forceinline__ void store16(void* p, Vec v) { *static_cast<Vec*>(p) = v; }

// out = in + t (in null: 0) over the structure's 3A values taken flat, 0 past
// num_atoms, with t = tv[b] * tscale (tv null: 0), tscale = 1 or 1/n (per_n).
// The translations and the centre's backward need no atom grouping, so each
// thread moves 16-byte blocks at consecutive addresses across the wave: one
// store instruction covers 1 KB of contiguous output.  Grid: nblk blocks of
// kThreads * kBlocksPerThread 16-byte blocks per structure.  RANGE: outputs out
// of range are reported (here and below only where a caller asks: looking took
// 0.6 of 5.5 us in a rotation of 2000 structures of 63 atoms, float64).
template <typename T, bool RANGE>
__global__ void __launch_bounds__(kThreads) xform_shift(T* out, const T* __restrict__ in,
                                                        const T* __restrict__ tv, int per_n,
                                                        const int32_t* __restrict__ num_atoms,
                                                        Report rep, int A, int nblk) {
    constexpr int E = 16 / (int)sizeof(T);  // values per 16-byte block
    const int b = blockIdx.x / nblk;
    const int64_t blk0 = (int64_t)(blockIdx.x - b * nblk) * kThreads * kBlocksPerThread;
    const int n = clamp_count(num_atoms[b], A, rep, blk0 == 0 && threadIdx.x == 0);
    const int64_t vals = 3 * (int64_t)A, valid = 3 * (int64_t)n;
    T* o = out + (size_t)b * vals;
    const T* p = in ? in + (size_t)b * vals : nullptr;
    T t[3] = {(T)0, (T)0, (T)0};
    if (tv && n > 0) {
        const T sc = per_n ? (T)(1.0 / (double)n) : (T)1;
#pragma unroll
        for (int c = 0; c < 3; ++c) t[c] = tv[3 * (size_t)b + c] * sc;
    }
    bool range = false;
#pragma unroll
    for (int r = 0; r < kBlocksPerThread; ++r) {
        const int64_t v0 = ((int64_t)blk0 + r * kThreads + threadIdx.x) * E;
        if (v0 >= vals) break;
        T v[E];
        if (v0 + E <= vals) {
            if (p && v0 < valid) {
                const Vec u = load16(p + v0);
                __builtin_memcpy(v, &u, 16);
            } else {
#pragma unroll
                for (int e = 0; e < E; ++e) v[e] = (T)0;
            }
            // v0 < 3A <= INT32_MAX here: a 32-bit remainder is exact (a 64-bit
            // one is a long software sequence on the GPU)
            int c = (int)((uint32_t)v0 % 3u);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                v[e] = v0 + e < valid ? v[e] + t[c] : (T)0;
                if (RANGE) range |= out_of_range(v[e]);
                c = c == 2 ? 0 : c + 1;
            }
            Vec u;
            __builtin_memcpy(&u, v, 16);
            store16(o + v0, u);
        } else {
            for (int e = 0; e < E && v0 + e < vals; ++e) {
                const int64_t i = v0 + e;
                const T v1 = i < valid ? (p ? p[i] : (T)0) + t[(uint32_t)i % 3u] : (T)0;
                if (RANGE) range |= out_of_range(v1);
                o[i] = v1;
            }
        }
    }
    if (RANGE && range) report_flag(rep, TPLX_XFORM_RANGE);
}

// out_i = M in_i + t for the atoms of the structure (M = R, R^T with
// transpose, or I when R is null; t = tv[b], or 0 when tv is null), 0 past
// num_atoms, with every global access a 16-byte one at consecutive addresses
// across the wave.  Each wave takes a chunk of kWaveAtoms atoms
// (3 * kWaveAtoms values): it loads the chunk into its own slice of LDS with
// coalesced 16-byte loads, each lane rotates four whole atoms there, and the
// wave stores the chunk back with coalesced 16-byte stores.  The slice is the
// wave's alone, so the wave needs no workgroup barrier; the wavefront fences
// and the wave barrier keep the LDS writes before the reads.  A chunk that
// runs past the structure's stride goes atom by atom.
// Grid: nblk blocks of 4 chunks per structure.
constexpr int kWaveAtoms = 256;

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T>
__device__ __forceinline__ void rotate_atom(const T m[9], int transpose, const T v[3], T w[3]) {
#pragma unroll
    for (int r = 0; r < 3; ++r)
        w[r] = transpose ? m[r] * v[0] + m[3 + r] * v[1] + m[6 + r] * v[2]
                         : m[3 * r] * v[0] + m[3 * r + 1] * v[1] + m[3 * r + 2] * v[2];
}

template <typename T, bool RANGE>
__global__ void __launch_bounds__(kThreads) xform_waves(T* out, const T* __restrict__ in,
                                                        const T* __restrict__ R, int transpose,
                                                        const T* __restrict__ tv,
                                                        const int32_t* __restrict__ num_atoms,
                                                        Report rep, int A, int nblk) {
    constexpr int E = 16 / (int)sizeof(T);  // values per 16-byte access
    constexpr int V = 3 * kWaveAtoms;       // values per chunk
    constexpr int kPerLane = kWaveAtoms / 64;
    __shared__ __align__(16) T s_buf[kThreads / 64][V];
    const int b = blockIdx.x / nblk;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int a0 = ((blockIdx.x - b * nblk) * (kThreads / 64) + wave) * kWaveAtoms;
    if (a0 >= A) return;  // the whole wave: no workgroup barrier follows
    const int n = clamp_count(num_atoms[b], A, rep, a0 == 0 && lane == 0);
    T* o = out + (size_t)b * 3 * A;
    const T* p = in + (size_t)b * 3 * A;
    T m[9], t[3] = {(T)0, (T)0, (T)0};
#pragma unroll
    for (int k = 0; k < 9; ++k) m[k] = R ? R[(size_t)b * 9 + k] : (T)(k % 4 == 0 ? 1 : 0);
    if (tv) {
#pragma unroll
        for (int c = 0; c < 3; ++c) t[c] = tv[3 * (size_t)b + c];
    }
    if (a0 + kWaveAtoms <= A) {
        T* buf = s_buf[wave];
        if (a0 < n) {
#pragma unroll
            for (int j = 0; j < V / (64 * E); ++j) {
                const int idx = (j * 64 + lane) * E;
                const Vec u = load16(p + 3 * (size_t)a0 + idx);
                __builtin_memcpy(__builtin_assume_aligned(buf + idx, 16), &u, 16);
            }
        }
        wave_lds_sync();
        bool range = false;
#pragma unroll
        for (int k = 0; k < kPerLane; ++k) {
            const int q = kPerLane * lane + k;
            T v[3] = {buf[3 * q], buf[3 * q + 1], buf[3 * q + 2]}, w[3] = {(T)0, (T)0, (T)0};
            if (a0 + q < n) {
                if (R) rotate_atom(m, transpose, v, w);
                else w[0] = v[0], w[1] = v[1], w[2] = v[2];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    w[c] += t[c];
                    if (RANGE) range |= out_of_range(w[c]);
                }
            }
            buf[3 * q] = w[0];
            buf[3 * q + 1] = w[1];
            buf[3 * q + 2] = w[2];
        }
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < V / (64 * E); ++j) {
            const int idx = (j * 64 + lane) * E;
            Vec u;
            __builtin_memcpy(&u, __builtin_assume_aligned(buf + idx, 16), 16);
            store16(o + 3 * (size_t)a0 + idx, u);
        }
        if (RANGE && range) report_flag(rep, TPLX_XFORM_RANGE);
        return;
    }
    bool range = false;
#pragma unroll
    for (int k = 0; k < kPerLane; ++k) {
        const int i = a0 + kPerLane * lane + k;
        if (i >= A) break;
        T v[3] = {(T)0, (T)0, (T)0}, w[3] = {(T)0, (T)0, (T)0};
        if (i < n) {
            v[0] = p[3 * (size_t)i];
            v[1] = p[3 * (size_t)i + 1];
            v[2] = p[3 * (size_t)i + 2];
            if (R) rotate_atom(m, transpose, v, w);
            else w[0] = v[0], w[1] = v[1], w[2] = v[2];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                w[c] += t[c];
                if (RANGE) range |= out_of_range(w[c]);
            }
        }
        o[3 * (size_t)i] = w[0];
        o[3 * (size_t)i + 1] = w[1];
        o[3 * (size_t)i + 2] = w[2];
    }
    if (RANGE && range) report_flag(rep, TPLX_XFORM_RANGE);
}

// center[b] = (sum of the first n atoms) / n, summed in FP64: each thread over
// a strided share of runs of kAtoms atoms (16-byte loads), then two levels
// through LDS.
template <typename T>
__global__ void __launch_bounds__(kThreads) xform_center(T* center, const T* __restrict__ in,
                                                         const int32_t* __restrict__ num_atoms,
                                                         Report rep, int A) {
    constexpr int kParts = 16;
    __shared__ double s_m[3 * kThreads];
    __shared__ double s_p[3 * kParts];
    const int b = blockIdx.x, tid = threadIdx.x;
    const int n = clamp_count(num_atoms[b], A, rep, tid == 0);
    const T* p = in + (size_t)b * 3 * A;
    constexpr int kPer16 = 16 / (int)sizeof(T);
    double acc[3] = {0.0, 0.0, 0.0};
    for (int a0 = tid * kAtoms; a0 < n; a0 += kThreads * kAtoms) {
        if (a0 + kAtoms <= n) {
            T v[3 * kAtoms];
#pragma unroll
            for (int k = 0; k < 3 * kAtoms; k += kPer16) {
                const Vec u = load16(p + 3 * (size_t)a0 + k);
                __builtin_memcpy(v + k, &u, 16);
            }
#pragma unroll
            for (int k = 0; k < 3 * kAtoms; ++k) acc[k % 3] += (double)v[k];
        } else {
            for (int i = a0; i < n && i < a0 + kAtoms; ++i) {
#pragma unroll
                for (int c = 0; c < 3; ++c) acc[c] += (double)p[3 * (size_t)i + c];
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) s_m[c * kThreads + tid] = acc[c];
    __syncthreads();
    if (tid < 3 * kParts) {
        const int c = tid / kParts, part = tid - c * kParts;
        double s = 0.0;
        for (int t = part; t < kThreads; t += kParts) s += s_m[c * kThreads + t];
        s_p[c * kParts + part] = s;
    }
    __syncthreads();
    if (tid < 3) {
        double s = 0.0;
#pragma unroll
        for (int part = 0; part < kParts; ++part) s += s_p[tid * kParts + part];
        const T c = (T)(s / (double)n);
        if (out_of_range(c)) report_flag(rep, TPLX_XFORM_RANGE);
        center[3 * (size_t)b + tid] = c;
    }
}

int check(int dtype, int B, int A) {
    if (dtype != TPL_XFORM_F32 && dtype != TPL_XFORM_F64) return TPL_XFORM_ERR_ARG;
    if (B < 0 || A < 0) return TPL_XFORM_ERR_ARG;
    if ((int64_t)3 * A > INT32_MAX || (int64_t)9 * B > INT32_MAX) return TPL_XFORM_ERR_SIZE;
    return TPL_XFORM_OK;
}

template <typename T, bool RANGE>
int launch_affine(void* out, const void* in, const void* R, int transpose, const void* tv, int per_n,
                  const int32_t* num_atoms, const Report& rep, int B, int A, hipStream_t s) {
    T* o = static_cast<T*>(out);
    const T *x = static_cast<const T*>(in), *r = static_cast<const T*>(R), *t = static_cast<const T*>(tv);
    if (x && !per_n) {
        const int64_t per = (int64_t)(kThreads / 64) * kWaveAtoms;
        const int64_t nb = ((int64_t)A + per - 1) / per;
        if (nb * B > INT32_MAX) return TPL_XFORM_ERR_SIZE;
        const int nblk = (int)nb;
        hipLaunchKernelGGL((xform_waves<T, RANGE>), dim3(nblk * B), dim3(kThreads), 0, s, o, x, r, transpose, t,
                           num_atoms, rep, A, nblk);
    } else if (!r) {
        const int64_t per = (int64_t)kThreads * kBlocksPerThread * (16 / (int)sizeof(T));
        const int64_t nb = (3 * (int64_t)A + per - 1) / per;
        if (nb * B > INT32_MAX) return TPL_XFORM_ERR_SIZE;
        const int nblk = (int)nb;
        hipLaunchKernelGGL((xform_shift<T, RANGE>), dim3(nblk * B), dim3(kThreads), 0, s, o, x, t, per_n, num_atoms,
                           rep, A, nblk);
    } else {
        return TPL_XFORM_ERR_ARG;  // a rotation needs an input
    }
    return hipGetLastError() == hipSuccess ? TPL_XFORM_OK : TPL_XFORM_ERR_LAUNCH;
}

int launch_affine(int dtype, void* out, const void* in, const void* R, int transpose,
                  const void* tv, int per_n, const int32_t* num_atoms, const Report& rep, int B,
                  int A, tpl_xform_stream_t stream) {
    const auto launch = dtype == TPL_XFORM_F32
                            ? (rep.flags ? launch_affine<float, true> : launch_affine<float, false>)
                            : (rep.flags ? launch_affine<double, true> : launch_affine<double, false>);
    return launch(out, in, R, transpose, tv, per_n, num_atoms, rep, B, A, static_cast<hipStream_t>(stream));
}

// The entry points, reporting as `rep` says.
int translate(int dtype, void* out, const void* in, const void* T, const int32_t* num_atoms, const Report& rep,
              int batch, int atoms_stride, tpl_xform_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_XFORM_OK) return rc;
    if (batch == 0 || atoms_stride == 0) return TPL_XFORM_OK;
    if (!out || !in || !T || !num_atoms) return TPL_XFORM_ERR_ARG;
    return launch_affine(dtype, out, in, nullptr, 0, T, 0, num_atoms, rep, batch, atoms_stride, stream);
}

int rotate(int dtype, void* out, const void* in, const void* R, int transpose, const int32_t* num_atoms,
           const Report& rep, int batch, int atoms_stride, tpl_xform_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_XFORM_OK) return rc;
    if (batch == 0 || atoms_stride == 0) return TPL_XFORM_OK;
    if (!out || !in || !R || !num_atoms) return TPL_XFORM_ERR_ARG;
    return launch_affine(dtype, out, in, R, transpose ? 1 : 0, nullptr, 0, num_atoms, rep, batch, atoms_stride,
                         stream);
}

int center_of(int dtype, void* center, const void* in, const int32_t* num_atoms, const Report& rep, int batch,
              int atoms_stride, tpl_xform_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_XFORM_OK) return rc;
    if (batch == 0) return TPL_XFORM_OK;
    if (!center || !num_atoms || (atoms_stride > 0 && !in)) return TPL_XFORM_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == TPL_XFORM_F32)
        hipLaunchKernelGGL(xform_center<float>, dim3(batch), dim3(kThreads), 0, s, static_cast<float*>(center),
                           static_cast<const float*>(in), num_atoms, rep, atoms_stride);
    else
        hipLaunchKernelGGL(xform_center<double>, dim3(batch), dim3(kThreads), 0, s, static_cast<double*>(center),
                           static_cast<const double*>(in), num_atoms, rep, atoms_stride);
    return hipGetLastError() == hipSuccess ? TPL_XFORM_OK : TPL_XFORM_ERR_LAUNCH;
}

int center_backward(int dtype, void* grad_in, const void* grad_center, const int32_t* num_atoms,
                    const Report& rep, int batch, int atoms_stride, tpl_xform_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_XFORM_OK) return rc;
    if (batch == 0 || atoms_stride == 0) return TPL_XFORM_OK;
    if (!grad_in || !grad_center || !num_atoms) return TPL_XFORM_ERR_ARG;
    return launch_affine(dtype, grad_in, nullptr, nullptr, 0, grad_center, 1, num_atoms, rep, batch,
                         atoms_stride, stream);
}

}  // namespace

extern "C" {

const char* tpl_xform_strerror(int code) {
    switch (code) {
        case TPL_XFORM_OK: return "ok";
        case TPL_XFORM_ERR_ARG: return "invalid argument (null pointer, negative size or unknown dtype)";
        case TPL_XFORM_ERR_LAUNCH: return "kernel launch failed";
        case TPL_XFORM_ERR_SIZE: return "sizes too large";
        default: return "unknown error code";
    }
}

int tpl_xform_translate(int dtype, void* out, const void* in, const void* T,
                        const int32_t* num_atoms, uint32_t* status, int batch, int atoms_stride,
                        tpl_xform_stream_t stream) {
    return translate(dtype, out, in, T, num_atoms, Report{status, nullptr}, batch, atoms_stride, stream);
}

int tpl_xform_translate_backward(int dtype, void* grad_in, const void* grad_out,
                                 const int32_t* num_atoms, uint32_t* status, int batch,
                                 int atoms_stride, tpl_xform_stream_t stream) {
    const int rc = check(dtype, batch, atoms_stride);
    if (rc != TPL_XFORM_OK) return rc;
    if (batch == 0 || atoms_stride == 0) return TPL_XFORM_OK;
    if (!grad_in || !grad_out || !num_atoms) return TPL_XFORM_ERR_ARG;
    return launch_affine(dtype, grad_in, grad_out, nullptr, 0, nullptr, 0, num_atoms, Report{status, nullptr},
                         batch, atoms_stride, stream);
}

int tpl_xform_rotate(int dtype, void* out, const void* in, const void* R, int transpose,
                     const int32_t* num_atoms, uint32_t* status, int batch, int atoms_stride,
                     tpl_xform_stream_t stream) {
    return rotate(dtype, out, in, R, transpose, num_atoms, Report{status, nullptr}, batch, atoms_stride, stream);
}

int tpl_xform_center(int dtype, void* center, const void* in, const int32_t* num_atoms,
                     uint32_t* status, int batch, int atoms_stride, tpl_xform_stream_t stream) {
    return center_of(dtype, center, in, num_atoms, Report{status, nullptr}, batch, atoms_stride, stream);
}

int tpl_xform_center_backward(int dtype, void* grad_in, const void* grad_center,
                              const int32_t* num_atoms, uint32_t* status, int batch,
                              int atoms_stride, tpl_xform_stream_t stream) {
    return center_backward(dtype, grad_in, grad_center, num_atoms, Report{status, nullptr}, batch, atoms_stride,
                           stream);
}

int tplx_xform_translate(int dtype, void* out, const void* in, const void* T, const int32_t* num_atoms,
                         uint32_t* flags, int batch, int atoms_stride, tpl_xform_stream_t stream) {
    return translate(dtype, out, in, T, num_atoms, Report{nullptr, flags}, batch, atoms_stride, stream);
}

int tplx_xform_rotate(int dtype, void* out, const void* in, const void* R, int transpose,
                      const int32_t* num_atoms, uint32_t* flags, int batch, int atoms_stride,
                      tpl_xform_stream_t stream) {
    return rotate(dtype, out, in, R, transpose, num_atoms, Report{nullptr, flags}, batch, atoms_stride, stream);
}

int tplx_xform_center(int dtype, void* center, const void* in, const int32_t* num_atoms, uint32_t* flags,
                      int batch, int atoms_stride, tpl_xform_stream_t stream) {
    return center_of(dtype, center, in, num_atoms, Report{nullptr, flags}, batch, atoms_stride, stream);
}

int tplx_xform_center_backward(int dtype, void* grad_in, const void* grad_center, const int32_t* num_atoms,
                               uint32_t* flags, int batch, int atoms_stride, tpl_xform_stream_t stream) {
    return center_backward(dtype, grad_in, grad_center, num_atoms, Report{nullptr, flags}, batch, atoms_stride,
                           stream);
}

}  // extern "C"
