// The tomography objective around the Eikonal path (scripts/inversion.jl):
// source initialisation (:48-60), receiver gather + misfit with its sparse
// adjoint source (:64-105), and the model parametrisation + smoothing
// regulariser (:42-43, :107-121).  All on the device, so an inversion step
// needs no host round trip between the solves.
#include "eikonal_device.hpp"
#include "kernels.hpp"
#include "misfit3.hpp"

namespace adt {

// Begin of part `q` of `parts` of an array: whole 16-byte pieces from its start.
template <typename T>
__device__ __forceinline__ int64_t part_begin(int64_t N, int q, int parts) {
  constexpr int V = 16 / (int)sizeof(T);
  if (q >= parts) return N;
  return (N / V) * q / parts * V;
}

// a[lo..hi) = v by one workgroup, in 16-byte stores where the address allows.
template <typename T>
__device__ __forceinline__ void fill_part(T* __restrict__ a, int64_t lo, int64_t hi, T v) {
  constexpr int V = 16 / (int)sizeof(T);
  using vec = __attribute__((ext_vector_type(16 / sizeof(T)))) T;
  if (((uintptr_t)(a + lo) & 15) == 0) {
    const int64_t nv = (hi - lo) / V;
    vec* const p = (vec*)(a + lo);
    for (int64_t q = threadIdx.x; q < nv; q += blockDim.x) p[q] = vec(v);
    lo += nv * V;
  }
  for (int64_t q = lo + threadIdx.x; q < hi; q += blockDim.x) a[q] = v;
}

// ------------------------------------------------------- source init ---

// u0 = 1000 everywhere, then the 8 grid nodes around a station at 1-based
// coordinates (x, y, z) get dist * h / vel0 * scale (scripts/inversion.jl:48-60;
// scale = vp/vs for S, scripts/inversion_joint.jl:65-73).  `parts` workgroups per
// station, each a contiguous part of u0 and those of the 8 nodes that lie in it (a
// node that several corners name gets the same value from each).
//
// Bound by the writes: one workgroup per station, 8 bytes a store, took 411 us
// for 32 stations of 200x200x80 FP64 (2.0 TB/s); this takes 131 us (6.2 TB/s).
template <typename T>
__global__ void __launch_bounds__(256) source_u0_kernel(SourceTable tab,
                                                        const T* __restrict__ vel0, int m, int n,
                                                        int l, T h, int parts) {
  const SourceDesc& s = tab.s[blockIdx.x / parts];
  T* __restrict__ u0 = (T*)s.u0;
  const int64_t nl = (int64_t)n * l, N = (int64_t)m * nl;
  const int64_t lo = part_begin<T>(N, blockIdx.x % parts, parts);
  const int64_t hi = part_begin<T>(N, blockIdx.x % parts + 1, parts);
  fill_part(u0, lo, hi, T(1000));
  __syncthreads();
  if (threadIdx.x < 8) {
    const T x = (T)s.x, y = (T)s.y, z = (T)s.z, sc = (T)s.scale;
    const int c = threadIdx.x;
    const int ix = (int)(c & 4 ? __builtin_floor(s.x) : __builtin_ceil(s.x));
    const int iy = (int)(c & 2 ? __builtin_floor(s.y) : __builtin_ceil(s.y));
    const int iz = (int)(c & 1 ? __builtin_floor(s.z) : __builtin_ceil(s.z));
    const T dx = x - (T)ix, dy = y - (T)iy, dz = z - (T)iz;
    const int64_t q = (int64_t)(ix - 1) * nl + (int64_t)(iy - 1) * l + (iz - 1);
    if (q >= lo && q < hi) {
      const T dist = Real<T>::sqrt_(dx * dx + dy * dy + dz * dz);
      u0[q] = dist * h / vel0[q] * sc;
    }
  }
}

// ------------------------------------------- receiver gather + misfit ---

// The misfit of several solves (stations) in two steps: seeds and loss (the first
// workgroup of each) beside grad_u = 0 (`parts` workgroups of 256 threads each,
// bound by the writes), then the node sums over many workgroups (each a chain of
// four dependent loads).  In one workgroup per solve 32 solves of 200x200x80
// FP64 with 500 receivers took 397 us, 310 of them zeros; the steps take
// 171 and 10 to 60 us.
template <typename T>
__global__ void __launch_bounds__(256) misfit_kernel(const MisfitDesc* __restrict__ d,
                                                     const MisfitNodes* __restrict__ nodes,
                                                     const double* __restrict__ rx,
                                                     const double* __restrict__ ry,
                                                     const double* __restrict__ rz, int nrec,
                                                     int parts) {
  const int e = blockIdx.x / (parts + 1), q = blockIdx.x % (parts + 1) - 1;
  const MisfitDesc& s = d[e];
  if (q < 0) {
    misfit_seeds<T>(s, nodes[e], rx, ry, rz, nrec);
    return;
  }
  if (!s.grad_u) return;
  const int64_t N = (int64_t)s.m * s.n * s.l;
  fill_part((T*)s.grad_u, part_begin<T>(N, q, parts), part_begin<T>(N, q + 1, parts), T(0));
}

template <typename T>
__global__ void __launch_bounds__(256) misfit_nodes_kernel(const MisfitDesc* __restrict__ d,
                                                           const MisfitNodes* __restrict__ nodes,
                                                           const double* __restrict__ rx,
                                                           const double* __restrict__ ry,
                                                           const double* __restrict__ rz, int parts) {
  const int e = blockIdx.x / parts;
  misfit_nodes<T>(d[e], nodes[e], rx, ry, rz, (int)((blockIdx.x % parts) * 256 + threadIdx.x),
                  parts * 256);
}

// ------------------------------------------------ model parametrisation ---

// fvar = 2 sigmoid(x) - 1 + vel0, f = 1 / fvar (scripts/inversion.jl:42-43,61).
template <typename T>
__global__ void model_kernel(const T* __restrict__ x, const T* __restrict__ vel0, int64_t N,
                             T* __restrict__ fvar, T* __restrict__ f) {
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (int64_t)gridDim.x * blockDim.x) {
    const T sg = T(1) / (T(1) + (T)exp(-(double)x[p]));
    const T v = T(2) * sg - T(1) + vel0[p];
    fvar[p] = v;
    if (f) f[p] = T(1) / v;
  }
}

// out = sum over k of in[k] (fixed order), e.g. dL/df over the stations; the
// arrays are tab's, or more's where they are too many for it.  Bound by the reads
// (32 arrays of 200x200x80 FP64: 216 us, 3.8 TB/s; 16-byte loads, more of them in
// flight or larger pieces of each array at a time gave 222-230).
template <typename T, bool MORE>
__global__ void __launch_bounds__(256) sum_arrays_kernel(ArrayTable tab, const void* const* more,
                                                         int nin, int64_t N, T* out) {
  auto in = [&](int k) { return (gptr<const T>)(MORE ? ((gptr<const void* const>)more)[k] : tab.a[k]); };
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (int64_t)gridDim.x * blockDim.x) {
    T s = in(0)[p];
    for (int k = 1; k < nin; ++k) s = s + in(k)[p];
    out[p] = s;
  }
}

// Box mean of a over a (2*rh+1)^2 x (2*rv+1) window with periodic wrap (the
// padded VALID conv3d of scripts/inversion.jl:107-118): calls
// f(node, its value, its mean) for the nodes that the thread takes.
__device__ __forceinline__ int wrap(int x, int ext) { return x < 0 ? x + ext : x >= ext ? x - ext : x; }

template <typename T, typename F>
__device__ __forceinline__ void box_means(const T* __restrict__ a, int m, int n, int l, int rh,
                                          int rv, T wgt, F f) {
  const int64_t N = (int64_t)m * n * l;
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = p / l;
    const int k = (int)(p - r * l), i = (int)(r / n), j = (int)(r - (int64_t)i * n);
    T s = T(0);
    for (int di = -rh; di <= rh; ++di) {
      for (int dj = -rh; dj <= rh; ++dj) {
        const T* const row = a + ((int64_t)wrap(i + di, m) * n + wrap(j + dj, n)) * l;
        for (int dk = -rv; dk <= rv; ++dk) s = s + wgt * row[wrap(k + dk, l)];
      }
    }
    f(p, a[p], s);
  }
}

// The 3x3x3 window: a thread takes kRun nodes along i and keeps the weighted
// values of three planes, so that each node loads nine and not 27.
constexpr int kRun = 8;
template <typename T, typename F>
__device__ __forceinline__ void box3_means(const T* __restrict__ a, int m, int n, int l, T wgt, F f) {
  const int64_t nl = (int64_t)n * l, all = (m + kRun - 1) / kRun * nl;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < all;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int i0 = (int)(q / nl) * kRun;
    const int64_t jk = q % nl;
    const int j = (int)(jk / l), k = (int)(jk - (int64_t)j * l);
    int64_t off[9];
#pragma unroll
    for (int c = 0; c < 9; ++c)
      off[c] = (int64_t)wrap(j + c / 3 - 1, n) * l + wrap(k + c % 3 - 1, l);
    T x[kRun + 2][9], mid[kRun + 2];
#pragma unroll
    for (int t = 0; t < kRun + 2; ++t) {
      const int i = i0 + t - 1;
      const T* const pl = a + (i <= m ? (int64_t)wrap(i, m) : 0) * nl;
#pragma unroll
      for (int c = 0; c < 9; ++c) {
        const T v = pl[off[c]];
        mid[t] = c == 4 ? v : mid[t];
        x[t][c] = wgt * v;
      }
      if (t < 2 || i - 1 >= m) continue;
      T s = T(0);
#pragma unroll
      for (int c = 0; c < 27; ++c) s = s + x[t - 2 + c / 9][c % 9];
      f((int64_t)(i - 1) * nl + jk, mid[t - 1], s);
    }
  }
}

template <typename T, int R, typename F>
__device__ __forceinline__ void windows(const T* __restrict__ a, int m, int n, int l, int rh, int rv,
                                        T wgt, F f) {
  if constexpr (R == 1)
    box3_means<T>(a, m, n, l, wgt, f);
  else
    box_means<T>(a, m, n, l, rh, rv, wgt, f);
}

// Sum over the 256 threads of a workgroup (fixed tree order), on thread 0.
template <typename T>
__device__ __forceinline__ T tree_sum(T x, T* part) {
  part[threadIdx.x] = x;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) part[threadIdx.x] = part[threadIdx.x] + part[threadIdx.x + off];
    __syncthreads();
  }
  return part[0];
}
// Sum of x[0..cnt) by one workgroup of 256 threads, on thread 0.
template <typename T>
__device__ __forceinline__ T sum_list(const T* __restrict__ x, int cnt, T* part) {
  T s = T(0);
  for (int b = threadIdx.x; b < cnt; b += 256) s = s + x[b];
  return tree_sum(s, part);
}

// Pass 1: d = fvar - box(fvar); sgn = sign(d); partial sums of |d| per block.
// Bound by the window's loads from the caches: with 27 of them a node and 64-bit
// remainders for the coordinates the 3x3x3 window took 94 us on 200x200x80 FP64;
// nine a node (box3_means) take 32.
template <typename T, int R>
__global__ void __launch_bounds__(256) smooth_pass1_kernel(const T* __restrict__ fvar, int m,
                                                           int n, int l, int rh, int rv, T wgt,
                                                           T* __restrict__ sgn,
                                                           T* __restrict__ partial) {
  __shared__ T part[256];
  T acc = T(0);
  windows<T, R>(fvar, m, n, l, rh, rv, wgt, [&](int64_t p, T v, T mean) {
    const T dv = v - mean;
    acc = acc + (dv < T(0) ? -dv : dv);
    sgn[p] = dv > T(0) ? T(1) : (dv < T(0) ? T(-1) : T(0));
  });
  const T s = tree_sum(acc, part);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// Pass 2: grad_fvar = lambda (sgn - box(sgn)) (the box with periodic wrap
// and a symmetric window is its own adjoint); value = lambda * sum(partial),
// by the first workgroup (one thread's serial sum of 4096 took most of 248 us;
// the pass now takes 25 us).
template <typename T, int R>
__global__ void __launch_bounds__(256) smooth_pass2_kernel(const T* __restrict__ sgn, int m,
                                                           int n, int l, int rh, int rv, T wgt,
                                                           T lambda, T* __restrict__ grad,
                                                           const T* __restrict__ partial,
                                                           int npart, T* __restrict__ value) {
  __shared__ T part[256];
  if (blockIdx.x == 0 && value) {
    const T s = sum_list(partial, npart, part);
    if (threadIdx.x == 0) *value = lambda * s;
  }
  if (!grad) return;  // value only
  windows<T, R>(sgn, m, n, l, rh, rv, wgt,
                [&](int64_t p, T v, T mean) { grad[p] = lambda * (v - mean); });
}

// grad_x = (grad_fvar - grad_f / fvar^2) * 2 sigmoid(x) (1 - sigmoid(x)):
// the chain rule through f = 1/fvar and fvar = 2 sigmoid(x) - 1 + vel0.
template <typename T>
__global__ void model_grad_kernel(const T* __restrict__ x, const T* __restrict__ fvar,
                                  const T* __restrict__ grad_f, const T* __restrict__ grad_fvar,
                                  int64_t N, T* __restrict__ grad_x) {
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (int64_t)gridDim.x * blockDim.x) {
    const T sg = T(1) / (T(1) + (T)exp(-(double)x[p]));
    T gv = grad_fvar ? grad_fvar[p] : T(0);
    if (grad_f) gv = gv - grad_f[p] / (fvar[p] * fvar[p]);
    grad_x[p] = gv * (T(2) * sg * (T(1) - sg));
  }
}

// f_s = scale / fvar: the S-wave slowness pvs ./ fvar of
// scripts/inversion_joint.jl:79 (one division, as written there).
template <typename T>
__global__ void slowness_kernel(const T* __restrict__ fvar, int64_t N, T scale,
                                T* __restrict__ f_s) {
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (int64_t)gridDim.x * blockDim.x)
    f_s[p] = scale / fvar[p];
}

// Adjoint of f_s = scale / fvar: grad_fvar += -scale grad_fs / fvar^2, and
// per-block partial sums of d/dscale = sum grad_fs / fvar (fixed tree order).
template <typename T>
__global__ void __launch_bounds__(256) slowness_grad_kernel(const T* __restrict__ fvar, int64_t N,
                                                            T scale, const T* __restrict__ grad_fs,
                                                            T* __restrict__ grad_fvar,
                                                            T* __restrict__ partial) {
  __shared__ T part[256];
  T acc = T(0);
  for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < N;
       p += (int64_t)gridDim.x * blockDim.x) {
    const T v = fvar[p], g = grad_fs[p];
    if (grad_fvar) grad_fvar[p] = grad_fvar[p] - scale * g / (v * v);
    acc = acc + g / v;
  }
  const T s = tree_sum(acc, part);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// out = sum of partial[0..npart) by one workgroup of 256 threads (one thread
// took 237 us for 4096).
template <typename T>
__global__ void __launch_bounds__(256) sum_partials_kernel(const T* __restrict__ partial, int npart,
                                                           T* __restrict__ out) {
  __shared__ T part[256];
  const T s = sum_list(partial, npart, part);
  if (threadIdx.x == 0) *out = s;
}

#define ADT_SMOOTH_INSTANTIATE(T, R)                                                               \
  template __global__ void smooth_pass1_kernel<T, R>(const T*, int, int, int, int, int, T, T*, T*); \
  template __global__ void smooth_pass2_kernel<T, R>(const T*, int, int, int, int, int, T, T, T*,   \
                                                     const T*, int, T*);
#define ADT_OBJ_INSTANTIATE(T)                                                                    \
  template __global__ void source_u0_kernel<T>(SourceTable, const T*, int, int, int, T, int);      \
  template __global__ void misfit_kernel<T>(const MisfitDesc*, const MisfitNodes*, const double*, \
                                            const double*, const double*, int, int);              \
  template __global__ void misfit_nodes_kernel<T>(const MisfitDesc*, const MisfitNodes*,          \
                                                  const double*, const double*, const double*, int); \
  template __global__ void model_kernel<T>(const T*, const T*, int64_t, T*, T*);                 \
  template __global__ void sum_arrays_kernel<T, false>(ArrayTable, const void* const*, int, int64_t, T*); \
  template __global__ void sum_arrays_kernel<T, true>(ArrayTable, const void* const*, int, int64_t, T*);  \
  ADT_SMOOTH_INSTANTIATE(T, 0) ADT_SMOOTH_INSTANTIATE(T, 1)                                      \
  template __global__ void slowness_kernel<T>(const T*, int64_t, T, T*);                         \
  template __global__ void slowness_grad_kernel<T>(const T*, int64_t, T, const T*, T*, T*);       \
  template __global__ void sum_partials_kernel<T>(const T*, int, T*);                            \
  template __global__ void model_grad_kernel<T>(const T*, const T*, const T*, const T*, int64_t, \
                                                T*);

ADT_OBJ_INSTANTIATE(double)
ADT_OBJ_INSTANTIATE(float)

}  // namespace adt
