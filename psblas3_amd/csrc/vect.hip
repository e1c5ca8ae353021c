// Device multivectors and the BLAS-1 vector path.
// Replaces cuda/vectordev.c, cuda/dvectordev.c, cuda/svectordev.c,
// cuda/ivectordev.c and the SPGPU BLAS-1 kernels (cuda/spgpu/kernels/
// daxpby.cu, dupd_xyz.cu, dxyzw.cu, axy_base.cuh, ddot.cu, dnrm2.cu,
// amax_base.cuh, asum_base.cuh, abs_base.cuh, scal_base.cuh,
// setscal_base.cuh, gath_base.cuh, scat_base.cuh).
//
// Elementwise kernels evaluate exactly the expressions of the CPU routines
// (psi_daxpbyv, psi_d_upd_xyz, psi_dxyzw, d_base_mlt_a_2) with contraction
// off, so their results are bit-identical to the CPU path.  Reductions keep
// partial sums on the device (DPP wave sums, one last-block pass); the kernel
// stores the scalar in pinned host memory and the host synchronises.
#include <math.h>
#include <string.h>

#include "psb_hip_internal.hpp"

#pragma clang fp contract(off)

namespace psbhip {

// ------------------------------------------------------------------ kernels
template <typename T>
__global__ __launch_bounds__(kBlock) void k_setscal(T* __restrict__ x, int64_t first, int64_t n,
                                                    T val) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    x[first + i] = val;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scal(T* __restrict__ x, int64_t n, T alpha) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    x[i] = alpha * x[i];
}

// Vectors of V entries (16 bytes where aligned, else single entries) walked
// grid-stride, two per thread in flight: BODY(vector indexes, whether there
// are two) for n / V of them, TAIL(entry index) for the rest.  FP64 axpbyz of
// 8M entries 35.1 -> 32.5 us (5.9 TB/s), the element product 32.0 -> 31.0 us.
#define PSB_WALK(V, N, BODY, TAIL)                                                      \
  {                                                                                     \
    const int nv_ = (N) / (V), st_ = gridDim.x * kBlock;                                \
    int k_ = blockIdx.x * kBlock + threadIdx.x;                                         \
    for (; k_ + (int64_t)st_ < nv_; k_ += 2 * st_) BODY(k_, k_ + st_, true)             \
    if (k_ < nv_) BODY(k_, k_, false)                                                   \
    if ((V) > 1 && blockIdx.x == 0)                                                     \
      for (int i_ = nv_ * (V) + threadIdx.x; i_ < (N); i_ += kBlock) TAIL(i_)           \
  }

// psi_daxpbyv: mode selects the branch of the CPU routine so that y is not
// read when beta == 0 and the single-term cases are a single product.
// z may alias y (axpby) or be a third vector (axpbyz).
template <typename T>
__device__ __forceinline__ T axpby1(T alpha, T xi, T beta, T yi) {
  if (alpha == T(0)) return (beta == T(0)) ? T(0) : (beta == T(1) ? yi : beta * yi);
  if (beta == T(0)) return (alpha == T(1)) ? xi : alpha * xi;
  return alpha * xi + beta * yi;
}
template <typename T, int V>
__global__ __launch_bounds__(kBlock) void k_axpby(int n, int pitch_x, int pitch_y, int pitch_z,
                                                  T alpha, const T* __restrict__ x, T beta,
                                                  const T* y, T* z) {
  typedef T vec __attribute__((ext_vector_type(V)));
  const int c = blockIdx.y;
  x += (int64_t)c * pitch_x;
  y += (int64_t)c * pitch_y;
  z += (int64_t)c * pitch_z;
  const bool rx = alpha != T(0), ry = beta != T(0);
  const vec* xp = reinterpret_cast<const vec*>(x);
  const vec* yp = reinterpret_cast<const vec*>(y);
  vec* zp = reinterpret_cast<vec*>(z);
#define PSB_BODY(A, B, TWO)                                                             \
  {                                                                                     \
    const vec x0 = rx ? xp[A] : vec(T(0)), x1 = rx ? xp[B] : vec(T(0));                 \
    const vec y0 = ry ? yp[A] : vec(T(0)), y1 = ry ? yp[B] : vec(T(0));                 \
    vec r0, r1;                                                                         \
    _Pragma("unroll") for (int e = 0; e < V; e++) {                                     \
      r0[e] = axpby1<T>(alpha, x0[e], beta, y0[e]);                                     \
      r1[e] = axpby1<T>(alpha, x1[e], beta, y1[e]);                                     \
    }                                                                                   \
    zp[A] = r0;                                                                         \
    if (TWO) zp[B] = r1;                                                                \
  }
#define PSB_TAIL(I) z[I] = axpby1<T>(alpha, rx ? x[I] : T(0), beta, ry ? y[I] : T(0));
  PSB_WALK(V, n, PSB_BODY, PSB_TAIL)
#undef PSB_BODY
#undef PSB_TAIL
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_upd_xyz(int n, T alpha, T beta, T gamma, T delta,
                                                    const T* __restrict__ x, T* __restrict__ y,
                                                    T* __restrict__ z) {
  const bool g = gamma != T(0) && !(alpha == T(0) && beta == T(0));
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    T yy;
    if (alpha != T(0) && beta != T(0)) yy = alpha * x[i] + beta * y[i];
    else if (alpha != T(0)) yy = alpha * x[i];
    else if (beta != T(0)) yy = beta * y[i];
    else yy = T(0);
    y[i] = yy;
    T zz;
    if (g && delta != T(0)) zz = gamma * yy + delta * z[i];
    else if (g) zz = gamma * yy;
    else if (delta != T(0)) zz = delta * z[i];
    else zz = T(0);
    z[i] = zz;
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_xyzw(int n, T a, T b, T c, T d, T e, T f,
                                                 const T* __restrict__ x, T* __restrict__ y,
                                                 T* __restrict__ z, T* __restrict__ w) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    T yy = a * x[i] + b * y[i];
    T zz = c * yy + d * z[i];
    T ww = e * zz + f * w[i];
    y[i] = yy;
    z[i] = zz;
    w[i] = ww;
  }
}

// d_base_mlt_a_2: z = alpha*y*x + beta*z with the CPU's branch structure.
template <typename T>
__device__ __forceinline__ T axybz1(T alpha, T xi, T yi, T beta, T zi) {
  if (alpha == T(0)) return beta != T(1) ? beta * zi : zi;
  if (alpha == T(1)) {
    if (beta == T(0)) return yi * xi;
    if (beta == T(1)) return zi + yi * xi;
    return beta * zi + yi * xi;
  }
  if (alpha == T(-1)) {
    if (beta == T(0)) return -yi * xi;
    if (beta == T(1)) return zi - yi * xi;
    return beta * zi - yi * xi;
  }
  if (beta == T(0)) return alpha * yi * xi;
  if (beta == T(1)) return zi + alpha * yi * xi;
  return beta * zi + alpha * yi * xi;
}
template <typename T, int V>
__global__ __launch_bounds__(kBlock) void k_axybz(int n, T alpha, const T* __restrict__ x,
                                                  const T* y, T beta, T* z) {
  typedef T vec __attribute__((ext_vector_type(V)));
  // as the CPU: alpha = 0 reads neither x nor y and always reads z, else z
  // only when beta is not 0; alpha = 0, beta = 1 leaves z alone
  const bool rxy = alpha != T(0), rz = beta != T(0) || !rxy;
  if (!rxy && beta == T(1)) return;
  const vec* xp = reinterpret_cast<const vec*>(x);
  const vec* yp = reinterpret_cast<const vec*>(y);
  vec* zp = reinterpret_cast<vec*>(z);
#define PSB_BODY(A, B, TWO)                                                             \
  {                                                                                     \
    const vec x0 = rxy ? xp[A] : vec(T(0)), x1 = rxy ? xp[B] : vec(T(0));               \
    const vec y0 = rxy ? yp[A] : vec(T(0)), y1 = rxy ? yp[B] : vec(T(0));               \
    const vec z0 = rz ? zp[A] : vec(T(0)), z1 = rz ? zp[B] : vec(T(0));                 \
    vec r0, r1;                                                                         \
    _Pragma("unroll") for (int e = 0; e < V; e++) {                                     \
      r0[e] = axybz1<T>(alpha, x0[e], y0[e], beta, z0[e]);                              \
      r1[e] = axybz1<T>(alpha, x1[e], y1[e], beta, z1[e]);                              \
    }                                                                                   \
    zp[A] = r0;                                                                         \
    if (TWO) zp[B] = r1;                                                                \
  }
#define PSB_TAIL(I)                                                                     \
  z[I] = axybz1<T>(alpha, rxy ? x[I] : T(0), rxy ? y[I] : T(0), beta, rz ? z[I] : T(0));
  PSB_WALK(V, n, PSB_BODY, PSB_TAIL)
#undef PSB_BODY
#undef PSB_TAIL
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_diag_inv(int n, int size, T* d) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < size; i += gridDim.x * kBlock) {
    if (i < n) d[i] = (d[i] == T(0)) ? T(1) : T(1) / d[i];
    else d[i] = T(1);
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_abs(int n, T alpha, const T* x, T* y) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    y[i] = alpha * fabs(x[i]);
}

// Reductions.  op: 0 dot, 1 sum of squares, 2 max |x|, 3 sum |x|, 4 scaled
// sum of squares (x/scale)^2 with scale read from device memory.  Accumulated
// in FP64.  VEC: 16-byte loads, four vectors per input in flight and four
// sums per thread (both inputs 16-byte aligned, over 65536 entries); else a
// thread's entries in order.  Against entry by entry, a fence and one arrival
// counter: FP64 dot of 1M entries 16.4 -> 7.3 us, nrm2 14.6 -> 5.6 us, FP32 dot
// of 3M 27.4 -> 6.8 us.  Small sizes are bound by the arrivals and the tail over
// the partials.
template <typename T, int OP>
__device__ __forceinline__ void red_step(double& acc, T xi, T yi, double inv) {
  const double a = (double)xi;
  if (OP == 0) acc += a * (double)yi;
  else if (OP == 1) acc += a * a;
  else if (OP == 2) acc = fmax(acc, fabs(a));
  else if (OP == 3) acc += fabs(a);
  else { const double t = a * inv; acc += t * t; }
}

template <typename T, int OP, bool VEC>
__global__ __launch_bounds__(kBlock) void k_reduce(int n, const T* __restrict__ x,
                                                   const T* __restrict__ y,
                                                   const double* __restrict__ scale_p,
                                                   double* partials, unsigned int* counter,
                                                   double* result, double* host_result) {
  constexpr int V = VEC ? 16 / (int)sizeof(T) : 1, U = 4;
  const int stride = gridDim.x * kBlock, t0 = blockIdx.x * kBlock + threadIdx.x;
  double acc[U] = {};
  double inv = 1.0;
  if (OP == 4) inv = 1.0 / *scale_p;
  if constexpr (VEC) {
    const int nv = n / V;
    typedef T vec __attribute__((ext_vector_type(V)));
    int64_t k = t0;
    for (; k + (U - 1) * (int64_t)stride < nv; k += U * (int64_t)stride) {
      vec a[U], b[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        a[u] = reinterpret_cast<const vec*>(x)[k + u * (int64_t)stride];
        b[u] = OP == 0 ? reinterpret_cast<const vec*>(y)[k + u * (int64_t)stride] : a[u];
      }
#pragma unroll
      for (int u = 0; u < U; u++)
#pragma unroll
        for (int e = 0; e < V; e++) red_step<T, OP>(acc[u], a[u][e], b[u][e], inv);
    }
    for (; k < nv; k += stride) {
      const vec a = reinterpret_cast<const vec*>(x)[k];
      const vec b = OP == 0 ? reinterpret_cast<const vec*>(y)[k] : a;
#pragma unroll
      for (int e = 0; e < V; e++) red_step<T, OP>(acc[0], a[e], b[e], inv);
    }
    if (blockIdx.x == 0)
      for (int i = nv * V + threadIdx.x; i < n; i += kBlock)
        red_step<T, OP>(acc[1], x[i], y[i], inv);
  } else {
    // one sum in entry order; eight loads (red_grid's entries a thread) on their
    // way at a time, the last ones past the end at the last entry
    constexpr int G = 8;
    for (int64_t k = t0; k < n; k += G * (int64_t)stride) {
      T a[G], b[G];
#pragma unroll
      for (int u = 0; u < G; u++) {
        const int64_t i = k + u * (int64_t)stride < n ? k + u * (int64_t)stride : n - 1;
        a[u] = x[i];
        b[u] = OP == 0 ? y[i] : a[u];
      }
#pragma unroll
      for (int u = 0; u < G; u++)
        if (k + u * (int64_t)stride < n) red_step<T, OP>(acc[0], a[u], b[u], inv);
    }
  }
  if (OP == 2)
    grid_reduce<true>(fmax(fmax(acc[0], acc[1]), fmax(acc[2], acc[3])), partials, counter, result,
                      host_result);
  else
    grid_reduce<false>((acc[0] + acc[1]) + (acc[2] + acc[3]), partials, counter, result,
                       host_result);
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_gath(int n, const int* __restrict__ idx, int base,
                                                 const T* __restrict__ x, T* __restrict__ out) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    out[i] = x[idx[i] - base];
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_scat(int n, const int* __restrict__ idx, int base,
                                                 const T* __restrict__ in, T beta, T* x) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    int j = idx[i] - base;
    x[j] = (beta == T(0)) ? in[i] : beta * x[j] + in[i];
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_ins_add(int n, const int* __restrict__ idx, int base,
                                                    const T* __restrict__ in, T* x) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
    atomicAdd(&x[idx[i] - base], in[i]);
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

__global__ __launch_bounds__(kBlock) void k_fill_uniform(double* x, int64_t n, uint64_t key) {
  for (int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock) {
    uint64_t h = mix64(key ^ (uint64_t)i);
    x[i] = 2.0 * ((double)(h >> 11) * 0x1.0p-53) - 1.0;
  }
}

// ------------------------------------------------------------------ host helpers
static inline MultiVec* MV(void* p) { return static_cast<MultiVec*>(p); }

static int check_pair(const MultiVec* a, const MultiVec* b, int n) {
  if (!a || !b) return PSB_HIP_INVALID;
  if (n > a->size || n > b->size) return PSB_HIP_UNSUPPORTED;
  if (a->elem_type != b->elem_type) return PSB_HIP_INVALID;
  return PSB_HIP_SUCCESS;
}

// Run one grid reduction and leave the scalar in red_result[slot] and
// host_result[slot].
template <typename T, int OP>
static int launch_reduce(int n, const T* x, const T* y, const double* scale_p, int slot) {
  Context& c = ctx();
  int g = red_grid(n);
  // Up to 65536 entries (32 blocks) the arrivals bound both forms alike (a CG
  // step's vector operations at 4096 34.2-35.0 us, at 65536 34.8-35.6, either
  // way), and single loads keep a thread's entries in one sum in order.
  const bool vec = n > 65536 &&
      ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
  if (vec)
    hipLaunchKernelGGL((k_reduce<T, OP, true>), dim3(g), dim3(kBlock), 0, c.stream, n, x, y,
                       scale_p, c.red_partials, c.red_counter + (size_t)slot * kRedCounter, c.red_result + slot,
                       c.host_result + slot);
  else
    hipLaunchKernelGGL((k_reduce<T, OP, false>), dim3(g), dim3(kBlock), 0, c.stream, n, x, y,
                       scale_p, c.red_partials, c.red_counter + (size_t)slot * kRedCounter, c.red_result + slot,
                       c.host_result + slot);
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

// The results of the reductions launched into slots 0 .. nslots-1.  A call that
// returns a host scalar synchronises: a dot of 4096 entries takes 15.0 us, of
// which the end of the kernel and its signal are 5.5 (read as soon as the slot
// changes, while the stream is still busy, it took 9.5; a copy back before the
// synchronisation takes 7 more).
static int fetch_results(int nslots, double* out) {
  Context& c = ctx();
  PSB_HIP_CHECK(hipStreamSynchronize(c.stream));
  memcpy(out, c.host_result, sizeof(double) * nslots);
  return check_waits("reduction");
}

// Slots of one batch of column reductions (host_result and red_result hold 64).
constexpr int kRedSlots = 32;

// op OP over the first n entries of cols columns of x (and y), all columns
// of a batch launched before the first result is waited for.
template <typename T, int OP>
static int reduce_cols(double* res, int n, int cols, const MultiVec* x, const MultiVec* y) {
  for (int c0 = 0; c0 < cols; c0 += kRedSlots) {
    const int nc = cols - c0 < kRedSlots ? cols - c0 : kRedSlots;
    for (int c = 0; c < nc; c++) {
      const int rc = launch_reduce<T, OP>(n, (const T*)x->v + (int64_t)(c0 + c) * x->pitch,
                                          (const T*)y->v + (int64_t)(c0 + c) * y->pitch, nullptr,
                                          c);
      if (rc) return rc;
    }
    const int rc = fetch_results(nc, res + c0);
    if (rc) return rc;
  }
  return PSB_HIP_SUCCESS;
}

template <int OP>
static int reduce_any(double* res, int n, int cols, const MultiVec* x, const MultiVec* y) {
  if (n <= 0) {
    for (int c = 0; c < cols; c++) res[c] = 0.0;
    return PSB_HIP_SUCCESS;
  }
  if (x->elem_type == PSB_HIP_TYPE_DOUBLE) return reduce_cols<double, OP>(res, n, cols, x, y);
  if (x->elem_type == PSB_HIP_TYPE_FLOAT) return reduce_cols<float, OP>(res, n, cols, x, y);
  return PSB_HIP_UNSUPPORTED;
}

// the scaled nrm2 of one column, for a sum of squares that over- or underflowed
template <typename T>
static int nrm2_scaled(int n, const T* x, double* res) {
  int rc = launch_reduce<T, 2>(n, x, x, nullptr, 0);
  if (rc) return rc;
  rc = launch_reduce<T, 4>(n, x, x, ctx().red_result, 1);
  if (rc) return rc;
  double r[2];
  rc = fetch_results(2, r);
  if (rc) return rc;
  *res = r[0] == 0.0 ? 0.0 : r[0] * sqrt(r[1]);
  return PSB_HIP_SUCCESS;
}

template <typename T>
static int setscal_impl(T val, int first, int last, int index_base, void* x) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  int64_t f = first - index_base, n = (int64_t)last - first + 1;
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (f < 0 || f + n > (int64_t)v->pitch * v->count) return PSB_HIP_UNSUPPORTED;
  hipLaunchKernelGGL((k_setscal<T>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream,
                     (T*)v->v, f, n, val);
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

template <int OP>
static int simple_reduce(double* res, int n, void* x) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  if (n > v->size) return PSB_HIP_UNSUPPORTED;
  return reduce_any<OP>(res, n, v->count, v, v);
}

// whether 16-byte accesses to every column of these vectors are aligned
template <typename T>
static bool vec16(const void* p, int64_t pitch, int cols) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && (cols <= 1 || pitch * sizeof(T) % 16 == 0);
}

}  // namespace psbhip

using namespace psbhip;


extern "C" {

int psb_hip_mv_alloc(void** mv, int count, int size, int elem_type) {
  PSB_ENSURE_INIT();
  *mv = nullptr;
  size_t es = elem_size(elem_type);
  if (es == 0 || count < 1 || size < 0) return set_error(PSB_HIP_UNSUPPORTED, __func__, "bad args");
  MultiVec* v = new MultiVec;
  v->count = count;
  v->size = size;
  v->elem_type = elem_type;
  // cuda/vectordev.c:83-145: pitch = size for one column, else 256-byte rows
  v->pitch = (count == 1) ? size : (int)((((size_t)size * es + 255) / 256) * 256 / es);
  size_t bytes = (size_t)v->pitch * count * es;
  if (bytes == 0) bytes = 256;
  hipError_t e = hipMalloc(&v->v, bytes);
  if (e != hipSuccess) {
    delete v;
    return set_error(PSB_HIP_OUTOFMEM, __func__, hipGetErrorString(e));
  }
  *mv = v;
  return PSB_HIP_SUCCESS;
}

void psb_hip_mv_free(void* mv) {
  if (!mv) return;
  MultiVec* v = MV(mv);
  if (ctx().initialized) hipStreamSynchronize(ctx().stream);
  hipFree(v->v);
  delete v;
}

int psb_hip_mv_size(void* mv) { return mv ? MV(mv)->size : -1; }
int psb_hip_mv_count(void* mv) { return mv ? MV(mv)->count : -1; }
int psb_hip_mv_pitch(void* mv) { return mv ? MV(mv)->pitch : -1; }
void* psb_hip_mv_data(void* mv) { return mv ? MV(mv)->v : nullptr; }

int psb_hip_mv_write_r2(void* mv, const void* host, int ld) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(mv);
  size_t es = elem_size(v->elem_type);
  if (v->size == 0) return PSB_HIP_SUCCESS;
  PSB_HIP_CHECK(hipMemcpy2DAsync(v->v, (size_t)v->pitch * es, host, (size_t)ld * es,
                                 (size_t)v->size * es, (size_t)v->count, hipMemcpyHostToDevice,
                                 ctx().stream));
  PSB_HIP_CHECK(hipStreamSynchronize(ctx().stream));
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_read_r2(void* mv, void* host, int ld) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(mv);
  size_t es = elem_size(v->elem_type);
  if (v->size == 0) return PSB_HIP_SUCCESS;
  PSB_HIP_CHECK(hipMemcpy2DAsync(host, (size_t)ld * es, v->v, (size_t)v->pitch * es,
                                 (size_t)v->size * es, (size_t)v->count, hipMemcpyDeviceToHost,
                                 ctx().stream));
  PSB_HIP_CHECK(hipStreamSynchronize(ctx().stream));
  return check_waits(__func__);
}

int psb_hip_mv_write(void* mv, const void* host) { return psb_hip_mv_write_r2(mv, host, MV(mv)->size); }
int psb_hip_mv_read(void* mv, void* host) { return psb_hip_mv_read_r2(mv, host, MV(mv)->size); }

int psb_hip_mv_write_first(void* mv, int first, int n, const void* host) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(mv);
  if (first < 1 || n < 0 || first - 1 + n > v->size) return PSB_HIP_UNSUPPORTED;
  size_t es = elem_size(v->elem_type);
  if (n == 0) return PSB_HIP_SUCCESS;
  PSB_HIP_CHECK(hipMemcpyAsync((char*)v->v + (size_t)(first - 1) * es, host, (size_t)n * es,
                               hipMemcpyHostToDevice, ctx().stream));
  PSB_HIP_CHECK(hipStreamSynchronize(ctx().stream));
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_read_first(void* mv, int first, int n, void* host) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(mv);
  if (first < 1 || n < 0 || first - 1 + n > v->size) return PSB_HIP_UNSUPPORTED;
  size_t es = elem_size(v->elem_type);
  if (n == 0) return PSB_HIP_SUCCESS;
  PSB_HIP_CHECK(hipMemcpyAsync(host, (char*)v->v + (size_t)(first - 1) * es, (size_t)n * es,
                               hipMemcpyDeviceToHost, ctx().stream));
  PSB_HIP_CHECK(hipStreamSynchronize(ctx().stream));
  return check_waits(__func__);
}

int psb_hip_mv_setscal_d(double val, int first, int last, int index_base, void* x) {
  if (MV(x)->elem_type != PSB_HIP_TYPE_DOUBLE) return PSB_HIP_INVALID;
  return setscal_impl<double>(val, first, last, index_base, x);
}
int psb_hip_mv_setscal_s(float val, int first, int last, int index_base, void* x) {
  if (MV(x)->elem_type != PSB_HIP_TYPE_FLOAT) return PSB_HIP_INVALID;
  return setscal_impl<float>(val, first, last, index_base, x);
}
int psb_hip_mv_setscal_i(int val, int first, int last, int index_base, void* x) {
  if (MV(x)->elem_type != PSB_HIP_TYPE_INT) return PSB_HIP_INVALID;
  return setscal_impl<int>(val, first, last, index_base, x);
}

int psb_hip_mv_geins(int n, void* irl, void* val, int dupl, int index_base, void* x) {
  PSB_ENSURE_INIT();
  MultiVec *vi = MV(irl), *vv = MV(val), *vx = MV(x);
  if (n > vi->size || n > vv->size) return PSB_HIP_UNSUPPORTED;
  if (vi->elem_type != PSB_HIP_TYPE_INT || vv->elem_type != vx->elem_type) return PSB_HIP_INVALID;
  if (n <= 0) return PSB_HIP_SUCCESS;
  int g = stream_grid(n);
  if (vx->elem_type == PSB_HIP_TYPE_DOUBLE) {
    if (dupl == PSB_HIP_INS_ADD)
      hipLaunchKernelGGL((k_ins_add<double>), dim3(g), dim3(kBlock), 0, ctx().stream, n,
                         (const int*)vi->v, index_base, (const double*)vv->v, (double*)vx->v);
    else
      hipLaunchKernelGGL((k_scat<double>), dim3(g), dim3(kBlock), 0, ctx().stream, n,
                         (const int*)vi->v, index_base, (const double*)vv->v, 0.0,
                         (double*)vx->v);
  } else if (vx->elem_type == PSB_HIP_TYPE_FLOAT) {
    if (dupl == PSB_HIP_INS_ADD)
      hipLaunchKernelGGL((k_ins_add<float>), dim3(g), dim3(kBlock), 0, ctx().stream, n,
                         (const int*)vi->v, index_base, (const float*)vv->v, (float*)vx->v);
    else
      hipLaunchKernelGGL((k_scat<float>), dim3(g), dim3(kBlock), 0, ctx().stream, n,
                         (const int*)vi->v, index_base, (const float*)vv->v, 0.0f,
                         (float*)vx->v);
  } else {
    return PSB_HIP_UNSUPPORTED;
  }
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_igath(void* x, int vector_id, int n, int first, const int* didx, int hfirst,
                     void* dhv, int index_base) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (vector_id < 0 || vector_id >= v->count) return PSB_HIP_UNSUPPORTED;
  int g = stream_grid(n);
  const int* idx = didx + (first - index_base);
  if (v->elem_type == PSB_HIP_TYPE_DOUBLE) {
    double* hv = (double*)dhv + (hfirst - index_base);
    hipLaunchKernelGGL((k_gath<double>), dim3(g), dim3(kBlock), 0, ctx().stream, n, idx,
                       index_base, (const double*)v->v + (int64_t)vector_id * v->pitch, hv);
  } else if (v->elem_type == PSB_HIP_TYPE_FLOAT) {
    float* hv = (float*)dhv + (hfirst - index_base);
    hipLaunchKernelGGL((k_gath<float>), dim3(g), dim3(kBlock), 0, ctx().stream, n, idx,
                       index_base, (const float*)v->v + (int64_t)vector_id * v->pitch, hv);
  } else {
    int* hv = (int*)dhv + (hfirst - index_base);
    hipLaunchKernelGGL((k_gath<int>), dim3(g), dim3(kBlock), 0, ctx().stream, n, idx,
                       index_base, (const int*)v->v + (int64_t)vector_id * v->pitch, hv);
  }
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_iscat(void* x, int vector_id, int n, int first, const int* didx, int hfirst,
                     const void* dhv, int index_base, double beta) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (vector_id < 0 || vector_id >= v->count) return PSB_HIP_UNSUPPORTED;
  int g = stream_grid(n);
  const int* idx = didx + (first - index_base);
  if (v->elem_type == PSB_HIP_TYPE_DOUBLE) {
    const double* hv = (const double*)dhv + (hfirst - index_base);
    hipLaunchKernelGGL((k_scat<double>), dim3(g), dim3(kBlock), 0, ctx().stream, n, idx,
                       index_base, hv, beta, (double*)v->v + (int64_t)vector_id * v->pitch);
  } else if (v->elem_type == PSB_HIP_TYPE_FLOAT) {
    const float* hv = (const float*)dhv + (hfirst - index_base);
    hipLaunchKernelGGL((k_scat<float>), dim3(g), dim3(kBlock), 0, ctx().stream, n, idx,
                       index_base, hv, (float)beta, (float*)v->v + (int64_t)vector_id * v->pitch);
  } else {
    const int* hv = (const int*)dhv + (hfirst - index_base);
    hipLaunchKernelGGL((k_scat<int>), dim3(g), dim3(kBlock), 0, ctx().stream, n, idx,
                       index_base, hv, (int)beta, (int*)v->v + (int64_t)vector_id * v->pitch);
  }
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_scal(double alpha, void* x) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  int64_t n = (int64_t)v->pitch * v->count;
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (v->elem_type == PSB_HIP_TYPE_DOUBLE)
    hipLaunchKernelGGL((k_scal<double>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream,
                       (double*)v->v, n, alpha);
  else if (v->elem_type == PSB_HIP_TYPE_FLOAT)
    hipLaunchKernelGGL((k_scal<float>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream,
                       (float*)v->v, n, (float)alpha);
  else
    return PSB_HIP_UNSUPPORTED;
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_dot(double* res, int n, void* x, void* y) {
  PSB_ENSURE_INIT();
  MultiVec *vx = MV(x), *vy = MV(y);
  int rc = check_pair(vx, vy, n);
  if (rc) return rc;
  return reduce_any<0>(res, n, vx->count < vy->count ? vx->count : vy->count, vx, vy);
}

int psb_hip_mv_nrm2(double* res, int n, void* x) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  if (n > v->size) return PSB_HIP_UNSUPPORTED;
  int rc = reduce_any<1>(res, n, v->count, v, v);
  for (int c = 0; c < v->count && !rc && n > 0; c++) {
    // the unscaled sum of squares is exact enough unless it over/underflowed;
    // then rescale by max|x| (the scaled dnrm2 of the CPU path)
    if (isfinite(res[c]) && (res[c] == 0.0 || res[c] > 1e-280))
      res[c] = sqrt(res[c]);
    else if (v->elem_type == PSB_HIP_TYPE_DOUBLE)
      rc = nrm2_scaled<double>(n, (const double*)v->v + (int64_t)c * v->pitch, &res[c]);
    else
      rc = nrm2_scaled<float>(n, (const float*)v->v + (int64_t)c * v->pitch, &res[c]);
  }
  return rc;
}

int psb_hip_mv_amax(double* res, int n, void* x) { return simple_reduce<2>(res, n, x); }
int psb_hip_mv_asum(double* res, int n, void* x) { return simple_reduce<3>(res, n, x); }

int psb_hip_mv_axpbyz(int n, double alpha, void* x, double beta, void* y, void* z) {
  PSB_ENSURE_INIT();
  MultiVec *vx = MV(x), *vy = MV(y), *vz = MV(z);
  int rc = check_pair(vx, vy, n);
  if (rc) return rc;
  rc = check_pair(vy, vz, n);
  if (rc) return rc;
  if (n <= 0) return PSB_HIP_SUCCESS;
  int cols = vz->count;
  if (vx->count < cols || vy->count < cols) return PSB_HIP_UNSUPPORTED;
  dim3 grid(stream_grid(n), cols);
#define PSB_AXPBY(T, V)                                                                      \
  hipLaunchKernelGGL((k_axpby<T, V>), grid, dim3(kBlock), 0, ctx().stream, n, vx->pitch,     \
                     vy->pitch, vz->pitch, (T)alpha, (const T*)vx->v, (T)beta, (const T*)vy->v, \
                     (T*)vz->v)
#define PSB_ALIGNED(T)                                                            \
  (vec16<T>(vx->v, vx->pitch, cols) && vec16<T>(vy->v, vy->pitch, cols) &&        \
   vec16<T>(vz->v, vz->pitch, cols))
  if (vx->elem_type == PSB_HIP_TYPE_DOUBLE) {
    if (PSB_ALIGNED(double)) PSB_AXPBY(double, 2);
    else PSB_AXPBY(double, 1);
  } else if (vx->elem_type == PSB_HIP_TYPE_FLOAT) {
    if (PSB_ALIGNED(float)) PSB_AXPBY(float, 4);
    else PSB_AXPBY(float, 1);
  } else {
    return PSB_HIP_UNSUPPORTED;
  }
#undef PSB_AXPBY
#undef PSB_ALIGNED
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_axpby(int n, double alpha, void* x, double beta, void* y) {
  return psb_hip_mv_axpbyz(n, alpha, x, beta, y, y);
}

int psb_hip_mv_upd_xyz(int n, double alpha, double beta, double gamma, double delta, void* x,
                       void* y, void* z) {
  PSB_ENSURE_INIT();
  MultiVec *vx = MV(x), *vy = MV(y), *vz = MV(z);
  int rc = check_pair(vx, vy, n);
  if (rc) return rc;
  rc = check_pair(vy, vz, n);
  if (rc) return rc;
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (vx->elem_type == PSB_HIP_TYPE_DOUBLE)
    hipLaunchKernelGGL((k_upd_xyz<double>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream,
                       n, alpha, beta, gamma, delta, (const double*)vx->v, (double*)vy->v,
                       (double*)vz->v);
  else if (vx->elem_type == PSB_HIP_TYPE_FLOAT)
    hipLaunchKernelGGL((k_upd_xyz<float>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream,
                       n, (float)alpha, (float)beta, (float)gamma, (float)delta,
                       (const float*)vx->v, (float*)vy->v, (float*)vz->v);
  else
    return PSB_HIP_UNSUPPORTED;
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_xyzw(int n, double a, double b, double c, double d, double e, double f, void* x,
                    void* y, void* z, void* w) {
  PSB_ENSURE_INIT();
  MultiVec *vx = MV(x), *vy = MV(y), *vz = MV(z), *vw = MV(w);
  int rc = check_pair(vx, vy, n);
  if (rc) return rc;
  rc = check_pair(vz, vw, n);
  if (rc) return rc;
  // psi_dxyzw: all six coefficients must be non-zero, else nothing is done
  if (a == 0.0 || b == 0.0 || c == 0.0 || d == 0.0 || e == 0.0 || f == 0.0)
    return PSB_HIP_SUCCESS;
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (vx->elem_type == PSB_HIP_TYPE_DOUBLE)
    hipLaunchKernelGGL((k_xyzw<double>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream, n,
                       a, b, c, d, e, f, (const double*)vx->v, (double*)vy->v, (double*)vz->v,
                       (double*)vw->v);
  else if (vx->elem_type == PSB_HIP_TYPE_FLOAT)
    hipLaunchKernelGGL((k_xyzw<float>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream, n,
                       (float)a, (float)b, (float)c, (float)d, (float)e, (float)f,
                       (const float*)vx->v, (float*)vy->v, (float*)vz->v, (float*)vw->v);
  else
    return PSB_HIP_UNSUPPORTED;
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_axybz(int n, double alpha, void* x, void* y, double beta, void* z) {
  PSB_ENSURE_INIT();
  MultiVec *vx = MV(x), *vy = MV(y), *vz = MV(z);
  int rc = check_pair(vx, vy, n);
  if (rc) return rc;
  rc = check_pair(vy, vz, n);
  if (rc) return rc;
  if (n <= 0) return PSB_HIP_SUCCESS;
  // one column of x (the diagonal) against every column of y and z
  int cols = vz->count;
  if (vx->count != 1 && vx->count != cols) return PSB_HIP_UNSUPPORTED;
  if (vy->count < cols || vy->pitch != vz->pitch) return PSB_HIP_UNSUPPORTED;
  for (int c = 0; c < cols; c++) {
    int64_t ox = (vx->count == 1) ? 0 : (int64_t)c * vx->pitch;
    int64_t oy = (int64_t)c * vy->pitch;
#define PSB_AXYBZ(T, V)                                                                    \
  hipLaunchKernelGGL((k_axybz<T, V>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream, n, \
                     (T)alpha, (const T*)vx->v + ox, (const T*)vy->v + oy, (T)beta,        \
                     (T*)vz->v + oy)
#define PSB_ALIGNED(T)                                                               \
  (vec16<T>((const T*)vx->v + ox, 0, 1) && vec16<T>((const T*)vy->v + oy, 0, 1) &&   \
   vec16<T>((const T*)vz->v + oy, 0, 1))
    if (vx->elem_type == PSB_HIP_TYPE_DOUBLE) {
      if (PSB_ALIGNED(double)) PSB_AXYBZ(double, 2);
      else PSB_AXYBZ(double, 1);
    } else if (vx->elem_type == PSB_HIP_TYPE_FLOAT) {
      if (PSB_ALIGNED(float)) PSB_AXYBZ(float, 4);
      else PSB_AXYBZ(float, 1);
    } else {
      return PSB_HIP_UNSUPPORTED;
    }
#undef PSB_AXYBZ
#undef PSB_ALIGNED
    PSB_HIP_LAUNCH_CHECK();
  }
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_axy(int n, double alpha, void* x, void* y) {
  return psb_hip_mv_axybz(n, alpha, x, y, 0.0, y);
}

int psb_hip_mv_diag_inv(int n, void* dv) {
  PSB_ENSURE_INIT();
  MultiVec* d = MV(dv);
  if (n > d->size) return PSB_HIP_UNSUPPORTED;
  if (d->size <= 0) return PSB_HIP_SUCCESS;
  if (d->elem_type == PSB_HIP_TYPE_DOUBLE)
    hipLaunchKernelGGL((k_diag_inv<double>), dim3(stream_grid(d->size)), dim3(kBlock), 0,
                       ctx().stream, n, d->size, (double*)d->v);
  else if (d->elem_type == PSB_HIP_TYPE_FLOAT)
    hipLaunchKernelGGL((k_diag_inv<float>), dim3(stream_grid(d->size)), dim3(kBlock), 0,
                       ctx().stream, n, d->size, (float*)d->v);
  else
    return PSB_HIP_UNSUPPORTED;
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_abs(int n, double alpha, void* x, void* y) {
  PSB_ENSURE_INIT();
  MultiVec *vx = MV(x), *vy = MV(y);
  int rc = check_pair(vx, vy, n);
  if (rc) return rc;
  if (n <= 0) return PSB_HIP_SUCCESS;
  if (vx->elem_type == PSB_HIP_TYPE_DOUBLE)
    hipLaunchKernelGGL((k_abs<double>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream, n,
                       alpha, (const double*)vx->v, (double*)vy->v);
  else if (vx->elem_type == PSB_HIP_TYPE_FLOAT)
    hipLaunchKernelGGL((k_abs<float>), dim3(stream_grid(n)), dim3(kBlock), 0, ctx().stream, n,
                       (float)alpha, (const float*)vx->v, (float*)vy->v);
  else
    return PSB_HIP_UNSUPPORTED;
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_mv_fill_uniform(void* x, uint64_t seed, uint32_t stream) {
  PSB_ENSURE_INIT();
  MultiVec* v = MV(x);
  if (v->elem_type != PSB_HIP_TYPE_DOUBLE) return PSB_HIP_UNSUPPORTED;
  if (v->size <= 0) return PSB_HIP_SUCCESS;
  for (int c = 0; c < v->count; c++) {
    // same key derivation as the host fill (host.cpp); column c uses stream + c
    uint64_t z = seed * 0xD1B54A32D192ED03ULL ^ ((uint64_t)(stream + (uint32_t)c) << 48);
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    const uint64_t key = z ^ (z >> 31);
    hipLaunchKernelGGL(k_fill_uniform, dim3(stream_grid(v->size)), dim3(kBlock), 0, ctx().stream,
                       (double*)v->v + (int64_t)c * v->pitch, (int64_t)v->size, key);
    PSB_HIP_LAUNCH_CHECK();
  }
  return PSB_HIP_SUCCESS;
}

}  // extern "C"
