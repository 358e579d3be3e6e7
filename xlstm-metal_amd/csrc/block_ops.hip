// The element-wise stages of a block around its projections, as one pass each:
//
//  * add_rmsnorm_kernel: s = x + r (the residual add; r optional) and y = RMSNorm(s) = s / rms(s) * w in
//    float32, rounded once (the block's _RMSNorm: x.float(), the norm, the cast back), with up to two
//    float32 state buffers copied along.
//  * silu_mul_kernel: y = silu(g) u, the SiLU rounded to the dtype before the product (the SwiGLU's two
//    modules).
//
// Every rounding of the modules they replace is kept, so results change only where the order of the
// sum of squares moves the last bit of rms.  Both are streams (bytes: x, r in, s, y out; g, u in, y
// out); at one token per sequence they are bound by the launch, and what they save is launches: in the
// mixed stack's decode step (d 2048, 8 tokens, 8 blocks, HIP graph, kernel trace) a residual add, three
// casts and the norm took 18.7 us, add_rmsnorm_kernel takes 4.9; with the SwiGLU product (9.6 -> 4.8) and the
// gate projections unstacked (two weight copies and two slices, ~18 us) the step went 1297 -> 1027 us.
// One workgroup of 256 threads per row, the row in registers (NV 16-byte vectors per thread, all loads
// issued before the first use), a row longer than 256 x 8 x 4 values re-read for the second pass.
#include "common.h"

namespace xl {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int BO_BLOCK = 256;
constexpr int BO_NV_MAX = 4;

template <typename T>
union V8 {
  u32x4 raw;
  T e[8];
};

template <typename T>
__device__ __forceinline__ u32x4 to_vec(const float (&a)[8]) {
  V8<T> v;
#pragma unroll
  for (int j = 0; j < 8; ++j) v.e[j] = from_f32<T>(a[j]);
  return v.raw;
}

// s (or x) of vector vi: the sum is rounded to T, as the residual add's output is
template <typename T>
__device__ __forceinline__ u32x4 add_vec(u32x4 a, u32x4 b) {
  V8<T> x, r;
  x.raw = a;
  r.raw = b;
  float f[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = to_f32(x.e[j]) + to_f32(r.e[j]);
  return to_vec<T>(f);
}

struct StateCopy {
  const float* src[2];
  float* dst[2];
  int n[2];
};

template <typename T, int NV>
__global__ __launch_bounds__(BO_BLOCK) void add_rmsnorm_kernel(const T* __restrict__ x, const T* __restrict__ r,
                                                               const T* __restrict__ w, T* __restrict__ s,
                                                               T* __restrict__ y, int D, float eps, StateCopy cp) {
  __shared__ float s_part[BO_BLOCK / 64];
  const int tid = threadIdx.x, nvec = D >> 3;
  const size_t row = (size_t)blockIdx.x * D;
  V8<T> v[NV];
  float ss = 0.f;
  if constexpr (NV <= BO_NV_MAX) {
    u32x4 rv[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int at = 8 * min(tid + BO_BLOCK * k, nvec - 1);
      v[k].raw = *(const u32x4*)(x + row + at);
      rv[k] = *(const u32x4*)((r ? r : x) + row + at);
    }
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      if (r) v[k].raw = add_vec<T>(v[k].raw, rv[k]);
      if (tid + BO_BLOCK * k < nvec) {
#pragma unroll
        for (int j = 0; j < 8; ++j) ss = fmaf(to_f32(v[k].e[j]), to_f32(v[k].e[j]), ss);
        if (r) *(u32x4*)(s + row + 8 * (tid + BO_BLOCK * k)) = v[k].raw;
      }
    }
  } else {
    for (int vi = tid; vi < nvec; vi += BO_BLOCK) {
      V8<T> a;
      a.raw = *(const u32x4*)(x + row + 8 * vi);
      if (r) {
        a.raw = add_vec<T>(a.raw, *(const u32x4*)(r + row + 8 * vi));
        *(u32x4*)(s + row + 8 * vi) = a.raw;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ss = fmaf(to_f32(a.e[j]), to_f32(a.e[j]), ss);
    }
  }
  ss = lane_of(wave_sum_dpp(ss), 63);
  if ((tid & 63) == 0) s_part[tid >> 6] = ss;
  __syncthreads();
  const float tot = s_part[0] + s_part[1] + s_part[2] + s_part[3];
  const float rstd = 1.0f / sqrtf(tot / (float)D + eps);
  auto norm = [&](const V8<T>& a, int vi) {
    V8<T> wv;
    wv.raw = *(const u32x4*)(w + 8 * vi);
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) f[j] = to_f32(a.e[j]) * rstd * to_f32(wv.e[j]);
    *(u32x4*)(y + row + 8 * vi) = to_vec<T>(f);
  };
  if constexpr (NV <= BO_NV_MAX) {
#pragma unroll
    for (int k = 0; k < NV; ++k)
      if (tid + BO_BLOCK * k < nvec) norm(v[k], tid + BO_BLOCK * k);
  } else {
    for (int vi = tid; vi < nvec; vi += BO_BLOCK) {  // each thread re-reads the vectors it wrote
      V8<T> a;
      a.raw = *(const u32x4*)((r ? s : x) + row + 8 * vi);
      norm(a, vi);
    }
  }
#pragma unroll
  for (int c = 0; c < 2; ++c)
    for (int64_t e = (int64_t)blockIdx.x * BO_BLOCK + tid; e < cp.n[c]; e += (int64_t)gridDim.x * BO_BLOCK)
      cp.dst[c][e] = cp.src[c][e];
}

template <typename T>
__global__ __launch_bounds__(BO_BLOCK) void silu_mul_kernel(const T* __restrict__ g, const T* __restrict__ u,
                                                            T* __restrict__ y, int64_t nvec) {
  for (int64_t vi = (int64_t)blockIdx.x * BO_BLOCK + threadIdx.x; vi < nvec; vi += (int64_t)gridDim.x * BO_BLOCK) {
    V8<T> a, b;
    a.raw = *(const u32x4*)(g + 8 * vi);
    b.raw = *(const u32x4*)(u + 8 * vi);
    float f[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float z = to_f32(a.e[j]);
      f[j] = round_to<T>(z / (1.0f + expf(-z))) * to_f32(b.e[j]);
    }
    *(u32x4*)(y + 8 * vi) = to_vec<T>(f);
  }
}

template <typename T>
void launch_norm(const void* x, const void* r, const void* w, void* s, void* y, int M, int D, float eps,
                 const StateCopy& cp, hipStream_t st) {
  const int nv = (D / 8 + BO_BLOCK - 1) / BO_BLOCK;
  const dim3 grid((unsigned)M), blk(BO_BLOCK);
  const T *xp = (const T*)x, *rp = (const T*)r, *wp = (const T*)w;
  T *sp = (T*)s, *yp = (T*)y;
  switch (nv) {
    case 1: hipLaunchKernelGGL((add_rmsnorm_kernel<T, 1>), grid, blk, 0, st, xp, rp, wp, sp, yp, D, eps, cp); break;
    case 2: hipLaunchKernelGGL((add_rmsnorm_kernel<T, 2>), grid, blk, 0, st, xp, rp, wp, sp, yp, D, eps, cp); break;
    case 3:
    case 4: hipLaunchKernelGGL((add_rmsnorm_kernel<T, 4>), grid, blk, 0, st, xp, rp, wp, sp, yp, D, eps, cp); break;
    default: hipLaunchKernelGGL((add_rmsnorm_kernel<T, 5>), grid, blk, 0, st, xp, rp, wp, sp, yp, D, eps, cp); break;
  }
}

}  // namespace
}  // namespace xl

extern "C" int xl_add_rmsnorm_fwd(const void* x, const void* residual, const void* weight, void* sum, void* y, int M,
                                  int D, float eps, const float* copy_src0, float* copy_dst0, int ncopy0,
                                  const float* copy_src1, float* copy_dst1, int ncopy1, int dtype, void* stream) {
  using namespace xl;
  clear_error();
  const char* who = "xl_add_rmsnorm_fwd";
  if (M < 0 || D < 0 || ncopy0 < 0 || ncopy1 < 0) return set_error(XL_ERR_INVALID_ARG, "%s: negative size", who);
  if (!dtype_ok(dtype)) return set_error(XL_ERR_INVALID_ARG, "%s: unknown dtype %d", who, dtype);
  if (dtype == XL_DTYPE_F32 || D < 8 || D % 8 != 0)
    return set_error(XL_ERR_UNSUPPORTED, "%s: dtype %d, D=%d (16-bit rows of a positive multiple of 8)", who, dtype, D);
  if (M == 0 && ncopy0 == 0 && ncopy1 == 0) return XL_OK;
  if (M == 0) return set_error(XL_ERR_INVALID_ARG, "%s: state copies need at least one row", who);
  if (!x || !weight || !y || (residual && !sum) || (ncopy0 && (!copy_src0 || !copy_dst0)) ||
      (ncopy1 && (!copy_src1 || !copy_dst1)))
    return set_error(XL_ERR_INVALID_ARG, "%s: null pointer", who);
  if (((uintptr_t)x | (uintptr_t)residual | (uintptr_t)weight | (uintptr_t)sum | (uintptr_t)y) & 15u)
    return set_error(XL_ERR_INVALID_ARG, "%s: pointers must be 16-byte aligned", who);
  const StateCopy cp{{copy_src0, copy_src1}, {copy_dst0, copy_dst1}, {ncopy0, ncopy1}};
  if (dtype == XL_DTYPE_BF16)
    launch_norm<bf16_t>(x, residual, weight, sum, y, M, D, eps, cp, (hipStream_t)stream);
  else
    launch_norm<f16_t>(x, residual, weight, sum, y, M, D, eps, cp, (hipStream_t)stream);
  return check_launch(who);
}

extern "C" int xl_silu_mul_fwd(const void* gate, const void* up, void* y, int64_t numel, int dtype, void* stream) {
  using namespace xl;
  clear_error();
  const char* who = "xl_silu_mul_fwd";
  if (numel < 0) return set_error(XL_ERR_INVALID_ARG, "%s: negative size", who);
  if (!dtype_ok(dtype)) return set_error(XL_ERR_INVALID_ARG, "%s: unknown dtype %d", who, dtype);
  if (dtype == XL_DTYPE_F32 || numel % 8 != 0)
    return set_error(XL_ERR_UNSUPPORTED, "%s: dtype %d, numel %lld (a 16-bit dtype, a multiple of 8)", who, dtype,
                     (long long)numel);
  if (numel == 0) return XL_OK;
  if (!gate || !up || !y) return set_error(XL_ERR_INVALID_ARG, "%s: null pointer", who);
  if (((uintptr_t)gate | (uintptr_t)up | (uintptr_t)y) & 15u)
    return set_error(XL_ERR_INVALID_ARG, "%s: pointers must be 16-byte aligned", who);
  const int64_t nvec = numel / 8;
  int64_t blocks = (nvec + BO_BLOCK - 1) / BO_BLOCK;
  if (blocks > 8192) blocks = 8192;  // 32 workgroups per CU, each striding over the rest
  const dim3 grid((unsigned)blocks), blk(BO_BLOCK);
  hipStream_t st = (hipStream_t)stream;
  if (dtype == XL_DTYPE_BF16)
    hipLaunchKernelGGL(silu_mul_kernel<bf16_t>, grid, blk, 0, st, (const bf16_t*)gate, (const bf16_t*)up, (bf16_t*)y, nvec);
  else
    hipLaunchKernelGGL(silu_mul_kernel<f16_t>, grid, blk, 0, st, (const f16_t*)gate, (const f16_t*)up, (f16_t*)y, nvec);
  return check_launch(who);
}
