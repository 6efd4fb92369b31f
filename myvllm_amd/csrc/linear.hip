// Linear layer of a few tokens: out (M, N) = x (M, K) w (N, K)^T, M <= 16,
// 16-bit operands, fp32 sums, one rounding.  The projections of a decode step
// (layers/linear_attention.py:86, :122 of yuyifanbupt/myvllm run them as
// torch linears).
//
// Bound by the read of w, so a workgroup takes 16 rows of w and its eight
// waves an eighth of K each: 64 KB of w in flight per workgroup.  The layer's
// in_proj is 772 workgroups, its out_proj only 128, on half the CUs.  The rows of w are
// the A operand (16x16x32 MFMA, fragments straight from memory, nothing
// staged), the tokens the B operand; the waves' partial tiles meet in LDS.
// Measured against the library's product with other weights in turn (us):
// 12,352 x 2,048 at 1 / 4 / 16 tokens 12.8 / 13.7 / 17.7 against 15.3 / 16.6 /
// 16.5, 2,048 x 4,096 6.8 / 7.4 / 9.4 against 11.3 / 11.8 / 11.5; 50 MB of
// weights in 12.8 us are 3.9 TB/s.  More tokens re-read x per row tile until
// that bounds it (64 tokens, two to four B tiles: 41 and 20 us against 18 and 11).
#include "gdn_common.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

template <typename T> struct Mfma;
template <> struct Mfma<bf16_t> {
  typedef bf16x8 v8;
  static GDN_DEVICE f32x4 mul(v8 a, v8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Mfma<f16_t> {
  typedef f16x8 v8;
  static GDN_DEVICE f32x4 mul(v8 a, v8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};

struct LinearArgs {
  const void* x; const void* w; void* out;
  int64_t x_s0, w_s0, o_s0;  // element strides
  int32_t M, N, K;           // K a multiple of 256
};

constexpr int kWaves = 8;

constexpr int kAhead = 8;  // k-steps of 32 in flight

template <typename T>
__global__ __launch_bounds__(64 * kWaves) void linear_kernel(LinearArgs a) {
  typedef typename Mfma<T>::v8 v8;
  typedef T v4 __attribute__((ext_vector_type(4)));
  __shared__ f32x4 part[kWaves][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int n0 = 16 * (int)blockIdx.x;
  const int steps = a.K / (32 * kWaves);
  // (rows past N and tokens past M are read from the last one: their products
  // stay in their own rows and columns, which are not stored)
  const int row = n0 + c < a.N ? n0 + c : a.N - 1, m = c < a.M ? c : a.M - 1;
  const int64_t k0 = (int64_t)wave * steps * 32 + 8 * q;
  const T* wp = reinterpret_cast<const T*>(a.w) + (int64_t)row * a.w_s0 + k0;
  const T* xp = reinterpret_cast<const T*>(a.x) + (int64_t)m * a.x_s0 + k0;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  int s = 0;
  for (; s + kAhead <= steps; s += kAhead) {
    v8 wf[kAhead], xf[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) wf[u] = *reinterpret_cast<const v8*>(wp + 32 * (s + u));
#pragma unroll
    for (int u = 0; u < kAhead; ++u) xf[u] = *reinterpret_cast<const v8*>(xp + 32 * (s + u));
#pragma unroll
    for (int u = 0; u < kAhead; ++u) acc = Mfma<T>::mul(wf[u], xf[u], acc);
  }
  for (; s < steps; ++s)
    acc = Mfma<T>::mul(*reinterpret_cast<const v8*>(wp + 32 * s), *reinterpret_cast<const v8*>(xp + 32 * s), acc);
  part[wave][lane] = acc;
  __syncthreads();
  // one wave sums: lane (c, q) holds token c, rows n0 + 4q..+3
  if (wave > 0) return;
  f32x4 sum = part[0][lane];
#pragma unroll
  for (int p = 1; p < kWaves; ++p) {
    const f32x4 y = part[p][lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) sum[r] += y[r];
  }
  const int n = n0 + 4 * q;
  if (c >= a.M) return;
  T* o = reinterpret_cast<T*>(a.out) + (int64_t)c * a.o_s0 + n;
  if (n + 4 <= a.N) {
    *reinterpret_cast<v4*>(o) = v4{(T)sum[0], (T)sum[1], (T)sum[2], (T)sum[3]};
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (n + r < a.N) o[r] = (T)sum[r];
  }
}

}  // namespace

// Called by the validated C entry point in gdn_capi.cpp.
hipError_t linear_launch(const gdn_tensor* x, const gdn_tensor* w, gdn_tensor* out, hipStream_t st) {
  LinearArgs a;
  a.x = x->data; a.w = w->data; a.out = out->data;
  a.x_s0 = x->stride[0]; a.w_s0 = w->stride[0]; a.o_s0 = out->stride[0];
  a.M = (int32_t)x->shape[0]; a.N = (int32_t)w->shape[0]; a.K = (int32_t)x->shape[1];
  if (a.M == 0 || a.N == 0) return hipSuccess;
  const dim3 grid((unsigned)((a.N + 15) / 16)), block(64 * kWaves);
  if (x->dtype == GDN_DTYPE_BF16) linear_kernel<bf16_t><<<grid, block, 0, st>>>(a);
  else linear_kernel<f16_t><<<grid, block, 0, st>>>(a);
  return hipGetLastError();
}
