// y = x W^T for a few rows of x (the decode step's projections), with the elementwise work
// that follows a projection of the decoder in its epilogue: relu(y)^2 (the MLP activation,
// nanochat/gpt.py:151-156) or a residual add (gpt.py:202-205).
//
// Bound by one pass over W (0.3-2.4 MB per projection, 25 MB for the head) and, for the small
// ones, by the latency of a workgroup: so a workgroup takes only 16 rows of W and its waves split
// the contraction, every wave with kAhead fragments of W and x in flight, straight from memory to
// the MFMA operands (a 16 x 32 fragment of W is one 16-byte load per lane).  The waves' partial
// tiles meet in LDS and are added in wave order.  x (a few KB) comes from L2.
// At 8 rows, weights of 2312 x 384, 384 x 1536 and 32768 x 384: 2.4 / 3.9 / 6.8 us against 3.5 /
// 4.7 / 9.1 us of the library GEMM (whose call also takes the host 18 us, this one 8).
#include "kda_device.hpp"
#include "kda_host.hpp"

namespace kda {

constexpr int kLinAhead = 3;  // 32-deep steps in flight per wave

enum LinEpilogue { kLinNone = 0, kLinRelu2 = 1, kLinAdd = 2 };

template <int MT, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void linear_rows_kernel(int M, int N, int K, long ldx, int epilogue,
                                                                    const bf16* __restrict__ x,
                                                                    const bf16* __restrict__ w,
                                                                    const bf16* __restrict__ res, long ldr,
                                                                    bf16* __restrict__ y) {
  __shared__ f32x4 part[WAVES][MT][kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, lr = lane % 16, kg = lane / 16;
  const int n0 = 16 * blockIdx.x;
  const bf16* wr = w + (size_t)min(n0 + lr, N - 1) * K + 8 * kg;
  const bf16* xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xr[t] = x + (size_t)min(16 * t + lr, M - 1) * ldx + 8 * kg;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = zero4();
  const int steps = K / 32;  // step s: columns 32 s ..; wave v takes s = v, v + WAVES, ...
  for (int s0 = wave; s0 < steps; s0 += kLinAhead * WAVES) {
    bf16x8 fw[kLinAhead], fx[kLinAhead][MT];
#pragma unroll
    for (int u = 0; u < kLinAhead; ++u) {
      const int s = min(s0 + u * WAVES, steps - 1);  // past the end: a valid step, not used
      fw[u] = *(const bf16x8*)(wr + 32 * s);
#pragma unroll
      for (int t = 0; t < MT; ++t) fx[u][t] = *(const bf16x8*)(xr[t] + 32 * s);
    }
#pragma unroll
    for (int u = 0; u < kLinAhead; ++u)
      if (s0 + u * WAVES < steps)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = mfma16(fw[u], fx[u][t], acc[t]);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) part[wave][t][lane] = acc[t];
  __syncthreads();
  // accumulator: rows of W 4 kg + r, row of x lr
  for (int t = wave; t < MT; t += WAVES) {
    f32x4 v = part[0][t][lane];
#pragma unroll
    for (int q = 1; q < WAVES; ++q) v += part[q][t][lane];
    const int m = 16 * t + lr, n = n0 + 4 * kg;
    if (m >= M || n >= N) continue;
    bf16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = to_bf16(v[r]);
    if (epilogue == kLinRelu2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = fmaxf((float)o[r], 0.f);
        o[r] = to_bf16(p * p);
      }
    } else if (epilogue == kLinAdd) {
      const bf16x4 a = *(const bf16x4*)(res + (size_t)m * ldr + n);
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = to_bf16((float)a[r] + (float)o[r]);
    }
    *(bf16x4*)(y + (size_t)m * N + n) = o;
  }
}

// The projection of a normed row with the norm in front of it: s = a x + b x2 (a = wa[0], b =
// wb[0], 1 where null) rounded to bf16, h = rms_norm(s), y = h W^T with linear_rows' epilogues.
// Every workgroup norms the (at most 16) rows for itself, 16 lanes a row as rms_norm_fwd_kernel
// does, while its first fragments of W are in flight, and keeps them in LDS; workgroup 0 also
// writes s.  At 8 rows of 384 the mix + norm launch and the projection's cost 2.3 + 2.4 us and
// two calls of the host; this one takes 4.0 us and one call (decoder step B8: 1011 -> 814 us).
template <int J>
__global__ __launch_bounds__(256) void norm_linear_rows_kernel(int M, int N, float eps, int epilogue,
                                                               const float* __restrict__ wa,
                                                               const float* __restrict__ wb,
                                                               const bf16* __restrict__ x,
                                                               const bf16* __restrict__ x2,
                                                               const bf16* __restrict__ w, bf16* __restrict__ s,
                                                               bf16* __restrict__ y) {
  constexpr int K = 128 * J, HP = K + 8, WAVES = 4, STEPS = K / 32, PER = STEPS / WAVES;
  constexpr int AHEAD = PER <= 4 ? PER : PER % 4 == 0 ? 4 : 3;
  static_assert(PER % AHEAD == 0, "whole rounds");
  __shared__ __attribute__((aligned(16))) bf16 sh[16 * HP];
  __shared__ f32x4 part[WAVES][kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, lr = lane % 16, kg = lane / 16;
  const int n0 = 16 * blockIdx.x;
  const bf16* wr = w + (size_t)min(n0 + lr, N - 1) * K + 8 * kg;
  bf16x8 fw[AHEAD];
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) fw[u] = *(const bf16x8*)(wr + 32 * (wave + u * WAVES));
  {
    const int row = threadIdx.x / 16, l = threadIdx.x % 16, rc = min(row, M - 1);
    bf16x8 xv[J], zv[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      xv[j] = *(const bf16x8*)(x + (size_t)rc * K + 128 * j + 8 * l);
      zv[j] = *(const bf16x8*)(x2 + (size_t)rc * K + 128 * j + 8 * l);
    }
    const float a = wa ? wa[0] : 1.f, b = wb ? wb[0] : 1.f;
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        xv[j][e] = to_bf16(fmaf(a, (float)xv[j][e], b * (float)zv[j][e]));
        ss = fmaf((float)xv[j][e], (float)xv[j][e], ss);
      }
      if (blockIdx.x == 0 && row < M) *(bf16x8*)(s + (size_t)row * K + 128 * j + 8 * l) = xv[j];
    }
    const float r = rsqrtf(group_sum<16>(ss) / K + eps);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      bf16x8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = to_bf16((float)xv[j][e] * r);
      *(bf16x8*)(sh + row * HP + 128 * j + 8 * l) = h;
    }
  }
  wait_lgkm0();
  ring_barrier();  // LDS only: the loads of W stay in flight
  f32x4 acc = zero4();
#pragma unroll
  for (int s0 = 0; s0 < PER; s0 += AHEAD) {
    bf16x8 nx[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (s0 + AHEAD < PER) nx[u] = *(const bf16x8*)(wr + 32 * (wave + (s0 + AHEAD + u) * WAVES));
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      acc = mfma16(fw[u], *(const bf16x8*)(sh + lr * HP + 32 * (wave + (s0 + u) * WAVES) + 8 * kg), acc);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (s0 + AHEAD < PER) fw[u] = nx[u];
  }
  part[wave][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  f32x4 v = part[0][lane];
#pragma unroll
  for (int q = 1; q < WAVES; ++q) v += part[q][lane];
  const int n = n0 + 4 * kg;
  if (lr >= M || n >= N) return;
  bf16x4 o;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    o[r] = to_bf16(v[r]);
    if (epilogue == kLinRelu2) {
      const float p = fmaxf((float)o[r], 0.f);
      o[r] = to_bf16(p * p);
    }
  }
  *(bf16x4*)(y + (size_t)lr * N + n) = o;
}

}  // namespace kda

extern "C" int kda_norm_linear_rows(int32_t rows, int32_t out_dim, int32_t in_dim, float eps, const float* a,
                                    const float* b, const void* x, const void* x2, const void* weight,
                                    int32_t epilogue, void* sum, void* y, hipStream_t stream) {
  using namespace kda;
  const int J = in_dim / 128;
  KDA_REQUIRE(rows >= 0 && rows <= 16, "norm_linear_rows: at most 16 rows");
  KDA_REQUIRE(in_dim > 0 && in_dim % 128 == 0 && (J <= 4 || J == 6 || J == 8),
              "norm_linear_rows: in_dim must be 128 x {1,2,3,4,6,8}");
  KDA_REQUIRE(out_dim > 0 && out_dim % 4 == 0, "norm_linear_rows: out_dim must be a multiple of 4");
  KDA_REQUIRE(epilogue == kLinNone || epilogue == kLinRelu2, "norm_linear_rows: unknown epilogue");
  if (rows == 0) return KDA_OK;
  KDA_REQUIRE(x && x2 && weight && sum && y && aligned16(x, x2, weight, sum, y),
              "norm_linear_rows: null or unaligned pointer");
  const dim3 grid((unsigned)((out_dim + 15) / 16));
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(256), 0, stream, rows, out_dim, eps, epilogue, a, b, (const bf16*)x,
                       (const bf16*)x2, (const bf16*)weight, (bf16*)sum, (bf16*)y);
  };
  switch (J) {
    case 1: go(norm_linear_rows_kernel<1>); break;
    case 2: go(norm_linear_rows_kernel<2>); break;
    case 3: go(norm_linear_rows_kernel<3>); break;
    case 4: go(norm_linear_rows_kernel<4>); break;
    case 6: go(norm_linear_rows_kernel<6>); break;
    default: go(norm_linear_rows_kernel<8>); break;
  }
  KDA_LAUNCH_CHECK("norm_linear_rows");
  return KDA_OK;
}

extern "C" int kda_linear_rows(int32_t rows, int32_t out_dim, int32_t in_dim, const void* x, int64_t x_row_stride,
                               const void* weight, int32_t epilogue, const void* residual,
                               int64_t residual_row_stride, void* y, hipStream_t stream) {
  using namespace kda;
  KDA_REQUIRE(rows >= 0 && rows <= 64, "linear_rows: at most 64 rows");
  KDA_REQUIRE(out_dim > 0 && out_dim % 4 == 0 && in_dim > 0 && in_dim % 32 == 0,
              "linear_rows: out_dim must be a multiple of 4, in_dim of 32");
  KDA_REQUIRE(epilogue >= kLinNone && epilogue <= kLinAdd, "linear_rows: unknown epilogue");
  KDA_REQUIRE(x_row_stride >= in_dim && x_row_stride % 8 == 0, "linear_rows: x rows must be 16-byte aligned");
  KDA_REQUIRE(epilogue != kLinAdd || (residual && ((uintptr_t)residual % 8) == 0 && residual_row_stride >= out_dim &&
                                      residual_row_stride % 4 == 0),
              "linear_rows: the residual must be 8-byte aligned rows of out_dim");
  if (rows == 0) return KDA_OK;
  KDA_REQUIRE(x && weight && y && aligned16(x, weight, y), "linear_rows: null or unaligned pointer");
  const dim3 grid((unsigned)((out_dim + 15) / 16));
  auto go = [&](auto kern, int waves) {
    hipLaunchKernelGGL(kern, grid, dim3(waves * kWave), 0, stream, rows, out_dim, in_dim, (long)x_row_stride, epilogue,
                       (const bf16*)x, (const bf16*)weight, (const bf16*)residual, (long)residual_row_stride,
                       (bf16*)y);
  };
  // a long contraction over few workgroups: twice the waves
  const bool deep = in_dim >= 1024;
  if (rows <= 16)
    deep ? go(linear_rows_kernel<1, 8>, 8) : go(linear_rows_kernel<1, 4>, 4);
  else if (rows <= 32)
    deep ? go(linear_rows_kernel<2, 8>, 8) : go(linear_rows_kernel<2, 4>, 4);
  else
    deep ? go(linear_rows_kernel<4, 8>, 8) : go(linear_rows_kernel<4, 4>, 4);
  KDA_LAUNCH_CHECK("linear_rows");
  return KDA_OK;
}
