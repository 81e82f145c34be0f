// Chains the segment maps of a segmented scan (forward state, reverse state gradient).
#pragma once

#include "chunk_layout.hpp"
#include "kda_device.hpp"

namespace kda {

// S_in(j+1) = P_j S_in(j) + Sigma_j over the segments of one recurrence.  One workgroup per
// (recurrence, V strip); wave w owns state tiles w * TPW .. (w + 1) * TPW - 1.  Each step the
// waves publish their tiles as B operands in LDS, one barrier, and every wave multiplies its
// rows of P_j (fragments written by the local kernel, requested several steps ahead) by the
// whole state.
// F32 = false (the forward): P_j in bf16, the state as hi + lo bf16 halves (about 16 mantissa bits).
// F32 = true (the reverse scan, whose one-pass form carries lam X in f32): both stay f32, on
// v_mfma_f32_16x16x4_f32.  The step (tile kt, r) contracts keys 16 kt + 4 (l / 16) + r: the
// state's operand is the accumulator register it already lies in.  At 23 dependent steps (B1
// T32768 H1, K = V = 128) the f32 form takes 39 us and the bf16 form 21; with the sets requested
// a batch at a time, so that each batch began with a memory round trip, 53 and 31.
constexpr int kCombThreads = 4 * kWave;

struct CombineArgs {
  int H, num_seqs;
  int fixed_T;           // > 0: every sequence has this length
  int seg_len, max_segs; // chunks per segment, segments of the longest sequence
  const int2* seqs;      // {first chunk, chunk count} per sequence (fixed_T == 0)
  const float* start;    // [num_seqs][H][V][K] value entering segment 0, or null (zero)
  const void* P;         // [rec][segment] K x K, rec = sequence * H + head: bf16 in perm_frag_elem
                         // order, F32: f32 in f32_frag_elem order
  const float* sigma;    // [rec][segment][V][K]
  float* out;            // [rec][segment][V][K], segments >= 1
};

template <int K, bool F32>
struct CombOps;

template <int K>
struct CombOps<K, false> {
  static constexpr int NB = K / 32, TPW = K / 64, kAhead = 8;
  static constexpr int lds = 2 * NB * kWave * 16;  // [hi/lo][fragment]
  bf16x8 p[TPW][NB];
  __device__ void load(const void* P, size_t seg, int wave, int lane) {
    const bf16* q = (const bf16*)P + seg * K * K;
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int s = 0; s < NB; ++s) p[t][s] = *(const bf16x8*)(q + (((size_t)(wave * TPW + t) * NB + s) * 64 + lane) * 8);
  }
  static __device__ void publish(char* buf, int kt, int lane, const f32x4& S) {
    bf16x4 hi, lo;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      hi[r] = to_bf16(S[r]);
      lo[r] = to_bf16(S[r] - to_f32(hi[r]));
    }
    char* d = buf + (kt / 2) * (kWave * 16) + lane * 16 + (kt % 2) * 8;
    *(bf16x4*)d = hi;
    *(bf16x4*)(d + NB * kWave * 16) = lo;
  }
  __device__ void apply(const char* buf, int lane, f32x4 (&acc)[TPW]) const {
    bf16x8 hi[NB], lo[NB];
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      hi[s] = *(const bf16x8*)(buf + (s * kWave + lane) * 16);
      lo[s] = *(const bf16x8*)(buf + ((NB + s) * kWave + lane) * 16);
    }
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int s = 0; s < NB; ++s) {
        acc[t] = mfma16(p[t][s], hi[s], acc[t]);
        acc[t] = mfma16(p[t][s], lo[s], acc[t]);
      }
  }
};

template <int K>
struct CombOps<K, true> {
  static constexpr int KT = K / 16, TPW = K / 64, kAhead = 4;
  static constexpr int lds = KT * kWave * 16;  // [tile] in accumulator order
  f32x4 p[TPW][KT];
  __device__ void load(const void* P, size_t seg, int wave, int lane) {
    const float* q = (const float*)P + seg * K * K;
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        p[t][kt] = *(const f32x4*)(q + (((size_t)(wave * TPW + t) * KT + kt) * 64 + lane) * 4);
  }
  static __device__ void publish(char* buf, int kt, int lane, const f32x4& S) {
    *(f32x4*)(buf + (kt * kWave + lane) * 16) = S;
  }
  __device__ void apply(const char* buf, int lane, f32x4 (&acc)[TPW]) const {
    f32x4 x[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) x[kt] = *(const f32x4*)(buf + (kt * kWave + lane) * 16);
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < TPW; ++t)
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(p[t][kt][r], x[kt][r], acc[t], 0, 0, 0);
  }
};

template <int K, int V, bool F32>
__global__ __launch_bounds__(kCombThreads) void seg_combine_kernel(CombineArgs a) {
  using Ops = CombOps<K, F32>;
  constexpr int VS = V / 16, TPW = Ops::TPW, kAhead = Ops::kAhead;
  const int max_segs = a.max_segs;
  __shared__ __attribute__((aligned(16))) char sB[2][Ops::lds];  // [parity]
  const int H = a.H;
  int rec, strip;
  if (!xcd_strip_coords(a.num_seqs * H, VS, rec, strip)) return;
  const int seq = rec / H, h = rec % H;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, lr = lane % 16, kg = lane / 16;
  const int n = a.fixed_T > 0 ? (a.fixed_T + kChunk - 1) / kChunk : a.seqs[seq].y;
  const int nseg = (n + a.seg_len - 1) / a.seg_len;
  if (nseg <= 1) return;
  const int v = 16 * strip + lr;
  f32x4 S[TPW];
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int kt = wave * TPW + t;
    if (a.start) {
      const float4 x = *(const float4*)(a.start + (((size_t)seq * H + h) * V + v) * K + 16 * kt + 4 * kg);
      S[t][0] = x.x; S[t][1] = x.y; S[t][2] = x.z; S[t][3] = x.w;
    } else {
      S[t] = zero4();
    }
  }
  const size_t seg0 = (size_t)rec * max_segs;
  const float* G0 = a.sigma + seg0 * V * K + (size_t)v * K;
  // the P rows and Sigma of the next kAhead steps in registers or in flight: a step's set is
  // requested again as soon as it is used
  Ops pa[kAhead];
  float4 sg[kAhead][TPW];
  auto fetch = [&](int b, int j) {
    const int jj = min(j, nseg - 2);
    pa[b].load(a.P, seg0 + jj, wave, lane);
#pragma unroll
    for (int t = 0; t < TPW; ++t) sg[b][t] = *(const float4*)(G0 + (size_t)jj * V * K + 16 * (wave * TPW + t) + 4 * kg);
  };
#pragma unroll
  for (int b = 0; b < kAhead; ++b) fetch(b, b);
  for (int j0 = 0;; j0 += kAhead) {
#pragma unroll
    for (int b = 0; b < kAhead; ++b) {
      const int j = j0 + b;
      if (j + 1 >= nseg) return;
      char* buf = sB[j & 1];
#pragma unroll
      for (int t = 0; t < TPW; ++t) Ops::publish(buf, wave * TPW + t, lane, S[t]);
      // LDS only: a fence-free barrier (the loads ahead and earlier stores stay in flight)
      wait_lgkm0();
      ring_barrier();
#pragma unroll
      for (int t = 0; t < TPW; ++t) {
        S[t][0] = sg[b][t].x; S[t][1] = sg[b][t].y; S[t][2] = sg[b][t].z; S[t][3] = sg[b][t].w;
      }
      pa[b].apply(buf, lane, S);
      fetch(b, j + kAhead);
      float* out = a.out + (seg0 + j + 1) * V * K + (size_t)v * K;
#pragma unroll
      for (int t = 0; t < TPW; ++t)
        *(float4*)(out + 16 * (wave * TPW + t) + 4 * kg) = make_float4(S[t][0], S[t][1], S[t][2], S[t][3]);
    }
  }
}

}  // namespace kda
