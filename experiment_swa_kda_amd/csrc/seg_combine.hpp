// Chains the segment maps of a segmented scan (forward state, reverse state gradient).
#pragma once

#include "chunk_layout.hpp"
#include "kda_device.hpp"

namespace kda {

// S_in(j+1) = P_j S_in(j) + Sigma_j over the segments of one recurrence.  One workgroup per
// (recurrence, V strip); wave w owns state tiles w * TPW .. (w + 1) * TPW - 1.  Each step the
// waves publish their tiles as hi + lo bf16 B-operand halves in LDS (about 16 mantissa
// bits of the state), one barrier, and every wave multiplies its rows of P_j (bf16
// fragments written by the local kernel, requested a batch of steps ahead) by the whole state.
// LO: P_j comes as hi + lo bf16 too (the reverse scan, whose one-pass form carries lam X in f32).
constexpr int kCombThreads = 4 * kWave;

struct CombineArgs {
  int H, num_seqs;
  int fixed_T;           // > 0: every sequence has this length
  int seg_len, max_segs; // chunks per segment, segments of the longest sequence
  const int2* seqs;      // {first chunk, chunk count} per sequence (fixed_T == 0)
  const float* start;    // [num_seqs][H][V][K] value entering segment 0, or null (zero)
  const bf16* P;         // [rec][segment] K x K (LO: then its low part), rec = sequence * H + head
  const float* sigma;    // [rec][segment][V][K]
  float* out;            // [rec][segment][V][K], segments >= 1
};

template <int K, int V, bool LO>
__global__ __launch_bounds__(kCombThreads) void seg_combine_kernel(CombineArgs a) {
  constexpr int kParts = LO ? 2 : 1, kCombBatch = LO ? 4 : 8;
  const int max_segs = a.max_segs;
  constexpr int KT = K / 16, NB = K / 32, VS = V / 16, TPW = KT / 4;
  __shared__ __attribute__((aligned(16))) char sB[2][2][NB][kWave * 16];  // [parity][hi/lo][frag]
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
  const bf16* P0 = a.P + (size_t)rec * max_segs * kParts * K * K;
  const float* G0 = a.sigma + (size_t)rec * max_segs * V * K + (size_t)v * K;
  // every step's P rows and Sigma for this wave, requested up front in batches of
  // kCombBatch steps (one memory round trip per batch instead of one per step)
  bf16x8 pa[kCombBatch][kParts][TPW][NB];
  float4 sg[kCombBatch][TPW];
  for (int j = 0; j + 1 < nseg; ++j) {
    const int jb = j % kCombBatch;
    if (jb == 0) {
#pragma unroll
      for (int b = 0; b < kCombBatch; ++b) {
        const int jj = min(j + b, nseg - 2);
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
          const int kt = wave * TPW + t;
#pragma unroll
          for (int u = 0; u < kParts; ++u)
#pragma unroll
            for (int s = 0; s < NB; ++s)
              pa[b][u][t][s] = *(const bf16x8*)(P0 + ((size_t)jj * kParts + u) * K * K + (((size_t)kt * NB + s) * 64 + lane) * 8);
          sg[b][t] = *(const float4*)(G0 + (size_t)jj * V * K + 16 * kt + 4 * kg);
        }
      }
    }
    char(*buf)[NB][kWave * 16] = sB[j & 1];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      const int kt = wave * TPW + t;
      bf16x4 hi, lo;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        hi[r] = to_bf16(S[t][r]);
        lo[r] = to_bf16(S[t][r] - to_f32(hi[r]));
      }
      *(bf16x4*)(buf[0][kt / 2] + lane * 16 + (kt % 2) * 8) = hi;
      *(bf16x4*)(buf[1][kt / 2] + lane * 16 + (kt % 2) * 8) = lo;
    }
    // LDS only: a fence-free barrier (the prefetched loads and earlier stores stay in flight)
    wait_lgkm0();
    ring_barrier();
    bf16x8 Bh[NB], Bl[NB];
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      Bh[s] = *(const bf16x8*)(buf[0][s] + lane * 16);
      Bl[s] = *(const bf16x8*)(buf[1][s] + lane * 16);
    }
    // pick this step's operands (jb is uniform; unrolled select keeps them in registers)
    bf16x8 pc[kParts][TPW][NB];
    float4 gc[TPW];
#pragma unroll
    for (int b = 0; b < kCombBatch; ++b)
      if (b == jb) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
          gc[t] = sg[b][t];
#pragma unroll
          for (int u = 0; u < kParts; ++u)
#pragma unroll
            for (int s = 0; s < NB; ++s) pc[u][t][s] = pa[b][u][t][s];
        }
      }
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
      f32x4 acc;
      acc[0] = gc[t].x; acc[1] = gc[t].y; acc[2] = gc[t].z; acc[3] = gc[t].w;
#pragma unroll
      for (int s = 0; s < NB; ++s) {
        acc = mfma16(pc[0][t][s], Bh[s], acc);
        acc = mfma16(pc[0][t][s], Bl[s], acc);
        if constexpr (LO) acc = mfma16(pc[kParts - 1][t][s], Bh[s], acc);
      }
      S[t] = acc;
    }
    float* out = a.out + ((size_t)rec * max_segs + j + 1) * V * K + (size_t)v * K;
#pragma unroll
    for (int t = 0; t < TPW; ++t)
      *(float4*)(out + 16 * (wave * TPW + t) + 4 * kg) = make_float4(S[t][0], S[t][1], S[t][2], S[t][3]);
  }
}

}  // namespace kda
