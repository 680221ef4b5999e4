// The second half of the split-K decodes: the float32 partials (o, m, l) of one
// (sequence, query head) row rescaled to a common maximum and summed.
#pragma once

#include "kf_common.h"

namespace kf {

// Wavefronts that share a row of `slots` partials (one workgroup per row when
// more than one).  Event-timed with 1 / 4 / 16 of them (32 query heads, 8 KV
// heads; an empty launch reads about 6 us): 16 partials 6.5 / 6.0 / 6.5 us, 32
// 8.5 / 6.1 / 6.1, 64 9.7 / 6.7 / 7.0, 128 14.0 / 8.2 / 7.9, 257 22.8 / 10.1 /
// 8.6; with 32 sequences (9 partials) 6.3 / 7.5 / 6.3.
inline int merge_waves(int slots) { return slots <= 16 ? 1 : slots <= 64 ? 4 : 16; }

// Sum of a row's `ns` partials: partial j's D outputs at ob + j * ost, its (m,
// l) at mb + j * mst (m in log2 units).  `sO` is WPR * D floats of LDS (WPR >
// 1 only).  On return every lane of wavefront 0 with (lane % (D / 4)) = c
// holds the outputs 4 c .. 4 c + 3, already divided by the row's sum.
//
// Bound by the latency of the dependent round trips to partials other XCDs
// wrote, so: every wavefront takes the maximum and the sum over all (m, l) by
// itself (a lane per partial, no exchange), the first partials' outputs are
// loaded beside them, and a 16-byte load covers 256 / D partials per
// instruction, MU instructions in flight, WPR wavefronts interleaved.  The
// previous form (one wavefront, one 4-byte load per lane and partial, empty
// slots tested one by one) took 75 us at B = 1, 8 KV heads, 1000 keys, 22 us
// at B = 16, 2 KV heads, 4096 keys and 132 us at B = 1, 8 KV heads, 65536
// keys; this one 6.8, 7.9 and 9.7 us.
constexpr int MU = 4;
template <int D, int WPR>
__device__ __forceinline__ f32x4 merge_row(const float* __restrict__ ob,
                                           const float* __restrict__ mb, int64_t ost,
                                           int64_t mst, int ns, float* sO, int wv, int lane) {
  // lanes per partial (a power of two; D 96 leaves 8 of 32 idle), partials per
  // instruction
  constexpr int LPS = D == 96 ? 32 : D / 4, SPI = 64 / LPS;
  const int sub = lane / LPS, col = min(4 * (lane % LPS), D - 4);
  f32x4 po[MU];
  float pm[MU];
  auto slot = [&](int i) { return (i * WPR + wv) * SPI + sub; };
  auto load = [&](int i0) {
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const int j = min(slot(i0 + u), ns - 1);  // a repeated partial gets no weight below
      po[u] = *(const f32x4*)(ob + j * ost + col);
      pm[u] = mb[j * mst];
    }
  };
  load(0);
  float2 ml[MU];
#pragma unroll
  for (int u = 0; u < MU; ++u) {
    const int j = 64 * u + lane;
    ml[u] = make_float2(-INFINITY, 0.f);
    if (j < ns) ml[u] = *(const float2*)(mb + j * mst);
  }
  float M = -INFINITY;
#pragma unroll
  for (int u = 0; u < MU; ++u) M = fmaxf(M, ml[u].x);
  for (int j = 64 * MU + lane; j < ns; j += 64) M = fmaxf(M, mb[j * mst]);
  M = wave_max(M);
  float l = 0.f;
#pragma unroll
  for (int u = 0; u < MU; ++u)
    if (64 * u + lane < ns) l += ml[u].y * fast_exp2(ml[u].x - M);
  for (int j = 64 * MU + lane; j < ns; j += 64) l += mb[j * mst + 1] * fast_exp2(mb[j * mst] - M);
  l = wave_sum(l);
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int i0 = 0; (i0 * WPR + wv) * SPI < ns; i0 += MU) {
    if (i0 > 0) load(i0);
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const float w = slot(i0 + u) < ns ? fast_exp2(pm[u] - M) : 0.f;
      // (a partial of weight 0 is left out, whatever it holds)
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += w != 0.f ? po[u][e] * w : 0.f;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll
    for (int x = LPS; x < 64; x <<= 1) o[e] += __shfl_xor(o[e], x, 64);
  if constexpr (WPR > 1) {
    if (sub == 0) *(f32x4*)(sO + wv * D + col) = o;
    __syncthreads();
    o = f32x4{0.f, 0.f, 0.f, 0.f};
    if (wv == 0) {
#pragma unroll
      for (int w = 0; w < WPR; ++w) o += *(const f32x4*)(sO + w * D + col);
    }
  }
  return o * (1.f / l);
}

}  // namespace kf
