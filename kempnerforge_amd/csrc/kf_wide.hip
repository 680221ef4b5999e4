// Attention for the head sizes the matrix-core kernels are not built for: D a
// multiple of 16 up to 128 (80, 96, 112, ...; D 32 and 96 in 16-bit types).
//
// The operands are copied to float32 rows padded to W, D rounded up to 32:
// each half of a row (the two sides of the RoPE pairs) is padded to W / 2 with
// zeros, which add nothing to any product.  q and k are rotated on the way, in
// the input type's eager rounding, so the copies hold exactly the values the
// generic kernels computed with; the float32 kernels (kf_f32.hip) then keep
// scores, probabilities, dS and all sums in float32, as the generic kernels
// do, and the results are rounded to the input type once.  B = 2, S = 1024, 16
// heads of 96 in bf16, forward and backward: 20.9 ms on the generic kernels
// (one wavefront per row, no matrix instruction), 0.40 ms here.
//
// The copies are passes over q, k, v, dout and the results only (no S^2 term);
// in each direction one launch widens every operand and one narrows every
// result (15 and 9 us of the 400).
#include "kf_common.h"
#include "kf_internal.h"

#include <algorithm>

namespace kf {

namespace {

int wide_dim(int D) { return (D + 31) / 32 * 32; }

// One [B, S, H, D] operand and its float32 copy.  Source element (b, s, h, d)
// at src + b sb + s ss + h sh + d; copy row (b, s, h) at dst + b db + s ds + h dh,
// rows s in [S, Sp) zero.
struct WideJob {
  const void* src;
  float* dst;
  int64_t sb, ss, sh, db, ds, dh;
  int S, Sp, H, rot;  // rot: RoPE at table row s
};
constexpr int MAX_JOBS = 4;
struct WideJobs {
  WideJob j[MAX_JOBS];
  int64_t n[MAX_JOBS];  // threads of each job
};

// 8 elements of T as floats (16-byte aligned source).
template <typename T>
__device__ __forceinline__ void load8(const T* p, float* x) {
  if constexpr (std::is_same<T, float>::value) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 v = *(const f32x4*)(p + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * h + e] = v[e];
    }
  } else {
    unpack8<T>(*(const u32x4*)p, x);
  }
}
__device__ __forceinline__ void store8(float* p, const float* x) {
  *(f32x4*)p = f32x4{x[0], x[1], x[2], x[3]};
  *(f32x4*)(p + 4) = f32x4{x[4], x[5], x[6], x[7]};
}

// Thread: 8 elements of the first half of a row and their RoPE partners
// (chunk c of W / 16, zero past D / 2).  With tcos, the first job's threads of
// batch row 0, head 0 also write the tables as the rotation used them (rounded
// to T) for the RoPE backward, [S][W / 2], padded columns 1 and 0.
template <typename T>
__global__ __launch_bounds__(256) void widen_kernel(WideJobs jobs, const float* __restrict__ cos,
                                                    const float* __restrict__ sin, int B, int D,
                                                    int W, float* __restrict__ tcos,
                                                    float* __restrict__ tsin) {
  const WideJob& a = jobs.j[blockIdx.y];
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= jobs.n[blockIdx.y]) return;
  const int nc = W / 16, half = D / 2;
  const int c = (int)(t % nc);
  const int64_t row = t / nc;
  const int h = (int)(row % a.H);
  const int s = (int)((row / a.H) % a.Sp), b = (int)(row / ((int64_t)a.H * a.Sp));
  float x1[8] = {}, x2[8] = {};
  if (s < a.S && 8 * c < half) {
    const T* p = (const T*)a.src + b * a.sb + s * a.ss + h * a.sh + 8 * c;
    load8<T>(p, x1);
    load8<T>(p + half, x2);
    if (a.rot) {
      const float* cr = cos + (int64_t)s * half + 8 * c;
      const float* sr = sin + (int64_t)s * half + 8 * c;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float r1, r2;
        rope_pair<T>(x1[e], x2[e], cr[e], sr[e], r1, r2);
        x1[e] = r1;
        x2[e] = r2;
      }
    }
  }
  float* q = a.dst + b * a.db + s * a.ds + h * a.dh + 8 * c;
  store8(q, x1);
  store8(q + W / 2, x2);
  if (tcos != nullptr && blockIdx.y == 0 && b == 0 && h == 0 && s < a.S) {
    float tc[8], ts[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool in = 8 * c < half;
      tc[e] = in ? round_to<T>(cos[(int64_t)s * half + 8 * c + e]) : 1.f;
      ts[e] = in ? round_to<T>(sin[(int64_t)s * half + 8 * c + e]) : 0.f;
    }
    store8(tcos + (int64_t)s * (W / 2) + 8 * c, tc);
    store8(tsin + (int64_t)s * (W / 2) + 8 * c, ts);
  }
}

// The padded float32 rows [rows][W] of a result as T [rows][D].
struct NarrowJobs {
  const float* src[3];
  void* dst[3];
  int64_t n[3];  // threads of each job: rows x D / 8
};
template <typename T>
__global__ __launch_bounds__(256) void narrow_kernel(NarrowJobs jobs, int D, int W) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int y = blockIdx.y;
  if (t >= jobs.n[y]) return;
  const int nc = D / 8, c = (int)(t % nc);
  const int64_t row = t / nc;
  const int col = 8 * c < D / 2 ? 8 * c : W / 2 + 8 * c - D / 2;
  float x[8];
  load8<float>(jobs.src[y] + row * W + col, x);
  T* q = (T*)jobs.dst[y] + row * D + 8 * c;
  if constexpr (std::is_same<T, float>::value)
    store8(q, x);
  else
    *(u32x4*)q = pack8<T>(x);
}

template <typename F>
int by_type(int dtype, F f) {
  if (dtype == BF16) return f(bf16{});
  if (dtype == F16) return f(f16{});
  return f(float{});
}

int widen(WideJobs& jobs, int n, int dtype, const float* cos, const float* sin, int B, int D,
          float* tcos, float* tsin, hipStream_t stream) {
  const int W = wide_dim(D);
  int64_t most = 0;
  for (int i = 0; i < n; ++i) {
    jobs.n[i] = (int64_t)B * jobs.j[i].Sp * jobs.j[i].H * (W / 16);
    most = std::max(most, jobs.n[i]);
  }
  KF_CHECK_ARG((most + 255) / 256 < (1LL << 31), "grid too large");
  return by_type(dtype, [&](auto t) {
    using T = decltype(t);
    KF_LAUNCH("widen", widen_kernel<T>, dim3((unsigned)((most + 255) / 256), n), dim3(256), 0,
              stream, jobs, cos, sin, B, D, W, tcos, tsin);
    KF_CHECK_LAUNCH();
    return KF_OK;
  });
}

int narrow(NarrowJobs& jobs, int n, int dtype, int D, hipStream_t stream) {
  int64_t most = 0;
  for (int i = 0; i < n; ++i) most = std::max(most, jobs.n[i]);
  KF_CHECK_ARG((most + 255) / 256 < (1LL << 31), "grid too large");
  return by_type(dtype, [&](auto t) {
    using T = decltype(t);
    KF_LAUNCH("narrow", narrow_kernel<T>, dim3((unsigned)((most + 255) / 256), n), dim3(256), 0,
              stream, jobs, D, wide_dim(D));
    KF_CHECK_LAUNCH();
    return KF_OK;
  });
}

// Sequences up to this length stay on the generic kernels: with one launch
// against three the forward takes 32 us per call there against 39 (S = 16, B =
// 1, 4 heads of 96, calls queued back to back), from 32 on 51 against 36.
constexpr int WIDE_MIN_KEYS = 17;

bool wide_size(int S, int D, int dtype, int Hq, int Hkv) {
  if (S < WIDE_MIN_KEYS || D % 16 != 0 || D > 128 || D < 16) return false;
  return Hkv > 0 && Hq % Hkv == 0 && Hq / Hkv <= 64 && (int64_t)Hq * wide_dim(D) <= (1 << 24) &&
         (dtype == F32 || dtype == BF16 || dtype == F16);
}

size_t al256(size_t n) { return (n + 255) / 256 * 256; }

// contiguous [B, S, H, W] copy of a job's operand
WideJob rows_job(const void* src, int64_t sb, int64_t ss, int64_t sh, float* dst, int S, int H,
                 int W, int rot) {
  return WideJob{src, dst, sb, ss, sh, (int64_t)S * H * W, (int64_t)H * W, W, S, S, H, rot};
}

struct FwdWide {
  float *q, *k, *v, *out;
  void* ws;  // fwd_f32's
  size_t bytes;
};
FwdWide carve_fwd(const FwdArgs& a, void* workspace) {
  const size_t W = wide_dim(a.D);
  const size_t nq = (size_t)a.B * a.Sq * a.Hq * W, nk = (size_t)a.B * a.Sk * a.Hkv * W;
  FwdWide w;
  w.q = (float*)workspace;
  w.k = w.q + nq;
  w.v = w.k + nk;
  w.out = w.v + nk;
  const size_t head = al256((2 * nq + 2 * nk) * sizeof(float));
  w.ws = (char*)workspace + head;
  w.bytes = head + fwd_f32_workspace(a.B, a.Sk, a.Hkv, (int)W);
  return w;
}

// a's operands widened, and the float32 call on them
int widen_fwd(const FwdArgs& a, const FwdWide& w, FwdArgs& f) {
  const int W = wide_dim(a.D);
  WideJobs jobs{};
  const int64_t qs = (int64_t)a.Hq * a.D;
  jobs.j[0] = rows_job(a.q, a.Sq * qs, qs, a.D, w.q, a.Sq, a.Hq, W, 1);
  jobs.j[1] = rows_job(a.k, a.ksb, a.kss, a.ksh, w.k, a.Sk, a.Hkv, W, !a.k_rotated);
  jobs.j[2] = rows_job(a.v, a.vsb, a.vss, a.vsh, w.v, a.Sk, a.Hkv, W, 0);
  const int rc = widen(jobs, 3, a.dtype, a.cos, a.sin, a.B, a.D, nullptr, nullptr, a.stream);
  if (rc) return rc;
  f = a;
  f.q = w.q; f.k = w.k; f.v = w.v; f.out = w.out;
  f.D = W;
  f.dtype = F32;
  f.k_rotated = f.q_rotated = 1;
  f.ksh = f.vsh = W;
  f.kss = f.vss = (int64_t)a.Hkv * W;
  f.ksb = f.vsb = (int64_t)a.Sk * a.Hkv * W;
  return KF_OK;
}

int narrow_out(const FwdArgs& a, const FwdWide& w) {
  NarrowJobs out{};
  out.src[0] = w.out;
  out.dst[0] = a.out;
  out.n[0] = (int64_t)a.B * a.Sq * a.Hq * (a.D / 8);
  return narrow(out, 1, a.dtype, a.D, a.stream);
}

struct BwdWide {
  float *v, *dout, *dq, *dk, *dv, *cos, *sin;
  void* ws;  // bwd_f32's
  size_t head;
};
BwdWide carve_bwd(const BwdArgs& a, void* workspace) {
  const size_t W = wide_dim(a.D);
  const size_t nq = (size_t)a.B * a.S * a.Hq * W, nk = (size_t)a.B * a.S * a.Hkv * W;
  BwdWide w;
  w.v = (float*)workspace;
  w.dout = w.v + nk;
  w.dq = w.dout + nq;
  w.dk = w.dq + nq;
  w.dv = w.dk + nk;
  w.cos = w.dv + nk;
  w.sin = w.cos + (size_t)a.S * (W / 2);
  w.head = al256((2 * nq + 3 * nk + (size_t)a.S * W) * sizeof(float));
  w.ws = (char*)workspace + w.head;
  return w;
}

}  // namespace

bool fwd_wide_supported(const FwdArgs& a) {
  if (a.rot || !wide_size(a.Sk, a.D, a.dtype, a.Hq, a.Hkv)) return false;
  if (a.dtype == F32 ? a.D % 32 == 0 : a.D == 64 || a.D == 128) return false;  // own kernels
  if ((a.ksb | a.kss | a.ksh | a.vsb | a.vss | a.vsh) & 7) return false;
  // what the float32 kernels take (the masks' conditions and the tile lists)
  FwdArgs f = a;
  f.dtype = F32;
  f.D = wide_dim(a.D);
  f.k_rotated = a.doc || a.kvalid ? 0 : a.k_rotated;
  return fwd_f32_supported(f);
}

size_t fwd_wide_workspace(const FwdArgs& a) { return carve_fwd(a, nullptr).bytes; }

int fwd_wide(const FwdArgs& a, void* workspace) {
  const FwdWide w = carve_fwd(a, workspace);
  FwdArgs f;
  int rc = widen_fwd(a, w, f);
  if (rc) return rc;
  rc = fwd_f32(f, w.ws);
  return rc ? rc : narrow_out(a, w);
}

int capture_wide(const FwdArgs& a, float* probs, void* workspace) {
  const FwdWide w = carve_fwd(a, workspace);
  FwdArgs f;
  int rc = widen_fwd(a, w, f);
  if (rc) return rc;
  rc = capture_f32(f, probs, w.ws);
  return rc ? rc : narrow_out(a, w);
}

bool bwd_wide_supported(const BwdArgs& a) {
  if (a.rot || !wide_size(a.S, a.D, a.dtype, a.Hq, a.Hkv)) return false;
  if (a.dtype == F32 ? a.D % 32 == 0 : a.D == 64 || a.D == 128) return false;
  BwdArgs f = a;
  f.dtype = F32;
  f.D = wide_dim(a.D);
  return bwd_f32_supported(f);
}

size_t bwd_wide_workspace(const BwdArgs& a, bool with_ds) {
  const int W = wide_dim(a.D);
  return carve_bwd(a, nullptr).head +
         (with_ds ? bwd_f32_workspace_ds(a.B, a.S, a.Hq, a.Hkv, W, a.causal)
                  : bwd_f32_workspace(a.B, a.S, a.Hq, a.Hkv, W));
}

int bwd_wide(const BwdArgs& a, void* workspace, size_t workspace_bytes) {
  const int W = wide_dim(a.D);
  const BwdWide w = carve_bwd(a, workspace);
  const F32BwdWs fw = bwd_f32_carve(a.B, a.S, a.Hq, a.Hkv, W, a.causal, a.doc != nullptr, w.ws,
                                    workspace_bytes - w.head);
  const int64_t qs = (int64_t)a.Hq * a.D, ks = (int64_t)a.Hkv * a.D;
  WideJobs jobs{};
  // q and k straight into the float32 backward's rotated rows [b h][Sp][W]
  const int64_t head = (int64_t)fw.Sp * W;
  jobs.j[0] = WideJob{a.q, fw.qrot, a.S * qs, qs, a.D, a.Hq * head, W, head, a.S, fw.Sp, a.Hq, 1};
  jobs.j[1] = WideJob{a.k, fw.krot, a.S * ks, ks, a.D, a.Hkv * head, W, head, a.S, fw.Sp, a.Hkv, 1};
  jobs.j[2] = rows_job(a.v, a.S * ks, ks, a.D, w.v, a.S, a.Hkv, W, 0);
  jobs.j[3] = rows_job(a.dout, a.S * qs, qs, a.D, w.dout, a.S, a.Hq, W, 0);
  int rc = widen(jobs, 4, a.dtype, a.cos, a.sin, a.B, a.D, w.cos, w.sin, a.stream);
  if (rc) return rc;
  rc = bwd_f32_stats(a.out, a.dout, a.lse, a.dtype, a.B, a.S, a.Hq, a.D, fw, a.stream);
  if (rc) return rc;
  BwdArgs f = a;
  f.q = f.k = nullptr;
  f.v = w.v; f.dout = w.dout; f.dq = w.dq; f.dk = w.dk; f.dv = w.dv; f.cos = w.cos; f.sin = w.sin;
  f.D = W;
  f.dtype = F32;
  rc = bwd_f32_kernels(f, fw, w.ws, workspace_bytes - w.head);
  if (rc) return rc;
  NarrowJobs out{};
  out.src[0] = w.dq; out.dst[0] = a.dq; out.n[0] = (int64_t)a.B * a.S * a.Hq * (a.D / 8);
  out.src[1] = w.dk; out.dst[1] = a.dk; out.n[1] = (int64_t)a.B * a.S * a.Hkv * (a.D / 8);
  out.src[2] = w.dv; out.dst[2] = a.dv; out.n[2] = out.n[1];
  return narrow(out, 3, a.dtype, a.D, a.stream);
}

}  // namespace kf
