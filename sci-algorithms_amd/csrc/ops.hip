// Forward model, adjoint, mask sum, layout conversion and squared-error
// reductions of the SCI forward model (PnP_SCI/python/utils.py:10-36,
// pnp_sci_algo.py:491-492).  All volumes are frame-major (T,H,W).
//
// These kernels are single-pass and HBM-bound: each reads and writes every
// byte once with 16-byte accesses along the contiguous pixel axis.

#include "scigap_internal.h"

#include <cstring>

namespace scigap {

namespace {
thread_local char g_err[512] = "";
}

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

void clear_error() { g_err[0] = 0; }

namespace {

constexpr int kThreads = 256;

// Blocks for a grid-stride loop over n items: enough to fill 256 CUs with
// several waves each, never more than the work needs.
inline unsigned grid_for(int64_t n, int per_thread = 1) {
  int64_t blocks = (n + int64_t(kThreads) * per_thread - 1) / (int64_t(kThreads) * per_thread);
  if (blocks > 256 * 16) blocks = 256 * 16;
  if (blocks < 1) blocks = 1;
  return unsigned(blocks);
}

// y = sum_t x_t * phi_t.  One thread handles 4 consecutive pixels (N % 4 == 0)
// or 1 pixel; the frame loop keeps the running sums in registers (fp64).
template <int V>
__global__ void __launch_bounds__(kThreads) k_forward(const float* __restrict__ x,
                                                      const float* __restrict__ phi,
                                                      float* __restrict__ y, int64_t N, int T) {
  const int64_t nv = N / V;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < nv;
       i += int64_t(gridDim.x) * blockDim.x) {
    if constexpr (V == 4) {
      double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
      for (int t = 0; t < T; ++t) {
        float4 a = reinterpret_cast<const float4*>(x + t * N)[i];
        float4 m = reinterpret_cast<const float4*>(phi + t * N)[i];
        s0 = acc_prod(a.x, m.x, s0);
        s1 = acc_prod(a.y, m.y, s1);
        s2 = acc_prod(a.z, m.z, s2);
        s3 = acc_prod(a.w, m.w, s3);
      }
      reinterpret_cast<float4*>(y)[i] = make_float4(float(s0), float(s1), float(s2), float(s3));
    } else {
      double acc = 0.0;
      for (int t = 0; t < T; ++t) acc = acc_prod(x[t * N + i], phi[t * N + i], acc);
      y[i] = float(acc);
    }
  }
}

template <int V>
__global__ void __launch_bounds__(kThreads) k_adjoint(const float* __restrict__ y,
                                                      const float* __restrict__ phi,
                                                      float* __restrict__ x, int64_t N, int T) {
  const int64_t nv = N / V;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < nv;
       i += int64_t(gridDim.x) * blockDim.x) {
    if constexpr (V == 4) {
      float4 v = reinterpret_cast<const float4*>(y)[i];
      for (int t = 0; t < T; ++t) {
        float4 m = reinterpret_cast<const float4*>(phi + t * N)[i];
        reinterpret_cast<float4*>(x + t * N)[i] = make_float4(v.x * m.x, v.y * m.y, v.z * m.z, v.w * m.w);
      }
    } else {
      float v = y[i];
      for (int t = 0; t < T; ++t) x[t * N + i] = v * phi[t * N + i];
    }
  }
}

__global__ void __launch_bounds__(kThreads) k_phi_sum(const float* __restrict__ phi,
                                                      float* __restrict__ s, int64_t N, int T) {
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < N;
       i += int64_t(gridDim.x) * blockDim.x) {
    // Sequential sum over t (the reference's np.sum over a length-T axis of a
    // C-order array also adds the T values of a pixel in order for T < 8).
    float acc = 0.f;
    for (int t = 0; t < T; ++t) acc += phi[t * N + i];
    s[i] = (acc == 0.f) ? 1.f : acc;
  }
}

// Tiled transpose of a rows x cols matrix (row-major) into cols x rows.
// (H,W,T) -> (T,H,W) is rows = H*W, cols = T; the reverse swaps them.
// grid.y is capped at 65535, so blocks stride over the row tiles.
constexpr int TT = 32;
__global__ void __launch_bounds__(TT * 8) k_transpose(const float* __restrict__ src,
                                                      float* __restrict__ dst,
                                                      int64_t rows, int64_t cols) {
  __shared__ float tile[TT][TT + 1];
  const int tx = threadIdx.x % TT, ty = threadIdx.x / TT;  // 32 x 8 threads
  const int64_t c0 = int64_t(blockIdx.x) * TT;
  const int64_t row_tiles = (rows + TT - 1) / TT;
  for (int64_t by = blockIdx.y; by < row_tiles; by += gridDim.y) {
    const int64_t r0 = by * TT;
    for (int k = ty; k < TT; k += 8) {
      int64_t r = r0 + k, c = c0 + tx;
      if (r < rows && c < cols) tile[k][tx] = src[r * cols + c];
    }
    __syncthreads();
    for (int k = ty; k < TT; k += 8) {
      int64_t c = c0 + k, r = r0 + tx;  // dst row = source column
      if (r < rows && c < cols) dst[c * rows + r] = tile[tx][k];
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Kernels on the reference's (H,W,T) layout.  A block takes P consecutive
// pixels, that is P*T consecutive floats: it moves them with 16-byte accesses
// in memory order and hands them to the pixels (or frames) through LDS, padded
// by one element every 32 so that reading with a stride of T meets the banks
// evenly.
//
// All are bound by memory, or by their launch.  A_ plus At_ of 256x256x8 on
// device tensors take 24 us; converting both operands first (six launches
// instead of two, three times the traffic) they took 55.  A conversion of
// 1024x1024x8 takes 11 us (6 TB/s, with what the caches hold); in 32x32 tiles, of
// which 8 frames fill a quarter, 35.
// ---------------------------------------------------------------------------

__host__ __device__ inline int pad32(int e) { return e + (e >> 5); }

inline size_t hwt_lds(int P, int64_t T, int bytes) {
  return size_t(pad32(int(P * T)) + 1) * size_t(bytes);
}

// Pixels of a block of k_forward_hwt: the most whose products leave room for
// several blocks on a CU; 0 when not even one wave's fit.
inline int forward_pixels(int64_t T) {
  for (int P : {256, 128, 64})
    if (int64_t(P) * T * 8 <= (P == 64 ? 60 : 40) * 1024) return P;
  return 0;
}

// y = sum_t x_t * phi_t on (H,W,T) arrays: exact products in fp64, summed in
// frame order (as k_forward).
template <bool VEC>
__global__ void __launch_bounds__(256) k_forward_hwt(const float* __restrict__ x,
                                                     const float* __restrict__ phi,
                                                     float* __restrict__ y, int64_t N, int T) {
  extern __shared__ double prod[];
  const int P = blockDim.x, tid = threadIdx.x;
  const int64_t p0 = int64_t(blockIdx.x) * P;
  const int64_t base = p0 * T;
  const int n = int(p0 + P <= N ? P : N - p0) * T;
  int done = 0;
  if constexpr (VEC) {
    const float4* const xv = reinterpret_cast<const float4*>(x + base);
    const float4* const fv = reinterpret_cast<const float4*>(phi + base);
    for (int i = tid; i < n / 4; i += P) {
      const float4 a = xv[i], b = fv[i];
      prod[pad32(4 * i)] = double(a.x) * double(b.x);
      prod[pad32(4 * i + 1)] = double(a.y) * double(b.y);
      prod[pad32(4 * i + 2)] = double(a.z) * double(b.z);
      prod[pad32(4 * i + 3)] = double(a.w) * double(b.w);
    }
    done = n & ~3;
  }
  for (int i = done + tid; i < n; i += P)
    prod[pad32(i)] = double(x[base + i]) * double(phi[base + i]);
  __syncthreads();
  if (p0 + tid < N) {
    double s = 0.0;
    for (int t = 0; t < T; ++t) s += prod[pad32(tid * T + t)];
    y[p0 + tid] = float(s);
  }
}

// The same for frame counts whose products do not fit the LDS: kChunk frames
// at a time, so that lanes read runs of a pixel's frames and not one frame each
// (512x512x160: 1130 us that way).
constexpr int kChunk = 16;
__global__ void __launch_bounds__(kThreads) k_forward_hwt_many(const float* __restrict__ x,
                                                               const float* __restrict__ phi,
                                                               float* __restrict__ y, int64_t N,
                                                               int T) {
  __shared__ double prod[kThreads][kChunk + 1];
  const int tid = threadIdx.x;
  const int64_t p0 = int64_t(blockIdx.x) * kThreads;
  const int np = int(p0 + kThreads <= N ? kThreads : N - p0);
  double s = 0.0;
  for (int t0 = 0; t0 < T; t0 += kChunk) {
    const int nt = T - t0 < kChunk ? T - t0 : kChunk;
    for (int i = tid; i < np * kChunk; i += kThreads) {
      const int p = i / kChunk, t = i % kChunk;
      const int64_t o = (p0 + p) * T + t0 + t;
      if (t < nt) prod[p][t] = double(x[o]) * double(phi[o]);
    }
    __syncthreads();
    if (tid < np)
      for (int t = 0; t < nt; ++t) s += prod[tid][t];
    __syncthreads();
  }
  if (tid < np) y[p0 + tid] = float(s);
}

// x_t = y * phi_t on (H,W,T) arrays; 256 pixels a block.
template <bool VEC>
__global__ void __launch_bounds__(kThreads) k_adjoint_hwt(const float* __restrict__ y,
                                                          const float* __restrict__ phi,
                                                          float* __restrict__ x, int64_t N,
                                                          int T) {
  __shared__ float ys[kThreads];
  const int64_t p0 = int64_t(blockIdx.x) * kThreads;
  const int tid = threadIdx.x;
  const int64_t base = p0 * T;
  const int64_t n = (p0 + kThreads <= N ? kThreads : N - p0) * int64_t(T);
  if (p0 + tid < N) ys[tid] = y[p0 + tid];
  __syncthreads();
  int64_t done = 0;
  if constexpr (VEC) {
    const float4* const fv = reinterpret_cast<const float4*>(phi + base);
    float4* const xv = reinterpret_cast<float4*>(x + base);
    for (unsigned i = tid; i < unsigned(n / 4); i += kThreads) {
      const float4 f = fv[i];
      unsigned p = 4 * i / unsigned(T), r = 4 * i - p * unsigned(T);
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        v[k] = ys[p];
        if (++r == unsigned(T)) {
          r = 0;
          p = p < kThreads - 1 ? p + 1 : p;
        }
      }
      xv[i] = make_float4(v[0] * f.x, v[1] * f.y, v[2] * f.z, v[3] * f.w);
    }
    done = n & ~int64_t(3);
  }
  for (int64_t i = done + tid; i < n; i += kThreads) x[base + i] = ys[i / T] * phi[base + i];
}

// (H,W,T) <-> (T,H,W).  FROM_HWT: src is (H,W,T).  P = 1 << logp pixels a
// block.  Vector accesses on both sides (host: N % 4 == 0, 16-byte pointers),
// full blocks only; the last block and other shapes go element by element.
template <bool FROM_HWT, bool VEC>
__global__ void __launch_bounds__(kThreads) k_relayout(const float* __restrict__ src,
                                                       float* __restrict__ dst, int64_t N, int T,
                                                       int logp) {
  extern __shared__ float buf[];
  const int P = 1 << logp, tid = threadIdx.x;
  const int64_t p0 = int64_t(blockIdx.x) * P, base = p0 * T;
  const int np = int(p0 + P <= N ? P : N - p0), n = np * T;
  const bool vec = VEC && np == P;
  // The (T,H,W) side: element i is frame i / P of pixel i % P.
  auto frames = [&](auto&& one) __attribute__((always_inline)) {
    for (int i = tid; i < P * T; i += kThreads) {
      const int t = i >> logp, q = i & (P - 1);
      if (q < np) one(t, q);
    }
  };
  auto frames4 = [&](auto&& four) __attribute__((always_inline)) {
    for (int i = tid; i < n / 4; i += kThreads)
      four(i >> (logp - 2), 4 * (i & ((P >> 2) - 1)));
  };
  if constexpr (FROM_HWT) {
    if (vec) {
      const float4* const v = reinterpret_cast<const float4*>(src + base);
      for (int i = tid; i < n / 4; i += kThreads) {
        const float4 a = v[i];
        buf[pad32(4 * i)] = a.x;
        buf[pad32(4 * i + 1)] = a.y;
        buf[pad32(4 * i + 2)] = a.z;
        buf[pad32(4 * i + 3)] = a.w;
      }
    } else {
      for (int i = tid; i < n; i += kThreads) buf[pad32(i)] = src[base + i];
    }
    __syncthreads();
    if (vec)
      frames4([&](int t, int q) {
        *reinterpret_cast<float4*>(dst + t * N + p0 + q) =
            make_float4(buf[pad32(q * T + t)], buf[pad32((q + 1) * T + t)],
                        buf[pad32((q + 2) * T + t)], buf[pad32((q + 3) * T + t)]);
      });
    else
      frames([&](int t, int q) { dst[t * N + p0 + q] = buf[pad32(q * T + t)]; });
  } else {
    if (vec)
      frames4([&](int t, int q) {
        const float4 a = *reinterpret_cast<const float4*>(src + t * N + p0 + q);
        buf[pad32(q * T + t)] = a.x;
        buf[pad32((q + 1) * T + t)] = a.y;
        buf[pad32((q + 2) * T + t)] = a.z;
        buf[pad32((q + 3) * T + t)] = a.w;
      });
    else
      frames([&](int t, int q) { buf[pad32(q * T + t)] = src[t * N + p0 + q]; });
    __syncthreads();
    if (vec) {
      float4* const v = reinterpret_cast<float4*>(dst + base);
      for (int i = tid; i < n / 4; i += kThreads)
        v[i] = make_float4(buf[pad32(4 * i)], buf[pad32(4 * i + 1)], buf[pad32(4 * i + 2)],
                           buf[pad32(4 * i + 3)]);
    } else {
      for (int i = tid; i < n; i += kThreads) dst[base + i] = buf[pad32(i)];
    }
  }
}

__global__ void k_fill_f64(double* p, int n, double v) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// sum((a-b)^2) over n contiguous elements per slice; slice = blockIdx.y.
__global__ void __launch_bounds__(kThreads) k_sq_error(const float* __restrict__ a,
                                                       const float* __restrict__ b,
                                                       double* __restrict__ out, int64_t n,
                                                       int per_slice_out) {
  const int64_t base = int64_t(blockIdx.y) * n;
  // As scikit-image's mean_squared_error for float32 images: the difference
  // is squared in fp32 and the squares are accumulated in fp64.
  double acc = 0.0;
  for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * blockDim.x) {
    const float d = a[base + i] - b[base + i];
    acc += double(d * d);
  }
  double s = wave_sum(acc);
  __shared__ double part[kThreads / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0;
    for (int w = 0; w < kThreads / 64; ++w) tot += part[w];
    atomicAdd(out + (per_slice_out ? blockIdx.y : 0), tot);
  }
}

// Per-frame SSIM sum over the interior pixels [3,H-3) x [3,W-3); fp64 like
// scikit-image (which converts both images to float64).  A 7x7 window
// centred on an interior pixel never leaves the image, so the reflect
// boundary of scipy's uniform_filter does not enter the cropped mean.
//
// Bound by fp64 arithmetic (4.4 cycles an instruction): a lane walks kSR rows
// of one column with the window's seven row sums of x, y, x^2, y^2 and x*y in
// registers, so each row costs seven taps, not 49.  253x317x7: 13.4 us,
// with all 49 taps per centre 33.7.  The walk ends with the last centre:
// in a stack of small frames most rows of a workgroup are beyond it.
constexpr int kSW = 4;  // waves per workgroup, one above the other
constexpr int kSR = 8;  // window centres per lane
__global__ void __launch_bounds__(64 * kSW) k_ssim(const float* __restrict__ a,
                                                   const float* __restrict__ b,
                                                   double* __restrict__ out, int H, int W,
                                                   double c1, double c2, double scale) {
  const int t = blockIdx.z;
  const size_t N = size_t(H) * W;
  const float* fa = a + t * N;
  const float* fb = b + t * N;
  const int w = threadIdx.x >> 6;
  const int c = 3 + blockIdx.x * 64 + (threadIdx.x & 63);
  const int r0 = 3 + (blockIdx.y * kSW + w) * kSR;  // first centre
  const int cc = c < W - 3 ? c : W - 4;             // (lanes beyond add nothing)
  double s = 0.0;
  double ring[7][5];
  auto row_step = [&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    const int row = r0 - 3 + i;
    const float* pa = fa + size_t(row) * W + cc - 3;
    const float* pb = fb + size_t(row) * W + cc - 3;
    double q[5] = {};
#pragma unroll
    for (int d = 0; d < 7; ++d) {
      const double x = pa[d], y = pb[d];
      q[0] += x;
      q[1] += y;
      q[2] = fma(x, x, q[2]);
      q[3] = fma(y, y, q[3]);
      q[4] = fma(x, y, q[4]);
    }
#pragma unroll
    for (int k = 0; k < 5; ++k) ring[i % 7][k] = q[k];
    if constexpr (i >= 6) {
      double m[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        m[k] = ring[0][k];
#pragma unroll
        for (int e = 1; e < 7; ++e) m[k] += ring[e][k];
      }
      const double np = 49.0, cov = np / (np - 1.0);
      const double ux = m[0] / np, uy = m[1] / np;
      const double vx = cov * (m[2] / np - ux * ux);
      const double vy = cov * (m[3] / np - uy * uy);
      const double vxy = cov * (m[4] / np - ux * uy);
      const double a1 = 2 * ux * uy + c1, a2 = 2 * vxy + c2;
      const double b1 = ux * ux + uy * uy + c1, b2 = vx + vy + c2;
      const double v = (a1 * a2) / (b1 * b2);
      if (c < W - 3) s += v;
    }
  };
  if (r0 + kSR <= H - 3)
    static_for<kSR + 6>(row_step);
  else  // the last rows, if any
    static_for<kSR + 6>([&](auto ic) __attribute__((always_inline)) {
      if (r0 < H - 3 && r0 - 3 + decltype(ic)::value < H) row_step(ic);
    });
  s = wave_sum(s);
  __shared__ double part[kSW];
  if ((threadIdx.x & 63) == 0) part[w] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0;
    for (int i = 0; i < kSW; ++i) tot += part[i];
    atomicAdd(out + t, tot * scale);
  }
}


}  // namespace

// Fill n doubles with v on `stream` (graph-capturable, unlike a memset node).
int fill_f64(double* p, int n, double v, hipStream_t s) {
  if (n <= 0) return SCIGAP_OK;
  k_fill_f64<<<(n + 255) / 256, 256, 0, s>>>(p, n, v);
  SCIGAP_LAUNCH_CHECK("fill kernel launch");
  return SCIGAP_OK;
}

}  // namespace scigap

using namespace scigap;

extern "C" {

int scigap_version(void) { return 10000; }

const char* scigap_last_error(void) { return scigap::g_err; }

int scigap_forward(const float* x, const float* phi, float* y, int64_t H, int64_t W, int64_t T,
                   void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!x || !phi || !y) return fail(SCIGAP_ENULL, "scigap_forward: null pointer");
  const int64_t N = H * W;
  if (overlaps(y, N * 4, x, N * T * 4) || overlaps(y, N * 4, phi, N * T * 4))
    return fail(SCIGAP_EALIAS, "scigap_forward: y overlaps an input");
  hipStream_t s = as_stream(stream);
  bool vec = (N % 4 == 0) && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(phi) |
                               reinterpret_cast<uintptr_t>(y)) % 16 == 0);
  if (vec)
    k_forward<4><<<grid_for(N / 4), kThreads, 0, s>>>(x, phi, y, N, int(T));
  else
    k_forward<1><<<grid_for(N), kThreads, 0, s>>>(x, phi, y, N, int(T));
  SCIGAP_LAUNCH_CHECK("scigap_forward launch");
  return SCIGAP_OK;
}

int scigap_adjoint(const float* y, const float* phi, float* x, int64_t H, int64_t W, int64_t T,
                   void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!x || !phi || !y) return fail(SCIGAP_ENULL, "scigap_adjoint: null pointer");
  const int64_t N = H * W;
  if (overlaps(x, N * T * 4, y, N * 4) || overlaps(x, N * T * 4, phi, N * T * 4))
    return fail(SCIGAP_EALIAS, "scigap_adjoint: x overlaps an input");
  hipStream_t s = as_stream(stream);
  bool vec = (N % 4 == 0) && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(phi) |
                               reinterpret_cast<uintptr_t>(y)) % 16 == 0);
  if (vec)
    k_adjoint<4><<<grid_for(N / 4), kThreads, 0, s>>>(y, phi, x, N, int(T));
  else
    k_adjoint<1><<<grid_for(N), kThreads, 0, s>>>(y, phi, x, N, int(T));
  SCIGAP_LAUNCH_CHECK("scigap_adjoint launch");
  return SCIGAP_OK;
}

int scigap_phi_sum(const float* phi, float* phi_sum, int64_t H, int64_t W, int64_t T,
                   void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!phi || !phi_sum) return fail(SCIGAP_ENULL, "scigap_phi_sum: null pointer");
  const int64_t N = H * W;
  if (overlaps(phi_sum, N * 4, phi, N * T * 4))
    return fail(SCIGAP_EALIAS, "scigap_phi_sum: output overlaps phi");
  k_phi_sum<<<grid_for(N), kThreads, 0, as_stream(stream)>>>(phi, phi_sum, N, int(T));
  SCIGAP_LAUNCH_CHECK("scigap_phi_sum launch");
  return SCIGAP_OK;
}

int scigap_forward_hwt(const float* x, const float* phi, float* y, int64_t H, int64_t W, int64_t T,
                       void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!x || !phi || !y) return fail(SCIGAP_ENULL, "scigap_forward_hwt: null pointer");
  const int64_t N = H * W;
  if (overlaps(y, N * 4, x, N * T * 4) || overlaps(y, N * 4, phi, N * T * 4))
    return fail(SCIGAP_EALIAS, "scigap_forward_hwt: y overlaps an input");
  hipStream_t s = as_stream(stream);
  const int P = forward_pixels(T);
  if (P == 0) {
    k_forward_hwt_many<<<unsigned((N + kThreads - 1) / kThreads), kThreads, 0, s>>>(x, phi, y, N,
                                                                               int(T));
  } else {
    const unsigned blocks = unsigned((N + P - 1) / P);
    const bool vec =
        (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(phi)) % 16 == 0;
    if (vec)
      k_forward_hwt<true><<<blocks, P, hwt_lds(P, T, 8), s>>>(x, phi, y, N, int(T));
    else
      k_forward_hwt<false><<<blocks, P, hwt_lds(P, T, 8), s>>>(x, phi, y, N, int(T));
  }
  SCIGAP_LAUNCH_CHECK("scigap_forward_hwt launch");
  return SCIGAP_OK;
}

int scigap_adjoint_hwt(const float* y, const float* phi, float* x, int64_t H, int64_t W, int64_t T,
                       void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!x || !phi || !y) return fail(SCIGAP_ENULL, "scigap_adjoint_hwt: null pointer");
  const int64_t N = H * W;
  if (overlaps(x, N * T * 4, y, N * 4) || overlaps(x, N * T * 4, phi, N * T * 4))
    return fail(SCIGAP_EALIAS, "scigap_adjoint_hwt: x overlaps an input");
  hipStream_t s = as_stream(stream);
  const unsigned blocks = unsigned((N + kThreads - 1) / kThreads);
  const bool vec = (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(phi)) % 16 == 0;
  if (vec)
    k_adjoint_hwt<true><<<blocks, kThreads, 0, s>>>(y, phi, x, N, int(T));
  else
    k_adjoint_hwt<false><<<blocks, kThreads, 0, s>>>(y, phi, x, N, int(T));
  SCIGAP_LAUNCH_CHECK("scigap_adjoint_hwt launch");
  return SCIGAP_OK;
}

// (H,W,T) <-> (T,H,W) through k_relayout; false where its pixels do not fit the
// LDS (over 240 frames) and where the 32x32 tiles of k_transpose, which such
// frame counts fill, are the better: from about 112 frames on where single
// elements are moved, since blocks then begin and end inside lines (1001x701x96:
// 180 us, in tiles 184; x128: 286 / 244; with 16-byte accesses 1024x1024x128:
// 204 / 276).  Blocks of few pixels, so that 8 or more share a CU: of
// 1001x701x64 with up to 40 KB of pixels a block 151 us, with as many threads
// as pixels besides 224, with 10 KB and 256 threads 106.
static bool relayout(bool from_hwt, const float* src, float* dst, int64_t N, int64_t T,
                     hipStream_t s) {
  const bool vec = N % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) % 16 == 0;
  if (T > (vec ? 240 : 112)) return false;
  int logp = 8;
  while (logp > 6 && (T << logp) * 4 > 10 * 1024) --logp;
  const unsigned blocks = unsigned((N + (1 << logp) - 1) >> logp);
  const size_t lds = hwt_lds(1 << logp, T, 4);
  if (from_hwt) {
    if (vec)
      k_relayout<true, true><<<blocks, kThreads, lds, s>>>(src, dst, N, int(T), logp);
    else
      k_relayout<true, false><<<blocks, kThreads, lds, s>>>(src, dst, N, int(T), logp);
  } else {
    if (vec)
      k_relayout<false, true><<<blocks, kThreads, lds, s>>>(src, dst, N, int(T), logp);
    else
      k_relayout<false, false><<<blocks, kThreads, lds, s>>>(src, dst, N, int(T), logp);
  }
  return true;
}

static int transpose(const float* src, float* dst, int64_t rows, int64_t cols, void* stream,
                     const char* name) {
  if (!src || !dst) return fail(SCIGAP_ENULL, "%s: null pointer", name);
  if (overlaps(src, rows * cols * 4, dst, rows * cols * 4))
    return fail(SCIGAP_EALIAS, "%s: src and dst overlap", name);
  // One side of the matrix is the frame axis: rows = H*W for (H,W,T) -> (T,H,W).
  const bool from_hwt = rows >= cols;
  if (relayout(from_hwt, src, dst, from_hwt ? rows : cols, from_hwt ? cols : rows,
               as_stream(stream))) {
    SCIGAP_LAUNCH_CHECK(name);
    return SCIGAP_OK;
  }
  int64_t gx = (cols + TT - 1) / TT, gy = (rows + TT - 1) / TT;
  if (gx > (int64_t(1) << 31) - 1) return fail(SCIGAP_EINVAL, "%s: volume too large", name);
  if (gy > 65535) gy = 65535;
  k_transpose<<<dim3(unsigned(gx), unsigned(gy)), TT * 8, 0, as_stream(stream)>>>(src, dst, rows,
                                                                                 cols);
  SCIGAP_LAUNCH_CHECK(name);
  return SCIGAP_OK;
}

int scigap_hwt_to_thw(const float* src, float* dst, int64_t H, int64_t W, int64_t T,
                      void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (T == 1) {
    if (!src || !dst) return fail(SCIGAP_ENULL, "scigap_hwt_to_thw: null pointer");
    hipError_t e = hipMemcpyAsync(dst, src, H * W * 4, hipMemcpyDeviceToDevice, as_stream(stream));
    return e == hipSuccess ? SCIGAP_OK : hip_fail(e, "scigap_hwt_to_thw copy");
  }
  return transpose(src, dst, H * W, T, stream, "scigap_hwt_to_thw");
}

int scigap_thw_to_hwt(const float* src, float* dst, int64_t H, int64_t W, int64_t T,
                      void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (T == 1) {
    if (!src || !dst) return fail(SCIGAP_ENULL, "scigap_thw_to_hwt: null pointer");
    hipError_t e = hipMemcpyAsync(dst, src, H * W * 4, hipMemcpyDeviceToDevice, as_stream(stream));
    return e == hipSuccess ? SCIGAP_OK : hip_fail(e, "scigap_thw_to_hwt copy");
  }
  return transpose(src, dst, T, H * W, stream, "scigap_thw_to_hwt");
}

int scigap_sq_error(const float* a, const float* b, double* out, int64_t H, int64_t W, int64_t T,
                    int per_frame, void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!a || !b || !out) return fail(SCIGAP_ENULL, "scigap_sq_error: null pointer");
  hipStream_t s = as_stream(stream);
  const int64_t N = H * W;
  if (int rc = fill_f64(out, per_frame ? int(T) : 1, 0.0, s)) return rc;
  if (per_frame) {
    unsigned gx = grid_for(N) / unsigned(T) + 1;
    if (gx > 1024) gx = 1024;
    k_sq_error<<<dim3(gx, unsigned(T)), kThreads, 0, s>>>(a, b, out, N, 1);
  } else {
    k_sq_error<<<dim3(grid_for(N * T), 1), kThreads, 0, s>>>(a, b, out, N * T, 0);
  }
  SCIGAP_LAUNCH_CHECK("scigap_sq_error launch");
  return SCIGAP_OK;
}

int scigap_ssim(const float* a, const float* b, double* out, int64_t H, int64_t W, int64_t T,
                float data_range, void* stream) {
  clear_error();
  if (int rc = check_shape(H, W, T)) return rc;
  if (!a || !b || !out) return fail(SCIGAP_ENULL, "scigap_ssim: null pointer");
  if (H < 7 || W < 7) return fail(SCIGAP_EINVAL, "win_size exceeds image extent (H, W >= 7 needed)");
  hipStream_t s = as_stream(stream);
  if (int rc = fill_f64(out, int(T), 0.0, s)) return rc;
  const double R = data_range, c1 = (0.01 * R) * (0.01 * R), c2 = (0.03 * R) * (0.03 * R);
  dim3 grid(unsigned((W - 6 + 63) / 64), unsigned((H - 6 + kSW * kSR - 1) / (kSW * kSR)),
            unsigned(T));
  k_ssim<<<grid, 64 * kSW, 0, s>>>(a, b, out, int(H), int(W), c1, c2,
                                   1.0 / (double(H - 6) * double(W - 6)));
  SCIGAP_LAUNCH_CHECK("scigap_ssim launch");
  return SCIGAP_OK;
}

}  // extern "C"
