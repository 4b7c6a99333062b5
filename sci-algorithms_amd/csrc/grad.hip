// Reverse-mode kernels of the unrolled, differentiable GAP-TV.
//
// Model (per sample; Phi is shared by the batch):
//   y     = sum_t Phi_t * truth_t            (or a given measurement)
//   S     = sum_t Phi_t
//   x_0   = Phi * y,  y1_0 = 0
//   for k < K:  yb = sum_t Phi_t x_k,  y1' = y1_k + (y - yb),
//               r = (y1' - yb)/S,  v = x_k + lambda_k * r * Phi,
//               x_{k+1} = TV_{w_k}(v)  (D = tv_iter_max-1 Chambolle updates,
//                                        no early exit)
// which is PnP_SCI/python/pnp_sci_algo.py:625-650 (accelerated GAP) with the
// TV step of scikit-image 0.18.3 _denoise.py:341-393 run for a fixed number
// of iterations, and per-iteration lambda_k / tv_weight_k.
//
// One Chambolle update, with G the forward difference (zero in the last row /
// column) and G^T its transpose (the "d" of _denoise.py:352-361):
//   out_u = v + G^T p_u,  g_u = G out_u,  n_u = |g_u|,  s_u = 1/(1 + c n_u),
//   a_u = p_u - tau g_u,  p_{u+1} = a_u * s_u,   c = tau / w,  tau = 1/4.
// Reverse of one update, given pbar_{u+1}:
//   abar_u = pbar_{u+1} * s_u,   sbar = <pbar_{u+1}, a_u>,
//   nbar = -c s_u^2 sbar,  cbar += -n_u s_u^2 sbar,
//   gbar_u = -tau abar_u + nbar g_u / n_u   (0 where n_u = 0),
//   obar_u = G^T gbar_u,  vbar += obar_u,  pbar_u = abar_u + G obar_u.
// The TV output out_D = v + G^T p_D starts the chain: vbar = xbar, pbar_D = G xbar.
//
// Activations are checkpointed once per outer iteration (x_k, y1' and the
// residual r_k the forward used); the TV step of one outer iteration is
// reversed by one fused tiled kernel (tv_bwd.hip) that forms v from x_k, r_k
// and Phi as the forward did and recomputes the inner dual fields in
// registers.  Layout (T,H,W) per sample.

#include <cmath>
#include <initializer_list>

#include "scigap_internal.h"

namespace scigap {

namespace {

constexpr int kThreads = 256;
constexpr int kSamples = 4;   // samples of one launch (a group), as a rule
constexpr int kSamplesMax = 8;

// Block reduction of one float into a gradient accumulator's slot.
__device__ __forceinline__ void block_atomic(float v, double* dst) {
  const float s = wave_sum(v);
  __shared__ float part[kThreads / 64];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int w = 0; w < kThreads / 64; ++w) tot += part[w];
    atomicAdd(grad_slot(dst), tot);
  }
}

// V consecutive floats of a plane.
template <int V>
struct Vec {
  float v[V];
};
template <int V>
__device__ __forceinline__ Vec<V> ldv(const float* p, int64_t i) {
  Vec<V> r;
  if constexpr (V == 4) {
    const float4 f = reinterpret_cast<const float4*>(p)[i];
    r.v[0] = f.x, r.v[1] = f.y, r.v[2] = f.z, r.v[3] = f.w;
  } else {
    r.v[0] = p[i];
  }
  return r;
}
template <int V>
__device__ __forceinline__ void stv(float* p, int64_t i, const Vec<V>& r) {
  if constexpr (V == 4)
    reinterpret_cast<float4*>(p)[i] = make_float4(r.v[0], r.v[1], r.v[2], r.v[3]);
  else
    p[i] = r.v[0];
}

// Reverse of the projection v = x + lambda*r*Phi, r = (y1' - yb)/S,
// y1' = y1 + y - yb, yb = sum_t Phi_t x_t (per pixel, all frames), given
// vbar = dL/dv.  The per-pixel part only: rbar = lambda sum_t vbar_t Phi_t,
// lambar += sum vbar r Phi, y1bar' = y1bar_next + rbar/S, ybb = -rbar/S - y1bar',
// ybar += y1bar', Sbar = -rbar r / S.  The frame part xbar_t = vbar_t + ybb Phi_t
// is never stored: the next reverse TV step forms it on load, and the mask
// gradient (k_ub_phibar) takes ybb and Sbar from the planes written here.
// blockIdx.y is the sample; planes of N, volumes of N*T floats per sample, r
// at its own distance.
//
// Memory-bound: V = 4 (16 bytes a lane) where that leaves waves enough; the
// loads of G frames are issued together (one memory latency per group), the
// sums keep frame order.  2 x 1024x1024x20: 58 us, against 78 us for each of two
// concurrent launches of one sample with one pixel a lane; 4 x 256x256x8: 6.5 us.
struct ProjArgs {
  const float* vbar;
  const float* phi;
  const float* S;
  const float* r;
  size_t r_b;
  float lam;
  const float* y1bar_in;  // null: 0
  float* y1bar_out;
  float* ybar;
  float* ybb;
  float* sbar;  // null: no mask gradient
  double* lambar;
  int64_t N;
  int T;
};

template <int V, int G>
__global__ void __launch_bounds__(kThreads) k_ub_proj(ProjArgs a) {
  const int b = blockIdx.y;
  const int64_t n = a.N / V;
  const size_t pl = size_t(b) * a.N;
  const float* const vbar = a.vbar + size_t(b) * a.N * a.T;
  float lsum = 0.f;
  for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * kThreads) {
    const Vec<V> ri = ldv<V>(a.r + b * a.r_b, i), si = ldv<V>(a.S, i);
    Vec<V> yb = ldv<V>(a.ybar + pl, i), y1{};
    if (a.y1bar_in) y1 = ldv<V>(a.y1bar_in + pl, i);
    double rsum[V] = {};
    float fsum[V] = {};
    for (int t0 = 0; t0 < a.T; t0 += G) {
      Vec<V> vb[G], f[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int t = t0 + g < a.T ? t0 + g : a.T - 1;
        vb[g] = ldv<V>(vbar + size_t(t) * a.N, i);
        f[g] = ldv<V>(a.phi + size_t(t) * a.N, i);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        if (t0 + g >= a.T) break;
#pragma unroll
        for (int k = 0; k < V; ++k) {
          rsum[k] = acc_prod(vb[g].v[k], f[g].v[k], rsum[k]);
          fsum[k] += f[g].v[k];
        }
      }
    }
    Vec<V> y1o, ybb, sb;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      float rbar = float(rsum[k]);
      lsum = fmaf(rbar, ri.v[k], lsum);  // dL/dlambda = sum_t vbar*r*Phi
      rbar *= a.lam;
      y1o.v[k] = y1.v[k] + rbar / si.v[k];
      yb.v[k] += y1o.v[k];
      ybb.v[k] = -rbar / si.v[k] - y1o.v[k];
      // S = sum_t Phi_t, except where that sum is 0 and S is the constant 1.
      sb.v[k] = fsum[k] != 0.f ? -rbar * ri.v[k] / si.v[k] : 0.f;
    }
    stv<V>(a.y1bar_out + pl, i, y1o);
    stv<V>(a.ybar + pl, i, yb);
    stv<V>(a.ybb + pl, i, ybb);
    if (a.sbar) stv<V>(a.sbar + pl, i, sb);
  }
  block_atomic(lsum, a.lambar);
}

// Mask gradient of one projection: phibar_t += sum over the group's samples of
// lambda r vbar_t + ybb x_t + Sbar.  One thread per pixel and frame
// (blockIdx.y), one pass over phibar for the whole group.
template <int V>
__global__ void __launch_bounds__(kThreads) k_ub_phibar(
    const float* __restrict__ vbar, const float* __restrict__ x, size_t x_b,
    const float* __restrict__ r, size_t r_b, float lam, const float* __restrict__ ybb,
    const float* __restrict__ sbar, float* __restrict__ phibar, int64_t N, int T, int nb) {
  const int64_t n = N / V;
  const size_t fr = size_t(blockIdx.y) * N;
  for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < n;
       i += int64_t(gridDim.x) * kThreads) {
    Vec<V> acc = ldv<V>(phibar + fr, i);
    for (int b = 0; b < nb; ++b) {
      const size_t pl = size_t(b) * N;
      const Vec<V> ri = ldv<V>(r + b * r_b, i), yb = ldv<V>(ybb + pl, i), sb = ldv<V>(sbar + pl, i);
      const Vec<V> vb = ldv<V>(vbar + pl * T + fr, i), xv = ldv<V>(x + b * x_b + fr, i);
#pragma unroll
      for (int k = 0; k < V; ++k)
        acc.v[k] += fmaf(lam * ri.v[k], vb.v[k], fmaf(yb.v[k], xv.v[k], sb.v[k]));
    }
    stv<V>(phibar + fr, i, acc);
  }
}

// End of the backward pass of a group.  Reverse of x_0 = Phi*y and, with
// truth, of y = sum_t Phi_t truth_t: with xbar_0 = vbar + ybb Phi,
//   ybar += sum_t xbar_0 Phi  (k_ub_end_y, blockIdx.y = sample),
//   phibar += xbar_0 y (+ ybar truth)  (k_ub_end_phi, blockIdx.y = frame);
// the last group writes the mask gradient itself (logits: times Phi (1 - Phi))
// and the lambda and weight gradients from their slots.
struct EndArgs {
  const float* vbar;
  const float* ybb;
  const float* phi;
  const float* y;
  size_t y_b;
  float* ybar;
  float* phibar;
  const float* truth;  // null: y was given
  float* grad_mask;    // last group only, else null
  int64_t N;
  int T, nb, logits;
  // last group only, else K = 0
  const double* slots;
  double* grad_lambda;
  double* grad_weight;
  int K;
};

__global__ void __launch_bounds__(kThreads) k_ub_end_y(EndArgs a) {
  const int b = blockIdx.y;
  const size_t pl = size_t(b) * a.N;
  for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < a.N;
       i += int64_t(gridDim.x) * kThreads) {
    const float yb = a.ybb[pl + i];
    double acc = 0.0;
#pragma unroll 8
    for (int t = 0; t < a.T; ++t) {
      const float f = a.phi[size_t(t) * a.N + i];
      acc = acc_prod(fmaf(yb, f, a.vbar[pl * a.T + size_t(t) * a.N + i]), f, acc);
    }
    a.ybar[pl + i] += float(acc);
  }
  if (b == 0)  // lambda and weight gradient of iteration k: the sums of their slots
    for (int k = blockIdx.x * kThreads + threadIdx.x; k < a.K; k += gridDim.x * kThreads) {
      double gl = 0.0, gw = 0.0;
      for (int j = 0; j < kGradSlots; ++j) {
        gl += a.slots[(size_t(k) * 2 * kGradSlots + j) * kGradSlotStride];
        gw += a.slots[((size_t(k) * 2 + 1) * kGradSlots + j) * kGradSlotStride];
      }
      a.grad_lambda[k] = gl;
      a.grad_weight[k] = gw;
    }
}

__global__ void __launch_bounds__(kThreads) k_ub_end_phi(EndArgs a) {
  const size_t fr = size_t(blockIdx.y) * a.N;
  for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < a.N;
       i += int64_t(gridDim.x) * kThreads) {
    const float f = a.phi[fr + i];
    float g = a.phibar[fr + i];
    for (int b = 0; b < a.nb; ++b) {
      const size_t pl = size_t(b) * a.N, vo = pl * a.T + fr + i;
      g = fmaf(fmaf(a.ybb[pl + i], f, a.vbar[vo]), a.y[b * a.y_b + i], g);
      if (a.truth) g = fmaf(a.ybar[pl + i], a.truth[vo], g);
    }
    if (a.grad_mask)
      a.grad_mask[fr + i] = a.logits ? g * f * (1.f - f) : g;
    else
      a.phibar[fr + i] = g;
  }
}

// Zeroes of a backward pass in one launch.
__global__ void k_zero(float* p, int64_t n, float* q, int64_t m, double* slots, int64_t ns) {
  const int64_t first = blockIdx.x * int64_t(blockDim.x) + threadIdx.x;
  const int64_t step = int64_t(gridDim.x) * blockDim.x;
  for (int64_t i = first; i < n; i += step) p[i] = 0.f;
  for (int64_t i = first; i < m; i += step) q[i] = 0.f;
  for (int64_t i = first; i < ns; i += step) slots[i] = 0.0;
}

unsigned grid1(int64_t n) {
  int64_t b = (n + 255) / 256;
  return unsigned(b < 1 ? 1 : (b > 4096 ? 4096 : b));
}

// phi = sigmoid(logits) when asked, and S = sum_t phi_t in frame order (a sum
// of 0 becomes 1), as scigap_phi_sum forms it.
__global__ void __launch_bounds__(kThreads) k_mask(const float* __restrict__ mask,
                                                   float* __restrict__ phi,
                                                   float* __restrict__ S, int64_t N, int T) {
  for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < N;
       i += int64_t(gridDim.x) * kThreads) {
    float acc = 0.f;
#pragma unroll 4
    for (int t = 0; t < T; ++t) {
      const size_t o = size_t(t) * N + i;
      float f = mask[o];
      if (phi) {
        f = 1.f / (1.f + expf(-f));
        phi[o] = f;
      }
      acc += f;
    }
    S[i] = acc == 0.f ? 1.f : acc;
  }
}

// Start of the forward pass, blockIdx.y = sample: y = sum_t Phi_t truth_t (or
// the given measurement), x_0 = Phi y, yb = A x_0, y1 = y - yb,
// r_0 = (y1 - yb)/S (the arithmetic of scigap_forward, scigap_adjoint and
// k_init).
struct StartArgs {
  const float* meas;
  int measure;
  const float* phi;
  const float* S;
  float* y;
  size_t y_b;
  float* x0;
  size_t x_b;
  float* r;
  size_t r_b;
  float* y1;
  size_t y1_b;
  int64_t N;
  int T;
};

__global__ void __launch_bounds__(kThreads) k_unrolled_start(StartArgs a) {
  const int b = blockIdx.y;
  const float* const meas = a.meas + size_t(b) * a.N * (a.measure ? a.T : 1);
  for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < a.N;
       i += int64_t(gridDim.x) * kThreads) {
    float y;
    if (a.measure) {
      double acc = 0.0;
#pragma unroll 4
      for (int t = 0; t < a.T; ++t)
        acc = acc_prod(meas[size_t(t) * a.N + i], a.phi[size_t(t) * a.N + i], acc);
      y = float(acc);
    } else {
      y = meas[i];
    }
    a.y[b * a.y_b + i] = y;
    double acc = 0.0;
#pragma unroll 4
    for (int t = 0; t < a.T; ++t) {
      const float f = a.phi[size_t(t) * a.N + i];
      const float x = y * f;
      a.x0[b * a.x_b + size_t(t) * a.N + i] = x;
      acc = acc_prod(x, f, acc);
    }
    const float yb = float(acc), y1 = y - yb;
    a.y1[b * a.y1_b + i] = y1;
    a.r[b * a.r_b + i] = (y1 - yb) / a.S[i];
  }
}

// Whether the per-pixel kernels take 4 pixels a lane: planes whose start and
// distances keep 16-byte alignment, and enough of them (at 1024x1024x20 the
// projection reverse takes 60-80 us with one pixel a lane; 4 pixels of a
// 256x256 plane would leave 3 of 4 SIMDs without a wave).
bool proj_vector(int64_t N, std::initializer_list<const void*> ptrs,
                 std::initializer_list<size_t> dists) {
  if (N % 4 != 0 || N < (int64_t(1) << 19)) return false;
  for (const void* p : ptrs)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
  for (size_t d : dists)
    if (d % 4 != 0) return false;
  return true;
}

}  // namespace

int64_t tv_backward_rounds(int D, int nb, int64_t H, int64_t W, int64_t T);
int tv_backward_tiles(int D, int nb, const float* x, size_t x_b, const float* phi, const float* r,
                      size_t r_b, float lam, const float* xbar, size_t xbar_b, const float* ybb,
                      size_t ybb_b, float* vbar, size_t vbar_b, int64_t H, int64_t W, int64_t T,
                      float w, double* wbar, hipStream_t s);

namespace {

// Scratch of the backward pass of a group of nb samples.
struct BwdScratch {
  float* vbar[2];
  float* y1bar[2];
  float* ybb[2];
  float* sbar;
  float* ybar;
};

size_t bwd_scratch(int64_t H, int64_t W, int64_t T, int nb, char* base, BwdScratch* out) {
  const size_t N = size_t(H) * W * nb, V = N * size_t(T);
  size_t off = 0;
  auto take = [&](size_t n) {
    float* q = base ? reinterpret_cast<float*>(base + off) : nullptr;
    off += align256(n * 4);
    return q;
  };
  BwdScratch b;
  for (auto& p : b.vbar) p = take(V);
  for (auto& p : b.y1bar) p = take(N);
  for (auto& p : b.ybb) p = take(N);
  b.sbar = take(N);
  b.ybar = take(N);
  if (out) *out = b;
  return off;
}

// Where the forward pass left a group's samples (the first one's planes and
// the distances to the next, in floats).
struct GroupCkpt {
  const float* x;
  size_t xstride, x_b;
  const float* r;
  size_t rstride, r_b;
  const float* y;
  size_t y_b;
};

// Backward through K unrolled iterations of nb samples.  phibar (null: no mask
// gradient) accumulates; grad_mask, grad_lambda and grad_weight are written by
// the last group.
int unrolled_backward(int64_t H, int64_t W, int64_t T, int K, int D, int nb, const float* lambdas,
                      const float* weights, const GroupCkpt& c, const float* phi, const float* S,
                      const float* grad_x, const float* truth, float* phibar, float* grad_mask,
                      int logits, bool last, double* slots, double* grad_lambda,
                      double* grad_weight, const BwdScratch& w, hipStream_t s) {
  const int64_t N = H * W;
  const size_t V = size_t(N) * T;
  // Adjoint of x_{k+1}: grad_x for k = K-1, else vbar_{k+1} + ybb_{k+1} Phi
  // (formed on load by the reverse TV step and by k_ub_end).
  const float* vb_in = grad_x;
  const float* ybb_in = nullptr;
  const float* y1b_in = nullptr;
  int sel = 0;
  for (int k = K - 1; k >= 0; --k) {
    const float lam = lambdas[k];
    const float* xk = c.x + size_t(k) * c.xstride;
    const float* r = c.r + size_t(k) * c.rstride;  // residual the forward used
    {
      ProfScope ps("unrolled_bwd_tv", s);
      if (int rc = tv_backward_tiles(D, nb, xk, c.x_b, phi, r, c.r_b, lam, vb_in, V, ybb_in,
                                     size_t(N), w.vbar[sel], V, H, W, T, weights[k],
                                     slots + size_t(2 * k + 1) * kGradSlots * kGradSlotStride, s))
        return rc;
    }
    {
      ProfScope ps("unrolled_bwd_proj", s);
      ProjArgs a{w.vbar[sel], phi,         S,          r,     c.r_b, lam, y1b_in,
                 w.y1bar[sel], w.ybar,     w.ybb[sel], phibar ? w.sbar : nullptr,
                 slots + size_t(2 * k) * kGradSlots * kGradSlotStride, N, int(T)};
      const bool vec = proj_vector(N, {a.vbar, phi, S, r, a.y1bar_in, a.y1bar_out, a.ybar, a.ybb,
                                       a.sbar}, {c.r_b});
      if (vec)
        k_ub_proj<4, 4><<<dim3(grid1(N / 4), unsigned(nb)), kThreads, 0, s>>>(a);
      else
        k_ub_proj<1, 8><<<dim3(grid1(N), unsigned(nb)), kThreads, 0, s>>>(a);
      SCIGAP_LAUNCH_CHECK("unrolled projection backward");
      if (phibar) {
        const bool pv = vec && proj_vector(N, {xk, phibar}, {c.x_b});
        if (pv)
          k_ub_phibar<4><<<dim3(grid1(N / 4), unsigned(T)), kThreads, 0, s>>>(
              w.vbar[sel], xk, c.x_b, r, c.r_b, lam, w.ybb[sel], w.sbar, phibar, N, int(T), nb);
        else
          k_ub_phibar<1><<<dim3(grid1(N), unsigned(T)), kThreads, 0, s>>>(
              w.vbar[sel], xk, c.x_b, r, c.r_b, lam, w.ybb[sel], w.sbar, phibar, N, int(T), nb);
        SCIGAP_LAUNCH_CHECK("unrolled mask gradient");
      }
    }
    vb_in = w.vbar[sel];
    ybb_in = w.ybb[sel];
    y1b_in = w.y1bar[sel];
    sel ^= 1;
  }
  EndArgs e{vb_in, ybb_in, phi, c.y, c.y_b, w.ybar, phibar, truth, grad_mask, N, int(T), nb, logits,
            slots, grad_lambda, grad_weight, last ? K : 0};
  k_ub_end_y<<<dim3(grid1(N), unsigned(nb)), kThreads, 0, s>>>(e);
  if (phibar) k_ub_end_phi<<<dim3(grid1(N), unsigned(T)), kThreads, 0, s>>>(e);
  SCIGAP_LAUNCH_CHECK("unrolled backward end");
  return SCIGAP_OK;
}

}  // namespace

}  // namespace scigap

// ---------------------------------------------------------------------------
// C entry points
// ---------------------------------------------------------------------------

namespace scigap {

int unrolled_forward_iterations(int64_t H, int64_t W, int64_t T, int K, int D, int nb,
                                const float* lambdas, const float* weights, const float* y,
                                size_t y_b, const float* phi, const float* S, float* xs,
                                size_t xstride, size_t x_b, float* y1b, size_t y1_b,
                                float* x_out, float* rs, size_t rstride, size_t r_b,
                                float* yb_part, size_t part_b, hipStream_t s);

namespace {

// Checkpoint of one sample: x_0..x_{K-1}, r_0..r_{K-1}, y; every plane set
// starts on a 256-byte boundary (strides in floats).
struct CkptLayout {
  size_t x = 0, r = 0, y = 0, per_sample = 0, total = 0, xstride = 0, rstride = 0;
};

CkptLayout ckpt_layout(const scigap_unrolled& u) {
  const size_t N = size_t(u.H) * u.W, V = N * size_t(u.T), K = size_t(u.iters);
  CkptLayout c;
  c.xstride = align256(V * 4) / 4;
  c.rstride = align256(N * 4) / 4;
  c.x = 0;
  c.r = K * c.xstride * 4;
  c.y = c.r + K * c.rstride * 4;
  c.per_sample = c.y + align256(N * 4);
  c.total = c.per_sample * size_t(u.batch);
  return c;
}

// Workspace: the samples of a batch run in groups (group_of), one launch per
// step for the whole group.
struct UWorkspace {
  float* phi = nullptr;      // sigmoid(logits), when logits
  float* S = nullptr;        // phi_sum
  float* phibar = nullptr;   // (T,H,W) dL/dphi
  double* gl = nullptr;      // K, when the caller passes no grad_lambda
  double* gw = nullptr;      // K, when the caller passes no grad_weight
  double* slots = nullptr;   // [K][lambda, weight][kGradSlots] gradient accumulators
  float* y1b = nullptr;      // two y1 planes per sample (forward)
  float* yb_part = nullptr;  // [min(T,8)][H*W] per sample: partial yb of frame-split launches
  size_t part_b = 0;
  BwdScratch bwd;
  size_t bytes = 0;
};

// Samples of a group: four fill the GPU and bound the scratch.  The reverse TV
// of 5 and 6 updates has one large workgroup per tile and CU, and a group waits
// for its last, partly empty round of them: there the size up to eight with the
// fewest rounds, a group's other launches counted as one round (36 us).  144
// workgroups a sample at 256x256x8, 6 updates: a batch of 8 takes 5 rounds, as
// 4 + 4 six; of 6 four, as 4 + 2 five.
int group_of(const scigap_unrolled& u) {
  const int D = u.tv_iter_max - 1;
  int best = u.batch < kSamples ? u.batch : kSamples;
  if (D <= 4) return best;
  auto cost = [&](int g) {
    const int64_t full = u.batch / g, rest = u.batch % g;
    return full * (tv_backward_rounds(D, g, u.H, u.W, u.T) + 1) +
           (rest ? tv_backward_rounds(D, int(rest), u.H, u.W, u.T) + 1 : 0);
  };
  int64_t least = cost(best);
  for (int g = 1; g <= u.batch && g <= kSamplesMax; ++g)
    if (cost(g) < least) {
      least = cost(g);
      best = g;
    }
  return best;
}

UWorkspace carve(const scigap_unrolled& u, char* base) {
  const size_t N = size_t(u.H) * u.W, V = N * size_t(u.T), K = size_t(u.iters);
  const size_t nb = size_t(group_of(u));
  UWorkspace w;
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* q = base ? base + off : nullptr;
    off += align256(bytes);
    return q;
  };
  if (u.logits) w.phi = reinterpret_cast<float*>(take(V * 4));
  w.S = reinterpret_cast<float*>(take(N * 4));
  w.phibar = reinterpret_cast<float*>(take(V * 4));
  w.gl = reinterpret_cast<double*>(take(K * 8));
  w.gw = reinterpret_cast<double*>(take(K * 8));
  w.slots = reinterpret_cast<double*>(take(K * 2 * kGradSlots * kGradSlotStride * 8));
  w.y1b = reinterpret_cast<float*>(take(2 * N * nb * 4));
  w.part_b = size_t(u.T < 8 ? u.T : 8) * N;
  w.yb_part = reinterpret_cast<float*>(take(w.part_b * nb * 4));
  const size_t bw = bwd_scratch(u.H, u.W, u.T, int(nb), base ? base + off : nullptr, &w.bwd);
  w.bytes = off + bw;
  return w;
}

int check_unrolled(const scigap_unrolled* u) {
  if (!u) return fail(SCIGAP_ENULL, "unrolled descriptor is NULL");
  if (int rc = check_shape(u->H, u->W, u->T)) return rc;
  if (u->H * u->W > (int64_t(1) << 30) - 8)
    return fail(SCIGAP_EINVAL, "H*W must be <= 2^30 - 8 (buffer-addressed planes)");
  if (u->batch < 1) return fail(SCIGAP_EINVAL, "batch must be >= 1");
  if (u->iters < 1) return fail(SCIGAP_EINVAL, "iters must be >= 1");
  if (u->tv_iter_max < 2 || u->tv_iter_max > 7)
    return fail(SCIGAP_EUNSUPPORTED, "tv_iter_max must be in [2, 7] (fused TV depth)");
  if (u->batch > 1 && (u->H * u->W * u->T) % 2 != 0)
    return fail(SCIGAP_EINVAL, "batch > 1 needs an even T*H*W (8-byte aligned samples)");
  return SCIGAP_OK;
}

int check_common(const scigap_unrolled* u, const float* lambdas, const float* weights,
                 const float* mask, const float* meas, const void* ckpt, size_t ckpt_bytes,
                 void* ws, size_t ws_bytes) {
  if (int rc = check_unrolled(u)) return rc;
  if (!lambdas || !weights || !mask || !meas || !ckpt)
    return fail(SCIGAP_ENULL, "unrolled: null argument");
  for (int k = 0; k < u->iters; ++k) {
    if (!(weights[k] > 0.f) || !std::isfinite(weights[k]))
      return fail(SCIGAP_EINVAL, "tv weight %d must be finite and > 0", k);
    if (!std::isfinite(lambdas[k])) return fail(SCIGAP_EINVAL, "lambda %d is not finite", k);
  }
  const size_t need = ckpt_layout(*u).total;
  if (ckpt_bytes < need)
    return fail(SCIGAP_EWORKSPACE, "checkpoint needs %zu bytes, got %zu", need, ckpt_bytes);
  const size_t wneed = carve(*u, nullptr).bytes;
  if (!ws || ws_bytes < wneed)
    return fail(SCIGAP_EWORKSPACE, "workspace needs %zu bytes, got %zu", wneed, ws_bytes);
  if ((reinterpret_cast<uintptr_t>(mask) | reinterpret_cast<uintptr_t>(ckpt)) % 8 != 0)
    return fail(SCIGAP_EINVAL, "device buffers must be 8-byte aligned");
  return SCIGAP_OK;
}

// phi (from logits when asked) and its frame sum.
int prepare_mask(const scigap_unrolled& u, const float* mask, const UWorkspace& w,
                 const float** phi, hipStream_t s) {
  const int64_t N = u.H * u.W;
  *phi = u.logits ? w.phi : mask;
  k_mask<<<grid1(N), kThreads, 0, s>>>(mask, u.logits ? w.phi : nullptr, w.S, N, int(u.T));
  SCIGAP_LAUNCH_CHECK("mask launch");
  return SCIGAP_OK;
}

}  // namespace
}  // namespace scigap

using namespace scigap;

extern "C" {

size_t scigap_unrolled_checkpoint_bytes(const scigap_unrolled* u) {
  if (check_unrolled(u) != SCIGAP_OK) return 0;
  return ckpt_layout(*u).total;
}

size_t scigap_unrolled_workspace_bytes(const scigap_unrolled* u) {
  if (check_unrolled(u) != SCIGAP_OK) return 0;
  return carve(*u, nullptr).bytes;
}

int scigap_unrolled_forward(const scigap_unrolled* u, const float* lambdas, const float* weights,
                            const float* mask, const float* meas, float* x_out, void* ckpt,
                            size_t ckpt_bytes, void* workspace, size_t workspace_bytes,
                            void* stream) {
  clear_error();
  if (int rc = check_common(u, lambdas, weights, mask, meas, ckpt, ckpt_bytes, workspace,
                            workspace_bytes))
    return rc;
  if (!x_out) return fail(SCIGAP_ENULL, "unrolled: null x_out");
  if (reinterpret_cast<uintptr_t>(x_out) % 8 != 0)
    return fail(SCIGAP_EINVAL, "device buffers must be 8-byte aligned");
  const int64_t N = u->H * u->W, V = N * u->T;
  const size_t outb = size_t(V) * 4 * u->batch;
  const CkptLayout cl = ckpt_layout(*u);
  if (overlaps(x_out, outb, ckpt, cl.total) || overlaps(x_out, outb, workspace, workspace_bytes))
    return fail(SCIGAP_EALIAS, "x_out overlaps the checkpoint or the workspace");
  hipStream_t s = as_stream(stream);
  const UWorkspace w = carve(*u, static_cast<char*>(workspace));
  const float* phi = nullptr;
  if (int rc = prepare_mask(*u, mask, w, &phi, s)) return rc;
  const size_t dist = cl.per_sample / 4;  // distance between samples in floats
  const int group = group_of(*u);
  for (int b = 0; b < u->batch; b += group) {
    const int nb = u->batch - b < group ? u->batch - b : group;
    char* cb = static_cast<char*>(ckpt) + cl.per_sample * b;
    float* xs = reinterpret_cast<float*>(cb + cl.x);
    float* rs = reinterpret_cast<float*>(cb + cl.r);
    float* yb = reinterpret_cast<float*>(cb + cl.y);
    StartArgs a{meas + size_t(b) * (u->measure ? V : N), u->measure ? 1 : 0, phi, w.S, yb, dist, xs,
                dist, rs, dist, w.y1b, size_t(2 * N), N, int(u->T)};
    k_unrolled_start<<<dim3(grid1(N), unsigned(nb)), kThreads, 0, s>>>(a);
    SCIGAP_LAUNCH_CHECK("unrolled start launch");
    if (int rc = unrolled_forward_iterations(
            u->H, u->W, u->T, u->iters, u->tv_iter_max - 1, nb, lambdas, weights, yb, dist, phi,
            w.S, xs, cl.xstride, dist, w.y1b, size_t(2 * N), x_out + size_t(b) * V, rs, cl.rstride,
            dist, w.yb_part, w.part_b, s))
      return rc;
  }
  return SCIGAP_OK;
}

int scigap_unrolled_backward(const scigap_unrolled* u, const float* lambdas, const float* weights,
                             const float* mask, const float* meas, const void* ckpt,
                             size_t ckpt_bytes, const float* grad_x, float* grad_mask,
                             float* grad_meas, double* grad_lambda, double* grad_weight,
                             void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  if (int rc = check_common(u, lambdas, weights, mask, meas, ckpt, ckpt_bytes, workspace,
                            workspace_bytes))
    return rc;
  if (!grad_x) return fail(SCIGAP_ENULL, "unrolled: null grad_x");
  if (u->measure && grad_meas)
    return fail(SCIGAP_EINVAL, "measure = 1: the truth videos get no gradient (grad_meas NULL)");
  const int64_t N = u->H * u->W, V = N * u->T;
  const int K = u->iters, D = u->tv_iter_max - 1;
  const CkptLayout cl = ckpt_layout(*u);
  if ((grad_mask && (overlaps(grad_mask, V * 4, workspace, workspace_bytes) ||
                     overlaps(grad_mask, V * 4, ckpt, cl.total))) ||
      (grad_meas && overlaps(grad_meas, size_t(N) * 4 * u->batch, workspace, workspace_bytes)))
    return fail(SCIGAP_EALIAS, "a gradient output overlaps the checkpoint or the workspace");
  hipStream_t s = as_stream(stream);
  const UWorkspace w = carve(*u, static_cast<char*>(workspace));
  const float* phi = nullptr;
  if (int rc = prepare_mask(*u, mask, w, &phi, s)) return rc;
  double* gl = grad_lambda ? grad_lambda : w.gl;
  double* gw = grad_weight ? grad_weight : w.gw;
  const size_t dist = cl.per_sample / 4;
  const int group = group_of(*u);
  float* const phibar = grad_mask ? w.phibar : nullptr;
  for (int b = 0; b < u->batch; b += group) {
    const int nb = u->batch - b < group ? u->batch - b : group;
    const char* cb = static_cast<const char*>(ckpt) + cl.per_sample * b;
    const GroupCkpt c{reinterpret_cast<const float*>(cb + cl.x), cl.xstride, dist,
                      reinterpret_cast<const float*>(cb + cl.r), cl.rstride, dist,
                      reinterpret_cast<const float*>(cb + cl.y), dist};
    const bool first = b == 0, last = b + nb >= u->batch;
    k_zero<<<grid1(first && phibar ? V : N * group), 256, 0, s>>>(
        w.bwd.ybar, N * group, phibar, first && phibar ? V : 0, w.slots,
        first ? int64_t(K) * 2 * kGradSlots * kGradSlotStride : 0);
    SCIGAP_LAUNCH_CHECK("gradient fill");
    if (int rc = unrolled_backward(u->H, u->W, u->T, K, D, nb, lambdas, weights, c, phi, w.S,
                                   grad_x + size_t(b) * V,
                                   u->measure ? meas + size_t(b) * V : nullptr, phibar,
                                   last ? grad_mask : nullptr, u->logits, last, w.slots, gl, gw,
                                   w.bwd, s))
      return rc;
    if (!u->measure && grad_meas) {
      hipError_t e = hipMemcpyAsync(grad_meas + size_t(b) * N, w.bwd.ybar, size_t(N) * nb * 4,
                                    hipMemcpyDeviceToDevice, s);
      if (e != hipSuccess) return hip_fail(e, "copy dL/dy");
    }
  }
  return SCIGAP_OK;
}

}  // extern "C"
