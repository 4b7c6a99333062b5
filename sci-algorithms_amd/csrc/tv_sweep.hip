// Chambolle TV of any depth as row sweeps (sweep.h), the default deep TV.
//
// The n_iter_max - 1 dual updates of a frame (scikit-image 0.18.3
// restoration/_denoise.py:341-393) run in passes of 3 to 6, split evenly
// (29 updates: 6, 6, 6, 6, 5).  One wave sweeps one 128-column strip of one
// frame: it reads the image and the dual field q = -4p of the pass before and
// writes the new dual field (the image on the last pass).  Frames and strips
// are independent waves, so a stack of small frames fills the device, which
// one workgroup per tile looping over the frames (tv_chunk.hip) cannot.  With
// 29 updates and no early stop (chunks of 6 / this): 440 / 75 us at 256x256x8,
// 546 / 152 us at 512x512x10, 3.2 / 2.0 ms at 2048x2048x20.
//
// What bounds it: at 2048x2048x20 a pass of 6 takes 440-480 us, 89% of the time
// the SIMDs need to issue its vector instructions one at a time (180 a row of
// 128 columns and wave, 24 of them square roots and reciprocals at half rate);
// its 20 B per pixel would take 325 us at the copy rate, so shallower passes
// lose (of 4: 3.3 ms).  At 256x256x8 it is the length of one wave's sweep.
//
// Early exit.  A pass stores its energies per strip; the launch after it
// decides.  With few strips (kInlineStrips) every wave sums the slots of its
// frame itself, always in the same order, so all waves of a frame agree and a
// pass is one launch.  With many, a decision kernel (one workgroup per frame)
// does it.  A frame that stopped at update s of pass c is recomputed by the
// waves of launch c + 1 from pass c's input, which the frame's later passes
// would have overwritten but no longer do.  A last launch decides and repairs
// for the final pass.  No atomics: results and exits do not depend on the
// order in which waves run.

#include "sweep.h"

#include <algorithm>
#include <atomic>
#include <cmath>

namespace scigap {

namespace {

using namespace sweep;

constexpr int kWaves = 4;   // independent waves of one workgroup
constexpr int kAheadTv = 2; // rows requested ahead of their use (4: no faster)

struct PassArgs {
  const float* img;    // (T,H,W)
  const float* q_in;   // [T][2][N] dual field of this pass, null: 0
  float* q_out;        // [T][2][N], null on the last pass
  float* out;          // (T,H,W)
  float* eslot;        // [T][kMaxPass][strips] energies of this pass
  // the pass before (nup_prev = 0: none)
  const float* q_prev; // its input dual field, null: 0
  const float* eslot_prev;
  int strips_prev, i0_prev, nup_prev;
  double* e0;          // [T] E_0
  double* elast;       // [2][T] last energy of the passes before, by parity
  int* stop;           // [T] exit iteration, -1 while running
  int* fix;            // [T] decision of the pass before: updates to redo, -1 none (many strips)
  int* stop_iter;      // optional result (last launch)
  int* early;          // optional count of frames that stopped early (last launch)
  int H, W, T, i0, par, ne, inline_decide;
  int R, strips_x, strips, per_xcd, items;
  float weight, tw;
  double eps;
};

// Exit test of the pass before for frame t (_denoise.py:384-391): updates of
// that pass to redo if the frame stops in it, else -1.  All lanes of the
// calling wave; every wave of a frame gets the same answer.  `keep`: this
// wave records E_0 and the pass's last energy for the launches after it.
__device__ __forceinline__ int exit_test(const PassArgs& a, int t, bool keep) {
  double prev = a.i0_prev > 0 ? a.elast[(a.par ^ 1) * a.T + t] : 0.0;
  double e0 = a.i0_prev > 0 ? a.e0[t] : 0.0;
  int f = -1;
  for (int u = 0; u < a.nup_prev; ++u) {
    const double e =
        slot_row_sum(a.eslot_prev + (size_t(t) * kMaxPass + u) * a.strips_prev, a.strips_prev);
    const int i = a.i0_prev + u;
    if (i == 0) e0 = e;
    if (i >= 1 && f < 0 && fabs(prev - e) < a.eps * e0) f = u;
    prev = e;
  }
  if (keep && (threadIdx.x & 63) == 0) {
    if (a.i0_prev == 0) a.e0[t] = e0;
    a.elast[a.par * a.T + t] = prev;
    if (f >= 0) a.stop[t] = a.i0_prev + f;
  }
  return __builtin_amdgcn_readfirstlane(f);
}

// What a pass does: the first and middle ones write the dual field, the last
// one and a repair (`lim` updates of the pass before redone) the image; the
// launch after the last pass only repairs.
enum Pass { FIRST, MIDDLE, LAST, REPAIR, FINISH };

// One strip of one frame, S updates.
template <int S, bool EDGE, int PASS>
__device__ __forceinline__ void pass_strip(const PassArgs& a, int strip, int t, int lim) {
  constexpr bool FROM_Q = PASS != FIRST, kRepair = PASS == REPAIR;
  constexpr bool kPutQ = PASS == FIRST || PASS == MIDDLE;
  using E = Rows<S, EDGE, !kRepair, FROM_Q, kRepair>;
  constexpr int HC = (S + 2) & ~1, TOP = E::kTop, FILL = E::kFill;
  constexpr int P = kAheadTv;
  const int H = a.H, W = a.W, N = H * W;
  const Strip st(strip, a.strips_x, H, W, a.R, HC, TOP, S);
  const StripPos& sp = st.sp;
  const int vo = (sp.row0 * W + sp.col) * 4;
  const float* qi = kRepair ? a.q_prev : a.q_in;
  const __amdgpu_buffer_rsrc_t ri = plane_rsrc(a.img + size_t(t) * N, N);
  // No dual field yet (pass 0): a descriptor of zero records reads as 0.
  const __amdgpu_buffer_rsrc_t r0 = plane_rsrc(qi + (qi ? size_t(t) * 2 * N : 0), qi ? N : 0);
  const __amdgpu_buffer_rsrc_t r1 = plane_rsrc(qi + (qi ? (size_t(t) * 2 + 1) * N : 0), qi ? N : 0);
  const unsigned vst = sp.owner ? unsigned(vo) : kNoStore;
  float* const qo = kPutQ ? a.q_out + size_t(t) * 2 * N : nullptr;
  const __amdgpu_buffer_rsrc_t w0 = plane_rsrc(qo, kPutQ ? N : 0);
  const __amdgpu_buffer_rsrc_t w1 = plane_rsrc(qo + (kPutQ ? N : 0), kPutQ ? N : 0);
  const __amdgpu_buffer_rsrc_t wo = plane_rsrc(a.out + size_t(t) * N, N);
  E rows;
  rows.lim = lim;
  f2 ni[P], n0[P], n1[P];
  auto request = [&](auto pc, int i) __attribute__((always_inline)) {
    constexpr int p = decltype(pc)::value;
    ni[p] = load_px<EDGE>(ri, sp, vo, i, H, W);
    if constexpr (FROM_Q) {
      n0[p] = load_px<EDGE>(r0, sp, vo, i, H, W);
      n1[p] = load_px<EDGE>(r1, sp, vo, i, H, W);
    }
  };
  static_for<P>([&](auto k) __attribute__((always_inline)) { request(k, decltype(k)::value); });
  const int rows_all = a.R + S + TOP;
  auto feed = [&](auto ic, int i) __attribute__((always_inline)) {
    constexpr int I = decltype(ic)::value, sl = I % kRing, p = I % P;
    rows.img[sl] = ni[p];
    if constexpr (FROM_Q) {
      rows.q[0][sl].q0 = n0[p];
      rows.q[0][sl].q1 = n1[p];
    }
    // The last rows' requests read the strip's last row again.
    const int k = i + P < rows_all ? i + P : rows_all - 1;
    request(std::integral_constant<int, p>{}, k);
  };
  const float tw = a.tw, w16 = uniform(16.f * a.weight);
  static_for<FILL>([&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
    feed(ic, i);
    rows.template step<i, true>(sp, sp.row0 + i, H, tw, w16, false);
    __builtin_amdgcn_sched_barrier(0);
  });
#pragma unroll 1
  for (int b = 0; b < a.R; b += kRing) {
    const bool last = b + kRing >= a.R;
    static_for<kRing>([&](auto mc) __attribute__((always_inline)) {
      constexpr int m = decltype(mc)::value, I = FILL + m;
      constexpr int j = (I + kRing - S) % kRing;  // slot of the finished row
      const int i = FILL + b + m;
      feed(std::integral_constant<int, I>{}, i);
      rows.template step<I, false>(sp, sp.row0 + i, H, tw, w16, last);
      if constexpr (kPutQ) {
        store_px<EDGE>(w0, sp, vst, i - S, H, W, rows.q[S][j].q0);
        store_px<EDGE>(w1, sp, vst, i - S, H, W, rows.q[S][j].q1);
      } else {
        store_px<EDGE>(wo, sp, vst, i - S, H, W, rows.out[S][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  if constexpr (!kRepair) {
    const int lane = threadIdx.x & 63;
    float* const slot = a.eslot + size_t(t) * kMaxPass * a.strips + strip;
#pragma unroll
    for (int g = 0; g < S; g += 4) {
      float s[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) s[u] = g + u < S && sp.owner ? rows.tot[g + u < S ? g + u : 0] : 0.f;
      const float k = wave_sum4(s);
      const int e = g + 2 * (lane & 1) + ((lane >> 1) & 1);
      if (lane < 4 && e < S) slot[size_t(e) * a.strips] = 0.0625f * k;
    }
  }
}

template <int S, int PASS>
__global__ void __launch_bounds__(64 * kWaves) k_tv_pass(PassArgs a) {
  const int wg = tile_of_block(blockIdx.x, a.per_xcd);
  const int item = wg * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= a.items) return;
  const int t = item / a.strips, strip = item - t * a.strips;
  int fix = -1;
  if (a.nup_prev > 0) {
    const int st = __builtin_amdgcn_readfirstlane(a.stop[t]);
    bool done = st >= 0 && st < a.i0_prev;  // stopped in an earlier pass
    if (!done) fix = a.inline_decide ? exit_test(a, t, strip == 0)
                                     : __builtin_amdgcn_readfirstlane(a.fix[t]);
    if (PASS == FINISH && strip == 0 && (threadIdx.x & 63) == 0) {
      const int s = done ? st : (fix >= 0 ? a.i0_prev + fix : a.ne);
      if (a.stop_iter) a.stop_iter[t] = s;
      if (a.early && s < a.ne) atomicAdd(a.early, 1);
    }
    if (done) return;
  } else if (strip == 0 && (threadIdx.x & 63) == 0) {
    a.stop[t] = -1;
  }
  const Strip st(strip, a.strips_x, a.H, a.W, a.R, (S + 2) & ~1, S + 1, S);
  if (fix >= 0) {
    if (st.edge)
      pass_strip<S, true, REPAIR>(a, strip, t, fix);
    else
      pass_strip<S, false, REPAIR>(a, strip, t, fix);
    return;
  }
  if constexpr (PASS != FINISH) {
    if (st.edge)
      pass_strip<S, true, PASS>(a, strip, t, S);
    else
      pass_strip<S, false, PASS>(a, strip, t, S);
  }
}

// The decision of one frame as its own launch (many strips; one workgroup per
// frame): wave u sums slot row u, then the exit test as in exit_test.
__global__ void __launch_bounds__(64 * kMaxPass) k_tv_decide(PassArgs a) {
  __shared__ double e[kMaxPass];
  const int t = blockIdx.x, w = threadIdx.x >> 6;
  const int st = a.stop[t];
  if (st >= 0 && st < a.i0_prev) return;  // workgroup-uniform
  if (w < a.nup_prev) {
    const double s =
        slot_row_sum(a.eslot_prev + (size_t(t) * kMaxPass + w) * a.strips_prev, a.strips_prev);
    if ((threadIdx.x & 63) == 0) e[w] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double prev = a.i0_prev > 0 ? a.elast[(a.par ^ 1) * a.T + t] : 0.0;
    const double e0 = a.i0_prev > 0 ? a.e0[t] : e[0];
    int f = -1;
    for (int u = 0; u < a.nup_prev; ++u) {
      const int i = a.i0_prev + u;
      if (i >= 1 && f < 0 && fabs(prev - e[u]) < a.eps * e0) f = u;
      prev = e[u];
    }
    if (a.i0_prev == 0) a.e0[t] = e0;
    a.elast[a.par * a.T + t] = prev;
    if (f >= 0) a.stop[t] = a.i0_prev + f;
    a.fix[t] = f;
  }
}

template <int S>
void launch_pass(const PassArgs& a, int pass, hipStream_t s) {
  const unsigned grid = unsigned(a.per_xcd * 8);
  switch (pass) {
    case FIRST: k_tv_pass<S, FIRST><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case MIDDLE: k_tv_pass<S, MIDDLE><<<grid, 64 * kWaves, 0, s>>>(a); break;
    case LAST: k_tv_pass<S, LAST><<<grid, 64 * kWaves, 0, s>>>(a); break;
    default: k_tv_pass<S, FINISH><<<grid, 64 * kWaves, 0, s>>>(a); break;
  }
}

int launch_pass_depth(int S, const PassArgs& a, int pass, hipStream_t s) {
  switch (S) {
    case 3: launch_pass<3>(a, pass, s); break;
    case 4: launch_pass<4>(a, pass, s); break;
    case 5: launch_pass<5>(a, pass, s); break;
    default: launch_pass<6>(a, pass, s); break;
  }
  SCIGAP_LAUNCH_CHECK("TV pass launch");
  return SCIGAP_OK;
}

// Most strips any pass geometry has (rows 8, the widest halo).
size_t max_strips(int64_t H, int64_t W) {
  int x = 0;
  for (int S = 3; S <= kMaxPass; ++S) x = std::max(x, strips_across(int(W), S));
  return size_t(x) * size_t((H + 7) / 8);
}

}  // namespace

int device_simds();

size_t tv_sweep_workspace(int64_t H, int64_t W, int64_t T) {
  const size_t N = size_t(H) * W, t = size_t(T);
  return 2 * align256(2 * t * N * 4) + 2 * align256(t * kMaxPass * max_strips(H, W) * 4) +
         3 * align256(t * 8) + 2 * align256(t * 4);
}

// TV of `image` (T,H,W) into `out` with n_iter_max = n >= 8.  `early`
// (optional) is increased by the number of frames that stopped early.
int tv_sweep(const float* image, float* out, int64_t H, int64_t W, int64_t T, float weight,
             float eps, int n, int* stop_iter, int* early, void* ws, hipStream_t s) {
  const size_t N = size_t(H) * W, t = size_t(T);
  const int ne = n - 1;
  const int passes = (ne + kMaxPass - 1) / kMaxPass;
  const int low = ne / passes, extra = ne % passes;  // the first `extra` passes run one more
  if (low < 3) return fail(SCIGAP_EUNSUPPORTED, "TV sweep of %d updates", ne);
  char* base = static_cast<char*>(ws);
  size_t off = 0;
  auto take = [&](size_t bytes) {
    char* q = base + off;
    off += align256(bytes);
    return q;
  };
  float* Q[2];
  for (auto& q : Q) q = reinterpret_cast<float*>(take(2 * t * N * 4));
  float* slot[2];
  for (auto& e : slot) e = reinterpret_cast<float*>(take(t * kMaxPass * max_strips(H, W) * 4));
  PassArgs a{};
  a.e0 = reinterpret_cast<double*>(take(t * 8));
  a.elast = reinterpret_cast<double*>(take(2 * t * 8));
  a.stop = reinterpret_cast<int*>(take(t * 4));
  a.fix = reinterpret_cast<int*>(take(t * 4));
  a.img = image;
  a.out = out;
  a.H = int(H);
  a.W = int(W);
  a.T = int(T);
  a.ne = ne;
  a.weight = weight;
  a.tw = float(0.25 / double(weight));
  a.eps = eps;
  a.R = strip_rows(H, W, T, low, device_simds());
  int i0 = 0;
  for (int c = 0; c <= passes; ++c) {
    const bool finish = c == passes;
    const int S = finish ? low : low + (c < extra ? 1 : 0);
    a.strips_x = strips_across(int(W), S);
    a.strips = a.strips_x * int((H + a.R - 1) / a.R);
    a.items = a.strips * int(T);
    a.per_xcd = ((a.items + kWaves - 1) / kWaves + 7) / 8;
    a.inline_decide = a.strips_prev <= kInlineStrips;
    a.i0 = i0;
    a.par = c & 1;
    a.q_in = c == 0 ? nullptr : Q[c & 1];
    a.q_out = c + 1 < passes ? Q[(c + 1) & 1] : nullptr;
    a.q_prev = c <= 1 ? nullptr : Q[(c - 1) & 1];
    a.eslot = slot[c & 1];
    a.eslot_prev = slot[(c + 1) & 1];
    a.stop_iter = finish ? stop_iter : nullptr;
    a.early = finish ? early : nullptr;
    if (c > 0 && !a.inline_decide) {
      ProfScope ps("tv_decide", s);
      k_tv_decide<<<unsigned(T), 64 * kMaxPass, 0, s>>>(a);
      SCIGAP_LAUNCH_CHECK("TV decision launch");
    }
    {
      ProfScope ps("tv_pass", s);
      const int pass = finish ? FINISH : c == 0 ? FIRST : c + 1 == passes ? LAST : MIDDLE;
      if (int rc = launch_pass_depth(S, a, pass, s)) return rc;
    }
    a.strips_prev = a.strips;
    a.i0_prev = i0;
    a.nup_prev = S;
    i0 += S;
  }
  return SCIGAP_OK;
}

// SIMDs of the current device (queried once per device).
int device_simds() {
  constexpr int kDevices = 64;
  static std::atomic<int> cached[kDevices];
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kDevices) return 1024;
  int v = cached[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      return 1024;
    v = 4 * cus;
    cached[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

}  // namespace scigap
