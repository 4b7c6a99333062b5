// Row-sweep engine of the Chambolle TV for gfx950: the device code of a strip, and
// how an image is cut into strips.
//
// One wavefront carries a 128-column strip of one frame down its rows with all
// S dual updates in flight at once, each one row behind the one before it:
//
//   step i:  image row i arrives, and for u = 1..S (j = i - u)
//     q_u[j]   = (q_{u-1}[j] + g) / (1 + tw |g|),  g = G out_{u-1}[j]
//     out_u[j] = image[j] - dq_u[j] / 4
//
// G out[j] needs out rows j and j+1, dq[j] needs q rows j-1 and j, so a stage
// holds two rows of what it reads and everything stays in registers: no LDS
// exchange, no barrier, and rows are loaded once per strip.  Horizontal
// neighbours come from the adjacent lane through DPP.  Stage u starts at step
// 2u-1, so a strip of R owned rows costs S*R + S*S row updates instead of the
// S*(R + 2S) of a square load tile.  The arithmetic of one pixel is that of
// tv_tile.h (q = -4p), operation for operation.
//
// A lane holds two adjacent columns.  The outermost S columns on each side
// that is not the image edge go stale (one per update), as in tv_tile.h, and
// strips are placed by the same col_place.
#pragma once

#include <algorithm>
#include <cmath>
#include <utility>

#include "fused.h"

namespace scigap {
namespace sweep {
namespace {

using namespace fused;

typedef float f2 __attribute__((ext_vector_type(2)));

// Two floats per lane in one buffer_store_dwordx2 (see raw_buffer_load_f2).
extern "C" __device__ void raw_buffer_store_f2(f2 v, __amdgpu_buffer_rsrc_t rsrc, int voffset,
                                               int soffset, int aux)
    __asm("llvm.amdgcn.raw.ptr.buffer.store.v2f32");

// A wave-uniform float as a scalar register: an FMA that reads two vector
// registers and a scalar issues at the rate of an add, one that reads three
// vector registers takes 4 cycles instead of 2.6 (two or more waves a SIMD).
__device__ __forceinline__ float uniform(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// ---------------------------------------------------------------------------
// Passes and strips of the deep TV (host)
// ---------------------------------------------------------------------------

constexpr int kMaxPass = 6;  // updates of a pass

// Strips up to which every wave sums its frame's energy slots itself: 6 slot
// rows of 128 are 12 loads a lane, about the launch they replace (512x512x10,
// 29 updates: 152 us with a limit of 64 or 128, 162 us with 300).
constexpr int kInlineStrips = 128;

// Strips across an image for passes of S updates (column halo HC(S)).
inline int strips_across(int W, int S) {
  const int HC = (S + 2) & ~1;
  return tiles_across(W, 128, HC, 128 - 2 * HC);
}

// Rows a strip owns: tall strips waste fewer halo rows, short ones give more
// waves.  The sweep of one strip costs S*(R + S) row updates; a SIMD works its
// waves off one after the other, and is about 2/3 busy with a single one.
// (29 updates, R = 8 / 16 / 32 / 64: 75 / 94 / 139 / - us at 256x256x8, 330 /
// 297 / 308 / - us at 1024x1024x8, 2.65 / 2.17 / 1.97 / 2.02 ms at
// 2048x2048x20.)
inline int strip_rows(int64_t H, int64_t W, int64_t T, int S, int simds) {
  int best = 8;
  double best_cost = 1e300;
  for (int R : {8, 16, 32, 64}) {
    const double waves = double(strips_across(int(W), S)) * double((H + R - 1) / R) * double(T);
    const double per_simd = std::max(1.5, std::ceil(waves / simds));
    const double cost = per_simd * double(R + S + 3);
    if (cost < best_cost * 0.999) {
      best_cost = cost;
      best = R;
    }
  }
  return best;
}

// ---------------------------------------------------------------------------

// Where a strip's pixels are.
struct StripPos {
  int row0;      // global row of step 0
  int col;       // global column of the lane's first pixel
  bool owner;    // the lane's columns are owned by the strip (both or neither)
  bool own1;     // ... and its second one lies inside the image
  bool in0, in1; // the lane's columns lie inside the image
  bool h0, h1;   // horizontal difference exists at the lane's columns
};

// Rows of one plane.  INSIDE strips lie in the image: one 8-byte load per row
// with the row step in the scalar offset (4-byte alignment is enough).  EDGE
// strips send every pixel outside the image past the end of the buffer, which
// reads as 0.
template <bool EDGE>
__device__ __forceinline__ f2 load_px(__amdgpu_buffer_rsrc_t rs, const StripPos& sp, int vo, int i,
                                      int H, int W) {
  if constexpr (!EDGE) {
    return raw_buffer_load_f2(rs, vo, i * W * 4, 0);
  } else {
    const int r = sp.row0 + i;
    const bool in = r >= 0 && r < H;  // wave-uniform
    const unsigned o = (unsigned(r) * unsigned(W) + unsigned(sp.col)) * 4u;
    const unsigned o0 = in && sp.in0 ? o : 0xFFFFFFF0u;
    const unsigned o1 = in && sp.in1 ? o + 4u : 0xFFFFFFF0u;
    f2 v;
    v.x = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o0, 0, 0));
    v.y = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o1, 0, 0));
    return v;
  }
}

// Offset that every plane's bounds check refuses, with room for a scalar
// offset: INSIDE strips are used for planes up to this many bytes only.
constexpr unsigned kNoStore = 0x80000000u;

// Store of one owned row of the strip (row i counted from sp.row0).  INSIDE:
// `vst` is the lane's offset, or kNoStore for lanes that own nothing -- a
// store without a branch, so that the number of memory operations in flight
// is the same on every path and a wait for the rows requested ahead does not
// wait for the latest stores too.  EDGE: lanes and rows are tested.
template <bool EDGE>
__device__ __forceinline__ void store_px(__amdgpu_buffer_rsrc_t rs, const StripPos& sp,
                                         unsigned vst, int i, int H, int W, f2 v) {
  if constexpr (!EDGE) {
    raw_buffer_store_f2(v, rs, int(vst), i * W * 4, 0);
  } else {
    const int r = sp.row0 + i;
    if (r >= H || !sp.owner) return;
    const unsigned o = (unsigned(r) * unsigned(W) + unsigned(sp.col)) * 4u;
    // (a bit_cast of a vector's element reads its first one: copy them out)
    const float x = v.x, y = v.y;
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, x), rs, o, 0, 0);
    if (sp.own1)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, y), rs, o + 4u, 0, 0);
  }
}

// State of one stage: what stage u keeps between steps.
struct Dual {
  f2 q0, q1;  // vertical and horizontal component of one row
};

// One dual update of row j from out rows `a` (j) and `b` (j+1).  e += 16 w |g|
// with ENERGY (scaled as the sum of dq^2 is, a power of two).
template <bool EDGE, bool ZERO, bool ENERGY>
__device__ __forceinline__ Dual dual_step(f2 a, f2 b, const Dual& p, const StripPos& sp, bool vrow,
                                          float tw, float w16, float& e) {
  const float right1 = from_next_lane(a.x);
  float g00 = b.x - a.x, g01 = b.y - a.y;
  float g10 = a.y - a.x, g11 = right1 - a.y;
  if constexpr (EDGE) {
    g00 = vrow ? g00 : 0.f;  // wave-uniform
    g01 = vrow ? g01 : 0.f;
    g10 = sp.h0 ? g10 : 0.f;
    g11 = sp.h1 ? g11 : 0.f;
  }
  const float n0 = fast_sqrt(fmaf(g00, g00, g10 * g10));
  const float n1 = fast_sqrt(fmaf(g01, g01, g11 * g11));
  if constexpr (ENERGY) {
    e = fmaf(w16, n0, e);
    e = fmaf(w16, n1, e);
  }
  const float i0 = fast_rcp(fmaf(tw, n0, 1.f));
  const float i1 = fast_rcp(fmaf(tw, n1, 1.f));
  Dual r;
  r.q0.x = (ZERO ? g00 : p.q0.x + g00) * i0;
  r.q1.x = (ZERO ? g10 : p.q1.x + g10) * i0;
  r.q0.y = (ZERO ? g01 : p.q0.y + g01) * i1;
  r.q1.y = (ZERO ? g11 : p.q1.y + g11) * i1;
  // Materialise the product here (tv_tile.h: the compiler would otherwise
  // fold the multiply into the divergence and change its rounding).
  float s0 = r.q0.x, s1 = r.q0.y, s2 = r.q1.x, s3 = r.q1.y;
  asm("" : "+v"(s0), "+v"(s1), "+v"(s2), "+v"(s3));
  r.q0.x = s0;
  r.q0.y = s1;
  r.q1.x = s2;
  r.q1.y = s3;
  return r;
}

// out = img - dq/4 with the vertical component of the row above in `up`;
// e += dq^2 with ENERGY.
template <bool ENERGY>
__device__ __forceinline__ f2 div_step(f2 img, const Dual& q, f2 up, float& e) {
  const float left0 = from_prev_lane(q.q1.y);
  const float d0 = (up.x - q.q0.x) + (left0 - q.q1.x);
  const float d1 = (up.y - q.q0.y) + (q.q1.x - q.q1.y);
  if constexpr (ENERGY) {
    e = fmaf(d0, d0, e);
    e = fmaf(d1, d1, e);
  }
  f2 o;
  o.x = fmaf(-0.25f, d0, img.x);
  o.y = fmaf(-0.25f, d1, img.y);
  return o;
}

// The rows in flight of one strip, S updates deep.  Rows are counted from the
// strip's first loaded row; every array is a ring over the row number modulo
// kRing, indexed at compile time, so that a loop over blocks of kRing rows
// keeps everything in registers without moving it.
//
// FROM_Q: the updates continue from a given dual field q_0 instead of 0 (then
// out_0 = image - dq_0/4 needs the row above and the column to the left: one
// more halo row at the top, kTop = S + 1, and column at the left).
constexpr int kRing = 8;

// LIMIT: only the first `lim` of the S updates run (a recomputation up to an
// exit iteration); the later stages hand their rows on.
template <int S, bool EDGE, bool ENERGY, bool FROM_Q, bool LIMIT = false>
struct Rows {
  static_assert(S >= 1 && S < kRing, "image rows live for S + 1 steps");
  static constexpr int kTop = S + (FROM_Q ? 1 : 0);   // halo rows above the owned ones
  static constexpr int kFill = S + kTop;              // steps before the first finished row
  f2 img[kRing];
  f2 out[S + 1][kRing];
  Dual q[S + 1][kRing];
  int lim = S;    // LIMIT only; wave-uniform
  // 16 times this lane's part of E_u over the owned rows: `acc` adds up kSumRows
  // rows, `tot` those sums, so that no chain of fp32 additions grows with the
  // strip's height (all terms of 64 rows in one chain: 1.9e-6 of the sum of a ramp).
  static constexpr int kSumRows = 4;
  float acc[S] = {}, tot[S] = {};

  // Step of row I (its image row and, with FROM_Q, dual row already stored in
  // img[I % kRing], q[0][I % kRing]); `row` is its global row.  FILL: one of
  // the first kFill steps (I is the row number); otherwise I only matters
  // modulo kRing, M = I - kFill counts from the start of the block, and `last`
  // marks the strip's last block (its lowest halo rows add no energy).
  template <int I, bool FILL>
  __device__ __forceinline__ void step(const StripPos& sp, int row, int H, float tw, float w16,
                                       bool last) {
    constexpr int o = FROM_Q ? 1 : 0;
    constexpr int M = FILL ? 0 : (I - kFill);
    const f2 im = img[I % kRing];
    if constexpr (!FROM_Q) {
      out[0][I % kRing] = im;
    } else if constexpr (!FILL || I >= 1) {
      constexpr bool en = ENERGY && (!FILL || I >= kTop);
      div<en, !FILL && (M >= kRing - S)>(im, q[0][I % kRing], q[0][(I + kRing - 1) % kRing].q0,
                                         last, acc[0], out[0][I % kRing]);
    }
    static_for<S>([&](auto uc) __attribute__((always_inline)) {
      constexpr int u = decltype(uc)::value + 1;
      if constexpr (!FILL || I >= 2 * u - 1 + o) {
        constexpr int j = (I + kRing * 8 - u) % kRing, jn = (j + 1) % kRing,
                      jp = (j + kRing - 1) % kRing;
        constexpr bool own = ENERGY && (!FILL || I - u >= kTop);
        constexpr bool cut = !FILL && (M >= kRing - S + u);  // not owned in the last block
        const bool vrow = !EDGE || (row - u >= 0 && row - u < H - 1);
        if constexpr (LIMIT) {
          // (values, not references, cross the branch: they stay registers)
          const f2 b0 = q[u - 1][j].q0, b1 = q[u - 1][j].q1, bo = out[u - 1][j];
          f2 n0 = b0, n1 = b1, no = bo;
          if (u <= lim) {
            const Dual p{b0, b1};
            float e = 0.f;
            const Dual d = dual_step<EDGE, false, false>(bo, out[u - 1][jn], p, sp, vrow, tw, w16, e);
            n0 = d.q0;
            n1 = d.q1;
            if constexpr (!FILL || I >= 2 * u + o) no = div_step<false>(img[j], d, q[u][jp].q0, e);
          }
          q[u][j].q0 = n0;
          q[u][j].q1 = n1;
          out[u][j] = no;
          return;
        }
        float e = acc[u - 1];
        q[u][j] = dual_step<EDGE, u == 1 && !FROM_Q, own>(out[u - 1][j], out[u - 1][jn],
                                                          q[u - 1][j], sp, vrow, tw, w16, e);
        if constexpr (own) acc[u - 1] = cut && last ? acc[u - 1] : e;
        if constexpr (!FILL || I >= 2 * u + o)
          div<own && (u < S), cut>(img[j], q[u][j], q[u][jp].q0, last, acc[u < S ? u : 0],
                                   out[u][j]);
      }
    });
    // The running energies are formed here: left alone, the compiler sinks
    // them into the branch that uses them and keeps every term live until then.
    if constexpr (ENERGY)
#pragma unroll
      for (int u = 0; u < S; ++u) {
        if constexpr (FILL ? I + 1 == kFill : (M + 1) % kSumRows == 0) {
          tot[u] += acc[u];
          acc[u] = 0.f;
          compute_here(tot[u]);
        } else {
          compute_here(acc[u]);
        }
      }
  }

  template <bool OWN, bool CUT>
  __device__ __forceinline__ void div(f2 im, const Dual& d, f2 up, bool last, float& a, f2& o) {
    float e = a;
    o = div_step<OWN>(im, d, up, e);
    if constexpr (OWN) a = CUT && last ? a : e;
  }
};

// Strip `tile` of the image (R owned rows, HC halo columns, `top` halo rows
// above); `edge` when it reaches outside the image or to its last column.
struct Strip {
  StripPos sp;
  int c0, r0, own_lo, own_hi;  // first loaded column, first owned row, owned columns
  bool edge;
  __device__ Strip(int tile, int tiles_x, int H, int W, int R, int HC, int top, int bottom) {
    const int ty = tile / tiles_x, tx = tile - ty * tiles_x;
    const ColPlace cp = col_place(tx, tiles_x, W, 128, HC, 128 - 2 * HC);
    c0 = cp.c0;
    r0 = ty * R;
    own_lo = cp.own_lo;
    own_hi = cp.own_hi;
    edge = c0 < 0 || r0 < top || c0 + 128 >= W || r0 + R + bottom > H ||
           unsigned(H) * unsigned(W) > kNoStore / 4u;
    const int lane = threadIdx.x & 63;
    sp.row0 = r0 - top;
    sp.col = c0 + 2 * lane;
    sp.owner = sp.col >= own_lo && sp.col < own_hi && sp.col < W;
    sp.own1 = sp.col + 1 < own_hi && sp.col + 1 < W;
    sp.in0 = sp.col >= 0 && sp.col < W;
    sp.in1 = sp.col + 1 >= 0 && sp.col + 1 < W;
    sp.h0 = sp.col >= 0 && sp.col < W - 1;
    sp.h1 = sp.col + 1 >= 0 && sp.col + 1 < W - 1;
  }
};

// Sums of four values over the wave: within each quad of lanes the values are
// exchanged so that lane l of the quad keeps value 2*(l&1) + (l>>1), then the
// sixteen quads are added.  Lane q < 4 returns the total of that value.
__device__ __forceinline__ float wave_sum4(const float (&s)[4]) {
  const int l = threadIdx.x & 63;
  const bool b0 = l & 1, b1 = (l >> 1) & 1;
  float a0 = b0 ? s[2] : s[0], c0 = b0 ? s[0] : s[2];
  float a1 = b0 ? s[3] : s[1], c1 = b0 ? s[1] : s[3];
  a0 += dpp_move<0xB1>(c0);
  a1 += dpp_move<0xB1>(c1);
  float k = b1 ? a1 : a0;
  const float c = b1 ? a0 : a1;
  k += dpp_move<0x4E>(c);
  k += dpp_move<0x124>(k);
  k += dpp_move<0x128>(k);
  k += __shfl_xor(k, 16, 64);
  k += __shfl_xor(k, 32, 64);
  return k;
}

}  // namespace
}  // namespace sweep
}  // namespace scigap
