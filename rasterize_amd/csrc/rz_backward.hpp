// Adjoint of the batched scene render: dL/d(layer RGBA) -> dL/d(control
// points, solid paint colours, gradient stop colours, transform). No
// counterpart in the reference.
//
// Forward per pixel, paths k in order (Scene::render, src/scene.rs:410-430,
// Rasterizer::fill, src/rasterize.rs:102-115):
//   W_k   = box-filtered winding of path k at the pixel (the signed area that
//           signed_difference_line deposits, src/rasterize.rs:365-470)
//   a_k   = alpha_from_winding(W_k) (src/path.rs:32-46); skipped if < 1e-6
//   s_k   = c_k * a_k                      (LinColor::with_alpha)
//   dst_k = s_k + dst_{k-1} * (1 - s_k.a)  (LinColor::blend_over)
// Backward, with T_k = prod_{j>k} (1 - s_j.a) and g = dL/d dst_N:
//   dL/ds_k = T_k * (g - e_alpha * <g, dst_{k-1}>)
//   dL/da_k = <c_k, dL/ds_k>,  dL/dc_k += a_k * dL/ds_k,  dL/dW_k = dL/da_k * a_k'(W_k)
// W_k(pixel) = integral over the pixel of the winding, which a line (p0, p1)
// changes when it moves: for a closed chain the endpoint terms cancel and
//   dL/dx0 = -I0, dL/dy0 = s I0, dL/dx1 = -I1, dL/dy1 = s I1,
//   I0 = int_{y0}^{y1} g_W(x(y), y) (1 - l(y)) dy, I1 = int g_W l dy,
// with l(y) = (y - y0) / (y1 - y0), s = dx/dy and g_W = dL/dW of the pixel the
// line passes through (piecewise constant, so the integrals are exact sums of
// trapezoids). A line's ends are the curve at t = bits / 2^depth of its
// subdivision leaf, so their gradients reach the control points through the
// Bernstein weights at those t; the subdivision is recomputed, not stored.
#pragma once
#include "rz_scene.hpp"

namespace rzk {

struct BwdTileArgs {
  SceneFineArgs f;              // the forward render's state
  const rzp::C4* grad_out;      // dL/d layer
  size_t grad_stride;           // pixels
  float* wbuf;                  // [entries * 256]: winding W, then dL/dW
  float* dbuf;                  // [entries * 256]: <dL/d layer, dst below the path>
  float* grad_colors;           // [n_paths * 4]
  float* stop_acc;              // [stops * 4] dL/d(stop as the paint reads it), or null
  const rzp::C4* stop_base;     // the scene's stop table (a paint's stops are a range of it)
};

__device__ inline float alpha_of(int rule, float W) {
  if (rule == 0) {
    const float a = fabsf(W);
    return a >= 1.0f ? 1.0f : (a < 1e-6f ? 0.0f : a);
  }
  const float f = (float)rzp::rem_euclid((double)W + 1.0, 2.0) - 1.0f;
  return fabsf(f);
}

// d alpha / d W where alpha is differentiable (0 on the clamped parts)
__device__ inline float dalpha_of(int rule, float W) {
  if (rule == 0) {
    const float a = fabsf(W);
    return (a >= 1e-6f && a < 1.0f) ? (W < 0.0f ? -1.0f : 1.0f) : 0.0f;
  }
  const float f = (float)rzp::rem_euclid((double)W + 1.0, 2.0) - 1.0f;
  return f < 0.0f ? -1.0f : 1.0f;
}

// Path q over canvas tile (TX, TY): its tile slot, record and event ranges
// and backdrop. Returns whether its winding can be nonzero anywhere on the
// tile (records, events, a backdrop, or pixels at or right of its right-edge
// column); where not, the path contributes nothing to the tile.
__device__ inline bool path_tile(const SceneFineArgs& a, uint32_t q, int TX, int TY, uint32_t* t,
                                 uint32_t* rb, uint32_t* re, uint32_t* eb, uint32_t* ee) {
  const PathInfo& P = a.pi[q];
  const int txl = TX - P.tx0, tyl = TY - P.ty0;
  *t = P.tile_base + (uint32_t)(tyl * P.g.tiles_x + txl);
  *rb = a.tile_off[*t];
  *re = a.tile_off[*t + 1];
  *eb = a.band_ev_off[P.band_base + tyl];
  *ee = a.band_ev_off[P.band_base + tyl + 1];
  const bool right = txl * 16 - P.g.phx + 15 >= P.redge_col;
  return *rb != *re || *eb != *ee || a.bd[*t] != 0 || right;
}

// Sum of v over the wave, in DPP steps (no LDS); the total is in lane 63.
__device__ inline float wave_sum_hi(float v) {
#define RZ_STEP(ctrl, rows) \
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, rows, 0xf, false))
  RZ_STEP(0x111, 0xf);
  RZ_STEP(0x112, 0xf);
  RZ_STEP(0x114, 0xf);
  RZ_STEP(0x118, 0xf);
  RZ_STEP(0x142, 0xa);
  RZ_STEP(0x143, 0xc);
#undef RZ_STEP
  return v;
}

// <c, dL/ds> / T of a solid paint c over a colour with <g, dst> = D; with D = 0
// the inner product <g, c>.
__device__ inline float solid_da(rzp::C4 c, rzp::C4 g, float D) {
  return rzp::madd(c.r, g.r, rzp::madd(c.g, g.g, rzp::madd(c.b, g.b, c.a * (g.a - D))));
}

// Per canvas tile: the forward composite again, keeping each path's winding
// and what its gradient needs of the colour below it; then the paths in
// reverse order with the transmittance of the paths above, giving dL/dW per
// pixel and path and dL/dc per path. Paths with zero winding over the tile
// (alpha 0 on all of it) change neither sweep; only their dL/dW slot is
// cleared.
//
// Bound by HBM: what the forward sweep keeps per (path, pixel) the reverse
// one reads. Of the colour below, dL/ds_k needs only its inner product with
// g = dL/d(layer), and as g is known before the sweep starts, that can be
// carried as a scalar,
//   D_k = <g, dst_k> = <g, s_k> + D_{k-1} (1 - s_k.a), D_0 = <g, bg>:
// 4 bytes a pixel instead of the colour's 16 (20 bytes of traffic a path and
// pixel instead of 44), and a composite of one channel instead of four.
// 256 paths of 32 cubics at 1024x1024: 3034 -> 1974 us. A solid paint, the
// same for all pixels, has sweeps of its own that load only its colour and
// rule and take g's inner product with it once a pixel (1117 -> 1041 us;
// 16 paths of 8 cubics at 256x256 63 -> 48 us). Each path is a chain of
// dependent loads, so waves in flight count: unbounded, the kernel took 129
// VGPRs and three waves per SIMD; 1041 -> 1002 us at four, 911 at five, which
// spill 39 registers where gradients are painted (240 shapes, two in five of
// them gradients with stop gradients: 7,486 us, 7,766 before all of this; the
// stops' atomics bound those).
__global__ __launch_bounds__(64, 5) void k_scene_bwd_tiles(BwdTileArgs b) {
  const SceneFineArgs& a = b.f;
  if (a.st->err || a.st->overflow) return;
  __shared__ TileLDS<kGroup> L;
  const int lane = threadIdx.x;
  const int TX = (int)(blockIdx.x % (uint32_t)a.tiles_x), TY = (int)(blockIdx.x / (uint32_t)a.tiles_x);
  const uint32_t nrow = a.row_count[TY];
  const uint32_t* row = a.rows + (size_t)TY * a.n_paths;
  // the lane's pixels in a path's tile slot
  const int pix = lane_row(lane) * 16 + lane_col(lane);
  rzp::C4 g[4];
  float D[4];
  const int x = TX * 16 + lane_col(lane), y = TY * 16 + lane_row(lane);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    g[i] = (x + i < a.lw && y < a.lh) ? b.grad_out[(size_t)y * b.grad_stride + x + i] : rzp::splat(0.0f);
    D[i] = g[i].r * a.bg.r + g[i].g * a.bg.g + g[i].b * a.bg.b + g[i].a * a.bg.a;
  }
  // forward sweep; a path with zero winding over the tile is skipped (the
  // reverse sweep writes its zero dL/dW)
  scene_paths(
      a, L, TX, TY, 0u, nrow, lane, [](int, auto w) { return (float)w * (1.0f / kFix); },
      [&](const rzp::DPaint* paint, int rule, uint32_t, uint32_t t, int xs, int ys, bool,
          const float* W) {
        const size_t e = (size_t)t * 256 + pix;
        *(float4*)(b.wbuf + e) = make_float4(W[0], W[1], W[2], W[3]);
        *(float4*)(b.dbuf + e) = make_float4(D[0], D[1], D[2], D[3]);
        if (load_const(&paint->kind) == rzp::PAINT_SOLID) {
          const rzp::C4 c = load_const(&paint->color);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float alpha = alpha_of(rule, W[i]);
            if (alpha >= 1e-6f)
              D[i] = rzp::madd(alpha, solid_da(c, g[i], 0.0f), D[i] * (1.0f - c.a * alpha));
          }
          return;
        }
        const rzp::DPaint p = load_const(paint);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float alpha = alpha_of(rule, W[i]);
          if (alpha >= 1e-6f) {
            const rzp::C4 s = rzp::mul(rzp::paint_at(p, xs + i, ys), alpha);
            D[i] = (g[i].r * s.r + g[i].g * s.g + g[i].b * s.b + g[i].a * s.a) + D[i] * (1.0f - s.a);
          }
        }
      });
  // reverse sweep
  float T[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) T[i] = 1.0f;
  const uint32_t nchunks = (nrow + 63) / 64;
  for (uint32_t ci = nchunks; ci-- > 0;) {
    const uint32_t j = ci * 64 + lane;
    uint32_t pid = 0;
    bool hit = false;
    if (j < nrow) {
      pid = row[j];
      const int4 r = a.rects[pid];
      hit = r.x <= TX && TX < r.z;
    }
    uint32_t lt = 0, lrb, lre, leb, lee;
    const bool draw = hit && path_tile(a, pid, TX, TY, &lt, &lrb, &lre, &leb, &lee);
    // paths skipped by the forward sweep: dL/dW = 0 on their tile slot
    uint64_t z = __ballot(hit && !draw);
    while (z) {
      const int src = __ffsll((unsigned long long)z) - 1;
      z &= z - 1;
      const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)lt, src);
      reinterpret_cast<float4*>(b.wbuf + (size_t)t * 256)[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    uint64_t m = __ballot(draw);
    // the next path's windings and inner products are loaded while the
    // current one is processed
    float4 nW, nD;
    auto prefetch = [&](uint64_t mm) {
      if (!mm) return;
      const int s2 = 63 - __clzll((long long)mm);
      const size_t base = (size_t)(uint32_t)__builtin_amdgcn_readlane((int)lt, s2) * 256 + pix;
      nW = *(const float4*)(b.wbuf + base);
      nD = *(const float4*)(b.dbuf + base);
    };
    prefetch(m);
    while (m) {
      const int src = 63 - __clzll((long long)m);
      m &= ~(1ull << src);
      const float cW[4] = {nW.x, nW.y, nW.z, nW.w}, cD[4] = {nD.x, nD.y, nD.z, nD.w};
      prefetch(m);
      const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)pid, src);
      const uint32_t t = (uint32_t)__builtin_amdgcn_readlane((int)lt, src);
      if (load_const(&a.pi[q].paint.kind) == rzp::PAINT_SOLID) {
        const rzp::C4 c = load_const(&a.pi[q].paint.color);
        const int rule = load_const(&a.pi[q].rule);
        rzp::C4 dc = rzp::splat(0.0f);
        float gWs[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          gWs[k] = 0.0f;
          const float alpha = alpha_of(rule, cW[k]);  // 0 outside the sub-view
          if (alpha >= 1e-6f) {
            gWs[k] = T[k] * solid_da(c, g[k], cD[k]) * dalpha_of(rule, cW[k]);
            const float u = alpha * T[k];
            dc = rzp::c4(rzp::madd(u, g[k].r, dc.r), rzp::madd(u, g[k].g, dc.g),
                         rzp::madd(u, g[k].b, dc.b), rzp::madd(u, g[k].a - cD[k], dc.a));
            T[k] *= 1.0f - c.a * alpha;
          }
        }
        *(float4*)(b.wbuf + (size_t)t * 256 + pix) = make_float4(gWs[0], gWs[1], gWs[2], gWs[3]);
        // dL/dc: sums over the wave, one atomic instruction for the channels
        // (a gradient paint's colour varies over the path: none)
        auto total = [](float v) { return __builtin_amdgcn_readlane(__float_as_int(wave_sum_hi(v)), 63); };
        const int r = total(dc.r), gr = total(dc.g), bl = total(dc.b), al = total(dc.a);
        if (lane < 4)
          atomicAdd(&b.grad_colors[4 * q + lane],
                    __int_as_float(lane == 0 ? r : lane == 1 ? gr : lane == 2 ? bl : al));
        continue;
      }
      const PathInfo P = load_const(a.pi + q);
      const int txl = TX - P.tx0, tyl = TY - P.ty0;
      const int xs = txl * 16 - P.g.phx + lane_col(lane);
      const int ys = tyl * 16 - P.g.phy + lane_row(lane);
      float gWs[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        float gW = 0.0f;
        if (xs + k >= 0 && xs + k < P.g.W && ys >= 0 && ys < P.g.H) {
          const float W = cW[k];
          const float alpha = alpha_of(P.rule, W);
          if (alpha >= 1e-6f) {
            const rzp::C4 cp = rzp::paint_at(P.paint, xs + k, ys);
            const rzp::C4 ds = rzp::c4(T[k] * g[k].r, T[k] * g[k].g, T[k] * g[k].b, T[k] * (g[k].a - cD[k]));
            const float da = cp.r * ds.r + cp.g * ds.g + cp.b * ds.b + cp.a * ds.a;
            gW = da * dalpha_of(P.rule, W);
            int i0, i1;
            float w1;
            rzp::C4 mixed;
            if (b.stop_acc && rzp::gradient_stops_at(P.paint, xs + k, ys, &i0, &i1, &w1, &mixed)) {
              // through into_linear and the stops' lerp (GradStops::at)
              rzp::C4 gm = rzp::mul(ds, alpha);
              if (!P.paint.linear_colors) gm = rzp::into_linear_vjp(mixed, gm);
              float* o = b.stop_acc + 4 * (size_t)(P.paint.stop_col - b.stop_base);
              const float w0 = 1.0f - w1;
              atomicAdd(o + 4 * i0 + 0, gm.r * w0);
              atomicAdd(o + 4 * i0 + 1, gm.g * w0);
              atomicAdd(o + 4 * i0 + 2, gm.b * w0);
              atomicAdd(o + 4 * i0 + 3, gm.a * w0);
              if (w1 != 0.0f) {
                atomicAdd(o + 4 * i1 + 0, gm.r * w1);
                atomicAdd(o + 4 * i1 + 1, gm.g * w1);
                atomicAdd(o + 4 * i1 + 2, gm.b * w1);
                atomicAdd(o + 4 * i1 + 3, gm.a * w1);
              }
            }
            T[k] *= 1.0f - cp.a * alpha;
          }
        }
        gWs[k] = gW;
      }
      *(float4*)(b.wbuf + (size_t)t * 256 + pix) = make_float4(gWs[0], gWs[1], gWs[2], gWs[3]);
    }
  }
}

// I0, I1 of one line (sub-view frame): for each pixel row it crosses and each
// pixel column of that row, g_W times the exact integral of (1 - l) and l
// over the y-range of the line inside the pixel. dxdy is the line's dx/dy
// (dy != 0).
//
// Rows and columns are one loop over the line's pixels: the lanes of a wave
// hold lines of different directions, and nested loops would take the longest
// row of any lane once per row. The pixel's g_W is asked for before its
// y-range is worked out, and the divisions (by dx and dy) are the line's, not
// the pixel's. 8,192 cubics of about 1,000 px at 1024x1024: k_scene_bwd_lines
// 473 -> 336 us, and 312 at four waves per SIMD (20 of 138 VGPRs spilled)
// instead of three.
__device__ inline void line_integrals(const PathInfo& P, const float* wbuf, Pt a, Pt c, double dxdy,
                                      double* I0, double* I1) {
  *I0 = *I1 = 0.0;
  const double dy = c.y - a.y;
  const double ylo = fmax(fmin(a.y, c.y), 0.0), yhi = fmin(fmax(a.y, c.y), (double)P.g.H);
  if (!(ylo < yhi)) return;
  const double inv_dy = 1.0 / dy, dydx = 1.0 / dxdy;
  // a line this steep stays in one column (or straddles x = 0, whose left
  // side has no pixels): nothing to cut
  const bool steep = !(fabs(dxdy) >= 1e-300);
  const int r1 = (int)ceil(yhi);
  const double sgn = dy > 0.0 ? 1.0 : -1.0;
  int r = (int)floor(ylo), cx = 0, ce = -1;
  double ya = ylo, yb = ylo, xb = a.x + (ylo - a.y) * dxdy;
  const float* row = nullptr;
  --r;
  while (true) {
    if (cx > ce) {
      if (++r >= r1) break;
      const double xa = xb;
      ya = yb;
      yb = fmin(yhi, (double)r + 1.0);
      xb = a.x + (yb - a.y) * dxdy;
      cx = max((int)floor(fmin(xa, xb)), 0);
      ce = min((int)floor(fmax(xa, xb)), P.g.W - 1);
      const int gy = r + P.g.phy;
      row = wbuf + (size_t)(P.tile_base + (uint32_t)((gy >> 4) * P.g.tiles_x)) * 256 + (gy & 15) * 16;
      if (cx > ce) continue;
    }
    const int gx = cx + P.g.phx;
    const float gw = row[(size_t)(gx >> 4) * 256 + (gx & 15)];
    double lo = ya, hi = yb;
    if (!steep) {
      const double y0 = a.y + ((double)cx - a.x) * dydx, y1 = a.y + ((double)cx + 1.0 - a.x) * dydx;
      lo = fmax(lo, fmin(y0, y1));
      hi = fmin(hi, fmax(y0, y1));
    }
    ++cx;
    if (!(lo < hi)) continue;
    const double len = sgn * (hi - lo);  // signed, in the line's direction
    const double lm = 0.5 * ((lo - a.y) * inv_dy + (hi - a.y) * inv_dy);
    *I0 += (double)gw * len * (1.0 - lm);
    *I1 += (double)gw * len * lm;
  }
}

struct BwdLineArgs {
  const PathInfo* pi;
  const uint32_t* slot_path;
  const uint32_t* subpaths;  // combined path: subpath -> first segment, [n_sub + 1]
  const float* wbuf;
  float* grad_points;        // [2 * points] of the combined path
  double* grad_tr_part;      // [waves * 6] per-wave partial dL/d transform
};

// Bernstein weights of a NP-point Bezier at t.
template <int NP>
__device__ inline void bernstein(double t, double* w) {
  const double u = 1.0 - t;
  if (NP == 2) {
    w[0] = u;
    w[1] = t;
  } else if (NP == 3) {
    w[0] = u * u;
    w[1] = 2.0 * t * u;
    w[2] = t * t;
  } else {
    w[0] = u * u * u;
    w[1] = 3.0 * t * u * u;
    w[2] = 3.0 * t * t * u;
    w[3] = t * t * t;
  }
}

// One flatten item of the backward pass: the same subtree as k_flat_lines, each
// leaf line's endpoint gradients pushed to the slot's control points.
template <int NP>
__device__ void bwd_line_item(const DPath& p, uint32_t slot, uint32_t j, int D0, bool active,
                              const Xform& x, double fl, const PathInfo* pi,
                              const uint32_t* slot_path, const BwdLineArgs& b, double* gtr) {
  rzg::Node<NP> n;
  bool walk, leaf;
  int err;
  uint32_t pid;
  flat_subtree<NP, true>(p, slot, j, D0, active, x, fl, pi, slot_path, &n, &walk, &leaf, &err, &pid);
  if (!walk && !leaf) return;
  const PathInfo& P = pi[pid];
  double gp[NP][2];
#pragma unroll
  for (int i = 0; i < NP; ++i) gp[i][0] = gp[i][1] = 0.0;
  auto on_leaf = [&](Pt a, Pt c, int depth, uint64_t bits) {
    if (c.y == a.y) return;
    double I0, I1;
    const double s = (c.x - a.x) / (c.y - a.y);
    line_integrals(P, b.wbuf, a, c, s, &I0, &I1);
    if (I0 == 0.0 && I1 == 0.0) return;
    const double ga[2] = {-I0, s * I0}, gc[2] = {-I1, s * I1};
    const double scale = ldexp(1.0, -depth);
    double wa[NP], wc[NP];
    bernstein<NP>((double)bits * scale, wa);
    bernstein<NP>((double)(bits + 1) * scale, wc);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      gp[i][0] += wa[i] * ga[0] + wc[i] * gc[0];
      gp[i][1] += wa[i] * ga[1] + wc[i] * gc[1];
    }
  };
  if (leaf) {
    // a leaf above the subtree depth: its bits are the top bits of j
    int k = 0;
    uint64_t bits = 0;
    // find the leaf depth again (the walk stopped where the node was flat)
    rzg::Node<NP> r = load_node<NP>(p, slot, P.m);
    while (k < D0 && !(rzg::flatness(r) < fl)) {
      rzg::Node<NP> ch;
      const int bit = (int)((j >> (D0 - 1 - k)) & 1u);
      rzg::child(r, bit, &ch);
      r = ch;
      bits = (bits << 1) | (uint64_t)bit;
      ++k;
    }
    on_leaf(n.p[0], n.p[NP - 1], k, bits);
  } else {
    rzg::traverse_db(n, fl, [&](Pt a, Pt c, int depth, uint64_t bits) {
      on_leaf(a, c, D0 + depth, ((uint64_t)j << depth) | bits);
    });
  }
  // control point indices of the slot (a closing line joins the subpath's
  // last point to its first)
  uint32_t idx[NP];
  const uint32_t item = p.slot_item[slot];
  if (item & 0x80000000u) {
    const uint32_t sub = item & 0x7fffffffu;
    const uint32_t s0 = b.subpaths[sub], s1 = b.subpaths[sub + 1];
    idx[0] = p.pt_off[s1 - 1] + (uint32_t)p.kinds[s1 - 1] + 1u;
    idx[NP - 1] = p.pt_off[s0];
  } else {
#pragma unroll
    for (int i = 0; i < NP; ++i) idx[i] = p.pt_off[item] + (uint32_t)i;
  }
  // transformed point p' = m p: dL/dp = M^T dL/dp', dL/dm += dL/dp' (x, y, 1)
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const double gx = gp[i][0], gy = gp[i][1];
    if (gx == 0.0 && gy == 0.0) continue;
    const double px = p.pts[2 * (size_t)idx[i]], py = p.pts[2 * (size_t)idx[i] + 1];
    atomicAdd(&b.grad_points[2 * (size_t)idx[i]], (float)(P.m[0] * gx + P.m[3] * gy));
    atomicAdd(&b.grad_points[2 * (size_t)idx[i] + 1], (float)(P.m[1] * gx + P.m[4] * gy));
    gtr[0] += gx * px;
    gtr[1] += gx * py;
    gtr[2] += gx;
    gtr[3] += gy * px;
    gtr[4] += gy * py;
    gtr[5] += gy;
  }
}

template <int NP>
__device__ inline void bwd_line_dispatch(const DPath& p, uint32_t slot, uint32_t j, int D0,
                                         bool active, const Xform& x, double fl,
                                         const PathInfo* pi, const uint32_t* slot_path,
                                         const BwdLineArgs& b, double* gtr) {
  bwd_line_item<NP>(p, slot, j, D0, active, x, fl, pi, slot_path, b, gtr);
}

__global__ __launch_bounds__(kBlock, 4) void k_scene_bwd_lines(DPath p, Xform x, double fl, uint32_t bl,
                                                             uint32_t bq, int dq, int dc,
                                                             const PathInfo* pi,
                                                             const uint32_t* slot_path,
                                                             BwdLineArgs b, const Status* st) {
  if (st->err || st->overflow) return;
  double gtr[6] = {0, 0, 0, 0, 0, 0};
  const uint32_t blk = blockIdx.x, t = threadIdx.x;
  if (blk < bl) {
    const uint32_t slot = p.order[blk * kBlock + t];
    bwd_line_dispatch<2>(p, slot, 0, 0, slot != ~0u, x, fl, pi, slot_path, b, gtr);
  } else if (blk < bl + bq) {
    const uint32_t v = (blk - bl) * kBlock + t;
    const uint32_t slot = p.order[p.blocks_line * kBlock + (v >> dq)];
    bwd_line_dispatch<3>(p, slot, v & ((1u << dq) - 1u), dq, slot != ~0u, x, fl, pi, slot_path, b,
                         gtr);
  } else {
    const uint32_t v = (blk - bl - bq) * kBlock + t;
    const uint32_t slot = p.order[(p.blocks_line + p.blocks_quad) * kBlock + (v >> dc)];
    bwd_line_dispatch<4>(p, slot, v & ((1u << dc) - 1u), dc, slot != ~0u, x, fl, pi, slot_path, b,
                         gtr);
  }
  // per-wave partial of dL/d transform
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    double v = gtr[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    gtr[k] = v;
  }
  if ((threadIdx.x & 63) == 0) {
    const size_t wave = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
#pragma unroll
    for (int k = 0; k < 6; ++k) b.grad_tr_part[wave * 6 + k] = gtr[k];
  }
}

// Sum the per-wave transform partials (one block). A run that failed or
// outgrew its buffers wrote no partials, and adds nothing.
__global__ __launch_bounds__(kBlock) void k_sum_tr(const double* part, size_t nwaves, double* out,
                                                    const Status* st) {
  if (st->err || st->overflow) return;
  __shared__ double sh[kBlock];
  for (int k = 0; k < 6; ++k) {
    double v = 0.0;
    for (size_t i = threadIdx.x; i < nwaves; i += kBlock) v += part[i * 6 + k];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = kBlock / 2; o > 0; o >>= 1) {
      if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
      __syncthreads();
    }
    if (threadIdx.x == 0) out[k] += sh[0];
    __syncthreads();
  }
}

}  // namespace rzk
