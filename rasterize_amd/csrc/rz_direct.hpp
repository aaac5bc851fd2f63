// Rasterizer::mask of a small path in one workgroup: flatten, signed-area
// accumulation (src/rasterize.rs:365-470) and row sums with the whole mask in
// LDS, without the binning stage. Used for the glyphs of an atlas whose masks
// fit (direct_lds); larger ones go through the tile pipeline.
#pragma once
#include "rz_scene.hpp"

namespace rzk {

constexpr int kDirectBlock = 256;
constexpr int kDirectSlots = 128;  // slots staged at once
constexpr int kDirectDepth = 10;   // subdivision depth at most (checked on the host)
// LDS of the accumulators at most: two workgroups per CU
constexpr size_t kDirectLds = 70 << 10;

// Accumulators: H rows of W | 1 ints (odd: neighbouring rows in different
// banks), 2^-20 fixed point.
inline size_t direct_lds(size_t W, size_t H) { return (W | 1) * H * sizeof(int); }

// A bound on the flatness of a curve's nodes: at depth k of its subdivision
// none is above bound / 16^k. A quad's second difference
// is quartered by every split; a cubic's two second differences a, b become
// convex combinations of a / 4 and b / 4, and its flatness vectors are 2a + b
// and a + 2b.
RZ_HD double flatness_bound(const rzg::Node<3>& n) { return rzg::flatness(n); }
RZ_HD double flatness_bound(const rzg::Node<4>& n) {
  const double ax = fabs(n.p[0].x - 2.0 * n.p[1].x + n.p[2].x), bx = fabs(n.p[1].x - 2.0 * n.p[2].x + n.p[3].x);
  const double ay = fabs(n.p[0].y - 2.0 * n.p[1].y + n.p[2].y), by = fabs(n.p[1].y - 2.0 * n.p[2].y + n.p[3].y);
  const double mx = fmax(ax, bx), my = fmax(ay, by);
  return 9.0 * (mx * mx + my * my);
}

// The depth at which every node is flat. The margin covers the rounding of
// the nodes' flatness: direct_ok keeps it below 2e-7 of the threshold.
RZ_HD int leaf_depth(double bound, double fl) {
  int k = 0;
  while (k < 31 && !(bound < fl * (1.0 - 1e-6))) {
    bound *= 0.0625;
    ++k;
  }
  return k;
}

// Whether curves with this flatness bound and these largest coordinates can be
// flattened to threshold fl by leaf_depth within kDirectDepth: a node's
// coordinates carry a rounding of a few ulps of the largest coordinate, which
// must stay small against the flatness vector's threshold sqrt(fl).
inline bool direct_ok(double bound, double max_coord, double fl) {
  return leaf_depth(bound, fl) <= kDirectDepth && max_coord * 1e-14 < 1e-7 * sqrt(fl);
}

struct DirectArgs {
  DPath p;
  const uint32_t* list;        // the glyphs of this launch
  const AtlasSlot* slots;
  const uint32_t* slot_begin;  // [glyphs + 1] a glyph's flatten slots
  double fl;
  int mode;
  float* out;
  size_t row_stride;
  Status* st;
};

// The child of a node at t = 1/2 (rzg::child, same operations), by selects.
__device__ inline double sel(bool c, double a, double b) { return c ? a : b; }
__device__ inline Pt sel(bool c, Pt a, Pt b) { return rzg::mkpt(sel(c, a.x, b.x), sel(c, a.y, b.y)); }
__device__ inline Pt half(Pt a, Pt b) { return rzg::mkpt(0.5 * a.x + 0.5 * b.x, 0.5 * a.y + 0.5 * b.y); }
__device__ inline Pt quarters(Pt a, Pt b, Pt c) {
  return rzg::mkpt(0.25 * a.x + 0.5 * b.x + 0.25 * c.x, 0.25 * a.y + 0.5 * b.y + 0.25 * c.y);
}
__device__ inline void to_child(rzg::Node<3>& n, bool r) {
  const Pt mid = quarters(n.p[0], n.p[1], n.p[2]);
  const Pt side = half(sel(r, n.p[1], n.p[0]), sel(r, n.p[2], n.p[1]));
  n.p[0] = sel(r, mid, n.p[0]);
  n.p[2] = sel(r, n.p[2], mid);
  n.p[1] = side;
}
__device__ inline void to_child(rzg::Node<4>& n, bool r) {
  const Pt mid = rzg::mkpt(0.125 * n.p[0].x + 0.375 * n.p[1].x + 0.375 * n.p[2].x + 0.125 * n.p[3].x,
                           0.125 * n.p[0].y + 0.375 * n.p[1].y + 0.375 * n.p[2].y + 0.125 * n.p[3].y);
  const Pt q0 = sel(r, n.p[1], n.p[0]), q1 = sel(r, n.p[2], n.p[1]), q2 = sel(r, n.p[3], n.p[2]);
  const Pt inner = quarters(q0, q1, q2), outer = half(sel(r, q1, q0), sel(r, q2, q1));
  n.p[0] = sel(r, mid, n.p[0]);
  n.p[3] = sel(r, n.p[3], mid);
  n.p[1] = sel(r, inner, outer);
  n.p[2] = sel(r, outer, inner);
}

// The leaf of the root's subdivision along the depth bits `bits`: the chord,
// if this thread owns it (a leaf above `depth` belongs to the bits that end in
// zeros). The same nodes, tests and leaves as PathFlattenIter's.
template <int NP>
__device__ inline bool leaf_line(const double2* root, uint32_t bits, int depth, double fl, Pt* a,
                                 Pt* b, bool* deep) {
  rzg::Node<NP> n;
#pragma unroll
  for (int i = 0; i < NP; ++i) n.p[i] = rzg::mkpt(root[i].x, root[i].y);
  for (int left = depth;; --left) {
    if (rzg::flatness(n) < fl) {
      *a = n.p[0];
      *b = n.p[NP - 1];
      return (bits & ((1u << left) - 1u)) == 0;
    }
    if (left == 0) {
      *deep = true;
      return false;
    }
    to_child(n, (bits >> (left - 1)) & 1u);
  }
}

// One glyph's accumulators.
struct DirectMask {
  int* acc;
  int stride, W, H;
  __device__ void add(int row, int col, int v) const {
    if ((unsigned)col < (unsigned)W) atomicAdd(&acc[row * stride + col], v);
  }
};

// A piece prepared for its row steps: lower end first.
struct DirectPiece {
  double x0, y0, x1, y1;
  int dir;  // +-1, 0: nothing to deposit
  int r0, r1;
};

__device__ inline DirectPiece direct_piece(Pt a, Pt b, int H) {
  DirectPiece q;
  const bool up = a.y > b.y;
  q.x0 = up ? b.x : a.x;
  q.y0 = up ? b.y : a.y;
  q.x1 = up ? a.x : b.x;
  q.y1 = up ? a.y : b.y;
  q.dir = up ? -1 : 1;
  const double lo = fmax(q.y0, 0.0), hi = fmin(q.y1, (double)H);
  q.r0 = q.r1 = 0;
  if (!(lo < hi)) {
    q.dir = 0;
    return q;
  }
  q.r0 = (int)floor(lo);
  q.r1 = (int)ceil(hi);
  return q;
}

// The deposits of the piece in pixel row r (0 <= x <= W). Positions are f64,
// the fractions inside the row's pixels f32. The row's total is the difference
// of its ends' heights in fixed point, so that what neighbouring lines of a
// closed chain deposit cancels exactly to the right of them; the last column
// takes what the others leave of it.
__device__ inline void direct_row(const DirectMask& M, const DirectPiece& q, double dxdy, int r) {
  const double rt = (double)r, rb = rt + 1.0;
  const bool in0 = q.y0 >= rt, in1 = q.y1 <= rb;  // the ends lie in this row
  const double xt = in0 ? q.x0 : q.x0 + dxdy * (rt - q.y0);
  const double xb = in1 ? q.x1 : q.x0 + dxdy * (rb - q.y0);
  const int f0 = in0 ? __float2int_rn((float)(q.y0 - rt) * kFix) : 0;
  const int f1 = in1 ? __float2int_rn((float)(q.y1 - rt) * kFix) : 1 << rzg::kFixShift;
  const int D = q.dir * (f1 - f0);
  const double xl = floor(fmax(fmin(xt, xb), 0.0));
  const int c = (int)xl;
  const float u = (float)(fmin(xt, xb) - xl), v = (float)(fmax(xt, xb) - xl);
  const float d = (float)D;
  if (v <= 1.0f) {
    const int A = __float2int_rn(d * (1.0f - 0.5f * (u + v)));
    M.add(r, c, A);
    M.add(r, c + 1, D - A);
    return;
  }
  // several columns: the area left of each column's right edge, differenced
  const float s = 1.0f / (v - u);
  const int n = (int)ceilf(v);  // columns c .. c + n - 1 are crossed
  float prev = 0.5f * s * (1.0f - u) * (1.0f - u);
  int sum = __float2int_rn(d * prev);
  M.add(r, c, sum);
  for (int k = 1; k < n; ++k) {
    // mean coverage of column k by the piece: exact trapezoid, 1 past its end
    const float e = fminf((float)(k + 1), v);
    const float in = s * (e - (float)k);                       // share of the piece inside
    const float cov = s * ((float)k - u) + in * (1.0f - 0.5f * (e - (float)k));
    const int A = __float2int_rn(d * cov) - sum;
    M.add(r, c + k, A);
    sum += A;
  }
  M.add(r, c + n, D - sum);
}

// A line per lane (have) into the accumulators: right clip and left split
// (rzg::effective_line), then each piece's rows: up to four by the lane
// itself, more by the whole wave. Every lane takes part.
__device__ inline void direct_line(const DirectMask& M, const rzg::BinGrid& g, bool have, Pt a, Pt b,
                                   int lane) {
  rzg::EffLine e;
  e.n = 0;
  if (have) e = rzg::effective_line(a, b, g);
  for (int pc = 0; __ballot(pc < e.n); ++pc) {
    DirectPiece q;
    q.dir = 0;
    q.r0 = q.r1 = 0;
    if (pc < e.n) q = direct_piece(pc ? e.p[1] : e.p[0], pc ? e.p[2] : e.p[1], M.H);
    const int rows = q.r1 - q.r0;
    double dxdy = 0.0;
    if (q.dir && (rows > 1 || q.y0 < 0.0 || q.y1 > (double)M.H)) dxdy = (q.x1 - q.x0) / (q.y1 - q.y0);
    if (q.dir && rows <= 4)
      for (int r = q.r0; r < q.r1; ++r) direct_row(M, q, dxdy, r);
    uint64_t m = __ballot(q.dir && rows > 4);
    while (m) {
      const int src = __ffsll((unsigned long long)m) - 1;
      m &= m - 1;
      auto of = [&](double v) {
        return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src),
                                __builtin_amdgcn_readlane(__double2loint(v), src));
      };
      DirectPiece w;
      w.x0 = of(q.x0);
      w.y0 = of(q.y0);
      w.x1 = of(q.x1);
      w.y1 = of(q.y1);
      w.dir = __builtin_amdgcn_readlane(q.dir, src);
      w.r0 = __builtin_amdgcn_readlane(q.r0, src);
      w.r1 = __builtin_amdgcn_readlane(q.r1, src);
      const double s = of(dxdy);
      for (int r = w.r0 + lane; r < w.r1; r += 64) direct_row(M, w, s, r);
    }
  }
}

// One glyph per workgroup. Its slots are staged kDirectSlots at a time with
// their control points under the glyph's transform; the leaves of all staged
// curves at their deepest level are dealt out to the lanes, each of which
// walks from the root to its leaf (three or four levels for a glyph's curves:
// less work than a depth-first walk whose lanes wait for the longest subtree)
// and deposits the line. Then a wave sums four rows at a time, 16 pixels each,
// and writes the mask.
// Bound by VALU issue. DIRECT
template <int RULE>
__global__ __launch_bounds__(kDirectBlock) void k_atlas_direct(DirectArgs a) {
  extern __shared__ int acc[];
  __shared__ double2 pts[kDirectSlots][4];
  __shared__ uint32_t pre[kDirectSlots + 1];
  __shared__ uint32_t kd[kDirectSlots];  // kind | depth << 8
  __shared__ uint32_t half_total;
  __shared__ int marks_all[kDirectBlock / 64][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int* marks = marks_all[wave];
  const uint32_t glyph = load_const(a.list + blockIdx.x);
  const AtlasSlot S = load_const(a.slots + glyph);
  rzg::BinGrid g{};
  g.mode = a.mode;
  g.W = S.w;
  g.H = S.h;
  g.wc = a.mode == rzg::EDGE_MASK ? (double)S.w - 1.0 : (double)S.w;
  const DirectMask M{acc, S.w | 1, S.w, S.h};
  for (int i = tid; i < M.H * M.stride; i += kDirectBlock) acc[i] = 0;
  const uint32_t s_end = load_const(a.slot_begin + glyph + 1);
  uint32_t lines = 0;
  bool deep = false;
  for (uint32_t s0 = load_const(a.slot_begin + glyph); s0 < s_end; s0 += kDirectSlots) {
    __syncthreads();  // the previous slots have been read
    uint32_t n = 0;
    if (tid < kDirectSlots) {
      const uint32_t slot = s0 + (uint32_t)tid;
      if (slot < s_end) {
        const uint32_t item = a.p.slot_item[slot];
        int kind = rzg::KIND_LINE, depth = 0;
        if (item & 0x80000000u) {
          const rzg::Node<2> q = load_node<2>(a.p, slot, S.m);
          pts[tid][0] = make_double2(q.p[0].x, q.p[0].y);
          pts[tid][1] = make_double2(q.p[1].x, q.p[1].y);
        } else {
          kind = a.p.kinds[item];
          const double* c = a.p.pts + 2 * (size_t)a.p.pt_off[item];
          rzg::Node<4> q;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int k = min(i, kind + 1);
            q.p[i] = rzg::tr_apply(S.m, rzg::mkpt(c[2 * k], c[2 * k + 1]));
            pts[tid][i] = make_double2(q.p[i].x, q.p[i].y);
          }
          if (kind == rzg::KIND_QUAD) {
            rzg::Node<3> t;
            t.p[0] = q.p[0];
            t.p[1] = q.p[1];
            t.p[2] = q.p[2];
            depth = leaf_depth(flatness_bound(t), a.fl);
          } else if (kind == rzg::KIND_CUBIC) {
            depth = leaf_depth(flatness_bound(q), a.fl);
          }
          if (depth > kDirectDepth) {
            deep = true;
            depth = kDirectDepth;
          }
        }
        kd[tid] = (uint32_t)kind | (uint32_t)depth << 8;
        n = 1u << depth;
      }
      uint32_t total;
      const uint32_t ex = wave_excl_scan(n, lane, &total);
      pre[tid] = ex;
      if (tid == 0) half_total = total;
      if (tid == kDirectSlots - 1) pre[kDirectSlots] = total;
    }
    __syncthreads();
    if (tid >= 64 && tid < kDirectSlots) pre[tid] += half_total;
    if (tid == 0) pre[kDirectSlots] += half_total;
    __syncthreads();
    const uint32_t total = pre[kDirectSlots];
    const uint32_t p0 = pre[lane], p1 = pre[64 + lane];
    const bool v0 = pre[lane + 1] > p0, v1 = pre[65 + lane] > p1;
    for (uint32_t j0 = (uint32_t)wave * 64u; j0 < total; j0 += kDirectBlock) {
      // owner of leaf j0 + lane: the last slot that starts at or before it
      marks[lane] = -1;
      wave_lds_sync();
      if (v0 && p0 >= j0 && p0 - j0 < 64u) marks[p0 - j0] = lane;
      if (v1 && p1 >= j0 && p1 - j0 < 64u) marks[p1 - j0] = 64 + lane;
      const uint64_t b1 = __ballot(v1 && p1 <= j0), b0 = __ballot(v0 && p0 <= j0);
      const int first = b1 ? 127 - __clzll((long long)b1) : 63 - __clzll((long long)b0);
      wave_lds_sync();
      const int o = max(dpp_max_scan(marks[lane]), first);
      const uint32_t j = j0 + (uint32_t)lane;
      Pt u = rzg::mkpt(0.0, 0.0), v = u;
      bool have = false;
      if (j < total) {
        const uint32_t bits = j - pre[o], q = kd[o];
        const int kind = (int)(q & 255u), depth = (int)(q >> 8);
        if (kind == rzg::KIND_QUAD) {
          have = leaf_line<3>(pts[o], bits, depth, a.fl, &u, &v, &deep);
        } else if (kind == rzg::KIND_CUBIC) {
          have = leaf_line<4>(pts[o], bits, depth, a.fl, &u, &v, &deep);
        } else {
          u = rzg::mkpt(pts[o][0].x, pts[o][0].y);
          v = rzg::mkpt(pts[o][1].x, pts[o][1].y);
          have = true;
        }
      }
      lines += (uint32_t)__popcll(__ballot(have));
      direct_line(M, g, have, u, v, lane);
    }
  }
  if (deep) set_err(a.st, rzg::ST_DEPTH);
  if (lane == 0 && lines) atomicAdd(&a.st->n_lines, lines);
  __syncthreads();
  // row sums: 16 lanes a row, 16 columns at a time, the sum so far carried
  // from lane 15 to lane 0 (row_ror:1)
  const int col = lane & 15;
  const int first_lane = col == 0 ? -1 : 0;
  for (int r0 = wave * 4; r0 < M.H; r0 += 4 * (kDirectBlock / 64)) {
    const int r = r0 + (lane >> 4);
    const bool in = r < M.H;
    const int* row = acc + r * M.stride;
    float* out = a.out + (size_t)(S.y + r) * a.row_stride + S.x;
    int run = 0;
    for (int c0 = 0; c0 < M.W; c0 += 16) {
      const int c = c0 + col;
      const bool px = in && c < M.W;
      int w = px ? row[c] : 0;
      w += __builtin_amdgcn_update_dpp(0, run, 0x121, 0xf, 0xf, false) & first_lane;
      w += __builtin_amdgcn_update_dpp(0, w, 0x111, 0xf, 0xf, false);
      w += __builtin_amdgcn_update_dpp(0, w, 0x112, 0xf, 0xf, false);
      w += __builtin_amdgcn_update_dpp(0, w, 0x114, 0xf, 0xf, false);
      w += __builtin_amdgcn_update_dpp(0, w, 0x118, 0xf, 0xf, false);
      run = w;
      if (px) out[c] = alpha_fix<RULE>(w);
    }
  }
}

}  // namespace rzk
