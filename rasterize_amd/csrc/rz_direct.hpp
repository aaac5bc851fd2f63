// Rasterizer::mask of a small path in one workgroup: flatten, signed-area
// accumulation (src/rasterize.rs:365-470) and row sums with the whole mask in
// LDS, without the binning stage. Used for the glyphs of an atlas whose masks
// fit (direct_lds) where that takes a set less time than the tile pipeline
// (DirectSet).
#pragma once
#include <algorithm>
#include <cmath>

#include "rz_scene.hpp"

namespace rzk {

constexpr int kDirectBlock = 512;  // threads at most (and at least kDirectSlots)
constexpr int kDirectSlots = 128;  // slots staged at once
constexpr int kDirectDepth = 10;   // subdivision depth at most (checked on the host)

// A workgroup's LDS beside its accumulators: the staged slots and the scans.
struct DirectLDS {
  double2 pts[kDirectSlots][4];  // control points under the glyph's transform
  uint32_t pre[kDirectSlots + 1];
  uint32_t kd[kDirectSlots];  // kind | depth << 8
  uint32_t half_total, nodes2[2];
  int marks[kDirectBlock / 64][64];
};
// LDS of the accumulators at most. Up to 70,640 bytes leave room for two
// workgroups a CU; a larger one runs alone (direct_cost).
constexpr size_t kDirectLds = 70 << 10;
constexpr size_t kCuLds = 160 << 10;

// Accumulators: H rows of direct_stride(W) ints, 2^-20 fixed point; four
// columns are a 16-byte read, and the odd number of them keeps neighbouring
// rows in different banks.
RZ_HD int direct_stride(int W) { return (((W + 3) >> 2) | 1) << 2; }
inline size_t direct_lds(size_t W, size_t H) { return (size_t)direct_stride((int)W) * H * sizeof(int); }

// Glyphs up to this size (24 KB: 76x76) are launched apart from larger ones,
// with two waves a workgroup instead of four. 16,384 glyphs of 16 to 128 px:
// these two classes 707 us, one class 792 (four waves) or 1079 (two), five
// classes 766 to 893, eight waves 1228. A set that the chip holds at once is
// one launch of eight waves a glyph, the shortest way through one: 400 glyphs
// 42 us, 46 with four waves, 77 with two.
constexpr size_t kDirectSmall = 24 << 10;

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

// What a glyph costs by this kernel and by the tile pipeline, in ns: of a full
// chip's time (direct, tiles), and of its workgroup's, with nothing beside it
// (chain). `lines`: what its curves and straight segments flatten into;
// straight ones longer than kDirectLong pixels are n_long and long_px in all.
//
// Fitted to sets of 20 to 30,000 equal glyphs of 8 to 1,500 px and 6 to 900
// segments. A workgroup costs 12 to 23 ns however little it does, or what
// its accumulators keep from the CU (two a CU at 132x133 px, 83 ns; one at
// 132x135, 150); a line little; but a long line takes all lanes for its rows,
// one line after the other, and a long side leaves most lanes of the row sums
// idle. Alone, a workgroup's time is its rounds of staged slots and nodes. The
// pipeline's price is in tiles, lines, and the records of long lines.
constexpr double kDirectLong = 16.0;
struct DirectCost {
  double direct = 0.0, tiles = 0.0, chain = 0.0;
};
inline DirectCost direct_cost(int w, int h, uint32_t n_slots, double lines, uint32_t n_long, double long_px) {
  DirectCost c;
  const size_t lds = direct_lds((size_t)w, (size_t)h), all = lds + sizeof(DirectLDS);
  const double kb = (double)all / 1024.0;
  double base = std::fmin(std::fmax(12.0, 0.25 * lines), 22.5);
  if (lds > kDirectSmall) base = (8.0 + 0.55 * kb) * (2 * all > kCuLds ? 2.0 : 1.0);
  c.direct = base + 0.015 * lines + (0.012 + 0.00018 * kb) * long_px + 0.15 * std::max(std::max(w, h) - 256, 0);
  c.tiles = 2.0 + 0.6 * ((w + 15) / 16) * ((h + 15) / 16) + 0.07 * lines + 0.012 * long_px;
  const double rounds = std::fmax((double)n_slots / kDirectSlots, lines / (4.0 * kDirectBlock));
  c.chain = 5000.0 + rounds * (9000.0 + 110.0 * std::min(std::max(w, h), 256)) + 400.0 * n_long +
            100.0 * std::max(w - 256, 0);
  return c;
}

// Whether a set's glyphs that this kernel can mask take less time here than
// with the others (n_binned of them) in the tile pipeline. The pipeline's
// launches cost 60 us and its longest path some; where it runs anyway, it
// still looks at every slot masked here. Measured, us here and there: 5,000
// glyphs of 16x16 and 20 segments 116, 95, 1,000 of them 30, 57; 10,000 of
// 48x48 of 20 225, 189, of 60 279, 336; 4,000 of 132x135 602, 454, 300 of
// them 61, 106; 2,000 polygons of 100 lines in 100x100 236, 218, of 30 127,
// 155; 2,000 of 1500x10 589, 286; 100 of 64x64 of 900 segments 126, 104, of 300
// 51, 67; 400 of 60x60 with one of 200x200 103, 82, 4,000 with one 231, 289.
constexpr double kTilesFixed = 60000.0, kTilesChain = 20.0, kTilesSlot = 0.13, kDirectFixed = 10000.0;
struct DirectSet {
  DirectCost sum;  // (chain: the longest)
  double slots = 0.0, most_slots = 0.0;
  void add(const DirectCost& c, uint32_t n_slots) {
    sum.direct += c.direct;
    sum.tiles += c.tiles;
    sum.chain = std::fmax(sum.chain, c.chain);
    slots += n_slots;
    most_slots = std::fmax(most_slots, (double)n_slots);
  }
  bool direct(uint32_t n_binned) const {
    // the longest chain lies beside the other workgroups only in part (400
    // polygons of 200 lines in 100x100: 155 us, 100 of them 131; 128 by the
    // pipeline)
    const double here =
        kDirectFixed + std::fmax(sum.chain, sum.direct) + 0.1 * std::fmin(sum.chain, sum.direct);
    if (n_binned) return here + kTilesSlot * slots < sum.tiles;
    return here < kTilesFixed + kTilesChain * most_slots + sum.tiles;
  }
};

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

// One lane's part of a curve's subdivision (PathFlattenIter's nodes, tests and
// leaves): the node reached from the root along `bits` (most significant
// first) in `levels` levels, and its leaves below. A curve's leaves lie at
// depth levels + 2 at most (leaf_depth), so they are the node itself, its
// children or its grandchildren.
enum { SUB_NONE = 0, SUB_LEAF = 1, SUB_SPLIT = 2 };
template <int NP>
__device__ inline int sub_node(const double2* root, uint32_t bits, int levels, double fl,
                               rzg::Node<NP>* n) {
#pragma unroll
  for (int i = 0; i < NP; ++i) n->p[i] = rzg::mkpt(root[i].x, root[i].y);
  for (int left = levels;; --left) {
    // a leaf above the node belongs to the bits that end in zeros
    if (rzg::flatness(*n) < fl) return (bits & ((1u << left) - 1u)) == 0 ? SUB_LEAF : SUB_NONE;
    if (left == 0) return SUB_SPLIT;
    to_child(*n, (bits >> (left - 1)) & 1u);
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

// Heights are rounded to 2^-20 of a pixel once per vertex (relative to any
// pixel row: the same everywhere), and a row's total deposit is the difference
// of two such heights, so that what the lines of a closed chain deposit in a
// row cancels exactly to the right of them.
__device__ inline int fix_height(double y) { return __double2int_rn(y * (double)(1 << rzg::kFixShift)); }

// The deposits of a piece with total D (2^-20) in pixel row r, from column c +
// u to c + v (0 <= u < 1): each column its share of the exact area, the last
// one what the others leave of D. Without a branch up to two columns, which
// nearly all lines of a flattened curve stay in; the reciprocal's error (one
// unit in the last place) is below the rounding to 2^-20.
__device__ inline void direct_cols(const DirectMask& M, int r, int c, float u, float v, int D) {
  const float d = (float)D;
  if (v > 2.0f) {
    // the mean coverage of each column by the piece, differenced
    const float s = 1.0f / (v - u);
    const int n = (int)ceilf(v);  // columns c .. c + n - 1 are crossed
    int sum = __float2int_rn(d * (0.5f * s * (1.0f - u) * (1.0f - u)));
    M.add(r, c, sum);
    for (int k = 1; k < n; ++k) {
      const float e = fminf((float)(k + 1), v);
      const float in = s * (e - (float)k);  // share of the piece inside column k
      const float cov = s * ((float)k - u) + in * (1.0f - 0.5f * (e - (float)k));
      const int A = __float2int_rn(d * cov) - sum;
      M.add(r, c + k, A);
      sum += A;
    }
    M.add(r, c + n, D - sum);
    return;
  }
  const bool one = v <= 1.0f;
  const float s = __builtin_amdgcn_rcpf(v - u), p = 1.0f - u, e = v - 1.0f;
  const float cov0 = one ? 1.0f - 0.5f * (u + v) : 0.5f * p * p * s;
  const int A0 = __float2int_rn(d * cov0);
  const int A1 = one ? D - A0 : __float2int_rn(d * ((p + e * (1.0f - 0.5f * e)) * s)) - A0;
  const int A2 = D - A0 - A1;
  M.add(r, c, A0);
  M.add(r, c + 1, A1);
  if (A2) M.add(r, c + 2, A2);
}

// A piece of a line with 0 <= x <= W, lower end first.
struct DirectPiece {
  double x0, y0, x1, y1;
  int dir;     // +-1
  int r0, r1;  // pixel rows [r0, r1), none: nothing to deposit
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
  if (lo < hi) {
    q.r0 = (int)floor(lo);
    q.r1 = (int)ceil(hi);
  }
  return q;
}

// A short piece, by its lane: at most four rows and 16 columns, so that f32
// positions relative to its first row and column are exact to 2^-20.
__device__ inline void direct_short(const DirectMask& M, const DirectPiece& q) {
  const double xl = floor(fmin(q.x0, q.x1)), yr = (double)q.r0;
  const float x0 = (float)(q.x0 - xl), x1 = (float)(q.x1 - xl);
  const int Y0 = fix_height(q.y0 - yr), Y1 = fix_height(q.y1 - yr);
  const int c0 = (int)xl;
  constexpr int one = 1 << rzg::kFixShift;
  // per 2^-20 of a row. The reciprocal (one unit in the last place) and the
  // two products move a cut of a piece of up to 16 px by up to 2^-18. Against
  // the oracle in f64 the masks are nearer than the tile pipeline's, which
  // rounds its records to f32: thirty triangles within 16 x 4 px 7.4e-7 of the mask's norm,
  // 2.6e-6 there, sixty within 16 x 1 2.1e-6, 9.4e-6, text 2.5e-7 to 4.7e-7, 6.5e-7 to 1.2e-6.
  const float slope = Y1 > Y0 ? (x1 - x0) * __builtin_amdgcn_rcpf((float)(Y1 - Y0)) : 0.0f;
  for (int r = q.r0; r < q.r1; ++r) {
    const int ry = (r - q.r0) << rzg::kFixShift;
    const int top = max(Y0, ry), bot = min(Y1, ry + one);
    const float xt = x0 + slope * (float)(top - Y0);
    const float xb = bot == Y1 ? x1 : x0 + slope * (float)(bot - Y0);
    const float lo = fmaxf(fminf(xt, xb), 0.0f);
    const float fl = floorf(lo);
    direct_cols(M, r, c0 + (int)fl, lo - fl, fmaxf(xt, xb) - fl, q.dir * (bot - top));
  }
}

// One row of a longer piece, positions in f64.
__device__ inline void direct_row(const DirectMask& M, const DirectPiece& q, double dxdy, int r) {
  const double rt = (double)r, rb = rt + 1.0;
  const bool in0 = q.y0 >= rt, in1 = q.y1 <= rb;  // the ends lie in this row
  const double xt = in0 ? q.x0 : q.x0 + dxdy * (rt - q.y0);
  const double xb = in1 ? q.x1 : q.x0 + dxdy * (rb - q.y0);
  const int f0 = in0 ? fix_height(q.y0 - rt) : 0, f1 = in1 ? fix_height(q.y1 - rt) : 1 << rzg::kFixShift;
  const double xl = floor(fmax(fmin(xt, xb), 0.0));
  direct_cols(M, r, (int)xl, (float)(fmax(fmin(xt, xb), 0.0) - xl), (float)(fmax(xt, xb) - xl), q.dir * (f1 - f0));
}

// A line per lane (have) into the accumulators: right clip and left split
// (rzg::effective_line) where a lane's line needs them, short pieces by their
// lanes, longer ones row by row by the whole wave. Every lane takes part.
__device__ inline void direct_line(const DirectMask& M, const rzg::BinGrid& g, bool have, Pt a, Pt b,
                                   int lane) {
  int left = have ? 1 : 0;  // pieces left: (a, b), then (b, c)
  Pt c = b;
  if (have && !(fmin(a.x, b.x) >= 0.0 && fmax(a.x, b.x) <= g.wc)) {
    const rzg::EffLine e = rzg::effective_line(a, b, g);
    left = e.n;
    a = e.p[0];
    b = e.p[1];
    c = e.p[2];
  }
  for (; __ballot(left > 0); --left, a = b, b = c) {
    DirectPiece q;
    q.x0 = q.y0 = q.x1 = q.y1 = 0.0;
    q.dir = 1;
    q.r0 = q.r1 = 0;
    if (left > 0) q = direct_piece(a, b, M.H);
    const int rows = q.r1 - q.r0;
    const bool small = rows <= 4 && fabs(q.x1 - q.x0) <= 16.0 && q.y1 - q.y0 <= 16.0;
    if (rows > 0 && small) direct_short(M, q);
    uint64_t m = __ballot(rows > 0 && !small);
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
      const double dxdy = (w.x1 - w.x0) / (w.y1 - w.y0);
      for (int r = w.r0 + lane; r < w.r1; r += 64) direct_row(M, w, dxdy, r);
    }
  }
}

// One glyph per workgroup. Its slots are staged kDirectSlots at a time with
// their control points under the glyph's transform. The subdivision nodes two
// levels above the deepest leaves (fewer where that leaves lanes idle) are
// dealt out to the lanes; a lane walks to its node (one or two levels for a
// glyph's curves) and deposits the up to four lines below it: no depth-first
// walk whose lanes wait for the longest subtree. Then a wave sums four rows at
// a time, 64 pixels each, and writes the mask.
// Bound by latency and VALU issue (40% of the SIMD cycles). Against the tile
// pipeline: 400 glyphs 114 -> 43 us, 16,384 glyphs 1178 -> 707 us.
// CUBIC: some path has cubics (a TrueType font's have none, and the kernel
// without them fits four waves per SIMD).
template <int RULE, bool CUBIC>
__global__ __launch_bounds__(kDirectBlock) void k_atlas_direct(DirectArgs a) {
  extern __shared__ int4 acc4[];
  int* acc = (int*)acc4;
  __shared__ DirectLDS L;
  auto& pts = L.pts;
  auto& pre = L.pre;
  auto& kd = L.kd;
  auto& half_total = L.half_total;
  auto& nodes2 = L.nodes2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nt = (int)blockDim.x;
  int* marks = L.marks[wave];
  const uint32_t glyph = load_const(a.list + blockIdx.x);
  const AtlasSlot S = load_const(a.slots + glyph);
  rzg::BinGrid g{};
  g.mode = a.mode;
  g.W = S.w;
  g.H = S.h;
  g.wc = a.mode == rzg::EDGE_MASK ? (double)S.w - 1.0 : (double)S.w;
  const DirectMask M{acc, direct_stride(S.w), S.w, S.h};
  for (int i = tid; i < M.H * (M.stride / 4); i += nt) ((int4*)acc)[i] = make_int4(0, 0, 0, 0);
  const uint32_t s_end = load_const(a.slot_begin + glyph + 1);
  uint32_t lines = 0;
  bool deep = false;
  for (uint32_t s0 = load_const(a.slot_begin + glyph); s0 < s_end; s0 += kDirectSlots) {
    __syncthreads();  // the previous slots have been read
    int my_depth = -1;
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
          } else if (CUBIC && kind == rzg::KIND_CUBIC) {
            depth = leaf_depth(flatness_bound(q), a.fl);
          }
          if (depth > kDirectDepth) {
            deep = true;
            depth = kDirectDepth;
          }
        }
        kd[tid] = (uint32_t)kind | (uint32_t)depth << 8;
        my_depth = depth;
      }
      uint32_t total;
      (void)wave_excl_scan(my_depth < 0 ? 0u : 1u << max(my_depth - 2, 0), lane, &total);
      if (lane == 0) nodes2[wave] = total;
    }
    __syncthreads();
    // levels a lane takes below its node
    const uint32_t n2 = nodes2[0] + nodes2[1];
    const int below = n2 * 4u <= (uint32_t)nt ? 0 : n2 * 2u <= (uint32_t)nt ? 1 : 2;
    if (tid < kDirectSlots) {
      const uint32_t n = my_depth < 0 ? 0u : 1u << max(my_depth - below, 0);
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
    for (uint32_t j0 = (uint32_t)wave * 64u; j0 < total; j0 += (uint32_t)nt) {
      // owner of node j0 + lane: the last slot that starts at or before it
      marks[lane] = -1;
      wave_lds_sync();
      if (v0 && p0 >= j0 && p0 - j0 < 64u) marks[p0 - j0] = lane;
      if (v1 && p1 >= j0 && p1 - j0 < 64u) marks[p1 - j0] = 64 + lane;
      const uint64_t b1 = __ballot(v1 && p1 <= j0), b0 = __ballot(v0 && p0 <= j0);
      const int first = b1 ? 127 - __clzll((long long)b1) : 63 - __clzll((long long)b0);
      wave_lds_sync();
      const int o = max(dpp_max_scan(marks[lane]), first);
      const uint32_t j = j0 + (uint32_t)lane;
      int sub = SUB_NONE;
      const uint32_t q = kd[o];
      const int kind = j < total ? (int)(q & 255u) : -1;
      rzg::Node<4> n;  // a line's or quad's points in the first two or three
#pragma unroll
      for (int i = 0; i < 4; ++i) n.p[i] = rzg::mkpt(0.0, 0.0);
      const int levels = max((int)(q >> 8) - below, 0);
      if (kind == rzg::KIND_QUAD) {
        rzg::Node<3> t;
        sub = sub_node(pts[o], j - pre[o], levels, a.fl, &t);
        n.p[0] = t.p[0];
        n.p[1] = t.p[1];
        n.p[2] = t.p[2];
      } else if (CUBIC && kind == rzg::KIND_CUBIC) {
        sub = sub_node(pts[o], j - pre[o], levels, a.fl, &n);
      } else if (kind == rzg::KIND_LINE) {
        n.p[0] = rzg::mkpt(pts[o][0].x, pts[o][0].y);
        n.p[1] = rzg::mkpt(pts[o][1].x, pts[o][1].y);
        sub = SUB_LEAF;
      }
      // the node's chord, or its children's, or its grandchildren's
#pragma unroll 1
      for (int h = 0; h < 2; ++h) {
        if (h && !__ballot(sub == SUB_SPLIT)) break;
        rzg::Node<4> c = n;
        bool leaf = true;  // c's chord is one of the lines
        if (sub == SUB_SPLIT) {
          if (!CUBIC || kind == rzg::KIND_QUAD) {
            rzg::Node<3> t;
            t.p[0] = n.p[0];
            t.p[1] = n.p[1];
            t.p[2] = n.p[2];
            to_child(t, h != 0);
            leaf = rzg::flatness(t) < a.fl;
            c.p[0] = t.p[0];
            c.p[1] = t.p[1];
            c.p[2] = t.p[2];
          } else {
            to_child(c, h != 0);
            leaf = rzg::flatness(c) < a.fl;
          }
        }
#pragma unroll 1
        for (int k = 0; k < 2; ++k) {
          bool have = sub == SUB_SPLIT || (sub == SUB_LEAF && h == 0);
          if (leaf && k) have = false;
          if (!__ballot(have)) break;
          Pt u = c.p[0], v = CUBIC && kind == rzg::KIND_CUBIC ? c.p[3] : kind == rzg::KIND_QUAD ? c.p[2] : c.p[1];
          if (have && !leaf) {
            if (!CUBIC || kind == rzg::KIND_QUAD) {
              rzg::Node<3> t;
              t.p[0] = c.p[0];
              t.p[1] = c.p[1];
              t.p[2] = c.p[2];
              to_child(t, k != 0);
              deep = deep || !(rzg::flatness(t) < a.fl);
              u = t.p[0];
              v = t.p[2];
            } else {
              rzg::Node<4> t = c;
              to_child(t, k != 0);
              deep = deep || !(rzg::flatness(t) < a.fl);
              u = t.p[0];
              v = t.p[3];
            }
          }
          lines += (uint32_t)__popcll(__ballot(have));
          direct_line(M, g, have, u, v, lane);
        }
      }
    }
  }
  if (deep) set_err(a.st, rzg::ST_DEPTH);
  if (lane == 0 && lines) atomicAdd(&a.st->n_lines, lines);
  __syncthreads();
  // row sums: 16 lanes a row, four columns a lane; the sum so far carried from
  // lane 15 to lane 0 (row_ror:1)
  const int first_lane = (lane & 15) == 0 ? -1 : 0;
  for (int r0 = wave * 4; r0 < M.H; r0 += nt >> 4) {
    const int r = r0 + (lane >> 4);
    const bool in = r < M.H;
    const int* row = acc + r * M.stride;
    float* out = a.out + (size_t)(S.y + r) * a.row_stride + S.x;
    int run = 0;
    for (int c0 = 0; c0 < M.W; c0 += 64) {
      const int c = c0 + ((lane & 15) << 2);
      int4 w = make_int4(0, 0, 0, 0);
      if (in && c < M.W) w = *(const int4*)(row + c);
      w.y += w.x;
      w.z += w.y;
      w.w += w.z;
      int t = w.w + (__builtin_amdgcn_update_dpp(0, run, 0x121, 0xf, 0xf, false) & first_lane);
      t += __builtin_amdgcn_update_dpp(0, t, 0x111, 0xf, 0xf, false);
      t += __builtin_amdgcn_update_dpp(0, t, 0x112, 0xf, 0xf, false);
      t += __builtin_amdgcn_update_dpp(0, t, 0x114, 0xf, 0xf, false);
      t += __builtin_amdgcn_update_dpp(0, t, 0x118, 0xf, 0xf, false);
      run = t;
      const int base = t - w.w;
      const float v[4] = {alpha_fix<RULE>(base + w.x), alpha_fix<RULE>(base + w.y),
                          alpha_fix<RULE>(base + w.z), alpha_fix<RULE>(base + w.w)};
      if (in && c < M.W) MaskOut{out, 0}.put(c, 0, min(4, M.W - c), v);
    }
  }
}

}  // namespace rzk
