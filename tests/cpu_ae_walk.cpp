// Host check of rzg::ae_piece, which skips and shortens the rows of an edge that
// cannot come out left of x = 0, against the walk of every row
// (ActiveEdgeIter, src/rasterize.rs:820-850): the same vertices, bit for bit,
// on edges that start, end, touch or cross near x = 0, steep and flat, from
// above the image to below it, both ways round. Prints the edges with vertices;
// exits 1 at the first difference.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>
#include "../rasterize_amd/csrc/rz_geom.hpp"

// The rows of the piece a -> b (one ActiveEdgeIter edge) below image row H:
// vertices after a up to (not including) b, through `to`.
template <typename To>
inline void ae_piece_rows(rzg::Pt a, rzg::Pt b, double H, To&& to) {
  if (fabs(a.y - b.y) < rzg::kEps) return;  // Edge::new: no rows
  const bool up = a.y <= b.y;
  const rzg::Pt lo = up ? a : b, hi = up ? b : a;
  const double dxdy = (hi.x - lo.x) / (hi.y - lo.y);
  rzg::Pt p = lo;
  if (p.y < 0.0) p = rzg::mkpt(p.x - p.y * dxdy, 0.0);
  if (!(fmin(p.x, hi.x) < rzg::kAeNear)) return;
  rzg::Pt rs[rzg::kAeRuns];
  bool rf[rzg::kAeRuns];
  int nr = 0;
  bool any = false;
  while (hi.y - p.y >= rzg::kEps && floor(p.y) < H) {
    const double ys = fmin(floor(p.y) + 1.0, hi.y);
    const rzg::Pt q = rzg::mkpt(p.x + dxdy * (ys - p.y), ys);
    const bool f = fmin(p.x, q.x) < 0.0;
    if ((nr == 0 || f != rf[nr - 1]) && nr < rzg::kAeRuns) {
      rs[nr] = p;
      rf[nr] = f;
      ++nr;
    }
    any = any || f;
    p = q;
  }
  if (!any) return;
  const rzg::Pt e = p;  // where the walk ended
  auto sh = [](rzg::Pt v) { return rzg::mkpt(v.x + 1.0, v.y); };
  if (up) {
    bool st = false;
    for (int k = 0; k < nr; ++k) {
      if (rf[k] == st) continue;
      if (rf[k]) {
        to(rs[k]);
        to(sh(rs[k]));
      } else {
        to(sh(rs[k]));
        to(rs[k]);
      }
      st = rf[k];
    }
    if (st) {
      to(sh(e));
      to(e);
    }
  } else {
    bool st = false;
    if (rf[nr - 1]) {
      to(e);
      to(sh(e));
      st = true;
    }
    for (int k = nr - 1; k >= 0; --k) {
      const bool below = k > 0 ? rf[k - 1] : false;
      if (rf[k] == below) continue;
      if (rf[k]) {
        to(sh(rs[k]));
        to(rs[k]);
      } else {
        to(rs[k]);
        to(sh(rs[k]));
      }
      st = below;
    }
    (void)st;
  }
}


int main() {
  std::mt19937_64 rng(3);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  long some = 0;
  for (int it = 0; it < 400000; ++it) {
    const double H = 1.0 + std::floor(U(rng) * 300.0);
    auto near0 = [&]() {
      const double k = U(rng);
      const double tiny = (U(rng) - 0.3) * std::pow(10.0, -7.0 - 10.0 * U(rng));
      return k < 0.4 ? tiny : k < 0.6 ? 0.0 : k < 0.7 ? -1e-17 * U(rng) : 300.0 * U(rng);
    };
    rzg::Pt a = rzg::mkpt(near0(), (H + 60.0) * U(rng) - 30.0);
    rzg::Pt b = rzg::mkpt(near0(), (H + 60.0) * U(rng) - 30.0);
    if (U(rng) < 0.3) b.x = std::pow(10.0, 4.0 * U(rng) - 2.0);
    if (U(rng) < 0.2) a.y = std::floor(a.y);
    if (U(rng) < 0.2) b.y = std::floor(b.y);
    if (U(rng) < 0.1) b.y = a.y + 1e-3 * U(rng);
    if (U(rng) < 0.5) std::swap(a, b);
    std::vector<rzg::Pt> v, w;
    rzg::ae_piece(a, b, H, [&](rzg::Pt p) { v.push_back(p); });
    ae_piece_rows(a, b, H, [&](rzg::Pt p) { w.push_back(p); });
    if (v.size() != w.size() || (v.size() && std::memcmp(v.data(), w.data(), v.size() * sizeof(rzg::Pt)))) {
      std::printf("edge (%.17g, %.17g) -> (%.17g, %.17g), H %g: %zu and %zu vertices\n", a.x, a.y, b.x, b.y,
                  H, v.size(), w.size());
      return 1;
    }
    some += !v.empty();
  }
  std::printf("%ld edges with moved rows\n", some);
  return some > 20000 ? 0 : 1;
}
