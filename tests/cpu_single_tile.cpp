// Host check of rzg::single_tile against the step-by-step decomposition
// (rzg::bin_piece) it stands for: where it answers, the piece must have
// exactly its record (bit for bit) and no band-bottom crossing. Lines start at
// random points, on tile and pixel edges and one rounding beside them, and run
// up to a few pixels, in every grid phase and edge mode. Prints the number of
// lines answered; exits 1 at the first difference.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>
#include "../rasterize_amd/csrc/rz_geom.hpp"

int main() {
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  auto coord = [&](double size) {
    double v = (size + 40.0) * U(rng) - 20.0;
    const double k = U(rng);
    if (k < 0.15) v = std::floor(v / 16.0) * 16.0;
    else if (k < 0.3) v = std::floor(v);
    if (U(rng) < 0.15) v = std::nextafter(v, U(rng) < 0.5 ? -1e9 : 1e9);
    return v;
  };
  long answered = 0, with_record = 0;
  for (int it = 0; it < 2000000; ++it) {
    rzg::BinGrid g;
    g.mode = it % 3;
    g.W = 1 + (int)(U(rng) * 100);
    g.H = 1 + (int)(U(rng) * 100);
    g.wc = g.mode == rzg::EDGE_MASK ? g.W - 1.0 : (double)g.W;
    g.phx = it % 4 ? (int)(U(rng) * 16) : 0;
    g.phy = it % 4 ? (int)(U(rng) * 16) : 0;
    g.tiles_x = (g.W + g.phx + 15) >> 4;
    g.tiles_y = (g.H + g.phy + 15) >> 4;
    // effective pieces have x in [0, wc]; with phases, tile edges sit at 16k - ph
    auto clampx = [&](double x) { return x < 0.0 ? 0.0 : (g.mode != rzg::EDGE_NONE && x > g.wc ? g.wc : x); };
    const double len = std::pow(10.0, 2.5 * U(rng) - 1.5);
    rzg::Pt a = rzg::mkpt(clampx(coord(g.W) - g.phx), coord(g.H) - g.phy), b;
    b.x = U(rng) < 0.1 ? a.x : clampx(a.x + len * (2 * U(rng) - 1));
    b.y = U(rng) < 0.1 ? a.y : a.y + len * (2 * U(rng) - 1);
    if (U(rng) < 0.1) b.x = clampx(coord(g.W));
    int tile;
    rzg::Rec r;
    if (!rzg::single_tile(a, b, g, &tile, &r)) continue;
    ++answered;
    std::vector<std::pair<int, rzg::Rec>> recs;
    int crossings = 0;
    rzg::bin_piece(a, b, g, [&](int t, rzg::Rec q) { recs.push_back({t, q}); },
                   [&](int, int, int) { ++crossings; });
    const bool same = crossings == 0 && (int)recs.size() == (tile >= 0 ? 1 : 0) &&
                      (tile < 0 || (recs[0].first == tile && std::memcmp(&recs[0].second, &r, sizeof(r)) == 0));
    if (!same) {
      std::printf("line (%.17g, %.17g) -> (%.17g, %.17g) W %d H %d ph %d %d mode %d: tile %d, %zu records, %d crossings\n",
                  a.x, a.y, b.x, b.y, g.W, g.H, g.phx, g.phy, g.mode, tile, recs.size(), crossings);
      return 1;
    }
    with_record += tile >= 0;
  }
  std::printf("%ld answered, %ld with a record\n", answered, with_record);
  return answered > 200000 && with_record > 100000 ? 0 : 1;
}
