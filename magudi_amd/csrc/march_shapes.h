// march_shapes.h -- the work-unit shapes of the 3-D marches that the autotuner tries, and how it
// picks one from their timings (host code without HIP).
#pragma once
#include <algorithm>
#include <vector>

namespace mgd {

// Rows of a march tile.
constexpr int kMarchRows = 16;

// Work units of a march over an nx x ny x nz grid: tiles of mtile x kMarchRows points, zc planes
// per unit.
inline int march_units(const int* n, int mtile, int zc) {
  return ((n[0] + mtile - 1) / mtile) * ((n[1] + kMarchRows - 1) / kMarchRows) *
         ((n[2] + zc - 1) / zc);
}

struct MarchShape {
  int tile, chunk;
};

// Tile widths of 16 and 32 points, unless one is fixed (opt_tile), with a fixed chunk
// (opt_chunk) as it is; else with chunks of 32, 64 and 128 planes, and shorter ones only where 32
// planes do not fill the GPU: their units spend most of their planes on the z windows' lead-in.
// Among those the one whose units just fill the GPU in one go (two work-groups of a 16-wide tile
// per CU, one of a 32-wide): forward and adjoint run of 64^3 8.1 ms at 8 planes, 5.8 at 4, 5.7 at
// 2; of 100^3 16.6 at 8, 14.5 at 10.  Chunks that leave half of the 256 CUs without a unit are not
// tried (64^3, forward step: 0.15 ms at 4 planes, 0.34 at 16, 0.62 at 32), but for the shortest.
inline std::vector<MarchShape> march_shapes(const int* n, int instances, int opt_tile,
                                            int opt_chunk) {
  std::vector<MarchShape> shapes;
  for (int tile : {16, 32}) {
    if (opt_tile != 0 && tile != opt_tile) continue;
    if (opt_chunk != 0) {
      shapes.push_back({tile, opt_chunk});
      continue;
    }
    const auto units = [&](int zc) { return (long)instances * march_units(n, tile, zc); };
    std::vector<int> chunks = {32, 64, 128};
    if (units(32) < 512) {
      const long columns = units(n[2]), room = tile == 32 ? 256 : 512;
      const int fill = columns <= room ? (int)((n[2] + room / columns - 1) / (room / columns)) : 0;
      chunks.push_back(8);
      chunks.push_back(16);
      if (units(8) < 256 || fill == 4) chunks.push_back(4);
      if (fill >= 2 && fill < 32 && fill != 4 && fill != 8 && fill != 16) chunks.push_back(fill);
    }
    const int least = *std::min_element(chunks.begin(), chunks.end());
    for (int chunk : chunks)
      if (chunk == least || units(chunk) >= 128) shapes.push_back({tile, chunk});
  }
  return shapes;
}

// The shapes of the least forward and the least adjoint time among n: sample(k, &f, &a) times
// shape k once and says whether it could.  Two rounds over every shape, since one sample in
// some is off by 10 % and more, then a third among those within a twentieth of the best (the
// samples of later rounds repeat within 1 %); the least sample of each counts.
template <class F>
bool pick_march_shapes(int n, F&& sample, int* forward, int* adjoint) {
  std::vector<float> f(n), a(n);
  for (int round = 0; round < 3; ++round) {
    const float fm = *std::min_element(f.begin(), f.end()), am = *std::min_element(a.begin(), a.end());
    for (int k = 0; k < n; ++k) {
      if (round == 2 && f[k] > 1.05f * fm && a[k] > 1.05f * am) continue;
      float fk = 0.f, ak = 0.f;
      if (!sample(k, &fk, &ak)) return false;
      f[k] = round == 0 ? fk : std::min(f[k], fk);
      a[k] = round == 0 ? ak : std::min(a[k], ak);
    }
  }
  *forward = (int)(std::min_element(f.begin(), f.end()) - f.begin());
  *adjoint = (int)(std::min_element(a.begin(), a.end()) - a.begin());
  return true;
}

}  // namespace mgd
