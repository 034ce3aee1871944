// The list build's quantised test against the exact one: no pair that belongs
// in a list may fail it, over grids from one cell to a million a side, radii
// from a hundredth of a cell to ten and skins up to two cells.
#include <cmath>
#include <cstdio>
#include <random>

#include "list_quant.hpp"

using namespace gg;

int main() {
  std::mt19937_64 rng(7);
  auto uni = [&](double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); };
  long pairs = 0, large = 0, all = 0, lost = 0, passed = 0, far = 0;
  for (int t = 0; t < 3000000; ++t) {
    const int side = (int)std::exp(uni(0.0, std::log(1.1e6)));
    const float L = (float)std::exp(uni(std::log(1e-3), std::log(1e3)));
    const float per_unit = (float)kQuantUnits / L;
    const float skin = (float)(L * (t % 4 ? uni(0.0, 0.3) : uni(0.0, 2.0)));
    float4 i, j;
    i.w = (float)(L * std::exp(uni(std::log(0.01), std::log(10.0))));
    j.w = t % 3 ? (float)(i.w * uni(0.5, 2.0)) : (float)(L * std::exp(uni(std::log(0.01), std::log(10.0))));
    // one end anywhere the stencil can be, the other at about the limit
    const double reach = (double)i.w + j.w + skin;
    double d[3], n2 = 0.0;
    for (double &c : d) c = uni(-1.0, 1.0), n2 += c * c;
    const double r = t % 2 ? reach * uni(0.0, 1.0) : reach * uni(0.999, 1.001);
    const double x[3] = {uni(-1.0, 2.0), uni(-1.0, 2.0), uni(-1.0, side + 1.0)};
    float *pi = &i.x, *pj = &j.x;
    for (int k = 0; k < 3; ++k) {
      pi[k] = (float)(L * x[k]);
      pj[k] = (float)(L * x[k] + d[k] / std::sqrt(n2) * r);
    }
    const float px = i.x - j.x, py = i.y - j.y, pz = i.z - j.z;
    const float d2 = px * px + py * py + pz * pz;
    const float lim = (i.w + j.w) + skin;
    const QuantLimit q = quant_limit(i, skin, per_unit, quant_margin(side));
    const bool pass = q.all || quant_test(q, quantise(j, per_unit)) < 0;
    if (!(d2 < lim * lim)) {
      ++far;
      continue;
    }
    ++pairs;
    large += quant_large(j.w, per_unit);
    all += q.all;
    passed += pass;
    if (!pass && !quant_large(j.w, per_unit)) {
      if (++lost < 5)
        std::printf("lost: side %d L %g r %g %g skin %g distance %g\n", side, L, i.w, j.w, skin,
                    std::sqrt(d2));
    }
  }
  std::printf("pairs %ld (large %ld, all %ld, passed %ld), beyond %ld, lost %ld\n", pairs, large,
              all, passed, far, lost);
  return lost || pairs < 1000000 || large < 1000 || all < 1000 || all > pairs / 2 ? 1 : 0;
}
