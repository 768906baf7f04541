// The colour scatter's corner-force slots (cpi::color_slots) on the host:
// every slot is written once, a node's slots belong to its own corners, and
// summing them in slot order adds the same forces in the same order as one
// read-modify-write pass per colour (compared bit for bit on random forces).
// Exit status 0 = pass.
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../cppimpact_amd/csrc/internal.h"
#include "../include/cppimpact_hip.h"

using namespace cpi;

static bool check(int n0, int n1, int n2, int quadratic, int extra, unsigned seed) {
  cpi_box_spec sp{n0, n1, n2, quadratic, 1.0, 1.0, 1.0, {0, 0, 0}, 0.0, 0};
  int nn = 0, ne = 0;
  if (cpi_mesh_box(&sp, &nn, &ne, nullptr, nullptr)) return false;
  const int npe = quadratic ? 10 : 4;
  std::vector<double> x(3 * (size_t)nn);
  std::vector<int32_t> conn((size_t)npe * ne);
  if (cpi_mesh_box(&sp, &nn, &ne, x.data(), conn.data())) return false;
  std::mt19937 rng(seed);
  for (int e = ne - 1; e > 0; e--) {  // any element order
    const int o = rng() % (e + 1);
    for (int k = 0; k < npe; k++) std::swap(conn[(size_t)npe * e + k], conn[(size_t)npe * o + k]);
  }
  nn += extra;  // nodes of no element
  std::vector<int32_t> color(ne), order;
  std::vector<uint32_t> slot, ptr;
  const int ncol = greedy_coloring(ne, npe, conn.data(), nn, color.data());
  color_slots(ne, npe, conn.data(), nn, color.data(), ncol, slot, ptr, order);
  if (ptr.size() != (size_t)nn + 1 || ptr[nn] != slot.size()) return false;
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  std::vector<double> f((size_t)npe * ne), buf(slot.size()), seq(nn, 0.0), sum(nn, 0.0);
  std::vector<int> hits(slot.size(), 0);
  for (int k = 0; k < npe; k++)
    for (int e = 0; e < ne; e++) {
      f[(size_t)k * ne + e] = u(rng);
      const uint32_t s = slot[(size_t)k * ne + e];
      const int n = conn[(size_t)npe * e + k];
      if (s < ptr[n] || s >= ptr[n + 1] || hits[s]++) return false;
      buf[s] = f[(size_t)k * ne + e];
    }
  for (int c = 0; c < ncol; c++)
    for (int e = 0; e < ne; e++)
      if (color[e] == c)
        for (int k = 0; k < npe; k++) seq[conn[(size_t)npe * e + k]] += f[(size_t)k * ne + e];
  for (int n = 0; n < nn; n++)
    for (uint32_t s = ptr[n]; s < ptr[n + 1]; s++) sum[n] += buf[s];
  if (sum != seq) return false;
  std::vector<int> seen(ne, 0);
  for (int e = 0; e < ne; e++) {
    if (order[e] < 0 || order[e] >= ne || seen[order[e]]++) return false;
    for (int d = 0; d < e; d++)
      if ((color[d] <= color[e]) != (order[d] < order[e])) return false;
  }
  return true;
}

int main() {
  int bad = 0;
  const int box[][3] = {{1, 1, 1}, {2, 1, 3}, {5, 4, 3}};
  for (int quadratic = 0; quadratic < 2; quadratic++)
    for (const auto &b : box)
      for (int extra = 0; extra < 3; extra += 2)
        if (!check(b[0], b[1], b[2], quadratic, extra, 7u + extra)) {
          std::fprintf(stderr, "FAIL %d %d %d quadratic %d extra %d\n", b[0], b[1], b[2], quadratic, extra);
          bad++;
        }
  if (!bad) std::printf("all slots hold\n");
  return bad != 0;
}
