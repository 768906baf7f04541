// The resident steps' messages (cpi::build_mail) on the host: every message
// is posted once and read by the block it is meant for, and a block that adds
// its own partial and the messages of a node in table order adds the same
// partials in the same order as the boundary-node kernel (compared bit for bit
// on random partials).  Exit status 0 = pass.
#include <cstdio>
#include <random>
#include <string>
#include <vector>

#include "../cppimpact_amd/csrc/internal.h"
#include "../include/cppimpact_hip.h"

using namespace cpi;

static bool check(const char *name, int nn, int ne, int npe, const std::vector<double> &x,
                  const std::vector<int32_t> &conn, int me, int mn) {
  BlockPlan P;
  std::string err;
  if (!build_block_plan(ne, npe, conn.data(), nn, x.data(), me, mn, P, err)) return false;
  const MailPlan M = build_mail(P);
  const int nb = P.nblocks, ml = P.max_local_nodes;
  const size_t total = M.dest.size();
  if ((int)M.first.size() != nb + 1 || M.first[nb] != (int)total) return false;
  std::mt19937 rng(3);
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  std::vector<double> part(P.n_slots), inbox(total), sum(P.n_boundary, 0.0);
  std::vector<int> hits(total, 0);
  for (double &v : part) v = u(rng);
  for (int i = 0; i < P.n_boundary; i++)
    for (int s = P.slot_ptr[i]; s < P.slot_ptr[i + 1]; s++) sum[i] += part[s];
  int most = 0;
  for (int b = 0; b < nb; b++) {
    most = std::max(most, M.first[b + 1] - M.first[b]);
    for (int m = M.first[b]; m < M.first[b + 1]; m++) {
      if (M.src[m] >= ml || M.dest[m] < 0 || M.dest[m] >= (int)total || hits[M.dest[m]]++)
        return false;
      const int s = P.slot_pad[(size_t)b * ml + M.src[m]];
      // a shared node's, and not to itself
      if (s < 0 || (M.dest[m] >= M.first[b] && M.dest[m] < M.first[b + 1])) return false;
      inbox[M.dest[m]] = part[s];
    }
  }
  if (most != M.most) return false;
  for (int b = 0; b < nb; b++) {
    int seen = 0;
    for (int l = 0; l < ml; l++) {
      const size_t i = (size_t)b * ml + l;
      if (P.nid_pad[i] < 0 || P.slot_pad[i] < 0) continue;
      const int node = P.nid_pad[i] - P.n_interior, s0 = P.slot_ptr[node];
      const int cnt = P.slot_ptr[node + 1] - s0 - 1, own = P.slot_pad[i] - s0;
      if (own < 0 || own > cnt || M.lo[i] != seen) return false;
      seen += cnt;
      if (M.first[b] + seen > M.first[b + 1]) return false;
      const uint16_t *idx = M.idx.data() + M.first[b] + M.lo[i];
      for (int k = 0; k < cnt; k++)
        if (idx[k] >= M.first[b + 1] - M.first[b]) return false;
      double f = 0.0;
      for (int k = 0; k < own; k++) f += inbox[M.first[b] + idx[k]];
      f += part[P.slot_pad[i]];
      for (int k = own; k < cnt; k++) f += inbox[M.first[b] + idx[k]];
      if (f != sum[node]) return false;
    }
    if (seen != M.first[b + 1] - M.first[b]) return false;
  }
  std::printf("ok %s: %d blocks, ml %d, %zu messages, most %d\n", name, nb, ml, total, M.most);
  return true;
}

static bool box(const char *name, int n0, int n1, int n2, int quadratic, int me, int mn) {
  cpi_box_spec sp{n0, n1, n2, quadratic, 1.0, 1.0, 1.0, {0, 0, 0}, 0.0, 0};
  int nn = 0, ne = 0;
  if (cpi_mesh_box(&sp, &nn, &ne, nullptr, nullptr)) return false;
  const int npe = quadratic ? 10 : 4;
  std::vector<double> x(3 * (size_t)nn);
  std::vector<int32_t> conn((size_t)npe * ne);
  if (cpi_mesh_box(&sp, &nn, &ne, x.data(), conn.data())) return false;
  return check(name, nn + 2, ne, npe, (x.resize(x.size() + 6, 0.5), x), conn, me, mn);
}

int main() {
  int bad = 0;
  bad += !box("one block", 4, 4, 4, 0, 384, 384);
  bad += !box("two blocks", 4, 4, 5, 0, 384, 384);
  bad += !box("tet4 cube", 10, 10, 10, 0, 384, 216);
  bad += !box("tet4 small blocks", 7, 5, 6, 0, 37, 64);
  bad += !box("tet10 box", 5, 4, 3, 1, 128, 512);
  bad += !box("tet10 small blocks", 4, 4, 4, 1, 17, 90);
  bad += !box("tet10 cube", 20, 20, 20, 1, 128, 512);
  if (bad) std::fprintf(stderr, "FAIL %d\n", bad);
  return bad != 0;
}
