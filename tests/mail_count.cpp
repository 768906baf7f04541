// The number of the resident steps' messages (cpi::count_mail) on the host: the
// tables' on a box in small blocks, and past what the tables' 32-bit words hold
// for a fan around one node that lies in every block.  Exit status 0 = pass.
#include <cstdio>
#include <string>
#include <vector>

#include "../cppimpact_amd/csrc/internal.h"
#include "../include/cppimpact_hip.h"

using namespace cpi;

static bool box(int n, int me) {
  cpi_box_spec sp{n, n, n, 0, 1.0, 1.0, 1.0, {0, 0, 0}, 0.0, 0};
  int nn = 0, ne = 0;
  if (cpi_mesh_box(&sp, &nn, &ne, nullptr, nullptr)) return false;
  std::vector<double> x(3 * (size_t)nn);
  std::vector<int32_t> conn(4 * (size_t)ne);
  if (cpi_mesh_box(&sp, &nn, &ne, x.data(), conn.data())) return false;
  x.resize(x.size() + 6, 0.5);  // two nodes of no element
  BlockPlan P;
  std::string err;
  if (!build_block_plan(ne, 4, conn.data(), nn + 2, x.data(), me, 384, P, err)) return false;
  const MailPlan M = build_mail(P);
  const MailCount N = count_mail(P);
  std::printf("box %d: %zu messages, most %zu\n", n, N.all, N.most);
  return N.all == M.dest.size() && N.most == (size_t)M.most;
}

// m blocks of three nodes: one that all share, and two of their own
static bool fan(int m) {
  BlockPlan P;
  P.nblocks = m;
  P.max_local_nodes = 3;
  P.n_interior = 2 * m;
  P.n_boundary = 1;
  P.n_slots = m;
  P.slot_ptr = {0, m};
  for (int b = 0; b < m; b++)
    for (int l = 0; l < 3; l++) {
      P.nid_pad.push_back(l == 0 ? 2 * m : 2 * b + l - 1);
      P.slot_pad.push_back(l == 0 ? b : -1);
    }
  const MailCount N = count_mail(P);
  std::printf("fan %d: %zu messages, most %zu\n", m, N.all, N.most);
  return N.all == (size_t)m * (m - 1) && N.most == (size_t)m - 1;
}

int main() {
  const bool ok = box(4, 384) && box(6, 37) && box(7, 1) && fan(300) && fan(70000);
  return ok ? 0 : 1;
}
