// Context management and the C ABI (include/cppimpact_hip.h) of
// libcppimpact_hip.so: device buffers, uploads/downloads between the
// reference's host layouts and the device layout, the hipGraph-captured
// step, timing and diagnostics.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <system_error>
#include <thread>
#include <vector>

#include "../../include/cppimpact_hip.h"
#include "device.h"
#include "internal.h"
#include "kernels.h"
#include "mlp_host.h"

namespace cpi {
void set_global_error(const std::string &s);
const char *global_error();
}  // namespace cpi

using namespace cpi;

struct cpi_ctx {
  int dev = 0;
  hipStream_t stream = nullptr;
  std::string err;
  int nn = 0, ne = 0, npe = 0, nq = 0, rule = 0, phys = 0, prec = 0, scatter = 0, mass_kind = 0;
  cpi_options opt{};
  cpi_material mat{};
  cpi_wall wall{};
  std::vector<int32_t> conn_u, color, slave_u;
  int ncol = 0;
  std::vector<int32_t> eperm, nperm, ninv;  // device->user elem, device->user node, user->device
  std::vector<int32_t> color_off;           // the colours' elements in d_by_color
  int32_t *d_by_color = nullptr;            // (null: the colour scatter has its slots)
  std::vector<int32_t> loose;               // user nodes of no element
  int32_t *d_last = nullptr;                // per user node: last element holding it (device id)
  int32_t *d_ninv = nullptr;                // user node -> device id
  uint32_t *d_spos = nullptr;               // per user element: its state (k_export_elems)
  size_t state_points = 0;                  // points the state arrays hold
  Vec3 *d_V0 = nullptr;                     // initial velocities, device order
  BlockPlan plan;
  std::vector<void *> allocs;
  double *d_tmp = nullptr;
  size_t tmp_len = 0;
  // pinned host words results come back through, and one event per chunk of
  // a large context's ring
  double *pin = nullptr;
  std::vector<hipEvent_t> ring;
  Params P{};
  int nblocks = 0, n_elem_rows = 0, n_node_rows = 0, n_rows = 0;
  size_t smem = 0;
  // captured steps: one plain step, the energy/output step, and kGraphRuns[k]
  // plain steps in one graph each
  struct GraphSet {
    hipGraphExec_t plain = nullptr, aux = nullptr;
    hipGraphExec_t run[2] = {nullptr, nullptr};
  } gs;
  // resident steps (k_resident): the plan allows them, and none has given up or
  // failed since cpi_init
  Resident res{};
  size_t res_smem = 0;
  bool res_able = false, resident = false;
  int res_min = 0;  // fewest plain steps of a call (kMinResident)
  hipEvent_t res_done[2] = {nullptr, nullptr};  // of every kAhead-th launch of a call, in turn
  // launches whose outcome the host has not seen, and the step that each call
  // since the first of them ends at (kMaxCalls at most)
  bool res_pending = false;
  std::vector<int64_t> calls;
  int64_t redone = 0;        // steps taken one by one instead, since cpi_init
  bool mass_ready = false, inited = false;
  double dt = 0.0;
  int64_t step = 0;
  MlpHost mlp;  // surrogate weights and sample buffer
};

// one workgroup: the minimum of the element partials and the smallest
// positive nodal mass (the wall spring's limit needs it)
__global__ void __launch_bounds__(256) k_dt_finish(const double *part, int nb, const double *m,
                                                   int nn, double *out) {
  __shared__ double r0[256], r1[256];
  double a = 1e300, b = 1e300;
  for (int i = threadIdx.x; i < nb; i += 256) a = fmin(a, part[i]);
  for (int i = threadIdx.x; i < nn; i += 256)
    if (m[i] > 0.0) b = fmin(b, m[i]);
  r0[threadIdx.x] = a;
  r1[threadIdx.x] = b;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      r0[threadIdx.x] = fmin(r0[threadIdx.x], r0[threadIdx.x + h]);
      r1[threadIdx.x] = fmin(r1[threadIdx.x], r1[threadIdx.x + h]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = r0[0];
    out[1] = r1[0];
  }
}

namespace {

hipError_t launch_dt_finish(const double *part, int nb, const double *m, int nn, double *out,
                            hipStream_t s) {
  hipLaunchKernelGGL(k_dt_finish, dim3(1), dim3(256), 0, s, part, nb, m, nn, out);
  return hipGetLastError();
}

#define HIPCHK(ctx, expr)                                                                  \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess) {                                                               \
      (ctx)->err = std::string(#expr) + " failed at " __FILE__ ":" + std::to_string(__LINE__) + \
                   ": " + hipGetErrorString(e_);                                          \
      return CPI_ERR_HIP;                                                                 \
    }                                                                                     \
  } while (0)

int fail(cpi_ctx *c, int code, const std::string &msg) {
  c->err = msg;
  return code;
}

template <typename T>
int dalloc(cpi_ctx *c, T **p, size_t n) {
  void *q = nullptr;
  hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
  if (e != hipSuccess) {
    c->err = "hipMalloc of " + std::to_string(n * sizeof(T)) + " bytes failed: " +
             hipGetErrorString(e);
    return CPI_ERR_ALLOC;
  }
  c->allocs.push_back(q);
  *p = (T *)q;
  if (c->opt.debug_fill_nan && c->stream)
    HIPCHK(c, hipMemsetAsync(q, 0xFF, std::max<size_t>(n, 1) * sizeof(T), c->stream));
  return CPI_OK;
}

void dfree(cpi_ctx *c, void *p) {
  const auto i = std::find(c->allocs.begin(), c->allocs.end(), p);
  if (p == nullptr || i == c->allocs.end()) return;
  c->allocs.erase(i);
  (void)hipFree(p);
}

// energy rows of a k_elem_direct launch on n elements, one per wave
int elem_direct_rows(int npe, int n) {
  const int nt = elem_direct_threads(npe);
  return nt / 64 * ((n + nt - 1) / nt);
}

template <typename T>
int upload(cpi_ctx *c, T *d, const std::vector<T> &h) {
  if (h.empty()) return CPI_OK;
  // on the context's stream: kernels there do not wait for the null stream,
  // and a pageable host-to-device copy may return before its DMA lands
  HIPCHK(c, hipMemcpyAsync(d, h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CPI_OK;
}

// the assembled forces that element kernels add to (the other scatters sum
// records of their own: 24 bytes a node saved, and their clearing at init)
int alloc_forces(cpi_ctx *c) {
  int rc = CPI_OK;
  for (int k = 0; k < 3 && !rc; k++) rc = dalloc(c, &c->P.f[k], c->nn);
  return rc;
}

int default_rule(int npe, int phys, int q) {
  if (q >= 0) return q;
  if (phys == CPI_PHYSICS_COMPAT) return CPI_QUAD_REF5;
  return npe == 4 ? CPI_QUAD_CENTROID : CPI_QUAD_EXACT4;
}

double rule_weight_sum(int rule) {
  switch (rule) {
    case CPI_QUAD_REF5: return -0.13333333333 + 0.075 + 0.075 + 0.075 + 0.075;
    case CPI_QUAD_REF4: return 0.041666667 + 0.041666667 + 0.041666667 + 0.041666667;
    case CPI_QUAD_EXACT4: return 4.0 / 24.0;
    default: return 1.0 / 6.0;
  }
}

// pinned words of a context: results up to kSmall come back in one transfer;
// a context whose nodal state is larger holds a ring of 1 MiB chunks, at most
// kRing of them (see bring_back_ring)
constexpr size_t kSmall = 512u << 10;
constexpr size_t kRing = 32;
constexpr int kCopyThreads = 6;
constexpr size_t kStateWords = (sizeof(Ctl) + 7) / 8;  // ahead of the exported arrays

// Words of d_tmp.  Nodal results pass at once where the device has room, else in
// parts of kTmpLow (16 MiB).  For an element state, which may be a third of the
// device's memory, it grows to kTmpMost (128 MiB) at most: a part costs 0.1 ms
// for its launch and copy threads, of the 4.6 ms its transfer takes.
constexpr size_t kTmpLow = 2u << 20, kTmpMost = 16u << 20;

// What passes through d_tmp goes in as many parts as it takes: n items of
// words doubles each, beside head words.  The first item and the number of
// items of each part to f.
template <class F>
int in_parts(cpi_ctx *c, size_t n, size_t words, size_t head, const F &f) {
  const size_t part = words ? std::max<size_t>(1, (c->tmp_len - head) / words) : n;
  for (size_t i = 0; i < n; i += part)
    if (int rc = f(i, std::min(part, n - i))) return rc;
  return CPI_OK;
}

// user-order [N][3] on the host -> nodal records in device node order
int put_nodes(cpi_ctx *c, const double *aos, Vec3 *d3, Node4 *d4) {
  int rc = in_parts(c, c->nn, 3, 0, [&](size_t i, size_t n) -> int {
    HIPCHK(c, hipMemcpyAsync(c->d_tmp, aos + 3 * i, 24 * n, hipMemcpyHostToDevice, c->stream));
    HIPCHK(c, launch_import_nodes(c->d_tmp, c->d_ninv + i, (int)n, d3, d4, c->stream));
    return CPI_OK;
  });
  if (rc) return rc;
  HIPCHK(c, hipStreamSynchronize(c->stream));  // d_tmp and the caller's array are free again
  return CPI_OK;
}

// Results that lie one after the other in d_tmp, to the caller's arrays.
// Waits for the stream.
struct Piece {
  void *host;
  size_t words;
};

// bytes [at, at + n) of the pieces' concatenation, from src
void spread(const Piece *p, size_t at, size_t n, const char *src) {
  for (; n; p++) {
    const size_t len = 8 * p->words;
    if (at >= len) {
      at -= len;
      continue;
    }
    const size_t k = std::min(n, len - at);
    std::memcpy((char *)p->host + at, src, k);
    src += k;
    n -= k;
    at = 0;
  }
}

// Results too large for one transfer: the chunks go through the pinned ring
// while a few threads copy those that have arrived to the caller's pages,
// which are fresh as a rule.  One thread (the runtime's staged copy) is bound
// by its page faults: the 239 MB of the 1.87M-node cylinder took 26 ms, this
// takes 8.4 (88 ms when the host also permuted them).
// false: no thread could be started and nothing was moved.
constexpr size_t kChunk = 1u << 20;
bool bring_back_ring(cpi_ctx *c, const Piece *p, size_t bytes, int *rc) {
  const size_t chunks = (bytes + kChunk - 1) / kChunk, ring = c->ring.size();
  std::atomic<size_t> issued{0}, next{0};
  std::unique_ptr<std::atomic<bool>[]> copied(new (std::nothrow) std::atomic<bool>[chunks]);
  if (!copied) return false;
  for (size_t i = 0; i < chunks; i++) copied[i] = false;
  std::atomic<int> err{(int)hipSuccess};
  auto work = [&] {
    (void)hipSetDevice(c->dev);
    for (;;) {
      const size_t i = next.fetch_add(1);
      if (i >= chunks) return;
      while (issued.load(std::memory_order_acquire) <= i) {
        if (err.load()) return;
        std::this_thread::yield();
      }
      const hipError_t e = hipEventSynchronize(c->ring[i % ring]);
      if (e != hipSuccess) {
        err = (int)e;
        return;
      }
      const size_t at = i * kChunk;
      spread(p, at, std::min(kChunk, bytes - at), (const char *)c->pin + (i % ring) * kChunk);
      copied[i].store(true, std::memory_order_release);
    }
  };
  std::vector<std::thread> team;
  const size_t want = std::min<size_t>(kCopyThreads, chunks);
  try {
    team.reserve(want);
    while (team.size() < want) team.emplace_back(work);
  } catch (const std::system_error &) {
  } catch (const std::bad_alloc &) {
  }
  if (team.empty()) return false;
  for (size_t i = 0; i < chunks && !err.load(); i++) {
    while (i >= ring && !copied[i - ring].load(std::memory_order_acquire) && !err.load())
      std::this_thread::yield();
    const size_t at = i * kChunk;
    hipError_t e = hipMemcpyAsync((char *)c->pin + (i % ring) * kChunk, (const char *)c->d_tmp + at,
                                  std::min(kChunk, bytes - at), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipEventRecord(c->ring[i % ring], c->stream);
    if (e != hipSuccess)
      err = (int)e;
    else
      issued.store(i + 1, std::memory_order_release);
  }
  for (auto &t : team) t.join();
  const hipError_t e = (hipError_t)err.load(), f = hipStreamSynchronize(c->stream);
  *rc = CPI_OK;
  if (e != hipSuccess || f != hipSuccess)
    *rc = fail(c, CPI_ERR_HIP, std::string("download: ") + hipGetErrorString(e != hipSuccess ? e : f));
  return true;
}

int bring_back(cpi_ctx *c, const Piece *p, int n) {
  size_t bytes = 0;
  for (int i = 0; i < n; i++) bytes += 8 * p[i].words;
  if (bytes <= kSmall) {
    HIPCHK(c, hipMemcpyAsync(c->pin, c->d_tmp, bytes, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    spread(p, 0, bytes, (const char *)c->pin);
    return CPI_OK;
  }
  int rc;
  if (!c->ring.empty() && bring_back_ring(c, p, bytes, &rc)) return rc;
  const double *src = c->d_tmp;
  for (int i = 0; i < n; src += p[i].words, i++)
    HIPCHK(c, hipMemcpyAsync(p[i].host, src, 8 * p[i].words, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CPI_OK;
}

// the control block
int get_ctl(cpi_ctx *c, Ctl *h) {
  HIPCHK(c, hipMemcpyAsync(c->pin, c->P.ctl, sizeof(Ctl), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  std::memcpy(h, c->pin, sizeof(Ctl));
  return CPI_OK;
}

bool all_finite(const double *v, size_t n) {
  double s[4] = {0.0, 0.0, 0.0, 0.0};  // v * 0 is NaN for an infinity or NaN
  size_t i = 0;
  for (; i + 4 <= n; i += 4)
    for (int k = 0; k < 4; k++) s[k] += v[i + k] * 0.0;
  for (; i < n; i++) s[0] += v[i] * 0.0;
  return s[0] + s[1] + s[2] + s[3] == 0.0;
}

// The element pass of the colour and atomic scatters: one launch, or, when the
// colour scatter's slots found no room, one per colour.
hipError_t elem_direct(cpi_ctx *c, Params p, int64_t *launches) {
  const int32_t *list = c->d_by_color;
  hipError_t e = hipSuccess;
  p.epart_base = 0;
  for (int k = 0; e == hipSuccess && k < (list ? c->ncol : 1); k++) {
    const int first = list ? c->color_off[k] : 0, n = (list ? c->color_off[k + 1] : c->ne) - first;
    e = launch_elem_direct(p, c->rule, c->prec, c->phys, list || c->scatter == CPI_SCATTER_ATOMIC,
                           list ? list + first : nullptr, n, c->stream);
    p.epart_base += elem_direct_rows(c->npe, n);
    if (launches) ++*launches;
  }
  return e;
}

int enqueue_step(cpi_ctx *c, bool aux) {
  Params p = c->P;
  p.store_aux = aux ? 1 : 0;
  hipError_t e = hipSuccess;
  if (c->scatter == CPI_SCATTER_BLOCK) {
    p.epart_base = 0;
    e = launch_elem_block(p, c->rule, c->prec, c->phys, aux, c->nblocks, c->smem, c->stream);
    if (e == hipSuccess) {
      p.epart_base = c->n_elem_rows;
      e = launch_node_bnd(p, c->prec, aux, c->stream);
    }
  } else {
    e = elem_direct(c, p, nullptr);
    if (e == hipSuccess) {
      p.epart_base = c->n_elem_rows;
      e = launch_node_all(p, c->prec, aux, c->stream);
    }
  }
  if (e == hipSuccess && aux) e = launch_energy_reduce(p, c->stream);
  if (e != hipSuccess) return fail(c, CPI_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(e));
  return CPI_OK;
}

// plain steps captured back to back in GraphSet::run: one graph launch, and
// no gap for the launch between the steps' kernels, per kGraphRuns[k]
// steps (measured at c2: ≈ 4 µs less per step than one graph per step)
constexpr int kGraphRuns[2] = {32, 4};

// Fewest plain steps of a call that go through the resident kernel: its launch
// and first loads cost as much as some steps.  With up to a block per CU calls
// of 5 steps take as long either way (energies read after each: 72-93 us, one
// launch per kernel 75-89), of 6 steps 4-12% less in the resident kernel.  With
// more blocks a call of 5 or 6 takes longer in it (196,608 tet4, FP32: 101 us
// against 87, 110 against 103; 48,000 tet10: 128 against 114, 139 against 135),
// one of 7 less (117 against 118; 148 against 155).
constexpr int kMinResident = 4, kMinResidentMany = 6;

// Most steps of one resident launch.  A longer call takes several: between them
// the chip is free for other streams' kernels (another context's ten steps, one
// launch per kernel, took 440 ms beside a call of 60,000 in one launch, 29 to 40
// ms so; its own resident launches wait for those queued before them, as
// cooperative launches do), and one that gives up loses the steps of one launch
// only.  A further launch takes 25 to 40 us: calls of 3,000 steps took 3-4%
// longer in launches of 128 steps, 1-2% in 256, 0.5% in 512, and in 1,024 no
// longer than in one.  At most 2 kAhead launches are queued, where a call of
// millions of steps would queue thousands.
constexpr int64_t kMaxResident = 1024;
constexpr int kAhead = 64;

// Polls after which a wait of a resident launch gives up: 24 ms (the last blocks
// may have to wait for another stream's kernels).  Some waits never end: 512
// blocks, two on every CU, that were launched while another context's step ran
// did not all get to run (some CU's room for the second is not the room it has
// when it starts empty).  The context's steps are then launched one by one until
// the next cpi_init.
constexpr unsigned kSpinLimit = 1u << 17;

// most calls queued on resident launches of unknown outcome (cpi_ctx::calls)
constexpr size_t kMaxCalls = 1024;

int capture(cpi_ctx *c, bool aux, hipGraphExec_t *out, int nrep = 1) {
  hipGraph_t g = nullptr;
  HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  int rc = CPI_OK;
  for (int i = 0; i < nrep && rc == CPI_OK; i++) rc = enqueue_step(c, aux);
  hipError_t e = hipStreamEndCapture(c->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (e != hipSuccess) return fail(c, CPI_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(e));
  e = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e != hipSuccess) return fail(c, CPI_ERR_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
  return CPI_OK;
}

void drop_graphs(cpi_ctx *c) {
  auto &G = c->gs;
  for (hipGraphExec_t *g : {&G.plain, &G.aux, &G.run[0], &G.run[1]}) {
    if (*g) (void)hipGraphExecDestroy(*g);
    *g = nullptr;
  }
}

// the step graphs (see cpi_ctx::gs)
int capture_graphs(cpi_ctx *c) {
  auto &G = c->gs;
  int rc;
  if ((rc = capture(c, false, &G.plain)) || (rc = capture(c, true, &G.aux)) ||
      (rc = capture(c, false, &G.run[0], kGraphRuns[0])) ||
      (rc = capture(c, false, &G.run[1], kGraphRuns[1])))
    return rc;
  return CPI_OK;
}

// d_tmp of n words at least, on the context's device whichever is current.  On
// failure it is what it was.
int ensure_tmp(cpi_ctx *c, size_t n) {
  if (c->tmp_len >= n) return CPI_OK;
  int cur = 0;
  HIPCHK(c, hipGetDevice(&cur));
  if (cur != c->dev) HIPCHK(c, hipSetDevice(c->dev));
  double *p = nullptr;
  int rc = dalloc(c, &p, n);
  if (rc) (void)hipGetLastError();  // not to be taken for a launch's
  if (cur != c->dev) HIPCHK(c, hipSetDevice(cur));
  if (rc) return rc;
  if (c->d_tmp) {
    HIPCHK(c, hipStreamSynchronize(c->stream));
    dfree(c, c->d_tmp);
  }
  c->d_tmp = p;
  c->tmp_len = n;
  return CPI_OK;
}

int compute_mass(cpi_ctx *c) {
  Params p = c->P;
  HIPCHK(c, hipMemsetAsync((void *)p.m, 0, sizeof(double) * c->nn, c->stream));
  const double rho = c->mat.rho;
  hipError_t e = hipSuccess;
  // CPI_SCATTER_* in launch_mass's numbering; colour by colour as elem_direct
  const int32_t *list = c->d_by_color;
  for (int k = 0; e == hipSuccess && k < (list ? c->ncol : 1); k++) {
    const int first = list ? c->color_off[k] : 0, n = (list ? c->color_off[k + 1] : c->ne) - first;
    e = launch_mass(p, c->rule, list ? CPI_SCATTER_ATOMIC : c->scatter, c->mass_kind, rho, c->nblocks,
                    list ? list + first : nullptr, n, c->stream);
  }
  if (e != hipSuccess) return fail(c, CPI_ERR_HIP, std::string("mass kernel: ") + hipGetErrorString(e));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->mass_ready = true;
  return CPI_OK;
}

// x = X0, v = v0, forces/aux/state zeroed (the mass, once assembled, stays)
int reset_state(cpi_ctx *c) {
  HIPCHK(c, launch_reset_nodes(c->P, c->d_V0, c->stream));
  const size_t rs = c->prec == CPI_PREC_F32 ? 4 : 8;
  if (c->phys != CPI_PHYSICS_COMPAT) {
    HIPCHK(c, hipMemsetAsync(c->P.sig, 0, rs * 6 * c->state_points, c->stream));
    HIPCHK(c, hipMemsetAsync(c->P.epbar, 0, rs * c->state_points, c->stream));
    if (c->P.yielded)
      HIPCHK(c, hipMemsetAsync(c->P.yielded, 0, 8 * (size_t)c->P.ywords * c->nblocks, c->stream));
    if (c->P.mlp_ctr) HIPCHK(c, hipMemsetAsync(c->P.mlp_ctr, 0, sizeof(unsigned long long), c->stream));
  }
  HIPCHK(c, hipMemsetAsync(c->P.epart, 0, sizeof(double) * EP_N * c->n_rows, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return CPI_OK;
}

// stable dt of the current device positions: element limit and the wall
// spring limit 2 sqrt(m_min / k)
constexpr int kMassMinBlocks = 256;
int stable_dt(cpi_ctx *c, double *dte, double *dtc) {
  const int nb = (c->ne + 255) / 256;
  int rc = ensure_tmp(c, (size_t)nb + kMassMinBlocks + 2);
  if (rc) return rc;
  double *mm = c->d_tmp + nb, *out = mm + kMassMinBlocks;
  HIPCHK(c, launch_elem_dt(c->P, c->d_tmp, c->stream));
  HIPCHK(c, launch_mass_min(c->P, mm, kMassMinBlocks, c->stream));
  HIPCHK(c, launch_dt_finish(c->d_tmp, nb, mm, kMassMinBlocks, out, c->stream));
  HIPCHK(c, hipMemcpyAsync(c->pin, out, 2 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  *dte = c->pin[0];
  *dtc = (c->wall.enabled && c->wall.stiffness > 0.0)
             ? 2.0 * std::sqrt(c->pin[1] / c->wall.stiffness)
             : INFINITY;
  return CPI_OK;
}

int report_flags(cpi_ctx *c, const Ctl &h) {
  if (h.flags & 2u) return fail(c, CPI_ERR_NUMERIC, "inverted or degenerate element (detJ <= 0) during the step");
  if (h.flags & 1u) return fail(c, CPI_ERR_NUMERIC, "non-finite value in the energy terms (NaN/Inf state)");
  if (h.flags & 4u)
    return fail(c, CPI_ERR_NUMERIC,
                "time step " + std::to_string(h.dt) + " above the stable limit " +
                    std::to_string(std::min(h.row[7], h.dt_contact)) +
                    " of the configuration (element CFL / wall spring)");
  return CPI_OK;
}

int steps_one_by_one(cpi_ctx *c, int64_t nsteps);

// The outcome of the resident launches is known (h).  The first launch to give up
// left out every step queued behind it; they are taken now, one launch per
// kernel of a step and call by call, so that each call's energies are those of
// its own last step.  Until that has succeeded the launches stay pending, and
// the next read tries again.
int settle(cpi_ctx *c, const Ctl &h, bool *missing) {
  int64_t done = h.step;
  *missing = done < c->step;
  if (h.decision & 1u) {
    c->resident = false;
    HIPCHK(c, hipMemsetAsync(&c->P.ctl->decision, 0, sizeof(uint32_t), c->stream));
  }
  for (const int64_t end : c->calls) {
    if (end <= done) continue;
    int rc = steps_one_by_one(c, end - done);
    if (rc) return rc;
    c->redone += end - done;
    done = end;
  }
  c->res_pending = false;
  c->calls.clear();
  return CPI_OK;
}

// the control block after all steps asked for
int settled_ctl(cpi_ctx *c, Ctl *h) {
  int rc = get_ctl(c, h);
  if (rc || !c->res_pending) return rc;
  bool missing;
  rc = settle(c, *h, &missing);
  return rc || !missing ? rc : get_ctl(c, h);
}

// before results are read by other ways than the control block
int settled(cpi_ctx *c) {
  Ctl h;
  return c->res_pending ? settled_ctl(c, &h) : CPI_OK;
}

int check_flags(cpi_ctx *c) {
  Ctl h;
  int rc = settled_ctl(c, &h);
  return rc ? rc : report_flags(c, h);
}

}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------

extern "C" void cpi_default_options(cpi_options *o) {
  if (!o) return;
  std::memset(o, 0, sizeof(*o));
  o->physics = CPI_PHYSICS_COMPAT;
  o->precision = CPI_PREC_F64;
  o->scatter = CPI_SCATTER_BLOCK;
  o->quadrature = CPI_QUAD_DEFAULT;
  o->mass = CPI_MASS_DEFAULT;
  o->stress_update = CPI_RETURN_EXACT;
  o->use_graph = 1;
  o->track_energy = 1;
  o->contact_slave_only = 0;
  o->fixed_bc = 0;
  o->debug_fill_nan = 0;
  o->stream_state = 0;
  o->block_elements = 0;
  o->device = 0;
  o->gravity[0] = 0.0;
  o->gravity[1] = 0.0;
  o->gravity[2] = -9.81;
  o->mlp_tolerance = 1e-3;
}

extern "C" const char *cpi_last_error(const cpi_ctx *c) {
  return c ? c->err.c_str() : cpi::global_error();
}

extern "C" void cpi_destroy(cpi_ctx *c) {
  if (!c) return;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  drop_graphs(c);
  for (void *p : c->allocs) (void)hipFree(p);
  if (c->pin) (void)hipHostFree(c->pin);
  for (hipEvent_t e : c->ring)
    if (e) (void)hipEventDestroy(e);
  for (hipEvent_t e : c->res_done)
    if (e) (void)hipEventDestroy(e);
  mlp_free(c->mlp);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

// The block kernels that read each corner as a 16-bit word, l | k << 9
// (local node, its contribution rank): the per-point tet10 kernel always,
// the tet4 kernels when the plan's blocks fit the words.
static bool corner_words(const cpi_ctx *c) {
  return c->scatter == CPI_SCATTER_BLOCK &&
         ((c->npe == 10 && c->nq == 4) || (c->npe == 4 && c->plan.corner_fits()));
}

static int create_impl(cpi_ctx *c, const cpi_mesh_desc *m, const cpi_material *mat,
                       const cpi_wall *wall, const cpi_options *opt) {
  c->opt = *opt;
  c->mat = *mat;
  if (wall) c->wall = *wall;
  c->nn = m->num_nodes;
  c->ne = m->num_elements;
  c->npe = m->nodes_per_element;
  const int npe = c->npe;
  if (c->nn <= 0 || c->ne <= 0 || (npe != 4 && npe != 10) || !m->xloc || !m->element_nodes)
    return fail(c, CPI_ERR_INVALID, "cpi_create: empty mesh or nodes_per_element not 4/10");
  if (opt->physics < 0 || opt->physics > 1 || opt->precision < 0 || opt->precision > 1 ||
      opt->scatter < 0 || opt->scatter > 2 || opt->stress_update < 0 || opt->stress_update > 1 ||
      opt->stream_state < 0 || opt->stream_state > 2)
    return fail(c, CPI_ERR_INVALID, "cpi_create: option out of range");
  if (!(mat->E > 0) || !(mat->rho > 0) || !(mat->nu > -1.0 && mat->nu < 0.5))
    return fail(c, CPI_ERR_INVALID, "cpi_create: material needs E > 0, rho > 0, -1 < nu < 0.5");
  if (wall && wall->enabled && (wall->dim < 0 || wall->dim > 2 || (wall->normal != 1 && wall->normal != -1)))
    return fail(c, CPI_ERR_INVALID, "cpi_create: wall dim must be 0..2 and normal +-1");
  c->phys = opt->physics;
  if (c->phys == CPI_PHYSICS_EP && opt->stress_update == CPI_RETURN_MLP) {
    if (npe != 4 || opt->precision != CPI_PREC_F32 || opt->scatter != CPI_SCATTER_BLOCK)
      return fail(c, CPI_ERR_INVALID, "the MLP surrogate runs on tet4, FP32, block scatter");
    c->phys = 2;
  }
  c->prec = opt->precision;
  c->scatter = opt->scatter;
  c->rule = default_rule(npe, opt->physics, opt->quadrature);
  if (c->rule < 0 || c->rule > 3) return fail(c, CPI_ERR_INVALID, "cpi_create: bad quadrature");
  if (npe == 10 && c->rule == CPI_QUAD_CENTROID)
    return fail(c, CPI_ERR_INVALID, "tet10 needs a 4- or 5-point rule");
  c->mass_kind = opt->mass >= 0 ? opt->mass
                                 : (opt->physics == CPI_PHYSICS_COMPAT ? CPI_MASS_ROWSUM : CPI_MASS_HRZ);
  c->nq = (npe == 4) ? 1 : (c->rule == CPI_QUAD_REF5 ? 5 : 4);
  // host copies and validation
  c->conn_u.assign(m->element_nodes, m->element_nodes + (long)npe * c->ne);
  for (int32_t v : c->conn_u)
    if (v < 0 || v >= c->nn) return fail(c, CPI_ERR_MESH, "element_nodes references a node out of range");
  const double *X0u = m->xloc;
  if (!all_finite(X0u, 3 * (size_t)c->nn)) return fail(c, CPI_ERR_MESH, "non-finite node coordinate");
  for (int e = 0; e < c->ne; e++) {
    const int32_t *ce = &c->conn_u[(long)npe * e];
    const int o = npe == 4 ? 0 : 2, i1 = npe == 4 ? 1 : 0, i2 = npe == 4 ? 2 : 1;
    double a[3], b[3], d[3];
    for (int k = 0; k < 3; k++) {
      a[k] = X0u[3L * ce[i1] + k] - X0u[3L * ce[o] + k];
      b[k] = X0u[3L * ce[i2] + k] - X0u[3L * ce[o] + k];
      d[k] = X0u[3L * ce[3] + k] - X0u[3L * ce[o] + k];
    }
    double v6 = a[0] * (b[1] * d[2] - b[2] * d[1]) - a[1] * (b[0] * d[2] - b[2] * d[0]) +
                a[2] * (b[0] * d[1] - b[1] * d[0]);
    if (!(v6 > 0.0))
      return fail(c, CPI_ERR_MESH, "element " + std::to_string(e) + " is inverted or degenerate");
  }
  // colouring (always: reported by cpi_get_coloring)
  c->color.assign(c->ne, 0);
  c->ncol = greedy_coloring(c->ne, npe, c->conn_u.data(), c->nn, c->color.data());
  // device
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= opt->device || opt->device < 0)
    return fail(c, CPI_ERR_NO_DEVICE, "no HIP device " + std::to_string(opt->device));
  HIPCHK(c, hipSetDevice(opt->device));
  hipDeviceProp_t prop;
  HIPCHK(c, hipGetDeviceProperties(&prop, opt->device));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(c, CPI_ERR_NO_DEVICE, std::string("device is ") + prop.gcnArchName +
                                          ", this library is built for gfx950 only");
  c->dev = opt->device;
  const int cus = prop.multiProcessorCount;
  HIPCHK(c, hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  {
    const size_t all = 8 * (kStateWords + 16 * (size_t)c->nn);
    size_t pinned = kSmall;
    if (all > kSmall && !(opt->debug_fill_nan & 4)) {
      c->ring.resize(std::min(kRing, (all + kChunk - 1) / kChunk), nullptr);
      pinned = std::max(pinned, c->ring.size() * kChunk);
      for (hipEvent_t &e : c->ring) HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    if (hipHostMalloc((void **)&c->pin, pinned, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      for (hipEvent_t e : c->ring) (void)hipEventDestroy(e);
      c->ring.clear();
      HIPCHK(c, hipHostMalloc((void **)&c->pin, kSmall, hipHostMallocDefault));
    }
  }
  // device orders
  if (c->scatter == CPI_SCATTER_BLOCK) {
    const int nt = elem_block_threads(npe, c->rule, c->prec, c->phys, 0, cus);
    const int dflt = elem_block_default_elements(npe);
    int me = opt->block_elements > 0 ? opt->block_elements : dflt;
    // the tet4 kernel gives each thread one element and at most one node,
    // the tet10 kernel of the 4-point rules each thread one point
    if (npe == 4 && me > nt)
      return fail(c, CPI_ERR_INVALID, "block_elements above " + std::to_string(nt) + " for tet4");
    if (npe == 10 && c->nq == 4 && 4 * me > nt)
      return fail(c, CPI_ERR_INVALID, "block_elements above " + std::to_string(nt / 4) +
                                          " for tet10 on a 4-point rule");
    // LDS budget per workgroup: three (FP64) or four (FP32) tet4 workgroups,
    // two tet10 ones per 160 KiB CU, never above the device's limit; node
    // records take 56 bytes each (slot offsets budgeted for 64 contributions
    // per node)
    const long share = npe == 4 ? (c->prec == CPI_PREC_F32 ? 40960 : 54272) : 81920;
    const long budget = std::min<long>((long)prop.sharedMemPerBlock, share);
    const long fixed = (long)elem_block_smem(npe, c->rule, c->prec, 0, me, 64);
    long mnl = (budget - fixed - 16) / 56;
    if (mnl < 4L * npe)
      return fail(c, CPI_ERR_INVALID, "block_elements " + std::to_string(me) +
                                          " does not fit the LDS budget");
    // the tet4 and the per-point tet10 kernels give each thread at most one
    // node; the five-point tet10 kernel loops over its nodes
    int mn = (int)std::min<long>(mnl, (npe == 4 || c->nq == 4) ? nt : 1024);
    std::string e;
    if (!build_block_plan(c->ne, npe, c->conn_u.data(), c->nn, X0u, me, mn, c->plan, e))
      return fail(c, CPI_ERR_INVALID, "partition: " + e);
    if (c->plan.max_local_nodes > mn)
      return fail(c, CPI_ERR_INVALID, "partition: a block holds more nodes than its kernel");
    // the per-point tet10 kernel reads each corner as a 16-bit word (local
    // node < 512, contribution rank < 128), which its limits of 128
    // elements and 512 nodes per block guarantee
    if (npe == 10 && c->nq == 4 && !c->plan.corner_fits())
      return fail(c, CPI_ERR_INVALID, "partition: a tet10 block exceeds its corner words");
    c->eperm = c->plan.elem_perm;
    c->nperm = c->plan.node_perm;
    c->ninv = c->plan.node_inv;
    c->nblocks = c->plan.nblocks;
  } else {
    c->nperm.resize(c->nn);
    c->ninv.resize(c->nn);
    for (int i = 0; i < c->nn; i++) c->nperm[i] = c->ninv[i] = i;
    c->eperm.resize(c->ne);
    for (int e = 0; e < c->ne; e++) c->eperm[e] = e;
  }
  Params &P = c->P;
  P.nn = c->nn;
  P.ne = c->ne;
  P.npe = npe;
  P.nq = c->nq;
  const double E = mat->E, nu = mat->nu;
  const double k = E / ((1 + nu) * (1 - 2 * nu));
  P.c11 = (1 - nu) * k;
  P.c12 = nu * k;
  P.c44 = ((1 - 2 * nu) / 2) * k;
  P.mu = E / (2.0 * (1.0 + nu));
  P.sy0 = mat->Y0;
  P.H = mat->H;
  P.wave_speed = std::sqrt(P.c11 / mat->rho);
  P.wall_on = (wall && wall->enabled) ? 1 : 0;
  P.wall_dim = wall ? wall->dim : 2;
  P.wall_normal = wall ? wall->normal : 1;
  P.wall_loc = wall ? wall->location : 0.0;
  P.wall_k = wall ? wall->stiffness : 0.0;
  P.wall_nk = wall ? wall->normal * wall->stiffness : 0.0;
  for (int i = 0; i < 3; i++) P.grav[i] = opt->gravity[i];
  P.wsum = rule_weight_sum(c->rule);
  int rc = CPI_OK;
  const int nn = c->nn, ne = c->ne;
  if (c->scatter == CPI_SCATTER_ATOMIC) rc = alloc_forces(c);
  if (!rc) rc = dalloc(c, &P.pos, nn);
  if (!rc) rc = dalloc(c, &P.vv, nn);
  if (!rc) rc = dalloc(c, &P.acc, nn);
  if (!rc) rc = dalloc(c, &P.du, nn);
  if (!rc) rc = dalloc(c, &P.xprev, nn);
  if (!rc) rc = dalloc(c, &P.X0, nn);
  double *dm = nullptr;
  if (!rc) rc = dalloc(c, &dm, nn);
  P.m = dm;
  if (rc) return rc;
  // connectivity [npe][ne] in device element and node order
  {
    std::vector<int32_t> cd((size_t)npe * ne);
    for (int e = 0; e < ne; e++)
      for (int j = 0; j < npe; j++)
        cd[(size_t)j * ne + e] = c->ninv[c->conn_u[(size_t)npe * c->eperm[e] + j]];
    int32_t *d = nullptr;
    if ((rc = dalloc(c, &d, cd.size())) || (rc = upload(c, d, cd))) return rc;
    P.conn = d;
  }
  // the element whose strain and stress a node reports
  {
    std::vector<int32_t> einv(ne), last(nn, -1);
    for (int e = 0; e < ne; e++) einv[c->eperm[e]] = e;
    for (int e = 0; e < ne; e++)
      for (int j = 0; j < npe; j++) last[c->conn_u[(size_t)npe * e + j]] = einv[e];
    for (int i = 0; i < nn; i++)
      if (last[i] < 0) c->loose.push_back(i);
    if ((rc = dalloc(c, &c->d_last, last.size())) || (rc = upload(c, c->d_last, last)) ||
        (rc = dalloc(c, &c->d_ninv, c->ninv.size())) || (rc = upload(c, c->d_ninv, c->ninv)) ||
        (rc = dalloc(c, &c->d_V0, nn)))
      return rc;
    HIPCHK(c, hipMemsetAsync(c->d_V0, 0, sizeof(Vec3) * nn, c->stream));
  }
  // per-node flags in device node order from a list of user node ids
  auto node_mask = [&](int n, const int32_t *ids, const char *what, const uint8_t **out) {
    std::vector<uint8_t> mask(nn, 0);
    for (int i = 0; i < n; i++) {
      const int s = ids ? ids[i] : -1;
      if (s < 0 || s >= nn) return fail(c, CPI_ERR_MESH, std::string(what) + " node out of range");
      mask[c->ninv[s]] = 1;
    }
    uint8_t *d = nullptr;
    int r = dalloc(c, &d, mask.size());
    if (!r) r = upload(c, d, mask);
    if (!r) *out = d;
    return r;
  };
  if (opt->contact_slave_only &&
      (rc = node_mask(m->num_slave_nodes, m->slave_nodes, "slave", &P.contact_mask)))
    return rc;
  if (opt->fixed_bc && (rc = node_mask(m->num_fixed_nodes, m->fixed_nodes, "fixed", &P.fixed_mask)))
    return rc;
  if (c->phys != CPI_PHYSICS_COMPAT) {
    const size_t rs = c->prec == CPI_PREC_F32 ? 4 : 8;
    char *s = nullptr, *q = nullptr;
    std::vector<uint32_t> spos(ne);
    c->state_points = c->nq * (size_t)ne;
    if (c->scatter == CPI_SCATTER_BLOCK) {
      // rows of a multiple of 64 points (five-point rule: 80); of a block
      // smaller than that, its points to the next power of two (times five),
      // so a row is never twice its block
      const BlockPlan &B = c->plan;
      int row = c->nq;
      while (row < 64 && row < c->nq * B.max_block_elems) row *= 2;
      P.state_ld = (c->nq * B.max_block_elems + row - 1) / row * row;
      c->state_points = (size_t)B.nblocks * P.state_ld;
      if (c->state_points / c->nq > UINT32_MAX)
        return fail(c, CPI_ERR_INVALID, "the stress state's rows pass 2^32 elements");
      for (int b = 0; b < B.nblocks; b++)
        for (int k = 0; k < B.meta[8 * (size_t)b + 1]; k++)
          spos[c->eperm[B.meta[8 * (size_t)b] + k]] = (uint32_t)((size_t)b * (P.state_ld / c->nq) + k);
    } else {
      for (int e = 0; e < ne; e++) spos[c->eperm[e]] = (uint32_t)e;
    }
    if ((rc = dalloc(c, &s, rs * 6 * c->state_points)) || (rc = dalloc(c, &q, rs * c->state_points)) ||
        (rc = dalloc(c, &c->d_spos, spos.size())) || (rc = upload(c, c->d_spos, spos)))
      return rc;
    P.sig = s;
    P.epbar = q;
    // when a step's working set (state, node records, partial forces,
    // connectivity) exceeds 192 MB, three quarters of the 256 MB Infinity
    // Cache, the block kernels stream the state past the caches, which then
    // keep the node records and partials that other blocks and the node
    // pass read again: the c3 cylinder (285 MB in FP32, 440 MB in FP64) and
    // the 128^3 tet4 cube (0.6-1 GB) step 4-6% faster; the c2 cube (89 and
    // 138 MB) stays cached, which streaming would make 6-9% slower
    const size_t slots = c->scatter == CPI_SCATTER_BLOCK ? (size_t)c->plan.n_slots : 0;
    const size_t conn = corner_words(c) ? 2 * (size_t)npe : 4 * (size_t)npe;
    const size_t ws = rs * 7 * c->nq * (size_t)ne + 56 * (size_t)c->nn +
                      slots * (c->prec == CPI_PREC_F32 ? 12 : 24) + conn * ne;
    P.stream_state = opt->stream_state == 1   ? 1
                     : opt->stream_state == 2 ? 0
                                              : (ws > ((size_t)192 << 20));
    // the tet4 kernels of plans beyond the corner words keep it cached
    if (npe == 4 && c->scatter == CPI_SCATTER_BLOCK && !corner_words(c)) P.stream_state = 0;
  }
  if (c->scatter == CPI_SCATTER_BLOCK) {
    BlockPlan &B = c->plan;
    if (npe == 4 && B.max_local_nodes > elem_block_threads(4, c->rule, c->prec, c->phys, B.nblocks, cus))
      return fail(c, CPI_ERR_INVALID, "partition: a tet4 block has more nodes than threads");
    if (npe == 10 && c->nq == 4 && 4 * B.max_block_elems > elem_block_threads(10, c->rule, c->prec, c->phys, B.nblocks, cus))
      return fail(c, CPI_ERR_INVALID, "partition: a tet10 block has more points than threads");
    int32_t *meta, *bn, *bs, *sp, *dn, *ds;
    uint16_t *cl, *ci, *cw = nullptr, *dg, *dof;
    Vec3 *part;
    // the five-point tet10 kernel reads no words, but its resident steps do:
    // a thread per node, its elements in one round, a block per CU
    const int nt5 = elem_block_threads(npe, c->rule, c->prec, c->phys, B.nblocks, cus);
    const bool five = npe == 10 && c->nq == 5 && B.nblocks <= cus &&
                      B.max_local_nodes <= nt5 && B.max_block_elems <= nt5 / 64 * 12 &&
                      B.corner_fits();
    const bool words = corner_words(c) || five;
    if ((rc = dalloc(c, &meta, B.meta.size())) || (rc = upload(c, meta, B.meta)) ||
        (rc = dalloc(c, &cl, B.conn_local.size())) || (rc = upload(c, cl, B.conn_local)) ||
        (rc = dalloc(c, &ci, B.csr_pos.size())) || (rc = upload(c, ci, B.csr_pos)) ||
        (words && ((rc = dalloc(c, &cw, B.corner.size())) || (rc = upload(c, cw, B.corner)))) ||
        (rc = dalloc(c, &bn, B.bnd_nodes.size())) || (rc = upload(c, bn, B.bnd_nodes)) ||
        (rc = dalloc(c, &bs, B.bnd_slot.size())) || (rc = upload(c, bs, B.bnd_slot)) ||
        (rc = dalloc(c, &sp, B.slot_ptr.size())) || (rc = upload(c, sp, B.slot_ptr)) ||
        (rc = dalloc(c, &dn, B.nid_pad.size())) || (rc = upload(c, dn, B.nid_pad)) ||
        (rc = dalloc(c, &ds, B.slot_pad.size())) || (rc = upload(c, ds, B.slot_pad)) ||
        (rc = dalloc(c, &dg, B.deg_pad.size())) || (rc = upload(c, dg, B.deg_pad)) ||
        (rc = dalloc(c, &dof, B.off_pad.size())) || (rc = upload(c, dof, B.off_pad)) ||
        (rc = dalloc(c, &part, (size_t)std::max(B.n_slots, 1))))
      return rc;
    P.meta = meta;
    P.conn_local = cl;
    P.csr_pos = ci;
    P.corner = cw;
    P.bnd_nodes = bn;
    P.bnd_slot = bs;
    P.slot_ptr = sp;
    P.nid_pad = dn;
    P.slot_pad = ds;
    P.deg_pad = dg;
    P.off_pad = dof;
    P.ml = B.max_local_nodes;
    P.kmax = B.kmax;
    P.partial = part;
    P.n_interior = B.n_interior;
    P.n_boundary = B.n_boundary;
    P.max_loc = B.max_local_nodes;
    P.max_el = B.max_block_elems;
    // the yielded bits, one per stress point: tet4 and the per-point tet10
    // kernel, exact return (the surrogate kernel reads ep always and keeps
    // no bits)
    if ((npe == 4 || c->nq == 4) && c->phys == CPI_PHYSICS_EP) {
      unsigned long long *yw = nullptr;
      P.ywords = (c->nq * B.max_block_elems + 63) / 64;
      if ((rc = dalloc(c, &yw, (size_t)P.ywords * B.nblocks))) return rc;
      P.yielded = yw;
    }
    // surrogate mode: the step's counter, the deferred-block list and the
    // network queue (one row per element at most, plus a tile of padding
    // the last tile reads)
    if (npe == 4 && c->phys == 2) {
      unsigned long long *ctr = nullptr;
      int2 *lst = nullptr;
      uint16_t *rows = nullptr;
      const size_t nrows = (size_t)ne + 16;
      if ((rc = dalloc(c, &ctr, 1)) || (rc = dalloc(c, &lst, (size_t)B.nblocks)) ||
          (rc = dalloc(c, &rows, nrows * 16)))
        return rc;
      HIPCHK(c, hipMemsetAsync(rows, 0, nrows * 32, c->stream));
      P.mlp_ctr = ctr;
      P.mlp_list = lst;
      P.mlp_rows = rows;
    }
    P.nblocks = B.nblocks;
    P.narrow5 = npe == 10 && c->nq == 5 && nt5 != elem_block_threads(npe, c->rule, c->prec, c->phys, 0, cus);
    // FP64 tet10 on a 4-point rule: the matrix units sum the corner forces
    // while the chip is not full twice over (whose blocks may be resident).
    // There the arithmetic counts (48k elements, resident: 13.1 -> 10.2 us a
    // step, 48 spilled registers down to 4); a larger mesh is bound by its state's
    // traffic, and sixteen elements a wave meet twice the LDS bank conflicts of
    // quads (1.2M elements: 165 us with quads, 170).
    P.matrix = npe == 10 && c->nq == 4 && c->prec != CPI_PREC_F32 &&
               B.nblocks <= 2 * cus;
    c->smem = elem_block_smem(npe, c->rule, c->prec, P.ml, P.max_el, P.kmax);
    if (c->smem > (size_t)prop.sharedMemPerBlock)
      return fail(c, CPI_ERR_INVALID, "element block needs " + std::to_string(c->smem) +
                                          " bytes of LDS; lower block_elements");
    hipError_t pe = prepare_elem_block(npe, c->rule, c->prec, c->phys, c->smem);
    if (pe != hipSuccess)
      return fail(c, CPI_ERR_HIP, std::string("LDS opt-in for the element kernel: ") +
                                      hipGetErrorString(pe));
    // resident steps when every block fits the chip at once
    // (asked with no mail first: most meshes are too large, and their messages
    // need not be counted)
    auto fits = [&](size_t smem) {
      return smem <= (size_t)prop.sharedMemPerBlock &&
             B.nblocks <= resident_capacity(npe, c->rule, c->prec, c->phys, smem,
                                            cus);
    };
    if (opt->use_graph && c->phys != 2 && words && prop.cooperativeLaunch &&
        (npe == 4 || five || c->prec == CPI_PREC_F32 || P.matrix) && fits(c->smem)) {
      const MailCount N = count_mail(B);
      const size_t n = N.all, bytes = mail_bytes(c->prec, n);
      const size_t smem = resident_smem(c->smem, c->prec, (int)std::min<size_t>(N.most, 65536));
      if (bytes <= (size_t)INT32_MAX && N.most <= 65535 && fits(smem)) {
        const MailPlan M = build_mail(B);
        char *mail = nullptr;
        int32_t *mf, *mlo, *md;
        uint16_t *ms, *mi;
        if ((rc = dalloc(c, &mail, bytes)) || (rc = dalloc(c, &mf, M.first.size())) ||
            (rc = upload(c, mf, M.first)) || (rc = dalloc(c, &mlo, M.lo.size())) ||
            (rc = upload(c, mlo, M.lo)) || (rc = dalloc(c, &md, n)) || (rc = upload(c, md, M.dest)) ||
            (rc = dalloc(c, &ms, n)) || (rc = upload(c, ms, M.src)) || (rc = dalloc(c, &mi, n)) ||
            (rc = upload(c, mi, M.idx)))
          return rc;
        c->res = Resident{mail, (int)n, M.most, mf, md, ms, mlo, mi, 0, 0, 0,
                          opt->debug_fill_nan & 2 ? 1u : kSpinLimit, (int)c->loose.size()};
        c->res_smem = smem;
        c->calls.reserve(kMaxCalls + 1);
        for (hipEvent_t &e : c->res_done)
          HIPCHK(c, hipEventCreateWithFlags(&e, hipEventDisableTiming));
        c->res_able = true;
        c->res_min = B.nblocks <= cus ? kMinResident : kMinResidentMany;
        P.resident = B.nblocks > 1;  // one block waits for nobody
      }
    }
    // one energy row per wave
    c->n_elem_rows = c->nblocks * (elem_block_threads(npe, c->rule, c->prec, c->phys, c->nblocks, cus) / 64);
    c->n_node_rows = 4 * std::max(1, (B.n_boundary + 255) / 256);
  } else {
    c->n_elem_rows = elem_direct_rows(npe, ne);
    if (c->scatter == CPI_SCATTER_COLOR) {
      std::vector<int32_t> order, by_color;
      color_order(ne, c->color.data(), c->ncol, order, by_color, c->color_off);
      int32_t *dor;
      if ((rc = dalloc(c, &dor, order.size())) || (rc = upload(c, dor, order))) return rc;
      P.sample_id = dor;
      // a record per corner, of 2^32 at most; before the first step, FP64 corner
      // masses
      const size_t corners = (size_t)npe * ne;
      uint32_t *ds = nullptr, *dp = nullptr;
      char *cf = nullptr;
      if (corners > UINT32_MAX || (opt->debug_fill_nan & 4))
        rc = CPI_ERR_ALLOC;
      else if (!(rc = dalloc(c, &ds, corners)) && !(rc = dalloc(c, &dp, (size_t)nn + 1)))
        rc = dalloc(c, &cf, corners * (c->prec == CPI_PREC_F32 ? sizeof(Vec3f) : sizeof(Vec3)));
      if (rc == CPI_OK) {
        std::vector<uint32_t> slot, ptr;
        color_slots(ne, npe, c->conn_u.data(), nn, c->color.data(), c->ncol, slot, ptr, order);
        if ((rc = upload(c, ds, slot)) || (rc = upload(c, dp, ptr))) return rc;
        P.fslot = ds;
        P.node_slot = dp;
        P.cforce = cf;
      } else if (rc == CPI_ERR_ALLOC) {
        // no room: the forces are added up colour by colour, a launch each
        (void)hipGetLastError();
        dfree(c, ds);
        dfree(c, dp);
        if ((rc = alloc_forces(c)) || (rc = dalloc(c, &c->d_by_color, by_color.size())) ||
            (rc = upload(c, c->d_by_color, by_color)))
          return rc;
        c->n_elem_rows = 0;
        for (int k = 0; k < c->ncol; k++)
          c->n_elem_rows += elem_direct_rows(npe, c->color_off[k + 1] - c->color_off[k]);
      } else {
        return rc;
      }
    }
    c->n_node_rows = 4 * ((nn + 255) / 256);
  }
  c->n_rows = std::max(c->n_elem_rows + c->n_node_rows, 4 * ((nn + 255) / 256));
  double *ep = nullptr, *hist = nullptr, *ered = nullptr;
  Ctl *ctl = nullptr;
  if ((rc = dalloc(c, &ep, (size_t)EP_N * c->n_rows)) || (rc = dalloc(c, &ctl, 1)) ||
      (rc = dalloc(c, &hist, 8 * 4096)) ||
      (rc = dalloc(c, &ered, (size_t)EP_N * energy_reduce_blocks())))
    return rc;
  P.ered = ered;
  P.epart = ep;
  P.n_epart = c->n_rows;
  P.ctl = ctl;
  P.hist = hist;
  P.hist_cap = 4096;
  P.mlp_tol = opt->mlp_tolerance;
  P.sample_keep = 1ull << 32;  // the recorder keeps every yielding point
  if (c->phys == 2) {
    if ((rc = mlp_alloc(c->mlp, c->nblocks, c->stream, c->err))) return rc;
    P.mlp = c->mlp.d_params;
    P.mlp_stats = c->mlp.d_stats;
  }
  // the words cpi_get_state brings back, allocated once, or what there is room
  // for
  const size_t whole = kStateWords + 16 * (size_t)nn;
  rc = opt->debug_fill_nan & 4 ? CPI_ERR_ALLOC : ensure_tmp(c, whole);
  if (rc) rc = ensure_tmp(c, opt->debug_fill_nan & 4 ? kStateWords + 100 : std::min(whole, kTmpLow));
  if (rc) return rc;
  // reference positions on the device
  if ((rc = put_nodes(c, X0u, nullptr, c->P.X0))) return rc;
  return reset_state(c);
}

extern "C" int cpi_create(const cpi_mesh_desc *m, const cpi_material *mat, const cpi_wall *wall,
                          const cpi_options *opt, cpi_ctx **out) {
  if (!out) {
    set_global_error("cpi_create: out is NULL");
    return CPI_ERR_INVALID;
  }
  *out = nullptr;
  if (!m || !mat) {
    set_global_error("cpi_create: mesh and material are required");
    return CPI_ERR_INVALID;
  }
  cpi_options def;
  cpi_default_options(&def);
  cpi_ctx *c = new (std::nothrow) cpi_ctx;
  if (!c) {
    set_global_error("cpi_create: out of host memory");
    return CPI_ERR_ALLOC;
  }
  int rc;
  try {
    rc = create_impl(c, m, mat, wall, opt ? opt : &def);
  } catch (const std::bad_alloc &) {
    c->err = "cpi_create: out of host memory";
    rc = CPI_ERR_ALLOC;
  } catch (const std::exception &e) {
    c->err = std::string("cpi_create: ") + e.what();
    rc = CPI_ERR_ALLOC;
  }
  if (rc) {
    set_global_error(c->err);
    cpi_destroy(c);
    return rc;
  }
  *out = c;
  return CPI_OK;
}

extern "C" int cpi_set_state(cpi_ctx *c, const double *x0, const double *v0) {
  if (!c) return CPI_ERR_INVALID;
  const size_t n = 3 * (size_t)c->nn;
  if (x0 && !all_finite(x0, n)) return fail(c, CPI_ERR_INVALID, "non-finite position");
  if (v0 && !all_finite(v0, n)) return fail(c, CPI_ERR_INVALID, "non-finite velocity");
  if (x0) c->mass_ready = false;
  c->inited = false;
  c->res_pending = false;  // steps of a state that is given up
  c->calls.clear();
  int rc = x0 ? put_nodes(c, x0, nullptr, c->P.X0) : CPI_OK;
  if (!rc && v0) rc = put_nodes(c, v0, c->d_V0, nullptr);
  return rc ? rc : reset_state(c);
}

extern "C" int cpi_stable_dt(cpi_ctx *c, double *dte, double *dtc) {
  if (!c || !dte || !dtc) return CPI_ERR_INVALID;
  if (!c->inited) {
    int rc = reset_state(c);
    if (!rc && !c->mass_ready) rc = compute_mass(c);
    if (rc) return rc;
  }
  int rc = settled(c);
  return rc ? rc : stable_dt(c, dte, dtc);
}

// ---------------------------------------------------------------------------
// cpi_stable_dt without allocation: the scratch of its reductions is a
// file-scope device array, one copy per GPU, held until the process ends.
// It takes the per-workgroup element minima of k_elem_dt (one per 256
// elements) and, in its last kNoallocOut words, the two results of
// k_dt_finish.  Calls that overlap on one GPU share it and race.
// ---------------------------------------------------------------------------
constexpr int kNoallocPartials = 65536;  // 16,777,216 elements at most
constexpr int kNoallocOut = 2;
static __device__ __align__(256) double scratch[kNoallocPartials + kNoallocOut];

namespace {

constexpr int kNoallocDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch[kNoallocDevices] = {};

// this device's copy of scratch, looked up once with the device current
int scratch_of(cpi_ctx *c, double **out) {
  if (c->dev < 0 || c->dev >= kNoallocDevices)
    return fail(c, CPI_ERR_INVALID, "cpi_stable_dt_noalloc: device ordinal out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch[c->dev]) {
    HIPCHK(c, hipSetDevice(c->dev));
    void *ptr = nullptr;
    HIPCHK(c, hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    g_scratch[c->dev] = static_cast<double *>(ptr);
  }
  *out = g_scratch[c->dev];
  return CPI_OK;
}

}  // namespace

extern "C" int cpi_stable_dt_noalloc(cpi_ctx *c, double *dte, double *dtc) {
  if (!c || !dte || !dtc) return CPI_ERR_INVALID;
  if (!c->inited)
    return fail(c, CPI_ERR_STATE, "cpi_stable_dt_noalloc: needs cpi_init (mass assembled)");
  const int nb = (c->ne + 255) / 256;
  if (nb > kNoallocPartials)
    return fail(c, CPI_ERR_INVALID,
                "cpi_stable_dt_noalloc: at most " + std::to_string(256L * kNoallocPartials) +
                    " elements (the mesh has " + std::to_string(c->ne) + ")");
  double *sp = nullptr;
  int rc = settled(c);
  if (!rc) rc = scratch_of(c, &sp);
  if (rc) return rc;
  HIPCHK(c, launch_elem_dt(c->P, sp, c->stream));
  HIPCHK(c, launch_dt_finish(sp, nb, c->P.m, c->nn, sp + kNoallocPartials, c->stream));
  double r[kNoallocOut];
  HIPCHK(c, hipMemcpyAsync(r, sp + kNoallocPartials, sizeof(r), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  *dte = r[0];
  *dtc = (c->wall.enabled && c->wall.stiffness > 0.0) ? 2.0 * std::sqrt(r[1] / c->wall.stiffness)
                                                      : INFINITY;
  return CPI_OK;
}

extern "C" int cpi_init(cpi_ctx *c, double dt) {
  if (!c) return CPI_ERR_INVALID;
  if (!std::isfinite(dt)) return fail(c, CPI_ERR_INVALID, "cpi_init: dt must be finite");
  if (c->phys == 2 && !c->mlp.ready)
    return fail(c, CPI_ERR_STATE, "cpi_init: CPI_RETURN_MLP needs cpi_set_surrogate first");
  c->inited = false;
  c->res_pending = false;  // steps of a state that is given up
  c->calls.clear();
  int rc = reset_state(c);
  if (!rc) rc = compute_mass(c);
  if (rc) return rc;
  double dtc = INFINITY;
  if (dt <= 0.0) {
    double dte;
    if ((rc = stable_dt(c, &dte, &dtc))) return rc;
    const double ds = 1.0 / std::sqrt(1.0 / (dte * dte) + 1.0 / (dtc * dtc));
    dt = (dt == 0.0 ? 0.5 : -dt) * ds;
    if (!(dt > 0.0) || !std::isfinite(dt)) return fail(c, CPI_ERR_NUMERIC, "stable dt is not positive");
  } else if (c->phys != CPI_PHYSICS_COMPAT) {
    double dte;
    if ((rc = stable_dt(c, &dte, &dtc))) return rc;
  }
  c->dt = dt;
  c->step = 0;
  c->redone = 0;
  Ctl h{};
  h.dt = dt;
  h.dt_contact = dtc;
  HIPCHK(c, hipMemcpyAsync(c->P.ctl, &h, sizeof(Ctl), hipMemcpyHostToDevice, c->stream));
  hipError_t e = launch_node_init(c->P, c->stream);
  if (e == hipSuccess) e = launch_energy_reduce(c->P, c->stream);
  if (e != hipSuccess) return fail(c, CPI_ERR_HIP, std::string("init kernels: ") + hipGetErrorString(e));
  HIPCHK(c, hipMemsetAsync(c->P.epart, 0, sizeof(double) * EP_N * c->n_rows, c->stream));
  c->resident = c->res_able;
  if (c->resident) {
    c->res.base = 0;
    c->res.launch = 0;
    HIPCHK(c, launch_mail_clear(c->res, c->prec, c->stream));
  }
  HIPCHK(c, hipStreamSynchronize(c->stream));
  // the step graphs hold the context's buffers, which a new initial state
  // does not change; what does change the launches drops them
  if (c->opt.use_graph && !c->gs.run[1]) {
    drop_graphs(c);
    if ((rc = capture_graphs(c))) return rc;
  }
  c->inited = true;
  return CPI_OK;
}

extern "C" int cpi_step(cpi_ctx *c, int32_t nsteps) {
  if (!c) return CPI_ERR_INVALID;
  if (!c->inited) return fail(c, CPI_ERR_STATE, "cpi_step before cpi_init");
  if (nsteps < 0) return fail(c, CPI_ERR_INVALID, "nsteps < 0");
  int64_t rest = nsteps;
  int rc = CPI_OK;
  auto may = [&]() {
    return c->resident && c->gs.plain && !c->P.samples && nsteps - 1 >= c->res_min;
  };
  // plain steps launched one by one run whatever became of the launches before
  // them: these have to be settled first
  if (c->res_pending && ((!may() && nsteps > 1) || !c->resident || c->calls.size() >= kMaxCalls) &&
      (rc = settled(c)))
    return rc;
  // the plain steps in a few launches (the last step of a call is the one with
  // the energies and outputs)
  int k = 0;
  for (bool go = may(); go && rest > 1; k++) {
    if (k % kAhead == 0) {
      const hipEvent_t e = c->res_done[(k / kAhead) & 1];
      if (k >= 2 * kAhead) HIPCHK(c, hipEventSynchronize(e));
      if (rest > kMaxResident) HIPCHK(c, hipEventRecord(e, c->stream));
    }
    c->res.steps = (int)std::min(rest - 1, kMaxResident);
    c->res.launch++;
    Params p = c->P;
    p.epart_base = 0;
    const hipError_t e = launch_resident(p, c->rule, c->prec, c->phys, c->res, c->nblocks,
                                         c->res_smem, c->stream);
    if (e == hipSuccess) {
      c->res.base ^= c->res.steps & 1;
      c->res_pending = c->P.resident;
      HIPCHK(c, launch_resident_loose(p, c->res, c->stream));
      rest -= c->res.steps;
    } else {
      // the per-step launches from here on, for all that has not been taken
      (void)hipGetLastError();
      go = c->resident = false;
      Ctl h;
      if ((rc = settled_ctl(c, &h))) return rc;
      rest = c->step + nsteps - h.step;
    }
  }
  rc = steps_one_by_one(c, rest);
  if (rc) return rc;
  c->step += nsteps;
  if (c->res_pending) c->calls.push_back(c->step);
  return CPI_OK;
}

namespace {
// nsteps steps in the stream, from the step graphs or kernel by kernel
int steps_one_by_one(cpi_ctx *c, int64_t nsteps) {
  for (int64_t i = 0; i < nsteps;) {
    const bool aux = (i == nsteps - 1);
    const auto &G = c->gs;
    if (G.plain) {
      int k = 0;
      while (k < 2 && !(G.run[k] && nsteps - 1 - i >= kGraphRuns[k])) k++;
      if (!aux && k < 2) {
        HIPCHK(c, hipGraphLaunch(G.run[k], c->stream));
        i += kGraphRuns[k];
        continue;
      }
      HIPCHK(c, hipGraphLaunch(aux ? G.aux : G.plain, c->stream));
    } else {
      int rc = enqueue_step(c, aux);
      if (rc) return rc;
    }
    i++;
  }
  return CPI_OK;
}
}  // namespace

extern "C" int cpi_synchronize(cpi_ctx *c) {
  if (!c) return CPI_ERR_INVALID;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return check_flags(c);
}

extern "C" int cpi_get_state(cpi_ctx *c, double *x, double *v, double *a, double *m, double *vi) {
  return cpi_get_state_mass3(c, x, v, a, m, vi, nullptr);
}

extern "C" int cpi_get_state_mass3(cpi_ctx *c, double *x, double *v, double *a, double *m,
                                   double *vi, double *m3) {
  if (!c) return CPI_ERR_INVALID;
  Ctl h;
  // the nodes i .. i + n, and the control block with each part
  auto part = [&](size_t i, size_t n) -> int {
    Piece p[7] = {{&h, sizeof(Ctl) / 8}};
    int k = 1;
    double *d = c->d_tmp + kStateWords;
    auto place = [&](double *host, size_t words) -> double * {
      if (!host) return nullptr;
      p[k++] = Piece{host + words * i, words * n};
      d += words * n;
      return d - words * n;
    };
    NodeExport o{};
    o.ctl = reinterpret_cast<Ctl *>(c->d_tmp);
    o.x = place(x, 3);
    o.v = place(v, 3);
    o.a = place(a, 3);
    o.m = place(m, 1);
    o.vi = place(vi, 3);
    o.m3 = place(m3, 3);
    o.half_dt = 0.5 * c->dt;
    HIPCHK(c, launch_export_nodes(c->P, c->d_ninv + i, (int)n, o, c->stream));
    return bring_back(c, p, k);
  };
  const size_t words = 3 * (!!x + !!v + !!a + !!vi + !!m3) + !!m;
  int rc = in_parts(c, c->nn, words, kStateWords, part);
  if (rc) return rc;
  if (c->res_pending) {
    bool missing;
    if ((rc = settle(c, h, &missing))) return rc;
    if (missing && (rc = in_parts(c, c->nn, words, kStateWords, part))) return rc;
  }
  return c->inited ? report_flags(c, h) : CPI_OK;
}

extern "C" int cpi_get_increment(cpi_ctx *c, double *du) {
  if (!c || !du) return CPI_ERR_INVALID;
  int rc = settled(c);
  if (rc) return rc;
  Params p = c->P;
  p.acc = c->P.du;
  NodeExport o{};
  o.a = c->d_tmp;
  return in_parts(c, c->nn, 3, 0, [&](size_t i, size_t n) -> int {
    HIPCHK(c, launch_export_nodes(p, c->d_ninv + i, (int)n, o, c->stream));
    const Piece q{du + 3 * i, 3 * n};
    return bring_back(c, &q, 1);
  });
}

extern "C" int cpi_get_element_state(cpi_ctx *c, double *sig, double *ep) {
  if (!c) return CPI_ERR_INVALID;
  const size_t n = (size_t)c->nq * c->ne;
  if (c->phys == CPI_PHYSICS_COMPAT) {
    if (sig) std::memset(sig, 0, sizeof(double) * 6 * n);
    if (ep) std::memset(ep, 0, sizeof(double) * n);
    return CPI_OK;
  }
  int rc = settled(c);
  if (rc || (!sig && !ep)) return rc;
  // an element's words
  const size_t ws = sig ? 6 * (size_t)c->nq : 0, we = ep ? (size_t)c->nq : 0;
  if (!(c->opt.debug_fill_nan & 4)) (void)ensure_tmp(c, std::min((ws + we) * c->ne, kTmpMost));
  return in_parts(c, c->ne, ws + we, 0, [&](size_t i, size_t ne) -> int {
    Piece p[2];
    int k = 0;
    if (sig) p[k++] = Piece{sig + ws * i, ws * ne};
    if (ep) p[k++] = Piece{ep + we * i, we * ne};
    HIPCHK(c, launch_export_elems(c->P, c->prec, c->d_spos + i, (int)ne, sig ? c->d_tmp : nullptr,
                                  ep ? c->d_tmp + ws * ne : nullptr, c->stream));
    return bring_back(c, p, k);
  });
}

extern "C" int cpi_get_stress_strain(cpi_ctx *c, double *strain, double *stress) {
  if (!c) return CPI_ERR_INVALID;
  if (!c->inited) return fail(c, CPI_ERR_STATE, "cpi_get_stress_strain before cpi_init");
  int rc = settled(c);
  if (rc) return rc;
  // nodes of no element keep what the caller's arrays hold
  double *out[2] = {strain, stress};
  std::vector<double> keep;
  try {
    for (double *o : out)
      if (o)
        for (int32_t n : c->loose) keep.insert(keep.end(), o + 6L * n, o + 6L * n + 6);
  } catch (const std::bad_alloc &) {
    return fail(c, CPI_ERR_ALLOC, "cpi_get_stress_strain: out of host memory");
  }
  rc = in_parts(c, c->nn, 6 * (!!strain + !!stress), 0, [&](size_t i, size_t n) -> int {
    Piece p[2];
    int k = 0;
    if (strain) p[k++] = Piece{strain + 6 * i, 6 * n};
    if (stress) p[k++] = Piece{stress + 6 * i, 6 * n};
    HIPCHK(c, launch_stress_node(c->P, c->d_last + i, (int)n, strain ? c->d_tmp : nullptr,
                                 stress ? c->d_tmp + (strain ? 6 * n : 0) : nullptr, c->stream));
    return bring_back(c, p, k);
  });
  const double *was = keep.data();
  for (double *o : out)
    if (o)
      for (int32_t n : c->loose) {
        std::memcpy(o + 6L * n, was, 6 * sizeof(double));
        was += 6;
      }
  return rc;
}

extern "C" int cpi_get_energy(cpi_ctx *c, double *row, int64_t *step) {
  if (!c || !row) return CPI_ERR_INVALID;
  Ctl h;
  int rc = settled_ctl(c, &h);
  if (rc) return rc;
  std::memcpy(row, h.row, sizeof(double) * CPI_NENERGY);
  if (step) *step = h.step;
  return CPI_OK;
}

extern "C" int cpi_get_energy_history(cpi_ctx *c, double *rows, int32_t cap, int32_t *count) {
  if (!c || !count || cap < 0) return CPI_ERR_INVALID;
  Ctl h;
  int rc = settled_ctl(c, &h);
  if (rc) return rc;
  const int64_t have = std::min<int64_t>(h.nrows, c->P.hist_cap);
  const int64_t n = std::min<int64_t>(have, cap);
  std::vector<double> all(8 * (size_t)c->P.hist_cap);
  HIPCHK(c, hipMemcpyAsync(all.data(), c->P.hist, sizeof(double) * all.size(), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  for (int64_t i = 0; i < n; i++) {
    int64_t r = h.nrows - n + i;
    std::memcpy(rows + 8 * i, &all[8 * (size_t)(r % c->P.hist_cap)], 8 * sizeof(double));
  }
  *count = (int32_t)n;
  return CPI_OK;
}

extern "C" int cpi_get_info(cpi_ctx *c, cpi_info *info) {
  if (!c || !info) return CPI_ERR_INVALID;
  std::memset(info, 0, sizeof(*info));
  info->num_nodes = c->nn;
  info->num_elements = c->ne;
  info->nodes_per_element = c->npe;
  info->num_quadrature_pts = c->nq;
  info->num_colors = c->ncol;
  info->num_blocks = c->scatter == CPI_SCATTER_BLOCK ? c->nblocks : 0;
  info->num_boundary_nodes = c->scatter == CPI_SCATTER_BLOCK ? c->plan.n_boundary : c->nn;
  info->num_partial_slots = c->scatter == CPI_SCATTER_BLOCK ? c->plan.n_slots : 0;
  // algorithmic bytes of an elastic step: connectivity 4 npe and the
  // stress read and written, 12 nq s, per element (ep is written only when
  // a point yields; the exact-return tet4 and per-point tet10 block kernels
  // read it only for points that have yielded, the other kernels read it
  // always), then per node what each pass must touch once
  const double s = c->prec == CPI_PREC_F32 ? 4 : 8;
  const bool block = c->scatter == CPI_SCATTER_BLOCK;
  const bool bits = block && c->phys == CPI_PHYSICS_EP && (c->npe == 4 || c->nq == 4);
  const double state =
      c->phys == CPI_PHYSICS_COMPAT ? 0.0 : (12.0 + (bits ? 0.0 : 1.0)) * c->nq * s;
  const double per_elem = 4.0 * c->npe + state;
  info->bytes_per_step = c->ne * per_elem + 224.0 * c->nn;
  if (block) {
    // corners as 16-bit words, or two u16 arrays
    const double nb = c->plan.n_boundary, ni = c->plan.n_interior;
    const double conn = corner_words(c) ? 2.0 * c->npe : 4.0 * c->npe;
    info->elem_kernel_bytes = c->ne * (conn + state) + ni * 104.0 + nb * 72.0;
    info->node_kernel_bytes = nb * 128.0;
  } else {
    info->elem_kernel_bytes = c->ne * per_elem + c->nn * 72.0;
    info->node_kernel_bytes = c->nn * 152.0;
  }
  info->dt = c->dt;
  info->step = c->step;
  return CPI_OK;
}

extern "C" int cpi_get_resident_steps(cpi_ctx *c, int64_t *taken, int64_t *redone) {
  if (!c) return CPI_ERR_INVALID;
  Ctl h{};
  int rc = c->inited ? settled_ctl(c, &h) : CPI_OK;
  if (rc) return rc;
  if (taken) *taken = h.resident;
  if (redone) *redone = c->redone;
  return CPI_OK;
}

extern "C" int cpi_get_coloring(cpi_ctx *c, int32_t *color, int32_t *ncol) {
  if (!c) return CPI_ERR_INVALID;
  if (color) std::memcpy(color, c->color.data(), sizeof(int32_t) * c->ne);
  if (ncol) *ncol = c->ncol;
  return CPI_OK;
}

extern "C" int cpi_time_steps(cpi_ctx *c, int32_t nsteps, double *ms) {
  if (!c || !ms) return CPI_ERR_INVALID;
  int rc = settled(c);  // the steps queued before have no part in the time
  if (rc) return rc;
  hipEvent_t a, b;
  HIPCHK(c, hipEventCreate(&a));
  HIPCHK(c, hipEventCreate(&b));
  HIPCHK(c, hipEventRecord(a, c->stream));
  rc = cpi_step(c, nsteps);
  HIPCHK(c, hipEventRecord(b, c->stream));
  HIPCHK(c, hipEventSynchronize(b));
  // steps that a resident launch left out belong to the time
  const int64_t redone = c->redone;
  if (!rc) rc = settled(c);
  if (c->redone != redone) {
    HIPCHK(c, hipEventRecord(b, c->stream));
    HIPCHK(c, hipEventSynchronize(b));
  }
  float t = 0.f;
  HIPCHK(c, hipEventElapsedTime(&t, a, b));
  (void)hipEventDestroy(a);
  (void)hipEventDestroy(b);
  *ms = t;
  return rc;
}

extern "C" int cpi_profile_kernels(cpi_ctx *c, int32_t nsteps, cpi_kernel_time *out, int32_t cap,
                                   int32_t *count) {
  if (!c || !out || !count) return CPI_ERR_INVALID;
  if (!c->inited) return fail(c, CPI_ERR_STATE, "cpi_profile_kernels before cpi_init");
  if (int rc = settled(c)) return rc;
  // with the surrogate the element pass is three launches: every other step
  // times them one by one, "elem_pass" (the elastic pass), "mlp_queue" (the
  // network on the queue) and "mlp_walk" (the deferred blocks), and the
  // steps between time the three together ("elem_block": from the start of
  // the first to the end of the last).  Block-scatter kernels are timed by
  // events their launch records at the kernel's own start and end
  // (hipExtLaunchKernel); the colour and atomic scatters' launches by events
  // recorded around them.
  const bool mlp = c->scatter == CPI_SCATTER_BLOCK && c->phys == 2;
  const char *names[5] = {c->scatter == CPI_SCATTER_BLOCK ? "elem_block" : "elem_direct",
                          c->scatter == CPI_SCATTER_BLOCK ? "node_bnd" : "node_all", "elem_pass",
                          "mlp_queue", "mlp_walk"};
  double tot[5] = {0, 0, 0, 0, 0};
  int64_t launches[5] = {0, 0, 0, 0, 0};
  // ev[0], ev[1] element pass start and end; ev[2], ev[3] node pass; ev[4..9]
  // the three surrogate launches one by one (destroyed on every return, and
  // no launch keeps them)
  struct Events {
    hipEvent_t e[10] = {};
    ~Events() {
      set_launch_events(nullptr, nullptr);
      for (auto &x : e)
        if (x) (void)hipEventDestroy(x);
    }
  } evs;
  hipEvent_t *ev = evs.e;
  for (int k = 0; k < 10; k++) HIPCHK(c, hipEventCreate(&ev[k]));
  auto elapsed = [&](int a, int b, float &ms) -> int {
    HIPCHK(c, hipEventElapsedTime(&ms, ev[a], ev[b]));
    return CPI_OK;
  };
  for (int i = 0; i < nsteps; i++) {
    Params p = c->P;
    p.store_aux = 0;
    const bool split = mlp && i % 2 == 0;
    hipError_t e = hipSuccess;
    p.epart_base = 0;
    if (mlp) {
      for (int part = 1; part <= 3 && e == hipSuccess; part++) {
        if (split)
          set_launch_events(ev[2 + 2 * part], ev[3 + 2 * part]);
        else
          set_launch_events(part == 1 ? ev[0] : nullptr, part == 3 ? ev[1] : nullptr);
        e = launch_elem_block(p, c->rule, c->prec, c->phys, false, c->nblocks, c->smem, c->stream,
                              part);
      }
      set_launch_events(nullptr, nullptr);
      if (split)
        for (int k = 2; k < 5; k++) launches[k] += 1;
      else
        launches[0] += 1;
    } else if (c->scatter == CPI_SCATTER_BLOCK) {
      set_launch_events(ev[0], ev[1]);
      e = launch_elem_block(p, c->rule, c->prec, c->phys, false, c->nblocks, c->smem, c->stream);
      set_launch_events(nullptr, nullptr);
      launches[0] += 1;
    } else {
      HIPCHK(c, hipEventRecord(ev[0], c->stream));
      e = elem_direct(c, p, &launches[0]);
      HIPCHK(c, hipEventRecord(ev[1], c->stream));
    }
    p.epart_base = c->n_elem_rows;
    if (e == hipSuccess) {
      if (c->scatter == CPI_SCATTER_BLOCK) {
        set_launch_events(ev[2], ev[3]);
        e = launch_node_bnd(p, c->prec, false, c->stream);
        set_launch_events(nullptr, nullptr);
      } else {
        HIPCHK(c, hipEventRecord(ev[2], c->stream));
        e = launch_node_all(p, c->prec, false, c->stream);
        HIPCHK(c, hipEventRecord(ev[3], c->stream));
      }
    }
    launches[1] += 1;
    if (e != hipSuccess) return fail(c, CPI_ERR_HIP, hipGetErrorString(e));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    float t = 0;
    int rc;
    if (split) {
      for (int k = 0; k < 3; k++) {
        if ((rc = elapsed(4 + 2 * k, 5 + 2 * k, t))) return rc;
        tot[2 + k] += t;
      }
    } else {
      if ((rc = elapsed(0, 1, t))) return rc;
      tot[0] += t;
    }
    if ((rc = elapsed(2, 3, t))) return rc;
    tot[1] += t;
  }
  c->step += nsteps;
  // one step only: the element pass is the sum of its launches
  if (launches[0] == 0 && launches[2] > 0) {
    tot[0] = tot[2] + tot[3] + tot[4];
    launches[0] = launches[2];
  }
  // the split entries only when some step was split
  int n = std::min<int>(cap, launches[2] > 0 ? 5 : 2);
  for (int k = 0; k < n; k++) {
    std::memset(out[k].name, 0, sizeof(out[k].name));
    std::strncpy(out[k].name, names[k], sizeof(out[k].name) - 1);
    out[k].total_ms = tot[k];
    out[k].launches = launches[k];
  }
  *count = n;
  return CPI_OK;
}

extern "C" int cpi_debug_strain(cpi_ctx *c, double alpha, int32_t dcase, double *W, double *V) {
  if (!c || !W || !V) return CPI_ERR_INVALID;
  if (dcase != 0 && dcase != 1) return fail(c, CPI_ERR_INVALID, "deformation case must be 0 or 1");
  const int nb = (c->ne + 255) / 256;
  int rc = ensure_tmp(c, 2 * (size_t)nb);
  if (rc) return rc;
  Params p = c->P;
  hipError_t e = launch_debug_strain(p, c->rule, alpha, dcase, c->mat.nu, c->d_tmp, c->stream);
  if (e != hipSuccess) return fail(c, CPI_ERR_HIP, hipGetErrorString(e));
  std::vector<double> h(2 * (size_t)nb);
  HIPCHK(c, hipMemcpyAsync(h.data(), c->d_tmp, sizeof(double) * h.size(), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  double w = 0, v = 0;
  for (int i = 0; i < nb; i++) {
    w += h[2 * i];
    v += h[2 * i + 1];
  }
  *W = w;
  *V = v;
  return CPI_OK;
}

extern "C" int cpi_bandwidth_probe(int32_t device, int64_t bytes, int32_t reps, double *gbs) {
  if (!gbs || bytes < 1024 || reps < 1) {
    set_global_error("cpi_bandwidth_probe: invalid arguments");
    return CPI_ERR_INVALID;
  }
  cpi_ctx tmp;  // only for error reporting through HIPCHK
  cpi_ctx *c = &tmp;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev) {
    set_global_error("cpi_bandwidth_probe: no HIP device " + std::to_string(device));
    return CPI_ERR_NO_DEVICE;
  }
  const long n4 = (long)(bytes / 32);
  void *a = nullptr, *b = nullptr;
  hipStream_t s = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = CPI_OK;
  auto run = [&]() -> int {
    HIPCHK(c, hipSetDevice(device));
    HIPCHK(c, hipMalloc(&a, n4 * 32));
    HIPCHK(c, hipMalloc(&b, n4 * 32));
    HIPCHK(c, hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    HIPCHK(c, hipMemsetAsync(a, 0, n4 * 32, s));
    HIPCHK(c, hipEventCreate(&e0));
    HIPCHK(c, hipEventCreate(&e1));
    HIPCHK(c, launch_stream_copy(a, b, n4, s));  // warm-up
    HIPCHK(c, hipEventRecord(e0, s));
    for (int i = 0; i < reps; i++) HIPCHK(c, launch_stream_copy(a, b, n4, s));
    HIPCHK(c, hipEventRecord(e1, s));
    HIPCHK(c, hipEventSynchronize(e1));
    float ms = 0.f;
    HIPCHK(c, hipEventElapsedTime(&ms, e0, e1));
    *gbs = 2.0 * 32.0 * (double)n4 * reps / (ms * 1e-3) / 1e9;
    return CPI_OK;
  };
  rc = run();
  if (rc) set_global_error(c->err);
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (s) (void)hipStreamDestroy(s);
  if (a) (void)hipFree(a);
  if (b) (void)hipFree(b);
  return rc;
}

// ---------------------------------------------------------------------------
// surrogate installation, counters and return-map samples
// ---------------------------------------------------------------------------

namespace {

bool same_value(double a, double b) { return std::fabs(a - b) <= 1e-12 * std::max(std::fabs(a), std::fabs(b)); }

// re-captures the step graphs after a change of the kernel arguments
int refresh_graphs(cpi_ctx *c) {
  drop_graphs(c);
  if (c->inited && c->opt.use_graph) return capture_graphs(c);
  return CPI_OK;
}

}  // namespace

extern "C" int cpi_set_surrogate(cpi_ctx *c, const cpi_mlp *m) {
  if (!c || !m) return CPI_ERR_INVALID;
  if (c->phys != 2)
    return fail(c, CPI_ERR_STATE, "cpi_set_surrogate: the context was not created with CPI_RETURN_MLP");
  if (m->dev != c->dev) return fail(c, CPI_ERR_INVALID, "cpi_set_surrogate: network is on another device");
  if (!m->scaled) return fail(c, CPI_ERR_STATE, "cpi_set_surrogate: network has no scaling (train or set it)");
  const MlpMaterial a = mlp_material(c->mat), &b = m->mm;
  if (!same_value(a.c11, b.c11) || !same_value(a.c12, b.c12) || !same_value(a.c44, b.c44) ||
      !same_value(a.sy0, b.sy0) || !same_value(a.H, b.H))
    return fail(c, CPI_ERR_INVALID, "cpi_set_surrogate: network was made for another material");
  HIPCHK(c, hipSetDevice(c->dev));
  HIPCHK(c, hipStreamSynchronize(m->stream));
  HIPCHK(c, hipMemcpyAsync(c->mlp.d_weights, m->W, sizeof(MlpWeights), hipMemcpyDeviceToDevice, c->stream));
  MlpParams h{};
  h.weights = c->mlp.d_weights;
  h.w1 = c->mlp.d_weights->w1;
  h.w2p = c->mlp.d_weights->w2p;
  h.w3p = c->mlp.d_weights->w3p;
  h.b1 = c->mlp.d_weights->b1;
  h.b2 = c->mlp.d_weights->b2;
  h.b3 = c->mlp.d_weights->b3;
  for (int k = 0; k < kMlpIn; k++) {
    h.in_mean[k] = m->in_mean[k];
    h.in_istd[k] = 1.0f / m->in_std[k];
  }
  for (int k = 0; k < kMlpOut; k++) {
    h.out_mean[k] = m->out_mean[k];
    h.out_std[k] = m->out_std[k];
  }
  h.c11 = (float)a.c11;
  h.c12 = (float)a.c12;
  h.c44 = (float)a.c44;
  h.sy0 = (float)a.sy0;
  h.H = (float)a.H;
  HIPCHK(c, hipMemcpyAsync(c->mlp.d_params, &h, sizeof(h), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->mlp.ready = true;
  return CPI_OK;
}

extern "C" int cpi_get_surrogate_stats(cpi_ctx *c, int64_t *accepted, int64_t *fallback) {
  if (!c) return CPI_ERR_INVALID;
  unsigned long long h[2] = {0, 0};
  if (c->mlp.d_stats) {
    std::vector<unsigned long long> all(2 * (size_t)c->mlp.nstats);
    HIPCHK(c, hipMemcpyAsync(all.data(), c->mlp.d_stats, sizeof(unsigned long long) * all.size(),
                             hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
    for (size_t i = 0; i < all.size(); i += 2) {
      h[0] += all[i];
      h[1] += all[i + 1];
    }
  }
  if (accepted) *accepted = (int64_t)h[0];
  if (fallback) *fallback = (int64_t)h[1];
  return CPI_OK;
}

extern "C" int cpi_reset_surrogate_stats(cpi_ctx *c) {
  if (!c) return CPI_ERR_INVALID;
  if (c->mlp.d_stats) {
    HIPCHK(c, hipMemsetAsync(c->mlp.d_stats, 0, 2 * sizeof(unsigned long long) * c->mlp.nstats,
                             c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  return CPI_OK;
}

extern "C" int cpi_samples_enable(cpi_ctx *c, int32_t cap) {
  if (!c || cap < 0) return CPI_ERR_INVALID;
  if (c->phys != CPI_PHYSICS_EP)
    return fail(c, CPI_ERR_STATE, "cpi_samples_enable: needs CPI_PHYSICS_EP with the exact return");
  HIPCHK(c, hipSetDevice(c->dev));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  int rc = settled(c);
  if (rc) return rc;
  rc = mlp_samples_alloc(c->mlp, cap, c->stream, c->err);
  if (rc) return rc;
  c->P.samples = c->mlp.d_samples;
  c->P.sample_count = c->mlp.d_sample_count;
  c->P.sample_cap = c->mlp.sample_cap;
  return refresh_graphs(c);
}

extern "C" int cpi_samples_subsample(cpi_ctx *c, double keep, uint64_t seed) {
  if (!c || !(keep >= 0.0 && keep <= 1.0)) return CPI_ERR_INVALID;
  c->P.sample_keep = keep >= 1.0 ? (1ull << 32) : (unsigned long long)(keep * 4294967296.0);
  c->P.sample_seed = seed;
  return refresh_graphs(c);
}

extern "C" int cpi_samples_get(cpi_ctx *c, float *out, int32_t cap, int32_t *recorded) {
  if (!c || cap < 0 || (cap > 0 && !out)) return CPI_ERR_INVALID;
  int cnt = 0;
  if (c->mlp.d_sample_count) {
    HIPCHK(c, hipMemcpyAsync(&cnt, c->mlp.d_sample_count, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  const int k = std::min(std::min(cnt, c->mlp.sample_cap), cap);
  if (k > 0) {
    HIPCHK(c, hipMemcpyAsync(out, c->mlp.d_samples, sizeof(float) * kSampleFloats * (size_t)k,
                             hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  if (recorded) *recorded = cnt;
  return CPI_OK;
}

extern "C" int cpi_samples_reset(cpi_ctx *c) {
  if (!c) return CPI_ERR_INVALID;
  if (c->mlp.d_sample_count) {
    HIPCHK(c, hipMemsetAsync(c->mlp.d_sample_count, 0, sizeof(int), c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));
  }
  return CPI_OK;
}
