// context.hip -- process-global state, init/finalize, errors, device memory.
//
// Replaces the reference's QPHIX_init/QPHIX_finalize (qphix_misc.cpp:427-594):
// the reference's thread pool, barriers and neighbour tables become one HIP
// device, one stream and on-the-fly neighbour index arithmetic.
#include "common.h"
#include "hostio.h"
#include <algorithm>
#include "qphix_mi355x.h"

#include <cstring>
#include <list>
#include <mutex>
#include <unordered_map>
#include <utility>

namespace qphix {

static Context g_ctx;
static char g_last_error[512] = {0};
static int g_error_count = 0;

Context &ctx() { return g_ctx; }

void fail(const char *file, int line, const char *msg) {
  std::snprintf(g_last_error, sizeof(g_last_error), "%s:%d: %s", file, line, msg);
  ++g_error_count;
  if (g_ctx.abort_on_error) {
    std::fprintf(stderr, "QPHIX ERROR %s\n", g_last_error);
    std::fflush(stderr);
    std::exit(1);
  }
}

bool failed() { return g_error_count != 0; }

bool require_init() { return g_ctx.initialised; }

void sync_if_needed() {
  if (g_ctx.sync_calls) HIP_CHECK(hipStreamSynchronize(g_ctx.stream));
}

// Allocation-failure injection for the error-path tests: after `n` more
// successful allocations every dev_alloc fails as if device memory were
// exhausted (negative: never).
static long g_fail_alloc_after = -1;

// Device blocks that handles and calls have freed, kept for the next one of the
// same size: hipMalloc and hipFree of a vector cost about 0.1 ms each and of a
// gigabyte up to 40 ms, more than the work of many calls.  At most DEV_KEEP
// bytes are held, the longest unused go first; all of them when an allocation
// fails and at finalize.  6 GiB: the scratch of a link preparation (LP_TOGETHER,
// 4 GiB) with link sets and their sloppy copies (24^3x32: 1.2 GB).  Work queued on
// a block before it was freed and after it was taken again is on the one library
// stream, in order.
constexpr size_t DEV_KEEP = (size_t)6 << 30, DEV_KEEP_BLOCKS = 256;

struct KeptBlocks {
  std::recursive_mutex m;  // a failed hipFree may end the process, whose exit handler finalizes
  std::unordered_map<void *, std::pair<size_t, int>> out;  // blocks handed out: bytes, device
  std::list<std::pair<void *, size_t>> kept;               // free, oldest first
  size_t held = 0;
};
static KeptBlocks &blocks() {
  static KeptBlocks *k = new KeptBlocks;  // outlives handles freed at process exit
  return *k;
}

// Gives kept blocks back until at most `most` bytes are held in fewer than
// DEV_KEEP_BLOCKS blocks (k.m is held).
static void shrink_blocks(KeptBlocks &k, size_t most) {
  while (k.held > most || k.kept.size() >= DEV_KEEP_BLOCKS) {
    void *const p = k.kept.front().first;
    k.held -= k.kept.front().second;
    k.kept.pop_front();
    HIP_CHECK(hipFree(p));
  }
}

static void *block_get(size_t bytes) {
  KeptBlocks &k = blocks();
  std::lock_guard<std::recursive_mutex> l(k.m);
  for (auto it = k.kept.begin(); it != k.kept.end(); ++it)
    if (it->second == bytes) {
      void *p = it->first;
      k.held -= bytes;
      k.kept.erase(it);
      k.out[p] = {bytes, g_ctx.device};
      return p;
    }
  void *p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    if (k.held == 0) return nullptr;
    shrink_blocks(k, 0);
    p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
      (void)hipGetLastError();
      return nullptr;
    }
  }
  k.out[p] = {bytes, g_ctx.device};
  return p;
}

void *dev_alloc(size_t bytes) {
  if (bytes == 0) return nullptr;
  if (g_fail_alloc_after == 0) {
    fail(__FILE__, __LINE__, "hipMalloc failed (device memory exhausted?) [injected]");
    return nullptr;
  }
  if (g_fail_alloc_after > 0) --g_fail_alloc_after;
  void *p = block_get(bytes);
  if (!p) fail(__FILE__, __LINE__, "hipMalloc failed (device memory exhausted?)");
  return p;
}

// Single-reduction CG steps: bit 0 the one-precision CG, bit 1 the mixed
// solver's sloppy steps.  QPHIX_FEWSUMS in the environment sets the initial
// value; QPHIX_MI355X_set_fewsums wins.
static int g_fewsums = -1;
int fewsums_mode() {
  if (g_fewsums < 0) {
    const char *e = std::getenv("QPHIX_FEWSUMS");
    g_fewsums = e ? (std::atoi(e) & 3) : 2;
  }
  return g_fewsums;
}
void set_fewsums_mode(int mode) { g_fewsums = mode & 3; }

void *dev_try_alloc(size_t bytes) {
  if (bytes == 0 || g_fail_alloc_after == 0) return nullptr;
  if (g_fail_alloc_after > 0) --g_fail_alloc_after;
  return block_get(bytes);
}

void dev_free(void *p) {
  if (!p) return;
  KeptBlocks &k = blocks();
  std::lock_guard<std::recursive_mutex> l(k.m);
  const auto it = k.out.find(p);
  const auto [bytes, device] = it == k.out.end() ? std::pair<size_t, int>{0, -1} : it->second;
  if (it != k.out.end()) k.out.erase(it);
  if (!g_ctx.initialised || device != g_ctx.device || bytes > DEV_KEEP) {
    HIP_CHECK(hipFree(p));
    return;
  }
  shrink_blocks(k, DEV_KEEP - bytes);
  k.kept.emplace_back(p, bytes);
  k.held += bytes;
}

// A workspace that grows: its old block has no next user of the same size.
static void ws_release(void *p) {
  if (!p) return;
  KeptBlocks &k = blocks();
  std::lock_guard<std::recursive_mutex> l(k.m);
  k.out.erase(p);
  HIP_CHECK(hipFree(p));
}

void *ws_get(size_t bytes) {
  Context &c = g_ctx;
  if (bytes > c.ws_bytes) {
    HIP_CHECK(hipStreamSynchronize(c.stream));
    ws_release(c.ws);
    c.ws = dev_alloc(bytes);
    c.ws_bytes = c.ws ? bytes : 0;
  }
  return c.ws;
}

void *ws2_get(size_t bytes) {
  Context &c = g_ctx;
  if (bytes > c.ws2_bytes) {
    HIP_CHECK(hipStreamSynchronize(c.stream));
    ws_release(c.ws2);
    c.ws2 = dev_alloc(bytes);
    c.ws2_bytes = c.ws2 ? bytes : 0;
  }
  return c.ws2;
}

void *ws2_try_get(size_t bytes) {
  Context &c = g_ctx;
  if (bytes > c.ws2_bytes) {
    HIP_CHECK(hipStreamSynchronize(c.stream));
    ws_release(c.ws2);
    c.ws2 = dev_try_alloc(bytes);
    c.ws2_bytes = c.ws2 ? bytes : 0;
  }
  return c.ws2;
}

// Gauge force kernel: 1 (default) the staple-product kernel where the links
// are SU(3) to rounding, 0 always the loop-walk kernel.
static int g_gf_staples = 1;
int gauge_force_staples_mode() { return g_gf_staples; }

static QPHIX_status_t init_common(QPHIX_layout_t *layout) {
  Context &c = g_ctx;
  if (c.initialised) return QPHIX_SUCCESS;  // F and D share one lattice (C14)
  // QPHIX_GRAPHS=0 starts the process with graph replay off (read once; a
  // later QPHIX_MI355X_set_graphs call wins)
  static bool env_read = false;
  if (!env_read) {
    env_read = true;
    if (const char *e = std::getenv("QPHIX_GRAPHS")) c.graphs = std::atoi(e) != 0;
  }
  if (!layout || layout->latdim != 4 || !layout->latsize) {
    fail(__FILE__, __LINE__, "QPHIX_init: need a 4-d layout");
    return QPHIX_FAIL;
  }
  if (layout->machdim != layout->latdim) {
    fail(__FILE__, __LINE__, "QPHIX_init: machine dimension must equal lattice dimension");
    return QPHIX_FAIL;
  }
  for (int d = 0; d < layout->machdim; ++d)
    if (layout->machsize && layout->machsize[d] != 1) {
      fail(__FILE__, __LINE__, "QPHIX_init: this build runs one lattice on one GPU (machsize must be 1)");
      return QPHIX_FAIL;
    }
  const int *L = layout->latsize;
  // qphix_misc.cpp:494-497: Nxh%2, Ny%4, Nz%4, Nt%4 (minimum lattice 4^4)
  if (L[0] % 4 || L[1] % 4 || L[2] % 4 || L[3] % 4 || L[0] <= 0) {
    fail(__FILE__, __LINE__, "QPHIX_init: every lattice extent must be a positive multiple of 4");
    return QPHIX_FAIL;
  }
  long long vol = 1LL * L[0] * L[1] * L[2] * L[3];
  if (vol / 2 > (1LL << 30)) {
    fail(__FILE__, __LINE__, "QPHIX_init: lattice too large for 32-bit site indices");
    return QPHIX_FAIL;
  }
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
    fail(__FILE__, __LINE__, "QPHIX_init: no HIP device visible");
    return QPHIX_FAIL;
  }
  const char *dv = std::getenv("QPHIX_DEVICE");
  c.device = dv ? std::atoi(dv) : 0;
  if (c.device < 0 || c.device >= ndev) c.device = 0;
  if (hipSetDevice(c.device) != hipSuccess) {
    fail(__FILE__, __LINE__, "QPHIX_init: hipSetDevice failed");
    return QPHIX_FAIL;
  }
  if (!faces_scratch_setup(c.device)) return QPHIX_FAIL;
  hipDeviceProp_t prop;
  HIP_CHECK(hipGetDeviceProperties(&prop, c.device));
  c.n_cu = prop.multiProcessorCount;
  HIP_CHECK(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking));

  Geometry &g = c.g;
  g.nx = L[0]; g.ny = L[1]; g.nz = L[2]; g.nt = L[3];
  g.nxh = g.nx / 2;
  g.vh = (int)(vol / 2);
  g.nxy = g.nxh * g.ny;
  g.nxyz = g.nxy * g.nz;
  if (layout->even_sites_on_node && (long long)layout->even_sites_on_node != vol / 2) {
    fail(__FILE__, __LINE__, "QPHIX_init: even_sites_on_node disagrees with latsize");
    return QPHIX_FAIL;
  }
  // Reduction scratch: enough partials for one block per 64 sites, 4 values
  // each, and for the multi-RHS kernels (8 sources, one 256-lane block per 32
  // sites, p.Ap and |r|^2 at once): vh / 2 values.
  c.max_blocks = (g.vh + 63) / 64 + 1024;
  c.partials_len = std::max((size_t)4 * c.max_blocks, (size_t)g.vh / 2 + 2048);
  c.partials = (double *)dev_alloc(sizeof(double) * c.partials_len);
  if (!c.partials) return QPHIX_MEM_ERROR;
  HIP_CHECK(hipHostMalloc(&c.pinned, PINNED_BYTES, hipHostMallocDefault));
  c.initialised = true;
  return QPHIX_SUCCESS;
}

static QPHIX_status_t finalize_common() {
  Context &c = g_ctx;
  if (!c.initialised) return QPHIX_SUCCESS;
  HIP_CHECK(hipStreamSynchronize(c.stream));
  host_io_release();
  ws_release(c.partials);
  ws_release(c.ws);
  ws_release(c.ws2);
  {
    KeptBlocks &k = blocks();
    std::lock_guard<std::recursive_mutex> l(k.m);
    shrink_blocks(k, 0);
  }
  if (c.pinned) HIP_CHECK(hipHostFree(c.pinned));
  HIP_CHECK(hipStreamDestroy(c.stream));
  const bool keep_abort = c.abort_on_error;
  const bool keep_sync = c.sync_calls;
  const bool keep_graphs = c.graphs;
  c = Context{};
  c.abort_on_error = keep_abort;
  c.sync_calls = keep_sync;
  c.graphs = keep_graphs;
  return QPHIX_SUCCESS;
}

} // namespace qphix

using namespace qphix;

extern "C" {

// qphix_misc.cpp:427-547 (F and D share the same lattice and device state)
QPHIX_status_t QPHIX_init_F(QPHIX_layout_t *layout) { return init_common(layout); }
QPHIX_status_t QPHIX_init_D(QPHIX_layout_t *layout) { return init_common(layout); }
// qphix_misc.cpp:583-586
QPHIX_status_t QPHIX_init(QPHIX_layout_t *layout) {
  const QPHIX_status_t f = QPHIX_init_F(layout);
  if (f != QPHIX_SUCCESS) return f;  // one report per failed init
  return QPHIX_init_D(layout);
}
QPHIX_status_t QPHIX_finalize_F() { return finalize_common(); }
QPHIX_status_t QPHIX_finalize_D() { return finalize_common(); }
QPHIX_status_t QPHIX_finalize() { return (QPHIX_status_t)(QPHIX_finalize_F() | QPHIX_finalize_D()); }

void QPHIX_MI355X_set_abort_on_error(int on) { g_ctx.abort_on_error = on != 0; }

int QPHIX_MI355X_last_error(char *buf, int len) {
  if (buf && len > 0) {
    std::strncpy(buf, g_last_error, (size_t)len - 1);
    buf[len - 1] = 0;
  }
  return g_error_count;
}

void QPHIX_MI355X_clear_error(void) {
  g_error_count = 0;
  g_last_error[0] = 0;
}

void QPHIX_MI355X_set_sync(int on) { g_ctx.sync_calls = on != 0; }
void QPHIX_MI355X_debug_fail_alloc(int after) { g_fail_alloc_after = after; }
void QPHIX_MI355X_set_fewsums(int mode) { qphix::set_fewsums_mode(mode); }
void QPHIX_MI355X_set_graphs(int on) { g_ctx.graphs = on != 0; }
void QPHIX_MI355X_set_gauge_force_staples(int on) { g_gf_staples = on != 0; }

void QPHIX_MI355X_sync(void) {
  if (g_ctx.initialised) HIP_CHECK(hipStreamSynchronize(g_ctx.stream));
}

void *QPHIX_MI355X_stream(void) { return (void *)g_ctx.stream; }

int QPHIX_MI355X_device_info(int *n_cu, double *hbm_gib) {
  if (!g_ctx.initialised) return 1;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, g_ctx.device) != hipSuccess) return 1;
  if (n_cu) *n_cu = prop.multiProcessorCount;
  if (hbm_gib) *hbm_gib = (double)prop.totalGlobalMem / (1024.0 * 1024.0 * 1024.0);
  return 0;
}

} // extern "C"
