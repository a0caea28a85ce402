// Host paths of libhpcgx.so without a GPU: this program defines the HIP
// runtime's functions itself, so the library's own calls land here.  Device
// memory is host memory, kernels do not run.  Launches are counted by name and
// checked as HIP checks them (an empty grid is an error); one may be made to
// fail, and so may one allocation.
//
//   host_path SCENARIO    exits 0 if it holds, else prints what did not
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <string>
#include <vector>

#include "hpcgx.h"

namespace {

constexpr unsigned kHostMallocCoherent = 0x40000000;
constexpr int kOk = 0, kOutOfMemory = 2, kInvalidConfiguration = 9, kNotReady = 600, kLaunchFailure = 719;

struct Dim3 {
  uint32_t x, y, z;
};

// Host stub -> mangled kernel name; the library registers its kernels before
// this program's own objects are made.
std::map<const void *, std::string> &kernels() {
  static std::map<const void *, std::string> k;
  return k;
}
std::map<std::string, int> launched;
int last_error = kOk;
int fail_malloc = 0;          // the coming hipMalloc that fails, counted from 1 (0: none)
std::string fail_launch;      // launches of a kernel whose name holds this fail
int fail_after = 0;           // once so many of them have run
int spmv_diag_one = -1;       // whether the last SpMV took the diagonals from the slot's value
int handle_count = 0;

int failed(int code) { return last_error = code; }
void *handle() { return reinterpret_cast<void *>((uintptr_t)(0x1000 + 16 * ++handle_count)); }

// Finishing kernels on the stream: where each leaves its total, and the total,
// which is the number of the launch.  They end one by one as the host asks
// after the stream, and all of them when it waits for it.
struct Total {
  double *host;
  double value;
};
std::deque<Total> under_way;
double totals = 0;
std::vector<std::pair<char *, size_t>> coherent;  // pinned memory made coherent by name
bool all_coherent = true;                         // totals have only gone to such memory
bool end_one() {
  if (under_way.empty()) return false;
  if (char *p = reinterpret_cast<char *>(under_way.front().host)) {
    bool in = false;
    for (const auto &m : coherent) in = in || (p >= m.first && p < m.first + m.second);
    all_coherent = all_coherent && in;
  }
  if (under_way.front().host) *under_way.front().host = under_way.front().value;
  under_way.pop_front();
  return true;
}

// Launches of kernels whose name holds `part`.
int launches(const char *part) {
  int n = 0;
  for (const auto &k : launched)
    if (k.first.find(part) != std::string::npos) n += k.second;
  return n;
}

}  // namespace

extern "C" {

void **__hipRegisterFatBinary(const void *) { return reinterpret_cast<void **>(handle()); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *, void *, void *, void *,
                           int *) {
  kernels()[stub] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

static struct {
  Dim3 grid, block;
  size_t shared;
  void *stream;
} config;
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) {
  config = {grid, block, shared, stream};
  return kOk;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
  *grid = config.grid;
  *block = config.block;
  *shared = config.shared;
  *stream = config.stream;
  return kOk;
}
int hipLaunchKernel(const void *stub, Dim3 grid, Dim3 block, void **args, size_t, void *) {
  const std::string &name = kernels()[stub];
  if (!grid.x || !grid.y || !grid.z || !block.x || !block.y || !block.z) {
    std::printf("empty launch: %s\n", name.c_str());
    return failed(kInvalidConfiguration);
  }
  if (!fail_launch.empty() && name.find(fail_launch) != std::string::npos && fail_after-- <= 0)
    return failed(kLaunchFailure);
  ++launched[name];
  if (name.find("k_spmvI") != std::string::npos)  // (ci, src, ..): ValSrc is four pointers and diag_one
    spmv_diag_one = *reinterpret_cast<int *>(static_cast<char *>(args[1]) + 4 * sizeof(void *));
  if (name.find("k_finish") != std::string::npos)  // (partials, G, scal, op, slot, host)
    under_way.push_back({*reinterpret_cast<double **>(args[5]), ++totals});
  return kOk;
}

int hipGetLastError() {
  const int e = last_error;
  last_error = kOk;
  return e;
}
const char *hipGetErrorString(int) { return "error"; }

int hipMalloc(void **p, size_t n) {
  if (fail_malloc && --fail_malloc == 0) return failed(kOutOfMemory);
  return (*p = std::calloc(n, 1)) ? kOk : failed(kOutOfMemory);
}
int hipFree(void *p) {
  std::free(p);
  return kOk;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  if (flags & kHostMallocCoherent) coherent.push_back({nullptr, n});
  const int e = hipMalloc(p, n);
  if (flags & kHostMallocCoherent) coherent.back().first = static_cast<char *>(*p);
  return e;
}
int hipHostFree(void *p) { return hipFree(p); }
int hipMemcpy(void *d, const void *s, size_t n, int) {
  std::memcpy(d, s, n);
  return kOk;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *) {
  std::memcpy(d, s, n);
  return kOk;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) {
  std::memset(d, v, n);
  return kOk;
}
int hipGetSymbolAddress(void **p, const void *) { return hipMalloc(p, (size_t)4 << 20); }
int hipFuncSetAttribute(const void *, int, int) { return kOk; }

int hipSetDevice(int) { return kOk; }
int hipStreamCreateWithFlags(void **s, unsigned) {
  *s = handle();
  return kOk;
}
int hipStreamDestroy(void *) { return kOk; }
int hipStreamSynchronize(void *) {
  while (end_one()) {}
  return kOk;
}
int hipStreamQuery(void *) { return end_one() ? kNotReady : kOk; }
int hipEventCreate(void **e) {
  *e = handle();
  return kOk;
}
int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void *) { return kOk; }
int hipEventRecord(void *, void *) { return kOk; }
int hipEventSynchronize(void *) { return kOk; }
int hipEventElapsedTime(float *ms, void *, void *) {
  *ms = 0;
  return kOk;
}
int hipStreamBeginCapture(void *, int) { return kOk; }
int hipStreamEndCapture(void *, void **g) {
  *g = handle();
  return kOk;
}
int hipGraphInstantiate(void **g, void *, void *, void *, size_t) {
  *g = handle();
  return kOk;
}
int hipGraphLaunch(void *, void *) { return kOk; }
int hipGraphDestroy(void *) { return kOk; }
int hipGraphExecDestroy(void *) { return kOk; }

}  // extern "C"

#define CHECK(what)                                          \
  do {                                                       \
    if (!(what)) {                                           \
      std::printf("line %d: not so: %s\n", __LINE__, #what); \
      return 1;                                              \
    }                                                        \
  } while (0)

// Levels with an empty colour block (grids of one plane) above the size that
// one workgroup takes: every call launches what there is and succeeds.
static int one_plane() {
  for (const int flat : {0, 1, 2}) {
    for (const int kappa : {0, 1}) {
      int d[3] = {128, 128, 1};
      std::swap(d[flat], d[2]);
      hpcgx_ctx *c;
      CHECK(hpcgx_create(0, &c) == HPCGX_OK);
      const std::vector<double> k((size_t)128 * 128, 1.0);
      CHECK(hpcgx_problem_generate(c, d[0], d[1], d[2], 1, kappa ? k.data() : nullptr) == HPCGX_OK);
      double *r, *x;
      CHECK(hpcgx_vec_alloc(c, 0, &r) == HPCGX_OK && hpcgx_vec_alloc(c, 0, &x) == HPCGX_OK);
      CHECK(hpcgx_symgs(c, 0, r, x) == HPCGX_OK);
      CHECK(hpcgx_mg(c, 0, r, x) == HPCGX_OK);
      for (const int prec : {HPCGX_PREC_FP32, HPCGX_PREC_FP16}) {
        CHECK(hpcgx_prepare_precision(c, prec) == HPCGX_OK);
        CHECK(hpcgx_mg_mixed(c, prec, r, x) == HPCGX_OK);
      }
      CHECK(launches("k_gs") > 0 && launches("k_tail") == 0);
      CHECK(hpcgx_destroy(c) == HPCGX_OK);
    }
  }
  return 0;
}

// The compact forms of three levels, with each of their allocations failing in
// turn, then a launch: nothing is kept of a failed attempt, the format stays what
// it was, and the next attempt builds every level.
static int forms_after_failure() {
  hpcgx_ctx *c;
  CHECK(hpcgx_create(0, &c) == HPCGX_OK);
  CHECK(hpcgx_set_column_format(c, HPCGX_COLS_EXPLICIT) == HPCGX_OK);
  CHECK(hpcgx_problem_generate(c, 32, 32, 32, 3, nullptr) == HPCGX_OK);
  double *x, *y;
  CHECK(hpcgx_vec_alloc(c, 0, &x) == HPCGX_OK && hpcgx_vec_alloc(c, 0, &y) == HPCGX_OK);
  const double bytes = hpcgx_memory_bytes(c);
  const auto still_explicit = [&] {
    const int before = launches("k_spmvIdddLi0E");
    bool ok = hpcgx_memory_bytes(c) == bytes && hpcgx_spmv(c, 0, x, y) == HPCGX_OK &&
              launches("k_spmvIdddLi0E") == before + 1;
    for (int l = 0; l < 3; ++l) {
      int64_t counts[4];
      ok = ok && hpcgx_level_column_forms(c, l, counts) == HPCGX_OK && !counts[3];
    }
    return ok;
  };
  int failures = 0;
  for (;; ++failures) {
    const int before = launches("k_compact_cols");
    fail_malloc = failures + 1;
    const int rc = hpcgx_set_column_format(c, HPCGX_COLS_COMPACT_ALWAYS);
    if (rc == HPCGX_OK) break;
    CHECK(rc == HPCGX_ENOMEM && fail_malloc == 0);
    CHECK(launches("k_compact_cols") == before);
    CHECK(still_explicit());
  }
  fail_malloc = 0;
  CHECK(failures >= 3);
  CHECK(launches("k_compact_cols") == 3);
  CHECK(hpcgx_destroy(c) == HPCGX_OK);

  CHECK(hpcgx_create(0, &c) == HPCGX_OK);
  CHECK(hpcgx_set_column_format(c, HPCGX_COLS_EXPLICIT) == HPCGX_OK);
  CHECK(hpcgx_problem_generate(c, 32, 32, 32, 3, nullptr) == HPCGX_OK);
  CHECK(hpcgx_vec_alloc(c, 0, &x) == HPCGX_OK && hpcgx_vec_alloc(c, 0, &y) == HPCGX_OK);
  for (const char *kernel : {"k_slot_values", "k_compact_cols", "k_slice_runs"}) {
    fail_launch = kernel;
    CHECK(hpcgx_set_column_format(c, HPCGX_COLS_COMPACT_ALWAYS) == HPCGX_EHIP);
    fail_launch.clear();
    CHECK(still_explicit());
  }
  const int before = launches("k_compact_cols");
  CHECK(hpcgx_set_column_format(c, HPCGX_COLS_COMPACT_ALWAYS) == HPCGX_OK);
  CHECK(launches("k_compact_cols") == before + 3);
  CHECK(hpcgx_destroy(c) == HPCGX_OK);
  return 0;
}

// A solve that fails after its finishing kernel was launched, the total still on
// its way: the next call that asks for one gets its own.
static int total_after_failure() {
  for (const int variant : {HPCGX_CG_FP64, HPCGX_CG_MIXED_FP32, HPCGX_CG_MIXED_FP16}) {
    hpcgx_ctx *c;
    CHECK(hpcgx_create(0, &c) == HPCGX_OK);
    CHECK(hpcgx_problem_generate(c, 16, 16, 16, 3, nullptr) == HPCGX_OK);
    CHECK(hpcgx_prepare_precision(c, HPCGX_PREC_FP32) == HPCGX_OK);
    CHECK(hpcgx_prepare_precision(c, HPCGX_PREC_FP16) == HPCGX_OK);
    double *b, *x, *w, got = 0;
    CHECK(hpcgx_vec_alloc(c, 0, &b) == HPCGX_OK && hpcgx_vec_alloc(c, 0, &x) == HPCGX_OK);
    CHECK(hpcgx_vec_alloc(c, 0, &w) == HPCGX_OK);
    int iters;
    double normr, normr0;
    fail_launch = "k_tail";  // the V-cycle of the second iteration, launched ahead
    fail_after = 1;
    CHECK(hpcgx_cg(c, variant, b, x, 10, 1e-30, 1, &iters, &normr, &normr0, nullptr, nullptr) == HPCGX_EHIP);
    fail_launch.clear();
    CHECK(!under_way.empty());
    CHECK(hpcgx_dot(c, 4096, b, x, &got) == HPCGX_OK);
    CHECK(got == totals);
    CHECK(hpcgx_waxpby_dot(c, 4096, 1.0, b, 2.0, x, w, &got) == HPCGX_OK);
    CHECK(got == totals);
    CHECK(hpcgx_destroy(c) == HPCGX_OK);
  }
  return 0;
}

// The host polls totals while the kernels that write them run: they go to
// memory that was asked to be coherent.
static int totals_coherent() {
  hpcgx_ctx *c;
  CHECK(hpcgx_create(0, &c) == HPCGX_OK);
  CHECK(hpcgx_problem_generate(c, 16, 16, 16, 3, nullptr) == HPCGX_OK);
  double *x, *y, got;
  CHECK(hpcgx_vec_alloc(c, 0, &x) == HPCGX_OK && hpcgx_vec_alloc(c, 0, &y) == HPCGX_OK);
  CHECK(hpcgx_dot(c, 4096, x, y, &got) == HPCGX_OK);
  CHECK(hpcgx_waxpby_dot(c, 4096, 1.0, x, 2.0, y, y, &got) == HPCGX_OK);
  CHECK(hpcgx_dot_noalloc(c, 4096, x, y, &got) == HPCGX_OK);
  int iters;
  double normr, normr0;
  CHECK(hpcgx_cg(c, HPCGX_CG_FP64, x, y, 3, 1e-30, 1, &iters, &normr, &normr0, nullptr, nullptr) == HPCGX_OK);
  CHECK(totals > 3 && all_coherent);
  CHECK(hpcgx_destroy(c) == HPCGX_OK);
  return 0;
}

// r.z is left by the finest level's steps alone: no such kernel is built for others
// (k_gs<VT, XT, ACC, ZK, FINE, CF, VF, GEN, RZ>, k_gs_run<ZK, FINE, VF, RZ>).
static int rz_kernels() {
  int fine = 0;
  for (const auto &k : kernels()) {
    const std::string &n = k.second;
    const bool gs = n.find("4k_gsI") != std::string::npos, run = n.find("8k_gs_runI") != std::string::npos;
    if ((!gs && !run) || n.find("ELb1EEEv") == std::string::npos) continue;  // RZ is the last argument
    CHECK(n.find(gs ? "IdddLin1ELb1E" : "ILin1ELb1E") != std::string::npos);
    ++fine;
  }
  CHECK(fine > 0);
  return 0;
}

// A diagonal that was replaced and could not be looked over is read from the
// value array, where it is, and not from the slot's value.
static int diagonal_after_failure() {
  hpcgx_ctx *c;
  CHECK(hpcgx_create(0, &c) == HPCGX_OK);
  CHECK(hpcgx_problem_generate(c, 16, 16, 16, 2, nullptr) == HPCGX_OK);
  double *x, *y;
  CHECK(hpcgx_vec_alloc(c, 0, &x) == HPCGX_OK && hpcgx_vec_alloc(c, 0, &y) == HPCGX_OK);
  const std::vector<double> diag(4096, 31.0);
  CHECK(hpcgx_spmv(c, 0, x, y) == HPCGX_OK && spmv_diag_one == 1);
  fail_launch = "k_check_diag";
  CHECK(hpcgx_level_set_diagonal(c, 0, diag.data()) == HPCGX_EHIP);
  fail_launch.clear();
  CHECK(hpcgx_spmv(c, 0, x, y) == HPCGX_OK && spmv_diag_one == 0);
  CHECK(hpcgx_level_set_diagonal(c, 0, diag.data()) == HPCGX_OK);
  CHECK(hpcgx_spmv(c, 0, x, y) == HPCGX_OK && spmv_diag_one == 1);
  CHECK(hpcgx_destroy(c) == HPCGX_OK);
  return 0;
}

int main(int argc, char **argv) {
  const std::string s = argc > 1 ? argv[1] : "";
  if (s == "one_plane") return one_plane();
  if (s == "forms_after_failure") return forms_after_failure();
  if (s == "total_after_failure") return total_after_failure();
  if (s == "totals_coherent") return totals_coherent();
  if (s == "rz_kernels") return rz_kernels();
  if (s == "diagonal_after_failure") return diagonal_after_failure();
  std::printf("no scenario: %s\n", s.c_str());
  return 2;
}
