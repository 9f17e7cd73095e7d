// The host engine on the CPU: gpu_cc_tb_amd/csrc/host/engine.cpp linked with
// these stand-ins for the HIP runtime and the kernel launchers (launchers that
// no scenario reaches stay undefined).  Device memory is host memory, work is
// done when it is queued, and an allocation or a launch can be made to fail.
// Each scenario prints "ok" or what it found.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <string>
#include <vector>

#include "../gpu_cc_tb_amd/csrc/device/launch.h"
#include "../include/gcctb.h"

namespace {
std::map<void*, size_t> live;  // allocation -> bytes
size_t fail_bytes = 0;         // the next hipMalloc of this size fails
int blocks(size_t bytes) {
  int n = 0;
  for (const auto& b : live) n += b.second == bytes;
  return n;
}
int launched = 0;              // execution launches over some transactions
int fail_launch = 0;           // this one fails
int error_at = 0;              // this one reports an error
int combined = 0;              // batches whose TPC-C queues were applied
bool waited = true;            // the host has waited since the last launch
std::string found;
void expect(bool ok, const char* what) {
  if (!ok && found.empty()) found = what;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) {
  if (n == fail_bytes) {
    fail_bytes = 0;
    return hipErrorOutOfMemory;
  }
  *p = std::calloc(1, n);
  live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  live.erase(p);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::calloc(1, n);
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  *v = 100000;
  return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
  waited = true;
  return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = nullptr;
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipStreamSynchronize(nullptr); }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 1;
  return hipSuccess;
}
}

namespace gcctb {
namespace launch {
hipError_t op_tx(const uint64_t*, uint64_t, uint32_t*, hipStream_t) { return hipSuccess; }
uint64_t scan_tmp_words(uint64_t n) { return n + 64; }
uint64_t radix_sort_tmp_words(uint64_t n) { return n + 1024; }
uint64_t seg_tmp_words(uint64_t n) { return n + 64; }
uint64_t comb_chunk_cap(uint64_t n, uint32_t min) { return n / min + 1; }
uint64_t comb_multi_cap(uint64_t n) { return n / 256 + 1; }
uint64_t comb_sum_words(uint64_t n, uint32_t cols) { return n / 128 * (cols + 1) + 16; }
uint64_t ord_flag_words(uint64_t n) { return n / 64 + 64; }
uint64_t ord_map_bytes(uint64_t rows) { return (rows + 31) / 32 * 32; }
hipError_t seed_table(uint64_t*, uint64_t, uint32_t, uint64_t, hipStream_t) { return hipSuccess; }
hipError_t fill_u32(uint32_t* v, uint64_t n, uint32_t x, hipStream_t) {
  for (uint64_t i = 0; i < n; ++i) v[i] = x;
  return hipSuccess;
}
hipError_t batch_begin(uint64_t*, hipStream_t) { return hipSuccess; }
hipError_t reset_rows(const uint32_t*, uint64_t n, uint64_t, uint64_t*, uint32_t*, hipStream_t, bool) {
  expect(n == 0 || launched, "rows are reset");
  return hipSuccess;
}
hipError_t run_begin(uint64_t* m, uint32_t*, uint64_t*, bool, hipStream_t) {
  std::memset(m, 0, METRIC_SLOTS * METRICS_WORDS * 8);
  return hipSuccess;
}
hipError_t run_end(const Metrics* m, const uint64_t*, const uint64_t*, const uint32_t*, RunResult* out, hipStream_t) {
  *out = RunResult{};
  out->metrics = m[0];
  out->metrics.error_flags &= 0xffffffffu;
  out->failed = m[0].error_flags >> 32;
  return hipSuccess;
}
uint32_t defer_threshold(uint64_t, uint64_t, uint32_t) { return 2; }
hipError_t defer_order(const uint64_t*, const uint64_t*, uint64_t n, uint64_t, uint32_t, uint32_t*, uint32_t*, hipStream_t) {
  expect(n == 0, "transactions are deferred");
  return hipSuccess;
}
// an execution launch commits its transactions
hipError_t exec(const ExecArgs& a, uint64_t n) {
  launched += n != 0;
  if (fail_launch && launched == fail_launch) return hipErrorLaunchFailure;
  waited = false;
  const uint64_t failed = a.metrics->error_flags >> 32;
  if (a.launch_no > 1 && failed != 0 && failed != a.launch_no) return hipSuccess;  // as txn_exec
  if (error_at && launched == error_at) {
    a.metrics->error_flags |= (uint64_t)a.launch_no << 32 | ERR_WATCHDOG;
    return hipSuccess;
  }
  a.metrics->committed += n;
  return hipSuccess;
}
hipError_t exec_tpcc(int, int, const ExecArgs& a, uint64_t n, int, hipStream_t) { return exec(a, n); }
hipError_t probe(const IndexView&, const uint64_t*, uint64_t, uint32_t*, hipStream_t, uint32_t*, uint32_t*, uint32_t,
                 const uint32_t*, uint32_t*, uint64_t*, uint32_t) {
  return hipSuccess;
}
hipError_t radix_sort_u32(uint32_t* k0, uint32_t* v0, uint32_t*, uint32_t*, uint64_t, int, uint32_t*, uint32_t** k,
                          uint32_t** v, hipStream_t, const uint32_t*) {
  *k = k0;
  *v = v0;
  return hipSuccess;
}
hipError_t seg_turns(const uint32_t*, const uint32_t*, uint64_t, int, uint32_t*, uint32_t*, uint32_t*, uint64_t,
                     const CombArgs& c, uint64_t*, hipStream_t, const uint32_t*) {
  combined += c.min && *c.error == 0;  // as k_seg_turns
  return hipSuccess;
}
hipError_t tpcc_combine(const CombArgs&, const uint32_t*, const uint32_t*, hipStream_t) { return hipSuccess; }
hipError_t fill_u64(uint64_t* v, uint64_t n, uint64_t x, hipStream_t) {
  for (uint64_t i = 0; i < n; ++i) v[i] = x;
  return hipSuccess;
}
hipError_t exec_tpl(bool, int, const ExecArgs& a, uint64_t n, int, bool, hipStream_t) { return exec(a, n); }
hipError_t exec_to(int, const ExecArgs& a, uint64_t n, int, bool, hipStream_t) { return exec(a, n); }
hipError_t exec_mvcc(int, const ExecArgs& a, uint64_t n, int, bool, hipStream_t) { return exec(a, n); }
hipError_t exec_silo(int, const ExecArgs& a, uint64_t n, int, bool, hipStream_t) { return exec(a, n); }
hipError_t exec_tictoc(int, const ExecArgs& a, uint64_t n, int, bool, hipStream_t) { return exec(a, n); }
hipError_t exec_ordered(int, const ExecArgs& a, uint64_t n, int, bool, hipStream_t) { return exec(a, n); }
}  // namespace launch
}  // namespace gcctb

namespace {
using namespace gcctb;

gcctb_ctx* make(const char* scheme, uint64_t rows, bool tpcc = false) {
  gcctb_config cfg{};
  cfg.cc_scheme = scheme;
  cfg.rows = rows;
  cfg.cols = tpcc ? TPCC_COLS : 1;
  cfg.tpcc = tpcc;
  cfg.warp_density = 3;
  cfg.block_size = 8;
  cfg.batch_size = 1 << 16;
  gcctb_ctx* c = nullptr;
  expect(gcctb_create(&cfg, &c) == GCCTB_OK, "create");
  expect(gcctb_seed_table(c) == GCCTB_OK, "seed");
  return c;
}

// ntx transactions of one read each
int load(gcctb_ctx* c, uint64_t ntx) {
  std::vector<uint64_t> ops(ntx), off(ntx + 1);
  for (uint64_t i = 0; i < ntx; ++i) ops[i] = make_op((uint32_t)(i % 1000), 0, false);
  for (uint64_t i = 0; i <= ntx; ++i) off[i] = i;
  return gcctb_load_ops(c, ops.data(), off.data(), ntx);
}

// A load whose allocation of the written-row bits, of their count or of the
// row map fails, then the same load again: it returns OK with all of them.
void load_after_failed_alloc(const char* scheme, int which) {
  const uint64_t rows = 3000017, ntx = 1 << 20;  // sizes that no other buffer has
  const size_t bits = (rows + 31) / 32 * 4, map = (rows + 31) / 32 * 32, count = 4;
  gcctb_ctx* c = make(scheme, rows);
  fail_bytes = which == 0 ? map : which == 1 ? bits : count;
  expect(load(c, ntx) == GCCTB_EDEVICE, "the failed allocation is reported");
  expect(load(c, ntx) == GCCTB_OK, "the second load fits");
  expect(blocks(map) == 1, "the row map is there");
  expect(blocks(bits) == 1, "the bits are there");
  expect(blocks(count) == (!std::strcmp(scheme, "gputx") ? 2 : 1), "the count is there");  // (GPUTx: and the highest rank)
  gcctb_destroy(c);
}

// A run after a load that failed (the context's first, or one after a smaller
// load) has no transactions.
void run_after_failed_load(const char* scheme, bool first) {
  const uint64_t ntx = 5003;
  for (const bool persist : {false, true}) {
    gcctb_ctx* c = make(scheme, 1000);
    if (!first) expect(load(c, 100) == GCCTB_OK, "the smaller load");
    fail_bytes = 4 * ntx;
    expect(load(c, ntx) == GCCTB_EDEVICE, "the failed allocation is reported");
    launched = 0;
    gcctb_stats st{};
    expect((persist ? gcctb_run_persistent(c, &st) : gcctb_run_plain(c, &st)) == GCCTB_OK, "the run");
    expect(st.txs == 0 && st.committed == 0 && st.total_ops == 0 && st.batches == (persist ? 1 : 0), "an empty run");
    expect(launched == 0, "nothing is launched");
    gcctb_destroy(c);
  }
}

// A launch that cannot be queued ends the run: the error is reported once the
// batches queued before it have ended, and the next run is whole.
void failed_launch(const char* scheme) {
  gcctb_ctx* c = make(scheme, 1000);
  const uint64_t sizes[4] = {10, 20, 30, 40};
  expect(load(c, 100) == GCCTB_OK, "load");
  expect(gcctb_set_batches(c, sizes, 4) == GCCTB_OK, "batches");
  fail_launch = 3;
  expect(gcctb_run_plain(c, nullptr) == GCCTB_EDEVICE, "the failed launch is reported");
  expect(launched == 3, "the batches after it are not queued");
  expect(waited, "the queued batches have ended");
  fail_launch = launched = 0;
  gcctb_stats st{};
  expect(gcctb_run_plain(c, &st) == GCCTB_OK && st.committed == 100 && st.batches == 4, "the next run");
  gcctb_destroy(c);
}

// TPC-C under GaccO, four batches, the second reports an error: the queues of
// the two behind it are not applied; the next run is whole.
void tpcc_error() {
  gcctb_ctx* c = make("gacco", 1000, true);
  const uint64_t sizes[4] = {10, 20, 30, 40};
  expect(load(c, 100) == GCCTB_OK, "load");
  const std::vector<uint32_t> params(100);
  expect(gcctb_load_params(c, params.data(), 100) == GCCTB_OK, "parameters");
  expect(gcctb_set_batches(c, sizes, 4) == GCCTB_OK, "batches");
  error_at = 2;
  gcctb_stats st{};
  expect(gcctb_run_plain(c, &st) == GCCTB_EKERNEL && st.committed == 10, "the error is reported");
  expect(st.batches == 2, "the count ends at the launch that reported it");
  expect(combined == 2, "the queues behind the error are left alone");
  combined = launched = error_at = 0;
  expect(gcctb_run_plain(c, &st) == GCCTB_OK && st.committed == 100 && st.batches == 4 && combined == 4, "the next run");
  gcctb_destroy(c);
}
}  // namespace

int main(int argc, char** argv) {
  if (argc < 2) return 2;
  const std::string what = argv[1];
  const char* scheme = argc > 2 ? argv[2] : "";
  if (what == "alloc") load_after_failed_alloc(scheme, std::atoi(argv[3]));
  if (what == "run") run_after_failed_load(scheme, !std::strcmp(argv[3], "first"));
  if (what == "launch") failed_launch(scheme);
  if (what == "tpcc") tpcc_error();
  std::printf("%s\n", found.empty() ? "ok" : found.c_str());
  return found.empty() ? 0 : 1;
}
