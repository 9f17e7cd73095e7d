// Calls launch::seg_turns and launch::tpcc_combine on buffers of its own (test
// plumbing: the arguments' layout comes from launch.h).
#include <hip/hip_runtime.h>

#include <vector>

#include "../gpu_cc_tb_amd/csrc/device/launch.h"

using namespace gcctb;

namespace {
// a device copy of host words, freed at the end of the call
struct Dev {
  void* p = nullptr;
  hipError_t put(const void* src, size_t bytes) {
    const hipError_t e = hipMalloc(&p, bytes);
    return e != hipSuccess ? e : hipMemcpy(p, src, bytes, hipMemcpyHostToDevice);
  }
  ~Dev() {
    if (p) (void)hipFree(p);
  }
};
}  // namespace

// nops accesses sorted by row (srow, sop) go through the turns and the TPC-C
// combiner, as a batch's do; cells holds nrows rows of TPCC_COLS.  Returns a HIP
// error; cells / reads / need change in place, *listed gets the queues.
extern "C" int combine_queues(const uint32_t* srow, const uint32_t* sop, uint32_t nops, const uint64_t* ops,
                              const uint32_t* params, uint64_t nrows, uint64_t* cells, uint64_t* reads, uint32_t* need,
                              uint64_t error, uint32_t* listed) {
  const std::vector<uint64_t> zero(4096);
  Dev d_chunks, d_ctr, d_srow, d_sop, d_ops, d_params, d_cells, d_reads, d_need, d_error, d_tmp, d_counters;
  hipError_t e = hipSuccess;
  auto put = [&](Dev& d, const void* p, size_t n) {
    if (e == hipSuccess) e = d.put(p, n);
  };
  if (nops > 1024 || nrows > 1024 || launch::seg_tmp_words(nops) * 4 > zero.size() * 8) return (int)hipErrorInvalidValue;
  put(d_chunks, zero.data(), zero.size() * 8);
  put(d_ctr, zero.data(), launch::COMB_WORDS * 4 + 8);
  put(d_tmp, zero.data(), zero.size() * 8);
  put(d_counters, zero.data(), slot_words(nrows) * 4);
  put(d_srow, srow, nops * 4ull);
  put(d_sop, sop, nops * 4ull);
  put(d_ops, ops, nops * 8ull);
  put(d_params, params, nops * 4ull);
  put(d_cells, cells, nrows * TPCC_COLS * 8);
  put(d_reads, reads, nops * 8ull);
  put(d_need, need, nops * 4ull);
  put(d_error, &error, 8);
  if (e != hipSuccess) return (int)e;
  launch::CombArgs c{};
  c.min = 2;
  c.whole = 1;
  c.chunk_cap = (uint32_t)(zero.size() / 2);
  c.chunks = static_cast<uint4*>(d_chunks.p);
  c.ctr = static_cast<uint32_t*>(d_ctr.p);
  c.ops = static_cast<uint64_t*>(d_ops.p);
  c.op_param = static_cast<uint32_t*>(d_params.p);
  c.cells = static_cast<uint64_t*>(d_cells.p);
  c.cols = TPCC_COLS;
  c.reads = static_cast<uint64_t*>(d_reads.p);
  c.need = static_cast<uint32_t*>(d_need.p);
  c.error = static_cast<uint64_t*>(d_error.p);
  auto* rows = static_cast<uint32_t*>(d_srow.p);
  auto* vals = static_cast<uint32_t*>(d_sop.p);
  e = launch::seg_turns(rows, vals, nops, 0, static_cast<uint32_t*>(d_tmp.p), c.need, static_cast<uint32_t*>(d_counters.p),
                        nrows, c, nullptr, nullptr);
  if (e == hipSuccess) e = launch::tpcc_combine(c, rows, vals, nullptr);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(cells, d_cells.p, nrows * TPCC_COLS * 8, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(reads, d_reads.p, nops * 8ull, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(need, d_need.p, nops * 4ull, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(listed, c.ctr + launch::COMB_CHUNKS, 4, hipMemcpyDeviceToHost);
  return (int)e;
}
