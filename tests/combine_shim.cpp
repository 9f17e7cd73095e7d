// Calls launch::tpcc_combine on buffers of its own (test plumbing: the
// arguments' layout comes from launch.h).
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

// nq queues of lens[q] updates, one after another in srow / sop; cells holds
// nrows rows of TPCC_COLS.  Returns a HIP error, cells / reads / need changed in place.
extern "C" int combine_queues(uint32_t nq, const uint32_t* lens, const uint32_t* srow, const uint32_t* sop, uint32_t nops,
                              const uint64_t* ops, const uint32_t* params, uint64_t nrows, uint64_t* cells,
                              uint64_t* reads, uint32_t* need, uint64_t error) {
  std::vector<uint4> chunks(nq);
  for (uint32_t q = 0, at = 0; q < nq; at += lens[q++]) chunks[q] = make_uint4(at, lens[q], 0u, 0u);
  const uint32_t ctr[launch::COMB_WORDS] = {nq};
  Dev d_chunks, d_ctr, d_srow, d_sop, d_ops, d_params, d_cells, d_reads, d_need, d_error;
  hipError_t e = hipSuccess;
  auto put = [&](Dev& d, const void* p, size_t n) {
    if (e == hipSuccess) e = d.put(p, n);
  };
  put(d_chunks, chunks.data(), nq * sizeof(uint4));
  put(d_ctr, ctr, sizeof ctr);
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
  c.chunk_cap = nq;
  c.chunks = static_cast<uint4*>(d_chunks.p);
  c.ctr = static_cast<uint32_t*>(d_ctr.p);
  c.ops = static_cast<uint64_t*>(d_ops.p);
  c.op_param = static_cast<uint32_t*>(d_params.p);
  c.cells = static_cast<uint64_t*>(d_cells.p);
  c.cols = TPCC_COLS;
  c.reads = static_cast<uint64_t*>(d_reads.p);
  c.need = static_cast<uint32_t*>(d_need.p);
  c.error = static_cast<uint64_t*>(d_error.p);
  e = launch::tpcc_combine(c, static_cast<uint32_t*>(d_srow.p), static_cast<uint32_t*>(d_sop.p), nullptr);
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(cells, d_cells.p, nrows * TPCC_COLS * 8, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(reads, d_reads.p, nops * 8ull, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(need, d_need.p, nops * 4ull, hipMemcpyDeviceToHost);
  return (int)e;
}
