// Host-side launch wrappers for the gfx950 kernels.  Every wrapper enqueues on
// the given stream and returns hipSuccess or the launch error.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../gcctb_common.h"

namespace gcctb {
namespace launch {

// --- execution kernels (one translation unit per scheme family) ---
// G must be 1, 2, 4, 8, 16 or 32; threads = block threads.
hipError_t exec_tpl(bool wait_die, int G, const ExecArgs& a, uint64_t nslots, int threads, bool persist, hipStream_t s);
hipError_t exec_to(int G, const ExecArgs& a, uint64_t nslots, int threads, bool persist, hipStream_t s);
hipError_t exec_mvcc(int G, const ExecArgs& a, uint64_t nslots, int threads, bool persist, hipStream_t s);
hipError_t exec_silo(int G, const ExecArgs& a, uint64_t nslots, int threads, bool persist, hipStream_t s);
hipError_t exec_tictoc(int G, const ExecArgs& a, uint64_t nslots, int threads, bool persist, hipStream_t s);
hipError_t exec_ordered(int G, const ExecArgs& a, uint64_t nslots, int threads, bool persist, hipStream_t s);
// kernel variants (plain form only), any scheme: whole-row mode, the event
// log, or both
hipError_t exec_row(int scheme, int G, const ExecArgs& a, uint64_t nslots, int threads, hipStream_t s);
hipError_t exec_evt(int scheme, int G, const ExecArgs& a, uint64_t nslots, int threads, hipStream_t s);
hipError_t exec_row_evt(int scheme, int G, const ExecArgs& a, uint64_t nslots, int threads, hipStream_t s);
// the latch schemes (slow_*), plain form, column mode: the CC arrays hold a
// 16-byte slot per row (the word, then the latch)
hipError_t exec_latch(int scheme, int G, const ExecArgs& a, uint64_t nslots, int threads, hipStream_t s);
// TPC-C kernels (plain form): every op updates its row in place (tpcc_apply)
hipError_t exec_tpcc(int scheme, int G, const ExecArgs& a, uint64_t nslots, int threads, hipStream_t s);

// --- table / index ---
hipError_t seed_table(uint64_t* cells, uint64_t rows, uint32_t cols, uint64_t seed, hipStream_t s);
// Insert n keys (keys == nullptr: key i) with values (vals == nullptr:
// value i) into a hash index whose nbuckets buckets start all free
// (every u32 IDX_EMPTY).  Keys must be unique and not IDX_EMPTY.
hipError_t index_insert(const uint32_t* keys, const uint32_t* vals, uint64_t n, uint32_t* buckets,
                        uint32_t nbuckets, hipStream_t s);
// rows_out[i] = row of ops[i]'s key (rows_out may be null); also into rows_copy when it is given;
// ids_out[i] = what op_ids(ops, n, id_base) writes, when it is given; with
// id_map, id_map[i] with the op's write flag in bit 31 instead; need[i] =
// NEED_FREE when given; nzero words (at most 256) at `zero` are cleared
hipError_t probe(const IndexView& ix, const uint64_t* ops, uint64_t n, uint32_t* rows_out,
                 hipStream_t s, uint32_t* rows_copy = nullptr, uint32_t* ids_out = nullptr,
                 uint32_t id_base = 0, const uint32_t* id_map = nullptr, uint32_t* need = nullptr,
                 uint64_t* zero = nullptr, uint32_t nzero = 0);

// --- per-op helpers ---
hipError_t op_tx(const uint64_t* tx_off, uint64_t ntx, uint32_t* op_tx, hipStream_t s);
// out[i] = (base + i) | OPID_WRITE if ops[base + i] writes: the values the
// GaccO / GPUTx sorts carry, so later passes read the flag in order.
hipError_t op_ids(const uint64_t* ops, uint64_t n, uint32_t base, uint32_t* out, hipStream_t s);
hipError_t fill_u32(uint32_t* v, uint64_t n, uint32_t x, hipStream_t s);
hipError_t fill_u64(uint64_t* v, uint64_t n, uint64_t x, hipStream_t s);

// --- stable LSD radix sort (8-bit digits) of (key, value) pairs ---
// Sorts bits [0, key_bits) of the keys.  Buffers: keys/vals in, alt buffers of
// the same size; the sorted result ends in (*keys_out, *vals_out), which point
// to one of the two buffer pairs.  tmp must hold radix_sort_tmp_words(n) u32.
// Here and below, nd (when given) is a device word that holds the actual
// element count, at most n.
uint64_t radix_sort_tmp_words(uint64_t n);
hipError_t radix_sort_u32(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, uint64_t n,
                          int key_bits, uint32_t* tmp, uint32_t** keys_out, uint32_t** vals_out,
                          hipStream_t s, const uint32_t* nd = nullptr);
// the same with the positions 0 .. n-1 as values (key_bits > 0): one pass (up to 8
// bits) only reads k0 and ends in (k1, v1)
hipError_t radix_sort_ids(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, uint64_t n, int key_bits,
                          uint32_t* tmp, uint32_t** keys_out, uint32_t** vals_out, hipStream_t s);
hipError_t radix_sort_u64(uint64_t* k0, uint32_t* v0, uint64_t* k1, uint32_t* v1, uint64_t n,
                          int key_bits, uint32_t* tmp, uint64_t** keys_out, uint32_t** vals_out,
                          hipStream_t s, const uint32_t* nd = nullptr);

// --- scans (u32) --- tmp must hold scan_tmp_words(n) u32.
uint64_t scan_tmp_words(uint64_t n);
hipError_t inclusive_max_u32(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* tmp, hipStream_t s);

// --- ordered-execution preprocessing ---
// From accesses sorted by (row, order), sop holding op_ids values: group-start
// flags (p or 0) and, when rowstart is given, row-start flags (p or 0).
hipError_t access_group_flags(const uint32_t* srow, const uint32_t* sop, uint64_t n, uint32_t* flags,
                              hipStream_t s, uint32_t* rowstart = nullptr);
// From accesses sorted by (row, order): key[p] >> rb is the row, val[p] an
// op id (op_ids).  need[op] (NEED_*) of every access that waits for another or
// is waited for (the caller fills need with NEED_FREE first), counters[row] =
// 0 for the rows where that happens.  With comb.min > 0 every row queue of at
// least comb.min accesses is listed for gacco_combine or tpcc_combine, none
// once a launch of the run reported an error.  conflicts (may be
// null): neighbours with equal keys where either writes, added to
// CONFLICT_SLOTS counters 16 words apart.  tmp holds seg_tmp_words(n) u32.
constexpr uint32_t CONFLICT_SLOTS = 16;
uint64_t seg_tmp_words(uint64_t n);
// GaccO's row combiners: what they read, and the lists that seg_turns files
// queues in (ctr: COMB_WORDS u32, zero before).  chunks[i]: {first position,
// length, its summary + 1 (0: the queue's only chunk), 0}; multi[i], queues
// of several chunks: {first position, first summary, chunks, 0}.
struct CombArgs {
  uint32_t min;          // shortest queue to combine (0: none)
  uint32_t whole;        // 1: a queue is one chunk whatever its length
  uint32_t chunk_cap, multi_cap;
  uint4* chunks;
  uint4* multi;
  uint64_t* sums;        // cols values and a mask of the columns written, per chunk
  uint32_t* ctr;
  const uint64_t* ops;
  const uint32_t* op_tx;
  const uint64_t* tx_off;
  const uint32_t* op_param;  // TPC-C
  uint64_t* cells;
  uint32_t cols;
  uint64_t seed;
  uint64_t* reads;
  uint32_t* need;
  unsigned long long* combined;
  const uint64_t* error;   // the run's error word (Metrics::error_flags; 0: none so far)
};
constexpr uint32_t COMB_CHUNKS = 0, COMB_SUMS = 1, COMB_MULTI = 2, COMB_WORDS = 4;
uint64_t comb_chunk_cap(uint64_t nops, uint32_t min);
uint64_t comb_multi_cap(uint64_t nops);
uint64_t comb_sum_words(uint64_t nops, uint32_t cols);
hipError_t seg_turns(const uint32_t* key, const uint32_t* val, uint64_t n, int rb, uint32_t* tmp, uint32_t* need,
                     uint32_t* counters, uint64_t nrows, const CombArgs& comb, uint64_t* conflicts, hipStream_t s,
                     const uint32_t* nd = nullptr);
hipError_t seg_turns64(const uint64_t* key, const uint32_t* val, uint64_t n, int rb, uint32_t* tmp, uint32_t* need,
                       uint32_t* counters, uint64_t nrows, uint64_t* conflicts, hipStream_t s,
                       const uint32_t* nd = nullptr);
// GPUTx one-pass rank (src/gputx.cu:5-27) from accesses sorted by (row, tx),
// val[p] the access's transaction with its write flag in bit 31: rank[tx] =
// max over tx's accesses of the access-group boundaries of their rows up to
// them (the caller zeroes rank and max_rank); max_rank = max.  tx_of (when
// given) maps val[p] without its flag to the transaction.
hipError_t seg_ranks(const uint32_t* row, const uint32_t* val, uint64_t n, uint32_t* tmp, uint64_t nrows,
                     uint32_t* rank, uint32_t* max_rank, hipStream_t s, const uint32_t* tx_of = nullptr,
                     const uint32_t* nd = nullptr);
// The accesses that can meet another one: those of rows that some op of
// ops[0, n) writes, in op order (rows: each op's row, null with a dense index:
// the key).  crow / cval get their rows and op ids (id_base + i, write flag in
// bit 31), *f.count their number, and need[i] = NEED_FREE for every op.  With
// f.crow set, cval gets the access's own index (with the flag) instead, and
// f.crow / f.cop / f.ctx its row, op id and transaction op_tx[i].  f.wmap
// (ord_map_bytes(nrows) bytes) is zero before and after; f.bits holds
// nrows / 32 words, f.flags ord_flag_words(n), tmp radix_sort_tmp_words(n).
struct OrdFilter {
  uint8_t* wmap;
  uint32_t* bits;
  uint64_t* flags;
  uint32_t* count;
  uint32_t* crow;
  uint32_t* cop;
  uint32_t* ctx;
};
uint64_t ord_flag_words(uint64_t n);
uint64_t ord_map_bytes(uint64_t nrows);
hipError_t ord_filter(const IndexView& ix, const uint64_t* ops, const uint32_t* rows, uint64_t n, uint64_t nrows,
                      uint32_t id_base, const uint32_t* op_tx, const OrdFilter& f, uint32_t* tmp, uint32_t* need,
                      uint32_t* crow, uint32_t* cval, hipStream_t s);
// GaccO, persistent form: run each listed row queue in order on the row's
// cells (cols <= 64), store its reads' results, mark its ops need = NEED_DONE
// and add the ops run to *combined.  srow, sop: the sorted accesses.
hipError_t gacco_combine(const CombArgs& c, const uint32_t* srow, const uint32_t* sop, hipStream_t s);
// TPC-C, GaccO: the same for queues of updates (c.whole), one wave per queue.
hipError_t tpcc_combine(const CombArgs& c, const uint32_t* srow, const uint32_t* sop, hipStream_t s);
// Open form, one admitted batch sorted by (row, op) with group starts gstart
// and row starts rstart: need[op] = base[row] + gstart[p] - rstart[p]; then
// row_base_add adds the batch's accesses of each row to base[row].
hipError_t access_need_open(const uint32_t* srow, const uint32_t* sop, const uint32_t* gstart, const uint32_t* rstart,
                            uint64_t n, uint64_t nrows, const uint32_t* base, uint32_t* need, hipStream_t s);
hipError_t row_base_add(const uint32_t* srow, const uint32_t* rstart, uint64_t n, uint64_t nrows, uint32_t* base,
                        hipStream_t s);
// composite key (rows[i] << rank_bits) | rank[tx[i]] for i in [0, n)
hipError_t gtx_exec_keys(const uint32_t* rows, const uint32_t* tx, const uint32_t* rank, uint64_t n, int rank_bits,
                         uint64_t* keys, hipStream_t s, const uint32_t* nd = nullptr);
// the same key cut to 32 bits, for row_bits + rank_bits <= 32
hipError_t gtx_exec_keys32(const uint32_t* rows, const uint32_t* tx, const uint32_t* rank, uint64_t n, int rank_bits,
                           uint32_t* keys, hipStream_t s, const uint32_t* nd = nullptr);
hipError_t rank_hist(const uint32_t* rank, uint64_t ntx, uint32_t nranks, uint32_t* hist, hipStream_t s);

// --- memory-system ceilings (microbench.hip) ---
hipError_t microbench(int which, uint64_t n_words, uint64_t threads_total, uint64_t iters, double* rate,
                      double* ms_out);

// --- hot-writer deferral (persistent form of the non-ordered schemes) ---
// map[slot] = the transaction the slot runs: the transactions that write no
// hot key from slot 0 up, those that do from slot ntx - 1 down (a key is hot
// when at least one transaction in `share` touches it, estimated from about
// DEFER_SAMPLE sampled ops).  cnt holds DEFER_WORDS u32, zero before
// (run_begin): DEFER_BUCKETS sampled counts, then the state words (cnt + DEFER_BUCKETS)[DEFER_ANY] (a
// key was hot) and [DEFER_NHOT] (the number deferred); map holds ntx u32.
constexpr uint32_t DEFER_BUCKETS = 1u << DEFER_BUCKET_BITS;
constexpr uint64_t DEFER_SAMPLE = 16384;
constexpr uint32_t DEFER_ANY = 0, DEFER_NCOLD = 1, DEFER_NHOT = 2;
constexpr uint64_t DEFER_WORDS = DEFER_BUCKETS + 8;
hipError_t defer_order(const uint64_t* tx_off, const uint64_t* ops, uint64_t ntx, uint64_t nops, uint32_t share,
                       uint32_t* cnt, uint32_t* map, hipStream_t s);
// the sampled-count threshold defer_order uses for a hot key
uint32_t defer_threshold(uint64_t ntx, uint64_t nops, uint32_t share);

// --- per-batch state ---
// clear the CC words (and MVCC chain heads) of rows[0, n) at their slots
// (arrays of slot_words(nrows_table) words); latch: the CC array holds two
// words per slot (the word and the row's latch)
hipError_t reset_rows(const uint32_t* rows, uint64_t n, uint64_t nrows_table, uint64_t* cc,
                      uint32_t* vprev, hipStream_t s, bool latch = false);
hipError_t batch_begin(uint64_t* ctrs, hipStream_t s);
// Start of a run: clear the metrics slots (and the deferral's counts, when
// given) and, with counters, do what batch_begin and persist_begin do.
hipError_t run_begin(uint64_t* metrics, uint32_t* defer, uint64_t* ctrs, bool counters, hipStream_t s);
// End of a run: what the host reports of it, written into host memory
// (pinned, read after the stream is waited for).  conflicts, combined and
// defer (the deferral's state words) may be null.
struct RunResult {
  Metrics metrics;  // sums over the slots (error_flags: or, flags alone)
  uint64_t conflicts, combined, deferred;
  uint64_t failed;  // plain form: the launch that reported an error, from 1 (0: none)
};
hipError_t run_end(const Metrics* metrics, const uint64_t* conflicts, const uint64_t* combined, const uint32_t* defer,
                   RunResult* out, hipStream_t s);
// admission state of a persistent launch (slot counter, gates, admission words)
hipError_t persist_begin(uint64_t* ctrs, hipStream_t s);
// *out = the device wall clock (100 MHz), written by a one-block kernel
hipError_t clock_sample(uint64_t* out, hipStream_t s);

}  // namespace launch
}  // namespace gcctb
