// Preprocessing and maintenance kernels for gfx950: table seeding, hash-index
// construction and probing, a stable LSD radix sort, scans, and the
// GaccO / GPUTx access-order passes that replace the reference's Thrust calls
// (include/gacco.cuh:307-336, include/gputx.cuh:252-281).
#include <cstddef>
#include <hip/hip_runtime.h>
#include <algorithm>
#include <stdint.h>
#include "dev_util.h"
#include "launch.h"

namespace gcctb {
namespace {

constexpr int BT = 256;  // threads per block for the streaming kernels

inline unsigned grid_for(uint64_t n, int per_block) {
  uint64_t g = (n + per_block - 1) / per_block;
  if (g == 0) g = 1;
  if (g > 0x7fffffffull) g = 0x7fffffffull;
  return (unsigned)g;
}
inline unsigned grid_stride_blocks(uint64_t n) {
  uint64_t g = (n + BT - 1) / BT;
  if (g > 65536 * 4) g = 65536 * 4;
  if (g == 0) g = 1;
  return (unsigned)g;
}

// Kernels that end in an atomic on one address run at most REDUCE_BLOCKS
// blocks and combine their waves in LDS first: one address sustains only
// ~1e8 atomics/s, so one atomic per wave of a 16M-element grid costs ~3 ms.
constexpr unsigned REDUCE_BLOCKS = 2048;
inline unsigned reduce_blocks(uint64_t n) {
  const unsigned g = grid_stride_blocks(n);
  return g < REDUCE_BLOCKS ? g : REDUCE_BLOCKS;
}
// Block-wide sum (Max = false) or max (Max = true) of one value per thread;
// the result is valid in thread 0.  Every thread of the block must call it.
template <bool Max>
__device__ __forceinline__ uint64_t block_reduce_u64(uint64_t v) {
  __shared__ uint64_t part[BT / 64];
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    const uint64_t o = dev::shfl_xor64(v, m);
    v = Max ? (o > v ? o : v) : v + o;
  }
  if (dev::lane_id() == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    v = part[0];
#pragma unroll
    for (int w = 1; w < BT / 64; ++w) v = Max ? (part[w] > v ? part[w] : v) : v + part[w];
  }
  return v;
}

__global__ void k_seed_table(uint64_t* cells, uint64_t rows, uint32_t cols, uint64_t seed) {
  const uint64_t n = rows * cols;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t r = i / cols;
    cells[i] = cell_init(seed, r, (uint32_t)(i - r * cols), cols);
  }
}

// Hash index build: each key takes the first free slot along its bucket
// sequence (CAS on the key word; a slot never frees again).  The table has
// about twice the slots it needs, so the sequence is short; it is bounded by
// nbuckets in any case.
__global__ void k_index_insert(const uint32_t* keys, const uint32_t* vals, uint64_t n, uint32_t* buckets,
                               uint32_t nbuckets) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t key = keys ? keys[i] : (uint32_t)i;
    const uint32_t val = vals ? vals[i] : (uint32_t)i;
    uint32_t b = idx_bucket(key, nbuckets);
    for (uint32_t step = 0; step < nbuckets; ++step) {
      uint32_t* bk = buckets + (size_t)b * (2 * IDX_SLOTS);
      int s = 0;
      while (s < IDX_SLOTS && atomicCAS(bk + s, IDX_EMPTY, key) != IDX_EMPTY) ++s;
      if (s < IDX_SLOTS) {
        bk[IDX_SLOTS + s] = val;
        break;
      }
      b = b + 1 == nbuckets ? 0u : b + 1;
    }
  }
}

// Quad (4 consecutive lanes) primitives over DPP quad permutes; every lane
// of the quad must be active.
template <int J>
__device__ __forceinline__ uint32_t quad_get(uint32_t v) {  // lane J's value
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, J * 0x55, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t quad_sum(uint32_t v) {
  v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, false);  // lanes 1,0,3,2
  v += (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, false);  // lanes 2,3,0,1
  return v;
}
__device__ __forceinline__ int quad_max(int v) {
  int o = __builtin_amdgcn_mov_dpp(v, 0xb1, 0xf, 0xf, false);
  v = o > v ? o : v;
  o = __builtin_amdgcn_mov_dpp(v, 0x4e, 0xf, 0xf, false);
  return o > v ? o : v;
}

// One bucket step of a quad-cooperative lookup: lane q holds the q-th 16
// bytes of the bucket (keys 0-3, keys 4-7, values 0-3, values 4-7).  Sets
// *val and returns true on a hit; *free_slot tells whether the bucket has a
// free slot (then the key is absent).
__device__ __forceinline__ bool quad_bucket_match(const uint4& w, uint32_t key, uint32_t q, uint32_t* val,
                                                  bool* free_slot) {
  const bool keys_here = q < 2;
  int h = -1;
  h = keys_here && w.x == key ? (int)q * 4 : h;
  h = keys_here && w.y == key ? (int)q * 4 + 1 : h;
  h = keys_here && w.z == key ? (int)q * 4 + 2 : h;
  h = keys_here && w.w == key ? (int)q * 4 + 3 : h;
  const int fr = keys_here && (w.x == IDX_EMPTY || w.y == IDX_EMPTY || w.z == IDX_EMPTY || w.w == IDX_EMPTY);
  h = quad_max(h);
  *free_slot = quad_max(fr) != 0;
  // the value of slot h sits in lane 2 + h / 4, component h % 4
  const uint32_t comp = (h & 3) == 0 ? w.x : (h & 3) == 1 ? w.y : (h & 3) == 2 ? w.z : w.w;
  const uint32_t from2 = quad_get<2>(comp), from3 = quad_get<3>(comp);
  *val = (h >> 2) ? from3 : from2;
  return h >= 0;
}

// Index probe (Find, include/index.cuh:74-91, over the hash index of
// dev::index_find).  A quad walks four probes at once: lane q loads op p0+q
// (a wave loads 64 consecutive ops), the quad shares the four keys, and lane
// q reads the q-th 16 bytes of each probe's home bucket, so one load
// instruction covers one line per probe and the four buckets are read at
// once.  A probe whose bucket is full without the key goes on bucket by
// bucket, the quad together.  A dense index (keys 0 .. length-1 on rows of
// the same number) maps each key to itself and reads no bucket.
// ids_out[i] (optional): the op's id (id_base + i), or id_map[i] when given,
// with the op's write flag in bit 31
// need[i] (optional) = NEED_FREE, and nzero words at `zero` are cleared: the
// ordered schemes' preparation starts here, and each fill of its own cost a
// launch per batch (16,384 TPC-C orders: 6 us and two launches of 17;
// 16.8 M ops: 81 -> 65 us).
__global__ __launch_bounds__(256) void k_probe(IndexView ix, const uint64_t* ops, uint64_t n, uint32_t* rows_out,
                                               uint32_t* rows_copy, uint32_t* ids_out, uint32_t id_base,
                                               const uint32_t* id_map, uint32_t* need, uint64_t* zero, uint32_t nzero) {
  if (blockIdx.x == 0 && threadIdx.x < nzero) zero[threadIdx.x] = 0;
  if (ix.dense) {  // direct addressing: no bucket to read
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
      const uint64_t op = ops[i];
      const uint32_t r = idx_dense_find(op_key(op), ix.length);
      if (rows_out) rows_out[i] = r;
      if (rows_copy) rows_copy[i] = r;
      if (ids_out) ids_out[i] = (id_map ? id_map[i] : id_base + (uint32_t)i) | (op_is_write(op) ? OPID_WRITE : 0u);
      if (need) need[i] = NEED_FREE;
    }
    return;
  }
  const uint32_t q = threadIdx.x & 3u;
  const uint4* bkt = reinterpret_cast<const uint4*>(ix.buckets);
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;  // a multiple of 4
  for (uint64_t p0 = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) & ~3ull; p0 < n; p0 += stride) {
    const uint64_t mine = p0 + q;
    const uint64_t myop = mine < n ? ops[mine] : 0ull;
    const uint32_t mykey = mine < n ? op_key(myop) : IDX_EMPTY;
    const uint32_t key[4] = {quad_get<0>(mykey), quad_get<1>(mykey), quad_get<2>(mykey), quad_get<3>(mykey)};
    uint32_t b[4];
    uint4 w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = idx_bucket(key[j], ix.nbuckets);
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = bkt[(size_t)b[j] * 4 + q];
    uint32_t res[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint32_t r = IDX_MISS;
      if (key[j] != IDX_EMPTY) {  // the reserved key is never stored
        uint4 cur = w[j];
        uint32_t bb = b[j];
        for (uint32_t step = 1;; ++step) {
          uint32_t val;
          bool free_slot;
          if (quad_bucket_match(cur, key[j], q, &val, &free_slot)) {
            r = val;
            break;
          }
          if (free_slot || step >= ix.nbuckets) break;
          bb = bb + 1 == ix.nbuckets ? 0u : bb + 1;
          cur = bkt[(size_t)bb * 4 + q];
        }
      }
      res[j] = r;
    }
    const uint32_t r = q == 0 ? res[0] : q == 1 ? res[1] : q == 2 ? res[2] : res[3];
    if (mine < n) {
      if (rows_out) rows_out[mine] = r;
      if (rows_copy) rows_copy[mine] = r;
      if (ids_out)
        ids_out[mine] = (id_map ? id_map[mine] : id_base + (uint32_t)mine) | (op_is_write(myop) ? OPID_WRITE : 0u);
      if (need) need[mine] = NEED_FREE;
    }
  }
}

__global__ void k_op_tx(const uint64_t* tx_off, uint64_t ntx, uint32_t* op_tx) {
  for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < ntx;
       t += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t b = tx_off[t], e = tx_off[t + 1];
    for (uint64_t i = b; i < e; ++i) op_tx[i] = (uint32_t)t;
  }
}
// Op ids for the GaccO / GPUTx sorts: base + i with the op's write flag in
// bit 31, so the passes over the sorted order read it without a random load.
__global__ void k_op_ids(const uint64_t* ops, uint64_t n, uint32_t base, uint32_t* out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    out[i] = (base + (uint32_t)i) | (op_is_write(ops[base + i]) ? OPID_WRITE : 0u);
}
__global__ void k_fill32(uint32_t* v, uint64_t n, uint32_t x) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    v[i] = x;
}
__global__ void k_fill64(uint64_t* v, uint64_t n, uint64_t x) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    v[i] = x;
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort, three launches per pass: per-tile digit histograms,
// the scan of each digit's row of the [digit][tile] matrix (one block per
// digit), then the scatter, whose blocks scan the 256 digit totals
// themselves (two launches for short inputs, RS_OWN_COUNTS).  The key bits are
// split evenly over ceil(bits / 8) passes (20 bits: 7 + 7 + 6), which shortens
// the per-item ballot loop and lengthens each digit's run.  A tile is 256 x
// RS_ITEMS elements; wave w of the block holds tile elements [w*RS_WSPAN,
// (w+1)*RS_WSPAN), lane-minor, so (wave, item, lane) order is input order.  The
// scatter ranks every element within its digit (ballots inside a wave, a
// per-wave LDS counter across its items, a prefix over waves), sorts the tile in
// LDS, and writes it out digit run by digit run, so consecutive lanes store to
// consecutive addresses.
// Bound: the stores of the digit runs (a pass over 2^24 u32 pairs moves 335
// MB in about 120 us, 2.8 TB/s) and, below 2^20 pairs, launch latency (about
// 4 us each).  Sort of u32 pairs by 24 bits against 5 launches a pass on
// 4,096-element tiles: 2^24 pairs 370 -> 368 us, 2^20 90 -> 73 us, 180,000 80 ->
// 39 us (with the scan's launch).
// ---------------------------------------------------------------------------
constexpr int RS_BT = 256;
constexpr int RS_WAVES = RS_BT / 64;
// Short inputs do without the scan's launch: the scatter's blocks read the
// whole matrix, laid out [tile][digit] then, with RS_OWN_LOADS 16-byte loads
// per thread, all in flight at once.  That costs them 1 to 4 us, growing with
// the matrix, against the launch's 4.  Sort of u32 pairs with / without the
// scan's launch, 24 loads: 16,384 pairs by 21 bits 34.5 -> 30.3 us, 65,536
// 34.9 -> 31.5, 131,072 35.9 -> 33.0, 180,000 (22,528 counts) 37.4 -> 33.8; by
// 24 bits 65,536 (16,384 counts) 36.8 -> 31.9.  In two rounds of 16 loads the
// gain ends there: 131,072 by 24 bits (32,768 counts) 38.0 -> 37.6, 262,144 by
// 21 bits (32,768) 38.3 -> 38.6, 262,144 by 24 bits (65,536) 43.5 -> 47.8.
constexpr int RS_OWN_LOADS = 24;
constexpr uint64_t RS_OWN_COUNTS = (uint64_t)RS_OWN_LOADS * 4 * RS_BT;
constexpr int RS_OWN_WIDTH = 5;  // digits of fewer bits would leave long sums to few threads

template <class KT, int RS_ITEMS>
__global__ __launch_bounds__(RS_BT) void k_rs_hist(const KT* keys, uint64_t n, int shift, uint32_t dmask,
                                                   uint32_t* hist, uint32_t nb, const uint32_t* nd, int by_tile) {
  __shared__ uint32_t h[256];
  constexpr int RS_TILE = RS_BT * RS_ITEMS;
  if (nd) n = *nd;
  h[threadIdx.x] = 0;
  const uint64_t base = (uint64_t)blockIdx.x * RS_TILE;
  if (base >= n) return;
  uint32_t d[RS_ITEMS];
#pragma unroll
  for (int i = 0; i < RS_ITEMS; ++i) {
    const uint64_t e = base + (uint64_t)i * RS_BT + threadIdx.x;
    d[i] = e < n ? (uint32_t)(keys[e] >> shift) & dmask : 256u;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RS_ITEMS; ++i)
    if (d[i] < 256u) atomicAdd(&h[d[i]], 1u);
  __syncthreads();
  if (by_tile) {  // [tile][digit], read by the scatter itself
    if (threadIdx.x <= dmask) hist[(uint64_t)blockIdx.x * (dmask + 1) + threadIdx.x] = h[threadIdx.x];
  } else if (threadIdx.x <= dmask) {
    hist[(uint64_t)threadIdx.x * nb + blockIdx.x] = h[threadIdx.x];
    if (base + RS_TILE >= n)  // the last tile also clears up to the next whole 16-byte load
      for (uint32_t b = blockIdx.x + 1; b & 3u; ++b) hist[(uint64_t)threadIdx.x * nb + b] = 0;
  }
}

// Columns of a row of the [digit][tile] matrix: padded to whole 16-byte loads.
inline uint32_t rs_stride(uint64_t nb) { return (uint32_t)((nb + 3) & ~3ull); }

// offs[d][0..nb) <- exclusive scan of itself, totals[d] <- its sum; block d.
// A thread takes 4 consecutive entries of each 1,024; the loads of 4,096
// entries (16.8M elements) are issued before the first is used.
__global__ __launch_bounds__(RS_BT) void k_rs_rowscan(uint32_t* offs, uint32_t nb, uint32_t* totals, uint32_t tile,
                                                      const uint32_t* nd) {
  constexpr int CH = 4;  // chunks of 4 * RS_BT entries per step
  __shared__ uint32_t wsum[2][RS_WAVES];
  uint4* row = reinterpret_cast<uint4*>(offs + (uint64_t)blockIdx.x * nb);
  const uint32_t t = threadIdx.x, lane = dev::lane_id(), wave = t / 64;
  const uint32_t n4 = nd ? ((*nd + tile - 1) / tile + 3) / 4 : nb / 4;
  uint32_t carry = 0;
  int buf = 0;
  for (uint32_t b0 = 0; b0 < n4; b0 += CH * RS_BT) {
    uint4 v[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const uint32_t i = b0 + c * RS_BT + t;
      v[c] = i < n4 ? row[i] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (b0 + c * RS_BT >= n4) break;  // the same for the whole block
      const uint32_t mine = v[c].x + v[c].y + v[c].z + v[c].w;
      uint32_t x = mine;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)x, d, 64);
        if (lane >= (uint32_t)d) x += o;
      }
      if (lane == 63) wsum[buf][wave] = x;
      __syncthreads();  // one per chunk: the two halves of wsum alternate
      uint32_t p = carry + x - mine;
#pragma unroll
      for (uint32_t w = 0; w < RS_WAVES; ++w) {
        const uint32_t q = wsum[buf][w];
        p += w < wave ? q : 0u;
        carry += q;
      }
      buf ^= 1;
      const uint32_t i = b0 + c * RS_BT + t;
      if (i < n4) row[i] = make_uint4(p, p + v[c].x, p + v[c].x + v[c].y, p + v[c].x + v[c].y + v[c].z);
    }
  }
  if (t == 0) totals[blockIdx.x] = carry;
}

// offs[d * nb + b]: where tile b's first element of digit d goes within the
// digit, totals[d] the elements of digit d; the digit is the `width` bits of
// the key from `shift` up.  OWN_SCAN: offs is the unscanned [tile][digit]
// matrix (16-byte rows) and totals is unused; the block adds the columns up.
template <class KT, int RS_ITEMS, bool OWN_SCAN>
__global__ __launch_bounds__(RS_BT) void k_rs_scatter(const KT* kin, const uint32_t* vin, KT* kout,
                                                      uint32_t* vout, uint64_t n, int shift, int width,
                                                      const uint32_t* offs, uint32_t nb, const uint32_t* totals,
                                                      const uint32_t* nd) {
  constexpr int RS_TILE = RS_BT * RS_ITEMS, RS_WSPAN = RS_ITEMS * 64;
  __shared__ KT skey[RS_TILE];
  __shared__ uint32_t sval[RS_TILE];
  __shared__ uint32_t wcnt[RS_WAVES][256];  // digit counts per wave, then each wave's start in the digit
  __shared__ uint32_t dstart[256];          // tile-local start of each digit
  __shared__ uint32_t gbase[256];           // global start of each digit's run from this tile
  __shared__ uint32_t wsum[RS_WAVES], wtot[RS_WAVES];
  const uint32_t dmask = (1u << width) - 1u;
  const uint32_t t = threadIdx.x, lane = dev::lane_id(), wave = t / 64;
  const uint64_t base = (uint64_t)blockIdx.x * RS_TILE;
  if (nd) n = *nd;
  if (base >= n) return;
  const uint32_t cnt = n - base < (uint64_t)RS_TILE ? (uint32_t)(n - base) : (uint32_t)RS_TILE;
#pragma unroll
  for (int w = 0; w < RS_WAVES; ++w) wcnt[w][t] = 0;
  // counts of four digits in the tiles before this one, and in all of them
  uint4 before = make_uint4(0, 0, 0, 0), every = before;
  if constexpr (OWN_SCAN) {
    const uint4* m = reinterpret_cast<const uint4*>(offs);
    const int qbits = width - 2;  // a row is 2^qbits loads; the thread's column is the same in every row it reads
    const uint32_t cells = (uint32_t)((n + RS_TILE - 1) / RS_TILE) << qbits;
    uint4 c[RS_OWN_LOADS];
#pragma unroll
    for (int i = 0; i < RS_OWN_LOADS; ++i) {
      const uint32_t j = i * RS_BT + t;
      c[i] = j < cells ? m[j] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < RS_OWN_LOADS; ++i) {
      const uint32_t f = (i * RS_BT + t) >> qbits < blockIdx.x ? ~0u : 0u;
      before.x += c[i].x & f, before.y += c[i].y & f, before.z += c[i].z & f, before.w += c[i].w & f;
      every.x += c[i].x, every.y += c[i].y, every.z += c[i].z, every.w += c[i].w;
    }
  }
  KT k[RS_ITEMS];
  uint32_t v[RS_ITEMS];
#pragma unroll
  for (int i = 0; i < RS_ITEMS; ++i) {
    const uint32_t e = wave * RS_WSPAN + i * 64 + lane;
    k[i] = e < cnt ? kin[base + e] : (KT)0;
    v[i] = e >= cnt ? 0u : vin ? vin[base + e] : (uint32_t)(base + e);  // no values: the positions
  }
  __syncthreads();
  // rank within (wave, digit): earlier items of the wave, then lower lanes
  uint32_t r[RS_ITEMS];
#pragma unroll
  for (int i = 0; i < RS_ITEMS; ++i) {
    const bool valid = wave * RS_WSPAN + i * 64 + lane < cnt;
    const uint32_t d = (uint32_t)(k[i] >> shift) & dmask;
    const uint64_t act = dev::ballot(valid);
    uint32_t plo = (uint32_t)act, phi = (uint32_t)(act >> 32);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      if (b >= width) break;
      const uint64_t bb = dev::ballot((d >> b) & 1u);
      const uint32_t m = (uint32_t)((int32_t)(d << (31 - b)) >> 31);  // all ones where the bit is set
      plo &= ~((uint32_t)bb ^ m);
      phi &= ~((uint32_t)(bb >> 32) ^ m);
    }
    const uint64_t peers = plo | ((uint64_t)phi << 32);
    const uint32_t below = __builtin_amdgcn_mbcnt_hi(phi, __builtin_amdgcn_mbcnt_lo(plo, 0u));
    uint32_t old = 0;
    if (valid && below == 0) old = atomicAdd(&wcnt[wave][d], (uint32_t)__popcll(peers));
    const int leader = peers ? __ffsll((unsigned long long)peers) - 1 : (int)lane;
    r[i] = (uint32_t)__shfl((int)old, leader, 64) + below;
  }
  __syncthreads();
  // digit t: each wave's start within the digit, the digit's tile total, and
  // the tile-local start of the digit (exclusive scan over digits)
  uint32_t tot = 0;
#pragma unroll
  for (int w = 0; w < RS_WAVES; ++w) {
    const uint32_t c = wcnt[w][t];
    wcnt[w][t] = tot;
    tot += c;
  }
  uint32_t all = 0, in_digit = 0;
  if constexpr (OWN_SCAN) {
    __shared__ uint4 part[2][RS_BT];
    part[0][t] = before;
    part[1][t] = every;
    __syncthreads();
    if (t <= dmask)  // column t / 4 was added up by every 2^(width-2)-th thread
      for (uint32_t j = t; j < 4 * RS_BT; j += dmask + 1) {
        in_digit += reinterpret_cast<const uint32_t*>(part[0])[j];
        all += reinterpret_cast<const uint32_t*>(part[1])[j];
      }
  } else if (t <= dmask) {
    all = totals[t];
    in_digit = offs[(uint64_t)t * nb + blockIdx.x];
  }
  uint32_t x = tot, y = all;
#pragma unroll
  for (int dd = 1; dd < 64; dd <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)x, dd, 64);
    const uint32_t q = (uint32_t)__shfl_up((int)y, dd, 64);
    if (lane >= (uint32_t)dd) {
      x += o;
      y += q;
    }
  }
  if (lane == 63) {
    wsum[wave] = x;
    wtot[wave] = y;
  }
  __syncthreads();
  uint32_t carry = 0, gcarry = 0;
  for (uint32_t w = 0; w < wave; ++w) {
    carry += wsum[w];
    gcarry += wtot[w];
  }
  dstart[t] = carry + x - tot;
  gbase[t] = gcarry + y - all + in_digit;  // the digit's start, then this tile's place in it
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RS_ITEMS; ++i) {
    if (wave * RS_WSPAN + i * 64 + lane < cnt) {
      const uint32_t d = (uint32_t)(k[i] >> shift) & dmask;
      const uint32_t lp = dstart[d] + wcnt[wave][d] + r[i];
      skey[lp] = k[i];
      sval[lp] = v[i];
    }
  }
  __syncthreads();
  for (uint32_t j = t; j < cnt; j += RS_BT) {
    const KT key = skey[j];
    const uint32_t d = (uint32_t)(key >> shift) & dmask;
    const uint32_t pos = gbase[d] + (j - dstart[d]);
    if (pos < n) {  // always true when the counts agree; keeps a logic error off foreign memory
      kout[pos] = key;
      vout[pos] = sval[j];
    }
  }
}

// ---------------------------------------------------------------------------
// Inclusive scans over u32 (max).  Three kernels: block totals, a single-block
// scan of the totals, and the block-local scan with its carry-in.
// ---------------------------------------------------------------------------
constexpr int SC_BT = 256;
constexpr int SC_ITEMS = 16;
constexpr int SC_TILE = SC_BT * SC_ITEMS;

struct OpMax {
  static __device__ __forceinline__ uint32_t id() { return 0u; }
  static __device__ __forceinline__ uint32_t f(uint32_t a, uint32_t b) { return a > b ? a : b; }
};

// inclusive scan across the block of one value per thread; returns inclusive,
// writes the block total to *total.
template <class Op>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t wsum[SC_BT / 64];
  const uint32_t lane = dev::lane_id(), wave = threadIdx.x / 64;
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)x, d, 64);
    if (lane >= (uint32_t)d) x = Op::f(o, x);
  }
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  uint32_t carry = Op::id();
  for (uint32_t w = 0; w < wave; ++w) carry = Op::f(carry, wsum[w]);
  uint32_t t = Op::id();
  for (int w = 0; w < SC_BT / 64; ++w) t = Op::f(t, wsum[w]);
  *total = t;
  __syncthreads();
  return Op::f(carry, x);
}

// Tile totals.  The operators are commutative, so the tile is read striped
// across the block (element i * SC_BT + t by thread t: every load coalesced).
template <class Op>
__global__ __launch_bounds__(SC_BT) void k_scan_reduce(const uint32_t* in, uint64_t n, uint32_t* sums) {
  const uint64_t base = (uint64_t)blockIdx.x * SC_TILE + threadIdx.x;
  uint32_t acc = Op::id();
#pragma unroll
  for (int i = 0; i < SC_ITEMS; ++i) {
    const uint64_t e = base + (uint64_t)i * SC_BT;
    acc = Op::f(acc, e < n ? in[e] : Op::id());
  }
  uint32_t total;
  block_scan<Op>(acc, &total);
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}
// exclusive scan of sums[0..nb) in place (single block)
template <class Op>
__global__ __launch_bounds__(SC_BT) void k_scan_top(uint32_t* sums, uint32_t nb) {
  __shared__ uint32_t tincl[SC_BT];
  const uint32_t per = (nb + SC_BT - 1) / SC_BT;
  const uint32_t b = threadIdx.x * per;
  uint32_t acc = Op::id();
  for (uint32_t i = 0; i < per; ++i)
    if (b + i < nb) acc = Op::f(acc, sums[b + i]);
  uint32_t total;
  const uint32_t incl = block_scan<Op>(acc, &total);
  tincl[threadIdx.x] = incl;
  __syncthreads();
  uint32_t c = threadIdx.x == 0 ? Op::id() : tincl[threadIdx.x - 1];
  for (uint32_t i = 0; i < per; ++i) {
    if (b + i < nb) {
      const uint32_t v = sums[b + i];
      sums[b + i] = c;
      c = Op::f(c, v);
    }
  }
}
// Tile scans.  The tile moves between global memory and LDS striped across
// the block (coalesced); thread t scans its SC_ITEMS consecutive elements out
// of LDS.  Element j sits at LDS word j + j / 16, so the 16 consecutive words
// of thread t start at 17 t and a wave's reads fall in distinct banks.  The
// whole tile is loaded before any of it is stored, so in may equal out.
template <class Op>
__global__ __launch_bounds__(SC_BT) void k_scan_down(const uint32_t* in, uint32_t* out, uint64_t n,
                                                     const uint32_t* sums) {
  static_assert(SC_ITEMS == 16, "the LDS padding assumes 16 items per thread");
  __shared__ uint32_t tile[SC_TILE + SC_TILE / 16];
  __shared__ uint32_t tincl[SC_BT];
  const uint32_t t = threadIdx.x;
  const uint64_t base = (uint64_t)blockIdx.x * SC_TILE;
#pragma unroll
  for (int i = 0; i < SC_ITEMS; ++i) {
    const uint32_t j = (uint32_t)i * SC_BT + t;
    tile[j + (j >> 4)] = base + j < n ? in[base + j] : Op::id();
  }
  __syncthreads();
  uint32_t vals[SC_ITEMS];
  uint32_t acc = Op::id();
#pragma unroll
  for (int i = 0; i < SC_ITEMS; ++i) {
    vals[i] = tile[t * 17 + i];
    acc = Op::f(acc, vals[i]);
  }
  uint32_t total;
  const uint32_t incl = block_scan<Op>(acc, &total);
  // exclusive prefix for this thread = block carry + (incl of previous threads)
  tincl[t] = incl;
  __syncthreads();
  uint32_t c = Op::f(sums[blockIdx.x], t == 0 ? Op::id() : tincl[t - 1]);
#pragma unroll
  for (int i = 0; i < SC_ITEMS; ++i) {
    c = Op::f(c, vals[i]);
    tile[t * 17 + i] = c;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < SC_ITEMS; ++i) {
    const uint32_t j = (uint32_t)i * SC_BT + t;
    if (base + j < n) out[base + j] = tile[j + (j >> 4)];
  }
}

template <class Op>
hipError_t scan_impl(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* tmp, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const uint64_t nb = (n + SC_TILE - 1) / SC_TILE;
  hipLaunchKernelGGL((k_scan_reduce<Op>), dim3((unsigned)nb), dim3(SC_BT), 0, s, in, n, tmp);
  hipLaunchKernelGGL((k_scan_top<Op>), dim3(1), dim3(SC_BT), 0, s, tmp, (uint32_t)nb);
  hipLaunchKernelGGL((k_scan_down<Op>), dim3((unsigned)nb), dim3(SC_BT), 0, s, in, out, n,
                     tmp);
  return hipGetLastError();
}

// Items per thread (a tile is 256 x items).  Up to 2^20 elements a 4,096-element
// tile leaves at most one block per CU, whose 16 items per wave then rank one
// after another with nothing to hide their latency; above, the longer tile's
// longer digit runs win.  24-bit sort, 16 / 4 items: 180,000 pairs 64 / 39 us,
// 2^20 73 / 71 us, 2^21 84 / 107 us, 2^24 363 / 741 us.
constexpr int RS_LONG = 16, RS_SHORT = 4;
constexpr uint64_t RS_SHORT_MAX = 1ull << 20;
template <class KT, int ITEMS>
hipError_t radix_impl(KT* k0, uint32_t* v0, KT* k1, uint32_t* v1, uint64_t n, int key_bits,
                      uint32_t* tmp, KT** kout, uint32_t** vout, const uint32_t* nd, hipStream_t s, bool ids = false) {
  KT* ka = k0;
  uint32_t* va = v0;
  KT* kb = k1;
  uint32_t* vb = v1;
  if (n > 1 && key_bits > 0) {
    const uint64_t nb = (n + RS_BT * ITEMS - 1) / (RS_BT * ITEMS);
    const uint32_t stride = rs_stride(nb);
    uint32_t* hist = tmp;
    uint32_t* totals = tmp + 256ull * stride;
    const int passes = (key_bits + 7) / 8;
    for (int p = 0, shift = 0; p < passes; ++p) {
      const int width = (key_bits - shift + passes - p - 1) / (passes - p);  // what is left, evenly
      const uint32_t dmask = (1u << width) - 1u;
      const uint32_t* vin = ids && p == 0 ? nullptr : va;
      const bool own = ITEMS == RS_SHORT && nb << width <= RS_OWN_COUNTS && width >= RS_OWN_WIDTH;
      hipLaunchKernelGGL((k_rs_hist<KT, ITEMS>), dim3((unsigned)nb), dim3(RS_BT), 0, s, ka, n, shift, dmask, hist, stride, nd,
                         own ? 1 : 0);
      if (own) {
        hipLaunchKernelGGL((k_rs_scatter<KT, RS_SHORT, true>), dim3((unsigned)nb), dim3(RS_BT), 0, s, ka, vin, kb, vb, n,
                           shift, width, hist, stride, totals, nd);
      } else {
        hipLaunchKernelGGL(k_rs_rowscan, dim3(dmask + 1), dim3(RS_BT), 0, s, hist, stride, totals,
                           (uint32_t)(RS_BT * ITEMS), nd);
        hipLaunchKernelGGL((k_rs_scatter<KT, ITEMS, false>), dim3((unsigned)nb), dim3(RS_BT), 0, s, ka, vin, kb, vb, n,
                           shift, width, hist, stride, totals, nd);
      }
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
      shift += width;
      KT* tk = ka;
      ka = kb;
      kb = tk;
      uint32_t* tv = va;
      va = vb;
      vb = tv;
    }
  }
  *kout = ka;
  *vout = va;
  return hipGetLastError();
}

template <class KT>
hipError_t radix_sort(KT* k0, uint32_t* v0, KT* k1, uint32_t* v1, uint64_t n, int key_bits, uint32_t* tmp, KT** kout,
                      uint32_t** vout, const uint32_t* nd, hipStream_t s) {
  return n <= RS_SHORT_MAX ? radix_impl<KT, RS_SHORT>(k0, v0, k1, v1, n, key_bits, tmp, kout, vout, nd, s)
                           : radix_impl<KT, RS_LONG>(k0, v0, k1, v1, n, key_bits, tmp, kout, vout, nd, s);
}

// ---------------------------------------------------------------------------
// Ordered-execution passes.
// ---------------------------------------------------------------------------
// rowstart (optional): p at the first access of a row, else 0
__global__ void k_access_group_flags(const uint32_t* srow, const uint32_t* sop, uint64_t n, uint32_t* flags,
                                     uint32_t* rowstart) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const bool row0 = (p == 0) || srow[p] != srow[p - 1];
    const bool start = row0 || ((sop[p] | sop[p - 1]) & OPID_WRITE) != 0u;
    flags[p] = start ? (uint32_t)p : 0u;
    if (rowstart) rowstart[p] = row0 ? (uint32_t)p : 0u;
  }
}
// ---------------------------------------------------------------------------
// Accesses that can meet another one.  A read of a row that nobody writes
// never waits, is never waited for and raises no rank, so it needs no place
// in its row's order: only the accesses of written rows are sorted.
//   k_ord_mark     a byte per row that some op writes; need = NEED_FREE
//   k_ord_pack     those bytes as bits (rows / 8 bytes, which every XCD's L2
//                  holds), the bytes cleared for the next time
//   k_ord_count    a bit per op and the count per tile of OT ops
//   (row scan)     each tile's place, and the total
//   k_ord_compact  the chosen ops' rows and ids (and transactions) in op order
// 1,048,576 transactions of 16 ops on 10,485,760 rows, theta 0.1, read ratio
// 0.9: 23% of the accesses are left, and GPUTx's preparation takes 0.73
// instead of 1.24 ms.
// ---------------------------------------------------------------------------
constexpr int OT = BT * 16;  // ops per tile, 64 words of op bits
__device__ __forceinline__ uint32_t ord_row(const IndexView& ix, const uint32_t* rows, uint64_t op, uint64_t i) {
  return rows ? rows[i] : idx_dense_find(op_key(op), ix.length);
}
__global__ void k_ord_mark(IndexView ix, const uint64_t* ops, const uint32_t* rows, uint64_t n, uint64_t nrows,
                           uint8_t* wmap, uint32_t* need) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t op = ops[i];
    const uint32_t r = ord_row(ix, rows, op, i);
    if (op_is_write(op) && r < nrows) wmap[r] = 1;
    need[i] = NEED_FREE;
  }
}
// 32 rows per thread; wmap holds a whole number of them
__global__ void k_ord_pack(uint4* wmap, uint64_t words, uint32_t* bits) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint4 a = wmap[2 * i], b = wmap[2 * i + 1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k)  // bytes of 0 or 1: the multiply gathers the four low bits
      m |= (((w[k] & 0x01010101u) * 0x10204080u) >> 28) << (4 * k);
    bits[i] = m;
    if (m) wmap[2 * i] = wmap[2 * i + 1] = make_uint4(0, 0, 0, 0);
  }
}
__global__ __launch_bounds__(BT) void k_ord_count(IndexView ix, const uint64_t* ops, const uint32_t* rows, uint64_t n,
                                                  uint64_t nrows, const uint32_t* bits, uint64_t* flags, uint32_t* cnt) {
  const uint64_t base = (uint64_t)blockIdx.x * OT;
  uint64_t mine = 0;
  uint32_t r[OT / BT];
#pragma unroll
  for (int i = 0; i < OT / BT; ++i) {
    const uint64_t e = base + (uint64_t)i * BT + threadIdx.x;
    r[i] = e < n ? ord_row(ix, rows, ops[e], e) : IDX_MISS;
  }
#pragma unroll
  for (int i = 0; i < OT / BT; ++i) {
    const uint64_t e = base + (uint64_t)i * BT + threadIdx.x;
    // an index miss stays among them (it sorts last and never executes, but
    // counts in the same-rank conflicts)
    const bool keep = r[i] < nrows ? ((bits[r[i] >> 5] >> (r[i] & 31u)) & 1u) != 0 : e < n;
    const uint64_t w = dev::ballot(keep);
    if (dev::lane_id() == 0) {
      if (e < n) flags[e / 64] = w;
      mine += (uint64_t)__popcll(w);
    }
  }
  mine = block_reduce_u64<false>(mine);
  if (threadIdx.x == 0) {
    cnt[blockIdx.x] = (uint32_t)mine;
    if (blockIdx.x + 1 == gridDim.x)  // up to the row scan's next whole 16-byte load
      for (uint32_t b = gridDim.x; b & 3u; ++b) cnt[b] = 0;
  }
}
// crow / cval: row and op id (id_base + i, write flag in bit 31) of each
// chosen op; cidx / cop / ctx (GPUTx, may be null): its own index with the
// write flag, the op id again, and the transaction
__global__ __launch_bounds__(BT) void k_ord_compact(IndexView ix, const uint64_t* ops, const uint32_t* rows, uint64_t n,
                                                    const uint64_t* flags, const uint32_t* place, uint32_t id_base,
                                                    const uint32_t* op_tx, uint32_t* crow, uint32_t* cval,
                                                    uint32_t* crow2, uint32_t* cop, uint32_t* ctx) {
  __shared__ uint32_t pre[OT / 64];
  const uint64_t base = (uint64_t)blockIdx.x * OT;
  const uint32_t t = threadIdx.x, wave = t / 64, lane = dev::lane_id();
  if (t < OT / 64) {
    const uint64_t w = base + 64ull * t < n ? flags[base / 64 + t] : 0;
    uint32_t x = (uint32_t)__popcll(w);
    const uint32_t own = x;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t o = (uint32_t)__shfl_up((int)x, d, 64);
      if (lane >= (uint32_t)d) x += o;
    }
    pre[t] = place[blockIdx.x] + x - own;
  }
  __syncthreads();
#pragma unroll 4
  for (int i = 0; i < OT / BT; ++i) {
    const uint64_t e = base + (uint64_t)i * BT + t;
    const uint64_t w = e < n ? flags[e / 64] : 0;
    if (!((w >> lane) & 1ull)) continue;
    const uint32_t p = pre[i * (BT / 64) + wave] + (uint32_t)__popcll(w & dev::lanemask_lt());
    const uint64_t op = ops[e];
    const uint32_t r = ord_row(ix, rows, op, e), wr = op_is_write(op) ? OPID_WRITE : 0u;
    const uint32_t id = (id_base + (uint32_t)e) | wr;
    crow[p] = r;
    if (crow2) {
      cval[p] = p | wr;
      crow2[p] = r;
      cop[p] = id;
      ctx[p] = op_tx[e];
    } else {
      cval[p] = id;
    }
  }
}

// ---------------------------------------------------------------------------
// Turns and local ranks from accesses sorted by (row, order): val[p] carries
// the access's write flag, key[p] >> rb is its row.  Position p starts a row
// (EV_ROW), or a new access group of its row (EV_GROUP: it or the access
// before it writes), or continues a run of reads (0).
//
// Two passes over tiles of TT elements, TT_ITEMS consecutive ones per thread:
// k_seg_tiles leaves each tile's last row start, last group start and the
// group starts after its last row start; then a tile's carry-in is found by
// reading the summaries before it backwards, 64 at a time (one step unless a
// row spans more than 64 tiles), and everything else lies inside the tile.
// This replaces group flags, two max-scans and a scatter over whole arrays
// (and, for GPUTx, a sum-scan, a key shift and a conflict pass): on 2^24
// accesses, theta 0.1, read ratio 0.9, GaccO's turns 432 -> 131 us (26 tiles,
// 86 turns, 19 fill), GPUTx's ranks 290 -> 128 us and turns 500 -> 138 us.
// Bound: the scattered need stores, which only accesses that meet another one
// still make (the others keep NEED_FREE from a streaming fill).
// ---------------------------------------------------------------------------
// Up to TT_SHORT_MAX accesses a thread takes TT_FEW for the turns, not
// TT_MANY: tiles of 2,048 left most of the chip idle at the sizes of a batch
// (180,224 accesses of 16,384 TPC-C orders, 88 tiles: 15.6 -> 12.3 us; the
// chosen accesses of 65,536 GPUTx transactions: 13.1 -> 8.5).  The ranks keep
// TT_MANY (9.0 us against 12.2: more blocks end in an atomic on one word).
constexpr int TT_MANY = 8, TT_FEW = 2;
constexpr uint64_t TT_SHORT_MAX = 1ull << 20;
inline bool tt_few(uint64_t n) { return n <= TT_SHORT_MAX; }
constexpr uint32_t EV_ROW = 1u, EV_GROUP = 2u;

template <class KT, int TT_ITEMS>
struct SegTile {
  static constexpr int TT = BT * TT_ITEMS;
  KT k[TT_ITEMS];
  uint32_t v[TT_ITEMS];
  KT pk;         // the access before the thread's first
  uint32_t pv;
  uint64_t p0;   // position of the thread's first access
  uint32_t cnt;  // how many it has

  __device__ __forceinline__ void load(const KT* key, const uint32_t* val, uint64_t n) {
    p0 = (uint64_t)blockIdx.x * TT + (uint64_t)threadIdx.x * TT_ITEMS;
    cnt = p0 >= n ? 0u : n - p0 < (uint64_t)TT_ITEMS ? (uint32_t)(n - p0) : (uint32_t)TT_ITEMS;
    if (cnt == (uint32_t)TT_ITEMS) {
      typedef uint32_t Wide __attribute__((ext_vector_type(TT_ITEMS < 4 ? TT_ITEMS : 4)));
      constexpr int W = (int)sizeof(Wide) / 4, Q = (int)sizeof(KT) / 4 * TT_ITEMS / W, V = TT_ITEMS / W;
      Wide q[Q], w[V];
#pragma unroll
      for (int i = 0; i < Q; ++i) q[i] = reinterpret_cast<const Wide*>(key + p0)[i];
#pragma unroll
      for (int i = 0; i < V; ++i) w[i] = reinterpret_cast<const Wide*>(val + p0)[i];
      __builtin_memcpy(k, q, sizeof k);
      __builtin_memcpy(v, w, sizeof v);
    } else {
#pragma unroll
      for (int i = 0; i < TT_ITEMS; ++i) {
        k[i] = (uint32_t)i < cnt ? key[p0 + i] : (KT)0;
        v[i] = (uint32_t)i < cnt ? val[p0 + i] : 0u;
      }
    }
    pk = cnt && p0 ? key[p0 - 1] : (KT)0;
    pv = cnt && p0 ? val[p0 - 1] : 0u;
  }
  // event of the thread's access i (0 past the end)
  __device__ __forceinline__ uint32_t event(int i, int rb) const {
    if ((uint32_t)i >= cnt) return 0u;
    const KT a = i ? k[i - 1] : pk;
    const uint32_t b = i ? v[i - 1] : pv;
    if (p0 + i == 0 || (k[i] >> rb) != (a >> rb)) return EV_ROW;
    return ((v[i] | b) & OPID_WRITE) ? EV_GROUP : 0u;
  }
};

// exclusive max / sum over the block's threads before this one (all lanes of
// the block take part); total: over the whole block
struct SegScan {
  uint32_t row, group;  // last row / group start + 1 (0: none)
  uint32_t cnt;         // group starts since the last row start (or since the tile's first access)
};
__device__ __forceinline__ SegScan seg_join(const SegScan& a, const SegScan& b) {  // a before b
  SegScan r;
  r.row = b.row ? b.row : a.row;
  r.group = b.group ? b.group : a.group;
  r.cnt = b.row ? b.cnt : a.cnt + b.cnt;
  return r;
}
__device__ __forceinline__ SegScan seg_block_scan(const SegScan& mine, SegScan* total) {
  __shared__ SegScan ws[BT / 64];
  const uint32_t lane = dev::lane_id(), wave = threadIdx.x / 64;
  SegScan x = mine;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    SegScan o;
    o.row = (uint32_t)__shfl_up((int)x.row, d, 64);
    o.group = (uint32_t)__shfl_up((int)x.group, d, 64);
    o.cnt = (uint32_t)__shfl_up((int)x.cnt, d, 64);
    if (lane >= (uint32_t)d) x = seg_join(o, x);
  }
  if (lane == 63) ws[wave] = x;
  SegScan e;
  e.row = (uint32_t)__shfl_up((int)x.row, 1, 64);
  e.group = (uint32_t)__shfl_up((int)x.group, 1, 64);
  e.cnt = (uint32_t)__shfl_up((int)x.cnt, 1, 64);
  if (lane == 0) e = SegScan{0, 0, 0};
  __syncthreads();
  SegScan before{0, 0, 0}, all{0, 0, 0};
#pragma unroll
  for (uint32_t w = 0; w < BT / 64; ++w) {
    if (w < wave) before = seg_join(before, ws[w]);
    all = seg_join(all, ws[w]);
  }
  *total = all;
  return seg_join(before, e);
}
// what the thread's own accesses add to the scan
template <class KT, int TT_ITEMS>
__device__ __forceinline__ SegScan seg_own(const SegTile<KT, TT_ITEMS>& t, int rb) {
  SegScan s{0, 0, 0};
#pragma unroll
  for (int i = 0; i < TT_ITEMS; ++i) {
    const uint32_t e = t.event(i, rb);
    const uint32_t p = (uint32_t)(t.p0 + i) + 1u;
    if (e) s.group = p;
    if (e == EV_ROW) {
      s.row = p;
      s.cnt = 0;
    } else if (e == EV_GROUP) {
      s.cnt++;
    }
  }
  return s;
}
// Carry-in of tile b: the join of the summaries before it, read backwards by
// the block's first wave until a row start is seen (the first access of all
// starts a row).  Every thread of the block calls it.
__device__ __forceinline__ SegScan seg_carry(const uint4* summ) {
  __shared__ SegScan in;
  if (threadIdx.x < 64) {
    SegScan c{0, 0, 0};
    const uint32_t lane = threadIdx.x;
    for (uint32_t b = blockIdx.x; b > 0 && c.row == 0;) {
      const bool has = lane < b;
      const uint4 s = has ? summ[b - 1 - lane] : make_uint4(0, 0, 0, 0);
      const uint64_t rows = dev::ballot(has && s.x != 0), groups = dev::ballot(has && s.y != 0);
      // the tiles from the nearest one with a row start on (all, if none has)
      const int rl = rows ? __ffsll((unsigned long long)rows) - 1 : 63;
      uint32_t n = lane <= (uint32_t)rl ? s.z : 0u;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) n += (uint32_t)__shfl_xor((int)n, d, 64);
      c.cnt += n;
      if (rows) c.row = (uint32_t)__shfl((int)s.x, rl, 64);
      if (groups && c.group == 0) c.group = (uint32_t)__shfl((int)s.y, __ffsll((unsigned long long)groups) - 1, 64);
      b = b > 64 ? b - 64 : 0;
    }
    if (lane == 0) in = c;
  }
  __syncthreads();
  return in;
}

template <class KT, int TT_ITEMS>
__global__ __launch_bounds__(BT) void k_seg_tiles(const KT* key, const uint32_t* val, uint64_t n, int rb, uint4* summ,
                                                  const uint32_t* nd) {
  constexpr int TT = BT * TT_ITEMS;
  if (nd) n = *nd;
  if ((uint64_t)blockIdx.x * TT >= n) return;
  SegTile<KT, TT_ITEMS> t;
  t.load(key, val, n);
  SegScan total;
  seg_block_scan(seg_own(t, rb), &total);
  if (threadIdx.x == 0) summ[blockIdx.x] = make_uint4(total.row, total.group, total.cnt, 0u);
}

// The row queues of a thread's accesses that end in it, filed block by block:
// one add per counter and block (a queue per atomic would pile onto them).
__device__ __forceinline__ uint32_t block_file(uint32_t n, uint32_t* ctr) {  // n places for this thread
  __shared__ uint32_t wsum[BT / 64], base;
  const uint32_t lane = dev::lane_id(), wave = threadIdx.x / 64;
  uint32_t x = n;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)x, d, 64);
    if (lane >= (uint32_t)d) x += o;
  }
  __syncthreads();  // the call before has read wsum and base
  if (lane == 63) wsum[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < BT / 64; ++w) {
    before += w < wave ? wsum[w] : 0u;
    all += wsum[w];
  }
  if (threadIdx.x == 0) base = all ? atomicAdd(ctr, all) : 0u;
  __syncthreads();
  return base + before + x - n;
}
constexpr uint32_t CB_BT = 256;  // accesses per combiner chunk, one per thread

// need[op] (op = val & OPID_MASK) of every access that waits or is waited
// for; the others keep NEED_FREE.  The counter of a row where that happens is
// set to 0 at the row's first access.  comb.min > 0: every row queue of at
// least comb.min accesses is listed for its combiner (CombArgs), unless an
// earlier launch of the run reported an error.
// conflicts (GPUTx): same-row neighbours of equal key (row and rank) where
// either writes, added to CONFLICT_SLOTS counters on lines of their own.
template <class KT, int TT_ITEMS>
__global__ __launch_bounds__(BT) void k_seg_turns(const KT* key, const uint32_t* val, uint64_t n, int rb,
                                                  const uint4* summ, uint32_t* need, uint32_t* counters,
                                                  uint64_t nrows, launch::CombArgs comb,
                                                  unsigned long long* conflicts, const uint32_t* nd) {
  constexpr int TT = BT * TT_ITEMS;
  if (nd) n = *nd;
  if ((uint64_t)blockIdx.x * TT >= n) return;
  __shared__ uint32_t wnext[BT / 64];
  SegTile<KT, TT_ITEMS> t;
  t.load(key, val, n);
  const uint32_t lane = dev::lane_id(), wave = threadIdx.x / 64;
  SegScan total, at = seg_block_scan(seg_own(t, rb), &total);
  at = seg_join(seg_carry(summ), at);
  // the first event at or after this thread's chunk, from the chunks after
  // it in the wave, then in the block, then the next tile's first access (a
  // run of reads that goes on there counts as followed: an unneeded
  // increment changes nothing)
  uint32_t first = 0;
#pragma unroll
  for (int i = TT_ITEMS - 1; i >= 0; --i) {
    const uint32_t e = t.event(i, rb);
    first = e ? e : first;
  }
  if (t.cnt < (uint32_t)TT_ITEMS && first == 0) first = EV_ROW;  // the end of the accesses
  const uint64_t some = dev::ballot(first != 0), grp = dev::ballot(first == EV_GROUP);
  if (lane == 0) wnext[wave] = some ? ((grp >> (__ffsll((unsigned long long)some) - 1)) & 1u ? EV_GROUP : EV_ROW) : 0u;
  __syncthreads();
  const uint64_t later = lane == 63 ? 0ull : some & (~0ull << (lane + 1));
  uint32_t next = 0;
  if (later) {
    next = (grp >> (__ffsll((unsigned long long)later) - 1)) & 1u ? EV_GROUP : EV_ROW;
  } else {
#pragma unroll
    for (uint32_t w = 0; w < BT / 64; ++w)
      if (w > wave && next == 0) next = wnext[w];
    if (next == 0) {
      const uint64_t e = (uint64_t)(blockIdx.x + 1) * TT;
      next = e >= n || (key[e] >> rb) != (key[e - 1] >> rb) ? EV_ROW : EV_GROUP;
    }
  }
  // does the chunk's last access end its row queue?
  KT nk = 0;
  {
    const uint32_t lo = (uint32_t)__shfl_down((int)(uint32_t)t.k[0], 1, 64);
    nk = (KT)lo;
    if constexpr (sizeof(KT) == 8)
      nk |= (KT)((uint64_t)(uint32_t)__shfl_down((int)(uint32_t)((uint64_t)t.k[0] >> 32), 1, 64) << 32);
    const uint64_t e = t.p0 + TT_ITEMS;
    if (lane == 63) nk = e < n ? key[e] : (KT)0;
  }
  // what follows each access: walk backwards
  uint32_t nx[TT_ITEMS];
#pragma unroll
  for (int i = TT_ITEMS - 1; i >= 0; --i) {
    if (i + 1 < TT_ITEMS) {
      const uint32_t e = t.event(i + 1, rb);
      nx[i] = e ? e : (uint32_t)i + 1 < t.cnt ? nx[i + 1] : (uint32_t)EV_ROW;
    } else {
      nx[i] = next;
    }
  }
  uint64_t same = 0;
  uint32_t qlen[TT_ITEMS] = {};  // length of the row queue that ends at access i
#pragma unroll
  for (int i = 0; i < TT_ITEMS; ++i) {
    if ((uint32_t)i >= t.cnt) break;
    const uint32_t e = t.event(i, rb), p = (uint32_t)(t.p0 + i);
    if (e) at.group = p + 1;
    if (e == EV_ROW) at.row = p + 1;
    const uint64_t row = (uint64_t)(t.k[i] >> rb);
    if (e == EV_GROUP && conflicts) same += t.k[i] == (i ? t.k[i - 1] : t.pk) ? 1u : 0u;
    if (row >= nrows) continue;  // an index miss never executes
    const uint32_t wait = at.group - at.row;
    const bool followed = nx[i] == EV_GROUP;
    if (wait || followed) need[t.v[i] & OPID_MASK] = wait | (followed ? 0u : NEED_LAST);
    if (e == EV_ROW && followed) counters[row_slot((uint32_t)row, slot_shift(nrows))] = 0u;
    if (comb.min) {
      const uint64_t q = t.p0 + i + 1;
      const KT k1 = i + 1 < TT_ITEMS ? t.k[i + 1] : nk;
      if (q == n || (k1 >> rb) != (t.k[i] >> rb)) qlen[i] = p + 2 - at.row;
    }
  }
  // After an error no queue is listed: a batch's launch will do nothing either
  // (txn_exec).  Asked here, in a kernel of many blocks: in k_tpcc_combine's own
  // few first instructions it moved the update loop, 61 -> 65 ns per payment.
  if (comb.min && *comb.error == 0) {
    // file the queues long enough: their chunks, and those of more than one
    // chunk once more for the carry between their chunks
    const uint32_t step = comb.whole ? 0x7fffffffu : CB_BT;
    uint32_t nch = 0, nmc = 0, nms = 0;
#pragma unroll
    for (int i = 0; i < TT_ITEMS; ++i) {
      if (qlen[i] < comb.min) qlen[i] = 0;
      const uint32_t c = (qlen[i] + step - 1) / step;
      nch += c;
      nmc += c > 1 ? c : 0u;
      nms += c > 1 ? 1u : 0u;
    }
    if (__syncthreads_or((int)nch)) {
      uint32_t ci = block_file(nch, comb.ctr + launch::COMB_CHUNKS);
      uint32_t si = block_file(nmc, comb.ctr + launch::COMB_SUMS);
      uint32_t mi = block_file(nms, comb.ctr + launch::COMB_MULTI);
#pragma unroll
      for (int i = 0; i < TT_ITEMS; ++i) {
        if (!qlen[i]) continue;
        const uint32_t first = (uint32_t)(t.p0 + i) + 1u - qlen[i], c = (qlen[i] + step - 1) / step;
        if (c > 1 && mi < comb.multi_cap) comb.multi[mi] = make_uint4(first, si, c, 0u);
        for (uint32_t x = 0; x < c; ++x)
          if (ci + x < comb.chunk_cap)
            comb.chunks[ci + x] = make_uint4(first + x * step, x + 1 < c ? step : qlen[i] - x * step,
                                             c > 1 ? si + x + 1u : 0u, 0u);
        ci += c;
        if (c > 1) {
          si += c;
          ++mi;
        }
      }
    }
  }
  if (conflicts) {
    same = block_reduce_u64<false>(same);
    if (threadIdx.x == 0 && same)
      atomicAdd(conflicts + 16 * (blockIdx.x % launch::CONFLICT_SLOTS), (unsigned long long)same);
  }
}

// GPUTx one-pass rank (src/gputx.cu:5-27): an access's local rank is the
// number of group starts in its row up to it; rank[tx] = max over tx's
// accesses, tx = val & OPID_MASK, or tx_of[val & OPID_MASK] when it is given;
// max_rank = max.
__global__ __launch_bounds__(BT) void k_seg_ranks(const uint32_t* key, const uint32_t* val, uint64_t n,
                                                  const uint4* summ, uint64_t nrows, uint32_t* rank,
                                                  uint32_t* max_rank, const uint32_t* tx_of, const uint32_t* nd) {
  constexpr int TT_ITEMS = TT_MANY, TT = BT * TT_ITEMS;
  if (nd) n = *nd;
  if ((uint64_t)blockIdx.x * TT >= n) return;
  SegTile<uint32_t, TT_ITEMS> t;
  t.load(key, val, n);
  SegScan total, at = seg_block_scan(seg_own(t, 0), &total);
  at = seg_join(seg_carry(summ), at);
  uint32_t mx = 0;
#pragma unroll
  for (int i = 0; i < TT_ITEMS; ++i) {
    const uint32_t e = t.event(i, 0);
    if (e == EV_ROW) at.cnt = 0;
    if (e == EV_GROUP) at.cnt++;
    // index misses (IDX_MISS sorts last) never execute and raise no rank
    if ((uint32_t)i < t.cnt && at.cnt && t.k[i] < nrows) {
      const uint32_t x = t.v[i] & OPID_MASK;
      atomicMax(&rank[tx_of ? tx_of[x] : x], at.cnt);  // ranks start at 0
      mx = at.cnt > mx ? at.cnt : mx;
    }
  }
  mx = (uint32_t)block_reduce_u64<true>(mx);
  // few blocks raise the maximum: look before the one-address atomic
  if (threadIdx.x == 0 && mx > dev::ld32(max_rank)) atomicMax(max_rank, mx);
}

// ---------------------------------------------------------------------------
// GaccO, persistent form: a row whose access queue (its accesses in
// transaction-id order) holds at least comb.min accesses is run in queue
// order by the row's combiner before the launch.  Every read returns the
// value of the last write to its column before it in transaction-id order,
// or the cell's value before the stream, and the row ends with the last write
// of each column: what the queue's turns produce one handoff at a time.  Its
// ops are marked done (need = NEED_DONE) and the launch skips them; no other
// op touches the row.  Column mode, cols <= 64.
//
// The queue is cut into chunks of CB_BT accesses that workgroups resolve
// independently, as a scan does:
//  1. k_comb_sums: the last write of each column in a chunk (queues of more
//     than one chunk only);
//  2. k_comb_carry, one workgroup per such queue: each column's value at the
//     start of every chunk, and the row's final cells;
//  3. k_comb_resolve: a chunk's reads.  Each wave resolves its own 64
//     accesses: per column written among them (one ballot each), a read
//     finds the last write below it, and the last write of each column is
//     the wave's summary; lane c of wave 0 carries column c through the
//     summaries from the chunk's start; the reads with no write below them
//     in their wave take that value.
// One workgroup per queue, chunk after chunk, took 3.4 us per 1,024 accesses,
// and the hottest row's queue was the whole time: 262,144 transactions of 4 to
// 32 ops at theta 0.99 (270,000 accesses to row 0) 944 us, now 178 us (26 + 36
// + 116; bound: the resolve pass's random op loads and result stores).
// ---------------------------------------------------------------------------
constexpr int CB_WAVES = CB_BT / 64;
// the value that op writes
__device__ __forceinline__ uint64_t comb_value(const launch::CombArgs& c, uint32_t opid) {
  const uint32_t tx = c.op_tx[opid];
  return write_value(c.seed, tx, (uint32_t)(opid - c.tx_off[tx]));
}

__global__ __launch_bounds__(CB_BT) void k_comb_sums(launch::CombArgs c, const uint32_t* sop) {
  __shared__ int last[64];
  const uint32_t nc = min(c.ctr[launch::COMB_CHUNKS], c.chunk_cap), tid = threadIdx.x;
  for (uint32_t x = blockIdx.x; x < nc; x += gridDim.x) {
    const uint4 ch = c.chunks[x];
    if (ch.z == 0) continue;  // the queue's only chunk
    if (tid < 64) last[tid] = -1;
    __syncthreads();
    if (tid < ch.y) {
      const uint32_t so = sop[ch.x + tid];
      if (so & OPID_WRITE) atomicMax(&last[op_col(c.ops[so & OPID_MASK])], (int)tid);
    }
    __syncthreads();
    if (tid < 64) {
      const int l = tid < c.cols ? last[tid] : -1;
      uint64_t* sum = c.sums + (uint64_t)(ch.z - 1) * (c.cols + 1);
      const uint64_t written = dev::ballot(l >= 0);
      if (tid == 0) sum[c.cols] = written;
      if (l >= 0) sum[tid] = comb_value(c, sop[ch.x + (uint32_t)l] & OPID_MASK);
    }
    __syncthreads();  // last is rewritten by the next chunk
  }
}

// Wave w takes the w-th part of the queue's chunks: the last write of each
// column in it, then (with the parts before it known) every chunk's carry-in
// in place of its summary.  Lane c holds column c.
constexpr int CC_WAVES = 16;
__global__ __launch_bounds__(CC_WAVES * 64) void k_comb_carry(launch::CombArgs c, const uint32_t* srow) {
  __shared__ uint64_t part[CC_WAVES][64];
  __shared__ uint64_t mask[CC_WAVES];
  const uint32_t nm = min(c.ctr[launch::COMB_MULTI], c.multi_cap);
  const uint32_t w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const bool col = lane < c.cols;
  for (uint32_t x = blockIdx.x; x < nm; x += gridDim.x) {
    const uint4 q = c.multi[x];
    uint64_t* rc = c.cells + (uint64_t)srow[q.x] * c.cols;
    const uint32_t per = (q.z + CC_WAVES - 1) / CC_WAVES;
    const uint32_t k0 = min(w * per, q.z), k1 = min(k0 + per, q.z);
    uint64_t* sum = c.sums + (uint64_t)q.y * (c.cols + 1);
    uint64_t cur = 0, seen = 0;
#pragma unroll 4
    for (uint32_t k = k0; k < k1; ++k) {
      const uint64_t m = sum[(uint64_t)k * (c.cols + 1) + c.cols];
      const uint64_t v = col ? sum[(uint64_t)k * (c.cols + 1) + lane] : 0;
      if ((m >> lane) & 1ull) cur = v;
      seen |= m;
    }
    part[w][lane] = cur;
    if (lane == 0) mask[w] = seen;
    __syncthreads();
    cur = col ? rc[lane] : 0;
    for (uint32_t y = 0; y < w; ++y)
      if ((mask[y] >> lane) & 1ull) cur = part[y][lane];
    if (w == CC_WAVES - 1 && col) {
      const uint64_t end = (mask[w] >> lane) & 1ull ? part[w][lane] : cur;
      part[w][lane] = end;  // the row's final cells, stored once every wave has read it
    }
#pragma unroll 4
    for (uint32_t k = k0; k < k1; ++k) {
      uint64_t* s = sum + (uint64_t)k * (c.cols + 1);
      const uint64_t m = s[c.cols];
      const uint64_t v = col ? s[lane] : 0;
      if (col) s[lane] = cur;
      if ((m >> lane) & 1ull) cur = v;
    }
    __syncthreads();
    if (w == CC_WAVES - 1 && col) rc[lane] = part[w][lane];
    __syncthreads();  // part and mask are rewritten by the next queue
  }
}

__global__ __launch_bounds__(CB_BT) void k_comb_resolve(launch::CombArgs c, const uint32_t* srow, const uint32_t* sop) {
  __shared__ uint64_t val[CB_BT];         // written values, by access
  __shared__ uint64_t sum[CB_WAVES][64];  // per wave: the last value it wrote to each column
  __shared__ uint64_t cin[CB_WAVES][64];  // per wave: each column's value at its first access
  __shared__ uint64_t wmask[CB_WAVES];    // per wave: the columns it wrote
  const uint32_t nc = min(c.ctr[launch::COMB_CHUNKS], c.chunk_cap);
  const uint32_t tid = threadIdx.x, w = tid / 64, lane = tid % 64;
  uint64_t done_ops = 0;
  for (uint32_t x = blockIdx.x; x < nc; x += gridDim.x) {
    const uint4 ch = c.chunks[x];
    const bool valid = tid < ch.y;
    uint32_t opid = 0, col = 0;
    bool isw = false;
    uint64_t wv = 0;
    if (valid) {
      const uint32_t so = sop[ch.x + tid];
      opid = so & OPID_MASK;
      isw = (so & OPID_WRITE) != 0;
      col = op_col(c.ops[opid]);
      if (isw) wv = comb_value(c, opid);
    }
    uint64_t* rc = c.cells + (uint64_t)srow[ch.x] * c.cols;
    const uint64_t* from = ch.z ? c.sums + (uint64_t)(ch.z - 1) * (c.cols + 1) : rc;
    const uint64_t start = tid < c.cols ? from[tid] : 0;
    int src = -1;  // the lane (of this wave) whose write this read sees
    uint64_t written = 0;
    uint64_t wm = dev::ballot(valid && isw);
    while (wm) {  // the columns written among the wave's 64 accesses
      const uint32_t cc = (uint32_t)__builtin_amdgcn_readlane((int)col, __ffsll((unsigned long long)wm) - 1);
      const uint64_t wc = dev::ballot(valid && isw && col == cc);
      if (valid && col == cc) {
        if (isw) {
          if ((wc >> lane) >> 1 == 0) sum[w][cc] = wv;  // the wave's last write of cc
        } else {
          const uint64_t below = wc & dev::lanemask_lt();
          if (below) src = 63 - __clzll((long long)below);
        }
      }
      written |= 1ull << cc;
      wm &= ~wc;
    }
    val[tid] = wv;
    if (lane == 0) wmask[w] = written;
    __syncthreads();
    if (tid < c.cols) {
      uint64_t cur = start;
      for (int y = 0; y < CB_WAVES; ++y) {
        cin[y][tid] = cur;
        if ((wmask[y] >> tid) & 1ull) cur = sum[y][tid];
      }
      if (ch.z == 0) rc[tid] = cur;  // the queue's only chunk: the row's final cells
    }
    __syncthreads();
    if (valid) {
      if (!isw) c.reads[opid] = src >= 0 ? val[w * 64 + (uint32_t)src] : cin[w][col];
      c.need[opid] = NEED_DONE;
    }
    done_ops += ch.y;
    __syncthreads();  // val / sum / cin / wmask are rewritten by the next chunk
  }
  if (tid == 0 && done_ops) atomicAdd(c.combined, (unsigned long long)done_ops);
}

// TPC-C under GaccO: a row queue of at least comb.min updates is run by one
// wave, which holds the row's cells in registers, gathers 64 updates at a
// time (the next 64 while it applies these) and applies them in order.  An
// update's turn in the launch is a handoff through memory of about 5 us
// (poll, load the row, store it, release, count); here it is a few dozen
// cycles (61 ns per payment of one warehouse's queue).  131,072 new orders at
// 16 warehouses 4.80 -> 1.04 ms, 262,144 payments at 16 warehouses 244 -> 1.44
// ms, 65,536 payments at 1 warehouse 546 -> 4.23 ms.
constexpr int TC_BT = 256;
// The updates of lanes 0 .. n - 1 in lane order on the row v, which every lane
// holds; returns this lane's result.  KIND: the updates' kind, known to be
// one for all of them (a queue's always are: a row belongs to one table), so
// that the loop carries that update's few operations alone, or -1.
template <int KIND>
__device__ __forceinline__ uint64_t tpcc_run(uint32_t kind, uint32_t param, uint32_t n, uint64_t (&v)[TPCC_COLS]) {
  const uint32_t lane = threadIdx.x % 64;
  uint64_t mine = 0;
#pragma unroll 8
  for (uint32_t j = 0; j < n; ++j) {
    const uint32_t k = KIND >= 0 ? (uint32_t)KIND : (uint32_t)__builtin_amdgcn_readlane((int)kind, (int)j);
    const uint64_t r = tpcc_apply(k, (uint32_t)__builtin_amdgcn_readlane((int)param, (int)j), v);
    mine = lane == j ? r : mine;
  }
  return mine;
}
__global__ __launch_bounds__(TC_BT) void k_tpcc_combine(launch::CombArgs c, const uint32_t* srow, const uint32_t* sop) {
  const uint32_t nq = min(c.ctr[launch::COMB_CHUNKS], c.chunk_cap);
  const uint32_t lane = threadIdx.x % 64;
  for (uint32_t x = (blockIdx.x * TC_BT + threadIdx.x) / 64; x < nq; x += gridDim.x * (TC_BT / 64)) {
    const uint4 q = c.chunks[x];
    uint64_t* row = c.cells + (uint64_t)srow[q.x] * TPCC_COLS;
    uint64_t v[TPCC_COLS];
#pragma unroll
    for (uint32_t i = 0; i < TPCC_COLS; ++i) v[i] = row[i];
    uint32_t op = lane < q.y ? sop[q.x + lane] & OPID_MASK : 0u;
    uint32_t kind = lane < q.y ? op_col(c.ops[op]) : 0u, param = lane < q.y ? c.op_param[op] : 0u;
    for (uint32_t b = 0; b < q.y; b += 64) {
      const uint32_t n = min(q.y - b, 64u), nb = b + 64 + lane;
      const bool more = nb < q.y;
      const uint32_t op1 = more ? sop[q.x + nb] & OPID_MASK : 0u;
      const uint32_t kind1 = more ? op_col(c.ops[op1]) : 0u, param1 = more ? c.op_param[op1] : 0u;
      uint64_t mine = 0;
      const uint32_t k0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)kind);
      const bool one_kind = dev::ballot(lane < n && kind != k0) == 0;
      if (one_kind && k0 == TPCC_PAY_W)
        mine = tpcc_run<TPCC_PAY_W>(kind, param, n, v);
      else if (one_kind && k0 == TPCC_PAY_D)
        mine = tpcc_run<TPCC_PAY_D>(kind, param, n, v);
      else if (one_kind && k0 == TPCC_PAY_C)
        mine = tpcc_run<TPCC_PAY_C>(kind, param, n, v);
      else if (one_kind && k0 == TPCC_NO_D)
        mine = tpcc_run<TPCC_NO_D>(kind, param, n, v);
      else if (one_kind && k0 == TPCC_NO_S)
        mine = tpcc_run<TPCC_NO_S>(kind, param, n, v);
      else
        mine = tpcc_run<-1>(kind, param, n, v);
      if (lane < n) {
        c.reads[op] = mine;
        c.need[op] = NEED_DONE;
      }
      op = op1;
      kind = kind1;
      param = param1;
    }
    if (lane == 0) {
#pragma unroll
      for (uint32_t i = 0; i < TPCC_COLS; ++i) row[i] = v[i];
    }
  }
}

// Open form (serving), one admitted batch at a time, accesses sorted by
// (row, op): the turn counts the accesses to the row that earlier batches of
// the launch queued (base[row]) plus the group start within the batch.
__global__ void k_access_need_open(const uint32_t* srow, const uint32_t* sop, const uint32_t* gstart,
                                   const uint32_t* rstart, uint64_t n, uint64_t nrows, const uint32_t* base,
                                   uint32_t* need) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t r = srow[p];
    if (r >= nrows) continue;  // an index miss never executes
    need[sop[p] & OPID_MASK] = base[r] + (gstart[p] - rstart[p]);
  }
}
// base[row] += the batch's accesses to the row, written once per row (at the
// row's last position); run after k_access_need_open.
__global__ void k_row_base_add(const uint32_t* srow, const uint32_t* rstart, uint64_t n, uint64_t nrows,
                               uint32_t* base) {
  for (uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n;
       p += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t r = srow[p];
    if (r >= nrows) continue;
    if (p + 1 == n || srow[p + 1] != r) base[r] += (uint32_t)(p - rstart[p] + 1);
  }
}

// keys[i] = (rows[i] << rank_bits) | rank[tx[i]]
template <class KT>
__global__ void k_gtx_exec_keys(const uint32_t* rows, const uint32_t* tx, const uint32_t* rank, uint64_t n,
                                int rank_bits, KT* keys, const uint32_t* nd) {
  if (nd) n = *nd;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    keys[i] = (KT)(((uint64_t)rows[i] << rank_bits) | rank[tx[i]]);
}
// Histogram of ranks (gputx_pre3, src/gputx.cu:30-38).  There are usually few
// ranks, so each block counts into LDS and adds its non-zero bins once.
constexpr uint32_t RANK_LDS_BINS = 8192;
__global__ __launch_bounds__(256) void k_rank_hist(const uint32_t* rank, uint64_t ntx, uint32_t nranks,
                                                   uint32_t* hist) {
  __shared__ uint32_t h[RANK_LDS_BINS];
  const bool in_lds = nranks <= RANK_LDS_BINS;
  if (in_lds)
    for (uint32_t b = threadIdx.x; b < nranks; b += blockDim.x) h[b] = 0;
  __syncthreads();
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ntx;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t r = rank[i];
    if (in_lds)
      atomicAdd(&h[r], 1u);
    else
      atomicAdd(&hist[r], 1u);
  }
  __syncthreads();
  if (in_lds)
    for (uint32_t b = threadIdx.x; b < nranks; b += blockDim.x)
      if (h[b]) atomicAdd(&hist[b], h[b]);
}

__global__ void k_reset_rows(const uint32_t* rows, uint64_t n, uint64_t nrows_table, uint32_t shift,
                             uint32_t wshift, uint64_t* cc, uint32_t* vprev) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t r = rows[i];
    if (r >= nrows_table) continue;
    const uint32_t w = row_slot(r, shift);
    if (cc) dev::st(cc + ((uint64_t)w << wshift), 0);
    if (vprev) dev::st32(vprev + w, 0);
  }
}
__device__ __forceinline__ void reset_batch(uint64_t* ctrs) {
  const int i = threadIdx.x;
  if (i == 0) {
    dev::st(ctrs + CTR_TICKET, 0);  // commit tickets
    dev::st(ctrs + CTR_POOL, 0);    // MVCC pool bump pointer
    dev::st(ctrs + CTR_T0, wall_clock64());
  }
  // timestamp allocators restart at 1 (timestamp.cuh:76-80)
  if (i < TS_SHARDS) dev::st(ctrs + CTR_TS0 + 16 * i, 1);
  if (i < GATE_SHARDS) dev::st(ctrs + CTR_GATE0 + 16 * i + 3, 0);  // groups that are through
}
__device__ __forceinline__ void reset_admission(uint64_t* ctrs) {
  const int i = threadIdx.x;
  if (i == 0) dev::st(ctrs + CTR_SLOT, 0);
  if (i < GATE_SHARDS) {
    dev::st(ctrs + CTR_GATE0 + 16 * i + 1, 0);
    dev::st(ctrs + CTR_GATE0 + 16 * i + 2, 0);
    dev::st(ctrs + CTR_GATE0 + 16 * i + 3, 0);
    dev::st(ctrs + CTR_ADMIT0 + 16 * i, 0);  // the u32 admission word and its neighbour
  }
}
__global__ void k_batch_begin(uint64_t* ctrs) { reset_batch(ctrs); }
__global__ void k_persist_begin(uint64_t* ctrs) { reset_admission(ctrs); }
// Start of a run: metrics (and the hot-key counts of a persistent run) to
// zero, and, with `counters`, what k_batch_begin and k_persist_begin set.
__global__ void k_run_begin(uint64_t* metrics, uint32_t* defer, uint64_t* ctrs, int counters) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
  for (uint32_t k = i; k < (uint32_t)METRIC_SLOTS * METRICS_WORDS; k += step) metrics[k] = 0;
  if (defer)
    for (uint32_t k = i; k < (uint32_t)launch::DEFER_WORDS; k += step) defer[k] = 0;
  if (counters && blockIdx.x == 0) {
    reset_batch(ctrs);
    reset_admission(ctrs);
  }
}
// End of a run: the metrics slots' totals, GPUTx's conflicts, the ops run by
// combiners and the deferral's state words, into host memory, so that the
// host reads them after its one wait for the stream and no copy follows.
// One block, since every run waits for it; bound by one load latency: thread t
// sums field t mod 16 of every 16th slot, all its loads (whole lines per 16
// threads) issued at once, and 16 threads add 16 sums each out of LDS.  An LDS
// atomic per slot and field took 15-22 us.
constexpr int RUN_FIELDS = 10;  // Metrics fields in use; the last is error_flags
static_assert(offsetof(Metrics, error_flags) == 8 * (RUN_FIELDS - 1) && METRICS_WORDS == 16, "the fields k_run_end sums");
__global__ __launch_bounds__(256) void k_run_end(const Metrics* metrics, const uint64_t* conflicts,
                                                 const uint64_t* combined, const uint32_t* defer,
                                                 launch::RunResult* out) {
  constexpr int STEP = 256 / METRICS_WORDS;  // slots that the block reads at once
  constexpr int N = METRIC_SLOTS / STEP;
  static_assert(METRIC_SLOTS % STEP == 0 && launch::CONFLICT_SLOTS == METRICS_WORDS, "no remainder");
  __shared__ uint64_t part[STEP + 1][METRICS_WORDS];
  const uint32_t f = threadIdx.x % METRICS_WORDS, g = threadIdx.x / METRICS_WORDS;
  const bool flags = f == RUN_FIELDS - 1;
  const uint64_t* m = reinterpret_cast<const uint64_t*>(metrics) + threadIdx.x;
  uint64_t v[N];
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = m[(size_t)i * 256];
  const uint64_t confl = g == 0 && conflicts ? conflicts[16 * f] : 0;
  const uint64_t comb = threadIdx.x == 0 && combined ? *combined : 0;
  const uint32_t any = threadIdx.x == 0 && defer ? defer[launch::DEFER_ANY] : 0;
  const uint32_t nhot = threadIdx.x == 0 && defer ? defer[launch::DEFER_NHOT] : 0;
  uint64_t x = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) x = flags ? x | v[i] : x + v[i];
  part[g][f] = x;
  if (g == 0) part[STEP][f] = confl;
  __syncthreads();
  uint64_t* o = reinterpret_cast<uint64_t*>(&out->metrics);
  if (threadIdx.x < RUN_FIELDS) {
    uint64_t y = 0;
#pragma unroll
    for (int i = 0; i < STEP; ++i) y = flags ? y | part[i][f] : y + part[i][f];
    dev::st(o + f, flags ? (uint32_t)y : y);
    if (flags) dev::st(&out->failed, y >> 32);
  }
  if (threadIdx.x == 0) {
    uint64_t c = 0;
#pragma unroll
    for (int i = 0; i < (int)launch::CONFLICT_SLOTS; ++i) c += part[STEP][i];
    dev::st(&out->conflicts, c);
    dev::st(&out->combined, comb);
    dev::st(&out->deferred, any ? nhot : 0);
  }
}

// Device wall clock now (for mapping commit stamps to host time).
__global__ void k_clock_sample(uint64_t* out) {
  if (threadIdx.x == 0) dev::st(out, wall_clock64());
}

// ---------------------------------------------------------------------------
// Hot-writer deferral (persistent form of the lock, timestamp and OCC
// schemes).  A transaction that writes a hot key conflicts with every
// concurrent transaction touching that key, and under high skew those writers
// hold up (2PL) or abort (OCC, T/O) the far larger number of transactions that
// only read the hot keys.  The launch therefore takes every other transaction
// first and the hot writers last.  A key is hot when its bucket (Fibonacci
// hash of the key) holds at least `thr` of a sample of the ops (every
// stride-th op); thr is scaled so that a key touched by at least one
// transaction in `share` qualifies.  The deferral only reorders admission:
// each scheme still reports its own serialization order.

// sampled access counts per bucket; the lanes of a wave that share a bucket
// add together (one atomic per distinct bucket of the wave)
__global__ __launch_bounds__(BT) void k_defer_count(const uint64_t* ops, uint64_t nsamp, uint64_t stride,
                                                    uint32_t* cnt, uint32_t thr, uint32_t* st) {
  for (uint64_t base = (uint64_t)blockIdx.x * BT; base < nsamp; base += (uint64_t)gridDim.x * BT) {
    const uint64_t i = base + threadIdx.x;
    const bool v = i < nsamp;
    const uint32_t b = v ? defer_bucket(op_key(ops[i * stride])) : 0u;
    uint64_t act = dev::ballot(v);
    while (act) {
      const int l = __ffsll((unsigned long long)act) - 1;
      const uint32_t lb = dev::shfl32(b, l);
      const uint64_t same = dev::ballot(b == lb) & act;
      if ((int)dev::lane_id() == l) {
        const uint32_t add = (uint32_t)__popcll(same), old = atomicAdd(cnt + lb, add);
        if (old < thr && old + add >= thr) st[launch::DEFER_ANY] = 1u;  // the add that makes the bucket hot
      }
      act &= ~same;
    }
  }
}

// map[slot] = transaction.  Nothing hot: the identity.  Otherwise a
// transaction that writes a hot key is deferred: the others fill the slots
// from 0 up, the deferred ones from ntx - 1 down, each class in the order its
// blocks claim their ranges (one pair of atomics per block step);
// st[DEFER_NHOT] ends as the number deferred.
__global__ __launch_bounds__(BT) void k_defer_order(const uint64_t* tx_off, const uint64_t* ops, uint64_t ntx,
                                                    const uint32_t* cnt, uint32_t thr, uint32_t* st, uint32_t* map) {
  __shared__ uint32_t wc[BT / 64], wh[BT / 64];
  __shared__ uint32_t bc, bh;
  const bool any = st[launch::DEFER_ANY] != 0;  // the same for every thread of the grid
  const uint32_t w = threadIdx.x / 64;
  for (uint64_t base = (uint64_t)blockIdx.x * BT; base < ntx; base += (uint64_t)gridDim.x * BT) {
    const uint64_t t = base + threadIdx.x;
    const bool v = t < ntx;
    if (!any) {
      if (v) map[t] = (uint32_t)t;
      continue;
    }
    bool h = false;
    if (v) {
      const uint64_t o1 = tx_off[t + 1];
      for (uint64_t o = tx_off[t]; o < o1; ++o) {
        const uint64_t op = ops[o];
        h |= op_is_write(op) && cnt[defer_bucket(op_key(op))] >= thr;
      }
    }
    const uint64_t mh = dev::ballot(h), mc = dev::ballot(v && !h);
    if (dev::lane_id() == 0) {
      wc[w] = (uint32_t)__popcll(mc);
      wh[w] = (uint32_t)__popcll(mh);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t sc = 0, sh = 0;
      for (int i = 0; i < BT / 64; ++i) {
        const uint32_t x = wc[i], y = wh[i];
        wc[i] = sc;
        wh[i] = sh;
        sc += x;
        sh += y;
      }
      bc = sc ? atomicAdd(st + launch::DEFER_NCOLD, sc) : 0u;
      bh = sh ? atomicAdd(st + launch::DEFER_NHOT, sh) : 0u;
    }
    __syncthreads();
    const uint64_t below = dev::lanemask_lt();
    if (h)
      map[ntx - 1 - (bh + wh[w] + (uint32_t)__popcll(mh & below))] = (uint32_t)t;
    else if (v)
      map[bc + wc[w] + (uint32_t)__popcll(mc & below)] = (uint32_t)t;
    __syncthreads();  // wc / wh / bc / bh are rewritten by the next step
  }
}

}  // namespace

namespace launch {

#define GC_LAUNCH(kern, n, ...)                                                    \
  do {                                                                            \
    hipLaunchKernelGGL(kern, dim3(grid_stride_blocks(n)), dim3(BT), 0, s, __VA_ARGS__); \
    return hipGetLastError();                                                     \
  } while (0)

hipError_t seed_table(uint64_t* cells, uint64_t rows, uint32_t cols, uint64_t seed, hipStream_t s) {
  GC_LAUNCH(k_seed_table, rows * cols, cells, rows, cols, seed);
}
hipError_t index_insert(const uint32_t* keys, const uint32_t* vals, uint64_t n, uint32_t* buckets,
                        uint32_t nbuckets, hipStream_t s) {
  GC_LAUNCH(k_index_insert, n, keys, vals, n, buckets, nbuckets);
}
hipError_t probe(const IndexView& ix, const uint64_t* ops, uint64_t n, uint32_t* rows_out,
                 hipStream_t s, uint32_t* rows_copy, uint32_t* ids_out, uint32_t id_base, const uint32_t* id_map,
                 uint32_t* need, uint64_t* zero, uint32_t nzero) {
  if (nzero > 256) return hipErrorInvalidValue;  // one word per thread of a block
  GC_LAUNCH(k_probe, n, ix, ops, n, rows_out, rows_copy, ids_out, id_base, id_map, need, zero, nzero);
}
hipError_t op_tx(const uint64_t* tx_off, uint64_t ntx, uint32_t* op_tx, hipStream_t s) {
  GC_LAUNCH(k_op_tx, ntx, tx_off, ntx, op_tx);
}
hipError_t op_ids(const uint64_t* ops, uint64_t n, uint32_t base, uint32_t* out, hipStream_t s) {
  GC_LAUNCH(k_op_ids, n, ops, n, base, out);
}
hipError_t fill_u32(uint32_t* v, uint64_t n, uint32_t x, hipStream_t s) { GC_LAUNCH(k_fill32, n, v, n, x); }
uint32_t defer_threshold(uint64_t ntx, uint64_t nops, uint32_t share) {
  const uint64_t stride = nops > DEFER_SAMPLE ? nops / DEFER_SAMPLE : 1;
  const uint64_t want = (ntx + (uint64_t)share * stride - 1) / ((uint64_t)share * stride);
  return (uint32_t)(want < 2 ? 2 : want > 0xffffffffull ? 0xffffffffull : want);
}
hipError_t defer_order(const uint64_t* tx_off, const uint64_t* ops, uint64_t ntx, uint64_t nops, uint32_t share,
                       uint32_t* cnt, uint32_t* map, hipStream_t s) {
  if (ntx == 0) return hipSuccess;
  // about DEFER_SAMPLE sampled ops
  const uint64_t stride = nops > DEFER_SAMPLE ? nops / DEFER_SAMPLE : 1;
  const uint64_t nsamp = nops / stride;
  const uint32_t thr = defer_threshold(ntx, nops, share);
  uint32_t* st = cnt + DEFER_BUCKETS;
  if (nsamp) {
    hipLaunchKernelGGL(k_defer_count, dim3(grid_stride_blocks(nsamp)), dim3(BT), 0, s, ops, nsamp, stride, cnt, thr, st);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(k_defer_order, dim3(reduce_blocks(ntx)), dim3(BT), 0, s, tx_off, ops, ntx, cnt, thr, st, map);
  return hipGetLastError();
}
hipError_t fill_u64(uint64_t* v, uint64_t n, uint64_t x, hipStream_t s) { GC_LAUNCH(k_fill64, n, v, n, x); }

uint64_t scan_tmp_words(uint64_t n) { return (n + SC_TILE - 1) / SC_TILE + 64; }
uint64_t radix_sort_tmp_words(uint64_t n) {
  const uint64_t nb = (n + RS_BT * RS_SHORT - 1) / (RS_BT * RS_SHORT);
  return 256ull * rs_stride(nb) + 256 + 64;
}
hipError_t radix_sort_u32(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, uint64_t n,
                          int key_bits, uint32_t* tmp, uint32_t** keys_out, uint32_t** vals_out,
                          hipStream_t s, const uint32_t* nd) {
  return radix_sort<uint32_t>(k0, v0, k1, v1, n, key_bits, tmp, keys_out, vals_out, nd, s);
}
hipError_t radix_sort_ids(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, uint64_t n, int key_bits,
                          uint32_t* tmp, uint32_t** keys_out, uint32_t** vals_out, hipStream_t s) {
  if (n == 1) {
    const hipError_t e = fill_u32(v0, 1, 0, s);
    if (e != hipSuccess) return e;
  }
  return n <= RS_SHORT_MAX
             ? radix_impl<uint32_t, RS_SHORT>(k0, v0, k1, v1, n, key_bits, tmp, keys_out, vals_out, nullptr, s, true)
             : radix_impl<uint32_t, RS_LONG>(k0, v0, k1, v1, n, key_bits, tmp, keys_out, vals_out, nullptr, s, true);
}
hipError_t radix_sort_u64(uint64_t* k0, uint32_t* v0, uint64_t* k1, uint32_t* v1, uint64_t n,
                          int key_bits, uint32_t* tmp, uint64_t** keys_out, uint32_t** vals_out,
                          hipStream_t s, const uint32_t* nd) {
  return radix_sort<uint64_t>(k0, v0, k1, v1, n, key_bits, tmp, keys_out, vals_out, nd, s);
}
hipError_t inclusive_max_u32(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* tmp, hipStream_t s) {
  return scan_impl<OpMax>(in, out, n, tmp, s);
}
hipError_t access_group_flags(const uint32_t* srow, const uint32_t* sop, uint64_t n, uint32_t* flags,
                              hipStream_t s, uint32_t* rowstart) {
  GC_LAUNCH(k_access_group_flags, n, srow, sop, n, flags, rowstart);
}
static unsigned seg_blocks(uint64_t n) {
  const uint64_t tile = BT * (tt_few(n) ? TT_FEW : TT_MANY);
  return (unsigned)((n + tile - 1) / tile);
}
// a smaller n may take the shorter tiles
uint64_t seg_tmp_words(uint64_t n) { return 4 * std::max<uint64_t>(seg_blocks(n), seg_blocks(std::min(n, TT_SHORT_MAX))); }
template <class KT>
static hipError_t seg_turns_impl(const KT* key, const uint32_t* val, uint64_t n, int rb, uint32_t* tmp, uint32_t* need,
                                 uint32_t* counters, uint64_t nrows, const CombArgs& comb, uint64_t* conflicts,
                                 const uint32_t* nd, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const unsigned nb = seg_blocks(n);
  uint4* summ = reinterpret_cast<uint4*>(tmp);
  auto* confl = reinterpret_cast<unsigned long long*>(conflicts);
  if (tt_few(n)) {
    hipLaunchKernelGGL((k_seg_tiles<KT, TT_FEW>), dim3(nb), dim3(BT), 0, s, key, val, n, rb, summ, nd);
    hipLaunchKernelGGL((k_seg_turns<KT, TT_FEW>), dim3(nb), dim3(BT), 0, s, key, val, n, rb, summ, need, counters, nrows,
                       comb, confl, nd);
  } else {
    hipLaunchKernelGGL((k_seg_tiles<KT, TT_MANY>), dim3(nb), dim3(BT), 0, s, key, val, n, rb, summ, nd);
    hipLaunchKernelGGL((k_seg_turns<KT, TT_MANY>), dim3(nb), dim3(BT), 0, s, key, val, n, rb, summ, need, counters, nrows,
                       comb, confl, nd);
  }
  return hipGetLastError();
}
hipError_t seg_turns(const uint32_t* key, const uint32_t* val, uint64_t n, int rb, uint32_t* tmp, uint32_t* need,
                     uint32_t* counters, uint64_t nrows, const CombArgs& comb, uint64_t* conflicts, hipStream_t s,
                     const uint32_t* nd) {
  return seg_turns_impl(key, val, n, rb, tmp, need, counters, nrows, comb, conflicts, nd, s);
}
hipError_t seg_turns64(const uint64_t* key, const uint32_t* val, uint64_t n, int rb, uint32_t* tmp, uint32_t* need,
                       uint32_t* counters, uint64_t nrows, uint64_t* conflicts, hipStream_t s,
                       const uint32_t* nd) {
  return seg_turns_impl(key, val, n, rb, tmp, need, counters, nrows, CombArgs{}, conflicts, nd, s);
}
hipError_t seg_ranks(const uint32_t* row, const uint32_t* val, uint64_t n, uint32_t* tmp, uint64_t nrows,
                     uint32_t* rank, uint32_t* max_rank, hipStream_t s, const uint32_t* tx_of, const uint32_t* nd) {
  if (n == 0) return hipSuccess;
  const unsigned nb = (unsigned)((n + BT * TT_MANY - 1) / (BT * TT_MANY));
  uint4* summ = reinterpret_cast<uint4*>(tmp);
  hipLaunchKernelGGL((k_seg_tiles<uint32_t, TT_MANY>), dim3(nb), dim3(BT), 0, s, row, val, n, 0, summ, nd);
  hipLaunchKernelGGL(k_seg_ranks, dim3(nb), dim3(BT), 0, s, row, val, n, summ, nrows, rank, max_rank, tx_of, nd);
  return hipGetLastError();
}
uint64_t comb_chunk_cap(uint64_t nops, uint32_t min) { return nops / min + nops / CB_BT + 1; }
uint64_t comb_multi_cap(uint64_t nops) { return nops / CB_BT + 1; }
uint64_t comb_sum_words(uint64_t nops, uint32_t cols) { return (2 * (nops / CB_BT) + 1) * (cols + 1ull); }
hipError_t tpcc_combine(const CombArgs& c, const uint32_t* srow, const uint32_t* sop, hipStream_t s) {
  const unsigned grid = c.chunk_cap < 8192 ? (c.chunk_cap + 3) / 4 : 2048;  // a wave per queue
  if (grid == 0) return hipSuccess;
  hipLaunchKernelGGL(k_tpcc_combine, dim3(grid), dim3(TC_BT), 0, s, c, srow, sop);
  return hipGetLastError();
}
hipError_t gacco_combine(const CombArgs& c, const uint32_t* srow, const uint32_t* sop, hipStream_t s) {
  if (c.cols == 0 || c.cols > 64 || c.chunk_cap == 0) return hipSuccess;
  // capped grids: with no queue listed every block leaves at once
  const unsigned grid = c.chunk_cap < 2048 ? c.chunk_cap : 2048;
  const unsigned mgrid = c.multi_cap < 256 ? c.multi_cap : 256;
  hipLaunchKernelGGL(k_comb_sums, dim3(grid), dim3(CB_BT), 0, s, c, sop);
  hipLaunchKernelGGL(k_comb_carry, dim3(mgrid), dim3(CC_WAVES * 64), 0, s, c, srow);
  hipLaunchKernelGGL(k_comb_resolve, dim3(grid), dim3(CB_BT), 0, s, c, srow, sop);
  return hipGetLastError();
}
hipError_t gtx_exec_keys(const uint32_t* rows, const uint32_t* tx, const uint32_t* rank,
                         uint64_t n, int rank_bits, uint64_t* keys, hipStream_t s, const uint32_t* nd) {
  GC_LAUNCH(k_gtx_exec_keys<uint64_t>, n, rows, tx, rank, n, rank_bits, keys, nd);
}
hipError_t gtx_exec_keys32(const uint32_t* rows, const uint32_t* tx, const uint32_t* rank,
                           uint64_t n, int rank_bits, uint32_t* keys, hipStream_t s, const uint32_t* nd) {
  GC_LAUNCH(k_gtx_exec_keys<uint32_t>, n, rows, tx, rank, n, rank_bits, keys, nd);
}
uint64_t ord_flag_words(uint64_t n) { return (n + OT - 1) / OT * (OT / 64); }
uint64_t ord_map_bytes(uint64_t nrows) { return (nrows + 31) / 32 * 32; }
hipError_t ord_filter(const IndexView& ix, const uint64_t* ops, const uint32_t* rows, uint64_t n, uint64_t nrows,
                      uint32_t id_base, const uint32_t* op_tx, const OrdFilter& f, uint32_t* tmp, uint32_t* need,
                      uint32_t* crow, uint32_t* cval, hipStream_t s) {
  if (n == 0) return hipSuccess;
  const unsigned nb = (unsigned)((n + OT - 1) / OT);
  const uint64_t words = (nrows + 31) / 32;
  hipLaunchKernelGGL(k_ord_mark, dim3(grid_stride_blocks(n)), dim3(BT), 0, s, ix, ops, rows, n, nrows, f.wmap, need);
  hipLaunchKernelGGL(k_ord_pack, dim3(grid_stride_blocks(words)), dim3(BT), 0, s, reinterpret_cast<uint4*>(f.wmap),
                     words, f.bits);
  hipLaunchKernelGGL(k_ord_count, dim3(nb), dim3(BT), 0, s, ix, ops, rows, n, nrows, f.bits, f.flags, tmp);
  hipLaunchKernelGGL(k_rs_rowscan, dim3(1), dim3(RS_BT), 0, s, tmp, rs_stride(nb), f.count, 0u,
                     (const uint32_t*)nullptr);
  hipLaunchKernelGGL(k_ord_compact, dim3(nb), dim3(BT), 0, s, ix, ops, rows, n, f.flags, tmp, id_base, op_tx, crow, cval,
                     f.crow, f.cop, f.ctx);
  return hipGetLastError();
}
hipError_t rank_hist(const uint32_t* rank, uint64_t ntx, uint32_t nranks, uint32_t* hist, hipStream_t s) {
  uint64_t blocks = (ntx + 4095) / 4096;
  if (blocks < 1) blocks = 1;
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL(k_rank_hist, dim3((unsigned)blocks), dim3(256), 0, s, rank, ntx, nranks, hist);
  return hipGetLastError();
}
hipError_t reset_rows(const uint32_t* rows, uint64_t n, uint64_t nrows_table, uint64_t* cc,
                      uint32_t* vprev, hipStream_t s, bool latch) {
  // Outside a run every CC word and chain head is zero, so clearing the whole
  // arrays leaves the same state.  That streams rows x 12 bytes instead of one
  // scattered line per op: the cheaper form once n >= rows / 8.  (A latch
  // array is zero outside a critical section, so its fill changes nothing.)
  const uint32_t wshift = latch ? 1 : 0;
  if (n * 8 >= nrows_table) {
    if (cc) {
      const hipError_t e = fill_u64(cc, slot_words(nrows_table) << wshift, 0, s);
      if (e != hipSuccess) return e;
    }
    if (vprev) return fill_u32(vprev, slot_words(nrows_table), 0, s);
    return hipSuccess;
  }
  GC_LAUNCH(k_reset_rows, n, rows, n, nrows_table, slot_shift(nrows_table), wshift, cc, vprev);
}
hipError_t access_need_open(const uint32_t* srow, const uint32_t* sop, const uint32_t* gstart, const uint32_t* rstart,
                            uint64_t n, uint64_t nrows, const uint32_t* base, uint32_t* need, hipStream_t s) {
  if (n == 0) return hipSuccess;
  GC_LAUNCH(k_access_need_open, n, srow, sop, gstart, rstart, n, nrows, base, need);
}
hipError_t row_base_add(const uint32_t* srow, const uint32_t* rstart, uint64_t n, uint64_t nrows, uint32_t* base,
                        hipStream_t s) {
  if (n == 0) return hipSuccess;
  GC_LAUNCH(k_row_base_add, n, srow, rstart, n, nrows, base);
}
hipError_t run_begin(uint64_t* metrics, uint32_t* defer, uint64_t* ctrs, bool counters, hipStream_t s) {
  hipLaunchKernelGGL(k_run_begin, dim3(defer ? 64 : 16), dim3(BT), 0, s, metrics, defer, ctrs, counters ? 1 : 0);
  return hipGetLastError();
}
hipError_t run_end(const Metrics* metrics, const uint64_t* conflicts, const uint64_t* combined, const uint32_t* defer,
                   RunResult* out, hipStream_t s) {
  hipLaunchKernelGGL(k_run_end, dim3(1), dim3(256), 0, s, metrics, conflicts, combined, defer, out);
  return hipGetLastError();
}
hipError_t persist_begin(uint64_t* ctrs, hipStream_t s) {
  hipLaunchKernelGGL(k_persist_begin, dim3(1), dim3(64), 0, s, ctrs);
  return hipGetLastError();
}
hipError_t clock_sample(uint64_t* out, hipStream_t s) {
  hipLaunchKernelGGL(k_clock_sample, dim3(1), dim3(64), 0, s, out);
  return hipGetLastError();
}

hipError_t batch_begin(uint64_t* ctrs, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_begin, dim3(1), dim3(64), 0, s, ctrs);
  return hipGetLastError();
}

}  // namespace launch
}  // namespace gcctb
