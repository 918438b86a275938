// ccp's cell list of a device position array with no allocation: the
// counterpart of ccp_cell_list for callers that cannot allocate device
// memory (code under hipGraph capture, serving loops, harnesses that forbid
// hipMalloc). The caller passes the positions and the four output arrays;
// the only other device memory the kernels use is `scratch` below, a
// file-scope array of fixed size that each GPU holds for the life of the
// process.
//
// Result: sci/soi are the cell keys and bead indices sorted stably by cell,
// beg/end the slot range of every cell with empty cells 0/0 -- the arrays of
// ccp's sugrid::generate_arrays (sugrid.cu:125-133: calc_indexes, a stable
// radix sort of (cell, index), set_cells_empty, find_cells_limits), bit for
// bit the arrays ccp_cell_list returns for the same positions and geometry.
//
// Method (a counting sort that keeps its state in the output arrays):
//   1. end[c] = 0 (a fill kernel, no memset), scratch words and flag = 0
//   2. key of bead i (ccp's floor(r / csl) + cps/2, clamped into the grid;
//      a bead outside raises the flag) into sci[i], end[key] += 1
//   3. exclusive scan of the counts: a block of 256 cells publishes its sum in
//      `scratch` and adds up those of the blocks before it (beyond NA_DIRECT
//      blocks: sums, their scan and the starts as three kernels), then its
//      cells get beg[c] = start and end[c] = start (the scatter cursor)
//   4. soi[atomicAdd(end[key], 1)] = i (arbitrary order within a cell)
//   5. one lane per cell sorts its slots by bead index (the stable order),
//      writes sci[s] = c over them and sets empty cells to 0/0.
// What bounds it is launches and their chains of loads, not bytes: at 100003
// beads over 2 sigma cells the call takes 57 us with five launches, 69 with
// seven (block sums and their scan as kernels of their own). Block sums added
// up by atomics in step 2 cost more than both: neighbouring words of a few
// cache lines, 98 us for that kernel.
// Calls on one GPU share its scratch array, and a scan block waits for words
// of it that another call's clearing would erase: a call holds the GPU's lock
// from its first launch until its stream is done, so that the calls of a
// process on one GPU run one after another, whatever their threads and streams.

#include "ccpmi.h"
#include "host.hpp"

#include <mutex>

namespace ccpmi {
namespace {

constexpr int NA_BLOCK = 256;
constexpr uint32_t NA_MAX_CELLS = 1u << 24; // cps <= 255
constexpr uint32_t NA_MAX_BLOCKS = NA_MAX_CELLS / NA_BLOCK;
constexpr uint32_t NA_FLAG = NA_MAX_BLOCKS; // word of the outside flag
constexpr uint32_t NA_TICKET = NA_FLAG + 1; // blocks of the scan that have started
constexpr uint32_t NA_WORDS = NA_MAX_BLOCKS + 64;
constexpr int NA_MAX_DEVICES = 64;

// 65536 block sums and the flag: 256.25 KiB per GPU
static __device__ __align__(256) uint32_t scratch[NA_WORDS];

__global__ __launch_bounds__(NA_BLOCK) void k_na_clear(uint32_t n_c, uint32_t *end, uint32_t *sc) {
  const uint32_t c = blockIdx.x * NA_BLOCK + threadIdx.x;
  if (c < n_c) end[c] = 0u;
  if (threadIdx.x == 0) sc[blockIdx.x] = 0u;
  if (c < 2u) sc[NA_FLAG + c] = 0u;
}

// ccp's cell coordinate floor(x / csl) + cps/2 (calc_indexes,
// sugrid.cu:26-34), clamped into the grid
__device__ __forceinline__ int na_coord(float x, float csl, int cps, bool &outside) {
  int c = (int)floorf(x / csl) + cps / 2;
  if (c < 0) { c = 0; outside = true; }
  if (c >= cps) { c = cps - 1; outside = true; }
  return c;
}

__global__ __launch_bounds__(NA_BLOCK) void k_na_key(const float *xyz, uint32_t n, float csl, int cps, uint32_t *key,
                                                     uint32_t *count, uint32_t *sc) {
  const uint32_t i = blockIdx.x * NA_BLOCK + threadIdx.x;
  if (i >= n) return;
  bool outside = false;
  const int gx = na_coord(xyz[3 * (size_t)i], csl, cps, outside);
  const int gy = na_coord(xyz[3 * (size_t)i + 1], csl, cps, outside);
  const int gz = na_coord(xyz[3 * (size_t)i + 2], csl, cps, outside);
  const uint32_t k = (uint32_t)((gz * cps + gy) * cps + gx);
  key[i] = k;
  atomicAdd(count + k, 1u);
  if (outside) atomicAdd(sc + NA_FLAG, 1u);
}

// exclusive scan of v over the block's 256 lanes, and the block total
__device__ __forceinline__ uint32_t na_block_scan(uint32_t v, uint32_t &total) {
  __shared__ uint32_t sums[NA_BLOCK / 64];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  uint32_t incl = v;
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t a = __shfl_up(incl, d);
    if (lane >= d) incl += a;
  }
  if (lane == 63) sums[wave] = incl;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for (int w = 0; w < NA_BLOCK / 64; ++w) {
    before += w < wave ? sums[w] : 0u;
    total += sums[w];
  }
  __syncthreads();
  return before + incl - v;
}

// one block: exclusive scan of the nblk block sums in place, each lane
// taking a contiguous run of them
__global__ __launch_bounds__(NA_BLOCK) void k_na_scan_sums(uint32_t nblk, uint32_t *sc) {
  const uint32_t per = (nblk + NA_BLOCK - 1) / NA_BLOCK;
  const uint32_t b0 = threadIdx.x * per, b1 = min(b0 + per, nblk);
  uint32_t part = 0;
  for (uint32_t b = b0; b < b1; ++b) part += sc[b];
  uint32_t total;
  uint32_t run = na_block_scan(part, total);
  for (uint32_t b = b0; b < b1; ++b) {
    const uint32_t v = sc[b];
    sc[b] = run;
    run += v;
  }
}

__global__ __launch_bounds__(NA_BLOCK) void k_na_block_sums(const uint32_t *count, uint32_t n_c, uint32_t *sc) {
  const uint32_t c = blockIdx.x * NA_BLOCK + threadIdx.x;
  uint32_t total;
  na_block_scan(c < n_c ? count[c] : 0u, total);
  if (threadIdx.x == 0) sc[blockIdx.x] = total;
}

__global__ __launch_bounds__(NA_BLOCK) void k_na_starts(uint32_t *count_cursor, uint32_t n_c, const uint32_t *sc,
                                                        uint32_t *beg) {
  const uint32_t c = blockIdx.x * NA_BLOCK + threadIdx.x;
  uint32_t total;
  const uint32_t ex = na_block_scan(c < n_c ? count_cursor[c] : 0u, total);
  if (c < n_c) {
    const uint32_t start = sc[blockIdx.x] + ex;
    beg[c] = start;
    count_cursor[c] = start;
  }
}

// The same in one launch for up to NA_DIRECT blocks (four words a lane, less
// than the two launches it saves). Blocks are numbered in the order in which
// they start, and each publishes its sum (below 2^31, bit 31 set: sum and flag
// are one word) before it waits for the blocks before it, so every wait ends:
// nothing else writes these words meanwhile (the lock of ccp_cell_list_noalloc).
constexpr uint32_t NA_DIRECT = 1024;
__global__ __launch_bounds__(NA_BLOCK) void k_na_starts_direct(uint32_t *count_cursor, uint32_t n_c, uint32_t *sc,
                                                               uint32_t *beg) {
  __shared__ uint32_t ticket;
  if (threadIdx.x == 0) ticket = atomicAdd(sc + NA_TICKET, 1u);
  __syncthreads();
  const uint32_t blk = ticket, c = blk * NA_BLOCK + threadIdx.x;
  uint32_t total, before;
  const uint32_t ex = na_block_scan(c < n_c ? count_cursor[c] : 0u, total);
  if (threadIdx.x == 0)
    __hip_atomic_store(sc + blk, total | 1u << 31, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  uint32_t part = 0;
  for (uint32_t b = threadIdx.x; b < blk; b += NA_BLOCK) {
    uint32_t v;
    do v = __hip_atomic_load(sc + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    while (!(v >> 31));
    part += v & ~(1u << 31);
  }
  na_block_scan(part, before);
  if (c < n_c) {
    beg[c] = before + ex;
    count_cursor[c] = before + ex;
  }
}

__global__ __launch_bounds__(NA_BLOCK) void k_na_scatter(const uint32_t *key, uint32_t n, uint32_t *cursor,
                                                         uint32_t *soi) {
  const uint32_t i = blockIdx.x * NA_BLOCK + threadIdx.x;
  if (i >= n) return;
  soi[atomicAdd(cursor + key[i], 1u)] = i;
}

__global__ __launch_bounds__(NA_BLOCK) void k_na_finish(uint32_t n_c, uint32_t *beg, uint32_t *end, uint32_t *soi,
                                                        uint32_t *sci) {
  const uint32_t c = blockIdx.x * NA_BLOCK + threadIdx.x;
  if (c >= n_c) return;
  const uint32_t s0 = beg[c], s1 = end[c];
  if (s0 == s1) {
    beg[c] = 0u;
    end[c] = 0u;
    return;
  }
  // insertion sort of the cell's bead indices (cells hold a few beads)
  for (uint32_t s = s0 + 1; s < s1; ++s) {
    const uint32_t v = soi[s];
    uint32_t t = s;
    while (t > s0 && soi[t - 1] > v) {
      soi[t] = soi[t - 1];
      --t;
    }
    soi[t] = v;
  }
  for (uint32_t s = s0; s < s1; ++s) sci[s] = c;
}

// each GPU's lock and the address of its scratch array, looked up once
struct NaDevice {
  std::mutex lock;
  uint32_t *scratch = nullptr;
};
NaDevice g_na[NA_MAX_DEVICES];

// One call on the current GPU: the lock is held until the launches on the
// stream are done, also when the call ends with an error behind them.
struct NaCall {
  std::unique_lock<std::mutex> lock;
  uint32_t *sc = nullptr;
  hipStream_t s;
  bool waiting = true;
  explicit NaCall(hipStream_t stream) : s(stream) {
    int dev = 0;
    host::hip_check(hipGetDevice(&dev));
    if (dev < 0 || dev >= NA_MAX_DEVICES) throw host::Error(CCP_ERR_ARG, "device index beyond the supported range");
    lock = std::unique_lock<std::mutex>(g_na[dev].lock);
    if (!g_na[dev].scratch) {
      void *p = nullptr;
      host::hip_check(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      g_na[dev].scratch = static_cast<uint32_t *>(p);
    }
    sc = g_na[dev].scratch;
  }
  void wait() {
    waiting = false;
    host::hip_check(hipStreamSynchronize(s));
  }
  ~NaCall() {
    if (waiting) (void)hipStreamSynchronize(s);
  }
};

unsigned na_blocks(uint32_t n) { return (n + NA_BLOCK - 1) / NA_BLOCK; }

} // namespace
} // namespace ccpmi

extern "C" int ccp_cell_list_noalloc(const float *xyz, uint32_t n, float csl, uint32_t cps, uint32_t *sci,
                                     uint32_t *soi, uint32_t *beg, uint32_t *end, void *stream) {
  using namespace ccpmi;
  try {
    if (!xyz || !sci || !soi || !beg || !end) throw host::Error(CCP_ERR_ARG, "null array");
    if (n == 0 || n >= (1u << 31)) throw host::Error(CCP_ERR_ARG, "number of objects out of range");
    if (!(csl > 0.0f)) throw host::Error(CCP_ERR_ARG, "cell side out of range");
    if (cps < 1 || (uint64_t)cps * cps * cps >= NA_MAX_CELLS)
      throw host::Error(CCP_ERR_ARG, "cells per side out of range: at most 255 (2^24 cells) without allocation");
    const uint32_t n_c = cps * cps * cps, nblk = na_blocks(n_c);
    hipStream_t s = static_cast<hipStream_t>(stream);
    NaCall call(s);
    uint32_t *sc = call.sc;
    k_na_clear<<<nblk, NA_BLOCK, 0, s>>>(n_c, end, sc);
    k_na_key<<<na_blocks(n), NA_BLOCK, 0, s>>>(xyz, n, csl, (int)cps, sci, end, sc);
    if (nblk <= NA_DIRECT) {
      k_na_starts_direct<<<nblk, NA_BLOCK, 0, s>>>(end, n_c, sc, beg);
    } else {
      k_na_block_sums<<<nblk, NA_BLOCK, 0, s>>>(end, n_c, sc);
      k_na_scan_sums<<<1, NA_BLOCK, 0, s>>>(nblk, sc);
      k_na_starts<<<nblk, NA_BLOCK, 0, s>>>(end, n_c, sc, beg);
    }
    k_na_scatter<<<na_blocks(n), NA_BLOCK, 0, s>>>(sci, n, end, soi);
    k_na_finish<<<nblk, NA_BLOCK, 0, s>>>(n_c, beg, end, soi, sci);
    host::hip_check(hipGetLastError());
    uint32_t outside = 0;
    host::hip_check(hipMemcpyAsync(&outside, sc + NA_FLAG, sizeof(outside), hipMemcpyDeviceToHost, s));
    call.wait();
    if (outside) throw host::Error(CCP_ERR_STATE, "bead left the cell grid");
    return CCP_OK;
  } catch (const host::Error &e) {
    ccpmi::host::set_null_error(e.what());
    return e.code;
  } catch (const std::exception &e) {
    ccpmi::host::set_null_error(e.what());
    return CCP_ERR_ARG;
  }
}
