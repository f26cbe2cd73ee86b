// Work items of the block-outer selection kernels: (block, chunk of its CSR
// query list), built on the GPU from the CSR offsets.  Shared by the
// selection forward (nsa_selbo.hip) and dK/dV (nsa_dkdv.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nsa {

// items[i] = {bh * n_blk + j, begin, end, 0}: pair range [begin, end) of q_of_block;
// n_items[0] = item count, n_items[1] = 0 (the work counter of next_item).
// The items of block e are items[first[e] .. first[e + 1]), in query order
// (first: nb + 1 ints, optional).  Every workgroup sums the items of the
// blocks before its own by itself, scans its own and writes their items one a
// thread: one workgroup whose threads each wrote their blocks' items took 190
// us over 4096 blocks (65k items) and 11 us over 2048; this takes 12 and 7.
constexpr int kItemTile = 1024;   // blocks scanned at a time
static inline unsigned sel_items_grid(int nb) {
  const int g = (nb + 31) / 32;
  return (unsigned)(g < 1 ? 1 : (g > 128 ? 128 : g));
}
static __global__ __launch_bounds__(256) void k_sel_items(const int32_t* __restrict__ offsets, int nb, int n_blk,
                                                          int chunk, int4* __restrict__ items,
                                                          int32_t* __restrict__ n_items,
                                                          int32_t* __restrict__ first = nullptr) {
  __shared__ int sfirst[kItemTile], sbeg[kItemTile], send[kItemTile];
  __shared__ int wsum[4];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int per = (nb + (int)gridDim.x - 1) / (int)gridDim.x;
  const int lo = (int)blockIdx.x * per < nb ? (int)blockIdx.x * per : nb;
  const int hi = lo + per < nb ? lo + per : nb;
  auto range = [&](int e, int& beg, int& end) {
    const int r = e + e / n_blk;   // row bh of n_blk + 1 offsets
    beg = offsets[r];
    end = offsets[r + 1];
  };
  // sum of x over the workgroup; excl: this thread's exclusive prefix
  auto scan = [&](int x, int& excl) {
    int incl = x;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(incl, off, 64);
      incl += lane >= off ? y : 0;
    }
    __syncthreads();   // wsum's last readers are done
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0, total = 0;
    for (int i = 0; i < 4; ++i) {
      before += i < w ? wsum[i] : 0;
      total += wsum[i];
    }
    excl = before + incl - x;
    return total;
  };
  int cnt = 0, ex;
#pragma unroll 4
  for (int e = tid; e < lo; e += 256) {
    int beg, end;
    range(e, beg, end);
    cnt += (end - beg + chunk - 1) / chunk;
  }
  int pos = scan(cnt, ex);   // items of the blocks before lo
  for (int t0 = lo; t0 < hi; t0 += kItemTile) {
    const int nt = hi - t0 < kItemTile ? hi - t0 : kItemTile;
    int n[4], mine = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = 4 * tid + u;
      n[u] = 0;
      if (i < nt) {
        int beg, end;
        range(t0 + i, beg, end);
        sbeg[i] = beg;
        send[i] = end;
        n[u] = (end - beg + chunk - 1) / chunk;
      }
      mine += n[u];
    }
    const int total = scan(mine, ex);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int i = 4 * tid + u;
      if (i < nt) {
        sfirst[i] = ex;
        if (first != nullptr) first[t0 + i] = pos + ex;
      }
      ex += n[u];
    }
    __syncthreads();
    for (int i = tid; i < total; i += 256) {
      int b = 0;   // the last block whose first item is at most i (the one that holds it)
      for (int step = kItemTile / 2; step > 0; step >>= 1)
        if (b + step < nt && sfirst[b + step] <= i) b += step;
      const int s0 = sbeg[b] + (i - sfirst[b]) * chunk;
      items[pos + i] = make_int4(t0 + b, s0, s0 + chunk < send[b] ? s0 + chunk : send[b], 0);
    }
    pos += total;
    __syncthreads();
  }
  if (blockIdx.x == gridDim.x - 1 && tid == 0) {
    n_items[0] = pos;
    n_items[1] = 0;
    if (first != nullptr) first[nb] = pos;
  }
}

// Next work item of a persistent grid over `total` items: the first
// gridDim.x go to the workgroups in order, each later one to the workgroup
// that asks first (the hardware dispatches workgroups as slots free up, so
// both halves balance dynamically).  Called by every thread of the workgroup
// after a barrier that follows its last read of *slot.
__device__ __forceinline__ int next_item(int32_t* counter, int* slot) {
  if (threadIdx.x == 0) *slot = (int)gridDim.x + atomicAdd(counter, 1);
  __syncthreads();
  return *slot;
}

// Selection blocks of the CSR consumed by the block-outer kernels: every
// block holding a key, the trailing partial one included (the forward attends
// to it when selected).
__host__ __device__ inline int sel_csr_blocks(int T, int block_size) { return (T + block_size - 1) / block_size; }

static inline size_t sel_items_cap(int B, int Hkv, int T, int S, int block_size, int chunk) {
  const size_t nb = (size_t)B * Hkv * sel_csr_blocks(T, block_size);
  const size_t pairs = (size_t)B * Hkv * T * S;
  return nb + (pairs + chunk - 1) / chunk + 1;
}

// CSR queries per selection work item: the largest power of two that still
// gives every resident slot of the kernel an item of a sequence this short, so
// that a few blocks' queries do not run on a few CUs.  An item costs its
// block's keys (forward: 64 keys of K and V^T; dK/dV: also K^T and 64 float
// rows of dK and dV written and summed again), which sets both ends.
// Measured, us, forward at chunks 128 / the rule's and dK/dV at 512 / the
// rule's: B1 T1301 Hq64 Hkv4 D128 163 / 103 (64); B1 T2048 Hq16 Hkv1 D128
// 159 / 62 (32) and 442 / 93 (64); T1024 Hq4 D64 float32 106 / 33 (16) and 445
// / 91 (32); T6011 Hq16 Hkv4 D64 dK/dV 297 / 242 (256); T32768 Hq64 Hkv4 D128
// dK/dV 4732 (512, four and more rounds of items) against 4790 at 256.
__host__ __device__ inline int sel_item_chunk(int64_t pairs, int64_t slots, int lo, int hi) {
  int c = lo;
  while (c < hi && pairs / slots >= 2 * c) c *= 2;
  return c;
}
// The slots are those of 256 compute units, whatever the device has: the chunk
// sizes workspaces too, and their queries are not told a stream.
static inline int sel_fwd_chunk(int64_t pairs) {
  return sel_item_chunk(pairs, 4 * 256, 16, 128);   // one wave per SIMD
}
static inline int sel_dkdv_chunk(int64_t pairs) {
  constexpr int64_t kSlots = 2 * 256;   // two workgroups per CU
  return pairs >= 4 * 512 * kSlots ? 512 : sel_item_chunk(pairs, kSlots, 32, 256);
}

// Most CSR entries in one selection work item (the kernels stage an item's
// entries in LDS); the item chunk passed to the entry points is capped here.
constexpr int kSelItemMax = 1024;

// Keys of a selection block handled per pass of the block-outer kernels; a
// block longer than this is split into ceil(L / kSelPass) partial slots.
constexpr int kSelPass = 64;

// Largest GQA group whose selection row tiles hold floor(32 / G) >= 3 entries
// (G heads each) instead of two queries x 16 head slots.
constexpr int kGroupPackMaxG = 10;
__host__ __device__ inline int sel_passes(int block_size) { return (block_size + kSelPass - 1) / kSelPass; }

// Packed (query, slot) entries of the CSR built with pack_slot:
// (t << sel_slot_bits(S)) | s, so that the kernels split them with a shift
// and a mask; they sort like (t, s).
__host__ __device__ inline int sel_slot_bits(int S) {
  int b = 0;
  while ((1 << b) < S) ++b;
  return b;
}

// Slot of a selected block j in row t is valid (has a CSR pair) iff
// 0 <= j < n_csr and j * L <= t.
__device__ __forceinline__ bool sel_slot_valid(int j, int n_csr, int L, int t) {
  return j >= 0 && j < n_csr && (int64_t)j * L <= t;
}

}  // namespace nsa
