// Edge-list preprocessing for the fused scatter (gfx950): range checks of the edge
// indices and a stable sort of edge ids by destination, giving CSR row pointers.
//
// The reference adds messages with scatter_add_ (e3nn/nn/models/v2106/points_convolution.py:13-17);
// grouping the edges of one destination lets one wavefront sum them in registers and
// write each output row exactly once.  The sort is integer-only and stable, so the
// permutation (and therefore the summation order) is unique for a given edge list.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <mutex>

#include <rocprim/rocprim.hpp>

#include "e3x_internal.h"

namespace {

constexpr int kBlock = 256;

__device__ int d_flag[4];  // range-check result of e3x_index_check (one copy per device)
std::mutex g_flag_mutex;   // one check at a time: concurrent callers would share the flag

// Sort buffers of e3x_csr_build_static.  Every device the library runs on holds its own copy of this array at its
// own address for the life of the process; host code must use the address hipGetSymbolAddress reports for the
// current device (static_scratch() below), never the array's name.
constexpr size_t kStaticScratchBytes = 64u << 20;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
constexpr int kMaxDevices = 64;
void* g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mutex;
// one call at a time per device: the callers of a device share its array, and a call ends with the stream synchronised
// (the range-check read-back), so holding the lock from the first launch to that point makes host threads take turns
std::mutex g_scratch_busy[kMaxDevices];

// device address of `scratch` on the current device, looked up once per device
int static_scratch(void** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return e3x::fail(E3X_ERR_HIP, "e3x_csr_build_static: no current HIP device");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
      return e3x::fail(E3X_ERR_HIP, "e3x_csr_build_static: hipGetSymbolAddress failed");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return E3X_OK;
}

template <typename IdxT>
__global__ __launch_bounds__(kBlock) void keys_kernel(const IdxT* __restrict__ dst, long long E, long long N,
                                                      unsigned* __restrict__ keys, int* __restrict__ ids,
                                                      int* __restrict__ flags) {
  bool bad = false;
  for (long long e = (long long)blockIdx.x * kBlock + threadIdx.x; e < E; e += (long long)gridDim.x * kBlock) {
    const long long d = (long long)dst[e];
    if (d < 0 || d >= N) bad = true;
    keys[e] = (unsigned)d;
    ids[e] = (int)e;
  }
  if (bad) atomicOr(&flags[0], 1);
}

template <typename IdxT>
__global__ __launch_bounds__(kBlock) void range_kernel(const IdxT* __restrict__ idx, long long E, long long N,
                                                       int* __restrict__ flags) {
  bool bad = false;
  for (long long e = (long long)blockIdx.x * kBlock + threadIdx.x; e < E; e += (long long)gridDim.x * kBlock) {
    const long long d = (long long)idx[e];
    if (d < -N || d >= N) bad = true;
  }
  if (bad) atomicOr(&flags[0], 1);
}

// src_rows[k] = source row of the edge at position k of the destination-sorted list, negative values wrapped
template <typename IdxT>
__global__ __launch_bounds__(kBlock) void src_rows_kernel(const IdxT* __restrict__ src, const int* __restrict__ perm,
                                                          long long E, long long n_src, int* __restrict__ src_rows) {
  for (long long k = (long long)blockIdx.x * kBlock + threadIdx.x; k < E; k += (long long)gridDim.x * kBlock) {
    long long s = (long long)src[perm ? perm[k] : k];
    if (s < 0) s += n_src;
    src_rows[k] = (int)s;
  }
}

// rowptr[n] = first position k with sorted_key[k] >= n   (n = 0..N)
__global__ __launch_bounds__(kBlock) void rowptr_kernel(const unsigned* __restrict__ sorted, long long E,
                                                        long long N, int* __restrict__ rowptr) {
  for (long long n = (long long)blockIdx.x * kBlock + threadIdx.x; n <= N; n += (long long)gridDim.x * kBlock) {
    long long lo = 0, hi = E;
    while (lo < hi) {
      const long long mid = (lo + hi) >> 1;
      if ((long long)sorted[mid] < n) lo = mid + 1; else hi = mid;
    }
    rowptr[n] = (int)lo;
  }
}

// key[n] = smallest source row among the in-edges of output row n (all ones for a row without edges), second[n] the
// smallest one above it, ids[n] = n
template <typename IdxT>
__global__ __launch_bounds__(kBlock) void rowkey_kernel(const IdxT* __restrict__ src, const int* __restrict__ rowptr,
                                                        const int* __restrict__ perm, long long N, long long n_src,
                                                        unsigned* __restrict__ keys, unsigned* __restrict__ second,
                                                        int* __restrict__ ids) {
  for (long long n = (long long)blockIdx.x * kBlock + threadIdx.x; n < N; n += (long long)gridDim.x * kBlock) {
    unsigned k1 = 0xffffffffu, k2 = 0xffffffffu;
    for (int k = rowptr[n]; k < rowptr[n + 1]; ++k) {
      long long s = (long long)src[perm ? perm[k] : k];
      if (s < 0) s += n_src;  // gather semantics: negative indices wrap
      const unsigned v = (unsigned)s;
      if (v < k1) {
        k2 = k1;
        k1 = v;
      } else if (v > k1 && v < k2) {
        k2 = v;
      }
    }
    keys[n] = k1;
    second[n] = k2;
    ids[n] = (int)n;
  }
}

// whether rows a and b, b next to a in an order, have the same two smallest sources
__device__ __forceinline__ bool counts_as_shared(const unsigned* __restrict__ keys, const unsigned* __restrict__ second, int a, int b) {
  return keys[a] != 0xffffffffu && keys[a] == keys[b] && second[a] != 0xffffffffu && second[a] == second[b];
}

// counts the neighbours in the order that agree in BOTH smallest sources: chance alone makes rows share one
// (a small id is the minimum of many rows), two in common mean overlapping source sets
__global__ __launch_bounds__(kBlock) void order_score_kernel(const int* __restrict__ order, const unsigned* __restrict__ keys,
                                                             const unsigned* __restrict__ second, long long N,
                                                             int* __restrict__ score) {
  int hits = 0;
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i + 1 < N; i += (long long)gridDim.x * kBlock) {
    if (counts_as_shared(keys, second, order[i], order[i + 1])) ++hits;
  }
  if (hits) atomicAdd(score, hits);
}

// One more level of the row key for graphs whose sources and destinations are the same node set:
// level[n] <- key[level[n]] (the smallest source of the row's current key node), and its value for the rows in
// their current order
__global__ __launch_bounds__(kBlock) void level_key_kernel(const int* __restrict__ order, const unsigned* __restrict__ keys,
                                                           unsigned* __restrict__ level, unsigned* __restrict__ by_position,
                                                           long long N, int first) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < N; i += (long long)gridDim.x * kBlock) {
    const int n = order[i];
    const unsigned prev = first ? keys[n] : level[n];  // each row appears once in `order`: no other thread touches level[n]
    const unsigned next = prev < (unsigned)N ? keys[prev] : 0xffffffffu;
    level[n] = next;
    by_position[i] = next;
  }
}

__global__ __launch_bounds__(kBlock) void fill_zero_kernel(int* p, int n) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

// one 16-byte element per thread and a grid that covers the buffer once
__global__ __launch_bounds__(kBlock) void copy16_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                        size_t n16) {
  const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n16) dst[i] = src[i];
}

// One wavefront per row: reads the row's in16 16-byte pieces (consecutive rows are stored one after the other) with
// non-temporal loads, eight 1 KB instructions in flight, folds them with XOR and writes out16 pieces of the fold.
typedef unsigned stream_u32x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(kBlock) void stream_rows_kernel(const stream_u32x4* __restrict__ in, long long in16,
                                                             long long n_rows, stream_u32x4* __restrict__ out, int out16) {
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * (kBlock / 64) + threadIdx.x / 64;
  if (row >= n_rows) return;
  const stream_u32x4* p = in + row * in16;
  stream_u32x4 acc = {0u, 0u, 0u, 0u};
  for (long long i = lane; i < in16; i += 64 * 8) {
    stream_u32x4 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
      v[k] = i + 64 * k < in16 ? __builtin_nontemporal_load(p + i + 64 * k) : stream_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 8; ++k) acc ^= v[k];
  }
  for (int q = lane; q < out16; q += 64) out[row * out16 + q] = acc;
}

__global__ __launch_bounds__(kBlock) void fill_zero_bytes_kernel(unsigned char* p, size_t n) {
  // 16-byte stores over the aligned middle, byte stores at the ragged ends
  const size_t head = (16 - ((uintptr_t)p & 15)) & 15;
  const size_t h = head < n ? head : n;
  const size_t n16 = (n - h) / 16;
  const size_t tid = (size_t)blockIdx.x * kBlock + threadIdx.x, stride = (size_t)gridDim.x * kBlock;
  uint4* mid = reinterpret_cast<uint4*>(p + h);
  for (size_t i = tid; i < n16; i += stride) mid[i] = make_uint4(0, 0, 0, 0);
  if (tid < h) p[tid] = 0;
  const size_t tail0 = h + n16 * 16;
  if (tid < n - tail0) p[tail0 + tid] = 0;
}

// ---- edge list in one pass: e3x_edges_build ---------------------------------------------------------------
// Counting sort by destination.  What bounds the set-up of a neighbour list is launches and host round trips, not bytes:
// 176 852 edges on 5 003 nodes took four library sorts (some 30 launches, 0.17 ms of kernels) and four stream
// synchronisations.  Here: counts, one or two scan kernels, placement, one pass over the rows, one ranking kernel, one
// read-back.
//   count    rank of an edge inside its row by an atomic on the row's counter; neighbouring lanes with the same
//            destination take one atomic together, so a list that is already grouped costs one atomic per run.  The
//            ranks depend on the order of the atomics;
//   place    edge ids at rowptr[row] + rank;
//   rows     a wavefront per row puts its ids in ascending order (the stable order, whatever the ranks were) and finds the
//            row's two smallest sources.  A list that was grouped already skips the sorting (perm is the identity);
//   order    rows ranked by their key by counting smaller keys.
constexpr int kScanTile = 4096;
// Up to here the second of the two scan kernels does without the first: adding up three tiles before one's own is less than a
// launch.  With the one ranking kernel below, set-up and step of a block on 5003 nodes 355 -> 339 us.
constexpr unsigned kScanTilesDirect = 4;
constexpr int kRowMax = 1024;  // longest row that is put in order here
enum { kBadSrc = 0, kBadDst, kUnsorted, kOverflow, kScore, kFlags };

__global__ __launch_bounds__(kBlock) void edges_zero_kernel(int* __restrict__ p, long long n) {
  for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long long)gridDim.x * kBlock) p[i] = 0;
}

// *flag = 1 where any thread of the workgroup says so.  One store a workgroup, none where it is set already: an atomic of
// every thread on the one word took 0.13 ms on a list of 1.9 million edges in no order.
__device__ __forceinline__ void raise(int* flag, bool set) {
  if (__syncthreads_or(set) && threadIdx.x == 0 && __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    __hip_atomic_store(flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename SrcT, typename DstT>
__global__ __launch_bounds__(kBlock) void edges_count_kernel(const SrcT* __restrict__ src, const DstT* __restrict__ dst, long long E,
                                                             long long N, long long n_src, int* __restrict__ counts,
                                                             int* __restrict__ rank, int* __restrict__ flags) {
  const int lane = threadIdx.x & 63;
  bool bad_s = false, bad_d = false, unsorted = false;
  const long long e_end = (E + 63) / 64 * 64;  // whole wavefronts: the shuffles run with every lane
  for (long long e = (long long)blockIdx.x * kBlock + threadIdx.x; e < e_end; e += (long long)gridDim.x * kBlock) {
    const bool live = e < E;
    long long d = -1;
    if (live) {
      d = (long long)dst[e];
      const long long s = (long long)src[e];
      if (s < -n_src || s >= n_src) bad_s = true;
      if (d < 0 || d >= N) {
        bad_d = true;
        d = -1;
      }
    }
    const int key = (int)d;
    int prev = __shfl_up(key, 1, 64);
    if (lane == 0 && e > 0 && live) prev = (int)(long long)dst[e - 1];
    if (live && e > 0 && prev > key) unsorted = true;
    const unsigned long long heads = __ballot(lane == 0 || prev != key);
    const unsigned long long upto = heads & (~0ull >> (63 - lane));
    const int head = 63 - __clzll((long long)upto);
    const unsigned long long after = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
    const int end = after ? __ffsll((long long)after) - 1 : 64;
    int base = 0;
    if (lane == head && key >= 0) base = atomicAdd(&counts[key], end - head);
    base = __shfl(base, head, 64);
    if (live) rank[e] = base + lane - head;
  }
  if (bad_s) atomicOr(&flags[kBadSrc], 1);
  if (bad_d) atomicOr(&flags[kBadDst], 1);
  raise(&flags[kUnsorted], unsorted);
}

// sums[b] = sum of tile b of the counts
__global__ __launch_bounds__(kBlock) void edges_scan_sums_kernel(const int* __restrict__ counts, long long N, int* __restrict__ sums) {
  __shared__ int part[kBlock / 64];
  const long long i0 = (long long)blockIdx.x * kScanTile;
  int v = 0;
  for (int i = threadIdx.x; i < kScanTile; i += kBlock) v += i0 + i < N ? counts[i0 + i] : 0;
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  if (threadIdx.x % 64 == 0) part[threadIdx.x / 64] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kBlock / 64; ++i) v += part[i];
    sums[blockIdx.x] = v;
  }
}

// rowptr[n] = sum of counts[0 .. n - 1], n = 0 .. N; every workgroup adds up the sums of the tiles before its own, or, where
// these are not given, the counts themselves
__global__ __launch_bounds__(kBlock) void edges_scan_kernel(const int* __restrict__ counts, long long N, const int* __restrict__ sums,
                                                            int* __restrict__ rowptr) {
  __shared__ int part[kBlock / 64], wsum[kBlock / 64];
  constexpr int PER = kScanTile / kBlock;
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  int before = 0;
  if (sums) {
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kBlock) before += sums[i];
  } else {
#pragma unroll 16
    for (int i = threadIdx.x; i < (int)blockIdx.x * kScanTile; i += kBlock) before += counts[i];
  }
  for (int off = 32; off >= 1; off >>= 1) before += __shfl_xor(before, off, 64);
  if (lane == 0) part[wave] = before;
  const long long i0 = (long long)blockIdx.x * kScanTile + threadIdx.x * PER;
  int c[PER], mine = 0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    c[k] = i0 + k < N ? counts[i0 + k] : 0;
    mine += c[k];
  }
  int incl = mine;
  for (int off = 1; off < 64; off <<= 1) {
    const int t = __shfl_up(incl, off, 64);
    if (lane >= off) incl += t;
  }
  if (lane == 63) wsum[wave] = incl;
  __syncthreads();
  int run = incl - mine;
  for (int i = 0; i < kBlock / 64; ++i) {
    run += part[i];
    if (i < wave) run += wsum[i];
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if (i0 + k <= N) rowptr[i0 + k] = run;
    run += c[k];
  }
}

template <typename DstT>
__global__ __launch_bounds__(kBlock) void edges_place_kernel(const DstT* __restrict__ dst, long long E, long long N,
                                                             const int* __restrict__ rowptr, const int* __restrict__ rank,
                                                             const int* __restrict__ flags, int* __restrict__ placed) {
  if (!flags[kUnsorted]) return;
  for (long long e = (long long)blockIdx.x * kBlock + threadIdx.x; e < E; e += (long long)gridDim.x * kBlock) {
    const long long d = (long long)dst[e];
    if (d >= 0 && d < N) placed[rowptr[d] + rank[e]] = (int)e;
  }
}

// smallest and second smallest distinct value of the two pairs
__device__ __forceinline__ void merge_two_smallest(unsigned& k1, unsigned& k2, unsigned a1, unsigned a2) {
  const unsigned lo = k1 < a1 ? k1 : a1, hi = k1 < a1 ? a1 : k1;  // lo <= hi
  const unsigned rest = k2 < a2 ? k2 : a2;
  k1 = lo;
  k2 = hi > lo && hi < rest ? hi : rest;  // (a pair's second is larger than its first, so rest > lo)
}

template <typename SrcT>
__global__ __launch_bounds__(kBlock) void edges_rows_kernel(const SrcT* __restrict__ src, const int* __restrict__ rowptr,
                                                            const int* __restrict__ placed, long long N, long long n_src,
                                                            int* __restrict__ perm, unsigned* __restrict__ keys,
                                                            unsigned* __restrict__ second, int* __restrict__ flags) {
  __shared__ int ids[kBlock / 64][kRowMax];
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  const long long row = (long long)blockIdx.x * (kBlock / 64) + wave;
  if (row >= N) return;
  const bool sorted = !flags[kUnsorted];
  const int beg = rowptr[row], n = rowptr[row + 1] - beg;
  if (!sorted && n > kRowMax) {  // the host takes the general sort
    if (lane == 0) atomicOr(&flags[kOverflow], 1);
    return;
  }
  unsigned k1 = 0xffffffffu, k2 = 0xffffffffu;
  for (int i = lane; i < n; i += 64) {
    const int id = sorted ? beg + i : placed[beg + i];
    if (!sorted) ids[wave][i] = id;
    else perm[beg + i] = id;
    long long s = (long long)src[id];
    if (s < 0) s += n_src;
    const unsigned v = (unsigned)s;
    if (v < k1) {
      k2 = k1;
      k1 = v;
    } else if (v > k1 && v < k2) {
      k2 = v;
    }
  }
  if (!sorted) {
    // (one wavefront wrote these and reads them back: its LDS operations complete in order)
    __builtin_amdgcn_wave_barrier();
    for (int i = lane; i < n; i += 64) {
      const int id = ids[wave][i];
      int smaller = 0;
      for (int j = 0; j < n; ++j) smaller += ids[wave][j] < id;
      perm[beg + smaller] = id;
    }
  }
  if (keys) {
    for (int off = 32; off >= 1; off >>= 1) {
      const unsigned a1 = (unsigned)__shfl_xor((int)k1, off, 64), a2 = (unsigned)__shfl_xor((int)k2, off, 64);
      merge_two_smallest(k1, k2, a1, a2);
    }
    if (lane == 0) {
      keys[row] = k1;
      second[row] = k2;
    }
  }
}

// The position of a row in the order of (key of the key of its key, key of its key, key, number), the last three levels
// only for one node set, found by counting the rows in front of it: N^2 comparisons spread over the chip.  The row that
// follows comes out of the same comparisons, and with it the pairs that order_score_kernel counts.  A workgroup takes ROWS
// rows, its 16 wavefronts a sixteenth of every tile of keys, and the 64 / ROWS groups of lanes of a wavefront every
// (64 / ROWS)th of these.
// A step of few rows has few workgroups, and waits for the vector ALU (and to look up levels in memory, when it did) of the CUs
// that have one.  Together with the count of the pairs as a kernel of its own, 64 rows a workgroup and 64-bit integers took
// 7.5 / 8.5 / 17.4 / 23.1 / 32.1 / 46.5 us for 200 / 1000 / 5003 / 8192 / 12 000 / 16 384 rows; 16 rows 4.5 / 4.9 / 12.0 /
// 17.2 / 31.3 / 50.6, 32 rows 5.3 / 5.5 / 12.5 / 16.8 / 32.0 / 42.7, 8 rows more from 1000 on (each workgroup reads all keys).
constexpr long long kRankMax = 16384, kRankNarrow = 8192;  // (up to which: 16 rows)
constexpr int kRankTile = 2048;
template <int ROWS>
__global__ __launch_bounds__(1024) void edges_order_kernel(const unsigned* __restrict__ keys, const unsigned* __restrict__ second,
                                                           int N, int levels, int* __restrict__ order, int* __restrict__ score) {
  constexpr int GROUPS = 64 / ROWS, PER_WAVE = kRankTile / 16;
  constexpr unsigned kNone = 0x7fe00000u;  // upper word of a number above every row's
  __shared__ unsigned short key_of[kRankMax];
  __shared__ double2 tile[kRankTile / 2];
  __shared__ double part_next[16][ROWS];
  __shared__ int part[16][ROWS];
  // the keys as 16 bits (sources are numbered below 65535; a row without edges 65535), so that the levels are looked up in LDS
  for (int i = threadIdx.x; i < N; i += 1024) key_of[i] = (unsigned short)keys[i];
  __syncthreads();
  // A row's levels and number as the bits of a positive normal double, whose order is that of the bits: one compare and one
  // minimum a key where 64-bit integers take twice the instructions
  auto composite = [&](int n) {
    const int k = key_of[n];
    int l1 = 0, l2 = 0;
    if (levels) {
      l1 = k < N ? key_of[k] : 0xffff;
      l2 = l1 < N ? min((int)key_of[l1], (int)kRankMax) : (int)kRankMax;  // (at least N where there is none)
    }
    return __hiloint2double((l2 + 0x10) << 16 | l1, k << 16 | n);
  };
  const int lane = threadIdx.x & 63, wave = threadIdx.x / 64;
  const int row = blockIdx.x * ROWS + lane % ROWS, group = lane / ROWS;
  const double mine = composite(row < N ? row : N - 1);
  double next = __hiloint2double((int)kNone, 0);
  int upto = 0;  // rows in front of this one, and itself
  auto take = [&](double k) {
    const bool le = k <= mine;
    upto += le;
    const double above = __hiloint2double(le ? (int)kNone : __double2hiint(k), __double2loint(k));
    asm("v_min_f64 %0, %1, %2" : "=v"(next) : "v"(next), "v"(above));
  };
  for (int t0 = 0; t0 < N; t0 += kRankTile) {
    __syncthreads();
    for (int i = threadIdx.x; i < kRankTile; i += 1024)
      reinterpret_cast<double*>(tile)[i] = t0 + i < N ? composite(t0 + i) : __hiloint2double((int)kNone, 0);
    __syncthreads();
#pragma unroll 8
    for (int i = 0; i < PER_WAVE / 2 / GROUPS; ++i) {
      const double2 k = tile[wave * (PER_WAVE / 2) + i * GROUPS + group];
      take(k.x);
      take(k.y);
    }
  }
  for (int off = 32; off >= ROWS; off >>= 1) {
    upto += __shfl_xor(upto, off, 64);
    next = fmin(next, __shfl_xor(next, off, 64));
  }
  if (group == 0) {
    part[wave][lane] = upto;
    part_next[wave][lane] = next;
  }
  __syncthreads();
  if (wave == 0) {
    bool hit = false;
    if (group == 0 && row < N) {
      for (int i = 1; i < 16; ++i) {
        upto += part[i][lane];
        next = fmin(next, part_next[i][lane]);
      }
      order[upto - 1] = row;
      if ((unsigned)__double2hiint(next) < kNone) hit = counts_as_shared(keys, second, row, __double2loint(next) & 0xffff);
    }
    const int hits = __popcll(__ballot(hit));
    if (lane == 0 && hits) atomicAdd(score, hits);
  }
}

unsigned grid_for(long long n, int per_block) {
  long long b = (n + per_block - 1) / per_block;
  if (b < 1) b = 1;
  if (b > 256 * 16) b = 256 * 16;
  return (unsigned)b;
}

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

int key_bits(long long N) {
  int b = 1;
  while ((1LL << b) < N) ++b;
  return b;
}

size_t sort_temp_bytes(long long E, long long N) {
  size_t temp = 0;
  (void)rocprim::radix_sort_pairs(nullptr, temp, (unsigned*)nullptr, (unsigned*)nullptr, (int*)nullptr, (int*)nullptr,
                            (size_t)E, 0, key_bits(N), (hipStream_t)0);
  return temp;
}

}  // namespace

int e3x::fill_zero_bytes(void* p, size_t n_bytes, void* stream) {
  if (n_bytes == 0) return E3X_OK;
  hipLaunchKernelGGL(fill_zero_bytes_kernel, dim3(grid_for((long long)(n_bytes / 16 + 1), kBlock)), dim3(kBlock), 0,
                     (hipStream_t)stream, (unsigned char*)p, n_bytes);
  return hipGetLastError() == hipSuccess ? E3X_OK : e3x::fail(E3X_ERR_HIP, "zero-fill launch failed");
}

extern "C" size_t e3x_csr_workspace_bytes(int64_t E, int64_t num_nodes) {
  if (E < 0 || num_nodes < 0) return 0;
  const size_t e4 = align_up((size_t)E * 4, 256);
  // flags | keys_in | keys_out | ids_in | rocPRIM temp
  return 256 + 3 * e4 + align_up(sort_temp_bytes(E > 0 ? E : 1, num_nodes > 1 ? num_nodes : 2), 256);
}

extern "C" int e3x_csr_build_static(const void* dst, int idx_bits, int64_t E, int64_t num_nodes, int32_t* rowptr,
                                    int32_t* perm, void* stream) {
  if (E < 0 || num_nodes < 0 || E >= (1LL << 31) || num_nodes >= (1LL << 31))
    return e3x::fail(E3X_ERR_INVALID, "e3x_csr_build_static: E and num_nodes must fit in int32");
  const size_t need = e3x_csr_workspace_bytes(E, num_nodes);
  if (need > kStaticScratchBytes) {
    char msg[200];
    snprintf(msg, sizeof msg,
             "e3x_csr_build_static: %lld edges need %zu bytes of sort buffers, the static buffer holds %zu "
             "(use e3x_csr_build with a workspace)", (long long)E, need, kStaticScratchBytes);
    return e3x::fail(E3X_ERR_INVALID, msg);
  }
  if (E == 0) return e3x_csr_build(dst, idx_bits, E, num_nodes, rowptr, perm, nullptr, kStaticScratchBytes, stream);  // touches no scratch
  void* ws = nullptr;
  const int rc = static_scratch(&ws);
  if (rc != E3X_OK) return rc;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return e3x::fail(E3X_ERR_HIP, "e3x_csr_build_static: no current HIP device");
  std::lock_guard<std::mutex> busy(g_scratch_busy[dev]);
  return e3x_csr_build(dst, idx_bits, E, num_nodes, rowptr, perm, ws, kStaticScratchBytes, stream);
}

extern "C" size_t e3x_csr_static_scratch_bytes(void) { return kStaticScratchBytes; }

extern "C" int e3x_csr_build(const void* dst, int idx_bits, int64_t E, int64_t num_nodes, int32_t* rowptr,
                             int32_t* perm, void* workspace, size_t workspace_bytes, void* stream) {
  if (E < 0 || num_nodes < 0 || E >= (1LL << 31) || num_nodes >= (1LL << 31))
    return e3x::fail(E3X_ERR_INVALID, "e3x_csr_build: E and num_nodes must fit in int32");
  if (idx_bits != 32 && idx_bits != 64) return e3x::fail(E3X_ERR_INVALID, "e3x_csr_build: idx_bits must be 32 or 64");
  if (!rowptr || (E > 0 && (!dst || !perm || !workspace)))
    return e3x::fail(E3X_ERR_INVALID, "e3x_csr_build: null pointer");
  if (workspace_bytes < e3x_csr_workspace_bytes(E, num_nodes))
    return e3x::fail(E3X_ERR_INVALID, "e3x_csr_build: workspace smaller than e3x_csr_workspace_bytes()");
  hipStream_t st = (hipStream_t)stream;
  if (E == 0) {
    hipLaunchKernelGGL(fill_zero_kernel, dim3(grid_for(num_nodes + 1, kBlock)), dim3(kBlock), 0, st, rowptr,
                       (int)(num_nodes + 1));
    return hipGetLastError() == hipSuccess ? E3X_OK : e3x::fail(E3X_ERR_HIP, "e3x_csr_build: launch failed");
  }
  const size_t e4 = align_up((size_t)E * 4, 256);
  char* ws = (char*)workspace;
  int* flags = (int*)ws;
  unsigned* keys_in = (unsigned*)(ws + 256);
  unsigned* keys_out = (unsigned*)(ws + 256 + e4);
  int* ids_in = (int*)(ws + 256 + 2 * e4);
  void* temp = ws + 256 + 3 * e4;
  size_t temp_bytes = sort_temp_bytes(E, num_nodes > 1 ? num_nodes : 2);

  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, st, flags, 2);
  if (idx_bits == 64)
    hipLaunchKernelGGL((keys_kernel<long long>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st,
                       (const long long*)dst, (long long)E, (long long)num_nodes, keys_in, ids_in, flags);
  else
    hipLaunchKernelGGL((keys_kernel<int>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, (const int*)dst,
                       (long long)E, (long long)num_nodes, keys_in, ids_in, flags);
  // stable LSD radix sort of (dst, edge id) over the significant key bits only
  hipError_t err = rocprim::radix_sort_pairs(temp, temp_bytes, keys_in, keys_out, ids_in, perm, (size_t)E, 0,
                                             key_bits(num_nodes > 1 ? num_nodes : 2), st);
  if (err != hipSuccess) return e3x::fail(E3X_ERR_HIP, "e3x_csr_build: radix sort failed");
  hipLaunchKernelGGL(rowptr_kernel, dim3(grid_for(num_nodes + 1, kBlock)), dim3(kBlock), 0, st, keys_out, (long long)E,
                     (long long)num_nodes, rowptr);
  int h_flags[2] = {0, 0};
  if (hipMemcpyAsync(h_flags, flags, sizeof(h_flags), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return e3x::fail(E3X_ERR_HIP, "e3x_csr_build: reading back the range flags failed");
  if (h_flags[0]) return e3x::fail(E3X_ERR_INDEX, "index out of range in scatter destination");
  return E3X_OK;
}

extern "C" size_t e3x_row_order_workspace_bytes(int64_t num_nodes) {
  if (num_nodes < 0) return 0;
  const size_t n4 = align_up((size_t)(num_nodes > 0 ? num_nodes : 1) * 4, 256);
  size_t temp = 0;
  (void)rocprim::radix_sort_pairs(nullptr, temp, (unsigned*)nullptr, (unsigned*)nullptr, (int*)nullptr, (int*)nullptr,
                                  (size_t)(num_nodes > 0 ? num_nodes : 1), 0, 32, (hipStream_t)0);
  return 256 + 6 * n4 + align_up(temp, 256);  // score | keys_in | keys_out | ids_in | second | level | level keys | rocPRIM temp
}

extern "C" int e3x_row_order_build(const void* src, int idx_bits, const int32_t* rowptr, const int32_t* perm, int64_t E,
                                   int64_t num_nodes, int64_t num_src_nodes, int32_t* row_order, int32_t* shared_pairs,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  if (E < 0 || num_nodes < 0 || num_src_nodes < 0 || num_nodes >= (1LL << 31) || num_src_nodes >= (1LL << 31))
    return e3x::fail(E3X_ERR_INVALID, "e3x_row_order_build: sizes must fit in int32");
  if (idx_bits != 32 && idx_bits != 64) return e3x::fail(E3X_ERR_INVALID, "e3x_row_order_build: idx_bits must be 32 or 64");
  if (shared_pairs) *shared_pairs = 0;
  if (num_nodes == 0) return E3X_OK;
  if (!rowptr || !row_order || !workspace || (E > 0 && !src)) return e3x::fail(E3X_ERR_INVALID, "e3x_row_order_build: null pointer");
  if (workspace_bytes < e3x_row_order_workspace_bytes(num_nodes))
    return e3x::fail(E3X_ERR_INVALID, "e3x_row_order_build: workspace smaller than e3x_row_order_workspace_bytes()");
  hipStream_t st = (hipStream_t)stream;
  const size_t n4 = align_up((size_t)num_nodes * 4, 256);
  char* ws = (char*)workspace;
  int* score = (int*)ws;
  unsigned* keys_in = (unsigned*)(ws + 256);
  unsigned* keys_out = (unsigned*)(ws + 256 + n4);
  int* ids_in = (int*)(ws + 256 + 2 * n4);
  unsigned* second = (unsigned*)(ws + 256 + 3 * n4);
  unsigned* level = (unsigned*)(ws + 256 + 4 * n4);
  unsigned* level_keys = (unsigned*)(ws + 256 + 5 * n4);
  void* temp = ws + 256 + 6 * n4;
  size_t temp_bytes = workspace_bytes - 256 - 6 * n4;
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, st, score, 1);
  if (idx_bits == 64)
    hipLaunchKernelGGL((rowkey_kernel<long long>), dim3(grid_for(num_nodes, kBlock)), dim3(kBlock), 0, st, (const long long*)src,
                       rowptr, perm, (long long)num_nodes, (long long)num_src_nodes, keys_in, second, ids_in);
  else
    hipLaunchKernelGGL((rowkey_kernel<int>), dim3(grid_for(num_nodes, kBlock)), dim3(kBlock), 0, st, (const int*)src, rowptr,
                       perm, (long long)num_nodes, (long long)num_src_nodes, keys_in, second, ids_in);
  if (hipGetLastError() != hipSuccess) return e3x::fail(E3X_ERR_HIP, "e3x_row_order_build: launch failed");
  // stable: rows with the same key keep their numbering
  hipError_t err = rocprim::radix_sort_pairs(temp, temp_bytes, keys_in, keys_out, ids_in, row_order, (size_t)num_nodes, 0, 32, st);
  if (err != hipSuccess) return e3x::fail(E3X_ERR_HIP, "e3x_row_order_build: radix sort failed");
  // Sources and destinations numbered alike (one node set): two more levels, key of the key.  Rows are then grouped
  // by (smallest source of the smallest source of their smallest source, ..., smallest source), which puts groups of
  // rows with neighbouring key nodes next to each other as well.  Two stable sorts, the most significant level last.
  if (num_src_nodes == num_nodes && num_nodes > 1) {
    int* cur = row_order;
    int* other = ids_in;
    for (int lev = 0; lev < 2; ++lev) {
      hipLaunchKernelGGL(level_key_kernel, dim3(grid_for(num_nodes, kBlock)), dim3(kBlock), 0, st, cur, keys_in, level, level_keys,
                         (long long)num_nodes, lev == 0 ? 1 : 0);
      if (hipGetLastError() != hipSuccess) return e3x::fail(E3X_ERR_HIP, "e3x_row_order_build: launch failed");
      err = rocprim::radix_sort_pairs(temp, temp_bytes, level_keys, keys_out, cur, other, (size_t)num_nodes, 0, 32, st);
      if (err != hipSuccess) return e3x::fail(E3X_ERR_HIP, "e3x_row_order_build: radix sort failed");
      std::swap(cur, other);
    }
    // two sorts: the result is back in row_order
  }
  if (shared_pairs) {
    hipLaunchKernelGGL(order_score_kernel, dim3(grid_for(num_nodes, kBlock)), dim3(kBlock), 0, st, row_order, keys_in, second,
                       (long long)num_nodes, score);
    if (hipMemcpyAsync(shared_pairs, score, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return e3x::fail(E3X_ERR_HIP, "e3x_row_order_build: reading back the score failed");
  }
  return E3X_OK;
}

// Where the counting sort pays and its kernels are safe: rows of moderate average length (a few long ones send the call to
// the general sort after the fact), tile sums that one workgroup adds up.  Whole set-up against the general sorts, 4 to 250
// edges per row: lists that are grouped already 0.16 to 0.98 of the time up to 2 million rows (4 million 1.11); others 0.27
// to 1.00 up to 1.9 million edges, 0.76 to 0.82 at 4 million with the rows ranked as well, else 0.87 to 1.44 at 4 and 8
// million (an atomic and a scattered store an edge against a few passes of a radix sort).  Such lists are therefore looked at
// first, for one read-back more.
static bool counting_sort_fits(int64_t E, int64_t N) { return E > 0 && N > 0 && N <= (1 << 21) && E / N <= 256; }
static bool rank_order_fits(int64_t N, int64_t n_src) { return N <= kRankMax && n_src < 65535; }
constexpr int64_t kCountUnseen = 2000000;

static size_t edges_small_bytes(int64_t E, int64_t N) {
  // flags | counts | tile sums | rank | placed | keys | second
  const size_t n4 = align_up((size_t)N * 4, 256), e4 = align_up((size_t)E * 4, 256);
  return 256 + n4 + align_up((size_t)((N + 1 + kScanTile - 1) / kScanTile) * 4, 256) + 2 * e4 + 2 * n4;
}

extern "C" size_t e3x_edges_workspace_bytes(int64_t E, int64_t num_nodes) {
  if (E < 0 || num_nodes < 0) return 0;
  const size_t general = std::max(e3x_csr_workspace_bytes(E, num_nodes), e3x_row_order_workspace_bytes(num_nodes));
  return std::max(general, counting_sort_fits(E, num_nodes) ? edges_small_bytes(E, num_nodes) : (size_t)256);
}

namespace {
template <typename SrcT, typename DstT>
void launch_edges(const SrcT* src, const DstT* dst, long long E, long long N, long long n_src, int* rowptr, int* perm, int* flags,
                  int* counts, int* sums, int* rank, int* placed, unsigned* keys, unsigned* second, hipStream_t st) {
  const unsigned tiles = (unsigned)((N + 1 + kScanTile - 1) / kScanTile);
  // flags and counters lie next to each other
  hipLaunchKernelGGL(edges_zero_kernel, dim3(grid_for(64 + N, kBlock)), dim3(kBlock), 0, st, flags, 64 + N);
  hipLaunchKernelGGL((edges_count_kernel<SrcT, DstT>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, src, dst, E, N, n_src, counts, rank, flags);
  if (tiles > kScanTilesDirect) hipLaunchKernelGGL(edges_scan_sums_kernel, dim3(tiles), dim3(kBlock), 0, st, counts, N, sums);
  else sums = nullptr;
  hipLaunchKernelGGL(edges_scan_kernel, dim3(tiles), dim3(kBlock), 0, st, counts, N, sums, rowptr);
  hipLaunchKernelGGL((edges_place_kernel<DstT>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, dst, E, N, rowptr, rank, flags, placed);
  hipLaunchKernelGGL((edges_rows_kernel<SrcT>), dim3((unsigned)((N + kBlock / 64 - 1) / (kBlock / 64))), dim3(kBlock), 0, st, src, rowptr,
                     placed, N, n_src, perm, keys, second, flags);
}

template <typename DstT>
__global__ __launch_bounds__(kBlock) void unsorted_kernel(const DstT* __restrict__ dst, long long E, int* __restrict__ flag) {
  bool unsorted = false;
  for (long long e = (long long)blockIdx.x * kBlock + threadIdx.x + 1; e < E; e += (long long)gridDim.x * kBlock)
    if (dst[e] < dst[e - 1]) unsorted = true;
  raise(flag, unsorted);
}

// whether dst is not non-decreasing; flag: a word of device scratch
int read_unsorted(const void* dst, int bits, int64_t E, int* flag, hipStream_t st, int* unsorted) {
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, st, flag, 1);
  if (bits == 64) hipLaunchKernelGGL((unsorted_kernel<long long>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, (const long long*)dst, (long long)E, flag);
  else hipLaunchKernelGGL((unsorted_kernel<int>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, (const int*)dst, (long long)E, flag);
  if (hipMemcpyAsync(unsorted, flag, sizeof(*unsorted), hipMemcpyDeviceToHost, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
    return e3x::fail(E3X_ERR_HIP, "e3x_edges_build: reading back the flags failed");
  return E3X_OK;
}
}  // namespace

extern "C" int e3x_edges_build(const void* src, int src_bits, const void* dst, int dst_bits, int64_t E, int64_t num_nodes,
                               int64_t num_src_nodes, int32_t* rowptr, int32_t* perm, int32_t* row_order, int32_t* grouped,
                               int32_t* shared_pairs, void* workspace, size_t workspace_bytes, void* stream) {
  if (E < 0 || num_nodes < 0 || num_src_nodes < 0 || E >= (1LL << 31) || num_nodes >= (1LL << 31))
    return e3x::fail(E3X_ERR_INVALID, "e3x_edges_build: E and num_nodes must fit in int32");
  if ((src_bits != 32 && src_bits != 64) || (dst_bits != 32 && dst_bits != 64))
    return e3x::fail(E3X_ERR_INVALID, "e3x_edges_build: index widths must be 32 or 64 bits");
  if (!rowptr || (E > 0 && (!src || !dst || !perm)) || !grouped || !shared_pairs || (workspace_bytes && !workspace))
    return e3x::fail(E3X_ERR_INVALID, "e3x_edges_build: null pointer");
  if (workspace_bytes < e3x_edges_workspace_bytes(E, num_nodes))
    return e3x::fail(E3X_ERR_INVALID, "e3x_edges_build: workspace smaller than e3x_edges_workspace_bytes()");
  hipStream_t st = (hipStream_t)stream;
  *grouped = 1;
  *shared_pairs = 0;
  bool order_done = false, counting = counting_sort_fits(E, num_nodes);
  int unsorted = -1;  // not known yet
  if (counting && E > kCountUnseen && !(row_order && rank_order_fits(num_nodes, num_src_nodes))) {
    const int rc = read_unsorted(dst, dst_bits, E, (int*)workspace, st, &unsorted);
    if (rc != E3X_OK) return rc;
    counting = !unsorted;
  }
  if (counting) {
    const size_t n4 = align_up((size_t)num_nodes * 4, 256), e4 = align_up((size_t)E * 4, 256);
    char* p = (char*)workspace;
    int* flags = (int*)p;
    int* counts = (int*)(p += 256);
    int* sums = (int*)(p += n4);
    int* rank = (int*)(p += align_up((size_t)((num_nodes + 1 + kScanTile - 1) / kScanTile) * 4, 256));
    int* placed = (int*)(p += e4);
    unsigned* keys = (unsigned*)(p += e4);
    unsigned* second = (unsigned*)(p += n4);
    const bool ranks = row_order && rank_order_fits(num_nodes, num_src_nodes);
    unsigned* k = ranks ? keys : nullptr;
#define E3X_EDGES(S, D) launch_edges((const S*)src, (const D*)dst, E, num_nodes, num_src_nodes, rowptr, perm, flags, counts, sums, rank, placed, k, second, st)
    if (src_bits == 64 && dst_bits == 64) E3X_EDGES(long long, long long);
    else if (src_bits == 64) E3X_EDGES(long long, int);
    else if (dst_bits == 64) E3X_EDGES(int, long long);
    else E3X_EDGES(int, int);
#undef E3X_EDGES
    if (ranks) {
      const int levels = num_src_nodes == num_nodes && num_nodes > 1 ? 1 : 0;
      const auto launch = [&](auto kernel, int rows) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)((num_nodes + rows - 1) / rows)), dim3(1024), 0, st, keys, second, (int)num_nodes, levels,
                           row_order, flags + kScore);
      };
      if (num_nodes <= kRankNarrow) launch(edges_order_kernel<16>, 16);
      else launch(edges_order_kernel<32>, 32);
    }
    int h[kFlags] = {0};
    if (hipGetLastError() != hipSuccess) return e3x::fail(E3X_ERR_HIP, "e3x_edges_build: launch failed");
    if (hipMemcpyAsync(h, flags, sizeof(h), hipMemcpyDeviceToHost, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
      return e3x::fail(E3X_ERR_HIP, "e3x_edges_build: reading back the flags failed");
    if (h[kBadSrc]) return e3x::fail(E3X_ERR_INDEX, "index out of range in gather source");
    if (h[kBadDst]) return e3x::fail(E3X_ERR_INDEX, "index out of range in scatter destination");
    *grouped = !h[kUnsorted];
    if (!h[kOverflow]) {
      *shared_pairs = ranks ? h[kScore] : 0;
      order_done = ranks;
    } else {  // a row too long to be put in order here
      const int rc = e3x_csr_build(dst, dst_bits, E, num_nodes, rowptr, perm, workspace, workspace_bytes, stream);
      if (rc != E3X_OK) return rc;
    }
  } else {
    int rc = e3x_index_check(src, src_bits, E, num_src_nodes, stream);
    if (rc != E3X_OK) return rc;
    if ((rc = e3x_csr_build(dst, dst_bits, E, num_nodes, rowptr, perm, workspace, workspace_bytes, stream)) != E3X_OK) return rc;
    if (E > 1) {
      if (unsorted < 0 && (rc = read_unsorted(dst, dst_bits, E, (int*)workspace, st, &unsorted)) != E3X_OK) return rc;
      *grouped = !unsorted;
    }
  }
  if (row_order && !order_done)
    return e3x_row_order_build(src, src_bits, rowptr, perm, E, num_nodes, num_src_nodes, row_order, shared_pairs, workspace, workspace_bytes, stream);
  return E3X_OK;
}

extern "C" int e3x_src_rows_build(const void* src, int idx_bits, const int32_t* perm, int64_t E, int64_t num_src_nodes,
                                   int32_t* src_rows, void* stream) {
  if (idx_bits != 32 && idx_bits != 64) return e3x::fail(E3X_ERR_INVALID, "e3x_src_rows_build: idx_bits must be 32 or 64");
  if (E < 0 || num_src_nodes < 0 || num_src_nodes >= (1LL << 31))
    return e3x::fail(E3X_ERR_INVALID, "e3x_src_rows_build: sizes must be in [0, 2^31)");
  if (E == 0) return E3X_OK;
  if (!src || !src_rows) return e3x::fail(E3X_ERR_INVALID, "e3x_src_rows_build: null pointer");
  hipStream_t st = (hipStream_t)stream;
  if (idx_bits == 64)
    hipLaunchKernelGGL((src_rows_kernel<long long>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st,
                       (const long long*)src, perm, (long long)E, (long long)num_src_nodes, src_rows);
  else
    hipLaunchKernelGGL((src_rows_kernel<int>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, (const int*)src, perm,
                       (long long)E, (long long)num_src_nodes, src_rows);
  return hipGetLastError() == hipSuccess ? E3X_OK : e3x::fail(E3X_ERR_HIP, "e3x_src_rows_build: launch failed");
}

extern "C" int e3x_index_check(const void* idx, int idx_bits, int64_t E, int64_t num_nodes, void* stream) {
  if (idx_bits != 32 && idx_bits != 64) return e3x::fail(E3X_ERR_INVALID, "e3x_index_check: idx_bits must be 32 or 64");
  if (E == 0) return E3X_OK;
  if (!idx) return e3x::fail(E3X_ERR_INVALID, "e3x_index_check: null pointer");
  hipStream_t st = (hipStream_t)stream;
  // zero, launch and read-back form one critical section (it ends with a stream synchronisation anyway)
  std::lock_guard<std::mutex> lock(g_flag_mutex);
  int* flag = nullptr;
  if (hipGetSymbolAddress((void**)&flag, HIP_SYMBOL(d_flag)) != hipSuccess)
    return e3x::fail(E3X_ERR_HIP, "e3x_index_check: hipGetSymbolAddress failed");
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(kBlock), 0, st, flag, 1);
  if (idx_bits == 64)
    hipLaunchKernelGGL((range_kernel<long long>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st,
                       (const long long*)idx, (long long)E, (long long)num_nodes, flag);
  else
    hipLaunchKernelGGL((range_kernel<int>), dim3(grid_for(E, kBlock)), dim3(kBlock), 0, st, (const int*)idx,
                       (long long)E, (long long)num_nodes, flag);
  int h = 0;
  if (hipMemcpyAsync(&h, flag, sizeof(int), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return e3x::fail(E3X_ERR_HIP, "e3x_index_check: reading back the range flag failed");
  if (h) return e3x::fail(E3X_ERR_INDEX, "index out of range in gather source");
  return E3X_OK;
}

extern "C" int e3x_copy_bytes(const void* src, void* dst, size_t n_bytes, void* stream) {
  if (n_bytes % 16 || ((uintptr_t)src % 16) || ((uintptr_t)dst % 16))
    return e3x::fail(E3X_ERR_INVALID, "e3x_copy_bytes: size and pointers must be multiples of 16");
  if (n_bytes == 0) return E3X_OK;
  const size_t blocks = (n_bytes / 16 + kBlock - 1) / kBlock;
  if (blocks > 0x7fffffffULL) return e3x::fail(E3X_ERR_INVALID, "e3x_copy_bytes: buffer too large for one launch");
  hipLaunchKernelGGL(copy16_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream, (const uint4*)src,
                     (uint4*)dst, n_bytes / 16);
  return hipGetLastError() == hipSuccess ? E3X_OK : e3x::fail(E3X_ERR_HIP, "e3x_copy_bytes: launch failed");
}

extern "C" int e3x_stream_rows(const void* in, size_t in_bytes_per_row, int64_t n_rows, void* out, size_t out_bytes_per_row,
                               void* stream) {
  if (in_bytes_per_row % 16 || out_bytes_per_row % 16 || ((uintptr_t)in % 16) || ((uintptr_t)out % 16) || n_rows < 0 ||
      out_bytes_per_row > (1u << 20))
    return e3x::fail(E3X_ERR_INVALID, "e3x_stream_rows: sizes and pointers must be multiples of 16, rows of output at most 1 MiB");
  if (n_rows == 0) return E3X_OK;
  if (!in || (out_bytes_per_row && !out)) return e3x::fail(E3X_ERR_INVALID, "e3x_stream_rows: null pointer");
  const int64_t blocks = (n_rows + kBlock / 64 - 1) / (kBlock / 64);
  if (blocks > 0x7fffffffLL) return e3x::fail(E3X_ERR_INVALID, "e3x_stream_rows: too many rows for one launch");
  hipLaunchKernelGGL(stream_rows_kernel, dim3((unsigned)blocks), dim3(kBlock), 0, (hipStream_t)stream,
                     (const stream_u32x4*)in, (long long)(in_bytes_per_row / 16), (long long)n_rows, (stream_u32x4*)out,
                     (int)(out_bytes_per_row / 16));
  return hipGetLastError() == hipSuccess ? E3X_OK : e3x::fail(E3X_ERR_HIP, "e3x_stream_rows: launch failed");
}
