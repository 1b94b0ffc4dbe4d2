// ks_bins.h - products with matrices whose rows gather x from all over.
//
// With random columns every gather of x is a cache line of its own: x does
// not fit an XCD's 4 MB L2, and even gathers that hit it come one line per
// lane.  Here the gathers are made from LDS instead.  Columns are cut into
// blocks of kBinCols, rows into segments of at most kBinEntries entries, and
// a product takes two passes:
//  1. k_bin_gather, column block by column block: the block's slice of x goes
//     to LDS, and the x of each entry (its 16-bit column within the block
//     streamed in) is written to xg.  xg is ordered by block, then segment.
//  2. k_bin_sum, segment by segment: the segment's runs of xg (one per
//     column block) go to LDS at their entries' places in CSR order
//     (`place`, 16 bits an entry, ordered by segment, then block), are
//     multiplied by the values, which stay in CSR order, and summed by row.
// All passes stream: 28 bytes an entry in FP64 and 16 in FP32 (the column and
// the place 2 each; xg written, then read; the value).  Rows of 4M columns and up
// to 4096 entries (196M in all): FP64 1.59 ms, FP32 0.97 ms.  Row sums form from
// products in CSR order in a fixed order: rows of at most kBinShort entries
// by one lane in CSR order, up to kBinMid by eight lanes and longer ones by a
// wavefront (lane l takes entries l, l + 8 or l + 64, .., then a fixed tree).
// The same first pass serves the SDDMM.
#pragma once
#include "ks_kernels.h"

namespace ks {

constexpr int kBinCols = 16384;    // columns of a block: 128 KB of FP64 x in LDS
constexpr int kBinEntries = 8192;  // entries of a segment: 64 KB of FP64 in LDS
constexpr int kBinRows = 4096;     // rows of a segment
constexpr int kBinBlocks = 1024;   // column blocks (n up to 16.7M)
constexpr int kBinUnit = 1 << 17;  // entries of one workgroup of the first pass
constexpr int kBinGather = 1024;   // threads of the first pass
constexpr int kBinSum = 512;       // threads of the second: two workgroups per CU
constexpr int kBinWords = kBinEntries / 64;
constexpr int kBinShort = 16;      // rows summed by one lane
constexpr int kBinMid = 256;       // rows summed by eight lanes

// The segments and runs of one side; device arrays.  Place p of a segment
// (its entries ordered by block) is the (r + 1)-th run's, r + 1 the number of
// run starts up to p, and its x is xg[p + shift of run r]: the starts are a
// bit mask with the count before each word, so a lane finds its entry without
// a search.
struct BinView {
  int64_t nseg = 0, nunit = 0;
  int nblk = 0;
  const int32_t* seg = nullptr;      // first row of each segment, nseg + 1
  const int32_t* snz = nullptr;      // first entry, nseg + 1
  const uint64_t* mask = nullptr;    // run starts, kBinWords per segment
  const uint16_t* before = nullptr;  // starts before each word
  const int32_t* shift = nullptr;    // xg index minus place, by run, nblk per segment (one 0 without entries)
  const int32_t* unit = nullptr;     // first pass: block, first and last + 1 entry of xg
  const uint16_t* lcol = nullptr;    // column within its block, in xg's order
  const uint16_t* place = nullptr;   // CSR place in the segment, ordered by segment, then block
  double* xg = nullptr;              // x by entry (FP64 or FP32), by block, then segment
};

// Counts the entries of each (block, segment): one workgroup per segment.
__global__ __launch_bounds__(kBlock) void k_bin_count(int nblk, int64_t nseg, const int32_t* __restrict__ snz,
                                                      const int32_t* __restrict__ col, int32_t* cnt) {
  __shared__ int h[kBinBlocks];
  const int64_t s = blockIdx.x;
  for (int b = threadIdx.x; b < nblk; b += kBlock) h[b] = 0;
  __syncthreads();
  for (int64_t j = snz[s] + (int64_t)threadIdx.x; j < snz[s + 1]; j += kBlock) atomicAdd(h + col[j] / kBinCols, 1);
  __syncthreads();
  for (int b = threadIdx.x; b < nblk; b += kBlock) cnt[b * nseg + s] = h[b];
}
// Where each block starts in xg.
__global__ void k_bin_starts(int nblk, int64_t nseg, const int32_t* __restrict__ run, int32_t* start) {
  for (int b = blockIdx.x * blockDim.x + threadIdx.x; b < nblk; b += gridDim.x * blockDim.x) start[b] = run[b * nseg];
}
// Writes lcol, place and the runs: an entry's rank in its run is the order in
// which its lane gets there, which no result depends on.
__global__ __launch_bounds__(kBlock) void k_bin_fill(int nblk, int64_t nseg, const int32_t* __restrict__ snz,
                                                     const int32_t* __restrict__ col,
                                                     const int32_t* __restrict__ run, uint16_t* lcol,
                                                     uint16_t* place, uint64_t* mask, uint16_t* before,
                                                     int32_t* shift) {
  __shared__ int at[kBinBlocks];   // next place of the run among the segment's entries
  __shared__ int out[kBinBlocks];  // run start in xg minus its first place
  __shared__ uint64_t start[kBinWords];
  const int64_t s = blockIdx.x;
  const int32_t j0 = snz[s], j1 = snz[s + 1];
  for (int b = threadIdx.x; b < nblk; b += kBlock) {
    out[b] = run[b * nseg + s];
    at[b] = run[b * nseg + s + 1] - out[b];  // its length, for now
  }
  for (int k = threadIdx.x; k < kBinWords; k += kBlock) start[k] = 0;
  __syncthreads();
  if (threadIdx.x == 0) {
    int p = 0, r = 0;
    for (int b = 0; b < nblk; ++b) {
      const int len = at[b];
      at[b] = p;
      out[b] -= p;
      if (len > 0) {
        start[p / 64] |= 1ull << (p % 64);
        shift[s * nblk + r++] = out[b];
      }
      p += len;
    }
    if (r == 0) shift[s * nblk] = 0;  // a segment without entries: BinLoad reads xg[0]
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kBinWords; k += kBlock) {
    int c = 0;
    for (int q = 0; q < k; ++q) c += __popcll(start[q]);
    mask[s * kBinWords + k] = start[k];
    before[s * kBinWords + k] = (uint16_t)c;
  }
  for (int64_t j = j0 + (int64_t)threadIdx.x; j < j1; j += kBlock) {
    const int32_t c = col[j], b = c / kBinCols;
    const int p = atomicAdd(at + b, 1);
    lcol[out[b] + p] = (uint16_t)(c - b * kBinCols);
    place[j0 + p] = (uint16_t)(j - j0);
  }
}

// First pass: xg[e] = x[column of e] over one unit, from LDS.  Bound by its
// stream (2 bytes read and sizeof(T) written an entry).
template <class T>
__global__ __launch_bounds__(kBinGather) void k_bin_gather(int64_t n, const int32_t* __restrict__ unit,
                                                           const uint16_t* __restrict__ lcol,
                                                           const T* __restrict__ x, T* __restrict__ xg, Gate g) {
  if (g.off()) return;
  __shared__ T xs[kBinCols];
  const int32_t b = unit[3 * blockIdx.x], e0 = unit[3 * blockIdx.x + 1], e1 = unit[3 * blockIdx.x + 2];
  const int64_t c0 = (int64_t)b * kBinCols;
  const int m = (int)(n - c0 < kBinCols ? n - c0 : kBinCols);
  for (int i = threadIdx.x; i < m; i += kBinGather) xs[i] = x[c0 + i];
  __syncthreads();
  // four entries per lane and step, from an aligned start, four steps' columns
  // in flight (lcol and xg are padded)
  typedef typename Chunk<uint16_t, 4>::type C4;
  constexpr int W = 16 / sizeof(T), U = 4, kStep = 4 * kBinGather;
  for (int64_t e4 = (e0 & ~3) + 4 * (int64_t)threadIdx.x; e4 < e1; e4 += U * kStep) {
    C4 c[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e4 + u * kStep < e1) c[u] = __builtin_nontemporal_load(reinterpret_cast<const C4*>(lcol + e4 + u * kStep));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t e = e4 + u * kStep;
      if (e >= e0 && e + 4 <= e1) {
#pragma unroll
        for (int h = 0; h < 4; h += W) {
          typename Chunk<T, W>::type q;
#pragma unroll
          for (int i = 0; i < W; ++i) q[i] = xs[c[u][h + i]];
          *reinterpret_cast<typename Chunk<T, W>::type*>(xg + e + h) = q;
        }
      } else {
#pragma unroll
        for (int h = 0; h < 4; ++h)
          if (e + h >= e0 && e + h < e1) xg[e + h] = xs[c[u][h]];
      }
    }
  }
}

// One segment's x on its way to LDS: the places of a lane are tid + kBinSum u
// (past the segment's end, its last place again, so that no load waits for a
// branch). 
template <class T>
struct BinLoad {
  static constexpr int U = kBinEntries / kBinSum;
  T x[U];
  int p[U];
  __device__ __forceinline__ static int at(int u, int cnt) {
    return min((int)threadIdx.x + u * kBinSum, max(cnt, 1) - 1);
  }
  // where a segment's loads start: at the matrix's first entry for a segment
  // without entries, so that they need no branch (which costs registers: six
  // to eight spilled in every FP64 k_bin_sum)
  __device__ __forceinline__ static int32_t first(int32_t j0, int cnt) { return cnt > 0 ? j0 : 0; }
  // run numbers first, then their shifts, then every entry; j0: first()
  __device__ __forceinline__ void load(const BinView& B, int64_t s, int32_t j0, int cnt, const T* __restrict__ xg) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint64_t* mask = B.mask + s * kBinWords + w;
    const uint16_t* before = B.before + s * kBinWords + w;
    const int32_t* shift = B.shift + s * B.nblk;
    int r[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint64_t m = mask[u * (kBinSum / 64)];
      r[u] = (int)before[u * (kBinSum / 64)] + __popcll(m & (~0ull >> (63 - lane))) - 1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = (int)threadIdx.x + u * kBinSum < cnt;
      r[u] = shift[in ? r[u] : 0] + (in ? (int)threadIdx.x + u * kBinSum : 0);
    }
    // ordinary loads: a run shares its first and last cache lines with the
    // next segment's runs, read at the same time on this XCD (streamed past
    // the L2 they cost 1.65 against 1.57 ms at 4M rows)
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = xg[r[u]];
#pragma unroll
    for (int u = 0; u < U; ++u) p[u] = __builtin_nontemporal_load(B.place + j0 + at(u, cnt));
  }
  __device__ __forceinline__ void stage(int cnt, T* sp) const {
#pragma unroll
    for (int u = 0; u < U; ++u)
      if ((int)threadIdx.x + u * kBinSum < cnt) sp[p[u]] = x[u];
  }
};

// 64 of a segment's rows, rb + kBinSum / 64 i, by one wavefront (the segment's
// wavefronts take its rows in turn: a segment of long rows has few of them):
// fn(row, first, end, lanes, sub) once for each row and lane that works on it,
// `lanes` lanes a row with this lane the sub-th: one to kBinShort entries, eight
// to kBinMid, else the wavefront.
// `list`: 64 bytes of the wavefront's own LDS.
template <class F>
__device__ __forceinline__ void bin_rows(int32_t rb, int32_t r1, int32_t j0, const int32_t* __restrict__ ptr,
                                         uint8_t* list, F fn) {
  constexpr int kW = kBinSum / 64;
  const int lane = threadIdx.x & 63;
  const int32_t r = rb + kW * lane;
  const int a = r < r1 ? ptr[r] - j0 : 0, e = r < r1 ? ptr[r + 1] - j0 : 0, len = e - a;
  if (r < r1 && len <= kBinShort) fn(r, a, e, std::integral_constant<int, 1>{}, 0);
  const uint64_t mid = __ballot(len > kBinShort && len <= kBinMid);
  if (mid) {
    if (mid >> lane & 1) list[__popcll(mid & ((1ull << lane) - 1))] = (uint8_t)lane;
    wave_sync();
    const int cnt = __popcll(mid);
    for (int i0 = 0; i0 < cnt; i0 += 8) {
      const int i = i0 + lane / 8;
      const int q = list[i < cnt ? i : 0];
      const int qa = __shfl(a, q, 64), qe = __shfl(e, q, 64);
      fn(i < cnt ? rb + kW * q : -1, qa, i < cnt ? qe : qa, std::integral_constant<int, 8>{}, lane & 7);
    }
    wave_sync();
  }
  for (uint64_t m = __ballot(len > kBinMid); m; m &= m - 1) {
    const int q = __ffsll((unsigned long long)m) - 1;
    fn(rb + kW * q, __shfl(a, q, 64), __shfl(e, q, 64), std::integral_constant<int, 64>{}, lane);
  }
}

// v summed over groups of L lanes, in every lane
template <int L, class T>
__device__ __forceinline__ T lanes_sum(T v) {
  if constexpr (L == 64 && sizeof(T) == 8) return wave_sum(v);
#pragma unroll
  for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Second pass of y = A x.
template <class T, int NV, class Epi>
__global__ __launch_bounds__(kBinSum) __attribute__((amdgpu_waves_per_eu(4))) void k_bin_sum(
    BinView B, const int32_t* __restrict__ ptr, const T* __restrict__ val, const T* __restrict__ xg, Epi epi, Gate g,
    RedArgs ra, StatArgs st) {
  if (g.off()) return;
  st.count();
  epi.prep();
  __shared__ T sp[kBinEntries];
  __shared__ uint8_t list[kBinSum / 64][64];
  double acc[NV > 0 ? NV : 1];
#pragma unroll
  for (int i = 0; i < (NV > 0 ? NV : 1); ++i) acc[i] = 0.0;
  constexpr int U = BinLoad<T>::U;
  const int tid = threadIdx.x, w = tid >> 6;
  RowBlocks rbs{B.nseg};
  int64_t s, end, step;
  rbs.range(s, end, step);
  for (; s < end; s += step) {
    const int32_t r0 = B.seg[s], r1 = B.seg[s + 1], j0 = B.snz[s], cnt = B.snz[s + 1] - j0;
    const int32_t jl = BinLoad<T>::first(j0, cnt);
    BinLoad<T> x;
    T v[U];
    x.load(B, s, jl, cnt, xg);
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = ld_stream(val + jl + BinLoad<T>::at(u, cnt));
    x.stage(cnt, sp);
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (tid + u * kBinSum < cnt) sp[tid + u * kBinSum] *= v[u];
    __syncthreads();
    for (int32_t rb = r0 + w; rb < r1; rb += kBinSum)
      bin_rows(rb, r1, j0, ptr, list[w], [&](int32_t r, int a, int e, auto lanes, int sub) {
        constexpr int L = decltype(lanes)::value;
        T t = T(0);
        int k = a + sub;
        for (; k + 3 * L < e; k += 4 * L) {  // four LDS reads at a time, added in order
          const T t0 = sp[k], t1 = sp[k + L], t2 = sp[k + 2 * L], t3 = sp[k + 3 * L];
          t = (((t + t0) + t1) + t2) + t3;
        }
        for (; k < e; k += L) t += sp[k];
        t = lanes_sum<L>(t);
        if (sub == 0 && r >= 0) epi.row(r, t, T(0), acc, epi.pre(r));
      });
    __syncthreads();
  }
  if constexpr (NV > 0) block_store<NV, kBinSum>(acc, ra);
}

// Second pass of the SDDMM: out[j] = (alpha u[row(j)]) v[col(j)], v in xg.
__global__ __launch_bounds__(kBinSum) __attribute__((amdgpu_waves_per_eu(4))) void k_bin_sddmm(
    BinView B, const int32_t* __restrict__ ptr, double alpha, const double* __restrict__ u,
    const double* __restrict__ xg, double* __restrict__ out, StatArgs st) {
  st.count();
  __shared__ double sp[kBinEntries];
  __shared__ uint8_t list[kBinSum / 64][64];
  const int tid = threadIdx.x, w = tid >> 6;
  RowBlocks rbs{B.nseg};
  int64_t s, end, step;
  rbs.range(s, end, step);
  for (; s < end; s += step) {
    const int32_t r0 = B.seg[s], r1 = B.seg[s + 1], j0 = B.snz[s], cnt = B.snz[s + 1] - j0;
    BinLoad<double> x;
    x.load(B, s, BinLoad<double>::first(j0, cnt), cnt, xg);
    x.stage(cnt, sp);
    __syncthreads();
    for (int32_t rb = r0 + w; rb < r1; rb += kBinSum)
      bin_rows(rb, r1, j0, ptr, list[w], [&](int32_t r, int a, int e, auto lanes, int sub) {
        constexpr int L = decltype(lanes)::value;
        const double ur = r >= 0 ? alpha * u[r] : 0.0;
        for (int k = a + sub; k < e; k += L) sp[k] *= ur;
      });
    __syncthreads();
    for (int k = tid; k < cnt; k += kBinSum) __builtin_nontemporal_store(sp[k], out + j0 + k);
    __syncthreads();
  }
}

}  // namespace ks
