// ks_rows.h - SpMV by row classes: matrices whose rows repeat, values included.
//
// A stencil whose coefficients are constant, or constant in parts, has few
// different rows: a 7-point box has 27, from its interior to its corners.  Such
// a matrix is kept as one byte per row, the number of the row's class, and a
// table of the at most kRowMax classes: offsets col - row and values in CSR
// order (kRowLen places per class), which every workgroup holds in LDS.  The
// product then streams x, y and a byte per row: a 7-point 160^3 product moves
// 70 MB in FP64 instead of 302 with row patterns (PatIx), whose values stream
// from memory.
//
// What bounds it then is the vector memory path of the CUs: seven gathers of
// 512 bytes per wavefront and row in FP64, whichever cache answers them (the
// 7-point 192^3 product takes 37 us; with one gather instead of seven 21 us,
// with the two of other planes left out still 35), and in FP32 about equally
// the bytes (18 us, 15 with one gather).  A thread takes kRowBatch rows, one
// of each of as many tiles, and gathers for all of them before it sums the
// first, with the codes of the next ones behind: 192^3 in FP32 takes 18.0 us
// with two, 18.5 with one and 19.7 with four, 96^3 in FP64 8.5, 7.8 and 8.5.
// Class data from scalar registers, for wavefronts of one class, gave nothing.
// Rows of at most two entries gather two (five, the next size, cost more than the
// entries' own format where x lies in the L2: one entry, 300000 rows, FP64 5.6 us, with
// two gathers 4.7; 2^22 rows 18.9 and 15.1).
// Measured against row patterns (7-point, us): FP64 96^3 18 -> 8.6, 128^3
// 28 -> 12.9, 160^3 57 -> 23; FP32 160^3 30 -> 11.3, 192^3 50 -> 18.2.
//
// Rows are summed entry for entry in CSR order, and tiles, grid and epilogues
// are k_spmv_stream's, so every result is bit for bit that of the other
// formats.
#pragma once
#include "ks_kernels.h"

namespace ks {

constexpr int64_t kRowMinNnz = 4096;          // fewer entries are not worth a table
constexpr int64_t kRowMaxN = int64_t(1) << 29;  // x is addressed by 32-bit byte offsets

// rows a thread takes at a time
template <class T, int NX>
constexpr int kRowBatch = NX == 2 ? 1 : 2;

template <class T, int NX, int NV, class Epi>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6))) void k_spmv_rows(
    int64_t n, int64_t ntiles, const int32_t* __restrict__ tiles, const int32_t* __restrict__ tab,
    const RowIx* __restrict__ code, const T* __restrict__ val, const T* __restrict__ x0, const T* __restrict__ x1,
    Epi epi, Gate g, RedArgs ra, StatArgs st) {
  if (g.off()) return;
  st.count();
  constexpr int B = kRowBatch<T, NX>;
  // the y of the workgroup's first tiles, for the projection (k_spmv_stream)
  constexpr int kYT = !HasProj<Epi>::value ? 0 : sizeof(T) == 4 ? 14 : 9;
  constexpr int kYW = kTileRows + 4;
  __shared__ __align__(16) T sval[kRowMax * kRowLen];
  __shared__ __align__(16) int32_t stab[kRowTab];
  __shared__ __align__(16) T sy[kYT > 0 ? kYT : 1][kYT > 0 ? kYW : 1];
  double acc[NV > 0 ? NV : 1];
#pragma unroll
  for (int i = 0; i < (NV > 0 ? NV : 1); ++i) acc[i] = 0.0;
  const int tid = threadIdx.x;
  RowBlocks rbs{ntiles};
  int64_t t, end, step;
  rbs.range(t, end, step);
  // rows of the batch's tiles, and this thread's codes; a tile past the end
  // has no rows and stands where the batch's first does
  int32_t r0[B], nr[B], cd[B];
  auto next = [&](int64_t u) {
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const bool in = u + b * step < end;
      const int64_t v = in ? u + b * step : u < end ? u : 0;
      r0[b] = tiles[v];
      nr[b] = in ? tiles[v + 1] - r0[b] : 0;
    }
#pragma unroll
    for (int b = 0; b < B; ++b) cd[b] = code[r0[b] + (tid < nr[b] ? tid : 0)].v;
  };
  next(t);
  for (int i = tid; i < kRowMax * kRowLen; i += kBlock) sval[i] = val[i];
  for (int i = tid; i < kRowTab; i += kBlock) stab[i] = tab[i];
  epi.prep();
  __syncthreads();
  const int most = __builtin_amdgcn_readfirstlane(stab[kRowTab - 1]);  // entries of the longest row
  // NK >= most entries gathered per row; places past a row's end hold offset 0
  auto sweep = [&](auto nk) {
    constexpr int NK = decltype(nk)::value;
    auto at = [](const T* x, uint32_t byte) {
      return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(x) + byte);
    };
    for (int slot = 0; t < end; t += B * step, slot += B) {
      T g0[B][NK], g1[B][NK];
      int32_t row[B], cls[B];
      bool act[B];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        act[b] = tid < nr[b];
        row[b] = r0[b] + (act[b] ? tid : 0);
        cls[b] = cd[b];
#pragma unroll
        for (int q = 0; q < NK; ++q) {
          const uint32_t c = (uint32_t)(row[b] + stab[cls[b] * kRowLen + q]) * (uint32_t)sizeof(T);
          g0[b][q] = at(x0, c);
          if (NX == 2) g1[b][q] = at(x1, c);
        }
      }
      decltype(epi.pre(0)) pv[B];
#pragma unroll
      for (int b = 0; b < B; ++b) pv[b] = epi.pre(row[b]);
      next(t + B * step);
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const int m = stab[kRowMax * kRowLen + cls[b]];
        const T* v = sval + cls[b] * kRowLen;
        T a0 = 0, a1 = 0;
#pragma unroll
        for (int q = 0; q < NK; ++q) {
          const T b0 = mul_add_rn(a0, v[q], g0[b][q]);
          a0 = q < m ? b0 : a0;
          if (NX == 2) {
            const T b1 = mul_add_rn(a1, v[q], g1[b][q]);
            a1 = q < m ? b1 : a1;
          }
        }
        if (act[b]) {
          if constexpr (kYT > 0) {
            if (slot + b < kYT) sy[slot + b][(row[b] - tid & 3) + tid] = epi.value(a0);
            else epi.row(row[b], a0, a1, acc, pv[b]);
          } else {
            epi.row(row[b], a0, a1, acc, pv[b]);
          }
        }
      }
    }
  };
  if (most <= 2) sweep(std::integral_constant<int, 2>{});
  else if (most <= 5) sweep(std::integral_constant<int, 5>{});
  else if (most <= 7) sweep(std::integral_constant<int, 7>{});
  else sweep(std::integral_constant<int, 8>{});
  if constexpr (NV > 0) block_store<NV>(acc, ra);
  if constexpr (HasProj<Epi>::value) {
    static_assert(NV == 0 && NX == 1, "projection epilogue takes a plain SpMV");
    __syncthreads();
    proj_tiles<T, kYT, kYW>(tiles, rbs, sy, epi, ra);
  }
}

}  // namespace ks
