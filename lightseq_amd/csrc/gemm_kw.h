// Products on blocked operands whose output is too small for one large tile per compute unit: the
// wavefronts of a workgroup split K between them and load their MFMA fragments straight from
// the L2.
//
//   C[M,N] = epilogue( sum_k A[M,k] * W[N,k] )      int8 x int8 -> int32 or fp16 x fp16 -> fp32
//
// Blocked operands (blocked_offset in ls_device.h): 16 rows x 64 bytes of K are 1 KB in the order in which the
// lanes of a wavefront hold an MFMA fragment, so a fragment is one load instruction over eight
// whole 128-byte lines.  From row-major operands the same instruction touches 16 rows, and the
// address unit takes about 55 clocks for it instead of 17: 525 x 768 x 3072 (int32 out) takes
// 8.2 us with row-major activations, 10.2 us with both row-major, 4.8 us blocked; 13 us was the
// persistent LDS kernel.
//
// What bounds it: the path from the L2 into a compute unit, (rows + columns) * K bytes per tile
// at about 100 KB/us when all compute units read, and the chain load -> product -> reduction ->
// epilogue of a launch of a few microseconds (2.5 us for 64 x 1024 x 1024).  So tiles are small
// (16 MB x 16 NB) and as many as the chip has compute units, K is a quarter per wavefront, D
// slices of loads are in flight, and no operand passes through LDS.  Only the partial sums of
// the four wavefronts meet there; the epilogue works on four neighbouring columns per thread,
// whose column never changes, so what it reads per column (bias, clip values) is requested
// before the first product.
// int8 and fp16 share everything but the instruction: v_mfma_i32_16x16x64_i8 and
// v_mfma_f32_16x16x32_f16 both take 64 bytes of K as 16 bytes per lane.
#pragma once
#include "gemm_tile.h"

#include <type_traits>

namespace lsh {

struct KwI8 {
  typedef v16i Acc16;  // of the LDS tile loop: sixteen neighbouring columns
  typedef v4i Acc;  // four neighbouring columns of one row
  static __device__ __forceinline__ Acc mma(const v4i& w, const v4i& a, const Acc& c) {
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(w, a, c, 0, 0, 0);
  }
};
struct KwF16 {
  typedef v16f Acc16;
  typedef v4f Acc;
  static __device__ __forceinline__ Acc mma(const v4i& w, const v4i& a, const Acc& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w),
                                                  __builtin_bit_cast(v8h, a), c, 0, 0, 0);
  }
};

// Epilogues: Col column(n, N) is what the columns n .. n + 3 need (requested before the first
// product; n is clamped to N - 4), store4(m, n, N, col, acc) finishes four elements of row m.
// kClips (optional): the epilogue needs values of device memory for all of its elements.  request()
// loads them ahead of the first product and nothing waits for them there; finish(raw) returns
// the epilogue that has them.
// kTable: 256 bytes per column are staged in LDS from table() and handed to store4 as `tab`, the
// table of column n (kw_table_index says where a code is).
// kBlockedOut: the output is a blocked int8 matrix; the lanes of a wavefront then take the 256
// bytes that 16 rows of one 16-column chunk are.
// kAddRanges (optional): the ranges of K add to the same elements instead of storing to planes.
template <typename Epi, typename = void>
constexpr bool kEpiAddsRanges = false;
template <typename Epi>
constexpr bool kEpiAddsRanges<Epi, std::void_t<decltype(Epi::kAddRanges)>> = Epi::kAddRanges;
// bytes of LDS: partial sums (a 16 x 16 block padded to 68 16-byte cells, so that the lanes that
// read neighbouring columns hit different banks) and the table rows
template <typename Epi, int MB, int NB>
constexpr int kw_lds_bytes() {
  return 4 * MB * NB * 68 * 16 + (Epi::kTable ? 16 * NB * 256 : 0);
}

// grid: tiles_m * tiles_n workgroups of 256, times ksplit in y (range y of K stores to rows
// [y M, (y + 1) M) of the output).  K in bytes, `slices` = the 64-byte slices of a range.
// D > 1: slices % (4 D) == 0; D == 1: any number.  Preconditions: K % 64 == 0, N % 4 == 0,
// operands 16-byte aligned and allocated in whole blocks of 16 rows.  A tile's operands have a
// 64-bit base and 32-bit offsets, so it is the tile (K below 2^24 bytes) and not the matrix that
// has to stay below 4 GiB.
template <typename Tr, typename Epi, int MB, int NB, int D>
__global__ void __launch_bounds__(256, 2)
gemm_kw_kernel(const int8_t* __restrict__ A, const int8_t* __restrict__ W, int M, int N, int K, int slices,
               int tiles_m, int tiles_n, Epi epi) {
  typedef typename Tr::Acc Acc;
  extern __shared__ __align__(16) int8_t smem[];
  constexpr int QN = 4 * NB;  // column quads of a tile
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  int tile_m, tile_n;
  tile_of((int)blockIdx.x, (int)gridDim.x, tiles_m, tiles_n, tile_m, tile_n);
  const int m0 = tile_m * (16 * MB), n0 = tile_n * (16 * NB);
  int8_t* tab = smem + 4 * MB * NB * 68 * 16;
  if constexpr (Epi::kTable) {
    // table rows straight into LDS, a quarter per wavefront (columns past N: the last row's)
    const uint32_t lds = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)tab);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int q = wave * NB + i, c = q * 4 + (lane >> 4);
      const uint32_t off = (uint32_t)min(n0 + c, N - 1) * 256u + (((lane ^ c) & 15) << 4);
      const uint32_t dst = __builtin_amdgcn_readfirstlane(lds + q * 1024);
      asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off),
                   "s"(epi.table())
                   : "memory");
    }
  }
  // the thread's column quad and its first row; further rows follow in steps of a fixed stride
  const int quad = Epi::kBlockedOut ? (wave % NB) * 4 + (lane & 3) : tid % QN;
  const int row0 = Epi::kBlockedOut ? (wave / NB) * 16 + (lane >> 2) : tid / QN;
  constexpr int ROWS = Epi::kBlockedOut ? (NB >= 4 ? 16 : 64 / NB) : 256 / QN;
  constexpr int PER = (16 * MB + ROWS - 1) / ROWS;
  const int n = n0 + 4 * quad;
  const typename Epi::Col col = epi.column(min(n, N - 4), N);
  const auto raw = epi_request(epi);
  decltype(epi_fetch(epi, 0, 0, 0)) fetched[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) fetched[j] = epi_fetch(epi, min(m0 + row0 + j * ROWS, M - 1), min(n, N - 4), N);

  // this wavefront's slices
  const int first = (int)blockIdx.y * slices;
  const int s0 = first + (D > 1 ? wave * (slices / 4) : wave * slices / 4);
  const int ns = D > 1 ? slices / 4 : (wave + 1) * slices / 4 - wave * slices / 4;
  const int8_t* a_base = A + (long)m0 * K + (long)s0 * 1024;
  const int8_t* w_base = W + (long)n0 * K + (long)s0 * 1024;
  uint32_t a_off[MB], w_off[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
    a_off[i] = (uint32_t)min(16 * i, ((M - 1) & ~15) - m0) * (uint32_t)K + lane * 16;
#pragma unroll
  for (int b = 0; b < NB; ++b)
    w_off[b] = (uint32_t)min(16 * b, ((N - 1) & ~15) - n0) * (uint32_t)K + lane * 16;
  v4i fa[D][MB], fw[D][NB];
  auto load = [&](int u, int s) {
    const int8_t* a = a_base + s * 1024;
    const int8_t* w = w_base + s * 1024;
#pragma unroll
    for (int b = 0; b < NB; ++b) fw[u][b] = *reinterpret_cast<const v4i*>(w + w_off[b]);
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[u][i] = *reinterpret_cast<const v4i*>(a + a_off[i]);
  };
  Acc acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[i][b] = (Acc)0;
  auto mma = [&](int u) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[i][b] = Tr::mma(fw[u][b], fa[u][i], acc[i][b]);
  };
  if constexpr (D > 1) {
#pragma unroll
    for (int u = 0; u < D; ++u) load(u, u);
    __builtin_amdgcn_sched_barrier(0);
    for (int s = D; s < ns; s += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        mma(u);
        load(u, s + u);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) mma(u);
  } else {
    for (int s = 0; s < ns; ++s) {
      load(0, s);
      mma(0);
    }
  }

  // lane (l16, kq) holds row 16 i + l16, columns 16 b + 4 kq .. + 3
  Acc* red = reinterpret_cast<Acc*>(smem);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b)
      red[(wave * MB * NB + i * NB + b) * 68 + kq * 17 + l16] = acc[i][b];
  if constexpr (Epi::kTable) wait_vmcnt<0>();
  __syncthreads();
  if (n >= N) return;
  const auto fin = epi_finish(epi, raw);
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const int row = row0 + j * ROWS;
    const int m = m0 + row;
    if (row < 16 * MB && m < M) {
      const int cell = ((row >> 4) * NB + (quad >> 2)) * 68 + (quad & 3) * 17 + (row & 15);
      const Acc c = (red[cell] + red[MB * NB * 68 + cell]) +
                    (red[2 * MB * NB * 68 + cell] + red[3 * MB * NB * 68 + cell]);
      const int mo = kEpiAddsRanges<Epi> ? m : m + (int)blockIdx.y * M;
      if constexpr (Epi::kTable) fin.store4(mo, n, N, col, c, tab + 4 * quad * 256);
      else epi_store4(fin, mo, n, N, col, c, fetched[j]);
    }
  }
}

// ---------------------------------------------------------------------------------
// The same without the split of K, for fp16: every output is one chain of products in ascending K.
// v_mfma_f32_16x16x32_f16 adds its 32 products in the order in which two v_mfma_f32_32x32x16_f16
// do (checked bit for bit over random operands of several ranges), so this kernel, the LDS tile
// loop and the row-major kernel all give the same bits; partial sums of K ranges do not, and in a
// stack of quantised layers one unit of fp16 in a few outputs grows into percents of the result.
// WM x WN wavefronts side by side, MB x NB blocks of 16 x 16 each; D slices in flight (slices % D
// == 0); fragments of the wavefronts of a workgroup meet in the vector cache.
// ---------------------------------------------------------------------------------
template <typename Tr, typename Epi, int WM, int WN, int MB, int NB, int D>
__global__ void __launch_bounds__(64 * WM * WN)
gemm_seq_kernel(const int8_t* __restrict__ A, const int8_t* __restrict__ W, int M, int N, int K, int slices,
                int tiles_m, int tiles_n, Epi epi) {
  typedef typename Tr::Acc Acc;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, kq = lane >> 4;
  int tile_m, tile_n;
  tile_of((int)blockIdx.x, (int)gridDim.x, tiles_m, tiles_n, tile_m, tile_n);
  const int m0 = (tile_m * WM + wave / WN) * (16 * MB), n0 = (tile_n * WN + wave % WN) * (16 * NB);
  if (m0 >= M || n0 >= N) return;  // (no barriers)
  typename Epi::Col col[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) col[b] = epi.column(min(n0 + 16 * b + 4 * kq, N - 4), N);
  decltype(epi_fetch(epi, 0, 0, 0)) fetched[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b)
      fetched[i][b] = epi_fetch(epi, min(m0 + 16 * i + l16, M - 1), min(n0 + 16 * b + 4 * kq, N - 4), N);
  const int8_t* a_base = A + (long)m0 * K;
  const int8_t* w_base = W + (long)n0 * K;
  uint32_t a_off[MB], w_off[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
    a_off[i] = (uint32_t)min(16 * i, ((M - 1) & ~15) - m0) * (uint32_t)K + lane * 16;
#pragma unroll
  for (int b = 0; b < NB; ++b)
    w_off[b] = (uint32_t)min(16 * b, ((N - 1) & ~15) - n0) * (uint32_t)K + lane * 16;
  v4i fa[D][MB], fw[D][NB];
  auto load = [&](int u, int s) {
    const int8_t* a = a_base + s * 1024;
    const int8_t* w = w_base + s * 1024;
#pragma unroll
    for (int b = 0; b < NB; ++b) fw[u][b] = *reinterpret_cast<const v4i*>(w + w_off[b]);
#pragma unroll
    for (int i = 0; i < MB; ++i) fa[u][i] = *reinterpret_cast<const v4i*>(a + a_off[i]);
  };
  Acc acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[i][b] = (Acc)0;
  auto mma = [&](int u) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[i][b] = Tr::mma(fw[u][b], fa[u][i], acc[i][b]);
  };
#pragma unroll
  for (int u = 0; u < D; ++u) load(u, u);
  __builtin_amdgcn_sched_barrier(0);
  for (int s = D; s < slices; s += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      mma(u);
      load(u, s + u);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int u = 0; u < D; ++u) mma(u);
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int m = m0 + 16 * i + l16;
    if (m >= M) continue;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int n = n0 + 16 * b + 4 * kq;
      if (n < N) epi_store4(epi, m, n, N, col[b], acc[i][b], fetched[i][b]);
    }
  }
}

// ---------------------------------------------------------------------------------
// host side: the estimated duration of a launch.  Its length is that of the compute unit with the
// most tiles: the first tile takes a + b k microseconds (k: K in units of 1024 bytes; b grows by a
// third when every compute unit works), each further one s0 + s1 k, and every one `table` more with
// the table epilogue, `arith` more with an epilogue that dequantises, adds and rounds to fp16.
// The constants are fits to a sweep of every tile over eight epilogues, hidden 512, 768 and 1024
// and 24 M from 16 to 7926: the tile with the smallest estimate is 1 to 2 % slower than the fastest
// on average, 5 to 8 % at the 95th percentile.  (One set of constants for all epilogues, fitted to
// the plain ones, was 5 % off for those and 5 to 12 % for the others.)
// ---------------------------------------------------------------------------------
enum class EpilogueCost { kPlain, kTable, kArith };
template <typename Epi>
constexpr EpilogueCost epilogue_cost() {
  return Epi::kTable ? EpilogueCost::kTable
                     : EpiHasColumn16<Epi>::value ? EpilogueCost::kArith : EpilogueCost::kPlain;
}
struct TileCost {
  int tm, tn;
  float a, b, s0, s1, table, arith;
};
inline float tile_us(const TileCost& c, int M, int N, int K, int ksplit, int cus, EpilogueCost epi) {
  const long tiles =
      (long)((M + c.tm - 1) / c.tm) * ((N + c.tn - 1) / c.tn) * ksplit;
  const float per = (float)((tiles + cus - 1) / cus), k = K / 1024.f;
  const float busy = tiles < cus ? (float)tiles / cus : 1.f;
  const float first = c.a + c.b * k * (1.f + 0.35f * busy);
  const float each = epi == EpilogueCost::kTable ? c.table : epi == EpilogueCost::kArith ? c.arith : 0.f;
  return first + (per - 1.f) * (c.s0 + c.s1 * k) + per * each;
}
constexpr TileCost kKwCost[] = {{16, 16, 2.4f, 0.15f, 0.f, 0.25f, 0.04f, 0.1f},
                                {32, 32, 2.5f, 0.39f, 0.02f, 0.54f, 0.1f, 0.15f},
                                {64, 32, 2.55f, 0.66f, 0.12f, 0.79f, 0.2f, 0.29f},
                                {64, 64, 2.8f, 1.0f, 0.65f, 0.98f, 0.79f, 0.61f}};
struct KwTile {
  int mb, nb;
  float us;
};
// Few rows: a generation step, whose weights come from the memory and not from the L2.  A compute
// unit draws about 37 KB/us of them (16 x 1024 x 4096: 64 KB of weights per tile 4.6 us, 16 KB
// 3.5 us), so a tile's weights are priced at that rate where it is more than the fitted slope.
// The other constants are those of an earlier fit: the sweep's small launches find their weights in
// the caches.
constexpr int kKwColdRows = 64;
constexpr TileCost kKwColdCost[] = {{16, 16, 2.3f, 0.2f, 0.05f, 0.2f, 0.03f, 0.1f},
                                    {32, 32, 2.3f, 0.3f, 0.1f, 0.6f, 0.12f, 0.15f},
                                    {64, 32, 2.65f, 0.6f, 0.25f, 0.9f, 0.35f, 0.3f},
                                    {64, 64, 3.0f, 0.9f, 0.8f, 1.15f, 2.0f, 0.6f}};
inline TileCost kw_cold_cost(TileCost c) {
  const float slope = (float)c.tn / 36.f;  // us per 1024 bytes of K
  c.b = c.b * 1.35f < slope ? slope / 1.35f : c.b;
  c.s1 = c.s1 < slope ? slope : c.s1;
  return c;
}
// K: the bytes of one of `ksplit` ranges
inline KwTile kw_choose_tile(int M, int N, int K, int ksplit, int cus, EpilogueCost epi) {
  KwTile best{0, 0, 0.f};
  for (int i = 0; i < 4; ++i) {
    const TileCost c = M <= kKwColdRows ? kw_cold_cost(kKwColdCost[i]) : kKwCost[i];
    const float us = tile_us(c, M, N, K, ksplit, cus, epi);
    if (best.mb == 0 || us < best.us) best = KwTile{c.tm / 16, c.tn / 16, us};
  }
  return best;
}

}  // namespace lsh
