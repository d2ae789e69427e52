// The kernels and the dispatch of products on blocked operands, shared by the files that bring
// epilogues (gemm_blocked.hip: the models', layer_gemm.hip: the layers').
#pragma once
#include "gemm_kw.h"
#include "ls_launch.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <mutex>

namespace lsh {

// one output tile per workgroup, both operands blocked
template <typename Tr, typename Epi, int WGM, int WGN, int MB, int NB, int NST>
__global__ void __launch_bounds__(64 * WGM * WGN)
gemm_blk_tile_kernel(const int8_t* __restrict__ A, const int8_t* __restrict__ W, int M, int N, int K,
                     int tiles_m, int tiles_n, Epi epi) {
  extern __shared__ __align__(16) int8_t smem[];
  asm volatile("" : "+s"(tiles_m) : "s"(A), "s"(W));
  constexpr int TM = WGM * MB * 32;
  int tm, tn;
  tile_of(blockIdx.x, tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
  tile_gemm<Epi, WGM, WGN, MB, NB, NST, false, true, typename Tr::Acc16>(A, W, epi, tm * TM, M, N, K, tn, smem);
}

template <auto Kern>
int raise_lds(size_t smem) {
  static std::mutex mu;
  static unsigned long long done = 0;  // bit per device index
  int dev = 0;
  if (int rc = lsh_check_hip(hipGetDevice(&dev), "hipGetDevice(gemm_blk)")) return rc;
  if (dev < 0 || dev >= 64) return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm: device index out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!(done >> dev & 1ull)) {
    if (smem > 64 * 1024)
      if (int rc = lsh_check_hip(hipFuncSetAttribute(reinterpret_cast<const void*>(Kern),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem),
                                 "hipFuncSetAttribute(gemm_blk)"))
        return rc;
    done |= 1ull << dev;
  }
  return LSH_OK;
}

// grid.x: output tiles, which tile_of counts in 24 bits
template <auto Kern, typename... Args>
int launch_blk(dim3 grid, int threads, size_t smem, hipStream_t s, Args... args) {
  if (grid.x >= (1u << 24)) return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm: more than 2^24 output tiles");
  if (int rc = raise_lds<Kern>(smem)) return rc;
  hipEvent_t e0, e1;
  if (gemm_take_timing_events(&e0, &e1))
    hipExtLaunchKernelGGL(Kern, grid, dim3(threads), (unsigned)smem, s, e0, e1, 0, args...);
  else
    Kern<<<grid, threads, smem, s>>>(args...);
  return lsh_check_launch("blocked gemm");
}

template <typename Tr, typename Epi, int MB, int NB>
int launch_kw(const int8_t* A, const int8_t* W, Epi epi, int M, int N, int K, int ksplit,
              hipStream_t s) {
  const int tm = (M + 16 * MB - 1) / (16 * MB), tn = (N + 16 * NB - 1) / (16 * NB);
  const dim3 grid(tm * tn, ksplit);
  constexpr size_t smem = kw_lds_bytes<Epi, MB, NB>();
  const int slices = K / 64 / ksplit;
#define LSH_KW(D)                                                                                   \
  return launch_blk<gemm_kw_kernel<Tr, Epi, MB, NB, D>>(grid, 256, smem, s, A, W, M, N, K, slices, tm, tn, epi)
  if (slices % 16 == 0) LSH_KW(4);
  if (slices % 12 == 0) LSH_KW(3);
  if (slices % 8 == 0) LSH_KW(2);
  LSH_KW(1);
#undef LSH_KW
}

template <typename Tr, typename Epi, int WGM, int WGN, int MB, int NB, int NST>
int launch_tile(const int8_t* A, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s) {
  constexpr int TM = WGM * MB * 32, TN = WGN * NB * 32;
  const int tm = (M + TM - 1) / TM, tn = (N + TN - 1) / TN;
  return launch_blk<gemm_blk_tile_kernel<Tr, Epi, WGM, WGN, MB, NB, NST>>(
      dim3(tm * tn), 64 * WGM * WGN, NST * (TM + TN) * kBK, s, A, W, M, N, K, tm, tn, epi);
}

// The LDS tile kernel: 8 wavefronts for tiles from 128 x 128 up, 4 for the small ones (several
// workgroups then share a compute unit and one's epilogue runs under the other's K loop).
constexpr TileCost kLdsCost[] = {{64, 64, 2.2f, 1.54f, 0.22f, 1.13f, 0.27f, 0.56f},
                                 {128, 64, 2.55f, 2.32f, 0.2f, 1.85f, 0.46f, 1.1f},
                                 {128, 128, 2.5f, 3.36f, 1.07f, 2.7f, 0.52f, 2.2f},
                                 {256, 128, 3.0f, 5.5f, 2.7f, 6.1f, 0.93f, 3.9f},
                                 {256, 192, 3.65f, 7.3f, 2.35f, 9.25f, 1.5f, 5.95f},
                                 {256, 256, 4.35f, 9.3f, 0.f, 14.2f, 2.2f, 7.4f}};
// (its third stage costs the 128 x 64 tile its third workgroup per compute unit)
constexpr int kLongK = 2048;
constexpr TileCost kLongKCost{128, 64, 2.55f, 2.32f, 0.2f, 2.35f, 0.46f, 1.1f};
struct LdsTile {
  int tm = 0, tn = 0;
  float us = 0;
};
inline LdsTile choose_lds_tile(int M, int N, int K, int cus, EpilogueCost epi) {
  LdsTile best;
  if (K % kBK != 0 || K / kBK < 3 || N % 16 != 0) return best;
  for (const auto& c : kLdsCost) {
    const bool long_k = K >= kLongK && c.tm == 128 && c.tn == 64;
    const float us = tile_us(long_k ? kLongKCost : c, M, N, K, 1, cus, epi);
    if (best.tm == 0 || us < best.us) best = LdsTile{c.tm, c.tn, us};
  }
  return best;
}

inline int check_blk(const int8_t* A, const int8_t* W, bool aligned, int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || !A || !W)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm: bad arguments");
  if (K % 64 != 0 || N % 4 != 0)
    return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm: needs K bytes % 64 == 0 and N % 4 == 0");
  if (((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15u) != 0 || !aligned)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm: operands must be 16-byte aligned");
  if (K >= (1 << 24) || M > 0x7fffff00 || N > 0x7fffff00 || (long)((M + 15) / 16) * ((N + 15) / 16) >= (1L << 31))
    return lsh_fail(LSH_ERR_UNSUPPORTED, "blocked gemm: operand too large");
  return LSH_OK;
}

template <typename Tr, typename Epi, bool TILES>
int dispatch_blk(const int8_t* A, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s,
                 int ksplit = 1) {
  if (int rc = check_blk(A, W, epi.aligned(), M, N, K)) return rc;
  if (ksplit < 1 || K % (64 * ksplit) != 0)
    return lsh_fail(LSH_ERR_INVALID, "blocked gemm: K does not split into whole 64-byte slices");
  const int cus = cu_count();
  constexpr EpilogueCost cost = epilogue_cost<Epi>();
  const KwTile kw = kw_choose_tile(M, N, K / ksplit, ksplit, cus, cost);
  if constexpr (TILES) {
    if (ksplit == 1) {
      const LdsTile t = choose_lds_tile(M, N, K, cus, cost);
      if (t.tm != 0 && t.us < kw.us) {
        if (t.tn == 256) return launch_tile<Tr, Epi, 2, 4, 4, 2, 2>(A, W, epi, M, N, K, s);
        if (t.tn == 192) return launch_tile<Tr, Epi, 4, 2, 2, 3, 2>(A, W, epi, M, N, K, s);
        if (t.tm == 256) return launch_tile<Tr, Epi, 4, 2, 2, 2, 3>(A, W, epi, M, N, K, s);
        // where a tile has a compute unit to itself the ring may fill its LDS: 2348 x 1024 x 1024 in 6.6
        // instead of 6.9 us (with two tiles a unit 2348 x 3072 x 1024 takes 12.1, not 10.4)
        if (t.tn == 128 && K >= 4 * kBK && (long)((M + 127) / 128) * ((N + 127) / 128) <= cus)
          return launch_tile<Tr, Epi, 4, 2, 1, 2, 4>(A, W, epi, M, N, K, s);
        if (t.tn == 128) return launch_tile<Tr, Epi, 4, 2, 1, 2, 2>(A, W, epi, M, N, K, s);
        if (t.tm == 64) return launch_tile<Tr, Epi, 2, 2, 1, 1, 3>(A, W, epi, M, N, K, s);
        // long K loops: a third stage instead of a third workgroup per compute unit
        if (K >= kLongK) return launch_tile<Tr, Epi, 4, 1, 1, 2, 3>(A, W, epi, M, N, K, s);
        return launch_tile<Tr, Epi, 2, 2, 2, 1, 2>(A, W, epi, M, N, K, s);
      }
    }
  }
  if (kw.mb == 1) return launch_kw<Tr, Epi, 1, 1>(A, W, epi, M, N, K, ksplit, s);
  if (kw.mb == 2) return launch_kw<Tr, Epi, 2, 2>(A, W, epi, M, N, K, ksplit, s);
  if (kw.nb == 2) return launch_kw<Tr, Epi, 4, 2>(A, W, epi, M, N, K, ksplit, s);
  return launch_kw<Tr, Epi, 4, 4>(A, W, epi, M, N, K, ksplit, s);
}


// fp16 products: every output one chain in ascending K (gemm_seq_kernel).  The estimates, in us with k
// = K in units of 1000 bytes, are fits to a sweep of hidden 512, 768 and 1024 (K of one and of
// four times that) over M from 4 to 8192 on 256 compute units; the smallest one is within 15 % of
// the fastest there.  What a launch takes beyond one round of the chip goes by the tiles per
// compute unit.
struct SeqTile {
  int kind;  // 0: a wavefront per 16 x 16, 1: per 32 x 32; 2 - 4: LDS tiles 64 x 64, 128 x 64,
             // 128 x 128; 5: the last with a third stage; 6, 7: 256 x 192, 256 x 256
  float us;
};
inline SeqTile choose_seq(int M, int N, int K, int cus) {
  const float k = (float)K / 1000.f;
  auto tiles = [&](int tm, int tn) {  // per compute unit
    return (float)((long)((M + tm - 1) / tm) * ((N + tn - 1) / tn)) / (float)cus;
  };
  auto lds = [&](float t, float first, float more) {
    return 2.f + first * k + (t > 1.f ? (t - 1.f) * (1.f + more * k) : 0.f);
  };
  SeqTile best{0, std::max(std::max(2.8f, 0.9f + 0.5f * k), 2.f + 0.2432f * tiles(16, 16) * k)};
  auto take = [&](int kind, float us) {
    if (us < best.us) best = SeqTile{kind, us};
  };
  take(1, std::max(1.f + 1.2f * k, 2.f + 0.5632f * tiles(32, 32) * k));
  if (K % kBK == 0 && K / kBK >= 3 && N % 16 == 0) {
    take(2, lds(tiles(64, 64), 1.9f, 1.4f));
    take(3, lds(tiles(128, 64), 3.7f, 1.8f));
    // with no more tiles than compute units a tile has a unit's LDS to itself: 3000 x 1024 x 4096 in
    // 33.7 us instead of 39.9 (beyond that two tiles a unit are better: 8192 rows 52.0, not 65.8)
    if (tiles(128, 128) <= 1.f) take(5, lds(tiles(128, 128), 3.85f, 0.f));
    else take(4, lds(tiles(128, 128), 4.5f, 2.2f));
    if (best.kind == 4) {
      // Several rounds of the chip: the larger tiles where theirs come out even, priced in whole rounds
      // (fits to the projections of keys and values, N = 6144 to 12288, M from 500 to 8000, to 5 %; us with
      // 128 x 128 and now: 976 x 12288 x 2048 28.8 and 25.8, 1200 x 12288 x 2048 36.1 and 30.8, 4096 x 12288
      // x 2048 103 and 95, 976 x 9216 x 1536 22.8 and 19.5).  3 % less at least, or the smaller tile stays.
      auto rounds = [&](int tm, int tn) { return std::ceil(tiles(tm, tn)); };
      const float small = 2.f + k + rounds(128, 128) * (1.65f + 3.22f * k);
      const float wide = rounds(256, 192) * (6.2f + 9.2f * k), square = rounds(256, 256) * (8.9f + 10.4f * k);
      if (std::min(wide, square) < 0.97f * small) best.kind = wide <= square ? 6 : 7;
    }
  }
  return best;
}

template <typename Epi, int MB, int D>
int launch_seq(const int8_t* A, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s) {
  const int tm = (M + 16 * MB - 1) / (16 * MB), tn = (N + 16 * MB - 1) / (16 * MB);
  return launch_blk<gemm_seq_kernel<KwF16, Epi, 1, 1, MB, MB, D>>(dim3(tm * tn), 64, 0, s, A, W, M, N, K,
                                                                  K / 64, tm, tn, epi);
}
// K in bytes
template <typename Epi>
int dispatch_f16(const int8_t* A, const int8_t* W, Epi epi, int M, int N, int K, hipStream_t s) {
  if (int rc = check_blk(A, W, epi.aligned(), M, N, K)) return rc;
  const int slices = K / 64;
  switch (choose_seq(M, N, K, cu_count()).kind) {
    case 0:
      if (slices % 16 == 0) return launch_seq<Epi, 1, 16>(A, W, epi, M, N, K, s);
      if (slices % 8 == 0) return launch_seq<Epi, 1, 8>(A, W, epi, M, N, K, s);
      return launch_seq<Epi, 1, 1>(A, W, epi, M, N, K, s);
    case 1:
      if (slices % 4 == 0) return launch_seq<Epi, 2, 4>(A, W, epi, M, N, K, s);
      return launch_seq<Epi, 2, 1>(A, W, epi, M, N, K, s);
    case 2: return launch_tile<KwF16, Epi, 2, 2, 1, 1, 3>(A, W, epi, M, N, K, s);
    case 3: return launch_tile<KwF16, Epi, 4, 1, 1, 2, 2>(A, W, epi, M, N, K, s);
    case 5: return launch_tile<KwF16, Epi, 2, 2, 2, 2, 3>(A, W, epi, M, N, K, s);
    case 6: return launch_tile<KwF16, Epi, 4, 2, 2, 3, 2>(A, W, epi, M, N, K, s);
    case 7: return launch_tile<KwF16, Epi, 2, 4, 4, 2, 2>(A, W, epi, M, N, K, s);
    default: return launch_tile<KwF16, Epi, 2, 2, 2, 2, 2>(A, W, epi, M, N, K, s);
  }
}

}  // namespace lsh
