// Pieces of the int8 GEMM shared by the stand-alone kernels (gemm_i8.hip) and the kernels that
// run a product as one phase of a longer launch (xcd_ffn_kernels.hip): the plain int32, the
// requantising and the tabulated epilogue, and the K loop of one large output tile.
#pragma once
#include "ls_device.h"
#include "tile_common.h"

#include <type_traits>

namespace lsh {

typedef float v4f __attribute__((ext_vector_type(4)));

// Where the table kernels of gemm_kw.h find code `code` of column `col` in the column's 256 bytes of
// LDS: the 16-byte chunks are permuted by the column, so that the lanes of one lookup, whose
// columns differ, spread over the banks.
__device__ __forceinline__ int kw_table_index(int code, int col) {
  return (code + 128) ^ ((col & 15) << 4);
}

// ---------------------------------------------------------------------------------
// Epilogues.  store16(m, n, N, c, full): c[0..15] are C[m, n .. n+15]; `full` means all
// 16 columns exist and the vector path may be used.
// ---------------------------------------------------------------------------------
struct EpiI32 {
  int32_t* C;
  __device__ __forceinline__ void store16(long m, int n, int N, const v16i& c, bool full) const {
    int32_t* p = C + m * N + n;
    if (full) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<int4*>(p + 4 * q) =
            make_int4(c[4 * q], c[4 * q + 1], c[4 * q + 2], c[4 * q + 3]);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (n + i < N) p[i] = c[i];
    }
  }
  // one element (the decode-step kernels give every thread one element of a 16 x 16 block)
  struct Pre1 {};
  __device__ __forceinline__ Pre1 prefetch1(int) const { return Pre1{}; }
  struct Blk1 {
    int n;
  };
  __device__ __forceinline__ Blk1 block1(int n) const { return Blk1{n}; }
  __device__ __forceinline__ void store1(long m, Blk1 blk, int N, int acc, Pre1, const int8_t*,
                                         int) const {
    C[m * N + blk.n] = acc;
  }
  // four neighbouring elements (gemm_kw.h)
  static constexpr bool kTable = false, kBlockedOut = false;
  struct Col {};
  __device__ __forceinline__ Col column(int, int) const { return Col{}; }
  __device__ __forceinline__ void store4(int m, int n, int N, Col, const v4i& c) const {
    *reinterpret_cast<v4i*>(C + (long)m * N + n) = c;
  }
  bool aligned() const { return C != nullptr && (reinterpret_cast<uintptr_t>(C) & 15u) == 0; }
  bool vec_ok(int N) const { return N % 4 == 0 && aligned(); }
  static const char* name() { return "EpiI32"; }
};

// int32 sums that start from zero and to which ranges of K add: exact in any order, and a reader has one
// plane to fetch instead of four.  That counts where every workgroup of the next product makes the
// layer norm (4 rows, us with planes and with sums: that product 5.2 and 4.5, this one, 4 x 1024 x 4096,
// 2.8 and 3.0) and where planes were no choice (16 x 768 x 3072: 3.4 in one range, 3.0).  In front
// of a layer norm of its own it costs more than it saves: 16 rows 3.3 and 3.5, 64 rows 3.7 and 5.3.
struct EpiI32Add : EpiI32 {
  static constexpr bool kAddRanges = true;
  __device__ __forceinline__ void store4(int m, int n, int N, Col, const v4i& c) const {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __hip_atomic_fetch_add(C + (long)m * N + n + i, c[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
};

__device__ __forceinline__ void store16_i8(int8_t* p, int n, int N, const int (&q)[16], bool full) {
  if (full) {
    uint4 o;
    o.x = pack4_i8(q[0], q[1], q[2], q[3]);
    o.y = pack4_i8(q[4], q[5], q[6], q[7]);
    o.z = pack4_i8(q[8], q[9], q[10], q[11]);
    o.w = pack4_i8(q[12], q[13], q[14], q[15]);
    *reinterpret_cast<uint4*>(p) = o;
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (n + i < N) p[i] = (int8_t)q[i];
  }
}

struct EpiI8 {
  int8_t* C;
  float alpha;
  __device__ __forceinline__ void store16(long m, int n, int N, const v16i& c, bool full) const {
    if (full) {
      *reinterpret_cast<uint4*>(C + m * N + n) = requant16_packed(c, alpha);
      return;
    }
    int q[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) q[i] = requant_acc(c[i], alpha);
    store16_i8(C + m * N + n, n, N, q, full);
  }
  struct Pre1 {};
  __device__ __forceinline__ Pre1 prefetch1(int) const { return Pre1{}; }
  struct Blk1 {
    int n;
  };
  __device__ __forceinline__ Blk1 block1(int n) const { return Blk1{n}; }
  __device__ __forceinline__ void store1(long m, Blk1 blk, int N, int acc, Pre1, const int8_t*,
                                         int) const {
    C[m * N + blk.n] = (int8_t)requant_acc_fast(acc, alpha);
  }
  static constexpr bool kTable = false, kBlockedOut = false;
  struct Col {};
  __device__ __forceinline__ Col column(int, int) const { return Col{}; }
  __device__ __forceinline__ void store4(int m, int n, int N, Col, const v4i& c) const {
    *reinterpret_cast<uint32_t*>(C + (long)m * N + n) =
        requant_acc_pack4(c[0], c[1], c[2], c[3], alpha);
  }
  bool aligned() const { return C != nullptr && (reinterpret_cast<uintptr_t>(C) & 15u) == 0; }
  bool vec_ok(int N) const { return N % 16 == 0 && aligned(); }
  static const char* name() { return "EpiI8"; }
};

// The same epilogue through a table.  After the requantisation an element is one of 255
// codes, and what follows (dequantise, add the column's bias, activation, requantise)
// depends only on that code and the column: table[n][code + 128], N x 256 bytes built once
// per weight matrix by build_act_lut with the very device function EpiActI8 evaluates, so
// the result is bit-identical.  The bias + GELU arithmetic costs ~35 vector instructions per
// element -- more than the matrix cores spend on a K = 768 product -- while the lookup is
// one byte load per element from a table that stays in L2 (768 KB for N = 3072); the lanes
// of one load instruction read two table rows, i.e. a handful of cache lines.
template <bool BLK>
struct EpiLut {
  int8_t* C;
  const int8_t* lut;
  float alpha;
  __device__ __forceinline__ void store16(long m, int n, int N, const v16i& c, bool full) const {
    int q[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int col = n + i < N ? n + i : N - 1;
      q[i] = lut[(long)col * 256 + requant_acc(c[i], alpha) + 128];
    }
    store16_i8(C + m * N + n, n, N, q, full);
  }
  // the same with the table rows of the tile's columns staged in LDS (`tab`: 256 bytes per
  // column, first row = the tile's first column; n_local = n - first column)
  __device__ __forceinline__ void store16_lds(long m, int n, int N, const v16i& c, bool full,
                                              const int8_t* tab, int n_local) const {
    int q[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
      q[i] = tab[(n_local + i) * 256 + requant_acc_fast(c[i], alpha) + 128];
    // blocked output: the 16 columns are one 16-byte chunk, and the lanes of consecutive rows
    // write consecutive chunks
    store16_i8(C + (BLK ? blocked_offset(m, n, N) : m * N + n), n, N, q, full);
  }
  // one element, the table rows of the workgroup's columns staged in LDS (n_local: the
  // element's column among them)
  struct Pre1 {};
  __device__ __forceinline__ Pre1 prefetch1(int) const { return Pre1{}; }
  struct Blk1 {
    int n;
  };
  __device__ __forceinline__ Blk1 block1(int n) const { return Blk1{n}; }
  __device__ __forceinline__ void store1(long m, Blk1 blk, int N, int acc, Pre1,
                                         const int8_t* tab, int n_local) const {
    C[m * N + blk.n] = tab[n_local * 256 + requant_acc_fast(acc, alpha) + 128];
  }
  static constexpr bool kTable = true, kBlockedOut = BLK;
  __device__ __forceinline__ const int8_t* table() const { return lut; }
  struct Col {};
  __device__ __forceinline__ Col column(int, int) const { return Col{}; }
  __device__ __forceinline__ void store4(int m, int n, int N, Col, const v4i& c,
                                         const int8_t* tab) const {
    int q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      q[i] = tab[i * 256 + kw_table_index(requant_acc_fast(c[i], alpha), n + i)];
    *reinterpret_cast<uint32_t*>(C + (BLK ? blocked_offset(m, n, N) : (long)m * N + n)) =
        pack4_i8(q[0], q[1], q[2], q[3]);
  }
  bool aligned() const { return C != nullptr && (reinterpret_cast<uintptr_t>(C) & 15u) == 0; }
  bool vec_ok(int N) const { return N % 16 == 0 && aligned(); }
  static const char* name() { return "EpiLutI8"; }
};
typedef EpiLut<false> EpiLutI8;
typedef EpiLut<true> EpiLutBlk;
template <typename Epi>
constexpr bool is_lut = std::is_same<Epi, EpiLutI8>::value || std::is_same<Epi, EpiLutBlk>::value;

template <typename Epi>
__device__ __forceinline__ const int8_t* epi_lut(const Epi& e) {
  if constexpr (is_lut<Epi>) return e.lut;
  else return nullptr;
}

// linear work index -> tile.  Workgroups (and the persistent kernel's work items) are
// dealt round-robin to the 8 XCDs; renumber so that each XCD (own L2) works on a
// contiguous run of tiles, walked in column-major order of 8-tile-tall groups so that a
// run shares W columns and A rows.
// Work-item counts stay below 2^24 (checked by the dispatcher): with both operands masked to
// 24 bits the compiler divides through a float reciprocal, a dozen instructions instead of
// the forty of a full 32-bit division -- this arithmetic runs before the first load of a
// launch and sits in the kernel four times.
__device__ __forceinline__ int div24(int a, int b) {
  return (int)(((unsigned)a & 0xffffffu) / ((unsigned)b & 0xffffffu));
}
__device__ __forceinline__ void tile_of(int t, int nblk, int tiles_m, int tiles_n, int& tile_m,
                                        int& tile_n) {
  const int per = nblk / 8, rem = nblk % 8;
  const int xcd = t % 8, loc = t / 8;
  const int pid = xcd * per + (xcd < rem ? xcd : rem) + loc;
  constexpr int GROUP = 8;
  const int group_sz = GROUP * tiles_n;
  const int grp = div24(pid, group_sz);
  const int in_grp = pid - grp * group_sz;
  const int first_m = grp * GROUP;
  const int gm = min(tiles_m - first_m, GROUP);
  tile_n = div24(in_grp, gm);
  tile_m = first_m + (in_grp - tile_n * gm);
}

// ---------------------------------------------------------------------------------
// One output tile of TM x TN = (WGM * MB * 32) x (WGN * NB * 32) on WGM * WGN wavefronts: rows
// row0 .. row0 + TM of A (clamped to row_end - 1 when read, not stored from row_end on) times
// rows tn * TN .. of W.  K steps of 128 bytes go through a ring of NST stages in `smem`
// ((TM + TN) * 128 bytes each) filled by global_load_lds_dwordx4; fragments are double-buffered
// per 32-byte slice and the issue order inside a slice is pinned (one LDS read after each of
// the first MFMAs); the step's barrier sits before the last slice's MFMAs, after it the freed
// stage is refilled with step kt + NST.  The tabulated epilogue brings its TN x 256-byte table
// into the stage that the second-to-last step frees, while the last step is multiplied.
// Every wavefront of the workgroup must call it (it holds workgroup barriers: tile_gemm_barriers
// of them); the caller separates two calls by a barrier of its own.
// Preconditions: K % 128 == 0, K / 128 >= NST, N % 16 == 0, operands 16-byte aligned and below 2^32
// bytes (BLOCKED: K below 2^24, the offsets count from the tile).  A_FROM_L2: the rows of A were
// written by other compute units of this XCD during this launch (read past the vector cache).
// BLOCKED: both operands in the blocked layout, row0 a multiple of 16.
// ---------------------------------------------------------------------------------
template <typename Epi, typename = void>
struct EpiHasClips : std::false_type {};
template <typename Epi>
struct EpiHasClips<Epi, std::enable_if_t<Epi::kClips>> : std::true_type {};
struct EpiNoRaw {};
template <typename Epi>
__device__ __forceinline__ auto epi_request(const Epi& e) {
  if constexpr (EpiHasClips<Epi>::value) return e.request();
  else return EpiNoRaw{};
}
template <typename Epi, typename Raw>
__device__ __forceinline__ Epi epi_finish(const Epi& e, const Raw& raw) {
  if constexpr (EpiHasClips<Epi>::value) return e.finish(raw);
  else return e;
}

// kFetch (optional): store4 needs values of its own elements (a residual, where a row goes).
// fetch(m, n, N) requests those of the columns n .. n + 3 of row m, ahead of the products or of the
// first store; store4 takes them as its last argument.
template <typename Epi, typename = void>
struct EpiHasFetch : std::false_type {};
template <typename Epi>
struct EpiHasFetch<Epi, std::enable_if_t<Epi::kFetch>> : std::true_type {};
struct EpiNoFetch {};
template <typename Epi>
__device__ __forceinline__ auto epi_fetch(const Epi& e, int m, int n, int N) {
  if constexpr (EpiHasFetch<Epi>::value) return e.fetch(m, n, N);
  else return EpiNoFetch{};
}
template <typename Epi, typename Acc, typename Fetched>
__device__ __forceinline__ void epi_store4(const Epi& e, int m, int n, int N, const typename Epi::Col& col,
                                           const Acc& c, const Fetched& x) {
  if constexpr (EpiHasFetch<Epi>::value) e.store4(m, n, N, col, c, x);
  else e.store4(m, n, N, col, c);
}
// kColumn16, kFetch16 (optional): what store16 needs of the columns n .. n + 15, and of row m or of its
// 16 elements, requested ahead of the K loop and handed to it.  An epilogue that asks for them when
// it needs them waits for one memory trip after another: 976 x 3072 x 1024 into heads 13.5 us so,
// 9.2 with both requested (and 9.9 with the rows laid out in LDS and stored 64 columns at a time,
// the accumulators' layout being no friend of whole lines).
template <typename Epi, typename = void>
struct EpiHasColumn16 : std::false_type {};
template <typename Epi>
struct EpiHasColumn16<Epi, std::enable_if_t<Epi::kColumn16>> : std::true_type {};
template <typename Epi>
__device__ __forceinline__ auto epi_column16(const Epi& e, int n) {
  if constexpr (EpiHasColumn16<Epi>::value) return e.column16(n);
  else return EpiNoFetch{};
}
template <typename Epi, typename = void>
struct EpiHasFetch16 : std::false_type {};
template <typename Epi>
struct EpiHasFetch16<Epi, std::enable_if_t<Epi::kFetch16>> : std::true_type {};
template <typename Epi>
__device__ __forceinline__ auto epi_fetch16(const Epi& e, int m, int n, int N) {
  if constexpr (EpiHasFetch16<Epi>::value) return e.fetch16(m, n, N);
  else return EpiNoFetch{};
}
// 32 x 32 products over 32 bytes of K: int8, or fp16 (the lanes hold the operands alike)
__device__ __forceinline__ v16i mma32(const v4i& w, const v4i& a, const v16i& c) {
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(w, a, c, 0, 0, 0);
}
__device__ __forceinline__ v16f mma32(const v4i& w, const v4i& a, const v16f& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, a),
                                                c, 0, 0, 0);
}
template <typename Epi, int NST>
constexpr int tile_gemm_barriers(int nk) {
  return nk + (is_lut<Epi> ? 1 : 0);
}

template <typename Epi, int WGM, int WGN, int MB, int NB, int NST, bool A_FROM_L2 = false,
          bool BLOCKED = false, typename Acc16 = v16i>
__device__ __forceinline__ void tile_gemm(const int8_t* __restrict__ A,
                                          const int8_t* __restrict__ W, const Epi& epi_arg, int row0,
                                          int row_end, int N, int K, int tn, int8_t* smem) {
  const auto raw = epi_request(epi_arg);
  constexpr bool LUT = is_lut<Epi>;
  // The operand order of the MFMA decides what a lane's 16 accumulators are: weight rows first,
  // 16 adjacent columns of one output row (one 16-byte store of int8 codes); activations first,
  // 16 rows of one column -- the layout for int32 output, whose stores then cover whole lines.
  constexpr bool ROWS_IN_REGS = std::is_same<Epi, EpiI32>::value;
  constexpr int NWV = WGM * WGN;
  constexpr int TM = WGM * MB * 32, TN = WGN * NB * 32;
  constexpr int STAGE = (TM + TN) * kBK;
  constexpr int NA = TM / 8 / NWV, NW = TN / 8 / NWV, PER = NA + NW;  // 1-KB loads per wavefront
  constexpr int NTAB = TN / 4 / NWV;  // table loads per wavefront
  constexpr int KSTEP = BLOCKED ? 2048 : kBK;  // bytes from one K step of a row to the next
  static_assert(TM % (8 * NWV) == 0 && TN % (8 * NWV) == 0, "stage rows split over the wavefronts");
  static_assert((NST - 1) * PER < 64, "vmcnt range");
  static_assert(!LUT || (TM >= TN && TN % (4 * NWV) == 0), "table fits a freed stage");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WGN, wn = wave % WGN, l32 = lane & 31, g = lane >> 5;
  const int nk = K / kBK;

  decltype(epi_column16(epi_arg, 0)) col16[NB];
  decltype(epi_fetch16(epi_arg, 0, 0, 0)) x16[MB][NB];
  auto first_col = [&](int j) { return min(tn * TN + wn * (NB * 32) + j * 32 + 16 * g, N - 16); };
  auto fetch16 = [&]() {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        x16[i][j] =
            epi_fetch16(epi_arg, min(row0 + wm * (MB * 32) + i * 32 + l32, row_end - 1), first_col(j), N);
  };
#pragma unroll
  for (int j = 0; j < NB; ++j) col16[j] = epi_column16(epi_arg, first_col(j));
  // (wavefronts of more than four blocks have no registers left for residuals until the loop is over)
  constexpr bool FETCH_AHEAD = MB * NB <= 4;
  if (FETCH_AHEAD) fetch16();

  const int8_t *a_tile = A, *w_tile = W;
  if (BLOCKED) {
    a_tile += (long)row0 * K;
    w_tile += (long)tn * TN * K;
  }
  uint32_t a_src[NA], w_src[NW];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int row = (wave + NWV * i) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ key_act(row);
    a_src[i] = (uint32_t)min(row0 + row, row_end - 1) * (uint32_t)K + c * 16;
    if (BLOCKED) {
      // one 1-KB block of 16 rows x 64 bytes per load, as it lies in memory: it is in fragment
      // order already, and 16 lanes of a fragment read are 256 contiguous bytes of LDS
      const int q = wave + NWV * i;
      a_src[i] = (uint32_t)min(q >> 1, ((row_end - 1) >> 4) - (row0 >> 4)) * 16u * (uint32_t)K +
                 (q & 1) * 1024 + lane * 16;
    }
  }
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const int row = (wave + NWV * i) * 8 + (lane >> 3);
    const int c = (lane & 7) ^ key_wgt(row);
    w_src[i] = (uint32_t)min(tn * TN + row, N - 1) * (uint32_t)K + c * 16;
    if (BLOCKED) {
      // the two halves of an odd block's rows change places: 16 lanes in sigma order read eight
      // rows of an even and the same eight of the odd block, which must not share their banks
      const int q = wave + NWV * i;
      w_src[i] = (uint32_t)min(q >> 1, ((N - 1) >> 4) - tn * (TN / 16)) * 16u * (uint32_t)K +
                 (q & 1) * 1024 + (lane ^ ((q >> 1) & 1) * 8) * 16;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) void*)smem);
  auto dma1 = [&](const int8_t* base, uint32_t voff, uint32_t lds) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff),
                 "s"(base)
                 : "memory");
  };
  // the same past this compute unit's vector cache (sc1: the line is taken from the L2), for an
  // operand that another compute unit of the XCD wrote during this launch
  auto dma1_l2 = [&](const int8_t* base, uint32_t voff, uint32_t lds) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2 sc1" ::"s"(lds), "v"(voff),
                 "s"(base)
                 : "memory");
  };
  auto issue = [&](int kt, int slot) {  // K step kt into ring slot `slot`
    const uint32_t base = lds0 + slot * STAGE;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      if (A_FROM_L2) dma1_l2(a_tile + kt * KSTEP, a_src[i], base + (wave + NWV * i) * 1024);
      else dma1(a_tile + kt * KSTEP, a_src[i], base + (wave + NWV * i) * 1024);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i)
      dma1(w_tile + kt * KSTEP, w_src[i], base + TM * kBK + (wave + NWV * i) * 1024);
  };
  // LDS byte offset of this lane's fragment chunk for K slice 0; slice ks is at (offset ^ (ks << 5)):
  // chunk index 2 * ks + g, swizzled by the row key, and 2 * ks only touches bits 1-2 of it
  int a_base[MB], w_base[NB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int row = wm * (MB * 32) + i * 32 + l32;
    a_base[i] = BLOCKED ? (row >> 4) * 2048 + g * 256 + (row & 15) * 16
                        : row * kBK + ((g ^ key_act(row)) << 4);
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int row = wn * (NB * 32) + j * 32 + sigma(l32);
    w_base[j] = TM * kBK + (BLOCKED ? (row >> 4) * 2048 + g * 256 + ((row & 15) ^ ((row >> 4) & 1) * 8) * 16
                                    : row * kBK + ((g ^ key_wgt(row)) << 4));
  }
  auto slice_at = [&](int base, int ks) {
    return BLOCKED ? base + (ks >> 1) * 1024 + (ks & 1) * 512 : base ^ (ks << 5);
  };
  struct Frag {
    v4i a[MB], w[NB];
  };
  auto load_frag = [&](Frag& f, const int8_t* stage, int ks) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
      f.a[i] = *reinterpret_cast<const v4i*>(stage + slice_at(a_base[i], ks));
#pragma unroll
    for (int j = 0; j < NB; ++j)
      f.w[j] = *reinterpret_cast<const v4i*>(stage + slice_at(w_base[j], ks));
  };
  Acc16 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = (Acc16)0;
  auto mma = [&](const Frag& f) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[i][j] = ROWS_IN_REGS ? mma32(f.a[i], f.w[j], acc[i][j]) : mma32(f.w[j], f.a[i], acc[i][j]);
  };
  // issue order of one slice: an LDS read of the next slice after each of the first MFMAs
  auto pattern = [&]() {
#pragma unroll
    for (int q = 0; q < MB + NB; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    if (MB * NB > MB + NB) __builtin_amdgcn_sched_group_barrier(0x008, MB * NB - (MB + NB), 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  Frag f[2];
  auto slices = [&](const int8_t* stage) {  // slices 1..3 read, slices 0..2 multiplied
#pragma unroll
    for (int ks = 1; ks < 4; ++ks) {
      load_frag(f[ks & 1], stage, ks);
      mma(f[(ks - 1) & 1]);
      pattern();
    }
  };

#pragma unroll
  for (int s = 0; s < NST; ++s) issue(s, s);
  wait_vmcnt<(NST - 1) * PER>();
  __builtin_amdgcn_s_barrier();
  load_frag(f[0], smem, 0);
  int slot = 0;
  // steady state: a step ends by refilling its own slot with step kt + NST
  for (int kt = 0; kt < nk - NST; ++kt) {
    slices(smem + slot * STAGE);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wavefront has read all of the stage
    wait_vmcnt<(NST - 2) * PER>();       // its own loads of step kt + 1 have landed ...
    __builtin_amdgcn_s_barrier();        // ... and everyone's; everyone is done with step kt
    issue(kt + NST, slot);
    __builtin_amdgcn_sched_barrier(0);
    if (++slot == NST) slot = 0;
    load_frag(f[0], smem + slot * STAGE, 0);
    mma(f[1]);
    pattern();
  }
  // drain: NST - 1 steps without a refill, then the last step
  int tab_slot = 0;
#pragma unroll
  for (int t = 0; t < NST - 1; ++t) {
    slices(smem + slot * STAGE);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    switch (NST - 2 - t) {  // stages that may still be on their way
      case 0: wait_vmcnt<0>(); break;
      case 1: wait_vmcnt<PER>(); break;
      case 2: wait_vmcnt<2 * PER>(); break;
      default: wait_vmcnt<3 * PER>();
    }
    __builtin_amdgcn_s_barrier();
    if (LUT && t == NST - 2) {
      // the slot of the second-to-last step is free: the tile's table rows go there
      tab_slot = slot;
      const long first = (long)tn * TN * 256, last = (long)N * 256 - 16;
#pragma unroll
      for (int i = 0; i < NTAB; ++i) {
        const int q = wave + NWV * i;
        const long off = min(first + q * 1024 + lane * 16, last);  // rows beyond N: never stored
        dma1(reinterpret_cast<const int8_t*>(epi_lut(epi_arg)), (uint32_t)off,
             lds0 + slot * STAGE + q * 1024);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (++slot == NST) slot = 0;
    load_frag(f[0], smem + slot * STAGE, 0);
    mma(f[1]);
    pattern();
  }
  slices(smem + slot * STAGE);
  mma(f[1]);
  if (LUT) {
    wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
  }
  const Epi epi = epi_finish(epi_arg, raw);
  if constexpr (ROWS_IN_REGS) {
    // int32 output: a lane holds column sigma(l32) of its block and the rows 8 (k / 4) + 4 g +
    // k % 4 in register k, so a store instruction writes two whole 128-byte lines (32 lanes, 32
    // adjacent columns of one row each)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int n = tn * TN + wn * (NB * 32) + j * 32 + sigma(l32);
        int32_t* cp = epi.C + n;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const long m = (long)row0 + wm * (MB * 32) + i * 32 + 8 * (k >> 2) + 4 * g + (k & 3);
          if (m < row_end && n < N) cp[m * N] = acc[i][j][k];
        }
      }
    return;
  }
  if (!FETCH_AHEAD) fetch16();
  const int8_t* tab = smem + tab_slot * STAGE;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const long m = (long)row0 + wm * (MB * 32) + i * 32 + l32;
    if (m < row_end) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int nl = wn * (NB * 32) + j * 32 + 16 * g;
        const int n = tn * TN + nl;
        if (n < N) {
          if constexpr (LUT) epi.store16_lds(m, n, N, acc[i][j], true, tab, nl);
          else if constexpr (EpiHasFetch16<Epi>::value) epi.store16(m, n, N, acc[i][j], col16[j], x16[i][j]);
          else if constexpr (EpiHasColumn16<Epi>::value) epi.store16(m, n, N, acc[i][j], col16[j]);
          else epi.store16(m, n, N, acc[i][j], true);
        }
      }
    }
  }
}

}  // namespace lsh
