// The 128x256 workgroup tile for K-contiguous operands whose rows lie at any alignment (an odd K): three LDS stages filled by
// loads that write LDS, two K tiles ahead.
//
// What bounds it: rows that do not start on a line have their K tiles of 128 bytes in two lines each, and a compute unit
// fetches such rows at 50 bytes a ns where whole lines come at 100 (256 units, rows 2 bytes off).  tile_gemm_kernel serves
// these operands through staging registers one K tile ahead: with operands that no cache holds it waits for memory on top
// (8 x 777 x 1000 x 3001 bf16: 67 us on one set of operands, 85 with eight in turn).  Here (59 and 77) a load has two K tiles
// to land, and eight wavefronts of 64x64, two a SIMD, multiply meanwhile.  bf16, f16 and int8 at 1 to 140 K tiles (12633 products,
// the mean of operands in a cache and not): 0.63 of the staged kernel's time with up to four K tiles, 0.65 to 0.74 up to sixteen,
// 0.8 up to 64, 0.88 beyond; slower, by 4 %, one of them (3160 x 4556 x 21).
#include "tile_gemm_launch.h"

namespace vecops_hip {

namespace {

constexpr int kThreads = 512;
constexpr int kRowsA = 128, kRowsB = 256;
constexpr int kStage = (kRowsA + kRowsB) * 128, kStages = 3;
constexpr int kLoads = kStage / 1024 / 8;          // loads of 1 KiB each of eight wavefronts has in a stage
constexpr int kLoadsA = kRowsA * 128 / 1024 / 8;   // the first of them A's
constexpr int kLds = kStage * kStages;
static_assert(kLds >= kEpilogueLdsBytes<2, 4, 2, 2>() && kLds <= 160 * 1024, "the epilogue lays C out in the stages");

template <int SRC>
__global__ __launch_bounds__(kThreads, 2) void tile_gemm_rows_kernel(const TileGemmParams p) {
  using T = SrcTraits<SRC>;
  constexpr bool INT = T::kInt;
  constexpr int KTILE = 8 * T::kElemsPerChunk;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  int batch, split, tm, tn;
  map_workgroup(p, blockIdx.x, gridDim.x, batch, split, tm, tn);
  batch = __builtin_amdgcn_readfirstlane(batch);
  split = __builtin_amdgcn_readfirstlane(split);
  tm = __builtin_amdgcn_readfirstlane(tm);
  tn = __builtin_amdgcn_readfirstlane(tn);
  const int m0 = tm * kRowsA, n0 = tn * kRowsB;
  // the walk over K as in tile_gemm_workgroup: a partial last K tile comes first
  const int total_k_tiles = (p.k + KTILE - 1) / KTILE, full_k_tiles = p.k / KTILE;
  const int kt_begin = split * p.k_tiles_per_split, kt_end = min(total_k_tiles, kt_begin + p.k_tiles_per_split);
  const int nk = __builtin_amdgcn_readfirstlane(max(kt_end - kt_begin, 0));
  const int has_tail = __builtin_amdgcn_readfirstlane(nk > 0 && kt_end > full_k_tiles ? 1 : 0);

  const char* a = static_cast<const char*>(p.a) + batch * p.a_bs * T::kSrcBytes;
  const char* b = static_cast<const char*>(p.b) + batch * p.b_bs * T::kSrcBytes;
  const u32x4 desc_a = tile_buffer_words((const VECOPS_GLOBAL char*)(a + static_cast<int64_t>(m0) * p.a_rs * T::kSrcBytes));
  const u32x4 desc_b = tile_buffer_words((const VECOPS_GLOBAL char*)(b + static_cast<int64_t>(n0) * p.b_rs * T::kSrcBytes));
  const uint32_t lds0 = lds_address_of(lds);
  // load i of this wavefront in a stage fills rows 64 i + 8 wave .. + 7 of the stage's A and B rows; lane l fetches the chunk
  // whose swizzled slot is l % 8.  Rows past the extent are clamped onto the last one: loaded, multiplied, never stored.
  uint32_t row_bytes[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const bool of_a = i < kLoadsA;
    const int tile_row = (of_a ? i : i - kLoadsA) * 64 + wave * 8 + (lane >> 3);
    const int chunk = ((lane & 7) ^ tile_row ^ (tile_row >> 3)) & 7;
    const int first = of_a ? m0 : n0, row = min(first + tile_row, (of_a ? p.m : p.n) - 1) - first;
    row_bytes[i] = static_cast<uint32_t>(static_cast<int64_t>(row) * (of_a ? p.a_rs : p.b_rs) * T::kSrcBytes + chunk * 16);
  }
  // position `t` of the walk into LDS stage `slot`; past the end: loads that fetch nothing, so that the count of loads in
  // flight holds
  auto load = [&](int i, int t, int slot) {
    u32x4 desc = i < kLoadsA ? desc_a : desc_b;
    desc[2] = __builtin_amdgcn_readfirstlane(t < nk ? desc[2] : 0u);
    load_16_bytes_into_lds(desc, __builtin_amdgcn_readfirstlane(lds0 + slot * kStage), __builtin_amdgcn_readfirstlane((i * 8 + wave) * 1024),
                           row_bytes[i], __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(max(kt_begin + t - has_tail, 0)) * 128u));
  };
  if (!has_tail)
#pragma unroll
    for (int i = 0; i < kLoads; ++i) load(i, 0, 0);
#pragma unroll
  for (int i = 0; i < kLoads; ++i) load(i, 1, 1);
  if (has_tail) {
    stage_rows_checked<SRC>(a, p.a_rs, 1, m0, p.m, kRowsA, (kt_end - 1) * KTILE, p.k, lds, tid, kThreads, 0u);
    stage_rows_checked<SRC>(b, p.b_rs, 1, n0, p.n, kRowsB, (kt_end - 1) * KTILE, p.k, lds + kRowsA * 128, tid, kThreads, 0u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // fragment reads: as in tile_gemm_kernel's 16x16 form, [k-step]
  const int frag_row = lane & 15, frag_chunk = ((lane >> 4) & 1) << 1 | (lane >> 5);
  uint32_t at_a[2][4], at_b[2][4];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      at_a[ks][f] = lds0 + lds_chunk_offset(wm * 64 + 16 * f + frag_row, 4 * ks + frag_chunk);
      at_b[ks][f] = lds0 + kRowsA * 128 + lds_chunk_offset(wn * 64 + 16 * f + frag_row, 4 * ks + frag_chunk);
    }
  typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
  u32x4 fa[2][4], fb[2][4];
  Accumulators<INT, 2, 2, true> acc;
  acc.clear();
  auto read = [&](auto ks_tag, uint32_t stage) {
    constexpr int KS = decltype(ks_tag)::value;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      fa[KS][f] = *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_a[KS][f] + stage));
      fb[KS][f] = *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_b[KS][f] + stage));
    }
  };
  auto multiply = [&](auto ks_tag, auto from, auto to) {
    constexpr int KS = decltype(ks_tag)::value, FROM = decltype(from)::value;
    static_for<decltype(to)::value - FROM>([&](auto cx) {
      constexpr int x = FROM + decltype(cx)::value;
      mfma_step16<SRC>(acc.t[x >> 2][x & 3], fb[KS][x & 3], fa[KS][x >> 2]);
    });
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using All = std::integral_constant<int, 16>;
  int slot = 0;
  // K tile t: its first k-step's fragments are read while the second k-step of the tile before is multiplied, and the stage
  // that the barrier has freed is refilled between those matrix instructions
  auto k_tile = [&](auto multiplies_tag, int t) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kLoads) : "memory");   // the next tile's loads may be in flight
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint32_t stage = static_cast<uint32_t>(slot * kStage);
    read(I0{}, stage);
    __builtin_amdgcn_sched_barrier(0);
    const int refill = slot == 0 ? kStages - 1 : slot - 1;
    static_for<kLoads>([&](auto ci) {
      constexpr int i = decltype(ci)::value;
      load(i, t + 2, refill);
      if constexpr (decltype(multiplies_tag)::value) {
        multiply(I1{}, std::integral_constant<int, i * 16 / kLoads>{}, std::integral_constant<int, (i + 1) * 16 / kLoads>{});
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    read(I1{}, stage);
    __builtin_amdgcn_sched_barrier(0);
    multiply(I0{}, I0{}, All{});
    slot = slot + 1 == kStages ? 0 : slot + 1;
  };
  if (nk > 0) {
    k_tile(std::false_type{}, 0);
#pragma unroll 1
    for (int t = 1; t < nk; ++t) k_tile(std::true_type{}, t);
    multiply(I1{}, I0{}, All{});
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // (the last trips' loads, before C is laid out in the stages)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  store_accumulators<SRC, 2, 4, 2, 2, kLds, true>(p, lds, acc, batch, split, m0, n0, wm, wn, wave, lane);
}

template <int SRC>
hipError_t launch(TileGemmParams p, hipStream_t stream) {
  auto kernel = tile_gemm_rows_kernel<SRC>;
  static thread_local int configured_device = -1;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  if (configured_device != device) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) return e;
    configured_device = device;
  }
  p.tiles_m = (p.m + kRowsA - 1) / kRowsA;
  p.tiles_n = (p.n + kRowsB - 1) / kRowsB;
  const int64_t grid = static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.batch * p.split_k;
  if (grid <= 0 || grid > INT32_MAX) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), kLds, stream, p);
  return hipGetLastError();
}

}  // namespace

bool launch_tile_gemm_rows_serves(int src, const TileGemmParams& p) {
  if (src != SRC_BF16 && src != SRC_F16 && src != SRC_I8) return false;
  if (p.m <= 0 || p.n <= 0 || p.k <= 0 || p.split_k < 1 || p.a_ks != 1 || p.b_ks != 1 || p.a_rs < 0 || p.b_rs < 0) return false;
  // 32-bit byte offsets inside a tile's rows
  const int64_t elem = src == SRC_I8 ? 1 : 2, most = (int64_t{1} << 31) - 256;
  return (kRowsA * p.a_rs + p.k) * elem < most && (kRowsB * p.b_rs + p.k) * elem < most;
}

hipError_t launch_tile_gemm_rows(int src, const TileGemmParams& p, hipStream_t stream) {
  switch (src) {
    case SRC_BF16: return launch<SRC_BF16>(p, stream);
    case SRC_F16: return launch<SRC_F16>(p, stream);
    case SRC_I8: return launch<SRC_I8>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vecops_hip
