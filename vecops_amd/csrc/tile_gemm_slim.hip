// Products whose tiles of 128x128 or 64x64 would leave the chip short of work or of loads in flight: workgroup tiles of 32,
// 64 or 128 rows by 16 to 64 columns (tile_gemm_slim_kernel), one workgroup a compute unit, each walking the whole K.
//
// What bounds it: the loads' way into LDS, (BM + BN) rows of K - a compute unit takes 137 bytes a ns of whole lines by
// itself and 100 where all do, 70 of 16-byte aligned rows that start inside a line and 50 of others - and for weights that
// no cache holds their way from memory (the walks of 128 x 11008 x 4096 and 512 x 4096 x 4096 bring in 60, at 4.3 and 2.7 TB/s of
// HBM, the matrix cores 0.25 and 0.33 busy).  So a tile is chosen by how many bytes the fullest unit fetches (take_slim_tile
// in capi.hip).
//   * Eight wavefronts split a stage's K in four and the tile's rows in two: a tile this narrow has too few fragments for
//     eight wavefronts side by side, and a product of one K part needs no partial sums in memory and no second launch.
//     The four sums meet in LDS at the end.
//   * A stage is two K tiles (256 bytes of a row).  Both operands arrive by loads that write LDS; the first four wavefronts
//     load A and the others B, so that each waits for loads of its own operand and B's ring can be as deep as LDS allows:
//     A's rows come from L2, where the other workgroups find them too, B's are weights that come from memory (one ring for
//     both, three stages: 35 us where this takes 33 at 128 x 11008 x 4096).
//   * A stage's fragments are read while the stage before is multiplied, the refills dealt between the matrix instructions
//     (all refills first: 34.5 us there; four wavefronts and stages of one K tile 37).
//   * A partial last K tile is walked first, through checked stores, as in tile_gemm_kernel.
// Measured (us, launch to launch, weights not in a cache / in one; before: the plan's own kernels with their K split):
// 17 x 412 x 1472 9.9 / 9.0 -> 5.7 / 5.3, 64 x 2048 x 1408 10.5 / 8.0 -> 5.8 / 5.3, 91 x 2011 x 640 10.1 / 9.1 -> 5.7 / 5.5,
// 128 x 1984 x 2048 13.3 / 9.9 -> 7.2 / 6.8, 100 x 4224 x 4672 40 / 26 -> 22 / 15, 512 x 1408 x 3520 25 / 21 -> 15 / 13,
// 128 x 11008 x 4096 37 / 25 -> 33 / 23.
#include "tile_gemm_launch.h"

namespace vecops_hip {

namespace {

constexpr int kParts = 4;                                        // of a stage's K: two wavefronts each
constexpr int kThreads = 128 * kParts;
constexpr int kStageTiles = 2;                                   // K tiles of 128 bytes in a stage

template <int BM, int BN>
struct SlimTile {
  static constexpr int kStageA = BM * 128 * kStageTiles, kStageB = BN * 128 * kStageTiles;
  static constexpr int kLoadsA = kStageA / 4096, kLoadsB = kStageB / 4096;  // loads of 1 KiB each of four wavefronts has in a stage
  static constexpr int kStagesA = BM == 128 ? 3 : 4;
  static constexpr int kFitB = (160 * 1024 - kStagesA * kStageA) / kStageB;
  static constexpr int kStagesB = kFitB < 16 ? kFitB : 16;
  static_assert(kStagesB >= 3, "a stage being multiplied, one in flight and one more");
  static_assert(kLoadsB * (kStagesB - 2) < 64, "the wait counts loads in flight in six bits");
  static constexpr int kBaseB = kStagesA * kStageA;
  static constexpr int kPitch = BN + 4;                          // words between the rows of the sums
  static constexpr int kSums = kParts * BM * kPitch * 4;
  static constexpr int kStages = kBaseB + kStagesB * kStageB;
  static constexpr int kLds = kStages > kSums ? kStages : kSums;
  static_assert(kLds <= 160 * 1024, "LDS of a compute unit");
};

// The work of one workgroup: number `pid` of the `total` that serve the problem `p`.
template <int SRC, int BM, int BN>
__device__ __forceinline__ void slim_workgroup(const TileGemmParams& p, int pid, int total) {
  using T = SrcTraits<SRC>;
  using L = SlimTile<BM, BN>;
  using Quad = typename AccQuad<T::kInt>::type;
  constexpr int KTILE = 8 * T::kElemsPerChunk;
  constexpr int FM = BM / 32, FN = BN / 16;  // 16-row fragments of a wavefront: half the rows, every column
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wk = wave >> 1;  // half of the rows, quarter of a stage's K
  int batch, split, tm, tn;
  map_workgroup(p, pid, total, batch, split, tm, tn);
  batch = __builtin_amdgcn_readfirstlane(batch);
  if (batch >= p.batch) return;  // a grouped launch rounds each group's run of workgroups up to a multiple of eight
  tm = __builtin_amdgcn_readfirstlane(tm);
  tn = __builtin_amdgcn_readfirstlane(tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int full = p.k / KTILE;
  const int has_tail = p.k % KTILE != 0 ? 1 : 0;
  const int nk = full + has_tail;
  const int stages = (nk + kStageTiles - 1) / kStageTiles;
  const char* a = static_cast<const char*>(p.a) + (batch * p.a_bs + static_cast<int64_t>(m0) * p.a_rs) * T::kSrcBytes;
  const char* b = static_cast<const char*>(p.b) + (batch * p.b_bs + static_cast<int64_t>(n0) * p.b_rs) * T::kSrcBytes;
  const u32x4 desc_a = tile_buffer_words((const VECOPS_GLOBAL char*)a), desc_b = tile_buffer_words((const VECOPS_GLOBAL char*)b);
  const uint32_t lds0 = lds_address_of(lds);

  // the first half of the wavefronts load A, the second B: each waits for loads of its own operand only
  const bool loads_a = wave < 4;
  const int loader = wave & 3;
  constexpr int kMostLoads = L::kLoadsA > L::kLoadsB ? L::kLoadsA : L::kLoadsB;
  uint32_t row_bytes[kMostLoads];
  {
    const int first_row = loads_a ? m0 : n0, last = (loads_a ? p.m : p.n) - 1;
    const int blocks = loads_a ? BM / 8 : BN / 8;   // of eight rows in a K tile
    const int64_t pitch = (loads_a ? p.a_rs : p.b_rs) * T::kSrcBytes;
#pragma unroll
    for (int i = 0; i < kMostLoads; ++i) {
      const int tile_row = (i * 4 + loader) % blocks * 8 + (lane >> 3);
      const int chunk = ((lane & 7) ^ tile_row ^ (tile_row >> 3)) & 7;
      row_bytes[i] = static_cast<uint32_t>((min(first_row + tile_row, last) - first_row) * pitch + chunk * 16);
    }
  }
  auto load_one = [&](auto rows_tag, const u32x4& descriptor, uint32_t base, int i, int s, bool first) {
    constexpr int ROWS = decltype(rows_tag)::value;
    const int block = i * 4 + loader, half = block >= ROWS / 8 ? 1 : 0;
    const int j = kStageTiles * s + half;
    if (first && has_tail && half == 0) return;
    u32x4 desc = descriptor;
    desc[2] = __builtin_amdgcn_readfirstlane(j < nk ? desc[2] : 0u);
    load_16_bytes_into_lds(desc, __builtin_amdgcn_readfirstlane(base), __builtin_amdgcn_readfirstlane(block * 1024), row_bytes[i],
                           __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(max(j - has_tail, 0)) * 128u));
  };
  using std::integral_constant;
  auto load_a = [&](int i, int s, int slot, bool first) {
    load_one(integral_constant<int, BM>{}, desc_a, lds0 + slot * L::kStageA, i, s, first);
  };
  auto load_b = [&](int i, int s, int slot, bool first) {
    load_one(integral_constant<int, BN>{}, desc_b, lds0 + L::kBaseB + slot * L::kStageB, i, s, first);
  };
  if (loads_a) {
#pragma unroll
    for (int s = 0; s < L::kStagesA - 1; ++s)
#pragma unroll
      for (int i = 0; i < L::kLoadsA; ++i) load_a(i, s, s, s == 0);
  } else {
#pragma unroll
    for (int s = 0; s < L::kStagesB - 1; ++s)
#pragma unroll
      for (int i = 0; i < L::kLoadsB; ++i) load_b(i, s, s, s == 0);
  }
  if (has_tail) {
    stage_rows_checked<SRC>(static_cast<const char*>(p.a) + batch * p.a_bs * T::kSrcBytes, p.a_rs, 1, m0, p.m, BM, full * KTILE, p.k, lds, tid, kThreads, 0u);
    stage_rows_checked<SRC>(static_cast<const char*>(p.b) + batch * p.b_bs * T::kSrcBytes, p.b_rs, 1, n0, p.n, BN, full * KTILE, p.k, lds + L::kBaseB, tid, kThreads, 0u);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // fragment reads: as in tile_gemm_kernel's 16x16 form
  const int frag_row = lane & 15, frag_chunk = ((lane >> 4) & 1) << 1 | (lane >> 5);
  uint32_t at_a[FM], at_b[FN];
  {
    const int chunk = (wk & 1) * 4 + frag_chunk;
#pragma unroll
    for (int f = 0; f < FM; ++f) at_a[f] = lds0 + (wk >> 1) * BM * 128 + lds_chunk_offset(wm * (BM / 2) + 16 * f + frag_row, chunk);
#pragma unroll
    for (int f = 0; f < FN; ++f) at_b[f] = lds0 + L::kBaseB + (wk >> 1) * BN * 128 + lds_chunk_offset(16 * f + frag_row, chunk);
  }
  typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
  u32x4 fa[2][FM], fb[2][FN];
  Quad acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = Quad{0, 0, 0, 0};

  int slot_a = 0, slot_b = 0;  // of the stage being read
  // Stage s: its fragments are read, the stage the barrier has freed is refilled, and stage s - 1 is multiplied meanwhile.
  auto step = [&](auto role_tag, auto set_tag, auto multiplies_tag, int s) {
    constexpr bool A = decltype(role_tag)::value;
    constexpr int SET = decltype(set_tag)::value;
    constexpr int LOADS = A ? L::kLoadsA : L::kLoadsB, STAGES = A ? L::kStagesA : L::kStagesB;
    // this stage has landed, and the reads of the one before it
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS * (STAGES - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint32_t offset_a = static_cast<uint32_t>(slot_a * L::kStageA), offset_b = static_cast<uint32_t>(slot_b * L::kStageB);
#pragma unroll
    for (int f = 0; f < FM; ++f) fa[SET][f] = *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_a[f] + offset_a));
#pragma unroll
    for (int f = 0; f < FN; ++f) fb[SET][f] = *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_b[f] + offset_b));
    __builtin_amdgcn_sched_barrier(0);
    static_for<LOADS>([&](auto ci) {
      constexpr int i = decltype(ci)::value;
      if constexpr (A) load_a(i, s + STAGES - 1, slot_a == 0 ? STAGES - 1 : slot_a - 1, false);
      else load_b(i, s + STAGES - 1, slot_b == 0 ? STAGES - 1 : slot_b - 1, false);
      if constexpr (decltype(multiplies_tag)::value) {
        constexpr int x0 = i * FM * FN / LOADS, x1 = (i + 1) * FM * FN / LOADS;
        static_for<x1 - x0>([&](auto cx) {
          constexpr int x = x0 + decltype(cx)::value;
          mfma_step16<SRC>(acc[x / FN][x % FN], fb[SET ^ 1][x % FN], fa[SET ^ 1][x / FN]);
        });
        __builtin_amdgcn_sched_barrier(0);
      }
    });
    slot_a = slot_a + 1 == L::kStagesA ? 0 : slot_a + 1;
    slot_b = slot_b + 1 == L::kStagesB ? 0 : slot_b + 1;
  };
  auto multiply = [&](auto set_tag) {
    constexpr int SET = decltype(set_tag)::value;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) mfma_step16<SRC>(acc[i][j], fb[SET][j], fa[SET][i]);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  auto walk = [&](auto role) {
    step(role, I0{}, std::false_type{}, 0);
    int s = 1;
    for (; s + 1 < stages; s += 2) {
      step(role, I1{}, std::true_type{}, s);
      step(role, I0{}, std::true_type{}, s + 1);
    }
    if (s < stages) {
      step(role, I1{}, std::true_type{}, s);
      multiply(I1{});
    } else {
      multiply(I0{});
    }
  };
  if (loads_a) walk(std::true_type{});
  else walk(std::false_type{});

  // the four quarters of K meet in LDS
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  uint32_t* sums = reinterpret_cast<uint32_t*>(lds);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
      *reinterpret_cast<u32x4*>(sums + (wk * BM + wm * (BM / 2) + 16 * i + frag_row) * L::kPitch + 16 * j + (lane >> 4) * 4) =
          __builtin_bit_cast(u32x4, acc[i][j]);
  __syncthreads();
  constexpr bool INT = T::kInt;
  const bool vec_c = c_takes_quads(p);
  const bool dequant = INT && p.row_scales != nullptr;
  // contiguous rows of C and of a C input: a quad at a time through the finishing step; else the general store
  const bool simple = vec_c && (p.cin == nullptr || (p.cin_cs == 1 && !dequant));
  const Finisher fin = make_finisher<INT>(p, dequant);
  constexpr int QUADS = BM * (BN / 4), PER = (QUADS + kThreads - 1) / kThreads;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int idx = i * kThreads + tid;
    const int row = idx / (BN / 4), quad = idx % (BN / 4), col = n0 + quad * 4, cols_left = p.n - col;
    if (idx >= QUADS || m0 + row >= p.m || cols_left <= 0) continue;
    u32x4 bits = *reinterpret_cast<const u32x4*>(sums + row * L::kPitch + quad * 4);
#pragma unroll
    for (int part = 1; part < kParts; ++part) {
      const u32x4 more = *reinterpret_cast<const u32x4*>(sums + (part * BM + row) * L::kPitch + quad * 4);
      if constexpr (INT) bits += more;
      else bits = __builtin_bit_cast(u32x4, __builtin_bit_cast(f32x4, bits) + __builtin_bit_cast(f32x4, more));
    }
    if (!simple || cols_left < 4) {
      store_quad_general<INT>(p, batch, 0, m0 + row, col, bits, vec_c, false);
      continue;
    }
    if constexpr (INT) {
      if (p.correction) {
#pragma unroll
        for (int e = 0; e < 4; ++e) bits[e] += static_cast<uint32_t>(p.correction[batch * p.correction_bs + col + e]);
      }
      if (dequant) {
        const float row_scale = p.row_scales[batch * p.row_scales_bs + m0 + row];
#pragma unroll
        for (int e = 0; e < 4; ++e)   // row scale first, then the column's
          bits[e] = __float_as_uint((static_cast<float>(static_cast<int32_t>(bits[e])) * row_scale) * p.column_scales[col + e]);
      }
    }
    f32x4 column_scales = {1.f, 1.f, 1.f, 1.f};
    if (p.fused && p.ep_column_scales) {
#pragma unroll
      for (int e = 0; e < 4; ++e) column_scales[e] = p.ep_column_scales[col + e];
    }
    uint32_t out[4];
    finish_quad(p, fin, bits, batch, m0 + row, col, 4, column_scales, out);
    store_quad_bits(p, batch * p.c_bs + static_cast<int64_t>(m0 + row) * p.c_rs + col, out);
  }
}

template <int SRC, int BM, int BN>
__global__ __launch_bounds__(kThreads, 2) void tile_gemm_slim_kernel(const TileGemmParams p) {
  slim_workgroup<SRC, BM, BN>(p, blockIdx.x, gridDim.x);
}

// Several problems in one launch: the groups of a grouped call that split K on their own.  Each of them a launch (and mostly
// two) of its own, a call over eighteen groups of 43 x 409 x 1985 took 155 us; together 15.
template <int SRC, int BM, int BN>
__global__ __launch_bounds__(kThreads, 2) void tile_gemm_slim_grouped_kernel(const GroupLaunch) {
  int begin = 0, end = 0;
  const TileGemmParams p = group_problem<SRC>(BM, BN, blockIdx.x, begin, end);
  slim_workgroup<SRC, BM, BN>(p, static_cast<int>(blockIdx.x) - begin, end - begin);
}

// > 64 KiB of dynamic LDS has to be enabled once per kernel and device; cheap enough to repeat per thread.
template <auto KERNEL, int LDS>
hipError_t allow_lds() {
  static thread_local int configured_device = -1;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  if (configured_device != device) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    if (e != hipSuccess) return e;
    configured_device = device;
  }
  return hipSuccess;
}

template <int SRC, int BM, int BN>
hipError_t launch_grouped(const GroupLaunch& t, int32_t workgroups, hipStream_t stream) {
  constexpr auto kernel = tile_gemm_slim_grouped_kernel<SRC, BM, BN>;
  constexpr int kLds = SlimTile<BM, BN>::kLds;
  if (hipError_t e = allow_lds<kernel, kLds>(); e != hipSuccess) return e;
  if (workgroups <= 0) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(workgroups)), dim3(kThreads), kLds, stream, t);
  return hipGetLastError();
}

template <int SRC>
hipError_t launch_grouped_tile(const GroupLaunch& t, int32_t workgroups, int bm, int bn, hipStream_t stream) {
  switch (bm * 1000 + bn) {
    case 32032: return launch_grouped<SRC, 32, 32>(t, workgroups, stream);
    case 32064: return launch_grouped<SRC, 32, 64>(t, workgroups, stream);
    case 64064: return launch_grouped<SRC, 64, 64>(t, workgroups, stream);
    case 128064: return launch_grouped<SRC, 128, 64>(t, workgroups, stream);
    default: return hipErrorInvalidValue;
  }
}

template <int SRC, int BM, int BN>
hipError_t launch(TileGemmParams p, hipStream_t stream) {
  constexpr auto kernel = tile_gemm_slim_kernel<SRC, BM, BN>;
  constexpr int kLds = SlimTile<BM, BN>::kLds;
  if (hipError_t e = allow_lds<kernel, kLds>(); e != hipSuccess) return e;
  p.tiles_m = (p.m + BM - 1) / BM;
  p.tiles_n = (p.n + BN - 1) / BN;
  p.split_k = 1;
  const int64_t grid = static_cast<int64_t>(p.tiles_m) * p.tiles_n * p.batch;
  if (grid <= 0 || grid > INT32_MAX) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(grid)), dim3(kThreads), kLds, stream, p);
  return hipGetLastError();
}

template <int SRC>
hipError_t launch_class(const TileGemmParams& p, int bm, int bn, hipStream_t stream) {
  switch (bm * 1000 + bn) {
    case 32016: return launch<SRC, 32, 16>(p, stream);
    case 32032: return launch<SRC, 32, 32>(p, stream);
    case 32048: return launch<SRC, 32, 48>(p, stream);
    case 32064: return launch<SRC, 32, 64>(p, stream);
    case 64048: return launch<SRC, 64, 48>(p, stream);
    case 64064: return launch<SRC, 64, 64>(p, stream);
    case 128048: return launch<SRC, 128, 48>(p, stream);
    case 128064: return launch<SRC, 128, 64>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

bool launch_tile_gemm_slim_serves(int src, const TileGemmParams& p) {
  if (src != SRC_BF16 && src != SRC_F16 && src != SRC_I8) return false;
  if (p.m <= 0 || p.n <= 0 || p.k <= 0 || p.a_ks != 1 || p.b_ks != 1 || p.a_rs < 0 || p.b_rs < 0) return false;
  // 32-bit byte offsets inside a tile's rows
  const int64_t elem = src == SRC_I8 ? 1 : 2;
  const int64_t most = (int64_t{1} << 31) - 256;
  return (128 * p.a_rs + p.k) * elem < most && (64 * p.b_rs + p.k) * elem < most;
}

hipError_t launch_tile_gemm_slim(int src, const TileGemmParams& p, int bm, int bn, hipStream_t stream) {
  switch (src) {
    case SRC_BF16: return launch_class<SRC_BF16>(p, bm, bn, stream);
    case SRC_F16: return launch_class<SRC_F16>(p, bm, bn, stream);
    case SRC_I8: return launch_class<SRC_I8>(p, bm, bn, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_tile_gemm_slim_grouped(int src, const GroupLaunch& t, int32_t workgroups, int bm, int bn, hipStream_t stream) {
  switch (src) {
    case SRC_BF16: return launch_grouped_tile<SRC_BF16>(t, workgroups, bm, bn, stream);
    case SRC_F16: return launch_grouped_tile<SRC_F16>(t, workgroups, bm, bn, stream);
    case SRC_I8: return launch_grouped_tile<SRC_I8>(t, workgroups, bm, bn, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vecops_hip
