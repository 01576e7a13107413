// Weight-only products (bf16 activations of up to 16 rows, int8 weights with a scale per row and group) for any K: a workgroup
// walks the whole K of 16 to 64 weight rows.
//
// What bounds it: the weights' way from memory.  Every byte of them is read once, so what counts is how many are under way:
// the weights arrive by loads that write LDS, in a ring of stages of 512 k, and the activations - which every workgroup reads
// whole, from L2 - in a ring of their own.  The first four wavefronts load activations, the others weights, so that each
// waits for loads of its own operand only; the workgroup's scales, one contiguous piece, are fetched into LDS once.  A stage's
// k are dealt to the eight wavefronts, whose sums meet in LDS at the end.  (skinny_w8a16_mfma_kernel loads weights,
// activations and scales as matrix-core fragments, 64 bytes of each of sixteen rows an instruction: four times the cycles a
// byte in the memory pipeline.)
#include "w8a16_ring.h"

#include "tile_gemm.h"

namespace vecops_hip {

namespace {

constexpr int kThreads = 512;
constexpr int kStageK = 512;                       // k of a stage: 64 for each wavefront
constexpr int kStageX = 16 * kStageK * 2, kStagesX = 3;
constexpr int kLoadsX = kStageX / 4096;            // loads of 1 KiB each of four wavefronts has in a stage
constexpr int kMostLds = 160 * 1024;

template <int BN>
struct RingTile {
  static constexpr int kStageW = BN * kStageK;
  static constexpr int kLoadsW = kStageW / 4096;
  static constexpr int kStagesW = BN == 64 ? 3 : BN == 48 ? 3 : BN == 32 ? 5 : 8;
  static constexpr int kBaseW = kStagesX * kStageX;
  static constexpr int kBaseScales = kBaseW + kStagesW * kStageW;
  static constexpr int kSums = 8 * BN * 16 * 4;
  static constexpr int kMostScales = kMostLds - kBaseScales;   // bytes of scales that fit behind the rings
  static_assert(kMostScales >= 8192 && kSums <= kBaseScales, "LDS of a compute unit");
};

template <int BN>
__global__ __launch_bounds__(kThreads, 2) void w8a16_ring_kernel(const SkinnyW8A16Params p, int group_shift) {
  using L = RingTile<BN>;
  constexpr int TILES = BN / 16;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = static_cast<int>(blockIdx.x) * BN;
  const int rows = min(BN, p.n - n0);
  const uint32_t lds0 = lds_address_of(lds);
  const int stages = (p.k + kStageK - 1) / kStageK;

  // the scales of the workgroup's rows, as they lie in memory; what lies past the last row arrives as zeros
  {
    u32x4 desc = tile_buffer_words((const VECOPS_GLOBAL char*)(p.scales + static_cast<int64_t>(n0) * p.groups));
    const uint32_t bytes = static_cast<uint32_t>(rows) * p.groups * 4u;
    desc[2] = __builtin_amdgcn_readfirstlane(bytes);
    for (uint32_t at = wave * 1024u; at < static_cast<uint32_t>(BN) * p.groups * 4u; at += 8192u)
      load_16_bytes_into_lds(desc, lds0 + L::kBaseScales, __builtin_amdgcn_readfirstlane(at), lane * 16, __builtin_amdgcn_readfirstlane(at));
  }

  // Weights: 128-byte pieces of BN rows (a K tile), four of them a stage; activations: 128-byte pieces of 16 rows, eight a
  // stage, one for each wavefront.  Rows are eight a load, the chunk of a lane permuted as in tile_gemm_kernel.
  const bool loads_x = wave < 4;
  const int loader = wave & 3;
  constexpr int kMostLoads = kLoadsX > L::kLoadsW ? kLoadsX : L::kLoadsW;
  uint32_t row_bytes[kMostLoads];
#pragma unroll
  for (int i = 0; i < kMostLoads; ++i) {
    const int tile_row = (i * 4 + loader) % (loads_x ? 2 : BN / 8) * 8 + (lane >> 3);
    const int chunk = ((lane & 7) ^ tile_row ^ (tile_row >> 3)) & 7;
    const int row = min(tile_row, (loads_x ? p.m : rows) - 1);   // rows past the extent: computed, never stored
    row_bytes[i] = static_cast<uint32_t>(row * (loads_x ? p.ldx * 2 : p.ldw) + chunk * 16);
  }
  // (the descriptors end with the operand's last row: the piece behind an odd multiple of 64 k reads zeros there)
  u32x4 desc_x = tile_buffer_words((const VECOPS_GLOBAL char*)p.x);
  u32x4 desc_w = tile_buffer_words((const VECOPS_GLOBAL char*)(p.w + static_cast<int64_t>(n0) * p.ldw));
  desc_x[2] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>((p.m - 1) * p.ldx * 2 + p.k * 2));
  desc_w[2] = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>((rows - 1) * p.ldw + p.k));
  auto load = [&](auto of_x, int i, int s, int slot) {
    constexpr bool X = decltype(of_x)::value;
    constexpr int BLOCKS = X ? 2 : BN / 8, PIECES = X ? 8 : 4, PIECE_K = X ? 64 : 128;
    const int block = i * 4 + loader, piece = s * PIECES + block / BLOCKS;
    u32x4 desc = X ? desc_x : desc_w;
    desc[2] = __builtin_amdgcn_readfirstlane(piece * PIECE_K < p.k ? desc[2] : 0u);
    load_16_bytes_into_lds(desc, __builtin_amdgcn_readfirstlane(lds0 + (X ? slot * kStageX : L::kBaseW + slot * L::kStageW)),
                           __builtin_amdgcn_readfirstlane(block * 1024), row_bytes[i],
                           __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(piece) * 128u));
  };

  const int row = lane & 15, chunk = ((lane >> 4) & 1) << 1 | (lane >> 5);  // (as in tile_gemm_kernel: no bank conflicts)
  uint32_t at_w[TILES], at_x[2];
#pragma unroll
  for (int t = 0; t < TILES; ++t)
    at_w[t] = lds0 + L::kBaseW + (wave >> 1) * BN * 128 + lds_chunk_offset(t * 16 + row, (wave & 1) * 4 + chunk);
#pragma unroll
  for (int h = 0; h < 2; ++h) at_x[h] = lds0 + wave * 2048 + lds_chunk_offset(row, 2 * chunk + h);
  typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
  typedef __attribute__((address_space(3))) float lds_float;
  f32x4 acc[TILES];
#pragma unroll
  for (int t = 0; t < TILES; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4 ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};  // eight bf16 1.0

  int slot_x = 0, slot_w = 0;
  auto step = [&](auto role, int s) {
    constexpr bool X = decltype(role)::value;
    constexpr int LOADS = X ? kLoadsX : L::kLoadsW, STAGES = X ? kStagesX : L::kStagesW;
    // this stage has landed (and, in front of the first, the scales), and every wavefront has left the one before it
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LOADS * (STAGES - 2)) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      load(role, i, s + STAGES - 1, X ? (slot_x == 0 ? STAGES - 1 : slot_x - 1) : (slot_w == 0 ? STAGES - 1 : slot_w - 1));
    const int k0 = s * kStageK + wave * 64;
    if (k0 < p.k) {
      const uint32_t stage_x = static_cast<uint32_t>(slot_x * kStageX), stage_w = static_cast<uint32_t>(slot_w * L::kStageW);
      u32x4 w[TILES];
#pragma unroll
      for (int t = 0; t < TILES; ++t) w[t] = *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_w[t] + stage_w));
      const bf16x8 b1 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_x[0] + stage_x)));
      const bf16x8 b2 = __builtin_bit_cast(bf16x8, *reinterpret_cast<const lds_u32x4*>(static_cast<uintptr_t>(at_x[1] + stage_x)));
      const int g = k0 >> group_shift;
      float scale[TILES][4];
#pragma unroll
      for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          scale[t][r] = *reinterpret_cast<const lds_float*>(
              static_cast<uintptr_t>(lds0 + L::kBaseScales + ((t * 16 + (lane >> 4) * 4 + r) * p.groups + g) * 4));
      // sum_k x * w = sum_k x * (w + 128) - 128 * sum_k x: the unsigned bytes convert exactly and cheaply
      f32x4 xs = {0.f, 0.f, 0.f, 0.f};
      xs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones), b1, xs, 0, 0, 0);
      xs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones), b2, xs, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < TILES; ++t) {
        uint32_t a[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint32_t wd = w[t][q] ^ 0x80808080u;
          const float f0 = static_cast<float>(wd & 0xffu), f1 = static_cast<float>((wd >> 8) & 0xffu);
          const float f2 = static_cast<float>((wd >> 16) & 0xffu), f3 = static_cast<float>(wd >> 24);
          // upper halves of two fp32 = two bf16 (exact: the values are integers below 256)
          a[2 * q] = __builtin_amdgcn_perm(__float_as_uint(f1), __float_as_uint(f0), 0x07060302u);
          a[2 * q + 1] = __builtin_amdgcn_perm(__float_as_uint(f3), __float_as_uint(f2), 0x07060302u);
        }
        const u32x4 a1 = {a[0], a[1], a[2], a[3]}, a2 = {a[4], a[5], a[6], a[7]};
        f32x4 dot = {0.f, 0.f, 0.f, 0.f};
        dot = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a1), b1, dot, 0, 0, 0);
        dot = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a2), b2, dot, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] = fmaf(scale[t][r], fmaf(-128.0f, xs[r], dot[r]), acc[t][r]);
      }
    }
    slot_x = slot_x + 1 == kStagesX ? 0 : slot_x + 1;
    slot_w = slot_w + 1 == L::kStagesW ? 0 : slot_w + 1;
  };
  auto walk = [&](auto role) {
    constexpr bool X = decltype(role)::value;
#pragma unroll
    for (int s = 0; s < (X ? kStagesX : L::kStagesW) - 1; ++s)
#pragma unroll
      for (int i = 0; i < (X ? kLoadsX : L::kLoadsW); ++i) load(role, i, s, s);
    for (int s = 0; s < stages; ++s) step(role, s);
  };
  if (loads_x) walk(std::true_type{});
  else walk(std::false_type{});

  // accumulator register r of lane l is output (weight row l / 16 * 4 + r, activation row l % 16) of its 16x16 tile
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t = 0; t < TILES; ++t) *reinterpret_cast<f32x4*>(sums + (wave * 16 + row) * BN + t * 16 + (lane >> 4) * 4) = acc[t];
  __syncthreads();
  for (int at = tid; at < 16 * BN; at += kThreads) {
    const int x_row = at / BN, n = at % BN;
    float total = sums[at];
#pragma unroll
    for (int w = 1; w < 8; ++w) total += sums[w * 16 * BN + at];
    if (x_row < p.m && n < rows) p.y[static_cast<int64_t>(x_row) * p.ldy + n0 + n] = static_cast<uint16_t>(bf16_bits_rne(total));
  }
}

template <int BN>
hipError_t launch(const SkinnyW8A16Params& p, hipStream_t stream) {
  auto kernel = w8a16_ring_kernel<BN>;
  static thread_local int configured_device = -1;
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  if (configured_device != device) {
    e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMostLds);
    if (e != hipSuccess) return e;
    configured_device = device;
  }
  // (the scales' last load of 1 KiB may end behind them)
  const int kLds = RingTile<BN>::kBaseScales + ((BN * p.groups * 4 + 1023) & ~1023);
  const int shift = p.group == 64 ? 6 : p.group == 128 ? 7 : 8;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((p.n + BN - 1) / BN)), dim3(kThreads), kLds, stream, p, shift);
  return hipGetLastError();
}

template <int BN>
bool scales_fit(const SkinnyW8A16Params& p) {
  return ((static_cast<int64_t>(BN) * p.groups * 4 + 1023) & ~int64_t{1023}) <= RingTile<BN>::kMostScales;
}

}  // namespace

bool launch_w8a16_ring_serves(const SkinnyW8A16Params& p, int bn) {
  if (p.group != 64 && p.group != 128 && p.group != 256) return false;
  if (p.m < 1 || p.m > 16 || p.n < 1 || p.k < 64 || p.ldx < 0 || p.ldw < 0) return false;
  // 32-bit byte offsets inside a workgroup's rows
  const int64_t most = (int64_t{1} << 31) - 1024;
  if (16 * p.ldx * 2 + p.k * 2 >= most || 64 * p.ldw + p.k >= most) return false;
  switch (bn) {
    case 16: return scales_fit<16>(p);
    case 32: return scales_fit<32>(p);
    case 48: return scales_fit<48>(p);
    case 64: return scales_fit<64>(p);
    default: return false;
  }
}

hipError_t launch_w8a16_ring(const SkinnyW8A16Params& p, int bn, hipStream_t stream) {
  switch (bn) {
    case 16: return launch<16>(p, stream);
    case 32: return launch<32>(p, stream);
    case 48: return launch<48>(p, stream);
    case 64: return launch<64>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace vecops_hip
