// The exact-order FP32 prefill GEMM on the FP32 matrix cores: every output is
// one FMA chain over ascending k from +0.0, bitwise the reference's FP32
// panels (src/kernels/panels/panel.rs:154-172).
//
// v_mfma_f32_16x16x4f32 adds its four products to the accumulator one after
// the other in ascending k, each as one fused multiply-add rounded to nearest
// even with subnormals kept: checked bit for bit against fmaf over normal,
// 2^+-30, subnormal, cancelling, infinite and NaN operands, and by the tests
// against the oracle. A chain of them over k = 0, 4, 8, ... is therefore the
// panels' chain itself.
#include <type_traits>
#include <utility>

#include "gemm_f32.hpp"

namespace focr {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

template <typename F, int... U>
__device__ __forceinline__ void steps(F &&f, std::integer_sequence<int, U...>) {
  (f(std::integral_constant<int, U>()), ...);
}

// (16 I WGM) x (16 J WGN) outputs per workgroup, WGM x WGN waves of I x J
// blocks of 16 x 16. Stages of KS k go HBM -> LDS by the LDS-DMA path into a
// ring of R slots (separate arrays, so that the compiler sees a step's reads
// never touch the slot being copied into), R - 1 stages ahead: A rows and W
// rows (FP32, or codes as they are) in 16-byte chunks ordered
// [16-row block][chunk of the row][row], so the 64 lanes of a fragment read
// (16 rows x 4 consecutive k) cover one contiguous run, and the stage's scale
// of each column. The row scale and fl(code * scale) are applied to the
// fragments as they are read. Rows past m and columns past n repeat the last
// one in bounds; their outputs are not written.
//
// Bound: the FP32 matrix cores (154 TFLOP/s measured from registers alone;
// 15.8 ns per 16 x 16 x 4 step of a lone dependent chain, 13.6 with two or
// more chains on a SIMD), to which the VALU work of forming the operands adds
// (FP32 matrix and vector instructions do not overlap here). A 16 x 16 block
// takes 8 matrix-core cycles per k, so small calls are bound by one block's
// chain and want one block per wave; large ones want more blocks per wave,
// which share the operand reads. INT16 codes, m = 144 / 1,501 / 6,544, us per
// call, SIMT chain tiles before -> this kernel: QKV 53 -> 15 / 78 -> 53 /
// 331 -> 229; WO 69 -> 10 / 73 -> 38 / 182 -> 115; W13 55 -> 22 / 174 -> 121 /
// 667 -> 484; W2 151 -> 21 / 161 -> 79 / 398 -> 239 (96 TFLOP/s). Tried
// without gain: fragments of the next stage read before the current products
// (a second register set), [row][chunk] order with 128-byte row segments,
// group-major scales, rings of six.
template <typename T, int EPI, bool SCALED, int WGM, int WGN, int I, int J, int KS, int R>
__global__ __launch_bounds__(64 * WGM *WGN) void chain_mfma_kernel(GemmArgs a, int row_tiles, int col_tiles) {
  constexpr bool kCodes = !std::is_same<T, float>::value;
  constexpr int W = WGM * WGN, BM = 16 * I * WGM, BN = 16 * J * WGN;
  constexpr int B = static_cast<int>(sizeof(T)), E = 16 / B;     // W values per 16-byte chunk
  constexpr int ABYTES = BM * KS * 4, BBYTES = BN * KS * B, SBYTES = kCodes ? 256 * W : 0;
  constexpr int NA = ABYTES / 1024, NB = BBYTES / 1024, PER = (NA + NB + W - 1) / W;  // copies of 1 KB
  constexpr int COPIES = PER + (kCodes ? 1 : 0);                 // per wave and stage
  constexpr int SLOT = ABYTES + BBYTES + SBYTES;
  static_assert(ABYTES % 1024 == 0 && BBYTES % 1024 == 0 && 16 * J <= 64, "whole copies");
  static_assert(R == 3 || R == 4, "ring slots");
  __shared__ __attribute__((aligned(1024))) char ring0[SLOT], ring1[SLOT], ring2[SLOT], ring3[R > 3 ? SLOT : 16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int l16 = lane & 15, g = lane >> 4;
  int rt, ct;
  xcd_tile(blockIdx.x, row_tiles, col_tiles, rt, ct);
  const int m0 = rt * BM, n0 = ct * BN;

  // Copy i of this wave is number wave + W i of the stage (the last one again
  // where there are fewer): 16-byte chunks 64 number + lane of A or W. Every
  // copy is a uniform base (the tile's first row at the stage's first k) plus
  // a 32-bit lane offset, so a copy costs no vector instruction but itself.
  const char *const abase = reinterpret_cast<const char *>(a.x + static_cast<size_t>(m0) * a.k);
  const char *const bbase =
      reinterpret_cast<const char *>(static_cast<const T *>(a.codes) + static_cast<size_t>(n0) * a.k);
  uint32_t off[PER];
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int number = wave + W * i < NA + NB ? wave + W * i : NA + NB - 1;
    if (number < NA) {
      const int q = 64 * number + lane;
      const int row = 16 * (q / (4 * KS)) + q % 16;
      off[i] = static_cast<uint32_t>(m0 + row < a.m ? row : a.m - 1 - m0) * a.k * 4 + 16 * ((q / 16) % (KS / 4));
    } else {
      const int q = 64 * (number - NA) + lane;
      const int col = 16 * (q / (16 * KS / E)) + q % 16;
      off[i] = static_cast<uint32_t>(n0 + col < a.n ? col : a.n - 1 - n0) * a.k * B + 16 * ((q / 16) % (KS / E));
    }
  }
  // This wave's columns' scales (lane = column), in its own 256 bytes.
  uint32_t soff = 0;
  int group_shift = 0;  // stages per scale group, as a power of two
  if constexpr (kCodes) {
    const int c = wn * 16 * J + lane % (16 * J);
    soff = static_cast<uint32_t>(n0 + c < a.n ? c : a.n - 1 - n0) * a.groups * 4;
    group_shift = __builtin_ctz(a.group / KS);
  }
  auto issue = [&](char *slot, int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < PER; i++) {
      const int number = wave + W * i < NA + NB ? wave + W * i : NA + NB - 1;
      const char *base = number < NA ? abase + static_cast<size_t>(stage) * (KS * 4)
                                     : bbase + static_cast<size_t>(stage) * (KS * B);
      __builtin_amdgcn_global_load_lds((global_void *)(base + off[i]), (lds_void *)(slot + 1024 * number), 16, 0, 0);
    }
    if constexpr (kCodes) {
      const char *base =
          reinterpret_cast<const char *>(a.scales + static_cast<size_t>(n0) * a.groups + (stage >> group_shift));
      __builtin_amdgcn_global_load_lds((global_void *)(base + soff),
                                       (lds_void *)(slot + ABYTES + BBYTES + 256 * wave), 4, 0, 0);
    }
  };

  float rs[I];
  if constexpr (SCALED) {
#pragma unroll
    for (int i = 0; i < I; i++) {
      const int row = m0 + 16 * (wm * I + i) + l16;
      rs[i] = a.row_scale[row < a.m ? row : a.m - 1];
    }
  }
  v4f acc[I][J];
#pragma unroll
  for (int i = 0; i < I; i++)
#pragma unroll
    for (int j = 0; j < J; j++) acc[i][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  // Lane group g supplies k = 4 t + g of step t.
  auto compute = [&](const char *slot) __attribute__((always_inline)) {
    float sc[J];
    if constexpr (kCodes) {
#pragma unroll
      for (int j = 0; j < J; j++)
        sc[j] = *reinterpret_cast<const float *>(slot + ABYTES + BBYTES + 256 * wave + 4 * (16 * j + l16));
    }
#pragma unroll
    for (int t = 0; t < KS / 4; t++) {
      float av[I], bv[J];
#pragma unroll
      for (int i = 0; i < I; i++) {
        av[i] = *reinterpret_cast<const float *>(slot + (((wm * I + i) * (KS / 4) + t) * 16 + l16) * 16 + 4 * g);
        if constexpr (SCALED) av[i] = av[i] * rs[i];
      }
#pragma unroll
      for (int j = 0; j < J; j++) {
        const T w = *reinterpret_cast<const T *>(slot + ABYTES + (((wn * J + j) * (KS / E) + 4 * t / E) * 16 + l16) * 16 +
                                                 (4 * t % E + g) * B);
        if constexpr (kCodes)
          bv[j] = static_cast<float>(static_cast<int32_t>(w)) * sc[j];
        else
          bv[j] = w;
      }
#pragma unroll
      for (int i = 0; i < I; i++)
#pragma unroll
        for (int j = 0; j < J; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
  };

  // Stage st sits in slot st % R. Step st: wait for this wave's copies of
  // stage st (those of the R - 2 stages after it may still fly) and its reads
  // of the slot before, meet the other waves, start stage st + R - 1 in that
  // slot (past the last stage the copy repeats it, so the counts stay the
  // same), then run stage st.
  const int stages = a.k / KS;
  char *const slots[4] = {ring0, ring1, ring2, ring3};
  auto run = [&](int st, auto uc) __attribute__((always_inline)) {
    constexpr int u = decltype(uc)::value;
    __builtin_amdgcn_s_waitcnt(wait_vm_lgkm0((R - 2) * COPIES));
    plain_barrier();
    issue(slots[(u + R - 1) % R], st + R - 1 < stages ? st + R - 1 : stages - 1);
    compute(slots[u]);
  };
#pragma unroll
  for (int u = 0; u < R - 1; u++) issue(slots[u], u < stages ? u : stages - 1);
  int st = 0;
  for (; st + R <= stages; st += R)
    steps([&](auto uc) __attribute__((always_inline)) { run(st + decltype(uc)::value, uc); },
          std::make_integer_sequence<int, R>());
  steps([&](auto uc) __attribute__((always_inline)) {
          if (st + decltype(uc)::value < stages) run(st + decltype(uc)::value, uc);
        },
        std::make_integer_sequence<int, R - 1>());
  // The repeated copies must land before the workgroup's LDS is released.
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)

  // D layout of 16x16: column = lane % 16, row = 4 (lane / 16) + r.
#pragma unroll
  for (int i = 0; i < I; i++)
#pragma unroll
    for (int j = 0; j < J; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const float v = acc[i][j][r];
        const float partner = EPI == FOCR_EPI_GLU ? __shfl_xor(v, 1) : 0.0f;
        emit<EPI>(a, m0 + 16 * (wm * I + i) + 4 * g + r, n0 + 16 * (wn * J + j) + l16, v, partner);
      }
}

template <typename T, int EPI, int WGM, int WGN, int I, int J, int KS, int R>
void launch_tile(const GemmArgs &a, hipStream_t stream) {
  const int rt = (a.m + 16 * I * WGM - 1) / (16 * I * WGM), ct = (a.n + 16 * J * WGN - 1) / (16 * J * WGN);
  const dim3 grid(static_cast<unsigned>(rt * ct)), block(64 * WGM * WGN);
  if (a.row_scale)
    hipLaunchKernelGGL((chain_mfma_kernel<T, EPI, true, WGM, WGN, I, J, KS, R>), grid, block, 0, stream, a, rt, ct);
  else
    hipLaunchKernelGGL((chain_mfma_kernel<T, EPI, false, WGM, WGN, I, J, KS, R>), grid, block, 0, stream, a, rt, ct);
}

// The tile by the number of 16 x 16 output blocks, against the chip's 1,024
// SIMDs: up to about one block each, one block per wave in the smallest
// workgroups; then wider workgroups, then two and four blocks per wave, then
// eight. Measured neighbours at the lines (INT16 codes, us): 1,200 blocks (WO,
// m = 400) 16 x 32 18.8, 16 x 64 19.4; 2,592 (W13, 144) 16 x 64 21.7, 32 x 64
// 23.2; 3,200 (QKV, 400) 32 x 64 22.8, 64 x 64 24.2; 4,512 (WO, 1,501) 32 x 64
// 37.8, 64 x 64 44.6; 8,064 (QKV, 1,000) 64 x 64 38.0, 32 x 64 43.5; 27,072
// (W13, 1,501) 64 x 64 121, 64 x 128 132; 45,216 (W13, 2,500) 64 x 128 195,
// 64 x 64 202. FP32 weights of k = 64, one or two stages, go on to the next form
// earlier: 150 x 64 -> 4,096 (2,560 blocks) 16 x 64 8.8, 32 x 64 6.6; 300 rows
// (4,864) 32 x 64 9.5, 64 x 64 6.5.
template <typename T, int EPI>
void launch_epilogue(const GemmArgs &a, hipStream_t stream) {
  const long blocks = static_cast<long>((a.m + 15) / 16) * ((a.n + 15) / 16);
  const bool brief = std::is_same<T, float>::value && a.k == 64;
  if (blocks <= 1280)
    launch_tile<T, EPI, 1, 2, 1, 1, 64, 4>(a, stream);
  else if (blocks <= (brief ? 2000 : 3100))
    launch_tile<T, EPI, 1, 4, 1, 1, 64, 4>(a, stream);
  else if (blocks <= (brief ? 4000 : 5500))
    launch_tile<T, EPI, 2, 2, 1, 2, 64, 3>(a, stream);
  else if (blocks <= 36000)
    launch_tile<T, EPI, 2, 2, 2, 2, 32, 3>(a, stream);
  else
    launch_tile<T, EPI, 2, 2, 2, 4, 32, 3>(a, stream);
}

template <typename T>
void launch_type(const GemmArgs &a, int epilogue, hipStream_t stream) {
  if (epilogue == FOCR_EPI_GLU)
    launch_epilogue<T, FOCR_EPI_GLU>(a, stream);
  else if (epilogue == FOCR_EPI_ADD)
    launch_epilogue<T, FOCR_EPI_ADD>(a, stream);
  else
    launch_epilogue<T, FOCR_EPI_STORE>(a, stream);
}

}  // namespace

// Whole 64-wide k stages (one scale group per stage for codes), 16-byte
// aligned rows, no exception columns (their values would have to replace the
// codes in k order), 32-bit offsets within a tile, and a grid whose tile
// count an int holds. FP32 weights of k = 64 past 12,500 blocks keep chain2's
// tiles, which do not repeat a ring of copies for two stages of work (us per
// call, here and there: 6,544 x 64 -> 4,096 67 and 56, 992 x 64 -> 2,048 7.0 and
// 9.2; at k = 128 39 and 44 for 2,400 rows; codes are faster here at any k).
bool launch_chain_mfma(const GemmArgs &a, int bits, int epilogue, hipStream_t stream) {
  const bool aligned = (reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.codes)) % 16 == 0;
  if (!aligned || a.k % 64 != 0 || a.k > (1 << 20) || a.n_exc != 0 || (bits != 32 && a.group % 64 != 0)) return false;
  const long blocks = static_cast<long>((a.m + 15) / 16) * ((a.n + 15) / 16);
  if (blocks >= (long(1) << 31) || (bits == 32 && a.k == 64 && blocks > 12500)) return false;
  if (bits == 8)
    launch_type<int8_t>(a, epilogue, stream);
  else if (bits == 16)
    launch_type<int16_t>(a, epilogue, stream);
  else
    launch_type<float>(a, epilogue, stream);
  return true;
}

}  // namespace focr
