// Fast-mode prefill projection: INT16 activations x INT8 weight codes, the
// reference's INT16 panels (src/kernels/panels/panel_i16.rs), bitwise.
//
// 1. quantize_kernel: every 64-input group of every row becomes INT16 codes
//    q and a step (quantize_group, panel_i16.rs:233-266; pack_rows 275-329:
//    exception columns zeroed first, step times the row scale, exception
//    inputs x * row_scale kept in FP32). Each code is split exactly as
//    q = 256*h + (l + 128) with h, l in [-128, 127], and h and l are written
//    as two int8 planes in the lane order of the 16x16x64 i8 matrix-core
//    operand, so every wave load in the GEMM is one contiguous 1 KB chunk.
// 2. gemm_kernel: per 16x16 output block and group, two i8 MFMAs give the
//    group's exact INT32 sum: H = sum h*w; C = (H << 8) + 128*sum(w) (the last
//    term precomputed per column at upload); S = C + sum l*w. |S| < 2^31 as
//    in the reference (64 * 32767 * 127). Then, in the reference's order,
//    acc = fma(f32(S), fl(s_w * s_a), acc) over ascending groups, the
//    exception FMAs ascending, and the epilogue (Store, Glu, Add).
// Because the group sums are exact integers, any summation order inside the
// matrix core gives the same S, and every output matches kernel_scalar bit
// for bit.
//
// Each group's A and B tiles, activation steps, column sums and scales are
// copied HBM -> LDS by the LDS-DMA path into one of two stages while the
// previous group is computed from the other; tiles are ordered per XCD so
// that the workgroups sharing an L2 share operands.
//
// Roofline: the i8 matrix cores do 2 x 64 MACs per output and group, the
// FP32 group epilogue 4 VALU ops per output and group (shift-add and convert
// issue at half the FMA rate). Measured, neither bounds it alone: without the
// epilogue it runs about 25 % faster, without the products about 15 %; the
// operand copies (L2 -> LDS, about 1 GB per 6544 x 1024 x 4096 call) and the
// per-group barrier take the rest.
#include <type_traits>

#include "focr_internal.hpp"

namespace focr {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int kMPad = 128;  // rows padded to a multiple of this
constexpr int kBM = 64;     // rows per workgroup tile

// One wave per (16-row block, group): lane l owns row l%16, inputs
// 16*(l/16) .. +16 of the group; the group's absmax is a 4-lane reduction.
__global__ __launch_bounds__(256) void quantize_kernel(const float *__restrict__ x, int m, int k, int groups,
                                                       int row_blocks, const float *__restrict__ row_scale,
                                                       const int16_t *__restrict__ exc_index, int n_exc,
                                                       int8_t *__restrict__ a_tiles, float *__restrict__ steps,
                                                       float *__restrict__ exc_inputs, int m_pad) {
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (wave >= row_blocks * groups) return;
  const int g = wave / row_blocks, mb = wave % row_blocks;
  const int lane = threadIdx.x & 63;
  const int row = mb * 16 + (lane & 15);
  const int k0 = g * 64 + 16 * (lane >> 4);
  float v[16];
  const bool live = row < m;
  if (live) {
    const float4 *src = reinterpret_cast<const float4 *>(x + static_cast<size_t>(row) * k + k0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float4 f = src[i];
      v[4 * i] = f.x;
      v[4 * i + 1] = f.y;
      v[4 * i + 2] = f.z;
      v[4 * i + 3] = f.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = 0.0f;
  }
  const float scale = live ? (row_scale ? row_scale[row] : 1.0f) : 0.0f;
  // Exception columns: keep x * row_scale, quantize the group without them.
  if (exc_index) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int e = exc_index[k0 + i];
      if (e >= 0) {
        if (live) exc_inputs[static_cast<size_t>(row) * n_exc + e] = v[i] * scale;
        v[i] = 0.0f;
      }
    }
  }
  // absmax from bit patterns (NaN and infinity order above every finite value).
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t b = __float_as_uint(v[i]) & 0x7fffffffu;
    top = b > top ? b : top;
  }
  {
    uint32_t o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), 16));
    top = o > top ? o : top;
    o = static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), 32));
    top = o > top ? o : top;
  }
  int q[16];
  float step;
  const float qmax = 32767.0f;
  if (top >= 0x7f800000u) {
#pragma unroll
    for (int i = 0; i < 16; i++) q[i] = 0;
    step = __builtin_nanf("");
  } else {
    const float absmax = __uint_as_float(top);
    const float inv = __fdiv_rn(qmax, absmax);
    if (!__builtin_isfinite(inv)) {
      if (absmax == 0.0f) {
#pragma unroll
        for (int i = 0; i < 16; i++) q[i] = 0;
        step = 0.0f;
      } else {
        // The reciprocal overflows: an f64 path with the step rounded up
        // where its rounding would clip the maximum.
        step = __fdiv_rn(absmax, qmax);
        const float tiny = __uint_as_float(1u);
        step = step > tiny ? step : tiny;
        if (static_cast<double>(step) * 32767.0 < static_cast<double>(absmax))
          step = __uint_as_float(__float_as_uint(step) + 1u);
#pragma unroll
        for (int i = 0; i < 16; i++) {
          double r = __builtin_rint(__ddiv_rn(static_cast<double>(v[i]), static_cast<double>(step)));
          r = r < -32767.0 ? -32767.0 : (r > 32767.0 ? 32767.0 : r);
          q[i] = static_cast<int>(r);
        }
      }
    } else {
      const float magic = 12582912.0f;  // 1.5 * 2^23
#pragma unroll
      for (int i = 0; i < 16; i++) {
        float y = v[i] * inv;
        y = y < -qmax ? -qmax : (y > qmax ? qmax : y);
        q[i] = static_cast<int>(__float_as_uint(y + magic)) - static_cast<int>(__float_as_uint(magic));
      }
      step = __fdiv_rn(absmax, qmax);
    }
  }
  // q = 256 * h + (l + 128), h = q >> 8, l = (q & 255) - 128.
  uint32_t hi[4], lo[4];
#pragma unroll
  for (int w = 0; w < 4; w++) {
    uint32_t hw = 0, lw = 0;
#pragma unroll
    for (int b = 0; b < 4; b++) {
      const int c = q[4 * w + b];
      hw |= (static_cast<uint32_t>(c >> 8) & 0xffu) << (8 * b);
      lw |= (static_cast<uint32_t>((c & 0xff) - 128) & 0xffu) << (8 * b);
    }
    hi[w] = hw;
    lo[w] = lw;
  }
  int8_t *dst = a_tiles + (static_cast<size_t>(g) * row_blocks + mb) * 2048;
  reinterpret_cast<uint4 *>(dst)[lane] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  reinterpret_cast<uint4 *>(dst + 1024)[lane] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  if (lane < 16) steps[static_cast<size_t>(g) * m_pad + row] = step * scale;
}

// One group's operands of a 64 x BN tile in LDS, filled by the LDS-DMA path;
// two stages (the group being computed and the next one).
template <int BN>
struct GroupTile {
  uint4 a[kBM / 16 * 2 * 64];  // [4 row blocks][hi, lo][64 lanes] x 16 B
  uint4 b[BN / 16 * 64];       // [column blocks][64 lanes] x 16 B
  float steps[kBM];            // activation steps of the tile's rows
  int32_t wsum[BN];            // 128 * sum of the group's codes per column
  float sw[BN];                // weight scales per column
};

// One output: its exception FMAs (ascending columns), then the epilogue.
// Whole waves call it (Glu exchanges neighbouring columns between lanes).
template <int EPI>
__device__ __forceinline__ void emit(float v, int row, int col, int m, int n, const float *__restrict__ exc_inputs,
                                     const float *__restrict__ exc_vals, int n_exc, float *__restrict__ out) {
  const bool live = row < m && col < n;
  if (n_exc && live)
    for (int e = 0; e < n_exc; e++)
      v = fmaf_(exc_inputs[static_cast<size_t>(row) * n_exc + e], exc_vals[static_cast<size_t>(col) * n_exc + e], v);
  if constexpr (EPI == FOCR_EPI_GLU) {
    const float up = __shfl_xor(v, 1);
    if (live && (col & 1) == 0) out[static_cast<size_t>(row) * (n / 2) + col / 2] = squared_relu_glu(v, up);
  } else if constexpr (EPI == FOCR_EPI_ADD) {
    if (live) {
      float *dst = out + static_cast<size_t>(row) * n + col;
      *dst = *dst + v;
    }
  } else {
    if (live) out[static_cast<size_t>(row) * n + col] = v;
  }
}

// 64 x BN outputs per workgroup of BN / 16 waves; wave (wm, wn) holds 32
// rows x 32 columns, 2 row blocks x 2 column blocks of 16 x 16. A wider tile
// moves fewer operand bytes per output (the activation planes are copied once
// per BN columns, the weights once per 64 rows).
//
// Step g: wait for this wave's copies of group g, meet the other waves
// (nobody still reads the other stage), start group g + 1's copies into it,
// then compute group g: per block two i8 matrix-core products and the FP32
// epilogue acc = fma(f32(S), fl(s_w * s_a), acc). 128-column tiles hold 8
// waves; at most 80 VGPRs keep three such workgroups (6 waves per SIMD) on a
// compute unit.
template <int EPI, int BN>
__global__ __launch_bounds__(BN * 4) __attribute__((amdgpu_waves_per_eu(BN == 128 ? 6 : 1)))
void gemm_kernel(const int8_t *__restrict__ a_tiles, const float *__restrict__ steps,
                                                   const float *__restrict__ exc_inputs, const int8_t *__restrict__ b_tiles,
                                                   const int32_t *__restrict__ wsum, const float *__restrict__ sw,
                                                   const float *__restrict__ exc_vals, int n_exc, int m, int n,
                                                   int groups, int row_blocks, int m_pad, int row_tiles, int col_tiles,
                                                   float *__restrict__ out) {
  constexpr int RB = kBM / 16, RW = 2, WAVES = BN / 16, THREADS = 64 * WAVES;
  constexpr int ACP = RB * 2 * 64 / THREADS;  // A copies per thread and group
  typedef GroupTile<BN> Tile;
  // Two distinct LDS objects (not one array): the compiler then sees that
  // reads of one stage do not alias copies into the other.
  __shared__ Tile ring0, ring1;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / (BN / 32), wn = wave % (BN / 32);
  int rt, ct;
  xcd_tile(blockIdx.x, row_tiles, col_tiles, rt, ct);
  const int mb0 = rt * RB;
  const int nb0 = ct * (BN / 16);
  const int col_blocks = n / 16;

  // Sources of this thread's copies per group, each a uniform base (scalar
  // registers, advanced by a group's stride) plus a 32-bit lane offset so that
  // every copy takes the scalar-base address form: ACP x 16 B of the A planes;
  // 16 B of column block nb0 + wave of B (blocks past n repeat the last one:
  // computed and discarded); and, for waves 0 .. 2 BN / 64, 4 B of the steps
  // (wave 0), of the column sums or of the scales (64 columns per wave).
  const char *abase = reinterpret_cast<const char *>(a_tiles) + static_cast<size_t>(mb0) * 2048;
  const uint32_t aoff = 16u * tid;
  const size_t a_stride = static_cast<size_t>(row_blocks) * 2048;
  const char *bbase = reinterpret_cast<const char *>(b_tiles) + static_cast<size_t>(nb0) * 1024;
  int blk = nb0 + wave;
  blk = blk < col_blocks ? blk : col_blocks - 1;
  const uint32_t boff = static_cast<uint32_t>((blk - nb0) * 64 + lane) * 16u;
  const size_t b_stride = static_cast<size_t>(col_blocks) * 1024;
  constexpr int XP = BN / 64;  // 64-column pieces of the sums and of the scales
  const bool x_copy = wave <= 2 * XP;
  const char *xbase = reinterpret_cast<const char *>(steps + mb0 * 16);
  uint32_t xoff = 4u * lane;
  size_t x_stride = static_cast<size_t>(m_pad) * sizeof(float);
  int x_dst = static_cast<int>(offsetof(Tile, steps));  // byte offset of the wave's 256 B in the stage
  if (wave != 0 && x_copy) {
    const bool scales = wave > XP;
    const int piece = scales ? wave - 1 - XP : wave - 1;
    int col = nb0 * 16 + 64 * piece + lane;
    col = col < n ? col : n - 1;
    xbase = scales ? reinterpret_cast<const char *>(sw + nb0 * 16) : reinterpret_cast<const char *>(wsum + nb0 * 16);
    xoff = 4u * static_cast<uint32_t>(col - nb0 * 16);
    x_stride = static_cast<size_t>(n) * 4;
    x_dst = (scales ? static_cast<int>(offsetof(Tile, sw)) : static_cast<int>(offsetof(Tile, wsum))) + 256 * piece;
  }
  auto issue = [&](Tile &t, int g) {
    const char *ga = abase + static_cast<size_t>(g) * a_stride;
#pragma unroll
    for (int i = 0; i < ACP; i++)
      __builtin_amdgcn_global_load_lds((global_void *)((ga + 16 * THREADS * i) + aoff),
                                       (lds_void *)(&t.a[64 * wave + THREADS * i]), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((global_void *)(bbase + static_cast<size_t>(g) * b_stride + boff),
                                     (lds_void *)(&t.b[64 * wave]), 16, 0, 0);
    if (x_copy)
      __builtin_amdgcn_global_load_lds((global_void *)(xbase + static_cast<size_t>(g) * x_stride + xoff),
                                       (lds_void *)(reinterpret_cast<char *>(&t) + x_dst), 4, 0, 0);
  };

  float acc[RW][2][4];
#pragma unroll
  for (int i = 0; i < RW; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;

  const int quad = lane >> 4, col_in = lane & 15;
  auto step = [&](Tile &cur, Tile &next, int g) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): group g landed
    plain_barrier();
    // Past the last group the copy repeats it into the free stage.
    issue(next, g + 1 < groups ? g + 1 : groups - 1);
    v4i ahi[RW], alo[RW], b[2];
#pragma unroll
    for (int i = 0; i < RW; i++) {
      const int rb = wm * RW + i;
      const uint4 hv = cur.a[(rb * 2) * 64 + lane], lv = cur.a[(rb * 2 + 1) * 64 + lane];
      ahi[i] = v4i{static_cast<int>(hv.x), static_cast<int>(hv.y), static_cast<int>(hv.z), static_cast<int>(hv.w)};
      alo[i] = v4i{static_cast<int>(lv.x), static_cast<int>(lv.y), static_cast<int>(lv.z), static_cast<int>(lv.w)};
    }
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const uint4 w = cur.b[(wn * 2 + j) * 64 + lane];
      b[j] = v4i{static_cast<int>(w.x), static_cast<int>(w.y), static_cast<int>(w.z), static_cast<int>(w.w)};
    }
    int32_t ws[2];
    float swv[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int c = (wn * 2 + j) * 16 + col_in;
      ws[j] = cur.wsum[c];
      swv[j] = cur.sw[c];
    }
    float sa[RW][4];
#pragma unroll
    for (int i = 0; i < RW; i++) {
      const float4 sv = *reinterpret_cast<const float4 *>(&cur.steps[(wm * RW + i) * 16 + 4 * quad]);
      sa[i][0] = sv.x;
      sa[i][1] = sv.y;
      sa[i][2] = sv.z;
      sa[i][3] = sv.w;
    }
    const v4i zero = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < RW; i++)
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const v4i hsum = __builtin_amdgcn_mfma_i32_16x16x64_i8(ahi[i], b[j], zero, 0, 0, 0);
        v4i c;
#pragma unroll
        for (int r = 0; r < 4; r++) c[r] = (hsum[r] << 8) + ws[j];
        const v4i sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(alo[i], b[j], c, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float scale = swv[j] * sa[i][r];
          acc[i][j][r] = fmaf_(static_cast<float>(sum[r]), scale, acc[i][j][r]);
        }
      }
  };
  issue(ring0, 0);
  int g = 0;
  for (; g + 2 <= groups; g += 2) {
    step(ring0, ring1, g);
    step(ring1, ring0, g + 1);
  }
  if (g < groups) step(ring0, ring1, g);
  // The repeated copies must land before the workgroup's LDS is released.
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)

#pragma unroll
  for (int i = 0; i < RW; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        emit<EPI>(acc[i][j][r], (mb0 + wm * RW + i) * 16 + 4 * quad + r, (nb0 + wn * 2 + j) * 16 + col_in, m, n,
                  exc_inputs, exc_vals, n_exc, out);
}

// Small grids: RB x CB blocks of 16 x 16 outputs per wave, WAVES such waves
// side by side in a workgroup (columns), every operand loaded straight into
// registers D groups ahead (a block of a group is one contiguous 1 KB run in
// operand order), no LDS and no barrier. Per output the same integers and the
// same chain over ascending groups as gemm_kernel.
// Bound: latency. With few tiles gemm_kernel's workgroups wait for each
// group's copies behind one barrier per group (0.5 us a group); here a group
// costs a wave its two dependent products and the FP32 step.
template <int EPI, int RB, int CB, int WAVES, int D>
__global__ __launch_bounds__(64 * WAVES) void gemm_small_kernel(
    const int8_t *__restrict__ a_tiles, const float *__restrict__ steps, const float *__restrict__ exc_inputs,
    const int8_t *__restrict__ b_tiles, const int32_t *__restrict__ wsum, const float *__restrict__ sw,
    const float *__restrict__ exc_vals, int n_exc, int m, int n, int groups, int row_blocks, int m_pad, int row_tiles,
    int col_tiles, float *__restrict__ out) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int quad = lane >> 4, col_in = lane & 15;
  int rt, ct;
  xcd_tile(blockIdx.x, row_tiles, col_tiles, rt, ct);
  const int mb0 = rt * RB, nb0 = (ct * WAVES + wave) * CB, col_blocks = n / 16;
  if (nb0 >= col_blocks) return;
  struct Group {
    v4i hi[RB], lo[RB], b[CB];
    float4 sa[RB];
    int32_t ws[CB];
    float sw[CB];
  };
  auto load = [&](Group &f, int group) __attribute__((always_inline)) {
    const size_t g = group < groups ? group : groups - 1;
#pragma unroll
    for (int i = 0; i < RB; i++) {
      const int mb = mb0 + i < row_blocks ? mb0 + i : row_blocks - 1;
      const v4i *src = reinterpret_cast<const v4i *>(a_tiles + (g * row_blocks + mb) * 2048);
      f.hi[i] = src[lane];
      f.lo[i] = src[64 + lane];
      f.sa[i] = *reinterpret_cast<const float4 *>(steps + g * m_pad + mb * 16 + 4 * quad);
    }
#pragma unroll
    for (int j = 0; j < CB; j++) {
      const int nb = nb0 + j < col_blocks ? nb0 + j : col_blocks - 1;
      f.b[j] = reinterpret_cast<const v4i *>(b_tiles + (g * col_blocks + nb) * 1024)[lane];
      f.ws[j] = wsum[g * n + nb * 16 + col_in];
      f.sw[j] = sw[g * n + nb * 16 + col_in];
    }
  };
  float acc[RB][CB][4];
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < CB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) acc[i][j][r] = 0.0f;
  Group f[D];
#pragma unroll
  for (int d = 0; d < D; d++) load(f[d], d);
  for (int g = 0; g < groups; g += D) {
#pragma unroll
    for (int d = 0; d < D; d++) {
      if (g + d < groups) {
#pragma unroll
        for (int i = 0; i < RB; i++)
#pragma unroll
          for (int j = 0; j < CB; j++) {
            const v4i zero = {0, 0, 0, 0};
            const v4i hsum = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[d].hi[i], f[d].b[j], zero, 0, 0, 0);
            v4i c;
#pragma unroll
            for (int r = 0; r < 4; r++) c[r] = (hsum[r] << 8) + f[d].ws[j];
            const v4i sum = __builtin_amdgcn_mfma_i32_16x16x64_i8(f[d].lo[i], f[d].b[j], c, 0, 0, 0);
            const float sa[4] = {f[d].sa[i].x, f[d].sa[i].y, f[d].sa[i].z, f[d].sa[i].w};
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const float scale = f[d].sw[j] * sa[r];
              acc[i][j][r] = fmaf_(static_cast<float>(sum[r]), scale, acc[i][j][r]);
            }
          }
        load(f[d], g + d + D);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RB; i++)
#pragma unroll
    for (int j = 0; j < CB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        emit<EPI>(acc[i][j][r], (mb0 + i) * 16 + 4 * quad + r, (nb0 + j) * 16 + col_in, m, n, exc_inputs, exc_vals, n_exc,
                  out);
}

}  // namespace

int launch_prefill_i16(Ctx *ctx, const Linear *lin, const float *x, size_t rows, const float *row_scale,
                       int epilogue, float *out) {
  const size_t m = rows, k = lin->k, n = lin->n, groups = lin->groups;
  FOCR_REQUIRE(m < (size_t(1) << 30) && n % 32 == 0 && k % 64 == 0, FOCR_E_SHAPE, "INT16 panel shape");
  const size_t m_pad = (m + kMPad - 1) / kMPad * kMPad;
  const size_t row_blocks = m_pad / 16;
  const size_t a_bytes = m_pad * k * 2;
  const size_t s_bytes = groups * m_pad * sizeof(float);
  const size_t e_bytes = m_pad * (lin->n_exc ? lin->n_exc : 1) * sizeof(float);
  int rc = ensure_scratch(ctx, a_bytes + s_bytes + e_bytes + 256);
  if (rc != FOCR_OK) return rc;
  int8_t *a_tiles = static_cast<int8_t *>(ctx->scratch);
  float *steps = reinterpret_cast<float *>(static_cast<char *>(ctx->scratch) + a_bytes);
  float *exc_inputs = reinterpret_cast<float *>(static_cast<char *>(ctx->scratch) + a_bytes + s_bytes);

  const size_t waves = row_blocks * groups;
  hipLaunchKernelGGL(quantize_kernel, dim3(static_cast<unsigned>((waves + 3) / 4)), dim3(256), 0, ctx->stream, x,
                     static_cast<int>(m), static_cast<int>(k), static_cast<int>(groups), static_cast<int>(row_blocks),
                     row_scale, lin->exc_index, static_cast<int>(lin->n_exc), a_tiles, steps, exc_inputs,
                     static_cast<int>(m_pad));
  FOCR_HIP_CHECK(hipGetLastError());
  // By 16 x 16 blocks of output, against the chip's 1,024 SIMDs (us, this form
  // and its neighbours, quantizer not counted): 432 (WO, m = 144) 16 x 16 per wave
  // 4.5, 16 x 32 5.8, gemm_kernel 10; 864 (W13, 48) 4.4, 5.0; 2,592 (W13, 144)
  // 16 x 32 7.1, 16 x 16 8.4, 32 x 32 8.4, gemm_kernel 9.7; 3,024 (W2, 1,000) 14.5,
  // 18.5, 18.2, 20. Larger grids share operands in LDS (gemm_kernel): from 4,000
  // blocks on where its tiles are 64 columns wide (us per call, 32 x 32 here and
  // gemm_kernel: W2, 1,664 rows 28.1 and 28.4, 2,432 32.7 and 29.6; k = 8,192, 2,432
  // rows 102 and 84); where they are 128 wide, from 5,500 on (W13, 320 rows 13.6 and
  // 13.9, 384 14.7 and 13.3; a k below 768 from 4,000 on: 256 -> 3,072, 304 rows 7 %
  // slower here), but not before 7,400 where its grid, padded to 128 rows, starts a
  // second round of one workgroup per compute unit (W13, 400 rows 14.9 and 16.1).
  const size_t blocks = (m + 15) / 16 * (n / 16);
  const bool wide = n >= 2048;  // gemm_kernel's tiles are 128 columns wide
  const size_t wide_tiles = m_pad / kBM * ((n + 127) / 128);
  if (blocks <= 4000 || (wide && ((blocks <= 5500 && k >= 768) || (blocks <= 7400 && wide_tiles > 256)))) {
    auto launch = [&](auto epi, auto rb, auto cb, auto wv, auto depth) {
      constexpr int E = decltype(epi)::value, RB = decltype(rb)::value, CB = decltype(cb)::value;
      constexpr int WV = decltype(wv)::value, D = decltype(depth)::value;
      const int rt = static_cast<int>((m + 16 * RB - 1) / (16 * RB));
      const int ct = static_cast<int>((n / 16 + CB * WV - 1) / (CB * WV));
      hipLaunchKernelGGL((gemm_small_kernel<E, RB, CB, WV, D>), dim3(static_cast<unsigned>(rt * ct)), dim3(64 * WV), 0,
                         ctx->stream, a_tiles, steps, exc_inputs, lin->i16_b, lin->i16_wsum, lin->i16_sw, lin->exc_vals,
                         static_cast<int>(lin->n_exc), static_cast<int>(m), static_cast<int>(n),
                         static_cast<int>(groups), static_cast<int>(row_blocks), static_cast<int>(m_pad), rt, ct, out);
    };
    using std::integral_constant;
    auto pick = [&](auto epi) {
      if (blocks <= 1000)
        launch(epi, integral_constant<int, 1>(), integral_constant<int, 1>(), integral_constant<int, 1>(),
               integral_constant<int, 4>());
      else if (blocks <= 4000)
        launch(epi, integral_constant<int, 1>(), integral_constant<int, 2>(), integral_constant<int, 2>(),
               integral_constant<int, 3>());
      else
        launch(epi, integral_constant<int, 2>(), integral_constant<int, 2>(), integral_constant<int, 2>(),
               integral_constant<int, 3>());
    };
    if (epilogue == FOCR_EPI_GLU)
      pick(integral_constant<int, FOCR_EPI_GLU>());
    else if (epilogue == FOCR_EPI_ADD)
      pick(integral_constant<int, FOCR_EPI_ADD>());
    else
      pick(integral_constant<int, FOCR_EPI_STORE>());
    FOCR_HIP_CHECK(hipGetLastError());
    return FOCR_OK;
  }
  // 128-column tiles where n gives at least 16 of them (fewer operand bytes
  // per output: +5 % on 1024 -> 4096), 64-column ones for narrow outputs
  // (n = 768: the wider tiles leave too few workgroups).
  const int row_tiles = static_cast<int>(m_pad / kBM);
#define FOCR_LAUNCH_I16(E, BN)                                                                                    \
  hipLaunchKernelGGL((gemm_kernel<E, BN>), dim3(static_cast<unsigned>(row_tiles * ((n + BN - 1) / BN))), dim3(BN * 4), \
                     0, ctx->stream, a_tiles, steps, exc_inputs, lin->i16_b, lin->i16_wsum, lin->i16_sw,             \
                     lin->exc_vals, static_cast<int>(lin->n_exc), static_cast<int>(m), static_cast<int>(n),          \
                     static_cast<int>(groups), static_cast<int>(row_blocks), static_cast<int>(m_pad), row_tiles,     \
                     static_cast<int>((n + BN - 1) / BN), out)
  if (epilogue == FOCR_EPI_GLU) {
    if (wide) FOCR_LAUNCH_I16(FOCR_EPI_GLU, 128); else FOCR_LAUNCH_I16(FOCR_EPI_GLU, 64);
  } else if (epilogue == FOCR_EPI_ADD) {
    if (wide) FOCR_LAUNCH_I16(FOCR_EPI_ADD, 128); else FOCR_LAUNCH_I16(FOCR_EPI_ADD, 64);
  } else {
    if (wide) FOCR_LAUNCH_I16(FOCR_EPI_STORE, 128); else FOCR_LAUNCH_I16(FOCR_EPI_STORE, 64);
  }
#undef FOCR_LAUNCH_I16
  FOCR_HIP_CHECK(hipGetLastError());
  return FOCR_OK;
}

}  // namespace focr
