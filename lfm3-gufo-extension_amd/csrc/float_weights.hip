// Float weights (BF16, F16, F32) with exact products on gfx950: the
// numerical reference precision of the model (BF16, README.md:24-27) and
// the other float formats the reference binds (weights.cpp:30-37): the
// projections of gpu::Dense / gpu::LaunchGEMV for such tensors
// (hip/ops.hip:876-890 F16Dense, 1799-1825, 1917-2005, 2243-2244) and the
// embedding gather (hip/ops.hip:858-875).
//
// Weights are repacked at load into tiles of 16 rows x 32 columns: lane
// L = 16 g + n of a wave holds row n's columns 8g..8g+7 (16 bytes for the
// 16-bit formats, 1 KB a tile; two 16-byte planes for F32, columns
// 8g..8g+3 in the first 1 KB and 8g+4..8g+7 in the second). Tiles are
// stored [row tile][column block], rows padded to 16 and columns to 32
// with zeros.
//
// Every product runs on v_mfma_f32_16x16x32_bf16 with exact BF16 x BF16
// products. The FP32 inputs split exactly into three BF16 parts,
// x = hi + mid + lo (hi = x truncated to BF16, mid = (x - hi) truncated,
// lo = the rest, which has at most 8 significant bits). A BF16 weight is
// one part; an F16 weight (11 significant bits) is hi + lo with lo of at
// most 3 bits; an F32 weight splits like the inputs. So the 3 x (1, 2 or
// 3) MFMAs per 32-column block give the exact products of the weights
// with the FP32 inputs; only the FP32 accumulation order differs from a
// scalar loop. Two kernels take these products. FloatGemvKernel (decode
// rows, and prompt rows of few blocks; up to 16 tokens a block): RT row tiles
// a block and, per wave, a contiguous range of column blocks; the waves' sums
// meet in LDS and add in wave order. FloatGemmKernel (prompt rows): a block
// owns 64 tokens (32 in the smallest shape) and splits their inputs once for
// all of its weight rows.
#include <cmath>
#include <cstring>
#include <utility>

#include "common.hpp"
#include "internal.hpp"

namespace lfm3amd {
namespace {

constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kTileCols = 32, kTileElems = 16 * kTileCols;

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

std::uint32_t ColBlocks(std::uint32_t cols) { return (cols + kTileCols - 1) / kTileCols; }
std::uint32_t RowTilesOf(std::uint32_t rows) { return (rows + 15) / 16; }

// x = hi + mid + lo exactly; returns the three BF16 bit patterns.
__device__ __forceinline__ void Split3(float x, unsigned& hi, unsigned& mid, unsigned& lo) {
  const unsigned b = __float_as_uint(x);
  const float r = x - __uint_as_float(b & 0xffff0000u);
  const unsigned rb = __float_as_uint(r);
  const float l = r - __uint_as_float(rb & 0xffff0000u);
  hi = b >> 16;
  mid = rb >> 16;
  lo = __float_as_uint(l) >> 16;
}

__device__ __forceinline__ f32x4 Mfma(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The A operands of one lane: 8 consecutive inputs of its token, split.
__device__ __forceinline__ void Operands(float4 p, float4 q, uint4& hi, uint4& mid, uint4& lo) {
  const float v[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
  unsigned h[8], m[8], l[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    Split3(v[i], h[i], m[i], l[i]);
  hi = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
  mid = make_uint4(m[0] | m[1] << 16, m[2] | m[3] << 16, m[4] | m[5] << 16, m[6] | m[7] << 16);
  lo = make_uint4(l[0] | l[1] << 16, l[2] | l[3] << 16, l[4] | l[5] << 16, l[6] | l[7] << 16);
}

// Weight formats (GGML type ids) and their tile geometry.
constexpr int kF32 = LFM3_TYPE_F32, kF16 = LFM3_TYPE_F16, kBf16 = LFM3_TYPE_BF16;
constexpr int WordsOf(int wf) { return wf == kF32 ? 2 : 1; }       // 16-byte words a lane
constexpr int PartsOf(int wf) { return wf == kBf16 ? 1 : wf == kF16 ? 2 : 3; }  // BF16 parts
constexpr int ElemBytes(int wf) { return wf == kF32 ? 4 : 2; }

// Eight weights of a lane (its tile words) -> their exact BF16 parts.
template<int WF>
__device__ __forceinline__ void WeightParts(const uint4 (&w)[WordsOf(WF)],
                                            uint4 (&part)[PartsOf(WF)]) {
  if constexpr (WF == kBf16) {
    part[0] = w[0];
  } else if constexpr (WF == kF16) {
    // v = f16 exactly in FP32; hi keeps its top 8 significant bits, and
    // lo = v - hi (at most 3 significant bits) is exact in BF16.
    const unsigned in[4] = {w[0].x, w[0].y, w[0].z, w[0].w};
    unsigned hi[4], lo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float v0 = HalfBitsToFloat(in[i] & 0xffffu), v1 = HalfBitsToFloat(in[i] >> 16);
      const unsigned b0 = __float_as_uint(v0) & 0xffff0000u, b1 = __float_as_uint(v1) & 0xffff0000u;
      const unsigned l0 = __float_as_uint(v0 - __uint_as_float(b0)) >> 16;
      const unsigned l1 = __float_as_uint(v1 - __uint_as_float(b1)) >> 16;
      hi[i] = (b0 >> 16) | b1;
      lo[i] = l0 | (l1 << 16);
    }
    part[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    part[1] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  } else {
    const float4 p = __builtin_bit_cast(float4, w[0]), q = __builtin_bit_cast(float4, w[1]);
    Operands(p, q, part[0], part[1], part[2]);
  }
}

// y[p][t][r] for tokens t of blockIdx.y's group of 16, row tiles
// [blockIdx.x * RT, + RT) and K part p = blockIdx.z (column blocks
// [p * nkb / parts, (p + 1) * nkb / parts)). With kSwiGLU the row tiles
// come in gate/up pairs (tile 2j gate, 2j + 1 up of output tile j) and
// y = silu(gate) * up, as the reference's SwiGLU (g / (1 + exp(-g))) * u.
template<int RT, bool kSwiGLU, int WF>
__launch_bounds__(kThreads) __global__
    void FloatGemvKernel(const uint4* __restrict__ tiles, int row_tiles, int nkb,
                        const float* __restrict__ x, int ldx, int batch, float* __restrict__ y,
                        int ldy, int out_rows, int parts, std::size_t part_stride) {
  __shared__ f32x4 s_red[kWaves][RT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = lane >> 4, m = lane & 15;
  const int tile0 = blockIdx.x * RT;
  const int token = blockIdx.y * 16 + m;
  const bool live = token < batch;
  const int part = blockIdx.z;
  const int p0 = part * nkb / parts, p1 = (part + 1) * nkb / parts;
  const int kb0 = p0 + wave * (p1 - p0) / kWaves, kb1 = p0 + (wave + 1) * (p1 - p0) / kWaves;
  const float* xr = x + std::size_t(live ? token : 0) * ldx + 8 * g;
  constexpr int NW = WordsOf(WF), NP = PartsOf(WF);
  // Tiles past the last one read the last one (unconditional 16-byte
  // loads); their rows are past out_rows, so their sums are never stored.
  const uint4* wt[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    wt[r] = tiles + (std::size_t(min(tile0 + r, row_tiles - 1)) * nkb) * 64 * NW + lane;

  f32x4 acc[3][RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    acc[0][r] = acc[1][r] = acc[2][r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const float4 zerof = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  // One block ahead: the next weights and inputs load while this block's
  // MFMAs run.
  uint4 wn[RT][NW];
  const auto load_w = [&](int kb, uint4 (&dst)[RT][NW]) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < NW; ++q)
        dst[r][q] = wt[r][std::size_t(kb) * 64 * NW + 64 * q];
  };
  float4 xa = zerof, xb = zerof;
  if (kb0 < kb1) {
    load_w(kb0, wn);
    if (live) {
      xa = *reinterpret_cast<const float4*>(xr + kb0 * kTileCols);
      xb = *reinterpret_cast<const float4*>(xr + kb0 * kTileCols + 4);
    }
  }
  for (int kb = kb0; kb < kb1; ++kb) {
    uint4 wc[RT][NW];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < NW; ++q)
        wc[r][q] = wn[r][q];
    const float4 ca = xa, cb = xb;
    if (kb + 1 < kb1) {
      load_w(kb + 1, wn);
      if (live) {
        xa = *reinterpret_cast<const float4*>(xr + (kb + 1) * kTileCols);
        xb = *reinterpret_cast<const float4*>(xr + (kb + 1) * kTileCols + 4);
      }
    }
    uint4 hi, mid, lo;
    Operands(ca, cb, hi, mid, lo);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      uint4 wp[NP];
      WeightParts<WF>(wc[r], wp);
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        acc[0][r] = Mfma(hi, wp[j], acc[0][r]);
        acc[1][r] = Mfma(mid, wp[j], acc[1][r]);
        acc[2][r] = Mfma(lo, wp[j], acc[2][r]);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
    s_red[wave][r][lane] = (acc[0][r] + acc[1][r]) + acc[2][r];
  __syncthreads();

  // Lane l of a tile holds tokens 4 (l >> 4) + i, weight row l & 15.
  float* yp = y + std::size_t(part) * part_stride;
  constexpr int kOut = kSwiGLU ? RT / 2 : RT;
  for (int e = threadIdx.x; e < kOut * 64; e += kThreads) {
    const int r = e >> 6, l = e & 63;
    const int t0 = blockIdx.y * 16 + 4 * (l >> 4);
    if (kSwiGLU) {
      f32x4 gs = s_red[0][2 * r][l], us = s_red[0][2 * r + 1][l];
      for (int v = 1; v < kWaves; ++v) {
        gs += s_red[v][2 * r][l];
        us += s_red[v][2 * r + 1][l];
      }
      const int row = ((tile0 >> 1) + r) * 16 + (l & 15);
      if (row >= out_rows)
        continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (t0 + i < batch)
          yp[std::size_t(t0 + i) * ldy + row] = (gs[i] / (1.0f + expf(-gs[i]))) * us[i];
    } else {
      f32x4 s = s_red[0][r][l];
      for (int v = 1; v < kWaves; ++v)
        s += s_red[v][r][l];
      const int row = (tile0 + r) * 16 + (l & 15);
      if (row >= out_rows)
        continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (t0 + i < batch)
          yp[std::size_t(t0 + i) * ldy + row] = s[i];
    }
  }
}

// f(0), f(1), .., f(N - 1) with constant indices.
template<int N, class F>
__device__ __forceinline__ void Unroll(F f) {
  [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) {
    (f(std::integral_constant<int, I>{}), ...);
  }(std::make_integer_sequence<int, N>{});
}

// y[p][t][r] for 16 TT tokens and 16 RT (8 / KG) weight rows a block, one K
// part p of `parts`: the prompt rows' products (64 tokens; 32 when there are
// no more).
//
// What bounds it: a decode-shaped block (16 tokens) reads every weight once
// per 16 tokens and splits every input once per 16 RT rows, which left the
// 512-token BF16 gate/up product (2 x 7680 x 2048) at 277-318 us; its 3 MFMAs
// per tile, token group and 32 columns take 39 us at the matrix peak. This
// kernel takes 85-88 us on weights from HBM (370 TFLOP/s, 1.1 PFLOP/s of
// MFMAs; 99 at the median between a pass's other launches), the down product
// in 2 parts 51 us against 238, F16 gate/up 185 against 369, F32 235 against
// 575; what is left is LDS latency at two waves a SIMD. A step of 128
// columns is split once per block into operand order in LDS (each lane's 16
// bytes at its own slot: no bank conflicts either way), double buffered, one
// barrier a step; each wave owns its weight rows, read straight into
// registers (the tiles are in operand order), so a weight byte enters a CU
// once per 64 tokens. The eight waves are KG groups along K times 8 / KG
// along the rows (256 rows a BF16 block when that fills the CUs; fewer rows
// and more K groups when it does not); the groups' sums meet in LDS.
//
// Every four column blocks are a segment: the products of the inputs' mid and
// lo parts first, then the hi parts', from zero, so that the small terms are
// not rounded at the size of the large ones; the finished segments add in K
// order. (A single chain over K = 2048 doubled the decode kernel's distance
// to float64.) The formats in several parts keep the small products apart.
constexpr int kStepKb = 4;  // column blocks a step

template<int RT, int KG, int TT, bool kSwiGLU, int WF>
__launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
__global__ void FloatGemmKernel(const uint4* __restrict__ tiles, int row_tiles, int nkb,
                                const float* __restrict__ x, int ldx, int batch,
                                float* __restrict__ y, int ldy, int out_rows, int row_blocks,
                                int token_blocks, int parts, std::size_t part_stride) {
  constexpr int NW = WordsOf(WF), NP = PartsOf(WF);
  constexpr int RG = kWaves / KG;          // waves along the rows
  constexpr int kMine = kStepKb / KG;      // column blocks of a step a wave takes
  constexpr int kBufs = KG == 1 ? kMine : 2 * kMine;  // weight buffers
  constexpr int kAhead = KG == 4 ? 2 : 1;  // steps the inputs are loaded ahead
  constexpr int kPairs = kStepKb * TT / kWaves;  // (column block, group) pairs a wave stages
  static_assert(kMine >= 1 && kPairs * kWaves == kStepKb * TT);
  constexpr int kStage = kStepKb * TT * 3 * 64;  // uint4 of one stage
  constexpr int kRed = KG > 1 ? kWaves * RT * TT * 64 : 0;
  __shared__ uint4 s_mem[2 * kStage > kRed ? 2 * kStage : kRed];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, m = lane & 15;
  const int kg = wave / RG, rg = wave % RG;
  const int item = XcdMajorItem(blockIdx.x, gridDim.x);
  const int tb = item % token_blocks, rb = (item / token_blocks) % row_blocks;
  const int part = item / (token_blocks * row_blocks);
  const int tile0 = (rb * RG + rg) * RT, tok0 = tb * 16 * TT;
  const int p0 = part * nkb / parts, p1 = (part + 1) * nkb / parts;
  const int steps = (p1 - p0 + kStepKb - 1) / kStepKb;

  // Inputs: the wave stages pairs kPairs w .. of a step; columns past the
  // part and tokens past the batch read zeros.
  const BufferResource x_res = MakeBuffer(x, unsigned(batch) * unsigned(ldx) * 4u);
  float4 xv[kAhead][kPairs][2];
  const auto load_x = [&](int step, float4 (&v)[kPairs][2]) {
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
      const int pair = wave * kPairs + j;
      const int kb = p0 + step * kStepKb + pair / TT, token = tok0 + 16 * (pair % TT) + m;
      const unsigned at = kb < p1 && token < batch
                              ? (unsigned(token) * unsigned(ldx) + unsigned(kb * kTileCols + 8 * g)) * 4u
                              : kOutOfRange;
      v[j][0] = LoadF4(x_res, at);
      v[j][1] = LoadF4(x_res, at + 16u);
    }
  };
  const auto store_x = [&](uint4* stage, const float4 (&v)[kPairs][2]) {
#pragma unroll
    for (int j = 0; j < kPairs; ++j) {
      uint4 hi, mid, lo;
      Operands(v[j][0], v[j][1], hi, mid, lo);
      uint4* at = stage + (wave * kPairs + j) * 3 * 64 + lane;
      at[0] = hi;
      at[64] = mid;
      at[128] = lo;
    }
  };
  // Weights: the wave's column blocks in order (block i of it is column
  // block p0 + kStepKb (i / kMine) + kg kMine + i % kMine); a buffer is
  // loaded again as soon as its products are issued. Column blocks past the
  // part read zeros, as their inputs do, so no step needs a branch.
  // Tiles past the last one read the last one; their rows are never stored.
  BufferResource w_res[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
    w_res[r] = MakeBuffer(tiles + std::size_t(min(tile0 + r, row_tiles - 1)) * nkb * (64 * NW),
                          unsigned(nkb) * (1024u * NW));
  const unsigned w_off = unsigned(lane) * 16u;
  uint4 wv[kBufs][RT][NW];
  const auto load_w = [&](int i, uint4 (&dst)[RT][NW]) {
    const int kb = p0 + kStepKb * (i / kMine) + kg * kMine + i % kMine;
    const unsigned off = kb < p1 ? w_off : kOutOfRange;
    const unsigned at = kb < p1 ? unsigned(kb * NW) * 1024u : 0u;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int q = 0; q < NW; ++q)
        dst[r][q] = LoadB128(w_res[r], off, at + unsigned(q) * 1024u);
  };

  // sum: the finished segments; acc: the open one; rest (formats in several
  // parts): every product but hi times the weight's first part.
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 sum[RT][TT], acc[RT][TT], rest[NP > 1 ? RT : 1][NP > 1 ? TT : 1];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      sum[r][t] = acc[r][t] = zero;
      if constexpr (NP > 1)
        rest[r][t] = zero;
    }

  // One step's products. In one part: a pass of the mid and lo parts over the
  // wave's column blocks, then one of the hi parts; each unit (a token group
  // of a pass) reads the next unit's operands from LDS before its MFMAs, so
  // that the matrix pipe does not wait for them, in a fixed order except at
  // two K groups (a quarter of the step's time more there: 52 us against 46
  // at 6144 x 2048, 512 rows; 27.8 against 29.3 at four groups, 256 rows).
  const auto multiply = [&]<int kFirst>(const uint4* a, int next_block)
                            __attribute__((always_inline)) {
    if constexpr (NP == 1) {
      constexpr int kUnits = 2 * kMine * TT;
      const auto read = [&](int u, uint4 (&v)[2]) {
        const uint4* at = a + u % (kMine * TT) * 3 * 64;
        if (u < kMine * TT) {
          v[0] = at[2 * 64];
          v[1] = at[64];
        } else {
          v[0] = at[0];
        }
      };
      constexpr bool kOrdered = KG != 2;
      uint4 op[2][2];
      if constexpr (kOrdered)
        read(0, op[0]);
      Unroll<kUnits>([&](auto unit) __attribute__((always_inline)) {
        constexpr int u = unit, j = u / TT % kMine, t = u % TT;
        constexpr bool small = u < kMine * TT;
        if constexpr (kOrdered) {
          if constexpr (u + 1 < kUnits)
            read(u + 1, op[(u + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
        } else {
          read(u, op[u & 1]);
        }
#pragma unroll
        for (int k = 0; k < (small ? 2 : 1); ++k)
#pragma unroll
          for (int r = 0; r < RT; ++r)
            acc[r][t] = Mfma(op[u & 1][k], wv[kFirst + j][r][0], acc[r][t]);
        if constexpr (!small && t == TT - 1)
          load_w(next_block + j, wv[kFirst + j]);
        if constexpr (kOrdered)
          __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      Unroll<kMine>([&](auto block) __attribute__((always_inline)) {
        constexpr int j = block;
        uint4 av[TT][3];
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int k = 0; k < 3; ++k)
            av[t][k] = a[((j * TT + t) * 3 + k) * 64];
#pragma unroll
        for (int r = 0; r < RT; ++r) {
          uint4 wp[NP];
          WeightParts<WF>(wv[kFirst + j][r], wp);
#pragma unroll
          for (int i = 0; i < NP; ++i)
#pragma unroll
            for (int k = 2; k >= 0; --k)
#pragma unroll
              for (int t = 0; t < TT; ++t)
                if (i + k > 0)
                  rest[r][t] = Mfma(av[t][k], wp[i], rest[r][t]);
                else
                  acc[r][t] = Mfma(av[t][k], wp[i], acc[r][t]);
        }
        load_w(next_block + j, wv[kFirst + j]);
      });
    }
  };
  const auto close_segment = [&]() {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        sum[r][t] += acc[r][t];
        acc[r][t] = zero;
        asm volatile("" : "+v"(sum[r][t]), "+v"(acc[r][t]));
      }
  };

  load_x(0, xv[0]);
  if constexpr (kAhead == 2)
    load_x(1, xv[1]);
#pragma unroll
  for (int i = 0; i < kBufs; ++i)
    load_w(i, wv[i]);
  store_x(s_mem, xv[0]);
  // One step: the stage is visible and every wave is done with the other
  // one; a later step's inputs load while this one multiplies (two steps
  // ahead where a step is one column block a wave, shorter than the load).
  const auto run_step = [&]<int kParity>(int step) __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(kWaitLgkm0);
    BlockBarrier();
    // Past the last step every offset is out of range: nothing is read.
    load_x(step + kAhead, xv[kAhead == 2 ? kParity : 0]);
    const uint4* stage = s_mem + (step & 1) * kStage + kg * kMine * TT * 3 * 64 + lane;
    multiply.template operator()<KG == 1 ? 0 : kParity * kMine>(stage, step * kMine + kBufs);
    if ((step + 1) % KG == 0)
      close_segment();
    if (step + 1 < steps)
      store_x(s_mem + ((step + 1) & 1) * kStage, xv[kAhead == 2 ? 1 - kParity : 0]);
  };
  int step = 0;
  if constexpr (KG == 1) {
    for (; step < steps; ++step)
      run_step.template operator()<0>(step);
  } else {
    for (; step + 2 <= steps; step += 2) {
      run_step.template operator()<0>(step);
      run_step.template operator()<1>(step + 1);
    }
    if (step < steps)
      run_step.template operator()<0>(step);
  }
  close_segment();
  if constexpr (NP > 1)
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        sum[r][t] += rest[r][t];

  // Lane l of a tile holds tokens 4 (l >> 4) + i, weight row l & 15.
  float* yp = y + std::size_t(part) * part_stride;
  constexpr int kOut = kSwiGLU ? RT / 2 : RT;  // output tiles a wave's rows give
  const auto store = [&](int r, int t, const f32x4& a, const f32x4& b) {
    const int row = ((kSwiGLU ? tile0 / 2 : tile0) + r) * 16 + m;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int token = tok0 + 16 * t + 4 * g + i;
      if (row < out_rows && token < batch)
        yp[std::size_t(token) * ldy + row] =
            kSwiGLU ? (a[i] / (1.0f + expf(-a[i]))) * b[i] : a[i];
    }
  };
  if constexpr (KG == 1) {
#pragma unroll
    for (int r = 0; r < kOut; ++r)
#pragma unroll
      for (int t = 0; t < TT; ++t)
        store(r, t, sum[kSwiGLU ? 2 * r : r][t], sum[kSwiGLU ? 2 * r + 1 : r][t]);
    return;
  }
  // The K groups' sums through LDS, added in group order; the groups share
  // the output tiles.
  f32x4* red = reinterpret_cast<f32x4*>(s_mem);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int t = 0; t < TT; ++t)
      red[((kg * RG + rg) * RT + r) * (TT * 64) + t * 64 + lane] = sum[r][t];
  __syncthreads();
  const auto total = [&](int r, int t) {
    f32x4 s = red[(rg * RT + r) * (TT * 64) + t * 64 + lane];
#pragma unroll
    for (int k = 1; k < KG; ++k)
      s += red[((k * RG + rg) * RT + r) * (TT * 64) + t * 64 + lane];
    return s;
  };
#pragma unroll
  for (int u = 0; u < (kOut * TT + KG - 1) / KG; ++u) {
    const int unit = u * KG + kg, r = unit / TT, t = unit % TT;
    if (unit >= kOut * TT)
      break;
    const f32x4 a = total(kSwiGLU ? 2 * r : r, t);
    store(r, t, a, kSwiGLU ? total(2 * r + 1, t) : a);
  }
}

// Element (n, k) of a tile (row n < 16, column k < 32), in elements from
// the tile's start.
__host__ __device__ inline std::size_t TileIndex(int wf, int n, int k) {
  return wf == kF32 ? std::size_t(((k & 7) >> 2) * 256 + (16 * (k >> 3) + n) * 4 + (k & 3))
                    : std::size_t((16 * (k >> 3) + n) * 8 + (k & 7));
}

// Row gather from the tiles: out[i] = row tokens[i] (or, with a row table,
// inputs[i] when not null), as FP32 (hip/ops.hip:858-875 Value for F32,
// F16 and BF16). Ids at or past the vocabulary give zero rows (the host
// refuses them before a launch).
template<int WF>
__global__ void FloatEmbedKernel(const void* __restrict__ tiles, int nkb, int cols,
                                 std::uint32_t vocab, const std::uint32_t* __restrict__ tokens,
                                 const float* const* inputs, float* __restrict__ out) {
  const int i = blockIdx.y;
  const float* row_in = inputs ? inputs[i] : nullptr;
  const std::uint32_t t = row_in ? 0u : tokens[i];
  const std::size_t base = (std::size_t(t >> 4) * nkb) * kTileElems;
  const int n = int(t & 15u);
  for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < cols; c += gridDim.x * blockDim.x) {
    float v;
    if (row_in) {
      v = row_in[c];
    } else if (t >= vocab) {
      v = 0.0f;
    } else {
      const std::size_t at = base + std::size_t(c / kTileCols) * kTileElems +
                             TileIndex(WF, n, c % kTileCols);
      if constexpr (WF == kF32)
        v = static_cast<const float*>(tiles)[at];
      else if constexpr (WF == kF16)
        v = HalfBitsToFloat(static_cast<const std::uint16_t*>(tiles)[at]);
      else
        v = __uint_as_float(unsigned(static_cast<const std::uint16_t*>(tiles)[at]) << 16);
    }
    out[std::size_t(i) * cols + c] = v;
  }
}

template<int RT, bool kSwiGLU, int WF>
void Launch(const void* tiles, std::uint32_t row_tiles, std::uint32_t nkb, const float* x,
            std::uint32_t ldx, std::uint32_t batch, float* y, std::uint32_t ldy,
            std::uint32_t out_rows, std::uint32_t parts, hipStream_t stream) {
  const dim3 grid((row_tiles + RT - 1) / RT, (batch + 15) / 16, parts);
  FloatGemvKernel<RT, kSwiGLU, WF><<<grid, kThreads, 0, stream>>>(
      static_cast<const uint4*>(tiles), int(row_tiles), int(nkb), x, int(ldx), int(batch), y,
      int(ldy), int(out_rows), int(parts), std::size_t(batch) * ldy);
}

// The prompt rows' launch. RT row tiles a wave: 4 for BF16, 2 for the formats
// whose weights split (their MFMAs per staged input are twice and three
// times as many, and the parts take registers).
template<int RT, int KG, int TT, bool kSwiGLU, int WF>
void LaunchGemm(const void* tiles, std::uint32_t row_tiles, std::uint32_t nkb, const float* x,
                std::uint32_t ldx, std::uint32_t batch, float* y, std::uint32_t ldy,
                std::uint32_t out_rows, std::uint32_t parts, hipStream_t stream) {
  constexpr std::uint32_t kBlockTiles = RT * kWaves / KG;
  const std::uint32_t row_blocks = (row_tiles + kBlockTiles - 1) / kBlockTiles;
  const std::uint32_t token_blocks = (batch + 16 * TT - 1) / (16 * TT);
  FloatGemmKernel<RT, KG, TT, kSwiGLU, WF><<<row_blocks * token_blocks * parts, kThreads, 0, stream>>>(
      static_cast<const uint4*>(tiles), int(row_tiles), int(nkb), x, int(ldx), int(batch), y,
      int(ldy), int(out_rows), int(row_blocks), int(token_blocks), int(parts),
      std::size_t(batch) * ldy);
}

// Rows that take the prompt kernel: more than one token group, and inputs
// that 32-bit buffer offsets reach.
constexpr std::uint32_t kGemmMinRows = 17;
bool PromptRows(std::uint32_t batch, std::uint32_t ldx) {
  return batch >= kGemmMinRows && BufferFits(std::size_t(batch) * ldx * 4);
}

// Calls that the prompt rows' kernel takes in blocks of 64 rows x 32 tokens:
// where one round of them does, and up to 32 tokens.
std::uint32_t SmallBlocks(std::uint32_t row_tiles, std::uint32_t batch) {
  return (row_tiles + 3) / 4 * ((batch + 31) / 32);
}
bool TakesSmallBlocks(std::uint32_t row_tiles, std::uint32_t batch, std::uint32_t parts) {
  return batch <= 32 || SmallBlocks(row_tiles, batch) * parts <= 256;
}

// Whether the decode rows' kernel takes prompt rows sooner: few blocks whose
// K is not split leave the prompt kernel a long chain of steps on a part of
// the CUs, while 16 rows x 16 tokens a block use them all. Both times in
// microseconds, fitted to 2430 pairs of launches (BF16, F16 and F32, 256 to
// 16384 rows, K 256 to 7680, 17 to 512 tokens, 1 to 8 parts): the kernel it
// picks is within 0.2% of the faster on average and 29% at worst, where the
// prompt kernel for every call was 15% slower on average. 2048 x 7680 at 17
// tokens in one part: BF16 18.2 us against 30.7, F16 18.7 against 56.2, F32
// 21.1 against 67.4; in 8 parts 15.9 against 8.5 (BF16). From 512 row tiles
// on (two or four tiles a decode block) the prompt kernel won every pair. The
// decode kernel sums a wave's products in one chain: 0.7-1.9e-7 of the result
// from float64 for BF16 (the prompt kernel 0.8-1.4e-7), 0.9-3.4e-7 for F16
// and F32 (0.6-1.1e-7), as decode rows have it.
bool DecodeKernelSooner(int wf, std::uint32_t row_tiles, std::uint32_t nkb, std::uint32_t batch,
                        std::uint32_t parts, bool swiglu) {
  if (row_tiles >= 512 || !TakesSmallBlocks(row_tiles, batch, parts))
    return false;
  const double k = double(kTileCols) * nkb / parts;
  const std::uint32_t decode =
      (swiglu ? (row_tiles + 1) / 2 : row_tiles) * ((batch + 15) / 16) * parts;
  const std::uint32_t rounds = (SmallBlocks(row_tiles, batch) * parts + 255) / 256;
  const double step = wf == kBf16 ? 0.0042 : wf == kF16 ? 0.0071 : 0.0085;
  return 2.7 + 0.0002 * k + std::max(decode, 256u) * (0.0009 + 7.9e-6 * k) <
         rounds * (3.7 + step * k);
}

// Blocks of the prompt rows' kernel when a block owns `block_tiles` row tiles.
std::uint32_t GemmBlocks(std::uint32_t row_tiles, std::uint32_t batch, std::uint32_t block_tiles) {
  return (row_tiles + block_tiles - 1) / block_tiles * ((batch + 63) / 64);
}

// The block shape whose rounds on the 256 CUs cost least: `cost` is a round's
// measured time at K = 2048, in microseconds (BF16, 64 tokens: 512 rows a
// block 83, 256 rows 46, 128 rows 27.5, 64 rows 19.5). Blocks of 64 rows x 32
// tokens where one round of them does (three fit a CU: 2048 x 2048 BF16 at
// 64 rows 5.8 us against 8.6, F32 8.4 against 12.1; past one round the
// weights' second read costs more, 7680 x 2048 at 96 rows 34.5 against 29.9)
// and up to 32 tokens (the BF16 gate/up at 17 rows 12.0 us against 25).
template<int WF, bool kSwiGLU>
void GemmFormat(const void* tiles, std::uint32_t row_tiles, std::uint32_t nkb, const float* x,
                std::uint32_t ldx, std::uint32_t batch, float* y, std::uint32_t ldy,
                std::uint32_t out_rows, std::uint32_t parts, hipStream_t s) {
  const auto cost = [&](std::uint32_t block_tiles, double round) {
    return double((GemmBlocks(row_tiles, batch, block_tiles) * parts + 255) / 256) * round;
  };
  const auto launch = [&](auto launcher) {
    launcher(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, s);
  };
  if (TakesSmallBlocks(row_tiles, batch, parts)) {
    launch(LaunchGemm<2, 4, 2, kSwiGLU, WF>);
  } else if constexpr (WF == kBf16) {
    const double c[4] = {cost(32, 83.0), cost(16, 46.0), cost(8, 27.5), cost(4, 19.5)};
    const auto best = std::min_element(c, c + 4) - c;
    if (best == 0)
      launch(LaunchGemm<4, 1, 4, kSwiGLU, WF>);
    else if (best == 1)
      launch(LaunchGemm<4, 2, 4, kSwiGLU, WF>);
    else if (best == 2)
      launch(LaunchGemm<4, 4, 4, kSwiGLU, WF>);
    else
      launch(LaunchGemm<2, 4, 4, kSwiGLU, WF>);
  } else {
    const double c[3] = {cost(16, 80.0), cost(8, 46.0), cost(4, 28.0)};
    const auto best = std::min_element(c, c + 3) - c;
    if (best == 0)
      launch(LaunchGemm<2, 1, 4, kSwiGLU, WF>);
    else if (best == 1)
      launch(LaunchGemm<2, 2, 4, kSwiGLU, WF>);
    else
      launch(LaunchGemm<2, 4, 4, kSwiGLU, WF>);
  }
}

template<int WF>
void LaunchFormat(const void* tiles, std::uint32_t row_tiles, std::uint32_t nkb, const float* x,
                  std::uint32_t ldx, std::uint32_t batch, float* y, std::uint32_t ldy,
                  std::uint32_t out_rows, std::uint32_t parts, bool swiglu, hipStream_t s) {
  if (PromptRows(batch, ldx) &&
      !DecodeKernelSooner(WF, row_tiles, nkb, batch, swiglu ? 1 : parts, swiglu)) {
    if (swiglu)
      GemmFormat<WF, true>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, 1, s);
    else
      GemmFormat<WF, false>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, s);
  } else if (swiglu) {
    if (row_tiles >= 1024)
      Launch<4, true, WF>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, 1, s);
    else
      Launch<2, true, WF>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, 1, s);
  } else if (row_tiles >= 1024) {
    Launch<4, false, WF>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, s);
  } else if (row_tiles >= 512) {
    Launch<2, false, WF>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, s);
  } else {
    Launch<1, false, WF>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, s);
  }
}

bool FloatFormat(std::uint32_t type) {
  return type == LFM3_TYPE_BF16 || type == LFM3_TYPE_F16 || type == LFM3_TYPE_F32;
}

}  // namespace
}  // namespace lfm3amd

using namespace lfm3amd;

extern "C" {

size_t lfm3_float_tiled_bytes(uint32_t type, uint32_t rows, uint32_t cols) {
  if (!FloatFormat(type))
    return 0;
  return std::size_t(RowTilesOf(rows)) * ColBlocks(cols) * kTileElems * ElemBytes(int(type));
}

int lfm3_float_pack_host(uint32_t type, const void* src, uint32_t rows, uint32_t cols,
                         void* tiles, uint32_t tile_offset, uint32_t tile_stride) {
  if (!FloatFormat(type) || !src || !tiles || !rows || !cols || !tile_stride)
    return Fail(LFM3_E_INVALID, "invalid LFM3 float-weight pack");
  const std::size_t eb = ElemBytes(int(type));
  const auto* in = static_cast<const std::uint8_t*>(src);
  auto* out = static_cast<std::uint8_t*>(tiles);
  const std::uint32_t nkb = ColBlocks(cols);
  for (std::uint32_t r = 0; r < rows; ++r) {
    const std::size_t tile = std::size_t(tile_offset) + std::size_t(r / 16) * tile_stride;
    const int n = int(r % 16);
    for (std::uint32_t c = 0; c < cols; ++c) {
      const std::size_t at = (tile * nkb + c / kTileCols) * kTileElems +
                             TileIndex(int(type), n, int(c % kTileCols));
      std::memcpy(out + at * eb, in + (std::size_t(r) * cols + c) * eb, eb);
    }
  }
  return LFM3_OK;
}

uint32_t lfm3_bf16_gemv_parts(uint32_t rows, uint32_t cols, uint32_t batch) {
  // Narrow outputs split K so that the grid reaches about 256 blocks; each
  // part keeps at least 16 column blocks (two a wave). Prompt rows count the
  // blocks of 128 rows x 64 tokens, up to 32 of them the blocks of 64 rows x
  // 32 tokens in parts of 8 column blocks and more: 2048 x 2048 at 17 rows
  // with the norm that adds the parts takes 10.7 us in 8 (F16; 12.4 in 4,
  // 11.8 unsplit), F32 12.0 (13.7, 12.5), BF16 9.8 (10.7, 11.9).
  const std::uint32_t tiles = RowTilesOf(rows);
  const std::uint32_t rt = tiles >= 1024 ? 4 : tiles >= 512 ? 2 : 1;
  const bool few = batch >= kGemmMinRows && batch <= 32;
  const std::uint32_t blocks = few                     ? SmallBlocks(tiles, batch)
                               : batch >= kGemmMinRows ? GemmBlocks(tiles, batch, 8)
                                                       : (tiles + rt - 1) / rt;
  const std::uint32_t least = few ? 8 : 16;
  std::uint32_t parts = 1;
  while (parts < 8 && blocks * parts * 2 <= 256 && ColBlocks(cols) / (parts * 2) >= least)
    parts *= 2;
  return parts;
}

int lfm3_float_gemv(uint32_t type, const void* tiles, uint32_t rows, uint32_t cols,
                    const float* x, uint32_t ldx, float* y, uint32_t ldy, uint32_t batch,
                    uint32_t parts, int swiglu, void* stream) {
  const std::uint32_t out_rows = rows;
  const std::uint32_t row_tiles = RowTilesOf(rows) * (swiglu ? 2 : 1);
  if (!FloatFormat(type) || !tiles || !x || !y || !rows || !cols || cols % kTileCols ||
      ldx < cols || ldx % 4 || ldy < out_rows || !batch || !parts || parts > 8 ||
      parts > ColBlocks(cols) || (swiglu && parts != 1) ||
      (reinterpret_cast<std::uintptr_t>(x) & 15))
    return Fail(LFM3_E_INVALID, "unsupported LFM3 float-weight GEMV shape");
  const auto s = static_cast<hipStream_t>(stream);
  const std::uint32_t nkb = ColBlocks(cols);
  if (type == LFM3_TYPE_BF16)
    LaunchFormat<kBf16>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, swiglu, s);
  else if (type == LFM3_TYPE_F16)
    LaunchFormat<kF16>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, swiglu, s);
  else
    LaunchFormat<kF32>(tiles, row_tiles, nkb, x, ldx, batch, y, ldy, out_rows, parts, swiglu, s);
  return HipStatus(hipGetLastError(), "LFM3 float-weight GEMV launch");
}

int lfm3_float_embed(uint32_t type, const void* tiles, uint32_t vocab, uint32_t cols,
                     const uint32_t* tokens, const float* const* inputs, uint32_t n, float* out,
                     void* stream) {
  if (!FloatFormat(type) || !tiles || !tokens || !out || !vocab || !cols || cols % kTileCols ||
      !n)
    return Fail(LFM3_E_INVALID, "unsupported LFM3 float-weight embedding");
  const dim3 grid((cols + 255) / 256, n);
  const auto s = static_cast<hipStream_t>(stream);
  const int nkb = int(ColBlocks(cols));
  if (type == LFM3_TYPE_BF16)
    FloatEmbedKernel<kBf16><<<grid, 256, 0, s>>>(tiles, nkb, int(cols), vocab, tokens, inputs, out);
  else if (type == LFM3_TYPE_F16)
    FloatEmbedKernel<kF16><<<grid, 256, 0, s>>>(tiles, nkb, int(cols), vocab, tokens, inputs, out);
  else
    FloatEmbedKernel<kF32><<<grid, 256, 0, s>>>(tiles, nkb, int(cols), vocab, tokens, inputs, out);
  return HipStatus(hipGetLastError(), "LFM3 float-weight embedding launch");
}

// The BF16 forms (the reference precision) of the entry points above.
size_t lfm3_bf16_tiled_bytes(uint32_t rows, uint32_t cols) {
  return lfm3_float_tiled_bytes(LFM3_TYPE_BF16, rows, cols);
}

int lfm3_bf16_pack_host(const void* src, uint32_t rows, uint32_t cols, void* tiles,
                        uint32_t tile_offset, uint32_t tile_stride) {
  return lfm3_float_pack_host(LFM3_TYPE_BF16, src, rows, cols, tiles, tile_offset, tile_stride);
}

int lfm3_bf16_gemv(const void* tiles, uint32_t rows, uint32_t cols, const float* x,
                   uint32_t ldx, float* y, uint32_t ldy, uint32_t batch, uint32_t parts,
                   int swiglu, void* stream) {
  return lfm3_float_gemv(LFM3_TYPE_BF16, tiles, rows, cols, x, ldx, y, ldy, batch, parts, swiglu,
                         stream);
}

int lfm3_bf16_embed(const void* tiles, uint32_t vocab, uint32_t cols, const uint32_t* tokens,
                    const float* const* inputs, uint32_t n, float* out, void* stream) {
  return lfm3_float_embed(LFM3_TYPE_BF16, tiles, vocab, cols, tokens, inputs, n, out, stream);
}

}  // extern "C"
