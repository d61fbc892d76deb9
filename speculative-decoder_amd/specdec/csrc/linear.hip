// Linear layers of few rows (decode, draft and verify steps) on gfx950 MFMA.
//
// Reference semantics: the q/k/v, o, gate/up and down projections of
// lm/forward.py:56-58,63-64 (transformers' nn.Linear without bias, bf16),
// here with the projections fused as the model stores them (one q|k|v
// weight, one gate|up weight) and, for the residual adds of :63-64, the
// add folded into the same rounding: out = bf16(x W^T + out).
//
// At decode sizes a projection reads a few MB of weights for one to 64
// rows, so its time is the latency of one pass over the weight with every
// load in flight.  Layout: the weight W [N, K] bf16 is split into 16-row
// feature tiles, one workgroup per tile; the K/32 k-steps of the tile are
// split between the workgroup's waves (up to 8), each wave streaming its
// steps' W rows and x rows in batches of 8 k-steps with the next batch's
// loads in flight while one is multiplied on v_mfma_f32_16x16x32_bf16:
//   D[feature 4g+i, row c] += W[feature c'][k 8g..] . x[row c][k 8g..]
// (A = the tile's W rows, lane 16g + c loading the 16 bytes of row c at
// k = 32s + 8g; B = x rows, the same layout, rows past M reading zeros
// through the buffer bound).  The waves' partial sums meet in LDS and are
// added in wave order; lane (c, g) then holds row c's features 4g .. 4g+3.
// More rows: linear_rows_kernel, several 16-row column tiles per wave
// with x through LDS.
// Each output element goes through the same operations whatever M is, so
// a row's result does not depend on the other rows of the call: a token
// verified among k+1 and decoded alone get the same bits.
#include "common.h"

#include <algorithm>

namespace specdec {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;

constexpr int kLinRows = 64;        // rows of a call, at most (four 16-row column tiles)
constexpr int kLinMaxWaves = 8;     // waves per workgroup (k-step split)
constexpr int kLinMaxSteps = 256;   // K / 32, at most (K <= 8192)

struct LinArgs {
  const uint16_t *x;  // [M, K] bf16
  int64_t x_stride;
  const uint16_t *w;  // [N, K] bf16
  int64_t w_stride;
  uint16_t *out;  // [M, N] bf16
  int64_t out_stride;
  int M, K, N;
  int steps;     // K / 32
  int per_wave;  // k-steps per wave (the last waves may take fewer or none)
  int accumulate;
  int w_tiled;  // W in the tiled layout (w_lane below), w_stride = K
};

__device__ __forceinline__ float bf16_bits_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// The byte offset in W of lane (c = lane % 16, g = lane / 16)'s 16 bytes at
// k-step 0 of feature row `row` (row c of feature tile `tile`), and the
// bytes from one k-step to the next.  Row-major W [N, w_stride]: row `row`,
// k 8g .. 8g+7.  Tiled W (N % 16 == 0): the 16 x 32 block of each (tile,
// k-step) is 1 KB contiguous in lane order, block (t, s) at (t * K/32 + s) KB,
// lane (c, g) holding row 16t + c, k 32s + 8g .. 32s + 8g + 7 -- every
// load instruction of a wave reads one contiguous KB instead of 64 bytes
// from each of 16 rows.
__device__ __forceinline__ void w_lane(const LinArgs &a, int tile, int row, int lane, unsigned &base,
                                       unsigned &step) {
  if (a.w_tiled) {
    base = (unsigned)(((int64_t)tile * a.steps * 64 + lane) * 16);
    step = 1024u;
  } else {
    base = (unsigned)(((int64_t)row * a.w_stride + 8 * (lane >> 4)) * 2);
    step = 64u;
  }
}

// At most 16 rows; KB k-steps per load batch.  PART workgroups per feature
// tile (weights with fewer tiles than compute units): each reads and stores
// 16 / PART of the tile's features, the other lanes' W operands read out of
// range (zeros); an output's operations are the same.
template <int KB, int PART>
__global__ __launch_bounds__(kLinMaxWaves * 64) void linear_kernel(LinArgs a) {
  __shared__ f32x4 s_acc[kLinMaxWaves][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int tile = PART == 1 ? blockIdx.x : blockIdx.x / PART;
  const int n0 = tile * 16, part = PART == 1 ? 0 : blockIdx.x % PART;
  const bool mine = PART == 1 || c / (16 / PART) == part;
  const int s_lo = wave * a.per_wave;
  const int cnt = max(min(a.per_wave, a.steps - s_lo), 0);
  // W rows past N read the last row (never stored); x rows past M read zeros
  const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.w), 0, (int)((int64_t)a.N * a.w_stride * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.x), 0, (int)(((int64_t)(a.M - 1) * a.x_stride + a.K) * 2), 0x00020000);
  const int row = min(n0 + c, a.N - 1);
  unsigned wbase, wstep;
  w_lane(a, tile, row, lane, wbase, wstep);
  const unsigned xbase = (unsigned)(((int64_t)c * a.x_stride + 8 * g) * 2);
  // accumulate: the values added before the rounding, loaded now so their
  // round trip overlaps the weight's
  // (through a buffer resource, by every wave and call, with no branch --
  // a branch would make the compiler convert, and so wait for, the values
  // right there: rows past M read zeros, features past N are read but never
  // stored, and only wave 0 uses them)
  const int f0 = n0 + 4 * g;
  uint16_t pre[4];
  {
    // (without accumulate the resource is empty: every read is out of range,
    // returns zero and touches no memory)
    const int obytes = a.accumulate ? (int)(((int64_t)(a.M - 1) * a.out_stride + a.N) * 2) : 0;
    const __amdgpu_buffer_rsrc_t ob = __builtin_amdgcn_make_buffer_rsrc(a.out, 0, obytes, 0x00020000);
    const unsigned obase = (unsigned)(((int64_t)c * a.out_stride + f0) * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) pre[i] = __builtin_amdgcn_raw_buffer_load_b16(ob, obase + 2u * i, 0, 0);
  }
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 A0[KB], A1[KB], B0[KB], B1[KB];
  // batch b's loads: steps s_lo + KB b .. (past the wave's last step, its
  // last step again; those are not multiplied)
  auto issue = [&](u32x4 (&A)[KB], u32x4 (&B)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const unsigned s = (unsigned)(s_lo + min(b * KB + j, cnt - 1));
      A[j] = __builtin_amdgcn_raw_buffer_load_b128(wb, mine ? wbase + s * wstep : 0xFFFFFF00u, 0, 0);
      B[j] = __builtin_amdgcn_raw_buffer_load_b128(xb, xbase + s * 64u, 0, 0);
    }
  };
  auto consume = [&](const u32x4 (&A)[KB], const u32x4 (&B)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j)
      if (b * KB + j < cnt)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, A[j]),
                                                      __builtin_bit_cast(bf16x8, B[j]), acc, 0, 0, 0);
  };
  if (cnt > 0) {
    const int nb = (cnt + KB - 1) / KB;
    issue(A0, B0, 0);
    __builtin_amdgcn_sched_barrier(0);
    int b = 0;
    for (; b + 2 < nb; b += 2) {
      issue(A1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(A0, B0, b);
      __builtin_amdgcn_sched_barrier(0);
      issue(A0, B0, b + 2);
      __builtin_amdgcn_sched_barrier(0);
      consume(A1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b + 1 < nb) {  // the last two batches
      issue(A1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(A0, B0, b);
      __builtin_amdgcn_sched_barrier(0);
      consume(A1, B1, b + 1);
    } else {  // the last batch
      consume(A0, B0, b);
    }
  }
  s_acc[wave][lane] = acc;
  __syncthreads();
  // the sums of the waves, in wave order
  if (wave == 0 && c < a.M && (PART == 1 || 4 * g / (16 / PART) == part)) {
    f32x4 t = s_acc[0][lane];
    for (int w = 1; w < nw; ++w) t += s_acc[w][lane];
    uint16_t *dst = a.out + (int64_t)c * a.out_stride + f0;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = t[i];
      if (a.accumulate && f0 + i < a.N) v += bf16_bits_to_f32(pre[i]);
      o[i] = __builtin_bit_cast(uint16_t, __float2bfloat16(v));  // round to nearest even
    }
    if (f0 + 3 < a.N && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f0 + i < a.N) dst[i] = o[i];
    }
  }
}

// At most 8 rows of a weight with fewer feature tiles than half the compute
// units: a workgroup takes 8 features.  A wave's MFMAs multiply two of
// linear_kernel's k-splits ("chains") at once, chain w in the operands' lanes
// c < 8 (8 features, 8 rows) and chain w + waves in lanes c >= 8: the diagonal
// blocks of D are the two chains' sums, the other two are not used.  Every lane
// loads (a tile cut in two left half of each load's lanes empty, of W and of x),
// so half the load instructions request the same bytes, and with KB = 16 a
// wave has all of K <= 8192 in flight at once.  The chains are added in order:
// the bits of linear_kernel.  1.7B down (33.5 MB), 1 / 5 / 8 rows: 8.6 / 9.5 /
// 11.0 us, 4.3 to 3.5 TB/s with the launch (one workgroup a tile 11.2 / 12.7 /
// 13.9, a tile in two with half the lanes empty 11.1 at 5 rows); what is left
// beyond W's bytes is the launch and x, which every workgroup reads.
template <int KB>
__global__ __launch_bounds__(kLinMaxWaves / 2 * 64) void linear_pairs_kernel(LinArgs a, int nw) {
  __shared__ f32x4 s_acc[kLinMaxWaves][16];  // [chain][8 (features / 4) + row]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4, r = c & 7;
  const int tile = blockIdx.x >> 1, half = blockIdx.x & 1;
  const int n0 = tile * 16 + 8 * half;
  const int chain = wave + (c >> 3) * waves, s_lo = chain * a.per_wave;
  const int cnt = chain < nw ? max(min(a.per_wave, a.steps - s_lo), 0) : 0;
  const int most = max(min(a.per_wave, a.steps - wave * a.per_wave), 0);  // the first chain has no fewer
  // W rows past N read the last row (never stored); x rows past M, and both
  // operands past a chain's steps, read zeros
  const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.w), 0, (int)((int64_t)a.N * a.w_stride * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.x), 0, (int)(((int64_t)(a.M - 1) * a.x_stride + a.K) * 2), 0x00020000);
  unsigned wbase, wstep;
  w_lane(a, tile, min(n0 + r, a.N - 1), (lane & 48) | (8 * half + r), wbase, wstep);
  const unsigned xbase = (unsigned)(((int64_t)r * a.x_stride + 8 * g) * 2);
  // the result: lane 8 f + row of wave 0, features n0 + 4f ..; accumulate's
  // values loaded now, as in linear_kernel
  const int f0 = n0 + 4 * ((lane >> 3) & 1);
  uint16_t pre[4];
  {
    const int obytes = a.accumulate ? (int)(((int64_t)(a.M - 1) * a.out_stride + a.N) * 2) : 0;
    const __amdgpu_buffer_rsrc_t ob = __builtin_amdgcn_make_buffer_rsrc(a.out, 0, obytes, 0x00020000);
    const unsigned obase = (unsigned)(((int64_t)r * a.out_stride + f0) * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) pre[i] = __builtin_amdgcn_raw_buffer_load_b16(ob, obase + 2u * i, 0, 0);
  }
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 A0[KB], A1[KB], B0[KB], B1[KB];
  auto issue = [&](u32x4 (&A)[KB], u32x4 (&B)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const int t = b * KB + j;
      const unsigned s = (unsigned)(s_lo + t);
      A[j] = __builtin_amdgcn_raw_buffer_load_b128(wb, t < cnt ? wbase + s * wstep : 0xFFFFFF00u, 0, 0);
      B[j] = __builtin_amdgcn_raw_buffer_load_b128(xb, t < cnt ? xbase + s * 64u : 0xFFFFFF00u, 0, 0);
    }
  };
  auto consume = [&](const u32x4 (&A)[KB], const u32x4 (&B)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j)
      if (b * KB + j < most)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, A[j]),
                                                      __builtin_bit_cast(bf16x8, B[j]), acc, 0, 0, 0);
  };
  const int nb = (most + KB - 1) / KB;
  if (nb > 0) {
    issue(A0, B0, 0);
    __builtin_amdgcn_sched_barrier(0);
    int b = 0;
    for (; b + 2 < nb; b += 2) {
      issue(A1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(A0, B0, b);
      __builtin_amdgcn_sched_barrier(0);
      issue(A0, B0, b + 2);
      __builtin_amdgcn_sched_barrier(0);
      consume(A1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b + 1 < nb) {
      issue(A1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(A0, B0, b);
      __builtin_amdgcn_sched_barrier(0);
      consume(A1, B1, b + 1);
    } else {
      consume(A0, B0, b);
    }
  }
  if ((g >> 1) == (c >> 3) && chain < nw) s_acc[chain][8 * (g & 1) + r] = acc;
  __syncthreads();
  if (wave == 0 && lane < 16 && r < a.M) {
    f32x4 t = s_acc[0][lane];
    for (int w = 1; w < nw; ++w) t += s_acc[w][lane];
    uint16_t *dst = a.out + (int64_t)r * a.out_stride + f0;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = t[i];
      if (a.accumulate && f0 + i < a.N) v += bf16_bits_to_f32(pre[i]);
      o[i] = __builtin_bit_cast(uint16_t, __float2bfloat16(v));  // round to nearest even
    }
    if (f0 + 3 < a.N && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f0 + i < a.N) dst[i] = o[i];
    }
  }
}

// linear_kernel<KB> of the attention rows a draft decode step left as
// split partials (attention_decode_parts_kernel: `nparts` per row and query
// head): each workgroup first folds them into its LDS copy of the rows --
// per (row, head, 4 dims) the max of the partials' m, then L and O summed
// in part order with the same exp2 and fma steps as the attention kernel's
// own fold, O / L rounded to bf16 (with kDecWaves parts, that kernel's
// bits) -- while the weight's first load batch is in flight, then projects
// them with the plain projection's k-split (x read from LDS instead of
// memory): the bits of those rows followed by specdec_linear.  Workgroup 0
// also writes the rows to attn_out when that is given.
template <int KB, int NP>
__global__ __launch_bounds__(kLinMaxWaves * 64) void linear_parts_kernel(LinArgs a, const float *parts, int heads,
                                                                          uint16_t *attn_out) {
  extern __shared__ __align__(16) uint16_t s_x[];  // [M][K] bf16
  __shared__ f32x4 s_acc[kLinMaxWaves][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int s_lo = wave * a.per_wave;
  const int cnt = max(min(a.per_wave, a.steps - s_lo), 0);
  const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.w), 0, (int)((int64_t)a.N * a.w_stride * 2), 0x00020000);
  const int row = min(n0 + c, a.N - 1);
  unsigned wbase, wstep;
  w_lane(a, blockIdx.x, row, lane, wbase, wstep);
  const int f0 = n0 + 4 * g;
  uint16_t pre[4];
  {
    const int obytes = a.accumulate ? (int)(((int64_t)(a.M - 1) * a.out_stride + a.N) * 2) : 0;
    const __amdgpu_buffer_rsrc_t ob = __builtin_amdgcn_make_buffer_rsrc(a.out, 0, obytes, 0x00020000);
    const unsigned obase = (unsigned)(((int64_t)c * a.out_stride + f0) * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) pre[i] = __builtin_amdgcn_raw_buffer_load_b16(ob, obase + 2u * i, 0, 0);
  }
  u32x4 A0[KB], A1[KB];
  auto issue = [&](u32x4 (&A)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const unsigned s = (unsigned)(s_lo + min(b * KB + j, cnt - 1));
      A[j] = __builtin_amdgcn_raw_buffer_load_b128(wb, wbase + s * wstep, 0, 0);
    }
  };
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  const int xrow = c * a.K;  // this lane's row of x in LDS (rows past M are zero)
  // the batch's x operands are read from LDS first, then its MFMAs run back
  // to back (reading each operand just before its MFMA waited out one LDS
  // round trip per k-step)
  auto consume = [&](const u32x4 (&A)[KB], int b) {
    u32x4 bv[KB];
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      bv[j] = u32x4{0u, 0u, 0u, 0u};
      if (c < a.M && b * KB + j < cnt)
        bv[j] = *reinterpret_cast<const u32x4 *>(&s_x[xrow + 32 * (s_lo + b * KB + j) + 8 * g]);
    }
#pragma unroll
    for (int j = 0; j < KB; ++j)
      if (b * KB + j < cnt)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, A[j]),
                                                      __builtin_bit_cast(bf16x8, bv[j]), acc, 0, 0, 0);
  };
  if (cnt > 0) issue(A0, 0);
  // ---- the fold: item (row r, head hq, dims d0 .. d0+3)
  const int items = a.M * heads * 16;
  for (int it = tid; it < items; it += blockDim.x) {
    const int r = it / (heads * 16), hq = (it / 16) % heads, d0 = (it % 16) * 4;
    const float *pp = parts + ((int64_t)r * heads + hq) * NP * kDecPart;
    // every part's values first, in one round trip
    float mw[NP], lw[NP];
    f32x4 ow[NP];
#pragma unroll
    for (int w = 0; w < NP; ++w) {
      const f32x2 ml = *reinterpret_cast<const f32x2 *>(pp + w * kDecPart);
      mw[w] = ml[0];
      lw[w] = ml[1];
      ow[w] = *reinterpret_cast<const f32x4 *>(pp + w * kDecPart + 4 + d0);
    }
    float M = mw[0];
#pragma unroll
    for (int w = 1; w < NP; ++w) M = fmaxf(M, mw[w]);
    float L = 0.0f, O[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NP; ++w) {
      const float f = (mw[w] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(mw[w] - M);
      L = __builtin_fmaf(f, lw[w], L);
#pragma unroll
      for (int i = 0; i < 4; ++i) O[i] = __builtin_fmaf(f, ow[w][i], O[i]);
    }
    uint16_t ob[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ob[i] = __builtin_bit_cast(uint16_t, from_f32<__hip_bfloat16>(O[i] / L));
    const u32x2 packed = u32x2{(uint32_t)ob[0] | ((uint32_t)ob[1] << 16), (uint32_t)ob[2] | ((uint32_t)ob[3] << 16)};
    *reinterpret_cast<u32x2 *>(&s_x[r * a.K + hq * 64 + d0]) = packed;
    if (attn_out && blockIdx.x == 0)
      *reinterpret_cast<u32x2 *>(attn_out + (int64_t)r * a.K + hq * 64 + d0) = packed;
  }
  __syncthreads();
  if (cnt > 0) {
    const int nb = (cnt + KB - 1) / KB;
    int b = 0;
    for (; b + 2 < nb; b += 2) {
      issue(A1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(A0, b);
      __builtin_amdgcn_sched_barrier(0);
      issue(A0, b + 2);
      __builtin_amdgcn_sched_barrier(0);
      consume(A1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b + 1 < nb) {
      issue(A1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(A0, b);
      __builtin_amdgcn_sched_barrier(0);
      consume(A1, b + 1);
    } else {
      consume(A0, b);
    }
  }
  s_acc[wave][lane] = acc;
  __syncthreads();
  // the sums of the waves, in wave order (wave 0 stores), then the value
  // added before the rounding
  if (wave == 0 && c < a.M) {
    f32x4 t = s_acc[0][lane];
    for (int w = 1; w < nw; ++w) t += s_acc[w][lane];
    uint16_t *dst = a.out + (int64_t)c * a.out_stride + f0;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = t[i];
      if (a.accumulate && f0 + i < a.N) v += bf16_bits_to_f32(pre[i]);
      o[i] = __builtin_bit_cast(uint16_t, __float2bfloat16(v));
    }
    if (f0 + 3 < a.N && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f0 + i < a.N) dst[i] = o[i];
    }
  }
}

// The gate/up projection with the MLP's activation in its epilogue: a
// workgroup computes feature tile t of the gate half (W rows 16 t ..) and
// of the up half (W rows inter + 16 t ..) of the fused [2 inter, K] weight
// with the k-split the plain projection of that weight takes, so each of
// its sums has the plain projection's bits; the sums are rounded to bf16
// (the projection's output) and turned into act = SiLU(bf16(s g)) *
// bf16(s u) with the row's post-attention norm scale s computed here from
// the residual row (row_rms_scale_bf16, the MLP norm kernel's arithmetic).
// So act has the bits of the projection followed by rms_silu_mul, in one
// launch, and the [rows, 2 inter] intermediate is never written.
template <int KB, int NVH>
__global__ __launch_bounds__(kLinMaxWaves * 64) void linear_silu_kernel(LinArgs a, const uint16_t *hid,
                                                                         int64_t hid_stride, int hdim, float eps,
                                                                         int inter) {
  __shared__ f32x4 s_acc[kLinMaxWaves][2][64];
  __shared__ float s_scale[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int s_lo = wave * a.per_wave;
  const int cnt = max(min(a.per_wave, a.steps - s_lo), 0);
  const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.w), 0, (int)((int64_t)a.N * a.w_stride * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.x), 0, (int)(((int64_t)(a.M - 1) * a.x_stride + a.K) * 2), 0x00020000);
  const int rg = min(n0 + c, inter - 1);  // past the gate half: its last row, never stored
  unsigned gbase, ubase, wstep;
  w_lane(a, blockIdx.x, rg, lane, gbase, wstep);
  w_lane(a, inter / 16 + blockIdx.x, inter + rg, lane, ubase, wstep);
  const unsigned xbase = (unsigned)(((int64_t)c * a.x_stride + 8 * g) * 2);
  // the first pass over this wave's first residual row (row `wave`), loaded
  // now so its round trip overlaps the weight's (rows past M: not used)
  // (and of its second row, wave + nw, when the call has more rows than waves)
  const int nvh = hdim / 8;
  const u32x4 *h0 = reinterpret_cast<const u32x4 *>(hid + (int64_t)min(wave, a.M - 1) * hid_stride);
  const u32x4 *h1 = reinterpret_cast<const u32x4 *>(hid + (int64_t)min(wave + nw, a.M - 1) * hid_stride);
  u32x4 hv0[NVH], hv1[NVH];
  row_pass_loads<NVH>(h0, 0, nvh, lane, hv0);
  row_pass_loads<NVH>(h1, 0, nvh, lane, hv1);
  f32x4 accg = f32x4{0.f, 0.f, 0.f, 0.f}, accu = accg;
  u32x4 G0[KB], G1[KB], U0[KB], U1[KB], B0[KB], B1[KB];
  auto issue = [&](u32x4 (&G)[KB], u32x4 (&U)[KB], u32x4 (&B)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      const unsigned s = (unsigned)(s_lo + min(b * KB + j, cnt - 1));
      G[j] = __builtin_amdgcn_raw_buffer_load_b128(wb, gbase + s * wstep, 0, 0);
      U[j] = __builtin_amdgcn_raw_buffer_load_b128(wb, ubase + s * wstep, 0, 0);
      B[j] = __builtin_amdgcn_raw_buffer_load_b128(xb, xbase + s * 64u, 0, 0);
    }
  };
  auto consume = [&](const u32x4 (&G)[KB], const u32x4 (&U)[KB], const u32x4 (&B)[KB], int b) {
#pragma unroll
    for (int j = 0; j < KB; ++j)
      if (b * KB + j < cnt) {
        accg = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, G[j]),
                                                       __builtin_bit_cast(bf16x8, B[j]), accg, 0, 0, 0);
        accu = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, U[j]),
                                                       __builtin_bit_cast(bf16x8, B[j]), accu, 0, 0, 0);
      }
  };
  if (cnt > 0) {
    const int nb = (cnt + KB - 1) / KB;
    issue(G0, U0, B0, 0);
    __builtin_amdgcn_sched_barrier(0);
    int b = 0;
    for (; b + 2 < nb; b += 2) {
      issue(G1, U1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(G0, U0, B0, b);
      __builtin_amdgcn_sched_barrier(0);
      issue(G0, U0, B0, b + 2);
      __builtin_amdgcn_sched_barrier(0);
      consume(G1, U1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b + 1 < nb) {
      issue(G1, U1, B1, b + 1);
      __builtin_amdgcn_sched_barrier(0);
      consume(G0, U0, B0, b);
      __builtin_amdgcn_sched_barrier(0);
      consume(G1, U1, B1, b + 1);
    } else {
      consume(G0, U0, B0, b);
    }
  }
  s_acc[wave][0][lane] = accg;
  s_acc[wave][1][lane] = accu;
  // the rows' norm scales, wave w taking rows w, w + nw, ...
  for (int r = wave; r < a.M; r += nw) {
    const u32x4 *hr = reinterpret_cast<const u32x4 *>(hid + (int64_t)r * hid_stride);
    const float sc = r == wave        ? row_rms_scale_bf16_from<NVH>(hr, hv0, nvh, hdim, eps, lane)
                     : r == wave + nw ? row_rms_scale_bf16_from<NVH>(hr, hv1, nvh, hdim, eps, lane)
                                      : row_rms_scale_bf16<NVH>(hr, nvh, hdim, eps, lane);
    if (lane == 0) s_scale[r] = sc;
  }
  __syncthreads();
  const int f0 = n0 + 4 * g;
  if (wave == 0 && c < a.M) {
    f32x4 tg = s_acc[0][0][lane], tu = s_acc[0][1][lane];
    for (int w = 1; w < nw; ++w) {
      tg += s_acc[w][0][lane];
      tu += s_acc[w][1][lane];
    }
    const float sc = s_scale[c];
    uint16_t *dst = a.out + (int64_t)c * a.out_stride + f0;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // the projection's bf16 outputs, then the activation
      const float gv = to_f32(from_f32<__hip_bfloat16>(tg[i]));
      const float uv = to_f32(from_f32<__hip_bfloat16>(tu[i]));
      o[i] = silu_mul_scaled_bf16(gv, uv, sc);
    }
    if (f0 + 3 < inter && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f0 + i < inter) dst[i] = o[i];
    }
  }
}

// Up to 64 rows: the same sums in the same order as linear_kernel's and
// linear_silu_kernel's (one k-split, the waves' sums folded in wave order),
// so a row's bits do not depend on which of them ran.
//
// Read as MFMA operands, 16 rows of x give 64 bytes each at a stride of 2 K
// bytes, and the vector cache serves such a load at about a sixth of a
// contiguous one's rate.  At one column tile W's bytes hide that; at 64 rows
// the 1.7B's qkv took 20.8 us, 100 MB of x operands at 5 TB/s.  Here a wave
// moves its x through LDS: rows of 256 (or 128) bytes, kRowSteps k-steps, in coalesced
// 16-byte loads, one load instruction for four (eight) rows, written with the
// 16-byte pieces of a row permuted by xor with its number, so that neither the writes nor
// the operand reads meet in a bank.  The buffer is the wave's own, so no
// barrier is needed before the fold, only an order within the wave
// (wave_lds_order).  The next chunk's x and W are in flight
// while one is multiplied.
// Several feature tiles of a workgroup (NT) share a wave's x operands, which
// halves what x costs where the weight has tiles for every compute unit
// anyway; where it has not, the column tiles go to workgroups of their own
// (blockIdx.y; they meet in W's lines of one L2).
struct NoSide {
  struct Chunk {};
  __device__ void issue(Chunk &, int) {}
  __device__ void consume(const Chunk &, int) {}
};

// The norm scales of a wave's residual rows (rows w, w + nw, ... of the
// workgroup's), Q of them carried with each chunk: their loads ride with the
// chunk's and their arithmetic runs under the next chunk's loads.  A scale has
// row_rms_scale_bf16's bits: the same order of sums; pieces past the row's end
// are read out of range, and their zeros add nothing.
template <int Q, int NVH> struct RowScales {
  struct Chunk {
    u32x4 h[Q][NVH];
  };
  __amdgpu_buffer_rsrc_t hb;
  unsigned stride, nvec;  // bytes of a row, 16-byte pieces of it
  int lane, wave, nw, row0, rows, hdim;
  float eps;
  float *scale;
  __device__ int row(int i) const { return min(wave + i * nw, rows - 1); }  // past the last: the last again
  __device__ void issue(Chunk &k, int chunk) {
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int v = 0; v < NVH; ++v) {
        const unsigned p = lane + 64u * v;
        k.h[q][v] = __builtin_amdgcn_raw_buffer_load_b128(
            hb, p < nvec ? (unsigned)(row0 + row(chunk * Q + q)) * stride + p * 16u : 0xFFFFFF00u, 0, 0);
      }
  }
  __device__ void consume(const Chunk &k, int chunk) {
#pragma clang fp contract(off)
    if (wave + chunk * Q * nw >= rows) return;
    float ss[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      ss[q] = 0.0f;
#pragma unroll
      for (int v = 0; v < NVH; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const unsigned w = k.h[q][v][e >> 1];
          const float x = __uint_as_float((e & 1) ? (w & 0xFFFF0000u) : (w << 16));
          const float sq = x * x;
          ss[q] += sq;
        }
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const float sc = rsqrtf(wave_sum_dpp(ss[q]) / (float)hdim + eps);
      if (lane == 0) scale[row(chunk * Q + q)] = sc;
    }
  }
};

// Orders a wave's LDS accesses before and after it across the wave's lanes.
// The hardware runs a wave's LDS operations in order, so this costs nothing
// there; without it the compiler may move one lane's read before another
// lane's store (it sees different addresses).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NCT, int NT, int RS, typename Side>
__device__ __forceinline__ void rows_mainloop(const LinArgs &a, const unsigned (&wbase)[NT], unsigned wstep, int row0,
                                              int lane, int s_lo, int cnt, u32x4 *s_xw, f32x4 (&acc)[NT][NCT],
                                              Side &side) {
  const __amdgpu_buffer_rsrc_t wb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.w), 0, (int)((int64_t)a.N * a.w_stride * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t xb = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t *>(a.x), 0, (int)(((int64_t)(a.M - 1) * a.x_stride + a.K) * 2), 0x00020000);
  // k-steps past the wave's last are read out of range: zeros, which add
  // exact zeros; rows past M repeat the last row (their sums are not stored)
  constexpr unsigned kNowhere = 0xFFFFFF00u;
  constexpr int kPieces = 4 * RS, kRows = 64 / kPieces;  // 16-byte pieces of a row, rows of a load instruction
  constexpr int NX = 16 * NCT / kRows;
  const int piece = lane % kPieces, sub = lane / kPieces;
  auto swizzle = [](int r) { return RS == 4 ? r & 15 : (r >> 1) & 7; };
  unsigned xrow[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i)
    xrow[i] = (unsigned)((int64_t)min(row0 + kRows * i + sub, a.M - 1) * a.x_stride * 2) +
              (unsigned)(s_lo * 64 + piece * 16);
  struct Chunk {
    u32x4 x[NX];
    u32x4 w[NT][RS];
    typename Side::Chunk side;
  };
  auto issue = [&](Chunk &k, int b) {
    const bool in = b + (piece >> 2) < cnt;
#pragma unroll
    for (int i = 0; i < NX; ++i)
      k.x[i] = __builtin_amdgcn_raw_buffer_load_b128(xb, in ? xrow[i] + (unsigned)b * 64u : kNowhere, 0, 0);
#pragma unroll
    for (int j = 0; j < RS; ++j)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        k.w[t][j] = __builtin_amdgcn_raw_buffer_load_b128(
            wb, b + j < cnt ? wbase[t] + (unsigned)(s_lo + b + j) * wstep : kNowhere, 0, 0);
    side.issue(k.side, b / RS);
  };
  const int c = lane & 15, g = lane >> 4;
  auto consume = [&](const Chunk &k, int b) {
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int r = kRows * i + sub;
      s_xw[r * kPieces + (piece ^ swizzle(r))] = k.x[i];
    }
    wave_lds_order();
#pragma unroll
    for (int j = 0; j < RS; ++j)
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        const u32x4 bv = s_xw[(ct * 16 + c) * kPieces + ((4 * j + g) ^ swizzle(c))];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[t][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, k.w[t][j]),
                                                               __builtin_bit_cast(bf16x8, bv), acc[t][ct], 0, 0, 0);
      }
    side.consume(k.side, b / RS);
    wave_lds_order();  // the next stores, of a chunk or of the sums, after these reads
  };
  Chunk k0, k1;
  issue(k0, 0);
  for (int b = 0; b < cnt; b += 2 * RS) {
    issue(k1, b + RS);
    __builtin_amdgcn_sched_barrier(0);
    consume(k0, b);
    __builtin_amdgcn_sched_barrier(0);
    issue(k0, b + 2 * RS);
    __builtin_amdgcn_sched_barrier(0);
    consume(k1, b + RS);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// 16-byte words of LDS a wave needs: its x chunk, then its sums
template <int NCT, int NT, int RS> constexpr int kRowsLds = NCT * 64 * (RS > NT ? RS : NT);

template <int NCT, int NT, int RS>
__global__ __launch_bounds__(kLinMaxWaves * 64) void linear_rows_kernel(LinArgs a) {
  extern __shared__ __align__(16) u32x4 s_rows[];
  constexpr int W16 = kRowsLds<NCT, NT, RS>;
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.y * 16 * NCT;
  const int s_lo = wave * a.per_wave;
  const int cnt = max(min(a.per_wave, a.steps - s_lo), 0);
  u32x4 *s_xw = s_rows + wave * W16;
  unsigned wbase[NT], wstep;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int tile = min((int)blockIdx.x * NT + t, (a.N - 1) / 16);  // past the last: that one, never stored
    w_lane(a, tile, min(tile * 16 + c, a.N - 1), lane, wbase[t], wstep);
  }
  // (feature tile, column tile) pairs are stored by waves in turn; the values
  // added before the rounding are loaded now for the wave's first pair (as in
  // linear_kernel: an empty resource without accumulate)
  auto f_of = [&](int pair) { return (int)(blockIdx.x * NT + pair / NCT) * 16 + 4 * g; };
  uint16_t pre[4];
  {
    const int obytes = a.accumulate ? (int)(((int64_t)(a.M - 1) * a.out_stride + a.N) * 2) : 0;
    const __amdgpu_buffer_rsrc_t ob = __builtin_amdgcn_make_buffer_rsrc(a.out, 0, obytes, 0x00020000);
    const int pair = min(wave, NT * NCT - 1);
    const unsigned obase = (unsigned)(((int64_t)(row0 + (pair % NCT) * 16 + c) * a.out_stride + f_of(pair)) * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) pre[i] = __builtin_amdgcn_raw_buffer_load_b16(ob, obase + 2u * i, 0, 0);
  }
  f32x4 acc[NT][NCT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) acc[t][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  NoSide none;
  rows_mainloop<NCT, NT, RS>(a, wbase, wstep, row0, lane, s_lo, cnt, s_xw, acc, none);
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
      s_xw[(t * NCT + ct) * 64 + lane] = __builtin_bit_cast(u32x4, acc[t][ct]);
  __syncthreads();
  for (int pair = wave; pair < NT * NCT; pair += nw) {
    const int r = row0 + (pair % NCT) * 16 + c, f0 = f_of(pair);
    if (r >= a.M) continue;
    f32x4 t = __builtin_bit_cast(f32x4, s_rows[pair * 64 + lane]);
    for (int w = 1; w < nw; ++w) t += __builtin_bit_cast(f32x4, s_rows[w * W16 + pair * 64 + lane]);
    uint16_t *dst = a.out + (int64_t)r * a.out_stride + f0;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v = t[i];
      if (a.accumulate && f0 + i < a.N) v += bf16_bits_to_f32(pair == wave ? pre[i] : dst[i]);
      o[i] = __builtin_bit_cast(uint16_t, __float2bfloat16(v));  // round to nearest even
    }
    if (f0 + 3 < a.N && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f0 + i < a.N) dst[i] = o[i];
    }
  }
}

// The gate/up form (linear_silu_kernel's sums and
// epilogue): NP gate tiles and their up tiles per workgroup, the rows' norm
// scales computed along the chunks (RowScales).
template <int NCT, int NP, int RS, int NVH, int Q, int TH>
__global__ __launch_bounds__(TH) void linear_silu_rows_kernel(LinArgs a, const uint16_t *hid, int64_t hid_stride,
                                                              int hdim, float eps, int inter) {
  extern __shared__ __align__(16) u32x4 s_rows[];
  __shared__ float s_scale[16 * NCT];
  constexpr int NT = 2 * NP, W16 = kRowsLds<NCT, NT, RS>;
  const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.y * 16 * NCT, rows = min(16 * NCT, a.M - row0);
  const int s_lo = wave * a.per_wave;
  const int cnt = max(min(a.per_wave, a.steps - s_lo), 0);
  u32x4 *s_xw = s_rows + wave * W16;
  unsigned wbase[NT], wstep;
#pragma unroll
  for (int t = 0; t < NP; ++t) {
    const int tile = min((int)blockIdx.x * NP + t, (inter - 1) / 16);  // past the last: that one, never stored
    const int rg = min(tile * 16 + c, inter - 1);  // past the gate half: its last row, never stored
    w_lane(a, tile, rg, lane, wbase[2 * t], wstep);
    w_lane(a, inter / 16 + tile, inter + rg, lane, wbase[2 * t + 1], wstep);
  }
  RowScales<Q, NVH> side{
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(hid), 0,
                                        (int)(((int64_t)(a.M - 1) * hid_stride + hdim) * 2), 0x00020000),
      (unsigned)(hid_stride * 2), (unsigned)(hdim / 8), lane, wave, nw, row0, rows, hdim, eps, s_scale};
  f32x4 acc[NT][NCT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct) acc[t][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  rows_mainloop<NCT, NT, RS>(a, wbase, wstep, row0, lane, s_lo, cnt, s_xw, acc, side);
  // rows past the chunks' (a short k-split with many rows a wave)
  for (int k = 2 * ((cnt + 2 * RS - 1) / (2 * RS)); wave + k * Q * nw < rows; ++k) {
    typename RowScales<Q, NVH>::Chunk h;
    side.issue(h, k);
    side.consume(h, k);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
      s_xw[(t * NCT + ct) * 64 + lane] = __builtin_bit_cast(u32x4, acc[t][ct]);
  __syncthreads();
  for (int pair = wave; pair < NP * NCT; pair += nw) {
    const int p = pair / NCT, ct = pair % NCT;
    const int r = ct * 16 + c, f0 = (int)(blockIdx.x * NP + p) * 16 + 4 * g;
    if (r >= rows) continue;
    f32x4 tg = __builtin_bit_cast(f32x4, s_rows[(2 * p * NCT + ct) * 64 + lane]);
    f32x4 tu = __builtin_bit_cast(f32x4, s_rows[((2 * p + 1) * NCT + ct) * 64 + lane]);
    for (int w = 1; w < nw; ++w) {
      tg += __builtin_bit_cast(f32x4, s_rows[w * W16 + (2 * p * NCT + ct) * 64 + lane]);
      tu += __builtin_bit_cast(f32x4, s_rows[w * W16 + ((2 * p + 1) * NCT + ct) * 64 + lane]);
    }
    const float sc = s_scale[r];
    uint16_t *dst = a.out + (int64_t)(row0 + r) * a.out_stride + f0;
    uint16_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float gv = to_f32(from_f32<__hip_bfloat16>(tg[i]));
      const float uv = to_f32(from_f32<__hip_bfloat16>(tu[i]));
      o[i] = silu_mul_scaled_bf16(gv, uv, sc);
    }
    if (f0 + 3 < inter && ((uintptr_t)dst & 7) == 0) {
      *reinterpret_cast<u32x2 *>(dst) =
          u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f0 + i < inter) dst[i] = o[i];
    }
  }
}

template <int NCT, int NT, int RS>
static void launch_linear_rows(const LinArgs &a, int64_t tiles, int waves, hipStream_t s) {
  const dim3 grid((unsigned)((tiles + NT - 1) / NT), (unsigned)((a.M + 16 * NCT - 1) / (16 * NCT)));
  linear_rows_kernel<NCT, NT, RS><<<grid, 64 * waves, (size_t)waves * kRowsLds<NCT, NT, RS> * 16, s>>>(a);
}

template <int NCT, int NP, int RS, int NVH, int Q>
static int launch_silu_rows_nvh(const LinArgs &a, int waves, const uint16_t *h, int64_t h_stride, int hd, float eps,
                                int inter, hipStream_t s) {
  const dim3 grid((unsigned)(((inter + 15) / 16 + NP - 1) / NP), (unsigned)((a.M + 16 * NCT - 1) / (16 * NCT)));
  const size_t lds = (size_t)waves * kRowsLds<NCT, 2 * NP, RS> * 16;
  // more than four waves: a weight of fewer than 128 tile pairs, whose column
  // tiles are one to a workgroup (specdec_linear_silu)
  constexpr int TH = NCT == 1 && NP == 1 ? 512 : 256;
  if (64 * waves > TH) return SPECDEC_EUNSUPPORTED;  // (no split of today's; an error, not a call left out)
  linear_silu_rows_kernel<NCT, NP, RS, NVH, Q, TH><<<grid, 64 * waves, lds, s>>>(a, h, h_stride, hd, eps, inter);
  return launch_status();
}

template <int NCT, int NP, int RS>
static int launch_silu_rows(const LinArgs &a, int waves, const uint16_t *h, int64_t h_stride, int hd, float eps,
                            int inter, hipStream_t s) {
  const int nvec = hd / 8;
  if (nvec <= 2 * 64) return launch_silu_rows_nvh<NCT, NP, RS, 2, 3>(a, waves, h, h_stride, hd, eps, inter, s);
  if (nvec <= 4 * 64) return launch_silu_rows_nvh<NCT, NP, RS, 4, 2>(a, waves, h, h_stride, hd, eps, inter, s);
  return launch_silu_rows_nvh<NCT, NP, RS, 8, 1>(a, waves, h, h_stride, hd, eps, inter, s);
}

// The k-split of a [N, K] weight: waves per workgroup and k-steps per wave.
static void linear_split(LinArgs &a, int64_t tiles, int &waves) {
  // The k-split depends on the weight's shape only (never on the rows), so
  // a row's sums are the same in every call.  Up to 8 k-steps per wave
  // (one load batch) while that takes at most 8 waves; with a feature tile
  // for every compute unit, 4 waves of up to 16 steps (more workgroups
  // resident at once, the whole weight requested in one pass); the steps of
  // wider weights spread evenly over 8 waves.
  const int max_waves = tiles >= cu_count() ? 4 : kLinMaxWaves;
  waves = std::min(max_waves, (a.steps + 7) / 8);
  a.per_wave = (a.steps + waves - 1) / waves;
}

}  // namespace specdec

using namespace specdec;

SPECDEC_API int specdec_linear(const void *x, int64_t x_stride, const void *w, int64_t w_stride, int32_t w_layout,
                               int64_t rows, int64_t in_features, int64_t out_features, void *out,
                               int64_t out_stride, int32_t accumulate, void *stream) {
  if (rows < 0 || in_features <= 0 || out_features <= 0) return SPECDEC_EINVAL;
  if (w_layout != SPECDEC_W_ROWS && w_layout != SPECDEC_W_TILED) return SPECDEC_EINVAL;
  if (w_layout == SPECDEC_W_TILED) {
    if (out_features % 16 != 0) return SPECDEC_EINVAL;
    w_stride = in_features;
  }
  if (rows == 0) return SPECDEC_OK;
  if (rows > kLinRows || in_features % 32 != 0 || in_features / 32 > kLinMaxSteps) return SPECDEC_EUNSUPPORTED;
  // one buffer resource addresses W, another the rows of x (32-bit offsets)
  if (out_features * w_stride * 2 > INT32_MAX || out_features > INT32_MAX / 2) return SPECDEC_EUNSUPPORTED;
  if ((int64_t)kLinRows * std::max(x_stride, out_stride) * 2 > INT32_MAX) return SPECDEC_EUNSUPPORTED;
  if (!x || !w || !out || x_stride < in_features || w_stride < in_features || out_stride < out_features)
    return SPECDEC_EINVAL;
  if (x_stride % 8 || w_stride % 8 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) || ((uintptr_t)out & 1))
    return SPECDEC_EINVAL;
  LinArgs a{};
  a.x = (const uint16_t *)x;
  a.x_stride = x_stride;
  a.w = (const uint16_t *)w;
  a.w_stride = w_stride;
  a.out = (uint16_t *)out;
  a.out_stride = out_stride;
  a.M = (int)rows;
  a.K = (int)in_features;
  a.N = (int)out_features;
  a.steps = (int)(in_features / 32);
  a.accumulate = accumulate != 0;
  a.w_tiled = w_layout == SPECDEC_W_TILED;
  const int64_t tiles = (out_features + 15) / 16;
  if (tiles > INT32_MAX) return SPECDEC_EUNSUPPORTED;
  int waves = 0;
  linear_split(a, tiles, waves);
  const dim3 grid((unsigned)tiles), block((unsigned)(64 * waves));
  hipStream_t s = as_stream(stream);
  const int cus = std::max(cu_count(), 1);
  if (rows <= 16) {
    // From 9 rows x outweighs W's latency where every compute unit has a tile:
    // two tiles share x through LDS (1.7B qkv, 16 rows: 8.1 against 9.5 us; 5
    // rows 7.7 against 7.6).  With less than half a tile for each, workgroups
    // of 8 features fill the chip: linear_pairs_kernel up to 8 rows (5 rows,
    // against a workgroup a tile: 1.7B down 9.5 and 12.7 us, o 4.3 and 5.4,
    // draft down 3.3 and 3.8, draft qkv 2.78 and 2.82; with more tiles its
    // launch is too many workgroups, 1.7B qkv 8.1 and 7.7), and above it, for
    // a long projection only, a tile in two (1.7B down, 9 / 16 rows: 10.9 /
    // 13.9 against 12.5 / 15.7; o from a row-major weight 5.7 / 6.7 against 6.3 /
    // 7.4, from a tiled one 5.01 / 6.02 against 4.97 / 5.98; draft down, 9 rows:
    // 4.1 against 3.9).
    if (rows > 8 && tiles >= cus) launch_linear_rows<1, 2, 4>(a, tiles, waves, s);
    else if (2 * tiles <= cus && rows <= 8) {
      const dim3 pg((unsigned)(2 * tiles)), pb((unsigned)(64 * ((waves + 1) / 2)));
      if (a.per_wave > 8) linear_pairs_kernel<16><<<pg, pb, 0, s>>>(a, waves);
      else linear_pairs_kernel<8><<<pg, pb, 0, s>>>(a, waves);
    } else if (2 * tiles <= cus && a.steps >= (a.w_tiled ? 65 : 64))
      linear_kernel<8, 2><<<dim3((unsigned)(2 * tiles)), block, 0, s>>>(a);
    else linear_kernel<8, 1><<<grid, block, 0, s>>>(a);
    return launch_status();
  }
  // 17 to 64 rows.  Few feature tiles: column tiles go to workgroups of their
  // own while those still fit one to a compute unit (1.7B down, 128 tiles, 64
  // rows: 16.1 us as two workgroups of two column tiles, 23.1 as one of four,
  // 19.3 as four of one).  A tile for every compute unit and more: two tiles a
  // workgroup (qkv, 384 tiles, 64 rows: 10.6 against 14.5 us).
  const int ct = (int)((rows + 15) / 16);
  const int groups = (int)std::min<int64_t>(ct, std::max<int64_t>(1, cus / tiles));
  const int nct = (ct + groups - 1) / groups;
  if (tiles >= cus) {
    if (nct == 2) launch_linear_rows<2, 2, 4>(a, tiles, waves, s);
    else if (nct == 3) launch_linear_rows<3, 2, 4>(a, tiles, waves, s);
    else launch_linear_rows<4, 2, 2>(a, tiles, waves, s);
  } else if (nct == 1) launch_linear_rows<1, 1, 4>(a, tiles, waves, s);
  else if (nct == 2) launch_linear_rows<2, 1, 4>(a, tiles, waves, s);
  else if (nct == 3) launch_linear_rows<3, 1, 4>(a, tiles, waves, s);
  else launch_linear_rows<4, 1, 4>(a, tiles, waves, s);
  return launch_status();
}

SPECDEC_API int specdec_linear_attn_parts(const float *parts, int64_t rows, int64_t n_heads, int32_t nparts,
                                         const void *w, int64_t w_stride, int32_t w_layout, int64_t out_features,
                                         void *out, int64_t out_stride, int32_t accumulate, void *attn_out,
                                         void *stream) {
  if (rows < 0 || n_heads <= 0 || out_features <= 0) return SPECDEC_EINVAL;
  if (nparts != 4 && nparts != 8 && nparts != 16) return SPECDEC_EINVAL;
  if (((uintptr_t)parts & 15) || (attn_out && ((uintptr_t)attn_out & 7))) return SPECDEC_EINVAL;
  if (w_layout != SPECDEC_W_ROWS && w_layout != SPECDEC_W_TILED) return SPECDEC_EINVAL;
  if (rows == 0) return SPECDEC_OK;
  const int64_t k = n_heads * 64;
  if (w_layout == SPECDEC_W_TILED) {
    if (out_features % 16 != 0) return SPECDEC_EINVAL;
    w_stride = k;
  }
  if (rows > 16 || k > 2048) return SPECDEC_EUNSUPPORTED;
  if (out_features * w_stride * 2 > INT32_MAX || out_features > INT32_MAX / 2) return SPECDEC_EUNSUPPORTED;
  if (16 * out_stride * 2 > INT32_MAX) return SPECDEC_EUNSUPPORTED;
  if (!parts || !w || !out || w_stride < k || out_stride < out_features) return SPECDEC_EINVAL;
  if (w_stride % 8 || ((uintptr_t)w & 15) || ((uintptr_t)out & 1)) return SPECDEC_EINVAL;
  LinArgs a{};
  a.w = (const uint16_t *)w;
  a.w_stride = w_stride;
  a.out = (uint16_t *)out;
  a.out_stride = out_stride;
  a.M = (int)rows;
  a.K = (int)k;
  a.N = (int)out_features;
  a.steps = (int)(k / 32);
  a.accumulate = accumulate != 0;
  a.w_tiled = w_layout == SPECDEC_W_TILED;
  const int64_t tiles = (out_features + 15) / 16;
  if (tiles > INT32_MAX) return SPECDEC_EUNSUPPORTED;
  int waves = 0;
  linear_split(a, tiles, waves);  // the plain projection's k-split
  const dim3 grid((unsigned)tiles), block((unsigned)(64 * waves));
  const size_t lds = (size_t)rows * k * 2;
  hipStream_t s = as_stream(stream);
  uint16_t *ao = (uint16_t *)attn_out;
  if (nparts == 4) linear_parts_kernel<8, 4><<<grid, block, lds, s>>>(a, parts, (int)n_heads, ao);
  else if (nparts == 8) linear_parts_kernel<8, 8><<<grid, block, lds, s>>>(a, parts, (int)n_heads, ao);
  else linear_parts_kernel<8, 16><<<grid, block, lds, s>>>(a, parts, (int)n_heads, ao);
  return launch_status();
}

SPECDEC_API int specdec_linear_silu(const void *x, int64_t x_stride, const void *w, int64_t w_stride,
                                    int32_t w_layout, int64_t rows, int64_t in_features, int64_t inter,
                                    const void *hidden, int64_t hidden_stride, int64_t hidden_dim, float eps,
                                    void *out, int64_t out_stride, void *stream) {
  if (rows < 0 || in_features <= 0 || inter <= 0 || hidden_dim <= 0) return SPECDEC_EINVAL;
  if (w_layout != SPECDEC_W_ROWS && w_layout != SPECDEC_W_TILED) return SPECDEC_EINVAL;
  if (w_layout == SPECDEC_W_TILED) {
    if (inter % 16 != 0) return SPECDEC_EINVAL;
    w_stride = in_features;
  }
  if (rows == 0) return SPECDEC_OK;
  if (rows > kLinRows || in_features % 32 != 0 || in_features / 32 > kLinMaxSteps) return SPECDEC_EUNSUPPORTED;
  if (hidden_dim % 8 != 0 || hidden_dim > 8 * 64 * 8) return SPECDEC_EUNSUPPORTED;
  const int64_t n = 2 * inter;
  if (n * w_stride * 2 > INT32_MAX || n > INT32_MAX / 2) return SPECDEC_EUNSUPPORTED;
  if ((int64_t)kLinRows * x_stride * 2 > INT32_MAX) return SPECDEC_EUNSUPPORTED;
  if (!x || !w || !out || !hidden || x_stride < in_features || w_stride < in_features || out_stride < inter ||
      hidden_stride < hidden_dim)
    return SPECDEC_EINVAL;
  if (x_stride % 8 || w_stride % 8 || hidden_stride % 8 || ((uintptr_t)x & 15) || ((uintptr_t)w & 15) ||
      ((uintptr_t)hidden & 15) || ((uintptr_t)out & 1))
    return SPECDEC_EINVAL;
  LinArgs a{};
  a.x = (const uint16_t *)x;
  a.x_stride = x_stride;
  a.w = (const uint16_t *)w;
  a.w_stride = w_stride;
  a.out = (uint16_t *)out;
  a.out_stride = out_stride;
  a.M = (int)rows;
  a.K = (int)in_features;
  a.N = (int)n;
  a.steps = (int)(in_features / 32);
  a.w_tiled = w_layout == SPECDEC_W_TILED;
  // the plain projection's k-split for this [2 inter, K] weight
  int waves = 0;
  linear_split(a, (n + 15) / 16, waves);
  const dim3 grid((unsigned)((inter + 15) / 16)), block((unsigned)(64 * waves));
  const uint16_t *h = (const uint16_t *)hidden;
  const int hd = (int)hidden_dim, nvec = hd / 8;
  hipStream_t s = as_stream(stream);
  // (linear_silu_rows_kernel addresses the residual rows by 32-bit offsets)
  if (rows > 12 && rows * hidden_stride * 2 > INT32_MAX) {
    for (int64_t r = 0; r < rows; r += 12) {
      const int st = specdec_linear_silu(a.x + r * x_stride, x_stride, w, w_stride, w_layout,
                                         std::min<int64_t>(12, rows - r), in_features, inter, h + r * hidden_stride,
                                         hidden_stride, hidden_dim, eps, a.out + r * out_stride, out_stride, stream);
      if (st != SPECDEC_OK) return st;
    }
    return SPECDEC_OK;
  }
  if (rows <= 12) {
    if (nvec <= 2 * 64) linear_silu_kernel<4, 2><<<grid, block, 0, s>>>(a, h, hidden_stride, hd, eps, (int)inter);
    else if (nvec <= 4 * 64) linear_silu_kernel<4, 4><<<grid, block, 0, s>>>(a, h, hidden_stride, hd, eps, (int)inter);
    else linear_silu_kernel<4, 8><<<grid, block, 0, s>>>(a, h, hidden_stride, hd, eps, (int)inter);
    return launch_status();
  }
  // 13 to 64 rows (at 16 the 1.7B's takes 17.0 against 18.3 us, the draft's 5.0
  // against 5.9, at 9 rows 16.6 and 4.4 either way).  Every workgroup computes
  // the norm scales of its rows, so with few tiles the column tiles are spread further than the plain
  // projection's (draft, 96 tiles, 32 rows: 5.0 us as one column tile a
  // workgroup, 7.2 as two), and with two tiles for every compute unit a
  // workgroup takes two (1.7B, 40 rows: 20.1 against 24.2 us).
  const int ct = (int)((rows + 15) / 16), cus = std::max(cu_count(), 1);
  const int64_t tiles = (inter + 15) / 16;
  const int groups = (int)std::min<int64_t>(ct, std::max<int64_t>(1, 2 * cus / tiles));
  const int nct = tiles >= 2 * cus ? ct : (ct + groups - 1) / groups;
#define SPECDEC_SILU_ROWS(NCT, NP, RS) \
  return launch_silu_rows<NCT, NP, RS>(a, waves, h, hidden_stride, hd, eps, (int)inter, s)
  if (tiles >= 2 * cus) {
    if (nct == 1) SPECDEC_SILU_ROWS(1, 2, 2);
    if (nct == 2) SPECDEC_SILU_ROWS(2, 2, 2);
    if (nct == 3) SPECDEC_SILU_ROWS(3, 2, 2);
    SPECDEC_SILU_ROWS(4, 2, 2);
  }
  if (nct == 1) SPECDEC_SILU_ROWS(1, 1, 4);
  if (nct == 2) SPECDEC_SILU_ROWS(2, 1, 4);
  if (nct == 3) SPECDEC_SILU_ROWS(3, 1, 2);
  SPECDEC_SILU_ROWS(4, 1, 2);
#undef SPECDEC_SILU_ROWS
}
