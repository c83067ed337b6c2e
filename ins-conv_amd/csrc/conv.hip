// Output-stationary sparse convolution (submanifold 3^3, strided 2^3, 1x1) and the size-2
// stride-2 deconvolution.
//
// Work unit: a tile of 32 output rows per wavefront.  For each filter offset k the wavefront
// looks up the 32 input rows (neighbour map), skips the offset when none exists, otherwise
// gathers the rows straight from HBM/L2 into registers (two lanes per row) and multiplies them with W[k]
// on the matrix cores: fp32 operands in three bf16 parts each, fp32 accumulate (see "fp32 products on the
// bf16 matrix cores").  Accumulators stay in registers for all offsets, so every output row is written
// exactly once and no atomics are needed: the result of a row does not depend on which other rows share
// its tile, nor on the launch shape.
#include <algorithm>

#include "common.h"

#include <atomic>
#include <type_traits>

namespace insc {

typedef float f16v __attribute__((ext_vector_type(16)));


constexpr int CONV_WAVES = 4;
constexpr int TILE_M = 32;
constexpr int MAXK = 27;

// ---------------------------------------------------------------------------------------
// generic kernel: any Cin / Cout, one thread per (row, output channel).  Used for shapes
// the MFMA kernel does not cover (the 3-channel stem).
// ---------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void conv_generic_kernel(const float *__restrict__ in, int64_t ld_in,
                                                           float *__restrict__ out, int64_t ld_out,
                                                           const float *__restrict__ W,
                                                           const float *__restrict__ bias,
                                                           const int32_t *__restrict__ map0,
                                                           const int32_t *__restrict__ map1, int mode, int K,
                                                           const int32_t *__restrict__ rows,
                                                           const int32_t *__restrict__ d_n_rows, int64_t n_rows,
                                                           int Cin, int Cout,
                                                           const uint8_t *__restrict__ row_mask, BnEpilogue ep) {
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  const int cpb = 256 / Cout > 0 ? 256 / Cout : 1;  // rows per block (Cout <= 256)
  const int lr = threadIdx.x / Cout, co = threadIdx.x % Cout;
  if (lr >= cpb) return;
  for (int64_t t = (int64_t)blockIdx.x * cpb + lr; t < n; t += (int64_t)gridDim.x * cpb) {
    const int row = rows ? rows[t] : (int)t;
    if (row < 0 || (row_mask && !row_mask[row])) continue;
    float acc = bias ? bias[co] : 0.0f;
    for (int k = 0; k < K; k++) {
      int src;
      if (mode == MAP_NBR)
        src = map0[(int64_t)row * K + k];
      else if (mode == MAP_IDENTITY)
        src = row;
      else
        src = (map1[row] == k) ? map0[row] : -1;
      if (src < 0) continue;
      const float *x = in + (int64_t)src * ld_in;
      const float *w = W + (int64_t)k * Cin * Cout + co;
      for (int ci = 0; ci < Cin; ci++) acc = fmaf(x[ci], w[(int64_t)ci * Cout], acc);
    }
    if (ep.res) acc += ep.res[(int64_t)row * ep.ldr + co];
    if (out) out[(int64_t)row * ld_out + co] = acc;
    if (ep.out2) {
      const float y = fmaf(acc, ep.w[co], ep.b[co]);
      ep.out2[(int64_t)row * ep.ld2 + co] = y * ((y > 0.0f) ? 1.0f : ep.leak);
    }
  }
}

// ---------------------------------------------------------------------------------------
// 3^3 layers with 1..4 input channels (the RGB stem of a U-Net): same thread layout - a thread per (row,
// output channel) - and the same order of operations as the generic kernel (so the same bits), but the
// 27 x CIN weights of a thread's output channel stay in registers over all its rows, and the neighbour ids
// and input values of a batch of rows are fetched once per block, one (row, offset) per thread, and read
// back from LDS by the threads of the row (one 16-byte broadcast read per offset): with every thread
// fetching its row's 27 ids and 81 values itself the kernel was bound by the number of load instructions
// (92 us for 150k rows and 32 output channels).  With three channels the fourth word of the values says whether the
// neighbour exists (a word of its own in LDS: 150k rows of 3 -> 16 channels 38 us, 34 so; with one channel nothing is gained).
// ---------------------------------------------------------------------------------------
constexpr int STEM_ROWS = 16;  // rows per batch at most (those of 256 / Cout rows that a block handles at a time)
template <int CIN>
__global__ __launch_bounds__(256) void conv_stem_kernel(const float *__restrict__ in, int64_t ld_in,
                                                        float *__restrict__ out, int64_t ld_out,
                                                        const float *__restrict__ W, const float *__restrict__ bias,
                                                        const int32_t *__restrict__ map0,
                                                        const int32_t *__restrict__ rows,
                                                        const int32_t *__restrict__ d_n_rows, int64_t n_rows,
                                                        int Cout, const uint8_t *__restrict__ row_mask,
                                                        BnEpilogue ep) {
  constexpr int K = 27;
  __shared__ float4 xs[2][STEM_ROWS][K];  // input values of (row, offset); two batches in turn
  constexpr bool FLAG = CIN == 3;         // whether a neighbour exists rides in the free fourth word
  __shared__ int vs[FLAG ? 1 : 2][FLAG ? 1 : STEM_ROWS][K];  // 1: the row has a neighbour at the offset
  __shared__ int rid[2][STEM_ROWS];       // row of the batch, -1: none
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  const int cpb = min(256 / Cout, STEM_ROWS);  // rows per batch (Cout <= 256)
  const int lr = threadIdx.x / Cout, co = threadIdx.x % Cout;
  const bool worker = lr < cpb;
  float w[K][CIN];
#pragma unroll
  for (int k = 0; k < K; k++)
#pragma unroll
    for (int ci = 0; ci < CIN; ci++) w[k][ci] = worker ? W[((int64_t)k * CIN + ci) * Cout + co] : 0.0f;
  const float bv = (bias && worker) ? bias[co] : 0.0f;
  const float ew = (ep.out2 && worker) ? ep.w[co] : 0.0f, eb = (ep.out2 && worker) ? ep.b[co] : 0.0f;
  int buf = 0;
  for (int64_t t0 = (int64_t)blockIdx.x * cpb; t0 < n; t0 += (int64_t)gridDim.x * cpb, buf ^= 1) {
    // fetch: one (row, offset) per thread
    for (int e = threadIdx.x; e < cpb * K; e += 256) {
      const int er = e / K, k = e - er * K;
      const int64_t t = t0 + er;
      int row = t < n ? (rows ? rows[t] : (int)t) : -1;
      if (row >= 0 && row_mask && !row_mask[row]) row = -1;
      const int src = row >= 0 ? map0[(int64_t)row * K + k] : -1;
      float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (src >= 0) {
        const float *p = in + (int64_t)src * ld_in;
#pragma unroll
        for (int ci = 0; ci < CIN; ci++) x[ci] = p[ci];
      }
      if constexpr (FLAG) x[3] = src >= 0 ? 1.0f : 0.0f;
      else vs[buf][er][k] = src >= 0 ? 1 : 0;
      xs[buf][er][k] = make_float4(x[0], x[1], x[2], x[3]);
      if (k == 0) rid[buf][er] = row;
    }
    __syncthreads();  // (one barrier per batch: the next batch fills the other buffer)
    const int row = worker ? rid[buf][lr] : -1;
    if (row < 0) continue;
    float acc = bv;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const float4 xv = xs[buf][lr][k];
      const float x[4] = {xv.x, xv.y, xv.z, xv.w};
      float a = acc;
#pragma unroll
      for (int ci = 0; ci < CIN; ci++) a = fmaf(x[ci], w[k][ci], a);
      bool there;
      if constexpr (FLAG) there = xv.w != 0.0f;
      else there = vs[buf][lr][k] != 0;
      acc = there ? a : acc;
    }
    if (ep.res) acc += ep.res[(int64_t)row * ep.ldr + co];
    if (out) out[(int64_t)row * ld_out + co] = acc;
    if (ep.out2) {
      const float y = fmaf(acc, ew, eb);
      ep.out2[(int64_t)row * ep.ld2 + co] = y * ((y > 0.0f) ? 1.0f : ep.leak);
    }
  }
}

// The same, a batch ahead.  A batch's values are two trips to memory away (three with a row list): they are asked for while the
// batch before is computed, its ids one batch earlier still, none under a condition.  Whether a neighbour exists rides in the
// fourth word where the input leaves it free.  (150k rows of 3 -> 32 channels 58.8 us batch by batch, 42.5 so.)  What it costs
// is a prologue, two batches of loads past the end and, with NE = 2, loads for pairs that a batch does not have; the
// rule at the launch says where that pays.  Four wavefronts a SIMD with one pair a thread; with two pairs 128 registers would
// spill.  (One kernel for both forms, its parts in shared lambdas, took 1 us more a launch.)
template <int CIN, int NE>
__global__ __launch_bounds__(256, CIN < 4 && NE == 1 ? 4 : 2) void conv_stem_ahead_kernel(const float *__restrict__ in, int64_t ld_in,
                                                        float *__restrict__ out, int64_t ld_out,
                                                        const float *__restrict__ W, const float *__restrict__ bias,
                                                        const int32_t *__restrict__ map0,
                                                        const int32_t *__restrict__ rows,
                                                        const int32_t *__restrict__ d_n_rows, int64_t n_rows,
                                                        int Cout, const uint8_t *__restrict__ row_mask,
                                                        BnEpilogue ep) {
  constexpr int K = 27;
  __shared__ float4 xs[2][STEM_ROWS][K];  // input values of (row, offset); two batches in turn
  __shared__ int vs[CIN == 4 ? 2 : 1][CIN == 4 ? STEM_ROWS : 1][K];  // 1: the row has a neighbour there (CIN < 4: xs[..].w)
  __shared__ int rid[2][STEM_ROWS];       // row of the batch, -1: none
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  const int cpb = min(256 / Cout, STEM_ROWS);  // rows per batch (Cout <= 256)
  const int lr = threadIdx.x / Cout, co = threadIdx.x % Cout;
  const bool worker = lr < cpb;
  const int64_t step = (int64_t)gridDim.x * cpb;
  if ((int64_t)blockIdx.x * cpb >= n) return;  // (the whole block)

  // fetch: NE (row, offset) pairs per thread, two where a batch has more than 256 of them
  int row_of[NE], src_of[NE];
  float x_of[NE][CIN];
  bool have[NE];
  auto load_ids = [&](int64_t t0) {
#pragma unroll
    for (int i = 0; i < NE; i++) {
      const int e = (int)threadIdx.x + i * 256, er = e / K, k = e - er * K;
      const int64_t t = t0 + er, tc = min(t, n - 1);
      const int r = rows ? rows[tc] : (int)tc;
      const bool on = t < n && r >= 0 && (!row_mask || row_mask[max(r, 0)]);
      const int src = map0[(int64_t)(on ? r : 0) * K + k];
      row_of[i] = on ? r : -1;
      src_of[i] = on ? src : -1;
    }
  };
  auto gather = [&]() {
#pragma unroll
    for (int i = 0; i < NE; i++) {
      have[i] = src_of[i] >= 0;
      const float *p = have[i] ? in + (int64_t)src_of[i] * ld_in : W;  // (no condition: any CIN words that exist)
#pragma unroll
      for (int ci = 0; ci < CIN; ci++) x_of[i][ci] = p[ci];
    }
  };

  int64_t t0 = (int64_t)blockIdx.x * cpb;
  load_ids(t0);
  float w[K][CIN];
#pragma unroll
  for (int k = 0; k < K; k++)
#pragma unroll
    for (int ci = 0; ci < CIN; ci++) w[k][ci] = worker ? W[((int64_t)k * CIN + ci) * Cout + co] : 0.0f;
  const float bv = (bias && worker) ? bias[co] : 0.0f;
  const float ew = (ep.out2 && worker) ? ep.w[co] : 0.0f, eb = (ep.out2 && worker) ? ep.b[co] : 0.0f;
  gather();
  int row_here[NE];
#pragma unroll
  for (int i = 0; i < NE; i++) row_here[i] = row_of[i];
  load_ids(t0 + step);  // (batches past the end read the last row's ids and hold no row)
  for (int buf = 0; t0 < n; t0 += step, buf ^= 1) {
#pragma unroll
    for (int i = 0; i < NE; i++) {
      const int e = (int)threadIdx.x + i * 256, er = e / K, k = e - er * K;
      if (e >= cpb * K) break;
      float x[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int ci = 0; ci < CIN; ci++) x[ci] = have[i] ? x_of[i][ci] : 0.0f;
      if constexpr (CIN < 4) x[3] = have[i] ? 1.0f : 0.0f;
      xs[buf][er][k] = make_float4(x[0], x[1], x[2], x[3]);
      if constexpr (CIN == 4) vs[buf][er][k] = have[i] ? 1 : 0;
      if (k == 0) rid[buf][er] = row_here[i];
    }
    __syncthreads();  // (one barrier per batch: the next batch fills the other buffer)
    // the next batch's values and the ids of the one after are in flight while this one is computed
    gather();
#pragma unroll
    for (int i = 0; i < NE; i++) row_here[i] = row_of[i];
    load_ids(t0 + 2 * step);
    __builtin_amdgcn_sched_barrier(0);
    const int row = worker ? rid[buf][lr] : -1;
    if (row < 0) continue;
    float acc = bv;
#pragma unroll
    for (int k = 0; k < K; k++) {
      const float4 xv = xs[buf][lr][k];
      const float x[4] = {xv.x, xv.y, xv.z, xv.w};
      float a = acc;
#pragma unroll
      for (int ci = 0; ci < CIN; ci++) a = fmaf(x[ci], w[k][ci], a);
      bool there;
      if constexpr (CIN == 4) there = vs[buf][lr][k] != 0;
      else there = xv.w != 0.0f;
      acc = there ? a : acc;
    }
    if (ep.res) acc += ep.res[(int64_t)row * ep.ldr + co];
    if (out) out[(int64_t)row * ld_out + co] = acc;
    if (ep.out2) {
      const float y = fmaf(acc, ew, eb);
      ep.out2[(int64_t)row * ep.ld2 + co] = y * ((y > 0.0f) ? 1.0f : ep.leak);
    }
  }
}

// ---------------------------------------------------------------------------------------
// fp32 products on the bf16 matrix cores.  A float is the exact sum of three bf16 numbers of eight
// significant bits each (x = x0 + x1 + x2, |x1| < 2^-7 |x0|, |x2| < 2^-7 |x1|), so a product of two floats is
// nine products of bf16 numbers, each exact in fp32; the smallest (x2 y2, at most 2^-30 of the product) is left out, the
// other eight are summed in fp32, so that a single product comes out as the fp32 instruction rounds it (worst error 6.0e-8,
// 2-norm 2.5e-8 either way; without x1 y2 and x2 y1 as well it would be 1.9e-7 and 3.1e-8, at 6 % less time for the
// U-Net on 6k voxels, 2 % on 150k).
// Exact needs the third part to be a bf16 number too: both operands are split 2^23 times their size, which takes the
// last bit of the smallest float to 2^-126, the smallest normal bf16 number.  (Unscaled, bits drop out of operands below
// 2^-110: 2-norm error 4.4e-6 at 2^-116, 4.5e-3 at 2^-126.)  The sums are 2^46 times the true ones until they are final.
// Why: v_mfma_f32_32x32x16_bf16 does 16 times the operations per cycle of v_mfma_f32_32x32x2_f32, eight
// of them still twice.  Measured for 32x32x32 blocks in a loop, three wavefronts per SIMD: 441 ns a
// block in fp32 (152 TFLOP/s), 291 ns as eight bf16 products, 365 ns with the split of the gathered operand in
// the loop (324 ns where two output blocks share it).  The rounding that counts is that of the running sum of the
// leading products x0 y0; the others go into a sum of their own (struct Sum), so it is rounded once per 16 channels,
// where the fp32 instruction rounds its sum eight times.  2-norm error against 64-bit sums, fp32 instruction -> here:
// four layers of 32 channels on 500k sites 1.63e-7 -> 0.69e-7, of 64 channels 1.33e-7 -> 0.73e-7, of 128 channels on
// 5k 1.35e-7 -> 0.77e-7; the seven-scale U-Net on 150k voxels 4.2e-7 -> 2.0e-7.
// The gathered operand is split by truncation (multiply, and, subtract, byte permute: 6.5 instructions a float; rounding
// to nearest - convert, unpack, subtract - takes as many and is slower), the weights, once, by rounding to nearest.
// What has no such sum - infinities, NaN, weights from 2^105, sums from 2^82 - comes out as NaN or infinity;
// those elements are summed again in plain fp32 (repair_sums), so an infinity stays one.
// (Times of variants that the comments below say were not taken are with six products instead of eight.)
// ---------------------------------------------------------------------------------------
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8v __attribute__((ext_vector_type(8)));

// 16 channels of one row (8 per half-wave) in three parts: the operand of one 32x32x16 instruction each
struct Parts {
  u32x4 p[3];
};

constexpr float SPLIT_SCALE = 0x1p23f;                            // of either operand
constexpr float SUM_SCALE = 0x1p46f, SUM_UNSCALE = 0x1p-46f;      // of their products

__device__ __forceinline__ void split_pair(float a, float b, unsigned &p0, unsigned &p1, unsigned &p2) {
  a *= SPLIT_SCALE;
  b *= SPLIT_SCALE;
  const unsigned ua = __float_as_uint(a), ub = __float_as_uint(b);
  p0 = __builtin_amdgcn_perm(ub, ua, 0x07060302);  // the upper halves of both
  const float ra = a - __uint_as_float(ua & 0xFFFF0000u), rb = b - __uint_as_float(ub & 0xFFFF0000u);
  const unsigned va = __float_as_uint(ra), vb = __float_as_uint(rb);
  p1 = __builtin_amdgcn_perm(vb, va, 0x07060302);
  const float qa = ra - __uint_as_float(va & 0xFFFF0000u), qb = rb - __uint_as_float(vb & 0xFFFF0000u);
  p2 = __builtin_amdgcn_perm(__float_as_uint(qb), __float_as_uint(qa), 0x07060302);
}

__device__ __forceinline__ Parts split8(const float4 &lo, const float4 &hi) {
  const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  Parts s;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    unsigned a, b, c;
    split_pair(x[2 * j], x[2 * j + 1], a, b, c);
    s.p[0][j] = a;
    s.p[1][j] = b;
    s.p[2][j] = c;
  }
  return s;
}

__device__ __forceinline__ f16v mfma_bf16(const u32x4 &a, const u32x4 &b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8v, a), __builtin_bit_cast(bf8v, b), c, 0, 0, 0);
}

// A running sum: the products of the leading parts, and apart from them all others, which are 2^-7 of these at most -
// so the sum that carries the rounding error is rounded once per 16 channels.  (Both times SUM_SCALE.)
struct Sum {
  f16v lead, rest;
};
__device__ __forceinline__ void sum_start(Sum &a, float bias) {
#pragma unroll
  for (int v = 0; v < 16; v++) {
    a.lead[v] = bias * SUM_SCALE;
    a.rest[v] = 0.0f;
  }
}
__device__ __forceinline__ f16v sum_of(const Sum &a) {
  f16v t;
#pragma unroll
  for (int v = 0; v < 16; v++) t[v] = a.lead[v] + a.rest[v];
  return t;
}

// the sums of products themselves, of a total of such sums
template <int N, class A>
__device__ __forceinline__ void unscale(A &a) {
#pragma unroll
  for (int j = 0; j < N; j++) a[j] *= SUM_UNSCALE;
}

// acc += 16 channels
__device__ __forceinline__ void mac16(const Parts &a, const Parts &b, Sum &acc) {
  acc.rest = mfma_bf16(a.p[1], b.p[2], acc.rest);
  acc.rest = mfma_bf16(a.p[2], b.p[1], acc.rest);
  acc.rest = mfma_bf16(a.p[2], b.p[0], acc.rest);
  acc.rest = mfma_bf16(a.p[1], b.p[1], acc.rest);
  acc.rest = mfma_bf16(a.p[0], b.p[2], acc.rest);
  acc.rest = mfma_bf16(a.p[1], b.p[0], acc.rest);
  acc.rest = mfma_bf16(a.p[0], b.p[1], acc.rest);
  acc.lead = mfma_bf16(a.p[0], b.p[0], acc.lead);
}

// ---------------------------------------------------------------------------------------
// Weight packing.  For filter offset k, input-channel chunk ch (32 channels) and output-channel block nb (32
// channels) the weight tile is six 1 KB pieces, one per half s of the chunk and bf16 part i (piece s * 3 + i):
// lane = h*32 + j reads from it, with one 16-byte load, the eight values W[k][ch*32 + s*16 + h*8 + 0..7][nb*32 + j].
// A chunk whose second half lies beyond Cin (Cin = 16, 48, ..) is read as its first three pieces only.  Channels
// beyond Cin / Cout are zero.
// ---------------------------------------------------------------------------------------
constexpr int WT_BYTES = 6144;  // a weight tile
__host__ __device__ static inline int conv_nch(int Cin) { return (Cin + 31) / 32; }
static inline int conv_nb_per_group(int Cout) {
  const int nbt = (Cout + 31) / 32;
  return nbt > 4 ? 4 : nbt;
}
static inline int conv_nbt_padded(int Cout) {
  const int nbt = (Cout + 31) / 32, nb = conv_nb_per_group(Cout);
  return (int)cdiv(nbt, nb) * nb;
}

// a float rounded to bf16, to nearest even
__device__ __forceinline__ unsigned bf16_part(float x) {
  return __builtin_bit_cast(uint16_t, (__bf16)x);
}

// A weight from its three parts, exactly (cold).
__device__ __forceinline__ float weight_of(unsigned p0, unsigned p1, unsigned p2) {
  if ((p0 & 0x7F80u) == 0x7F80u) return __uint_as_float((p1 << 16) | p2);
  return (__uint_as_float(p0 << 16) + __uint_as_float(p1 << 16) + __uint_as_float(p2 << 16)) * (1.0f / SPLIT_SCALE);
}

// The fp32 layout of insc_conv_pack_weights: a tile is 4 KB, four 1 KB quarters; quarter q holds, for lane 0..63 in
// turn, the values W[k][ch*32 + h*16 + s][nb*32 + j], s = 4q..4q+3.
__global__ void pack_weights_kernel(const float *__restrict__ W, int K, int Cin, int Cout, int nch, int nbtp,
                                    float *__restrict__ Wp) {
  const int64_t total = (int64_t)K * nch * nbtp * 1024;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int s = (int)(((e >> 8) & 3) * 4 + (e & 3)), lane = (int)((e >> 2) & 63);
    int64_t q = e >> 10;
    const int nb = (int)(q % nbtp);
    q /= nbtp;
    const int ch = (int)(q % nch), k = (int)(q / nch);
    const int cin = ch * 32 + (lane >> 5) * 16 + s, col = nb * 32 + (lane & 31);
    Wp[e] = (cin < Cin && col < Cout) ? W[((int64_t)k * Cin + cin) * Cout + col] : 0.0f;
  }
}

// The three-part layout.
__global__ void split_weights_kernel(const float *__restrict__ W, int K, int Cin, int Cout, int nch, int nbtp,
                                     uint16_t *__restrict__ Ws) {
  const int64_t total = (int64_t)K * nch * nbtp * 1024;  // one (lane, value) of all three parts per thread
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int j8 = (int)(e & 7), lane = (int)((e >> 3) & 63), s = (int)((e >> 9) & 1);
    const int64_t tile = e >> 10;
    int64_t q = tile;
    const int nb = (int)(q % nbtp);
    q /= nbtp;
    const int ch = (int)(q % nch), k = (int)(q / nch);
    const int cin32 = s * 16 + (lane >> 5) * 8 + j8, cin = ch * 32 + cin32, col = nb * 32 + (lane & 31);
    float x = (cin < Cin && col < Cout) ? W[((int64_t)k * Cin + cin) * Cout + col] : 0.0f;
    uint16_t *to = Ws + tile * (WT_BYTES / 2) + s * 1536 + lane * 8 + j8;
    // (weights that the scale would take to the end of the range, infinities and NaN: NaN in the first part, so that their
    // sums are formed again, and the weight itself in the other two)
    const unsigned u = __float_as_uint(x);
    unsigned p0 = bf16_part(x * SPLIT_SCALE), p1 = u >> 16, p2 = u & 0xFFFFu;
    if ((p0 & 0x7F80u) == 0x7F80u) {
      p0 = 0x7FC0u;
    } else {
      x = x * SPLIT_SCALE - __uint_as_float(p0 << 16);  // (exact)
      p1 = bf16_part(x);
      p2 = bf16_part(x - __uint_as_float(p1 << 16));
    }
    to[0] = (uint16_t)p0;
    to[512] = (uint16_t)p1;
    to[1024] = (uint16_t)p2;
  }
}

// The lane's number, formed where it is asked for: what rarely runs or runs once per tile would otherwise have its
// addresses formed ahead of the kernel's loop and kept, or spilled, across it (the sums formed again below took
// conv_wshare_kernel from 1455 to 1736 us, 64 -> 64 at 500k sites).
__device__ __forceinline__ int lane_again() {
  int all = -1;
  asm volatile("" : "+s"(all));
  return (int)__builtin_amdgcn_mbcnt_hi((unsigned)all, __builtin_amdgcn_mbcnt_lo((unsigned)all, 0));
}

// Rows of a tile that the elements of this lane's 32x32 sums belong to (element v: row 8 * (v / 4) + 4 * h + v % 4), from
// the lanes that hold them.
__device__ __forceinline__ void rows_of_elements(int my_row, int (&rid)[16]) {
  const int base = (lane_again() >> 5) * 16;
#pragma unroll
  for (int v = 0; v < 16; v++) rid[v] = __builtin_amdgcn_ds_bpermute(base + 4 * (8 * (v >> 2) + (v & 3)), my_row);
}

// Elements whose sum of bf16 products is not finite (an infinity or NaN among the inputs or weights, or an overflow on
// the way) are formed again in plain fp32: tile_sums() gives them for the wavefront's tile (add_plain_products below), v0
// is the first of this lane's N elements among its sixteen.  Which elements these are depends on the element's own sum
// alone - but for an infinite weight, which makes NaN of the zeros of rows without its offset as well: these come out right,
// with the rounding of this sum.  One multiply-add per element finds out that there are none.
__device__ __forceinline__ bool is_bad(float x) { return (__float_as_uint(x) & 0x7F800000u) == 0x7F800000u; }
template <int N, class A>
__device__ __forceinline__ float not_finite(const A &a, float t) {  // NaN as soon as one is infinite or NaN
#pragma unroll
  for (int j = 0; j < N; j++) t = fmaf(a[j], 0.0f, t);
  return t;
}
template <int N, class A, class F>
__device__ __forceinline__ void repair_sums(A &a, int v0, const F &tile_sums) {
  const float t = not_finite<N>(a, 0.0f);
  if (__builtin_expect(!__any(t != t), 1)) return;
  const f16v x = tile_sums();
#pragma unroll
  for (int j = 0; j < N; j++) {
    float y = x[j];
    if (N < 16) {
#pragma unroll
      for (int v = 0; v < 16; v++) y = v == v0 + j ? x[v] : y;
    }
    a[j] = is_bad(a[j]) ? y : a[j];
  }
}

// ---------------------------------------------------------------------------------------
// MFMA kernel.  Cin % 16 == 0, rows of `in` 16-byte aligned, packed weights.
// Software pipeline: while the 16*NB MFMAs of one (offset, channel chunk) run, the gather of
// the next chunk's input rows and the next weight tile are already in flight.
// ---------------------------------------------------------------------------------------
// Gathered row chunk: lane (r, h) holds channels h*8 .. h*8+7 of the chunk's first half (q[0], q[1]) and of its
// second half (q[2], q[3]).
struct Frag {
  float4 q[4];
};
// A weight tile as it is loaded.  PW: from the packed fp32 layout (what insc_conv_pack_weights makes and callers of the C
// ABI may hold): sixteen weights a lane, which are split as split_weights_kernel does it, so either layout gives the same
// bits.  Costs about as many instructions per tile as the gathered chunk's parts: 64 -> 64 at 500k sites 411 us against 337,
// 39k sites 54 against 48; in scratch memory, once per call, it would cost a launch, an allocation now and then, and
// so capture into a graph.
template <bool PW>
struct WFrag {
  Parts s[2];
};
template <>
struct WFrag<true> {
  float4 q[4];
};
constexpr int pw_pieces(bool pw, int halves) { return pw ? 4 : 3 * halves; }  // of a tile: 1 KB each
constexpr int wt_bytes(bool pw) { return pw ? 4096 : WT_BYTES; }

typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
typedef float fl2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {  // (one instruction)
  const fl2v v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf2v));
}
// eight weights, as split_weights_kernel
__device__ __forceinline__ Parts split8_nearest(const float4 &lo, const float4 &hi) {
  const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  Parts s;
#pragma unroll
  for (int j = 0; j < 4; j++) {
    float a = x[2 * j] * SPLIT_SCALE, b = x[2 * j + 1] * SPLIT_SCALE;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const unsigned p = bf16_pair(a, b);
      s.p[i][j] = p;
      a -= __uint_as_float(p << 16);
      b -= __uint_as_float(p & 0xFFFF0000u);
    }
  }
  return s;
}
__device__ __forceinline__ const Parts &parts_of(const WFrag<false> &w, int half) { return w.s[half]; }
__device__ __forceinline__ Parts parts_of(const WFrag<true> &w, int half) {
  return split8_nearest(w.q[2 * half], w.q[2 * half + 1]);
}

// acc += chunk a times weight tile b; full: the chunk's second half exists
template <bool PW>
__device__ __forceinline__ void mac_chunk(Sum &acc, const Parts (&a)[2], const WFrag<PW> &b, bool full) {
  mac16(a[0], parts_of(b, 0), acc);
  if (full) mac16(a[1], parts_of(b, 1), acc);
}

// Gather: every lane reads the 64 bytes of its own input row that the MFMA A operand needs, with
// buffer loads: one 32-bit offset per item, rows without a neighbour get an out-of-range offset
// and the hardware returns zeros, and the weight tile is addressed by a scalar offset.
// offsets at or beyond this bound make a buffer load return zeros
constexpr uint32_t BUF_OOB = 0xFFFFF000u;  // room for the per-load immediate on top

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float4 buf_load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

// The 32-channel chunk at byte offset `base` (BUF_OOB: zeros) of a lane's own row, every lane its 64 bytes of it.
__device__ __forceinline__ Frag gather_chunk(__amdgpu_buffer_rsrc_t rin, bool on, uint32_t base, int h, bool full) {
  const uint32_t v0 = on ? base + (uint32_t)(h * 32) : BUF_OOB, v1 = on && full ? base + (uint32_t)(64 + h * 32) : BUF_OOB;
  Frag f;
  f.q[0] = buf_load16(rin, v0, 0);
  f.q[1] = buf_load16(rin, v0 + 16u, 0);
  f.q[2] = buf_load16(rin, v1, 0);
  f.q[3] = buf_load16(rin, v1 + 16u, 0);
  return f;
}

// The same chunk two lanes at a time: loads 0 and 1 of an even lane and its odd neighbour bring 32 consecutive bytes of the
// even and of the odd lane's row (loads 2 and 3: 64 bytes further on), and the two lanes exchange what is the other's
// (own_rows).  Why: the address unit takes a quad of lanes per cycle and line they touch, whatever they read of it, so four
// rows a quad are four cycles for 64 bytes: rows that all lie in L1 came in at 9.3 TB/s that way and at 13.7 two rows a quad;
// 500k sites of 32 channels at 8.5 and 11.1.  (A line a quad reaches 17.0 and 12.3, but its exchange over four lanes takes 32
// instructions and not 16: 32 -> 32 at 500k sites 104, 99 and 102 us a layer with one, two and four lanes a row.)
// Kernels whose launches are shorter than a few wavefronts per SIMD wait for their own instructions, not for the address
// unit, and gather row by row (U-Net on 6k voxels 977 us, two lanes a row 1020).  So do the kernels that split packed fp32 weights
// as they go, which wait for their vector instructions: 112 -> 112 at 60k sites 230 us two lanes a row, 209 row by row.
template <int CTRL>
__device__ __forceinline__ uint32_t lane_perm(uint32_t x) {  // (an operand modifier of the instruction that uses it)
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}
__device__ __forceinline__ uint32_t pair_piece(int lane) { return (uint32_t)((lane & 1) * 16 + (lane & 32)); }
__device__ __forceinline__ Frag gather_pairs(__amdgpu_buffer_rsrc_t rin, bool on, uint32_t base, uint32_t piece, bool full) {
  const uint32_t b = on ? base : BUF_OOB;
  const uint32_t v0 = lane_perm<0xA0>(b) + piece, v1 = lane_perm<0xF5>(b) + piece;  // quad_perm [0,0,2,2] and [1,1,3,3]
  Frag f;
  f.q[0] = buf_load16(rin, v0, 0);
  f.q[1] = buf_load16(rin, v1, 0);
  f.q[2] = buf_load16(rin, full ? v0 + 64u : BUF_OOB, 0);
  f.q[3] = buf_load16(rin, full ? v1 + 64u : BUF_OOB, 0);
  return f;
}
// x of even lanes stays, x of odd ones goes to their even neighbour's y; y the other way round.  Eight v_cndmask with a lane
// permutation on one operand, a form that the compiler does not make by itself.  (The wait states in front are those
// of an operand that the instruction before has written; every lane is active where this is called.)
__device__ __forceinline__ void exchange(float4 &x, float4 &y) {
  float4 t, u;
  asm("s_nop 0\n\ts_mov_b64 vcc, %16\n\t"
      "v_cndmask_b32_dpp %0, %12, %8, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %1, %13, %9, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %2, %14, %10, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %3, %15, %11, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "s_not_b64 vcc, vcc\n\t"
      "v_cndmask_b32_dpp %4, %8, %12, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %5, %9, %13, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %6, %10, %14, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_cndmask_b32_dpp %7, %11, %15, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "=&v"(t.x), "=&v"(t.y), "=&v"(t.z), "=&v"(t.w), "=&v"(u.x), "=&v"(u.y), "=&v"(u.z), "=&v"(u.w)
      : "v"(x.x), "v"(x.y), "v"(x.z), "v"(x.w), "v"(y.x), "v"(y.y), "v"(y.z), "v"(y.w), "s"(0x5555555555555555ull)
      : "vcc", "scc");
  x = t;
  y = u;
}
// what gather_pairs has loaded, sorted out: as gather_chunk gives it
__device__ __forceinline__ Frag own_rows(Frag f) {
  exchange(f.q[0], f.q[1]);
  exchange(f.q[2], f.q[3]);
  return f;
}
// either of the two; PAIRS: two lanes a row
template <bool PAIRS>
__device__ __forceinline__ Frag gather_rows(__amdgpu_buffer_rsrc_t rin, bool on, uint32_t base, int lane, uint32_t piece, bool full) {
  return PAIRS ? gather_pairs(rin, on, base, piece, full) : gather_chunk(rin, on, base, lane >> 5, full);
}
template <bool PAIRS>
__device__ __forceinline__ Frag rows_of(const Frag &f) {
  return PAIRS ? own_rows(f) : f;
}
// weight tile `tile` of the filter (on false: zeros)
template <bool PW>
__device__ __forceinline__ WFrag<PW> load_wtile(__amdgpu_buffer_rsrc_t rw, int tile, bool on, uint32_t lane16) {
  const uint32_t soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)tile * (uint32_t)wt_bytes(PW)));
  WFrag<PW> f;
  if constexpr (PW) {
    // (half s, channels h * 8 ..: quarters 2h and 2h + 1, there at lane s * 32 + column)
    const uint32_t voff = on ? (lane16 & 512u) * 4u + (lane16 & 511u) : BUF_OOB;
#pragma unroll
    for (int i = 0; i < 4; i++) f.q[i] = buf_load16(rw, voff + (i >> 1) * 512u + (i & 1) * 1024u, soff);
  } else {
    const uint32_t voff = on ? lane16 : BUF_OOB;
#pragma unroll
    for (int i = 0; i < 6; i++)
      f.s[i / 3].p[i % 3] = __builtin_bit_cast(u32x4, buf_load16(rw, voff + 1024u * (i & 3), soff + (i >= 4 ? 4096u : 0u)));
  }
  return f;
}

// sums += the products of a tile's rows with output block nb in plain fp32 (v_mfma_f32_32x32x2_f32), offsets and channels
// ascending: what repair_sums falls back to.  id_of(k): input row of offset k of tile row lane & 31, -1: none.  A row
// takes no part in an offset that it does not have (its zeros would turn an infinite weight into NaN).
// Cold, so it waits for every load; but one NaN of a scan reaches whole scales, which then pass through it: 32 -> 32 at
// 500k sites 0.15 ms finite, 0.34 all NaN (element by element in scalar code: 12.9), 64 -> 64 at 500k 0.42 and 1.25 (54.5),
// 96 -> 96 at 10k 0.07 and 0.21 (3.7).
template <bool PW, class Ids>
__device__ __forceinline__ void add_plain_products(f16v &sums, const Ids &id_of, int K, __amdgpu_buffer_rsrc_t rin,
                                                   uint32_t ld4, __amdgpu_buffer_rsrc_t rw, int Cin, int nch, int nbtp,
                                                   int nb) {
  const int lane = lane_again(), h = lane >> 5;
#pragma unroll 1
  for (int k = 0; k < K; k++) {
    const int src = id_of(k);
    const unsigned have = (unsigned)__ballot(src >= 0) >> (4 * h);  // (the two half-waves agree; bit of this lane's rows)
    if (!__any(have != 0)) continue;
    const f16v before = sums;
#pragma unroll 1
    for (int c16 = 0; c16 * 16 < Cin; c16++) {
      const uint32_t voff = src >= 0 ? (uint32_t)src * ld4 + (uint32_t)(c16 * 64 + h * 32) : BUF_OOB;
      const float4 lo = buf_load16(rin, voff, 0), hi = buf_load16(rin, voff + 16u, 0);
      const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      const int tile = (k * nch + (c16 >> 1)) * nbtp + nb;
      const uint32_t soff = (uint32_t)__builtin_amdgcn_readfirstlane(
          (int)((uint32_t)tile * (uint32_t)wt_bytes(PW) + (uint32_t)((c16 & 1) * (PW ? 512 : 3072))));
      float wv[8];
      if constexpr (PW) {
        const uint32_t wo = (uint32_t)(h * 2048 + (lane & 31) * 16);
        const float4 wlo = buf_load16(rw, wo, soff), whi = buf_load16(rw, wo + 1024u, soff);
        const float t[8] = {wlo.x, wlo.y, wlo.z, wlo.w, whi.x, whi.y, whi.z, whi.w};
#pragma unroll
        for (int j = 0; j < 8; j++) wv[j] = t[j];
      } else {
        u32x4 p[3];
#pragma unroll
        for (int i = 0; i < 3; i++) p[i] = __builtin_bit_cast(u32x4, buf_load16(rw, (uint32_t)lane * 16u + 1024u * i, soff));
#pragma unroll
        for (int j = 0; j < 8; j++) {
          unsigned q[3];
#pragma unroll
          for (int i = 0; i < 3; i++) q[i] = j & 1 ? p[i][j >> 1] >> 16 : p[i][j >> 1] & 0xFFFFu;
          wv[j] = weight_of(q[0], q[1], q[2]);
        }
      }
#pragma unroll
      for (int j = 0; j < 8; j++)
        sums = __builtin_amdgcn_mfma_f32_32x32x2f32(x[j], wv[j], sums, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 16; v++) sums[v] = have & (1u << (8 * (v >> 2) + (v & 3))) ? sums[v] : before[v];
  }
}

// The first six 64-byte lines of the kernel's arguments, asked for at once and waited for once.  They are in no cache when a
// launch begins, and the compiler loads them where they are used: a trip to memory per line, one after the other.  (U-Net of
// 16 channels on 6k voxels 577 -> 567 us, of 32 on 150k 2170 -> 2130.  The kernels whose blocks stay for many tiles gain
// nothing.)
__device__ __forceinline__ void request_six_lines_of_arguments() {
  const __attribute__((address_space(4))) uint32_t *a =
      (const __attribute__((address_space(4))) uint32_t *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" ::"s"(a[0]), "s"(a[16]), "s"(a[32]), "s"(a[48]), "s"(a[64]), "s"(a[80]));
}

// The rows of a tile: residual sum, the raw rows, the batch norm's rows - whole passes over the sixteen rows of a lane, so
// that nothing branches per row.  Rows that do not exist (my_row < 0) go out of range.
__device__ __forceinline__ void element_offsets(int my_row, uint32_t ld4, uint32_t (&off)[16]) {
  int o[16];
  rows_of_elements((int)(my_row >= 0 ? __umul24((unsigned)my_row, ld4) : BUF_OOB), o);
  const uint32_t col4 = (uint32_t)(lane_again() & 31) * 4u;
#pragma unroll
  for (int v = 0; v < 16; v++) off[v] = (uint32_t)o[v] + col4;
}
// block: the first column (a multiple of 32); on: this lane's column exists
__device__ __forceinline__ void store_tile(f16v &sum, int my_row, int block, bool on, __amdgpu_buffer_rsrc_t rout,
                                           uint32_t ldo4, __amdgpu_buffer_rsrc_t rout2, uint32_t ld24,
                                           __amdgpu_buffer_rsrc_t rres, uint32_t ldr4, float ew, float eb, float leak,
                                           bool has_out, bool has_out2, bool has_res) {
  uint32_t off[16];
  if (has_res) {
    element_offsets(my_row, ldr4, off);
    if (on) {
      float rv[16];
#pragma unroll
      for (int v = 0; v < 16; v++)
        rv[v] = __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(rres, (int)off[v], block * 4, 0));
      __builtin_amdgcn_sched_barrier(0);  // (all of them requested before the first is waited for)
#pragma unroll
      for (int v = 0; v < 16; v++) sum[v] += rv[v];
    }
    __builtin_amdgcn_sched_barrier(0);  // (the sums stay above the stores)
  }
  if (has_out) {
    element_offsets(my_row, ldo4, off);
    if (on) {
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const float x = sum[v];  // (a bit cast applied to the vector element itself reads element 0)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), rout, (int)off[v], block * 4, 0);
      }
    }
  }
  if (has_out2) {
    // fused batch norm + leaky ReLU
    element_offsets(my_row, ld24, off);
    if (on) {
#pragma unroll
      for (int v = 0; v < 16; v++) {
        const float y = fmaf(sum[v], ew, eb);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y * ((y > 0.0f) ? 1.0f : leak)), rout2, (int)off[v], block * 4, 0);
      }
    }
  }
}

// Narrow 3^3 layers (fewer than 64 input channels, so one or two chunks): a row's sum is formed as two partial sums, of the even
// offsets and of the odd ones - each ascending, with one chunk the odd ones beginning with the centre, whose weights the
// filter-in-LDS kernel has no room for -, the bias in the former, added at the end.  So a tile can go to one wavefront, which
// forms them one after the other, or to two: what a launch of few tiles lasts is its longest wavefront.
constexpr unsigned EVEN_OFFSETS = 0x5555555u, ODD_OFFSETS = 0x2AAAAAAu;  // of 27
__device__ __forceinline__ int pick_offset(unsigned rest, bool centre_first) {
  return centre_first && ((rest >> 13) & 1u) ? 13 : __builtin_ctz(rest);
}

// S == 1: every wavefront of the block owns a tile and walks all of its filter offsets (a narrow 3^3 layer: partial sum by
//         partial sum).
// S  > 1: the S wavefronts of a block share ONE tile (and NB output blocks of it); the (offset, channel chunk) items are dealt
//         out round robin and the partial sums are added in wavefront order at the end.  This is for
//         the coarse scales of a U-Net, where a layer has a handful of tiles but hundreds of
//         channels and a single wavefront would run tens of thousands of dependent MFMAs.  Which
//         terms a wavefront sums depends on k and ch only, never on the tile a row happens to sit in.
//         How a row's sum is grouped depends on the layer shape alone: S * G partial sums of a wide
//         layer, two of a narrow one, whether one wavefront forms both (S == 1) or each has its own (S == 2).
//         With gridDim.z = G > 1 the deal goes over S * G wavefronts in G blocks (different
//         compute units): a coarse scale has so few tiles that the matrix cores of the few
//         units holding them would bound the layer.
template <int NB, int K, int MODE, int S, bool PW, bool PAIRS>
__global__ __launch_bounds__((S == 1 ? CONV_WAVES : S) * 64, S == 8 && PW ? 4 /* two blocks a compute unit */ : NB == 3 || (NB == 2 && K == 27) ? 2 : 1) void conv_mfma_kernel(
    const float *__restrict__ in, int64_t ld_in, float *__restrict__ out, int64_t ld_out,
    const float *__restrict__ Wp, const float *__restrict__ bias, const int32_t *__restrict__ map0,
    const int32_t *__restrict__ map1, const int32_t *__restrict__ rows,
    const int32_t *__restrict__ d_n_rows, int64_t n_rows, int Cin, int Cout, int nbtp,
    const uint8_t *__restrict__ tile_flags, uint32_t in_bytes, uint32_t wp_bytes, BnEpilogue ep,
    float *__restrict__ part, int32_t *__restrict__ pcount, TilePlan plan) {
  constexpr int WAVES = S == 1 ? CONV_WAVES : S;
  constexpr int NSTAGE = (TILE_M * K + 64 * S - 1) / (64 * S);
  __shared__ int nbl[S == 1 ? WAVES : 1][NSTAGE * 64 * S];  // (whole passes: the last one's store needs no condition)
  __shared__ float red[S > 1 ? S : 1][S > 1 ? NB * 16 * 64 : 1];  // (slot S - 1: only when all wavefronts share the tail)
  __shared__ unsigned wmask[S];
  request_six_lines_of_arguments();  // (they take 360 bytes)
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  // (the wavefront's number as a scalar: the item cursor below then runs on the scalar unit)
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int r = lane & 31, h = lane >> 5;
  // (with a tile schedule the blocks of a split launch take the tiles by falling cost: blocks go to the
  // compute units round robin, so every unit then holds a mix of expensive and cheap tiles)
  // Which (tile slot, output block, share of the split) this block works on.  Split launches with a
  // tile schedule renumber their blocks: the hardware hands out blocks in the order x, y, z, round robin
  // over the compute units, so block L goes - all blocks being resident at once - to unit L mod CUS.
  // Ranked by cost (tile slot major: the output blocks and shares of a tile cost the same), the first CUS
  // blocks take ranks in order, the next CUS in reverse order and so on in turns, so that the compute unit
  // that drew the most expensive block of one turn gets the cheapest of the next.
  unsigned bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  if (S > 1 && MODE == MAP_NBR && K == 27 && plan.map != nullptr && plan.sched != nullptr) {
    const unsigned CUS = plan.cus;
    const unsigned gyz = gridDim.y * gridDim.z;
    const unsigned total = (unsigned)((n + TILE_M - 1) / TILE_M) * gyz;
    const unsigned L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    if (L >= total) return;  // (launches are sized by an upper bound of the row count)
    const unsigned rnd = L / CUS, pos = L % CUS, m = min(CUS, total - rnd * CUS);
    const unsigned R = rnd * CUS + ((rnd & 1u) ? m - 1 - pos : pos);
    bx = R / gyz;
    const unsigned rem = R - bx * gyz;
    by = rem / gridDim.z;
    bz = rem - by * gridDim.z;
  }
  const int64_t slot = S == 1 ? (int64_t)bx * WAVES + wave : (int64_t)bx;
  const bool by_cost = MODE == MAP_NBR && K == 27 && plan.map != nullptr && plan.sched != nullptr && slot * TILE_M < n;
  const int64_t t0 = (by_cost ? (int64_t)plan.sched[slot] : slot) * TILE_M;
  const int cb0 = by * NB;  // first output-channel block of this column group
  const int nch = conv_nch(Cin);
  // the items of a tile are dealt to S wavefronts in each of G blocks; gridDim.z = GZ holds G blocks
  // per source (two sources: the blocks from G on gather from the second one, through its own map)
  const int GZ = S == 1 ? 1 : (int)gridDim.z;
  const bool second = S > 1 && ep.src2_in != nullptr && (int)bz >= GZ / 2;
  const float *const in0 = in, *const bias0 = bias;  // (the first source, whichever this block reads)
  const int64_t ld_in0 = ld_in;
  const uint32_t in_bytes0 = in_bytes;
  const int32_t *const map00 = map0;
  const int G = (S > 1 && ep.src2_in != nullptr) ? GZ / 2 : GZ, ST = S * G;
  const int ws = wave * G + (S == 1 ? 0 : (int)bz - (second ? G : 0));
  if (second) {
    in = ep.src2_in;
    ld_in = ep.src2_ld;
    in_bytes = (uint32_t)(ep.src2_rows * ep.src2_ld * 4);
    map0 = ep.src2_map;
    bias = nullptr;
  }

  // blocks beyond the row count leave at once (launches are sized by an upper bound of it)
  if ((S == 1 ? (int64_t)bx * WAVES : (int64_t)bx) * TILE_M >= n) return;
  // a tile is skipped when it lies beyond the row count or, with tile flags, is not marked: the whole block (S > 1) or one
  // wavefront, and barriers are among the wavefronts of one tile only
  if (t0 >= n || (tile_flags && !tile_flags[t0 >> 5])) return;
  // Up to the first gather a small launch does little but wait for memory that no cache holds yet, so nothing here loads
  // under a condition of its own (each such load would be waited for before the next) and what needs no map goes first:
  // the bias and the per-channel scale / shift of the fused batch norms, zero beyond Cout.  Then the row ids, the tile's
  // slice of the neighbour map and its offsets in one trip.  (3^3 layers of 16, 32 and 48 channels at 6k, 1.5k and 400
  // sites 12.3 -> 10.7, 13.7 -> 12.2 and 19.1 -> 17.3 us, with the arguments asked for at once.)
  float bias_of[NB], ew[NB], eb[NB], sw[NB], sb[NB];
  {
    const uint32_t width = (uint32_t)Cout * 4u;
    const bool side = MODE == MAP_PARENT && ep.side_in;
    const __amdgpu_buffer_rsrc_t rbias = make_rsrc(bias, bias && (S == 1 || ws == 0) ? width : 0u),
                                 rew = make_rsrc(ep.w, ep.out2 ? width : 0u), reb = make_rsrc(ep.b, ep.out2 ? width : 0u),
                                 rsw = make_rsrc(ep.side_w, side ? width : 0u), rsb = make_rsrc(ep.side_b, side ? width : 0u);
    auto at = [&](__amdgpu_buffer_rsrc_t from, int b) {
      return __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(from, ((cb0 + b) * 32 + r) * 4, 0, 0));
    };
#pragma unroll
    for (int b = 0; b < NB; b++) {
      bias_of[b] = at(rbias, b);
      ew[b] = at(rew, b);
      eb[b] = at(reb, b);
      sw[b] = sb[b] = 0.0f;
      if (MODE == MAP_PARENT) {
        sw[b] = at(rsw, b);
        sb[b] = at(rsb, b);
      }
    }
  }
  const bool in_range = t0 + r < n;
  int listed = (int)min(t0 + r, n - 1), my_row;
  if (rows) listed = rows[listed];

  // Stage the tile's slice of the neighbour map in LDS and find the offsets it uses.  With a tile plan (the map transposed
  // into processing order, one 128-byte run per (offset, tile), and the offsets of every tile) the loads are coalesced, need
  // no row id and the LDS copy is offset-major.
  const bool planned = MODE == MAP_NBR && K == 27 && plan.map != nullptr;
  int *nl = nbl[S == 1 ? wave : 0];
  unsigned mymask = 0;
  int staged[NSTAGE];
  if (planned) {
    // (the launch checked that 32-bit offsets reach all of the plan; entries beyond the 27th offset are out of range)
    const uint32_t pld4 = (uint32_t)plan.ld * 4u;
    const __amdgpu_buffer_rsrc_t rplan = make_rsrc(plan.map, 27u * pld4);
    const uint32_t first = (uint32_t)t0 * 4u + (uint32_t)r * 4u + (uint32_t)h * pld4;
    mymask = plan.tmask[t0 >> 5];
#pragma unroll
    for (int i = 0; i < NSTAGE; i++)  // entry e = k * 32 + row, e = (i * S + wave) * 64 + lane
      staged[i] = (int)__builtin_amdgcn_raw_buffer_load_b32(rplan, (int)(first + (uint32_t)((S == 1 ? i : i * S + wave) * 2) * pld4), 0, 0);
    asm volatile("" : "+v"(listed));  // (not waited for until the map is on its way)
    my_row = in_range ? listed : -1;
#pragma unroll
    for (int i = 0; i < NSTAGE; i++) nl[(S == 1 ? i : i * S + wave) * 64 + lane] = staged[i];
  } else {
    my_row = in_range ? listed : -1;
    // (rows that do not exist read the map of one that does)
    const int some_row = max(__builtin_amdgcn_readfirstlane(my_row), 0);
    // (a row of a deconvolution has one input row, at one offset)
    int my_offset = -1, my_parent = -1;
    if (MODE == MAP_PARENT) {
      my_offset = map1[my_row < 0 ? some_row : my_row];
      my_parent = map0[my_row < 0 ? some_row : my_row];
    }
    if constexpr (MODE == MAP_NBR && K == 27) {
      // A lane stays with one offset, half a wavefront with a row: the row ids come from their lanes through the scalar
      // unit, and the offsets in use are what the ballots of all rows have in common, without a reduction over the lanes.
      constexpr int PAIRS_OF_ROWS = TILE_M / (2 * S);
      const int kk = min(r, K - 1);
      int v[PAIRS_OF_ROWS];
#pragma unroll
      for (int i = 0; i < PAIRS_OF_ROWS; i++) {
        const int rr = (S == 1 ? i : i * S + wave) * 2;
        const int ra = __builtin_amdgcn_readlane(my_row, rr), rb = __builtin_amdgcn_readlane(my_row, rr + 1), rid = h ? rb : ra;
        v[i] = map0[(int64_t)(rid < 0 ? some_row : rid) * K + kk];
      }
      uint64_t used = 0;
#pragma unroll
      for (int i = 0; i < PAIRS_OF_ROWS; i++) {
        const int rr = (S == 1 ? i : i * S + wave) * 2;
        const int ra = __builtin_amdgcn_readlane(my_row, rr), rb = __builtin_amdgcn_readlane(my_row, rr + 1);
        if ((h ? rb : ra) < 0) v[i] = -1;
        used |= __ballot(v[i] >= 0);
      }
      mymask = (unsigned)(used | used >> 32) & 0x7FFFFFFu;
      if (r < K) {
#pragma unroll
        for (int i = 0; i < PAIRS_OF_ROWS; i++) nl[((S == 1 ? i : i * S + wave) * 2 + h) * K + r] = v[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < NSTAGE; i++) {
        const int e = (S == 1 ? i : i * S + wave) * 64 + lane;
        const int rr = (e / K) & (TILE_M - 1), kk = e - (e / K) * K;
        const int rid = __shfl(my_row, rr, 64);
        if (MODE == MAP_NBR) {
          const int v = map0[(int64_t)(rid < 0 ? some_row : rid) * K + kk];
          staged[i] = rid < 0 || e >= TILE_M * K ? -1 : v;
        } else if (MODE == MAP_IDENTITY) {
          staged[i] = e < TILE_M * K ? rid : -1;
        } else {
          const int offset_of = __shfl(my_offset, rr, 64), parent_of = __shfl(my_parent, rr, 64);
          staged[i] = rid >= 0 && offset_of == kk ? parent_of : -1;
        }
      }
#pragma unroll
      for (int i = 0; i < NSTAGE; i++) {
        const int e = (S == 1 ? i : i * S + wave) * 64 + lane;
        nl[e] = staged[i];
        mymask |= (staged[i] >= 0 ? 1u : 0u) << (e % K);
      }
      // (every entry of a lane is at the same offset)
      static_assert((MODE == MAP_NBR && K == 27) || 64 % K == 0, "");
      uint64_t some = __ballot(mymask != 0);
#pragma unroll
      for (int d = 32; d >= K; d >>= 1) some |= some >> d;
      mymask = (unsigned)some & ((1u << K) - 1u);
    }
    if (S > 1 && lane == 0) wmask[wave] = mymask;
  }
  if (S > 1) {
    __syncthreads();
  } else {
    // (a wavefront's own entries)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // Split launches: what the tail of this wavefront will read besides the sums - the other operand of a
  // folded element-wise sum, the saved rows of a residual frame's batch norm - is asked for here, for
  // the rows the wavefront finishes, so that the main loop hides these loads.  (Rows and columns that do
  // not exist get the values of ones that do, and are not written.)
  constexpr int NVP = S > 1 ? 16 / S : 1;
  float pre_res[NB][NVP], pre_pin[NVP], pre_pout[NVP];
  int pre_pe[NVP];
  if (S > 1) {
    const int c = cb0 * 32 + r;
#pragma unroll
    for (int j = 0; j < NVP; j++) {
      pre_pe[j] = -1;
      pre_pin[j] = pre_pout[j] = 0.0f;
#pragma unroll
      for (int b = 0; b < NB; b++) pre_res[b][j] = 0.0f;
    }
    if (ep.res) {
#pragma unroll
      for (int j = 0; j < NVP; j++) {
        const int v = wave * NVP + j, row = __shfl(my_row, 8 * (v >> 2) + 4 * h + (v & 3), 64);
#pragma unroll
        for (int b = 0; b < NB; b++) pre_res[b][j] = ep.res[(int64_t)max(row, 0) * ep.ldr + min(c + b * 32, Cout - 1)];
      }
    }
    if (MODE == MAP_NBR && K == 27 && ep.pre_exist) {
      const int pe = ep.pre_exist[max(my_row, 0)], my_pe = my_row < 0 ? -1 : pe;
#pragma unroll
      for (int j = 0; j < NVP; j++) {
        const int v = wave * NVP + j;
        pre_pe[j] = __shfl(my_pe, 8 * (v >> 2) + 4 * h + (v & 3), 64);
      }
      const uint64_t saved = __ballot(my_pe >= 0);
      if (saved) {  // (the saved matrices may have no rows at all)
        const int some_saved = __builtin_amdgcn_readlane(my_pe, __builtin_ctzll(saved)), cc = min(c, Cout - 1);
#pragma unroll
        for (int j = 0; j < NVP; j++) {
          const int64_t row = pre_pe[j] < 0 ? some_saved : pre_pe[j];
          pre_pin[j] = ep.pre_in[row * ep.ld_pin + cc];
          pre_pout[j] = ep.pre_out[row * ep.ld_pout + cc];
        }
      }
    }
  }
  // Offsets some row of the tile uses.  With S wavefronts per tile, the (offset k, chunk ch)
  // items are dealt out by (k * nch + ch) % S: wavefront w takes, of offset k, the chunks
  // ch0(k), ch0(k) + S, ... with ch0(k) = (w - k * nch) mod S.  The deal depends on k, ch and
  // the layer shape only, so a row's sum is formed the same way whatever tile it sits in.
  unsigned rest;  // offsets that hold at least one item of this wavefront
  int nitems = 0;
  if (S == 1) {
    rest = (unsigned)__builtin_amdgcn_readfirstlane((int)mymask);
    nitems = __builtin_popcount(rest) * nch;
  } else {
    unsigned act = mymask;
    if (!planned) {
#pragma unroll
      for (int w = 0; w < S; w++) act |= wmask[w];
    }
    act = (unsigned)__builtin_amdgcn_readfirstlane((int)act);
    // (lane k looks at offset k: ballots instead of a scalar loop over the offsets; an offset holds nch / ST items of this
    // wavefront, one more where c0 is below the remainder)
    // (two wavefronts: a narrow layer's two partial sums)
    const int c0 = S == 2 ? ((ws ^ lane) & 1) * nch : (ws - lane * nch) & (ST - 1);
    const bool has = lane < K && ((act >> (lane & 31)) & 1u) && c0 < nch;
    rest = (unsigned)__ballot(has);
    if (S == 2) {
      nitems = __builtin_popcount(rest) * nch;
    } else {
      const unsigned more = (unsigned)__ballot(has && c0 < (nch & (ST - 1)));
      nitems = __builtin_popcount(act) * (nch >> __builtin_ctz(ST)) + __builtin_popcount(more);
    }
  }

  // (one wavefront, two partial sums: the running one and the finished one.  With three output blocks a wavefront the finished
  // one waits in LDS: in registers it goes over the 256 that leave a second wavefront per SIMD, and the 34 that spilled cost
  // more than the loads here or, without a cap, that wavefront: 48 -> 96 at 150k sites 232, 185 and 155 us, 16 -> 96 112, 91 and 75.
  // Two and four blocks take the same time either way.)
  constexpr bool SEQ = S == 1 && K == 27 && MODE == MAP_NBR, HELD = SEQ && NB == 3;
  __shared__ float held[HELD ? WAVES : 1][HELD ? NB * 16 * 64 : 1];
  Sum sums[NB];
  f16v total[SEQ && !HELD ? NB : 1];
  int cur = 0;  // the partial sum in sums
#pragma unroll
  for (int b = 0; b < NB; b++) sum_start(sums[b], bias_of[b]);

  if (rest) {
    // Work items of this tile: (active offset k, 32-channel chunk ch), offsets ascending, chunks
    // inside.  A cursor walks them with scalar selects only (no branches: a branchy iterator
    // splits the loop body into many blocks and the load/MFMA overlap below is lost).  Past the
    // last item it yields k = -1, and loads for such an item are sent out of range: they
    // return zeros and move no data.
    struct Cursor {
      int k, ch, p;
      unsigned rest;
    };
    const bool centre_first = K == 27 && nch == 1;
    auto ch0 = [&](int k) -> int { return S <= 2 ? 0 : ((ws - k * nch) & (ST - 1)); };
    auto step = [&](const Cursor &c) -> Cursor {
      Cursor n = c;
      if (SEQ) {
        const bool next = c.ch + 1 >= nch, over = next && c.rest == 0 && c.p == 0;
        const unsigned left = over ? rest & ODD_OFFSETS : c.rest;
        const int nk = left ? pick_offset(left, centre_first) : -1;
        n.ch = next ? 0 : c.ch + 1;
        n.p = over ? 1 : c.p;
        n.k = next ? nk : c.k;
        n.rest = next ? left & ~(1u << (nk & 31)) : c.rest;
        return n;
      }
      const int stride = S == 2 ? 1 : ST;
      const bool wrap = c.ch + stride >= nch;
      const int nk = c.rest ? __builtin_ctz(c.rest) : -1;
      n.ch = wrap ? ch0(nk) : c.ch + stride;
      n.k = wrap ? nk : c.k;
      n.rest = wrap ? (c.rest & (c.rest - 1)) : c.rest;
      return n;
    };
    Cursor first;
    if (SEQ) {
      first.k = first.p = 0;
      first.ch = nch;
      first.rest = rest & EVEN_OFFSETS;
      first = step(first);
    } else {
      first.k = pick_offset(rest, centre_first);
      first.ch = ch0(first.k);
      first.p = 0;
      first.rest = rest & ~(1u << first.k);
    }

    const __amdgpu_buffer_rsrc_t rin = make_rsrc(in, in_bytes), rw = make_rsrc(Wp, wp_bytes);
    const uint32_t ld4 = (uint32_t)ld_in * 4u, lane16 = (uint32_t)lane * 16u, piece = pair_piece(lane);
    auto gather = [&](const Cursor &c) -> Frag {
      const int kk = c.k < 0 ? 0 : c.k;
      const int src = nl[planned ? kk * TILE_M + r : r * K + kk];
      const bool on = c.k >= 0 && src >= 0, full = Cin - c.ch * 32 >= 32;
      const uint32_t base = (uint32_t)src * ld4 + (uint32_t)(c.ch * 128);
      return gather_rows<PAIRS>(rin, on, base, lane, piece, full);
    };
    auto wload = [&](const Cursor &c, int b) -> WFrag<PW> {
      return load_wtile<PW>(rw, ((c.k < 0 ? 0 : c.k) * nch + c.ch) * nbtp + cb0 + b, c.k >= 0, lane16);
    };

    // Pipeline: while item t runs on the matrix cores, the gathers of item t+1 are in flight; so are its weights when a
    // wavefront owns a single output block (otherwise the weight tiles of the (item, block) sequence are fetched one step
    // ahead).  Register slots are compile-time (the body is unrolled over the two turns of the rings) because
    // copying a fragment would wait for the load that fills it.  Every load is issued
    // unconditionally: a load under a branch would force the wait before the MFMAs to drain
    // all outstanding loads.  The sched_barrier / memory-clobber pairs keep the loads above the
    // MFMAs they overlap and their consumers below.
    // (Rings of three and four items spill or leave room for fewer wavefronts; a list of the items in LDS instead of the
    // cursor, and the next item split between the MFMAs of this one, measured the same at 32 channels and slower above.)
    Frag g[2];
    WFrag<PW> bw[2];
    g[0] = gather(first);
    bw[0] = wload(first, 0);
    Cursor c0 = first, c1 = step(first);  // item on the matrix cores and its successor
    auto turn = [&](auto U) -> bool {
      constexpr int u = decltype(U)::value;
      g[u ^ 1] = gather(c1);
      if constexpr (NB == 1) bw[u ^ 1] = wload(c1, 0);
      const bool full = Cin - c0.ch * 32 >= 32;
      if (SEQ && c0.p != cur) {
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const f16v part = sum_of(sums[b]);
#pragma unroll
          for (int v = 0; v < 16; v++) {
            if constexpr (HELD) held[wave][(b * 16 + v) * 64 + lane] = part[v];
            else total[b][v] = part[v];
          }
          sum_start(sums[b], 0.0f);
        }
        cur = c0.p;
      }
      Parts as[2];
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const int nn = u * NB + b;
        if constexpr (NB > 1) bw[(nn + 1) & 1] = (b + 1 < NB) ? wload(c0, b + 1) : wload(c1, 0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (b == 0) {
          const Frag a = rows_of<PAIRS>(g[u]);
          as[0] = split8(a.q[0], a.q[1]);
          as[1] = split8(a.q[2], a.q[3]);
        }
        mac_chunk(sums[b], as, bw[NB == 1 ? u : nn & 1], full);
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      c0 = c1;
      c1 = step(c1);
      return --nitems > 0;
    };
    while (turn(std::integral_constant<int, 0>()) && turn(std::integral_constant<int, 1>())) {
    }
  }

  // input row of this lane's output row at offset k (cold: from memory, through a source's own map)
  auto id_at = [&](const int32_t *map, int k) -> int {
    if (planned) return plan.map[(int64_t)k * plan.ld + t0 + (lane_again() & 31)];
    if (my_row < 0) return -1;
    return MODE == MAP_NBR ? map[(int64_t)my_row * K + k] : MODE == MAP_IDENTITY ? my_row : map1[my_row] == k ? map[my_row] : -1;
  };
  f16v acc[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    acc[b] = sum_of(sums[b]);
    if (SEQ && cur != 0) {
#pragma unroll
      for (int v = 0; v < 16; v++) acc[b][v] = (HELD ? held[wave][(b * 16 + v) * 64 + lane] : total[HELD ? 0 : b][v]) + acc[b][v];
    }
  }
  // (rows whose byte offsets fit 32 bits, through 24-bit multiplies, in every matrix that is written or added)
  const int64_t widest = 4 * max(max(ld_out, ep.ld2), max(ep.ldr, ep.ld_side));
  const bool fits = widest < (1 << 24) && __all(my_row < (1 << 24) && (int64_t)my_row * widest + 4 * (int64_t)Cout <= (int64_t)BUF_OOB);
  if (S == 1) {
    // (one block at a time: copies of all blocks' repeated sums would cost NB = 3 its second wavefront per SIMD, 32 -> 96 at
    // 200k sites 99 -> 124 us)
    float t = 0.0f;
#pragma unroll
    for (int b = 0; b < NB; b++) {
      unscale<16>(acc[b]);
      t = not_finite<16>(acc[b], t);
    }
    if (__builtin_expect(__any(t != t), 0)) {
#pragma unroll 1
      for (int bb = 0; bb < NB; bb++) {
        const int c = (cb0 + bb) * 32 + r;
        f16v x;
#pragma unroll
        for (int v = 0; v < 16; v++) x[v] = (bias && c < Cout) ? bias[c] : 0.0f;
        add_plain_products<PW>(x, [&](int k) { return id_at(map0, k); }, K, make_rsrc(in, in_bytes), (uint32_t)ld_in * 4u,
                           make_rsrc(Wp, wp_bytes), Cin, nch, nbtp, cb0 + bb);
#pragma unroll
        for (int b = 0; b < NB; b++) {
          if (b != bb) continue;
#pragma unroll
          for (int v = 0; v < 16; v++) acc[b][v] = is_bad(acc[b][v]) ? x[v] : acc[b][v];
        }
      }
    }
  }

  if (S > 1) {
    // Every wavefront leaves its partial sum in LDS; each then adds up - in wavefront order - and
    // finishes 16 / S of the rows of the tile, so that the tail of the block (partial sums through
    // memory, residual loads, two stores per row with a fused batch norm) is shared by all of them.
    // D layout of the 32x32 MFMA: lane holds column (lane & 31), rows 8*(v/4) + 4*(lane>>5) + (v&3).
    constexpr int NV = 16 / (S > 1 ? S : 16);
#pragma unroll
    for (int b = 0; b < NB; b++) {
#pragma unroll
      for (int v = 0; v < 16; v++) red[wave][(b * 16 + v) * 64 + lane] = acc[b][v];
    }
    __syncthreads();
    float a[NB][NV];
    int rid[NV];
#pragma unroll
    for (int j = 0; j < NV; j++) {
      const int v = wave * NV + j;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        a[b][j] = red[0][(b * 16 + v) * 64 + lane];
#pragma unroll
        for (int w = 1; w < S; w++) a[b][j] += red[w][(b * 16 + v) * 64 + lane];
      }
      rid[j] = __shfl(my_row, 8 * (v >> 2) + 4 * h + (v & 3), 64);
    }
    if (GZ > 1) {
      // The blocks of a (tile, output block) leave their sums in memory; of the wavefronts that
      // hold the same rows, the one that arrives last adds the sums in block order (so the result
      // does not depend on the arrival order), writes the rows and puts the arrival counter back to
      // zero.  Nobody waits for anybody.
      // (stores and loads of the sums go past the XCD-local L2 - device-scope atomics - so that no
      // cache write-back or invalidation is needed: a full fence flushes the whole L2 and costs
      // more than the layer)
      // Why the last arrival sees every sum.  (1) The sums are written with agent-scope atomic stores:
      // on this part such a store is not kept in the writer's XCD-local L2 but written through to the
      // level all XCDs share, and it is acknowledged from there.  (2) vmcnt(0) makes the wavefront wait
      // for those acknowledgements before it issues the counter's read-modify-write, which is performed
      // at that same shared level: a wavefront's increment is ordered after its own sums.  (3) The
      // wavefront that reads GZ - 1 back has therefore been preceded by all other increments, hence by
      // all other sums.  (4) Its loads below are issued only after that value has returned (the branch
      // depends on it; wavefronts issue in order) and are agent-scope atomic loads, which do not hit a
      // stale line of the reader's own L2.  The compiler fences pin the program order this relies on
      // (they emit no instructions).  An acquire/release pair at agent scope would say the same in the
      // language's terms but writes back and invalidates the whole L2.
      const int unit = (int)(bx * gridDim.y + by);
      float *mine = part + ((int64_t)unit * GZ + bz) * (NB * 1024) + (wave * NV) * 64 + lane;
#pragma unroll
      for (int b = 0; b < NB; b++) {
#pragma unroll
        for (int j = 0; j < NV; j++)
          __hip_atomic_store(mine + b * 1024 + j * 64, a[b][j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the stores have been acknowledged
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      int old = 0;
      if (lane == 0) old = atomicAdd(pcount + unit * S + wave, 1);
      if (__builtin_amdgcn_readfirstlane(old) != GZ - 1) return;
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      const float *all = part + (int64_t)unit * GZ * (NB * 1024) + (wave * NV) * 64 + lane;
      // (the sums of eight blocks at a time are requested together and added in block order: one trip
      // to memory per eight blocks instead of one per block)
      constexpr int GP = NB == 1 ? 8 : 4;
      for (int g0 = 0; g0 < GZ; g0 += GP) {
        float pv[GP][NB][NV];
#pragma unroll
        for (int gg = 0; gg < GP; gg++) {
          if (g0 + gg < GZ) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
#pragma unroll
              for (int j = 0; j < NV; j++)
                pv[gg][b][j] = __hip_atomic_load(all + ((g0 + gg) * NB + b) * 1024 + j * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
        }
#pragma unroll
        for (int gg = 0; gg < GP; gg++) {
          if (g0 + gg < GZ) {
#pragma unroll
            for (int b = 0; b < NB; b++) {
#pragma unroll
              for (int j = 0; j < NV; j++) a[b][j] = (g0 + gg == 0) ? pv[0][b][j] : a[b][j] + pv[gg][b][j];
            }
          }
        }
      }
      if (lane == 0) pcount[unit * S + wave] = 0;
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
    const int c = (cb0 + b) * 32 + r;
    unscale<NV>(a[b]);
    repair_sums<NV>(a[b], wave * NV, [&]() -> f16v {
      f16v t;
#pragma unroll
      for (int v = 0; v < 16; v++) t[v] = (bias0 && c < Cout) ? bias0[c] : 0.0f;
      const __amdgpu_buffer_rsrc_t rw = make_rsrc(Wp, wp_bytes);
      add_plain_products<PW>(t, [&](int k) { return id_at(map00, k); }, K, make_rsrc(in0, in_bytes0), (uint32_t)ld_in0 * 4u, rw, Cin,
                         nch, nbtp, cb0 + b);
      if (ep.src2_in)
        add_plain_products<PW>(t, [&](int k) { return id_at(ep.src2_map, k); }, K,
                           make_rsrc(ep.src2_in, (uint32_t)(ep.src2_rows * ep.src2_ld * 4)), (uint32_t)ep.src2_ld * 4u, rw, Cin, nch,
                           nbtp, cb0 + b);
      return t;
    });
    if (c >= Cout) continue;
    if (ep.res) {
#pragma unroll
      for (int j = 0; j < NV; j++) a[b][j] += pre_res[b][j];
    }
    float sv[NV];
    if (MODE == MAP_PARENT && ep.side_in) {
#pragma unroll
      for (int j = 0; j < NV; j++) sv[j] = rid[j] >= 0 ? ep.side_in[(int64_t)rid[j] * ep.ld_side + c] : 0.0f;
      __builtin_amdgcn_sched_barrier(0);  // (all loads above the stores)
    }
    if (MODE == MAP_NBR && K == 27 && ep.pre_exist && ep.out2) {
      // batch norm of a residual frame, with the saved input and output of the rows that existed
#pragma unroll
      for (int j = 0; j < NV; j++) {
        if (rid[j] < 0) continue;
        if (out) out[(int64_t)rid[j] * ld_out + c] = a[b][j];
        const float o = fmaf(a[b][j], ew[b], eb[b]);
        const float y =
            pre_pe[j] >= 0 ? sub_exact(leaky(fmaf(pre_pin[j], ew[b], o), ep.leak), pre_pout[j]) : leaky(o, ep.leak);
        ep.out2[(int64_t)rid[j] * ep.ld2 + c] = y;
      }
      continue;
    }
    if (!(MODE == MAP_PARENT && ep.side_in) && fits) {
      const uint32_t c4 = (uint32_t)c * 4u;
      if (out) {
        const __amdgpu_buffer_rsrc_t rout = make_rsrc(out, BUF_OOB);
#pragma unroll
        for (int j = 0; j < NV; j++)
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(a[b][j]), rout,
                                                (int)(rid[j] < 0 ? BUF_OOB : __umul24((unsigned)rid[j], (uint32_t)ld_out * 4u) + c4), 0, 0);
      }
      if (ep.out2) {
        const __amdgpu_buffer_rsrc_t rout2 = make_rsrc(ep.out2, BUF_OOB);
#pragma unroll
        for (int j = 0; j < NV; j++) {
          const float y = fmaf(a[b][j], ew[b], eb[b]);  // fused batch norm + leaky ReLU
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y * ((y > 0.0f) ? 1.0f : ep.leak)), rout2,
                                                (int)(rid[j] < 0 ? BUF_OOB : __umul24((unsigned)rid[j], (uint32_t)ep.ld2 * 4u) + c4), 0, 0);
        }
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < NV; j++) {
      if (rid[j] < 0) continue;
      if (out) out[(int64_t)rid[j] * ld_out + c] = a[b][j];
      if (ep.out2) {
        const float y = fmaf(a[b][j], ew[b], eb[b]);  // fused batch norm + leaky ReLU
        ep.out2[(int64_t)rid[j] * ep.ld2 + c] = y * ((y > 0.0f) ? 1.0f : ep.leak);
      }
      if (MODE == MAP_PARENT && ep.side_in) {
        const float y = fmaf(sv[j], sw[b], sb[b]);  // batch norm of the other half of a joined matrix
        ep.side_out[(int64_t)rid[j] * ep.ld2 + c] = y * ((y > 0.0f) ? 1.0f : ep.leak);
      }
    }
    }
    return;
  }

  // Such rows go out in whole passes without a branch per row: with one, the 16 stores of every matrix
  // and block, and the loads of a joined matrix's other half, went one by one.  A deconvolution's map (two words a row) is
  // loaded once and handed round for the same reason, not 8 times under a condition.  Deconvolutions of 6k, 37k and 150k
  // sites to one block of columns 15.9 -> 7.5, 17.6 -> 8.9 and 54 -> 29 us, of 1k sites to two 20.9 -> 11.9.
  {
    if (__builtin_expect(fits, 1)) {
      const __amdgpu_buffer_rsrc_t rout = make_rsrc(out, out ? BUF_OOB : 0u), rout2 = make_rsrc(ep.out2, ep.out2 ? BUF_OOB : 0u),
                                   rres = make_rsrc(ep.res, ep.res ? BUF_OOB : 0u);
      const uint32_t ldo4 = (uint32_t)ld_out * 4u, ld24 = (uint32_t)ep.ld2 * 4u, ldr4 = (uint32_t)ep.ldr * 4u;
#pragma unroll
      for (int b = 0; b < NB; b++) {
        const int block = (cb0 + b) * 32;
        const bool on = block + r < Cout;
        float sv[16];
        if (MODE == MAP_PARENT && ep.side_in) {
          // (the other half of a joined matrix: asked for before this block's rows are stored)
          uint32_t off[16];
          element_offsets(my_row, (uint32_t)ep.ld_side * 4u, off);
          const __amdgpu_buffer_rsrc_t rside = make_rsrc(ep.side_in, BUF_OOB);
#pragma unroll
          for (int v = 0; v < 16; v++)
            sv[v] = __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(rside, (int)(on ? off[v] : BUF_OOB), block * 4, 0));
          __builtin_amdgcn_sched_barrier(0);
        }
        store_tile(acc[b], my_row, block, on, rout, ldo4, rout2, ld24, rres, ldr4, ew[b], eb[b], ep.leak, out != nullptr,
                   ep.out2 != nullptr, ep.res != nullptr);
        if (MODE == MAP_PARENT && ep.side_in) {
          uint32_t off[16];
          element_offsets(my_row, ld24, off);
          const __amdgpu_buffer_rsrc_t rto = make_rsrc(ep.side_out, BUF_OOB);
          if (on) {
#pragma unroll
            for (int v = 0; v < 16; v++) {
              const float y = fmaf(sv[v], sw[b], sb[b]);
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y * ((y > 0.0f) ? 1.0f : ep.leak)), rto, (int)off[v], block * 4, 0);
            }
          }
        }
      }
      return;
    }
  }

  // D layout of the 32x32 MFMA: lane holds column (lane & 31), rows 8*(v/4) + 4*(lane>>5) + (v&3).
  // All row ids are fetched from their lanes first, then the stores go out back to back.
  int rid[16];
  rows_of_elements(my_row, rid);
  // (the values of the residual input are all fetched before the first store: a store may alias them
  // as far as the compiler knows, and loads issued between the stores would wait one by one)
  if (ep.res) {
    float rv[NB][16];
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const float *rp = ep.res + (int64_t)(rid[v] < 0 ? 0 : rid[v]) * ep.ldr + cb0 * 32 + r;
#pragma unroll
      for (int b = 0; b < NB; b++) rv[b][v] = (rid[v] >= 0 && (cb0 + b) * 32 + r < Cout) ? rp[b * 32] : 0.0f;
    }
#pragma unroll
    for (int v = 0; v < 16; v++) {
#pragma unroll
      for (int b = 0; b < NB; b++) acc[b][v] += rv[b][v];
    }
    __builtin_amdgcn_sched_barrier(0);  // (the sums stay above the stores)
  }
#pragma unroll
  for (int v = 0; v < 16; v++) {
    if (rid[v] < 0) continue;
    if (out) {
      float *op = out + (int64_t)rid[v] * ld_out + cb0 * 32 + r;
#pragma unroll
      for (int b = 0; b < NB; b++)
        if ((cb0 + b) * 32 + r < Cout) op[b * 32] = acc[b][v];
    }
    if (ep.out2) {
      // fused batch norm + leaky ReLU
      float *op2 = ep.out2 + (int64_t)rid[v] * ep.ld2 + cb0 * 32 + r;
#pragma unroll
      for (int b = 0; b < NB; b++)
        if ((cb0 + b) * 32 + r < Cout) {
          const float y = fmaf(acc[b][v], ew[b], eb[b]);
          op2[b * 32] = y * ((y > 0.0f) ? 1.0f : ep.leak);
        }
    }
  }
  if (MODE == MAP_PARENT && ep.side_in) {
    // batch norm of the other half of a joined matrix, same rows and columns
#pragma unroll
    for (int v = 0; v < 16; v++) {
      float x[NB];
#pragma unroll
      for (int b = 0; b < NB; b++)
        x[b] = (rid[v] >= 0 && (cb0 + b) * 32 + r < Cout) ? ep.side_in[(int64_t)rid[v] * ep.ld_side + (cb0 + b) * 32 + r] : 0.0f;
      if (rid[v] < 0) continue;
#pragma unroll
      for (int b = 0; b < NB; b++)
        if ((cb0 + b) * 32 + r < Cout) {
          const float y = fmaf(x[b], sw[b], sb[b]);
          ep.side_out[(int64_t)rid[v] * ep.ld2 + (cb0 + b) * 32 + r] = y * ((y > 0.0f) ? 1.0f : ep.leak);
        }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Narrow 3^3 layers (Cin <= 32, Cout <= 32): the packed filter stays in LDS for the life of the block - 26
// tiles of 6 KB; the centre's, which every tile of a submanifold layer starts with, is read through L1 (all
// 27 would be 2 KB more than a compute unit has) - so the only traffic between L2 and the CU is the gather and
// the map.  Blocks are persistent: block b owns every gridDim.x-th tile and its wavefronts draw them one by one.
// The neighbour ids go from the tile plan straight into registers, a ring of them ahead of the gathers (LDS has no
// room for a copy, and none is needed: lane r only ever wants the ids of row r).
// The sums are formed exactly as in conv_mfma_kernel<1, 27, MAP_NBR, 1> (centre, then offsets ascending, same
// MFMA sequence; the odd offsets' partial sum, with the centre, before the even ones'), so both kernels give the same bits.
// What bounds it: the gather - 500k sites, 32 -> 32: 640 MB of rows through L1 in 94 us a layer (6.8 TB/s; a gather alone, two
// lanes a row, reaches 11.1), against 35 us of matrix-core time; 103 us with one lane a row, 115 with fp32 instructions.
// (A contiguous eighth of the tiles per XCD instead of interleaved ones: 531 against 511 us for four layers.)
// ---------------------------------------------------------------------------------------
// (32 -> 32 in four layers with their batch norms, 500k / 150k sites: eight wavefronts 542 / 228 us, twelve 538 / 201;
// rings of three and four items, which spill at twelve wavefronts, 589 / 232 and 667 / 253)
constexpr int WL_WAVES = 12;
constexpr int WL_DEPTH = 2;
constexpr int WL_MIN_TILES = 2048;  // smaller launches go to conv_mfma_kernel (default of the knob below)
constexpr int WL_SCHED = 256;  // a block orders up to this many tiles of its own by cost

// KS: halves of the 32-channel chunk that exist (1: 16 input channels, 2: 32)
template <int KS, bool PW>
__global__ __launch_bounds__(WL_WAVES * 64) void conv_wlds_kernel(
    const float *__restrict__ in, int64_t ld_in, float *__restrict__ out, int64_t ld_out,
    const float *__restrict__ Wp, const float *__restrict__ bias, const int32_t *__restrict__ map0,
    const int32_t *__restrict__ rows, const int32_t *__restrict__ d_n_rows, int64_t n_rows, int Cin, int Cout,
    const uint8_t *__restrict__ tile_flags, uint32_t in_bytes, uint32_t map_bytes, uint32_t wp_bytes, BnEpilogue ep,
    TilePlan plan) {
  constexpr int K = 27, D = WL_DEPTH, AHEAD = 2 * D - 2;  // gathers D - 1 items ahead, neighbour ids D - 1 before those
  constexpr int PIECES = KS * 3, TILE16 = PIECES * 64;    // of a weight tile: 1 KB pieces, 16-byte units
  __shared__ u32x4 wl[(K - 1) * TILE16];
  __shared__ int next_turn;
  __shared__ int cost_l[WL_SCHED], sched_l[WL_SCHED];
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 31;

  // The order of a tile's offsets: q = 0 the centre, 1 .. 12 the other odd ones, 13 .. 26 the even ones; offset q > 0 has its
  // weights in LDS slot q - 1.
  auto k_of = [](int q) -> int { return 2 * q + (q == 0 ? 13 : q <= 6 ? -1 : q <= 12 ? 1 : -26); };

  // the filter but for the centre, in per-lane order
  if constexpr (PW) {
    const __amdgpu_buffer_rsrc_t rw = make_rsrc(Wp, wp_bytes);
    for (int i = threadIdx.x; i < (K - 1) * KS * 64; i += WL_WAVES * 64) {
      const int slot = i / (KS * 64), e = i - slot * (KS * 64), half = e >> 6, l = e & 63;
      const uint32_t from = (uint32_t)(k_of(slot + 1) * 4096 + (l >> 5) * 2048 + half * 512 + (l & 31) * 16);
      const Parts p = split8_nearest(buf_load16(rw, from, 0), buf_load16(rw, from + 1024u, 0));
#pragma unroll
      for (int q = 0; q < 3; q++) wl[slot * TILE16 + (half * 3 + q) * 64 + l] = p.p[q];
    }
  } else {
    const u32x4 *src = reinterpret_cast<const u32x4 *>(Wp);
    for (int i = threadIdx.x; i < (K - 1) * TILE16; i += WL_WAVES * 64) {
      const int slot = i / TILE16, e = i - slot * TILE16;
      wl[i] = src[k_of(slot + 1) * (WT_BYTES / 16) + e];
    }
  }
  if (threadIdx.x == 0) next_turn = 0;
  const int64_t ntiles = (n + TILE_M - 1) / TILE_M;
  // Blocks are dealt to the eight XCDs round robin (block b runs on XCD b % 8) and every XCD has an
  // L2 of its own: rank the blocks XCD by XCD, so that the tiles an XCD works on at any time are
  // neighbours in the processing order and share gathered rows in its L2.
  const int G8 = gridDim.x >> 3;
  const int brank = (gridDim.x & 7) == 0 ? (int)(blockIdx.x & 7) * G8 + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  // The block of rank q owns the tiles q, q + gridDim.x, ...  With a tile plan it takes them most
  // expensive first (cost = offsets the tile uses; ties in tile order): its wavefronts then finish
  // within a cheap tile of each other instead of an average one.
  const int my_tiles = ntiles > brank ? (int)((ntiles - brank + gridDim.x - 1) / gridDim.x) : 0;
  const bool lpt = plan.map != nullptr && my_tiles > WL_WAVES && my_tiles <= WL_SCHED;
  if (lpt) {
    for (int j = threadIdx.x; j < my_tiles; j += WL_WAVES * 64) {
      const int64_t tt = (int64_t)j * gridDim.x + brank;
      cost_l[j] = (!tile_flags || tile_flags[tt]) ? __builtin_popcount(plan.tmask[tt]) : -1;
    }
  }
  __syncthreads();
  if (lpt) {
    for (int j = threadIdx.x; j < my_tiles; j += WL_WAVES * 64) {
      const int c = cost_l[j];
      int rank = 0;
      for (int i = 0; i < my_tiles; i++) {
        const int ci = cost_l[i];
        rank += (ci > c || (ci == c && i < j)) ? 1 : 0;
      }
      sched_l[rank] = j;
    }
    __syncthreads();
  }

  const __amdgpu_buffer_rsrc_t rin = make_rsrc(in, in_bytes), rw = make_rsrc(Wp, wp_bytes);
  // the outputs are addressed with 32-bit byte offsets as well; rows that do not exist get an
  // out-of-range offset and the hardware drops the store
  const __amdgpu_buffer_rsrc_t rout = make_rsrc(out, out ? BUF_OOB : 0u), rout2 = make_rsrc(ep.out2, ep.out2 ? BUF_OOB : 0u), rres = make_rsrc(ep.res, ep.res ? BUF_OOB : 0u);
  const uint32_t ld4 = (uint32_t)ld_in * 4u, ldo4 = (uint32_t)ld_out * 4u, ldo24 = (uint32_t)ep.ld2 * 4u, ldr4 = (uint32_t)ep.ldr * 4u;
  const uint32_t piece = pair_piece(lane);
  const int col = r;
  const float bv = (bias && col < Cout) ? bias[col] : 0.0f;
  const float ew = (ep.out2 && col < Cout) ? ep.w[col] : 0.0f;
  const float eb = (ep.out2 && col < Cout) ? ep.b[col] : 0.0f;

  // The wavefronts of a block draw its tiles from a counter in LDS
  // (tile costs differ by 3x: a fixed deal per wavefront leaves the slowest one far behind).
  // draw(): the next tile of this block that has work, or ntiles.
  // With fewer than three tiles per wavefront the draws ahead of the tile pipeline (up to three tiles
  // in hand per wavefront) would leave late wavefronts with nothing: then the turns are dealt instead,
  // back and forth: wavefront w takes w, 2 WL_WAVES - 1 - w, 2 WL_WAVES + w, ...  (What a block lasts is the
  // matrix core of its busiest SIMD, which three wavefronts share - w, w + 4, w + 8; with the turns going
  // round the same way, w + WL_WAVES next, the SIMD that starts with the three most expensive tiles also
  // gets the first of the second round.)
  const bool dealt = my_tiles < 3 * WL_WAVES;
  int my_turn = wave, my_round = 0;
  auto draw = [&]() -> int {
    for (;;) {
      int turn;
      if (dealt) {
        turn = my_turn;
        my_round++;
        my_turn = my_round * WL_WAVES + ((my_round & 1) ? WL_WAVES - 1 - wave : wave);
      } else {
        int v = 0;
        if (lane == 0) v = atomicAdd(&next_turn, 1);
        turn = v;
      }
      turn = __builtin_amdgcn_readfirstlane(turn);
      if (turn >= my_tiles) return (int)ntiles;
      const int t = (lpt ? __builtin_amdgcn_readfirstlane(sched_l[turn]) : turn) * (int)gridDim.x + brank;
      if (!tile_flags || tile_flags[t]) return t;
    }
  };
  auto load_row = [&](int t) -> int {
    const int64_t p = (int64_t)t * TILE_M + r;
    return (t < ntiles && p < n) ? (rows ? rows[p] : (int)p) : -1;
  };
  // Where a lane finds the neighbour id of offset k: at base + k * pitch of the tile plan (the map transposed into
  // processing order: one 128-byte run per (offset, tile)), or without a plan of its own row of the map.
  const bool planned = plan.map != nullptr;
  const __amdgpu_buffer_rsrc_t rids = planned ? make_rsrc(plan.map, (uint32_t)(plan.ld * K * 4)) : make_rsrc(map0, map_bytes);
  const uint32_t pitch = planned ? (uint32_t)plan.ld * 4u : 4u;
  auto id_base = [&](int t, int row) -> uint32_t {
    return planned ? (uint32_t)(t * TILE_M + r) * 4u : row >= 0 ? (uint32_t)row * (K * 4u) : BUF_OOB;
  };
  // the offsets a tile uses, bit q
  auto every_other = [](unsigned x) -> unsigned {  // bits 0, 2, .. 30 of x
    x &= 0x55555555u;
    x = (x | x >> 1) & 0x33333333u;
    x = (x | x >> 2) & 0x0F0F0F0Fu;
    x = (x | x >> 4) & 0x00FF00FFu;
    return (x | x >> 8) & 0xFFFFu;
  };
  auto offsets_of = [&](int t, uint32_t base, int v) -> unsigned {
    unsigned m = 0;
    if (t >= ntiles) return 0u;
    if (planned) {
      m = (unsigned)__builtin_amdgcn_readfirstlane(v) & 0x7FFFFFFu;
    } else {
      for (int k = 0; k < K; k++) {
        const int id = base == BUF_OOB ? -1 : (int)__builtin_amdgcn_raw_buffer_load_b32(rids, (int)(base + k * pitch), 0, 0);
        m |= __any(id >= 0) ? 1u << k : 0u;
      }
    }
    const unsigned odd = every_other(m >> 1), even = every_other(m);
    return ((odd >> 6) & 1u) | ((odd & 0x3Fu) << 1) | ((odd >> 7) << 7) | (even << 13);
  };
  auto next_q = [](unsigned &rest) -> int {  // past the end: -1
    const int q = rest ? __builtin_ctz(rest) : -1;
    rest &= rest - 1;
    return q;
  };
  auto id_load = [&](int q, uint32_t base) -> int {
    const uint32_t k = (uint32_t)k_of(q);
    return (int)__builtin_amdgcn_raw_buffer_load_b32(rids, (int)(q >= 0 && base != BUF_OOB ? base : BUF_OOB),
                                                     (int)(q >= 0 ? k * pitch : 0u), 0);
  };
  auto gather = [&](int q, int src, uint32_t base) -> Frag {
    const bool on = q >= 0 && src >= 0 && base != BUF_OOB;  // (a load sent out of range returns 0, which would pass for a site)
    return gather_rows<!PW>(rin, on, (uint32_t)src * ld4, lane, piece, KS == 2);
  };

  // Software pipeline over tiles: while tile t is computed, the neighbour ids of the first items of the next
  // tile and the row ids and offset mask of the one after it are in flight; the gathers of the next tile's first
  // items go out before this tile's rows are stored.
  int t = draw();
  if (t >= ntiles) return;  // (no workgroup barrier below)
  int my_row = load_row(t);
  uint32_t base = id_base(t, my_row);
  unsigned rest = offsets_of(t, base, planned ? (int)plan.tmask[t] : 0);
  int ids[AHEAD];  // ids of the items 0 .. AHEAD - 1 of tile t
  {
    unsigned rr = rest;
#pragma unroll
    for (int i = 0; i < AHEAD; i++) ids[i] = id_load(next_q(rr), base);
  }
  int tn = draw();
  int my_row_n = load_row(tn);
  int mask_n_v = planned && tn < ntiles ? (int)plan.tmask[tn] : 0;
  Frag g[D];
  WFrag<false> bw;  // of the item on the matrix cores
  WFrag<PW> cw;     // the centre's
  auto prime = [&](unsigned rr, uint32_t b) {  // the gathers of the first items, and the centre's weights
    const uint32_t lane16 = (uint32_t)lane_again() * 16u;  // (not a constant of the loop: the weights would be, and spilled)
#pragma unroll
    for (int i = 0; i < D - 1; i++) g[i] = gather(next_q(rr), ids[i], b);
    if constexpr (PW) {
      cw = load_wtile<PW>(rw, 13, true, lane16);
    } else {
#pragma unroll
      for (int i = 0; i < PIECES; i++)
        bw.s[i / 3].p[i % 3] = __builtin_bit_cast(u32x4, buf_load16(rw, lane16, 13u * WT_BYTES + 1024u * i));
    }
  };
  prime(rest, base);

  while (t < ntiles) {
    const uint32_t base_n = id_base(tn, my_row_n);
    const unsigned rest_n = offsets_of(tn, base_n, mask_n_v);
    // ring of neighbour ids: the item i's is in slot i % D from the step it is loaded in to its gather
    int ix[D];
#pragma unroll
    for (int i = D - 1; i < AHEAD; i++) ix[i % D] = ids[i];
    {
      unsigned rr = rest_n;
#pragma unroll
      for (int i = 0; i < AHEAD; i++) ids[i] = id_load(next_q(rr), base_n);
    }
    const int tnn = tn < ntiles ? draw() : (int)ntiles;
    const int my_row_nn = load_row(tnn);
    const int mask_nn_v = planned && tnn < ntiles ? (int)plan.tmask[tnn] : 0;

    // the odd offsets' partial sum, then - with the bias - the even ones'
    Sum sum;
    f16v total;
    bool second = false;
    sum_start(sum, 0.0f);
    auto fold = [&]() {
      total = sum_of(sum);
      sum_start(sum, bv);
      second = true;
    };

    if (rest) {
      // three cursors over the tile's items: the one computed, the one gathered, the one whose id is loaded
      unsigned rc = rest, rg = rest, ri = rest;
#pragma unroll
      for (int i = 0; i < D - 1; i++) (void)next_q(rg);
#pragma unroll
      for (int i = 0; i < AHEAD; i++) (void)next_q(ri);
      // step of the item in slot U of the rings
      auto issue = [&](auto U) {
        constexpr int u = decltype(U)::value;
        const int qg = next_q(rg), qi = next_q(ri);
        // (the id first: its wait, a step on, is then not one for the gathers behind it as well)
        const int here = ix[(u + D - 1) % D];
        ix[(u + AHEAD) % D] = id_load(qi, base);
        __builtin_amdgcn_sched_barrier(0);
        g[(u + D - 1) % D] = gather(qg, here, base);
      };
      auto compute = [&](auto U) {
        constexpr int u = decltype(U)::value;
        Parts as[2];
        const Frag a = rows_of<!PW>(g[u]);
        as[0] = split8(a.q[0], a.q[1]);
        if constexpr (KS == 2) as[1] = split8(a.q[2], a.q[3]);
        mac_chunk(sum, as, bw, KS == 2);
      };
      auto wread = [&](int q) {
        const u32x4 *p = wl + (q - 1) * TILE16 + lane;
#pragma unroll
        for (int i = 0; i < PIECES; i++) bw.s[i / 3].p[i % 3] = p[i * 64];
      };
      {
        const int q = next_q(rc);
        if (q >= 13) fold();
        if (q != 0) {  // (a tile without the centre; bw or cw holds the centre's weights otherwise)
          wread(q);
        } else if constexpr (PW) {
#pragma unroll
          for (int i = 0; i < KS; i++) bw.s[i] = parts_of(cw, i);
        }
        __builtin_amdgcn_sched_barrier(0);
        issue(std::integral_constant<int, 0>());
        __builtin_amdgcn_sched_barrier(0);
        compute(std::integral_constant<int, 0>());
      }
      // one turn: the slots 1 .. D - 1, 0
      auto one = [&](auto U) -> bool {
        if (!rc) return false;
        const int q = next_q(rc);
        if (q >= 13 && !second) fold();
        wread(q);
        __builtin_amdgcn_sched_barrier(0);
        issue(U);
        __builtin_amdgcn_sched_barrier(0);
        compute(U);
        return true;
      };
      static_assert(D == 2, "the turns of the rings are written out");
      while (one(std::integral_constant<int, 1>()) && one(std::integral_constant<int, 0>())) {
      }
    }
    // the next tile's first gathers and the centre's weights, in flight over this tile's stores
    prime(rest_n, base_n);
    __builtin_amdgcn_sched_barrier(0);
    if (!second) fold();
    f16v acc = sum_of(sum);
#pragma unroll
    for (int v = 0; v < 16; v++) acc[v] += total[v];
    unscale<16>(acc);

    // D layout of the 32x32 MFMA: lane holds column (lane & 31), rows 8*(v/4) + 4*(lane>>5) + (v&3)
    repair_sums<16>(acc, 0, [&]() -> f16v {
      f16v x;
#pragma unroll
      for (int v = 0; v < 16; v++) x[v] = bv;
      add_plain_products<PW>(
          x, [&](int k) { return base == BUF_OOB ? -1 : (int)__builtin_amdgcn_raw_buffer_load_b32(rids, (int)(base + k * pitch), 0, 0); },
          K, rin, ld4, rw, Cin, 1, 1, 0);
      return x;
    });
    store_tile(acc, my_row, 0, col < Cout, rout, ldo4, rout2, ldo24, rres, ldr4, ew, eb, ep.leak, out != nullptr, ep.out2 != nullptr, ep.res != nullptr);
    t = tn;
    my_row = my_row_n;
    base = base_n;
    rest = rest_n;
    tn = tnn;
    my_row_n = my_row_nn;
    mask_n_v = mask_nn_v;
  }
}

// ---------------------------------------------------------------------------------------
// Wide 3^3 layers with many tiles: the four wavefronts of a block work on four consecutive tiles and walk the union
// of their offsets in step: the weight tile of a step goes from L2 into LDS once per block (buffer loads that write
// LDS directly, 1 KB pieces dealt to the wavefronts) and is read from there by all four, and a wavefront
// computes NB output blocks from one gathered chunk, split into parts once.  A wavefront owns its tile: no partial
// sums cross wavefronts.  To give the bits of conv_mfma_kernel<1, 27, MAP_NBR, ST> it forms that kernel's ST partial
// sums - the items (k, ch) with (k * nch + ch) % ST == p, in ascending order, bias in sum 0 - one after the other and
// adds each to the total when it is done: two accumulators per output block, whatever ST.
// Blocks are persistent over units (group of four tiles, NB output blocks) taken from the cost-
// ordered group schedule: block b takes the units b, 2B - 1 - b, 2B + b, ..
// Weights and gathers of two steps are in flight over the step on the matrix cores; the three weight buffers and A
// slots are compile-time choices (the step loop is unrolled by three): the compiler then knows that a read of one
// weight buffer cannot touch a load into another that is still in flight (for a single array it would wait for every
// outstanding load before each LDS read).
// What bounds it (64 -> 64 at 500k sites, a launch 414 us in fp32, 325 now; four layers with batch norms 1920 and
// 1530): 2.2 GB from L2 into L1 per launch at 6.5 TB/s; matrix cores busy 41 %.  Not taken: eight tiles per block,
// which halves the weight bytes, 1542 us instead of 1436 (the wavefronts wait for one another); units in site order per
// XCD, which would hit L2, 1741 instead of 1460 (unbalanced).
// ---------------------------------------------------------------------------------------
#define INSC_LDS_PTR(x) ((__attribute__((address_space(3))) void *)(x))
template <int NB, int ST, bool PW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB > 1 ? 2 : 3, NB > 1 ? 2 : 3))) void conv_wshare_kernel(
    const float *__restrict__ in, int64_t ld_in, float *__restrict__ out, int64_t ld_out,
    const float *__restrict__ Wp, const float *__restrict__ bias, const int32_t *__restrict__ rows,
    const int32_t *__restrict__ d_n_rows, int64_t n_rows, int Cin, int Cout, int nbt, int nbtp,
    const uint8_t *__restrict__ tile_flags, uint32_t in_bytes, uint32_t wp_bytes, BnEpilogue ep, TilePlan plan) {
  constexpr int K = 27, WV = 4;
  constexpr int NSTAGE = (TILE_M * K + 63) / 64;  // 14 loads of 64 entries; the last one half empty
  constexpr int PC = pw_pieces(PW, 2);            // pieces of a weight tile
  __shared__ int nl[WV][NSTAGE * 64];
  __shared__ u32x4 wl0[NB][PC * 64];
  __shared__ u32x4 wl1[NB][PC * 64];
  __shared__ u32x4 wl2[NB][PC * 64];
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  const int ntiles = (int)((n + TILE_M - 1) / TILE_M), ngroups = (ntiles + WV - 1) / WV;
  const int nug = (nbt + NB - 1) / NB;  // units per group
  const int64_t units = (int64_t)ngroups * nug;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int r = lane & 31, h = lane >> 5;
  const int nch = conv_nch(Cin);
  // offsets that hold items of partial sum p
  unsigned hm[ST];
#pragma unroll
  for (int p = 0; p < ST; p++) hm[p] = (unsigned)__ballot(lane < K && ((p - lane * nch) & (ST - 1)) < nch);
  const int64_t B = gridDim.x, b = blockIdx.x;
  const __amdgpu_buffer_rsrc_t rplan = make_rsrc(plan.map, (uint32_t)(plan.ld * K * 4));
  const __amdgpu_buffer_rsrc_t rsched = make_rsrc(plan.sched + (plan.ld + 31) / 32, (uint32_t)ngroups * 4u);  // group schedule
  const __amdgpu_buffer_rsrc_t rtmask = make_rsrc(plan.tmask, (uint32_t)ntiles * 4u);
  const __amdgpu_buffer_rsrc_t rflag = make_rsrc(tile_flags, tile_flags ? (uint32_t)ntiles : 0u);
  const __amdgpu_buffer_rsrc_t rin = make_rsrc(in, in_bytes), rw = make_rsrc(Wp, wp_bytes);
  const __amdgpu_buffer_rsrc_t rout = make_rsrc(out, out ? BUF_OOB : 0u), rout2 = make_rsrc(ep.out2, ep.out2 ? BUF_OOB : 0u);
  const __amdgpu_buffer_rsrc_t rres = make_rsrc(ep.res, ep.res ? BUF_OOB : 0u);
  const __amdgpu_buffer_rsrc_t rbias = make_rsrc(bias, bias ? (uint32_t)Cout * 4u : 0u);
  const __amdgpu_buffer_rsrc_t rew = make_rsrc(ep.w, ep.out2 ? (uint32_t)Cout * 4u : 0u);
  const __amdgpu_buffer_rsrc_t reb = make_rsrc(ep.b, ep.out2 ? (uint32_t)Cout * 4u : 0u);
  const uint32_t ld4 = (uint32_t)ld_in * 4u, ldo4 = (uint32_t)ld_out * 4u, ldo24 = (uint32_t)ep.ld2 * 4u,
                 ldr4 = (uint32_t)ep.ldr * 4u;
  const uint32_t piece = pair_piece(lane);
  int *nlw = nl[wave];

  auto unit_at = [&](int64_t j) -> int64_t { return j * B + ((j & 1) ? B - 1 - b : b); };
  auto group_issue = [&](int64_t u) -> int {
    return __builtin_amdgcn_raw_buffer_load_b32(rsched, (int)(u < units ? (uint32_t)(u / nug) * 4u : BUF_OOB), 0, 0);
  };
  // offset masks of the four tiles of a group (0 for a tile that does not exist or is not flagged):
  // lanes 0..3 fetch one each, every wavefront the same four
  auto masks_issue = [&](int g, int &mv, int &fv) {
    const int t = g * WV + (lane & 3);
    const bool ok = g >= 0 && t < ntiles;
    mv = __builtin_amdgcn_raw_buffer_load_b32(rtmask, (int)(ok ? (uint32_t)t * 4u : BUF_OOB), 0, 0);
    fv = tile_flags ? (int)__builtin_amdgcn_raw_buffer_load_b8(rflag, (int)(ok ? (uint32_t)t : BUF_OOB), 0, 0) : (ok ? 1 : 0);
  };
  // this wavefront's slice of the map, straight into LDS (entry e = k * 32 + row at nlw[e])
  // (load i covers the offsets 2i and 2i + 1: one per half-wave; the lane's part of the address is the
  // same for every i, the rest is a scalar)
  auto stage_issue = [&](int tile) {
    if (tile < 0) return;  // no such tile: its wavefront never reads the slice
    const int l = lane_again();
    const uint32_t base = (uint32_t)((l >> 5) * (int)plan.ld + tile * TILE_M + (l & 31)) * 4u;
    const uint32_t pair = (uint32_t)plan.ld * 8u;
#pragma unroll
    for (int i = 0; i < NSTAGE; i++) {
      const uint32_t voff = (2 * i + 1 < K || l < 32) ? base : BUF_OOB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rplan, INSC_LDS_PTR(nlw + i * 64), 4, (int)voff, (int)(i * pair), 0, 0);
    }
  };
  auto row_of = [&](int tile) -> int {
    const int64_t p = (int64_t)tile * TILE_M + r;
    return (tile >= 0 && p < n) ? (rows ? rows[p] : (int)p) : -1;
  };
  struct Step {
    int k, ch, p;
    unsigned rest;
  };

  int64_t j = 0, u = unit_at(0);
  int g_c = u < units ? __builtin_amdgcn_readfirstlane(group_issue(u)) : -1;
  int g_n = unit_at(1) < units ? __builtin_amdgcn_readfirstlane(group_issue(unit_at(1))) : -1;
  int mv_c, fv_c;
  masks_issue(g_c, mv_c, fv_c);
  int tile = g_c >= 0 && g_c * WV + wave < ntiles ? g_c * WV + wave : -1;
  stage_issue(tile);
  int my_row = row_of(tile);

  while (u < units) {
    const int ob0 = (int)(u % nug) * NB;
    const int64_t un = unit_at(j + 1), unn = unit_at(j + 2);
    const int g_nn_v = group_issue(unn);
    int mv_n, fv_n;
    masks_issue(g_n, mv_n, fv_n);
    const int tile_n = g_n >= 0 && g_n * WV + wave < ntiles ? g_n * WV + wave : -1;
    const int my_row_n = row_of(tile_n);
    // masks of the group: mine and the union
    unsigned mt[WV];
#pragma unroll
    for (int w = 0; w < WV; w++)
      mt[w] = __builtin_amdgcn_readlane(fv_c, w) ? (unsigned)__builtin_amdgcn_readlane(mv_c, w) : 0u;
    unsigned mine = 0, uni = 0;
#pragma unroll
    for (int w = 0; w < WV; w++) {
      uni |= mt[w];
      if (w == wave) mine = mt[w];
    }
    if (tile < 0) mine = 0;

    if (uni) {
      // bias and the fused batch norm's coefficients of this lane's columns
      float bv[NB], ew[NB], eb[NB];
#pragma unroll
      for (int o = 0; o < NB; o++) {
        const uint32_t off = (uint32_t)((ob0 + o) * 32 + r) * 4u;
        bv[o] = __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(rbias, (int)off, 0, 0));
        ew[o] = __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(rew, (int)off, 0, 0));
        eb[o] = __uint_as_float((unsigned)__builtin_amdgcn_raw_buffer_load_b32(reb, (int)off, 0, 0));
      }
      // the running partial sum and the sum of the finished ones; bias in partial sum 0
      Sum acc[NB];
      f16v total[NB];
#pragma unroll
      for (int o = 0; o < NB; o++) sum_start(acc[o], bv[o]);
      int cur = 0;  // the partial sum in acc
      auto step_next = [&](const Step &c) -> Step {  // past the end: k = -1
        Step nx = c;
        nx.ch = c.ch + ST;
        if (nx.ch >= nch || c.k < 0) {
#pragma unroll
          for (int p = 1; p < ST; p++) {
            if (nx.rest == 0 && nx.p < p) {
              nx.p = p;
              nx.rest = uni & hm[p];
            }
          }
          nx.k = nx.rest ? __builtin_ctz(nx.rest) : -1;
          nx.ch = (nx.p - nx.k * nch) & (ST - 1);
          nx.rest &= nx.rest - 1;
        }
        return nx;
      };
      // weight tiles of a step -> LDS, their 1 KB pieces dealt to the four wavefronts
      auto w_issue = [&](const Step &c, u32x4 (*wl)[PC * 64]) {
#pragma unroll
        for (int i = 0; i < (PC * NB + WV - 1) / WV; i++) {
          const int piece = i * WV + wave, o = piece / PC;
          if (piece >= PC * NB) break;
          const uint32_t soff = (uint32_t)(((c.k < 0 ? 0 : c.k) * nch + c.ch) * nbtp + ob0 + o) * (uint32_t)wt_bytes(PW);
          const bool ok = c.k >= 0 && ob0 + o < nbt;
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              rw, INSC_LDS_PTR(&wl[0][piece * 64]), 16,
              (int)(ok ? (uint32_t)((piece - o * PC) * 1024 + lane * 16) : BUF_OOB), (int)soff, 0, 0);
        }
      };
      auto gather = [&](const Step &c) -> Frag {
        const int kk = c.k < 0 ? 0 : c.k;
        const int src = nlw[kk * TILE_M + r];
        const bool on = c.k >= 0 && ((mine >> kk) & 1u) && src >= 0;
        return gather_rows<!PW>(rin, on, (uint32_t)src * ld4 + (uint32_t)(c.ch * 128), lane, piece, Cin - c.ch * 32 >= 32);
      };
      auto compute = [&](const Step &c, const Frag &a, const u32x4 (*wl)[PC * 64]) {
        if (c.k < 0 || !((mine >> c.k) & 1u)) return;  // (the same for every lane of the wavefront)
        const bool full = Cin - c.ch * 32 >= 32;
        if (c.p != cur) {
#pragma unroll
          for (int o = 0; o < NB; o++) {
            const f16v part = sum_of(acc[o]);
#pragma unroll
            for (int v = 0; v < 16; v++) total[o][v] = cur == 0 ? part[v] : total[o][v] + part[v];
            sum_start(acc[o], 0.0f);
          }
          cur = c.p;
        }
        const Frag w = rows_of<!PW>(a);
        const Parts as[2] = {split8(w.q[0], w.q[1]), split8(w.q[2], w.q[3])};
#pragma unroll
        for (int o = 0; o < NB; o++) {
          if (ob0 + o >= nbt) break;
          WFrag<PW> bf;
          if constexpr (PW) {
#pragma unroll
            for (int i = 0; i < 4; i++)
              bf.q[i] = __builtin_bit_cast(float4, wl[o][(2 * h + (i & 1)) * 64 + (i >> 1) * 32 + r]);
          } else {
#pragma unroll
            for (int i = 0; i < 6; i++) bf.s[i / 3].p[i % 3] = wl[o][i * 64 + lane];
          }
          mac_chunk(acc[o], as, bf, full);
        }
      };
      // Two steps' weights and gathers are in flight over the step on the matrix cores; weight buffers and gather
      // slots go round in three turns, each a compile-time choice.
      Step c0, c1, c2;
      c0.k = -1;
      c0.ch = nch;
      c0.p = 0;
      c0.rest = uni & hm[0];
      c0 = step_next(c0);
      c1 = step_next(c0);
      __builtin_amdgcn_sched_barrier(0);
      w_issue(c0, wl0);
      __builtin_amdgcn_sched_barrier(0);
      Frag a0 = gather(c0), a1, a2;
      __builtin_amdgcn_sched_barrier(0);
      w_issue(c1, wl1);
      __builtin_amdgcn_sched_barrier(0);
      a1 = gather(c1);
      __builtin_amdgcn_sched_barrier(0);
      // Before a barrier every wavefront waits until its own pieces of the step's weight tiles have
      // landed in LDS: everything but what was issued after them - the step's four gather loads and the next
      // step's (at least PC * NB / 4) pieces and four gather loads; the order of the loads is pinned.
      auto turn = [&](Step &c, Step &cp2, const Frag &a, Frag &ap2, const Step &cp1, u32x4 (*wl)[PC * 64],
                      u32x4 (*wlp2)[PC * 64]) {
        __builtin_amdgcn_s_waitcnt(0x0F70 | (8 + PC * NB / WV));
        __syncthreads();  // the step's weights are complete for every wavefront, and nobody reads the oldest buffer any more
        __builtin_amdgcn_sched_barrier(0);
        cp2 = step_next(cp1);
        w_issue(cp2, wlp2);
        __builtin_amdgcn_sched_barrier(0);
        ap2 = gather(cp2);
        __builtin_amdgcn_sched_barrier(0);
        compute(c, a, wl);
        __builtin_amdgcn_sched_barrier(0);
      };
      for (;;) {
        turn(c0, c2, a0, a2, c1, wl0, wl2);
        if (c1.k < 0) break;
        turn(c1, c0, a1, a0, c2, wl1, wl0);
        if (c2.k < 0) break;
        turn(c2, c1, a2, a1, c0, wl2, wl1);
        if (c0.k < 0) break;
      }
      __syncthreads();  // the weight buffers are free for the next unit

      // this unit's rows; the next unit's map slice goes out first (nobody reads nl any more)
      stage_issue(tile_n);
      if (mine) {
#pragma unroll
        for (int o = 0; o < NB; o++) {
          const int cc = (ob0 + o) * 32 + r;
          if (ob0 + o >= nbt) break;
          f16v sum = sum_of(acc[o]);
          if (cur != 0) {
#pragma unroll
            for (int v = 0; v < 16; v++) sum[v] = total[o][v] + sum[v];
          }
          unscale<16>(sum);
          repair_sums<16>(sum, 0, [&]() -> f16v {
            f16v x;
#pragma unroll
            for (int v = 0; v < 16; v++) x[v] = bv[o];
            add_plain_products<PW>(x, [&](int k) { return plan.map[(int64_t)k * plan.ld + (int64_t)tile * TILE_M + (lane_again() & 31)]; }, K, rin, ld4,
                               rw, Cin, nch, nbtp, ob0 + o);
            return x;
          });
          store_tile(sum, my_row, (ob0 + o) * 32, cc < Cout, rout, ldo4, rout2, ldo24, rres, ldr4, ew[o], eb[o], ep.leak, out != nullptr,
                     ep.out2 != nullptr, ep.res != nullptr);
        }
      }
    } else {
      stage_issue(tile_n);
    }
    j++;
    u = un;
    g_c = g_n;
    g_n = unn < units ? __builtin_amdgcn_readfirstlane(g_nn_v) : -1;
    mv_c = mv_n;
    fv_c = fv_n;
    tile = tile_n;
    my_row = my_row_n;
  }
}

__global__ void count_rules_kernel(const int32_t *__restrict__ map0, int K, const int32_t *__restrict__ rows,
                                   const int32_t *__restrict__ d_n_rows, int64_t n_rows,
                                   unsigned long long *__restrict__ total) {
  const int64_t n = d_n_rows ? min((int64_t)*d_n_rows, n_rows) : n_rows;
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int c = 0;
  if (t < n) {
    const int row = rows ? rows[t] : (int)t;
    if (row >= 0)
      for (int k = 0; k < K; k++) c += map0[(int64_t)row * K + k] >= 0 ? 1 : 0;
  }
  for (int d = 32; d > 0; d >>= 1) c += __shfl_down(c, d, 64);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(total, (unsigned long long)c);
}

// map[k * ld + p] = nbr[order[p]][k] for p < n, -1 up to the end of the last tile; tmask[t] = OR of
// the offsets the rows of tile t have.  One thread per position; the writes of one offset are
// coalesced across the wavefront.
__device__ __forceinline__ void tile_plan_body(const int32_t *__restrict__ nbr, const int32_t *__restrict__ order,
                                               const int32_t *__restrict__ d_n, int64_t n_rows, int64_t ld,
                                               int32_t *__restrict__ map, uint32_t *__restrict__ tmask) {
  // A block transposes the rows of 256 positions through LDS: the rows are read 27 consecutive words at a
  // time (consecutive threads, consecutive offsets), the plan is written one 1 KB run per offset.  (With a
  // thread per position reading its own row every load instruction touched 64 different lines.)
  __shared__ int site_l[256];
  __shared__ int row_l[256 * 27];  // [position][offset]: stride 27, odd, so the reads below are conflict-free
  const int64_t n = d_n ? min((int64_t)*d_n, n_rows) : n_rows;
  const int64_t padded = (n + TILE_M - 1) / TILE_M * TILE_M;
  const int64_t p0 = (int64_t)blockIdx.x * 256, p = p0 + threadIdx.x;
  if (p0 >= padded) return;  // (the whole block)
  site_l[threadIdx.x] = p < n ? (order ? order[p] : (int)p) : -1;
  __syncthreads();
  // (positions beyond the sites read the row of the block's first site: a load under a condition would be waited for
  // before the next is issued; the plans of 6k sites 12.0 us, 5.4 so, of 150k 16.7, 13.1, of 500k 45, 36.5)
  {
    const int some = site_l[0];
    int v[27];
    unsigned none = 0;
#pragma unroll
    for (int i = 0; i < 27; i++) {
      const int e = i * 256 + threadIdx.x, lp = e / 27, k = e - lp * 27;
      const int site = site_l[lp];
      none |= (site < 0 ? 1u : 0u) << i;
      v[i] = nbr[(int64_t)(site < 0 ? some : site) * 27 + k];
    }
#pragma unroll
    for (int i = 0; i < 27; i++) row_l[i * 256 + threadIdx.x] = (none >> i) & 1u ? -1 : v[i];
  }
  __syncthreads();
  if (p >= padded) return;  // whole 32-lane groups leave together (padded is a multiple of 32)
  unsigned m = 0;
#pragma unroll
  for (int k = 0; k < 27; k++) {
    const int v = row_l[threadIdx.x * 27 + k];
    map[(int64_t)k * ld + p] = v;
    if (v >= 0) m |= 1u << k;
  }
#pragma unroll
  for (int d = 16; d > 0; d >>= 1) m |= (unsigned)__shfl_xor((int)m, d, 64);
  if ((threadIdx.x & 31) == 0) tmask[p >> 5] = m;
}
__global__ __launch_bounds__(256) void tile_plan_kernel(const int32_t *__restrict__ nbr,
                                                        const int32_t *__restrict__ order,
                                                        const int32_t *__restrict__ d_n, int64_t n_rows, int64_t ld,
                                                        int32_t *__restrict__ map, uint32_t *__restrict__ tmask) {
  tile_plan_body(nbr, order, d_n, n_rows, ld, map, tmask);
}
// the plans of several maps (the scales of a network) in one launch: blockIdx.y picks the map
__global__ __launch_bounds__(256) void tile_plan_batch_kernel(TilePlanBatch b) {
  const TilePlanJob &j = b.job[blockIdx.y];
  if (!j.nbr) return;  // this plan is up to date: only its schedule is wanted
  tile_plan_body(j.nbr, j.order, j.d_n, j.n_rows, j.ld, j.map, j.tmask);
}

// The columns of the sites added by the last insert, appended to a plan that holds the older
// sites already: positions [first, end of the last tile) of every offset row (first = site count
// before the insert; positions follow the processing order, in which new sites come last).  The
// offset masks of the tiles they open have been cleared beforehand; the mask of a tile is the OR
// over its rows.  One thread per (position, offset).
__global__ __launch_bounds__(256) void tile_plan_append_batch_kernel(TilePlanBatch b) {
  const TilePlanJob &j = b.job[blockIdx.y];
  if (!j.map) return;
  const int64_t first = j.d_n[1], n = j.d_n[0];
  // one wavefront per tile, from the tile that holds position `first` on; lane = (row of the tile,
  // parity of the offset)
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int64_t tile = first / TILE_M + (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (tile * TILE_M >= n) return;
  const int64_t p = tile * TILE_M + r;
  const bool mine = p >= first;  // (older positions of the first tile keep their entries)
  const int site = (mine && p < n) ? (j.order ? j.order[p] : (int)p) : -1;
  unsigned m = 0;
  for (int k = h; k < 28; k += 2) {
    const int v = (site >= 0 && k < 27) ? j.nbr[(int64_t)site * 27 + k] : -1;
    if (mine && k < 27) j.map[(int64_t)k * j.ld + p] = v;
    const unsigned long long bal = __ballot(v >= 0);
    if ((unsigned)bal) m |= 1u << k;
    if ((unsigned)(bal >> 32)) m |= 1u << (k + 1);
  }
  if (lane == 0 && m) atomicOr(&j.tmask[tile], m);
}

int tile_plan_append_batch(const TilePlanBatch &b, int64_t n_new_upper, hipStream_t s) {
  if (b.n <= 0 || n_new_upper <= 0) return INSC_OK;
  // (the new sites touch at most n_new_upper / 32 + 2 tiles; four tiles per block)
  hipLaunchKernelGGL(tile_plan_append_batch_kernel, dim3(grid_for(n_new_upper / TILE_M + 2, 4), (unsigned)b.n), dim3(256),
                     0, s, b);
  INSC_LAUNCH_CHECK();
  return INSC_OK;
}

// sched = the tiles by falling number of active offsets (a counting sort over the 28 classes; the order inside a class is the order of arrival and has no influence on any result).
__device__ __forceinline__ void tile_sched_body(const uint32_t *__restrict__ tmask, const int32_t *__restrict__ d_n,
                                                int64_t n_rows, int32_t *__restrict__ sched,
                                                int32_t *__restrict__ gsched, bool groups) {
  // One workgroup for the tiles, another (groups) for groups of four consecutive tiles, by the offsets any of the four uses
  // (their schedule follows the tile schedule at gsched).  The lanes of a wavefront that hold the same class send one
  // atomic between them - one each, on a few addresses, was most of the time - and the masks are asked for eight at a
  // time, without a condition.  (One workgroup for both, an atomic per tile: 6k sites 4.2 us, 150k 12.4, 500k 32;
  // now 4.0, 7.6 and 17.)
  __shared__ int cnt[28], base[28];
  const int64_t n = d_n ? min((int64_t)*d_n, n_rows) : n_rows;
  const int64_t ntiles = (n + TILE_M - 1) / TILE_M, ngroups = (ntiles + 3) / 4;
  const int tid = threadIdx.x, lane = tid & 63;
  if (tid < 28) cnt[tid] = 0;
  __syncthreads();
  // an entry's place among those of its class
  auto draw = [&](int *counter, bool valid, int c) -> int {
    uint64_t peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 5; b++) {
      const uint64_t m = __ballot((c >> b) & 1);
      peers &= ((c >> b) & 1) ? m : ~m;
    }
    const int below = __popcll(peers & ((1ull << lane) - 1ull));
    int at = 0;
    if (valid && below == 0) at = atomicAdd(&counter[c], __popcll(peers));
    return __shfl(at, peers ? __builtin_ctzll(peers) : lane, 64) + below;
  };
  auto each_tile = [&](auto f) {
    for (int64_t t0 = tid - lane; t0 < ntiles; t0 += 8 * 1024) {  // (whole wavefronts)
      unsigned m[8];
#pragma unroll
      for (int u = 0; u < 8; u++) m[u] = tmask[min(t0 + lane + u * 1024, ntiles - 1)];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int64_t t = t0 + lane + u * 1024;
        if (t - lane < ntiles) f(t, t < ntiles, 27 - __builtin_popcount(m[u] & 0x7FFFFFFu));
      }
    }
  };
  auto each_group = [&](auto f) {
    for (int64_t g0 = tid - lane; g0 < ngroups; g0 += 4 * 1024) {
      unsigned m[4][4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
#pragma unroll
        for (int q = 0; q < 4; q++) m[u][q] = tmask[min((g0 + lane + u * 1024) * 4 + q, ntiles - 1)];
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int64_t g = g0 + lane + u * 1024;
        if (g - lane < ngroups) f(g, g < ngroups, 27 - __builtin_popcount((m[u][0] | m[u][1] | m[u][2] | m[u][3]) & 0x7FFFFFFu));
      }
    }
  };
  auto count = [&](int64_t, bool valid, int c) { draw(cnt, valid, c); };
  if (groups)
    each_group(count);
  else
    each_tile(count);
  __syncthreads();
  if (tid < 28) {
    int a = 0;
#pragma unroll
    for (int c = 0; c < 27; c++) a += c < tid ? cnt[c] : 0;
    base[tid] = a;
  }
  __syncthreads();
  int32_t *const out = groups ? gsched : sched;
  auto place = [&](int64_t t, bool valid, int c) {
    const int at = draw(base, valid, c);
    if (valid) out[at] = (int32_t)t;
  };
  if (groups)
    each_group(place);
  else
    each_tile(place);
}
__global__ __launch_bounds__(1024) void tile_sched_kernel(const uint32_t *__restrict__ tmask,
                                                          const int32_t *__restrict__ d_n, int64_t n_rows,
                                                          int32_t *__restrict__ sched, int32_t *__restrict__ gsched) {
  tile_sched_body(tmask, d_n, n_rows, sched, gsched, blockIdx.y != 0);
}
__global__ __launch_bounds__(1024) void tile_sched_batch_kernel(TilePlanBatch b) {
  const TilePlanJob &j = b.job[blockIdx.x];
  if (j.sched) tile_sched_body(j.tmask, j.d_n, j.n_rows, j.sched, j.sched + (j.ld + 31) / 32, blockIdx.y != 0);
}

int build_tile_plans(const TilePlanBatch &b, hipStream_t s) {
  int64_t most = 0;
  bool any_sched = false;
  for (int i = 0; i < b.n; i++) {
    if (b.job[i].nbr) most = std::max(most, cdiv(b.job[i].n_rows, TILE_M) * TILE_M);
    any_sched = any_sched || b.job[i].sched;
  }
  if (b.n <= 0) return INSC_OK;
  if (most > 0) hipLaunchKernelGGL(tile_plan_batch_kernel, dim3(grid_for(most, 256), (unsigned)b.n), dim3(256), 0, s, b);
  if (any_sched) hipLaunchKernelGGL(tile_sched_batch_kernel, dim3((unsigned)b.n, 2), dim3(1024), 0, s, b);
  INSC_LAUNCH_CHECK();
  return INSC_OK;
}

int build_tile_plan(const int32_t *nbr, const int32_t *order, const int32_t *d_n, int64_t n_rows, int64_t ld,
                    int32_t *map, uint32_t *tmask, int32_t *sched, hipStream_t s) {
  if (n_rows <= 0) return INSC_OK;
  const int64_t padded = cdiv(n_rows, TILE_M) * TILE_M;
  hipLaunchKernelGGL(tile_plan_kernel, dim3(grid_for(padded, 256)), dim3(256), 0, s, nbr, order, d_n, n_rows, ld, map,
                     tmask);
  if (sched)
    hipLaunchKernelGGL(tile_sched_kernel, dim3(1, 2), dim3(1024), 0, s, tmask, d_n, n_rows, sched, sched + (ld + 31) / 32);
  INSC_LAUNCH_CHECK();
  return INSC_OK;
}

static bool conv_uses_mfma(const float *in, int64_t ld_in, int Cin, int K) {
  return Cin % 16 == 0 && ((uintptr_t)in % 16 == 0) && (ld_in % 4 == 0) && (K == 27 || K == 8 || K == 1);
}

int64_t packed_floats(int K, int Cin, int Cout) {
  return (int64_t)K * conv_nch(Cin) * conv_nbt_padded(Cout) * 1024;
}
int64_t split_floats(int K, int Cin, int Cout) { return packed_floats(K, Cin, Cout) / 1024 * (WT_BYTES / 4); }

static int pack_weights(const float *W, int K, int Cin, int Cout, float *Wp, hipStream_t s) {
  const int64_t total = packed_floats(K, Cin, Cout);
  hipLaunchKernelGGL(pack_weights_kernel, dim3(grid_for(total, 256, 4096)), dim3(256), 0, s, W, K, Cin, Cout,
                     conv_nch(Cin), conv_nbt_padded(Cout), Wp);
  INSC_LAUNCH_CHECK();
  return INSC_OK;
}

int split_weights(const float *W, int K, int Cin, int Cout, float *Ws, hipStream_t s) {
  const int64_t total = packed_floats(K, Cin, Cout);
  hipLaunchKernelGGL(split_weights_kernel, dim3(grid_for(total, 256, 4096)), dim3(256), 0, s, W, K, Cin, Cout,
                     conv_nch(Cin), conv_nbt_padded(Cout), reinterpret_cast<uint16_t *>(Ws));
  INSC_LAUNCH_CHECK();
  return INSC_OK;
}

// Launch policy of wide 3^3 layers (64..159 input channels, a tile schedule).  All kernels give the same
// bits; the bounds only move time.
// With at least this many (group of four tiles, output block) units, and at most two output blocks: the kernel whose blocks
// share the weight tiles through LDS.  64 -> 64, four layers with batch norms, shared / two blocks a split wavefront: 60k sites
// 282 / 268 us, 90k 346 / 391, 150k 567 / 580.  With three and four output blocks the split kernel, which gathers once for all
// or for two of them, is ahead everywhere: 96 -> 96 at 39k sites 437 / 315, at 333k 2335 / 2133, 112 -> 112 at 60k 714 / 686.
constexpr int64_t SHARED_MIN_UNITS = 1100;
static std::atomic<int64_t> g_shared_min_units{SHARED_MIN_UNITS};
// (Between the two lay a kernel with a wavefront for every (tile, output block): 64 -> 32 at 60k sites 52 us against 40 in the split
// kernel, which gathers two lanes a row as well, at 100k 74 / 63, at 200k 131 / 130; 64 -> 160 at 25k 70 / 65.)
constexpr int64_t NARROW_SPLIT_WAVES = 8192, MANY_BLOCKS_MIN_WAVES = 2400;  // (see the launch shapes below)
// Narrow 3^3 layers (Cin, Cout <= 32) with at least this many 32-row tiles run on the persistent
// kernel that keeps the whole filter in LDS; smaller ones on the one-wavefront-per-tile kernel.
// Same bits either way.
static std::atomic<int64_t> g_wl_min_tiles{WL_MIN_TILES};

// W: raw [K,Cin,Cout] weights (always needed by the generic kernel); Wp: split weights (split_ref), packed
// fp32 ones, or null, in which case the raw ones are split (or, where that layout would pass 4 GB, packed) into scratch
// memory first.
// Whether one launch can gather from two sources (BnEpilogue::src2_*): the shapes that the split
// kernel serves - 3^3 layers of a residual frame (latency != 0) and stride-2 deconvolutions, from 32
// input channels on.
bool conv_two_sources_ok(int mode, int K, const float *in, int64_t ld_in, const float *in2, int64_t ld_in2,
                         int64_t in2_rows, int Cin, int latency) {
  if (!in2 || Cin < 32 || !conv_uses_mfma(in, ld_in, Cin, K) || !conv_uses_mfma(in2, ld_in2, Cin, K)) return false;
  if (in2_rows < 0 || in2_rows * ld_in2 * 4 >= (int64_t)BUF_OOB) return false;
  return (mode == MAP_NBR && K == 27 && latency) || (mode == MAP_PARENT && K == 8);
}

int launch_conv(const float *in, int64_t ld_in, int64_t in_rows, float *out, int64_t ld_out, const float *W,
                const float *Wp, const float *bias, const int32_t *map0, const int32_t *map1, int mode, int K,
                const int32_t *rows, const int32_t *d_n_rows, int64_t n_rows, int Cin, int Cout,
                const uint8_t *tile_flags, const uint8_t *row_mask, hipStream_t s, BnEpilogue ep, TilePlan plan,
                int latency, int64_t expect_rows) {
  if (n_rows == 0) return INSC_OK;
  if (ep.side_in && !(mode == MAP_PARENT && K == 8 && conv_uses_mfma(in, ld_in, Cin, K) && ep.side_out && ep.side_w && ep.side_b)) {
    set_error("conv: a second batch norm in the epilogue is for deconvolutions on the matrix-core kernel only");
    return INSC_ERR_ARG;
  }
  if (ep.src2_in && !conv_two_sources_ok(mode, K, in, ld_in, ep.src2_in, ep.src2_ld, ep.src2_rows, Cin, latency)) {
    set_error("conv: no kernel with two sources for this shape (K=%d, map mode %d, Cin=%d)", K, mode, Cin);
    return INSC_ERR_ARG;
  }
  if (ep.src2_in) plan = TilePlan();  // (a plan describes the first source's map only)
  if (ep.pre_exist && !(ep.out2 && ep.pre_in && ep.pre_out && latency && mode == MAP_NBR && K == 27 && Cin >= 32 &&
                        conv_uses_mfma(in, ld_in, Cin, K))) {
    set_error("conv: the batch norm of a residual frame is fused into 3^3 layers on the split kernel only (Cin=%d)", Cin);
    return INSC_ERR_ARG;
  }
  if (expect_rows <= 0 || expect_rows > n_rows) expect_rows = n_rows;
  if (plan.map && (mode != MAP_NBR || K != 27 || plan.ld * 27 * 4 >= (int64_t)BUF_OOB || plan.ld < cdiv(n_rows, TILE_M) * TILE_M))
    plan = TilePlan();  // only the 3^3 map has a plan; an unusable one is ignored
  plan.cus = (unsigned)device_cus();
  if (conv_uses_mfma(in, ld_in, Cin, K)) {
    // the gather addresses rows with 32-bit byte offsets (buffer loads)
    const int64_t split_bytes = split_floats(K, Cin, Cout) * 4, packed_bytes = packed_floats(K, Cin, Cout) * 4;
    const bool pw = is_split(Wp) ? false : Wp ? true : split_bytes >= (int64_t)BUF_OOB;
    const int64_t in_bytes64 = in_rows * ld_in * 4, wp_bytes64 = pw ? packed_bytes : split_bytes;
    if (in_rows < 0 || in_bytes64 >= (int64_t)BUF_OOB || wp_bytes64 >= (int64_t)BUF_OOB) {
      set_error("conv: input matrix (%lld rows x %lld floats) or weights exceed the 4 GB the kernel addresses",
                (long long)in_rows, (long long)ld_in);
      return INSC_ERR_ARG;
    }
    const uint32_t in_bytes = (uint32_t)in_bytes64, wp_bytes = (uint32_t)wp_bytes64;
    if (is_split(Wp)) {
      Wp = split_address(Wp);
    } else if (!Wp) {
      void *ws;
      int rc = workspace(WS_API, s, (size_t)wp_bytes64, &ws);
      if (rc) return rc;
      rc = pw ? pack_weights(W, K, Cin, Cout, (float *)ws, s) : split_weights(W, K, Cin, Cout, (float *)ws, s);
      if (rc) return rc;
      Wp = (const float *)ws;
    }
    const int64_t tiles = cdiv(n_rows, TILE_M);
    // Rows of the neighbour map and of the outputs: one per listed row, or - with a row list,
    // which only 3^3 layers over one site set use - one per input site.  (The two differ when a
    // layer gathers from another site set than the one it writes.)
    const int64_t out_rows = rows ? in_rows : std::max(in_rows, n_rows);
    const int64_t map_bytes64 = out_rows * 27 * 4;
    // (row ids and row strides go through 24-bit multiplies)
    const bool small_ids = in_rows < (1 << 24) && out_rows < (1 << 24) && ld_out * 4 < (1 << 24) &&
                           ep.ld2 * 4 < (1 << 24) && out_rows * ld_out * 4 < (int64_t)BUF_OOB &&
                           out_rows * ep.ld2 * 4 < (int64_t)BUF_OOB && ep.ldr * 4 < (1 << 24) &&
                           out_rows * ep.ldr * 4 < (int64_t)BUF_OOB;
    // (below some two thousand tiles the persistent kernel's start-up - every block copies the whole filter into LDS -
    // costs more than it saves; without a plan every tile looks its offsets up first: four times as many.  Of 32 input
    // channels, split ahead, the filter takes all of LDS, one block a compute unit, and the bound is three and a half times as high: filter
    // in LDS / per tile 66k sites 41 / 27 us, 100k 47 / 38, 200k 71 / 69, 300k 108 / 112; 16 -> 32 at 66k 24 / 22, at 100k 28 / 31, 32 -> 32 with
    // packed weights 35 / 33 and 40 / 40, at 130k 46 / 53.  Both kernels give the same bits.)
    const int64_t wl_set = g_wl_min_tiles.load(std::memory_order_relaxed);
    const int64_t wl_min = Cin > 16 && !pw && plan.map ? 1 + (wl_set - 1) * 7 / 2 : wl_set;
    if (mode == MAP_NBR && K == 27 && Cin <= 32 && Cout <= 32 && map_bytes64 < (int64_t)BUF_OOB && small_ids &&
        cdiv(expect_rows, TILE_M) / (plan.map ? 1 : 4) >= wl_min && !latency) {
      const uint32_t map_bytes = (uint32_t)map_bytes64;
      // persistent blocks, a multiple of the XCD count, at most one per compute unit
      const int64_t want = cdiv(tiles, WL_WAVES);
      const unsigned nblk = (unsigned)std::min<int64_t>(device_cus(), want);
      auto kernel = Cin == 16 ? (pw ? conv_wlds_kernel<1, true> : conv_wlds_kernel<1, false>)
                              : (pw ? conv_wlds_kernel<2, true> : conv_wlds_kernel<2, false>);
      hipLaunchKernelGGL(kernel, dim3(nblk), dim3(WL_WAVES * 64), 0, s, in, ld_in, out, ld_out, Wp, bias, map0, rows,
                         d_n_rows, n_rows, Cin, Cout, tile_flags, in_bytes, map_bytes, wp_bytes, ep, plan);
      INSC_LAUNCH_CHECK();
      return INSC_OK;
    }
    const int nbt = (Cout + 31) / 32;
    // Launch shape.  How a row's sum is grouped is a function of the layer shape only (so results never depend on the scene);
    // how many wavefronts and output blocks go with that depends on the size as well.
    //  Cin < 64: two partial sums (3^3), formed by one wavefront for up to three output blocks of its tile or, in
    //    small launches, by a wavefront each and per block;
    //  wider layers sit at the coarse scales of a U-Net, which have few tiles: for 3^3 / 2^3 maps the items of a tile are
    //    dealt to S wavefronts (four for 3^3) in each of G blocks, with one output block per wavefront or,
    //    where that leaves enough wavefronts, two or three.
    // latency != 0 (residual frames: a few thousand rows at most, so a launch lasts as long as
    // its most expensive tile): the items of every 3^3 tile are dealt to four wavefronts whatever
    // the width, and to more blocks for the wide layers.
    const bool lat = latency && mode == MAP_NBR && K == 27 && Cin >= 32;
    const bool two = ep.src2_in != nullptr;  // (checked above: a shape that the split kernel serves)
    const bool split = lat || two || (Cin >= 64 && K > 1 && (mode == MAP_NBR || (mode == MAP_PARENT && Cin >= 96)));
    const int NB0 = split ? 1 : conv_nb_per_group(Cout);
    const int nbtp = conv_nbt_padded(Cout);
    int S = 1;
    const bool narrow = mode == MAP_NBR && K == 27 && !split;  // (two partial sums, whoever forms them)
    if (split) S = K == 27 ? (Cin >= 160 ? 8 : 4) : ((Cin >= 96 || two) ? 4 : 1);  // K == 8: conv and deconv
    int NB = (S == 1 && Cin >= 96) ? 1 : NB0;
    // (four blocks and two partial sums leave one wavefront a SIMD, two blocks two: 48 -> 128 without a plan at 100k sites 295 / 253 us,
    // 16 -> 112 140 / 112, with one at 60k 89 / 88 and 48 / 42)
    if (narrow && NB == 4) NB = 2;
    // (the split across blocks is for scales with few tiles; in a U-Net the width grows with the depth,
    // and a layer that narrows to at most 96 channels sits at a fine scale with many tiles)
    // (eight blocks from 224 -> 192 channels: the two coarsest scales of a seven-scale U-Net, a few tiles,
    // where a wavefront's item loop is most of the launch - 224 -> 224 at 70 sites 15 -> 12 us; at 192 input
    // channels, and for 256 -> 128 and 320 -> 160 with their more numerous tiles, it gains nothing)
    int G = (split && K == 27 && Cout > 96) ? ((Cin >= 224 && Cout >= 192) ? 8 : Cin >= 160 ? 4 : Cin >= 128 ? 2 : 1) : 1;
    if (lat) {
      G = Cin >= 128 ? 4 : Cin >= 64 ? 2 : 1;
      S = 4;
    }
    if (G > 1) S = 4;
    // A tile of a narrow layer: a wavefront for each partial sum and output block up to NARROW_SPLIT_WAVES of them, one wavefront
    // for all beyond.  Kernel times, split / not: 32 -> 32 at 6k sites 13 / 20 us, 48 -> 48 at 2k 18 / 41; four layers with
    // batch norms 48 -> 48 at 60k (7504 wavefronts) 247 / 253, 32 -> 32 at 37k 165 / 173.  (Four partial sums for two-chunk
    // layers: U-Net of 16 channels on 6k voxels 648 us and not 690, but 48 -> 48 at 150k 540 and not 424.)
    // Without a plan every wavefront stages the map by itself, and more of them than fit the chip at once are slower:
    // 32 -> 64 at 25k sites (3128) 33 / 29, 32 -> 32 at 60k (3752) 39 / 35, 48 -> 48 91 / 75, but 32 -> 32 at 40k (2500) 27 / 33.
    if (narrow && !pw && tiles * nbt * 2 <= (plan.map ? NARROW_SPLIT_WAVES : (int64_t)plan.cus * 12)) {
      S = 2;
      NB = 1;
    }
    // Wide layers: two or three output blocks a wavefront, which gathers and splits a row for all of them, while that
    // leaves MANY_BLOCKS_MIN_WAVES wavefronts.  Kernel times, several / one: 64 -> 64 at 39k sites (4848 wavefronts left) 41 /
    // 48 us, 192 -> 96 at 10k (2528) 49 / 64, 128 -> 64 at 39k (4848) 64 / 73, but
    // 96 -> 96 at 10k (1264) 37 / 32 and 128 -> 128 at 2.6k (1296) 22 / 19.
    if (mode == MAP_NBR && K == 27 && !latency && !pw) {
      const int many = S == 4 ? (nbt % 2 == 0 ? 2 : nbt % 3 == 0 ? 3 : 1) : S == 8 && nbt == 3 ? 3 : 1;
      if (many > 1 && tiles * (nbt / many) * S * G >= MANY_BLOCKS_MIN_WAVES) NB = many;
    }
    const bool wide_planned = mode == MAP_NBR && K == 27 && Cin >= 64 && S == 4 && G == 1 && !lat && plan.map && plan.sched &&
                              small_ids;
    // (Twice as high a bound for a layer with one output block, which has half the weight bytes per gathered row to share
    // (64 -> 32 at 60k sites, shared / split 60 / 39 us, at 100k 70 / 62, at 200k 137 / 137), and for the five or seven blocks that are
    // taken one a wavefront; not with packed weights.
    // Kernel times, shared / split: 64 -> 160 at 40k sites (1565 units) 101 / 99 us, 96 -> 160 144 / 138, at 60k (2345) 143 / 145 and
    // 203 / 209, at 100k 240 / 264 and 350 / 383.)
    const int64_t shared_min = g_shared_min_units.load(std::memory_order_relaxed) * (nbt == 1 || (nbt > 2 && !pw) ? 2 : 1);
    if (wide_planned && (NB == 1 || nbt == 2) && cdiv(tiles, 4) * nbt >= shared_min) {
      // blocks of four tiles that share the weight tiles through LDS
      // with enough units left, two output blocks per gathered chunk (eight accumulators: two
      // wavefronts per SIMD instead of three, but a third fewer bytes per MFMA)
      if (nbt >= 2 && cdiv(tiles, 4) * cdiv(nbt, 2) * 3 >= g_shared_min_units.load(std::memory_order_relaxed) * 2) {
        static int per_cu4_of[2] = {0, 0};
        int &per_cu4 = per_cu4_of[pw];
        auto kernel = pw ? conv_wshare_kernel<2, 4, true> : conv_wshare_kernel<2, 4, false>;
        if (!per_cu4) {
          INSC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu4, kernel, 256, 0));
          if (per_cu4 < 1) per_cu4 = 1;
        }
        const int64_t wunits = cdiv(tiles, 4) * cdiv(nbt, 2);
        const unsigned nblk = (unsigned)std::min<int64_t>((int64_t)device_cus() * per_cu4, wunits);
        hipLaunchKernelGGL(kernel, dim3(nblk), dim3(256), 0, s, in, ld_in, out, ld_out, Wp, bias, rows,
                           d_n_rows, n_rows, Cin, Cout, nbt, nbtp, tile_flags, in_bytes, wp_bytes, ep, plan);
        INSC_LAUNCH_CHECK();
        return INSC_OK;
      }
      static int per_cu2_of[2] = {0, 0};
      int &per_cu2 = per_cu2_of[pw];
      auto kernel = pw ? conv_wshare_kernel<1, 4, true> : conv_wshare_kernel<1, 4, false>;
      if (!per_cu2) {
        INSC_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu2, kernel, 256, 0));
        if (per_cu2 < 1) per_cu2 = 1;
      }
      const int64_t wunits = cdiv(tiles, 4) * nbt;
      const unsigned nblk = (unsigned)std::min<int64_t>((int64_t)device_cus() * per_cu2, wunits);
      hipLaunchKernelGGL(kernel, dim3(nblk), dim3(256), 0, s, in, ld_in, out, ld_out, Wp, bias, rows,
                         d_n_rows, n_rows, Cin, Cout, nbt, nbtp, tile_flags, in_bytes, wp_bytes, ep, plan);
      INSC_LAUNCH_CHECK();
      return INSC_OK;
    }
    const unsigned gx = (unsigned)(S == 1 ? cdiv(tiles, CONV_WAVES) : tiles);
    const int GZ = two ? 2 * G : G;  // blocks per (tile, output block): G per source
    dim3 grid(gx, (unsigned)cdiv(nbt, NB), (unsigned)GZ), block((S == 1 ? CONV_WAVES : S) * 64);
    float *part = nullptr;
    int32_t *pcount = nullptr;
    if (GZ > 1) {
      const size_t units = (size_t)gx * grid.y;
      void *ws;
      int rc = workspace(WS_CONV, s, units * GZ * NB * 1024 * sizeof(float), &ws);
      if (rc) return rc;
      part = (float *)ws;
      if ((rc = zero_counters(s, units * (size_t)S, &pcount))) return rc;  // one counter per wavefront of a unit
    }
    bool shape_ok = true;
    // (two lanes a row from one wavefront per SIMD on; layers of a residual frame are short whatever their grids)
    const bool pairs = !latency && (int64_t)grid.x * grid.y * grid.z * (block.x / 64) >= (int64_t)plan.cus * 4;
#define INSC_CONV_LAUNCH(NBV, KV, MV, SV)                                                                       \
  hipLaunchKernelGGL((pw ? conv_mfma_kernel<NBV, KV, MV, SV, true, false> : pairs ? conv_mfma_kernel<NBV, KV, MV, SV, false, true> : conv_mfma_kernel<NBV, KV, MV, SV, false, false>), grid, block, 0, s, in, ld_in, out, ld_out, Wp, bias,  \
                     map0, map1, rows, d_n_rows, n_rows, Cin, Cout, nbtp, tile_flags, in_bytes, wp_bytes, ep, part,  \
                     pcount, plan)
#define INSC_CONV_LAUNCH_MANY(NBV, SV)                                                                            \
  hipLaunchKernelGGL((conv_mfma_kernel<NBV, 27, MAP_NBR, SV, false, true>), grid, block, 0, s, in, ld_in, out, ld_out, Wp, bias,  \
                     map0, map1, rows, d_n_rows, n_rows, Cin, Cout, nbtp, tile_flags, in_bytes, wp_bytes, ep, part,  \
                     pcount, plan)
#define INSC_CONV_CASE(NBV)                                      \
  case NBV:                                                      \
    if (mode == MAP_NBR && K == 27)                              \
      INSC_CONV_LAUNCH((NBV > 3 ? 2 : NBV), 27, MAP_NBR, 1);     \
    else if (mode == MAP_NBR && K == 8)                          \
      INSC_CONV_LAUNCH(NBV, 8, MAP_NBR, 1);                      \
    else if (mode == MAP_PARENT && K == 8)                       \
      INSC_CONV_LAUNCH(NBV, 8, MAP_PARENT, 1);                   \
    else if (mode == MAP_IDENTITY && K == 1)                     \
      INSC_CONV_LAUNCH(NBV, 1, MAP_IDENTITY, 1);                 \
    else                                                         \
      shape_ok = false;                                          \
    break;
    if (S > 1 && mode == MAP_NBR && K == 27) {
      switch (S) {
        case 2: INSC_CONV_LAUNCH(1, 27, MAP_NBR, 2); break;
        case 4:
          if (NB == 1) INSC_CONV_LAUNCH(1, 27, MAP_NBR, 4);
          else if (NB == 2) INSC_CONV_LAUNCH_MANY(2, 4);
          else INSC_CONV_LAUNCH_MANY(3, 4);
          break;
        case 8:
          if (NB == 3) INSC_CONV_LAUNCH_MANY(3, 8);
          else INSC_CONV_LAUNCH(1, 27, MAP_NBR, 8);
          break;
        default: shape_ok = false;
      }
    } else if (S > 1 && mode == MAP_NBR && K == 8) {
      switch (S) {
        case 4: INSC_CONV_LAUNCH(1, 8, MAP_NBR, 4); break;
        default: shape_ok = false;
      }
    } else if (S == 4 && mode == MAP_PARENT && K == 8) {
      INSC_CONV_LAUNCH(1, 8, MAP_PARENT, 4);
    } else if (S > 1) {
      shape_ok = false;
    } else {
      switch (NB) {
        INSC_CONV_CASE(1)
        INSC_CONV_CASE(2)
        INSC_CONV_CASE(3)
        INSC_CONV_CASE(4)
        default:
          shape_ok = false;
      }
    }
    if (!shape_ok) {
      set_error("conv: no matrix-core kernel for K=%d with map mode %d", K, mode);
      return INSC_ERR_ARG;
    }
#undef INSC_CONV_LAUNCH
#undef INSC_CONV_LAUNCH_MANY
#undef INSC_CONV_CASE
  } else {
    if (!W) {
      set_error("conv: this shape (Cin=%d) runs on the generic kernel, which needs the unpacked weights", Cin);
      return INSC_ERR_ARG;
    }
    if (Cout > 256) {
      set_error("conv: Cout=%d > 256 is not supported for Cin=%d", Cout, Cin);
      return INSC_ERR_ARG;
    }
    const int cpb = 256 / Cout;
    if (mode == MAP_NBR && K == 27 && Cin <= 4) {
      // enough blocks to fill the machine, few enough that the weights are fetched rarely
      const dim3 sg(grid_for(n_rows, std::min(cpb, STEM_ROWS), (unsigned)device_cus() * 8));
#define INSC_STEM(...)                                                                                         \
  hipLaunchKernelGGL((__VA_ARGS__), sg, dim3(256), 0, s, in, ld_in, out, ld_out, W, bias, map0, rows, d_n_rows, n_rows, Cout, row_mask, ep)
      // A batch ahead or batch by batch (same bits).  Up to 256 (row, offset) pairs a batch, one a thread: with three channels
      // always ahead (3 -> 32, us batch by batch / ahead: 6k rows 6.7 / 6.3, 37k 17.9 / 15.6, 400k 131 / 87); with two or four from
      // some five batches a block (2 -> 64: 37k rows, four batches, 20.1 / 21.6, 100k, twelve, 52.5 / 47.5; 4 -> 64: 37k 32.0 /
      // 32.6, 100k 82 / 70); with one, whose batches are short, from twelve (1 -> 32: 100k 20.4 / 20.2, 400k 63.8 / 58.7).
      // Two pairs a thread: ahead with two channels (2 -> 16: 37k 11.0 / 12.4, 100k 23.1 / 22.7, 400k 80 / 65), else batch by
      // batch (1 -> 16: 37k 7.7 / 10.3, 400k 45 / 57; 3 -> 16: 37k 12.5 / 16.7, 400k 82 / 87; 4 -> 16: 37k 18.7 / 24.1, 400k 125 / 119).
      const int batch = std::min(cpb, STEM_ROWS);
      const int64_t batches = expect_rows / ((int64_t)batch * sg.x);  // of a block
      const bool two = batch * 27 > 256;
      if (Cin == 1) {
        if (!two && batches >= 12) INSC_STEM(conv_stem_ahead_kernel<1, 1>);
        else INSC_STEM(conv_stem_kernel<1>);
      } else if (Cin == 2) {
        if (batches < 5) INSC_STEM(conv_stem_kernel<2>);
        else if (two) INSC_STEM(conv_stem_ahead_kernel<2, 2>);
        else INSC_STEM(conv_stem_ahead_kernel<2, 1>);
      } else if (Cin == 3) {
        if (!two) INSC_STEM(conv_stem_ahead_kernel<3, 1>);
        else INSC_STEM(conv_stem_kernel<3>);
      } else {
        if (!two && batches >= 5) INSC_STEM(conv_stem_ahead_kernel<4, 1>);
        else INSC_STEM(conv_stem_kernel<4>);
      }
#undef INSC_STEM
      INSC_LAUNCH_CHECK();
      return INSC_OK;
    }
    hipLaunchKernelGGL(conv_generic_kernel, dim3(grid_for(n_rows, cpb, 65536)), dim3(256), 0, s, in, ld_in, out,
                       ld_out, W, bias, map0, map1, mode, K, rows, d_n_rows, n_rows, Cin, Cout, row_mask, ep);
  }
  INSC_LAUNCH_CHECK();
  return INSC_OK;
}

}  // namespace insc

using namespace insc;

extern "C" {

// (bounds are held to what the rules can multiply: "never" may be asked for as the largest integer)
constexpr int64_t BOUND_MAX = int64_t(1) << 48;

// (this and the next but one are kept for callers: the kernels that these bounds chose were the slower ones at every size and are gone)
int insc_conv_set_persistent_min_units(int64_t units) {
  INSC_REQUIRE(units >= 1, INSC_ERR_ARG, "insc_conv_set_persistent_min_units: units must be >= 1");
  return INSC_OK;
}

int insc_conv_set_shared_weights_min_units(int64_t units) {
  INSC_REQUIRE(units >= 1, INSC_ERR_ARG, "insc_conv_set_shared_weights_min_units: units must be >= 1");
  g_shared_min_units.store(std::min(units, BOUND_MAX), std::memory_order_relaxed);
  return INSC_OK;
}

int insc_conv_set_wavefront_per_unit_min_units(int64_t units) {
  INSC_REQUIRE(units >= 1, INSC_ERR_ARG, "insc_conv_set_wavefront_per_unit_min_units: units must be >= 1");
  return INSC_OK;
}

int insc_conv_set_filter_lds_min_tiles(int64_t tiles) {
  INSC_REQUIRE(tiles >= 1, INSC_ERR_ARG, "insc_conv_set_filter_lds_min_tiles: tiles must be >= 1");
  g_wl_min_tiles.store(std::min(tiles, BOUND_MAX), std::memory_order_relaxed);
  return INSC_OK;
}

int insc_conv_reset_launch_policy(void) {
  g_shared_min_units.store(SHARED_MIN_UNITS, std::memory_order_relaxed);
  g_wl_min_tiles.store(WL_MIN_TILES, std::memory_order_relaxed);
  return INSC_OK;
}

int64_t insc_conv_packed_floats(int K, int Cin, int Cout) {
  if (K <= 0 || Cin <= 0 || Cout <= 0) return 0;
  return packed_floats(K, Cin, Cout);
}

int insc_conv_pack_weights(const float *d_W, int K, int Cin, int Cout, float *d_Wp, void *stream) {
  INSC_REQUIRE(d_W && d_Wp && K > 0 && K <= MAXK && Cin > 0 && Cout > 0, INSC_ERR_ARG,
               "insc_conv_pack_weights: bad arguments");
  return pack_weights(d_W, K, Cin, Cout, d_Wp, (hipStream_t)stream);
}

int64_t insc_conv_split_floats(int K, int Cin, int Cout) {
  if (K <= 0 || Cin <= 0 || Cout <= 0) return 0;
  return split_floats(K, Cin, Cout);
}

int insc_conv_split_weights(const float *d_W, int K, int Cin, int Cout, float *d_Ws, void *stream) {
  INSC_REQUIRE(d_W && d_Ws && K > 0 && K <= MAXK && Cin > 0 && Cout > 0 && ((uintptr_t)d_Ws & 15) == 0, INSC_ERR_ARG,
               "insc_conv_split_weights: bad arguments");
  return split_weights(d_W, K, Cin, Cout, d_Ws, (hipStream_t)stream);
}

int insc_conv_nbr(const float *d_in, int64_t ld_in, int64_t n_in_rows, float *d_out, int64_t ld_out,
                  const float *d_W, const float *d_Wp, const float *d_bias, const int32_t *d_nbr, int K,
                  const int32_t *d_rows, const int32_t *d_n_rows, int64_t n_rows, int Cin, int Cout,
                  double *h_muladds, void *stream) {
  INSC_REQUIRE(n_rows >= 0 && Cin > 0 && Cout > 0 && K > 0 && K <= MAXK, INSC_ERR_ARG,
               "insc_conv_nbr: bad sizes (n_rows=%lld Cin=%d Cout=%d K=%d)", (long long)n_rows, Cin, Cout, K);
  INSC_REQUIRE(ld_in >= Cin && ld_out >= Cout, INSC_ERR_ARG, "insc_conv_nbr: row stride smaller than channel count");
  INSC_REQUIRE(n_rows == 0 || (d_in && d_out && (d_W || d_Wp)), INSC_ERR_ARG, "insc_conv_nbr: null pointer");
  INSC_REQUIRE(d_nbr || K == 1, INSC_ERR_ARG, "insc_conv_nbr: a null map needs K == 1");
  hipStream_t s = (hipStream_t)stream;
  INSC_REQUIRE(n_in_rows >= 0, INSC_ERR_ARG, "insc_conv_nbr: n_in_rows is negative");
  int rc = launch_conv(d_in, ld_in, n_in_rows, d_out, ld_out, d_W, d_Wp, d_bias, d_nbr, nullptr,
                       d_nbr ? MAP_NBR : MAP_IDENTITY, K, d_rows, d_n_rows, n_rows, Cin, Cout, nullptr, nullptr, s);
  if (rc) return rc;
  if (h_muladds) {
    unsigned long long h = 0;
    if (n_rows > 0 && d_nbr) {
      void *ws;
      rc = workspace(WS_API, s, 256, &ws);
      if (rc) return rc;
      rc = insc_fill_i32((int32_t *)ws, 2, 0, stream);
      if (rc) return rc;
      hipLaunchKernelGGL(count_rules_kernel, dim3(grid_for(n_rows, 256)), dim3(256), 0, s, d_nbr, K, d_rows, d_n_rows,
                         n_rows, (unsigned long long *)ws);
      INSC_LAUNCH_CHECK();
      INSC_HIP(hipMemcpyAsync(&h, ws, 8, hipMemcpyDeviceToHost, s));
      INSC_HIP(hipStreamSynchronize(s));
    } else if (n_rows > 0) {
      int32_t hn = (int32_t)n_rows;
      if (d_n_rows) {
        INSC_HIP(hipMemcpyAsync(&hn, d_n_rows, 4, hipMemcpyDeviceToHost, s));
        INSC_HIP(hipStreamSynchronize(s));
      }
      h = (unsigned long long)hn;
    }
    *h_muladds = (double)h * Cin * Cout;
  }
  return INSC_OK;
}

int insc_plan_build(const int32_t *d_nbr, const int32_t *d_order, const int32_t *d_n_rows, int64_t n_rows,
                    int64_t plan_ld, int32_t *d_plan, uint32_t *d_tmask, int32_t *d_sched, void *stream) {
  INSC_REQUIRE(n_rows >= 0 && plan_ld >= cdiv(n_rows, TILE_M) * TILE_M, INSC_ERR_ARG,
               "insc_plan_build: plan_ld must cover the rows rounded up to a multiple of 32");
  INSC_REQUIRE(n_rows == 0 || (d_nbr && d_plan && d_tmask), INSC_ERR_ARG, "insc_plan_build: null pointer");
  return build_tile_plan(d_nbr, d_order, d_n_rows, n_rows, plan_ld, d_plan, d_tmask, d_sched, (hipStream_t)stream);
}

int insc_conv_ssc_plan(const float *d_in, int64_t ld_in, int64_t n_in_rows, float *d_out, int64_t ld_out,
                       const float *d_W, const float *d_Wp, const float *d_bias, const int32_t *d_nbr,
                       const int32_t *d_plan, int64_t plan_ld, const uint32_t *d_tmask, const int32_t *d_sched,
                       const int32_t *d_order, const int32_t *d_n_rows, int64_t n_rows, int Cin, int Cout,
                       void *stream) {
  INSC_REQUIRE(n_rows >= 0 && Cin > 0 && Cout > 0 && n_in_rows >= 0, INSC_ERR_ARG, "insc_conv_ssc_plan: bad sizes");
  INSC_REQUIRE(ld_in >= Cin && ld_out >= Cout, INSC_ERR_ARG, "insc_conv_ssc_plan: row stride smaller than channel count");
  INSC_REQUIRE(n_rows == 0 || (d_in && d_out && (d_W || d_Wp) && d_nbr && d_plan && d_tmask), INSC_ERR_ARG,
               "insc_conv_ssc_plan: null pointer");
  INSC_REQUIRE(plan_ld >= cdiv(n_rows, TILE_M) * TILE_M, INSC_ERR_ARG, "insc_conv_ssc_plan: plan_ld too small");
  TilePlan plan;
  plan.map = d_plan;
  plan.ld = plan_ld;
  plan.tmask = d_tmask;
  plan.sched = d_sched;
  return launch_conv(d_in, ld_in, n_in_rows, d_out, ld_out, d_W, d_Wp, d_bias, d_nbr, nullptr, MAP_NBR, 27, d_order,
                     d_n_rows, n_rows, Cin, Cout, nullptr, nullptr, (hipStream_t)stream, BnEpilogue(), plan);
}

int insc_deconv_down2(const float *d_in, int64_t ld_in, int64_t n_in_rows, float *d_out, int64_t ld_out,
                      const float *d_W, const float *d_Wp, const float *d_bias, const int32_t *d_parent,
                      const int32_t *d_offset, const int32_t *d_rows, const int32_t *d_n_rows, int64_t n_rows,
                      int Cin, int Cout, void *stream) {
  INSC_REQUIRE(n_rows >= 0 && Cin > 0 && Cout > 0, INSC_ERR_ARG, "insc_deconv_down2: bad sizes");
  INSC_REQUIRE(ld_in >= Cin && ld_out >= Cout, INSC_ERR_ARG, "insc_deconv_down2: row stride too small");
  INSC_REQUIRE(n_rows == 0 || (d_in && d_out && (d_W || d_Wp) && d_parent && d_offset), INSC_ERR_ARG,
               "insc_deconv_down2: null pointer");
  INSC_REQUIRE(n_in_rows >= 0, INSC_ERR_ARG, "insc_deconv_down2: n_in_rows is negative");
  return launch_conv(d_in, ld_in, n_in_rows, d_out, ld_out, d_W, d_Wp, d_bias, d_parent, d_offset, MAP_PARENT, 8, d_rows,
                     d_n_rows, n_rows, Cin, Cout, nullptr, nullptr, (hipStream_t)stream);
}

}  // extern "C"
