// Block floats on the GPU: the cast into the plain planes, the exact unpacker, and the one-time repack into the
// columns tiles that the matmul kernels read.
//
// Rules (restated from the reference, in code of our own):
//   cast   models/gpt2.py:19-30, kernels.py:1074-1081 (NIBBLE), kernels.py:1108-1114 (put's bfp8 rule): round to bf16
//          (nearest even), take the run's largest exponent field `top`, keep 7 (bfp8) or 3 (bfp4) bits of magnitude
//          below it, rounding half up (bfp8) or to nearest with ties up (bfp4), saturating at 127 / 7. A zero keeps no
//          sign.
//   decode tensor.py:1093-1104 (_bf16s): normalize the magnitude, exponent (e - shift) mod 256.
#include "common.h"

namespace bt {

// A run of 16 bf16 values with its largest exponent field `top` into the plain planes: the exponent byte, then the
// 16 signed magnitudes (bfp8: a byte each; bfp4: two to a byte, the first in the low nibble).
template <int FMT>
__device__ __forceinline__ void store_run(const uint32_t (&bits)[16], uint32_t top, uint8_t *exp, uint8_t *val) {
  *exp = (uint8_t)top;
  if (FMT == BT_BFP8) {
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) w[i / 4] |= ((uint32_t)bfp_signed<8>(bits[i], top) & 255u) << (8 * (i % 4));
    *(uint4 *)val = make_uint4(w[0], w[1], w[2], w[3]);
  } else {
    uint32_t w[2] = {0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) w[i / 8] |= ((uint32_t)bfp_signed<4>(bits[i], top) & 15u) << (4 * (i % 8));
    *(uint2 *)val = make_uint2(w[0], w[1]);
  }
}

// One thread a run: 16 values of one row sharing an exponent, at any column stride (a transposed view).
template <int FMT>
__global__ void __launch_bounds__(256) pack_kernel(const void *src, int src_dtype, int64_t batch, int64_t rows,
                                                   int64_t cols, int64_t sb, int64_t sr, int64_t sc, uint8_t *exps,
                                                   uint8_t *vals) {
  int64_t runs = (cols + 15) / 16;
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= batch * rows * runs) return;
  int64_t j = t % runs, r = t / runs % rows, b = t / runs / rows;
  uint32_t bits[16];
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    int64_t c = j * 16 + i;
    uint32_t v = 0;
    if (c < cols) {
      int64_t at = b * sb + r * sr + c * sc;
      v = src_dtype == BT_BF16 ? ((const uint16_t *)src)[at] : bf16_rne(((const float *)src)[at]);
    }
    bits[i] = v;
    top = max(top, (v >> 7) & 255u);
  }
  store_run<FMT>(bits, top, exps + t, vals + t * (FMT == BT_BFP8 ? 16 : 8));
}

// The same for contiguous columns: two neighbouring threads a run, 8 values each, so that every load of a wave is one
// contiguous stretch (a thread a run reads 32 bytes apart, value by value). The bound is HBM: 2 bytes read and 1 1/16
// (bfp8) or 9/16 (bfp4) written a value. Loads of A bytes, the widest that every row's start is aligned to; a piece
// that crosses the row's end goes value by value. 4096 x 14336 bf16 to bfp4 (154 MB): 107 us with a thread a
// run, 41 us so (3.7 TB/s).
template <int FMT, int SRC, int A>
__global__ void __launch_bounds__(256) pack_half_kernel(const void *src, uint32_t halves, FastDiv runs, FastDiv rows,
                                                        int64_t cols, int64_t sb, int64_t sr, uint8_t *exps,
                                                        uint8_t *vals) {
  constexpr int SIZE = SRC == BT_BF16 ? 2 : 4, W = SIZE * 2;  // words of 4 bytes a piece
  typedef uint32_t words __attribute__((ext_vector_type(W)));
  const uint32_t t = blockIdx.x * 256u + threadIdx.x, u = min(t, halves - 1u);  // every lane stays, for the exchange
  const uint32_t run = u >> 1, br = fdiv(run, runs), b = fdiv(br, rows);
  const int64_t c0 = (int64_t)(run - br * runs.d) * 16 + 8 * (u & 1u);
  const uint8_t *p = (const uint8_t *)src + ((int64_t)b * sb + (int64_t)(br - b * rows.d) * sr + c0) * SIZE;
  uint32_t bits[8];
  if (c0 + 8 <= cols) {
    words w;
    if constexpr (A >= 4) {
      typedef uint32_t piece __attribute__((ext_vector_type(A / 4)));
#pragma unroll
      for (int i = 0; i < 4 * W / A; i++) {
        const piece x = ((const piece *)p)[i];
#pragma unroll
        for (int k = 0; k < A / 4; k++) w[i * (A / 4) + k] = x[k];
      }
    } else {
#pragma unroll
      for (int i = 0; i < W; i++) w[i] = ((const uint16_t *)p)[2 * i] | (uint32_t)((const uint16_t *)p)[2 * i + 1] << 16;
    }
#pragma unroll
    for (int i = 0; i < 8; i++)
      bits[i] = SRC == BT_BF16 ? w[i / 2 % W] >> (16 * (i & 1)) & 0xFFFFu : bf16_rne(__uint_as_float(w[i % W]));
  } else {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      bits[i] = 0;
      if (c0 + i < cols) bits[i] = SRC == BT_BF16 ? ((const uint16_t *)p)[i] : bf16_rne(((const float *)p)[i]);
    }
  }
  uint32_t top = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) top = max(top, bits[i] >> 7 & 255u);
  top = max(top, (uint32_t)__builtin_amdgcn_update_dpp((int)top, (int)top, 0xB1, 0xF, 0xF, false));  // the run's other half
  if (t >= halves) return;
  uint32_t w[2] = {0, 0};
#pragma unroll
  for (int i = 0; i < 8; i++) {
    if (FMT == BT_BFP8) w[i / 4] |= ((uint32_t)bfp_signed<8>(bits[i], top) & 255u) << (8 * (i % 4));
    else w[0] |= ((uint32_t)bfp_signed<4>(bits[i], top) & 15u) << (4 * i);
  }
  if (FMT == BT_BFP8) *(uint2 *)(vals + (int64_t)t * 8) = make_uint2(w[0], w[1]);
  else *(uint32_t *)(vals + (int64_t)t * 4) = w[0];
  if (!(t & 1u)) exps[t >> 1] = (uint8_t)top;
}

// One row of x (bf16) put into a plain block-float tensor at each place (Tensor.put into a block-float cache,
// kernels.py:1083-1168): a block a row of x, a thread a run of 16 of it in every batch entry, rounded as the cast
// rounds. A later duplicate place wins: the block first looks for a j > i with the same place. Strides are in
// values (multiples of 16); the planes hold a value's exponent byte at its index / 16 and its q at its index (bfp8)
// or index / 2 (bfp4).
template <int FMT>
__global__ void __launch_bounds__(256) put_bfp_kernel(uint8_t *exps, uint8_t *vals, int64_t dst_rows, int64_t cols,
                                                      int64_t dst_sb, int64_t dst_sr, const int32_t *ids, int64_t n,
                                                      const uint16_t *x, int64_t x_sb, int64_t x_sr, int64_t batch) {
  __shared__ int later;
  const int64_t i = blockIdx.x;
  const int32_t p = ids[i];
  if (p < 0 || p >= dst_rows) return;
  if (threadIdx.x == 0) later = 0;
  __syncthreads();
  bool found = false;
  for (int64_t j = i + 1 + threadIdx.x; j < n; j += blockDim.x) found |= ids[j] == p;
  if (found) later = 1;
  __syncthreads();
  if (later) return;
  const int64_t runs = cols / 16;
  for (int64_t e = threadIdx.x; e < batch * runs; e += blockDim.x) {
    const int64_t b = e / runs, j = e % runs;
    const uint16_t *src = x + b * x_sb + i * x_sr + j * 16;
    uint32_t bits[16], top = 0;
#pragma unroll
    for (int k = 0; k < 16; k++) bits[k] = src[k], top = max(top, (bits[k] >> 7) & 255u);
    const int64_t at = b * dst_sb + (int64_t)p * dst_sr + j * 16;  // the run's first value
    store_run<FMT>(bits, top, exps + at / 16, vals + (FMT == BT_BFP8 ? at : at / 2));
  }
}

// Counts, into *bad, the runs of the plain planes that hold a nonzero value under an exponent the matmul kernels can't
// read: they take the exponent byte as the signed power (e - 133) (bfp8) or (e - 120) (bfp4), so bfp8 needs e >= 5 and
// bfp4 e <= 247; and a bfp4 B decoded in registers needs e >= 3, where every value is a normal bf16. A run of zeros
// multiplies to zero under any exponent, so it never counts. One thread a run.
template <int FMT>
__global__ void __launch_bounds__(256) range_kernel(const uint8_t *exps, const uint8_t *vals, int64_t runs,
                                                   uint32_t *bad) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= runs) return;
  const uint32_t e = exps[t];
  if (FMT == BT_BFP8 ? e >= 5u : e >= 3u && e <= 247u) return;
  uint32_t any = 0;
  if (FMT == BT_BFP8) {
    const uint4 v = *(const uint4 *)(vals + t * 16);
    any = v.x | v.y | v.z | v.w;
  } else {
    const uint2 v = *(const uint2 *)(vals + t * 8);
    any = v.x | v.y;
  }
  if (any) atomicAdd(bad, 1u);
}

__global__ void zero_word_kernel(uint32_t *word) {
  if (threadIdx.x == 0) word[0] = 0;
}

// Signed q of value c in row r of matrix b of the plain planes.
template <int FMT>
__device__ __forceinline__ int plain_q(const uint8_t *vals, int64_t row_bytes, int64_t b_rows_r, int64_t c) {
  if (FMT == BT_BFP8) return (int)(int8_t)vals[b_rows_r * row_bytes + c];
  uint32_t byte = vals[b_rows_r * row_bytes + c / 2];
  int nib = (int)((byte >> (4 * (c & 1))) & 15u);
  return nib >= 8 ? nib - 16 : nib;
}

// One thread a value: bf16 bits exactly as the unpacker gives them.
template <int FMT>
__global__ void __launch_bounds__(256) unpack_kernel(const uint8_t *exps, const uint8_t *vals, int64_t batch,
                                                     int64_t rows, int64_t cols, uint16_t *dst) {
  int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= batch * rows * cols) return;
  int64_t c = t % cols, br = t / cols;  // br = b * rows + r
  int64_t runs = (cols + 15) / 16, cols16 = runs * 16;
  int q = plain_q<FMT>(vals, FMT == BT_BFP8 ? cols16 : cols16 / 2, br, c);
  uint32_t e = exps[br * runs + c / 16];
  dst[t] = (uint16_t)unpacked_bits(FMT == BT_BFP8 ? q : q * 16, e);
}

// Row of exponent byte p of a columns tile, and row of value j (of 8) for lane l, half h.
__device__ __forceinline__ int tile_row_of_exp(int p) { return 32 * ((p >> 3) & 1) + 8 * (p >> 4) + (p & 7); }
__device__ __forceinline__ int tile_row(int l, int h, int j) { return 32 * h + 8 * (l >> 4) + j; }

// A columns tile keeps each run's exponent as d = (e - bias) mod 256, read by the matmul as a signed byte: the
// power of two it applies to the integer magnitude (bfp8: q * 2^d) or to q * 2^-9, what a bfp4 value's fp8 form
// converts to (bfp4: q * 2^-9 * 2^d). The map is a bijection, so readback recovers e exactly.
template <int FMT> __device__ __forceinline__ uint32_t exp_bias() { return FMT == BT_BFP8 ? 133u : 120u; }

// Where value j (0..7) of a lane's half sits in its 4 bytes of a bfp4 columns tile, as sign and magnitude: for j < 4
// byte j's bit 7 and bits 0-2; for j >= 4 bits 4-6 of byte j - 4 and bit 3 of byte (j - 3) % 4. The matmul reads
// these as fp8 bytes with one mask, and with one rotate and a mask.
__device__ __forceinline__ uint32_t nibble_bits(int q, int j) {
  const uint32_t mag = (uint32_t)(q < 0 ? -q : q), sgn = q < 0 ? 1u : 0u;
  return j < 4 ? mag << (8 * j) | sgn << (8 * j + 7) : mag << (8 * (j - 4) + 4) | sgn << (8 * ((j - 3) & 3) + 3);
}
__device__ __forceinline__ int nibble_q(uint32_t w, int j) {  // the inverse: value j's signed q from the 4 bytes
  const uint32_t mag = (w >> (j < 4 ? 8 * j : 8 * (j - 4) + 4)) & 7u;
  const uint32_t sgn = (w >> (j < 4 ? 8 * j + 7 : 8 * ((j - 3) & 3) + 3)) & 1u;
  return sgn ? -(int)mag : (int)mag;
}

// A block re-lays 16 neighbouring runs of one 64-row chunk through LDS: it reads the chunk's rows as whole stretches of
// the planes (a run's 8 or 16 bytes a thread, 128 or 256 bytes a row), and each of its 4 waves then gathers 4 tiles from
// LDS and writes each as one contiguous stretch. One block a tile, each lane fetching its 16 values a byte at a time from
// 16 rows, left the loads' lines mostly unused. The bound is HBM: 9/16 (bfp4) or 17/16 (bfp8) bytes a value each way.
// LDS rows are 8 bytes longer than their runs, so that the 4 lane groups' rows, 8 apart, start 16 banks apart. WIDE: the
// value plane starts on 8 bytes (it is byte addressed otherwise). 4096 x 14336 in bfp4: 53 us a block a tile, 25 us so
// (2.9 TB/s). RUNS: the block's runs; 4, a tile a wave, where there would be fewer than 256 blocks of 16, each a chain of
// 4 tiles a wave (bfp4, 15 x 1817: 3.9 us on 16 runs, 3.3 a block a tile, 2.4 on 4; 1024 x 2048 4.5, 5.1 and 2.8).
constexpr int RUNS_B = 16;
template <int FMT, bool WIDE, int RUNS>
__global__ void __launch_bounds__(256) columns_kernel(const uint8_t *exps, const uint8_t *vals, int64_t rows,
                                                      uint32_t runs, uint32_t chunks, FastDiv groups, FastDiv chunks_d,
                                                      uint8_t *dst) {
  constexpr int TB = FMT == BT_BFP8 ? 1088 : 576, RB = FMT == BT_BFP8 ? 16 : 8, S = RUNS * RB + 8;
  __shared__ __attribute__((aligned(16))) uint8_t lv[64 * S];
  __shared__ __attribute__((aligned(16))) uint8_t le[RUNS][64];  // a tile's exponent bytes, as it stores them
  const uint32_t q = fdiv(blockIdx.x, groups), b = fdiv(q, chunks_d), chunk = q - b * chunks, run0 = (blockIdx.x - q * groups.d) * RUNS;
  const int t = threadIdx.x;
  const int64_t k0 = (int64_t)chunk * 64;
#pragma unroll
  for (int i = 0; i < RUNS / 4; i++) {
    const int row = t / RUNS + 256 / RUNS * i, run = t % RUNS;
    const bool in = k0 + row < rows && run0 + run < runs;
    const int64_t at = ((int64_t)b * rows + k0 + row) * runs + run0 + run;  // the run's number in the planes
    uint2 w[RB / 8];
#pragma unroll
    for (int k = 0; k < RB / 8; k++) {
      w[k] = make_uint2(0, 0);
      if (!in) continue;
      const uint8_t *p = vals + at * RB + 8 * k;
      if (WIDE) w[k] = *(const uint2 *)p;
      else w[k] = make_uint2(p[0] | p[1] << 8 | p[2] << 16 | (uint32_t)p[3] << 24, p[4] | p[5] << 8 | p[6] << 16 | (uint32_t)p[7] << 24);
    }
    const uint32_t e = in ? exps[at] : 0u;
    le[run][16 * (row >> 3 & 3) + 8 * (row >> 5) + (row & 7)] = (uint8_t)(e - exp_bias<FMT>());
#pragma unroll
    for (int k = 0; k < RB / 8; k++) *(uint2 *)(lv + row * S + run * RB + 8 * k) = w[k];
  }
  __syncthreads();
  const int l = t & 63, n = l & 15;
#pragma unroll
  for (int i = 0; i < RUNS / 4; i++) {
    const uint32_t run = (t >> 6) + 4 * i;
    if (run0 + run >= runs) break;  // uniform in the wave
    uint8_t *out = dst + ((int64_t)((int64_t)b * runs + run0 + run) * chunks + chunk) * TB;
    if (l < 16) ((uint32_t *)out)[l] = ((const uint32_t *)le[run])[l];
    uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const uint8_t *p = lv + tile_row(l, h, j) * S + run * RB;
        if (FMT == BT_BFP8) w[(h * 8 + j) / 4] |= (uint32_t)p[n] << (8 * (j % 4));
        else w[h] |= nibble_bits((int32_t)((uint32_t)p[n / 2] << (28 - 4 * (n & 1))) >> 28, j);
      }
    if (FMT == BT_BFP8) *(uint4 *)(out + 64 + 16 * l) = make_uint4(w[0], w[1], w[2], w[3]);
    else *(uint2 *)(out + 64 + 8 * l) = make_uint2(w[0], w[1]);
  }
}

__global__ void __launch_bounds__(64) bf16_columns_kernel(const uint16_t *src, int64_t rows, int64_t cols, int64_t sb,
                                                          int64_t sr, int64_t sc, int64_t chunks, int64_t nruns,
                                                          uint16_t *dst) {
  int64_t tile = blockIdx.x;
  int64_t chunk = tile % chunks, run = tile / chunks % nruns, b = tile / chunks / nruns;
  int l = threadIdx.x;
  int64_t n = run * 16 + (l & 15);
  uint32_t w[8];
#pragma unroll
  for (int i = 0; i < 16; i += 2) {
    uint32_t pair = 0;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      int h = (i + u) / 8, j = (i + u) % 8;
      int64_t k = chunk * 64 + tile_row(l, h, j);
      uint32_t v = (k < rows && n < cols) ? src[b * sb + k * sr + n * sc] : 0;
      pair |= v << (16 * u);
    }
    w[i / 2] = pair;
  }
  uint4 *out = (uint4 *)(dst + tile * 1024 + 16 * l);
  out[0] = make_uint4(w[0], w[1], w[2], w[3]);
  out[1] = make_uint4(w[4], w[5], w[6], w[7]);
}

// Readback a thread a value: finds it in its tile, decodes it exactly. For small results, where a block's chain of the
// kernel below is longer than the byte loads it saves.
template <int FMT>
__global__ void __launch_bounds__(256) columns_value_kernel(const uint8_t *src, int64_t total, int64_t rows, int64_t cols,
                                                            int64_t chunks, int64_t runs, uint16_t *dst) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  const int64_t n = t % cols, k = t / cols % rows, b = t / cols / rows;
  const int kk = (int)(k % 64), h = kk / 32, g = (kk % 32) / 8, j = kk % 8, l = g * 16 + (int)(n % 16);
  const int64_t tile = (b * runs + n / 16) * chunks + k / 64;
  if (FMT == BT_BF16) {
    dst[t] = ((const uint16_t *)src)[tile * 1024 + 16 * l + 8 * h + j];
    return;
  }
  const uint8_t *tp = src + tile * (FMT == BT_BFP8 ? 1088 : 576);
  const uint32_t e = (tp[16 * g + 8 * h + j] + exp_bias<FMT>()) & 255u;
  const int q = FMT == BT_BFP8 ? (int)(int8_t)tp[64 + 16 * l + 8 * h + j] : nibble_q(*(const uint32_t *)(tp + 64 + 8 * l + 4 * h), j) * 16;
  dst[t] = (uint16_t)unpacked_bits(q, e);
}

// Readback of 16 neighbouring runs of one chunk a block: each of its 4 waves loads 4 tiles as contiguous stretches, every
// lane decoding its 16 values exactly, and the block stores the 64 rows' 256 columns from LDS as whole 512-byte
// stretches (WIDE: every row of the result starts on 16 bytes; otherwise a thread a column). A thread a value took its
// exponent and value a byte at a time from tiles that lie `chunks` apart. The bound is HBM: 2 bytes written a value and
// 9/16 to 2 read. 4096 x 14336 in bfp4: 187 us a thread a value, 37 us
// so (4.1 TB/s).
template <int FMT, bool WIDE>
__global__ void __launch_bounds__(256) columns_unpack_kernel(const uint8_t *src, int64_t rows, int64_t cols,
                                                             uint32_t runs, uint32_t chunks, FastDiv groups,
                                                             FastDiv chunks_d, uint16_t *dst) {
  constexpr int TB = FMT == BT_BF16 ? 2048 : FMT == BT_BFP8 ? 1088 : 576, S = 16 * RUNS_B + 4;  // rows 130 dwords apart
  __shared__ __attribute__((aligned(16))) uint16_t lds[64 * S];
  const uint32_t q = fdiv(blockIdx.x, groups), b = fdiv(q, chunks_d), chunk = q - b * chunks, run0 = (blockIdx.x - q * groups.d) * RUNS_B;
  const int t = threadIdx.x, l = t & 63, g = l >> 4, n = l & 15;
#pragma unroll
  for (int i = 0; i < RUNS_B / 4; i++) {
    const uint32_t run = (t >> 6) + 4 * i;
    if (run0 + run >= runs) break;  // uniform in the wave
    const uint8_t *tp = src + ((int64_t)((int64_t)b * runs + run0 + run) * chunks + chunk) * TB;
    uint32_t v[16];  // value 8h + j: row 32h + 8g + j of the tile, column n
    if (FMT == BT_BF16) {
      const uint4 w0 = ((const uint4 *)(tp + 32 * l))[0], w1 = ((const uint4 *)(tp + 32 * l))[1];
      const uint32_t w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
      for (int k = 0; k < 16; k++) v[k] = w[k / 2] >> (16 * (k & 1));
    } else {
      const uint4 ew = *(const uint4 *)(tp + 16 * g);
      const uint32_t es[4] = {ew.x, ew.y, ew.z, ew.w};
      uint32_t w[4];
      if (FMT == BT_BFP8) {
        const uint4 x = *(const uint4 *)(tp + 64 + 16 * l);
        w[0] = x.x, w[1] = x.y, w[2] = x.z, w[3] = x.w;
      } else {
        const uint2 x = *(const uint2 *)(tp + 64 + 8 * l);
        w[0] = x.x, w[1] = x.y, w[2] = w[3] = 0;
      }
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const uint32_t e = ((es[k / 4] >> (8 * (k % 4))) + exp_bias<FMT>()) & 255u;
        const int mag = FMT == BT_BFP8 ? (int32_t)(w[k / 4] << (24 - 8 * (k % 4))) >> 24 : nibble_q(w[k / 8], k % 8) * 16;
        // for e in 7..254 the value is a normal float whose top half is the exact bf16; mag * 2^(e - 133) in both formats
        v[k] = e - 7u <= 247u ? __float_as_uint((float)mag * __uint_as_float((e - 6u) << 23)) >> 16 : unpacked_bits(mag, e);
      }
    }
#pragma unroll
    for (int k = 0; k < 16; k++) lds[(32 * (k / 8) + 8 * g + k % 8) * S + 16 * run + n] = (uint16_t)v[k];
  }
  __syncthreads();
  const int64_t k0 = (int64_t)chunk * 64, c0 = (int64_t)run0 * 16;
  uint16_t *out = dst + ((int64_t)b * rows + k0) * cols + c0;
  if (WIDE) {  // cols is a multiple of 8
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int row = t / 32 + 8 * i, c = t % 32 * 8;
      const uint2 x = *(const uint2 *)(lds + row * S + c), y = *(const uint2 *)(lds + row * S + c + 4);
      if (k0 + row < rows && c0 + c < cols) *(uint4 *)(out + row * cols + c) = make_uint4(x.x, x.y, y.x, y.y);
    }
  } else {
    if (c0 + t >= cols) return;
#pragma unroll 8
    for (int row = 0; row < 64; row++)
      if (k0 + row < rows) out[row * cols + t] = lds[row * S + t];
  }
}

static int check_fmt(int fmt) {
  if (fmt != BT_BFP8 && fmt != BT_BFP4) return fail(BT_EINVAL, "block-float format must be bfp8 or bfp4, not %d", fmt);
  return BT_OK;
}

static int check_shape(int64_t batch, int64_t rows, int64_t cols) {
  if (batch <= 0 || rows <= 0 || cols <= 0)
    return fail(BT_EINVAL, "shape %lld x %lld x %lld must be positive", (long long)batch, (long long)rows,
                (long long)cols);
  return BT_OK;
}

static unsigned blocks_for(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

// pack_half_kernel with the widest loads (16, 8, 4 or 2 bytes) that every row's start is aligned to.
template <int FMT>
static void launch_pack_half(uint64_t src, int src_dtype, int64_t batch, int64_t rows, int64_t cols, int64_t sb, int64_t sr,
                             uint64_t exps, uint64_t vals, hipStream_t s) {
  const int64_t size = src_dtype == BT_BF16 ? 2 : 4, runs = (cols + 15) / 16;
  const uint32_t halves = (uint32_t)(2 * batch * rows * runs);
  uint64_t at = src | 16u;  // the starts' common alignment; strides that no second row or matrix uses don't count
  if (rows > 1) at |= (uint64_t)(sr * size);
  if (batch > 1) at |= (uint64_t)(sb * size);
  const uint64_t align = at & (~at + 1);
  const FastDiv rd = make_fastdiv((uint32_t)runs), wd = make_fastdiv((uint32_t)rows);
#define BT_PACK(SRC, A)                                                                                              \
  pack_half_kernel<FMT, SRC, A><<<blocks_for(halves, 256), 256, 0, s>>>((const void *)src, halves, rd, wd, cols, sb, \
                                                                        sr, (uint8_t *)exps, (uint8_t *)vals)
  if (src_dtype == BT_FP32) {
    if (align >= 16) BT_PACK(BT_FP32, 16);
    else BT_PACK(BT_FP32, 4);
  } else if (align >= 16) BT_PACK(BT_BF16, 16);
  else if (align >= 4) BT_PACK(BT_BF16, 4);
  else BT_PACK(BT_BF16, 2);
#undef BT_PACK
}

}  // namespace bt

using namespace bt;

extern "C" {

int bt_bfp_pack(bt_runtime *rt, int fmt, uint64_t src, int src_dtype, int64_t batch, int64_t rows, int64_t cols,
                int64_t sb, int64_t sr, int64_t sc, uint64_t exps, uint64_t vals) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (int s = check_fmt(fmt)) return s;
  if (int s = check_shape(batch, rows, cols)) return s;
  if (src_dtype != BT_BF16 && src_dtype != BT_FP32) return fail(BT_EINVAL, "a block float is cast from bf16 or fp32");
  if (vals % 16) return fail(BT_EINVAL, "the value plane must be 16-byte aligned");
  const int64_t runs = (cols + 15) / 16, n = batch * rows * runs;
  if (sc == 1 && 2 * n < (1ll << 31)) {
    if (fmt == BT_BFP8) launch_pack_half<BT_BFP8>(src, src_dtype, batch, rows, cols, sb, sr, exps, vals, r->stream);
    else launch_pack_half<BT_BFP4>(src, src_dtype, batch, rows, cols, sb, sr, exps, vals, r->stream);
  } else if (fmt == BT_BFP8)
    pack_kernel<BT_BFP8><<<blocks_for(n, 256), 256, 0, r->stream>>>((const void *)src, src_dtype, batch, rows, cols,
                                                                     sb, sr, sc, (uint8_t *)exps, (uint8_t *)vals);
  else
    pack_kernel<BT_BFP4><<<blocks_for(n, 256), 256, 0, r->stream>>>((const void *)src, src_dtype, batch, rows, cols,
                                                                     sb, sr, sc, (uint8_t *)exps, (uint8_t *)vals);
  BT_LAUNCHED("bfp_pack");
  return BT_OK;
}

int bt_bfp_unpack(bt_runtime *rt, int fmt, uint64_t exps, uint64_t vals, int64_t batch, int64_t rows, int64_t cols,
                  uint64_t dst) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (int s = check_fmt(fmt)) return s;
  if (int s = check_shape(batch, rows, cols)) return s;
  int64_t n = batch * rows * cols;
  if (fmt == BT_BFP8)
    unpack_kernel<BT_BFP8><<<blocks_for(n, 256), 256, 0, r->stream>>>((const uint8_t *)exps, (const uint8_t *)vals,
                                                                       batch, rows, cols, (uint16_t *)dst);
  else
    unpack_kernel<BT_BFP4><<<blocks_for(n, 256), 256, 0, r->stream>>>((const uint8_t *)exps, (const uint8_t *)vals,
                                                                       batch, rows, cols, (uint16_t *)dst);
  BT_LAUNCHED("bfp_unpack");
  return BT_OK;
}

int bt_bfp_columns(bt_runtime *rt, int fmt, uint64_t exps, uint64_t vals, int64_t batch, int64_t rows, int64_t cols,
                   uint64_t dst) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (int s = check_fmt(fmt)) return s;
  if (int s = check_shape(batch, rows, cols)) return s;
  if (dst % 16) return fail(BT_EINVAL, "columns tiles must be 16-byte aligned");
  int64_t chunks = (rows + 63) / 64, nruns = (cols + 15) / 16, tiles = batch * nruns * chunks;
  if (tiles >= (1ll << 31)) return fail(BT_EINVAL, "too many tiles");
  const bool few = batch * chunks * ((nruns + RUNS_B - 1) / RUNS_B) < 256;
  const int per = few ? 4 : RUNS_B;
  const int64_t groups = (nruns + per - 1) / per;
  const FastDiv gd = make_fastdiv((uint32_t)groups), cd = make_fastdiv((uint32_t)chunks);
  const unsigned blocks = (unsigned)(batch * chunks * groups);
#define BT_COLUMNS_N(FMT, WIDE, RUNS)                                                                                \
  columns_kernel<FMT, WIDE, RUNS><<<blocks, 256, 0, r->stream>>>((const uint8_t *)exps, (const uint8_t *)vals, rows,   \
                                                                 (uint32_t)nruns, (uint32_t)chunks, gd, cd, (uint8_t *)dst)
#define BT_COLUMNS(FMT, WIDE)                                                                                        \
  do {                                                                                                               \
    if (few) BT_COLUMNS_N(FMT, WIDE, 4);                                                                             \
    else BT_COLUMNS_N(FMT, WIDE, RUNS_B);                                                                            \
  } while (0)
  if (fmt == BT_BFP8 && vals % 8 == 0) BT_COLUMNS(BT_BFP8, true);
  else if (fmt == BT_BFP8) BT_COLUMNS(BT_BFP8, false);
  else if (vals % 8 == 0) BT_COLUMNS(BT_BFP4, true);
  else BT_COLUMNS(BT_BFP4, false);
#undef BT_COLUMNS
#undef BT_COLUMNS_N
  BT_LAUNCHED("bfp_columns");
  return BT_OK;
}

int bt_bfp_range(bt_runtime *rt, int fmt, uint64_t exps, uint64_t vals, int64_t batch, int64_t rows, int64_t cols,
                 uint64_t bad) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (int s = check_fmt(fmt)) return s;
  if (int s = check_shape(batch, rows, cols)) return s;
  if (vals % 16 || bad % 4) return fail(BT_EINVAL, "the value plane must be 16-byte aligned and the count 4-byte aligned");
  const int64_t runs = batch * rows * ((cols + 15) / 16);
  zero_word_kernel<<<1, 64, 0, r->stream>>>((uint32_t *)(uintptr_t)bad);
  BT_LAUNCHED("bfp_range");
  if (fmt == BT_BFP8)
    range_kernel<BT_BFP8><<<blocks_for(runs, 256), 256, 0, r->stream>>>((const uint8_t *)exps, (const uint8_t *)vals,
                                                                         runs, (uint32_t *)(uintptr_t)bad);
  else
    range_kernel<BT_BFP4><<<blocks_for(runs, 256), 256, 0, r->stream>>>((const uint8_t *)exps, (const uint8_t *)vals,
                                                                         runs, (uint32_t *)(uintptr_t)bad);
  BT_LAUNCHED("bfp_range");
  return BT_OK;
}

int bt_bf16_columns(bt_runtime *rt, uint64_t src, int64_t batch, int64_t rows, int64_t cols, int64_t sb, int64_t sr,
                    int64_t sc, uint64_t dst) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (int s = check_shape(batch, rows, cols)) return s;
  if (dst % 16) return fail(BT_EINVAL, "columns tiles must be 16-byte aligned");
  int64_t chunks = (rows + 63) / 64, nruns = (cols + 15) / 16, tiles = batch * nruns * chunks;
  if (tiles >= (1ll << 31)) return fail(BT_EINVAL, "too many tiles");
  bf16_columns_kernel<<<(unsigned)tiles, 64, 0, r->stream>>>((const uint16_t *)src, rows, cols, sb, sr, sc, chunks,
                                                              nruns, (uint16_t *)dst);
  BT_LAUNCHED("bf16_columns");
  return BT_OK;
}

int bt_columns_unpack(bt_runtime *rt, int fmt, uint64_t src, int64_t batch, int64_t rows, int64_t cols,
                      uint64_t dst) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (fmt != BT_BF16 && fmt != BT_BFP8 && fmt != BT_BFP4) return fail(BT_EINVAL, "columns format %d", fmt);
  if (int s = check_shape(batch, rows, cols)) return s;
  const int64_t chunks = (rows + 63) / 64, nruns = (cols + 15) / 16, groups = (nruns + RUNS_B - 1) / RUNS_B;
  if (batch * nruns * chunks >= (1ll << 31)) return fail(BT_EINVAL, "too many tiles");
  const FastDiv gd = make_fastdiv((uint32_t)groups), cd = make_fastdiv((uint32_t)chunks);
  const bool wide = cols % 8 == 0 && dst % 16 == 0;
  // a thread a value up to where both take the same: 1.5 million values of block floats and of rows stored a column a
  // thread, half a million of bf16 in whole words (bfp4, a thread a value and in blocks: 60 x 204 2.4 and 9.7 us, 1024 x
  // 1024 5.1 and 7.6, 1024 x 2048 8.7 and 7.8, 4096 x 4096 52 and 13; bf16, 300 x 2000 3.4 and 3.3, 1024 x 1024 4.6 and
  // 3.2); also tiles that don't start on the blocks' 16-byte loads
  const int64_t total = batch * rows * cols;
  if (total < (fmt == BT_BF16 && wide ? 1 << 19 : 3 << 19) || src % 16) {
    const unsigned blocks = blocks_for(total, 256);
    if (fmt == BT_BF16) columns_value_kernel<BT_BF16><<<blocks, 256, 0, r->stream>>>((const uint8_t *)src, total, rows, cols, chunks, nruns, (uint16_t *)dst);
    else if (fmt == BT_BFP8) columns_value_kernel<BT_BFP8><<<blocks, 256, 0, r->stream>>>((const uint8_t *)src, total, rows, cols, chunks, nruns, (uint16_t *)dst);
    else columns_value_kernel<BT_BFP4><<<blocks, 256, 0, r->stream>>>((const uint8_t *)src, total, rows, cols, chunks, nruns, (uint16_t *)dst);
    BT_LAUNCHED("columns_unpack");
    return BT_OK;
  }
#define BT_UNPACK(FMT, WIDE)                                                                                         \
  columns_unpack_kernel<FMT, WIDE><<<(unsigned)(batch * chunks * groups), 256, 0, r->stream>>>(                      \
    (const uint8_t *)src, rows, cols, (uint32_t)nruns, (uint32_t)chunks, gd, cd, (uint16_t *)dst)
  if (fmt == BT_BF16 && wide) BT_UNPACK(BT_BF16, true);
  else if (fmt == BT_BF16) BT_UNPACK(BT_BF16, false);
  else if (fmt == BT_BFP8 && wide) BT_UNPACK(BT_BFP8, true);
  else if (fmt == BT_BFP8) BT_UNPACK(BT_BFP8, false);
  else if (wide) BT_UNPACK(BT_BFP4, true);
  else BT_UNPACK(BT_BFP4, false);
#undef BT_UNPACK
  BT_LAUNCHED("columns_unpack");
  return BT_OK;
}

int bt_put_bfp(bt_runtime *rt, int fmt, uint64_t exps, uint64_t vals, int64_t batch, int64_t dst_rows, int64_t cols,
               int64_t dst_sb, int64_t dst_sr, uint64_t ids, int64_t n, uint64_t x, int64_t x_sb, int64_t x_sr) {
  Runtime *r;
  if (int s = enter(rt, &r)) return s;
  if (fmt != BT_BFP8 && fmt != BT_BFP4) return fail(BT_EINVAL, "put_bfp writes bfp8 or bfp4, not %d", fmt);
  if (!exps || !vals || !ids || !x) return fail(BT_EINVAL, "put_bfp needs its planes, ids and x");
  if (batch < 1 || dst_rows < 1 || cols < 16 || cols % 16 || n < 0 || dst_sb % 16 || dst_sr % 16)
    return fail(BT_EINVAL, "put_bfp shape: batch %lld, %lld rows of %lld (a multiple of 16), strides %lld %lld",
                (long long)batch, (long long)dst_rows, (long long)cols, (long long)dst_sb, (long long)dst_sr);
  if (ids % 4 || x % 2) return fail(BT_EINVAL, "put_bfp needs aligned ids and x");
  if (n == 0) return BT_OK;
  if (n >= (1ll << 31)) return fail(BT_EINVAL, "put_bfp: too many rows");
  if (fmt == BT_BFP8)
    put_bfp_kernel<BT_BFP8><<<(unsigned)n, 256, 0, r->stream>>>((uint8_t *)exps, (uint8_t *)vals, dst_rows, cols, dst_sb,
                                                               dst_sr, (const int32_t *)ids, n, (const uint16_t *)x, x_sb,
                                                               x_sr, batch);
  else
    put_bfp_kernel<BT_BFP4><<<(unsigned)n, 256, 0, r->stream>>>((uint8_t *)exps, (uint8_t *)vals, dst_rows, cols, dst_sb,
                                                               dst_sr, (const int32_t *)ids, n, (const uint16_t *)x, x_sb,
                                                               x_sr, batch);
  BT_LAUNCHED("put_bfp");
  return BT_OK;
}

}  // extern "C"
