// Blockwise quantiser: the producer of the MatMulNBits weight format, on the device.
//
// Restates BlockwiseQuantizer::quantizeAndTranspose for column-wise blocks
// (onnxruntime/core/mlas/lib/q4_dq.cpp:468-574) with range2scalezp / range2scale (:347-386):
//   asymmetric  min = min(min, 0), max = max(max, 0); scale = (max - min) / (2^bits - 1);
//               zp = clamp(roundf(-min / scale)) (min itself when the scale is 0);
//   symmetric   s = the extreme with the larger magnitude; scale = -s / 2^(bits-1); zp = 2^(bits-1);
//   q = clamp(roundf(v * (1 / stored scale) + zp), 0, 2^bits - 1), all in fp32, no fused multiply-add.
// fp16 models widen every element to fp32 and store the scale rounded to fp16; the reciprocal is taken from the
// stored scale, the zero point from the unrounded one.  Output is the canonical operand layout of the operator.
// Positions k >= K of the last block (left unwritten by the reference) receive the zero point: they dequantise to 0.
//
// A workgroup owns 128 neighbouring columns and the 8/bits consecutive blocks that share one zero-point byte.  Each
// block is first copied to LDS with 16-byte loads (rows of the source are contiguous across the 128 columns: 256-byte
// pieces of fp16 rows; 128-byte pieces - 64 columns - were measured 8 % slower, 512-byte pieces 20 % slower), so the
// source is read from HBM exactly once.  Four threads per column take one quarter of the block each: a thread reads
// its quarter from LDS, keeps it widened to fp32 in registers across the range scan, and quantises from there
// (the block size is a template parameter for that reason; quarters of 16 and more elements are read a second time
// instead).  Whole blocks - all but a ragged last one - run without per-element conditions.  (Reading a thread's
// elements straight from global memory into registers - no LDS tile, one barrier per block - was measured at less
// than half the speed: 2-byte loads per lane put too few bytes in flight.)  Blocks of 64 and fewer elements run on a
// second kernel that lays several blocks of a column side by side in one workgroup (mnb_quantize_small_kernel), fp16
// blocks of 256 on a third (mnb_quantize_pairs_kernel).
//
// The 16-byte loads ask for no more alignment than the element has: rows of odd widths go the same way as aligned ones, a
// tenth slower (the hardware takes a cache line more per piece).  Only the last strip, of fewer than 128 columns, is filled
// element by element, 16 loads in flight a thread; a compile-time form without that path serves the widths that have no
// such strip, for its registers cost a wavefront a SIMD.  [K, N] from HBM, before (odd fp32 rows one element in flight, odd
// fp16 rows as pairs of 2-byte loads) -> now, us: fp32 [5824, 10235] 4-bit blocks of 64 142 -> 60, [12128, 3534] blocks of 128
// with zero points 116 -> 47, [8192, 7001] 139 -> 59; fp16 [4832, 12825] blocks of 32 with zero points 135 -> 48, 8-bit
// blocks of 64 96 -> 54, [14336, 4095] blocks of 128 57 -> 39, [8192, 33] blocks of 64 with zero points 9.2 -> 4.9.
#include <hip/hip_runtime.h>

#include "mnb_buffer.hip.h"
#include "mnb_internal.h"
#include "mnb_quant_grid.h"

namespace {

constexpr int kCols = 128;     // columns per workgroup
constexpr int kQuarters = 4;   // threads per column (each takes one quarter of the block)

// A 16-byte piece of a row, whose address is a multiple of the element's size only (the hardware splits what it has to).
template <typename T>
struct PieceOf;
template <>
struct PieceOf<_Float16> {
  typedef uint32_t type __attribute__((ext_vector_type(4), aligned(2)));
};
template <>
struct PieceOf<float> {
  typedef uint32_t type __attribute__((ext_vector_type(4), aligned(4)));
};

// The strip of columns and the group of blocks of a workgroup (see mnb_quant_grid.h).
__device__ __forceinline__ MnbQuantTile quant_tile(int strips, int groups, int run) {
  if (run == 0) return {blockIdx.x, blockIdx.y};
  return mnb_quant_run_tile(blockIdx.x, gridDim.x, strips, groups, run);
}

// The rows of a tile that 16-byte loads cannot read: EACH elements a thread, 16 loads in flight.  Rows and columns beyond the
// matrix re-read its last ones (and are never used).
template <typename T, int EACH, int THREADS>
__device__ __forceinline__ void fill_by_elements(T* tile, const T* src, int64_t ld, int rows, int64_t cols, int tid) {
  const int cc = tid % kCols;
  const T* const column = src + (cc < cols ? cc : cols - 1);
  constexpr int STEP = THREADS / kCols, AT_ONCE = EACH < 16 ? EACH : 16;
#pragma unroll
  for (int u0 = 0; u0 < EACH; u0 += AT_ONCE) {
    if (u0 * STEP >= rows) break;
    T v[AT_ONCE];
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) {
      const int r = tid / kCols + (u0 + u) * STEP;
      v[u] = column[(int64_t)(r < rows ? r : rows - 1) * ld];
    }
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) tile[(tid / kCols + (u0 + u) * STEP) * kCols + cc] = v[u];
  }
}

// A tile of ROWS rows of which only `rows` exist: behind the others' fill the missing ones become NaN, which the scan skips
// (as the reference's comparisons do), so that it needs no condition.  (With a condition on every element, one LDS read after
// the other, a ragged last block was most of a small matrix's time: fp16 [200, 13] 4-bit blocks of 32 6.9 us, now 5.0;
// [600, 1001] 2-bit blocks of 64 11.6 and 5.2; fp32 [300, 1001] blocks of 256 11.0 and 7.8.)
template <typename T, int ROWS, int THREADS>
__device__ __forceinline__ void clear_missing_rows(T* tile, int rows, int tid) {
  const uint32_t nan = sizeof(T) == 2 ? 0x7e007e00u : 0x7fc00000u;
  constexpr int CH = kCols * (int)sizeof(T) / 16;  // 16-byte pieces of a row
  __syncthreads();
  for (int i = rows * CH + tid; i < ROWS * CH; i += THREADS)
    reinterpret_cast<uint4*>(tile)[i] = make_uint4(nan, nan, nan, nan);
}

// The first zero of a column of zeros (and NaN).
template <typename T>
__device__ __forceinline__ float first_zero(const T* column, int rows) {
  float f = (float)column[0];
  for (int e = 1; !(f == 0.f) && e < rows; ++e) f = (float)column[e * kCols];
  return f;
}

// ... and their part of the weights is the zero point: `mine` elements of the words are the matrix's.
template <int BITS, int WORDS>
__device__ __forceinline__ void zero_point_behind(uint32_t (&word)[WORDS], int mine, int z) {
  const uint32_t fill = (uint32_t)z * (0xffffffffu / ((1u << BITS) - 1));
#pragma unroll
  for (int w = 0; w < WORDS; ++w) {
    const int bits = (mine - w * (32 / BITS)) * BITS;  // of this word
    const uint32_t keep = bits <= 0 ? 0u : bits >= 32 ? 0xffffffffu : (1u << bits) - 1;
    word[w] = (word[w] & keep) | (fill & ~keep);
  }
}

// ALL: no strip of fewer than 128 columns.  (The wavefronts a SIMD asked for are those that the LDS tile leaves room for, for
// fp16 blocks of 128 six of the eight: with fewer registers the loads of the scan come in smaller batches, [4096, 14336] 4-bit
// with zero points 38.9 us and 37.3.)
// QROWS = block size / 4: the elements of a thread's quarter.  A compile-time constant so that the quarter, widened
// to fp32, stays in registers between the range scan and the quantisation (each element leaves LDS once).
template <typename T, int BITS, int QROWS, bool ALL>
__global__ void __launch_bounds__(kCols * kQuarters) __attribute__((amdgpu_waves_per_eu(
    sizeof(T) == 2 ? 6 : QROWS <= 32 ? 4 : 2, sizeof(T) == 2 ? (QROWS <= 16 ? 8 : 6) : QROWS <= 32 ? 4 : 2)))
                                                     mnb_quantize_kernel(uint8_t* __restrict__ B, T* __restrict__ scales,
                                                                         uint8_t* __restrict__ zp,
                                                                         const T* __restrict__ src, int64_t K, int64_t N,
                                                                         int64_t ld, int nsub, int strips,
                                                                         int groups, int run) {
  constexpr int PER_BYTE = 8 / BITS;  // blocks per zero-point byte, elements per weight byte
  constexpr int MAXQ = (1 << BITS) - 1;
  constexpr int MID = 1 << (BITS - 1);
  constexpr int VEC = 16 / (int)sizeof(T);  // elements per 16-byte load
  constexpr int bs = QROWS * kQuarters;
  constexpr int blob = bs * BITS / 8;
  constexpr int QBITS = QROWS * BITS;       // bits a thread produces per block: 8 (2-bit, block 16), 16, or words
  constexpr int QWORDS = (QBITS + 31) / 32;
  extern __shared__ __align__(16) unsigned char smem[];
  T* tile = reinterpret_cast<T*>(smem);                                    // [bs][kCols]
  float* red = reinterpret_cast<float*>(smem + (size_t)bs * kCols * sizeof(T));  // [2][kQuarters][kCols]

  const int tid = threadIdx.x;
  const int c = tid % kCols, qr = tid / kCols;
  const MnbQuantTile qt = quant_tile(strips, groups, run);
  const int64_t n0 = qt.strip * kCols;
  const int64_t n = n0 + c;
  const int64_t kbc = (K + bs - 1) / bs;
  const int64_t zrow = (kbc * BITS + 7) / 8;
  const int64_t kb0 = qt.group * nsub;
  const int nb = (int)(kbc - kb0 < nsub ? kbc - kb0 : nsub);  // blocks of this workgroup, consecutive along K
  const bool fast = ALL || n0 + kCols <= N;
  const int q0 = qr * QROWS;
  uint32_t zbyte = 0;

  // The next block travels from global memory into registers while the current one is worked on from LDS.
  constexpr int CH = kCols / VEC;                                // 16-byte chunks per row
  constexpr int PRE = (bs * CH + kCols * kQuarters - 1) / (kCols * kQuarters);  // chunks per thread and block
  // chunk u of a thread: row (tid + 256 u) / CH of the block (rows beyond the block's last re-read that row and are
  // never used, so that no load sits under a condition), 16-byte piece (tid + 256 u) % CH of the strip
  using piece_t = typename PieceOf<T>::type;
  auto chunk_ptr = [&](int64_t kb, int u) -> const piece_t* {
    const int64_t k0 = kb * bs;
    const int rows = (int)(k0 + bs < K ? bs : K - k0);
    const int i = tid + u * kCols * kQuarters;
    const int r = i / CH < rows ? i / CH : rows - 1;
    return reinterpret_cast<const piece_t*>(src + (k0 + r) * ld + n0 + (i % CH) * VEC);
  };
  u4_t pre[PRE];
#pragma unroll
  for (int u = 0; u < PRE; ++u) pre[u] = fast ? (u4_t)*chunk_ptr(kb0, u) : u4_t{0, 0, 0, 0};

  for (int sb = 0; sb < nb; ++sb) {
    const int sub = sb % PER_BYTE;
    const int64_t kb = kb0 + sb;
    const int64_t k0 = kb * bs;
    const int rows = (int)(k0 + bs < K ? bs : K - k0);
    __syncthreads();  // the previous block's tile is no longer read
    if (fast) {
#pragma unroll
      for (int u = 0; u < PRE; ++u) {
        const int i = tid + u * kCols * kQuarters;
        if (bs * CH % (kCols * kQuarters) == 0 || i < bs * CH)
          *reinterpret_cast<u4_t*>(tile + (i / CH) * kCols + (i % CH) * VEC) = pre[u];
      }
      if (sb + 1 < nb) {
#pragma unroll
        for (int u = 0; u < PRE; ++u) pre[u] = *chunk_ptr(kb + 1, u);
      }
    } else {
      fill_by_elements<T, bs / kQuarters, kCols * kQuarters>(tile, src + k0 * ld + n0, ld, rows, N - n0, tid);
    }
    if (rows < bs) clear_missing_rows<T, bs, kCols * kQuarters>(tile, rows, tid);  // (a ragged last block)
    __syncthreads();
    // range of this thread's quarter, then of the whole block
    // blocks of 64 and more elements read the tile a second time when they quantise instead of holding their
    // quarter in registers (which, with the registers of the load in flight, keeps wavefronts off the SIMD)
    constexpr bool kHold = QROWS < 16;
    float held[kHold ? QROWS : 1];
    float mn = 3.402823466e+38f, mx = -3.402823466e+38f;
#pragma unroll
    for (int e = 0; e < QROWS; ++e) {
      const float v = (float)tile[(q0 + e) * kCols + c];
      mn = __builtin_fminf(v, mn);  // one instruction each; like the reference's comparisons they skip a NaN
      mx = __builtin_fmaxf(v, mx);
      if constexpr (kHold) held[e] = v;
    }
    // The reference's scan (if (v < min) min = v) keeps the first zero it meets, whatever its sign, where the
    // minimum instruction prefers -0.  Only an all-zero block shows it (the sign of its stored scale): the first zero is
    // looked up there.
    if (mn == 0.f && mx == 0.f) mn = mx = first_zero(tile + q0 * kCols + c, QROWS);
    red[qr * kCols + c] = mn;
    red[(kQuarters + qr) * kCols + c] = mx;
    __syncthreads();
#pragma unroll
    for (int q2 = 0; q2 < kQuarters; ++q2) {
      const float a = red[q2 * kCols + c], b = red[(kQuarters + q2) * kCols + c];
      mn = a < mn ? a : mn;
      mx = b > mx ? b : mx;
    }
    float scale;
    int z;
    if (zp) {
      mn = mn < 0.f ? mn : 0.f;
      mx = mx > 0.f ? mx : 0.f;
      scale = (mx - mn) / (float)MAXQ;
      float zf = mn;
      if (scale != 0.f) zf = 0.f - mn / scale;
      zf = zf < 0.f ? 0.f : zf;
      zf = zf > (float)MAXQ ? (float)MAXQ : zf;
      z = (int)roundf(zf);
    } else {
      const float smax = fabsf(mx) > fabsf(mn) ? mx : mn;
      scale = -smax / (float)MID;
      z = MID;
    }
    zbyte |= (uint32_t)z << (sub * BITS);
    if (zp && (sub == PER_BYTE - 1 || kb == kbc - 1)) {
      // the unused part of the last zero-point byte keeps the reference's filler, the default zero point
      for (int f = sub + 1; f < PER_BYTE; ++f) zbyte |= (uint32_t)MID << (f * BITS);
      if (n < N && qr == 0) zp[n * zrow + kb / PER_BYTE] = (uint8_t)zbyte;
      zbyte = 0;
    }
    const T stored = (T)scale;
    const float sf = (float)stored;
    const float rscale = sf != 0.f ? 1.0f / sf : 0.f;
    const float zf32 = (float)z;
    if (n < N) {
      if (qr == 0) scales[n * kbc + kb] = stored;
      uint32_t word[QWORDS];
#pragma unroll
      for (int w = 0; w < QWORDS; ++w) word[w] = 0;
      // clamp(roundf(t), 0, MAXQ), roundf rounding halves away from zero: for t >= 0 that is trunc(t + 0.49999997f)
      // (the largest float below one half: a sum that lands exactly between two floats rounds to the even one,
      // which is the integer, only when t itself is a tie), everything below 0.5 ends at 0 either way, and the clamp
      // commutes with the truncation because its bounds are integers.
      auto quantise = [&](float v) -> uint32_t {
        float t = v * rscale;  // separate statements: the product is rounded before the addition
        t = t + zf32;
        t = t + 0.49999997f;
        t = __builtin_amdgcn_fmed3f(t, 0.f, (float)MAXQ);
        return (uint32_t)t;
      };
#pragma unroll
      for (int e = 0; e < QROWS; ++e) {
        const float v = kHold ? held[e] : (float)tile[(q0 + e) * kCols + c];
        word[(e * BITS) / 32] |= quantise(v) << ((e * BITS) % 32);
      }
      if (rows < bs) zero_point_behind<BITS>(word, rows - q0, z);
      uint8_t* out = B + (n * kbc + kb) * blob + qr * (QBITS / 8);
      if constexpr (QBITS == 8) {
        *out = (uint8_t)word[0];
      } else if constexpr (QBITS == 16) {
        *reinterpret_cast<uint16_t*>(out) = (uint16_t)word[0];
      } else if constexpr (QWORDS % 4 == 0) {
        // 16-byte stores (the quarter starts at a multiple of 16 bytes of a 16-byte aligned blob)
#pragma unroll
        for (int w = 0; w < QWORDS; w += 4)
          *reinterpret_cast<uint4*>(out + 4 * w) = make_uint4(word[w], word[w + 1], word[w + 2], word[w + 3]);
      } else {
#pragma unroll
        for (int w = 0; w < QWORDS; ++w) *reinterpret_cast<uint32_t*>(out + 4 * w) = word[w];
      }
    }
  }
}

// fp16 blocks of 256.  A wavefront owns 32 rows of 128 columns, two columns a lane, and loads them straight into registers: 32
// loads of 256 bytes a wavefront are in flight, six wavefronts a SIMD, no tile and no copy through LDS.  A pair of elements
// is compared by one packed fp16 minimum and maximum (exact) before it is widened to be quantised.  PARTS = block size / 32
// wavefronts share a block and exchange their ranges.  Arithmetic and outputs are those of the kernel above, whose tile for
// this block size, 64 KiB of LDS, leaves two workgroups a compute unit: [8192, 8192] 4-bit 50.9 us there, 40.9 here.
// Bound by the memory path (4.2 TB/s; stores of 16 bytes a column).  Rows at odd addresses are read by dwords all the same:
// [8192, 8191] 4-bit 65.5 -> 45.3 us, 8-bit 73.9 -> 56.1; where they begin at multiples of four the row goes into a scalar offset
// ([8000, 4100] 2-bit with zero points 39.4, by addresses of their own 42.5).  Shorter blocks are faster through the tile, on odd rows as well
// ([14336, 4095] blocks of 128 39.0 us there, 40.9 here; [4832, 12825] blocks of 32 with zero points 47.9 and 61.8).
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

// What a launch can count on: kAnyPairs nothing, kDwords rows at multiples of four bytes, kAllDwords besides that every
// workgroup has its 128 columns and every block its rows (the registers of the other cases' loads cost wavefronts).
enum PairsForm { kAnyPairs, kDwords, kAllDwords };

template <int BITS, int PARTS, PairsForm FORM>
__global__ void __launch_bounds__(64 * PARTS) mnb_quantize_pairs_kernel(uint8_t* __restrict__ B,
                                                                        _Float16* __restrict__ scales,
                                                                        uint8_t* __restrict__ zp,
                                                                        const _Float16* __restrict__ src, int64_t K,
                                                                        int64_t N, int64_t ld, int nsub,
                                                                        int strips, int groups, int run) {
  constexpr bool ALL = FORM == kAllDwords;
  constexpr int PER_BYTE = 8 / BITS, MAXQ = (1 << BITS) - 1, MID = 1 << (BITS - 1);
  constexpr int ROWS = 32, BS = ROWS * PARTS, BLOB = BS * BITS / 8, WORDS = ROWS * BITS / 32;
  __shared__ float2 red_min[PARTS][64], red_max[PARTS][64];
  const int lane = threadIdx.x & 63, part = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const MnbQuantTile qt = quant_tile(strips, groups, run);
  const int64_t n0 = qt.strip * kCols, n = n0 + 2 * lane;
  const int64_t kbc = (K + BS - 1) / BS, zrow = (kbc * BITS + 7) / 8, kb0 = qt.group * nsub;
  const int nb = (int)(kbc - kb0 < nsub ? kbc - kb0 : nsub);
  const bool fast = n0 + kCols <= N;
  float minus_zero = -0.f;
  asm volatile("" : "+v"(minus_zero));  // opaque: see `quantise`
  uint32_t zbyte[2] = {0, 0};

  for (int sb = 0; sb < nb; ++sb) {
    const int sub = sb % PER_BYTE;
    const int64_t kb = kb0 + sb, k0 = kb * BS + part * ROWS;
    const int mine = (int)(K - k0 < ROWS ? K - k0 : ROWS);  // rows of this part that exist (may be <= 0)
    const _Float16* const rows = src + k0 * ld + n0;  // (uniform over the wavefront)
    half2_t v[ROWS];
    if (ALL || (fast && mine >= ROWS)) {
      if constexpr (FORM != kAnyPairs) {
        const rsrc_t block_rows = mnb_rsrc(rows);
        const uint32_t pitch = (uint32_t)ld * 2;
#pragma unroll
        for (int e = 0; e < ROWS; ++e)  // (the row in a scalar offset: no address registers for each load)
          v[e] = __builtin_bit_cast(half2_t, mnb_buffer_load_b32(block_rows, 4 * lane, e * pitch));
      } else {
        typedef uint32_t pair_t __attribute__((aligned(2)));
#pragma unroll
        for (int e = 0; e < ROWS; ++e)
          v[e] = __builtin_bit_cast(half2_t, (uint32_t)*reinterpret_cast<const pair_t*>(rows + e * ld + 2 * lane));
      }
    } else {
      // what does not exist is a NaN for the scan, which skips it (as the reference's comparisons do), and zero afterwards
#pragma unroll
      for (int e = 0; e < ROWS; ++e)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          v[e][h] = e < mine && n + h < N ? rows[e * ld + 2 * lane + h] : (_Float16)__builtin_nanf("");
    }
    half2_t lo = {(_Float16)__builtin_inff(), (_Float16)__builtin_inff()}, hi = -lo;
#pragma unroll
    for (int e = 0; e < ROWS; ++e) {
      v[e] = __builtin_elementwise_canonicalize(v[e]);  // (in place: the comparisons would keep a second, quieted copy)
      lo = __builtin_elementwise_min(lo, v[e]);
      hi = __builtin_elementwise_max(hi, v[e]);
    }
    if (!ALL && mine < ROWS) {
#pragma unroll
      for (int e = 0; e < ROWS; ++e)
        if (e >= mine) v[e] = half2_t{};  // quantised to the zero point
    }
    float mn[2], mx[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      mn[h] = __builtin_fminf(3.402823466e+38f, (float)lo[h]);
      mx[h] = __builtin_fmaxf(-3.402823466e+38f, (float)hi[h]);
      // all zeros: the scan keeps the first it meets, whatever its sign (it is the sign of the stored scale)
      if (mn[h] == 0.f && mx[h] == 0.f) {
        int e = 0;
        float f = (float)rows[2 * lane + h];
        while (!(f == 0.f) && ++e < mine && e < ROWS) f = (float)rows[e * ld + 2 * lane + h];
        mn[h] = mx[h] = f;
      }
    }
    if (sb > 0) __syncthreads();  // the previous block's ranges are no longer read
    red_min[part][lane] = make_float2(mn[0], mn[1]);
    red_max[part][lane] = make_float2(mx[0], mx[1]);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PARTS; ++q) {
      const float2 a = red_min[q][lane], b = red_max[q][lane];
      mn[0] = a.x < mn[0] ? a.x : mn[0];
      mn[1] = a.y < mn[1] ? a.y : mn[1];
      mx[0] = b.x > mx[0] ? b.x : mx[0];
      mx[1] = b.y > mx[1] ? b.y : mx[1];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float scale;
      int z;
      if (zp) {
        const float low = mn[h] < 0.f ? mn[h] : 0.f, high = mx[h] > 0.f ? mx[h] : 0.f;
        scale = (high - low) / (float)MAXQ;
        float zf = low;
        if (scale != 0.f) zf = 0.f - low / scale;
        zf = zf < 0.f ? 0.f : zf;
        zf = zf > (float)MAXQ ? (float)MAXQ : zf;
        z = (int)roundf(zf);
      } else {
        const float smax = fabsf(mx[h]) > fabsf(mn[h]) ? mx[h] : mn[h];
        scale = -smax / (float)MID;
        z = MID;
      }
      zbyte[h] |= (uint32_t)z << (sub * BITS);
      if (zp && (sub == PER_BYTE - 1 || kb == kbc - 1)) {
        for (int f = sub + 1; f < PER_BYTE; ++f) zbyte[h] |= (uint32_t)MID << (f * BITS);
        if (n + h < N && part == 0) zp[(n + h) * zrow + kb / PER_BYTE] = (uint8_t)zbyte[h];
        zbyte[h] = 0;
      }
      const _Float16 stored = (_Float16)scale;
      const float sf = (float)stored;
      const float rscale = sf != 0.f ? 1.0f / sf : 0.f;
      const float zf32 = (float)z;
      if (ALL || n + h < N) {
        if (part == 0) scales[(n + h) * kbc + kb] = stored;
        uint32_t word[WORDS];
#pragma unroll
        for (int w = 0; w < WORDS; ++w) word[w] = 0;
        // as in the kernel above; the product is one instruction with its widening (v_fma_mix: adding -0 changes nothing)
        auto quantise = [&](_Float16 x) -> uint32_t {
          float t = __builtin_fmaf((float)x, rscale, minus_zero);
          t = t + zf32;
          t = t + 0.49999997f;
          t = __builtin_amdgcn_fmed3f(t, 0.f, (float)MAXQ);
          return (uint32_t)t;
        };
#pragma unroll
        for (int e = 0; e < ROWS; ++e) word[e * BITS / 32] |= quantise(v[e][h]) << (e * BITS % 32);
        uint8_t* out = B + ((n + h) * kbc + kb) * BLOB + part * (ROWS * BITS / 8);
        if constexpr (WORDS % 4 == 0) {
#pragma unroll
          for (int w = 0; w < WORDS; w += 4)
            *reinterpret_cast<uint4*>(out + 4 * w) = make_uint4(word[w], word[w + 1], word[w + 2], word[w + 3]);
        } else {
#pragma unroll
          for (int w = 0; w < WORDS; ++w) *reinterpret_cast<uint32_t*>(out + 4 * w) = word[w];
        }
      }
    }
  }
}

// Blocks of 16, 32 and 64 elements: with one block per workgroup the tile is a few KiB, a thread has four to sixteen
// elements between three barriers, and a column's output arrives in pieces of 2 to 8 bytes (measured 52 us for
// blocks of 32 where blocks of 128 take 29 us on the same matrix).  Here a workgroup owns 128 columns x BPW blocks
// side by side along K (128 rows; 64 rows for blocks of 16): a thread takes a whole block of its column (half of a
// block of 64), so blocks of up to 32 need no exchange of ranges at all, the source is still read in 256-byte pieces
// of 64 or 128 rows, a column's BPW blobs are contiguous in B, and the zero points of the blocks that share a byte
// meet in LDS.  One pass per workgroup; the arithmetic is that of the kernel above, statement for statement.
// SLOTS = threads per column
template <typename T, int BITS, int BS, int TPB, int SLOTS, bool ALL>
__global__ void __launch_bounds__(kCols * SLOTS) mnb_quantize_small_kernel(uint8_t* __restrict__ B, T* __restrict__ scales,
                                                                            uint8_t* __restrict__ zp,
                                                                            const T* __restrict__ src, int64_t K,
                                                                            int64_t N, int64_t ld, int strips,
                                                                            int groups, int run) {
  constexpr int PER_BYTE = 8 / BITS;
  constexpr int MAXQ = (1 << BITS) - 1;
  constexpr int MID = 1 << (BITS - 1);
  constexpr int VEC = 16 / (int)sizeof(T);
  constexpr int EPT = BS / TPB;        // elements per thread
  constexpr int BPW = SLOTS / TPB;    // blocks per workgroup
  constexpr int ROWS = BPW * BS;
  constexpr int blob = BS * BITS / 8;
  constexpr int QWORDS = EPT * BITS / 32;
  static_assert(EPT * BITS % 32 == 0 && BPW % PER_BYTE == 0,
                "a thread writes whole words; a zero-point byte stays in one workgroup");
  extern __shared__ __align__(16) unsigned char smem[];
  T* tile = reinterpret_cast<T*>(smem);                                              // [ROWS][kCols]
  float* red = reinterpret_cast<float*>(smem + (size_t)ROWS * kCols * sizeof(T));    // [2][SLOTS][kCols]
  uint32_t* zs = reinterpret_cast<uint32_t*>(red + 2 * SLOTS * kCols);              // [BPW][kCols]

  const int tid = threadIdx.x;
  const int c = tid % kCols, slot = tid / kCols;
  const int bi = slot / TPB, part = slot % TPB;
  const MnbQuantTile qt = quant_tile(strips, groups, run);
  const int64_t n0 = qt.strip * kCols;
  const int64_t n = n0 + c;
  const int64_t kbc = (K + BS - 1) / BS;
  const int64_t zrow = (kbc * BITS + 7) / 8;
  const int64_t kb0 = qt.group * BPW;
  const int64_t k0 = kb0 * BS;
  const int rows = (int)(k0 + ROWS < K ? ROWS : K - k0);  // rows of the tile that exist (>= 1)
  const bool whole = rows == ROWS;

  if (ALL || n0 + kCols <= N) {
    constexpr int CH = kCols / VEC;                       // 16-byte chunks per row
    constexpr int PRE = ROWS * CH / (kCols * SLOTS);     // chunks per thread
    static_assert(ROWS * CH % (kCols * SLOTS) == 0, "whole chunks per thread");
    u4_t pre[PRE];
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const int i = tid + u * kCols * SLOTS;
      const int r = i / CH < rows ? i / CH : rows - 1;    // rows beyond K re-read the last one and are never used
      pre[u] = *reinterpret_cast<const typename PieceOf<T>::type*>(src + (k0 + r) * ld + n0 + (i % CH) * VEC);
    }
#pragma unroll
    for (int u = 0; u < PRE; ++u) {
      const int i = tid + u * kCols * SLOTS;
      *reinterpret_cast<u4_t*>(tile + (i / CH) * kCols + (i % CH) * VEC) = pre[u];
    }
  } else {
    fill_by_elements<T, ROWS / SLOTS, kCols * SLOTS>(tile, src + k0 * ld + n0, ld, rows, N - n0, tid);
  }
  if (!whole) clear_missing_rows<T, ROWS, kCols * SLOTS>(tile, rows, tid);
  __syncthreads();

  const int64_t kb = kb0 + bi;
  const bool exists = kb < kbc;
  const int e0 = bi * BS + part * EPT;                               // first row of this thread's elements
  float mn = 3.402823466e+38f, mx = -3.402823466e+38f;
#pragma unroll
  for (int e = 0; e < EPT; ++e) {
    const float v = (float)tile[(e0 + e) * kCols + c];
    mn = __builtin_fminf(v, mn);
    mx = __builtin_fmaxf(v, mx);
  }
  if (mn == 0.f && mx == 0.f) mn = mx = first_zero(tile + e0 * kCols + c, EPT);  // (see the kernel above)
  if constexpr (TPB > 1) {
    red[slot * kCols + c] = mn;
    red[(SLOTS + slot) * kCols + c] = mx;
    __syncthreads();
#pragma unroll
    for (int q2 = 0; q2 < TPB; ++q2) {
      const float a = red[(bi * TPB + q2) * kCols + c], b = red[(SLOTS + bi * TPB + q2) * kCols + c];
      mn = a < mn ? a : mn;
      mx = b > mx ? b : mx;
    }
  }
  float scale;
  int z;
  if (zp) {
    mn = mn < 0.f ? mn : 0.f;
    mx = mx > 0.f ? mx : 0.f;
    scale = (mx - mn) / (float)MAXQ;
    float zf = mn;
    if (scale != 0.f) zf = 0.f - mn / scale;
    zf = zf < 0.f ? 0.f : zf;
    zf = zf > (float)MAXQ ? (float)MAXQ : zf;
    z = (int)roundf(zf);
  } else {
    const float smax = fabsf(mx) > fabsf(mn) ? mx : mn;
    scale = -smax / (float)MID;
    z = MID;
  }
  if (zp) {
    // blocks beyond the last one leave the reference's filler, the default zero point, in their part of the byte
    if (part == 0) zs[bi * kCols + c] = exists ? (uint32_t)z : (uint32_t)MID;
    __syncthreads();
    if (part == 0 && bi % PER_BYTE == 0 && exists && n < N) {
      uint32_t zbyte = 0;
#pragma unroll
      for (int f = 0; f < PER_BYTE; ++f) zbyte |= zs[(bi + f) * kCols + c] << (f * BITS);
      zp[n * zrow + kb / PER_BYTE] = (uint8_t)zbyte;
    }
  }
  if (!exists || n >= N) return;
  const T stored = (T)scale;
  const float sf = (float)stored;
  const float rscale = sf != 0.f ? 1.0f / sf : 0.f;
  const float zf32 = (float)z;
  if (part == 0) scales[n * kbc + kb] = stored;
  auto quantise = [&](float v) -> uint32_t {  // clamp(roundf(v * rscale + zp), 0, MAXQ): see the kernel above
    float t = v * rscale;
    t = t + zf32;
    t = t + 0.49999997f;
    t = __builtin_amdgcn_fmed3f(t, 0.f, (float)MAXQ);
    return (uint32_t)t;
  };
  uint32_t word[QWORDS];
#pragma unroll
  for (int w = 0; w < QWORDS; ++w) word[w] = 0;
#pragma unroll
  for (int e = 0; e < EPT; ++e)
    word[(e * BITS) / 32] |= quantise((float)tile[(e0 + e) * kCols + c]) << ((e * BITS) % 32);
  if (!whole) zero_point_behind<BITS>(word, rows - e0, z);
  uint8_t* out = B + (n * kbc + kb) * blob + part * (EPT * BITS / 8);
  if constexpr (QWORDS % 4 == 0) {
#pragma unroll
    for (int w = 0; w < QWORDS; w += 4)
      *reinterpret_cast<uint4*>(out + 4 * w) = make_uint4(word[w], word[w + 1], word[w + 2], word[w + 3]);
  } else if constexpr (QWORDS % 2 == 0) {
#pragma unroll
    for (int w = 0; w < QWORDS; w += 2) *reinterpret_cast<uint2*>(out + 4 * w) = make_uint2(word[w], word[w + 1]);
  } else {
#pragma unroll
    for (int w = 0; w < QWORDS; ++w) *reinterpret_cast<uint32_t*>(out + 4 * w) = word[w];
  }
}

// Which order of the tiles (see mnb_quant_grid.h).  Runs of 16 groups pay where the writes weigh (8-bit weights, and the short blobs
// of fp16 blocks of 64 and fewer) and where neighbouring strips share the lines at their seam (rows at odd addresses), given
// enough tiles for eight XCDs; strips side by side read better.  Measured, side by side / runs, us, [4096, 14336] unless
// said: 8-bit blocks of 128 45.5 / 40.0, blocks of 64 49.8 / 42.2, fp32 66.9 / 60.4; 4-bit blocks of 32 38.4 / 37.1, blocks of
// 64 38.2 / 35.9, with zero points 37.8 / 37.3; odd fp16 rows [4832, 12825] blocks of 32 61.0 / 48.2, [4096, 4099] 15.9 / 14.3;
// but 4-bit blocks of 128 32.0 / 33.4, fp32 4-bit 55.2 / 57.2, [4096, 4096] fp32 19.4 / 20.9, blocks of 16 34.0 / 35.5, fp16
// blocks of 256 41.1 / 43.7.
MnbQuantGrid quant_grid(const void* src, int elem, int bits, int bs, int64_t N, int64_t ld, int64_t groups, int threads) {
  const int64_t strips = (N + kCols - 1) / kCols, tiles = strips * groups, cus = mnb_device_info().cus;
  const bool pieces = reinterpret_cast<uintptr_t>(src) % 16 == 0 && ld * elem % 16 == 0;
  bool runs = elem == 2 && !pieces ? tiles >= 4 * cus : tiles >= 8 * cus && (bits == 8 || (elem == 2 && bs <= 64));
  if (bs == 16 || (bs == 256 && pieces)) runs = false;
  if (const char* e = mnb_tuning_env("MNB_QUANT_RUNS")) runs = e[0] == '1';  // calibration
  return mnb_quant_grid(strips, groups, threads, runs);
}

template <typename T, int BITS, int BS>
hipError_t launch_small(void* B, void* scales, void* zp, const void* src, int64_t K, int64_t N, int64_t ld,
                        hipStream_t s) {
  constexpr int TPB = (BS == 64 && BITS != 2) ? 2 : 1;  // 2-bit blocks of 64: four blocks share a zero-point byte
  constexpr int SLOTS = 4;  // (eight for blocks of 16 - 128 rows again - was measured: no difference)
  constexpr int BPW = SLOTS / TPB, ROWS = BPW * BS;
  const auto kernel = N % kCols == 0 ? mnb_quantize_small_kernel<T, BITS, BS, TPB, SLOTS, true>
                                     : mnb_quantize_small_kernel<T, BITS, BS, TPB, SLOTS, false>;
  const size_t smem = (size_t)ROWS * kCols * sizeof(T) + 2 * SLOTS * kCols * sizeof(float) + (size_t)BPW * kCols * 4;
  if (smem > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)smem);
    if (e != hipSuccess) return e;
  }
  const int64_t kbc = (K + BS - 1) / BS;
  const int64_t strips = (N + kCols - 1) / kCols, groups = (kbc + BPW - 1) / BPW;
  const MnbQuantGrid g = quant_grid(src, sizeof(T), BITS, BS, N, ld, groups, kCols * SLOTS);
  if (!g.ok) return hipErrorInvalidConfiguration;
  kernel<<<dim3(g.x, g.y), dim3(kCols * SLOTS), smem, s>>>((uint8_t*)B, (T*)scales, (uint8_t*)zp, (const T*)src, K, N, ld,
                                                   (int)strips, (int)groups, g.run);
  return hipGetLastError();
}

template <typename T, int BITS, int QROWS>
hipError_t launch_k(void* B, void* scales, void* zp, const void* src, int64_t K, int64_t N, int64_t ld, hipStream_t s) {
  constexpr int bs = QROWS * kQuarters;
  // (fp32 blocks of 256, two wavefronts a SIMD whatever the registers: the form without the other fill is faster where a
  // workgroup takes several blocks, [8192, 8192] 4-bit with zero points 70.5 us and 75.0, and slower where it takes one, 8-bit
  // [4096, 8192] 49.1 us and 47.4)
  constexpr bool kForms = QROWS <= 32 || BITS < 8;
  const bool whole_strips = N % kCols == 0 && (QROWS <= 32 || zp != nullptr);
  const auto kernel = kForms && whole_strips ? mnb_quantize_kernel<T, BITS, QROWS, kForms> : mnb_quantize_kernel<T, BITS, QROWS, false>;
  const size_t smem = (size_t)bs * kCols * sizeof(T) + 2 * kQuarters * kCols * sizeof(float);
  // fp32 sources with 256-deep blocks need 66 KiB of LDS: above the default limit, within the CU's 160 KiB
  if (smem > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)smem);
    if (e != hipSuccess) return e;
  }
  const int64_t kbc = (K + bs - 1) / bs;
  // Blocks per workgroup: the 8/bits blocks of one zero-point byte when zero points are written, else one.  Many
  // small workgroups beat few long ones here: [4096, 14336] fp16 to 4 bits, blocks of 128, took 36 us with one
  // block per workgroup, 41 us with two and 44-46 us with four to eight (64-column workgroups).
  const int nsub = zp ? 8 / BITS : 1;
  const int64_t strips = (N + kCols - 1) / kCols, groups = (kbc + nsub - 1) / nsub;
  const MnbQuantGrid g = quant_grid(src, sizeof(T), BITS, bs, N, ld, groups, kCols * kQuarters);
  if (!g.ok) return hipErrorInvalidConfiguration;
  kernel<<<dim3(g.x, g.y), dim3(kCols * kQuarters), smem, s>>>((uint8_t*)B, (T*)scales, (uint8_t*)zp, (const T*)src, K, N, ld,
                                                       nsub, (int)strips, (int)groups, g.run);
  return hipGetLastError();
}

template <int BITS, int PARTS>
hipError_t launch_pairs(void* B, void* scales, void* zp, const void* src, int64_t K, int64_t N, int64_t ld, hipStream_t s) {
  const int64_t kbc = (K + 32 * PARTS - 1) / (32 * PARTS);
  const int nsub = zp ? 8 / BITS : 1;  // (as above)
  const int64_t strips = (N + kCols - 1) / kCols, groups = (kbc + nsub - 1) / nsub;
  const MnbQuantGrid g = quant_grid(src, 2, BITS, 32 * PARTS, N, ld, groups, 64 * PARTS);
  if (!g.ok) return hipErrorInvalidConfiguration;
  // (dwords at multiples of four, 32-bit offsets within the 32 rows of a wavefront)
  const bool dwords = (reinterpret_cast<uintptr_t>(src) % 4 == 0) && (ld % 2 == 0) && ld < (1 << 25);
  const bool all = dwords && N % kCols == 0 && K % (32 * PARTS) == 0;
  // (a matrix of fewer than 128 columns is read element by element in either form: [9182, 33] 2-bit 21.7 us and 22.7)
  const auto kernel = all                   ? mnb_quantize_pairs_kernel<BITS, PARTS, kAllDwords>
                      : dwords || N < kCols ? mnb_quantize_pairs_kernel<BITS, PARTS, kDwords>
                                            : mnb_quantize_pairs_kernel<BITS, PARTS, kAnyPairs>;
  kernel<<<dim3(g.x, g.y), dim3(64 * PARTS), 0, s>>>((uint8_t*)B, (_Float16*)scales, (uint8_t*)zp, (const _Float16*)src, K, N, ld,
                                                     nsub, (int)strips, (int)groups, g.run);
  return hipGetLastError();
}

template <typename T, int BITS>
hipError_t launch_b(void* B, void* scales, void* zp, const void* src, int64_t K, int64_t N, int64_t ld, int bs,
                    hipStream_t s) {
  switch (bs) {
    case 16: return launch_small<T, BITS, 16>(B, scales, zp, src, K, N, ld, s);
    case 32: return launch_small<T, BITS, 32>(B, scales, zp, src, K, N, ld, s);
    case 64:
      // measured on [4096, 14336]: the side-by-side kernel is 3-25 % faster, except for fp16 sources to 8 bits
      // (5-7 % slower), and for fp16 to 2 bits while there are few tiles, for a thread there has all 64 elements of a block
      // (side by side / one block a workgroup: [1000, 2048] 7.1 / 4.5 us, [4096, 130] 8.2 / 5.7, [2048, 2048] 6.0 / 5.3;
      // [1500, 3000], three tiles a unit, 8.7 / 8.9, [4096, 14336] 33.9 / 40.4)
      if constexpr (BITS == 2 && sizeof(T) == 2)
        if (zp == nullptr && (N + kCols - 1) / kCols * ((K + 63) / 64) <= 2 * mnb_device_info().cus)
          return launch_k<T, BITS, 16>(B, scales, zp, src, K, N, ld, s);
      if constexpr (BITS == 8 && sizeof(T) == 2) return launch_k<T, BITS, 16>(B, scales, zp, src, K, N, ld, s);
      else return launch_small<T, BITS, 64>(B, scales, zp, src, K, N, ld, s);
    case 128: return launch_k<T, BITS, 32>(B, scales, zp, src, K, N, ld, s);
    case 256:
      if constexpr (sizeof(T) == 2) return launch_pairs<BITS, 8>(B, scales, zp, src, K, N, ld, s);
      else return launch_k<T, BITS, 64>(B, scales, zp, src, K, N, ld, s);
    default: return hipErrorInvalidValue;
  }
}

template <typename T>
hipError_t launch_t(void* B, void* scales, void* zp, const void* src, int64_t K, int64_t N, int64_t ld, int bits,
                    int bs, hipStream_t s) {
  if (bits == 2) return launch_b<T, 2>(B, scales, zp, src, K, N, ld, bs, s);
  return bits == 4 ? launch_b<T, 4>(B, scales, zp, src, K, N, ld, bs, s) : launch_b<T, 8>(B, scales, zp, src, K, N, ld, bs, s);
}

}  // namespace

hipError_t mnb_launch_quantize(void* B, void* scales, void* zp, const void* src, int64_t K, int64_t N, int64_t ld,
                               int bits, int bs, int dtype, hipStream_t s) {
  if (K == 0 || N == 0) return hipSuccess;
  return dtype == kMnbDtypeFloat16 ? launch_t<_Float16>(B, scales, zp, src, K, N, ld, bits, bs, s)
                                   : launch_t<float>(B, scales, zp, src, K, N, ld, bits, bs, s);
}
