// The streaming kernel whose wavefronts share the activations in LDS.  A workgroup of eight wavefronts owns 32 RT rows and
// 32 CW columns; a wavefront owns 32 of the columns and all the rows.  K goes in chunks of 128: TEAMS = 8 / CW teams of
// CW wavefronts each take their own 128 / TEAMS k of every chunk, and their sums meet in LDS at the end, in team order.
//
// Why this shape.  A weight costs two vector instructions to dequantise, and beside a matrix instruction of 32 cycles only
// six vector instructions are free (measured: four add 6 % to a loop of matrix instructions, ten 60 %): a wavefront
// multiplies each dequantised operand (16 k x 32 columns) with RT row tiles.  The activations of a chunk come through the
// address unit at 64 bytes a cycle and compute unit, once per workgroup, straight into LDS (no registers); four stages,
// three chunks ahead.  The weights are loaded as whole 16-byte vectors, 1 KB an instruction, three chunks ahead.
//
// Measured before / now (us, weights from HBM): 128 rows of 11008 x 4096 4-bit 30.7 / 21.3, 256 rows of 6144 x 4096 27.2 / 21.1
// (bfloat16, called eagerly, 26.7 / 17.6 to 19.1 by the card, where the products alone need 8.1; mnb_mid.hip holds the times by tile).  What bounds it by
// the counters: matrix and vector instructions, 16.5 K cycles a SIMD each, hardly overlap in the 38 to 41 K that a compute unit is
// busy, a quarter of the units has no workgroup, and 4 to 7 us are launch, first chunks and sums at the end.
// Tried and not kept: a team of producer wavefronts, the fills spread between the matrix instructions, eight stages, weights
// with the non-temporal hint, tiles in launch order: each 0 to 6 % slower.
#pragma once
#include <atomic>
#include <type_traits>

#include "mnb_mfma16_common.hip.h"

namespace {

constexpr int kRowsChunk = 128, kRowsStages = 4;

// exact (q - zp) * scale for the 8 weights of one 4-bit word / the 8 weights of two 8-bit words
template <int BITS>
__device__ __forceinline__ h8_t dequant_word(uint32_t w0, uint32_t w1, const UnpackConsts& uc, h2_t z_lo, h2_t z_hi,
                                             h2_t s2) {
  uint4 r;
  if constexpr (BITS == 4) {
    const uint32_t w8 = w0 >> 8;
    const h2_t p0 = mnb_as_h2((w0 & uc.mask_lo) | uc.magic_lo);  // 1024 + q
    const h2_t p1 = mnb_as_h2((w0 & uc.mask_hi) | uc.magic_hi);  //   64 + q
    const h2_t p2 = mnb_as_h2((w8 & uc.mask_lo) | uc.magic_lo);
    const h2_t p3 = mnb_as_h2((w8 & uc.mask_hi) | uc.magic_hi);
    r.x = mnb_as_u32((p0 + z_lo) * s2);
    r.y = mnb_as_u32((p1 + z_hi) * s2);
    r.z = mnb_as_u32((p2 + z_lo) * s2);
    r.w = mnb_as_u32((p3 + z_hi) * s2);
  } else {
    const h2_t p0 = mnb_as_h2(__builtin_amdgcn_perm(kMagic, w0, 0x07010700u));
    const h2_t p1 = mnb_as_h2(__builtin_amdgcn_perm(kMagic, w0, 0x07030702u));
    const h2_t p2 = mnb_as_h2(__builtin_amdgcn_perm(kMagic, w1, 0x07010700u));
    const h2_t p3 = mnb_as_h2(__builtin_amdgcn_perm(kMagic, w1, 0x07030702u));
    r.x = mnb_as_u32((p0 + z_lo) * s2);
    r.y = mnb_as_u32((p1 + z_lo) * s2);
    r.z = mnb_as_u32((p2 + z_lo) * s2);
    r.w = mnb_as_u32((p3 + z_lo) * s2);
  }
  return __builtin_bit_cast(h8_t, r);
}


struct MidRowsParams {
  SkinnyParams s;
  int row_blocks;
  // ANY alone:
  int ragged;        // 1: the last chunk of K is not whole (K a multiple of 8, rows that 16-byte loads can read)
  uint32_t a_bytes;  // of A, from its first value to its last: what lies behind reads as zeros
  int split_chunks;  // K is cut along the grid's second dimension, so many chunks each (an even number); 0: it is not
  f4_t* partial;     // ... and the sums go here, [cut][tile][quad of rows][lane], for mnb_mid_rows_sum_kernel
};

template <int RT>
constexpr size_t kMidRowsLds = (size_t)kRowsStages * RT * 32 * kRowsChunk * 2;

typedef uint32_t u4_any_t __attribute__((ext_vector_type(4), aligned(2)));  // a 16-byte store to any 16-bit element

// A finished tile of ROWS x COLS values in the output's type: `put(out, pitch)` lays the workgroup's values side by side in LDS, then
// 512 threads write 16 bytes each.  What a workgroup does once is bound by its branches and by fetching its instructions, so: no
// branch around a single value, one path for each kind of output, shifts for rows and pieces, the bias asked for ahead of the
// sums.  Behind the loop a workgroup took 4650 cycles with 64 x 128 tiles and 5900 with 128 x 64 (2.1 and 2.6 us), now 3400 and
// 4800: half a microsecond of 18 to 20 (128 rows of 11008 x 4096 and 256 rows of 6144 x 4096 in bfloat16, side by side on one card).
template <int ROWS, int COLS, class F>
__device__ __forceinline__ void store_rows(const SkinnyParams& p, _Float16* out, int thread, int m0, int64_t n0, F&& put) {
  constexpr int PITCH = COLS + 8, PER_ROW = COLS / 8, STEP = 512 / PER_ROW;
  put(out, PITCH);
  // the thread's columns, the same in all its rows (packed columns of fused outputs begin at multiples of 16)
  const int piece = thread % PER_ROW, row = thread / PER_ROW;
  int64_t n = n0 + piece * 8, limit = p.epi.kind == kMnbFusedNone ? p.N : p.epi.n0, ld = p.ldc;
  _Float16* dst = p.C;
  if (p.epi.kind == kMnbFusedQkv && n >= p.epi.start1) {
    const bool third = n >= p.epi.start2;
    dst = third ? p.epi.out2 : p.epi.out1, ld = third ? p.epi.ld2 : p.epi.ld1;
    limit = third ? p.epi.n2 : p.epi.n1, n -= third ? p.epi.start2 : p.epi.start1;
  }
  dst += (int64_t)(m0 + row) * ld + n;
  const _Float16* src = out + row * PITCH + piece * 8;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < ROWS; r += STEP, dst += STEP * ld, src += STEP * PITCH) {
    if ((ROWS % STEP != 0 && row + r >= ROWS) || m0 + row + r >= p.M) break;  // (96 rows in steps of 64: half a step too many)
    if (n + 8 <= limit) {
      *reinterpret_cast<u4_any_t*>(dst) = *reinterpret_cast<const u4_t*>(src);
    } else {
#pragma unroll 1
      for (int e = 0; n + e < limit; ++e) dst[e] = src[e];
    }
  }
}

// Wavefronts a SIMD: two workgroups' for up to two row tiles.  Small 4-bit tiles fit four workgroups by themselves, but for those
// without zero points, which took 65 registers unasked (with zero points the demand would spill).
// ANY: K with a ragged last chunk, or cut over workgroups.  (A form of its own: what it has to know before its first loads costs the
// other one 0.3 us of 9.5, 300 rows of 1024 x 3072 in bfloat16.)
template <int BITS, bool HAS_ZP, int RT, int CW, int IO, bool ANY>
__global__ void __launch_bounds__(512, RT == 1 && BITS == 4 && !HAS_ZP ? 8 : RT <= 2 ? 4 : 2) mnb_mid_shared_rows_kernel(MidRowsParams mp) {
  const SkinnyParams& p = mp.s;
  constexpr bool WIDE = IO != kMnbIoModel;
  constexpr int TEAMS = 8 / CW, STAGES = kRowsStages, ROWS = 32 * RT, COLS = 32 * CW;
  constexpr int SLABS = 8 / TEAMS;              // operands of 16 k that a wavefront makes of a chunk
  constexpr int STAGE_BYTES = ROWS * kRowsChunk * 2;
  constexpr bool PAIRS = BITS == 4 && CW == 2;  // weights of two chunks at a time
  constexpr int VECS = BITS == 8 && CW == 4 ? 2 : 1;
  constexpr int META_BYTES = (WIDE ? 2 : 1) * (HAS_ZP ? 4 : 2);
  constexpr int W_LOADS = 2 * VECS;
  using meta_t = std::conditional_t<WIDE && HAS_ZP, u2_t, uint32_t>;
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int team = wave / CW, cw = wave % CW;
  const int li = lane & 31, kq = lane >> 5;

  // Workgroups go to the eight XCDs round-robin: each XCD takes a contiguous run of tiles, row blocks of a slab side by side,
  // so that its level-2 cache serves the slab's weights to all but the first.
  const int tiles = gridDim.x, xcd = blockIdx.x & 7;
  const int tile = xcd * (tiles >> 3) + min(xcd, tiles & 7) + (int)(blockIdx.x >> 3);
  const int m0 = tile % mp.row_blocks * ROWS;
  const int64_t n0 = (int64_t)(tile / mp.row_blocks) * COLS;
  // the workgroup's chunks of K
  const int c0 = ANY ? (int)blockIdx.y * mp.split_chunks : 0;
  const int chunks = ANY && mp.split_chunks ? min(mp.split_chunks, p.chunks - c0) : p.chunks;
  const int last = chunks - 1;

  // Every address is a fixed base, a fixed offset per lane and one scalar: activations, weights and entries lie within 4 GiB
  // of their bases (the host checks).
  // ---- activations: a chunk's 256 bytes of every row; one instruction covers four rows.  16-byte pieces are
  // XOR-swizzled with the row, so that the 16 rows that an operand read takes at a time hit all banks.
  uint32_t a_off[RT];
#pragma unroll
  for (int u = 0; u < RT; ++u) {
    const int row = (wave * RT + u) * 4 + (lane >> 4);
    const int grow = m0 + row < p.M ? m0 + row : p.M - 1;  // rows beyond M re-read the last row and are never stored
    a_off[u] = (uint32_t)(((int64_t)grow * p.lda + ((lane & 15) ^ (row & 15)) * 8) * 2);
  }
  // A ragged last chunk goes first, so that the loop knows nothing of it: step 0 takes chunk `last`, whose pieces beyond K lie
  // behind the buffer's end and arrive as zeros (what stands there may be no number), and step c chunk c - 1.
  const int ragged = ANY && c0 + chunks == p.chunks ? mp.ragged : 0;
  auto chunk_of = [&](int c) __attribute__((always_inline)) {
    if (c > last) c = last;
    return ANY ? max(c - ragged, 0) : c;
  };
  const rsrc_t a_rsrc = ANY ? mnb_rsrc_bytes(p.A + c0 * kRowsChunk, mp.a_bytes - (uint32_t)c0 * (kRowsChunk * 2)) : mnb_rsrc(p.A);
  auto fill = [&](int c, int stage) __attribute__((always_inline)) {
    const uint32_t k = (uint32_t)chunk_of(c) * (kRowsChunk * 2);
#pragma unroll
    for (int u = 0; u < RT; ++u)
      mnb_buffer_load_lds_b128(a_rsrc, a_off[u], (lds_ptr_t)(smem + stage * STAGE_BYTES + (wave * RT + u) * 1024), k);
  };
  auto fill_first = [&]() __attribute__((always_inline)) {
    const int first = ragged ? last : 0, pieces = (p.K - (c0 + first) * kRowsChunk) / 8;  // of 16 bytes, up to K
#pragma unroll
    for (int u = 0; u < RT; ++u) {
      const int piece = (lane & 15) ^ (((wave * RT + u) * 4 + (lane >> 4)) & 15);
      const uint32_t off = a_off[u] + (uint32_t)first * (kRowsChunk * 2);
      mnb_buffer_load_lds_b128(a_rsrc, !ragged || piece < pieces ? off : 0xFFFFFFF0u, (lds_ptr_t)(smem + (wave * RT + u) * 1024));
    }
  };
  // The k of a lane's operands are those of its weights: any permutation of them will do, the same on both sides.
  uint32_t a_rd[SLABS];
#pragma unroll
  for (int s = 0; s < SLABS; ++s) {
    const int piece = CW == 2 ? 4 * team + 2 * kq + s : BITS == 4 ? 8 * team + 4 * kq + s : 8 * team + 4 * (s >> 1) + 2 * kq + (s & 1);
    a_rd[s] = (uint32_t)(li * 256 + ((piece ^ (li & 15)) << 4));
  }
  auto read_a = [&](int stage, int s, h8_t (&f)[RT]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < RT; ++t) f[t] = *reinterpret_cast<const h8_t*>(smem + a_rd[s] + stage * STAGE_BYTES + t * 8192);
  };

  // ---- weights: lane (column li, half kq of the wavefront) takes a vector of k-group ...
  //   CW = 4, 4-bit  2 team + kq: four words, the operands of the four slabs
  //   CW = 4, 8-bit  4 team + 2 v + kq, v = 0, 1: two words a slab
  //   CW = 2, 8-bit  2 team + kq
  //   CW = 2, 4-bit  team, of chunk c + kq (c even): exchanging halves of the wavefront leaves every lane the two words of its
  //                  own half of the k-group, of both chunks
  // of its chunk, and the meta entry of its block (blocks of 32 and more).
  struct Raw {
    u4_t w[VECS];
    meta_t m[VECS];
  };
  constexpr int GROUPS = BITS == 4 ? 4 : 8;  // k-groups of a chunk
  const int col = cw * 32 + li;
  const uint32_t w_pitch = (uint32_t)(p.Npad * 16), m_pitch = (uint32_t)(p.Npad * META_BYTES);
  const rsrc_t w_rsrc = mnb_rsrc(reinterpret_cast<const uint8_t*>(p.W) + n0 * 16 + (int64_t)(c0 * GROUPS) * w_pitch);
  const rsrc_t m_rsrc = mnb_rsrc(p.meta + n0 * META_BYTES + (int64_t)((c0 * kRowsChunk) >> p.bs_shift) * m_pitch);
  const uint32_t m_byte = (uint32_t)(mnb_meta_col(col) * META_BYTES), m_shift = (m_byte & 2u) * 8;
  const uint32_t w_one = (uint32_t)col * 16, m_one = WIDE ? m_byte : (m_byte & ~3u);
  const uint32_t w_two = w_one + (kq ? (PAIRS ? GROUPS : 1) * w_pitch : 0u);
  // (blocks of 256: the second chunk of a pair lies in the next block where the pairs begin at odd chunks)
  const uint32_t m_step = PAIRS ? (uint32_t)((kRowsChunk << (p.bs_shift == 8 ? ragged : 0)) >> p.bs_shift) : 32u >> p.bs_shift;
  const uint32_t m_two = m_one + (kq && BITS == 4 ? m_step * m_pitch : 0u);
  // vector v and its entry: a lane's offsets, and the chunk that the scalar ones are of
  auto load_one = [&](Raw& R, int v, int c, uint32_t w_off, uint32_t m_off) __attribute__((always_inline)) {
    const uint32_t g = (uint32_t)(c * GROUPS + team * (GROUPS / TEAMS) + 2 * v);
    R.w[v] = mnb_buffer_load_b128(w_rsrc, w_off, g * w_pitch);
    const uint32_t at = ((uint32_t)(c * kRowsChunk + team * (kRowsChunk / TEAMS) + v * 32) >> p.bs_shift) * m_pitch;
    if constexpr (WIDE && HAS_ZP) R.m[v] = mnb_buffer_load_b64(m_rsrc, m_off, at);
    else R.m[v] = mnb_buffer_load_b32(m_rsrc, m_off, at);
  };
  auto load_w = [&](int c_raw, Raw& R) __attribute__((always_inline)) {
    const bool two = !PAIRS || c_raw < last;  // (behind the last chunk there is none)
#pragma unroll
    for (int v = 0; v < VECS; ++v) load_one(R, v, chunk_of(c_raw), two ? w_two : w_one, two ? m_two : m_one);
  };
  auto load_first = [&](Raw& R) __attribute__((always_inline)) {  // step 0: chunk `last` where that is ragged (PAIRS: with chunk 0)
    if constexpr (PAIRS) {
      const uint32_t from = (uint32_t)(team * 32);
      const uint32_t m_ahead = (((uint32_t)(last * kRowsChunk) + from) >> p.bs_shift) - (from >> p.bs_shift);
      const bool ahead = ragged && !kq;
      const bool two = last > 0 && !ragged;
      load_one(R, 0, 0, ahead ? w_one + (uint32_t)(last * GROUPS) * w_pitch : two ? w_two : w_one,
               ahead ? m_one + m_ahead * m_pitch : two ? m_two : m_one);
    } else {
#pragma unroll
      for (int v = 0; v < VECS; ++v) load_one(R, v, ragged ? last : 0, w_two, m_two);
    }
  };
  meta_t pair_m[2];  // PAIRS: entries of the two chunks
  auto arrange = [&](Raw& R) __attribute__((always_inline)) {
    auto swap = [](uint32_t& a, uint32_t& b) __attribute__((always_inline)) {  // upper half of a with lower half of b
#if defined(__HIP_DEVICE_COMPILE__)
      const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
      a = r[0], b = r[1];
#endif
    };
    uint32_t w0 = R.w[0][0], w1 = R.w[0][1], w2 = R.w[0][2], w3 = R.w[0][3];
    swap(w0, w2);
    swap(w1, w3);
    R.w[0] = u4_t{w0, w1, w2, w3};  // words 0, 1: chunk c, words 2, 3: chunk c + 1
    if constexpr (WIDE && HAS_ZP) {
      uint32_t s0 = R.m[0][0], s1 = s0, z0 = R.m[0][1], z1 = z0;
      swap(s0, s1);
      swap(z0, z1);
      pair_m[0] = u2_t{s0, z0}, pair_m[1] = u2_t{s1, z1};
    } else {
      uint32_t e0 = R.m[0], e1 = e0;
      swap(e0, e1);
      pair_m[0] = e0, pair_m[1] = e1;
    }
  };
  const UnpackConsts uc = make_unpack_consts();
  auto make_b = [&](const Raw& R, int odd, int s) __attribute__((always_inline)) {
    const int v = VECS == 2 ? s >> 1 : 0;
    const uint32_t w0 = PAIRS ? R.w[0][2 * odd + (s & 1)] : BITS == 4 ? R.w[0][s & 3] : R.w[v][2 * (s & 1)];
    const uint32_t w1 = BITS == 4 ? 0u : R.w[v][2 * (s & 1) + 1];
    meta_t m;
    if constexpr (PAIRS) m = pair_m[odd];
    else m = R.m[v];
    if constexpr (WIDE) {
      float sc, zp;
      if constexpr (HAS_ZP) {
        const uint32_t sc_bits = m[0], zp_bits = m[1];
        sc = __uint_as_float(sc_bits), zp = __uint_as_float(zp_bits);
      } else {
        sc = __uint_as_float(m), zp = (float)(1 << (BITS - 1));
      }
      return dequant_word_wide<BITS, IO == kMnbIoBf16>(w0, w1, sc, -zp * sc);
    } else {
      _Float16 sc, nz;
      decode_meta<BITS, HAS_ZP>(HAS_ZP ? (uint32_t)m : (uint32_t)m >> m_shift, sc, nz);
      return dequant_word<BITS>(w0, w1, uc, mnb_h2(nz), mnb_h2(nz + (_Float16)960.0f), mnb_h2(sc));
    }
  };

  f16_t acc[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;
  auto multiply = [&](const h8_t (&a)[RT], h8_t b) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < RT; ++t) {
#if defined(__HIP_DEVICE_COMPILE__)
      if constexpr (IO == kMnbIoBf16)
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8_t, a[t]), __builtin_bit_cast(bf8_t, b), acc[t], 0, 0, 0);
      else
        acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t], b, acc[t], 0, 0, 0);
#endif
    }
  };
  // RT matrix instructions with the vector instructions of one operand between them
  auto interleave = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, (WIDE ? 28 : 18) / RT, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // Order of the vector-memory operations: step c issues the activations of chunk c + 3 at its begin and the weights of chunk
  // c + 4 at its end (PAIRS: of chunks c + 3 and c + 4, where c is odd).
  Raw R[PAIRS ? 2 : STAGES];
  h8_t a[2][RT], b[2];  // operands of the even and the odd slabs
#pragma unroll
  for (int t = 0; t < RT; ++t) a[1][t] = h8_t{};
  b[1] = h8_t{};
  auto load_at = [&](int c) __attribute__((always_inline)) {  // the weights that step c loads, from - 4 on
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PAIRS) {
      if (ANY && c == -3) load_first(R[0]);
      else if ((c & 1) != 0) load_w(c + 3, R[((c + 3) >> 1) & 1]);
    } else {
      if (ANY && c == -4) load_first(R[0]);
      else load_w(c + STAGES, R[c & (STAGES - 1)]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (!PAIRS) load_at(-4);
#pragma unroll
  for (int i = 0; i < STAGES - 1; ++i) {
    if (ANY && i == 0) fill_first();
    else fill(i, i);
    load_at(i - 3);
  }
  // (stage = c modulo 4.  TAIL: the last chunks, up to three: all that they need has been asked for, and they ask for
  // nothing.  The compiler would drop loads that nothing uses, and the counts of the waits would no longer hold.)
  auto step = [&](int c, auto stage_of, auto tail) __attribute__((always_inline)) {
    constexpr int stage = decltype(stage_of)::value, odd = stage & 1;
    constexpr bool TAIL = decltype(tail)::value;
    Raw& W = R[PAIRS ? stage >> 1 : stage];
    // Behind the barrier: the activations of chunk c are in LDS (younger are those of the next two chunks and the weights
    // loaded since), and nobody reads those of chunk c - 1 any more, whose stage is filled again.
    constexpr int kFills = TAIL ? 2 - stage : STAGES - 2;
    constexpr int kLoads = PAIRS ? (TAIL ? (stage == 0 ? 2 : 1) : odd ? 1 : 2) : (TAIL ? 3 - stage : 3);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lds0(kFills * RT + kLoads * W_LOADS));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < SLABS; ++s) {
      read_a(stage, s, a[s & 1]);
      __builtin_amdgcn_sched_barrier(0);
      if (s == 0) {
        if constexpr (!TAIL) fill(c + STAGES - 1, (stage + STAGES - 1) % STAGES);
        if constexpr (PAIRS && !odd) arrange(W);
      }
      multiply(a[(s & 1) ^ 1], b[(s & 1) ^ 1]);  // the slab before, of the step before if need be (zeros in front of the first)
      b[s & 1] = make_b(W, odd, s);
      interleave();
    }
    if constexpr (!TAIL && PAIRS && odd) load_w(c + 3, W);
    if constexpr (!TAIL && !PAIRS) load_w(c + STAGES, W);
  };
  using std::integral_constant;
  constexpr integral_constant<int, 0> s0{};
  constexpr integral_constant<int, 1> s1{};
  constexpr integral_constant<int, 2> s2{};
  constexpr integral_constant<int, 3> s3{};
  int c = 0;
  for (; c + STAGES <= chunks; c += STAGES) {
    step(c, s0, std::false_type{});
    step(c + 1, s1, std::false_type{});
    step(c + 2, s2, std::false_type{});
    step(c + 3, s3, std::false_type{});
  }
  // (nested, not a loop with exits: behind a join the number of loads in flight would not be known)
  if (c < chunks) {
    step(c, s0, std::true_type{});
    if (c + 1 < chunks) {
      step(c + 1, s1, std::true_type{});
      if (c + 2 < chunks) step(c + 2, s2, std::true_type{});
    }
  }
  multiply(a[1], b[1]);

  // ---- sums of the teams.  Register 4 q + i of acc[t]: row 32 t + 8 q + 4 kq + i, column li of the wavefront's 32.
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lds0(0));  // the last prefetches write LDS the sums are about to reuse
  __syncthreads();
  int own = lane, thread = threadIdx.x;
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (RT == 1 && BITS == 4) {  // the lane's number anew: no register of it through the loop of the tiles that have 64
    own = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    thread = wave * 64 + own;
  }
#endif
  const int own_col = cw * 32 + (own & 31);
  constexpr bool bf16 = IO == kMnbIoBf16;
  const float bias = p.bias && n0 + own_col < p.N ? widen16(p.bias[n0 + own_col], bf16) : 0.f;  // (arrives during the sums)
  float* const red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<f4_t*>(red + ((((cw * RT + t) * 4 + q) * TEAMS + team) * 64 + own) * 4) =
          f4_t{acc[t][4 * q], acc[t][4 * q + 1], acc[t][4 * q + 2], acc[t][4 * q + 3]};
  __syncthreads();
  // The wavefronts of a column share out its 4 RT quads of rows (unit = 4 t + q).
  constexpr int UNITS = 4 * RT / TEAMS;
  f4_t sum[UNITS];
#pragma unroll
  for (int u = 0; u < UNITS; ++u) {
    sum[u] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < TEAMS; ++k)
      sum[u] += *reinterpret_cast<const f4_t*>(red + (((cw * RT * 4 + team + TEAMS * u) * TEAMS + k) * 64 + own) * 4);
  }
  if (ANY && mp.split_chunks) {
    f4_t* const dst = mp.partial + ((int64_t)blockIdx.y * tiles + tile) * (ROWS * COLS / 4) + (cw * RT * 4 + team) * 64 + own;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) dst[TEAMS * u * 64] = sum[u];
    return;
  }
  __syncthreads();
  auto row_of = [&](int u) __attribute__((always_inline)) {
    const int unit = team + TEAMS * u;
    return (unit >> 2) * 32 + (unit & 3) * 8 + 4 * (own >> 5);
  };
  if (p.epi.kind == kMnbFusedMlp) {
    store_rows<ROWS, COLS / 2>(p, reinterpret_cast<_Float16*>(smem), thread, m0, n0 / 2, [&](_Float16* out, int pitch) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // lanes l and l + 16: gate and up of the same output column
          const float v = sum[u][i] + bias, up = __shfl_xor(v, 16, 64);
          if ((own & 31) < 16) out[(row_of(u) + i) * pitch + cw * 16 + (own & 31)] = narrow16(v / (1.0f + __expf(-v)) * up, bf16);
        }
    });
  } else {
    store_rows<ROWS, COLS>(p, reinterpret_cast<_Float16*>(smem), thread, m0, n0, [&](_Float16* out, int pitch) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) out[(row_of(u) + i) * pitch + own_col] = narrow16(sum[u][i] + bias, bf16);
    });
  }
}

// The sums of `splits` cuts of K, in their order, bias and narrowing: a workgroup takes 256 quads of rows of a tile, a thread one.  Bound by
// its launch (2 us) and by the partial sums, which come from the level-2 caches and the Infinity Cache.
template <int RT, int CW>
__global__ void __launch_bounds__(256) mnb_mid_rows_sum_kernel(MidRowsParams mp, int splits, int tiles) {
  const SkinnyParams& p = mp.s;
  const int tile = blockIdx.x / (RT * CW), quad = blockIdx.x % (RT * CW) * 256 + threadIdx.x;
  const int lane = quad & 63, unit = (quad >> 6) % (4 * RT), cw = (quad >> 6) / (4 * RT);
  const int m = tile % mp.row_blocks * (32 * RT) + (unit >> 2) * 32 + (unit & 3) * 8 + 4 * (lane >> 5);
  const int64_t n = (int64_t)(tile / mp.row_blocks) * (32 * CW) + cw * 32 + (lane & 31);
  if (n >= p.N || m >= p.M) return;
  const f4_t* src = mp.partial + (int64_t)tile * (256 * RT * CW) + quad;
  const float bias = p.bias ? widen16(p.bias[n], p.io_bf16) : 0.f;
  f4_t sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k = 0; k < splits; ++k) sum += src[(int64_t)k * tiles * (256 * RT * CW)];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (m + i < p.M) p.C[(int64_t)(m + i) * p.ldc + n] = narrow16(sum[i] + bias, p.io_bf16);
}

// One workgroup of 512 threads a tile, in one dimension of the grid, which ends below 2^32 threads.  (Products of more tiles of every
// size, 137 GB of output and more, stay with mnb_mid_kernel, whose rows and columns are dimensions of their own.)
constexpr int64_t kMidRowsMaxTiles = (int64_t)1 << 23;

// 32-row tiles and 32-column slabs of a workgroup, and (ANY) the cuts of K with the place of their sums
struct MidRowsLaunch {
  int rt, cw, splits;
  f4_t* partial;
};

template <int BITS, bool HAS_ZP, int RT, int CW, int IO, bool ANY>
hipError_t launch_rows_one(const SkinnyParams& params, const MidRowsLaunch& l, hipStream_t s) {
  MidRowsParams mp{};
  mp.s = params;
  mp.s.chunks = (params.K + kRowsChunk - 1) / kRowsChunk;
  mp.row_blocks = (params.M + 32 * RT - 1) / (32 * RT);
  mp.ragged = params.K % kRowsChunk != 0;
  mp.a_bytes = (uint32_t)(((int64_t)(params.M - 1) * params.lda + params.K) * 2);  // (below 4 GiB: mid_rows_plan)
  auto kernel = mnb_mid_shared_rows_kernel<BITS, HAS_ZP, RT, CW, IO, ANY>;
  // more than 64 KB of dynamic LDS has to be asked for, once per device (the attribute is kept per device)
  static std::atomic<unsigned long long> asked{0};
  int device = 0;
  if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return e;
  if (device >= 64 || !((asked.load(std::memory_order_relaxed) >> device) & 1ull)) {
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kMidRowsLds<RT>);
        e != hipSuccess)
      return e;
    if (device < 64) asked.fetch_or(1ull << device, std::memory_order_relaxed);
  }
  const int64_t grid = (int64_t)((params.N + 32 * CW - 1) / (32 * CW)) * mp.row_blocks;
  if (grid >= kMidRowsMaxTiles) return hipErrorInvalidValue;
  if constexpr (ANY) {
    if (l.splits > 1) {
      mp.split_chunks = ((mp.s.chunks + l.splits - 1) / l.splits + 1) / 2 * 2;
      mp.partial = l.partial;
      kernel<<<dim3((unsigned)grid, (unsigned)l.splits), dim3(512), kMidRowsLds<RT>, s>>>(mp);
      if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
      mnb_mid_rows_sum_kernel<RT, CW><<<dim3((unsigned)(grid * RT * CW)), dim3(256), 0, s>>>(mp, l.splits, (int)grid);
      return hipGetLastError();
    }
  }
  kernel<<<dim3((unsigned)grid), dim3(512), kMidRowsLds<RT>, s>>>(mp);
  return hipGetLastError();
}

template <int BITS, bool HAS_ZP, int CW, int IO, bool ANY>
hipError_t launch_rows_rt(const SkinnyParams& p, const MidRowsLaunch& l, hipStream_t s) {
  switch (l.rt) {
    case 1: return launch_rows_one<BITS, HAS_ZP, 1, CW, IO, ANY>(p, l, s);
    case 2: return launch_rows_one<BITS, HAS_ZP, 2, CW, IO, ANY>(p, l, s);
    case 3: return launch_rows_one<BITS, HAS_ZP, 3, CW, IO, ANY>(p, l, s);
    case 4: return launch_rows_one<BITS, HAS_ZP, 4, CW, IO, ANY>(p, l, s);
    default: return hipErrorInvalidValue;
  }
}

template <int BITS, bool HAS_ZP, int IO, bool ANY>
hipError_t launch_rows_cw(const SkinnyParams& p, const MidRowsLaunch& l, hipStream_t s) {
  return l.cw == 4 ? launch_rows_rt<BITS, HAS_ZP, 4, IO, ANY>(p, l, s) : launch_rows_rt<BITS, HAS_ZP, 2, IO, ANY>(p, l, s);
}

template <int BITS, bool HAS_ZP, bool ANY>
hipError_t launch_rows_io(const SkinnyParams& p, int io, const MidRowsLaunch& l, hipStream_t s) {
  if (io == kMnbIoBf16) return launch_rows_cw<BITS, HAS_ZP, kMnbIoBf16, ANY>(p, l, s);
  if (io == kMnbIoF16Wide) {  // zero points in the activation type: 4-bit with zero points
    if constexpr (BITS == 4 && HAS_ZP) return launch_rows_cw<BITS, HAS_ZP, kMnbIoF16Wide, ANY>(p, l, s);
    else return hipErrorInvalidValue;
  }
  return launch_rows_cw<BITS, HAS_ZP, kMnbIoModel, ANY>(p, l, s);
}

template <bool ANY>
hipError_t launch_rows(const SkinnyParams& p, int bits, bool has_zp, int io, const MidRowsLaunch& l, hipStream_t s) {
  if (bits == 4) return has_zp ? launch_rows_io<4, true, ANY>(p, io, l, s) : launch_rows_io<4, false, ANY>(p, io, l, s);
  return has_zp ? launch_rows_io<8, true, ANY>(p, io, l, s) : launch_rows_io<8, false, ANY>(p, io, l, s);
}

}  // namespace

// The form ANY, in a translation unit of its own (mnb_mid_any.hip); `params` and `launch` are a SkinnyParams and a MidRowsLaunch.
hipError_t mnb_mid_launch_any(const void* params, const void* launch, int bits, bool has_zp, int io, hipStream_t s);
