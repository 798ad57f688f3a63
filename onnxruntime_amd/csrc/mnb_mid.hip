// fp16 kernel for 16 < M <= a few hundred rows: the regime between decode and prefill, where the reference runs its
// strip-wise dequantise + SGEMM loop (SQ4BitGemm_CompFp32, onnxruntime/core/mlas/lib/qnbitgemm.cpp:563-732) and the
// work is still dominated by streaming the weights once.
//
// Same structure as the decode kernel (mnb_skinny.hip): a workgroup owns 16*T output columns and a block of 16*MT rows,
// K is split over its wavefronts (reduced through LDS at the end, fixed order), and every lane feeds its own 16-byte
// weight vector to v_mfma_f32_16x16x32_f16 as the B operand -- no LDS on the weight path.  The difference is that each
// dequantised operand is used by MT row tiles, so the weights are dequantised exactly ((q - zp) * scale in fp16, the
// reference's fp16 dequantisation bit for bit) and the matrix cores accumulate across blocks; the VALU cost of the
// dequantisation is amortised over MT * 4 matrix instructions per word.
//
// 16-bit models on a matrix packed with fp32 meta entries (IO = kMnbIoBf16, kMnbIoF16Wide: bfloat16, and fp16 with zero
// points in the activation type) run the same kernel: the weights are dequantised in fp32, fma(float(q), scale,
// -zp * scale), narrowed to the activation type, and multiplied by the matrix instruction of that type.
//
// The A operand of lane (j, kq) is 16 bytes of row j at a 64-byte stride between lanes -- read from the row-major
// activations, one load instruction would touch 64 cache lines.  A small staging kernel therefore first rewrites A
// into operand order in the caller's workspace, [chunk][word i][row tile][kq][j] in 16-byte units (zero-filled beyond
// M and K, any alignment of the source), so that every operand load of a wavefront is 1 KiB contiguous.  The staged
// copy is M x K halves (at most a few MB) and is re-read from L2 by every workgroup.
#include <atomic>

#include "mnb_mfma16_common.hip.h"

namespace {

struct MidParams {
  SkinnyParams s;
  const uint4* As;  // staged activations
  int row_tiles;    // 16-row tiles in the staged copy (multiple of the kernel's MT)
};

// A (row-major, lda, any alignment) -> rows of `pieces` 16-byte pieces, zeros beyond K: what the kernel of mnb_mid_rows.hip.h
// reads where it cannot read A itself.  One thread per piece; bound by its launch (2 us), then by memory (1000 rows of 4088 3 us).
__global__ void __launch_bounds__(256) mnb_mid_pad_a_kernel(const _Float16* __restrict__ A, int64_t lda, int M, int K, int pieces,
                                                            u4_t* __restrict__ rows) {
  typedef uint32_t piece_t __attribute__((ext_vector_type(4), aligned(2)));
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= (int64_t)M * pieces) return;
  const int64_t row = u / pieces;
  const int k0 = (int)(u - row * pieces) * 8;
  const _Float16* const src = A + row * lda + k0;
  u4_t out = {0, 0, 0, 0};
  if (k0 + 8 <= K) {
    out = *reinterpret_cast<const piece_t*>(src);
  } else if (k0 < K) {
    _Float16 tmp[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) tmp[e] = k0 + e < K ? src[e] : (_Float16)0.0f;
    out = __builtin_bit_cast(u4_t, tmp);
  }
  rows[u] = out;
}

// A (row-major, lda) -> operand order.  One thread per 16-byte unit.
template <int BITS>
__global__ void __launch_bounds__(256) mnb_mid_stage_a_kernel(const _Float16* __restrict__ A, int64_t lda, int M, int K,
                                                              int chunks, int row_tiles, int vec_ok,
                                                              uint4* __restrict__ As) {
  constexpr int GK = 128 / BITS, NI = GK / 8, CK = 4 * GK;
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t total = (int64_t)chunks * NI * row_tiles * 64;
  if (u >= total) return;
  const int j = (int)(u & 15), kq = (int)((u >> 4) & 3);
  const int64_t v = u >> 6;
  const int rt = (int)(v % row_tiles);
  const int i = (int)((v / row_tiles) % NI);
  const int c = (int)(v / ((int64_t)row_tiles * NI));
  const int row = rt * 16 + j;
  const int k0 = c * CK + kq * GK + 8 * i;
  uint4 out = make_uint4(0u, 0u, 0u, 0u);
  if (row < M && k0 < K) {
    const _Float16* src = A + (int64_t)row * lda + k0;
    if (vec_ok && k0 + 8 <= K) {
      out = *reinterpret_cast<const uint4*>(src);
    } else {
      __align__(16) _Float16 tmp[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) tmp[e] = (k0 + e < K) ? src[e] : (_Float16)0.0f;
      out = *reinterpret_cast<const uint4*>(tmp);
    }
  }
  As[u] = out;
}

}  // namespace
#include "mnb_mid_rows.hip.h"
namespace {

// One chunk: word step i of every column tile against the MT row tiles, then -- the A operands of step i being dead --
// their reload for the wavefront's next chunk (a_next, when NEXT_A).  The activations are thus prefetched
// three quarters of a chunk ahead without a second register set.  NEXT_A is a compile-time flag on purpose: a load
// under a run-time condition makes the number of outstanding loads unknown to the compiler at the join, and every
// later wait then degenerates to "wait for all loads", the weight prefetch issued just before included.
template <int BITS, bool HAS_ZP, int T, int MT, bool NEXT_A, int IO>
__device__ __forceinline__ void mid_compute_chunk(const ChunkRegs<BITS, T>& R, h8_t (*af)[(128 / BITS) / 8],
                                                  const uint4* a_next, int64_t a_step, const UnpackConsts& uc,
                                                  f4_t (*y)[T]) {
  constexpr int NI = (128 / BITS) / 8;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const bool second = (BITS == 4) && i >= 2;  // words 2, 3 of a 4-bit vector may belong to the next block
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const uint32_t wd[4] = {R.w[t].x, R.w[t].y, R.w[t].z, R.w[t].w};
      h8_t b;
      if constexpr (IO != kMnbIoModel) {
        const float sc = __uint_as_float(second ? R.m1[t] : R.m0[t]);
        const float zp = HAS_ZP ? __uint_as_float(second ? R.z1[t] : R.z0[t]) : (float)(1 << (BITS - 1));
        b = BITS == 4 ? dequant_word_wide<BITS, IO == kMnbIoBf16>(wd[i], 0u, sc, -zp * sc)
                      : dequant_word_wide<BITS, IO == kMnbIoBf16>(wd[(2 * i) & 3], wd[(2 * i + 1) & 3], sc, -zp * sc);
      } else {
        _Float16 sc, nz;
        decode_meta<BITS, HAS_ZP>(second ? R.m1[t] : R.m0[t], sc, nz);
        const h2_t s2 = mnb_h2(sc);
        const h2_t z_lo = mnb_h2(nz);                     // -(1024 + zp)
        const h2_t z_hi = mnb_h2(nz + (_Float16)960.0f);  // -(64 + zp), exact
        b = BITS == 4 ? dequant_word<4>(wd[i], 0u, uc, z_lo, z_hi, s2)
                      : dequant_word<8>(wd[(2 * i) & 3], wd[(2 * i + 1) & 3], uc, z_lo, z_hi, s2);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        if constexpr (IO == kMnbIoBf16)
          y[mt][t] = mfma16_bf16(af[mt][i], b, y[mt][t]);
        else
          y[mt][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[mt][i], b, y[mt][t], 0, 0, 0);
      }
    }
    // Nothing moves across the end of a word step: loads hoisted above the matrix instructions that still read
    // af[.][i] would need a second register set, and so would dequantised operands prepared steps ahead.
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (NEXT_A) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) af[mt][i] = __builtin_bit_cast(h8_t, a_next[i * a_step + mt * 64]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// What a wavefront needs to issue its first loads comes as leading scalar kernel arguments, which the build asks the
// compiler to have preloaded into SGPRs at wavefront start; the parameter block carries the rest.
// DIRECT: the activations are read from the caller's row-major A (16-byte aligned rows, K a multiple of 8) and
// brought into operand order inside the kernel, so the staging pass and its launch drop out: a wavefront reads its
// chunk of a 16-row tile row-contiguously (64 lanes x 16 bytes = 4 rows x 256 bytes with 4-bit weights: 8 cache lines
// per instruction), passes it through a private 4 KiB of LDS and picks its operands up from there, tile after tile (LDS
// executes a wavefront's accesses in order: no barrier).  The loads of the next chunk are issued before the current one
// is computed and wait in registers (MT x NI vectors).  A ragged last chunk (K no multiple of 128 with 4-bit weights, 64
// with 8-bit) costs a clamped address and a uniform test per chunk, in a form of its own (DIRECT = 2: in the form for whole
// chunks they took up to 9 % of short products), and saves the staging launch that such a K used to need (K = 2880, 4-bit,
// blocks of 32, through the Python operator: N = 32, one row 12.1 -> 9.3 us; N = 5003, 37 rows 12.3 -> 11.0 us).
template <int BITS, bool HAS_ZP, int T, int MT, int NW, int IO, int DIRECT>
__global__ void __launch_bounds__(NW * 64) mnb_mid_kernel(const uint4* hot_W, int64_t hot_Npad, const uint4* hot_As,
                                                          const uint8_t* hot_meta, int hot_row_tiles, int hot_chunks,
                                                          int hot_bs_shift, MidParams rest) {
  MidParams mp = rest;
  mp.s.W = hot_W;
  mp.s.Npad = hot_Npad;
  mp.As = hot_As;
  mp.s.meta = hot_meta;
  mp.row_tiles = hot_row_tiles;
  mp.s.chunks = hot_chunks;
  mp.s.bs_shift = hot_bs_shift;
  const SkinnyParams& p = mp.s;
  constexpr int GK = 128 / BITS;
  constexpr int NI = GK / 8;
  constexpr int LOAD_MODE = IO == kMnbIoModel ? 1 : 2;  // which meta entries a chunk's loads fetch (load_chunk)
  extern __shared__ __align__(16) unsigned char smem[];
  float* red = reinterpret_cast<float*>(smem);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, kq = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * T);
  const int64_t col0 = n0 + j;
  const int m0 = blockIdx.y * (16 * MT);

  // staged A: unit index = (((c * NI + i) * row_tiles + rt) * 4 + kq) * 16 + j
  const uint4* a_lane = mp.As + ((int64_t)blockIdx.y * MT * 4 + kq) * 16 + j;
  const int64_t a_step = (int64_t)mp.row_tiles * 64;  // units between consecutive (c, i)
  f4_t y[MT][T];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t) y[mt][t] = f4_t{0.f, 0.f, 0.f, 0.f};
  const UnpackConsts uc = make_unpack_consts();

  h8_t af[MT][NI];
  auto load_a = [&](int c) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < NI; ++i)
        af[mt][i] = __builtin_bit_cast(h8_t, a_lane[((int64_t)c * NI + i) * a_step + mt * 64]);
  };
  // DIRECT: 16-byte pieces of a chunk's row: PIECES; rows one load instruction covers: RPI (16 / RPI == NI instructions
  // per 16-row tile).  Pieces are XOR-swizzled with the row so that neither the row-contiguous writes nor the operand
  // reads conflict on LDS banks.
  constexpr int PIECES = 4 * NI, RPI = 64 / PIECES;
  const int piece = lane % PIECES, r0 = lane / PIECES;
  auto swz = [](int row) { return PIECES == 16 ? row : (row >> 1); };
  h8_t* const mine = reinterpret_cast<h8_t*>(smem + (size_t)NW * T * 4 * 64 * sizeof(float)) + wave * (16 * PIECES);
  h8_t g[MT][NI];  // the next chunk's activations on their way (DIRECT)
  auto fetch_a = [&](int c) {
    // ragged: pieces beyond K (K is a multiple of 8) re-read the row's last one and are cleared before they are used
    const int64_t k = DIRECT == 2 ? min(c * 4 * GK + piece * 8, p.K - 8) : (int64_t)c * 4 * GK + piece * 8;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int I = 0; I < NI; ++I) {
        int row = m0 + mt * 16 + I * RPI + r0;
        row = row < p.M ? row : p.M - 1;  // rows beyond M re-read the last row and are never stored
        g[mt][I] = *reinterpret_cast<const h8_t*>(p.A + (int64_t)row * p.lda + k);
      }
  };
  auto pass_a = [&](int c) {
    if (DIRECT == 2 && (c + 1) * 4 * GK > p.K) {  // wave-uniform: the ragged last chunk
      const bool exists = c * 4 * GK + piece * 8 < p.K;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int I = 0; I < NI; ++I) g[mt][I] = exists ? g[mt][I] : h8_t{};
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int I = 0; I < NI; ++I) {
        const int row = I * RPI + r0;
        mine[row * PIECES + (piece ^ swz(row))] = g[mt][I];
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) af[mt][i] = mine[j * PIECES + ((kq * NI + i) ^ swz(j))];
    }
  };

  // Weights two chunks ahead (double buffer), activations reloaded word step by word step inside the chunk.  No load
  // of the loop sits under a condition, so every wait counts exactly the loads it needs and leaves the younger
  // prefetches in flight; a prefetch beyond the wavefront's last chunk is clamped to the last chunk of the matrix
  // instead of skipped (valid memory that another wavefront of the workgroup is reading anyway, never used here).
  auto a_of = [&](int c) -> const uint4* { return a_lane + (int64_t)c * NI * a_step; };
  ChunkRegs<BITS, T> R0, R1;
  const int last = p.chunks - 1;
  int c = wave;
  if constexpr (DIRECT != 0) {
    // weights two chunks ahead, activations one: fetched into g before a chunk is computed, passed through LDS after
    load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c, last), kq, col0, R0);
    fetch_a(min(c, last));
    load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c + NW, last), kq, col0, R1);
    pass_a(min(c, last));
    __builtin_amdgcn_sched_barrier(0);
    for (; c + NW < p.chunks; c += 2 * NW) {
      fetch_a(c + NW);
      __builtin_amdgcn_sched_barrier(0);
      mid_compute_chunk<BITS, HAS_ZP, T, MT, false, IO>(R0, af, nullptr, a_step, uc, y);
      load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c + 2 * NW, last), kq, col0, R0);
      __builtin_amdgcn_sched_barrier(0);
      pass_a(c + NW);
      fetch_a(min(c + 2 * NW, last));
      __builtin_amdgcn_sched_barrier(0);
      mid_compute_chunk<BITS, HAS_ZP, T, MT, false, IO>(R1, af, nullptr, a_step, uc, y);
      load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c + 3 * NW, last), kq, col0, R1);
      __builtin_amdgcn_sched_barrier(0);
      pass_a(min(c + 2 * NW, last));
    }
    if (c < p.chunks) mid_compute_chunk<BITS, HAS_ZP, T, MT, false, IO>(R0, af, nullptr, a_step, uc, y);
  } else {
    load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c, last), kq, col0, R0);
    load_a(min(c, last));
    load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c + NW, last), kq, col0, R1);
    __builtin_amdgcn_sched_barrier(0);
    for (; c + NW < p.chunks; c += 2 * NW) {
      mid_compute_chunk<BITS, HAS_ZP, T, MT, true, IO>(R0, af, a_of(c + NW), a_step, uc, y);
      load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c + 2 * NW, last), kq, col0, R0);
      __builtin_amdgcn_sched_barrier(0);
      mid_compute_chunk<BITS, HAS_ZP, T, MT, true, IO>(R1, af, a_of(min(c + 2 * NW, last)), a_step, uc, y);
      load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(c + 3 * NW, last), kq, col0, R1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (c < p.chunks) mid_compute_chunk<BITS, HAS_ZP, T, MT, false, IO>(R0, af, nullptr, a_step, uc, y);
  }

  // reduce over the wavefronts, one row tile at a time: lane (j, kq), register r of y[mt][t] holds
  // row m0 + 16 mt + 4 kq + r, column n0 + 16 t + j
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (mt > 0) __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[(wave * T * 4 + t * 4 + r) * 64 + lane] = y[mt][t][r];
    __syncthreads();
    reduce_and_store_tiles<T, NW>(p, red, m0 + mt * 16, n0);
  }
}

// ---- activations shared through LDS ---------------------------------------------------------------------------------
// The kernel above re-reads the activations once per 16 T columns: every workgroup walks all of K, and its wavefronts,
// which split K between them, share nothing.  For wide matrices that stream is several times the weights' (64 rows,
// K = 4096, N = 28672, 64 columns per workgroup: 448 x 512 KB = 229 MB against 59 MB of weights) and it is the level-2
// caches, busy 70 % of the launch, that set the pace.  Here a workgroup's eight wavefronts form KGS = 4 teams of NG = 2:
// the teams split K as before, the two wavefronts of a team own neighbouring slabs of 16 T columns and walk the same
// chunks, and the chunk's activations (16 MT rows x 256 bytes) are fetched ONCE per team, from the caller's row-major A
// straight into LDS (buffer_load ... lds, 16-byte pieces XOR-swizzled with the row so that neither the row-contiguous
// fills nor the operand reads conflict on banks), one round ahead of the arithmetic, into one of two buffers.  Per
// round: wait for the own fills of this round, barrier, start the fills of the next round, pick the operands up from
// LDS, compute, reload the weight registers for the round after next.  No staged copy of A, no staging launch.
// Needs K a whole number of chunks and 16-byte aligned rows of A; everything else takes the kernel above.
// Anatomy of a round (64 rows, N = 28672, K = 4096, 4-bit, time stamps of the shader clock in a calibration build):
// the older wavefront of a SIMD needs 2800 cycles for its arithmetic (64 matrix instructions, 1024 cycles of the matrix
// pipe, and 320 vector instructions, 1280 issue cycles), the younger one, which gets the issue slots the older
// leaves, 4250; then both wait about 1300 cycles for the fills they issued when the round began: 24 of 1 KB a wavefront
// at once, which the address unit takes at 64 bytes a cycle, and a round trip.  (A read probe gets 110 to 120 GB/s a compute
// unit, 28 to 31 TB/s over the chip, out of the level-2 caches into LDS: their bandwidth is not what these rounds wait for.)  A
// third buffer (fills two rounds ahead) does not fit the 160 KB of LDS.  Ablations: without the arithmetic the launch takes
// 16.0 us, without fills, operand reads and arithmetic 10.9 us (the weights alone), all together 29.7 us.
// The kernel of mnb_mid_rows.hip.h, smaller chunks in four stages and larger matrix instructions, takes 4-bit weights over; this
// one keeps 8-bit weights of K > 2048, whose stream is what both wait for, and blocks of 16 (see mid_rows_plan).
// Tried on top and not kept: dequantising the next operand between the matrix instructions of the current one (a
// software pipeline inside mid_compute_chunk, also with the order forced by scheduling groups) -- bit-identical
// results and the same times (+-1 %) on eight shapes of both kernels; cutting K into parts across workgroups for
// matrices too narrow to fill the chip (fp32 partial tiles, an arrival counter per tile, the last workgroup to arrive
// adds the parts in part order) -- correct, and slower than the kernel above on every narrow shape (N = 4096,
// K = 14336, 64 rows: 27.5 against 19.7 us; K = 4096: 18.6 against 7.9 us), because a round costs 2.0 to 2.3 us
// whatever the grid (the same with 32 workgroups as with 224) on top of about 8 us per launch.
template <int BITS, bool HAS_ZP, int T, int MT, int KGS, int NG, int IO>
__global__ void __launch_bounds__(KGS * NG * 64) mnb_mid_shared_kernel(const uint4* hot_W, int64_t hot_Npad,
                                                                        const _Float16* hot_A, const uint8_t* hot_meta,
                                                                        int64_t hot_lda, int hot_chunks,
                                                                        int hot_bs_shift, MidParams rest) {
  MidParams mp = rest;
  mp.s.W = hot_W;
  mp.s.Npad = hot_Npad;
  mp.s.A = hot_A;
  mp.s.meta = hot_meta;
  mp.s.lda = hot_lda;
  mp.s.chunks = hot_chunks;
  mp.s.bs_shift = hot_bs_shift;
  const SkinnyParams& p = mp.s;
  constexpr int GK = 128 / BITS, NI = GK / 8, CK = 4 * GK;
  constexpr int PIECES = 4 * NI;                   // 16-byte pieces per row of a chunk
  constexpr int ROWS = 16 * MT;                    // rows of A a workgroup works on
  constexpr int CHUNK_BYTES = ROWS * PIECES * 16;  // one team's activations of one chunk
  constexpr int RPI = 64 / PIECES;                 // rows one fill instruction covers
  constexpr int A_PER_WAVE = ROWS / RPI / NG;      // fill instructions per wavefront and round
  constexpr int LOAD_MODE = IO == kMnbIoModel ? 1 : 2;  // which meta entries a chunk's loads fetch (load_chunk)
  // vector-memory instructions of load_chunk: T of weights and, per half vector (4-bit) or vector, the T entries of meta
  // data in one (4 bytes or fewer each) or two (fp32 scale and zero point)
  static_assert(T == 4, "the count of loads below");
  constexpr int W_LOADS = T + (BITS == 4 ? 2 : 1) * (IO != kMnbIoModel && HAS_ZP ? 2 : 1);
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / NG, ng = wave % NG;
  const int j = lane & 15, kq = lane >> 4;
  const int64_t n0 = ((int64_t)blockIdx.x * NG + ng) * (16 * T);
  const int64_t col0 = n0 + j;
  const int m0 = blockIdx.y * ROWS;
  auto swz = [](int row) { return PIECES == 16 ? (row & 15) : ((row >> 1) & 7); };

  // this wavefront's share of a round's fills: instruction q covers rows q * RPI + lane / PIECES
  uint32_t a_off[A_PER_WAVE];
#pragma unroll
  for (int u = 0; u < A_PER_WAVE; ++u) {
    const int row = (ng * A_PER_WAVE + u) * RPI + lane / PIECES;
    const int piece = (lane % PIECES) ^ swz(row);
    const int grow = m0 + row < p.M ? m0 + row : p.M - 1;  // rows beyond M re-read the last row and are never stored
    a_off[u] = (uint32_t)(((int64_t)grow * p.lda + piece * 8) * 2);
  }
  unsigned char* const team = smem + kg * CHUNK_BYTES;  // buffer b of the team: team + b * KGS * CHUNK_BYTES
  auto fill = [&](int c, int b) {
    const rsrc_t r = mnb_rsrc(p.A + (int64_t)c * CK);
#pragma unroll
    for (int u = 0; u < A_PER_WAVE; ++u)
      mnb_buffer_load_lds_b128(r, a_off[u],
                               (lds_ptr_t)(team + b * (KGS * CHUNK_BYTES) + (ng * A_PER_WAVE + u) * RPI * PIECES * 16));
  };
  f4_t y[MT][T];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t) y[mt][t] = f4_t{0.f, 0.f, 0.f, 0.f};
  const UnpackConsts uc = make_unpack_consts();
  h8_t af[MT][NI];
  auto pick = [&](int b) {
    const unsigned char* buf = team + b * (KGS * CHUNK_BYTES);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int row = mt * 16 + j;
        af[mt][i] = *reinterpret_cast<const h8_t*>(buf + (row * PIECES + ((kq * NI + i) ^ swz(row))) * 16);
      }
  };

  const int last = p.chunks - 1;
  const int rounds = (p.chunks + KGS - 1) / KGS;
  auto chunk_of = [&](int r) { return r * KGS + kg; };
  ChunkRegs<BITS, T> R0, R1;
  // One round.  On entry the fills of round r (issued a round earlier) are followed in issue order by exactly one
  // set of weight loads, so "at most W_LOADS outstanding" means they have landed; the barrier makes that true of the
  // team-mate's share, and tells everybody that the other buffer's readers are done with it.
  auto round = [&](int r, ChunkRegs<BITS, T>& R, int b) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(W_LOADS));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    fill(min(chunk_of(r + 1), last), b ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    pick(b);
    if (chunk_of(r) < p.chunks) mid_compute_chunk<BITS, HAS_ZP, T, MT, false, IO>(R, af, nullptr, 0, uc, y);
    __builtin_amdgcn_sched_barrier(0);
    load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(chunk_of(r + 2), last), kq, col0, R);
    __builtin_amdgcn_sched_barrier(0);
  };
  load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(chunk_of(0), last), kq, col0, R0);
  __builtin_amdgcn_sched_barrier(0);
  fill(min(chunk_of(0), last), 0);
  __builtin_amdgcn_sched_barrier(0);
  load_chunk<BITS, HAS_ZP, LOAD_MODE, T>(p, min(chunk_of(1), last), kq, col0, R1);
  for (int r = 0; r < rounds; r += 2) {
    round(r, R0, 0);
    round(r + 1, R1, 1);  // (past the end: loads of valid memory, a barrier everybody reaches, no arithmetic)
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lds0(0));  // the last prefetches write LDS the reduction is about to reuse
  __syncthreads();

  // Sums of the teams in team order, all row tiles at once; the KGS wavefronts of a slab share out its quads of rows: two column
  // tiles (a pair of gate and up) and every other row tile each.  (One row tile after the other, two barriers each and values of two
  // bytes stored one by one between branches: 64 rows of 28672 x 4096 in 8-bit weights 30.5 us; so 28.4, with twice the LDS.)
  constexpr bool bf16 = IO == kMnbIoBf16;
  constexpr int COLS = NG * 16 * T, PAIRS = T / 2, SHARE = KGS / PAIRS;  // wavefronts of a pair
  static_assert(KGS % PAIRS == 0 && MT % SHARE == 0, "row tiles shared out evenly");
  const int pair = kg / SHARE, mt0 = kg % SHARE;
  const int64_t block0 = (int64_t)blockIdx.x * COLS;
  float bias[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t n = n0 + (2 * pair + h) * 16 + j;
    bias[h] = p.bias && n < p.N ? widen16(p.bias[n], bf16) : 0.f;  // (arrives during the sums)
  }
  f4_t* const red = reinterpret_cast<f4_t*>(smem) + ng * (MT * T * KGS * 64);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < T; ++t) red[((mt * T + t) * KGS + kg) * 64 + lane] = y[mt][t];
  __syncthreads();
  constexpr int UNITS = MT / SHARE;
  f4_t sum[UNITS][2];
#pragma unroll
  for (int u = 0; u < UNITS; ++u)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sum[u][h] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KGS; ++k) sum[u][h] += red[(((mt0 + SHARE * u) * T + 2 * pair + h) * KGS + k) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[u][h][i] += bias[h];
    }
  __syncthreads();
  const int thread = wave * 64 + lane;
  if (p.epi.kind == kMnbFusedMlp) {
    store_rows<ROWS, COLS / 2>(p, reinterpret_cast<_Float16*>(smem), thread, m0, block0 / 2, [&](_Float16* out, int pitch) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = sum[u][0][i], up = sum[u][1][i];
          out[((mt0 + SHARE * u) * 16 + 4 * kq + i) * pitch + (ng * PAIRS + pair) * 16 + j] = narrow16(g / (1.0f + __expf(-g)) * up, bf16);
        }
    });
  } else {
    store_rows<ROWS, COLS>(p, reinterpret_cast<_Float16*>(smem), thread, m0, block0, [&](_Float16* out, int pitch) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < UNITS; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            out[((mt0 + SHARE * u) * 16 + 4 * kq + i) * pitch + ng * 16 * T + (2 * pair + h) * 16 + j] = narrow16(sum[u][h][i], bf16);
    });
  }
}

struct MidPlan {
  int t, mt, nw;
};

MidPlan mid_plan(const MnbLayout& L, int64_t M, int min_t = 1) {
  MidPlan pl;
  const int CK = 4 * L.group_k;
  const int chunks = (int)((L.K + CK - 1) / CK);
  const int64_t tiles = (L.N + 15) / 16;
  // A workgroup's tile of 16 T columns x 16 MT rows decides how often a dequantised weight (MT) and a loaded
  // activation operand (T) are reused; the grid has to give every CU a workgroup first.  Among the shapes that
  // reach 192 workgroups the largest tile wins, at equal area the wider one (measured: the activations are the
  // larger stream); if none does, the shape with the most workgroups.
  int64_t best_wgs = -1;
  int best_area = 0;
  pl.t = min_t;
  pl.mt = 2;
  for (int t = 4; t >= min_t; t >>= 1) {
    for (int mt = M <= 32 ? 2 : 4; mt >= 2; mt >>= 1) {
      const int64_t wgs = ((tiles + t - 1) / t) * ((M + 16 * mt - 1) / (16 * mt));
      const int area = t * mt;
      const bool full = wgs >= 192, best_full = best_wgs >= 192;
      const bool better = best_wgs < 0 || (full && !best_full) || (full && best_full && area > best_area) ||
                          (!full && !best_full && (wgs > best_wgs || (wgs == best_wgs && area > best_area)));
      if (better) {
        best_wgs = wgs;
        best_area = area;
        pl.t = t;
        pl.mt = mt;
      }
    }
  }
  // eight wavefronts split K further and hide more latency in a single round of workgroups; with several rounds of
  // the largest tile, two workgroups of four wavefronts share a CU instead
  pl.nw = chunks < 16 || (best_area == 16 && best_wgs >= 384) ? 4 : 8;
  if (const char* e = mnb_tuning_env("MNB_MID_PLAN")) {  // calibration builds: "<T>,<MT>,<NW>"
    int t = 0, mt = 0, nw = 0;
    if (sscanf(e, "%d,%d,%d", &t, &mt, &nw) == 3 && (t == 1 || t == 2 || t == 4) && (mt == 2 || mt == 4) &&
        (nw == 4 || nw == 8)) {
      pl.t = t;
      pl.mt = mt;
      pl.nw = nw;
    }
  }
  if (pl.t < min_t) pl.t = min_t;  // gate/up pairs live in one workgroup
  return pl;
}

// whether the direct form of an instantiation exists: the widest tiles have no registers left for the activations in
// flight
template <int BITS, int T, int MT>
constexpr bool kMidHasDirect = !(MT == 4 && T == 4);

// direct: 0 from the staged copy, 1 in place, 2 in place with a ragged last chunk
template <int BITS, bool HAS_ZP, int T, int MT, int IO>
hipError_t launch_nw(const MidParams& mp, const MidPlan& pl, int direct, hipStream_t s) {
  const SkinnyParams& p = mp.s;
  dim3 grid((unsigned)((p.N + 16 * T - 1) / (16 * T)), (unsigned)((p.M + 16 * MT - 1) / (16 * MT)));
  // the sums of the wavefronts, and with activations in place 16 rows of one chunk for each
  const size_t smem = (size_t)pl.nw * T * 4 * 64 * sizeof(float) + (direct ? (size_t)pl.nw * 16 * (128 / BITS / 2) * 16 : 0);
  auto launch = [&](auto kernel) {
    kernel<<<grid, dim3(64 * pl.nw), smem, s>>>(p.W, p.Npad, mp.As, p.meta, mp.row_tiles, p.chunks, p.bs_shift, mp);
    return hipGetLastError();
  };
  if constexpr (kMidHasDirect<BITS, T, MT>) {
    if (direct == 1)
      return pl.nw == 8 ? launch(mnb_mid_kernel<BITS, HAS_ZP, T, MT, 8, IO, 1>) : launch(mnb_mid_kernel<BITS, HAS_ZP, T, MT, 4, IO, 1>);
    if (direct == 2)
      return pl.nw == 8 ? launch(mnb_mid_kernel<BITS, HAS_ZP, T, MT, 8, IO, 2>) : launch(mnb_mid_kernel<BITS, HAS_ZP, T, MT, 4, IO, 2>);
  }
  return pl.nw == 8 ? launch(mnb_mid_kernel<BITS, HAS_ZP, T, MT, 8, IO, 0>) : launch(mnb_mid_kernel<BITS, HAS_ZP, T, MT, 4, IO, 0>);
}

template <int BITS, bool HAS_ZP, int T, int IO>
hipError_t launch_mt(const MidParams& p, const MidPlan& pl, int direct, hipStream_t s) {
  return pl.mt == 2 ? launch_nw<BITS, HAS_ZP, T, 2, IO>(p, pl, direct, s) : launch_nw<BITS, HAS_ZP, T, 4, IO>(p, pl, direct, s);
}

template <int BITS, bool HAS_ZP, int IO>
hipError_t launch_t(const MidParams& p, const MidPlan& pl, int direct, hipStream_t s) {
  switch (pl.t) {
    case 4: return launch_mt<BITS, HAS_ZP, 4, IO>(p, pl, direct, s);
    case 2: return launch_mt<BITS, HAS_ZP, 2, IO>(p, pl, direct, s);
    default: return launch_mt<BITS, HAS_ZP, 1, IO>(p, pl, direct, s);
  }
}

template <int BITS, bool HAS_ZP>
hipError_t launch_io(const MidParams& p, const MidPlan& pl, int io, int direct, hipStream_t s) {
  if (io == kMnbIoBf16) return launch_t<BITS, HAS_ZP, kMnbIoBf16>(p, pl, direct, s);
  if (io == kMnbIoF16Wide) {  // zero points in the activation type: 4-bit with zero points
    if constexpr (BITS == 4 && HAS_ZP) return launch_t<BITS, HAS_ZP, kMnbIoF16Wide>(p, pl, direct, s);
    else return hipErrorInvalidValue;
  }
  return launch_t<BITS, HAS_ZP, kMnbIoModel>(p, pl, direct, s);
}

int mid_row_tiles(int64_t M, int mt) { return (int)((M + 16 * mt - 1) / (16 * mt)) * mt; }

// ---- the kernel with activations shared through LDS: when it applies, and its launch
constexpr int kSharedT = 4, kSharedKgs = 4, kSharedNg = 2;  // 128 columns per workgroup, eight wavefronts

bool mid_shared_fills(const MnbLayout& L, int64_t M, int64_t cus) {
  const int64_t slabs = (L.N + 16 * kSharedT * kSharedNg - 1) / (16 * kSharedT * kSharedNg);
  const int rows = M <= 32 ? 32 : 64;
  const int64_t wgs = slabs * ((M + rows - 1) / rows);
  return wgs * 8 >= cus * 5 && wgs <= cus && L.K / (4 * L.group_k) >= 2 * kSharedKgs;
}

bool mid_shared_applies(const MnbGemmArgs& a) {
  const MnbLayout& L = a.L;
  if (!mnb_mid_applicable(a) || a.M <= 16) return false;
  const int CK = 4 * L.group_k;
  const bool vec_ok = (reinterpret_cast<uintptr_t>(a.A) % 16 == 0) && (a.lda % 8 == 0);
  // the fills address A with 32-bit byte offsets from the chunk's first column
  const bool reach = (uint64_t)a.M * (uint64_t)a.lda * 2 + 512 < ((uint64_t)1 << 32);
  if (!vec_ok || !reach || L.K % CK != 0) return false;
  bool use;
  if (const char* e = mnb_tuning_env("MNB_MID_SHARED")) {
    use = e[0] != '0';
  } else {
    // Asked after mid_rows_plan, so of 8-bit weights and blocks of 16 (the 4-bit figures are against the kernel above alone).
    // A workgroup here needs the same time whatever the grid (eight rounds of 2 - 3 us at K = 4096), so the kernel pays
    // where its 128-column slabs make one well-filled round of workgroups -- which is also where the activations'
    // stream through the level-2 caches is largest.  Measured against the kernel above (K = 4096, 4-bit):
    // N = 28672: M = 17 21.9 -> 17.7 us, M = 32 22.8 -> 17.6, M = 64 28.5 -> 25.5; N = 14336, M = 128 28.1 -> 24.8;
    // N = 11008, M = 128 30.2 -> 25.2; N = 6144, M = 256 27.4 -> 24.0; with fewer workgroups than 5/8 of the compute
    // units, or more than all of them, it loses (N = 14336, M = 64: 16.9 -> 24.0; N = 28672, M = 256: 82 -> 100).
    // bfloat16 (fp32 scales, weights narrowed one by one: bound by the vector instructions) by the same rule, 4-bit:
    // N = 28672: M = 17 25.1 -> 21.1 us, M = 32 25.8 -> 21.3, M = 64 29.0 -> 28.3; N = 11008, M = 128 31.0 -> 27.8;
    // N = 6144, M = 256 27.8 -> 26.8; 8-bit: N = 28672, M = 64 41.0 -> 31.1; N = 6144, M = 256 28.3 -> 25.4.
    use = mid_shared_fills(L, a.M, mnb_device_info().cus);
  }
  return use;
}

template <int BITS, bool HAS_ZP, int MT, int IO>
hipError_t launch_shared_mt(const MidParams& mp, hipStream_t s) {
  const SkinnyParams& p = mp.s;
  constexpr int T = kSharedT, KGS = kSharedKgs, NG = kSharedNg, NW = KGS * NG;
  constexpr size_t chunk_bytes = (size_t)16 * MT * (128 / BITS / 2) * 16;
  constexpr size_t fills = 2 * KGS * chunk_bytes, red = (size_t)NW * T * MT * 4 * 64 * sizeof(float);
  constexpr size_t smem = fills > red ? fills : red;
  auto kernel = mnb_mid_shared_kernel<BITS, HAS_ZP, T, MT, KGS, NG, IO>;
  // more than 64 KB of dynamic LDS has to be asked for, once per device (the attribute is kept per device)
  static std::atomic<unsigned long long> asked{0};
  int device = 0;
  if (hipError_t e = hipGetDevice(&device); e != hipSuccess) return e;
  if (device >= 64 || !((asked.load(std::memory_order_relaxed) >> device) & 1ull)) {
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        e != hipSuccess)
      return e;
    if (device < 64) asked.fetch_or(1ull << device, std::memory_order_relaxed);
  }
  const dim3 grid((unsigned)((p.N + 16 * T * NG - 1) / (16 * T * NG)), (unsigned)((p.M + 16 * MT - 1) / (16 * MT)));
  kernel<<<grid, dim3(NW * 64), smem, s>>>(p.W, p.Npad, p.A, p.meta, p.lda, p.chunks, p.bs_shift, mp);
  return hipGetLastError();
}

template <int BITS, bool HAS_ZP, int IO>
hipError_t launch_shared_rows(const MidParams& mp, hipStream_t s) {
  return mp.s.M <= 32 ? launch_shared_mt<BITS, HAS_ZP, 2, IO>(mp, s) : launch_shared_mt<BITS, HAS_ZP, 4, IO>(mp, s);
}

template <int BITS, bool HAS_ZP>
hipError_t launch_shared(const MidParams& mp, int io, hipStream_t s) {
  if (io == kMnbIoBf16) return launch_shared_rows<BITS, HAS_ZP, kMnbIoBf16>(mp, s);
  if (io == kMnbIoF16Wide) {  // zero points in the activation type: 4-bit with zero points
    if constexpr (BITS == 4 && HAS_ZP) return launch_shared_rows<BITS, HAS_ZP, kMnbIoF16Wide>(mp, s);
    else return hipErrorInvalidValue;
  }
  return launch_shared_rows<BITS, HAS_ZP, kMnbIoModel>(mp, s);
}

// ---- the kernel of mnb_mid_rows.hip.h: when it applies, its tile, and its launch
// Time of a launch (us) with tiles of 32 rt rows and 32 cw columns: `start`, then turns of as many workgroups as the compute
// units hold (mid_rows_per_cu), each of K / 128 steps of
//     step * (1 + load * share of the units at work) + more * (workgroups a unit - 1)
// and `turn` in front of every further one.  Fitted to 594 problems of 17 to 1400 rows, 200 to 28672 columns, K to 14336 on each
// of the eight tiles (8-bit, 32 x 128: 178 problems of 17 to 2200 rows; mean error 3 to 7 %, also on 600 others up to 2200 rows); the tile that the estimate picks is 0.3 % behind the best one on the average, 16 % at
// most.
struct MidRowsTime {
  double start, step, load, more, turn;
};
constexpr MidRowsTime kMidRowsTime[4][2][4] = {
    {{{3.39, 0.200, 0.27, 0.210, 2.2}, {4.03, 0.224, 0.40, 0.332, 2.6}, {4.73, 0.264, 0.57, 0.000, 3.2}, {5.40, 0.339, 0.57, 0.000, 3.9}},
     {{3.90, 0.312, 0.23, 0.359, 3.6}, {5.00, 0.347, 0.44, 0.557, 3.7}, {5.97, 0.408, 0.67, 0.000, 5.1}, {7.02, 0.535, 0.68, 0.000, 6.0}}},  // 4-bit, fp16 entries
    {{{3.36, 0.259, 0.20, 0.238, 1.8}, {4.01, 0.284, 0.28, 0.313, 2.5}, {4.75, 0.326, 0.34, 0.000, 3.0}, {5.35, 0.365, 0.43, 0.000, 3.9}},
     {{3.80, 0.436, 0.15, 0.415, 2.9}, {4.81, 0.473, 0.24, 0.533, 3.8}, {5.82, 0.541, 0.34, 0.000, 4.7}, {6.84, 0.600, 0.43, 0.000, 6.0}}},  // 4-bit, fp32 entries
    {{{3.74, 0.204, 0.36, 0.266, 2.5}, {4.32, 0.251, 0.45, 0.401, 2.0}, {5.01, 0.311, 0.53, 0.000, 3.3}, {5.60, 0.368, 0.59, 0.000, 4.4}},
     {{4.26, 0.364, 0.17, 0.460, 2.4}, {5.58, 0.406, 0.41, 0.662, 3.2}, {6.48, 0.461, 0.67, 0.000, 6.0}, {7.36, 0.561, 0.74, 0.000, 6.0}}},  // 8-bit, fp16 entries
    {{{3.82, 0.215, 0.45, 0.273, 1.1}, {4.35, 0.247, 0.59, 0.374, 1.8}, {5.04, 0.326, 0.44, 0.000, 3.1}, {5.54, 0.387, 0.53, 0.000, 3.8}},
     {{4.10, 0.422, 0.36, 0.395, 2.3}, {5.55, 0.461, 0.32, 0.643, 3.0}, {6.45, 0.523, 0.43, 0.000, 5.0}, {7.49, 0.604, 0.53, 0.000, 6.0}}},  // 8-bit, fp32 entries
};

int64_t mid_rows_tiles(const MnbLayout& L, int64_t M, int rt, int cw) {
  return ((L.N + 32 * cw - 1) / (32 * cw)) * ((M + 32 * rt - 1) / (32 * rt));
}
// Workgroups of eight wavefronts that a compute unit holds: by LDS (32 KB a row tile), 8-bit weights in 128-column slabs with one row
// tile by their 86 to 94 registers, five wavefronts a SIMD.
int mid_rows_per_cu(int bits, int rt, int cw) { return rt == 1 ? (bits == 8 && cw == 4 ? 2 : 4) : rt == 2 ? 2 : 1; }

// Chunks of each of `splits` cuts of K: an even number, so that blocks of 256 begin with a cut.
int64_t mid_rows_split_chunks(const MnbLayout& L, int splits) {
  const int64_t steps = (L.K + kRowsChunk - 1) / kRowsChunk;
  return ((steps + splits - 1) / splits + 1) / 2 * 2;
}

double mid_rows_us(const MnbLayout& L, int64_t M, int rt, int cw, int64_t cus, int splits = 1) {
  const bool wide = L.dtype == kMnbDtypeFloat;
  const MidRowsTime& t = kMidRowsTime[(L.bits == 8 ? 2 : 0) + (wide ? 1 : 0)][cw == 4][rt - 1];
  const int64_t steps = splits > 1 ? mid_rows_split_chunks(L, splits) : (L.K + kRowsChunk - 1) / kRowsChunk;
  const int64_t most = mid_rows_per_cu(L.bits, rt, cw);
  int64_t left = mid_rows_tiles(L, M, rt, cw) * splits;
  double us = t.start;
  auto turn = [&](int64_t per_cu, double share) {
    return (double)steps * (t.step * (1.0 + t.load * share) + t.more * (double)(per_cu - 1));
  };
  if (const int64_t full = (left - 1) / (most * cus); full > 0) {
    us += (double)full * (turn(most, 1.0) + t.turn);
    left -= full * most * cus;
  }
  const int64_t per_cu = (left + cus - 1) / cus;
  us += turn(per_cu, (double)left / (double)(per_cu * cus));
  // Activations beyond the level-2 caches: an XCD's workgroups, cus / 8 units of them, are row blocks of one slab side by side, and
  // only where they are several slabs' is a row block read once for these.  Each such pass goes through the fabric, at 6.5 TB/s
  // (150 timings, mean error 21 -> 10 %: 2030 rows of 495 x 9216 26.6 estimated without, 43.9 measured).
  if (const double mb = (double)M * (double)L.K * 2e-6; mb > 8) {
    const double shared = (double)(cus / 8 * most) / (double)((M + 32 * rt - 1) / (32 * rt));
    const double fabric = t.start + mb * (double)((L.N + 32 * cw - 1) / (32 * cw)) / (shared > 1 ? shared : 1.0) / 6.5;
    if (fabric > us) us = fabric;
  }
  // the second launch, which reads what the first one has written
  if (splits > 1) us += 2.5 + (double)(mid_rows_tiles(L, M, rt, cw) * splits * rt * cw) * 4096.0 * 2.0 / 4.0e6;
  return us;
}

// The same for mnb_mid_kernel with the plan's tile (16 t columns, 16 mt rows, nw wavefronts that share out the chunks), within
// 10 % on the average (432 problems, weights from HBM): start + rounds * round * (1 + up * load + over * what is beyond one), load
// in workgroups of eight wavefronts a compute unit; 8-bit rounds (half as many k) 0.57 of it.
double mid_us(const MnbLayout& L, int64_t M, const MidPlan& pl, int64_t cus) {
  struct Time {
    double start, round, up, over, wide;
  };
  const Time t = pl.t == 1 ? Time{2.59, 0.698, 0.84, 3.54, 1.04} : pl.t == 2 ? Time{3.75, 0.276, 4.39, 9.0, 1.25} :
                 pl.mt == 2 ? Time{4.54, 0.585, 2.70, 9.0, 1.12} : Time{9.31, 0.426, 6.0, 8.98, 1.20};
  const int64_t chunks = (L.K + 4 * L.group_k - 1) / (4 * L.group_k), rounds = (chunks + pl.nw - 1) / pl.nw;
  const int64_t wgs = (((L.N + 15) / 16 + pl.t - 1) / pl.t) * ((M + 16 * pl.mt - 1) / (16 * pl.mt));
  const double load = (double)(wgs * pl.nw) / (8.0 * (double)cus);
  const double waits = 1.0 + t.up * (load < 1 ? load : 1.0) + t.over * (load < 1 ? 0.0 : load - 1.0);
  return t.start + (double)rounds * t.round * waits * (L.bits == 8 ? 0.57 : 1.0) * (L.dtype == kMnbDtypeFloat ? t.wide : 1.0);
}

size_t mid_operand_bytes(const MnbLayout& L, int64_t M) {
  const int CK = 4 * L.group_k;
  const int64_t chunks = (L.K + CK - 1) / CK;
  return (size_t)chunks * (L.group_k / 8) * mid_row_tiles(M, 4) * 64 * 16;  // the larger of the two row blockings
}

struct MidRowsPlan {
  int rt, cw;  // 32-row tiles and 32-column slabs of a workgroup; rt = 0: not this kernel
  double us;   // estimate
  bool padded = false;  // reads a padded copy of A
  int splits = 1;       // cuts of K
};

size_t mid_rows_split_bytes(const MnbLayout& L, int64_t M, int rt, int cw, int splits) {
  return (size_t)mid_rows_tiles(L, M, rt, cw) * splits * rt * cw * 4096;
}

// K a multiple of 8, blocks of 32 and more (a lane holds one entry for its weights), rows that 16-byte loads can read.
// (A ragged last chunk costs nothing: it goes first, from an address past the buffer's end where it has no values.  By the kernels
// before, with their rows in place or a copy / so, called eagerly: 37 rows of 5003 x 2880 11.1 / 8.1 us, 124 rows of 7572 x 5344 18.2 / 15.8; mnb_mid_any.hip.)
// Measured, the kernels before / this one, us, weights from HBM (4-bit unless said, K = 4096): 128 rows of 11008 columns 30.7 / 21.3,
// 256 rows of 6144 27.2 / 21.1, 64 rows of 28672 29.3 / 25.1; 415 rows of 3147 x 3584 in bfloat16 31.3 / 17.1.  Long K goes the other way
// in both directions: few columns are cut finer by mnb_mid_kernel, whose tiles of 16 columns are four times as many (85 rows of
// 2706 x 9344 17.5 / 20.9; 29 rows of 298 x 8576 10.3 / 17.4), hence the estimate of that one; and 8-bit weights of K > 2048 in slabs that
// fill the units once stream no better here than through mnb_mid_shared_kernel (64 rows of 28672 31.8 / 34.9, 256 rows of 6144
// 24.7 / 25.3, 17 rows of 28672 in bfloat16 25.1 / 25.2; out of the Infinity Cache 28.6 / 27.4 and 23.7 / 21.6; but 64 rows of 20000 x 2048 25.9 / 17.6, 100 rows of 14000 x 1024 13.2 / 11.8).
// Those slabs are not cut into 64 columns by up to 64 rows either: with several such workgroups a unit and K of 512 to 1024 their
// estimate is 10 to 25 % short.  Measured on 110 problems where it would have them, their time / that of the tile taken instead is
// 1.05 on the average, 0.89 to 1.30 (681 rows of 2113 x 512 9.8 / 7.6, 46 rows of 21411 x 768 10.3 / 9.3, 58 rows of 28085 x 512 9.1 / 10.3).
//
// Rows of A that it cannot read (K no multiple of 8, an odd pitch or address) are copied first, padded with zeros to whole chunks, into the
// scratch that such calls bring for the copy in operand order: a launch and a pass, so only where the kernel gains them
// back.  Measured, the kernels before / copy and this one, us, 4-bit: 2048 rows of 14336 x 4088 320 / 267, in bfloat16 1055 rows of
// 22849 x 2508 210 / 169, 1366 rows of 2378 x 4056 54 / 40, 138 rows of 12513 x 272 14.9 / 8.9 (all but the second read in place by now);
// small products the other way (45 rows of 534 x 5411 10.6 / 14.5).
MidRowsPlan mid_rows_plan(const MnbGemmArgs& a, bool in_place_only = false) {
  const MnbLayout& L = a.L;
  MidRowsPlan best{0, 0, 0.0};
  if (!mnb_mid_applicable(a) || a.M <= 16 || L.bs < 32) return best;
  const bool vec_ok = (reinterpret_cast<uintptr_t>(a.A) % 16 == 0) && (a.lda % 8 == 0);
  const bool padded = !vec_ok || L.K % 8 != 0;  // (these calls bring scratch)
  if (padded && in_place_only) return best;
  const int64_t K = (L.K + kRowsChunk - 1) / kRowsChunk * kRowsChunk, lda = padded ? K : a.lda;
  // 32-bit byte offsets of activations, weights and entries
  constexpr uint64_t kReach = (uint64_t)1 << 32;
  const bool reach = (uint64_t)a.M * (uint64_t)lda * 2 < kReach && (uint64_t)L.w_bytes < kReach &&
                     (uint64_t)L.KBp * (uint64_t)L.Npad * L.meta_bytes < kReach;
  if (!reach || (padded && (size_t)a.M * K * 2 > mid_operand_bytes(L, a.M))) return best;
  // (a cut needs scratch for its sums; fused outputs are made of whole ones)
  bool split_ok = !padded && !a.uncut && a.epi.kind == kMnbFusedNone && reinterpret_cast<uintptr_t>(a.workspace) % 16 == 0;
  if (const char* e = mnb_tuning_env("MNB_MID_ROWS")) {  // calibration: "<rt>,<cw>"; "0,0" switches the kernel off
    const int n = sscanf(e, "%d,%d,%d", &best.rt, &best.cw, &best.splits);  // (and "<cuts of K>", where they fit)
    if (n < 2) best.rt = 0;
    best.padded = padded;
    const int64_t per = mid_rows_split_chunks(L, best.splits > 0 ? best.splits : 1);
    best.splits = (int)((K / kRowsChunk + per - 1) / per);
    if (n < 3 || best.rt == 0 || !split_ok || mid_rows_split_bytes(L, a.M, best.rt, best.cw, best.splits) > a.workspace_bytes) best.splits = 1;
    return best;
  }
  const int64_t cus = mnb_device_info().cus;
  // (never more than such calls ask for, so that more scratch is no other plan)
  const size_t room = a.workspace_bytes < mid_operand_bytes(L, a.M) ? a.workspace_bytes : mid_operand_bytes(L, a.M);
  const bool wide_slabs = !padded && L.K % (4 * L.group_k) == 0 && mid_shared_fills(L, a.M, cus);
  if (wide_slabs && L.bits == 8 && L.K > 2048) return best;
  const int most = a.M > 96 ? 4 : (int)((a.M + 31) / 32);
  for (int rt = 1; rt <= most; ++rt)
    for (int cw = 2; cw <= 4; cw += 2) {
      if (wide_slabs && rt <= 2 && cw == 2) continue;
      if (mid_rows_tiles(L, a.M, rt, cw) >= kMidRowsMaxTiles) continue;
      const double us = mid_rows_us(L, a.M, rt, cw, cus);
      if (best.rt == 0 || us < best.us) best = MidRowsPlan{rt, cw, us, padded};
      // Narrow matrices of long K leave units idle, or give each a long way through K: cut K, and sum the cuts in a launch of their
      // own, where the scratch that the call brings holds the sums.  Uncut (or on the other kernels) / so, us, called eagerly: 168 rows of
      // 745 x 7680 17.2 / 10.6, 48 rows of 512 x 14336 15.5 / 8.9, 401 rows of 989 x 7592 in bfloat16 19.7 / 16.4, 32 rows of 1024 x 8192 in 8
      // bits 10.1 / 8.6, 17 rows of 4096 x 14336 15.0 / 14.2.  The estimate has to promise a tenth: close ones go either way (256 rows
      // of 2048 x 8192 18.5 uncut, 17.0 with two cuts of 64 x 64 tiles).
      for (int splits = 2; split_ok && splits <= 8; ++splits) {
        const int64_t per = mid_rows_split_chunks(L, splits);
        if (per < 4 || per * (splits - 1) >= K / kRowsChunk) break;
        if (mid_rows_split_bytes(L, a.M, rt, cw, splits) > room) break;
        const double cut = mid_rows_us(L, a.M, rt, cw, cus, splits);
        if (cut >= 0.9 * best.us) continue;
        if (mnb_prefer_gemm256(L, a.M)) { split_ok = false; break; }  // (sizes of the tile GEMM ask for no scratch)
        best = MidRowsPlan{rt, cw, cut, padded, splits};
      }
    }
  if (padded) best.us += 2.5 + (double)a.M * (double)K * 1.3e-6;
  // (a cut is two launches for the host: 29 rows of 298 x 8576 9.8 us so, 9.5 uncut, called eagerly.  That is the close call: of 40 products
  // between 0.85 and 0.93 39 are faster cut as graphs, 27 % on the average, and 37 called eagerly, 18 %: 57 rows of 142 x 9832 in 8 bits 16.3 /
  // 9.0 and 15.6 / 9.9; the others are up to 10 % slower, 482 rows of 483 x 8576 14.8 / 16.2.)
  if (!wide_slabs && best.us >= (best.splits > 1 ? 0.85 : padded ? 0.9 : 0.93) * mid_us(L, a.M, mid_plan(L, a.M, a.epi.kind == kMnbFusedMlp ? 2 : 1), cus))
    best.rt = 0;
  return best;
}

}  // namespace

bool mnb_mid_applicable(const MnbGemmArgs& a) {
  // fp16 models, and 16-bit ones (a.io) on a matrix packed with fp32 meta entries
  return (a.io != kMnbIoModel ? a.L.dtype == kMnbDtypeFloat : a.L.dtype == kMnbDtypeFloat16) && a.M >= 1;
}

// bytes of the staged copy of A
size_t mnb_mid_workspace_bytes(const MnbLayout& L, int64_t M) { return mid_operand_bytes(L, M); }

const char* mnb_mid_kernel_name(const MnbGemmArgs& a) {
  if (mid_rows_plan(a).rt > 0) return "mnb_mid_shared_rows_kernel";
  return mid_shared_applies(a) ? "mnb_mid_shared_kernel" : "mnb_mid_kernel";
}

// Estimate (seconds) of the streaming kernel's many-row form where it would run this call; negative where it would not.
double mnb_mid_rows_seconds(const MnbGemmArgs& a) {
  const MidRowsPlan rows = mid_rows_plan(a, true);
  return rows.rt > 0 ? rows.us * 1e-6 : -1.0;
}

// Activations straight from A when its rows allow 16-byte loads and K is a multiple of 8 (the kernel then reorders them
// itself, and no workspace is touched); otherwise, and for the widest tiles, a staging pass writes them in operand
// order first.
//
// A ragged K saves that pass and its launch, 1.5-2.5 us of a product, 10-38 % of the small ones, more where the host's
// launches set the pace (37 rows of 5003 x 2880, called eagerly: 12.3 -> 11.1 us).  Where the workgroups are more than the
// compute units and the product is long some of that goes the other way, for the activations in flight leave room for one
// workgroup of eight wavefronts a unit where the staged form has two (4-bit, 130 registers and more against 80 to 134), and
// rows whose pitch is no multiple of 128 bytes cost a cache line more with every piece of a chunk.  So these keep the staged
// copy, staged -> in place measured (us, fp16, weights from HBM, launches in a graph, 600 ragged shapes):
//   4-bit, two-tile slabs of 32 rows, more than 24 chunks, tiles of up to 128 rows that are three quarters full
//                                        -8 to +10 (48 rows, K = 3640 +10; 128 rows of 2498 x 6920 21.9 -> 23.2); the
//                                        emptier ones, whose missing rows re-read one line, -18 to +3
//   4-bit, four-tile slabs, more than 90 chunks   -5 to +8 (97 rows of 5988 x 13960 49.7 -> 53.0)
//   8-bit, slabs of one and two tiles, more than 96 chunks, up to 32 rows more than 64   -13 to +18 (31 rows of 4778 x 7400
//                                        26.2 -> 30.9; 32 rows of 11309 x 5816 28.2 -> 31.9; 59 rows of 2633 x 11976 30.8
//                                        -> 35.0; 98 rows of 2834 x 13232 41.5 -> 45.8)
//   8-bit, four-tile slabs               -10 to +8, on the average -1 % (232 rows of 2678 x 4040 22.3 -> 24.1)
// The other forms gain on the average: 4-bit single tiles 8 %, 8-bit slabs below 96 chunks 15 %, 4-bit four-tile slabs 3 %,
// tiles of 64 rows 6-10 %, workgroups of four wavefronts 10-24 %.
static bool ragged_in_place_pays(const MnbLayout& L, int64_t M, const MidPlan& pl) {
  const int64_t chunks = (L.K + 4 * L.group_k - 1) / (4 * L.group_k), row_tiles = (M + 16 * pl.mt - 1) / (16 * pl.mt);
  const int64_t wgs = (((L.N + 15) / 16 + pl.t - 1) / pl.t) * row_tiles;
  if (wgs <= mnb_device_info().cus || pl.mt != 2 || pl.nw != 8) return true;
  if (L.bits == 8) return pl.t != 4 && chunks <= (M <= 32 ? 64 : 96);
  if (pl.t == 2) return chunks <= 24 || M > 128 || 4 * M < 3 * 32 * row_tiles;
  return pl.t == 1 || chunks <= 90;
}

static bool mid_direct(const MnbGemmArgs& a, const MidPlan& pl) {
  const bool vec_ok = (reinterpret_cast<uintptr_t>(a.A) % 16 == 0) && (a.lda % 8 == 0);
  bool direct = vec_ok && a.L.K % 8 == 0 && !(pl.mt == 4 && pl.t == 4) &&
                (a.L.K % (4 * a.L.group_k) == 0 || ragged_in_place_pays(a.L, a.M, pl));
  if (const char* e = mnb_tuning_env("MNB_MID_DIRECT")) direct = direct && e[0] != '0';  // calibration
  return direct;
}

bool mnb_mid_direct(const MnbGemmArgs& a) {
  // (the kernels that share activations read A in place as well)
  const bool whole = a.L.K % kRowsChunk == 0;  // (a ragged K brings scratch unless mnb_mid_kernel reads it in place, whichever kernel runs)
  return mid_direct(a, mid_plan(a.L, a.M, a.epi.kind == kMnbFusedMlp ? 2 : 1)) || (whole && mid_rows_plan(a, true).rt > 0) ||
         mid_shared_applies(a);
}

hipError_t mnb_launch_mid(const MnbGemmArgs& a, hipStream_t s) {
  const MnbLayout& L = a.L;
  if (!mnb_mid_applicable(a) || (a.io != kMnbIoModel && a.epi.kind != kMnbFusedNone)) return hipErrorInvalidValue;
  const MidPlan pl = mid_plan(L, a.M, a.epi.kind == kMnbFusedMlp ? 2 : 1);
  const int CK = 4 * L.group_k;
  MidParams mp{};
  SkinnyParams& p = mp.s;
  p.A = reinterpret_cast<const _Float16*>(a.A);
  p.W = reinterpret_cast<const uint4*>(a.packed);
  p.meta = reinterpret_cast<const uint8_t*>(a.packed) + L.meta_off;
  p.bias = reinterpret_cast<const _Float16*>(a.bias);
  p.C = reinterpret_cast<_Float16*>(a.C);
  p.lda = a.lda;
  p.ldc = a.ldc;
  p.Npad = L.Npad;
  p.M = (int)a.M;
  p.N = (int)L.N;
  p.K = (int)L.K;
  p.bs_shift = mnb_log2i(L.bs);
  p.chunks = (int)((L.K + CK - 1) / CK);
  p.io_bf16 = a.io == kMnbIoBf16;
  p.epi.kind = a.epi.kind;
  if (a.epi.kind != kMnbFusedNone) {
    p.C = reinterpret_cast<_Float16*>(a.epi.out[0]);
    p.ldc = a.epi.ld[0];
    p.epi.start1 = (int)a.epi.start[1];
    p.epi.start2 = (int)a.epi.start[2];
    p.epi.n0 = (int)a.epi.n[0];
    p.epi.n1 = (int)a.epi.n[1];
    p.epi.n2 = (int)a.epi.n[2];
    p.epi.out1 = reinterpret_cast<_Float16*>(a.epi.out[1]);
    p.epi.out2 = reinterpret_cast<_Float16*>(a.epi.out[2]);
    p.epi.ld1 = a.epi.ld[1];
    p.epi.ld2 = a.epi.ld[2];
  }
  if (const MidRowsPlan rows = mid_rows_plan(a); rows.rt > 0) {
    if (rows.padded) {
      if (a.workspace == nullptr || a.workspace_bytes < mnb_mid_workspace_bytes(L, a.M)) return hipErrorInvalidValue;
      const int pieces = (p.K + kRowsChunk - 1) / kRowsChunk * (kRowsChunk / 8);
      const int64_t units = (int64_t)p.M * pieces;
      mnb_mid_pad_a_kernel<<<dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s>>>(p.A, p.lda, p.M, p.K, pieces,
                                                                                       reinterpret_cast<u4_t*>(a.workspace));
      if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
      p.A = reinterpret_cast<const _Float16*>(a.workspace);
      p.lda = p.K = pieces * 8;
    }
    const MidRowsLaunch l{rows.rt, rows.cw, rows.splits, reinterpret_cast<f4_t*>(a.workspace)};  // (no cuts where A is padded there)
    if (p.K % kRowsChunk != 0 || rows.splits > 1) return mnb_mid_launch_any(&p, &l, L.bits, L.has_zp, a.io, s);
    return launch_rows<false>(p, L.bits, L.has_zp, a.io, l, s);
  }
  if (mid_shared_applies(a)) {
    if (L.bits == 4) return L.has_zp ? launch_shared<4, true>(mp, a.io, s) : launch_shared<4, false>(mp, a.io, s);
    return L.has_zp ? launch_shared<8, true>(mp, a.io, s) : launch_shared<8, false>(mp, a.io, s);
  }
  mp.As = reinterpret_cast<const uint4*>(a.workspace);
  mp.row_tiles = mid_row_tiles(a.M, pl.mt);
  const int vec_ok = (reinterpret_cast<uintptr_t>(a.A) % 16 == 0) && (a.lda % 8 == 0);
  const int direct = !mid_direct(a, pl) ? 0 : L.K % (4 * L.group_k) == 0 ? 1 : 2;
  if (!direct) {
    if (a.workspace == nullptr || a.workspace_bytes < mnb_mid_workspace_bytes(L, a.M)) return hipErrorInvalidValue;
    const int64_t units = (int64_t)p.chunks * (L.group_k / 8) * mp.row_tiles * 64;
    const dim3 sgrid((unsigned)((units + 255) / 256));
    uint4* staged = reinterpret_cast<uint4*>(a.workspace);
    if (L.bits == 4)
      mnb_mid_stage_a_kernel<4><<<sgrid, dim3(256), 0, s>>>(p.A, p.lda, p.M, p.K, p.chunks, mp.row_tiles, vec_ok, staged);
    else
      mnb_mid_stage_a_kernel<8><<<sgrid, dim3(256), 0, s>>>(p.A, p.lda, p.M, p.K, p.chunks, mp.row_tiles, vec_ok, staged);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  }
  if (L.bits == 4)
    return L.has_zp ? launch_io<4, true>(mp, pl, a.io, direct, s) : launch_io<4, false>(mp, pl, a.io, direct, s);
  return L.has_zp ? launch_io<8, true>(mp, pl, a.io, direct, s) : launch_io<8, false>(mp, pl, a.io, direct, s);
}
