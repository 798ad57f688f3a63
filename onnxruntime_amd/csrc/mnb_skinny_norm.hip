// Decode of one row with its (Skip)SimplifiedLayerNormalization inside the projection: what MatMulNBitsMlp and
// MatMulNBitsQkv run for one token.
//
// The separate normalisation is one workgroup's work: 2.3 us of launch, load latency and reduction on a chip that waits,
// then the projection starts from nothing.  Here every workgroup of the decode kernel normalises the row for itself - a
// row is 2 K bytes, read from the level-2 cache - while the weights of its first chunks are on their way from memory:
// the row, skip and scale are requested first and the weights behind them, so the normalisation waits for its own loads
// only.  The normalised row is kept in LDS and the operands are picked up there (the sixteen rows of a matrix instruction
// all read the one row that exists).  Rounding is that of mnb_fused.hip: sums in fp32, the row narrowed to fp16 once.
// Bound like the decode kernel by the weights' bytes.  Measured, one row, all projections of a layer with K = 4096, 14336
// feed-forward columns: replayed as a graph with weights from HBM 41.8 -> 38.6 us (8-bit 58.0 -> 54.4); called eagerly, where
// the host's launches set the pace, 49.5 -> 45.2 us.  More rows keep the separate normalisation: every workgroup would
// repeat all of them.
#include "mnb_skinny_kernels.hip.h"

namespace {

struct RowNorm {
  const _Float16* skip;   // optional
  const _Float16* scale;
  _Float16* sum_out;      // optional: A + skip, written by the first workgroup
  float eps;
};

// K <= NW * 64 * 8 * VPT and a whole number of chunks; D = chunks of weights in flight per wavefront
template <int BITS, int MODE, int T, int NW, int VPT, int D>
__global__ void __launch_bounds__(NW * 64) mnb_skinny_norm_kernel(MNB_SKINNY_HOT_PARAMS, RowNorm nm, SkinnyParams rest) {
  const SkinnyParams p = with_hot_params(rest, MNB_SKINNY_HOT_NAMES);
  constexpr int GK = 128 / BITS, NI = GK / 8, THREADS = NW * 64;
  extern __shared__ __align__(16) unsigned char smem[];
  float* red = reinterpret_cast<float*>(smem);                           // [NW][T][4][64], also the sums of squares
  h8_t* row = reinterpret_cast<h8_t*>(red + NW * T * 4 * 64);            // the normalised row, K halves
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kq = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * (16 * T);
  const int64_t col0 = n0 + (lane & 15);

  // the row's loads: vectors beyond K re-read the last one and are left out of the sum
  const int vectors = p.chunks * (4 * GK / 8);
  h8_t av[VPT], gv[VPT], sv[VPT];
#pragma unroll
  for (int v = 0; v < VPT; ++v) {
    const int i = min(v * THREADS + (int)threadIdx.x, vectors - 1);
    av[v] = reinterpret_cast<const h8_t*>(p.A)[i];
    gv[v] = reinterpret_cast<const h8_t*>(nm.scale)[i];
  }
  if (nm.skip) {
#pragma unroll
    for (int v = 0; v < VPT; ++v)
      sv[v] = reinterpret_cast<const h8_t*>(nm.skip)[min(v * THREADS + (int)threadIdx.x, vectors - 1)];
  } else {
#pragma unroll
    for (int v = 0; v < VPT; ++v) sv[v] = h8_t{};
  }
  __builtin_amdgcn_sched_barrier(0);

  ChunkRegs<BITS, T> R[D];
  const int last = p.chunks - 1;
  const int own = wave < p.chunks ? (p.chunks - wave + NW - 1) / NW : 0;  // chunks of this wavefront
  auto load = [&](int c, ChunkRegs<BITS, T>& r) {
    __builtin_amdgcn_sched_barrier(0);
    load_chunk<BITS, false, MODE, T>(p, c, kq, col0, r);
    __builtin_amdgcn_sched_barrier(0);
  };
  // (no load sits under a condition, see skinny_chunks: clamped to the last chunk, which is valid and not used)
#pragma unroll
  for (int s = 0; s < D; ++s) load(min(wave + s * NW, last), R[s]);

  float x[VPT][8], ss = 0.f;
#pragma unroll
  for (int v = 0; v < VPT; ++v) {
    const int i = v * THREADS + (int)threadIdx.x;
    const bool exists = i < vectors;
    h8_t sum_h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float val = (float)av[v][e];
      if (nm.skip) val += (float)sv[v][e];
      x[v][e] = val;
      sum_h[e] = (_Float16)val;
      ss += exists ? val * val : 0.f;
    }
    if (nm.sum_out && blockIdx.x == 0 && exists) reinterpret_cast<h8_t*>(nm.sum_out)[i] = sum_h;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  // The barriers of the prologue order LDS accesses only: the weights stay in flight across them.
  auto lds_barrier = [] {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (lane == 0) red[wave] = ss;
  lds_barrier();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) total += red[w];
  const float denom = sqrtf(total / (float)p.K + nm.eps);
#pragma unroll
  for (int v = 0; v < VPT; ++v) {
    const int i = v * THREADS + (int)threadIdx.x;
    h8_t o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (_Float16)(x[v][e] / denom * (float)gv[v][e]);
    if (i < vectors) row[i] = o;
  }
  lds_barrier();  // (also: every wavefront has read the sums of squares before the reduction buffer is reused)

  f4_t y[T];
#pragma unroll
  for (int t = 0; t < T; ++t) y[t] = f4_t{0.f, 0.f, 0.f, 0.f};
  const BConst bconst = make_bconst<BITS, false>();
  const UnpackConsts uc = make_unpack_consts();
  const UnpackConsts2 uc2 = make_unpack_consts2();
  auto run = [&](int c, const ChunkRegs<BITS, T>& r) {
    h8_t af[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) af[i] = row[(c * 4 + kq) * NI + i];
    compute_chunk<BITS, false, MODE, T>(r, af, bconst, uc, uc2, y);
  };
  int q = 0, c = wave;
  for (; q + 2 * D - 1 < own; q += D, c += D * NW) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      run(c + s * NW, R[s]);
      load(c + (s + D) * NW, R[s]);
    }
  }
  const int left = own - q;  // 0 .. 2 D - 1: straight-line code for each, so that every wait counts its loads
#pragma unroll
  for (int n = 1; n < 2 * D; ++n) {
    if (left == n) {
#pragma unroll
      for (int s = 0; s < n; ++s) {
        run(c + s * NW, R[s % D]);
        if (s + D < n) load(c + (s + D) * NW, R[s % D]);
      }
    }
  }
#if defined(MNB_STAMPS)
  unsigned long long stamp[kStampPoints] = {};
#endif
  skinny_epilogue<T, NW>(p, red, y, wave, lane, n0 MNB_STAMP_ARG);
}

template <int BITS, int MODE, int T, int NW, int VPT, int D>
hipError_t launch_one(const SkinnyParams& p, const RowNorm& nm, hipStream_t s) {
  const dim3 grid((unsigned)((p.N + 16 * T - 1) / (16 * T)));
  const size_t smem = (size_t)NW * T * 4 * 64 * sizeof(float) + (size_t)p.K * 2;
  mnb_skinny_norm_kernel<BITS, MODE, T, NW, VPT, D><<<grid, dim3(NW * 64), smem, s>>>(MNB_SKINNY_HOT_ARGS(p), nm, p);
  return hipGetLastError();
}

template <int BITS, int MODE, int T, int NW, int D>
hipError_t launch_k(const SkinnyParams& p, const RowNorm& nm, hipStream_t s) {
  return p.K <= NW * 64 * 8 * (8 / NW) ? launch_one<BITS, MODE, T, NW, 8 / NW, D>(p, nm, s)
                                       : launch_one<BITS, MODE, T, NW, 16 / NW, D>(p, nm, s);
}

template <int BITS, int MODE>
hipError_t launch_t(const SkinnyParams& p, const RowNorm& nm, int t, hipStream_t s) {
  switch (t) {
    case 4: return launch_k<BITS, MODE, 4, 4, 2>(p, nm, s);
    case 2: return launch_k<BITS, MODE, 2, 8, 4>(p, nm, s);
    default: return launch_k<BITS, MODE, 1, 8, 4>(p, nm, s);
  }
}

}  // namespace

hipError_t mnb_skinny_launch_norm(const void* params, int bits, int mode, int t, const void* skip, const void* scale,
                                  void* sum_out, float eps, hipStream_t s) {
  const SkinnyParams& p = *static_cast<const SkinnyParams*>(params);
  const RowNorm nm{static_cast<const _Float16*>(skip), static_cast<const _Float16*>(scale),
                   static_cast<_Float16*>(sum_out), eps};
  if (bits == 4) return mode == 0 ? launch_t<4, 0>(p, nm, t, s) : launch_t<4, 1>(p, nm, t, s);
  return mode == 0 ? launch_t<8, 0>(p, nm, t, s) : launch_t<8, 1>(p, nm, t, s);
}
