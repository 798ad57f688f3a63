// fp16 decode kernel for 1 <= M <= 16: which calls it serves, its plan and the dispatch to the translation unit that
// holds the kernels of the call's weight format.  The design is described at the top of mnb_skinny_kernels.hip.h.
#include "mnb_skinny_kernels.hip.h"

bool mnb_skinny_applicable(const MnbGemmArgs& a) {
  // fp16 models, and 16-bit ones (a.io) on a matrix packed with fp32 meta entries
  return (a.io != kMnbIoModel ? a.L.dtype == kMnbDtypeFloat : a.L.dtype == kMnbDtypeFloat16) && a.M >= 1 && a.M <= 16;
}

bool mnb_skinny_native2(const MnbGemmArgs& a) {
  const MnbLayout& L = a.L;
  return L.src_bits == 2 && L.w2_bytes > 0 && a.io == kMnbIoModel && a.M <= 16 &&
         (reinterpret_cast<uintptr_t>(a.A) % 16 == 0) && (a.lda % 8 == 0) && (L.K % 256 == 0);
}

namespace {

// operands, extents and outputs of a call; the chunks are those of the packed nibbles or bytes
SkinnyParams skinny_params(const MnbGemmArgs& a) {
  const MnbLayout& L = a.L;
  SkinnyParams p{};
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
  p.chunks = (int)((L.K + 4 * L.group_k - 1) / (4 * L.group_k));
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
  return p;
}

bool overlap(const void* a, size_t na, const void* b, size_t nb) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return x < y + nb && y < x + na;
}

// Tiles of a slab of the kernel that normalises the row itself (mnb_skinny_norm.hip: slabs of one, two and four tiles), or
// 0 where the separate normalisation and the decode kernel are the faster pair: the decode kernel has plans that the
// other lacks, and with little work behind it the prologue that every workgroup repeats is not hidden.  Measured as graphs
// with weights from HBM, K = 1024 ... 8192, the pair against the one kernel, us:
//   single-tile slabs                             7-32 % faster everywhere (N = 3072, K = 4096 6.9 -> 5.4)
//   two-tile slabs up to 512 tiles                0-27 % faster everywhere (N = 6144, K = 4096, blocks of 128 9.0 -> 6.8);
//     beyond (only the MLP's, the others have three tiles) 8-bit and exact 4-bit operands of more than 32 chunks 7-22 %
//     faster, raw 4-bit ones slower (N = 11008, K = 2048 7.4 -> 9.1, K = 8192 16.5 -> 18.9)
//   three-tile slabs, here of two tiles           8-bit 3-13 % faster; exact 4-bit operands equal or up to 14 % faster up to
//     32 chunks, slower from 48 on; raw 4-bit ones always slower (N = 9216, K = 4096 10.3 -> 11.3, K = 8192 14.1 -> 18.8)
//   one to 1.6 rounds of four-tile slabs, which the decode plan narrows to two tiles: 8-bit up to 64 chunks 2-10 % faster;
//     4-bit slower (N = 20480, K = 4096, blocks of 32 17.5 -> 20.1; K = 8192 27.4 -> 33.0)
//   one round of four-tile slabs or less          up to 16 chunks 0-14 % faster, else slower (N = 16384, K = 4096, blocks of
//     32 13.6 -> 15.2, K = 8192, blocks of 128 18.4 -> 20.4; 8-bit, K = 4096 17.4 -> 18.1)
//   more four-tile slabs                          0-18 % faster (N = 28672, K = 4096 17.0 -> 15.4); beyond two rounds with
//     up to 16 chunks slower (N = 57344, K = 2048 16.9 -> 17.8)
int norm_slab(const MnbLayout& L, int min_t) {
  const SkinnyPlan pl = skinny_plan(L, kMnbIoModel, 1, true, min_t);
  const int64_t tiles = (L.N + 15) / 16, slabs4 = (tiles + 3) / 4, cus = mnb_device_info().cus;
  const int chunks = (int)(L.K / (4 * L.group_k));
  const bool raw4 = L.bits == 4 && pl.mode == 0;
  if (pl.t == 1) return 1;
  if (pl.t == 2 && tiles < 800) return tiles <= 512 || L.bits == 8 || (!raw4 && chunks > 32) ? 2 : 0;
  if (pl.t == 3) return L.bits == 8 || (!raw4 && chunks <= 32) ? 2 : 0;
  if (pl.t == 2) return L.bits == 8 && chunks <= 64 ? 4 : 0;
  if (slabs4 <= cus) return chunks <= 16 ? 4 : 0;
  return slabs4 > 2 * cus && chunks <= 16 ? 0 : 4;
}

}  // namespace

bool mnb_skinny_norm_applicable(const MnbGemmArgs& a, const MnbNormPrologue& n) {
  const MnbLayout& L = a.L;
  auto al16 = [](const void* q) { return reinterpret_cast<uintptr_t>(q) % 16 == 0; };
  if (a.M != 1 || a.io != kMnbIoModel || L.dtype != kMnbDtypeFloat16 || L.has_zp || a.epi.kind == kMnbFusedNone) return false;
  if (L.K % (4 * L.group_k) != 0 || L.K > 8192 || !al16(a.A) || !al16(n.norm_scale_dev) || !al16(n.skip_dev) ||
      !al16(n.skip_sum_dev))
    return false;
  if (norm_slab(L, a.epi.kind == kMnbFusedMlp ? 2 : 1) == 0) return false;
  // Every workgroup reads the row while others may have stored their results already: no output may lie on the row,
  // its skip row or the scales (the separate normalisation has read them all before the projection starts).
  const size_t bytes = (size_t)L.K * 2;
  const void* outs[4] = {n.skip_sum_dev, a.epi.out[0], a.epi.out[1], a.epi.out[2]};
  const size_t sizes[4] = {bytes, (size_t)a.epi.n[0] * 2, (size_t)a.epi.n[1] * 2, (size_t)a.epi.n[2] * 2};
  for (int i = 0; i < 4; ++i)
    if (outs[i] != nullptr && (overlap(outs[i], sizes[i], a.A, bytes) || overlap(outs[i], sizes[i], n.norm_scale_dev, bytes) ||
                               (n.skip_dev != nullptr && overlap(outs[i], sizes[i], n.skip_dev, bytes))))
      return false;
  return true;
}

hipError_t mnb_launch_skinny_norm(const MnbGemmArgs& a, const MnbNormPrologue& n, hipStream_t s) {
  if (!mnb_skinny_norm_applicable(a, n)) return hipErrorInvalidValue;
  const SkinnyParams p = skinny_params(a);
  const int t = norm_slab(a.L, a.epi.kind == kMnbFusedMlp ? 2 : 1);  // (gate/up pairs live in one workgroup)
  return mnb_skinny_launch_norm(&p, a.L.bits, a.L.bs >= 4 * a.L.group_k ? 0 : 1, t, n.skip_dev, n.norm_scale_dev,
                                n.skip_sum_dev, n.epsilon, s);
}

hipError_t mnb_launch_skinny(const MnbGemmArgs& a, hipStream_t s) {
  const MnbLayout& L = a.L;
  if (!mnb_skinny_applicable(a) || (a.io != kMnbIoModel && a.epi.kind != kMnbFusedNone)) return hipErrorInvalidValue;
  const bool direct = L.K >= 4 * L.group_k;
  // 2-bit sources: the copy in their own width (half the bytes to stream) when the matrix has one and whole chunks
  // of 256 k can be read straight from aligned activations; else the nibble copy
  const bool native2 = mnb_skinny_native2(a);
  MnbLayout L2 = L;
  if (native2) {
    L2.bits = 2;
    L2.group_k = 64;
  }
  const bool words = reinterpret_cast<uintptr_t>(a.A) % 4 == 0 && (a.lda % 2 == 0 || a.M == 1);
  SkinnyPlan pl = skinny_plan(native2 ? L2 : L, a.io, a.M, direct, a.epi.kind == kMnbFusedMlp ? 2 : 1, words);
  SkinnyParams p = skinny_params(a);
  const int CK = 4 * (native2 ? L2.group_k : L.group_k);
  p.chunks = (int)(direct ? L.K / CK : 1);
  if (native2) p.W = reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(a.packed) + L.w2_off);
  p.phase_chunks = pl.phase_chunks;
  p.mtr = pl.mtr;
  p.whole_chunks = direct;
  if (native2) return mnb_skinny_launch_w2(&p, &pl, s);
  if (L.bits == 4) return L.has_zp ? mnb_skinny_launch_w4zp(&p, &pl, s) : mnb_skinny_launch_w4(&p, &pl, s);
  return mnb_skinny_launch_w8(&p, &pl, L.has_zp, s);
}
