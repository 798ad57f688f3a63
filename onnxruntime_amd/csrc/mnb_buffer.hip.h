// Buffer addressing, loads straight into LDS and hand-written wait counts: shared by the tile GEMMs.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint32_t u4_t __attribute__((ext_vector_type(4)));  // plain register quad (HIP's uint4 struct resists SROA)
typedef uint32_t u2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Buffer addressing: a 128-bit resource (uniform base, no range check: every offset is valid by construction) plus a
// 32-bit per-lane byte offset, so a load costs no 64-bit address arithmetic in the vector unit.  The host pass of the
// compiler knows these builtins but not the target features they need, and silently drops a whole kernel, launch
// stub included, that calls one: the calls are for the device pass only.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t rsrc_t;
__device__ __forceinline__ rsrc_t mnb_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00020000);
}
__device__ __forceinline__ u2_t mnb_buffer_load_b64(rsrc_t r, uint32_t off, uint32_t uniform_off = 0) {
  return __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, (int)uniform_off, 0);
}
__device__ __forceinline__ u4_t mnb_buffer_load_b128(rsrc_t r, uint32_t off, uint32_t uniform_off = 0) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, (int)uniform_off, 0);
}
__device__ __forceinline__ uint32_t mnb_buffer_load_b32(rsrc_t r, uint32_t off, uint32_t uniform_off = 0) {
  return __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, (int)uniform_off, 0);
}
// The same of a range that ends: what lies behind it reads as zeros, also into LDS.
__device__ __forceinline__ rsrc_t mnb_rsrc_bytes(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}
// Output rows of `pitch` elements of `size` bytes as a buffer that begins at row m0, column n0 and ends behind the last of m rows of n
// columns: stores beyond the end are dropped, so the rows of a last tile need no branch.  Offsets into it must stay below 4 GiB
// (mnb_rows_reach), and columns beyond n within a row are the caller's to leave out.
__device__ __forceinline__ rsrc_t mnb_rsrc_rows(void* base, int64_t pitch, int size, int64_t m0, int64_t n0, int64_t m, int64_t n) {
  const int64_t left = ((m - 1 - m0) * pitch + n - n0) * size;  // (a tile begins inside the matrix: positive)
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<uint8_t*>(base) + (m0 * pitch + n0) * size, 0,
                                           (int)(uint32_t)(left < 0xFFFFFFFF ? left : 0xFFFFFFFF), 0x00020000);
}
__device__ __forceinline__ void mnb_buffer_store_b32(rsrc_t r, uint32_t v, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b32(v, r, (int)off, 0, 0);
}
// 16 bytes per lane from the buffer straight into LDS: lane L's bytes land at `lds` (uniform) + 16 L.
__device__ __forceinline__ void mnb_buffer_load_lds_b128(rsrc_t r, uint32_t off, lds_ptr_t lds, uint32_t uniform_off = 0) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds, 16, (int)off, (int)uniform_off, 0, 0);
}
#else
struct rsrc_t {};
__host__ __device__ inline rsrc_t mnb_rsrc(const void*) { return {}; }
__host__ __device__ inline u2_t mnb_buffer_load_b64(rsrc_t, uint32_t, uint32_t = 0) { return u2_t{0, 0}; }
__host__ __device__ inline u4_t mnb_buffer_load_b128(rsrc_t, uint32_t, uint32_t = 0) { return u4_t{0, 0, 0, 0}; }
__host__ __device__ inline uint32_t mnb_buffer_load_b32(rsrc_t, uint32_t, uint32_t = 0) { return 0; }
__host__ __device__ inline void mnb_buffer_load_lds_b128(rsrc_t, uint32_t, lds_ptr_t, uint32_t = 0) {}
__host__ __device__ inline rsrc_t mnb_rsrc_bytes(const void*, uint32_t) { return {}; }
__host__ __device__ inline rsrc_t mnb_rsrc_rows(void*, int64_t, int, int64_t, int64_t, int64_t, int64_t) { return {}; }
__host__ __device__ inline void mnb_buffer_store_b32(rsrc_t, uint32_t, uint32_t) {}
#endif
// every element of `rows` rows lies below 4 GiB of the first one (each row being shorter than its pitch)
__host__ __device__ inline bool mnb_rows_reach(int64_t pitch, int size, int rows) { return (uint64_t)pitch * rows * size < (1ull << 32); }

// s_waitcnt immediate that waits until at most VM vector-memory operations are outstanding and every LDS operation
// of the wavefront has completed (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] << 14).
constexpr int waitcnt_vm_lds0(int vm) { return (vm & 15) | (7 << 4) | (0 << 8) | ((vm >> 4) << 14); }
// The same for vector-memory operations only (LDS and scalar-memory counters untouched).
constexpr int waitcnt_vm(int vm) { return (vm & 15) | (7 << 4) | (15 << 8) | ((vm >> 4) << 14); }

