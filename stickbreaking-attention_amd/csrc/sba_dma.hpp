// Loads from global memory straight into LDS, and reads of the layout they leave there: panels of [row][32 columns], 16-bit, 64-byte rows
// whose 16-byte chunks are XORed with (row >> 2) & 3, so that row reads and transposing reads meet no bank twice.
#pragma once
#include "sba_device.hpp"

namespace sba {

typedef __attribute__((address_space(3))) unsigned char lds_u8;

template <typename V>
__device__ __forceinline__ V lds_load(lds_u8* p) { return *reinterpret_cast<__attribute__((address_space(3))) V*>(p); }

__device__ __forceinline__ u32x4 buffer_desc(const void* base, int bytes) {
  const uint64_t a = (uint64_t)base;
  return u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, (uint32_t)bytes, 0x00020000u};
}
// The scalars of a vector-memory instruction must not have been written by a vector instruction (as a reloaded spill is) in the
// five wait states before it.  The compiler sees to that for its own instructions, not for those in inline assembly: each of
// these statements begins with its own five.
//
// 64 x 16 bytes from a buffer straight into LDS, lane i's to lds + 16 i; twice, kStep bytes apart there.
template <int kStep>
__device__ __forceinline__ void dma16x2(int lds, int voff, u32x4 desc, int soff0, int soff1) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\t"
               "s_mov_b32 m0, %5\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %4 offen lds"
               ::"s"(lds), "v"(voff), "s"(desc), "s"(soff0), "s"(soff1), "s"(lds + kStep) : "memory");
}
template <int kLeft>
__device__ __forceinline__ void vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLeft) : "memory"); }

template <typename T>
__device__ __forceinline__ typename Elem<T>::vec8 tr_pair(lds_u8* p0, lds_u8* p1) {
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p0);
  s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p1);
  s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(typename Elem<T>::vec8, v);
}

}  // namespace sba
