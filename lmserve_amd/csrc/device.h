// Device-side helpers shared by the HIP sources of libkvcache.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace kvc {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Store policies: the cache bits of the instruction. What a kernel leaves dirty in the L2s of the 8 XCDs is written
// back when it ends; a store at device scope is written through to the last-level cache, where a reader on any
// XCD finds it. The non-temporal forms are for more rows than the caches would hold for their next reader.
enum StorePolicy : int { kPlain = 0, kNonTemporal = 2, kThrough = 16, kThroughNt = 16 | 2 };

// A run of bytes that one workgroup writes, `base` and `bytes` uniform over it. A store at or past `bytes` is dropped by
// the hardware's own range check, so a lane past the end needs no branch. Through the compiler's buffer store and not in
// inline asm: an instruction that overwrites the data of a 16-byte store too soon behind it corrupts the store, and
// only for stores it knows does the compiler keep the two apart.
struct OutRow {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ OutRow(char* base, uint32_t bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(base, 0, (int)bytes, 0x00020000)) {}
  template <StorePolicy POLICY>
  __device__ __forceinline__ void store(uint32_t offset, u32x4 v) const {
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, offset, 0, POLICY);
  }
};

// The same for addresses that differ from lane to lane by more than an offset: 16 bytes, kThrough and kThroughNt. The two wait
// states behind the store keep a later instruction off its data registers.
__device__ __forceinline__ void st_through(char* p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}
__device__ __forceinline__ void st_through_nt(char* p, u32x4 v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1 nt\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

// A kernel launch whose arguments go straight to the runtime. The launch by <<<>>> and its macro first store the
// configuration for a host stub that fetches it again, 0.1 to 0.15 us of the 2.3 a launch costs, and a launch per layer at
// decode sizes is bound by that. Errors are in hipGetLastError, as with the macro.
template <typename T>
struct Same {
  using type = T;
};
template <typename... P>
inline void launch(void (*kernel)(P...), dim3 grid, dim3 block, size_t lds, hipStream_t stream,
                   const typename Same<P>::type&... args) {
  void* pointers[] = {const_cast<void*>(static_cast<const void*>(&args))..., nullptr};
  (void)hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, pointers, lds, stream);
}

}  // namespace kvc
