// Pieces shared by the GEMM kernels that keep several LDS stages in flight (kg_fp8_ring.hip, kg_bf16_batched.hip).
#pragma once
#include "kg_device.h"

#include <type_traits>
#include <utility>

// Waits until at most N of this wave's vector-memory operations and none of its LDS reads are in flight, then for
// the workgroup.
template <int N>
KG_DEV void kg_ring_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// One copy instruction: 16 bytes a lane from VGPR offset v (range-checked) + ko of resource r to 1 KB of LDS.
KG_DEV void kg_ring_copy(__amdgpu_buffer_rsrc_t r, u8* dst, unsigned v, int ko) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, v, ko, 0, 0);
}

// f(0), f(1), ... with the index a compile-time constant.
template <class F, int... T>
KG_DEV void kg_unroll(F f, std::integer_sequence<int, T...>) {
  (f(std::integral_constant<int, T>{}), ...);
}
