// Loads from memory straight into LDS.
#pragma once
#include "common.cuh"

namespace dinfer {
namespace {

// 16 bytes a lane from `at` to LDS, lane after lane from byte `lds` on. (Not the builtin: behind it the compiler waits for all loads
// on their way before every read of LDS.)
__device__ __forceinline__ void load_to_lds(uint32_t lds, const char* at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(at) : "m0");
}

}  // namespace
}  // namespace dinfer
