// Shared by the bf16 products that bring their operands through a ring of LDS stages: loads straight from global memory into
// LDS, 64 columns of 8 rows an instruction, and the waits that go with them (see gemm_tile.hip for the layout).
#pragma once
#include "dispatch.h"

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx4_t __attribute__((ext_vector_type(4)));

union TFrag {
    uint4 u;
    bf16x8_t v;
};

#define GT_KC 64                    // columns of a chunk: 128 bytes a row
#define GT_WAIT_VMCNT(N) __builtin_amdgcn_s_waitcnt(0x0f70 | ((N) & 15) | (((N) >> 4) << 14))
#define GT_XCDS 8

// 16 bytes per lane from global memory straight into LDS: lane l's bytes land at lds_base + 16 l.
// Written as assembly so that the compiler neither counts nor guards it: the waits are the
// explicit ones below (the vector memory counter retires in order).
__device__ __forceinline__ void gt_load_to_lds(const void* src, __attribute__((address_space(3))) void* lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(src), "s"(lds_base)
                 : "memory", "m0");
}

// The same from a scalar base and 32 bits a lane.
__device__ __forceinline__ void gt_load_to_lds_from(const void* base, uint32_t offset, __attribute__((address_space(3))) void* lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(offset), "s"(base), "s"(lds_base)
                 : "memory", "m0");
}
