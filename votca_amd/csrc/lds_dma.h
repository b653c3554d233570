// Global-to-LDS loads (gfx950) and the LDS row layout that the direct-to-LDS GEMM kernels share.
//
// global_load_lds_dwordx4 moves 16 bytes per lane from L2 / HBM straight into LDS (lane l lands at
// base + 16 l), so tiles in flight hold no registers. An LDS row is 128 bytes of one operand row (64
// BF16, 32 of the hi plane and the same 32 of the lo plane, or 16 doubles); one load instruction fills
// eight rows, the eight lanes of a row fetching 128 contiguous bytes (64 per plane). The 16-byte
// chunk c of row r sits at slot c ^ ((r & 7) ^ ((r >> 3) & 1)): a fragment read (16 rows, one chunk)
// touches 16 distinct 16-byte bank groups (measured: 8 cycles per ds_read_b128 of a wave, as for a
// linear read; 32 without the swizzle).
#pragma once
#include "gemm_kernels.h"

namespace xg {

// 16-byte-aligned zeros that out-of-range lanes load from (never written)
__device__ __attribute__((aligned(64))) unsigned int g_zero_page[16];

typedef __attribute__((address_space(3))) uint4 lds_u4;

// 16 bytes per lane from global memory into LDS at (uniform) byte offset `lds_off` + 16 * lane.
// Issued as inline assembly so that the compiler's wait-count pass does not tie every later LDS
// read to these loads; completion is tracked explicitly with s_waitcnt vmcnt in the main loops.
__device__ __forceinline__ void dma16(const void* g, unsigned lds_off) {
  const unsigned o = __builtin_amdgcn_readfirstlane(lds_off);
  // one wait state between the M0 write and the LDS-DMA load that reads it
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(o), "v"(g) : "memory", "m0");
}

__device__ __forceinline__ int lds_slot(int row, int c) { return c ^ ((row & 7) ^ ((row >> 3) & 1)); }

// Usable for BF16 operands that are K-contiguous planes (hi and, for SPLIT, lo) with 16-byte aligned
// rows: ld, batch stride and K multiples of 8, K chunks multiples of the stage's k.
inline bool lds_ok(const Opnd<unsigned short>& A, const Opnd<unsigned short>& B, int K, bool split) {
  auto al = [](const void* p) { return p != nullptr && (reinterpret_cast<uintptr_t>(p) % 16) == 0; };
  return al(A.p) && al(B.p) && (!split || (al(A.lo) && al(B.lo))) && A.ld % 8 == 0 && B.ld % 8 == 0 &&
         A.bs % 8 == 0 && B.bs % 8 == 0 && K % 8 == 0;
}

}  // namespace xg
