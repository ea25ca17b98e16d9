// Weights of the next product into the XCDs' L2s, from blocks of a kernel before it that leaves
// the memory idle.  Lines that are only read stay there from kernel to kernel, and blocks go
// round the XCDs by their numbers, so a block that is to read rows of W finds them on its own:
// one row of 4096 into 4096 8.4 us from memory, 5.0 so.
#pragma once

#include "hip_common.h"

// 16 bytes a lane from memory to LDS (at + 16 * lane).  The compiler does not know of the
// load, which would have it wait for all before reads of LDS; no register is written.  Nor does
// it look into the text: a load to LDS may not read M0 in the cycle behind the scalar unit's
// write of it, so that one idle instruction lies between.
__device__ __forceinline__ void to_lds(const char* from, unsigned at) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(at),
               "v"(from)
               : "memory", "m0");
}

struct Warm {
  const char* w;  // null: none
  long ld;        // bytes from row to row
  int rows, O, K; // of W of a block of the product, in all; columns
  int chunks;     // of 64 columns of a row that are fetched, from where the block begins
  int blocks;     // of the product
  unsigned turn;  // where they begin (first_column)
};

// The chunk of n that a block begins at (linear_few_kernel.h).
__device__ __forceinline__ int first_chunk(unsigned turn, int whole, int n, unsigned block) {
  if (!turn) return 0;
  const unsigned at = (block >> 3) * 3;
  return max(min((int)(at - __umulhi(at, turn) * whole), n - 1), 0);
}

// Block `block` of which those from `base` to `end` fetch; lds: 1 KB of a wave's that nothing
// reads.  Ends when all loads have come.
__device__ __forceinline__ void warm_rows(const Warm& a, int block, int base, int end, int wid,
                                          int waves, unsigned lds) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int xcd = block & 7, least = base + ((xcd - base) & 7);
  const int step = (end - least + 7) / 8 * 8;  // blocks of the product between two of this one's
  const int all = (a.K + 63) / 64, loads = a.chunks * (a.rows / 8);
  for (int b = xcd + (block - least); b < a.blocks; b += step) {
    const int first = first_chunk(a.turn, all, all, b);
    // a load is 8 rows of 128 bytes
    for (int i = wid; i < loads; i += waves) {
      int c = i / (a.rows / 8) + first;
      c = c >= all ? c - all : c;
      const int row = min(b * a.rows + i % (a.rows / 8) * 8 + (lane >> 3), a.O - 1);
      const char* from = a.w + (long)row * a.ld + min(c * 64 + (lane & 7) * 8, a.K - 8) * 2;
      to_lds(from, lds);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

extern "C" {
// How a product of M rows, on its own, reads W [O, K] of rows ld elements apart, if it is one
// that this helps.
bool linear_own_warm(long M, long O, long K, long ld, const void* w, Warm* out);
}
