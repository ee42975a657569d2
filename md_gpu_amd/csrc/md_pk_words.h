// md_pk_words.h -- the 64-bit words in which the persistent kernel (persist.hip) publishes
// positions and sums: data, and above them the number of the step they belong to.
//   position word   48 bits of data, 3 flag bits, the step number's low 13 bits
//   sum word        32 bits of data, 3 zero bits, the step number's low 29 bits
// A reader of step n finds the word of step n or n - 2 (or zero: nothing yet), so the low
// bits tell them apart however long the run is.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#define MD_PK_FN __host__ __device__ __forceinline__
#else
#define MD_PK_FN inline
#endif

namespace pk {

// the upper 32 bits; fl: flag bits (0..7); d16: the upper 16 of a position word's 48 data bits
MD_PK_FN uint32_t pos_tag(unsigned n, unsigned fl, unsigned d16) { return (((n << 3) | fl) << 16) | d16; }
MD_PK_FN uint32_t sum_tag(unsigned n) { return n << 3; }

MD_PK_FN uint64_t word(uint32_t data, uint32_t tag) { return (uint64_t)data | ((uint64_t)tag << 32); }
MD_PK_FN bool pos_of_step(uint64_t w, unsigned n) { return (unsigned)(w >> 51) == (n & 0x1fffu); }
MD_PK_FN bool sum_of_step(uint64_t w, unsigned n) { return (unsigned)(w >> 35) == (n & 0x1fffffffu); }

}  // namespace pk
