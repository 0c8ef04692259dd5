// 16 bytes of a row that may start at any address (gemm_bytes.hip). The index arithmetic and the byte moves alone, on v4i of
// common.h (or of a host program that checks the addresses).
#pragma once
#include <cstdint>

namespace sofie {

// Bytes k .. k + 15 of a row of K >= 16 bytes that starts at any address, zero behind K. load_row_chunk requests the dwords
// they lie in (loads from odd addresses are taken apart lane by lane: 256 x 1000 x 1001 in k_gemm_bytes_direct took 13.6 us
// with them and 5.7 us with K = 1000), row_chunk puts them together once they are there. A chunk that would run over the
// end of the row is requested so that it ends there and is moved down. No byte outside the aligned dwords of the row is
// touched. SHIFTS: some row or K is no multiple of four bytes (without it the fifth dword is not requested).
struct RowChunk {
   v4i d;
   int e;
};
template <bool SHIFTS>
__device__ __forceinline__ void load_row_chunk(RowChunk &c, const unsigned char *row, int k, int K)
{
   const unsigned char *p = row + (k < K - 16 ? k : K - 16);
   const int sh = (int)(reinterpret_cast<uintptr_t>(p) & 3u);
   p -= sh;
   __builtin_memcpy(&c.d, __builtin_assume_aligned(p, 4), 16);
   if constexpr (SHIFTS) c.e = *reinterpret_cast<const int *>(p + (sh ? 16 : 12));
}
template <bool SHIFTS>
__device__ __forceinline__ v4i row_chunk(const RowChunk &c, const unsigned char *row, int k, int K)
{
   v4i v = c.d;
   if constexpr (SHIFTS) {
      const unsigned sh = (unsigned)((reinterpret_cast<uintptr_t>(row) + (k < K - 16 ? k : K - 16)) & 3u);
#pragma unroll
      for (int i = 0; i < 4; ++i)
         v[i] = (int)__builtin_amdgcn_alignbyte((unsigned)(i < 3 ? c.d[i + 1] : c.e), (unsigned)c.d[i], sh);
   }
   return v;
}
// Moves of whole dwords, then of bytes. No 64-bit shift: where the allocator gave its amount the last vector register of the
// wavefront's allocation, v_lshrrev_b64 shifted by what was in v0 (912 x 272 x 46, k_gemm_bytes_direct with 128 registers: by
// the thread index).
__device__ __forceinline__ v4i trim_row_chunk(v4i v, int k, int K)
{
   const int drop = k - (K - 16);      // bytes in front of k that load_row_chunk had to take along
   if (drop <= 0) return v;
   if (drop >= 16) return v4i{0, 0, 0, 0};
   if (drop & 8) v = v4i{v[2], v[3], 0, 0};
   if (drop & 4) v = v4i{v[1], v[2], v[3], 0};
#pragma unroll
   for (int i = 0; i < 4; ++i) v[i] = (int)__builtin_amdgcn_alignbyte((unsigned)(i < 3 ? v[i + 1] : 0), (unsigned)v[i], (unsigned)drop & 3u);
   return v;
}

}  // namespace sofie
