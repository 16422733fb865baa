// The row partition inside a GEMM: every workgroup counts the mask itself and finds the token rows of its own tile.
//
// A partition of its own (route.hip) is a launch ahead of the GEMM, and the GEMM then waits for two loads that depend on each
// other, the counts and its rows of perm.  Up to kScanMaxRows rows the whole mask is 16 or 32 bytes per thread: one load, a
// prefix sum over the workgroup, and the tile's rows are in LDS.
#pragma once
#include "common.hpp"
#include "gemm_args.hpp"
#include "gemm_sched.hpp"

namespace ffnk {

// 16-bit mask of the non-zero bytes of a 16-byte vector (bit j = byte j).
__device__ __forceinline__ uint32_t nonzero_bytes16(uint4 v) {
  uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t bits = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t t = (w[i] | ((w[i] & 0x7f7f7f7fu) + 0x7f7f7f7fu)) & 0x80808080u;  // bit 7 of each non-zero byte
    uint32_t nib = (((t >> 7) * 0x01020408u) >> 24) & 0xFu;                     // gather to 4 bits
    bits |= nib << (4 * i);
  }
  return bits;
}

// Inclusive prefix sum over the 64 lanes.
__device__ __forceinline__ int wave_prefix_sum(int v) {
#if defined(__HIP_DEVICE_COMPILE__)
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1, 2, 4, 8: inside 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15: the last of rows 0 and 2 to rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31: the last of row 1 to rows 2 and 3
#endif
  return v;
}

// Index of set bit number n (0 = lowest) of a word that has more than n.
__device__ __forceinline__ int nth_set_bit(uint32_t word, int n) {
  int at = 0;
#pragma unroll
  for (int half = 16; half >= 1; half >>= 1) {
    const int c = __popc((word >> at) & ((1u << half) - 1u));
    if (n >= c) {
      n -= c;
      at += half;
    }
  }
  return at;
}

// A thread counts the rows of its own word of ROWS rows; the words and the visual rows ahead of each stay in LDS, and the row of a
// position is found from there: the wave's segment of 64 words, one of its eights, the word, the bit - three dependent LDS reads
// for a position per thread, whatever the mask.  (Threads that walk their own rows and write those of the tile take up to 32
// steps of 150 cycles with nothing to hide them: 2-3 us of a tile.)
template <int NT>
struct RowScan {
  static constexpr int ROWS = kScanMaxRows / NT;  // consecutive rows of a thread
  static constexpr int NWAVES = NT / kWave;
  static_assert(ROWS == 16 || ROWS == 32, "one or two 16-byte loads per thread");
  // LDS (ints): visual rows per wave | ahead of every eighth word | ahead of every word | words | the tile's token rows
  static constexpr int kEighths = NWAVES, kAhead = kEighths + NWAVES * 8, kWords = kAhead + NT, kRows = kWords + NT;
  static_assert(kEighths % 4 == 0 && (kRows + 256) * 4 <= 64 * 128, "16-byte aligned, inside the smallest token panel");

  int start[NWAVES];  // visual rows ahead of each wave's words
  int n_vis;          // of all M (uniform)

  // `lds`: free until the caller's next barrier but one.  Rows past M count as neither.
  __device__ __forceinline__ void scan(const uint8_t* mask, int M, uint8_t* lds) {
    const int t = (int)threadIdx.x, first = t * ROWS;
    uint32_t bits = 0;
    if (first < M) {
      // (whole aligned 16-byte vectors that hold a row: never past the page of the mask's last byte)
      const uint4* v = reinterpret_cast<const uint4*>(mask + first);
      const uint4 a = v[0];
      uint4 b = make_uint4(0, 0, 0, 0);
      if (ROWS == 32 && first + 16 < M) b = v[1];
      bits = nonzero_bytes16(a) | (ROWS == 32 ? nonzero_bytes16(b) << 16 : 0u);
      const int n = M - first;
      if (n < ROWS) bits &= (1u << n) - 1u;
    }
    const int own = __popc(bits), incl = wave_prefix_sum(own);
    int* s = reinterpret_cast<int*>(lds);
    s[kWords + t] = (int)bits;
    s[kAhead + t] = incl - own;
    if (t % 8 == 0) s[kEighths + t / 8] = incl - own;
    if (t % kWave == kWave - 1) s[t / kWave] = incl;
    __syncthreads();
    int total = 0;
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) {
      start[w] = total;
      total += __builtin_amdgcn_readfirstlane(s[w]);
    }
    n_vis = total;
  }

  // Token row of member q (0 <= q < the group's rows) of group grp.
  __device__ __forceinline__ int find(int grp, int q, const uint8_t* lds) const {
    const int* s = reinterpret_cast<const int*>(lds);
    auto ahead = [&](int word, int visual) { return grp == 0 ? visual : word * ROWS - visual; };  // members ahead of a word
    int w = 0;
#pragma unroll
    for (int k = 1; k < NWAVES; ++k) w = ahead(k * kWave, start[k]) <= q ? k : w;
    int from = 0;  // visual rows ahead of the wave's words
#pragma unroll
    for (int k = 1; k < NWAVES; ++k) from = w == k ? start[k] : from;
    auto last_of_eight = [&](const int* at, int word, int step) {  // the last of eight words `step` apart with at most q members ahead
      const int4 lo = *reinterpret_cast<const int4*>(at), hi = *reinterpret_cast<const int4*>(at + 4);
      const int v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      int k = 0;
#pragma unroll
      for (int i = 1; i < 8; ++i) k = ahead(word + i * step, from + v[i]) <= q ? i : k;
      return word + k * step;
    };
    const int eighth = last_of_eight(s + kEighths + w * 8, w * kWave, 8);
    const int word = last_of_eight(s + kAhead + eighth, eighth, 1);
    const uint32_t bits = (uint32_t)s[kWords + word];
    const int before = ahead(word, from + s[kAhead + word]);
    return word * ROWS + nth_set_bit(grp == 0 ? bits : ~bits, q - before);
  }

  // Token rows of routed positions [lo, hi) of group grp -> LDS, position lo first.
  __device__ __forceinline__ void place(int grp, int lo, int hi, uint8_t* lds) const {
    for (int p = lo + (int)threadIdx.x; p < hi; p += NT) reinterpret_cast<int*>(lds)[kRows + p - lo] = find(grp, grp == 0 ? p : p - n_vis, lds);
  }
  static __device__ __forceinline__ int row(const uint8_t* lds, int p) { return reinterpret_cast<const int*>(lds)[kRows + p]; }
};

}  // namespace ffnk
