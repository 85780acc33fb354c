// What the matrix-core attention kernels share: fragments, transposing reads of value
// tiles, and the search for a block's rows.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "common.h"

#define LOG2E 1.44269504f

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

union frag_u {
  shortx8 s;
  shortx4 h[2];
  unsigned int u[4];
  bf16x8 v;
};

template <int N, typename F>
DEVINL void static_for(F&& f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

DEVINL unsigned int cvt2_bf16(float lo, float hi) {
  const floatx2 f = {lo, hi};
  const bf16x2 b = __builtin_convertvector(f, bf16x2);
  return __builtin_bit_cast(unsigned int, b);
}

typedef __attribute__((ext_vector_type(2))) unsigned short ushortx2;
DEVINL unsigned max_halves(unsigned a, unsigned b) {
  return __builtin_bit_cast(unsigned, __builtin_elementwise_max(__builtin_bit_cast(ushortx2, a),
                                                                __builtin_bit_cast(ushortx2, b)));
}

// Two weights p >= 0 (or NaN) as three bf16 numbers each whose sum is p to its last bit: the
// first eight, the next eight and the last eight bits. A term that would be 0 beside p > 0 is
// 2^-126, so that a weight times an infinite value is that infinity, as in fp32.
DEVINL void split3(float p0, float p1, unsigned (&u)[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const unsigned a = __builtin_bit_cast(unsigned, p0), b = __builtin_bit_cast(unsigned, p1);
    u[k] = __builtin_amdgcn_perm(b, a, 0x07060302);  // the upper halves
    p0 -= __builtin_bit_cast(float, a & 0xffff0000u);
    p1 -= __builtin_bit_cast(float, b & 0xffff0000u);
  }
  const ushortx2 least = __builtin_elementwise_min(__builtin_bit_cast(ushortx2, u[0]),
                                                   ushortx2{0x80, 0x80});
  u[1] = max_halves(u[1], __builtin_bit_cast(unsigned, least));
  u[2] = max_halves(u[2], __builtin_bit_cast(unsigned, least));
}

// Transposing reads of two V^T fragments, of each the halves HALF bytes apart. Written out
// because the compiler puts a wait for all global loads in flight, the next tiles' among
// them, before the builtin form. Nothing may touch v before await_values: no branch and
// nothing that could run out of registers stands between the two.
template <int AT, int HALF>
DEVINL void read_values(shortx4 (&v)[4], unsigned a0, unsigned a1) {
  asm volatile(
      "ds_read_b64_tr_b16 %0, %4 offset:%6\n\t"
      "ds_read_b64_tr_b16 %1, %4 offset:%7\n\t"
      "ds_read_b64_tr_b16 %2, %5 offset:%6\n\t"
      "ds_read_b64_tr_b16 %3, %5 offset:%7"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(a0), "v"(a1), "n"(AT), "n"(AT + HALF)
      : "memory");
}

DEVINL void await_values(shortx4 (&v)[4]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])::"memory");
}

// Sequence and first row of the nb-th block of ``rows`` rows, counted through the
// sequences; false past the last. A lane per sequence.
DEVINL bool find_block(const int* cu, int S, int rows, int nb, int lane, int& seq, int& off) {
  for (int s0 = 0; s0 < S; s0 += WAVE) {
    const int s = s0 + lane;
    const int n = s < S ? (cu[s + 1] - cu[s] + rows - 1) / rows : 0;
    int end = n;
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
      const int before = __shfl_up(end, d, WAVE);
      if (lane >= d) end += before;
    }
    const unsigned long long past = __ballot(end > nb);
    if (past) {
      const int at = __builtin_ctzll(past);
      seq = s0 + at;
      off = (nb - __builtin_amdgcn_readlane(end - n, at)) * rows;
      return true;
    }
    nb -= __builtin_amdgcn_readlane(end, WAVE - 1);
  }
  return false;
}
