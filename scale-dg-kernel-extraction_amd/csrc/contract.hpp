// Contraction of one pencil held in a lane's registers with an operator that is
// the same for every lane, read through the scalar cache (stage_pencil,
// stage_aug).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

namespace dgk {

// The order in which a contraction adds its products: row n of n < N is l(n).
template <int NQ>
struct RowsAscending {
  static constexpr int N = NQ;
  static constexpr int l(int n) { return n; }
};

// acc[c] = sum over n of a[l(n)] B(l(n), c), n ascending, every product fused
// into the sum; B(l, c) = D[c + l NQ] for l < NQ, ell[c + (l - NQ) NQ] above.
//
// B's entries are scalar operands, read in batches of 128 bytes (32 scalar
// registers), a batch ahead.  Scalar loads return out of order, so a wait for
// one is a wait for all: the batch in use is waited for (the pins on `cur`)
// before the next one is asked for, which then has a batch of arithmetic to
// arrive in.  Without the pins the compiler waits for both at once; without the
// opaque addresses and the ties on acc it loads all of B first and spills it.
template <class T, int NQ, class Rows>
struct Contract {
  static constexpr int W = 128 / (int)sizeof(T);
  static constexpr int TOTAL = Rows::N * NQ;
  static constexpr int BATCHES = (TOTAL + W - 1) / W;
  typedef const T __attribute__((address_space(4))) *uniform_ptr;
  uniform_ptr pd, pe;
  T buf[2][W];

  template <int B>
  __device__ __forceinline__ void load(T (&to)[W]) {
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const int t = B * W + k;
      if (t < TOTAL) {
        const int l = Rows::l(t / NQ), c = t % NQ;
        to[k] = l < NQ ? pd[l * NQ + c] : pe[(l - NQ) * NQ + c];
      }
    }
  }
  template <int B, int NA>
  __device__ __forceinline__ void step(const T (&a)[NA], T (&acc)[NQ]) {
    T(&cur)[W] = buf[B & 1];
    if constexpr (B + 1 < BATCHES) {
#pragma unroll
      for (int k = 0; k < W; ++k)
        if (B * W + k < TOTAL) asm volatile("" : : "s"(cur[k]));
      asm volatile("" : "+s"(pd), "+s"(pe));
#pragma unroll
      for (int c = 0; c < NQ; ++c) asm volatile("" : "+v"(acc[c]));
      load<B + 1>(buf[(B + 1) & 1]);
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
      const int t = B * W + k;
      if (t < TOTAL) {
        const int n = t / NQ, c = t % NQ;
        if constexpr (std::is_same<T, float>::value)
          acc[c] = __builtin_fmaf(a[Rows::l(n)], cur[k], acc[c]);
        else
          acc[c] = __builtin_fma(a[Rows::l(n)], cur[k], acc[c]);
      }
    }
  }
  template <int NA, int... B>
  __device__ __forceinline__ void steps(const T (&a)[NA], T (&acc)[NQ],
                                        std::integer_sequence<int, B...>) {
    (step<B>(a, acc), ...);
  }
  template <int NA>
  __device__ __forceinline__ void run(const T *D, const T *ell, const T (&a)[NA], T (&acc)[NQ]) {
    pd = (uniform_ptr)D;
    pe = (uniform_ptr)ell;
    load<0>(buf[0]);
#pragma unroll
    for (int c = 0; c < NQ; ++c) acc[c] = (T)0;
    steps(a, acc, std::make_integer_sequence<int, BATCHES>());
  }
};

}  // namespace dgk
