// Generated by gen_dpp_fma.py; do not edit.
//
// Multiply-adds with a wave-uniform table operand held in vector registers.
// A table of n values sits in ceil(n / 16) registers, value i in lanes
// l % 16 == i % 16 of register i / 16 (every row of 16 lanes holds a copy),
// and v_fmac reads value i through its DPP row_newbcast modifier, which
// hands one lane of a row to the row's 16 lanes at the full FMA rate
// (measured 62.8 against 62.5 TFLOP/s for the plain FP64 instruction).  A
// contraction then waits for no table load at all, where scalar loads of
// its rows cost a scalar-cache round trip each.
//
// dpp_fma<OFF, STRIDE>(t, x, a): a[i] += table[OFF + i STRIDE] x for the
// LEN values of a.  One asm block per call: its leading s_nop keeps the two
// wait states a DPP read needs after any VALU write of a table register
// (the compiler does not look into the block).  DPP reads an inactive
// lane's register as invalid, so every lane of the wave must be active: call
// it in uniform control flow only, and mask loads and stores instead.
#pragma once

#include <hip/hip_runtime.h>

namespace femtc
{

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[1])
{
  static_assert(OFF + 0 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %1, %3 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[2])
{
  static_assert(OFF + 1 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %2, %6 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %4, %6 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[3])
{
  static_assert(OFF + 2 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %3, %9 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %5, %9 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %7, %9 row_newbcast:%8 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[4])
{
  static_assert(OFF + 3 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %4, %12 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %6, %12 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %8, %12 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %10, %12 row_newbcast:%11 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[5])
{
  static_assert(OFF + 4 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %5, %15 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %7, %15 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %9, %15 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %11, %15 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %13, %15 row_newbcast:%14 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[6])
{
  static_assert(OFF + 5 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %6, %18 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %8, %18 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %10, %18 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %12, %18 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %14, %18 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %5, %16, %18 row_newbcast:%17 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(t[(OFF + 5 * STRIDE) / 16]), "n"((OFF + 5 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[7])
{
  static_assert(OFF + 6 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %7, %21 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %9, %21 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %11, %21 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %13, %21 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %15, %21 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %5, %17, %21 row_newbcast:%18 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %6, %19, %21 row_newbcast:%20 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(t[(OFF + 5 * STRIDE) / 16]), "n"((OFF + 5 * STRIDE) % 16),
        "v"(t[(OFF + 6 * STRIDE) / 16]), "n"((OFF + 6 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const double (&t)[NR], double x,
                                        double (&a)[8])
{
  static_assert(OFF + 7 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %8, %24 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %10, %24 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %12, %24 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %14, %24 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %4, %16, %24 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %5, %18, %24 row_newbcast:%19 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %6, %20, %24 row_newbcast:%21 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %7, %22, %24 row_newbcast:%23 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(t[(OFF + 5 * STRIDE) / 16]), "n"((OFF + 5 * STRIDE) % 16),
        "v"(t[(OFF + 6 * STRIDE) / 16]), "n"((OFF + 6 * STRIDE) % 16),
        "v"(t[(OFF + 7 * STRIDE) / 16]), "n"((OFF + 7 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[1])
{
  static_assert(OFF + 0 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %1, %3 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[2])
{
  static_assert(OFF + 1 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %2, %6 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %4, %6 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[3])
{
  static_assert(OFF + 2 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %3, %9 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %5, %9 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %7, %9 row_newbcast:%8 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[4])
{
  static_assert(OFF + 3 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %4, %12 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %6, %12 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %8, %12 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %10, %12 row_newbcast:%11 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[5])
{
  static_assert(OFF + 4 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %5, %15 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %7, %15 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %9, %15 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %11, %15 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %13, %15 row_newbcast:%14 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[6])
{
  static_assert(OFF + 5 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %6, %18 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %8, %18 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %10, %18 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %12, %18 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %14, %18 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %5, %16, %18 row_newbcast:%17 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(t[(OFF + 5 * STRIDE) / 16]), "n"((OFF + 5 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[7])
{
  static_assert(OFF + 6 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %7, %21 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %9, %21 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %11, %21 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %13, %21 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %15, %21 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %5, %17, %21 row_newbcast:%18 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %6, %19, %21 row_newbcast:%20 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(t[(OFF + 5 * STRIDE) / 16]), "n"((OFF + 5 * STRIDE) % 16),
        "v"(t[(OFF + 6 * STRIDE) / 16]), "n"((OFF + 6 * STRIDE) % 16),
        "v"(x));
}

template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const float (&t)[NR], float x,
                                        float (&a)[8])
{
  static_assert(OFF + 7 * STRIDE < 16 * NR, "value inside the table");
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %8, %24 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %10, %24 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %2, %12, %24 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %3, %14, %24 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %4, %16, %24 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %5, %18, %24 row_newbcast:%19 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %6, %20, %24 row_newbcast:%21 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %7, %22, %24 row_newbcast:%23 row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
      : "v"(t[(OFF + 0 * STRIDE) / 16]), "n"((OFF + 0 * STRIDE) % 16),
        "v"(t[(OFF + 1 * STRIDE) / 16]), "n"((OFF + 1 * STRIDE) % 16),
        "v"(t[(OFF + 2 * STRIDE) / 16]), "n"((OFF + 2 * STRIDE) % 16),
        "v"(t[(OFF + 3 * STRIDE) / 16]), "n"((OFF + 3 * STRIDE) % 16),
        "v"(t[(OFF + 4 * STRIDE) / 16]), "n"((OFF + 4 * STRIDE) % 16),
        "v"(t[(OFF + 5 * STRIDE) / 16]), "n"((OFF + 5 * STRIDE) % 16),
        "v"(t[(OFF + 6 * STRIDE) / 16]), "n"((OFF + 6 * STRIDE) % 16),
        "v"(t[(OFF + 7 * STRIDE) / 16]), "n"((OFF + 7 * STRIDE) % 16),
        "v"(x));
}

} // namespace femtc
