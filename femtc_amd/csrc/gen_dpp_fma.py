"""Writes dpp_fma.hpp: multiply-adds whose table operand is broadcast from a
register (see the generated header's comment).

    python3 gen_dpp_fma.py > dpp_fma.hpp
"""

HEADER = """// Generated by gen_dpp_fma.py; do not edit.
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
"""

MAX = 8  # lines of at most 8 dofs or points


def block(ctype, op, n):
    x = 3 * n  # operand numbers: n accumulators, n (table, lane) pairs, x
    lines = ['"s_nop 1\\n\\t"']
    for i in range(n):
        lines.append(f'"{op} %{i}, %{n + 2 * i}, %{x} row_newbcast:%{n + 2 * i + 1} '
                     f'row_mask:0xf bank_mask:0xf{"" if i == n - 1 else chr(92) + "n" + chr(92) + "t"}"')
    body = "\n      ".join(lines)
    outs = ", ".join(f'"+v"(a[{i}])' for i in range(n))
    ins = ",\n        ".join(
        f'"v"(t[(OFF + {i} * STRIDE) / 16]), "n"((OFF + {i} * STRIDE) % 16)'
        for i in range(n))
    return f"""
template <int OFF, int STRIDE, int NR>
__device__ __forceinline__ void dpp_fma(const {ctype} (&t)[NR], {ctype} x,
                                        {ctype} (&a)[{n}])
{{
  static_assert(OFF + {n - 1} * STRIDE < 16 * NR, "value inside the table");
  asm({body}
      : {outs}
      : {ins},
        "v"(x));
}}
"""


def main():
    out = HEADER
    for ctype, op in (("double", "v_fmac_f64_dpp"), ("float", "v_fmac_f32_dpp")):
        for n in range(1, MAX + 1):
            out += block(ctype, op, n)
    out += "\n} // namespace femtc"
    print(out)


if __name__ == "__main__":
    main()
