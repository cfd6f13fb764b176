// The contraction chain of one cell group of the chain kernels
// (apply_chain.hpp), stage by stage, on the schedule, axis order and LDS
// layout that apply_kernel.hpp describes.  The caller synchronises between
// the stages.
//
// Tables in registers.  A contraction walks its table one row at a time,
// acc[m] += T[k][m] in[k], and the wave-uniform T[k][m] come from vector
// registers through dpp_fma (dpp_fma.hpp): the table set is loaded once per
// wave (2 N Q values in 2 N Q / 16 registers: 14 VGPRs for FP64 at N = Q =
// 7).  Against scalar loads of each row as in apply_kernel.hpp (MI355X, us
// per gathered apply): affine FP64 K+M at P=5, 97,290 cells, 235 -> 218; FP32
// mass at P=3, Q=5, 290,177 cells, 113 -> 110.  (In the fused kernels of
// apply_kernel.hpp scalar rows are as fast or faster: FP32 even-odd cell pass
// 134 against 166.)
//
// Every stage therefore runs in all lanes of the wave.  Lanes outside a
// stage's role read a line that another lane owns and have their stores
// masked (the `on` arguments).
#pragma once

#include "cell_common.hpp"
#include "common.hpp"
#include "dpp_fma.hpp"
#include "lds_layout.hpp"

namespace femtc
{

// The table registers of a wave: SIZE values of a table in global memory.
template <typename T, int SIZE>
struct TableRegs
{
  static constexpr int NR = (SIZE + 15) / 16;
  T r[NR];

  __device__ __forceinline__ void load(const T* __restrict__ tab)
  {
    const int l = (int)(threadIdx.x & 15);
#pragma unroll
    for (int i = 0; i < NR; ++i)
    {
      const int k = i * 16 + l;
      r[i] = 16 * (i + 1) <= SIZE ? tab[k] : tab[k < SIZE ? k : 0];
    }
  }
};

// out[m] += sum_k T(k, m) in[k] with T(k, m) = table[OFF + k KS + m MS]
template <int OFF, int KS, int MS, int NR, typename T, int K, int M,
          int k = 0>
__device__ __forceinline__ void contract(const T (&t)[NR], const T (&in)[K],
                                         T (&out)[M])
{
  if constexpr (k < K)
  {
    dpp_fma<OFF + k * KS, MS>(t, in[k], out);
    contract<OFF, KS, MS, NR, T, K, M, k + 1>(t, in, out);
  }
}

template <typename T, int M>
__device__ __forceinline__ void clear(T (&a)[M])
{
#pragma unroll
  for (int m = 0; m < M; ++m)
    a[m] = T(0);
}

// One cell's stages for operator OP (correct mode) in precision T.
template <typename T, int N, int Q, int OP>
struct CellChain
{
  static constexpr bool AFF = OP >= OP_MASS_AFF; // geometry per cell
  static constexpr int OPB = AFF ? OP - OP_MASS_AFF : OP;
  static constexpr bool MASSTERM = (OPB == OP_MASS || OPB == OP_KPM);
  static constexpr bool GRAD = (OPB != OP_MASS);
  static constexpr bool GEO = GRAD && !AFF; // geometry streamed per point
  // table registers: [phi | dphi] (phi alone for the mass operator)
  static constexpr int TABLE = GRAD ? 2 * N * Q : N * Q;
  using Tab = TableRegs<T, TABLE>;
  static constexpr int NR = Tab::NR;
  // the Gauss weights in the table set in memory
  static constexpr int WOFF = 2 * N * Q;
  static constexpr int NX = GRAD ? 2 : 1; // X tensors
  static constexpr int NY = GRAD ? 3 : 1; // Y tensors
  // X[qb][c][a] and Y[a][qb][qc] with bank-conflict-minimising strides
  static constexpr LdsLayout LY = lds_layout<(int)sizeof(T), N, Q>();
  static constexpr int XQ = LY.XQ, XC = LY.XC, YQ = LY.YQ, YA = LY.YA;
  static constexpr int SX = Q * XQ; // one X tensor
  static constexpr int SY = N * YA; // one Y tensor
  // LDS slots
  static constexpr int X_P = 0, X_G = 1;             // F1 -> F2
  static constexpr int Y_PP = 0, Y_PG = 1, Y_GP = 2; // F2 -> F3
  static constexpr int Y_RA = 0, Y_RB = 1, Y_RC = 2; // B3 -> B2
  static constexpr int X_S0 = 0, X_SB = 1;           // B2 -> B1

  // Per-cell LDS elements of a group of CPB cells: the tuned strides where
  // the table has them, else the cell's own footprint.  X and Y share it.
  template <int CPB>
  static constexpr int wcell()
  {
    constexpr int X = CPB > 1 && LY.XCELL ? LY.XCELL : NX * SX;
    constexpr int Y = CPB > 1 && LY.YCELL ? LY.YCELL : NY * SY;
    static_assert(X >= NX * SX && Y >= NY * SY, "layout fits");
    return X > Y ? X : Y;
  }

  // out = phi in (D = 0) or g in (D = 1), dofs to points
  template <int D>
  static __device__ __forceinline__ void fwd(const Tab& t, const T (&in)[N],
                                             T (&out)[Q])
  {
    clear(out);
    contract<D * N * Q, Q, 1>(t.r, in, out);
  }

  // out = sum of phi' in0 (HAS0) and g' in1 (HAS1), points to dofs
  template <bool HAS0, bool HAS1>
  static __device__ __forceinline__ void bwd(const Tab& t, const T (&in0)[Q],
                                             const T (&in1)[Q], T (&out)[N])
  {
    clear(out);
    if constexpr (HAS0)
      contract<0, 1, Q>(t.r, in0, out);
    if constexpr (HAS1)
      contract<N * Q, 1, Q>(t.r, in1, out);
  }

  // F1: contract axis b of the line (a, c) and store it into X.
  static __device__ __forceinline__ void f1(const Tab& t, const T (&u)[N],
                                            T* Xc, int a, int c, bool on)
  {
    T ap[Q], ag[Q];
    fwd<0>(t, u, ap);
    if constexpr (GRAD)
      fwd<1>(t, u, ag);
    if (on)
    {
#pragma unroll
      for (int q = 0; q < Q; ++q)
      {
        Xc[X_P * SX + q * XQ + c * XC + a] = ap[q];
        if constexpr (GRAD)
          Xc[X_G * SX + q * XQ + c * XC + a] = ag[q];
      }
    }
  }

  // F2: contract axis c of the line (qb, a) of X.
  static __device__ __forceinline__ void f2(const Tab& t, const T* Xc, int qb,
                                            int a, T (&bpp)[Q], T (&bpg)[Q],
                                            T (&bgp)[Q])
  {
    T inp[N], ing[N];
#pragma unroll
    for (int c = 0; c < N; ++c)
    {
      inp[c] = Xc[X_P * SX + qb * XQ + c * XC + a];
      if constexpr (GRAD)
        ing[c] = Xc[X_G * SX + qb * XQ + c * XC + a];
    }
    fwd<0>(t, inp, bpp);
    if constexpr (GRAD)
    {
      fwd<1>(t, inp, bpg);
      fwd<0>(t, ing, bgp);
    }
  }

  static __device__ __forceinline__ void f2_store(T* Yc, int qb, int a,
                                                  bool on, const T (&bpp)[Q],
                                                  const T (&bpg)[Q],
                                                  const T (&bgp)[Q])
  {
    const int o = a * YA + qb * YQ;
    if (on)
    {
#pragma unroll
      for (int q = 0; q < Q; ++q)
      {
        Yc[Y_PP * SY + o + q] = bpp[q];
        if constexpr (GRAD)
        {
          Yc[Y_PG * SY + o + q] = bpg[q];
          Yc[Y_GP * SY + o + q] = bgp[q];
        }
      }
    }
  }

  // F3 reads the line (qb, qc) of Y at offset yo = qb YQ + qc.
  static __device__ __forceinline__ void f3_load(const T* Yc, int yo,
                                                 T (&ipp)[N], T (&ipg)[N],
                                                 T (&igp)[N])
  {
#pragma unroll
    for (int a = 0; a < N; ++a)
    {
      ipp[a] = Yc[Y_PP * SY + a * YA + yo];
      if constexpr (GRAD)
      {
        ipg[a] = Yc[Y_PG * SY + a * YA + yo];
        igp[a] = Yc[Y_GP * SY + a * YA + yo];
      }
    }
  }

  // F3: contract axis a.
  static __device__ __forceinline__ void
  f3(const Tab& t, const T (&ipp)[N], const T (&ipg)[N], const T (&igp)[N],
     T (&uq)[Q], T (&da)[Q], T (&db)[Q], T (&dc)[Q])
  {
    if constexpr (MASSTERM)
      fwd<0>(t, ipp, uq);
    if constexpr (GRAD)
    {
      fwd<1>(t, ipp, da);
      fwd<0>(t, igp, db);
      fwd<0>(t, ipg, dc);
    }
  }

  // Point q: v = S(q) d (+ detJw u).  g and dw are filled from the cell's
  // values cg (w = w(qa) w(qb) w(qc)) on affine cells.
  static __device__ __forceinline__ void
  point(int q, T (&g)[6], T& dw, const T* cg, T w, const T (&uq)[Q],
        const T (&da)[Q], const T (&db)[Q], const T (&dc)[Q], T (&va)[Q],
        T (&vb)[Q], T (&vc)[Q], T (&vm)[Q])
  {
    if constexpr (AFF)
    {
      // G(q) = w(qa) w(qb) w(qc) S, detJw(q) = w(qa) w(qb) w(qc) detJ
      if constexpr (GRAD)
      {
#pragma unroll
        for (int k = 0; k < 6; ++k)
          g[k] = w * cg[k];
      }
      if constexpr (MASSTERM)
        dw = w * cg[6];
    }
    if constexpr (GRAD)
    {
      // S = [[G5,G4,G2],[G4,G3,G1],[G2,G1,G0]] on (d_a, d_b, d_c)
      va[q] = g[5] * da[q] + g[4] * db[q] + g[2] * dc[q];
      vb[q] = g[4] * da[q] + g[3] * db[q] + g[1] * dc[q];
      vc[q] = g[2] * da[q] + g[1] * db[q] + g[0] * dc[q];
    }
    if constexpr (MASSTERM)
      vm[q] = dw * uq[q];
  }

  // B3: contract axis a (transposed).
  static __device__ __forceinline__ void
  b3(const Tab& t, const T (&va)[Q], const T (&vb)[Q], const T (&vc)[Q],
     const T (&vm)[Q], T (&ra)[N], T (&rb)[N], T (&rc)[N])
  {
    bwd<MASSTERM, GRAD>(t, vm, va, ra);
    if constexpr (GRAD)
    {
      bwd<true, false>(t, vb, vb, rb);
      bwd<true, false>(t, vc, vc, rc);
    }
  }

  static __device__ __forceinline__ void b3_store(T* Yc, int yo, bool on,
                                                  const T (&ra)[N],
                                                  const T (&rb)[N],
                                                  const T (&rc)[N])
  {
    if (on)
    {
#pragma unroll
      for (int a = 0; a < N; ++a)
      {
        const int o = a * YA + yo;
        Yc[Y_RA * SY + o] = ra[a];
        if constexpr (GRAD)
        {
          Yc[Y_RB * SY + o] = rb[a];
          Yc[Y_RC * SY + o] = rc[a];
        }
      }
    }
  }

  static __device__ __forceinline__ void b2_load(const T* Yc, int qb, int a,
                                                 T (&ra)[Q], T (&rb)[Q],
                                                 T (&rc)[Q])
  {
    const int o = a * YA + qb * YQ;
#pragma unroll
    for (int q = 0; q < Q; ++q)
    {
      ra[q] = Yc[Y_RA * SY + o + q];
      if constexpr (GRAD)
      {
        rb[q] = Yc[Y_RB * SY + o + q];
        rc[q] = Yc[Y_RC * SY + o + q];
      }
    }
  }

  // B2: contract axis c (transposed) of the line (qb, a), stored into X.
  static __device__ __forceinline__ void b2(const Tab& t, const T (&ra)[Q],
                                            const T (&rb)[Q],
                                            const T (&rc)[Q], T* Xc, int qb,
                                            int a, bool on)
  {
    T s0[N], sb[N];
    bwd<true, GRAD>(t, ra, rc, s0);
    if constexpr (GRAD)
      bwd<true, false>(t, rb, rb, sb);
    if (on)
    {
#pragma unroll
      for (int c = 0; c < N; ++c)
      {
        const int xo = qb * XQ + c * XC + a;
        Xc[X_S0 * SX + xo] = s0[c];
        if constexpr (GRAD)
          Xc[X_SB * SX + xo] = sb[c];
      }
    }
  }

  // B1: contract axis b (transposed) of the line (a, c) of X.
  static __device__ __forceinline__ void b1(const Tab& t, const T* Xc, int a,
                                            int c, T (&w)[N])
  {
    T s0[Q], sb[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q)
    {
      s0[q] = Xc[X_S0 * SX + q * XQ + c * XC + a];
      if constexpr (GRAD)
        sb[q] = Xc[X_SB * SX + q * XQ + c * XC + a];
    }
    bwd<true, GRAD>(t, s0, sb, w);
  }
};

} // namespace femtc
