// Chain kernel: the continuous operator through any dofmap, with the faces
// that consecutive cells share summed in LDS.
//
// What bounds the gathered kernel of apply_kernel.hpp is mostly its scatter:
// N^3 memory-side atomics per cell in runs of N addresses (61-77 G/s; runs of
// 33 sustain 141 G/s).  Mesh numberings, lexicographic or in the order a
// reader meets the cells, mostly list neighbours one after another, so here
// one workgroup takes a chain of S consecutive cells.  Each cell's right
// face (c = P) and the next cell's left face (c = 0) share one slot of a box
// [N][N][S P + 1] in LDS wherever the dofmap gives both the same dofs; the
// box then goes to y with one atomic per slot, consecutive lanes on
// consecutive dofs.
//
//  * Any dofmap is correct: a left-face dof that is not its left neighbour's
//    right-face dof is added to y on its own.  The check reads only the
//    dofmap entries that the neighbour's lanes read anyway.
//  * No LDS atomics: slot c >= 1 of a cell belongs to that cell (its lanes
//    store it), and after a barrier the left faces are added to their
//    neighbours' slots, one owner each.  LDS FP32 atomics made the P=6 FP32
//    K+M pass 385 us against 248.
//  * The write order of the box follows the numbering: along z through the
//    whole chain when the middle row continues from cell to cell, else cell
//    by cell (a reader's numbering gives each cell's new dofs one run).
//
// Cell groups.  Up to Q = 8 every wave takes 64 / Q^2 cells of the chain in
// its own LDS work area with wave-local stage syncs.  At Q = 6 that leaves 28
// of 64 lanes idle, so the workgroup's 4 waves take 7 cells together (252 of
// 256 lanes): affine FP64 K+M at P=5, 97,290 cells, 248 -> 218 us.  At Q = 5
// and 7 (50 and 49 lanes) the same packing was neutral or slower.
//
// Where the numbering does not chain (shuffled cells, cells one after another
// along another axis, plates of one cell) the box would write runs of P and
// single left-face values where the lanes hold runs of N.  A workgroup
// therefore looks at its first two pairs of cells, and if neither shares the
// dof of row (1, 1) every lane adds its values to y as the gathered kernel's
// do: FP32 mass P=7, local axes rotated, 213 -> 56 us, P=3, shuffled, 196 ->
// 114.  The dofs wait in the box's place: held in registers they took 1-2
// waves per SIMD from many shapes.
//
// Measured (MI355X, overwriting applies with the clear of y, 3e6 dofs, us, the
// gathered kernel of apply_kernel.hpp against this one; cells and dofs
// lexicographic, in reader order, and lexicographic dofs with shuffled cells):
//   FP32 mass P=3          115 /  42   188 /  55   114 / 114
//   FP32 stiffness P=4      96 /  54   141 /  55    94 /  90
//   FP64 mass P=7           66 /  53    89 /  56    70 /  65
//   affine FP64 K+M P=5     89 /  71   120 /  71    89 / 103
//   FP32 mass P=1          299 /  87   298 /  87   622 / 620
#pragma once

#include "cell_chain.hpp"

namespace femtc
{

// Waves of a chain workgroup: 4; 2 where a wave holds 7 or 16 cells and two
// already make long rows (affine FP64 stiffness P=2, 1.6e7 dofs: 403 -> 371
// us; mass P=1: 627 -> 557).
template <int Q>
constexpr int chain_waves()
{
  return Q <= 3 ? 2 : 4;
}

template <typename T, int N, int Q, int OP>
struct ChainShape
{
  using Ch = CellChain<T, N, Q, OP>;
  static constexpr int P = N - 1;
  static constexpr int BT = 64 * chain_waves<Q>();
  static constexpr bool PACK = Q == 6;         // cells straddle waves
  static constexpr int GT = PACK ? BT : 64;    // threads of a cell group
  static constexpr int NG = BT / GT;           // groups
  static constexpr int CPB = GT / (Q * Q);     // cells of a group
  static constexpr int S = NG * CPB;           // cells of the chain
  static constexpr int Z = S * P + 1;          // dofs of a box row
  // row (a, b) at a SA + b Z: SA spreads the lanes (a, c) of a store over
  // the LDS banks
  static constexpr int SLOTS = sizeof(T) == 8 ? 32 : 64;
  static constexpr int SA = N * Z + ((N - N * Z) % SLOTS + SLOTS) % SLOTS;
  static constexpr int BOX = N * SA;
  static constexpr int WC = Ch::template wcell<CPB>();
  // geometry of a group in pieces of two elements, in two halves of
  // qa-planes [0, QA1) and [QA1, Q)
  static constexpr int QA1 = geometry_split<Q>();
  static constexpr int GP0 = Ch::GEO ? 3 * QA1 * Q * Q * CPB : 0;
  static constexpr int GP1 = Ch::GEO ? 3 * (Q - QA1) * Q * Q * CPB : 0;
  static constexpr int GPT0 = (GP0 + GT - 1) / GT, GPT1 = (GP1 + GT - 1) / GT;
  static constexpr int WORK = CPB * WC > 2 * GP0 ? CPB * WC : 2 * GP0;
  static constexpr int LDSW = (WORK + 1) / 2; // pieces per group
  static constexpr size_t LDS = sizeof(Piece<T>) * (size_t)NG * LDSW +
                                (sizeof(T) + sizeof(int32_t)) * (size_t)BOX;
  // an unchained workgroup keeps its dofs [b][cell][a][c] in the place of the
  // box and its dofs, and (PACK) its values in the work area
  static_assert((size_t)S * N * N * N * sizeof(int32_t) <=
                    (sizeof(T) + sizeof(int32_t)) * (size_t)BOX,
                "the dofs fit the box");
  static_assert(!PACK || S * N * N * N <= 2 * LDSW,
                "the values fit the work area");
};

template <typename T, int N, int Q, int OP>
__global__ void __launch_bounds__((64 * chain_waves<Q>()))
    chain_cells(const T* __restrict__ tab, const T* __restrict__ x,
                T* __restrict__ y, const T* __restrict__ G,
                const T* __restrict__ detJw, const int32_t* __restrict__ dofmap,
                long long num_cells, int nblk, const int* __restrict__ skip)
{
  if (skip && *skip)
    return;
  using Sh = ChainShape<T, N, Q, OP>;
  using Ch = typename Sh::Ch;
  constexpr int P = N - 1, NN = N * N, N3 = N * NN, Q2 = Q * Q, Q3 = Q2 * Q;
  constexpr int GT = Sh::GT, CPB = Sh::CPB, Z = Sh::Z, SA = Sh::SA;
  extern __shared__ __align__(16) unsigned char femtc_lds_dyn[];
  // contiguous ranges of chains per XCD (workgroups are dealt round-robin):
  // neighbouring chains share x lines and y lines in one L2
  const long long per = (nblk + 7) / 8;
  const long long blk = (long long)(blockIdx.x % 8) * per + blockIdx.x / 8;
  if (blk >= nblk)
    return; // uniform over the workgroup
  const int grp =
      Sh::PACK ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  Piece<T>* Ls = reinterpret_cast<Piece<T>*>(femtc_lds_dyn) + grp * Sh::LDSW;
  T* box = reinterpret_cast<T*>(reinterpret_cast<Piece<T>*>(femtc_lds_dyn) +
                                Sh::NG * Sh::LDSW);
  int32_t* gid = reinterpret_cast<int32_t*>(box + Sh::BOX);
  auto sync = [] {
    if constexpr (Sh::PACK)
      lds_barrier();
    else
      stage_sync<true>();
  };

  // the chain's cells, this group's first one, and this lane's; a lane
  // without a cell repeats the chain's last one and stores nothing
  const long long chain0 = blk * Sh::S;
  const int ncell =
      num_cells - chain0 < Sh::S ? (int)(num_cells - chain0) : Sh::S;
  const int k0 = grp * CPB;
  const int tid = (int)(threadIdx.x & (GT - 1));
  const int lc = tid / Q2, ln = tid - lc * Q2;
  const bool live = lc < CPB && k0 + lc < ncell;
  const int k = live ? k0 + lc : ncell - 1;
  const long long cell = chain0 + k;
  T* Xc = reinterpret_cast<T*>(Ls) + (lc < CPB ? lc : 0) * Sh::WC;
  // thread roles (lanes past a role's lines take its line 0)
  const int ln1 = ln < NN ? ln : 0, ln2 = ln < N * Q ? ln : 0;
  const int r1a = ln1 / N, r1c = ln1 - r1a * N; // F1/B1: (a, c)
  const int r2q = ln2 / N, r2a = ln2 - r2q * N; // F2/B2: (qb, a)
  const int q3b = ln / Q, q3c = ln - q3b * Q;   // F3/B3: (qb, qc)
  const int yo3 = q3b * Ch::YQ + q3c;
  const bool on1 = live && ln < NN, on2 = live && ln < N * Q;
  const int slot0 = r1a * SA + k * P + r1c;

  // the dofs of row (1, 1) on either side of the chain's first two pairs of
  // neighbours (scalar loads; a cell alone is compared with itself)
  int32_t here[2], there[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
  {
    const int kk = i + 1 < ncell ? i + 1 : ncell - 1;
    const int32_t* d = dofmap + (chain0 + kk) * N3 + NN + N;
    here[i] = d[0];
    there[i] = d[ncell > 1 ? P - N3 : 0];
  }

  // ---------------- loads ----------------------------------------------
  typename Ch::Tab tabs;
  tabs.load(tab);
  const int32_t* dm = dofmap + cell * N3 + r1a * NN;
  int32_t idx[N];
#pragma unroll
  for (int b = 0; b < N; ++b)
    idx[b] = dm[r1c + b * N];
  // bit b: (a, b, 0) is not the left neighbour's (a, b, P)
  const bool face = r1c == 0 && k > 0;
  unsigned miss = 0;
  {
    const int off = face ? P - N3 : r1c;
#pragma unroll
    for (int b = 0; b < N; ++b)
      miss |= (dm[off + b * N] != idx[b] ? 1u : 0u) << b;
  }
  T u[N];
#pragma unroll
  for (int b = 0; b < N; ++b)
    u[b] = x[idx[b]];
  Piece<T> gp0[Ch::GEO ? Sh::GPT0 : 1], gp1[Ch::GEO ? Sh::GPT1 : 1];
  if constexpr (Ch::GEO)
  {
    // lane-contiguous pieces of the group's cells, as they are laid out in
    // LDS: [cell][plane][qb][qc][6]
    const int left = ncell - 1 - k0; // last cell, from the group's first
#pragma unroll
    for (int h = 0; h < 2; ++h)
    {
      const int pc = 3 * (h ? Q - Sh::QA1 : Sh::QA1) * Q2; // pieces per cell
      const int tot = h ? Sh::GP1 : Sh::GP0;
      const T* Gh = G + (chain0 + k0) * 6 * Q3 + (h ? 6 * Sh::QA1 * Q2 : 0);
#pragma unroll
      for (int i = 0; i < (h ? Sh::GPT1 : Sh::GPT0); ++i)
      {
        int p = i * GT + tid;
        if (GT * (i + 1) > tot)
          p = p < tot ? p : tot - 1;
        const int c = CPB > 1 ? (int)((unsigned)p / (unsigned)pc) : 0;
        const int r = p - c * pc;
        const Piece<T>* src = reinterpret_cast<const Piece<T>*>(
            Gh + (long long)(c < left ? c : left) * 6 * Q3);
        (h ? gp1[i] : gp0[i]) = stream_load(src + r);
      }
    }
  }
  T cg[Ch::AFF ? CELLGEO : 1];
  T wbc = T(1);
  if constexpr (Ch::AFF)
  {
#pragma unroll
    for (int i = 0; i < CELLGEO; ++i)
      cg[i] = G[cell * CELLGEO + i];
    wbc = tab[Ch::WOFF + q3b] * tab[Ch::WOFF + q3c];
  }
  T dw[Ch::MASSTERM ? Q : 1];
  if constexpr (Ch::MASSTERM && !Ch::AFF)
  {
    const T* Dp = detJw + cell * Q3 + ln;
#pragma unroll
    for (int q = 0; q < Q; ++q)
      dw[q] = stream_load(Dp + q * Q2);
  }
  // Whether the numbering chains here.  Looked at only now: a wait for the
  // scalar loads before the gather of x cost 10 % at P=1.
  __builtin_amdgcn_sched_barrier(0);
  const bool chained = here[0] == there[0] || here[1] == there[1];
  // The line's dofs: to the box's slots, or to the lane's own place.  Packed
  // cells branch, the others choose the address, each the faster by up to 6 %:
  // affine FP64 K+M P=5, 97,290 cells, 242 us against 252; FP32 mass P=1, Q=4.
  int32_t* own = reinterpret_cast<int32_t*>(box) + k * NN + ln1;
  int32_t* ids = chained || Sh::PACK ? gid + slot0 : own;
  const int idstep = chained || Sh::PACK ? Z : Sh::S * NN;
  if (!chained)
    miss = 0;
  if (Sh::PACK && !chained)
  {
    if (on1)
    {
#pragma unroll
      for (int b = 0; b < N; ++b)
        own[b * (Sh::S * NN)] = idx[b];
    }
  }
  else if (on1)
  {
#pragma unroll
    for (int b = 0; b < N; ++b)
      if (!((miss >> b) & 1u))
        ids[b * idstep] = idx[b];
  }

  // ---------------- the cells' contraction chain ------------------------
  Ch::f1(tabs, u, Xc, r1a, r1c, on1);
  sync();
  T bpp[Q], bpg[Q], bgp[Q];
  Ch::f2(tabs, Xc, r2q, r2a, bpp, bpg, bgp);
  sync(); // X is read; Y overwrites the same LDS
  Ch::f2_store(Xc, r2q, r2a, on2, bpp, bpg, bgp);
  sync();
  T ipp[N], ipg[N], igp[N];
  Ch::f3_load(Xc, yo3, ipp, ipg, igp);
  sync();
  if constexpr (Ch::GEO)
  {
#pragma unroll
    for (int i = 0; i < Sh::GPT0; ++i)
      if (i * GT + tid < Sh::GP0)
        Ls[i * GT + tid] = gp0[i];
    sync();
  }
  T uq[Q], da[Q], db[Q], dc[Q];
  Ch::f3(tabs, ipp, ipg, igp, uq, da, db, dc);
  T va[Q], vb[Q], vc[Q], vm[Q];
  auto point = [&](int q, int qa0, int planes) {
    T g[6];
    T dwq = T(0), w = T(0);
    if constexpr (Ch::GEO)
    {
      const Piece<T>* Lg = Ls + (lc < CPB ? lc : 0) * 3 * planes * Q2 +
                           ((q - qa0) * Q2 + ln) * 3;
#pragma unroll
      for (int j = 0; j < 3; ++j)
      {
        const Piece<T> pc = Lg[j];
        g[2 * j] = pc.x;
        g[2 * j + 1] = pc.y;
      }
    }
    if constexpr (Ch::AFF)
      w = tab[Ch::WOFF + q] * wbc;
    else if constexpr (Ch::MASSTERM)
      dwq = dw[q];
    Ch::point(q, g, dwq, cg, w, uq, da, db, dc, va, vb, vc, vm);
  };
#pragma unroll
  for (int q = 0; q < Sh::QA1; ++q)
    point(q, 0, Sh::QA1);
  if constexpr (Ch::GEO)
  {
    sync();
#pragma unroll
    for (int i = 0; i < Sh::GPT1; ++i)
      if (i * GT + tid < Sh::GP1)
        Ls[i * GT + tid] = gp1[i];
    sync();
  }
#pragma unroll
  for (int q = Sh::QA1; q < Q; ++q)
    point(q, Sh::QA1, Q - Sh::QA1);
  T ra_[N], rb_[N], rc_[N];
  Ch::b3(tabs, va, vb, vc, vm, ra_, rb_, rc_);
  if constexpr (Ch::GEO)
    sync(); // the geometry in LDS is consumed; Y may be rewritten
  Ch::b3_store(Xc, yo3, live, ra_, rb_, rc_);
  sync();
  T ra[Q], rb[Q], rc[Q];
  Ch::b2_load(Xc, r2q, r2a, ra, rb, rc);
  sync(); // Y is read; X overwrites the same LDS
  Ch::b2(tabs, ra, rb, rc, Xc, r2q, r2a, on2);
  sync();
  T w[N];
  Ch::b1(tabs, Xc, r1a, r1c, w);

  // ---------------- the chain's box, then y ------------------------------
  if (!chained)
  {
    // nothing to merge: every value from its lane, the N^2 lines of a cell in
    // one instruction (packed cells straddle the waves and change lanes for
    // that: FP32 mass P=4, Q=6, local axes rotated, 107 -> 86 us)
    if constexpr (Sh::PACK)
    {
      lds_barrier(); // X is read
      T* val = reinterpret_cast<T*>(Ls);
      int tt = threadIdx.x; // not kept from above through the contractions
      asm volatile("" : "+v"(tt));
      const int c1 = tt / Q2, l1 = tt - c1 * Q2;
      if (c1 < ncell && l1 < NN)
      {
#pragma unroll
        for (int b = 0; b < N; ++b)
          val[(b * Sh::S + c1) * NN + l1] = w[b];
      }
      lds_barrier();
      const int l = (int)(threadIdx.x & 63);
      for (int c = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
           c < ncell; c += Sh::BT / 64)
        if (l < NN)
        {
#pragma unroll
          for (int b = 0; b < N; ++b)
          {
            const int o = (b * Sh::S + c) * NN + l;
            atomic_add(y + reinterpret_cast<int32_t*>(box)[o], val[o]);
          }
        }
    }
    else if (on1)
    {
      int32_t id[N];
#pragma unroll
      for (int b = 0; b < N; ++b)
        id[b] = own[b * (Sh::S * NN)];
#pragma unroll
      for (int b = 0; b < N; ++b)
        atomic_add(y + id[b], w[b]);
    }
    return; // uniform over the workgroup
  }
  if (on1 && !face)
  {
#pragma unroll
    for (int b = 0; b < N; ++b)
      box[slot0 + b * Z] = w[b];
  }
  lds_barrier();
  if (on1 && face)
  {
#pragma unroll
    for (int b = 0; b < N; ++b)
    {
      if ((miss >> b) & 1u)
        atomic_add(y + dm[b * N], w[b]);
      else
        box[slot0 + b * Z] += w[b];
    }
  }
  lds_barrier();
  const int zlen = ncell * P + 1;
  const int mid = SA + Z; // row (1, 1)
  const bool along_z = ncell < 2 || gid[mid + P + 1] == gid[mid + P] + 1;
  for (int i = threadIdx.x; i < NN * Z; i += Sh::BT)
  {
    int ab, z;
    if (along_z)
    {
      ab = i / Z;
      z = i - ab * Z;
    }
    else if (i < NN)
    {
      ab = i; // the first cell's left face
      z = 0;
    }
    else
    {
      const int j = i - NN;
      const int kc = j / (NN * P), r = j - kc * (NN * P);
      ab = r / P;
      z = kc * P + 1 + (r - ab * P);
    }
    const int a = ab / N;
    const int s = a * SA + (ab - a * N) * Z + z;
    if (z < zlen)
      atomic_add(y + gid[s], box[s]);
  }
}

template <typename T, int N, int Q, int OP>
int launch_chain(const ApplyReq& r)
{
  if constexpr (!chain_pays(OP, sizeof(T) == 8, N, Q))
    return FEMTC_ERR_INVALID_ARGUMENT;
  else
  {
    using Sh = ChainShape<T, N, Q, OP>;
    if (!r.gather || r.reference_mode || r.energy)
      return FEMTC_ERR_INVALID_ARGUMENT;
    const long long nblk = (r.num_cells + Sh::S - 1) / Sh::S;
    if (nblk == 0)
      return FEMTC_OK;
    if (nblk > 0x7ffffff0LL)
      return FEMTC_ERR_INVALID_ARGUMENT;
    static_assert(Sh::LDS <= 64 * 1024, "chain workgroup LDS");
    hipLaunchKernelGGL((chain_cells<T, N, Q, OP>),
                       dim3((unsigned)(8 * ((nblk + 7) / 8))), dim3(Sh::BT),
                       Sh::LDS, r.stream, (const T*)r.tab, (const T*)r.x,
                       (T*)r.y, (const T*)r.G, (const T*)r.detJw, r.dofmap,
                       (long long)r.num_cells, (int)nblk, r.skip);
    return hip_status(hipGetLastError());
  }
}

template <typename T, int N, int Q>
int chain_op(const ApplyReq& r)
{
  switch (r.op)
  {
  case OP_MASS: return launch_chain<T, N, Q, OP_MASS>(r);
  case OP_STIFF: return launch_chain<T, N, Q, OP_STIFF>(r);
  case OP_KPM: return launch_chain<T, N, Q, OP_KPM>(r);
  case OP_MASS_AFF: return launch_chain<T, N, Q, OP_MASS_AFF>(r);
  case OP_STIFF_AFF: return launch_chain<T, N, Q, OP_STIFF_AFF>(r);
  case OP_KPM_AFF: return launch_chain<T, N, Q, OP_KPM_AFF>(r);
  }
  return FEMTC_ERR_INVALID_ARGUMENT;
}

template <int N, int Q>
int chain_dtype(const ApplyReq& r)
{
  return r.dtype == FEMTC_F64 ? chain_op<double, N, Q>(r)
                              : chain_op<float, N, Q>(r);
}

// Q in {N, N+1, N+2}
template <int N>
int chain_q(const ApplyReq& r)
{
  switch (r.Q - N)
  {
  case 0: return chain_dtype<N, N>(r);
  case 1: return chain_dtype<N, N + 1>(r);
  case 2: return chain_dtype<N, N + 2>(r);
  }
  return FEMTC_ERR_INVALID_ARGUMENT;
}

} // namespace femtc
