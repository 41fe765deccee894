// CG of systems whose iterations are bound by launches and latency, not by
// memory: the loop of spmv::cg (spmv/cg.cpp:50-80) in one workgroup (cg_tiny),
// or in two kernels per iteration (cg_direction, cg_residual).
#pragma once

#include "handles.hpp"

namespace spmvx
{

// ---------------------------------------------------------------- sums
// Sum of v over the 64 lanes by DPP moves (a shuffle through LDS costs several
// times their latency), in all lanes; fixed order.
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_move(float v)
{
  return __uint_as_float(static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
      0, static_cast<int>(__float_as_uint(v)), CTRL, ROWS, 0xF, false)));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_move(double v)
{
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(u), CTRL, ROWS, 0xF, false));
  const uint32_t hi = static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), CTRL, ROWS, 0xF, false));
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}
__device__ __forceinline__ float lane_value(float v, int lane)
{
  return __uint_as_float(static_cast<uint32_t>(
      __builtin_amdgcn_readlane(static_cast<int>(__float_as_uint(v)), lane)));
}
__device__ __forceinline__ double lane_value(double v, int lane)
{
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u), lane));
  const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(u >> 32), lane));
  return __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
}
// Lanes 15 (31, 47, 63) get the sum of their row of 16.
template <typename T>
__device__ __forceinline__ T row_sums(T v)
{
  v += dpp_move<0x111, 0xF>(v); // row_shr:1
  v += dpp_move<0x112, 0xF>(v); // row_shr:2
  v += dpp_move<0x114, 0xF>(v); // row_shr:4
  v += dpp_move<0x118, 0xF>(v); // row_shr:8
  return v;
}
template <typename T>
__device__ __forceinline__ T wave_total(T v)
{
  v = row_sums(v);
  return (lane_value(v, 15) + lane_value(v, 31)) + (lane_value(v, 47) + lane_value(v, 63));
}

// Sum of v over a workgroup of NW <= 16 wavefronts, in all threads; `red` (16
// values of LDS) is not used by another sum whose readers may still be on
// their way, so one barrier is enough.
template <int NW, typename T>
__device__ __forceinline__ T group_total(T v, T* red)
{
  v = wave_total(v);
  const int lane = threadIdx.x & 63;
  if (lane == 0)
    red[threadIdx.x >> 6] = v;
  lds_barrier();
  T s = lane < NW ? red[lane] : T(0);
  return lane_value(row_sums(s), 15);
}

// Sum of n partials by every workgroup for itself (blockDim.x = BS): each
// thread's loads all in flight, fixed order, valid in all threads.
template <int BS, int U = 4, typename Acc>
__device__ __forceinline__ Acc partials_sum(const Acc* __restrict__ part, int32_t n, Acc* red)
{
  Acc s0 = Acc(0), s1 = Acc(0);
  for (int32_t i = threadIdx.x; i < n; i += U * BS)
  {
    Acc v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = i + u * BS < n ? part[i + u * BS] : Acc(0);
#pragma unroll
    for (int u = 0; u < U; u += 2)
    {
      s0 += v[u];
      s1 += v[u + 1];
    }
  }
  return group_total<BS / 64>(s0 + s1, red);
}

// ---------------------------------------------------------------- one workgroup
// The whole solve in one workgroup: p in LDS, r and x of a thread's RPT rows and
// the matrix in registers (KW entries per row, columns as 16-bit LDS slots, two
// to a register; entries a row does not have are zeros times a zero slot behind
// p).  An iteration is a product out of LDS and two workgroup sums, with no
// launch and no memory round trip.
// At most kTinySlice iterations per launch (r, p and x go through memory between
// launches), so that a solve that does not converge never holds the GPU for
// long.
// Bound by the latency of its sums and divisions and by one CU's LDS gathers.
// FP64 us per iteration, here and in the five kernels of larger systems: 5-point
// 16^2 0.9 and 12.1, 64^2 2.0 and 13.9; 7-point 16^3 3.1 and 13.7; 27-point 10^3 1.7
// and 14.0.
constexpr int kTinyBS = 512;
constexpr int32_t kTinyRows = 8 * kTinyBS;
constexpr int32_t kTinySlice = 2048;
// Widest row kept in registers with RPT rows per thread (56 entries: 140 of a
// thread's 256 registers in FP64, with 8 rows another 64 for their state).
constexpr int tiny_width(int rpt) { return 56 / rpt; }

template <typename V, typename X, typename Acc, int RPT, int KW>
__global__ __launch_bounds__(kTinyBS) void cg_tiny(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ colidx,
    const V* __restrict__ val, int32_t n, const X* __restrict__ b, X* __restrict__ x,
    X* __restrict__ r, X* __restrict__ p, CgState<Acc>* st, Acc* __restrict__ hist, int32_t first,
    int32_t kmax, Acc rtol2)
{
  extern __shared__ __align__(16) char tiny_lds[];
  X* lp = reinterpret_cast<X*>(tiny_lds); // p of all rows, then a zero
  __shared__ Acc red[3][16];
  constexpr int NW = kTinyBS / 64;
  const int t = threadIdx.x;
  X rv[RPT], xv[RPT];
  constexpr int KC = (KW + 1) / 2;
  V av[RPT][KW];
  uint32_t ac[RPT][KC];
  Acc part = Acc(0);
#pragma unroll
  for (int j = 0; j < RPT; ++j)
  {
    const int32_t i = t + j * kTinyBS;
    const bool in = i < n;
    const int32_t ra = in ? rowptr[i] : 0, re = in ? rowptr[i + 1] : 0;
    rv[j] = in ? (first ? b[i] : r[i]) : X(0);
    xv[j] = in && !first ? x[i] : X(0);
    if (in)
      lp[i] = first ? rv[j] : p[i];
    part += static_cast<Acc>(rv[j]) * static_cast<Acc>(rv[j]);
#pragma unroll
    for (int u = 0; u < KC; ++u)
      ac[j][u] = 0;
#pragma unroll
    for (int u = 0; u < KW; ++u)
    {
      const bool on = ra + u < re;
      av[j][u] = on ? val[ra + u] : V{};
      const uint32_t c = static_cast<uint32_t>(on ? colidx[ra + u] : n);
      ac[j][u / 2] |= c << (16 * (u & 1));
    }
  }
  if (t == 0)
    lp[n] = X(0);
  Acc rr, rr0;
  int32_t k;
  bool converged = false, stopped;
  if (first)
  {
    rr = rr0 = group_total<NW>(part, red[2]);
    k = 0;
    stopped = kmax <= 0;
    if (t == 0 && hist)
      hist[0] = rr;
  }
  else
  {
    rr = st->rnorm_old;
    rr0 = st->rnorm0;
    k = st->k;
    stopped = st->stopped != 0;
    lds_barrier(); // p complete
  }
  for (int32_t done = 0; done < kTinySlice && !stopped; ++done)
  {
    // y = A p (cg.cpp:56), every row in stored order
    X yv[RPT];
    Acc s[RPT];
    Acc pdy = Acc(0);
#pragma unroll
    for (int j = 0; j < RPT; ++j)
      s[j] = Acc(0);
#pragma unroll
    for (int u = 0; u < KW; ++u)
    {
      // (8 gathers in flight: more would not fit the registers)
      if (u % (8 / RPT) == 0)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < RPT; ++j)
        s[j] += static_cast<Acc>(widen(av[j][u]))
                * static_cast<Acc>(lp[(ac[j][u / 2] >> (16 * (u & 1))) & 0xFFFFu]);
    }
#pragma unroll
    for (int j = 0; j < RPT; ++j)
    {
      // (the zero slot past the last row)
      const int32_t i = t + j * kTinyBS;
      yv[j] = static_cast<X>(s[j]);
      pdy += static_cast<Acc>(lp[i < n ? i : n]) * static_cast<Acc>(yv[j]);
    }
    // (the sum's barrier: every thread has read p)
    const Acc alpha = rr / group_total<NW>(pdy, red[0]); // cg.cpp:61-62
    const X al = static_cast<X>(alpha);
    Acc rn = Acc(0);
#pragma unroll
    for (int j = 0; j < RPT; ++j)
    {
      const int32_t i = t + j * kTinyBS;
      xv[j] = xv[j] + al * lp[i < n ? i : n];
      rv[j] = rv[j] - al * yv[j];
      rn += static_cast<Acc>(rv[j]) * static_cast<Acc>(rv[j]);
    }
    // Past the last row an infinite alpha has made a NaN of 0 - alpha 0.  It shows in the
    // history alone (alpha is NaN in the next step either way, and x and r with it): without
    // one the test is left out (1.6% of the solve, 5-point 64^2).
    if (hist && !(alpha - alpha == Acc(0)))
    {
      rn = Acc(0);
#pragma unroll
      for (int j = 0; j < RPT; ++j)
        rn += t + j * kTinyBS < n ? static_cast<Acc>(rv[j]) * static_cast<Acc>(rv[j]) : Acc(0);
    }
    rn = group_total<NW>(rn, red[1]);
    const X be = static_cast<X>(rn / rr);
    rr = rn;
    ++k;
    if (t == 0 && hist)
      hist[k] = rr;
    converged = rr / rr0 < rtol2; // cg.cpp:79
    stopped = converged || k >= kmax;
#pragma unroll
    for (int j = 0; j < RPT; ++j)
    {
      const int32_t i = t + j * kTinyBS;
      if (i < n)
        lp[i] = lp[i] * be + rv[j]; // cg.cpp:76
    }
    lds_barrier();
  }
#pragma unroll
  for (int j = 0; j < RPT; ++j)
  {
    const int32_t i = t + j * kTinyBS;
    if (i < n)
    {
      x[i] = xv[j];
      r[i] = rv[j];
      p[i] = lp[i];
    }
  }
  if (t == 0)
  {
    st->rnorm0 = rr0;
    st->rnorm_old = rr;
    st->k = k;
    st->converged = converged ? 1 : 0;
    st->stopped = stopped ? 1 : 0;
  }
}

// Rows per thread of cg_tiny for n rows.
inline int tiny_rows(int64_t n)
{
  return n <= kTinyBS ? 1 : (n <= 2 * kTinyBS ? 2 : (n <= 4 * kTinyBS ? 4 : 8));
}
inline bool cg_is_tiny(const Pattern& P)
{
  return P.nrows > 0 && P.nrows <= kTinyRows && P.nrows == P.ncols
         && P.longest <= tiny_width(tiny_rows(P.nrows));
}

// Launches a slice of the solve on s.
template <typename V, typename X, typename Acc>
void launch_cg_tiny(const Pattern& P, hipStream_t s, const V* val, const X* b, X* x, X* r, X* p,
                    CgState<Acc>* st, Acc* hist, bool first, int32_t kmax, Acc rtol2)
{
  const int32_t n = static_cast<int32_t>(P.nrows);
  const uint32_t lds = static_cast<uint32_t>(sizeof(X)) * static_cast<uint32_t>(n + 1);
  using std::integral_constant;
  auto run = [&](auto rpt, auto kw) {
    cg_tiny<V, X, Acc, decltype(rpt)::value, decltype(kw)::value><<<1, kTinyBS, lds, s>>>(
        P.rowptr.as<int32_t>(), P.colidx.as<int32_t>(), val, n, b, x, r, p, st, hist, first ? 1 : 0,
        kmax, rtol2);
  };
  // the narrowest compiled width that holds the longest row
  auto width = [&](auto rpt, auto k1, auto k2, auto k3) {
    if (P.longest <= decltype(k1)::value)
      run(rpt, k1);
    else if (P.longest <= decltype(k2)::value)
      run(rpt, k2);
    else
      run(rpt, k3);
  };
  switch (tiny_rows(n))
  {
  case 1:
    width(integral_constant<int, 1>{}, integral_constant<int, 7>{}, integral_constant<int, 27>{},
          integral_constant<int, tiny_width(1)>{});
    break;
  case 2:
    width(integral_constant<int, 2>{}, integral_constant<int, 5>{}, integral_constant<int, 9>{},
          integral_constant<int, tiny_width(2)>{});
    break;
  case 4:
    width(integral_constant<int, 4>{}, integral_constant<int, 5>{}, integral_constant<int, 7>{},
          integral_constant<int, tiny_width(4)>{});
    break;
  default:
    width(integral_constant<int, 8>{}, integral_constant<int, 3>{}, integral_constant<int, 5>{},
          integral_constant<int, tiny_width(8)>{});
    break;
  }
  check_launch("cg_tiny");
}

// ---------------------------------------------------------------- two kernels per iteration
// State of an iteration.  Iteration j (from 1) has slot j & 1: cg_direction
// reads the other slot (iteration j - 1) and writes this one, cg_residual adds
// alpha, so that no kernel reads what a workgroup of the same launch writes.
template <typename Acc>
struct CgSlot
{
  Acc rr;          // ||r_{j-1}||^2
  Acc alpha;       // of iteration j
  int32_t k;       // iterations completed before j; -1: nothing yet
  int32_t stopped; // no iteration j: x is final
};

constexpr int kSmallBS = 256;

// x = 0, r = b, p = 0, partial ||b||^2
template <typename X, typename Acc>
__global__ __launch_bounds__(kSmallBS) void cg_small_init(int64_t n, const X* __restrict__ b,
                                                          X* __restrict__ x, X* __restrict__ r,
                                                          X* __restrict__ p,
                                                          Acc* __restrict__ partials,
                                                          CgSlot<Acc>* slot)
{
  __shared__ Acc red[16];
  Acc part = Acc(0);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * kSmallBS;
  for (int64_t i = blockIdx.x * static_cast<int64_t>(kSmallBS) + threadIdx.x; i < n; i += stride)
  {
    const X bi = b[i];
    x[i] = X(0);
    r[i] = bi;
    p[i] = X(0);
    part += static_cast<Acc>(bi) * static_cast<Acc>(bi);
  }
  part = block_sum(part, red);
  if (threadIdx.x == 0)
  {
    partials[blockIdx.x] = part;
    if (blockIdx.x == 0)
      *slot = CgSlot<Acc>{Acc(0), Acc(0), -1, 0};
  }
}

// Iteration j, first kernel: completes iteration j - 1 (||r||^2 from its npr
// partials, convergence, x += alpha p), forms the new direction q = beta p + r
// and its product y = A q, partial q.y.  One lane per row; the direction of a
// row's columns is formed again by every row that needs it (the same two
// operations, so the same value), which saves a kernel per iteration.  KR > 0:
// columns from the row masks over KR offsets (see csr_wave), so that the gathers
// need not wait for indices; KR = 0: from colidx.
template <typename V, typename X, typename Acc, int KR>
__global__ __launch_bounds__(kSmallBS) void cg_direction(
    const int32_t* __restrict__ rowptr, const int32_t* __restrict__ colidx,
    const int32_t* __restrict__ masks, const int32_t* __restrict__ offs,
    const V* __restrict__ val, int32_t n, const X* __restrict__ r, const X* __restrict__ p,
    X* __restrict__ q, X* __restrict__ x, X* __restrict__ y, const Acc* __restrict__ part_r,
    int32_t npr, Acc* __restrict__ part_s, CgState<Acc>* st, const CgSlot<Acc>* prev,
    CgSlot<Acc>* cur, Acc* __restrict__ hist)
{
  __shared__ Acc red[2][16];
  const CgSlot<Acc> in = *prev;
  const int64_t nblk = (n + kSmallBS - 1) / kSmallBS;
  const int64_t blk = xcd_block(blockIdx.x, nblk);
  const int32_t row = static_cast<int32_t>(blk) * kSmallBS + static_cast<int32_t>(threadIdx.x);
  const bool has = row < n;
  if (in.stopped)
  {
    if (blockIdx.x == 0 && threadIdx.x == 0)
      *cur = in;
    return;
  }
  // everything that does not depend on the sum below is requested before it
  constexpr int U = KR == 0 ? 4 : KR;
  const int32_t ra = has ? rowptr[row] : 0, re = has ? rowptr[row + 1] : 0;
  X rc[U], pc[U];
  V a[U];
  uint32_t mask = 0;
  auto request = [&](int32_t e) {
    if constexpr (KR == 0)
    {
      int32_t c[U];
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        const int32_t k = e + u < re ? e + u : (re > ra ? re - 1 : -1);
        c[u] = k >= 0 ? colidx[k] : 0;
        a[u] = k >= 0 ? val[k] : V{};
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        rc[u] = r[c[u]];
        pc[u] = p[c[u]];
      }
    }
    else
    {
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        // an entry the row does not have: its own row and first value instead
        const bool on = (mask >> u) & 1;
        const int32_t c = on ? row + offs[u] : (has ? row : 0);
        rc[u] = r[c];
        pc[u] = p[c];
        a[u] = val[e]; // padded past the last entry
        e += on ? 1 : 0;
      }
    }
  };
  if constexpr (KR > 0)
    mask = has ? static_cast<uint32_t>(masks[row]) : 0u;
  const X xi = has ? x[row] : X(0), pi = has ? p[row] : X(0), ri = has ? r[row] : X(0);
  request(ra);
  const Acc rr = partials_sum<kSmallBS>(part_r, npr, red[0]); // cg.cpp:69
  const int32_t k = in.k + 1;
  const bool first = k == 0;
  const Acc rr0 = first ? rr : st->rnorm0;
  const bool converged = !first && rr / rr0 < st->rtol2; // cg.cpp:79
  const bool stop = converged || k >= st->kmax;
  const X beta = first ? X(0) : static_cast<X>(rr / in.rr); // cg.cpp:70
  if (blockIdx.x == 0 && threadIdx.x == 0)
  {
    *cur = CgSlot<Acc>{rr, Acc(0), k, stop ? 1 : 0};
    if (first)
      st->rnorm0 = rr;
    if (hist)
      hist[k] = rr;
  }
  if (has && !first)
    x[row] = xi + static_cast<X>(in.alpha) * pi; // cg.cpp:65
  if (stop)
    return;
  const X qi = pi * beta + ri; // cg.cpp:76
  if (has)
    q[row] = qi;
  Acc s = Acc(0);
  if constexpr (KR > 0)
  {
#pragma unroll
    for (int u = 0; u < U; ++u)
    {
      const X d = pc[u] * beta + rc[u];
      const Acc t = static_cast<Acc>(widen(a[u])) * static_cast<Acc>(d);
      s = (mask >> u) & 1 ? s + t : s;
    }
  }
  else
    for (int32_t e = ra;;)
    {
#pragma unroll
      for (int u = 0; u < U; ++u)
      {
        const X d = pc[u] * beta + rc[u];
        const Acc t = static_cast<Acc>(widen(a[u])) * static_cast<Acc>(d);
        s = e + u < re ? s + t : s;
      }
      e += U;
      if (e >= re)
        break;
      request(e);
    }
  const X yi = static_cast<X>(s);
  if (has)
    y[row] = yi;
  const Acc part =
      group_total<kSmallBS / 64>(has ? static_cast<Acc>(qi) * static_cast<Acc>(yi) : Acc(0), red[1]);
  if (threadIdx.x == 0)
    part_s[blk] = part;
}

// Iteration j, second kernel: alpha = rr / (q.y) from the nps partials,
// r -= alpha y, partial ||r||^2 (cg.cpp:61-69).
template <typename X, typename Acc>
__global__ __launch_bounds__(kSmallBS) void cg_residual(int32_t n, X* __restrict__ r,
                                                        const X* __restrict__ y,
                                                        const Acc* __restrict__ part_s,
                                                        int32_t nps, Acc* __restrict__ part_r,
                                                        CgSlot<Acc>* cur)
{
  __shared__ Acc red[2][16];
  if (cur->stopped)
    return;
  const Acc rr = cur->rr;
  const int64_t nblk = (n + 2 * kSmallBS - 1) / (2 * kSmallBS);
  const int32_t blk = static_cast<int32_t>(xcd_block(blockIdx.x, nblk));
  const int32_t i0 = blk * 2 * kSmallBS + static_cast<int32_t>(threadIdx.x), i1 = i0 + kSmallBS;
  X ra = i0 < n ? r[i0] : X(0), rb = i1 < n ? r[i1] : X(0);
  const X ya = i0 < n ? y[i0] : X(0), yb = i1 < n ? y[i1] : X(0);
  const Acc alpha = rr / partials_sum<kSmallBS>(part_s, nps, red[0]);
  const X al = static_cast<X>(alpha);
  ra = ra - al * ya;
  rb = rb - al * yb;
  if (i0 < n)
    r[i0] = ra;
  if (i1 < n)
    r[i1] = rb;
  Acc part = static_cast<Acc>(ra) * static_cast<Acc>(ra);
  part += i1 < n ? static_cast<Acc>(rb) * static_cast<Acc>(rb) : Acc(0);
  part = group_total<kSmallBS / 64>(i0 < n ? part : Acc(0), red[1]);
  if (threadIdx.x == 0)
  {
    part_r[blk] = part;
    if (blockIdx.x == 0)
      cur->alpha = alpha;
  }
}

// Systems the two-kernel iteration takes: those where its fewer launches gain
// more than its second gather per entry and its uncoalesced values cost.  FP64
// us per iteration, two kernels and five: masks, 5-point 256^2 7.4 and 15.0, 512^2
// 10.3 and 17.4, 1024^2 (5.2M entries) 31.7 and 36.1, 1448^2 (10.5M) 67 and 54; 7-point
// 100^3 (6.9M) 36.5 and 39.6; 27-point 32^3 (0.8M) 11.0 and 15.4, 48^3 (2.9M) 19.1 and
// 17.9.  Irregular rows (power law of 3-64 entries), from colidx: 4000 rows 16.7 and
// 18.4, 30000 (0.29M) 18.6 and 21.4, 100000 (0.96M) 25.3 and 24.9.
constexpr int64_t kSmallRows = 1024 * 1024;
constexpr int32_t kSmallWidth = 64;
// By size alone: what decides about the workspace, which must not change while the
// masks of a shared pattern are being built.
inline bool cg_may_be_small(const Pattern& P)
{
  return P.nrows > 0 && P.nrows <= kSmallRows && P.nrows == P.ncols;
}

// How a solve iterates: in one workgroup, in two kernels (over the row masks of KR
// offsets, 0: from colidx), or neither.  Taken once per solve, under the pattern's
// lock: another thread may be building the masks for another matrix of the pattern.
struct CgForm
{
  bool tiny = false, small = false;
  int kr = 0;
};
inline CgForm cg_form(Pattern& P, bool alone)
{
  CgForm f;
  if (!alone)
    return f;
  f.tiny = cg_is_tiny(P);
  if (f.tiny || !cg_may_be_small(P))
    return f;
  std::lock_guard<std::recursive_mutex> lock(P.lazy_mu);
  if (P.masked && P.all_masked)
  {
    f.kr = kWaveClasses[P.wave].kr;
    f.small = P.nnz <= (f.kr <= 9 ? 6000000 : 2000000);
  }
  else
    f.small = P.longest <= kSmallWidth && P.nnz <= 600000;
  return f;
}

inline int small_blocks(int64_t n) { return static_cast<int>((n + kSmallBS - 1) / kSmallBS); }
inline int small_partials(int64_t n)
{
  return static_cast<int>((n + 2 * kSmallBS - 1) / (2 * kSmallBS));
}

// Vectors and partial sums of the two-kernel iteration: p[0] is the direction
// of even iterations and of the start, p[1] of odd ones.
template <typename X, typename Acc>
struct SmallArgs
{
  X *r, *y, *p[2], *x;
  Acc *part_s, *part_r;
  CgState<Acc>* st;
  CgSlot<Acc>* slot; // two
  Acc* hist;
};

// Iteration j (its parity matters) on stream s, in the form f.
template <typename V, typename X, typename Acc>
void launch_small_iteration(const Pattern& P, const CgForm& f, hipStream_t s, const V* val,
                            const SmallArgs<X, Acc>& a, int j)
{
  const int32_t n = static_cast<int32_t>(P.nrows);
  const int par = j & 1;
  auto go = [&](auto kr) {
    cg_direction<V, X, Acc, decltype(kr)::value><<<small_blocks(n), kSmallBS, 0, s>>>(
        P.rowptr.as<int32_t>(), P.colidx.as<int32_t>(), P.wrows.as<int32_t>(),
        P.woffs.as<int32_t>(), val, n, a.r, a.p[par ^ 1], a.p[par], a.x, a.y, a.part_r,
        small_partials(n), a.part_s, a.st, a.slot + (par ^ 1), a.slot + par, a.hist);
  };
  using std::integral_constant;
  switch (f.kr)
  {
  case 3: go(integral_constant<int, 3>{}); break;
  case 5: go(integral_constant<int, 5>{}); break;
  case 7: go(integral_constant<int, 7>{}); break;
  case 9: go(integral_constant<int, 9>{}); break;
  case 15: go(integral_constant<int, 15>{}); break;
  case 27: go(integral_constant<int, 27>{}); break;
  default: go(integral_constant<int, 0>{}); break;
  }
  cg_residual<X, Acc><<<small_partials(n), kSmallBS, 0, s>>>(n, a.r, a.y, a.part_s,
                                                              small_blocks(n), a.part_r,
                                                              a.slot + par);
}

} // namespace spmvx
