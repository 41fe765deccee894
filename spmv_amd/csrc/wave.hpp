// CSR product for matrices whose rows are short and alike (stencils, meshes):
// one wavefront per 64 rows.  Included by kernels.hpp, whose CSR variants run
// it where it suits the matrix (Pattern::wave_class).
#pragma once

namespace spmvx
{

// csr_wave: block b is rows [64 b, 64 b + 64), at most E - 7 - KR entries.  One
// wavefront per workgroup, lane l owns row l of a block, and every wavefront
// walks a strided list of blocks:
//   1  the block's values (and, where needed, 16-bit column indices) have
//      landed in LDS (buffer loads that write LDS directly, no registers);
//   2  the lanes issue all gathers of x (adjacent lanes hold adjacent rows: for
//      stencils the gathers of one entry position are contiguous), then read
//      their rows' values from LDS;
//   3  the next block's values and indices are requested into the same LDS,
//      which is free from here on;
//   4  the products are formed and summed in stored order from 0, rounded
//      separately: bit-identical to csr_stream.
// Loads return in order, so the gathers of step 2, issued before step 3, do
// not wait for the stream, and a wavefront's buffer is being filled while it
// waits for them and sums.  There is no barrier anywhere.
//
// Columns (HM = 0): the 16-bit indices of the block (IM 1 or 2, see csr_stream),
// row extents from rowptr.
// Columns (HM = 1): stencils and structured meshes have one short list of column
// offsets (col - row), of which every row uses some.  Blocks whose rows all do
// store a mask per row over that list instead of indices: 4 bytes per row in
// place of 2 per entry and 4 of rowptr (27-point FP64: 236 instead of 290 bytes
// per row, 7-point FP32 40 instead of 54).  The other blocks keep their 16-bit
// indices, with the row's length in the mask's place; a row's start is the sum
// of the lengths before it.
//
// Results (burst > 0): a product that streams its matrix from HBM loses far more to
// its y stores than their bytes (27-point 160^3: 157 us for the matrix alone,
// 189 with a store per block).  So a wavefront keeps the results of `burst` blocks
// in LDS and stores them together, non-temporal.  Few wavefronts per CU stream
// best then (wave_plan).  burst = 0: every block's results are stored at once,
// for matrices with too few blocks to fill bursts.
//
// Complex values: only matrices whose blocks all have masks (complex_wave).
//
// Bound by HBM.  27-point 160^3, FP64: csr_stream 222 us, here with indices 176,
// with masks 150 (0.97 GB: 6.5 TB/s, a streaming read runs at 7.0).  7-point 256^3:
// FP64 313 to 218 us, FP32 188 to 117, BF16 168 to 89.  Complex FP64, csr_stream's 129
// to 90 us (7-point 160^3), 9.0 to 6.8 (63x65x61), 123 to 67 (27-point 100^3); complex
// FP32, 7-point 160^3, 83 to 51.
constexpr int kWaveRows = 64;

// 1 KiB LDS loads (64 lanes of 16 bytes) that hold n entries of es bytes.
__host__ __device__ constexpr int wave_loads(int n, int es) { return (n * es + 1023) / 1024; }

// Cache bits of a buffer load: allocate as usual, or stream (non-temporal).
constexpr int kLoadKeep = 0, kLoadStream = 2;

// Requests `bytes` bytes (a multiple of 16, at most N KiB) from g (16-byte
// aligned) into LDS; lanes past the end are out of the buffer's range and read
// nothing.  A load's whole distance from g is in the lane's offset: the scalar
// offset of a buffer load takes no part in the range check, and with i KiB there
// the last loads of a short block would read up to N KiB past the arrays.  The caller
// waits (lds_filled): the compiler does not order LDS reads after these loads.
typedef __attribute__((address_space(3))) char* lds_ptr;
template <int N, int AUX>
__device__ __forceinline__ void lds_fill(const char* g, int32_t bytes, lds_ptr lds)
{
  __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(g), 0, bytes, 0x00020000);
  int32_t off = static_cast<int32_t>(threadIdx.x) * 16;
  asm volatile("" : "+v"(off)); // (the sums below are formed here, not kept in N registers)
#pragma unroll
  for (int i = 0; i < N; ++i)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, lds + i * 1024, 16, off + i * 1024, 0, 0, AUX);
}

// Waits for every vector memory operation of this wavefront (the loads of
// lds_fill among them); LDS reads stay behind it.
__device__ __forceinline__ void lds_filled()
{
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Sizes of csr_wave: E entries staged per block, KR entries of a row gathered
// at once, and the wavefronts per CU of a streaming product (B > 0) for 16-, 8-,
// 4- and 2-byte values.  KR are the widths of the 3-, 5-, 7-, 9- and 27-point
// operators and one between; E holds 64 such rows, up to 7 entries before the
// block (aligned loads) and KR entries read past the last row.
// Wavefronts per CU: the best of the counts tried, matrices of the KR's width
// with row masks in HBM (FP64 7-point 256^3 6 / 7 / 9 wavefronts: 223 / 218 / 235 us,
// 27-point 160^3 3 / 4 / 5: 152 / 149 / 163; FP32 7-point 10 / 12 / 16: 123 / 117 /
// 127, 27-point 6 / 8 / 10: 83 / 82 / 85; complex FP64 7-point 160^3 4 / 5 / 6: 92.2 /
// 90.5 / 91.7, 27-point 100^3 2 / 3 / 4: 73 / 67 / 69; complex FP32 stays within 2% of
// its best with FP64's).  Enough loads must be in flight, and
// each further stream costs HBM efficiency: wide rows (more bytes and gathers
// per wavefront) want fewer.
struct WaveClass
{
  int e, kr, per_cu16, per_cu8, per_cu4, per_cu2;
};
#define SPMVX_WAVE_CLASSES(X)                                                                \
  X(0, 256, 3, 10, 12, 20, 20)                                                              \
  X(1, 384, 5, 7, 9, 16, 20)                                                                \
  X(2, 512, 7, 5, 7, 12, 16)                                                                \
  X(3, 640, 9, 4, 7, 12, 12)                                                                \
  X(4, 1024, 15, 3, 4, 8, 12)                                                               \
  X(5, 1792, 27, 3, 4, 8, 12)
constexpr int kNumWaveClasses = 6;
#define SPMVX_WAVE_ENTRY(i, E, K, W16, W8, W4, W2) {E, K, W16, W8, W4, W2},
constexpr WaveClass kWaveClasses[kNumWaveClasses] = {SPMVX_WAVE_CLASSES(SPMVX_WAVE_ENTRY)};
#undef SPMVX_WAVE_ENTRY
// Stored entries that a block of a class may hold.
constexpr int wave_block_nnz(int c) { return kWaveClasses[c].e - 7 - kWaveClasses[c].kr; }

// LDS of a wavefront: the staged values, the 16-bit indices (when any block has
// them), a zero value, the kept results.
struct WaveLds
{
  int col_at, zero_at, kept_at, bytes;
};
constexpr WaveLds wave_lds(int e, int vbytes, int xbytes, bool cols, int burst)
{
  WaveLds L{};
  L.col_at = 1024 * wave_loads(e, vbytes);
  L.zero_at = L.col_at + (cols ? 1024 * wave_loads(e, 2) : 0);
  L.kept_at = L.zero_at + 16;
  L.bytes = L.kept_at + burst * kWaveRows * xbytes;
  return L;
}
// Wavefronts with that much LDS that fit a CU (160 KiB in steps of 1280 bytes,
// at most 32).
constexpr int wave_per_cu(int lds)
{
  return 163840 / ((lds + 1279) / 1280 * 1280) < 32 ? 163840 / ((lds + 1279) / 1280 * 1280) : 32;
}

// Wavefronts per SIMD that the registers must allow: what the LDS allows, as far
// as the KR gathers and values of a lane in flight (and about 48 registers
// beside them) fit.
constexpr int wave_per_simd(int e, int kr, int vbytes, int xbytes, bool cols)
{
  const int lds = (wave_per_cu(wave_lds(e, vbytes, xbytes, cols, 0).bytes) + 3) / 4;
  const int reg = 512 / (kr * xbytes / 2 + 48);
  return lds < reg ? lds : reg;
}

// The element `off` bytes into x, 0 where that is past its `bytes` bytes (nothing
// is read then).
template <typename X>
__device__ __forceinline__ X ld_buffer(const X* x, uint32_t bytes, uint32_t off)
{
  __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<X*>(x), 0, static_cast<int32_t>(bytes), 0x00020000);
  if constexpr (sizeof(X) == 16)
    return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  else if constexpr (sizeof(X) == 8)
    return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  else
    return __builtin_bit_cast(X, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}

// A non-temporal store.
template <typename T>
__host__ __device__ __forceinline__ void store_streamed(T* p, T v)
{
  __builtin_nontemporal_store(v, p);
}
template <typename T>
__host__ __device__ __forceinline__ void store_streamed(cplx<T>* p, cplx<T> v)
{
  store_streamed(&p->re, v.re);
  store_streamed(&p->im, v.im);
}

// This lane's share of storing the results of nkept blocks (first, first + nw, ...) kept
// in LDS, kWaveRows of each: 16 bytes at a time where y allows it.  Lanes past the last
// kept block read nothing: a burst need not fill the blocks of one store.
template <typename X>
__host__ __device__ __forceinline__ void store_burst(const X* kept, int32_t nkept, int32_t first,
                                                     int32_t nw, int32_t nrows, X* y, int lane)
{
  if ((reinterpret_cast<uintptr_t>(y) & 15) == 0)
  {
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    constexpr int N = 16 / sizeof(X), LPB = kWaveRows / N; // per lane; lanes per block
    const int32_t step = kWaveRows / LPB;                  // blocks per store
#pragma unroll 4
    for (int32_t t0 = 0; t0 < nkept; t0 += step)
    {
      const int32_t t = t0 + lane / LPB;
      if (t < nkept)
      {
        const X* k = kept + t0 * kWaveRows + lane * N;
        const int32_t row = (first + t * nw) * kWaveRows + (lane % LPB) * N;
        if (row + N <= nrows)
          __builtin_nontemporal_store(*reinterpret_cast<const u4*>(k),
                                      reinterpret_cast<u4*>(y + row));
        else
          for (int i = 0; row + i < nrows; ++i)
            y[row + i] = k[i];
      }
    }
  }
  else
#pragma unroll 1
    for (int32_t t = 0; t < nkept; ++t)
    {
      const int32_t row = (first + t * nw) * kWaveRows + lane;
      if (row < nrows)
        store_streamed(y + row, kept[t * kWaveRows + lane]);
    }
}

// Sum of v (< 2^BITS) over the lanes below this one.
template <int BITS>
__device__ __forceinline__ int32_t lanes_before(int32_t v)
{
  int32_t s = 0;
#pragma unroll
  for (int j = 0; j < BITS; ++j)
  {
    const uint64_t m = __ballot((v >> j) & 1);
    s += static_cast<int32_t>(__builtin_amdgcn_mbcnt_hi(
             static_cast<uint32_t>(m >> 32),
             __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0)))
         << j;
  }
  return s;
}

// HM = 0: rows is rowptr, blocks holds (first row, first entry).
// HM = 1: rows holds a mask or a length per row, blocks (1 where the block's
// rows have masks, first entry), offs the list of column offsets (KR entries).
template <typename V, typename X, typename Acc, int MODE, int IM, int HM, int E, int KR>
__global__ __launch_bounds__(kWaveRows, wave_per_simd(E, KR, sizeof(V), sizeof(X), HM == 0))
void csr_wave(const int32_t* __restrict__ rows, const int2* __restrict__ blocks,
              const int32_t* __restrict__ offs, const uint16_t* __restrict__ col16,
              const int4* __restrict__ wbase, int32_t nrows, int32_t ncols,
              const V* __restrict__ val, const X* __restrict__ x, X* __restrict__ y,
              const X* __restrict__ b, Acc* __restrict__ partials, const CgState<Acc>* st,
              int32_t it, WaveLds at, int32_t burst, int32_t keep)
{
  if (MODE != kPlain && !cg_live(st, it))
    return;
  constexpr int NV = wave_loads(E, sizeof(V)), NX = wave_loads(E, 2);
  constexpr int AL = 8; // entries: 16 bytes of indices
  constexpr bool ALL = kIsComplex<V>; // every block has masks (complex_wave)
  extern __shared__ __align__(16) char buf[];
  const lds_ptr fill_at = (lds_ptr)buf;
  const V* lval = reinterpret_cast<const V*>(buf);
  const uint16_t* lcol = reinterpret_cast<const uint16_t*>(buf + at.col_at);
  X* kept = reinterpret_cast<X*>(buf + at.kept_at);
  const int32_t zero = at.zero_at / static_cast<int32_t>(sizeof(V)); // slot of a zero value
  const int lane = threadIdx.x;
  // this wavefront's blocks: XCD x (dispatch order modulo 8) walks one
  // contiguous range, its wavefronts side by side in it
  const int32_t nblocks = (nrows + kWaveRows - 1) / kWaveRows;
  const int32_t xcd = blockIdx.x % kNumXcd, j = blockIdx.x / kNumXcd;
  const int32_t nw = (static_cast<int32_t>(gridDim.x) + kNumXcd - 1 - xcd) / kNumXcd;
  const int32_t q = nblocks / kNumXcd, rem = nblocks % kNumXcd;
  int32_t bi = xcd * q + (xcd < rem ? xcd : rem) + j;
  const int32_t bend = bi - j + q + (xcd < rem ? 1 : 0);
  Acc part = Acc(0);
  if (bi < bend)
  {
    if (HM && lane < 4)
      reinterpret_cast<uint32_t*>(buf + at.zero_at)[lane] = 0u;
    // entry range [k0, k1) and kind of the block at hand, its column bases,
    // row extents (HM = 1: mask or length in ra) and x / b entry; idle lanes of
    // the last block hold an empty row
    int32_t k0, k1, kind, ra, re = 0;
    int4 w = make_int4(0, 0, 0, 0);
    X xr = X(0);
    auto load_rows = [&](int32_t blk, int32_t& a, int32_t& e, X& xe) {
      const int32_t row = blk * kWaveRows + lane;
      if constexpr (HM)
        a = ld_stream<true>(rows + row); // padded to whole blocks
      else
      {
        a = ld_stream<true>(rows + (row < nrows ? row : nrows));
        e = ld_stream<true>(rows + (row < nrows ? row + 1 : nrows));
      }
      if constexpr (MODE == kDot)
        xe = x[row < nrows ? row : nrows - 1];
      else if constexpr (MODE == kResid)
        xe = b[row < nrows ? row : nrows - 1];
    };
    int32_t turn = 5 * j; // spreads the kept blocks over wavefronts and time
    auto fill = [&](int32_t a, int32_t e, int32_t masked) {
      const int32_t kb = a & ~(AL - 1);
      const int32_t n = (e - kb + AL - 1) & ~(AL - 1);
      if (!ALL && (!HM || !masked))
        lds_fill<NX, kLoadStream>(reinterpret_cast<const char*>(col16 + kb), n * 2, fill_at + at.col_at);
      const char* g = reinterpret_cast<const char*>(val + kb);
      const int32_t bytes = n * static_cast<int32_t>(sizeof(V));
      if ((turn++ & 31) < keep) // (wave_keep)
        lds_fill<NV, kLoadKeep>(g, bytes, fill_at);
      else
        lds_fill<NV, kLoadStream>(g, bytes, fill_at);
    };
    int32_t of[KR]; // the list of column offsets, as byte offsets into x
#pragma unroll
    for (int k = 0; k < KR; ++k)
      of[k] = HM ? static_cast<int32_t>(static_cast<uint32_t>(offs[k])
                                        * static_cast<uint32_t>(sizeof(X)))
                 : 0;
    kind = blocks[bi].x;
    k0 = blocks[bi].y;
    k1 = blocks[bi + 1].y;
    if constexpr (!ALL)
      w = wbase[bi];
    load_rows(bi, ra, re, xr);
    fill(k0, k1, kind);

    // results waiting to be stored: blocks kfirst, kfirst + nw, ... (burst > 0), or
    // the last block's (burst = 0; behind the next block's gathers: a store issued
    // after the refill would be waited for with it)
    int32_t nkept = 0, kfirst = bi;
    int32_t yrow = -1;
    X yval = X(0);
    auto store_kept = [&]() {
      if (burst > 0)
      {
        store_burst(kept, nkept, kfirst, nw, nrows, y, lane);
        nkept = 0;
      }
      else if (yrow >= 0)
        store_result(y + yrow, yval);
    };

    auto block = [&](auto refill, auto masked, int32_t nb) {
      lds_filled();
      int32_t n0 = 0, n1 = 0, nkind = 0;
      int4 nwb = w;
      if constexpr (refill.value)
      {
        nkind = blocks[nb].x;
        n0 = blocks[nb].y;
        n1 = blocks[nb + 1].y;
        if constexpr (!ALL)
          nwb = wbase[nb];
      }
      // row's first entry in LDS and its length
      int32_t pos, len;
      if constexpr (masked.value)
      {
        len = __popc(ra);
        pos = k0 % AL + lanes_before<5>(len);
      }
      else if constexpr (HM)
      {
        len = ra;
        pos = k0 % AL + lanes_before<11>(len);
      }
      else
      {
        len = re - ra;
        pos = ra - (k0 & ~(AL - 1));
      }
      const int32_t row = bi * kWaveRows + lane;
      Acc s = Acc(0);
      X xv[KR];
      V v[KR];
      int32_t c0 = 0;
      // gathers of KR list offsets (masked) or of entries p0 .. p0 + KR of the
      // row, then their values
      auto request = [&](int32_t p0) {
        if constexpr (masked.value)
        {
          // a lane without the k-th offset gathers out of x's range (0, no read)
          // and takes the zero kept behind the staged entries: its product adds 0
          const uint32_t at = static_cast<uint32_t>(row) * static_cast<uint32_t>(sizeof(X));
          const uint32_t xbytes = static_cast<uint32_t>(ncols) * static_cast<uint32_t>(sizeof(X));
#pragma unroll
          for (int k = 0; k < KR; ++k)
          {
            const uint32_t o = at + static_cast<uint32_t>(of[k]);
            xv[k] = ld_buffer(x, xbytes, (ra >> k) & 1 ? o : 0xFFFFFFF0u);
          }
#pragma unroll
          for (int k = 0; k < KR; ++k)
          {
            v[k] = lval[(ra >> k) & 1 ? p0 : zero];
            p0 += (ra >> k) & 1;
          }
        }
        else
        {
          // decoded column, clamped into [0, ncols): positions outside the row
          // (or the block) hold some other entry, whose product is not added
          auto column = [&](uint32_t c16) -> uint32_t {
            uint32_t cc;
            if constexpr (IM == 1)
              cc = static_cast<uint32_t>(w.x) + c16;
            else
            {
              const int32_t lo = (c16 & 0x4000u) ? w.y : w.x, hi = (c16 & 0x4000u) ? w.w : w.z;
              cc = static_cast<uint32_t>((c16 & 0x8000u) ? hi : lo) + (c16 & 0x3FFFu);
            }
            const uint32_t top = static_cast<uint32_t>(ncols) - 1u;
            return cc < top ? cc : top;
          };
#pragma unroll
          for (int k = 0; k < KR; ++k)
            xv[k] = x[column(lcol[p0 + k])];
#pragma unroll
          for (int k = 0; k < KR; ++k)
            v[k] = lval[p0 + k];
        }
      };
      auto add = [&]() {
#pragma unroll
        for (int k = 0; k < KR; ++k)
        {
          const Acc p = static_cast<Acc>(widen(v[k])) * static_cast<Acc>(xv[k]);
          if constexpr (masked.value)
            s += p;
          else
            s = c0 + k < len ? s + p : s;
        }
      };
      if constexpr (!masked.value)
        for (; __any(len > c0 + KR); c0 += KR) // rows longer than KR: KR entries at a time
        {
          request(pos + (c0 < len ? c0 : 0));
          add();
        }
      request(pos + (c0 < len ? c0 : 0));
      if (nkept == burst)
        store_kept();
      int32_t nra = 0, nre = 0;
      X nxr = X(0);
      if constexpr (refill.value)
      {
        load_rows(nb, nra, nre, nxr);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the LDS reads are done
        fill(n0, n1, nkind);
        __builtin_amdgcn_sched_barrier(0);
      }
      add();
      yrow = row < nrows ? row : -1;
      yval = MODE == kResid ? xr - static_cast<X>(s) : static_cast<X>(s);
      if (yrow >= 0)
      {
        if (MODE == kResid)
          part += static_cast<Acc>(yval) * static_cast<Acc>(yval);
        else if (MODE == kDot)
          part += static_cast<Acc>(xr) * static_cast<Acc>(yval);
      }
      if (burst > 0)
      {
        if (nkept == 0)
          kfirst = bi;
        kept[nkept * kWaveRows + lane] = yval;
        ++nkept;
      }
      bi = nb;
      k0 = n0;
      k1 = n1;
      kind = nkind;
      w = nwb;
      ra = nra;
      re = nre;
      xr = nxr;
    };
    auto step = [&](auto refill, int32_t nb) {
      if constexpr (ALL)
        block(refill, std::true_type{}, nb);
      else if (HM && kind)
        block(refill, std::bool_constant<HM != 0>{}, nb);
      else
        block(refill, std::false_type{}, nb);
    };
    for (int32_t nb = bi + nw; nb < bend; nb += nw)
      step(std::true_type{}, nb);
    step(std::false_type{}, 0);
    store_kept();
  }
  if constexpr (MODE != kPlain)
  {
    part = wave_sum(part);
    if (lane == 0)
      partials[blockIdx.x] = part;
  }
}

// How csr_wave runs a matrix of nblocks blocks: blocks per store of results (as
// many as the LDS of its wavefronts holds, at most 24: 16 were 1-4% slower),
// workgroups.  From 8 blocks per wavefront on, bursts are the faster (FP64
// 7-point 112^3, 12 blocks: 18.6 against 19.7 us, 27-point 90^3, 11: 30.5 against
// 34.7; BF16 7-point 128^3, 8: 13.0 against 12.6); with fewer, every wavefront
// that fits takes part (FP64 5-point 1024^2, 7: 11.4 against 11.8).
struct WavePlan
{
  int burst;
  int64_t grid;
};
constexpr int64_t kWaveMaxGrid = 8192; // 32 wavefronts on each of 256 CUs
inline WavePlan wave_plan(int c, int vbytes, bool cols, int64_t nblocks, int ncu)
{
  const WaveClass& k = kWaveClasses[c];
  const int xbytes = vbytes >= 8 ? vbytes : 4;
  const int per = vbytes == 16 ? k.per_cu16
                  : vbytes == 8 ? k.per_cu8
                                : (vbytes == 4 ? k.per_cu4 : k.per_cu2);
  const int64_t stream = static_cast<int64_t>(ncu) * per;
  if (nblocks >= 8 * stream)
  {
    const int room = 163840 / per / 1280 * 1280 - wave_lds(k.e, vbytes, xbytes, cols, 0).bytes;
    return WavePlan{std::min(24, room / (kWaveRows * xbytes)), stream};
  }
  const int64_t all = int64_t(4) * ncu * wave_per_simd(k.e, k.kr, vbytes, xbytes, cols);
  return WavePlan{0, std::min(nblocks, std::min(all, kWaveMaxGrid))};
}

// Of every 32 blocks, how many keep their values in the 256 MB last-level cache for
// the next product of a solve; the others are streamed past it.  Loading all of a
// larger matrix as usual would evict each line before its next use.  The kept share
// is what fits beside the vectors in use (x, p, r and y of CG): from 160 to 240 MB in
// all were within 2% of each other.  Below 64 MB the loads are left as streams
// (27-point 64^3, 55 MB: kept 13.0, streamed 12.4 us).
// Only CG's products do this: a product that may be the only one on its matrix loses
// (27-point 160^3 after other work: 152 streamed, 156 us).
// Streamed and by this rule, an iteration of FP64 CG, 27-point 112^3 (303 MB): 95 and
// 83 us; FP32 CG, 7-point 256^3 (470 MB beside 268 MB of vectors): 3% less.  Repeated
// products, us: 27-point 96^3 35.3 and 32.5, 128^3 78.4 and 72, 7-point 112^3 20.4 and
// 19.0, FP32 256^3 121 and 115, BF16 93 and 88.
constexpr double kKeepBytes = 208e6, kKeepLeast = 48e6, kKeepFrom = 64e6;
inline int32_t wave_keep(int64_t nnz, size_t vbytes, double vector_bytes)
{
  const double bytes = static_cast<double>(nnz) * static_cast<double>(vbytes);
  if (bytes < kKeepFrom)
    return 0;
  const double room = std::max(kKeepLeast, kKeepBytes - vector_bytes);
  return std::min(32, static_cast<int32_t>(32.0 * room / bytes + 0.5));
}

// Launches csr_wave on M.nparts workgroups.
template <typename V, typename X, typename Acc, int MODE>
void launch_csr_wave(const CsrView& M, hipStream_t s, const V* val, const X* x, X* y, const X* b,
                     Acc* partials, const CgState<Acc>* st, int32_t it, hipEvent_t ev0,
                     hipEvent_t ev1)
{
  const dim3 grid(static_cast<unsigned>(M.nparts));
  const bool hm = M.wrows != nullptr;
  const int32_t keep =
      MODE == kDot ? wave_keep(M.nnz, sizeof(V), 4.0 * sizeof(X) * M.ncols) : 0;
  auto go = [&](auto im, auto masks, auto e, auto kr) {
    const WaveLds at = wave_lds(decltype(e)::value, sizeof(V), sizeof(X), M.wcols, M.burst);
    launch_timed(&csr_wave<V, X, Acc, MODE, decltype(im)::value, decltype(masks)::value,
                           decltype(e)::value, decltype(kr)::value>,
                 grid, dim3(kWaveRows), static_cast<uint32_t>(at.bytes), s, ev0, ev1,
                 hm ? M.wrows : M.rowptr, hm ? M.wblocks : M.blocks, M.woffs, M.col16, M.wbase,
                 M.nrows, M.ncols, val, x, y, b, partials, st, it, at, M.burst,
                 keep);
  };
  using std::integral_constant;
  auto kinds = [&](auto e, auto kr) {
    if (kIsComplex<V> || hm)
      go(integral_constant<int, 2>{}, integral_constant<int, 1>{}, e, kr);
    else if constexpr (kIsComplex<V>)
      return;
    else if (M.short_kind == 1)
      go(integral_constant<int, 1>{}, integral_constant<int, 0>{}, e, kr);
    else
      go(integral_constant<int, 2>{}, integral_constant<int, 0>{}, e, kr);
  };
  switch (M.wave)
  {
#define SPMVX_WAVE_CASE(i, EE, K, W16, W8, W4, W2)                                             \
  case i: kinds(integral_constant<int, EE>{}, integral_constant<int, K>{}); break;
    SPMVX_WAVE_CLASSES(SPMVX_WAVE_CASE)
#undef SPMVX_WAVE_CASE
  default: break;
  }
}

} // namespace spmvx
