// Sparse triangular solves on the device:
//  - BJAC / ILU(0) preconditioner application:
//    y = alpha * U^-1 (d .* L^-1 x) + beta * y with L unit lower, U unit upper
//    (psb_d_bjac_apply_vect, prec/impl/psb_d_bjacprec_impl.f90:166-173:
//    psb_spsm with scale 'L' and the inverse pivots, then psb_spsm on U);
//  - the CSR matrix's own solve y = alpha * op(T)^-1 x + beta * y, T lower or
//    upper, unit or not, op 'N', 'T' or 'C' (psb_d_cuda_csrg_inner_vect_sv,
//    cuda/impl/psb_d_cuda_csrg_inner_vect_sv.F90; the CPU algorithm it must
//    equal is psb_d_csr_cssv, base/serial/impl/psb_d_csr_impl.F90:782-1039),
//    FP64 and FP32.
//
// Each triangle is solved by levels: the host analysis gives every row the
// length of its longest dependency chain.  A row's sum runs in its CSR order,
// y(i) = x(i) - sum_j val(j) y(ja(j)) with separate multiply and add, as the
// reference's inner_csrsv (base/serial/impl/psb_d_csr_impl.F90:890-941), so
// the result equals the sequential CPU solve bit for bit.
//
// A non-unit row divides by its diagonal, (x(i) - sum) / a(i,i), as the CPU
// does.  The transposed solve (op 'T' / 'C') is solved as the triangle of the
// transpose, whose row c lists the entries (i, c) of T in the order the CPU
// applies them (rows in solve order, CSR order inside a row); its rows are
// computed as the CPU updates them, by running subtraction
// y(c) = ((x(c) - v1 y(i1)) - v2 y(i2)) ..., then the division.
//
// The triangle is cut into tiles of about kTileRows rows and one workgroup
// solves a tile: its rows in steps (the levels inside the tile, 64 rows at a
// time, one wavefront), with the entries, the right-hand side and the solution
// staged in LDS, so a step costs LDS traffic and arithmetic only.  A row's
// dependencies outside its tile (its halo) are polled from the solution array
// itself, which starts out filled with one NaN bit pattern that no solve
// stores (is_unset): an entry is ready once it holds anything else, so a
// value needs no flag and no fence (8- or 4-byte agent-scope loads and
// stores).  Three wavefronts of the workgroup poll while the fourth solves.
// Workgroups take their tiles by a ticket, in an order where a tile depends
// only on tiles before it, so a workgroup waits only for tiles whose
// workgroups already run: every wait ends whatever the number of resident
// workgroups.  Two solution arrays alternate; a tile resets its rows of the
// other one for the solve after.
//
// Tiles follow the grid when the triangle's entries sit at the offsets of a
// regular grid in natural order (1, p and q, p dividing q: 5- and 7-point
// stencils and their ILU(0) factors), as boxes of 8 x 8 x 8 or 24 x 24 rows;
// otherwise they are runs of consecutive rows, and a row of more than 1024
// entries is a tile of its own (wide_row).  The chain of dependencies
// then crosses tiles once in 8 (24) rows along each axis, and only a crossing
// pays the way through memory between XCDs.
//
// Measured against one workgroup walking runs of small levels and a launch for
// each larger one, which this replaced (7-point stencil, lower, non-unit,
// FP64): L = 32 156 -> 41 us, L = 64 438 -> 91 us, L = 110 903 -> 204 us (boxes of
// 10 x 10 x 10 53 / 114 / 228 us, of 8 x 8 x 4 44 / 106 / 224 us); 5-point
// 1000 x 1000 2562 -> 647 us; 27-point L = 40, runs of rows, 1373 -> 407 us.
//
// A triangle of at most kFewLevels levels, or with the launch-per-level variant
// set, is solved in level order instead: renumbered so that level l holds
// positions lev_ptr[l] .. lev_ptr[l+1]-1 (rows ascending inside a level), x
// gathered into that order, one launch per level (one thread per row), the
// solution scattered back; captured once into a graph that works on internal
// buffers.
#pragma clang fp contract(off)

#include <string.h>

#include <algorithm>
#include <new>
#include <vector>

#include "host_parallel.hpp"
#include "psb_hip_internal.hpp"

namespace psbhip {

// Limits of a tile that is a run of rows: rows, stored entries, halo entries; and
// of any tile (boxes have up to 576 rows): LDS bytes (64 KB lets two workgroups
// share a CU; an 8 x 8 x 8 tile takes about 31 KB).
constexpr int kTileRows = 512;
constexpr int kTileEntries = 2048;
constexpr int kTileHalo = 1024;
constexpr size_t kTileLds = (size_t)64 << 10;
constexpr int kTileThreads = 256;
// polls of memory by a wavefront before its halo entries are given up (they
// then count as NaN, and the next call that brings a result to the host fails);
// a poll takes about a microsecond.  A tile waits for those whose workgroups
// run beside it: at most 2048 of them, of 512 steps of 0.26 us, one after
// another, are 0.3 s.
constexpr int kTilePolls = 1 << 23;

// A tile: its rows at positions row0 .. row0+nrow-1 of the tile-ordered
// arrays, its entries at ent0 .., its steps at step0 .., its halo at halo0 ..
struct TriTile {
  int row0, nrow, ent0, nent, step0, nstep, halo0, nhalo;
};

template <typename T>
struct TriLevels {
  int n = 0, nnz = 0, nlev = 0;
  // level order (one launch per level)
  int* perm = nullptr;          // level position -> row
  int* irp = nullptr;           // level-ordered CSR, 0-based; columns are level positions
  int* ja = nullptr;
  T* val = nullptr;
  std::vector<int> lev_ptr;     // host: level l = positions lev_ptr[l] .. lev_ptr[l+1]-1
  // tiles (ntiles > 0: this form is used)
  int ntiles = 0;
  int width = 0;                // entries of every row, padding included; 0: per step
  size_t lds = 0;               // LDS bytes of the largest tile
  TriTile* tiles = nullptr;     // in ticket order
  int* trow = nullptr;          // row of each position
  T* tdv = nullptr;             // diagonal of each position (non-unit triangles)
  T* tval = nullptr;            // entry k of a step's t-th row at ent + k*count + t
  uint16_t* tdep = nullptr;     // LDS slot of the entry's dependency
  int2* tstep = nullptr;        // {first row | rows << 16, first entry | width << 16}
  int* thalo = nullptr;         // rows of earlier tiles the tile reads
  T* sol = nullptr;             // two solution arrays, sol_stride entries apart
  unsigned long long* ticket = nullptr;
};

// 0: tiles (default); 1: one launch per level.
static int g_trsv_variant = 0;

struct IluDev {
  int n = 0;
  TriLevels<double> L, U;
  double* d = nullptr;          // inverse pivots
  double* t1 = nullptr;         // L^-1 x (row order)
  // launch-per-level form
  double* xa = nullptr;         // right-hand side of the triangle being solved (level order)
  double* ya = nullptr;         // its solution (level order)
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

// A CSR matrix's triangle prepared for op(T)^-1 x: the strict part (or, for
// op 'T' / 'C', the strict part of the transpose), and the diagonal when the
// triangle is not unit.
template <typename T>
struct TriSolve {
  int n = 0, key = -1;          // key: lower | unit << 1 | transposed << 2
  bool run = false;             // transposed: rows by running subtraction
  TriLevels<T> tl;
  // launch-per-level form
  T* dv = nullptr;              // diagonal in level order (non-unit), else null
  T* xa = nullptr;              // right-hand side (level order)
  T* ya = nullptr;              // solution (level order)
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

// dst[p] = src[perm[p]], times d[perm[p]] when d is given (the pivot scaling
// y(i) * d(i) of the reference's 'L' scale)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_perm_gather(int n, const int* __restrict__ perm,
                                                        const T* __restrict__ src,
                                                        const T* __restrict__ d,
                                                        T* __restrict__ dst) {
  for (int p = blockIdx.x * kBlock + threadIdx.x; p < n; p += gridDim.x * kBlock) {
    const int i = perm[p];
    dst[p] = d ? src[i] * d[i] : src[i];
  }
}

// dst[perm[p]] = src[p]
template <typename T>
__global__ __launch_bounds__(kBlock) void k_perm_scatter(int n, const int* __restrict__ perm,
                                                         const T* __restrict__ src,
                                                         T* __restrict__ dst) {
  for (int p = blockIdx.x * kBlock + threadIdx.x; p < n; p += gridDim.x * kBlock)
    dst[perm[p]] = src[p];
}

// alpha * s + beta * *y with the special cases of the library's axpby (alpha or
// beta 0 or 1; y not read for beta == 0), separately rounded; beta == 0 and
// alpha == -1 negate, as the CPU solve's scaling does
template <typename T>
__device__ __forceinline__ T axpby_y(T alpha, T s, T beta, const T* y) {
  if (alpha == T(0)) return (beta == T(0)) ? T(0) : (beta == T(1) ? *y : beta * *y);
  if (beta == T(0)) return (alpha == T(1)) ? s : alpha * s;
  return alpha * s + beta * *y;
}

// y[perm[p]] = alpha * src[p] + beta * y[perm[p]]
template <typename T>
__global__ __launch_bounds__(kBlock) void k_perm_scatter_axpby(int n, const int* __restrict__ perm,
                                                               const T* __restrict__ src,
                                                               T alpha, T beta, T* y) {
  for (int p = blockIdx.x * kBlock + threadIdx.x; p < n; p += gridDim.x * kBlock) {
    const int i = perm[p];
    y[i] = axpby_y(alpha, src[p], beta, y + i);
  }
}

// One level: positions p0 .. p0+count-1, one thread each.  RUN: running
// subtraction from x (the transposed solve); DIV: divide by the diagonal.
template <typename T, bool DIV, bool RUN>
__global__ __launch_bounds__(kBlock) void k_trsv_level(int p0, int count,
                                                       const int* __restrict__ irp,
                                                       const int* __restrict__ ja,
                                                       const T* __restrict__ val,
                                                       const T* __restrict__ dv,
                                                       const T* __restrict__ x, T* y) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= count) return;
  const int p = p0 + t;
  T r;
  if (RUN) {
    r = x[p];
    for (int e = irp[p]; e < irp[p + 1]; e++) r = r - val[e] * y[ja[e]];
  } else {
    T acc = T(0);
    for (int e = irp[p]; e < irp[p + 1]; e++) acc = acc + val[e] * y[ja[e]];
    r = x[p] - acc;
  }
  y[p] = DIV ? r / dv[p] : r;
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_tri_unset(int64_t n, T* __restrict__ sol) {
  const T u = __builtin_bit_cast(T, MarkBits<T>::unset);
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock)
    sol[i] = u;
}

// Entries from one solution array to the other: n rounded up to whole 128-byte
// lines.  A solve polls one array while it sets the other back with plain
// stores, and a plain access leaves its line in the XCD's L2, where polls of
// entries in the same line would find it unchanged.
template <typename T>
inline size_t sol_stride(int n) {
  constexpr size_t line = 128 / sizeof(T);
  return ((size_t)n + line - 1) / line * line;
}

// LDS of a tile, in this order (each part 16-byte aligned): solution slots
// (rows, halo, a zero slot), entry values, diagonals, rows, steps, entry
// slots.  The host's tile_lds adds up the same parts.
__host__ __device__ inline size_t lds16(size_t b) { return (b + 15) & ~(size_t)15; }
template <typename T>
__host__ __device__ inline size_t tile_lds(int nrow, int nhalo, int nent, int nstep, bool dv) {
  return lds16(sizeof(T) * (size_t)(nrow + nhalo + 1)) + lds16(sizeof(T) * (size_t)nent) +
         (dv ? lds16(sizeof(T) * (size_t)nrow) : 0) + lds16(sizeof(int) * (size_t)nrow) +
         lds16(sizeof(int2) * (size_t)nstep) + lds16(sizeof(uint16_t) * (size_t)nent);
}

// Registers of one row's step: the operands that do not depend on the
// solution, loaded a step ahead.
template <typename T, int W, bool DIV>
struct TileStep {
  int roff, cnt;
  int dep[W];
  T v[W];
  T xi, dv;
  int row;
};

// A row of more entries than a tile stages, a tile of its own (no steps; its halo
// lists the row of every entry): the workgroup polls the entries in chunks and
// leaves the products in LDS, one thread adds them in CSR order (product and sum
// rounded separately, as everywhere).  Bound by that chain of adds.  One such row
// used to send the whole triangle to a launch per level: FP64, a chain of 20,000
// rows under one of 1500 entries 31.5 -> 5.2 ms, the 7-point lower triangle at
// L = 40 under one of 3000 955 -> 124 us and under 64 of 5000 45.8 -> 0.6 ms, a full
// triangle of 2496 rows 398 -> 12.9 ms.
constexpr int kWideChunk = 1024;
template <typename T, bool DIV, bool RUN>
__device__ __forceinline__ void wide_row(const TriTile& t, const int* __restrict__ trow,
                                         const T* __restrict__ tdv, const T* __restrict__ tval,
                                         const int* __restrict__ thalo, T* sol, T* next,
                                         const T* x, const T* __restrict__ scale, T alpha, T beta,
                                         T* y, T* prod, const Waits& waits) {
  const int i = trow[t.row0];
  T xi = x[i];
  if (scale) xi = xi * scale[i];
  T acc = RUN ? xi : T(0);
  for (int c = 0; c < t.nent; c += kWideChunk) {
    const int m = t.nent - c < kWideChunk ? t.nent - c : kWideChunk;
    for (int e = threadIdx.x; e < m; e += kTileThreads) {
      const T* from = sol + thalo[t.halo0 + c + e];
      const T v = ld_stream(tval + t.ent0 + c + e);
      T s = ld_agent(from);
      for (int polls = 1; is_unset(s); polls++) {
        if (polls >= waits.polls) {
          give_up(waits);
          s = __builtin_bit_cast(T, MarkBits<T>::nan);
          break;
        }
        __builtin_amdgcn_s_sleep(16);
        s = ld_agent(from);
      }
      prod[e] = v * s;
    }
    __syncthreads();
    if (threadIdx.x == 0)
      for (int e = 0; e < m; e++) acc = RUN ? acc - prod[e] : acc + prod[e];
    __syncthreads();
  }
  if (threadIdx.x != 0) return;
  T r = RUN ? acc : xi - acc;
  if (DIV) r = r / tdv[t.row0];
  r = set_value(r);
  next[i] = __builtin_bit_cast(T, MarkBits<T>::unset);
  st_agent(sol + i, r);
  y[i] = axpby_y(alpha, r, beta, y + i);
}

// One tile per workgroup.  Bound by the chain of dependencies: a step (the
// LDS reads of W solution entries, W multiply-adds and, when DIV, a division)
// is 0.26 us with the division (a chain of 20,000 rows 5.1 ms), a crossing
// into the next tile one store and one load through memory between XCDs,
// 1-2 us; the bytes (40 a row) would take 2 us at L = 64, not 91.  Polling by
// every lane from the start instead of by the first ones until an entry
// comes: 97 and 254 us at L = 64 and 110.  W > 0: every row has W entries
// (padding: value 0 times the zero slot, which leaves the sum's bits
// unchanged; the sum starts at +0, so it is never -0 there, and the running
// form subtracts +0); W == 0: the step's own width.  Rows sum in CSR order.
template <typename T, int W, bool DIV, bool RUN>
__global__ __launch_bounds__(kTileThreads) void k_trsv_tiles(
    size_t stride, int ntiles, const TriTile* __restrict__ tiles, const int* __restrict__ trow,
    const T* __restrict__ tdv, const T* __restrict__ tval, const uint16_t* __restrict__ tdep,
    const int2* __restrict__ tstep, const int* __restrict__ thalo, T* sol2,
    unsigned long long* ticket, const T* x, const T* __restrict__ scale, T alpha, T beta, T* y,
    Waits waits) {
  extern __shared__ __align__(16) char lds[];
  __shared__ unsigned long long my;
  if (threadIdx.x == 0) my = atomicAdd(ticket, 1ull);
  __syncthreads();
  // a launch draws exactly ntiles tickets, so all of its tickets share one epoch
  const unsigned long long epoch = my / (unsigned)ntiles;
  const TriTile t = tiles[(int)(my - epoch * (unsigned)ntiles)];
  T* sol = sol2 + (epoch & 1 ? stride : 0);    // no line of one in the other: sol_stride
  T* next = sol2 + (epoch & 1 ? 0 : stride);
  T* ys = reinterpret_cast<T*>(lds);
  if (t.nstep == 0) {
    wide_row<T, DIV, RUN>(t, trow, tdv, tval, thalo, sol, next, x, scale, alpha, beta, y, ys,
                          waits);
    return;
  }
  char* at = lds + lds16(sizeof(T) * (size_t)(t.nrow + t.nhalo + 1));
  T* ev = reinterpret_cast<T*>(at);
  at += lds16(sizeof(T) * (size_t)t.nent);
  T* dvs = reinterpret_cast<T*>(at);
  if (DIV) at += lds16(sizeof(T) * (size_t)t.nrow);
  int* rows = reinterpret_cast<int*>(at);
  at += lds16(sizeof(int) * (size_t)t.nrow);
  int2* steps = reinterpret_cast<int2*>(at);
  at += lds16(sizeof(int2) * (size_t)t.nstep);
  uint16_t* ed = reinterpret_cast<uint16_t*>(at);
  const T unset = __builtin_bit_cast(T, MarkBits<T>::unset);

  for (int p = threadIdx.x; p < t.nrow; p += kTileThreads) {
    const int r = trow[t.row0 + p];
    rows[p] = r;
    T xv = x[r];
    if (scale) xv = xv * scale[r];
    ys[p] = xv;
    if (DIV) dvs[p] = tdv[t.row0 + p];
    next[r] = unset;
  }
  for (int h = threadIdx.x; h < t.nhalo; h += kTileThreads) ys[t.nrow + h] = unset;
  if (threadIdx.x == 0) ys[t.nrow + t.nhalo] = T(0);
  for (int e = threadIdx.x; e < t.nent; e += kTileThreads) {
    ev[e] = ld_stream(tval + t.ent0 + e);
    ed[e] = tdep[t.ent0 + e];
  }
  for (int q = threadIdx.x; q < t.nstep; q += kTileThreads) steps[q] = tstep[t.step0 + q];
  __syncthreads();

  if (threadIdx.x >= kWave) {
    // Pollers: each lane walks its halo entries (step order) and passes every
    // one on to LDS as it comes.  Until the first entry is there only the
    // first lanes poll, so tiles whose turn is far off load the memory little.
    constexpr int kPollers = kTileThreads - kWave;
    constexpr int kFirst = 8;
    const int lane = threadIdx.x - kWave;
    int h = lane, polls = 0;
    int src = h < t.nhalo ? thalo[t.halo0 + h] : 0;
    bool open = lane < kFirst;
    while (__any(h < t.nhalo)) {
      if (!open) open = !is_unset(ld_lds(ys + t.nrow));
      const bool look = open && h < t.nhalo;
      if (look) {
        const T v = ld_agent(sol + src);
        if (!is_unset(v)) {
          st_lds(ys + t.nrow + h, v);
          h += kPollers;
          if (h < t.nhalo) src = thalo[t.halo0 + h];
        }
      } else {
        __builtin_amdgcn_s_sleep(2);
      }
      if (__any(look) && ++polls > waits.polls) {
        give_up(waits);
        for (; h < t.nhalo; h += kPollers)
          st_lds(ys + t.nrow + h, __builtin_bit_cast(T, MarkBits<T>::nan));
      }
    }
  } else {
    const int lane = threadIdx.x;
    constexpr int WR = W > 0 ? W : 4;
    auto step = [&](int q) { return steps[q < t.nstep ? q : t.nstep - 1]; };
    auto fetch = [&](int2 d, TileStep<T, WR, DIV>& s) {
      s.roff = d.x & 0xffff;
      s.cnt = d.x >> 16;
      const int ln = lane < s.cnt ? lane : s.cnt - 1;
      s.xi = ys[s.roff + ln];
      s.row = rows[s.roff + ln];
      if (DIV) s.dv = dvs[s.roff + ln];
      if (W > 0) {
#pragma unroll
        for (int k = 0; k < WR; k++) {
          const int e = W * s.roff + k * s.cnt + ln;
          s.dep[k] = ed[e];
          s.v[k] = ev[e];
        }
      }
    };
    // reads the solution entries; whether all of the step's have arrived
    auto read = [&](const int (&dep)[WR], T (&yk)[WR]) {
#pragma unroll
      for (int k = 0; k < WR; k++) yk[k] = ld_lds(ys + dep[k]);
    };
    auto wait = [&](const int (&dep)[WR], T (&yk)[WR]) {
      for (;;) {
        bool ready = true;
#pragma unroll
        for (int k = 0; k < WR; k++) ready = ready && !is_unset(yk[k]);
        if (__all(ready)) break;
        __builtin_amdgcn_s_sleep(1);
        read(dep, yk);
      }
    };
    auto add = [&](T& acc, const T (&v)[WR], const T (&yk)[WR]) {
#pragma unroll
      for (int k = 0; k < WR; k++) acc = RUN ? acc - v[k] * yk[k] : acc + v[k] * yk[k];
    };
    TileStep<T, WR, DIV> cur, nxt;
    int2 d0 = step(0), d1 = step(1);
    fetch(d0, cur);
    for (int q = 0; q < t.nstep; q++) {
      const int2 d2 = step(q + 2);
      T acc = RUN ? cur.xi : T(0);
      T yk[WR];
      if constexpr (W > 0) {
        read(cur.dep, yk);   // the critical reads first, the next step's behind them
        fetch(d1, nxt);
        wait(cur.dep, yk);
        add(acc, cur.v, yk);
      } else {
        fetch(d1, nxt);
        const int e0 = d0.y & 0xffff, w = d0.y >> 16;
        const int ln = lane < cur.cnt ? lane : cur.cnt - 1;
        for (int k0 = 0; k0 < w; k0 += WR) {
          int dep[WR];
          T v[WR];
#pragma unroll
          for (int k = 0; k < WR; k++) {   // past the width: the zero slot, value 0
            const bool in = k0 + k < w;
            const int e = e0 + (in ? k0 + k : 0) * cur.cnt + ln;
            dep[k] = in ? (int)ed[e] : t.nrow + t.nhalo;
            v[k] = in ? ev[e] : T(0);
          }
          read(dep, yk);
          wait(dep, yk);
          add(acc, v, yk);
        }
      }
      T r = RUN ? acc : cur.xi - acc;
      if (DIV) r = r / cur.dv;
      r = set_value(r);
      if (lane < cur.cnt) {
        st_lds(ys + cur.roff + lane, r);
        st_agent(sol + cur.row, r);
      }
      cur = nxt;
      d0 = d1;
      d1 = d2;
    }
  }
  __syncthreads();
  for (int p = threadIdx.x; p < t.nrow; p += kTileThreads) {
    const int i = rows[p];
    y[i] = axpby_y(alpha, ys[p], beta, y + i);
  }
}

// Level of every row (longest chain of dependencies through the triangle);
// the number of levels.
static int count_levels(int n, bool lower, const int* irp, const int* ja, std::vector<int>& lev) {
  lev.assign(n, 0);
  int nlev = 0;
  for (int t = 0; t < n; t++) {
    const int i = lower ? t : n - 1 - t;
    int l = 0;
    for (int p = irp[i] - 1; p < irp[i + 1] - 1; p++) l = std::max(l, lev[ja[p] - 1] + 1);
    lev[i] = l;
    nlev = std::max(nlev, l + 1);
  }
  return nlev;
}

// Rows grouped by level, in ascending row order within a level.
static void order_levels(int n, int nlev, const std::vector<int>& lev, std::vector<int>& rows,
                         std::vector<int>& lev_ptr) {
  lev_ptr.assign(nlev + 1, 0);
  for (int i = 0; i < n; i++) lev_ptr[lev[i] + 1]++;
  for (int l = 0; l < nlev; l++) lev_ptr[l + 1] += lev_ptr[l];
  rows.assign(n, 0);
  std::vector<int> fill(lev_ptr.begin(), lev_ptr.end() - 1);
  for (int i = 0; i < n; i++) rows[fill[lev[i]]++] = i;
}

constexpr int kHostMin = 32768;   // rows from which the planning uses threads

// A row that takes a tile of its own (wide_row).
static bool is_wide(int len) { return len > kTileEntries / 2; }

// The offsets of a regular grid in natural order: every entry of the triangle
// sits 1, p or q rows before its row (in solve order), q a multiple of p.
// Returns the number of distinct offsets (2 or 3), 0 for any other triangle.
static int grid_offsets(int n, bool lower, const int* irp, const int* ja, int (&o)[3]) {
  int m = 0;
  for (int i = 0; i < n; i++)
    for (int e = irp[i] - 1; e < irp[i + 1] - 1; e++) {
      const int d = lower ? i - (ja[e] - 1) : (ja[e] - 1) - i;
      int k = 0;
      while (k < m && o[k] != d) k++;
      if (k < m) continue;
      if (m == 3) return 0;
      o[m++] = d;
    }
  std::sort(o, o + m);
  if (m < 2 || o[0] != 1 || o[1] < 8 || (m == 3 && o[2] % o[1] != 0)) return 0;
  return m;
}

// Tile of every row in solve order t (row t of a lower triangle, n-1-t of an
// upper one), tile numbers ascending along the dependencies; the number of
// tiles.  Boxes of the grid when the triangle is one and no entry leaves a box
// against its order (an entry that wraps round a grid line can), else runs of
// consecutive rows within the limits of a tile.
static int assign_tiles(int n, bool lower, const int* irp, const int* ja,
                        std::vector<int>& tile) {
  tile.assign(n, 0);
  auto row = [&](int t) { return lower ? t : n - 1 - t; };
  auto dep = [&](int e) { return lower ? ja[e] - 1 : n - ja[e]; };   // solve order of entry e
  int o[3] = {1, 0, 0};
  const int m = grid_offsets(n, lower, irp, ja, o);
  if (m > 0) {
    // 8 x 8 x 8 (512 rows): a level of the box is at most 48 rows, one step; in
    // two dimensions 24 x 24 (576 rows), at most 24 a level
    const int nx = o[1], ny = m == 3 ? o[2] / nx : (n + nx - 1) / nx;
    const int bx = m == 3 ? 8 : 24, by = bx, bz = 8;
    const int tx = (nx + bx - 1) / bx, ty = (ny + by - 1) / by;
    const int pl = nx * ny;
    int nt[kHostThreads] = {};
    host_parallel(n, kHostMin, [&](int th, int lo, int hi) {
      int most = 0;
      for (int t = lo; t < hi; t++) {
        const int z = m == 3 ? t / pl : 0, r = m == 3 ? t - z * pl : t;
        const int yy = r / nx, xx = r - yy * nx;
        tile[t] = ((z / bz) * ty + yy / by) * tx + xx / bx;
        most = std::max(most, tile[t] + 1);
      }
      nt[th] = most;
    });
    bool bad[kHostThreads] = {};
    host_parallel(n, kHostMin, [&](int th, int lo, int hi) {
      bool any = false;
      for (int t = lo; t < hi; t++) {
        const int b = irp[row(t)] - 1, m = irp[row(t) + 1] - 1 - b;
        any = any || is_wide(m);   // an entry stored over and over
        for (int e = b; e < b + m; e++) any = any || tile[dep(e)] > tile[t];
      }
      bad[th] = any;
    });
    if (!*std::max_element(bad, bad + kHostThreads))
      return *std::max_element(nt, nt + kHostThreads);
  }
  std::vector<int> seen(n > 0 ? n : 1, -1);
  int nt = 0, rows = 0, ent = 0, halo = 0, t0 = 0;
  bool wide = false;   // the tile holds a wide row: nothing joins it
  for (int t = 0; t < n; t++) {
    const int b = irp[row(t)] - 1, e = irp[row(t) + 1] - 1;
    const bool w = is_wide(e - b);
    if (rows > 0 && (wide || w)) {
      nt++;
      rows = ent = halo = 0;
      t0 = t;
    }
    wide = w;
    if (w) {
      rows = 1;
      tile[t] = nt;
      continue;
    }
    for (;;) {
      int fresh = 0;   // halo entries this row would add
      for (int k = b; k < e; k++) {
        const int d = dep(k);
        if (d < t0 && seen[d] != nt) {
          seen[d] = nt;
          fresh++;
        }
      }
      if (rows == 0 || (rows < kTileRows && ent + (e - b) <= kTileEntries / 2 &&
                        halo + fresh <= kTileHalo)) {
        rows++;
        ent += e - b;
        halo += fresh;
        break;
      }
      nt++;   // a new tile starts at this row
      rows = ent = halo = 0;
      t0 = t;
    }
    tile[t] = nt;
  }
  return nt + (n > 0 ? 1 : 0);
}

template <typename V>
static int upload(V** dst, const V* src, size_t count) {
  PSB_HIP_CHECK(hipMalloc((void**)dst, sizeof(V) * std::max<size_t>(count, 1)));
  if (count > 0)
    PSB_HIP_CHECK(hipMemcpyAsync(*dst, src, sizeof(V) * count, hipMemcpyHostToDevice,
                                 ctx().stream));
  return PSB_HIP_SUCCESS;
}

// The tiles [q0, q1) as one host thread packs them, offsets from its own start.
template <typename V>
struct TilePack {
  int q0 = 0, q1 = 0;
  size_t lds = 0;
  std::vector<V> val;
  std::vector<uint16_t> dep;
  std::vector<int2> step;
  std::vector<int> halo;
};
constexpr unsigned kHaloHash = 4 * kTileHalo;   // a tile has at most kTileHalo halo entries

// Cuts the triangle into tiles and uploads them (T.ntiles > 0 then); leaves
// T.ntiles at 0 when a tile does not fit LDS.
template <typename V>
static int plan_tiles(TriLevels<V>& T, bool lower, const int* irp, const int* ja, const V* val,
                      const V* diag, const std::vector<int>& lev) {
  const int n = T.n;
  if (n == 0) return PSB_HIP_SUCCESS;
  int wmax = 0;   // of the rows that share tiles
  for (int i = 0; i < n; i++)
    if (!is_wide(irp[i + 1] - irp[i])) wmax = std::max(wmax, irp[i + 1] - irp[i]);
  auto row = [&](int t) { return lower ? t : n - 1 - t; };
  auto dep = [&](int e) { return lower ? ja[e] - 1 : n - ja[e]; };
  std::vector<int> tile;
  const int nt = assign_tiles(n, lower, irp, ja, tile);
  // ticket order: tiles by their level in the graph of tiles, so that the
  // tiles that run together are the ones whose turn it is
  std::vector<int> ptr(nt + 1, 0), order(n), tlev(nt, 0), tnew(nt);
  for (int t = 0; t < n; t++) ptr[tile[t] + 1]++;
  for (int k = 0; k < nt; k++) ptr[k + 1] += ptr[k];
  {
    std::vector<int> fill(ptr.begin(), ptr.end() - 1);
    for (int t = 0; t < n; t++) order[fill[tile[t]]++] = t;
  }
  int nlev = 0;
  for (int k = 0; k < nt; k++) {
    int l = 0;
    for (int p = ptr[k]; p < ptr[k + 1]; p++) {
      const int i = row(order[p]);
      for (int e = irp[i] - 1; e < irp[i + 1] - 1; e++) {
        const int q = tile[dep(e)];
        if (q != k) l = std::max(l, tlev[q] + 1);
      }
    }
    tlev[k] = l;
    nlev = std::max(nlev, l + 1);
  }
  std::vector<int> lptr(nlev + 1, 0), byl(nt);
  for (int k = 0; k < nt; k++) lptr[tlev[k] + 1]++;
  for (int l = 0; l < nlev; l++) lptr[l + 1] += lptr[l];
  for (int k = 0; k < nt; k++) byl[lptr[tlev[k]]++] = k;
  // pack the tiles: a step is the tile's rows of one level of the whole
  // triangle, at most 64.  (By levels inside the tile a row whose own chain
  // starts in an earlier tile would sit in the first step and hold up rows
  // that are ready long before: runs of consecutive rows of the L = 110
  // stencil took 70 ms that way.)
  const int width = wmax <= 2 ? 2 : (wmax <= 4 ? wmax : 0);
  std::vector<TriTile> tiles(nt);
  for (int q = 0, pos = 0; q < nt; q++) {
    tiles[q].row0 = pos;
    pos += tiles[q].nrow = ptr[byl[q] + 1] - ptr[byl[q]];
  }
  std::vector<int> trow(n), at(n);   // at: position of a row (solve order) inside its tile
  std::vector<V> tdv(diag ? n : 0);
  TilePack<V> pack[kHostThreads];
  host_parallel(nt, (kHostMin + kTileRows - 1) / kTileRows, [&](int th, int q0, int q1) {
    TilePack<V>& P = pack[th];
    P.q0 = q0;
    P.q1 = q1;
    std::vector<int> begin, fill, trs, key(kHaloHash, 0), where(kHaloHash);
    std::vector<unsigned> stamp(kHaloHash, 0);
    auto lv = [&](int t) { return lev[row(t)]; };
    auto len = [&](int t) { return irp[row(t) + 1] - irp[row(t)]; };
    for (int q = q0; q < q1; q++) {
      const int k = byl[q], nrow = ptr[k + 1] - ptr[k];
      TriTile& D = tiles[q];
      D.ent0 = (int)P.val.size();
      D.step0 = (int)P.step.size();
      D.halo0 = (int)P.halo.size();
      if (nrow == 1 && is_wide(len(order[ptr[k]]))) {   // wide_row
        const int i = row(order[ptr[k]]), b = irp[i] - 1, m = len(order[ptr[k]]);
        trow[D.row0] = i;
        if (diag) tdv[D.row0] = diag[i];
        P.val.insert(P.val.end(), val + b, val + b + m);
        P.dep.resize(P.val.size(), 0);
        for (int e = b; e < b + m; e++) P.halo.push_back(ja[e] - 1);
        D.nent = D.nhalo = m;
        D.nstep = 0;
        P.lds = std::max(P.lds, sizeof(V) * kWideChunk);
        continue;
      }
      // the tile's rows by level; begin: where each level that occurs begins
      trs.assign(order.begin() + ptr[k], order.begin() + ptr[k + 1]);
      int l0 = lv(trs[0]), l1 = l0;
      for (int t : trs) {
        l0 = std::min(l0, lv(t));
        l1 = std::max(l1, lv(t));
      }
      begin.clear();
      if (l1 - l0 < 4 * nrow) {
        fill.assign(l1 - l0 + 2, 0);
        for (int t : trs) fill[lv(t) - l0 + 1]++;
        for (int l = 0; l <= l1 - l0; l++) {
          if (fill[l + 1] > 0) begin.push_back(fill[l]);
          fill[l + 1] += fill[l];
        }
        for (int p = ptr[k]; p < ptr[k + 1]; p++) trs[fill[lv(order[p]) - l0]++] = order[p];
      } else {
        std::stable_sort(trs.begin(), trs.end(), [&](int x, int z) { return lv(x) < lv(z); });
        for (int p = 0; p < nrow; p++)
          if (p == 0 || lv(trs[p]) != lv(trs[p - 1])) begin.push_back(p);
      }
      const int nl = (int)begin.size();
      begin.push_back(nrow);
      if (width == 0)   // longest rows first: a step's rows are at least half as long as its widest
        for (int l = 0; l < nl; l++)
          std::stable_sort(trs.begin() + begin[l], trs.begin() + begin[l + 1],
                           [&](int x, int z) { return len(x) > len(z); });
      for (int p = 0; p < nrow; p++) {
        at[trs[p]] = p;
        trow[D.row0 + p] = row(trs[p]);
        if (diag) tdv[D.row0 + p] = diag[row(trs[p])];
      }
      int nhalo = 0;
      auto slot = [&](int d) {   // LDS slot of the row at d in solve order
        if (tile[d] == k) return at[d];
        unsigned h = (unsigned)d * 2654435761u % kHaloHash;
        while (stamp[h] == (unsigned)q + 1 && key[h] != d) h = (h + 1) % kHaloHash;
        if (stamp[h] != (unsigned)q + 1) {   // first use of an entry outside the tile
          stamp[h] = (unsigned)q + 1;
          key[h] = d;
          where[h] = nrow + nhalo++;
          P.halo.push_back(row(d));
        }
        return where[h];
      };
      for (int l = 0; l < nl; l++)
        for (int r0 = begin[l], c = 0; r0 < begin[l + 1]; r0 += c) {
          const int w = width > 0 ? width : len(trs[r0]);
          c = std::min(kWave, begin[l + 1] - r0);
          if (width == 0)
            for (int p = 1; p < c; p++)
              if (2 * len(trs[r0 + p]) < w) c = p;
          const int e0 = (int)P.val.size() - D.ent0;
          P.step.push_back(make_int2(r0 | c << 16, e0 | w << 16));
          P.val.resize(P.val.size() + (size_t)w * c, V(0));
          P.dep.resize(P.dep.size() + (size_t)w * c, 0xffff);   // padding, set below
          for (int p = r0; p < r0 + c; p++) {
            const int b = irp[row(trs[p])] - 1, m = len(trs[p]);
            for (int u = 0; u < m; u++) {
              const size_t x = (size_t)D.ent0 + e0 + (size_t)u * c + (p - r0);
              P.val[x] = val[b + u];
              P.dep[x] = (uint16_t)slot(dep(b + u));
            }
          }
        }
      D.nhalo = nhalo;
      D.nent = (int)P.val.size() - D.ent0;
      D.nstep = (int)P.step.size() - D.step0;
      for (int e = D.ent0; e < D.ent0 + D.nent; e++)
        if (P.dep[e] == 0xffff) P.dep[e] = (uint16_t)(nrow + nhalo);   // the zero slot
      P.lds = std::max(P.lds, tile_lds<V>(nrow, nhalo, D.nent, D.nstep, diag != nullptr));
    }
  });
  size_t lds = 0, ents = 0, steps = 0, halos = 0;
  for (TilePack<V>& P : pack) {
    for (int q = P.q0; q < P.q1; q++) {
      tiles[q].ent0 += (int)ents;
      tiles[q].step0 += (int)steps;
      tiles[q].halo0 += (int)halos;
    }
    lds = std::max(lds, P.lds);
    ents += P.val.size();
    steps += P.step.size();
    halos += P.halo.size();
    if (ents > (size_t)INT32_MAX) return PSB_HIP_SUCCESS;
  }
  if (lds > kTileLds) return PSB_HIP_SUCCESS;
  int rc = upload(&T.tiles, tiles.data(), tiles.size());
  if (!rc) rc = upload(&T.trow, trow.data(), trow.size());
  if (!rc && diag) rc = upload(&T.tdv, tdv.data(), tdv.size());
  if (rc) return rc;
  hipStream_t s = ctx().stream;
  PSB_HIP_CHECK(hipMalloc((void**)&T.tval, sizeof(V) * std::max<size_t>(ents, 1)));
  PSB_HIP_CHECK(hipMalloc((void**)&T.tdep, sizeof(uint16_t) * std::max<size_t>(ents, 1)));
  PSB_HIP_CHECK(hipMalloc((void**)&T.tstep, sizeof(int2) * std::max<size_t>(steps, 1)));
  PSB_HIP_CHECK(hipMalloc((void**)&T.thalo, sizeof(int) * std::max<size_t>(halos, 1)));
  size_t e0 = 0, s0 = 0, h0 = 0;
  for (const TilePack<V>& P : pack) {
    if (!P.val.empty()) {
      PSB_HIP_CHECK(hipMemcpyAsync(T.tval + e0, P.val.data(), sizeof(V) * P.val.size(),
                                   hipMemcpyHostToDevice, s));
      PSB_HIP_CHECK(hipMemcpyAsync(T.tdep + e0, P.dep.data(), sizeof(uint16_t) * P.dep.size(),
                                   hipMemcpyHostToDevice, s));
    }
    if (!P.step.empty())
      PSB_HIP_CHECK(hipMemcpyAsync(T.tstep + s0, P.step.data(), sizeof(int2) * P.step.size(),
                                   hipMemcpyHostToDevice, s));
    if (!P.halo.empty())
      PSB_HIP_CHECK(hipMemcpyAsync(T.thalo + h0, P.halo.data(), sizeof(int) * P.halo.size(),
                                   hipMemcpyHostToDevice, s));
    e0 += P.val.size();
    s0 += P.step.size();
    h0 += P.halo.size();
  }
  const unsigned long long zero = 0;
  rc = upload(&T.ticket, &zero, 1);
  if (rc) return rc;
  const int64_t nsol = 2 * (int64_t)sol_stride<V>(n);
  PSB_HIP_CHECK(hipMalloc((void**)&T.sol, sizeof(V) * (size_t)nsol));
  hipLaunchKernelGGL((k_tri_unset<V>), dim3(stream_grid(nsol)), dim3(kBlock), 0, s, nsol, T.sol);
  PSB_HIP_LAUNCH_CHECK();
  PSB_HIP_CHECK(hipStreamSynchronize(s));   // the host vectors go out of scope
  T.width = width;
  T.lds = lds;
  T.ntiles = nt;
  return PSB_HIP_SUCCESS;
}

// y = alpha * T^-1 (scale .* x) + beta * y by tiles (scale null: x itself).
// x and y may be the same vector: a tile reads its rows of x before it writes
// its rows of y, and no other tile's.
template <typename V, bool DIV, bool RUN>
static int solve_tiles_t(const TriLevels<V>& T, const V* x, const V* scale, V alpha, V beta, V* y,
                         hipStream_t s) {
#define PSB_TILE_LAUNCH(W)                                                                    \
  hipLaunchKernelGGL((k_trsv_tiles<V, W, DIV, RUN>), dim3(T.ntiles), dim3(kTileThreads), T.lds, \
                     s, sol_stride<V>(T.n), T.ntiles, T.tiles, T.trow, T.tdv, T.tval, T.tdep, T.tstep, T.thalo, \
                     T.sol, T.ticket, x, scale, alpha, beta, y, waits(kTilePolls))
  switch (T.width) {
    case 2: PSB_TILE_LAUNCH(2); break;
    case 3: PSB_TILE_LAUNCH(3); break;
    case 4: PSB_TILE_LAUNCH(4); break;
    default: PSB_TILE_LAUNCH(0); break;
  }
#undef PSB_TILE_LAUNCH
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

template <typename V>
static int solve_tiles(const TriLevels<V>& T, bool run, const V* x, const V* scale, V alpha,
                       V beta, V* y, hipStream_t s) {
  if (T.tdv && run) return solve_tiles_t<V, true, true>(T, x, scale, alpha, beta, y, s);
  if (T.tdv) return solve_tiles_t<V, true, false>(T, x, scale, alpha, beta, y, s);
  if (run) return solve_tiles_t<V, false, true>(T, x, scale, alpha, beta, y, s);
  return solve_tiles_t<V, false, false>(T, x, scale, alpha, beta, y, s);
}

// How a triangle is solved: as its shape decides, as tiles where they can, or
// by levels.
enum TriForm { TRI_AUTO, TRI_TILES, TRI_LEVELS };

// Levels up to which a launch per level is at least as fast as tiles: 2
// levels of 500,000 rows 61 against 71 us, a diagonal of a million rows 36
// against 40 us; a launch is about 3 us, so from 5 levels on tiles win (38
// levels of 20,000 rows 634 against 182 us).
constexpr int kFewLevels = 4;

// The triangle (diag: its diagonal, null for a unit one) as tiles, or in level
// order with the launch-per-level variant, with few levels and where tiles
// refuse.
template <typename V>
static int upload_tri(TriLevels<V>& T, int n, bool lower, const int* irp, const int* ja,
                      const V* val, const V* diag, TriForm form = TRI_AUTO) {
  T.n = n;
  T.nnz = irp[n] - 1;
  for (int i = 0; i < n; i++)
    for (int p = irp[i] - 1; p < irp[i + 1] - 1; p++) {
      const int c = ja[p];
      if (c < 1 || c > n || (lower ? c > i : c < i + 2))
        return set_error(PSB_HIP_INVALID, "trsv", "entry outside its triangle");
    }
  std::vector<int> lev;
  T.nlev = count_levels(n, lower, irp, ja, lev);
  if (form != TRI_LEVELS && g_trsv_variant != 1 && (form == TRI_TILES || T.nlev > kFewLevels)) {
    const int rc = plan_tiles(T, lower, irp, ja, val, diag, lev);
    if (rc || T.ntiles > 0) return rc;
  }
  std::vector<int> rows;
  order_levels(n, T.nlev, lev, rows, T.lev_ptr);
  std::vector<int> pos(n > 0 ? n : 1, 0);
  for (int p = 0; p < n; p++) pos[rows[p]] = p;
  // the triangle in level order: row rows[p] becomes position p, its entries
  // keep their CSR order and point at the positions of their columns
  std::vector<int> pirp(n + 1, 0), pja(T.nnz > 0 ? T.nnz : 1, 0);
  std::vector<V> pval(T.nnz > 0 ? T.nnz : 1, V(0));
  for (int p = 0; p < n; p++) {
    const int i = rows[p], b = irp[i] - 1, c = irp[i + 1] - 1 - b;
    for (int k = 0; k < c; k++) {
      pja[pirp[p] + k] = pos[ja[b + k] - 1];
      pval[pirp[p] + k] = val[b + k];
    }
    pirp[p + 1] = pirp[p] + c;
  }
  int rc = upload(&T.irp, pirp.data(), pirp.size());
  if (!rc) rc = upload(&T.ja, pja.data(), pja.size());
  if (!rc) rc = upload(&T.val, pval.data(), pval.size());
  if (!rc) rc = upload(&T.perm, rows.data(), rows.size());
  if (rc) return rc;
  PSB_HIP_CHECK(hipStreamSynchronize(ctx().stream));   // the host vectors go out of scope
  return PSB_HIP_SUCCESS;
}

// x and y in level order; dv the diagonal in level order (null: unit);
// run: rows by running subtraction (the transposed solve)
template <typename V, bool DIV, bool RUN>
static void enqueue_levels_t(const TriLevels<V>& T, const V* dv, const V* x, V* y,
                             hipStream_t s) {
  for (int l = 0; l < T.nlev; l++) {
    const int count = T.lev_ptr[l + 1] - T.lev_ptr[l];
    hipLaunchKernelGGL((k_trsv_level<V, DIV, RUN>), dim3((count + kBlock - 1) / kBlock),
                       dim3(kBlock), 0, s, T.lev_ptr[l], count, T.irp, T.ja, T.val, dv, x, y);
  }
}

template <typename V>
static void enqueue_levels(const TriLevels<V>& T, const V* dv, bool run, const V* x, V* y,
                           hipStream_t s) {
  if (dv && run) enqueue_levels_t<V, true, true>(T, dv, x, y, s);
  else if (dv) enqueue_levels_t<V, true, false>(T, dv, x, y, s);
  else if (run) enqueue_levels_t<V, false, true>(T, dv, x, y, s);
  else enqueue_levels_t<V, false, false>(T, dv, x, y, s);
}

// The captured part of a launch-per-level application: x in L level order (xa) -> U^-1
// (d .* L^-1 x) in U level order (ya).  The gather of the caller's x and the
// scatter into the caller's y (with alpha and beta) run around it.
static void enqueue_apply(IluDev* F, hipStream_t s) {
  const int n = F->n, g = stream_grid(n);
  enqueue_levels<double>(F->L, nullptr, false, F->xa, F->ya, s);
  hipLaunchKernelGGL(k_perm_scatter<double>, dim3(g), dim3(kBlock), 0, s, n, F->L.perm, F->ya,
                     F->t1);
  hipLaunchKernelGGL(k_perm_gather<double>, dim3(g), dim3(kBlock), 0, s, n, F->U.perm, F->t1,
                     F->d, F->xa);
  enqueue_levels<double>(F->U, nullptr, false, F->xa, F->ya, s);
}

// The host planning f behind a C entry point, out of host memory as a return code.
template <typename F>
static int plan(F f) {
  try {
    return f();
  } catch (const std::bad_alloc&) {
    return set_error(PSB_HIP_OUTOFMEM, "trsv", "host memory");
  } catch (const std::exception& e) {
    return set_error(PSB_HIP_RUNTIME, "trsv", e.what());
  }
}

template <typename V>
static void free_tri(TriLevels<V>& T) {
  void* p[] = {T.perm, T.irp, T.ja, T.val, T.tiles, T.trow, T.tdv, T.tval, T.tdep, T.tstep,
               T.thalo, T.sol, T.ticket};
  for (void* q : p)
    if (q) (void)hipFree(q);
  T = TriLevels<V>{};
}

static void destroy_ilu(IluDev* F) {
  if (!F) return;
  if (ctx().initialized) (void)hipStreamSynchronize(ctx().stream);
  if (F->exec) (void)hipGraphExecDestroy(F->exec);
  if (F->graph) (void)hipGraphDestroy(F->graph);
  free_tri(F->L);
  free_tri(F->U);
  void* p[] = {F->d, F->xa, F->ya, F->t1};
  for (void* q : p)
    if (q) (void)hipFree(q);
  delete F;
}

template <typename V>
static void destroy_sv(TriSolve<V>* S) {
  if (!S) return;
  if (ctx().initialized) (void)hipStreamSynchronize(ctx().stream);
  if (S->exec) (void)hipGraphExecDestroy(S->exec);
  if (S->graph) (void)hipGraphDestroy(S->graph);
  free_tri(S->tl);
  void* p[] = {S->dv, S->xa, S->ya};
  for (void* q : p)
    if (q) (void)hipFree(q);
  delete S;
}

// Prepares op(T)^-1 for the CSR triangle (irp, ja, val), 1-based host
// arrays: the diagonal of a non-unit row (its last entry if lower, first if
// upper, the entries psb_d_csr_cssv divides by) is taken out, the rest must
// lie strictly inside the triangle.  For op 'T' / 'C' the strict part is
// transposed with row c's entries in the CPU's update order: the rows i of T
// in solve order (descending for a lower triangle), CSR order within a row.
template <typename V>
static int build_sv(TriSolve<V>* S, int n, const int* irp, const int* ja, const V* val,
                    bool lower, bool unit, bool trans) {
  S->n = n;
  S->run = trans;
  const int nnz = irp[n] - 1;
  std::vector<int> sirp(n + 1, 1), sja;
  std::vector<V> sval, dv;
  sja.reserve(nnz > 0 ? nnz : 1);
  sval.reserve(nnz > 0 ? nnz : 1);
  if (!unit) dv.resize(n > 0 ? n : 1);
  for (int i = 0; i < n; i++) {
    int b = irp[i] - 1, e = irp[i + 1] - 1;
    if (!unit) {
      if (e <= b) return set_error(PSB_HIP_INVALID, "trsv", "non-unit row without entries");
      if (lower) dv[i] = val[--e];
      else dv[i] = val[b++];
    }
    for (int k = b; k < e; k++) {
      sja.push_back(ja[k]);
      sval.push_back(val[k]);
    }
    sirp[i + 1] = (int)sja.size() + 1;
  }
  bool tlower = lower;
  if (trans) {
    for (int i = 0; i < n; i++)   // the strict part must be a triangle before it is turned
      for (int k = sirp[i] - 1; k < sirp[i + 1] - 1; k++)
        if (sja[k] < 1 || sja[k] > n || (lower ? sja[k] > i : sja[k] < i + 2))
          return set_error(PSB_HIP_INVALID, "trsv", "entry outside its triangle");
    const int snz = sirp[n] - 1;
    std::vector<int> cnt(n + 1, 0);
    for (int k = 0; k < snz; k++) cnt[sja[k]]++;
    std::vector<int> tirp(n + 1, 1);
    for (int c = 0; c < n; c++) tirp[c + 1] = tirp[c] + cnt[c + 1];
    std::vector<int> fill(tirp.begin(), tirp.end() - 1), tja(snz > 0 ? snz : 1);
    std::vector<V> tval(snz > 0 ? snz : 1);
    for (int t = 0; t < n; t++) {
      const int i = lower ? n - 1 - t : t;   // the CPU's order of the rows
      for (int k = sirp[i] - 1; k < sirp[i + 1] - 1; k++) {
        const int q = fill[sja[k] - 1]++ - 1;
        tja[q] = i + 1;
        tval[q] = sval[k];
      }
    }
    sirp.swap(tirp);
    sja.swap(tja);
    sval.swap(tval);
    tlower = !lower;
  }
  int rc = upload_tri(S->tl, n, tlower, sirp.data(), sja.data(), sval.data(),
                      unit ? (const V*)nullptr : dv.data());
  if (rc || S->tl.ntiles > 0) return rc;
  const size_t nb = sizeof(V) * (size_t)(n > 0 ? n : 1);
  hipError_t e = hipSuccess;
  V** bufs[] = {&S->xa, &S->ya};
  for (V** b : bufs)
    if (e == hipSuccess) e = hipMalloc((void**)b, nb);
  hipStream_t s = ctx().stream;
  if (e == hipSuccess && !unit && n > 0) {   // the diagonal, gathered into level order
    e = hipMalloc((void**)&S->dv, nb);
    if (e == hipSuccess) e = hipMemcpy(S->xa, dv.data(), nb, hipMemcpyHostToDevice);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(k_perm_gather<V>, dim3(stream_grid(n)), dim3(kBlock), 0, s, n,
                         S->tl.perm, S->xa, (const V*)nullptr, S->dv);
      e = hipStreamSynchronize(s);
    }
  }
  if (e == hipSuccess && n > 0) {
    e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
      enqueue_levels<V>(S->tl, S->dv, S->run, S->xa, S->ya, s);
      e = hipStreamEndCapture(s, &S->graph);
    }
    if (e == hipSuccess) e = hipGraphInstantiate(&S->exec, S->graph, nullptr, nullptr, 0);
  }
  if (e != hipSuccess)
    return set_error(e == hipErrorOutOfMemory ? PSB_HIP_OUTOFMEM : PSB_HIP_RUNTIME, "trsv",
                     hipGetErrorString(e));
  return PSB_HIP_SUCCESS;
}

template <typename V>
static int csr_sv_build(TriSolve<V>* S, const CsrDev* m, int key) {
  std::vector<int> irp(m->rows + 1), ja(m->nnz > 0 ? m->nnz : 1);
  std::vector<V> val(m->nnz > 0 ? m->nnz : 1);
  hipStream_t s = ctx().stream;
  PSB_HIP_CHECK(hipMemcpyAsync(irp.data(), m->irp, sizeof(int) * irp.size(),
                               hipMemcpyDeviceToHost, s));
  if (m->nnz > 0) {
    PSB_HIP_CHECK(hipMemcpyAsync(ja.data(), m->ja, sizeof(int) * (size_t)m->nnz,
                                 hipMemcpyDeviceToHost, s));
    PSB_HIP_CHECK(hipMemcpyAsync(val.data(), m->val, sizeof(V) * (size_t)m->nnz,
                                 hipMemcpyDeviceToHost, s));
  }
  PSB_HIP_CHECK(hipStreamSynchronize(s));
  return build_sv<V>(S, m->rows, irp.data(), ja.data(), val.data(), (key & 1) != 0,
                     (key & 2) != 0, (key & 4) != 0);
}

// The CSR matrix's prepared solve for key (lower | unit << 1 | trans << 2),
// built from the device copy of the matrix on first use and kept until the
// matrix is rewritten, freed or asked for another triangle or op.
template <typename V>
static int csr_sv_get(CsrDev* m, int key, TriSolve<V>** out) {
  TriSolve<V>* S = (TriSolve<V>*)m->sv;
  if (S && S->key == key) {
    *out = S;
    return PSB_HIP_SUCCESS;
  }
  release_csr_sv(m);
  S = new TriSolve<V>();
  const int rc = plan([&] { return csr_sv_build(S, m, key); });
  if (rc) {
    destroy_sv(S);
    return rc;
  }
  S->key = key;
  m->sv = S;
  *out = S;
  return PSB_HIP_SUCCESS;
}

template <typename V>
static int csr_sv_apply(CsrDev* m, int key, V alpha, const MultiVec* x, V beta, MultiVec* y) {
  TriSolve<V>* S = nullptr;
  int rc = csr_sv_get<V>(m, key, &S);
  if (rc) return rc;
  hipStream_t s = ctx().stream;
  const int n = S->n, g = stream_grid(n);
  for (int c = 0; c < x->count; c++) {
    const V* xc = (const V*)x->v + (size_t)c * x->pitch;
    V* yc = (V*)y->v + (size_t)c * y->pitch;
    if (S->tl.ntiles > 0) {
      if ((rc = solve_tiles<V>(S->tl, S->run, xc, nullptr, alpha, beta, yc, s))) return rc;
      continue;
    }
    hipLaunchKernelGGL(k_perm_gather<V>, dim3(g), dim3(kBlock), 0, s, n, S->tl.perm, xc,
                       (const V*)nullptr, S->xa);
    PSB_HIP_LAUNCH_CHECK();
    PSB_HIP_CHECK(hipGraphLaunch(S->exec, s));
    hipLaunchKernelGGL(k_perm_scatter_axpby<V>, dim3(g), dim3(kBlock), 0, s, n, S->tl.perm,
                       S->ya, alpha, beta, yc);
    PSB_HIP_LAUNCH_CHECK();
  }
  return PSB_HIP_SUCCESS;
}

void release_csr_sv(CsrDev* m) {
  if (!m || !m->sv) return;
  if (m->elem_type == PSB_HIP_TYPE_DOUBLE) destroy_sv((TriSolve<double>*)m->sv);
  else destroy_sv((TriSolve<float>*)m->sv);
  m->sv = nullptr;
}

}  // namespace psbhip

using namespace psbhip;

extern "C" {

int psb_hip_ilu_alloc(void** ilu, int n, const int* lirp, const int* lja, const double* lval,
                      const int* uirp, const int* uja, const double* uval, const double* d) {
  PSB_ENSURE_INIT();
  if (!ilu || n < 0 || !lirp || !uirp || !d) return PSB_HIP_INVALID;
  *ilu = nullptr;
  IluDev* F = new IluDev();
  F->n = n;
  int rc = PSB_HIP_SUCCESS;
  for (TriForm form : {TRI_AUTO, TRI_TILES, TRI_LEVELS}) {   // both factors in the same form
    free_tri(F->L);
    free_tri(F->U);
    rc = plan([&] {
      const int rl = upload_tri(F->L, n, true, lirp, lja, lval, (const double*)nullptr, form);
      return rl ? rl : upload_tri(F->U, n, false, uirp, uja, uval, (const double*)nullptr, form);
    });
    if (rc || (F->L.ntiles > 0) == (F->U.ntiles > 0)) break;
  }
  if (rc) {
    destroy_ilu(F);
    return rc;
  }
  const size_t nb = sizeof(double) * (size_t)(n > 0 ? n : 1);
  hipError_t e = hipSuccess;
  // both factors as tiles, or the levels of both in one graph
  const bool tiled = F->L.ntiles > 0 && F->U.ntiles > 0;
  double** bufs[] = {&F->d, &F->t1, &F->xa, &F->ya};
  for (int k = 0; k < (tiled ? 2 : 4); k++)
    if (e == hipSuccess) e = hipMalloc((void**)bufs[k], nb);
  if (e == hipSuccess && n > 0)
    e = hipMemcpy(F->d, d, sizeof(double) * (size_t)n, hipMemcpyHostToDevice);
  if (e == hipSuccess && n > 0 && !tiled) {
    hipStream_t s = ctx().stream;
    e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
      enqueue_apply(F, s);
      e = hipStreamEndCapture(s, &F->graph);
    }
    if (e == hipSuccess) e = hipGraphInstantiate(&F->exec, F->graph, nullptr, nullptr, 0);
  }
  if (e != hipSuccess) {
    destroy_ilu(F);
    return set_error(e == hipErrorOutOfMemory ? PSB_HIP_OUTOFMEM : PSB_HIP_RUNTIME, __func__,
                     hipGetErrorString(e));
  }
  *ilu = F;
  return PSB_HIP_SUCCESS;
}

int psb_hip_ilu_set_variant(int variant) {
  const int old = g_trsv_variant;
  if (variant == 0 || variant == 1) g_trsv_variant = variant;
  return old;
}

int psb_hip_ilu_segments(void* ilu, int* lower_segments, int* upper_segments) {
  IluDev* F = (IluDev*)ilu;
  if (!F) return PSB_HIP_INVALID;
  if (lower_segments) *lower_segments = F->L.ntiles;
  if (upper_segments) *upper_segments = F->U.ntiles;
  return PSB_HIP_SUCCESS;
}

int psb_hip_ilu_free(void* ilu) {
  destroy_ilu((IluDev*)ilu);
  return PSB_HIP_SUCCESS;
}

int psb_hip_ilu_levels(void* ilu, int* lower_levels, int* upper_levels) {
  IluDev* F = (IluDev*)ilu;
  if (!F) return PSB_HIP_INVALID;
  if (lower_levels) *lower_levels = F->L.nlev;
  if (upper_levels) *upper_levels = F->U.nlev;
  return PSB_HIP_SUCCESS;
}

int psb_hip_ilu_apply(void* ilu, double alpha, void* xv, double beta, void* yv) {
  PSB_ENSURE_INIT();
  IluDev* F = (IluDev*)ilu;
  MultiVec *x = (MultiVec*)xv, *y = (MultiVec*)yv;
  if (!F || !x || !y || x->elem_type != PSB_HIP_TYPE_DOUBLE || y->elem_type != PSB_HIP_TYPE_DOUBLE ||
      x->size < F->n || y->size < F->n || x->count != 1 || y->count != 1)
    return set_error(PSB_HIP_INVALID, __func__, "x/y type or size");
  if (F->n == 0) return PSB_HIP_SUCCESS;
  hipStream_t s = ctx().stream;
  if (!F->exec) {   // t1 = L^-1 x, then y = alpha U^-1 (d .* t1) + beta y
    int rc = solve_tiles<double>(F->L, false, (const double*)x->v, nullptr, 1.0, 0.0, F->t1, s);
    if (!rc)
      rc = solve_tiles<double>(F->U, false, F->t1, F->d, alpha, beta, (double*)y->v, s);
    return rc;
  }
  const int n = F->n, g = stream_grid(n);
  hipLaunchKernelGGL(k_perm_gather<double>, dim3(g), dim3(kBlock), 0, s, n, F->L.perm,
                     (const double*)x->v, (const double*)nullptr, F->xa);
  PSB_HIP_LAUNCH_CHECK();
  PSB_HIP_CHECK(hipGraphLaunch(F->exec, s));
  hipLaunchKernelGGL(k_perm_scatter_axpby<double>, dim3(g), dim3(kBlock), 0, s, n, F->U.perm,
                     F->ya, alpha, beta, (double*)y->v);
  PSB_HIP_LAUNCH_CHECK();
  return PSB_HIP_SUCCESS;
}

int psb_hip_csr_spsv(void* dmat, int lower, int unit, int trans, double alpha, void* xv,
                     double beta, void* yv) {
  PSB_ENSURE_INIT();
  CsrDev* m = (CsrDev*)dmat;
  MultiVec *x = (MultiVec*)xv, *y = (MultiVec*)yv;
  if (!m || !x || !y) return set_error(PSB_HIP_INVALID, __func__, "null argument");
  if (m->rows != m->cols) return set_error(PSB_HIP_INVALID, __func__, "matrix not square");
  if (trans < 0 || trans > 2) return set_error(PSB_HIP_INVALID, __func__, "trans");
  if (x->elem_type != m->elem_type || y->elem_type != m->elem_type || x->size < m->rows ||
      y->size < m->rows || x->count != y->count)
    return set_error(PSB_HIP_INVALID, __func__, "x/y type, size or count");
  if (m->rows == 0) return PSB_HIP_SUCCESS;
  const int key = (lower ? 1 : 0) | (unit ? 2 : 0) | (trans ? 4 : 0);
  if (m->elem_type == PSB_HIP_TYPE_DOUBLE)
    return csr_sv_apply<double>(m, key, alpha, x, beta, y);
  return csr_sv_apply<float>(m, key, (float)alpha, x, (float)beta, y);
}

int psb_hip_csr_spsv_levels(void* dmat, int* levels, int* segments) {
  CsrDev* m = (CsrDev*)dmat;
  if (!m) return PSB_HIP_INVALID;
  int nl = 0, ns = 0;
  if (m->sv && m->elem_type == PSB_HIP_TYPE_DOUBLE) {
    nl = ((TriSolve<double>*)m->sv)->tl.nlev;
    ns = ((TriSolve<double>*)m->sv)->tl.ntiles;
  } else if (m->sv) {
    nl = ((TriSolve<float>*)m->sv)->tl.nlev;
    ns = ((TriSolve<float>*)m->sv)->tl.ntiles;
  }
  if (levels) *levels = nl;
  if (segments) *segments = ns;
  return PSB_HIP_SUCCESS;
}

}  // extern "C"
