// qh_comp.hip -- RK4 of a constant generator, one closed set of rows per workgroup.
//
// Generators of open systems often fall apart: a jump and the coherent term that
// goes with it move a row index of rho and its column index together, so a
// conserved difference (excitation numbers, the bits in which the two indices
// differ) splits the rows into sets that no entry connects.  Within such a set the
// whole integration needs nobody else: a workgroup keeps the set's vector in LDS
// and its matrix entries in registers and runs every step of a call, so a call
// reads and writes the state once instead of three vector passes and a launch per
// stage.
//
// Plan (once per matrix): connected components of the sparsity pattern (the
// lock-free union find of Anderson & Woll 1991 with the path halving of Tarjan & van
// Leeuwen 1984), components packed into bins of whole components, rows sorted within a bin.
// A bin's rows are stored in slices of 64 (one wavefront): the diagonal apart, and
// every other entry as one or two real entries, first the imaginary parts (an even
// number of slots a slice), then the real parts, each a value and the 16-bit index
// of its column within the bin.
//
// A set too large for that keeps its vector in LDS and reads its entries at every
// stage, as 32-bit words of a column and an index into the bin's table of distinct
// values (an entry repeats a few products of couplings and square roots).
//
// What bounds it: at few bins the chain of LDS reads of one stage and its barrier
// (0.3 to 1.5 us a stage, where a launch a stage takes 2.6 to 4.3 us), at many
// the LDS reads, 16 B an entry: 12-qubit circuit (decay and dephasing), 10 steps of
// 16.8 M rows in 1.4 ms, four launches a step of 233 us before; 512 systems of 100 to
// 230 400 rows in FP32, 10 steps of 16 M rows in 3.7 ms, 8.4 ms before.
#include <algorithm>
#include <memory>
#include <string>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "qh_common.h"
#include "qh_comp_plan.h"
#include "qh_optional.h"

namespace {

const int CP_GRAN = 64;         // rows of a granule: the components that start in 64 consecutive sorted rows
const int CP_DICT_W = 12;       // words of a row fetched ahead
const size_t CP_SCRATCH = (size_t)64 << 20;  // workspace taken from the library's scratch
const int CP_PROBE_ROWS = 16384;  // rows looked at before a large matrix as a whole
const int CP_PACK_ROWS = 512;   // bins of small components are filled to this size once they outnumber the CUs

// -------------------------------------------------------------- components
// Parents only ever decrease.  The loads are ordinary cached ones: a value read late
// is still an ancestor, and only the device-scope exchange that hangs one root below
// another has to see the present one, which it returns when it fails.  (With every
// load at device scope the 16 M rows of a sweep of 512 systems took 20 ms.)
__device__ inline int32_t cc_load(const int32_t *p, int32_t i) {
  return __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline void cc_store(int32_t *p, int32_t i, int32_t v) {
  __hip_atomic_store(p + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ inline int32_t cc_find(int32_t *p, int32_t i) {
  int32_t q = cc_load(p, i);
  while (q != i) {
    const int32_t g = cc_load(p, q);
    if (g != q) cc_store(p, i, g);
    i = q;
    q = g;
  }
  return i;
}

__global__ void k_cc_init(int32_t *parent, int32_t *size, int32_t n) {
  for (int64_t r = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
    parent[r] = (int32_t)r;
    size[r] = 0;
  }
}

// rows r0 .. r0 + n, and the entries between them (indices from r0)
__global__ void __launch_bounds__(256) k_cc_hook(int32_t *parent, const int32_t *__restrict__ rp,
                                                 const int32_t *__restrict__ col, int32_t r0, int32_t n) {
  const int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (r >= n) return;
  int32_t a = (int32_t)r;
  const int32_t end = rp[r0 + r + 1];
  for (int32_t e = rp[r0 + r]; e < end; e += 4) {
    int32_t c[4];  // four entries' columns and their parents in flight together
#pragma unroll
    for (int k = 0; k < 4; k++) c[k] = e + k < end ? col[e + k] - r0 : (int32_t)r;
#pragma unroll
    for (int k = 0; k < 4; k++) c[k] = c[k] < 0 || c[k] >= n ? (int32_t)r : c[k];
#pragma unroll
    for (int k = 0; k < 4; k++) c[k] = c[k] == (int32_t)r ? a : cc_load(parent, c[k]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      int32_t b = c[k];
      while (b != a) {  // the larger root below the smaller one; the larger index decreases every round
        a = cc_find(parent, a);
        b = cc_find(parent, b);
        if (a == b) break;
        const int32_t hi = a > b ? a : b, lo = a > b ? b : a;
        const int32_t old = atomicCAS(parent + hi, hi, lo);
        if (old == hi) {
          a = lo;
          break;
        }
        cc_store(parent, hi, old);  // what this die's cache still held as a root
        a = lo;
        b = old;
      }
    }
  }
}

// The root of every row, and the rows of every root.  A block counts its 1024 rows by
// root in an LDS table first: a few large components would otherwise queue a global
// atomic per row (0.25 ms for 230 400 rows in 67 of them).
const int CC_LABEL_ROWS = 1024;
__global__ void __launch_bounds__(256) k_cc_label(int32_t *parent, int32_t *lab, int32_t *size, int32_t n) {
  __shared__ int32_t key[2 * CC_LABEL_ROWS], cnt[2 * CC_LABEL_ROWS];
  for (int i = threadIdx.x; i < 2 * CC_LABEL_ROWS; i += 256) {
    key[i] = -1;
    cnt[i] = 0;
  }
  __syncthreads();
  for (int k = 0; k < CC_LABEL_ROWS; k += 256) {
    const int64_t r = (int64_t)blockIdx.x * CC_LABEL_ROWS + k + threadIdx.x;
    if (r >= n) break;
    const int32_t l = cc_find(parent, (int32_t)r);
    lab[r] = l;
    unsigned h = ((unsigned)l * 2654435761u) >> 21;  // 11 bits: the table's size, half of it used at most
    for (;;) {
      const int32_t old = atomicCAS(&key[h], -1, l);
      if (old == -1 || old == l) break;
      h = (h + 1) & (2 * CC_LABEL_ROWS - 1);
    }
    atomicAdd(&cnt[h], 1);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 2 * CC_LABEL_ROWS; i += 256)
    if (cnt[i]) atomicAdd(size + key[i], cnt[i]);
}

__global__ void k_cc_largest(const int32_t *size, int32_t *out, int32_t n) {
  int32_t m = 0;
  for (int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x; r < n; r += (int64_t)gridDim.x * 256) m = max(m, size[r]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(out, m);
}

__global__ void k_cc_granules(const int32_t *size, const int32_t *off, int32_t *gsize, int32_t n) {
  const int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (r < n && size[r]) atomicAdd(gsize + off[r] / CP_GRAN, size[r]);
}

// ------------------------------------------------------------------- plan
__global__ void k_cp_keys(const int32_t *lab, const int32_t *off, const int32_t *gbin, int32_t *key, int32_t *row,
                          int32_t n) {
  const int64_t r = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (r >= n) return;
  key[r] = gbin[off[lab[r]] / CP_GRAN];
  row[r] = (int32_t)r;
}

__global__ void k_cp_fill_order(int32_t *order, int64_t n) {
  const int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (i < n) order[i] = -1;
}

// sorted position q -> padded position, and the row's index within its bin
__global__ void k_cp_place(const int32_t *key, const int32_t *row, const int32_t *brow, const int32_t *bslice,
                           int32_t *order, int32_t *pos, int32_t n) {
  const int64_t q = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (q >= n) return;
  const int32_t b = key[q], at = (int32_t)q - brow[b];
  order[(int64_t)bslice[b] * 64 + at] = row[q];
  pos[row[q]] = at;
}

__device__ inline int32_t cp_wave_max(int32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// f(column, value) of row r's entries off the diagonal, the loads of four entries in
// flight together; the diagonal entry (zero where there is none) is returned
template <typename F>
__device__ __forceinline__ double2 cp_entries(int32_t r, const int32_t *__restrict__ rp,
                                              const int32_t *__restrict__ col, const double2 *__restrict__ val, F &&f) {
  double2 d = make_double2(0.0, 0.0);
  const int32_t end = rp[r + 1];
  for (int32_t e = rp[r]; e < end; e += 4) {
    int32_t c[4];
    double2 v[4];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int32_t q = min(e + k, end - 1);
      c[k] = col[q];
      v[k] = val[q];
    }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (e + k >= end) break;
      if (c[k] == r)
        d = v[k];
      else
        f(c[k], v[k]);
    }
  }
  return d;
}

// slots of every slice: imaginary parts (made even) and all (count: the slices'
// number where only the device has it)
__global__ void __launch_bounds__(256) k_cp_width(const int32_t *order, const int32_t *__restrict__ rp,
                                                  const int32_t *__restrict__ col, const double2 *__restrict__ val,
                                                  int32_t *width, int32_t *nim, int32_t nslices,
                                                  const int32_t *count) {
  const int32_t s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= (count ? *count : nslices)) return;
  const int32_t r = order[(int64_t)s * 64 + lane];
  int32_t ni = 0, nr = 0;
  if (r >= 0)
    cp_entries(r, rp, col, val, [&](int32_t, double2 v) {
      ni += v.y != 0.0;
      nr += v.x != 0.0;
    });
  ni = (cp_wave_max(ni) + 1) & ~1;
  nr = cp_wave_max(nr);
  if (lane == 0) {
    width[s] = ni + nr;
    nim[s] = ni;
  }
}

// the diagonal of every slice, and the entries of those whose bin holds them in
// registers; zc[s]: index of the bin's zero cell, read by the slots that a row does
// not fill, or -1 where the bin reads words
__global__ void __launch_bounds__(256) k_cp_fill(const int32_t *order, const int32_t *pos,
                                                 const int32_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                 const double2 *__restrict__ val, const int32_t *soff,
                                                 const int32_t *width, const int32_t *nim, const int32_t *zc,
                                                 double2 *diag, double *ev, uint16_t *ec, int32_t nslices) {
  const int32_t s = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (s >= nslices) return;
  const int32_t r = order[(int64_t)s * 64 + lane];
  const bool reg = zc[s] >= 0;
  const int64_t s0 = soff[s], s1 = s0 + width[s];
  int64_t pi = s0, pr = s0 + nim[s];
  double2 d = make_double2(0.0, 0.0);
  auto put = [&](int64_t slot, double v, int32_t c) {
    ev[slot * 64 + lane] = v;
    ec[slot * 64 + lane] = (uint16_t)c;
  };
  if (r >= 0)
    d = cp_entries(r, rp, col, val, [&](int32_t q, double2 v) {
      if (!reg) return;
      const int32_t c = pos[q];
      if (v.y != 0.0) put(pi++, v.y, c);
      if (v.x != 0.0) put(pr++, v.x, c);
    });
  diag[(int64_t)s * 64 + lane] = d;
  if (!reg) return;
  for (; pi < s0 + nim[s]; pi++) put(pi, 0.0, zc[s]);
  for (; pr < s1; pr++) put(pr, 0.0, zc[s]);
}

// The table and the words of one bin a workgroup: every distinct value of an entry
// goes through a hash table in LDS (open addressing; the host takes the plan back
// when a bin has more than CP_DICT - 1).  A word is the column's index plus one
// (cell 0 is the zero cell) and, above it, the byte offset of the value.
__global__ void __launch_bounds__(1024) k_cp_dict(const int32_t *bins, const int32_t *bslice, const int32_t *order,
                                                  const int32_t *pos, const int32_t *__restrict__ rp,
                                                  const int32_t *__restrict__ col, const double2 *__restrict__ val,
                                                  const int32_t *soff, const int32_t *width, const int32_t *nim,
                                                  uint32_t *ew, double *dict, int32_t *overflow) {
  const int CELLS = 4 * CP_DICT;
  __shared__ unsigned long long key[CELLS];
  __shared__ int32_t id[CELLS], count;
  const int32_t sl0 = bslice[bins[blockIdx.x]], nsl = bslice[bins[blockIdx.x] + 1] - sl0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < CELLS; i += 1024) key[i] = 0ull;
  if (threadIdx.x == 0) count = 0;
  __syncthreads();
  auto cell = [&](double v, bool insert) -> int {
    const unsigned long long k = (unsigned long long)__double_as_longlong(v);
    unsigned h = (unsigned)((k * 0x9E3779B97F4A7C15ull) >> 52) & (CELLS - 1);
    for (int i = 0; i < CELLS; i++, h = (h + 1) & (CELLS - 1)) {
      unsigned long long old = *(volatile unsigned long long *)&key[h];
      if (old == 0ull && insert) {
        old = atomicCAS(&key[h], 0ull, k);
        if (old == 0ull) {
          atomicAdd(&count, 1);
          return (int)h;
        }
      }
      if (old == k) return (int)h;
    }
    return 0;  // full: the bin overflows
  };
  // a bin over the limit stops taking values, long before the table is full
  for (int32_t s = wave; s < nsl; s += 16) {
    const int32_t r = order[(int64_t)(sl0 + s) * 64 + lane];
    if (r < 0 || *(volatile int32_t *)&count >= CP_DICT) continue;
    cp_entries(r, rp, col, val, [&](int32_t, double2 v) {
      if (v.y != 0.0) cell(v.y, true);
      if (v.x != 0.0) cell(v.x, true);
    });
  }
  __syncthreads();
  const bool over = count >= CP_DICT;
  __syncthreads();
  if (threadIdx.x == 0) {
    if (over) overflow[0] = 1;
    count = 1;
    dict[(int64_t)blockIdx.x * CP_DICT] = 0.0;
  }
  if (over) return;  // the whole workgroup
  __syncthreads();
  for (int i = threadIdx.x; i < CELLS; i += 1024)
    if (key[i]) {
      id[i] = atomicAdd(&count, 1);
      dict[(int64_t)blockIdx.x * CP_DICT + id[i]] = __longlong_as_double((long long)key[i]);
    }
  __syncthreads();
  for (int32_t s = wave; s < nsl; s += 16) {
    const int32_t r = order[(int64_t)(sl0 + s) * 64 + lane];
    const int64_t s0 = soff[sl0 + s], s1 = s0 + width[sl0 + s];
    int64_t pi = s0, pr = s0 + nim[sl0 + s];
    const int64_t p1 = pr;
    auto put = [&](int64_t slot, double v, int32_t c) {
      ew[slot * 64 + lane] = (uint32_t)(pos[c] + 1) | ((uint32_t)id[cell(v, false)] * 8u) << 16;
    };
    if (r >= 0)
      cp_entries(r, rp, col, val, [&](int32_t c, double2 v) {
        if (v.y != 0.0) put(pi++, v.y, c);
        if (v.x != 0.0) put(pr++, v.x, c);
      });
    for (; pi < p1; pi++) ew[pi * 64 + lane] = 0u;
    for (; pr < s1; pr++) ew[pr * 64 + lane] = 0u;
  }
}

// ------------------------------------------------------- plan of a small matrix
// A matrix of up to CP_SMALL_ROWS rows has its components, bins and order formed by
// one workgroup in LDS and its offsets by another, so that a new parameter set waits
// for the device once (four integers) and not for a dozen launches and three round
// trips: 2^2 x 23 rows from its terms to its populations 0.56 -> 0.44 ms.
const int CP_SMALL_ROWS = 16384, CP_SMALL_GRAN = CP_SMALL_ROWS / CP_GRAN + 1;
enum { CPS_BINS = 0, CPS_SLICES, CPS_ROWS, CPS_WIDTH, CPS_SLOTS, CPS_N };  // rows: the largest bin's, whole slices

// inclusive sum over the wavefront
__device__ inline int32_t cp_wave_scan(int32_t v, int lane) {
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int32_t u = __shfl_up(v, o, 64);
    if (lane >= o) v += u;
  }
  return v;
}

__global__ void __launch_bounds__(1024) k_cp_small(const int32_t *__restrict__ rp, const int32_t *__restrict__ col,
                                                   int32_t n, int32_t *order, int32_t *pos, int32_t *bslice,
                                                   int32_t *bins, int32_t *info) {
  extern __shared__ int32_t ls[];
  int32_t *parent = ls, *size = ls + n;  // size: rows of a root, then its offset in the sorted order
  __shared__ int32_t hist[16][CP_SMALL_GRAN], gsize[CP_SMALL_GRAN], gbin[CP_SMALL_GRAN], first[CP_SMALL_GRAN + 1];
  __shared__ int32_t part[16];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int32_t ngran = n / CP_GRAN + 1;
  for (int32_t r = t; r < n; r += 1024) {
    parent[r] = r;
    size[r] = 0;
  }
  for (int32_t g = t; g < ngran; g += 1024) {
    gsize[g] = 0;
    for (int w = 0; w < 16; w++) hist[w][g] = 0;
  }
  __syncthreads();
  volatile int32_t *vp = parent;
  auto find = [&](int32_t i) {
    int32_t q = vp[i];
    while (q != i) {
      const int32_t g = vp[q];
      if (g != q) vp[i] = g;
      i = q;
      q = g;
    }
    return i;
  };
  for (int32_t r = t; r < n; r += 1024) {
    int32_t a = r;
    const int32_t end = rp[r + 1];
    for (int32_t e0 = rp[r]; e0 < end; e0 += 8) {
      int32_t c[8];  // in flight together
#pragma unroll
      for (int k = 0; k < 8; k++) c[k] = e0 + k < end ? col[e0 + k] : r;
#pragma unroll 1
      for (int k = 0; k < 8; k++) {
        int32_t b = c[0];
#pragma unroll
        for (int q = 0; q < 7; q++) c[q] = c[q + 1];
        if (b == r) continue;
        for (;;) {
          a = find(a);
          b = find(b);
          if (a == b) break;
          const int32_t hi = a > b ? a : b, lo = a > b ? b : a;
          const int32_t old = atomicCAS(parent + hi, hi, lo);
          a = lo;
          if (old == hi) break;
          b = old;
        }
      }
    }
  }
  __syncthreads();
  for (int32_t r = t; r < n; r += 1024) {
    const int32_t l = find(r);
    vp[r] = l;
    atomicAdd(size + l, 1);
  }
  __syncthreads();
  // offsets of the components in the order of their roots, and the granules' rows
  const int32_t per = (n + 1023) / 1024, b0 = min(t * per, n), b1 = min(b0 + per, n);
  int32_t own = 0;
  for (int32_t r = b0; r < b1; r++) own += size[r];
  const int32_t inc = cp_wave_scan(own, lane);
  if (lane == 63) part[wave] = inc;
  __syncthreads();
  int32_t run = inc - own;
  for (int w = 0; w < wave; w++) run += part[w];
  for (int32_t r = b0; r < b1; r++) {
    const int32_t s = size[r];
    if (s) atomicAdd(gsize + run / CP_GRAN, s);
    size[r] = run;
    run += s;
  }
  __syncthreads();
  if (wave == 0) {  // a bin for every granule with rows
    int32_t nb = 0, sl = 0, most = 0;
    for (int32_t g0 = 0; g0 < ngran; g0 += 64) {
      const int32_t v = g0 + lane < ngran ? gsize[g0 + lane] : 0;
      const uint64_t m = __ballot(v > 0);
      const int32_t b = nb + (int32_t)__popcll(m & ((1ull << lane) - 1ull)), k = (v + 63) / 64;
      const int32_t at = sl + cp_wave_scan(k, lane) - k;
      if (v > 0) {
        gbin[g0 + lane] = b;
        first[b] = at;
        bslice[b] = at;
        bins[b] = b;
      }
      most = max(most, cp_wave_max(k));
      nb += (int32_t)__popcll(m);
      sl = __shfl(at + k, 63, 64);
    }
    if (lane == 0) {
      first[nb] = sl;
      bslice[nb] = sl;
      info[CPS_BINS] = nb;
      info[CPS_SLICES] = sl;
      info[CPS_ROWS] = most * 64;
    }
    part[0] = nb;
  }
  __syncthreads();
  const int32_t nb = part[0];
  for (int32_t p = t; p < first[nb] * 64; p += 1024) order[p] = -1;
  for (int32_t r = t; r < n; r += 1024) parent[r] = gbin[size[parent[r]] / CP_GRAN];  // the row's bin
  __syncthreads();
  // rows in increasing order within a bin: wavefront w takes the w-th part of them
  const int32_t c = ((n + 15) / 16 + 63) / 64 * 64, r0 = min(wave * c, n), r1 = min(r0 + c, n);
  for (int32_t r = r0 + lane; r < r1; r += 64) atomicAdd(&hist[wave][parent[r]], 1);
  __syncthreads();
  for (int32_t b = t; b < nb; b += 1024) {
    int32_t s = 0;
    for (int w = 0; w < 16; w++) {
      const int32_t v = hist[w][b];
      hist[w][b] = s;
      s += v;
    }
  }
  __syncthreads();
  for (int32_t rr = r0; rr < r1; rr += 64) {
    const int32_t r = rr + lane;
    const int32_t b = r < r1 ? parent[r] : -1;
    uint64_t left = __ballot(b >= 0);
    int32_t at = 0;
    while (left) {
      const int32_t f = __shfl(b, __ffsll((unsigned long long)left) - 1, 64);
      const uint64_t m = __ballot(b == f);
      if (b == f) at = hist[wave][f] + (int32_t)__popcll(m & ((1ull << lane) - 1ull));
      __builtin_amdgcn_wave_barrier();
      if (lane == 0) hist[wave][f] += (int32_t)__popcll(m);
      __builtin_amdgcn_wave_barrier();
      left &= ~m;
    }
    if (b >= 0) {
      pos[r] = at;
      order[(int64_t)first[b] * 64 + at] = r;
    }
  }
}

// offsets of the slices' slots, their bins' zero cells, the widest slice and all slots
__global__ void __launch_bounds__(64) k_cp_small_offsets(const int32_t *width, const int32_t *bslice, int32_t *soff,
                                                         int32_t *zc, int32_t *info) {
  const int lane = threadIdx.x;
  const int32_t nsl = info[CPS_SLICES], nb = info[CPS_BINS];
  int32_t run = 0, most = 0;
  for (int32_t s0 = 0; s0 < nsl; s0 += 64) {
    const int32_t w = s0 + lane < nsl ? width[s0 + lane] : 0;
    const int32_t inc = cp_wave_scan(w, lane);
    if (s0 + lane < nsl) soff[s0 + lane] = run + inc - w;
    most = max(most, cp_wave_max(w));
    run += __shfl(inc, 63, 64);
  }
  for (int32_t b = lane; b < nb; b += 64)
    for (int32_t s = bslice[b]; s < bslice[b + 1]; s++) zc[s] = (bslice[b + 1] - bslice[b]) * 64;
  if (lane == 0) {
    info[CPS_WIDTH] = most;
    info[CPS_SLOTS] = run;
  }
}

// ------------------------------------------------------------------ stepping
struct CpArgs {
  const int32_t *bins, *bslice;  // this launch's bins; first slice of every bin
  const int32_t *soff, *width, *nim, *order;
  const double2 *diag;
  const double *ev;    // entries held in registers: values and columns
  const uint16_t *ec;
  const uint32_t *ew;  // entries read as words, and this launch's first table
  const double *dict;
  void *x;
  float2 *xlo;   // the low words of an FP32 state, else null
  int32_t cells;  // entries of one LDS buffer
  double h;
  int64_t nsteps;
};

// entry r of the state as complex128, and back (an FP32 state is the sum of two words)
__device__ inline double2 cp_load(const CpArgs &a, int32_t r) {
  if (!a.xlo) return ((const double2 *)a.x)[r];
  const float2 hi = ((const float2 *)a.x)[r], lo = a.xlo[r];
  return make_double2((double)hi.x + (double)lo.x, (double)hi.y + (double)lo.y);
}
__device__ inline void cp_store(const CpArgs &a, int32_t r, double2 v) {
  if (!a.xlo) {
    ((double2 *)a.x)[r] = v;
    return;
  }
  const float hr = (float)v.x, hm = (float)v.y;
  ((float2 *)a.x)[r] = make_float2(hr, hm);
  a.xlo[r] = make_float2((float)(v.x - (double)hr), (float)(v.y - (double)hm));
}
// the imaginary parts of a row are summed first, then the sum is turned by i and the
// real parts follow
__device__ inline void cp_times_i(double &p, double &r) {
  const double u = p;
  p = -r;
  r = u;
}

// A thread owns S rows of the bin, wavefront w the slices w, w + waves, ...; the W
// slots of a row live in registers (2.5 dwords each), so that a step reads LDS only.
// RK4 on a linear autonomous system in nested form, y <- x + c A y with c = h/4,
// h/3, h/2, h, double buffered: one barrier a stage.  SKIP: pairs of slots that none
// of the slice's rows fills are passed over, which pays where the LDS is the bound
// (bins on every CU); without it more reads are in flight at once.
template <int S, int W, bool SKIP>
__global__ void __launch_bounds__(1024) k_comp_rk4(CpArgs a) {
  extern __shared__ double2 sm[];
  const int b = a.bins[blockIdx.x];
  const int32_t sl0 = a.bslice[b], nsl = a.bslice[b + 1] - sl0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  double2 x[S], y[S], d[S];
  int32_t row[S], nim[S], wid[S];
  double v[S * W];
  uint32_t c2[S * W / 2];
#pragma unroll
  for (int k = 0; k < S; k++) {
    const int32_t sl = wave + k * waves;
    int32_t s0 = 0;
    row[k] = -1;
    nim[k] = wid[k] = 0;
    x[k] = d[k] = make_double2(0.0, 0.0);
    if (sl < nsl) {
      const int64_t p = (int64_t)(sl0 + sl) * 64 + lane;
      row[k] = a.order[p];
      s0 = a.soff[sl0 + sl];
      wid[k] = a.width[sl0 + sl];
      nim[k] = a.nim[sl0 + sl];
      d[k] = a.diag[p];
      if (row[k] >= 0) x[k] = cp_load(a, row[k]);
      sm[sl * 64 + lane] = x[k];
    }
    y[k] = x[k];
#pragma unroll
    for (int e = 0; e < W; e += 2) {
      const bool f = e < wid[k], g = e + 1 < wid[k];
      const int64_t at = (int64_t)(s0 + e) * 64 + lane;
      v[k * W + e] = f ? a.ev[at] : 0.0;
      v[k * W + e + 1] = g ? a.ev[at + 64] : 0.0;
      const uint32_t z = (uint32_t)nsl * 64u;
      const uint32_t lo = f ? a.ec[at] : z, hi = g ? a.ec[at + 64] : z;
      c2[(k * W + e) / 2] = lo | (hi << 16);
    }
  }
  if (threadIdx.x == 0) sm[nsl * 64] = sm[a.cells + nsl * 64] = make_double2(0.0, 0.0);
  __syncthreads();
  const double cs[4] = {a.h / 4.0, a.h / 3.0, a.h / 2.0, a.h};
  for (int64_t st = 0; st < a.nsteps; st++) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const char *in = (const char *)(sm + (q & 1 ? a.cells : 0));
      double2 *out = sm + (q & 1 ? 0 : a.cells);
#pragma unroll
      for (int k = 0; k < S; k++) {
        const int32_t sl = wave + k * waves;
        if (sl < nsl) {
          double p = 0.0, r = 0.0;
          // LDS reads in flight (a divisor of W; the registers allow fewer beside more slots)
          constexpr int CH = SKIP ? 2 : S > 1 || W > 16 ? (W == 10 || W == 12 ? 2 : 4) : W == 12 || W == 16 ? W / 2 : W;
          static_assert(W % CH == 0 && CH % 2 == 0, "whole chunks");
#pragma unroll
          for (int e0 = 0; e0 < W; e0 += CH) {
            if (SKIP && e0 >= wid[k]) continue;
            double2 t[CH];
#pragma unroll
            for (int j = 0; j < CH; j++) {
              const uint32_t w = c2[(k * W + e0 + j) / 2];
              const uint32_t at = j & 1 ? (w >> 12) & 0xFFFF0u : (w << 4) & 0xFFFF0u;
              t[j] = *(const double2 *)(in + at);
            }
#pragma unroll
            for (int j = 0; j < CH; j++) {
              if (!(j & 1) && nim[k] == e0 + j) cp_times_i(p, r);
              p = fma(v[k * W + e0 + j], t[j].x, p);
              r = fma(v[k * W + e0 + j], t[j].y, r);
            }
          }
          if (nim[k] == W || (SKIP && nim[k] > 0 && nim[k] >= wid[k])) cp_times_i(p, r);
          p = fma(d[k].x, y[k].x, fma(-d[k].y, y[k].y, p));
          r = fma(d[k].x, y[k].y, fma(d[k].y, y[k].x, r));
          y[k].x = fma(cs[q], p, x[k].x);
          y[k].y = fma(cs[q], r, x[k].y);
          out[sl * 64 + lane] = y[k];
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < S; k++) x[k] = y[k];
  }
#pragma unroll
  for (int k = 0; k < S; k++)
    if (row[k] >= 0) cp_store(a, row[k], x[k]);
}

// a wavefront's scalar, kept from being expanded into one condition per slot ahead of
// the step loop (they would spill)
__device__ inline int32_t cp_opaque(int32_t v) {
  asm volatile("" : "+s"(v));
  return v;
}

// The same steps with the entries read as words at every stage, the next slice's
// CP_DICT_W words in flight during the products of this one.  Y: the stage vectors
// in LDS (complex64 for an FP32 state, whose x stays in 64 bits); products and sums
// in 64 bits.  1024 threads, S rows each (even, so that the two word buffers keep
// their parity from stage to stage).
template <typename Y, int S>
__global__ void __launch_bounds__(1024) k_comp_dict(CpArgs a) {
  static_assert(S % 2 == 0, "two word buffers");
  extern __shared__ double2 sm[];
  constexpr int WC = CP_DICT_W;
  Y *buf = (Y *)sm;
  double *dict = (double *)(buf + 2 * a.cells);
  const int b = a.bins[blockIdx.x];
  const int32_t sl0 = a.bslice[b], nsl = a.bslice[b + 1] - sl0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int i = threadIdx.x; i < CP_DICT; i += 1024) dict[i] = a.dict[(int64_t)blockIdx.x * CP_DICT + i];
  double2 x[S], d[S];
  int32_t wn[S], s0[S];  // width << 16 | imaginary slots; first slot
  uint32_t w[2][WC];
#pragma unroll
  for (int k = 0; k < S; k++) {
    const int32_t sl = wave + k * 16;
    wn[k] = s0[k] = 0;
    x[k] = d[k] = make_double2(0.0, 0.0);
    if (sl < nsl) {
      const int64_t p = (int64_t)(sl0 + sl) * 64 + lane;
      const int32_t row = a.order[p];
      s0[k] = a.soff[sl0 + sl];
      wn[k] = a.width[sl0 + sl] << 16 | a.nim[sl0 + sl];
      d[k] = a.diag[p];
      if (row >= 0) x[k] = cp_load(a, row);
      Y t;
      t.x = x[k].x;
      t.y = x[k].y;
      buf[sl * 64 + lane + 1] = t;
    }
  }
  // words past a slice's last slot read as zero: the zero cell times zero
  auto fetch = [&](int k, uint32_t(&to)[WC]) {
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t *>(a.ew + (int64_t)cp_opaque(s0[k]) * 64), (short)0, (cp_opaque(wn[k]) >> 16) * 256,
        0x00020000);
#pragma unroll
    for (int e = 0; e < WC; e++)
      to[e] = __builtin_amdgcn_raw_buffer_load_b32(rs, (uint32_t)(lane * 4 + e * 256), 0, 0);
  };
  fetch(0, w[0]);
  if (threadIdx.x == 0) {
    Y z;
    z.x = z.y = 0;
    buf[0] = buf[a.cells] = z;
  }
  __syncthreads();
  const double cs[4] = {a.h / 4.0, a.h / 3.0, a.h / 2.0, a.h};
  for (int64_t st = 0; st < a.nsteps; st++) {
#pragma unroll 1
    for (int q = 0; q < 4; q++) {
      const Y *in = buf + (q & 1 ? a.cells : 0);
      Y *out = buf + (q & 1 ? 0 : a.cells);
      const double c = q == 0 ? cs[0] : q == 1 ? cs[1] : q == 2 ? cs[2] : cs[3];
#pragma unroll
      for (int k = 0; k < S; k++) {
        const int32_t sl = wave + k * 16;
        if (k + 1 == S)
          fetch(0, w[0]);
        else if (sl + 16 < nsl)
          fetch((k + 1) % S, w[(k + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // issued before this slice's products
        if (sl < nsl) {
          const int32_t wnk = cp_opaque(wn[k]), wid = wnk >> 16, nim = wnk & 0xFFFF;
          double p = 0.0, r = 0.0;
          auto term = [&](uint32_t u) {
            const Y t = in[u & 0xFFFFu];
            const double v = *(const double *)((const char *)dict + (u >> 16));
            p = fma(v, (double)t.x, p);
            r = fma(v, (double)t.y, r);
          };
#pragma unroll
          for (int e = 0; e < WC; e += 2) {
            if (e >= wid) continue;
            if (nim == e) cp_times_i(p, r);
            term(w[k & 1][e]);
            term(w[k & 1][e + 1]);
          }
          for (int32_t e = WC; e < wid; e++) {
            if (nim == e) cp_times_i(p, r);
            term(a.ew[(int64_t)(s0[k] + e) * 64 + lane]);
          }
          if (nim > 0 && nim >= wid) cp_times_i(p, r);
          const Y own = in[sl * 64 + lane + 1];
          p = fma(d[k].x, (double)own.x, fma(-d[k].y, (double)own.y, p));
          r = fma(d[k].x, (double)own.y, fma(d[k].y, (double)own.x, r));
          p = fma(c, p, x[k].x);
          r = fma(c, r, x[k].y);
          if (q == 3) x[k] = make_double2(p, r);
          Y t;
          t.x = p;
          t.y = r;
          out[sl * 64 + lane + 1] = t;
        }
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int k = 0; k < S; k++) {
    const int32_t sl = wave + k * 16;
    if (sl >= nsl) continue;
    const int32_t row = a.order[(int64_t)(sl0 + sl) * 64 + lane];
    if (row >= 0) cp_store(a, row, x[k]);
  }
}

int cp_launch(void (*kernel)(CpArgs), const CpClass &c, const CpArgs &a, size_t lds, hipStream_t s) {
  if (lds > 64 * 1024)
    QH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds));
  hipLaunchKernelGGL(kernel, dim3(c.count), dim3(c.threads), lds, s, a);
  QH_HIP(hipGetLastError());
  return QH_OK;
}

}  // namespace

struct qh_comp {
  void *buf = nullptr, *slots = nullptr;  // the plan's arrays; its entries
  CpArgs a{};
  double *trace = nullptr;  // QH_COMP_TRACE doubles for the trace renormalisation
  std::vector<CpClass> classes, brief;  // brief: of a call of up to brief_steps steps
  int64_t brief_steps = 0;
  int64_t slots_of[2] = {0, 0};  // in registers, as words
  // launches of fewer blocks than CUs run on a stream of their own beside the
  // others (disjoint rows), between two events of the library stream
  hipStream_t side = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
};

void qh_comp_free(qh_comp *c) {
  if (!c) return;
  if (c->side) (void)hipStreamSynchronize(c->side);
  for (hipEvent_t e : c->ev)
    if (e) (void)hipEventDestroy(e);
  if (c->side) (void)hipStreamDestroy(c->side);
  qh_free_ptr(c->buf);
  qh_free_ptr(c->slots);
  delete c;
}

namespace {

// a workspace handed out in 256-byte aligned pieces; two passes: sizes, then pointers
struct Carve {
  char *p = nullptr;
  size_t n = 0;
  template <typename T>
  T *take(size_t count) {
    T *q = reinterpret_cast<T *>(p + n);
    n += (count * sizeof(T) + 255) & ~(size_t)255;
    return q;
  }
};

// the rules of qh_comp_plan.h on this device and matrix
bool cp_worth(double most, double all, int64_t n) { return ::cp_worth(most, all, n, qh_num_cus()); }
double cp_least(int64_t rows, const qh_mat *A) { return ::cp_least(rows, (double)A->nnz / (double)A->rows - 1.0); }

// The plan of a matrix of at most CP_SMALL_ROWS rows with one shape for all bins
// (*done = 0 where it needs the general builder)
int cp_build_small(qh_mat *A, int f32, int *done) {
  *done = 0;
  const int32_t n = (int32_t)A->rows;
  hipStream_t s = qh_stream();
  const int32_t ngran = n / CP_GRAN + 1, maxsl = n / 64 + ngran;
  int32_t *order, *pos, *bslice, *bins, *soff, *nim, *zc, *width, *info;
  double2 *diag;
  double *trace;
  auto arrays = [&](Carve &q) {
    order = q.take<int32_t>((size_t)maxsl * 64);
    pos = q.take<int32_t>(n);
    bslice = q.take<int32_t>(ngran + 1);
    bins = q.take<int32_t>(ngran);
    soff = q.take<int32_t>(maxsl);
    nim = q.take<int32_t>(maxsl);
    zc = q.take<int32_t>(maxsl);
    width = q.take<int32_t>(maxsl);
    info = q.take<int32_t>(CPS_N);
    diag = q.take<double2>((size_t)maxsl * 64);
    trace = q.take<double>(QH_COMP_TRACE);
  };
  Carve size, at;
  arrays(size);
  // freed on every return before it is handed to A (the free waits for the device)
  std::unique_ptr<qh_comp, void (*)(qh_comp *)> c(new qh_comp(), qh_comp_free);
  auto fail = [&](int code) {
    (void)hipStreamSynchronize(s);
    return code;
  };
  int32_t *h = nullptr;
  int rc = qh_alloc(&c->buf, size.n);
  if (!rc) rc = qh_scratch(0, nullptr, CPS_N * sizeof(int32_t), (void **)&h);
  if (rc) return fail(rc);
  at.p = (char *)c->buf;
  arrays(at);
#define CP_HIP(call)                                                                  \
  do {                                                                                \
    hipError_t e_ = (call);                                                           \
    if (e_ != hipSuccess) {                                                           \
      qh_set_error("%s:%d %s: %s", __FILE__, __LINE__, #call, hipGetErrorString(e_)); \
      return fail(QH_EHIP);                                                           \
    }                                                                                 \
  } while (0)
  const size_t lds = (size_t)2 * n * sizeof(int32_t);
  if (lds > 40 * 1024)
    CP_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_cp_small), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds));
  hipLaunchKernelGGL(k_cp_small, dim3(1), dim3(1024), lds, s, A->rowptr, A->col, n, order, pos, bslice, bins, info);
  hipLaunchKernelGGL(k_cp_width, dim3(qh_blocks(maxsl, 4)), dim3(256), 0, s, order, A->rowptr, A->col, A->val, width,
                     nim, maxsl, (const int32_t *)(info + CPS_SLICES));
  hipLaunchKernelGGL(k_cp_small_offsets, dim3(1), dim3(64), 0, s, width, bslice, soff, zc, info);
  CP_HIP(hipGetLastError());
  CP_HIP(hipMemcpyAsync(h, info, CPS_N * sizeof(int32_t), hipMemcpyDeviceToHost, s));
  CP_HIP(hipStreamSynchronize(s));
  const int nb = h[CPS_BINS], nsl = h[CPS_SLICES], rows = h[CPS_ROWS], W = cp_width_class(h[CPS_WIDTH], false);
  const int64_t slots = h[CPS_SLOTS];
  if (!cp_fits_registers(rows, W) && cp_worth(cp_least(rows, A), 0.0, n)) return fail(QH_OK);
  *done = 1;
  if (!cp_fits_registers(rows, W)) {
    A->comp_state[f32] = -1;
    return fail(QH_OK);
  }
  if (!cp_worth(CP_CLK_REG * W * (rows / 64) + CP_CLK_FIXED, CP_CLK_REG * W * nsl, n)) {
    A->comp_state[f32] = -1;
    return fail(QH_OK);
  }
  double *ev;
  uint16_t *ec;
  auto entries = [&](Carve &q) {
    ev = q.take<double>((size_t)slots * 64 + 1);
    ec = q.take<uint16_t>((size_t)slots * 64 + 1);
  };
  Carve em, ep;
  entries(em);
  rc = qh_alloc(&c->slots, em.n);
  if (rc) return fail(rc);
  ep.p = (char *)c->slots;
  entries(ep);
  hipLaunchKernelGGL(k_cp_fill, dim3(qh_blocks(nsl, 4)), dim3(256), 0, s, order, pos, A->rowptr, A->col, A->val,
                     soff, width, nim, zc, diag, ev, ec, nsl);
  CP_HIP(hipGetLastError());
#undef CP_HIP
  const int S = rows > 1024 ? 2 : 1;
  c->slots_of[0] = slots;
  c->classes.push_back(CpClass{cp_threads(rows), S, W, false, false, 0, nb, rows + 1});
  c->a = CpArgs{};
  c->a.bins = bins;
  c->a.bslice = bslice;
  c->a.soff = soff;
  c->a.width = width;
  c->a.nim = nim;
  c->a.order = order;
  c->a.diag = diag;
  c->a.ev = ev;
  c->a.ec = ec;
  c->trace = trace;
  A->comp[f32] = c.release();
  A->comp_state[f32] = 1;
  return QH_OK;
}

int cp_build(qh_mat *A, int f32) {
  const int32_t max_rows = f32 ? CP_MAX_ROWS32 : CP_MAX_ROWS64;
  int &state = A->comp_state[f32];
  const int32_t n = (int32_t)A->rows;
  hipStream_t s = qh_stream();
  const unsigned nb256 = qh_blocks(n, 256);
  const int32_t ngran = n / CP_GRAN + 1;
  size_t scan_b = 0, sort_b = 0;
  QH_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan_b, (int32_t *)nullptr, (int32_t *)nullptr, n, s));
  int bits = 1;
  while ((1 << bits) < ngran && bits < 31) bits++;
  QH_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_b, (int32_t *)nullptr, (int32_t *)nullptr,
                                            (int32_t *)nullptr, (int32_t *)nullptr, n, 0, bits, s));
  int32_t *parent, *size, *lab, *off, *gsize, *gbin, *key, *row, *pos, *brow;
  char *tmp;
  auto layout = [&](Carve &c) {
    parent = c.take<int32_t>(n);
    size = c.take<int32_t>(n);
    lab = c.take<int32_t>(n);
    off = c.take<int32_t>(n);
    key = c.take<int32_t>(n);
    row = c.take<int32_t>(n);
    pos = c.take<int32_t>(n);
    gsize = c.take<int32_t>(ngran);
    gbin = c.take<int32_t>(ngran);
    brow = c.take<int32_t>(ngran + 1);
    tmp = c.take<char>(std::max(scan_b, sort_b) + 1);
  };
  Carve meas, work;
  layout(meas);
  // (an allocation of some MB and its release take up to a millisecond: the library's
  // scratch, kept, up to CP_SCRATCH bytes)
  void *wbuf = nullptr, *own = nullptr;
  int rc = meas.n <= CP_SCRATCH ? qh_scratch(meas.n, &wbuf, 0, nullptr) : qh_alloc(&own, meas.n);
  if (rc) return rc;
  if (own) wbuf = own;
  work.p = (char *)wbuf;
  layout(work);
  // freed on every return before it is handed to A (the frees wait for the device)
  std::unique_ptr<void, void (*)(void *)> owned(own, qh_free_ptr);
  std::unique_ptr<qh_comp, void (*)(qh_comp *)> c(new qh_comp(), qh_comp_free);
  auto fail = [&](int code) {
    (void)hipStreamSynchronize(s);
    return code;
  };
#define CP_HIP(call)                                                                             \
  do {                                                                                           \
    hipError_t e_ = (call);                                                                      \
    if (e_ != hipSuccess) {                                                                      \
      qh_set_error("%s:%d %s: %s", __FILE__, __LINE__, #call, hipGetErrorString(e_));            \
      return fail(QH_EHIP);                                                                      \
    }                                                                                            \
  } while (0)
  // A large matrix is probed first: the rows of its largest block, or its first
  // CP_PROBE_ROWS ones.  Rows that hang together there do so in the whole (10-qubit
  // chain, 1 M rows: 0.1 ms for the probe, 1.2 ms for all rows; 16 M rows of a sweep 10 ms).
  if (n > 4 * CP_PROBE_ROWS) {
    int32_t r0 = 0, m = CP_PROBE_ROWS;
    if (A->blk_off.size() > 2) {
      size_t big = 0;
      for (size_t i = 0; i + 1 < A->blk_off.size(); i++)
        if (A->blk_off[i + 1] - A->blk_off[i] > A->blk_off[big + 1] - A->blk_off[big]) big = i;
      r0 = (int32_t)A->blk_off[big];
      m = (int32_t)(A->blk_off[big + 1] - A->blk_off[big]);
    }
    const unsigned nbp = qh_blocks(m, 256);
    int32_t most = 0;
    hipLaunchKernelGGL(k_cc_init, dim3(std::min(nbp, 4096u)), dim3(256), 0, s, parent, size, m);
    hipLaunchKernelGGL(k_cc_hook, dim3(nbp), dim3(256), 0, s, parent, A->rowptr, A->col, r0, m);
    hipLaunchKernelGGL(k_cc_label, dim3(qh_blocks(m, CC_LABEL_ROWS)), dim3(256), 0, s, parent, lab, size, m);
    CP_HIP(hipMemsetAsync(off, 0, sizeof(int32_t), s));
    hipLaunchKernelGGL(k_cc_largest, dim3(std::min(nbp, 256u)), dim3(256), 0, s, size, off, m);
    CP_HIP(hipMemcpyAsync(&most, off, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    CP_HIP(hipStreamSynchronize(s));
    if (most > max_rows || !cp_worth(cp_least(most, A), 0.0, n)) {
      fail(0);
      state = -1;
      return QH_OK;
    }
  }
  // components, and the rows that start in each granule of the sorted order
  CP_HIP(hipMemsetAsync(gsize, 0, sizeof(int32_t) * ngran, s));
  hipLaunchKernelGGL(k_cc_init, dim3(std::min(nb256, 4096u)), dim3(256), 0, s, parent, size, n);
  hipLaunchKernelGGL(k_cc_hook, dim3(nb256), dim3(256), 0, s, parent, A->rowptr, A->col, 0, n);
  hipLaunchKernelGGL(k_cc_label, dim3(qh_blocks(n, CC_LABEL_ROWS)), dim3(256), 0, s, parent, lab, size, n);
  size_t tb = std::max(scan_b, sort_b);
  CP_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, tb, size, off, n, s));
  hipLaunchKernelGGL(k_cc_granules, dim3(nb256), dim3(256), 0, s, size, off, gsize, n);
  std::vector<int32_t> hg(ngran);
  CP_HIP(hipMemcpyAsync(hg.data(), gsize, sizeof(int32_t) * ngran, hipMemcpyDeviceToHost, s));
  CP_HIP(hipStreamSynchronize(s));
  // bins: consecutive granules up to CP_PACK_ROWS where there are many, else one each
  const int64_t cus = qh_num_cus();
  const int32_t pack = (int64_t)n > 2 * cus * CP_PACK_ROWS ? CP_PACK_ROWS : 0;
  std::vector<int32_t> hbin(ngran), hrow{0}, hslice{0};
  int32_t cur = 0, largest = 0;
  auto close = [&] {
    if (!cur) return;
    hrow.push_back(hrow.back() + cur);
    hslice.push_back(hslice.back() + (cur + 63) / 64);
    largest = std::max(largest, cur);
    cur = 0;
  };
  for (int32_t g = 0; g < ngran; g++) {
    if (!hg[g]) {
      hbin[g] = 0;
      continue;
    }
    if (cur && cur + hg[g] > pack) close();
    hbin[g] = (int32_t)hrow.size() - 1;
    cur += hg[g];
  }
  close();
  if (largest > max_rows || !cp_worth(cp_least(largest, A), 0.0, n)) {
    fail(0);
    state = -1;
    return QH_OK;
  }
  const int32_t nbins = (int32_t)hrow.size() - 1, nsl = hslice.back();
  // order the rows by bin
  CP_HIP(hipMemcpyAsync(gbin, hbin.data(), sizeof(int32_t) * ngran, hipMemcpyHostToDevice, s));
  CP_HIP(hipMemcpyAsync(brow, hrow.data(), sizeof(int32_t) * (nbins + 1), hipMemcpyHostToDevice, s));
  // `parent` and `size` are free from here: the sort's second buffers
  hipLaunchKernelGGL(k_cp_keys, dim3(nb256), dim3(256), 0, s, lab, off, gbin, key, row, n);
  CP_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, key, parent, row, size, n, 0, bits, s));
  int32_t *order, *bslice, *soff, *nim, *zc, *width, *bins, *over;
  double2 *diag;
  double *trace;
  auto head = [&](Carve &q) {
    order = q.take<int32_t>((size_t)nsl * 64);
    bslice = q.take<int32_t>(nbins + 1);
    soff = q.take<int32_t>((size_t)nsl + 1);
    nim = q.take<int32_t>(nsl);
    zc = q.take<int32_t>(nsl);
    width = q.take<int32_t>(nsl);
    bins = q.take<int32_t>(nbins);
    over = q.take<int32_t>(1);
    diag = q.take<double2>((size_t)nsl * 64);
    trace = q.take<double>(QH_COMP_TRACE);
  };
  Carve hm;
  head(hm);
  void *hbuf = nullptr;
  rc = qh_alloc(&hbuf, hm.n);
  if (rc) return fail(rc);
  Carve hw;
  hw.p = (char *)hbuf;
  head(hw);
  c->buf = hbuf;
  CP_HIP(hipMemcpyAsync(bslice, hslice.data(), sizeof(int32_t) * (nbins + 1), hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_cp_fill_order, dim3(qh_blocks((int64_t)nsl * 64, 256)), dim3(256), 0, s, order,
                     (int64_t)nsl * 64);
  hipLaunchKernelGGL(k_cp_place, dim3(nb256), dim3(256), 0, s, parent, size, brow, bslice, order, pos, n);
  hipLaunchKernelGGL(k_cp_width, dim3(qh_blocks(nsl, 4)), dim3(256), 0, s, order, A->rowptr, A->col, A->val, width,
                     nim, nsl, nullptr);
  CP_HIP(hipGetLastError());
  std::vector<int32_t> hwid(nsl), hoff(nsl), hzc(nsl);
  CP_HIP(hipMemcpyAsync(hwid.data(), width, sizeof(int32_t) * nsl, hipMemcpyDeviceToHost, s));
  CP_HIP(hipStreamSynchronize(s));
  // the shape of every bin's launch, and what the largest bin and all of them take
  std::vector<CpBin> hbn(nbins);
  for (int32_t b = 0; b < nbins; b++) {
    hbn[b] = CpBin{(hslice[b + 1] - hslice[b]) * 64, 0, 0};
    for (int32_t i = hslice[b]; i < hslice[b + 1]; i++) {
      hbn[b].width = std::max(hbn[b].width, (int)hwid[i]);
      hbn[b].slots += hwid[i];
    }
  }
  const CpShapes sh = cp_shapes(hbn, f32, (int)cus);
  int64_t slots[2] = {0, 0};  // held in registers, read as words
  for (int32_t b = 0; b < nbins; b++)
    for (int32_t i = hslice[b]; i < hslice[b + 1]; i++) {
      hoff[i] = (int32_t)slots[sh.words[b]];
      slots[sh.words[b]] += hwid[i];
      hzc[i] = sh.words[b] ? -1 : hbn[b].rows;
      if (slots[sh.words[b]] > (int64_t)0x7fffffff) {
        fail(0);
        state = -1;
        return QH_OK;
      }
    }
  if (!sh.runnable || !cp_worth(sh.most, sh.all, n)) {
    fail(0);
    state = -1;
    return QH_OK;
  }
  c->classes = sh.classes;
  c->brief = sh.brief;
  c->brief_steps = sh.brief_steps;
  std::copy_n(slots, 2, c->slots_of);
  for (const CpClass &k : c->classes)
    if (k.side && !c->side) {
      CP_HIP(hipStreamCreateWithFlags(&c->side, hipStreamNonBlocking));
      for (hipEvent_t &e : c->ev) CP_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
  const int ndict = c->classes[0].W == 0 ? c->classes[0].count : 0;  // these bins come first
  double *ev, *dict;
  uint16_t *ec;
  uint32_t *ew;
  auto entries = [&](Carve &q) {
    ev = q.take<double>((size_t)slots[0] * 64 + 1);
    ec = q.take<uint16_t>((size_t)slots[0] * 64 + 1);
    ew = q.take<uint32_t>((size_t)slots[1] * 64 + 1);
    dict = q.take<double>((size_t)ndict * CP_DICT + 1);
  };
  Carve em, ep;
  entries(em);
  rc = qh_alloc(&c->slots, em.n);
  if (rc) return fail(rc);
  ep.p = (char *)c->slots;
  entries(ep);
  CP_HIP(hipMemcpyAsync(zc, hzc.data(), sizeof(int32_t) * nsl, hipMemcpyHostToDevice, s));
  CP_HIP(hipMemcpyAsync(soff, hoff.data(), sizeof(int32_t) * nsl, hipMemcpyHostToDevice, s));
  CP_HIP(hipMemcpyAsync(bins, sh.bins.data(), sizeof(int32_t) * nbins, hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_cp_fill, dim3(qh_blocks(nsl, 4)), dim3(256), 0, s, order, pos, A->rowptr, A->col, A->val,
                     soff, width, nim, zc, diag, ev, ec, nsl);
  int32_t hover = 0;
  if (ndict) {
    CP_HIP(hipMemsetAsync(over, 0, sizeof(int32_t), s));
    hipLaunchKernelGGL(k_cp_dict, dim3(ndict), dim3(1024), 0, s, bins, bslice, order, pos, A->rowptr, A->col, A->val,
                       soff, width, nim, ew, dict, over);
    CP_HIP(hipMemcpyAsync(&hover, over, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  }
  CP_HIP(hipGetLastError());
  CP_HIP(hipStreamSynchronize(s));  // the host vectors and the workspace go
  if (hover) {  // more values than a table holds
    fail(0);
    state = -1;
    return QH_OK;
  }
#undef CP_HIP
  c->a.bslice = bslice;
  c->a.bins = bins;
  c->a.soff = soff;
  c->a.width = width;
  c->a.ew = ew;
  c->a.dict = dict;
  c->a.nim = nim;
  c->a.order = order;
  c->a.diag = diag;
  c->a.ev = ev;
  c->a.ec = ec;
  c->trace = trace;
  A->comp[f32] = c.release();
  state = 1;
  return QH_OK;
}

// The matrices whose plan was refused, by precision, rows and entries, for the rest of
// the process, so that of the matrices of a sweep (one structure, other values) one is
// looked at; the entry decides only the speed.
struct CpRefused {
  int prec;
  int64_t rows, nnz;
};
CpRefused g_refused[64];
unsigned g_nrefused = 0;

bool cp_refused(const qh_mat *A, int prec) {
  for (unsigned i = 0; i < g_nrefused && i < 64; i++)
    if (g_refused[i].prec == prec && g_refused[i].rows == A->rows && g_refused[i].nnz == A->nnz) return true;
  return false;
}

}  // namespace

int qh_comp_prepare(qh_mat *A, int prec, int64_t nsteps, int graph_len, bool layout, int *usable) {
  const int f32 = prec == QH_FP32;
  *usable = 0;
  if (A->comp_state[f32] == 0 && cp_refused(A, prec)) A->comp_state[f32] = -1;
  if (A->comp_state[f32] == 0 && (nsteps < 0 || cp_pays(A->rows, A->comp_seen, nsteps, graph_len, layout))) {
    const std::string text = qh_last_error();
    bool fits = true;
    auto build = [&]() -> int {
      int rc = QH_OK, done = 0;
      // row and slot numbers are 32-bit
      if (A->rows < 1 || A->rows > (int64_t)1 << 30)
        A->comp_state[f32] = -1;
      else if (A->rows <= CP_SMALL_ROWS)
        rc = cp_build_small(A, f32, &done);
      if (!rc && A->comp_state[f32] == 0 && !done) rc = cp_build(A, f32);
      return rc;
    };
    auto none = [&] {
      (void)hipGetLastError();
      qh_set_error("%s", text.c_str());
      A->comp_state[f32] = -1;  // the stage kernels run without the plan
      fits = false;
    };
    const int rc = qh_optional(QH_ENOMEM, build, none);
    if (rc) return rc;
    if (A->comp_state[f32] == -1 && fits) g_refused[g_nrefused++ % 64] = CpRefused{prec, A->rows, A->nnz};
  }
  *usable = A->comp_state[f32] == 1;
  return QH_OK;
}

int qh_comp_rk4(qh_mat *A, qh_vec *x, double dt, int64_t nsteps) {
  const int f32 = x->prec == QH_FP32;
  const qh_comp &c = *A->comp[f32];
  hipStream_t s = qh_stream();
  auto fork = [&]() -> int {
    QH_HIP(hipEventRecord(c.ev[0], s));
    QH_HIP(hipStreamWaitEvent(c.side, c.ev[0], 0));
    return QH_OK;
  };
  auto join = [&]() -> int {
    if (hipEventRecord(c.ev[1], c.side) == hipSuccess && hipStreamWaitEvent(s, c.ev[1], 0) == hipSuccess) return QH_OK;
    QH_HIP(hipStreamSynchronize(c.side));
    return QH_OK;
  };
  auto launch = [&](const CpClass &k) -> int {
    CpArgs a = c.a;
    a.bins += k.first;
    a.x = x->d;
    a.xlo = f32 ? x->lo : nullptr;
    a.cells = k.cells;
    a.h = dt;
    a.nsteps = nsteps;
    hipStream_t ks = k.side ? c.side : s;
    const size_t table = CP_DICT * sizeof(double);
    if (k.W == 0 && f32)
      return cp_launch(k_comp_dict<float2, 8>, k, a, (size_t)2 * k.cells * sizeof(float2) + table, ks);
    if (k.W == 0) return cp_launch(k_comp_dict<double2, 6>, k, a, (size_t)2 * k.cells * sizeof(double2) + table, ks);
#define CP_CASE(SS, WW, SK)                   \
  if (k.S == SS && k.W == WW && k.skip == SK) \
    return cp_launch(k_comp_rk4<SS, WW, SK>, k, a, (size_t)2 * k.cells * sizeof(double2), ks);
    CP_REG_KERNELS(CP_CASE)
#undef CP_CASE
    qh_set_error("no kernel for bins of %d rows a thread and %d slots", k.S, k.W);
    return QH_EINVAL;
  };
  return cp_run(nsteps <= c.brief_steps ? c.brief : c.classes, launch, fork, join);
}

double *qh_comp_trace(const qh_mat *A, int prec) { return A->comp[prec == QH_FP32]->trace; }

extern "C" int qh_mat_closed_info(const qh_mat *m, int prec, int64_t *bins, int64_t *word_bins, int64_t *launches,
                                  int64_t *slots, int64_t *word_slots) {
  QH_REQUIRE(m && (prec == QH_FP64 || prec == QH_FP32), QH_EINVAL,
             "qh_mat_closed_info: a matrix and a precision required");
  const qh_comp *c = m->comp[prec == QH_FP32];
  int64_t all = 0, words = 0;
  if (c)
    for (const CpClass &k : c->classes) {
      all += k.count;
      if (k.W == 0) words += k.count;
    }
  if (bins) *bins = all;
  if (word_bins) *word_bins = words;
  if (launches) *launches = c ? (int64_t)c->classes.size() : 0;
  if (slots) *slots = c ? c->slots_of[0] : 0;
  if (word_slots) *word_slots = c ? c->slots_of[1] : 0;
  return QH_OK;
}
