// qh_ks.h -- device pieces shared by the sliced-layout stage kernels
// (qh_spmv.hip: one row per lane; qh_ks2.hip: two rows per lane).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "qh_common.h"

namespace {

// stage epilogues: SpMV only; RK4 stages 1-3 and stage 4 of the form that keeps
// the stage derivatives (time-dependent terms); Bogacki-Shampine stage 3 (k3 and
// the 3rd-order candidate); Bogacki-Shampine error stage (k4 and the weighted
// error norm); a stage of the nested RK4 polynomial of a constant generator
// (y = x + c A y'); its last stage on an FP32 state (hi + lo updated, products in
// FP64)
enum {
  MODE_SPMV = 0,
  MODE_STAGE = 1,
  MODE_FINAL = 2,
  MODE_BS3 = 3,
  MODE_BS3E = 4,
  MODE_AXPY = 5,
  MODE_LAST = 6
};

// Raw buffer resource over n elements (gfx9 descriptor word 3: 32-bit data
// format).  A buffer load whose byte offset is at or beyond n * sizeof(T)
// returns zero instead of touching memory: inactive lanes load with offset
// QH_KS_OOB and so contribute exact zeros without any per-lane select.
#define QH_KS_OOB 0x80000000u
__device__ inline __amdgpu_buffer_rsrc_t ks_rsrc(const void *p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

// slot groups of a slice (KS_SC1: real values, one per lane for both of its rows)
enum { KS_UNI = 0, KS_SCA = 1, KS_CPX = 2, KS_SC1 = 3 };

// The metadata of a slice's slots held in registers: lane k loads slot k (one
// trip to memory for the whole slice, at most 64 slots), and a pass reads the slots
// it needs with v_readlane into scalar registers.  With the metadata behind scalar
// loads every pass waits for its own before it can issue its gathers; where the
// metadata streams (they miss the scalar cache each time) those waits are a large part
// of a wavefront's time, and where the caches hold it the trip ahead of the first pass
// and the reads of lanes are the longer way.  Per launch, from memory / in registers:
// 10-qubit chain FP64 28.7 / 24.7 us, 12-qubit circuit FP64 262 / 235 us and FP32 154 /
// 140 us; 9-qubit chain FP64 7.8 / 8.7 us, three 9-level cavities FP32 12.9 / 13.7 us.
template <typename M>
struct KsRegs {
  static constexpr int ND = sizeof(M) / 4;
  int32_t r[ND];
  // slots m[0 .. n), n <= 64
  __device__ __forceinline__ void load(const M *m, int32_t n, int lane) {
    const int32_t *p = (const int32_t *)(m + lane);
#pragma unroll
    for (int i = 0; i < ND; i++) r[i] = 0;
    if (lane < n) {
#pragma unroll
      for (int i = 0; i < ND; i++) r[i] = p[i];
    }
  }
  __device__ __forceinline__ M get(int32_t k) const {
    struct W {
      int32_t w[ND];
    } w;
#pragma unroll
    for (int i = 0; i < ND; i++) w.w[i] = __builtin_amdgcn_readlane(r[i], k);
    return __builtin_bit_cast(M, w);
  }
};

// where a pass takes its slots from: slot k of the registers (RL), or memory
template <typename M, bool RL>
struct KsSrc;
template <typename M>
struct KsSrc<M, true> {
  const KsRegs<M> &regs;
  int32_t k;  // slot of the slice
  __device__ __forceinline__ M get(int j) const { return regs.get(k + j); }
  __device__ __forceinline__ void skip(int n) { k += n; }
};
template <typename M>
struct KsSrc<M, false> {
  const M *mp;
  __device__ __forceinline__ M get(int j) const { return mp[j]; }
  __device__ __forceinline__ void skip(int n) { mp += n; }
};

// row sum of a one-row-per-lane pass (FP64)
struct KsAcc {
  double re, im;
};

// The last rem (< U) slots of a group: for U <= 4 a pass of exactly rem slots
// (no load is issued for a slot that is not there), else a masked pass of U.
// before() runs between the issue and the products (the pipelined driver
// multiplies its pending pass there).
template <int U, typename Ops, typename F>
__device__ __forceinline__ void ks_tail(Ops &ops, int32_t rem, F &&before, typename Ops::Acc &acc) {
  if constexpr (U <= 4) {
    if (rem == 1) {
      typename Ops::template Buf<1> t;
      ops.template issue<1>(t);
      __builtin_amdgcn_sched_barrier(0);
      before();
      ops.fma(t, acc);
    }
    if constexpr (U > 2) {
      if (rem == 2) {
        typename Ops::template Buf<2> t;
        ops.template issue<2>(t);
        __builtin_amdgcn_sched_barrier(0);
        before();
        ops.fma(t, acc);
      }
    }
    if constexpr (U > 3) {
      if (rem == 3) {
        typename Ops::template Buf<3> t;
        ops.template issue<3>(t);
        __builtin_amdgcn_sched_barrier(0);
        before();
        ops.fma(t, acc);
      }
    }
  } else {
    typename Ops::template Buf<U> t;
    ops.template issue<U, true>(t, rem);
    __builtin_amdgcn_sched_barrier(0);
    before();
    ops.fma(t, acc);
  }
}

// all n slots of one group of a slice, U per pass.  PIPE: the loads of pass p+1
// are issued before the products of pass p (two passes in flight; the passes
// alternate between two buffers so no loaded register is copied while its load
// is outstanding, and the scheduling barriers keep the compiler from moving
// the products of a pass above the issue of the next one).  The products are
// summed in pass order either way; ops.flush(acc) marks where the ops may move
// partial sums into their final accumulators (after every second pass and at
// the end).
template <int U, bool PIPE, typename Ops>
__device__ __forceinline__ void ks_run(Ops ops, int32_t n, typename Ops::Acc &acc) {
  static_assert(U - 1 <= QH_KS_PAD, "tail pass reads past the padding");
  typename Ops::template Buf<U> a, b;
  const int32_t np = n / U, rem = n % U;
  if (!PIPE || np == 0) {
    for (int32_t p = 0; p < np; p++) {
      ops.template issue<U>(a);
      ops.fma(a, acc);
      ops.flush(acc);
    }
    if (rem) ks_tail<U>(ops, rem, [] {}, acc);
    ops.flush(acc);
    return;
  }
  ops.template issue<U>(a);
  int32_t p = 1;
  for (; p + 1 < np; p += 2) {
    ops.template issue<U>(b);
    __builtin_amdgcn_sched_barrier(0);
    ops.fma(a, acc);
    ops.template issue<U>(a);
    __builtin_amdgcn_sched_barrier(0);
    ops.fma(b, acc);
    ops.flush(acc);
  }
  if (p < np) {  // a in flight, one full pass left
    ops.template issue<U>(b);
    __builtin_amdgcn_sched_barrier(0);
    ops.fma(a, acc);
    if (rem)
      ks_tail<U>(ops, rem, [&] { ops.fma(b, acc); }, acc);
    else
      ops.fma(b, acc);
  } else {  // a in flight, no full pass left
    if (rem)
      ks_tail<U>(ops, rem, [&] { ops.fma(a, acc); }, acc);
    else
      ops.fma(a, acc);
  }
  ops.flush(acc);
}

__device__ inline uint64_t wave_min_u64(uint64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint64_t o = __shfl_xor(v, off, 64);
    v = o < v ? o : v;
  }
  return v;
}


}  // namespace
