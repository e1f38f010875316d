// Whole-record output through LDS for the one-lane-per-knot kernels (device
// code).  A wave's 64 consecutive knots have one contiguous block of records
// (64 x 105 floats = 26,880 bytes); the lanes hand their records over in LDS
// (at the record stride, 105 floats: odd, so their writes fall in different
// banks), and the wave copies them out with consecutive lanes on consecutive
// 16-byte pieces: every store covers 1 KB of contiguous output instead of 64
// records' cache lines.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fdgrad_knot.hpp"

namespace rbd {

constexpr int kRecordBlockFloats = 64 * kOutPerKnot;   // one wave's records

// A store that the caches treat as streaming (non-temporal) when NT: the
// outputs are written once and not read again by the kernel.
template <bool NT, typename T>
__device__ inline void put(T* dst, T x) {
  if constexpr (NT) __builtin_nontemporal_store(x, dst);
  else *dst = x;
}

// Copy `words` floats from the LDS block to dst (the first record of the
// wave's knots): 16-byte pieces when dst is 16-byte aligned, single floats
// otherwise.  Called by the whole wave after a wave_lds_sync.  NT: streaming
// stores (whole lines here, unlike a lane's own record stores, which leave
// lines partly written); the flat one-lane kernel at 2^20 knots measured 189
// against 201 us with them.
template <bool NT = false>
__device__ inline void copy_record_block(const float* rec, float* dst, int words, int lane) {
  typedef float v4f __attribute__((ext_vector_type(4)));
  if ((reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
    v4f* d4 = reinterpret_cast<v4f*>(dst);
    const v4f* s4 = reinterpret_cast<const v4f*>(rec);
    for (int e = lane; e < words / 4; e += 64) put<NT>(d4 + e, s4[e]);
    for (int e = (words / 4) * 4 + lane; e < words; e += 64) put<NT>(dst + e, rec[e]);
  } else {
    for (int e = lane; e < words; e += 64) put<NT>(dst + e, rec[e]);
  }
}

// Whether a one-lane kernel of precision P keeps a knot's outputs in registers
// until they are complete: with FP32 columns they fit (255 registers, no
// spills, two waves per SIMD: what the derivative pass no longer needs makes
// room for them); with FP64 columns they go into LDS as they come.
template <class P> constexpr bool kHoldOutputs = kWavesPerSimd<P> == 2;
// Floats of LDS for records of REC floats
template <class P, int REC> constexpr int kRecordLds = (kHoldOutputs<P> ? 32 : 64) * REC;

// A one-lane kernel's loop over the wave's blocks of 64 knots with records of
// REC floats: load(k, in) reads knot k's inputs into registers, compute(in, p,
// k0, nk) computes the knot and stores its record at p, and the wave writes
// the nk records of knots k0.. to out.
//
// With the outputs in registers, 32 records go through LDS at a time, so a
// wave needs 13,440 bytes and a CU runs 8 waves; with the whole block in LDS
// it ran 6 (2^20 knots: HOLD_NOTE).  The next block's loads are issued before
// the copies: a wave's vector-memory counter retires loads and stores in the
// order they were issued, so waiting for loads also waits for every store
// issued before them.  Lanes past the last knot compute a copy of it; only nk
// records are written out.  rec: kRecordLds<P, REC> floats or more, which
// compute may use too until it returns.
template <class P, int REC, class In, class Load, class Compute>
__device__ RBD_INLINE void one_lane_records(long n, float* out, float* rec, Load&& load, Compute&& compute) {
  const int lane = int(threadIdx.x);
  const long stride = long(gridDim.x) * 64;
  long k0 = long(blockIdx.x) * 64;
  if (k0 >= n) return;
  In in;
  load(k0 + lane < n ? k0 + lane : n - 1, in);
  for (; k0 < n; k0 += stride) {
    const int nk = int(n - k0 < 64 ? n - k0 : 64);
    float r[kHoldOutputs<P> ? REC : 1];
    compute(in, kHoldOutputs<P> ? r : rec + REC * lane, k0, nk);
    const long k1 = k0 + stride + lane;
    if (k0 + stride < n) load(k1 < n ? k1 : n - 1, in);
    __builtin_amdgcn_sched_barrier(0);
    wave_lds_sync();
    if constexpr (kHoldOutputs<P>) {
      static_for<0, 2>([&](auto Hc) {
        constexpr int h = decltype(Hc)::value;
        if ((lane >> 5) == h) {
          float* d = rec + REC * (lane & 31);
          static_for<0, REC>([&](auto Jc) { d[decltype(Jc)::value] = r[decltype(Jc)::value]; });
        }
        wave_lds_sync();
        const int left = nk - 32 * h;
        copy_record_block<true>(rec, out + (k0 + 32 * h) * REC, (left < 0 ? 0 : left < 32 ? left : 32) * REC, lane);
        wave_lds_sync();                    // read out before the next records overwrite it
      });
    } else {
      copy_record_block<true>(rec, out + k0 * REC, nk * REC, lane);
      wave_lds_sync();
    }
  }
}

}  // namespace rbd
