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

// A store that the caches treat as streaming (non-temporal) when NT: the
// outputs are written once and not read again by the kernel.
template <bool NT, typename T>
__device__ inline void put(T* dst, T x) {
  if constexpr (NT) __builtin_nontemporal_store(x, dst);
  else *dst = x;
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));   // 16 bytes at a 4-byte-aligned address

// Copy `words` floats from the LDS block to dst (the first record of the
// wave's knots) in 16-byte pieces, whatever dst's alignment.  Called by the
// whole wave after a wave_lds_sync.  NT: streaming
// stores (whole lines here, unlike a lane's own record stores, which leave
// lines partly written); the flat one-lane kernel at 2^20 knots measured 189
// against 201 us with them.  WORDS: the words of a whole block, whose pieces
// are read from LDS kCopyAhead at a time ahead of their stores, so that a
// block's copy meets the LDS latency 4 times and not 28 (0: one by one): array
// of structures, 20,000 knots 10.8 -> 9.8 us, 1,000,003 knots 105.7 -> 102.0;
// external forces, 150,001 knots 27.1 -> 24.7.
constexpr int kCopyAhead = 7;
template <bool NT = false, int WORDS = 0>
__device__ inline void copy_record_block(const float* rec, float* dst, int words, int lane) {
  v4u* d4 = reinterpret_cast<v4u*>(dst);
  const v4f* s4 = reinterpret_cast<const v4f*>(rec);
  if (WORDS > 0 && words == WORDS) {
    constexpr int pieces = (WORDS / 4 + 63) / 64;
    static_for<0, (pieces + kCopyAhead - 1) / kCopyAhead>([&](auto Gc) {
      constexpr int g = decltype(Gc)::value * kCopyAhead;
      v4f x[kCopyAhead];
      static_for<0, kCopyAhead>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value, p = g + j;
        if (p < pieces && (64 * p + 63 < WORDS / 4 || lane < WORDS / 4 - 64 * p)) x[j] = s4[64 * p + lane];
      });
      static_for<0, kCopyAhead>([&](auto Jc) {
        constexpr int j = decltype(Jc)::value, p = g + j;
        if (p < pieces && (64 * p + 63 < WORDS / 4 || lane < WORDS / 4 - 64 * p)) put<NT>(d4 + 64 * p + lane, v4u(x[j]));
      });
    });
  } else {
    for (int e = lane; e < words / 4; e += 64) put<NT>(d4 + e, v4u(s4[e]));
  }
  const int rest = words & 3;
  if (lane < rest) put<NT>(dst + (words - rest) + lane, rec[words - rest + lane]);
}

// `words` (4 to F) contiguous floats from memory to LDS through the wave's
// registers in 16-byte pieces, piece 64 j + lane in x[j] and the last few
// floats one to a lane: load_block issues every load, put_block writes what
// arrived.  In a short block the places past the end take the last whole piece
// again, in place of a branch around each.  Read float by float, a short or
// unaligned block cost a round trip to memory for every 64 floats
// (33,000 knots, 40 in the last block: finish with the gradient
// before it 25.2 -> 14.5 us, the split layout's three calls 52.9 -> 24.7).
template <int F> constexpr int kBlockPieces = F / 4;
template <int F> constexpr int kLanePieces = (kBlockPieces<F> + 63) / 64;
template <int F> struct BlockPieces {
  v4f x[kLanePieces<F>];
  float rest;
};
template <int F>
__device__ RBD_INLINE void load_block(const float* src, int words, int lane, BlockPieces<F>& b) {
  const v4u* s4 = reinterpret_cast<const v4u*>(src);
  if (words == F) {
    static_for<0, kLanePieces<F>>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      if (64 * j + 63 < kBlockPieces<F> || lane < kBlockPieces<F> - 64 * j) b.x[j] = s4[64 * j + lane];
    });
  } else {
    const int last = words / 4 - 1;
    static_for<0, kLanePieces<F>>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      b.x[j] = s4[min(64 * j + lane, last)];
    });
  }
  if (lane < (words & 3)) b.rest = src[(words & ~3) + lane];
}
template <int F>
__device__ RBD_INLINE void put_block(const BlockPieces<F>& b, int words, int lane, float* rec) {
  v4f* r4 = reinterpret_cast<v4f*>(rec);
  if (words == F) {
    static_for<0, kLanePieces<F>>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      if (64 * j + 63 < kBlockPieces<F> || lane < kBlockPieces<F> - 64 * j) r4[64 * j + lane] = b.x[j];
    });
  } else {
    const int last = words / 4 - 1;
    static_for<0, kLanePieces<F>>([&](auto Jc) {
      constexpr int j = decltype(Jc)::value;
      r4[min(64 * j + lane, last)] = b.x[j];
    });
  }
  if (lane < (words & 3)) rec[(words & ~3) + lane] = b.rest;
}

// Whether a one-lane kernel of precision P keeps a knot's outputs in registers
// until they are complete: with FP32 columns they fit in the 256 registers of
// two waves per SIMD (what the derivative pass no longer needs makes room for
// them; the iiwa's array-of-structures kernel 253 and none spilled, external
// forces 1 spilled, the 147 floats of the WAFR layout 23; the synthetic arm's
// kernels 34 to 53); with FP64 columns they go into LDS as they come.
template <class P> constexpr bool kHoldOutputs = kWavesPerSimd<P> == 2;
// Floats of LDS for records of REC floats
template <class P, int REC> constexpr int kRecordLds = (kHoldOutputs<P> ? 32 : 64) * REC;

// The records of a wave's 64 knots to dst, nk of them: each lane's from the
// registers at r, 32 at a time through LDS (kHoldOutputs), or from the LDS
// block they were written to.  rec: kRecordLds<P, REC> floats, free when the
// call returns.
template <class P, int REC>
__device__ RBD_INLINE void put_records(const float* r, float* rec, float* dst, int nk, int lane) {
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
      copy_record_block<true, 32 * REC>(rec, dst + 32 * h * REC, (left < 0 ? 0 : left < 32 ? left : 32) * REC, lane);
      wave_lds_sync();                    // read out before the next records overwrite it
    });
  } else {
    (void)r;
    copy_record_block<true, 64 * REC>(rec, dst, nk * REC, lane);
    wave_lds_sync();
  }
}

// A one-lane kernel's loop over the wave's blocks of 64 knots with records of
// REC floats: load(k, in) reads knot k's inputs into registers, compute(in, p,
// k0, nk) computes the knot and stores its record at p, and the wave writes
// the nk records of knots k0.. to out.
//
// With the outputs in registers, 32 records go through LDS at a time, so a
// wave needs 13,440 bytes and a CU runs 8 waves; with the whole block in LDS
// it ran 6 (array of structures, 100,003 knots 20.5 -> 15.2 us: one round of
// waves instead of two; 1,000,003 knots 114 -> 106).  The next block's loads are issued before
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
    put_records<P, REC>(r, rec, out + k0 * REC, nk, lane);
  }
}

}  // namespace rbd
