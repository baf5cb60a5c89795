// Runs of consecutive elements per lane, moved through LDS by the whole wave.
//
// In a scan every lane owns a run of consecutive elements.  Read by the lane
// itself, each 16-byte load of a wave touches 64 cache lines and uses an eighth
// of each; the runs of a CU's waves outgrow its 32 KiB L1, so the lines come
// again for every piece.  Here the wave moves chunks of E elements of all its
// runs: P = 2 E neighbouring lanes take one chunk's 16-byte pieces, so an
// instruction touches whole lines only, and the pieces change hands in LDS.
//
// The buffer is the wave's own: in LDS a wave's operations complete in order,
// so only the compiler has to be kept from reordering them (stage_sync), and
// no barrier is needed.  Slots are XOR-swizzled: both the pieces of
// neighbouring lanes and one piece of eight neighbouring runs fall into all
// eight 16-byte bank groups.
//
// It pays where a sweep waits for its lines (the division's, 2^24: 331 -> 266
// us); the grand product's sweeps, bound by products and by the registers their
// local prefixes hold, were slower with it (2^20 rows 37.7 -> 44, 2^21 prefix
// products 63.8 -> 66.8), as was the mid-size division (24.8 -> 25.4).
#pragma once
#include "fr29.hpp"

namespace pl {

__device__ __forceinline__ void stage_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

template <int E>
struct RunStage {
  static_assert(E == 4, "the swizzle is made for chunks of 128 bytes");
  static constexpr int P = 2 * E;        // pieces per chunk
  static constexpr int kRuns = 64 / P;   // runs per instruction
  static constexpr int kSlots = 64 * P;  // 16-byte slots per wave
  uint4* lds;
  int lane;

  __device__ __forceinline__ int slot(int run, int p) const { return run * P + (p ^ (run & (P - 1))); }

  // The chunks at src + stride * run, run < 64: raw[q] is piece lane % P of
  // run q * kRuns + lane / P.  lim: elements that may be read from src on (the
  // pieces past them are zero); all (wave-uniform): every piece may be.
  __device__ __forceinline__ void fetch(const fr* src, int stride, int64_t lim, bool all, uint4 (&raw)[P]) const {
    const int run = lane / P, p = lane % P;
    const uint4* s = (const uint4*)src + (2 * stride * run + p);
    if (all) {
#pragma unroll
      for (int q = 0; q < P; q++) raw[q] = s[2 * stride * kRuns * q];
    } else {
#pragma unroll
      for (int q = 0; q < P; q++)
        raw[q] = stride * (run + kRuns * q) + p / 2 < lim ? s[2 * stride * kRuns * q] : make_uint4(0, 0, 0, 0);
    }
  }
  // the fetched pieces into the buffer, for every lane to take its own chunk
  __device__ __forceinline__ void put(const uint4 (&raw)[P]) const {
    stage_sync();
#pragma unroll
    for (int q = 0; q < P; q++) lds[slot(lane / P + kRuns * q, lane % P)] = raw[q];
    stage_sync();
  }
  // element e of the lane's chunk
  __device__ __forceinline__ fr get(int e) const {
    const uint4 a = lds[slot(lane, 2 * e)], b = lds[slot(lane, 2 * e + 1)];
    fr v;
    v.l[0] = a.x; v.l[1] = a.y; v.l[2] = a.z; v.l[3] = a.w;
    v.l[4] = b.x; v.l[5] = b.y; v.l[6] = b.z; v.l[7] = b.w;
    return v;
  }
  __device__ __forceinline__ void set(int e, const fr& v) const {
    lds[slot(lane, 2 * e)] = make_uint4(v.l[0], v.l[1], v.l[2], v.l[3]);
    lds[slot(lane, 2 * e + 1)] = make_uint4(v.l[4], v.l[5], v.l[6], v.l[7]);
  }
  // the buffer's chunks to dst + stride * run, bounds as for fetch
  __device__ __forceinline__ void store(fr* dst, int stride, int64_t lim, bool all) const {
    stage_sync();
    const int run = lane / P, p = lane % P;
    uint4* d = (uint4*)dst + (2 * stride * run + p);
#pragma unroll
    for (int q = 0; q < P; q++) {
      const uint4 v = lds[slot(run + kRuns * q, p)];
      if (all || stride * (run + kRuns * q) + p / 2 < lim) d[2 * stride * kRuns * q] = v;
    }
  }
};

}  // namespace pl
