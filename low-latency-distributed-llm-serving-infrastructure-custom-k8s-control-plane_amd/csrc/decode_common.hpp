// What the decode partition kernels share: the split-K partials' merge, in
// the partition launch and for the merge kernel.
#pragma once

#include "pa_common.hpp"
#include "pa_launch.hpp"

namespace pa {

constexpr int kDecodeThreads = 256;
constexpr int kDecodeWaves = kDecodeThreads / kWave;
// Largest split-K partition (context tokens per workgroup) the kernels take.
constexpr int kMaxPartition = PA_DECODE_MAX_PARTITION;
// Query heads one workgroup of the matrix-core kernel serves.
constexpr int kMfmaHeads = 16;

// K output elements of one head of a multi-partition sequence from its
// split-K partials: ml addresses the head's (max, sum) pair in item 0, acc
// the first element's accumulator and out its output; element k sits
// k * estride elements further.  Partitions 0 .. nfull-1 are items first ..
// first + nfull - 1, partition nfull (when nparts > nfull) is item rem;
// ml_stride / stride step one item.  kMergeBatch partitions per round trip,
// with a running maximum (the stored maxima are already in the exp2
// domain); slots past the last partition read the first one again and get
// no weight.  The elements share each partial's (max, sum), loaded once for
// all of them, and their loads go out together: one round trip per batch
// for the K elements (one after the other, eight heads of 128 took four).
// Each element's arithmetic is the same whatever K, and both merge paths
// (the merge kernel, K = 1, and the in-launch merge of the partition
// kernel) run this, so they give the same bits.
constexpr int kMergeBatch = 8;
constexpr int kMergeOutputs = 4;  // elements a thread of the in-launch merge merges at once

// Partials read by the in-launch merge are written by workgroups on other
// XCDs in the same launch: they are stored and loaded as device-scope
// relaxed atomics, which write through and read past the XCD's L2, so no
// L2 write-back or invalidate is needed (see the partition kernel's tail).
__device__ __forceinline__ void store_device(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float load_device(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T, int K, bool DEVICE_LOADS = false>
__device__ __forceinline__ void merge_partials(const float* ml, const float* acc, int estride, int64_t ml_stride,
                                               int64_t stride, int64_t first, int nfull, int64_t rem, int nparts,
                                               T* out) {
  auto item_of = [&](int p) -> int64_t { return p < nfull ? first + p : rem; };
  auto ld = [&](const float* q) { return DEVICE_LOADS ? load_device(q) : *q; };
  float mx = kScoreFloor, sum = 0.f, o[K];
#pragma unroll
  for (int k = 0; k < K; ++k) o[k] = 0.f;
  for (int p = 0; p < nparts; p += kMergeBatch) {
    float mp[kMergeBatch], lp[kMergeBatch], xp[kMergeBatch][K];
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const int64_t it = item_of(p + u < nparts ? p + u : 0);
      mp[u] = ld(ml + it * ml_stride);
      lp[u] = ld(ml + it * ml_stride + 1);
#pragma unroll
      for (int k = 0; k < K; ++k) xp[u][k] = ld(acc + it * stride + k * estride);
    }
    float mn = mx;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      if (u > 0 && p + u >= nparts) {
        mp[u] = kScoreFloor;
        lp[u] = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k) xp[u][k] = 0.f;
      }
      mn = fmaxf(mn, mp[u]);
    }
    const float r = fast_exp2(mx - mn);
    sum *= r;
#pragma unroll
    for (int k = 0; k < K; ++k) o[k] *= r;
#pragma unroll
    for (int u = 0; u < kMergeBatch; ++u) {
      const float w = fast_exp2(mp[u] - mn);
      sum = fmaf(lp[u], w, sum);
#pragma unroll
      for (int k = 0; k < K; ++k) o[k] = fmaf(xp[u][k], w, o[k]);
    }
    mx = mn;
  }
#pragma unroll
  for (int k = 0; k < K; ++k) store_scalar<T>(out + k * estride, sum > 0.f ? o[k] / sum : 0.f);
}

// The last of a sequence's partition workgroups (for this unit and
// sub-group) to finish merges the sequence's partials; no workgroup waits
// for another.  The workgroups run on different XCDs, whose L2s are
// separate: the partials above are device-scope stores (written through
// past the L2), and every wave waits for its stores to complete before
// the barrier.  Then one thread adds the workgroup's arrival to the
// sequence's 64-bit record with one device-scope atomic: bits 0-15 count
// arrivals, bits 16-39 hold 1 + the item of the partial last partition
// (added by that workgroup) and bits 40-63 1 + the item of partition 0,
// the first of the sequence's full partitions, which pa_pack lists as
// consecutive items (added by that workgroup; the host passes records
// only for fewer than 65535 items, so every field fits).  The workgroup
// whose addition brings the count to nparts has every field in the value
// the atomic returns; it resets the record for the next launch (the
// records start at zero and every launch leaves them at zero) and merges
// as the merge kernel does, with device-scope loads that read past its
// L2.  An agent-scope release or acquire fence here instead writes back or
// invalidates a whole L2 per workgroup, and made the decode slower than a
// second launch.
//
// Called by all kDecodeThreads threads of a workgroup that stored its
// partials of a sequence of nparts > 1 partitions for G query heads from h0
// on (of hq); record: the index of the sequence's record for them.
//
// KC elements of one head per thread, ODM / KC apart, so that the lanes of a
// wave read consecutive floats of each partial; the thread's group r = tid,
// tid + 256, ... covers elements j + k * ODM / KC (k < KC) of head
// r / (ODM / KC), j = r % (ODM / KC).
template <typename T, int ODM, int KC>
__device__ __forceinline__ void merge_in_launch(const DecodeArgs& a, int G, int part, int64_t item, int ctx,
                                                int nparts, int64_t record, int h0, int hq, T* out_row) {
  __shared__ int64_t s_merge[3];
  const int tid = threadIdx.x;
  const int nfull = ctx / a.partition;
  const bool has_rem = nfull * a.partition < ctx;
  uint64_t* rec = reinterpret_cast<uint64_t*>(a.merge_state) + record;
  uint64_t add = 1;
  if (part == 0) add += static_cast<uint64_t>(item + 1) << 40;
  if (part == nfull) add += static_cast<uint64_t>(item + 1) << 16;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const uint64_t now = __hip_atomic_fetch_add(rec, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + add;
    const bool last = static_cast<int>(now & 0xffff) == nparts;
    if (last) {
      __hip_atomic_store(rec, uint64_t{0}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_merge[1] = static_cast<int64_t>(now >> 40) - 1;
      s_merge[2] = static_cast<int64_t>((now >> 16) & 0xffffff) - 1;
    }
    s_merge[0] = last;
  }
  __syncthreads();
  if (s_merge[0]) {
    const int64_t first = s_merge[1];
    const int64_t rem = has_rem ? s_merge[2] : -1;
    const bool ok = first >= 0 && first + nfull <= a.num_items && (!has_rem || (rem >= 0 && rem < a.num_items));
    if (ok) {
      constexpr int RUN = ODM / KC;  // groups per head
      static_assert(ODM % KC == 0, "a group's elements stay inside one head");
      T* out = out_row + static_cast<int64_t>(h0) * ODM;
      for (int r = tid; r < G * RUN; r += kDecodeThreads) {
        const int g = r / RUN;
        const int e = g * ODM + (r - g * RUN);
        merge_partials<T, KC, true>(a.part_ml + 2 * (h0 + g), a.part_acc + static_cast<int64_t>(h0) * ODM + e,
                                    RUN, 2 * static_cast<int64_t>(hq), static_cast<int64_t>(hq) * ODM, first,
                                    nfull, rem, nparts, out + e);
      }
    }
  }
}

// decode_mfma.hip
hipError_t launch_decode_mfma(const DecodeArgs& a, int dtype, int head_dim, int unit_heads, int64_t num_items, hipStream_t stream);
hipError_t decode_mfma_workgroups_per_cu(int dtype, int head_dim, bool shared, int unit_heads, int* per_cu);

}  // namespace pa
