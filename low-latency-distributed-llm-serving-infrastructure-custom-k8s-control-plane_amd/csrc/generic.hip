// Generic paged attention: one wavefront per (query token, query head).
//
// Covers every shape the tuned kernels do not (head dims other than 64 and
// 128 up to 256, groups above 64, block sizes that are not powers of two)
// and, with flat_attention_kernel below, implements the reference C ABI
// (csrc/include/paged_kernels.h:22-34) over a flat gather list plus a dense
// uint8 mask.  Semantics follow csrc/src/paged_kernels.cpp:30-104: masked
// context tokens are skipped, a row with no attended token and an empty
// context produce zeros.  Softmax is computed online (running max and sum)
// in base 2, accumulation is fp32.
//
// Context tokens are visited in chunks of 64: each lane resolves one token's
// slot (from the mask + gather list, or from the block table), a ballot
// keeps the attended ones, and the wave then walks them in ascending order,
// the lanes splitting the head dimension.
#include "pa_common.hpp"
#include "pa_launch.hpp"

namespace pa {

template <typename T, int EPL, bool kMasked>
__global__ __launch_bounds__(kWave) void generic_attention_kernel(GenericArgs a) {
  const int lane = threadIdx.x;
  const int hq = a.num_query_heads;
  const int64_t rowid = blockIdx.x;
  const int t = static_cast<int>(rowid / hq);
  const int h = static_cast<int>(rowid - static_cast<int64_t>(t) * hq);
  const int group = hq / a.num_kv_heads;
  const int kvh = h / group;
  const int D = a.head_dim;
  const int64_t row_stride = static_cast<int64_t>(a.num_kv_heads) * D;

  int seq = 0;
  int64_t trow = 0;
  int n_ctx;
  if constexpr (kMasked) {
    n_ctx = a.num_context_tokens;
  } else {
    // Largest s with cu_seqlens[s] <= t.
    int lo = 0, hi = a.num_seqs;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (a.cu_seqlens[mid] <= t) lo = mid; else hi = mid;
    }
    seq = lo;
    trow = a.rows != nullptr ? a.rows[seq] : seq;
    const int64_t first = a.cu_seqlens[seq];
    const int64_t count = a.cu_seqlens[seq + 1] - first;
    if ((a.filter == 1 && count != 1) || (a.filter == 2 && count == 1)) return;
    const int64_t pos = a.context_lens[seq] - count + (t - first);
    n_ctx = static_cast<int>(pos + 1);
    if (n_ctx < 0) n_ctx = 0;
  }

  const T* qrow = reinterpret_cast<const T*>(a.query) + t * a.q_token_stride + h * a.q_head_stride;
  float q[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const int d = lane + e * kWave;
    q[e] = d < D ? load_scalar<T>(qrow + d) : 0.f;
  }
  const T* kbase = reinterpret_cast<const T*>(a.key_cache) + kvh * D;
  const T* vbase = reinterpret_cast<const T*>(a.value_cache) + kvh * D;

  float m = kScoreFloor, l = 0.f;
  float acc[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = 0.f;

  for (int c0 = 0; c0 < n_ctx; c0 += kWave) {
    const int c = c0 + lane;
    int64_t slot = -1;
    if (c < n_ctx) {
      if constexpr (kMasked) {
        if (a.mask[static_cast<int64_t>(t) * n_ctx + c] != 0) {
          slot = a.gather_slots[c];
          if (slot >= static_cast<int64_t>(a.total_blocks) * a.block_size) slot = -1;
        }
      } else {
        const int col = c / a.block_size;
        if (trow >= 0 && trow < a.num_table_rows && col < a.block_table_stride) {
          const int b = a.block_tables[trow * a.block_table_stride + col];
          if (b >= 0 && b < a.total_blocks)
            slot = static_cast<int64_t>(b) * a.block_size + (c - col * a.block_size);
        }
      }
    }
    uint64_t live = __ballot(slot >= 0);
    while (live) {
      const int src = __builtin_ctzll(live);
      live &= live - 1;
      const int64_t s = __shfl(slot, src, kWave);
      const T* krow = kbase + s * row_stride;
      const T* vrow = vbase + s * row_stride;
      float part = 0.f;
      float v[EPL];
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        const int d = lane + e * kWave;
        const bool in = d < D;
        part = fmaf(q[e], in ? load_scalar<T>(krow + d) : 0.f, part);
        v[e] = in ? load_scalar<T>(vrow + d) : 0.f;
      }
      const float score = wave_sum(part) * a.scale_log2e;
      const float m_new = fmaxf(m, score);
      const float alpha = fast_exp2(m - m_new);
      const float p = fast_exp2(score - m_new);
      l = l * alpha + p;
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[e] = fmaf(p, v[e], acc[e] * alpha);
      m = m_new;
    }
  }

  T* orow = reinterpret_cast<T*>(a.output) + (static_cast<int64_t>(t) * hq + h) * D;
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const int d = lane + e * kWave;
    if (d < D) store_scalar<T>(orow + d, acc[e] * inv);
  }
}

// The reference ABI's flat call for fp32 rows of whole 16-byte pieces: one
// workgroup of W waves per (query token, GH query heads of one KV head).
//
// The call is a chain of dependent reads, not bytes: 8 tokens x 8 heads over
// 2000 gathered slots touch 4 MB.  One wave walking a row's attended tokens
// one at a time (generic_attention_kernel) took 168 us for that call, each
// token a K round trip, a 64-lane sum and the softmax recurrence.  Here
//  * the waves scan the mask row together, kIter * 64 consecutive slots a
//    wave with all their bytes in flight, and compact the attended slots into
//    an LDS list (ascending), so that the attended tokens are dealt evenly
//    over the workgroup whatever their position in the row;
//  * a row group of LPR lanes holds a K/V row, 16 bytes a lane, and keeps its
//    own (max, sum, acc) over kUnroll tokens a step, whose K and V loads go
//    out together; the groups combine once at the end;
//  * GH heads share each K/V row and the scan.
// Measured from a HIP graph, one wave per row -> this kernel: 8 tokens x 8
// heads of 64 over 1471 slots 165 -> 7.7 us.  One head per workgroup against
// the group's four: 32 tokens x 32/8 heads of 128 over 17K slots 99 -> 44 us,
// 128 tokens over 37K 413 -> 102 us; 8 tokens (64 workgroups) 33 -> 35 us.
template <int LPR, int W, int GH>
__global__ __launch_bounds__(W* kWave) void flat_attention_kernel(GenericArgs a) {
  constexpr int kIter = W == 4 ? 16 : 8;      // mask bytes a lane reads per segment
  constexpr int kWaveSlots = kIter * kWave;   // consecutive slots a wave scans
  constexpr int kSegment = W * kWaveSlots;    // slots per pass over the list
  constexpr int RPW = kWave / LPR;            // rows per wave load
  constexpr int kGroups = W * RPW;
  constexpr int kUnroll = 4;
  // The list of a segment, and after the last one the waves' accumulators
  // [W][GH][LPR] (16 bytes each).
  constexpr int kAccInts = W * GH * LPR * 4;
  __shared__ __align__(16) int s_buf[kSegment > kAccInts ? kSegment : kAccInts];
  __shared__ int s_count[W];
  __shared__ float s_m[W][GH], s_l[W][GH];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int hq = a.num_query_heads;
  const int units = hq / GH;  // workgroups per query token
  const int64_t unit = blockIdx.x;
  const int t = static_cast<int>(unit / units);
  const int h0 = static_cast<int>(unit - static_cast<int64_t>(t) * units) * GH;
  const int kvh = h0 / (hq / a.num_kv_heads);
  const int D = a.head_dim;
  const int64_t row_stride = static_cast<int64_t>(a.num_kv_heads) * D;
  const int n_ctx = a.num_context_tokens;
  const int64_t num_slots = static_cast<int64_t>(a.total_blocks) * a.block_size;
  const uint8_t* mask = a.mask + static_cast<int64_t>(t) * n_ctx;

  // Lanes whose piece lies past D read the row's first piece, add nothing to
  // the scores and are never stored.
  const int lig = lane % LPR;
  const bool in = lig * 4 < D;
  const int piece = in ? lig * 4 : 0;
  const float* kbase = reinterpret_cast<const float*>(a.key_cache) + kvh * D + piece;
  const float* vbase = reinterpret_cast<const float*>(a.value_cache) + kvh * D + piece;
  const int group = wave * RPW + lane / LPR;
  float4 q[GH], acc[GH];
  float m[GH], l[GH];
#pragma unroll
  for (int g = 0; g < GH; ++g) {
    q[g] = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(a.query) + t * a.q_token_stride +
                                            (h0 + g) * a.q_head_stride + piece);
    m[g] = kScoreFloor;
    l[g] = 0.f;
    acc[g] = make_float4(0.f, 0.f, 0.f, 0.f);
  }

  for (int64_t seg = 0; seg < n_ctx; seg += kSegment) {
    // The attended slots of this segment -> s_buf.
    const int left = static_cast<int>(min<int64_t>(kSegment, n_ctx - seg));
    const int c0 = wave * kWaveSlots + lane;
    int slot[kIter];
#pragma unroll
    for (int i = 0; i < kIter; ++i) {
      const int c = c0 + i * kWave;
      slot[i] = c < left ? mask[seg + c] : 0;
    }
#pragma unroll
    for (int i = 0; i < kIter; ++i) slot[i] = slot[i] != 0 ? a.gather_slots[seg + c0 + i * kWave] : -1;
    uint64_t live[kIter];
    int count = 0;
#pragma unroll
    for (int i = 0; i < kIter; ++i) {
      live[i] = __ballot(slot[i] >= 0 && slot[i] < num_slots);
      count += __popcll(live[i]);
    }
    if (lane == 0) s_count[wave] = count;
    __syncthreads();
    int at = 0, n = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      if (w < wave) at += s_count[w];
      n += s_count[w];
    }
#pragma unroll
    for (int i = 0; i < kIter; ++i) {
      if ((live[i] >> lane) & 1)
        s_buf[at + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(live[i] >> 32),
                                             __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(live[i]), 0))] = slot[i];
      at += __popcll(live[i]);
    }
    __syncthreads();

    // Row group g takes tokens g, g + kGroups, ... of the list.
    for (int base = 0; base < n; base += kGroups * kUnroll) {
      float4 k[kUnroll], v[kUnroll];
      bool ok[kUnroll];
#pragma unroll
      for (int u = 0; u < kUnroll; ++u) {
        const int i = base + u * kGroups + group;
        ok[u] = i < n;
        const int64_t off = s_buf[ok[u] ? i : 0] * row_stride;
        k[u] = *reinterpret_cast<const float4*>(kbase + off);
        v[u] = *reinterpret_cast<const float4*>(vbase + off);
      }
      // A slot past the list repeats the first one: no weight, and its V
      // (which may hold an infinity) stays out of the product.
#pragma unroll
      for (int u = 0; u < kUnroll; ++u)
        v[u] = make_float4(ok[u] ? v[u].x : 0.f, ok[u] ? v[u].y : 0.f, ok[u] ? v[u].z : 0.f, ok[u] ? v[u].w : 0.f);
#pragma unroll
      for (int g = 0; g < GH; ++g) {
        float s[kUnroll];
        float m_new = m[g];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const float dot = fmaf(q[g].x, k[u].x, fmaf(q[g].y, k[u].y, fmaf(q[g].z, k[u].z, q[g].w * k[u].w)));
          float x = group_sum<16>(in ? dot : 0.f);
          if constexpr (LPR >= 32) x = sum_row_pairs(x);
          if constexpr (LPR >= 64) x = sum_halves(x);
          s[u] = ok[u] ? x * a.scale_log2e : -INFINITY;
          m_new = fmaxf(m_new, s[u]);
        }
        const float alpha = fast_exp2(m[g] - m_new);
        m[g] = m_new;
        l[g] *= alpha;
        acc[g] = make_float4(acc[g].x * alpha, acc[g].y * alpha, acc[g].z * alpha, acc[g].w * alpha);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
          const float p = fast_exp2(s[u] - m_new);
          l[g] += p;
          acc[g].x = fmaf(p, v[u].x, acc[g].x);
          acc[g].y = fmaf(p, v[u].y, acc[g].y);
          acc[g].z = fmaf(p, v[u].z, acc[g].z);
          acc[g].w = fmaf(p, v[u].w, acc[g].w);
        }
      }
    }
    __syncthreads();  // the list is rewritten by the next segment
  }

  // Row groups of the wave, then the waves.
  float4* s_acc = reinterpret_cast<float4*>(s_buf);
#pragma unroll
  for (int g = 0; g < GH; ++g) {
#pragma unroll
    for (int o = LPR; o < kWave; o <<= 1) {
      const float mo = __shfl_xor(m[g], o, kWave), lo = __shfl_xor(l[g], o, kWave);
      const float mn = fmaxf(m[g], mo);
      const float wa = fast_exp2(m[g] - mn), wb = fast_exp2(mo - mn);
      m[g] = mn;
      l[g] = l[g] * wa + lo * wb;
      acc[g].x = acc[g].x * wa + __shfl_xor(acc[g].x, o, kWave) * wb;
      acc[g].y = acc[g].y * wa + __shfl_xor(acc[g].y, o, kWave) * wb;
      acc[g].z = acc[g].z * wa + __shfl_xor(acc[g].z, o, kWave) * wb;
      acc[g].w = acc[g].w * wa + __shfl_xor(acc[g].w, o, kWave) * wb;
    }
    if (lane < LPR) s_acc[(wave * GH + g) * LPR + lane] = acc[g];
    if (lane == 0) {
      s_m[wave][g] = m[g];
      s_l[wave][g] = l[g];
    }
  }
  __syncthreads();
  const float* accs = reinterpret_cast<const float*>(s_acc);
  for (int i = threadIdx.x; i < GH * D; i += W * kWave) {
    const int g = i / D, d = i - g * D;
    float mx = s_m[0][g];
#pragma unroll
    for (int w = 1; w < W; ++w) mx = fmaxf(mx, s_m[w][g]);
    float sum = 0.f, o = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float f = fast_exp2(s_m[w][g] - mx);
      sum = fmaf(s_l[w][g], f, sum);
      o = fmaf(accs[(w * GH + g) * LPR * 4 + d], f, o);
    }
    reinterpret_cast<float*>(a.output)[(static_cast<int64_t>(t) * hq + h0 + g) * D + d] =
        o * (sum > 0.f ? 1.f / sum : 0.f);
  }
}

bool generic_supported(int dtype, int head_dim) {
  if (dtype != PA_DTYPE_F32 && dtype != PA_DTYPE_BF16 && dtype != PA_DTYPE_F16) return false;
  return head_dim >= 1 && head_dim <= 256;
}

template <typename T, bool kMasked>
static hipError_t launch_generic_t(const GenericArgs& a, hipStream_t s) {
  const int64_t rows = static_cast<int64_t>(a.num_query_tokens) * a.num_query_heads;
  if (rows <= 0) return hipSuccess;
  const dim3 grid(static_cast<uint32_t>(rows));
  if (a.head_dim <= 64)
    hipLaunchKernelGGL((generic_attention_kernel<T, 1, kMasked>), grid, dim3(kWave), 0, s, a);
  else if (a.head_dim <= 128)
    hipLaunchKernelGGL((generic_attention_kernel<T, 2, kMasked>), grid, dim3(kWave), 0, s, a);
  else
    hipLaunchKernelGGL((generic_attention_kernel<T, 4, kMasked>), grid, dim3(kWave), 0, s, a);
  return hipGetLastError();
}

// Most workgroups that get 16 waves each (segments of 8192 slots) instead of
// 4 (4096): few units leave CUs idle, so a unit's tokens want more loads in
// flight; many fill the chip with 4.  16 / 4 waves, us: 64 units 7.8 / 9.2,
// 160 units 22.5 / 30.0, 256 units 43.9 / 67.0 (64 of short contexts 10.6 /
// 8.5), 512 units 57.7 / 54.2, 1024 units 139.6 / 102.3.
#ifndef PA_FLAT_WIDE_UNITS
#define PA_FLAT_WIDE_UNITS 384
#endif
constexpr int64_t kFlatWideUnits = PA_FLAT_WIDE_UNITS;

static bool flat_fast_path_supported(const GenericArgs& a) {
  const auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  return a.head_dim % 4 == 0 && a.head_dim <= 256 && aligned(a.query) && aligned(a.key_cache) &&
         aligned(a.value_cache);
}

template <int LPR, int GH>
static hipError_t launch_flat_units(const GenericArgs& a, hipStream_t s) {
  const int64_t units = static_cast<int64_t>(a.num_query_tokens) * (a.num_query_heads / GH);
  if (units <= 0) return hipSuccess;
  const dim3 grid(static_cast<uint32_t>(units));
  if (units <= kFlatWideUnits)
    hipLaunchKernelGGL((flat_attention_kernel<LPR, 16, GH>), grid, dim3(16 * kWave), 0, s, a);
  else
    hipLaunchKernelGGL((flat_attention_kernel<LPR, 4, GH>), grid, dim3(4 * kWave), 0, s, a);
  return hipGetLastError();
}

template <int LPR>
static hipError_t launch_flat_rows(const GenericArgs& a, hipStream_t s) {
  const int group = a.num_query_heads / a.num_kv_heads;
  return group % 4 == 0   ? launch_flat_units<LPR, 4>(a, s)
         : group % 3 == 0 ? launch_flat_units<LPR, 3>(a, s)
         : group % 2 == 0 ? launch_flat_units<LPR, 2>(a, s)
                          : launch_flat_units<LPR, 1>(a, s);
}

hipError_t launch_flat(const GenericArgs& a, hipStream_t s) {
  if (!flat_fast_path_supported(a)) return launch_generic_t<float, true>(a, s);
  return a.head_dim <= 64    ? launch_flat_rows<16>(a, s)
         : a.head_dim <= 128 ? launch_flat_rows<32>(a, s)
                             : launch_flat_rows<64>(a, s);
}

hipError_t launch_generic(const GenericArgs& a, int dtype, hipStream_t s) {
  switch (dtype) {
    case PA_DTYPE_F32:
      return launch_generic_t<float, false>(a, s);
    case PA_DTYPE_BF16:
      return launch_generic_t<bf16_t, false>(a, s);
    case PA_DTYPE_F16:
      return launch_generic_t<f16_t, false>(a, s);
    default:
      return hipErrorNotSupported;
  }
}

}  // namespace pa
