// Paged-attention decode for gfx950 on the vector units: one workgroup per
// (sequence, context partition of up to 4096 tokens, KV head), split-K merge
// after.  fp32 caches and 16-bit heads of 256 run here; 16-bit heads of 64 to
// 128 run on the matrix cores (decode_mfma.hip).
//
// The workgroup (4 waves) serves the G = H_q / H_kv query heads that share
// one KV head, so every K/V row of the partition is read from HBM once
// (groups above 8 run as sub-groups of at most 8 on SHARED instances, whose
// re-reads are ordered to meet in one XCD's L2).  Heads of 64, 128 and 256
// have their own instances; heads of 80 and 96 run those of 128 with the
// pieces past the head masked (DM below).
// The partition is cut into 32-token tiles (16 for groups above 4 and for
// 512-byte rows) dealt round-robin to the waves;
// each wave runs flash-style online softmax over its tiles with no
// workgroup barrier inside the loop:
//
//  K (QK layout)  a "row group" of kL lanes holds one token's K row, each
//                 lane two 16-byte pieces (the group's loads cover the row
//                 contiguously); a wave covers 64 / kL tokens per load.
//                 Dots with the G query slices use v_dot2_f32_bf16 /
//                 v_dot2_f32_f16 (16-bit types) and a DPP butterfly sums
//                 each group; groups of more than 4 on fp32 heads of 64 (row
//                 groups of 8 lanes) use a reduce-scatter instead, after
//                 which each lane holds one head's scores (qk_softmax_rs).
//  V (PV layout)  one wave load covers one V row (4 bytes per lane of 256-byte
//                 rows, 8 of 512), so the row address of a load is
//                 wave-uniform and is formed in scalar registers from the
//                 block id fetched with v_readlane.  Every lane owns a fixed
//                 slice of the head dimension for all G heads.
//  softmax        per tile: wave-wide max per head (DPP + shuffles), rescale
//                 of the running sum / accumulator only when the max moved,
//                 p = exp2(s - max) staged in LDS.  For bf16/fp16 the p of
//                 two tokens are packed as a pair of the cache type and the
//                 PV product uses v_dot2 on the matching V pair (one v_perm_b32 per
//                 two elements); fp32 keeps fp32 FMAs throughout.
//
// At the end the four waves combine (max, sum, acc) through LDS.  A sequence
// whose context fits one partition gets its normalised output directly;
// otherwise the partials go to the workspace and decode_merge_kernel
// combines them.
//
// The reference computes the same quantity with its CPU loop nest
// (csrc/src/paged_kernels.cpp:49-104) over a flat gather list and dense mask.
#include "decode_common.hpp"

namespace pa {

constexpr int kMaxDecodeGroup = 8;  // query heads one workgroup serves
#ifndef PA_DECODE_TILE
#define PA_DECODE_TILE 32  // context tokens per wave iteration (at least 2 rows per group)
#endif
#ifndef PA_DECODE_TILE_WIDE
#define PA_DECODE_TILE_WIDE 16  // the same for groups of more than 4 query heads
#endif

// Tuning switches (compile-time; the defaults are the shipped choice).
#ifndef PA_DECODE_NT
#define PA_DECODE_NT 1  // non-temporal K/V loads
#endif
#ifndef PA_DECODE_MIN_WAVES
#define PA_DECODE_MIN_WAVES 4  // occupancy floor per SIMD for groups of up to 4 heads
#endif
// Occupancy floor for a group of G query heads: the register budget of the
// wider groups does not fit four waves per SIMD without spilling.
#ifndef PA_DECODE_MIN_WAVES_WIDE
#define PA_DECODE_MIN_WAVES_WIDE 2  // the same for wider groups or rows
#endif
#ifndef PA_DECODE_MIN_WAVES_ROW512
#define PA_DECODE_MIN_WAVES_ROW512 3  // the same for 16-bit rows of 512 bytes (D 256)
#endif
#define PA_DECODE_OCCUPANCY(T, D, G)                                                          \
  __attribute__((amdgpu_waves_per_eu(                                                         \
      ((G) <= 4 && sizeof(T) == 2 && (D) * sizeof(T) > 256) ? PA_DECODE_MIN_WAVES_ROW512      \
      : ((G) <= 4 && (D) * sizeof(T) <= 256)                ? PA_DECODE_MIN_WAVES             \
                                                            : PA_DECODE_MIN_WAVES_WIDE)))

typedef unsigned int u32x2v __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4v __attribute__((ext_vector_type(4)));

// K/V loads.  NT: streaming (non-temporal) loads, for rows no other
// workgroup reads; plain cached loads where sibling workgroups re-read them.
template <typename V, bool NT>
__device__ __forceinline__ V kv_load(const void* p);
template <>
__device__ __forceinline__ uint4 kv_load<uint4, true>(const void* p) {
  const u32x4v v = __builtin_nontemporal_load(reinterpret_cast<const u32x4v*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}
template <>
__device__ __forceinline__ uint2 kv_load<uint2, true>(const void* p) {
  const u32x2v v = __builtin_nontemporal_load(reinterpret_cast<const u32x2v*>(p));
  return make_uint2(v.x, v.y);
}
template <>
__device__ __forceinline__ uint32_t kv_load<uint32_t, true>(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(p));
}
template <>
__device__ __forceinline__ uint4 kv_load<uint4, false>(const void* p) {
  return *reinterpret_cast<const uint4*>(p);
}
template <>
__device__ __forceinline__ uint2 kv_load<uint2, false>(const void* p) {
  return *reinterpret_cast<const uint2*>(p);
}
template <>
__device__ __forceinline__ uint32_t kv_load<uint32_t, false>(const void* p) {
  return *reinterpret_cast<const uint32_t*>(p);
}

template <typename T, int D, int TILE>
struct DecodeShape {
  static constexpr bool kHalf = Elem<T>::kBytes == 2;  // bf16 or fp16
  static constexpr int kE = Elem<T>::kBytes;
  static constexpr int kRowBytes = D * kE;
  // QK layout
  static constexpr int kChunkElems = 16 / kE;  // elements per 16-byte piece
  static constexpr int kL = kRowBytes / 32;    // lanes per K row
  static constexpr int kGpw = kWave / kL;      // K rows per wave load
  static constexpr int kTile = TILE >= 2 * kGpw ? TILE : 2 * kGpw;
  static constexpr int kLog2Gpw = kGpw == 4 ? 2 : 3;
  static constexpr int kTpg = kTile / kGpw;    // tile tokens per row group
  // PV layout: a V row per wave load
  static constexpr int kPvBytes = kRowBytes / kWave;
  static constexpr int kPe = kPvBytes / kE;  // elements per lane
  static_assert(kL == 8 || kL == 16, "rows of 256 or 512 bytes");
  static_assert(kTpg >= 2 && kTpg % 2 == 0, "token pairs need an even count per group");
};

template <int NB>
struct VRaw;
template <>
struct VRaw<4> {
  using type = uint32_t;
};
template <>
struct VRaw<8> {
  using type = uint2;
};

// 32-bit word w of a lane's V piece (a pair of 16-bit elements).
__device__ __forceinline__ uint32_t v_word(uint32_t v, int) { return v; }
__device__ __forceinline__ uint32_t v_word(uint2 v, int w) { return w == 0 ? v.x : v.y; }

// Dot product of one lane's K slice (two 16-byte pieces) with its q slice.
template <typename T>
__device__ __forceinline__ float slice_dot(const uint4 (&q)[2], const uint4 (&k)[2]) {
  float acc = 0.f;
  if constexpr (Elem<T>::kBytes == 2) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      acc = dot2_half<T>(q[c].x, k[c].x, acc);
      acc = dot2_half<T>(q[c].y, k[c].y, acc);
      acc = dot2_half<T>(q[c].z, k[c].z, acc);
      acc = dot2_half<T>(q[c].w, k[c].w, acc);
    }
  } else {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      acc = fmaf(__uint_as_float(q[c].x), __uint_as_float(k[c].x), acc);
      acc = fmaf(__uint_as_float(q[c].y), __uint_as_float(k[c].y), acc);
      acc = fmaf(__uint_as_float(q[c].z), __uint_as_float(k[c].z), acc);
      acc = fmaf(__uint_as_float(q[c].w), __uint_as_float(k[c].w), acc);
    }
  }
  return acc;
}

// Max over the lanes of a wave that share (lane % L): every row group.
// Every step pairs lanes of equal (lane % L) only (a rotation by 8 within a
// row of 16, then the row and half swaps), so the lanes of one row group may
// hold different values (the reduce-scatter score layout).
template <int L>
__device__ __forceinline__ float across_groups_max(float x) {
  if constexpr (L == 8) x = fmaxf(x, dpp<kDppRowRor8>(x));
  return max_halves(max_row_pairs(x));
}

// SHARED: the workgroup is one of several sub-groups of a KV head's query
// heads, whose siblings read the same K/V rows (cached loads).
// DM: the head dim in memory, when smaller than the lane layout's D (heads
// of 80 and 96 on the layout of 128).  Lanes whose K pieces or V slice lie
// past DM read the row's first piece or slice instead (always in bounds);
// their q pieces are zero, so those K pieces add nothing to the scores, and
// their accumulators are never stored.
template <typename T, int D, int G, bool SHARED, int DM>
__global__ __launch_bounds__(kDecodeThreads) PA_DECODE_OCCUPANCY(T, D, G) void decode_partition_kernel(DecodeArgs a) {
  // Tiles of 16 tokens for wide groups and for 16-bit rows of 512 bytes
  // (the same bytes per tile as 32 tokens of 256-byte rows).
  using S = DecodeShape<T, D,
                        ((G > 4 || (Elem<T>::kBytes == 2 && D * sizeof(T) > 256)) ? PA_DECODE_TILE_WIDE
                                                                                   : PA_DECODE_TILE)>;
  using VR = typename VRaw<S::kPvBytes>::type;
  // Nontemporal K/V loads, except where other workgroups re-read the same
  // lines: sibling sub-groups (SHARED), and the rows of heads of 80 and 96,
  // whose 128-byte lines straddle two KV heads.
  constexpr bool kNt = PA_DECODE_NT && !SHARED && DM == D;
  constexpr int L = S::kL;
  constexpr int GPW = S::kGpw;
  constexpr int TPG = S::kTpg;
  constexpr int CE = S::kChunkElems;
  constexpr int PE = S::kPe;
  constexpr bool HALF = S::kHalf;  // 16-bit elements (bf16 or fp16)
  // p staging per wave: 16-bit pairs [16 pairs][G] or fp32 [32 tokens][G]
  constexpr int kTile = S::kTile;
  constexpr int PWORDS = HALF ? (kTile / 2) * G : kTile * G;
  constexpr bool MASKD = DM < D;
  constexpr int KPM = DM / S::kChunkElems;  // 16-byte pieces of a row in memory
  static_assert(!MASKD || (!HALF && DM % S::kChunkElems == 0 && KPM >= S::kL && DM % S::kPe == 0),
                "masked head dims: fp32, whole 16-byte pieces, at least one piece per lane");
  // RS: reduce-scatter scores, for groups of more than half a row group of 8
  // lanes: a score position per lane, and lane lig of every row group ends
  // with the scores of query head lig alone (see qk_softmax_rs).
  constexpr bool RS = L == 8 && G > 4;
  static_assert(!RS || (!HALF && G <= 8), "rows of 256 bytes are fp32 heads of 64");

  // Block ids of the partition; its tail from kParkStart holds the new
  // token's pieces and their destinations from the staging to the last tile
  // (pa_decode_append): a 16-byte piece and an 8-byte address per lane.
  constexpr int kBlkInts = kMaxPartition + 2;
  constexpr int kParkStart = (kBlkInts - kWave * 6) & ~3;  // 16-byte aligned
  __shared__ __align__(16) int s_blk[kBlkInts];
  __shared__ uint4 s_q[(RS ? L : G) * D * S::kE / 16];
  __shared__ uint32_t s_p[kDecodeWaves][PWORDS];
  __shared__ float s_m[kDecodeWaves][G];
  __shared__ float s_l[kDecodeWaves][G];
  __shared__ float s_acc[kDecodeWaves][G * D];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int hkv = a.num_kv_heads;
  // Workgroup -> (item, KV head, sub-group of G of the head's a.group query
  // heads; one sub-group unless a.group exceeds the largest kernel group).
  int64_t item;
  int kvh, sg = 0;
  if (a.sub_groups == 1) {
    item = blockIdx.x / hkv;
    kvh = static_cast<int>(blockIdx.x - item * hkv);
  } else {
    // Sibling sub-groups read the same K/V rows.  Workgroup ids are dealt to
    // the XCDs round-robin, so siblings get ids that are equal modulo the XCD
    // count and close together: the later reads hit that XCD's L2.  Runs of
    // kXcds (item, KV head) units, each run repeated once per sub-group; the
    // last run may be shorter.
    const int64_t span = static_cast<int64_t>(kXcds) * a.sub_groups;
    const int64_t run = blockIdx.x / span;
    const int64_t base = run * kXcds;
    const int width = static_cast<int>(min<int64_t>(kXcds, gridDim.x / a.sub_groups - base));
    const int r = static_cast<int>(blockIdx.x - run * span);
    sg = r / width;
    const int64_t u = base + (r - sg * width);
    item = u / hkv;
    kvh = static_cast<int>(u - item * hkv);
  }
  const int h0 = kvh * a.group + sg * G;  // first query head
  const int seq = a.items[2 * item];
  const int part = a.items[2 * item + 1];
  const int64_t trow = a.rows != nullptr ? a.rows[seq] : seq;
  const bool row_ok = trow >= 0 && trow < a.num_table_rows;
  int ctx = a.context_lens[seq];
  int64_t qtok = a.cu_seqlens[seq];
  const int p0 = part * a.partition;
  const int log2_bs = a.log2_block_size;
  const int bs_mask = (1 << log2_bs) - 1;

  // Block ids covering this partition -> LDS (invalid ids become -1).  The
  // whole partition's span is read, whatever the context length, so that
  // the reads do not wait for it (entries past the context are never used);
  // each thread's first entry is loaded here, beside the context length and
  // the query token, and stored with the first query piece below.
  const int first_blk = p0 >> log2_bs;
  const int nblk = ((p0 + a.partition - 1) >> log2_bs) - first_blk + 1;
  auto table_entry = [&](int i) {
    const int col = first_blk + i;
    return row_ok && col < a.block_table_stride ? a.block_tables[trow * a.block_table_stride + col] : -1;
  };
  auto valid_block = [&](int b) { return b < 0 || b >= a.total_blocks ? -1 : b; };
  const int b0 = tid < nblk ? table_entry(tid) : -1;
  // (both scalar loads issued before either is waited for: one round trip)
  asm volatile("" : "+s"(ctx), "+s"(qtok));
  const int n = max(0, min(a.partition, ctx - p0));
  const int64_t row_stride = static_cast<int64_t>(hkv) * DM;
  const T* kbase = reinterpret_cast<const T*>(a.key_cache) + kvh * DM;
  const T* vbase = reinterpret_cast<const T*>(a.value_cache) + kvh * DM;

  // pa_decode_append: the workgroups of the partition holding the new token
  // (position ctx - 1) write its K and V rows of this KV head into
  // the cache, as pa_reshape_and_cache would; sibling
  // sub-groups write the same bytes.  The wave that attends the partition's
  // last tile (the one holding that position) does it, a lane per 16-byte
  // piece: it loads the piece here, so the load overlaps the staging below,
  // parks it in the tail of s_blk (past the partition's block ids) and
  // stores it in the tile loop just before that tile's loads, with a
  // barrier of the wave between them, which orders the stores before its
  // own reads of that position; no other wave or workgroup of the launch
  // reads it.  (Stored at the top of the launch, the rows were counted by
  // every later wait of the wave's loads.)  When the block ids leave no
  // room (more than kParkStart of them: one-token blocks and a partition
  // above 3712 tokens), the pieces are stored before the staging barrier
  // instead, which orders them before the whole workgroup's reads.
  constexpr int kPieceElems = 16 / static_cast<int>(sizeof(T));
  constexpr int kAppendPieces = DM / kPieceElems;  // 16-byte pieces of the unit's row
  static_assert(2 * kAppendPieces <= kWave, "one piece of K or V per lane of a wave");
  const bool append = a.new_key != nullptr && n > 0 && p0 + n == ctx;
  const int last_tile = (n + S::kTile - 1) / S::kTile - 1;
  const int append_wave = append ? last_tile % kDecodeWaves : -1;
  // Lane l's piece: l < kAppendPieces of K, the rest of V; its element in
  // the token's row, and where it goes given the block b holding ctx - 1.
  auto append_elem = [&](int l) { return kvh * DM + (l >= kAppendPieces ? l - kAppendPieces : l) * kPieceElems; };
  auto append_target = [&](int b, int l) {
    const int64_t slot = (static_cast<int64_t>(b) << log2_bs) + ((ctx - 1) & bs_mask);
    return const_cast<T*>(reinterpret_cast<const T*>(l >= kAppendPieces ? a.value_cache : a.key_cache)) +
           slot * row_stride + append_elem(l);
  };
  T* append_dst = nullptr;
  uint4 append_piece = make_uint4(0, 0, 0, 0);
  if (wave == append_wave && lane < 2 * kAppendPieces) {
    const int col = (ctx - 1) >> log2_bs;
    const int b = row_ok && col < a.block_table_stride ? a.block_tables[trow * a.block_table_stride + col] : -1;
    if (b >= 0 && b < a.total_blocks) {
      const bool is_v = lane >= kAppendPieces;
      const T* src = reinterpret_cast<const T*>(is_v ? a.new_value : a.new_key) +
                     qtok * (is_v ? a.new_value_token_stride : a.new_key_token_stride) +
                     static_cast<int64_t>(kvh) * (is_v ? a.new_value_head_stride : a.new_key_head_stride) +
                     (append_elem(lane) - kvh * DM);
      append_dst = append_target(b, lane);
      append_piece = ld16(src);
    }
  }

  // The G query rows of this KV head -> LDS (read back per tile, one head
  // at a time, so they do not occupy registers across the loop).
  const int lig = lane % L;  // lane within its row group
  const int gi = lane / L;   // row group within the wave
  constexpr int QCHUNKS = G * D / CE;  // 16-byte pieces of the G query rows
  constexpr int QN = RS ? 2 * L * L : QCHUNKS;  // 16-byte pieces staged
  auto query_piece = [&](int i) -> uint4 {
    if constexpr (RS) {
      // Per (position p, lane l) of a row group, the two pieces (l and l + L)
      // lane l dots at position p: those of query head p ^ l, zero past G.  A
      // lane's reads for p = 0 .. 7 are then one base address plus constants.
      const int piece = i & 1;
      const int ln = (i >> 1) % L;
      const int g = ((i >> 1) / L) ^ ln;
      const T* qrow = reinterpret_cast<const T*>(a.query) + qtok * a.q_token_stride +
                      static_cast<int64_t>(h0 + min(g, G - 1)) * a.q_head_stride;
      return (g < G && (!MASKD || ln + piece * L < KPM)) ? ld16(qrow + (ln + piece * L) * CE)
                                                        : make_uint4(0, 0, 0, 0);
    } else {
      const int g = i / (D / CE);
      const int c = i - g * (D / CE);
      const T* qrow = reinterpret_cast<const T*>(a.query) + qtok * a.q_token_stride +
                      static_cast<int64_t>(h0 + g) * a.q_head_stride;
      return (!MASKD || c < KPM) ? ld16(qrow + c * CE) : make_uint4(0, 0, 0, 0);
    }
  };
  // Each thread's first table entry and first query piece are both loaded
  // before either is stored, so that the two round trips overlap; the rest
  // (partitions of more than kDecodeThreads blocks, more query pieces than
  // threads) follow.
  {
    const uint4 q0 = tid < QN ? query_piece(tid) : make_uint4(0, 0, 0, 0);
    if (tid < nblk) s_blk[tid] = valid_block(b0);
    if (tid < QN) s_q[tid] = q0;
  }
  for (int i = tid + kDecodeThreads; i < nblk; i += kDecodeThreads) s_blk[i] = valid_block(table_entry(i));
  for (int i = tid + kDecodeThreads; i < QN; i += kDecodeThreads) s_q[i] = query_piece(i);
  // The new token's pieces: parked past the block ids with their
  // destinations (null: none), or (no room there) stored now, before the
  // barrier.
  uint4* const park_piece = reinterpret_cast<uint4*>(s_blk + kParkStart);
  T** const park_dst = reinterpret_cast<T**>(s_blk + kParkStart + kWave * 4);
  const bool park = nblk <= kParkStart;
  // Whether the last tile's wave stores parked pieces (the array's last
  // word, past every block id).
  if (tid == 0) s_blk[kBlkInts - 1] = append && park ? 1 : 0;
  if (wave == append_wave && lane < 2 * kAppendPieces) {
    if (park) {
      park_piece[lane] = append_piece;
      park_dst[lane] = append_dst;
    } else if (append_dst != nullptr) {
      st16(append_dst, append_piece);
    }
  }
  __syncthreads();

  const float scale = a.scale_log2e;
  float m[G], acc[G][PE];
#pragma unroll
  for (int g = 0; g < G; ++g) m[g] = kScoreFloor;
#pragma unroll
  for (int j = 0; j < G; ++j)
#pragma unroll
    for (int e = 0; e < PE; ++e) acc[j][e] = 0.f;

  // ---- per-tile work ------------------------------------------------------
  // A lane's K pieces are lig and lig + L (16-byte pieces of the row).
  // Softmax exponentials are spread over the L lanes of a row group: lane
  // lig owns "combos" k = lig + L*r, each one (token pair,
  // head) for bf16 or (token, head) for fp32, and computes, sums and stages
  // only those.
  constexpr int NC = (HALF ? TPG / 2 : TPG) * G;  // combos per lane group
  constexpr int CPL = (NC + L - 1) / L;           // combos per lane
  float lsum[G];  // this lane's share of the softmax denominators
#pragma unroll
  for (int j = 0; j < G; ++j) lsum[j] = 0.f;
  float ml = kScoreFloor;  // RS: running maximum of the lane's own head (its sum in lsum[0])

  uint4 kb[TPG][2];
  bool kok[TPG];
  VR vb[kTile];

  auto tile_blocks = [&](int tile) {
    const int t = tile * kTile + (lane & (kTile - 1));
    return t < n ? s_blk[((p0 + t) >> log2_bs) - first_blk] : -1;
  };
  // Per-lane element offset of its K slice within a wave load: row group gi
  // reads row gi of the load (GPW consecutive tokens).
  const int64_t koff = static_cast<int64_t>(gi) * row_stride + lig * CE;
  // Second K piece of the lane (its first piece again past DM).
  const int kp1 = (!MASKD || lig + L < KPM) ? lig + L : lig;
  const bool k_uniform = log2_bs >= S::kLog2Gpw;  // a load's GPW tokens share a block
  auto issue_k = [&](int tile, int blk_lane) {
    const int t0 = tile * kTile;
#pragma unroll
    for (int i = 0; i < TPG; ++i) {
      const int t = t0 + gi + GPW * i;
      if (k_uniform) {
        // Block id and row base of the load are wave-uniform (scalar regs).
        // Lanes past the end of the partition still read a row of the same
        // (valid) block; their scores are masked.
        const int b = __builtin_amdgcn_readlane(blk_lane, GPW * i);
        kok[i] = t < n && b >= 0;
        if (b >= 0) {
          const int64_t slot0 =
              (static_cast<int64_t>(b) << log2_bs) | ((p0 + t0 + GPW * i) & bs_mask);
          const T* row = kbase + slot0 * row_stride + koff;
          kb[i][0] = kv_load<uint4, kNt>(row);
          kb[i][1] = kv_load<uint4, kNt>(row + (MASKD ? (kp1 - lig) * CE : L * CE));
        } else {
          kb[i][0] = make_uint4(0, 0, 0, 0);
          kb[i][1] = make_uint4(0, 0, 0, 0);
        }
      } else {
        int b = -1;
        if (t < n) b = s_blk[((p0 + t) >> log2_bs) - first_blk];
        kok[i] = b >= 0;
        if (kok[i]) {
          const int64_t slot = (static_cast<int64_t>(b) << log2_bs) | ((p0 + t) & bs_mask);
          const T* row = kbase + slot * row_stride;
          kb[i][0] = kv_load<uint4, kNt>(row + lig * CE);
          kb[i][1] = kv_load<uint4, kNt>(row + (MASKD ? kp1 : lig + L) * CE);
        } else {
          kb[i][0] = make_uint4(0, 0, 0, 0);
          kb[i][1] = make_uint4(0, 0, 0, 0);
        }
      }
    }
  };
  // V rows.  Fast path (blocks of >= 16 tokens):
  // rows come in runs of 16 consecutive tokens inside one block, so the
  // block lookup and the 64-bit row address are formed once per run in
  // scalar registers and each further row is one scalar pointer increment.
  // Rows past the end of the partition are zeroed (p = 0 must not meet
  // uninitialised cache contents).
  constexpr int kRun = 16;
  const bool v_runs = log2_bs >= 4;
  // Element offset of the lane's V slice (formed at each use: a value kept
  // across the loop costs registers).
  auto v_slice = [&]() -> int {
    if constexpr (MASKD) {
      return lane * PE < DM ? lane * PE : 0;
    } else {
      return lane * PE;
    }
  };
  auto issue_v = [&](int tile, int blk_lane, bool full) {
    const int t0 = tile * kTile;
    if (v_runs) {
#pragma unroll
      for (int run = 0; run < kTile / kRun; ++run) {
        const int b = __builtin_amdgcn_readlane(blk_lane, run * kRun);
        if (b >= 0) {
          const int64_t slot0 =
              (static_cast<int64_t>(b) << log2_bs) | ((p0 + t0 + run * kRun) & bs_mask);
          const T* rowp = vbase + slot0 * row_stride + v_slice();
          if (full) {
#pragma unroll
            for (int r = 0; r < kRun; ++r) {
              vb[run * kRun + r] = kv_load<VR, kNt>(rowp);
              rowp += row_stride;
            }
          } else {
#pragma unroll
            for (int r = 0; r < kRun; ++r) {
              const int u = run * kRun + r;
              vb[u] = t0 + u < n ? kv_load<VR, kNt>(rowp) : VR{};
              rowp += row_stride;
            }
          }
        } else {
#pragma unroll
          for (int r = 0; r < kRun; ++r) vb[run * kRun + r] = VR{};
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < kTile; ++u) {
        const int b = __builtin_amdgcn_readlane(blk_lane, u);
        if (b >= 0) {
          const int64_t slot = (static_cast<int64_t>(b) << log2_bs) | ((p0 + t0 + u) & bs_mask);
          vb[u] = kv_load<VR, kNt>(vbase + slot * row_stride + v_slice());
        } else {
          vb[u] = VR{};
        }
      }
    }
  };

  // Scores of the loaded K tile, online-softmax update, p -> LDS.
  // Scores stay unscaled (the max commutes with the positive scale); the
  // scale is applied inside the exponent: p = exp2(s * scale - max * scale).
  //
  // RS layout: position p of lane lig dots the query head p ^ lig, so after
  // the 8 partial dots every lane holds one partial of each head.  Halving
  // steps over the row group each add the partner lane's partial of the heads
  // the lane keeps: partners lig ^ 7 (row half-mirror), ^ 2, ^ 1.  The partner
  // holds head h at position h ^ (lig ^ c), so for a kept position p it is
  // p ^ c, in the discarded half.  After the steps (7 adds instead of 3 per
  // head) position 0 of lane lig holds the score of head lig.  The tile maxima
  // are then one reduction over the row groups, and the lane computes, sums
  // and stages its own head's exponentials with no selection among heads.
  auto qk_softmax_rs = [&](bool full) {
    float s[TPG];
    {
      float x[TPG][L];
      const uint4* sq = s_q + 2 * lig;
#pragma unroll
      for (int p = 0; p < L; ++p) {
        const uint4 qg[2] = {sq[2 * L * p], sq[2 * L * p + 1]};
#pragma unroll
        for (int i = 0; i < TPG; ++i) x[i][p] = slice_dot<T>(qg, kb[i]);
      }
#pragma unroll
      for (int i = 0; i < TPG; ++i) {
#pragma unroll
        for (int q = 0; q < 4; ++q) x[i][q] += dpp<kDppRowHalfMirror>(x[i][q ^ 7]);
#pragma unroll
        for (int q = 0; q < 2; ++q) x[i][q] += dpp<kDppQuadXor2>(x[i][q ^ 2]);
        x[i][0] += dpp<kDppQuadXor1>(x[i][1]);
        s[i] = (full || kok[i]) ? x[i][0] : -INFINITY;
      }
    }
    // Head lig's tile maximum, in every row group; head g's is read from lane
    // g (row group 0).
    float tm = s[0];
#pragma unroll
    for (int i = 1; i < TPG; ++i) tm = fmaxf(tm, s[i]);
    tm = across_groups_max<L>(tm);
    bool moved = false;
    float m_new[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m_new[g] = fmaxf(m[g], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tm), g)));
      moved |= m_new[g] != m[g];
    }
    const float ml_new = fmaxf(ml, tm);  // m_new of the lane's head (those below G)
    if (moved) {  // wave-uniform
      float alpha[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        alpha[g] = fast_exp2((m[g] - m_new[g]) * scale);
        m[g] = m_new[g];
      }
      lsum[0] *= fast_exp2((ml - ml_new) * scale);
#pragma unroll
      for (int j = 0; j < G; ++j)
#pragma unroll
        for (int e = 0; e < PE; ++e) acc[j][e] *= alpha[j];
    }
    uint32_t* sp = s_p[wave];
    ml = ml_new;
    const float mc = -ml * scale;
    if (lig < G) {
#pragma unroll
      for (int i = 0; i < TPG; ++i) {
        const float pa = fast_exp2(fmaf(s[i], scale, mc));
        lsum[0] += pa;
        sp[(gi + GPW * i) * G + lig] = __float_as_uint(pa);
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  auto qk_softmax = [&](bool full) {
    float s[TPG][G];
    float tmax[G];
#pragma unroll
    for (int j = 0; j < G; ++j) tmax[j] = -INFINITY;
#pragma unroll
    for (int j = 0; j < G; ++j) {
      const uint4 qg[2] = {s_q[j * (D / CE) + lig], s_q[j * (D / CE) + lig + L]};
#pragma unroll
      for (int i = 0; i < TPG; ++i) {
        float v = group_sum<L>(slice_dot<T>(qg, kb[i]));
        if (!full) v = kok[i] ? v : -INFINITY;
        s[i][j] = v;
        tmax[j] = fmaxf(tmax[j], v);
      }
    }
    // Tile maxima over the row groups.
    bool moved = false;
    float m_new[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      m_new[g] = __int_as_float(
          __builtin_amdgcn_readfirstlane(__float_as_int(fmaxf(m[g], across_groups_max<L>(tmax[g])))));
      moved |= m_new[g] != m[g];
    }
    if (moved) {  // wave-uniform
      float alpha[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        alpha[g] = fast_exp2((m[g] - m_new[g]) * scale);
        lsum[g] *= alpha[g];
        m[g] = m_new[g];
      }
#pragma unroll
      for (int j = 0; j < G; ++j)
#pragma unroll
        for (int e = 0; e < PE; ++e) acc[j][e] *= alpha[j];
    }
    float mneg[G];
#pragma unroll
    for (int g = 0; g < G; ++g) mneg[g] = -m[g] * scale;
    uint32_t* sp = s_p[wave];
#pragma unroll
    for (int r = 0; r < CPL; ++r) {
      const int c = lig + L * r;
      if (NC % L != 0 && c >= NC) break;
      float sa = -INFINITY, sb = -INFINITY, mc = 0.f;  // mc: -max * scale of the head
#pragma unroll
      for (int cc = 0; cc < NC; ++cc) {
        const bool mine = c == cc;
        if constexpr (HALF) {
          sa = mine ? s[2 * (cc / G)][cc % G] : sa;
          sb = mine ? s[2 * (cc / G) + 1][cc % G] : sb;
        } else {
          sa = mine ? s[cc / G][cc % G] : sa;
        }
      }
      const int g = c % G;
#pragma unroll
      for (int gg = 0; gg < G; ++gg) mc = g == gg ? mneg[gg] : mc;
      if constexpr (HALF) {
        const float pa = fast_exp2(fmaf(sa, scale, mc));
        const float pb = fast_exp2(fmaf(sb, scale, mc));
#pragma unroll
        for (int gg = 0; gg < G; ++gg) lsum[gg] += g == gg ? pa + pb : 0.f;
        sp[((c / G) * GPW + gi) * G + g] = pack_half2<T>(pa, pb);
      } else {
        const float pa = fast_exp2(fmaf(sa, scale, mc));
#pragma unroll
        for (int gg = 0; gg < G; ++gg) lsum[gg] += g == gg ? pa : 0.f;
        sp[(gi + GPW * (c / G)) * G + g] = __float_as_uint(pa);
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  // Accumulate P x V of the loaded V tile.
  auto pv = [&]() {
    const uint32_t* sp = s_p[wave];
    if constexpr (HALF) {
#pragma unroll
      for (int t = 0; t < kTile; ++t) {
        if (t % (2 * GPW) >= GPW) continue;
        const int pidx = (t / (2 * GPW)) * GPW + (t % GPW);
        uint32_t pw[G];
#pragma unroll
        for (int j = 0; j < G; ++j) pw[j] = sp[pidx * G + j];
#pragma unroll
        for (int w = 0; w < PE / 2; ++w) {
          // Element 2w (lo) and 2w+1 (hi) of tokens t and t + GPW, paired.
          const uint32_t va = v_word(vb[t], w), vbb = v_word(vb[t + GPW], w);
          const uint32_t lo = __builtin_amdgcn_perm(vbb, va, 0x05040100u);
          const uint32_t hi = __builtin_amdgcn_perm(vbb, va, 0x07060302u);
#pragma unroll
          for (int j = 0; j < G; ++j) {
            acc[j][2 * w] = dot2_half<T>(pw[j], lo, acc[j][2 * w]);
            acc[j][2 * w + 1] = dot2_half<T>(pw[j], hi, acc[j][2 * w + 1]);
          }
        }
      }
    } else {
#pragma unroll
      for (int t = 0; t < kTile; ++t) {
        float v[PE];
        if constexpr (PE == 1) {
          v[0] = __uint_as_float(vb[t]);
        } else {
          v[0] = __uint_as_float(vb[t].x);
          v[1] = __uint_as_float(vb[t].y);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
          const float p = __uint_as_float(sp[t * G + g]);
#pragma unroll
          for (int e = 0; e < PE; ++e) acc[g][e] = fmaf(p, v[e], acc[g][e]);
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  // Each wave walks its tiles: all K and V loads of a tile are issued at
  // the top of the iteration (several waves per SIMD hide the latency; a
  // pipeline carrying the next tile's loads across the loop did not fit the
  // register budget).
  const int ntiles = (n + kTile - 1) / kTile;
  for (int tile = wave; tile < ntiles; tile += kDecodeWaves) {
    if (tile == ntiles - 1) {
      // The new token's parked pieces, stored by the wave that attends the
      // last tile just before its loads.  (The flag and the pieces are read
      // here, with the index made opaque, so that nothing of them is held
      // in registers across the loop.)
      int l = lane, flag = kBlkInts - 1;
      asm volatile("" : "+v"(l), "+v"(flag));
      if (s_blk[flag] != 0) {
        if (l < 2 * kAppendPieces) {
          T* const dst = park_dst[l];
          if (dst != nullptr) st16(dst, park_piece[l]);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      }
    }
    const int blk_lane = tile_blocks(tile);
    // Tile fully inside the partition with every block valid: no masking.
    const bool full = (tile + 1) * kTile <= n && __ballot(lane < kTile && blk_lane < 0) == 0;
    issue_k(tile, blk_lane);
    issue_v(tile, blk_lane, full);
    if constexpr (RS) {
      qk_softmax_rs(full);
    } else {
      qk_softmax(full);
    }
    pv();
  }

  // ---- combine the waves -------------------------------------------------
  // Each (token, head) exponential was summed by exactly one lane.
  float ltot[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float l = RS ? (lig == g ? lsum[0] : 0.f) : lsum[g];
#pragma unroll
    for (int o = kWave / 2; o >= 1; o >>= 1) l += __shfl_xor(l, o, kWave);
    ltot[g] = l;
  }
#pragma unroll
  for (int j = 0; j < G; ++j)
#pragma unroll
    for (int e = 0; e < PE; ++e) s_acc[wave][j * D + lane * PE + e] = acc[j][e];
  if (lane < G) {
#pragma unroll
    for (int g = 0; g < G; ++g)
      if (lane == g) {
        s_m[wave][g] = m[g] * scale;
        s_l[wave][g] = ltot[g];
      }
  }
  __syncthreads();

  // This workgroup's G query heads are h0 .. h0 + G-1.
  const int hq = hkv * a.group;
  const int nparts = (ctx + a.partition - 1) / a.partition;
  float* pacc = a.part_acc + (item * hq + h0) * DM;
  T* out = reinterpret_cast<T*>(a.output) + (qtok * hq + h0) * DM;
  for (int i = tid; i < G * DM; i += kDecodeThreads) {
    const int g = i / DM;
    const int si = MASKD ? g * D + (i - g * DM) : i;  // its s_acc element
    float mx = s_m[0][g];
#pragma unroll
    for (int w = 1; w < kDecodeWaves; ++w) mx = fmaxf(mx, s_m[w][g]);
    float o = 0.f, l = 0.f;
#pragma unroll
    for (int w = 0; w < kDecodeWaves; ++w) {
      const float f = fast_exp2(s_m[w][g] - mx);
      o = fmaf(s_acc[w][si], f, o);
      l = fmaf(s_l[w][g], f, l);
    }
    if (nparts <= 1) {
      store_scalar<T>(out + i, l > 0.f ? o / l : 0.f);
    } else {
      store_device(pacc + i, o);
      if (i % DM == 0) {
        float* pml = a.part_ml + (item * hq + h0 + g) * 2;
        store_device(pml, mx);
        store_device(pml + 1, l);
      }
    }
  }

  // ---- in-launch split-K merge ---------------------------------------------
  if (nparts > 1 && n > 0 && a.merge_state != nullptr && seq >= 0 && seq < a.num_seqs) {
    // (fp32 heads of 80 and 96 merge one element at a time, which keeps
    // their occupancy.)
    constexpr int KO = (G * DM + kDecodeThreads - 1) / kDecodeThreads;
    constexpr int KM = MASKD && sizeof(T) == 4 ? 1 : kMergeOutputs;
    constexpr int KC = KO >= 4 && KM >= 4 ? 4 : KO >= 2 && KM >= 2 ? 2 : 1;
    merge_in_launch<T, DM, KC>(a, G, part, item, ctx, nparts,
                                   (static_cast<int64_t>(seq) * hkv + kvh) * a.sub_groups + sg, h0, hq,
                                   reinterpret_cast<T*>(a.output) + qtok * hq * DM);
  }
}

// Combines the split-K partials (max, sum, unnormalised acc) of one
// multi-partition sequence for the G heads of one KV head.  One workgroup
// per (entry of the merge list, KV head, 256 of the G*D outputs); an entry,
// written by pa_pack, is (first full-partition item, number of full
// partitions, sequence, item of the partial last partition or -1): the full
// partitions of a sequence are contiguous items, its partial one sits among
// the short work at the end.  Every thread owns one output (merge_partials):
// no LDS and no barrier, so the only dependent global round trips are the
// entry and then the partials.  (With several outputs per thread their
// round trips queued one behind the other: eight heads of 128 at partition
// 2048 took 19 us.)
template <typename T>
__global__ __launch_bounds__(kDecodeThreads) void decode_merge_kernel(DecodeArgs a, int G, int D) {
  const int hkv = a.num_kv_heads;
  const int64_t m = blockIdx.x / hkv;
  const int kvh = static_cast<int>(blockIdx.x - m * hkv);
  const int4 e = reinterpret_cast<const int4*>(a.merge_items)[m];
  const int64_t first = e.x;
  const int nfull = static_cast<int>(min(static_cast<int64_t>(e.y), a.num_items - first));
  const bool has_rem = e.w >= 0 && e.w < a.num_items;
  const int nparts = nfull + (has_rem ? 1 : 0);
  if (nfull < 0 || nparts <= 1) return;
  const int hq = hkv * G;
  T* out = reinterpret_cast<T*>(a.output) + (a.cu_seqlens[e.z] * hq + kvh * G) * D;
  const int i = static_cast<int>(blockIdx.y) * kDecodeThreads + static_cast<int>(threadIdx.x);
  if (i >= G * D) return;
  const int h = kvh * G + i / D;
  merge_partials<T, 1>(a.part_ml + 2 * h, a.part_acc + static_cast<int64_t>(kvh) * G * D + i, 0,
                       2 * static_cast<int64_t>(hq), static_cast<int64_t>(hq) * D, first, nfull, has_rem ? e.w : -1,
                       nparts, out + i);
}

// ---- host-side dispatch ------------------------------------------------

// The merge phase, unless the partition launch merged in place (merge
// records given): all a.group query heads of a KV head merge in one
// workgroup row; out_d: elements per query head in memory.
template <typename T>
static hipError_t launch_merge_t(const DecodeArgs& a, int out_d, int phases, hipStream_t stream) {
  const int64_t grid = a.num_merge * a.num_kv_heads;
  if (!(phases & PA_DECODE_PHASE_MERGE) || grid <= 0) return hipSuccess;
  if ((phases & PA_DECODE_PHASE_PARTITIONS) && a.merge_state != nullptr) return hipSuccess;
  const int chunks = (a.group * out_d + kDecodeThreads - 1) / kDecodeThreads;
  hipLaunchKernelGGL((decode_merge_kernel<T>), dim3(static_cast<uint32_t>(grid), static_cast<uint32_t>(chunks)),
                     dim3(kDecodeThreads), 0, stream, a, a.group, out_d);
  return hipGetLastError();
}

static hipError_t launch_merge(const DecodeArgs& a, int dtype, int out_d, int phases, hipStream_t stream) {
  return dtype == PA_DTYPE_BF16  ? launch_merge_t<bf16_t>(a, out_d, phases, stream)
         : dtype == PA_DTYPE_F16 ? launch_merge_t<f16_t>(a, out_d, phases, stream)
                                 : launch_merge_t<float>(a, out_d, phases, stream);
}

// Launches both phases of one kernel instance.  D, G: the kernel's head dim
// and group.
struct LaunchOp {
  const DecodeArgs& a;
  int64_t num_items;
  int phases;
  hipStream_t stream;
  template <typename T, int D, int G, bool SHARED, int DM>
  hipError_t run() const {
    const int64_t grid = num_items * a.num_kv_heads * a.sub_groups;
    if (phases & PA_DECODE_PHASE_PARTITIONS) {
      hipLaunchKernelGGL((decode_partition_kernel<T, D, G, SHARED, DM>), dim3(static_cast<uint32_t>(grid)),
                         dim3(kDecodeThreads), 0, stream, a);
      const hipError_t err = hipGetLastError();
      if (err != hipSuccess) return err;
    }
    return launch_merge_t<T>(a, DM, phases, stream);
  }
};

// Resident partition workgroups per CU of one kernel instance.
struct OccupancyOp {
  int* per_cu;
  template <typename T, int D, int G, bool SHARED, int DM>
  hipError_t run() const {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, decode_partition_kernel<T, D, G, SHARED, DM>,
                                                        kDecodeThreads, 0);
  }
};

template <typename T, int D, bool SHARED, int DM, typename Op>
static hipError_t visit_group(int G, const Op& op) {
  switch (G) {
    case 1: return op.template run<T, D, 1, SHARED, DM>();
    case 2: return op.template run<T, D, 2, SHARED, DM>();
    case 3: return op.template run<T, D, 3, SHARED, DM>();
    case 4: return op.template run<T, D, 4, SHARED, DM>();
    case 5: return op.template run<T, D, 5, SHARED, DM>();
    case 6: return op.template run<T, D, 6, SHARED, DM>();
    case 7: return op.template run<T, D, 7, SHARED, DM>();
    case 8: return op.template run<T, D, 8, SHARED, DM>();
    default: return hipErrorNotSupported;
  }
}

template <bool SHARED, typename Op>
static hipError_t visit_shape(int dtype, int head_dim, int g, const Op& op) {
  if (dtype == PA_DTYPE_BF16) {
    if (head_dim == 256) return visit_group<bf16_t, 256, SHARED, 256>(g, op);
  } else if (dtype == PA_DTYPE_F16) {
    if (head_dim == 256) return visit_group<f16_t, 256, SHARED, 256>(g, op);
  } else if (dtype == PA_DTYPE_F32) {
    if (head_dim == 128) return visit_group<float, 128, SHARED, 128>(g, op);
    if (head_dim == 64) return visit_group<float, 64, SHARED, 64>(g, op);
    if (head_dim == 96) return visit_group<float, 128, SHARED, 96>(g, op);
    if (head_dim == 80) return visit_group<float, 128, SHARED, 80>(g, op);
  }
  return hipErrorNotSupported;
}

// The kernel instance of a shape: a group above the largest kernel group
// runs as decode_sub_groups(group) workgroups per KV head, on the SHARED
// instances (cached K/V loads: the siblings' re-reads hit L2).
template <typename Op>
static hipError_t visit_decode(int dtype, int head_dim, int group, const Op& op) {
  if (group < 1) return hipErrorNotSupported;
  const int nsub = decode_sub_groups(group);
  return nsub > 1 ? visit_shape<true>(dtype, head_dim, group / nsub, op)
                  : visit_shape<false>(dtype, head_dim, group, op);
}

int decode_unit_heads(int dtype, int head_dim, int num_kv_heads, int group) {
  return decode_uses_mfma(dtype, head_dim) && head_dim % 64 == 0 && num_kv_heads % 2 == 0 && group >= 1 && group <= 4
             ? 2
             : 1;
}

int decode_sub_groups(int group) {
  // The fewest equal sub-groups of at most kMaxDecodeGroup query heads.
  int n = (group + kMaxDecodeGroup - 1) / kMaxDecodeGroup;
  while (n < group && group % n != 0) ++n;
  return n > 0 ? n : 1;
}

int decode_workgroups_per_head(int dtype, int head_dim, int group) {
  if (!decode_uses_mfma(dtype, head_dim)) return decode_sub_groups(group);
  int n = (group + kMfmaHeads - 1) / kMfmaHeads;
  while (n < group && group % n != 0) ++n;
  return n > 0 ? n : 1;
}

bool decode_fast_path_supported(int dtype, int head_dim, int group, int block_size,
                                int partition) {
  if (dtype != PA_DTYPE_F32 && dtype != PA_DTYPE_BF16 && dtype != PA_DTYPE_F16) return false;
  // Rows of up to 512 bytes: heads of 64 and 128, and of 256 in 16-bit types;
  // heads of 80 and 96 on the lane layout of 128.
  const bool wide16 = dtype != PA_DTYPE_F32 && head_dim == 256;
  if (head_dim != 64 && head_dim != 128 && head_dim != 80 && head_dim != 96 && !wide16) return false;
  if (group < 1 || group > kMaxDecodeQueryGroup) return false;
  if (block_size <= 0 || (block_size & (block_size - 1)) != 0) return false;
  if (partition <= 0 || partition > kMaxPartition || partition % 32 != 0) return false;
  return true;
}

hipError_t launch_decode(const DecodeArgs& a, int dtype, int head_dim, int group,
                         int64_t num_items, int phases, hipStream_t stream) {
  if (num_items <= 0) return hipSuccess;
  if (decode_uses_mfma(dtype, head_dim)) {
    if (phases & PA_DECODE_PHASE_PARTITIONS) {
      const int heads = decode_unit_heads(dtype, head_dim, a.num_kv_heads, group);
      const hipError_t err = launch_decode_mfma(a, dtype, head_dim, heads, num_items, stream);
      if (err != hipSuccess) return err;
    }
    return launch_merge(a, dtype, head_dim, phases, stream);
  }
  return visit_decode(dtype, head_dim, group, LaunchOp{a, num_items, phases, stream});
}

hipError_t decode_workgroups_per_cu(int dtype, int head_dim, int num_kv_heads, int group, int* per_cu) {
  *per_cu = 0;
  if (!decode_uses_mfma(dtype, head_dim)) return visit_decode(dtype, head_dim, group, OccupancyOp{per_cu});
  const int wgs = decode_workgroups_per_head(dtype, head_dim, group);
  const hipError_t err = decode_mfma_workgroups_per_cu(
      dtype, head_dim, wgs > 1, decode_unit_heads(dtype, head_dim, num_kv_heads, group), per_cu);
  *per_cu *= decode_sub_groups(group) / wgs;
  return err;
}

}  // namespace pa
