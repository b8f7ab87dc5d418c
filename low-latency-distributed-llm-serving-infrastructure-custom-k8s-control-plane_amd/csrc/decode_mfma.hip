// Paged-attention decode of 16-bit caches on the matrix cores (heads of 64 and
// 128, and of 80 and 96 on the LDS rows of 128): one workgroup per (sequence,
// context partition, KV head or two adjacent ones), up to 16 query heads of a
// KV head in one pass (larger groups run as sub-groups of at most 16).
//
// What bounds it is HBM: every K/V byte is read once for all 16 heads, and a
// 32-token tile costs a wave 24 MFMAs (heads of 128) and about 120 vector
// instructions whatever the group.  The vector kernel (decode.hip) serves at most 8 heads a
// pass (groups above 8 read K/V again through L2) at a dot2 per head, token
// and pair of dims.  Vector kernel -> this one, steps of one layer: 48
// sequences of 512-8192 tokens, 128/8 heads of 128, fp16, 227 -> 148 us (5.4
// TB/s); 64 of 128-8192, 14/2 heads of 64, 39.3 -> 30.3 us; 256 of 32-8192,
// 64/8 heads of 128, 734 -> 723 us (6.3 TB/s), 9/3 of 64, 144 -> 133 us.  A
// workgroup alone reads three times as fast (8 sequences of 2048 tokens, 64/8
// heads of 128 in whole partitions: 75 -> 25 us).
//
// v_mfma_f32_16x16x32: lane l = 16 c + r (c = 0..3) holds row r and the 8
// k-values of its quarter c of the A operand, column r and the same k-values
// of B, and column r, rows 4c .. 4c+3 of the result.  The order of k is free
// as long as both operands agree, which makes the other operands a lane's
// own registers:
//  S^T = K Q^T   A: lane (r, c) holds token r's 16-byte pieces 4j + c, read
//                from LDS, B: the same pieces of query head r (kept in
//                registers).  The result gives the lane tokens 4c .. 4c+3 of
//                head r.
//  O^T = V^T P^T B: head r's probabilities of tokens 4c .. 4c+3 of both
//                16-token halves of the tile -- the lane's own scores,
//                exponentiated and packed, no exchange.  A: the same 8 tokens
//                of V, which the lane loads as whole pieces (16 lanes read a
//                row); dim PE * r + b of block b is then element b of the
//                lane's pieces, so the transpose is v_perm_b32 on its own
//                registers.  The result gives the lane PE * 4 consecutive
//                dims of head r, whose softmax state it also holds.
// A probability goes into the product as two terms of the cache type, itself
// rounded and what the rounding left, so that the result is off by its own
// rounding alone: rounded once, it was exact only where its token set the
// running maximum, and the error grew with longer partitions and fewer waves a
// head.  Off 64 bits in bf16 (2-norm), one term -> two: 16 sequences of
// 256-1024 tokens, 32/8 heads of 128, 2.1e-3 -> 1.7e-3; 48 of 512-8192, 128/8,
// fp16, 2.7e-4 -> 2.1e-4.  The 8 MFMAs and 20 vector instructions more a tile
// hide behind the loads: 16 sequences 117.4 -> 118.1 us for 8 layers, 256 of
// 32-8192 tokens 258.3 -> 258.6, 64 with 32/32 heads 341.7 -> 341.8.
// Heads of 96, 64 sequences of 128-4096 tokens, 32/32: 347 -> 311 us; of 80, 32
// sequences: 177 -> 148 us; 96/8 heads of 96, 32 sequences: 77 -> 52 us.
// K as operand loads straight from HBM (64 bytes of 16 rows an instruction,
// no LDS) took 164 us in the first of those steps; streaming (nontemporal)
// loads are worth 11-13 % where no sibling reads the rows again.
// HEADS 2 (groups of up to 4, an even KV head count): half of the waves take
// each of two adjacent KV heads, so that both halves of a token's 512 (or 256)
// contiguous bytes are read by one workgroup at about the same time.  Against
// the vector kernel that read them as one row: 256 sequences of 32-8192
// tokens, 32/8 heads of 128, 268 -> 258 us (6.6 TB/s), 64 sequences, 32/32
// heads, 343 -> 341; one workgroup per head took 274 and 356.
// A short context is its workgroup's latency: the prologue has one round trip
// after the other (item; row, context and token; block ids, query and new rows;
// K and V), so it divides by multiplication, has one barrier and no load that
// waits for a block id but K and V.  With divisions, a three-barrier reduction
// and the new rows loaded after their block id: 138 sequences of 25-49 tokens,
// 32/8 heads of 128, 10.9 -> 9.4 us, 8/8 10.1 -> 8.6; 131 of 22-88, 32/32 heads
// of 96, 35.5 -> 30.9.  (Three workgroups per CU at heads of 128, where the
// vector kernel had four or five for groups of 1: 96 sequences of 55 tokens,
// 20/20 heads, 960 workgroups, take 14.7 us and took 13.5 there.  At four the
// registers spill 38.)
// Each wave runs its own online softmax over every fourth tile (every second
// one of its head's with HEADS 2), no barrier in the loop.
#include <type_traits>

#include "decode_common.hpp"

namespace pa {

constexpr int kMfmaTile = 32;   // context tokens per wave iteration

typedef float f32x4m __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8m __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8m __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4m __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2m __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ f32x4m mfma16(u32x4m a, u32x4m b, f32x4m c);
template <>
__device__ __forceinline__ f32x4m mfma16<bf16_t>(u32x4m a, u32x4m b, f32x4m c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8m, a), __builtin_bit_cast(bf16x8m, b), c,
                                                 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4m mfma16<f16_t>(u32x4m a, u32x4m b, f32x4m c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8m, a), __builtin_bit_cast(f16x8m, b), c, 0,
                                                0, 0);
}

// A lane's piece of a V row: D / 16 elements.
template <int D>
struct VPiece;
template <>
struct VPiece<64> {
  using type = u32x2m;
};
template <>
struct VPiece<128> {
  using type = u32x4m;
};

// NT: streaming loads, for rows no other workgroup reads.
template <typename V, bool NT>
__device__ __forceinline__ V row_load(const void* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const V*>(p));
  return *reinterpret_cast<const V*>(p);
}

// The K operands of a tile from the wave's LDS rows, at[j] the LDS address of
// piece 4j + c of token r and the second half of the tile HALF bytes further.
// Waits until at most VM vector memory operations are outstanding, the copies
// into those rows among the ones that are done: the compiler orders an LDS
// read after such a copy only where it can tell the two by their alias
// scopes, and then waits for every load in flight.
template <int KJ, int HALF, int VM>
__device__ __forceinline__ void read_k(const uint32_t (&at)[KJ], u32x4m (&k)[2][KJ]) {
  static_assert(KJ >= 2 && KJ <= 4, "heads of 64 to 128");
  if constexpr (KJ == 2)
    asm volatile(
        "s_waitcnt vmcnt(%7)\n\t"
        "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\t"
        "ds_read_b128 %2, %4 offset:%6\n\tds_read_b128 %3, %5 offset:%6\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[1][0]), "=&v"(k[1][1])
        : "v"(at[0]), "v"(at[1]), "n"(HALF), "n"(VM)
        : "memory");
  else if constexpr (KJ == 3)
    asm volatile(
        "s_waitcnt vmcnt(%10)\n\t"
        "ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\tds_read_b128 %2, %8\n\t"
        "ds_read_b128 %3, %6 offset:%9\n\tds_read_b128 %4, %7 offset:%9\n\tds_read_b128 %5, %8 offset:%9\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[1][0]), "=&v"(k[1][1]), "=&v"(k[1][2])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "n"(HALF), "n"(VM)
        : "memory");
  else
    asm volatile(
        "s_waitcnt vmcnt(%13)\n\t"
        "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\tds_read_b128 %3, %11\n\t"
        "ds_read_b128 %4, %8 offset:%12\n\tds_read_b128 %5, %9 offset:%12\n\t"
        "ds_read_b128 %6, %10 offset:%12\n\tds_read_b128 %7, %11 offset:%12\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(k[0][0]), "=&v"(k[0][1]), "=&v"(k[0][2]), "=&v"(k[0][3]), "=&v"(k[1][0]), "=&v"(k[1][1]),
          "=&v"(k[1][2]), "=&v"(k[1][3])
        : "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3]), "n"(HALF), "n"(VM)
        : "memory");
}

// n / d, with rcp = (2^32 - 1) / d from the host: the product's high half is
// the quotient or one less.  (A division by a runtime value is a chain of some
// 30 dependent instructions, and the prologue's stood in front of every load.)
__device__ __forceinline__ uint32_t quotient(uint32_t n, uint32_t d, uint32_t rcp) {
  const uint32_t q = __umulhi(n, rcp);
  return n - q * d >= d ? q + 1 : q;
}

template <typename T, int D, int DM, bool SHARED, int HEADS>
__global__ __launch_bounds__(kDecodeThreads) __attribute__((amdgpu_waves_per_eu(3))) void
decode_mfma_kernel(DecodeArgs a) {
  static_assert(sizeof(T) == 2, "16-bit caches");
  // (Rows of 160 or 192 bytes share 128-byte lines with the next head's.)
  constexpr bool kNt = !SHARED && DM == D;
  constexpr int KJ = (DM + 31) / 32;  // MFMAs of a 16-token half's scores
  constexpr int PE = D / 16;       // V elements of a lane's piece, blocks of the output
  constexpr int kRowBytes = D * 2;   // an LDS row
  constexpr int kMemBytes = DM * 2;  // a cache row
  constexpr int kAccRow = D + 4;   // padded LDS row of one head's accumulators
  using VP = typename VPiece<D>::type;

  __shared__ int s_blk[kMaxPartition + 2];
  __shared__ int s_hole[kDecodeWaves];  // a wave met a missing block
  __shared__ float s_m[kDecodeWaves][kMfmaHeads];
  __shared__ float s_l[kDecodeWaves][kMfmaHeads];
  // Per wave: the K rows of its tile, and after the last tile its
  // accumulators.
  constexpr int kWaveBytes = kMfmaHeads * kAccRow * 4;
  static_assert(kWaveBytes >= kMfmaTile * kRowBytes, "a tile's K rows fit");
  __shared__ __align__(16) char s_wave[kDecodeWaves][kWaveBytes];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int r = lane & 15;  // token of a K load, query head elsewhere
  const int c = lane >> 4;
  constexpr int kHeadWaves = kDecodeWaves / HEADS;  // waves per KV head
  const int hkv = a.num_kv_heads;
  const uint32_t sub_groups = SHARED ? a.sub_groups : 1;
  const int G = SHARED ? a.group / a.sub_groups : a.group;
  // Workgroup -> (item, KV head, sub-group).  Ids are dealt to the XCDs
  // round-robin: the members of a gang get ids that are equal modulo the XCD
  // count and close together, gang after gang going to the next XCD (runs of
  // 8 gangs, the last may be shorter).  Sub-groups that read the same rows
  // form a gang, whose later reads hit that XCD's L2; so do all of an item's
  // heads of 64, whose rows of 128 bytes share HBM bursts (128 sequences, 16/8
  // heads: 208 -> 196 us), but not its heads of 128 (256 sequences, 32/8 heads:
  // 258 us spread over the XCDs, 265 as one gang).
  const uint32_t units = static_cast<uint32_t>(hkv) / HEADS;
  constexpr bool kGangUnits = kMemBytes % 256 != 0;
  uint32_t g_id = blockIdx.x, member = 0;
  if constexpr (kGangUnits || SHARED) {
    const uint32_t gang = (kGangUnits ? units : 1) * sub_groups;
    const uint32_t gangs = static_cast<uint32_t>(a.num_items) * (kGangUnits ? 1 : units);
    const uint32_t run = quotient(blockIdx.x, kXcds * gang, a.run_rcp);
    const uint32_t at_run = blockIdx.x - run * (kXcds * gang);
    const uint32_t width = min(static_cast<uint32_t>(kXcds), gangs - run * kXcds);
    member = width == kXcds ? at_run / kXcds : at_run / width;
    g_id = run * kXcds + (at_run - member * width);
  }
  const int64_t item = kGangUnits ? g_id : quotient(g_id, units, a.unit_rcp);
  const int unit = static_cast<int>(!kGangUnits ? g_id - static_cast<uint32_t>(item) * units
                                    : SHARED    ? member / sub_groups
                                                : member);
  const int sg = !SHARED ? 0 : static_cast<int>(kGangUnits ? member - unit * sub_groups : member);
  const int kvh = unit * HEADS + wave / kHeadWaves;
  const int h0 = kvh * a.group + sg * G;  // first query head of the wave
  const int seq = a.items[2 * item];
  const int part = a.items[2 * item + 1];
  const int64_t trow = a.rows != nullptr ? a.rows[seq] : seq;
  const bool row_ok = trow >= 0 && trow < a.num_table_rows;
  int ctx = a.context_lens[seq];
  int64_t qtok = a.cu_seqlens[seq];
  const int p0 = part * a.partition;
  const int log2_bs = a.log2_block_size;
  const int bs_mask = (1 << log2_bs) - 1;
  // Block ids of the partition -> LDS (invalid ids become -1).  The whole
  // span is read, whatever the context length, so that the reads do not wait
  // for it.
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
  const int64_t row_bytes = static_cast<int64_t>(hkv) * kMemBytes;
  const char* kbase = reinterpret_cast<const char*>(a.key_cache) + kvh * kMemBytes;
  const char* vbase = reinterpret_cast<const char*>(a.value_cache) + kvh * kMemBytes;

  // The query heads (lanes past the group repeat its last one, and their
  // results are never stored; zero past the head dim).
  u32x4m q[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j) {
    const T* qrow = reinterpret_cast<const T*>(a.query) + qtok * a.q_token_stride +
                    static_cast<int64_t>(h0 + min(r, G - 1)) * a.q_head_stride;
    const bool in = DM % 32 == 0 || (4 * j + c) * 8 < DM;
    q[j] = *reinterpret_cast<const u32x4m*>(qrow + (in ? (4 * j + c) * 8 : 0));
    if constexpr (DM % 32 != 0) q[j] = in ? q[j] : u32x4m{0, 0, 0, 0};
  }

  // pa_decode_append: the wave that attends the partition's last tile (which
  // holds position ctx - 1) writes the new token's K and V rows of this KV
  // head, a lane per 16-byte piece, just before that tile's loads; it loads
  // the pieces here, beside the block ids.  No other wave or workgroup of the
  // launch reads the position (sibling sub-groups write the same bytes).
  constexpr int kAppendPieces = kMemBytes / 16;
  const int ntiles = (n + kMfmaTile - 1) / kMfmaTile;
  const bool append = a.new_key != nullptr && n > 0 && p0 + n == ctx;
  const bool append_wave = append && (ntiles - 1) % kHeadWaves == wave % kHeadWaves;
  const bool append_v = lane >= kAppendPieces;
  const int append_at = (append_v ? lane - kAppendPieces : lane) * 8;  // element of the piece
  uint4 append_piece = make_uint4(0, 0, 0, 0);
  if (append_wave && lane < 2 * kAppendPieces)
    append_piece = ld16(reinterpret_cast<const T*>(append_v ? a.new_value : a.new_key) +
                        qtok * (append_v ? a.new_value_token_stride : a.new_key_token_stride) +
                        static_cast<int64_t>(kvh) * (append_v ? a.new_value_head_stride : a.new_key_head_stride) +
                        append_at);

  bool hole = false;  // a block the partition needs is missing
  {
    auto stage = [&](int i, int b) {
      s_blk[i] = b;
      hole |= b < 0 && (i << log2_bs) < n + (p0 & bs_mask);
    };
    if (tid < nblk) stage(tid, valid_block(b0));
    for (int i = tid + kDecodeThreads; i < nblk; i += kDecodeThreads) stage(i, valid_block(table_entry(i)));
  }
  hole = __any(hole);
  if (lane == 0) s_hole[wave] = hole;
  __syncthreads();
  hole = false;
#pragma unroll
  for (int w = 0; w < kDecodeWaves; ++w) hole |= s_hole[w] != 0;

  VP vt[8];  // V of a tile: tokens 4c .. 4c+3 of the first half, then of the second
  // K goes straight into LDS, whole rows per load (in the operand's layout a
  // load would touch 64 bytes of 16 rows, 12 % slower), the 16-byte chunks of
  // token t at position chunk ^ swizzle(t), which spreads the 16 rows of an
  // operand read over the banks.
  constexpr int kChunks = kRowBytes / 16;
  constexpr int kRowsPerLoad = kWave / kChunks;
  constexpr int kLoads = 16 / kRowsPerLoad;  // per 16-token half
  auto swizzle = [](int t) { return kChunks == 16 ? 4 * (t & 3) + ((t >> 2) & 3) : (t >> 1) & 7; };
  char* const s_k = s_wave[wave];
  // Row of the lane within load i of a half, and its bytes from the half's
  // first row.
  auto k_row = [&](int i) { return kRowsPerLoad * i + lane / kChunks; };
  auto k_chunk = [&](int i) { return static_cast<uint32_t>(((lane % kChunks) ^ swizzle(k_row(i))) * 16); };
  // Lanes whose chunk lies past the head dim load nothing; the chunks past it
  // that the scores read (10 and 11 of a head of 80) stay zero.
  if constexpr (DM % 32 != 0) {
    static_assert((KJ * 32 - DM) / 8 * kMfmaTile == kWave, "a lane per chunk");
    const int t = lane % kMfmaTile, chunk = DM / 8 + lane / kMfmaTile;
    st16(s_k + t * kRowBytes + 16 * (chunk ^ swizzle(t & 15)), make_uint4(0, 0, 0, 0));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
  auto load_k_lds = [&](const char* src, int s, int i) {
    if (DM < D && k_chunk(i) >= kMemBytes) return;
    typedef const __attribute__((address_space(1))) void* global_ptr;
    typedef __attribute__((address_space(3))) void* lds_ptr;
    __builtin_amdgcn_global_load_lds((global_ptr)(src), (lds_ptr)(s_k + (s * kLoads + i) * (kWave * 16)), 16, 0,
                                     kNt ? 2 : 0);
  };
  uint32_t koff[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) koff[i] = static_cast<uint32_t>(k_row(i) * static_cast<int>(row_bytes)) + k_chunk(i);
  // (Lanes past the head dim read the row's first piece; their output rows
  // are never stored.)
  const uint32_t vcol = DM == D || r * PE < DM ? r * (PE * 2) : 0;
  const uint32_t voff = static_cast<uint32_t>(4 * c * static_cast<int>(row_bytes)) + vcol;
  auto write_new_rows = [&](int tile) {
    if (append_wave && tile == ntiles - 1) {
      const int b = __builtin_amdgcn_readfirstlane(s_blk[((ctx - 1) >> log2_bs) - first_blk]);
      const int64_t slot = (static_cast<int64_t>(b) << log2_bs) + ((ctx - 1) & bs_mask);
      if (b >= 0 && lane < 2 * kAppendPieces)
        st16(const_cast<char*>(append_v ? vbase : kbase) + slot * row_bytes + append_at * 2, append_piece);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
  };
  // Blocks of 16 tokens or more, all of them there: a 16-token half lies in
  // one block, so it takes one scalar base and per-lane offsets.  Tokens past
  // the partition's end read rows of its last half's block.
  int64_t at[2];  // byte offset of each half's first row
  auto locate = [&](int tile) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int t = min(tile * kMfmaTile + 16 * s, (n - 1) & ~15);
      const int b = __builtin_amdgcn_readfirstlane(s_blk[((p0 + t) >> log2_bs) - first_blk]);
      at[s] = ((static_cast<int64_t>(b) << log2_bs) | ((p0 + t) & bs_mask)) * row_bytes;
    }
  };
  auto load_k = [&]() {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < kLoads; ++i) load_k_lds(kbase + at[s] + koff[i], s, i);
  };
  auto load_v = [&]() {
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 4; ++i) vt[4 * s + i] = row_load<VP, kNt>(vbase + at[s] + i * row_bytes + voff);
  };
  // Any block size, blocks missing: a slot per lane; a token without a block
  // (or past the end) reads slot 0.
  auto slot_of = [&](int t) -> int64_t {
    const int b = t < n ? s_blk[((p0 + t) >> log2_bs) - first_blk] : -1;
    return b < 0 ? 0 : (static_cast<int64_t>(b) << log2_bs) | ((p0 + t) & bs_mask);
  };
  auto load_any = [&](int tile) {
    const int t0 = tile * kMfmaTile;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        load_k_lds(kbase + slot_of(t0 + 16 * s + k_row(i)) * row_bytes + k_chunk(i), s, i);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        vt[4 * s + i] = row_load<VP, kNt>(vbase + slot_of(t0 + 16 * s + 4 * c + i) * row_bytes + vcol);
    }
  };

  const float scale = a.scale_log2e;
  float m = kScoreFloor, l = 0.f;  // head r; l: this lane's tokens only
  f32x4m acc[PE];                  // acc[b][i]: dim PE * (4c + i) + b of head r
#pragma unroll
  for (int b = 0; b < PE; ++b) acc[b] = f32x4m{0.f, 0.f, 0.f, 0.f};

  f32x4m s[2];  // scores of tokens 4c .. 4c+3 of each half, head r
  // LDS addresses of the lane's K operands in the first half.
  uint32_t k_at[KJ];
#pragma unroll
  for (int j = 0; j < KJ; ++j)
    k_at[j] = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)s_k)) +
              r * kRowBytes + 16 * ((4 * j + c) ^ swizzle(r));
  // VM: the operations issued after the tile's K copies (its V loads).
  auto scores = [&](auto vm) {
    u32x4m k[2][KJ];
    read_k<KJ, 16 * kRowBytes, decltype(vm)::value>(k_at, k);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      s[h] = f32x4m{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < KJ; ++j) s[h] = mfma16<T>(k[h][j], q[j], s[h]);
    }
  };
  using AllDone = std::integral_constant<int, 0>;
  using VInFlight = std::integral_constant<int, 8>;
  // Tokens past the end or without a block get no weight, and their V rows
  // (uninitialised or infinite, perhaps) are zeroed.
  auto mask = [&](int tile) {
    const int t = tile * kMfmaTile + (lane & (kMfmaTile - 1));
    const uint32_t live =
        static_cast<uint32_t>(__ballot(t < n && s_blk[((p0 + min(t, n - 1)) >> log2_bs) - first_blk] >= 0));
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool on = (live >> (16 * h + 4 * c + i)) & 1u;
        s[h][i] = on ? s[h][i] : -INFINITY;
        if (!on) vt[4 * h + i] = VP{};
      }
  };
  auto attend = [&]() {
    float tm = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                     fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
    tm = max_halves(max_row_pairs(tm));
    const float m_new = fmaxf(m, tm);
    if (__any(m_new != m)) {
      const float alpha = fast_exp2((m - m_new) * scale);
      l *= alpha;
#pragma unroll
      for (int b = 0; b < PE; ++b) acc[b] *= alpha;
      m = m_new;
    }
    const float mc = -m * scale;
    u32x4m p, rest;  // the probabilities, and what rounding them left
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float pa = fast_exp2(fmaf(s[h][2 * i], scale, mc));
        const float pb = fast_exp2(fmaf(s[h][2 * i + 1], scale, mc));
        l += pa + pb;
        const uint32_t w = pack_half2<T>(pa, pb);
        p[2 * h + i] = w;
        rest[2 * h + i] = pack_half2<T>(pa - half_lo<T>(w), pb - half_hi<T>(w));
      }
#pragma unroll
    for (int w = 0; w < PE / 2; ++w) {
      u32x4m lo, hi;  // elements 2w and 2w + 1 of the 8 tokens
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lo[i] = __builtin_amdgcn_perm(vt[2 * i + 1][w], vt[2 * i][w], 0x05040100u);
        hi[i] = __builtin_amdgcn_perm(vt[2 * i + 1][w], vt[2 * i][w], 0x07060302u);
      }
      acc[2 * w] = mfma16<T>(lo, rest, mfma16<T>(lo, p, acc[2 * w]));
      acc[2 * w + 1] = mfma16<T>(hi, rest, mfma16<T>(hi, p, acc[2 * w + 1]));
    }
  };

  if (wave % kHeadWaves < ntiles) {
    int tile = wave % kHeadWaves;
    if (log2_bs < 4 || hole) {
      for (; tile < ntiles; tile += kHeadWaves) {
        write_new_rows(tile);
        load_any(tile);
        scores(AllDone());
        mask(tile);
        attend();
      }
    } else {
      // The next tile's K copies go out once the scores have used the current
      // K, its V loads once the product has used the current V: V is in flight
      // under the scores, the next K under the product.  (The scheduling
      // barriers keep them there.  With a copy into LDS outstanding the
      // compiler waits for everything in flight at the first use of a loaded
      // register, so the empty statements make it wait for the query before
      // the first copies and for V ahead of the next ones: 1-4 % of a
      // latency-bound step.)
#pragma unroll
      for (int j = 0; j < KJ; ++j) asm volatile("" : "+v"(q[j]));
      write_new_rows(tile);
      locate(tile);
      load_k();
      __builtin_amdgcn_sched_barrier(0);
      load_v();
      __builtin_amdgcn_sched_barrier(0);
      for (; tile + kHeadWaves < ntiles; tile += kHeadWaves) {
        locate(tile + kHeadWaves);
        scores(VInFlight());
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" : "+v"(vt[i]));
        write_new_rows(tile + kHeadWaves);
        __builtin_amdgcn_sched_barrier(0);
        load_k();
        __builtin_amdgcn_sched_barrier(0);
        attend();
        load_v();
        __builtin_amdgcn_sched_barrier(0);
      }
      scores(VInFlight());
      mask(tile);
      attend();
    }
  }

  // ---- combine the waves -------------------------------------------------
  l = sum_halves(sum_row_pairs(l));
  float* acc_row = reinterpret_cast<float*>(s_k) + r * kAccRow + 4 * PE * c;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int b = 0; b < PE; b += 4)
      *reinterpret_cast<float4*>(acc_row + PE * i + b) =
          make_float4(acc[b][i], acc[b + 1][i], acc[b + 2][i], acc[b + 3][i]);
  if (lane < kMfmaHeads) {
    s_m[wave][lane] = m * scale;
    s_l[wave][lane] = l;
  }
  __syncthreads();

  const int hq = hkv * a.group;
  const int nparts = ctx <= a.partition ? 1 : (ctx + a.partition - 1) / a.partition;
  const int hu = unit * HEADS * a.group + sg * G;  // first query head of the workgroup
  float* pacc = a.part_acc + (item * hq + hu) * DM;
  T* out = reinterpret_cast<T*>(a.output) + (qtok * hq + hu) * DM;
  for (int i = tid; i < HEADS * G * DM; i += kDecodeThreads) {
    const int hg = i / DM;
    const bool second = HEADS == 2 && hg >= G;
    const int w0 = second ? kHeadWaves : 0;  // the head's first wave
    const int g = second ? hg - G : hg;
    const int e = g * kAccRow + (i - hg * DM);
    float mx = s_m[w0][g];
#pragma unroll
    for (int w = 1; w < kHeadWaves; ++w) mx = fmaxf(mx, s_m[w0 + w][g]);
    float o = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < kHeadWaves; ++w) {
      const float f = fast_exp2(s_m[w0 + w][g] - mx);
      o = fmaf(reinterpret_cast<const float*>(s_wave[w0 + w])[e], f, o);
      sum = fmaf(s_l[w0 + w][g], f, sum);
    }
    if (nparts <= 1) {
      store_scalar<T>(out + i, sum > 0.f ? o / sum : 0.f);
    } else {
      store_device(pacc + i, o);
      if (i % DM == 0) {
        float* pml = a.part_ml + (item * hq + hu + hg) * 2;
        store_device(pml, mx);
        store_device(pml + 1, sum);
      }
    }
  }
  if (nparts > 1 && n > 0 && a.merge_state != nullptr && seq >= 0 && seq < a.num_seqs)
    merge_in_launch<T, DM, kMergeOutputs>(a, HEADS * G, part, item, ctx, nparts,
                                         (static_cast<int64_t>(seq) * units + unit) * a.sub_groups + sg, hu, hq,
                                         reinterpret_cast<T*>(a.output) + qtok * hq * DM);
}

bool decode_uses_mfma(int dtype, int head_dim) {
  return (dtype == PA_DTYPE_BF16 || dtype == PA_DTYPE_F16) &&
         (head_dim == 64 || head_dim == 80 || head_dim == 96 || head_dim == 128);
}

template <typename T, int D, int DM, typename Op>
static hipError_t visit_mfma_t(bool shared, int heads, const Op& op) {
  if constexpr (DM == D)
    if (heads == 2) return op.template run<T, D, DM, false, 2>();
  return shared ? op.template run<T, D, DM, true, 1>() : op.template run<T, D, DM, false, 1>();
}

// Heads of 80 and 96 run on the LDS rows of 128.
template <typename T, typename Op>
static hipError_t visit_mfma_dim(int head_dim, bool shared, int heads, const Op& op) {
  switch (head_dim) {
    case 64: return visit_mfma_t<T, 64, 64>(shared, heads, op);
    case 80: return visit_mfma_t<T, 128, 80>(shared, heads, op);
    case 96: return visit_mfma_t<T, 128, 96>(shared, heads, op);
    case 128: return visit_mfma_t<T, 128, 128>(shared, heads, op);
    default: return hipErrorNotSupported;
  }
}

template <typename Op>
static hipError_t visit_mfma(int dtype, int head_dim, bool shared, int heads, const Op& op) {
  if (dtype == PA_DTYPE_BF16) return visit_mfma_dim<bf16_t>(head_dim, shared, heads, op);
  if (dtype == PA_DTYPE_F16) return visit_mfma_dim<f16_t>(head_dim, shared, heads, op);
  return hipErrorNotSupported;
}

struct MfmaLaunch {
  const DecodeArgs& a;
  int64_t num_items;
  hipStream_t stream;
  template <typename T, int D, int DM, bool SHARED, int HEADS>
  hipError_t run() const {
    const uint32_t units = a.num_kv_heads / HEADS;
    const int64_t grid = num_items * units * a.sub_groups;
    const uint32_t gang = (DM * 2 % 256 != 0 ? units : 1) * a.sub_groups;
    DecodeArgs b = a;
    b.unit_rcp = 0xffffffffu / units;
    b.run_rcp = 0xffffffffu / (kXcds * gang);
    hipLaunchKernelGGL((decode_mfma_kernel<T, D, DM, SHARED, HEADS>), dim3(static_cast<uint32_t>(grid)),
                       dim3(kDecodeThreads), 0, stream, b);
    return hipGetLastError();
  }
};

struct MfmaOccupancy {
  int* per_cu;
  template <typename T, int D, int DM, bool SHARED, int HEADS>
  hipError_t run() const {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, decode_mfma_kernel<T, D, DM, SHARED, HEADS>,
                                                        kDecodeThreads, 0);
  }
};

hipError_t launch_decode_mfma(const DecodeArgs& a, int dtype, int head_dim, int unit_heads, int64_t num_items,
                              hipStream_t stream) {
  return visit_mfma(dtype, head_dim, a.sub_groups > 1, unit_heads, MfmaLaunch{a, num_items, stream});
}

hipError_t decode_mfma_workgroups_per_cu(int dtype, int head_dim, bool shared, int unit_heads, int* per_cu) {
  return visit_mfma(dtype, head_dim, shared, unit_heads, MfmaOccupancy{per_cu});
}

}  // namespace pa
