// A7/A8: sparse MLA prefill over selected token records, bf16 MFMA with an
// online softmax, from either flat bf16 records (576 x bf16 = 1152 B/token)
// or the fp8 paged cache (656 B/token: 512 e4m3 + 4 fp32 tile scales + 64
// bf16 RoPE, 64 tokens per page).
//
// Semantics: operators/deepseek_v32/attention/reference/torch.py:13-28 - per
// query row r, every selected id in [0, N) (duplicates count per slot) gives
// a record; P = softmax(q[r,h] . rec * scale); out[r,h] = P @ rec[:512],
// rounded to bf16; a row with no valid id is zero.
//
// Mapping (gfx950, wave64). A work-group owns one query row and 64 heads
// and walks the selection in blocks of 32 keys with 4 waves, one per SIMD,
// in two roles:
// * Score waves 0 and 1 compute S^T = K Q^T for all 32 keys and heads
//   32 sw .. 32 sw + 31 with v_mfma_f32_32x32x16_bf16 (Q^T of their 32 heads
//   stays in 144 AGPRs, read by the MFMAs as the B operand), and the online
//   softmax of their heads, writing P^T (bf16) and per-head rescale factors
//   to LDS.
// * Load waves 2 and 3 stage the records: lane (kk, j) (kk = 16 (w - 2) +
//   lane / 4, j = lane % 4) loads a quarter of key kk's record with 16-byte
//   loads, kLookahead blocks ahead, and converts it into bf16 rows of a
//   block buffer in LDS (fp8 records by v_cvt_scalef32_pk_bf16_fp8 with
//   their tile scales; e4m3 x 2^k is exact in bf16), once per key.
// * All four accumulate O^T += V^T P^T (v_mfma_f32_16x16x32_bf16, V^T from
//   ds_read_b64_tr_b16) over all 64 heads: score waves for 96 dims each,
//   load waves for 160 each. Row sums come from the same MFMA pipe: each
//   wave adds P^T of one head tile against a row of ones, so l sums exactly
//   the bf16 P the product used.
// The work is software-pipelined so that every wave has matrix work and
// independent VALU / LDS work in the same step, which its SIMD runs side by
// side (the code issues them interleaved): in step `it` the score waves
// compute S(it) and the softmax of block it - 1 (its scores kept in
// registers) and the PV product of block it - 2; the load waves convert the
// rows of block it + 1 and run the PV product of block it - 2. One barrier
// per step; four block buffers (S reads it, PV reads it - 2, it + 1 is
// written); P and the rescale factors are double buffered by block parity.
// The physical rows of the selection live in a ring of 8 blocks in LDS that
// the load waves keep 6 blocks ahead (the id and page-table loads each
// land two steps before use, ahead of the record loads).
//
// Online softmax in log2 units with lazy rescaling (only when a block raises
// a head's running max by more than 8, so p <= 2^8).
#include <type_traits>

#include "dsa_common.h"
#include "../../include/dsa_gfx950.h"

namespace dsa {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v2u __attribute__((ext_vector_type(2)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
// 16 bytes of `out`, which callers need only align to kOutAlign.
constexpr int kOutAlign = 8;
typedef uint32_t v4u_out __attribute__((ext_vector_type(4), aligned(kOutAlign)));
static_assert(alignof(v4u_out) == kOutAlign && alignof(uint2) <= kOutAlign, "stores of out");

constexpr int kQkDim = 576;
constexpr int kVDim = 512;
constexpr int kHeadsPerGroup = 64;
constexpr int kBlock = 32;            // keys per block
constexpr int kThreads = 256;
constexpr int kMaxSelected = 4096;    // widest selection per query row
constexpr int kPageTokens = 64;
constexpr float kRescaleThreshold = 8.0f;

template <bool kFp8>
struct Format {
  static constexpr int kRecordBytes = kFp8 ? 656 : kQkDim * 2;
  // 16-byte loads per lane per block: the two load waves fetch 16 keys each,
  // four lanes per key (fp8: 8 latent + scales + 2 RoPE; bf16: 16 + 2).
  static constexpr int kLoads = kFp8 ? 11 : 18;
};

// bf16 K/V rows of one block in LDS: key r at kRowBytes r, its 576 dims in
// order. 1168 bytes = 292 dwords = 36 (mod 64): the 16 keys read by a 16-lane
// group of the score operands land on 16 distinct 4-bank groups, and the 8
// even (or odd) keys of a V^T transpose read on disjoint 8-bank windows.
constexpr int kRowBytes = kQkDim * 2 + 16;
constexpr int kBufBytes = kBlock * kRowBytes;
constexpr int kBuffers = 4;
// Physical rows of the selected keys, by block, in a ring of kRing blocks
// filled kRingAhead blocks ahead of the block being scored.
constexpr int kRing = 8;
constexpr int kRingAhead = 6;
// 16-dim tiles of O^T per score wave and per load wave (two of each).
constexpr int kScoreDimTiles = 6;
constexpr int kLoadDimTiles = (kVDim / 16 - 2 * kScoreDimTiles) / 2;

struct __align__(16) Lds {
  uint8_t kv[kBuffers][kBufBytes];
  // P^T in PV B-operand order, by block parity: [parity][head tile][lane]
  // 16 bytes: lane (c, g) of tile t holds head 16t + c, k-index j = key
  // 2(j & 3) + 8(g & 1) + (g >> 1) + 16(j >> 2), bf16.
  uint8_t p[2][4][64][16];
  float alpha[2][kHeadsPerGroup];  // per-head rescale factor of the block, by parity
  float row_sum[kHeadsPerGroup];
  int32_t wave_last[2];  // last position in range seen by each load wave
  int32_t ring[kRing][kBlock];  // block b at slot b % kRing: record row per key, -1 = padding
};

// Key order inside a block. Row m = 8a + 4h + i of the 32x32 score tile holds
// key 2i + 8(a & 1) + h + 16(a >> 1); k-index j of the PV operands of lane
// row-group g is key 2(j & 3) + 8(g & 1) + (g >> 1) + 16(j >> 2). With these,
// the four results a score lane holds in registers 4a'..4a'+3 are exactly
// the four consecutive k-indices 4(a' >> 1) .. +3 of one PV operand slot.
__device__ __forceinline__ int score_key(int m) {
  return 2 * (m & 3) + 8 * ((m >> 3) & 1) + ((m >> 2) & 1) + 16 * (m >> 4);
}

// Source of padding slots and invalid ids: a zero record (zero scales), so
// that their V^T operands are zeros rather than whatever the cache holds.
__device__ __align__(16) uint8_t zero_record[kQkDim * 2];

__device__ __forceinline__ v8bf as_v8bf(v4u v) { return __builtin_bit_cast(v8bf, v); }

// Two floats -> packed bf16 pair, round-to-nearest-even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2f){lo, hi}, v2bf));
}

template <bool kHigh>
__device__ __forceinline__ uint32_t dequant_pair(uint32_t word, float scale) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(word, scale, kHigh));
}

typedef float v16f __attribute__((ext_vector_type(16)));

typedef v4s __attribute__((address_space(3))) * lds_v4s;

template <typename T>
__device__ __forceinline__ T lds_load(uint32_t addr) {
  return *(T __attribute__((address_space(3)))*)(uintptr_t)addr;
}
template <typename T>
__device__ __forceinline__ void lds_store(uint32_t addr, T v) {
  *(T __attribute__((address_space(3)))*)(uintptr_t)addr = v;
}

// 16 or 4 bytes of global memory at an address kept as an integer (a pointer
// read back from LDS would be a generic one, whose loads count as LDS traffic
// too and would be waited for at every barrier).
template <typename T>
__device__ __forceinline__ T global_read(uint64_t addr) {
  return *(const T __attribute__((address_space(1)))*)addr;
}

// LDS barrier: finish this wave's LDS traffic, then s_barrier. The memory
// clobber keeps the compiler from moving memory accesses across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <bool kFp8>
__global__ __launch_bounds__(kThreads, 1) void sparse_mla_fwd(
    const uint16_t* __restrict__ q, const uint8_t* __restrict__ kv,
    const int32_t* __restrict__ page_table, int64_t n_tokens, int64_t pages,
    const int32_t* __restrict__ indices, int64_t rows, int64_t heads, int64_t topk,
    float scale_log2, uint16_t* __restrict__ out) {
  using F = Format<kFp8>;
  __shared__ Lds lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4;
  const int c = lane & 15;
  // Work-groups go to the XCDs round-robin by linear id: the head groups of a
  // row, which gather the same records, are 8 ids apart, on one XCD and about
  // the same time. Later rows first: a causal prompt's later rows see more
  // tokens, and the long work-groups should not be the last to start.
  const uint32_t groups = (uint32_t)(heads / kHeadsPerGroup);
  const uint32_t tile = blockIdx.x >> 3;
  const int64_t row = rows - 1 - ((int64_t)(tile / groups) * 8 + (blockIdx.x & 7));
  if (row < 0) return;
  const int64_t head0 = (int64_t)(tile % groups) * kHeadsPerGroup;
  const int32_t* ids = indices + row * topk;
  const float neg_inf = -__builtin_inff();
  // Blocks of 32 selected positions, rounded up to an even count (the loop
  // takes two per trip; a padding block has no valid key and adds nothing).
  // A row that ends in padding (a selection longer than what the row sees)
  // stops at its last id in range: the blocks past it would add nothing
  // (a prompt's first 2,048 rows: 1,261 -> 770 us). Only such rows look for
  // it; looking in every row cost a full one 4 us.
  int n_blocks = (int)((topk + 2 * kBlock - 1) / (2 * kBlock)) * 2;
  const int32_t last_id = ids[topk - 1];
  const bool trim = last_id < 0 || last_id >= n_tokens;

  // Physical record row of a selected id and its page (-1 for padding, an id
  // outside [0, n_tokens) or a page outside the cache).
  auto phys_from = [&](int32_t id, int32_t page) -> int32_t {
    if (id < 0 || id >= n_tokens) return -1;
    if (!kFp8) return id;
    return page >= 0 && page < pages ? (int32_t)((int64_t)page * kPageTokens + id % kPageTokens) : -1;
  };

  // Roles: waves 0 and 1 score (32 heads each, all 32 keys of a block, with
  // 32x32x16 MFMAs) and run the softmax; waves 2 and 3 stage the records
  // (HBM -> registers -> bf16 rows in LDS). All four accumulate O^T for their
  // share of the 512 dims over all 64 heads.
  const bool scorer = wave < 2;
  const int sw = wave & 1;           // score wave: heads 32 sw .. + 31
  const int n = lane & 31;           // score lane: head 32 sw + n
  const int h = lane >> 5;           // score lane: row half
  // Staged record bytes of the load waves (fp8: two sets of kLoads at 0 and
  // kLoads, bf16: one set).
  constexpr int kPool = (kFp8 ? 2 : 1) * F::kLoads;
  v4u pool[kPool];
  // Q^T operands of the score waves (k-step ks: dims 16 ks + 8h), 144
  // registers held in AGPRs: loaded straight into them, and read from
  // there as the B operand of the S MFMAs, so that the score waves' VGPRs
  // hold O^T, S, the softmax state and the operand read-ahead without
  // spilling (in VGPRs, about ten of the 36 operands were reloaded from AGPR
  // spill slots every step).
  constexpr int kQOps = kQkDim / 16;
  v4u q_ops[kQOps];
  float m_run = neg_inf;  // score lane: running max of its head (scaled)
  // Row sums of heads 16 wave + c (P^T against ones; every row alike).
  v4f l_acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  // Load role: key kk of each block, quarter j of its record.
  const int kk = 16 * (wave & 1) + (lane >> 2);
  const int j = lane & 3;
  const uint32_t ring_base = (uint32_t)(uintptr_t)&lds.ring[0][0];
  const uint32_t kv_base = (uint32_t)(uintptr_t)&lds.kv[0][0];
  const uint32_t p_base = (uint32_t)(uintptr_t)&lds.p[0][0][0][0];
  auto buf_of = [&](int bl) -> uint32_t { return kv_base + (uint32_t)(bl & (kBuffers - 1)) * kBufBytes; };

  // Per-block base addresses are formed once and hidden from the optimizer
  // (an identity DPP move it cannot see through): otherwise it hoists (lane
  // offset + constant) out of the loop and pays an add per LDS access instead
  // of using the instruction's offset field. Unlike an empty asm statement it
  // does not cut the scheduling region.
  auto lane_base = [](uint32_t buf, uint32_t lane_off) -> uint32_t {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(buf + lane_off), 0xE4, 0xF, 0xF, false);
  };
  auto row_of = [&](int bl) -> int32_t {
    return bl < n_blocks ? lds_load<int32_t>(ring_base + 4 * (uint32_t)((bl % kRing) * kBlock + kk)) : -1;
  };
  // Block b's record bytes of this lane -> registers. Blocks past the end
  // (and invalid ids) read the zero record, so the load count per block is
  // fixed. fp8 latent loads i cover record bytes 64i + 16j (64 contiguous
  // bytes per key and instruction); bf16 loads 2i + u cover 128i + 32j + 16u.
  auto fetch = [&](auto set, int32_t phys) __attribute__((always_inline)) {
    v4u* st = pool + decltype(set)::value;
    const uint8_t* rec = phys >= 0 ? kv + (int64_t)phys * F::kRecordBytes : zero_record;
    if (kFp8) {
#pragma unroll
      for (int i = 0; i < 8; ++i) st[i] = *reinterpret_cast<const v4u*>(rec + 64 * i + 16 * j);
      st[8] = *reinterpret_cast<const v4u*>(rec + kVDim);
      st[9] = *reinterpret_cast<const v4u*>(rec + kVDim + 16 + 32 * j);
      st[10] = *reinterpret_cast<const v4u*>(rec + kVDim + 32 + 32 * j);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        st[i] = *reinterpret_cast<const v4u*>(rec + 128 * (i >> 1) + 32 * j + 16 * (i & 1));
      st[16] = *reinterpret_cast<const v4u*>(rec + 2 * kVDim + 32 * j);
      st[17] = *reinterpret_cast<const v4u*>(rec + 2 * kVDim + 16 + 32 * j);
    }
  };
  // Landed record bytes -> bf16 rows of a block buffer (fp8: e4m3 x tile
  // scale, exact in bf16).
  auto unpack = [&](auto set, uint32_t buf) __attribute__((always_inline)) {
    const v4u* st = pool + decltype(set)::value;
    const uint32_t rec = lane_base(buf, (uint32_t)kk * kRowBytes + 32 * j);
    if (kFp8) {
      const v4f sc = __builtin_bit_cast(v4f, st[8]);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float s_i = sc[i >> 1];
        const v4u w = st[i];
        const v4u lo{dequant_pair<false>(w.x, s_i), dequant_pair<true>(w.x, s_i),
                     dequant_pair<false>(w.y, s_i), dequant_pair<true>(w.y, s_i)};
        const v4u hi{dequant_pair<false>(w.z, s_i), dequant_pair<true>(w.z, s_i),
                     dequant_pair<false>(w.w, s_i), dequant_pair<true>(w.w, s_i)};
        lds_store<v4u>(rec + 128 * i, lo);
        lds_store<v4u>(rec + 128 * i + 16, hi);
      }
      lds_store<v4u>(rec + 2 * kVDim, st[9]);
      lds_store<v4u>(rec + 2 * kVDim + 16, st[10]);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) lds_store<v4u>(rec + 128 * (i >> 1) + 16 * (i & 1), st[i]);
      lds_store<v4u>(rec + 2 * kVDim, st[16]);
      lds_store<v4u>(rec + 2 * kVDim + 16, st[17]);
    }
  };

  // Score A operand (K): lane l reads key score_key(l % 32), dims 16 ks + 8h.
  const uint32_t k_lane = (uint32_t)score_key(n) * kRowBytes + 16 * h;
  // O^T dims of the wave: score waves take fewer (they also run S and the
  // softmax), so that both roles spend about the same time per block.
  const int dim0 = scorer ? 16 * kScoreDimTiles * sw : 16 * (2 * kScoreDimTiles + kLoadDimTiles * (wave & 1));
  // V^T rows (ds_read_b64_tr_b16): lane 4 jj + qq of row group g addresses
  // key 2 jj + 8 (g & 1) + (g >> 1) (and + 16) at dims dim0 + 16m + 4qq.
  const int jj = c >> 2;
  const int qq = c & 3;
  const int vkey = 2 * jj + 8 * (g & 1) + (g >> 1);
  const uint32_t v_lane = (uint32_t)vkey * kRowBytes + 2 * dim0 + 8 * qq;
  constexpr uint32_t kHalf = 16 * kRowBytes;

  // Record loads run kLookahead blocks ahead of the block being scored: two
  // register sets for fp8 (blocks it + 2 and it + 3 in flight), one for the
  // bf16 record, whose two sets would not fit beside O^T.
  constexpr int kLookahead = kFp8 ? 3 : 2;
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, kFp8 ? F::kLoads : 0>;

  // The id and page loads of a load lane's key kk are branch-free (clamped
  // addresses, out-of-range results replaced).
  auto id_load = [&](int bl) -> int32_t {
    const int i = bl * kBlock + kk;
    const bool in = bl < n_blocks && i < topk;
    const int32_t id = ids[in ? i : 0];
    return in ? id : -1;
  };
  auto page_load = [&](int32_t id) -> int32_t {
    if (!kFp8) return 0;
    const bool in = id >= 0 && id < n_tokens;
    const int32_t page = page_table[in ? id / kPageTokens : 0];
    return in ? page : -1;
  };
  // Ring state per step parity: the id and page of the block whose row the
  // step stores, and the id loaded for the block two steps after it.
  int32_t ring_id[2] = {-1, -1}, ring_page[2] = {-1, -1}, id_keep[2] = {-1, -1};
  int32_t phys_next = -1;
  // Prologue, up to one barrier: each load lane takes its key's rows of blocks
  // 0 .. kRingAhead - 1 through its own id, page and record loads and puts
  // them into the ring (which the load waves then keep kRingAhead blocks
  // ahead; the four lanes of a key store the same value), and stages block 0;
  // the score waves load their Q beside that. With the ring filled by all
  // waves and Q loaded behind its barrier, 16.7k of a 2,048-key tile's 185k
  // cycles passed before the first step, then 11.7k (1,024 rows of 128 heads,
  // eight rounds: 648 -> 636 us, with 64 keys 109.7 -> 106.0).
  if (!scorer) {
    int32_t rows0[kRingAhead], pages0[kRingAhead];
#pragma unroll
    for (int b = 0; b < kRingAhead; ++b) rows0[b] = id_load(b);
    id_keep[0] = id_load(kRingAhead);
    id_keep[1] = id_load(kRingAhead + 1);
    ring_id[0] = id_load(kRingAhead + 2);
    ring_id[1] = id_load(kRingAhead + 3);
#pragma unroll
    for (int b = 0; b < kRingAhead; ++b) pages0[b] = page_load(rows0[b]);
    ring_page[0] = page_load(id_keep[0]);
    ring_page[1] = page_load(id_keep[1]);
    rows0[0] = phys_from(rows0[0], pages0[0]);
    fetch(Set0{}, rows0[0]);
    rows0[1] = phys_from(rows0[1], pages0[1]);
    if (kFp8) fetch(Set1{}, rows0[1]);
#pragma unroll
    for (int b = 2; b < kRingAhead; ++b) rows0[b] = phys_from(rows0[b], pages0[b]);
#pragma unroll
    for (int b = 0; b < kRingAhead; ++b) lds.ring[b][kk] = rows0[b];
    if (trim) {
      int last = -1;
#pragma unroll 4
      for (int i0 = 0; i0 < (int)topk; i0 += kThreads / 2) {
        const int i = i0 + (int)threadIdx.x - kThreads / 2;
        const int32_t id = ids[i < topk ? i : 0];
        const uint64_t in = __builtin_amdgcn_ballot_w64(i < topk && id >= 0 && id < n_tokens);
        if (in) last = i0 + 64 * (wave & 1) + 63 - __builtin_clzll(in);
      }
      if (lane == 0) lds.wave_last[wave & 1] = last;
    }
    unpack(Set0{}, buf_of(0));
    fetch(Set0{}, rows0[kLookahead - 1]);
    phys_next = rows0[kLookahead];
  } else {
    // Q^T of the score wave's heads (72 KiB per work-group), loaded only once
    // the row's last id is there: issued at the start, the Q loads of all
    // work-groups would queue ahead of the id loads that start the pipeline.
    asm volatile("" ::"s"(__builtin_amdgcn_readfirstlane(last_id)) : "memory");
    const uint16_t* qrow = q + ((row * heads + head0 + 32 * sw + n) * kQkDim) + 8 * h;
#pragma unroll
    for (int ks = 0; ks < kQOps; ++ks)
      asm volatile("global_load_dwordx4 %0, %1, off" : "=a"(q_ops[ks]) : "v"(qrow + 16 * ks) : "memory");
    // These loads are outside the compiler's load counting: wait here.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  lds_barrier();
  if (trim) {
    const int last = max(lds.wave_last[0], lds.wave_last[1]);
    n_blocks = __builtin_amdgcn_readfirstlane((max(last, 0) / (2 * kBlock) + 1) * 2);
  }

  // Software pipeline, one barrier per step. Step `it`:
  //   score waves: S(it) = K Q^T of block it, the softmax of block it - 1
  //     (its scores kept in registers from the previous step), the PV
  //     product of block it - 2 for their dims;
  //   load waves: rows of block it + 1 into LDS, records of block
  //     it + kLookahead into registers, the PV product of block it - 2.
  // Each wave thus has matrix work (S, PV) and independent VALU / LDS work
  // (softmax, conversion and row stores) in the same step, which the SIMD
  // runs side by side. Buffers: S reads it, PV reads it - 2, the load waves
  // write it + 1 (last read by PV(it - 3), before the previous barrier): four
  // buffers. P and the rescale factors of block b sit at parity b & 1.
  auto step = [&](int it, auto set, auto parity, auto role, auto parts, auto& o, v16f& s_prev)
                  __attribute__((always_inline)) {
    constexpr bool kScore = decltype(role)::value;
    constexpr int kParts = decltype(parts)::value;
    constexpr bool kS = (kParts & 1) != 0;     // score waves: S(it); load waves: rows of it + 1
    constexpr bool kSoft = (kParts & 2) != 0;  // score waves: softmax(it - 1)
    constexpr bool kPV = (kParts & 4) != 0;    // PV(it - 2)
    constexpr int kM = kScore ? kScoreDimTiles : kLoadDimTiles;

    // ---- the step's first LDS reads, before any wait or branch: block
    // it - 2's rescale factors, block it - 1's padding mask, P^T of the four
    // head tiles (and of this wave's tile for its row sums), the first V^T
    // operands (two ds_read_b64_tr_b16 per 16-dim tile, kAheadV tiles ahead)
    // and the first K operands of S(it).
    const uint32_t par_pv = (uint32_t)(it & 1);
    // Load waves read all their V^T operands up front: their row stores
    // later in the step would otherwise sit ahead of V^T reads in the LDS.
    constexpr int kAheadV = kScore ? 3 : kLoadDimTiles;  // score waves: 2 / 3 / 4 measured 160.36 / 160.11 / 160.41 us
    constexpr int kAheadK = 6;
    float al[4];
    int32_t prow = 0;
    v8bf pb[4], p_own;
    v4s vlo[kAheadV], vhi[kAheadV];
    v4u ka[kAheadK];
    uint32_t vbase = 0, kbase = 0;
    if constexpr (kPV) {
#pragma unroll
      for (int t = 0; t < 4; ++t) al[t] = lds.alpha[par_pv][16 * t + c];
    }
    if constexpr (kScore && kSoft)
      prow = lds_load<int32_t>(ring_base + 4 * (uint32_t)(((it - 1) % kRing) * kBlock + n));
    if constexpr (kPV) {
      if constexpr (kScore) {
#pragma unroll
        for (int t = 0; t < 4; ++t)
          pb[t] = as_v8bf(lds_load<v4u>(p_base + par_pv * 4096 + (uint32_t)(t * 64 + lane) * 16));
        p_own = as_v8bf(lds_load<v4u>(p_base + par_pv * 4096 + (uint32_t)(wave * 64 + lane) * 16));
      } else {
        // Load waves: P^T straight into AGPRs (read from there as the MFMA
        // B operand), which frees 20 VGPRs of the role that spills (its
        // AGPR reloads per two steps 43 -> 27; layer -0.3 us). The reads go
        // out before the V^T reads, so any wait that covers a V^T operand
        // covers them too; the explicit wait below states it.
        v4u t4[5];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t addr = p_base + par_pv * 4096 + (uint32_t)(t * 64 + lane) * 16;
          asm volatile("ds_read_b128 %0, %1" : "=a"(t4[t]) : "v"(addr) : "memory");
        }
        const uint32_t own = p_base + par_pv * 4096 + (uint32_t)(wave * 64 + lane) * 16;
        asm volatile("ds_read_b128 %0, %1" : "=a"(t4[4]) : "v"(own) : "memory");
#pragma unroll
        for (int t = 0; t < 4; ++t) pb[t] = as_v8bf(t4[t]);
        p_own = as_v8bf(t4[4]);
      }
      vbase = lane_base(buf_of(it - 2), v_lane);
#pragma unroll
      for (int d = 0; d < kAheadV; ++d) {
        vlo[d] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(vbase + 32 * d));
        vhi[d] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(vbase + 32 * d + kHalf));
      }
    }
    if constexpr (kScore && kS) {
      kbase = lane_base(buf_of(it), k_lane);
#pragma unroll
      for (int d = 0; d < kAheadK; ++d) ka[d] = lds_load<v4u>(kbase + 32 * d);
    }

    // The step's two data-dependent checks, placed after some independent
    // work so that their LDS reads have landed: rescale O^T (and the row
    // sums) by block it - 2's factors if any head's running max rose, and
    // turn the padding keys of block it - 1 into -inf before its softmax.
    auto checks = [&]() __attribute__((always_inline)) {
      if constexpr (kPV) {
        bool rescale = false;
#pragma unroll
        for (int t = 0; t < 4; ++t) rescale |= al[t] != 1.0f;
        if (__builtin_amdgcn_ballot_w64(rescale)) {
#pragma unroll
          for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int m = 0; m < kM; ++m) o[t][m] *= al[t];
          l_acc *= lds.alpha[par_pv][16 * wave + c];
        }
      }
      if constexpr (kScore && kSoft) {
        const uint32_t vmask = (uint32_t)__builtin_amdgcn_ballot_w64(h == 0 && prow >= 0);
        if (vmask != 0xFFFFFFFFu) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = score_key(8 * (r >> 2) + 4 * h + (r & 3));
            s_prev[r] = (vmask >> key) & 1u ? s_prev[r] : neg_inf;
          }
        }
      }
    };
    // PV MFMA number k of this step (k < 4 kM: dim tile k / 4, head tile
    // k % 4; k = 4 kM: the row sums of this wave's head tile).
    auto pv_mfma = [&](int k) __attribute__((always_inline)) {
      if (k == 4 * kM) {
        const v4u ones = v4u{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
        l_acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_v8bf(ones), p_own, l_acc, 0, 0, 0);
        return;
      }
      const int m = k >> 2, t = k & 3;
      const v8bf va = __builtin_bit_cast(
          v8bf, __builtin_shufflevector(vlo[m % kAheadV], vhi[m % kAheadV], 0, 1, 2, 3, 4, 5, 6, 7));
      o[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb[t], o[t][m], 0, 0, 0);
      if (t == 3 && m + kAheadV < kM) {
        vlo[m % kAheadV] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(vbase + 32 * (m + kAheadV)));
        vhi[m % kAheadV] =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(vbase + 32 * (m + kAheadV) + kHalf));
      }
    };
    constexpr int kPvMfmas = kPV ? 4 * kM + 1 : 0;

    if constexpr (kScore) {
      // ---- S(it) = K Q^T (32 keys x heads 32 sw .. + 31, 36 k-steps of 16
      // dims, back to back), the PV MFMAs and the softmax of block it - 1 in
      // one instruction stream: each k-step issues its MFMA(s), then a slice
      // of the softmax's VALU work, which runs while the MFMAs execute.
      //
      // Softmax of head 32 sw + n: this lane holds keys score_key(8(r / 4) +
      // 4h + r % 4), the other half (lane ^ 32) the rest. Maxima on raw
      // scores (scale_log2 > 0), so that p = exp2(s * scale_log2 - m) is one
      // FMA and one exp2. Row sums come from the PV product (P^T against a
      // row of ones).
      v16f sa = {};
      float mx = neg_inf, alpha = 1.0f, neg_m = 0.0f;
      uint32_t pk[8];
      const uint32_t par_soft = (uint32_t)((it - 1) & 1);
      auto soft_slice = [&](int ks) __attribute__((always_inline)) {
        if (ks < 8) {
          mx = fmaxf(fmaxf(mx, s_prev[2 * ks]), s_prev[2 * ks + 1]);
        } else if (ks == 8) {
          const uint32_t u = __float_as_uint(mx);
          const auto sw32 = __builtin_amdgcn_permlane32_swap(u, u, false, false);
          mx = fmaxf(__uint_as_float(sw32[0]), __uint_as_float(sw32[1])) * scale_log2;
          const bool need = mx > m_run + kRescaleThreshold || (m_run == neg_inf && mx != neg_inf);
          const float m_new = need ? fmaxf(m_run, mx) : m_run;
          // exp2(-inf) = 0 covers the first valid block.
          alpha = need ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
          m_run = m_new;
          // With no valid key so far every score is -inf and p = 0.
          neg_m = m_run == neg_inf ? 0.0f : -m_run;
        } else if (ks < 17) {
          const int r = 2 * (ks - 9);
          pk[ks - 9] = pack_bf16(__builtin_amdgcn_exp2f(__builtin_fmaf(s_prev[r], scale_log2, neg_m)),
                                 __builtin_amdgcn_exp2f(__builtin_fmaf(s_prev[r + 1], scale_log2, neg_m)));
        } else if (ks == 17) {
          // Both row halves hold the same factor; both write it.
          lds.alpha[par_soft][32 * sw + n] = alpha;
          // P^T -> LDS: registers 4a' .. 4a' + 3 are k-indices 4(a' >> 1) ..
          // +3 of operand slot (c = n % 16, g = 2h + (a' & 1)) of head tile
          // 2 sw + n / 16.
          const uint32_t p_tile = p_base + par_soft * 4096 + (uint32_t)((2 * sw + (n >> 4)) * 64 + (n & 15)) * 16;
#pragma unroll
          for (int ap = 0; ap < 4; ++ap) {
            const int gg = 2 * h + (ap & 1);
            lds_store<v2u>(p_tile + (uint32_t)gg * 256 + 8 * (ap >> 1), v2u{pk[2 * ap], pk[2 * ap + 1]});
          }
        }
      };
      // The first kHead k-steps run S alone (the checks' reads land
      // meanwhile); then PV MFMAs and softmax slices join.
      constexpr int kHead = kS ? 3 : 0;
      constexpr int kBody = kPvMfmas > 18 ? kPvMfmas : 18;
      constexpr int kSteps = kS ? kQkDim / 16 : kBody;
      if constexpr (kHead == 0) checks();
#pragma unroll
      for (int ks = 0; ks < kSteps; ++ks) {
        if constexpr (kS) {
          const v8bf a = as_v8bf(ka[ks % kAheadK]);
          if (ks + kAheadK < kQkDim / 16) ka[ks % kAheadK] = lds_load<v4u>(kbase + 32 * (ks + kAheadK));
          sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, as_v8bf(q_ops[ks]), sa, 0, 0, 0);
        }
        if (kHead > 0 && ks == kHead - 1) checks();
        const int kb = ks - kHead;
        if (kb >= 0 && kb < kPvMfmas) pv_mfma(kb);
        if constexpr (kSoft) {
          if (kb >= 0) soft_slice(kb);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = kSteps - kHead; k < kPvMfmas; ++k) pv_mfma(k);
      static_assert(!kS || kQkDim / 16 - kHead >= 18, "softmax slices must fit the S k-steps");
      if constexpr (kS) s_prev = sa;
    } else {
      // ---- rows of block it + 1 (its buffer last held block it - 3) in
      // 32 quarters beside the PV MFMAs; the records of block it +
      // kLookahead into the freed registers.
      const uint32_t rec = kS ? lane_base(buf_of(it + 1), (uint32_t)kk * kRowBytes + 32 * j) : 0;
      const v4u* st = pool + decltype(set)::value;
      auto unpack_round = [&](int i) __attribute__((always_inline)) {
        if (kFp8) {
          const float s_i = __builtin_bit_cast(v4f, st[8])[i >> 1];
          const v4u w = st[i];
          const v4u lo{dequant_pair<false>(w.x, s_i), dequant_pair<true>(w.x, s_i),
                       dequant_pair<false>(w.y, s_i), dequant_pair<true>(w.y, s_i)};
          const v4u hi{dequant_pair<false>(w.z, s_i), dequant_pair<true>(w.z, s_i),
                       dequant_pair<false>(w.w, s_i), dequant_pair<true>(w.w, s_i)};
          lds_store<v4u>(rec + 128 * i, lo);
          lds_store<v4u>(rec + 128 * i + 16, hi);
          if (i == 7) {
            lds_store<v4u>(rec + 2 * kVDim, st[9]);
            lds_store<v4u>(rec + 2 * kVDim + 16, st[10]);
          }
        } else {
          lds_store<v4u>(rec + 128 * i, st[2 * i]);
          lds_store<v4u>(rec + 128 * i + 16, st[2 * i + 1]);
          if (i == 7) {
            lds_store<v4u>(rec + 2 * kVDim, st[16]);
            lds_store<v4u>(rec + 2 * kVDim + 16, st[17]);
          }
        }
      };
      // The rounds in quarters (two conversions each; the row's two 16-byte
      // halves stored after quarters 1 and 3), one quarter after each PV
      // MFMA: a 16-cycle MFMA hides about two VALU instructions, so whole
      // rounds (eight conversions) after every sixth MFMA stalled its pipe.
      v4u part_lo = v4u{0u, 0u, 0u, 0u}, part_hi = v4u{0u, 0u, 0u, 0u};
      auto unpack_quarter = [&](int i, int u) __attribute__((always_inline)) {
        if (kFp8) {
          const float s_i = __builtin_bit_cast(v4f, st[8])[i >> 1];
          const v4u w = st[i];
          if (u == 0) {
            part_lo.x = dequant_pair<false>(w.x, s_i);
            part_lo.y = dequant_pair<true>(w.x, s_i);
          } else if (u == 1) {
            part_lo.z = dequant_pair<false>(w.y, s_i);
            part_lo.w = dequant_pair<true>(w.y, s_i);
            lds_store<v4u>(rec + 128 * i, part_lo);
          } else if (u == 2) {
            part_hi.x = dequant_pair<false>(w.z, s_i);
            part_hi.y = dequant_pair<true>(w.z, s_i);
          } else {
            part_hi.z = dequant_pair<false>(w.w, s_i);
            part_hi.w = dequant_pair<true>(w.w, s_i);
            lds_store<v4u>(rec + 128 * i + 16, part_hi);
            if (i == 7) {
              lds_store<v4u>(rec + 2 * kVDim, st[9]);
              lds_store<v4u>(rec + 2 * kVDim + 16, st[10]);
            }
          }
        } else if (u == 3) {
          unpack_round(i);  // bf16 records: stores only
        }
      };
      checks();
      // P^T of the load waves landed: 20 V^T reads follow them.
      if constexpr (kPV) asm volatile("s_waitcnt lgkmcnt(15)" ::: "memory");
      constexpr int kQuarters = kS ? 32 : 0;
      constexpr int kSteps = kPvMfmas > kQuarters ? kPvMfmas : kQuarters;
#pragma unroll
      for (int k = 0; k < kSteps; ++k) {
        if (k < kPvMfmas) pv_mfma(k);
        if (k < kQuarters) unpack_quarter(k / 4, k % 4);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (kS) {
        // Ring: row of block it + kRingAhead (its slot held block it - 2)
        // from its id and page, both landed two steps ago; then the page of
        // block it + kRingAhead + 2 from its id (loaded two steps ago, kept
        // for the row two steps from now) and the id of block it +
        // kRingAhead + 4. Each link of the id -> page -> row chain thus has
        // two steps to land (with one step each, the load waves waited
        // ~640 ticks per step here). These loads go out before the record
        // loads, so that waiting for them waits for nothing the step does not
        // wait for anyway. Loaded values live in one register per step parity
        // and are copied only once landed; the four lanes of a key store the
        // same value.
        constexpr int kP = decltype(parity)::value;
        lds.ring[(it + kRingAhead) % kRing][kk] = phys_from(id_keep[kP], ring_page[kP]);
        id_keep[kP] = ring_id[kP];
        ring_page[kP] = page_load(ring_id[kP]);
        ring_id[kP] = id_load(it + kRingAhead + 4);
        fetch(set, phys_next);
        phys_next = row_of(it + kLookahead + 1);
      }
    }
    lds_barrier();
  };
  using Pre0 = std::integral_constant<int, 1>;   // S / rows only
  using Pre1 = std::integral_constant<int, 3>;   // + softmax
  using Full = std::integral_constant<int, 7>;   // + PV
  using Tail0 = std::integral_constant<int, 6>;  // softmax + PV
  using Tail1 = std::integral_constant<int, 4>;  // PV only
  auto run = [&](auto role) __attribute__((always_inline)) {
    constexpr int kM = decltype(role)::value ? kScoreDimTiles : kLoadDimTiles;
    // O^T: head tile t (heads 16t + c), dims dim0 + 16m + 4g + r.
    v4f o[4][kM];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int m = 0; m < kM; ++m) o[t][m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    v16f s_prev = {};
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    step(0, Set1{}, Even{}, role, Pre0{}, o, s_prev);
    step(1, Set0{}, Odd{}, role, Pre1{}, o, s_prev);
    // Two blocks per trip so that each register set stays a fixed register set.
    for (int it = 2; it < n_blocks; it += 2) {
      step(it, Set1{}, Even{}, role, Full{}, o, s_prev);
      step(it + 1, Set0{}, Odd{}, role, Full{}, o, s_prev);
    }
    step(n_blocks, Set1{}, Even{}, role, Tail0{}, o, s_prev);
    step(n_blocks + 1, Set0{}, Odd{}, role, Tail1{}, o, s_prev);
    // The fetches past the last block are never read; let them land before
    // the registers are released.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- row sums of all 64 heads, then O / l.
    if (g == 0) lds.row_sum[16 * wave + c] = l_acc[0];
    __syncthreads();
    // Two dim tiles at a time: the row groups swap halves, so that a lane
    // holds 8 consecutive dims (of tile m + (g & 1)) and a head's 64 bytes go
    // out in one instruction. With 8 bytes a lane (32 of a head) the stores
    // took 7.5k cycles to land, now 3.9k (1,024 rows of 128 heads: 636 -> 631
    // us, with 64 keys 106.0 -> 94.4).
    uint16_t* obase = out + ((row * heads + head0 + c) * kVDim) + dim0 + 16 * (g & 1) + 8 * (g >> 1);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float lt = lds.row_sum[16 * t + c];
      const float inv_l = lt > 0.0f ? 1.0f / lt : 0.0f;
      uint16_t* orow = obase + (int64_t)16 * t * kVDim;
#pragma unroll
      for (int m = 0; m < kM; m += 2) {
        const auto lo = __builtin_amdgcn_permlane16_swap(
            pack_bf16(o[t][m][0] * inv_l, o[t][m][1] * inv_l),
            pack_bf16(o[t][m + 1][0] * inv_l, o[t][m + 1][1] * inv_l), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(
            pack_bf16(o[t][m][2] * inv_l, o[t][m][3] * inv_l),
            pack_bf16(o[t][m + 1][2] * inv_l, o[t][m + 1][3] * inv_l), false, false);
        *reinterpret_cast<v4u_out*>(orow + 16 * m) = v4u_out{lo[0], hi[0], lo[1], hi[1]};
      }
    }
  };
  if (scorer) run(std::true_type{});
  else run(std::false_type{});
}

// ---- few query rows: scores and values in two launches.
//
// (row, 64 heads) work-groups leave most CUs idle below 128 rows x 128 heads,
// and a row's 64 key blocks are one serial chain of ~1.1 us steps. Splitting
// the keys of one accumulation would make the fp32 sums depend on the batch
// size; the work is split where it changes no sum, so the results have the
// bits of sparse_mla_fwd:
// * mla_scores: the scores of any key block are independent of the others.
//   A work-group takes a row, 64 or 128 heads and a run of key blocks and
//   writes the blocks' scores (fp32, -inf at padding) in the order of the PV
//   operands, and each block's maximum per head.
// * mla_values: the value dims are independent of each other. A work-group
//   takes a row, 64 heads and 64 or 128 of the 512 dims, replays the running-max
//   chain from the block maxima, forms P^T straight in the operand registers
//   and runs the PV products block by block, in sparse_mla_fwd's order.
// A block without a valid key changes no sum and is skipped.
//
// What bounds them: mla_scores (9.6 us for one row of 128 heads, 16.4 for 16) is
// a chain of load latencies, ids -> pages -> records -> LDS, in front of one to
// eight 1,152-cycle MFMA steps. mla_values (23.0 us for one row, 25.3 for 16, 32.2 for 32
// with 128 dims) is one wave per SIMD issuing ~65 instructions per block (~650
// cycles with the LDS waits). The workspace holds 1 MB of fp32 scores per row of
// 128 heads and 2,048 selected (34 MB with the maxima at the 32 rows of a quarter round).
constexpr int kScoreThreads = 512;
constexpr int kScoreKeys = 1024;                      // most keys per work-group of mla_scores
constexpr int kSplitSelected = 2048;                  // widest selection of the split form
constexpr int kValueThreads = 256;
constexpr int kValueBlocks = 2;                       // key blocks per step of mla_values
constexpr int kValueKeys = kValueBlocks * kBlock;
constexpr int kValueDepth = 4;                        // steps of mla_values' loads in flight

// The records of positions first + tid + kThreadsN u (u < kBatch) of a
// selection; the zero record for padding, an id outside [0, n_tokens) or a
// page outside the cache. Ids, then pages, are loaded all at once.
template <bool kFp8, int kThreadsN, int kBatch>
__device__ __forceinline__ void resolve_records(const int32_t* __restrict__ ids, int first, int end,
                                                const uint8_t* __restrict__ kv,
                                                const int32_t* __restrict__ page_table,
                                                int64_t n_tokens, int64_t pages,
                                                uint64_t (&rec)[kBatch], bool (&valid)[kBatch]) {
  int32_t id[kBatch], page[kBatch];
#pragma unroll
  for (int u = 0; u < kBatch; ++u) {
    const int i = first + (int)threadIdx.x + kThreadsN * u;
    id[u] = ids[i < end ? i : 0];
    if (i >= end) id[u] = -1;
  }
#pragma unroll
  for (int u = 0; u < kBatch; ++u) {
    valid[u] = id[u] >= 0 && id[u] < n_tokens;
    page[u] = kFp8 ? page_table[valid[u] ? id[u] / kPageTokens : 0] : 0;
  }
#pragma unroll
  for (int u = 0; u < kBatch; ++u) {
    valid[u] = valid[u] && (!kFp8 || (page[u] >= 0 && page[u] < pages));
    const int64_t at = kFp8 ? (int64_t)page[u] * kPageTokens + id[u] % kPageTokens : (int64_t)id[u];
    rec[u] = (uint64_t)(uintptr_t)(valid[u] ? kv + at * Format<kFp8>::kRecordBytes : zero_record);
  }
}

// Scores of the split form: [row][block][head / 16][64 lanes][8] floats, lane
// 16 g + c holding head c's key 2(j & 3) + 8(g & 1) + (g >> 1) + 16(j >> 2) at
// j; block maxima (scaled): [row][block][head].
constexpr int kScoreTile = 64 * 8;

// Key blocks of a selection in the split form: whole rounds of mla_values
// (blocks past the selection hold -inf scores).
constexpr int kValueRound = 8;
__host__ __device__ constexpr int padded_blocks(int64_t topk) {
  return (int)((topk + kBlock * kValueRound - 1) / (kBlock * kValueRound)) * kValueRound;
}

// One work-group: kTiles head tiles of 32 (waves 0-3: tile wave % kTiles of
// block wave / kTiles of the step), the K rows of a step's 4 / kTiles blocks
// staged once as bf16 rows in LDS by waves 4-7, a step ahead.
template <bool kFp8, int kTiles>
__global__ __launch_bounds__(kScoreThreads, 1) void mla_scores(
    const uint16_t* __restrict__ q, const uint8_t* __restrict__ kv,
    const int32_t* __restrict__ page_table, int64_t n_tokens, int64_t pages,
    const int32_t* __restrict__ indices, int64_t heads, int64_t topk, float scale_log2,
    int32_t chunks, int32_t chunk_steps, float* __restrict__ scores,
    float* __restrict__ block_max) {
  constexpr int kStepBlocks = 4 / kTiles;
  constexpr int kStepKeys = kStepBlocks * kBlock;
  // Staging: kLanes lanes per key, each 16-byte pieces of its record.
  constexpr int kLanes = 256 / kStepKeys;
  constexpr int kLatent = (kFp8 ? kVDim : 2 * kQkDim) / (16 * kLanes);
  constexpr int kRope = kFp8 ? 8 / kLanes : 0;
  // Register sets of records in flight: a step's records are loaded kDepth
  // steps before they are staged.
  constexpr int kDepth = kLatent + kRope > 10 ? 1 : kLatent + kRope > 6 ? 2 : 3;
  __shared__ __align__(16) uint8_t rows_lds[2][kStepKeys * kRowBytes];
  // This work-group's records (and the staging's look-ahead past them).
  __shared__ uint64_t records[kScoreKeys + kDepth * kStepKeys];
  __shared__ uint32_t valid_bits[kScoreKeys / 32];  // by block, bit = key
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float neg_inf = -__builtin_inff();
  const uint32_t groups = (uint32_t)(heads / (32 * kTiles));
  const uint32_t chunk = blockIdx.x % (uint32_t)chunks;
  const uint32_t rest = blockIdx.x / (uint32_t)chunks;
  const int64_t head0 = (int64_t)(rest % groups) * (32 * kTiles);
  const int64_t row = rest / groups;
  const int n_blocks = padded_blocks(topk);
  const int all_steps = n_blocks / kStepBlocks;
  const int step0 = (int)chunk * chunk_steps;
  const int steps = min(chunk_steps, all_steps - step0);
  if (steps <= 0) return;
  const int32_t* ids = indices + row * topk;
  const int first = step0 * kStepKeys;

  // The score waves' Q^T operands (k-step ks: dims 16 ks + 8h of head n), on
  // their way while the records are looked up.
  constexpr int kQOps = kQkDim / 16;
  const int tile = wave % kTiles;
  const int n = lane & 31;
  const int h = lane >> 5;
  v4u q_ops[kQOps];
  if (wave < 4) {
    const uint16_t* qrow = q + ((row * heads + head0 + 32 * tile + n) * kQkDim) + 8 * h;
#pragma unroll
    for (int ks = 0; ks < kQOps; ++ks) q_ops[ks] = *reinterpret_cast<const v4u*>(qrow + 16 * ks);
  }
  for (int i0 = 0; i0 < (steps + kDepth) * kStepKeys; i0 += kScoreThreads) {
    uint64_t rec[1];
    bool valid[1];
    const int end = (int)(topk < first + steps * kStepKeys ? topk : first + steps * kStepKeys);
    resolve_records<kFp8, kScoreThreads, 1>(ids, first + i0, end, kv, page_table, n_tokens, pages, rec, valid);
    const int i = i0 + (int)threadIdx.x;
    const uint64_t bits = __builtin_amdgcn_ballot_w64(valid[0]);
    if (i < (steps + kDepth) * kStepKeys) records[i] = rec[0];
    if (i < steps * kStepKeys && (lane & 31) == 0) valid_bits[i / 32] = (uint32_t)(bits >> (lane & 32));
  }
  __syncthreads();

  if (wave < 4) {
    // ---- score wave
    const int blk = wave / kTiles;
    constexpr int kQAgprs = 32;  // operands held in AGPRs (256 registers per wave, split 128 / 128)
#pragma unroll
    for (int ks = 0; ks < kQAgprs; ++ks) asm volatile("" : "+a"(q_ops[ks]));
    const uint32_t k_lane = (uint32_t)(uintptr_t)&rows_lds[0][0] +
                            (uint32_t)(blk * kBlock + score_key(n)) * kRowBytes + 16 * h;
    // The scores of the previous step, finished (padding keys, maximum,
    // stores) in slices under this step's MFMAs.
    v16f prev = {};
    uint32_t prev_mask = 0;
    int prev_block = 0;
    float mx = neg_inf;
    auto finish = [&](int slice) __attribute__((always_inline)) {
      if (slice < 8) {
        mx = fmaxf(fmaxf(mx, prev[2 * slice]), prev[2 * slice + 1]);
      } else if (slice == 8) {
        const uint32_t ub = __float_as_uint(mx);
        const auto sw32 = __builtin_amdgcn_permlane32_swap(ub, ub, false, false);
        mx = fmaxf(__uint_as_float(sw32[0]), __uint_as_float(sw32[1])) * scale_log2;
      } else if (slice < 13) {
        const int ap = slice - 9;
        float* dst = scores + (((row * n_blocks + prev_block) * (heads / 16)) + (head0 + 32 * tile) / 16 + (n >> 4)) * kScoreTile;
        *reinterpret_cast<v4f*>(dst + ((2 * h + (ap & 1)) * 16 + (n & 15)) * 8 + 4 * (ap >> 1)) =
            v4f{prev[4 * ap], prev[4 * ap + 1], prev[4 * ap + 2], prev[4 * ap + 3]};
      } else if (slice == 13) {
        if (h == 0) block_max[(row * n_blocks + prev_block) * heads + head0 + 32 * tile + n] = mx;
      }
    };
    auto mask_padding = [&]() __attribute__((always_inline)) {
      mx = neg_inf;
      if (prev_mask != 0xFFFFFFFFu) {
        // Key of register r: score_key(8 (r / 4) + 4 h + r % 4).
        const uint32_t mine = prev_mask >> h;
#pragma unroll
        for (int r = 0; r < 16; ++r) prev[r] = mine & (1u << score_key(8 * (r >> 2) + (r & 3))) ? prev[r] : neg_inf;
      }
    };
    lds_barrier();  // step 0's rows
    for (int t = 0; t < steps; ++t) {
      const uint32_t kbase = k_lane + (uint32_t)(t & 1) * (uint32_t)sizeof(rows_lds[0]);
      constexpr int kAheadK = 12;
      v4u ka[kAheadK];
#pragma unroll
      for (int d = 0; d < kAheadK; ++d) ka[d] = lds_load<v4u>(kbase + 32 * d);
      const uint32_t step_bits = valid_bits[t * kStepBlocks + blk];
      v16f s = {};
      if (t > 0) mask_padding();
#pragma unroll
      for (int ks = 0; ks < kQOps; ++ks) {
        const v8bf a = as_v8bf(ka[ks % kAheadK]);
        if (ks + kAheadK < kQOps) ka[ks % kAheadK] = lds_load<v4u>(kbase + 32 * (ks + kAheadK));
        s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, as_v8bf(q_ops[ks]), s, 0, 0, 0);
        if (ks >= 2 && ks < 11) finish(ks - 2);
        if (ks == 11 && t > 0) {
#pragma unroll
          for (int i = 9; i < 14; ++i) finish(i);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      prev = s;
      prev_mask = __builtin_amdgcn_readfirstlane(step_bits);
      prev_block = (step0 + t) * kStepBlocks + blk;
      lds_barrier();
    }
    mask_padding();
#pragma unroll
    for (int i = 0; i < 14; ++i) finish(i);
    for (int t = steps; t % kDepth != 0; ++t) lds_barrier();  // the staging waves' whole rounds
    return;
  }

  // ---- staging wave
  const int slot = threadIdx.x - 256;
  const int kk = slot / kLanes;
  const int j = slot % kLanes;
  v4u raw[kDepth][kLatent + kRope];
  v4f tile_scales[kDepth] = {};
  auto fetch = [&](int t, int set) __attribute__((always_inline)) {
    const uint64_t rec = records[t * kStepKeys + kk];
    const uint64_t mine = rec + 16 * j;
#pragma unroll
    for (int i = 0; i < kLatent; ++i) raw[set][i] = global_read<v4u>(mine + 16 * kLanes * i);
#pragma unroll
    for (int i = 0; i < kRope; ++i) raw[set][kLatent + i] = global_read<v4u>(mine + kVDim + 16 + 16 * kLanes * i);
    if (kFp8) tile_scales[set] = global_read<v4f>(rec + kVDim);
  };
  auto stage = [&](int t, int set) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)(uintptr_t)&rows_lds[0][0] + (uint32_t)(t & 1) * (uint32_t)sizeof(rows_lds[0]) +
                        (uint32_t)kk * kRowBytes;
#pragma unroll
    for (int i = 0; i < kLatent; ++i) {
      if (kFp8) {
        const float sc = tile_scales[set][16 * kLanes * i / 128];
        const v4u w = raw[set][i];
        const uint32_t to = at + 32 * (uint32_t)(kLanes * i + j);
        lds_store<v4u>(to, v4u{dequant_pair<false>(w.x, sc), dequant_pair<true>(w.x, sc),
                               dequant_pair<false>(w.y, sc), dequant_pair<true>(w.y, sc)});
        lds_store<v4u>(to + 16, v4u{dequant_pair<false>(w.z, sc), dequant_pair<true>(w.z, sc),
                                    dequant_pair<false>(w.w, sc), dequant_pair<true>(w.w, sc)});
      } else {
        lds_store<v4u>(at + 16 * (uint32_t)(kLanes * i + j), raw[set][i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kRope; ++i)
      lds_store<v4u>(at + 2 * kVDim + 16 * (uint32_t)(kLanes * i + j), raw[set][kLatent + i]);
  };
#pragma unroll
  for (int u = 0; u < kDepth; ++u) fetch(min(u, steps), u);
  // Step t's rows are staged before the barrier that starts S(t); their
  // buffer's last reader, S(t - 2), ended before the barrier before that one.
  for (int t0 = 0; t0 < steps; t0 += kDepth) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) {
      stage(t0 + u, u);  // past the last step: zero rows nobody reads
      __builtin_amdgcn_sched_barrier(0);
      fetch(min(t0 + u + kDepth, steps), u);
      lds_barrier();
    }
  }
  lds_barrier();  // the barrier after S(steps - 1)
}

// One work-group: a row, 64 heads (wave w: heads 16 w .. + 15) and kDv of the
// value dims, in steps of kValueBlocks key blocks. Latency rules it (records,
// scores and maxima come from the last-level cache or HBM), so all loads of a
// step go out kValueDepth steps ahead.
template <bool kFp8, int kDv>
__global__ __launch_bounds__(kValueThreads, 2) void mla_values(
    const uint8_t* __restrict__ kv, const int32_t* __restrict__ page_table, int64_t n_tokens,
    int64_t pages, const int32_t* __restrict__ indices, int64_t rows, int64_t heads, int64_t topk,
    float scale_log2, const float* __restrict__ scores, const float* __restrict__ block_max,
    uint16_t* __restrict__ out) {
  // Value rows of a step, by parity: rows 4 or 36 (mod 64) dwords apart, so
  // that the 8 even (or odd) keys of a V^T transpose read are on disjoint
  // 8-bank windows.
  constexpr int kStride = 2 * kDv + 16;
  static_assert(kStride / 4 % 64 == 4 || kStride / 4 % 64 == 36, "bank windows of the transpose reads");
  __shared__ __align__(16) uint8_t v_lds[2][kValueKeys * kStride];
  __shared__ uint64_t records[kSplitSelected + (kValueDepth + 1) * kValueKeys];  // + the look-ahead
  __shared__ int32_t wave_last[kValueThreads / 64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15;
  const int g = lane >> 4;
  const float neg_inf = -__builtin_inff();
  // Work-groups go to the XCDs round-robin by linear id: the parts of one
  // (row, 64 heads), which read the same scores, are 8 ids apart and share an
  // XCD's L2.
  constexpr uint32_t kParts = kVDim / kDv;
  const uint32_t groups = (uint32_t)(heads / 64);
  const uint32_t tile = (blockIdx.x / (8 * kParts)) * 8 + (blockIdx.x & 7);
  const int d0 = (int)((blockIdx.x >> 3) % kParts) * kDv;
  const int64_t row = tile / groups;
  if (row >= rows) return;
  const int64_t head0 = (int64_t)(tile % groups) * 64 + 16 * wave;
  const int32_t* ids = indices + row * topk;
  const int n_blocks = padded_blocks(topk);

  // Scores and maxima of this wave's 16 heads (uniform base, lane offset).
  v4f s_lo[kValueDepth][kValueBlocks], s_hi[kValueDepth][kValueBlocks];
  float mb[kValueDepth][kValueBlocks];
  // (A row's scores are n_blocks x heads x 128 bytes: 32-bit offsets.)
  const int64_t tiles16 = heads / 16;
  const uint8_t* s_base = reinterpret_cast<const uint8_t*>(scores + (row * n_blocks * tiles16 + head0 / 16) * kScoreTile);
  const uint8_t* m_base = reinterpret_cast<const uint8_t*>(block_max + row * n_blocks * heads + head0);
  auto load_scores = [&](int t, int b, int set) __attribute__((always_inline)) {
    // Past the last block: the last one again, not used.
    const uint32_t block = (uint32_t)min(t * kValueBlocks + b, n_blocks - 1);
    const uint32_t at = block * (uint32_t)(tiles16 * kScoreTile * 4) + 32u * (uint32_t)lane;
    s_lo[set][b] = *reinterpret_cast<const v4f*>(s_base + at);
    s_hi[set][b] = *reinterpret_cast<const v4f*>(s_base + at + 16);
    mb[set][b] = *reinterpret_cast<const float*>(m_base + (block * (uint32_t)(heads * 4) + 4u * (uint32_t)c));
  };

  // Record rows of the whole selection, and the last valid position.
  {
    int32_t last = -1;
    constexpr int kBatch = 8;
    const int total = n_blocks * kBlock;
    for (int i = threadIdx.x; i < (kValueDepth + 1) * kValueKeys; i += kValueThreads)
      records[total + i] = (uint64_t)(uintptr_t)zero_record;
    for (int i0 = 0; i0 < total; i0 += kBatch * kValueThreads) {
      uint64_t rec[kBatch];
      bool valid[kBatch];
      resolve_records<kFp8, kValueThreads, kBatch>(ids, i0, (int)topk, kv, page_table, n_tokens, pages, rec, valid);
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int i = i0 + (int)threadIdx.x + kValueThreads * u;
        if (i < total) records[i] = rec[u] + (kFp8 ? d0 : 2 * d0);
        if (valid[u]) last = i;
      }
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) last = max(last, __shfl_xor(last, m));
    if (lane == 0) wave_last[wave] = last;
  }
  __syncthreads();
  const int last = __builtin_amdgcn_readfirstlane(
      max(max(wave_last[0], wave_last[1]), max(wave_last[2], wave_last[3])));
  static_assert(kValueRound % (kValueDepth * kValueBlocks) == 0, "whole rounds of the register sets");
  // Steps up to the last valid position, in whole rounds of the register sets.
  const int steps = (last + kValueDepth * kValueKeys) / (kValueDepth * kValueKeys) * kValueDepth;

  // Staging: four lanes per key.
  static_assert(4 * kValueKeys == kValueThreads, "a step's keys by four lanes each");
  const int kk = threadIdx.x >> 2;
  const int j = threadIdx.x & 3;
  constexpr int kRaw = kDv / 64 * (kFp8 ? 1 : 2);
  constexpr int kScales = kFp8 ? (kDv + 127) / 128 : 1;
  v4u raw[kValueDepth][kRaw];
  float tile_scale[kValueDepth][kScales] = {};
  uint64_t rec_next = records[kk];  // of the next step to fetch
  const int scale_at = kVDim + 4 * (d0 / 128) - d0;  // from the record's first value byte here
  auto fetch = [&](int t, int set) __attribute__((always_inline)) {
    const uint64_t rec = rec_next;
    rec_next = records[(t + 1) * kValueKeys + kk];
#pragma unroll
    for (int u = 0; u < kRaw; ++u) raw[set][u] = global_read<v4u>(rec + 16 * j + 64 * u);
    if (kFp8) {
#pragma unroll
      for (int u = 0; u < kScales; ++u) tile_scale[set][u] = global_read<float>(rec + scale_at + 4 * u);
    }
  };
  const uint32_t v_base = (uint32_t)(uintptr_t)&v_lds[0][0];
  auto stage = [&](int t, int set) __attribute__((always_inline)) {
    const uint32_t to = v_base + (uint32_t)(t & 1) * (uint32_t)sizeof(v_lds[0]) + (uint32_t)kk * kStride;
#pragma unroll
    for (int u = 0; u < kRaw; ++u) {
      const v4u w = raw[set][u];
      if (kFp8) {
        const float sc = tile_scale[set][u / 2];
        lds_store<v4u>(to + 128 * u + 32 * j, v4u{dequant_pair<false>(w.x, sc), dequant_pair<true>(w.x, sc),
                                                  dequant_pair<false>(w.y, sc), dequant_pair<true>(w.y, sc)});
        lds_store<v4u>(to + 128 * u + 32 * j + 16, v4u{dequant_pair<false>(w.z, sc), dequant_pair<true>(w.z, sc),
                                                       dequant_pair<false>(w.w, sc), dequant_pair<true>(w.w, sc)});
      } else {
        lds_store<v4u>(to + 64 * u + 16 * j, w);
      }
    }
  };

  constexpr int kM = kDv / 16;
  v4f o[kM], l_acc = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int m = 0; m < kM; ++m) o[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = neg_inf;
  const v8bf ones = as_v8bf(v4u{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
  const int vkey = 2 * (c >> 2) + 8 * (g & 1) + (g >> 1);
  const uint32_t v_lane = v_base + (uint32_t)vkey * kStride + 8 * (c & 3);
  // The running max of this lane's head through one block, as sparse_mla_fwd
  // takes it, and the block's P^T operand; the rescale factor stays in alpha.
  float alpha = 1.0f;
  auto softmax = [&](float mx, const v4f& lo, const v4f& hi) __attribute__((always_inline)) -> v8bf {
    const bool need = (mx > m_run + kRescaleThreshold) | ((m_run == neg_inf) & (mx != neg_inf));
    const float m_new = (need & (mx > m_run)) ? mx : m_run;
    alpha = need ? __builtin_amdgcn_exp2f(m_run - m_new) : 1.0f;
    m_run = m_new;
    const float neg_m = m_run == neg_inf ? 0.0f : -m_run;
    auto p = [&](float v) { return __builtin_amdgcn_exp2f(__builtin_fmaf(v, scale_log2, neg_m)); };
    return as_v8bf(v4u{pack_bf16(p(lo[0]), p(lo[1])), pack_bf16(p(lo[2]), p(lo[3])),
                       pack_bf16(p(hi[0]), p(hi[1])), pack_bf16(p(hi[2]), p(hi[3]))});
  };
  if (steps > 0) {
#pragma unroll
    for (int u = 0; u < kValueDepth; ++u) {
      fetch(u, u);
#pragma unroll
      for (int b = 0; b < kValueBlocks; ++b) load_scores(u, b, u);
    }
    // The softmax runs one block ahead of the PV products: its VALU work
    // fills the LDS latency and the MFMAs of the block before.
    v8bf p_next = softmax(mb[0][0], s_lo[0][0], s_hi[0][0]);
    for (int t0 = 0; t0 < steps; t0 += kValueDepth) {
#pragma unroll
      for (int u = 0; u < kValueDepth; ++u) {
        const int t = t0 + u;
        stage(t, u);  // the buffer's last readers passed the previous barrier
        __builtin_amdgcn_sched_barrier(0);
        fetch(t + kValueDepth, u);
        lds_barrier();
        const uint32_t vb = v_lane + (uint32_t)(t & 1) * (uint32_t)sizeof(v_lds[0]);
#pragma unroll
        for (int b = 0; b < kValueBlocks; ++b) {
          if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
            l_acc *= alpha;
#pragma unroll
            for (int m = 0; m < kM; ++m) o[m] *= alpha;
          }
          const v8bf pb = p_next;
          v4s v0[kM], v1[kM];
#pragma unroll
          for (int m = 0; m < kM; ++m) {
            const uint32_t at = vb + (uint32_t)(b * kBlock) * kStride + 32 * m;
            v0[m] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)at);
            v1[m] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s)(uintptr_t)(at + 16 * kStride));
          }
          // The next block's scores: in this step's set or the next one's.
          const int nu = b + 1 < kValueBlocks ? u : (u + 1) % kValueDepth;
          const int nb = b + 1 < kValueBlocks ? b + 1 : 0;
          v4u p_regs = __builtin_bit_cast(v4u, softmax(mb[nu][nb], s_lo[nu][nb], s_hi[nu][nb]));
          asm volatile("" : "+v"(p_regs));  // here, ahead of the MFMAs that wait for the V^T reads
          p_next = as_v8bf(p_regs);
          l_acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, pb, l_acc, 0, 0, 0);
#pragma unroll
          for (int m = 0; m < kM; ++m) {
            const v8bf va = __builtin_bit_cast(v8bf, __builtin_shufflevector(v0[m], v1[m], 0, 1, 2, 3, 4, 5, 6, 7));
            o[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pb, o[m], 0, 0, 0);
          }
        }
        // Into the registers just read: loads into others would be copied
        // here, and the copies would wait for them.
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < kValueBlocks; ++b) load_scores(t + kValueDepth, b, u);
      }
    }
  }

  const float lt = l_acc[0];
  const float inv_l = lt > 0.0f ? 1.0f / lt : 0.0f;
  uint16_t* orow = out + ((row * heads + head0 + c) * kVDim) + d0 + 4 * g;
#pragma unroll
  for (int m = 0; m < kM; ++m)
    *reinterpret_cast<uint2*>(orow + 16 * m) = make_uint2(pack_bf16(o[m][0] * inv_l, o[m][1] * inv_l),
                                                          pack_bf16(o[m][2] * inv_l, o[m][3] * inv_l));
}

// How a call's rows are run: rows [0, wide_rows) by sparse_mla_fwd, the rest in
// the split form with kDv = dv.
//
// sparse_mla_fwd takes about 71 us (2,048 selected; 40 us at 1,024, 24 at 512, 18
// at 320) for each round of one (row, 64 heads) work-group per CU, however few
// there are. The split form's scores go through memory instead of LDS, so the
// rows after the last full round go there while they are few enough. Rows of
// 128 heads over fp8 / bf16 records, us, the split form beside the wide one:
//   2,048 selected  4 rows 34 / 32 (71)  16 rows 43 / 40 (72)  32 rows 54 / 56 (72)
//                   36 rows 78 / 88 (71 / 73)  64 rows 83 / 100 (73)
// so never above a quarter of a round. Below it the form of less time goes, by
// costs fitted to both (us; 17 selections of 256 .. 2,048, 33 counts of rows of 64, 128 and
// 192 heads, both formats; the form taken is within 5 % of the faster one in
// each): the wide form by its 64-key steps, the split form by its tiles (row, 64
// heads) and 256-key rounds. At 320 selected 16 rows take 18.2 / 17.9 wide (split 21.8 /
// 20.0), at 512 24.4 / 24.0 (21.9 / 20.9), 32 rows at 768 32.1 / 32.6 (32.7 / 33.2), at 1,024
// 39.9 / 40.4 (37.2 / 37.1). Below 320 selected the split form gains at most 1 us.
struct MlaPlan {
  int64_t wide_rows, split_rows;
  int dv;
  int64_t score_floats, bytes;  // of the split rows' workspace: scores, then block maxima
};

constexpr int64_t kSplitMinSelected = 320;

MlaPlan mla_plan(int64_t rows, int64_t heads, int64_t topk) {
  MlaPlan p{rows, 0, 0, 0, 0};
  const int64_t cus = device_cu_count();
  const int64_t per_row = heads / kHeadsPerGroup;
  if (topk > kSplitSelected || per_row * 4 > cus) return p;
  const int64_t round = cus / per_row;  // rows of a full round
  const int64_t tail = rows % round;
  const int64_t tiles = tail * per_row;
  if (tail == 0 || tiles * 4 > cus) return p;
  const double t = (double)tiles, steps = (double)((topk + 63) / 64), rounds = (double)((topk + 255) / 256);
  const double wide_us = 8.9 + 1.98 * steps;
  const double split_us = tiles * 8 <= cus ? 12.5 + 0.049 * t + (2.28 + 0.0453 * t) * rounds
                                           : 12.8 + 0.065 * t + (3.39 + 0.0304 * t) * rounds;
  if (topk < kSplitMinSelected || split_us >= wide_us) return p;
  p.wide_rows = rows - tail;
  p.split_rows = tail;
  // One round of mla_values work-groups at 64 dims up to an eighth of the
  // CUs' tiles; above, 128 dims halve the softmax work, which each part of the
  // dims repeats (2,048 selected: 16 rows of 128 heads 42.9 / 40.4 us with 64 dims and 47.0 / 46.1
  // with 128, 20 rows 61.4 / 57.4 and 58.1 / 56.6).
  p.dv = tiles * 8 <= cus ? 64 : 128;
  p.score_floats = tail * padded_blocks(topk) * heads * kBlock;
  p.bytes = (p.score_floats + tail * padded_blocks(topk) * heads) * 4;
  return p;
}

template <bool kFp8>
int launch_split(const MlaPlan& p, const uint16_t* q, int64_t heads, const uint8_t* kv,
                 const int32_t* page_table, int64_t n_tokens, int64_t pages, const int32_t* indices,
                 int64_t topk, float scale_log2, uint16_t* out, float* scores, hipStream_t stream) {
  const int64_t rows = p.split_rows;
  float* block_max = scores + p.score_floats;
  // mla_scores: all heads of a multiple of 128 share a staged block, and the
  // blocks are dealt out for at most one work-group per CU: runs a step shorter
  // than that leave a few work-groups to a second round (12 rows of 128 heads,
  // 2,048 selected, 47.7 us as 264 work-groups, 39.8 as 192; 24 rows 59.7, 50.9).
  const int tiles = heads % 128 == 0 ? 4 : 2;
  const int64_t steps = padded_blocks(topk) * tiles / 4;
  const int64_t units = rows * (heads / (32 * tiles));
  const int64_t most = kScoreKeys / kBlock * tiles / 4;
  const int64_t fit = device_cu_count() / units;  // runs per unit in one round
  int64_t chunk = (steps + (fit > 1 ? fit : 1) - 1) / (fit > 1 ? fit : 1);
  if (chunk > most) chunk = most;
  const int64_t chunks = (steps + chunk - 1) / chunk;
  hipLaunchKernelGGL((tiles == 4 ? mla_scores<kFp8, 4> : mla_scores<kFp8, 2>),
                     dim3((unsigned)(units * chunks)), dim3(kScoreThreads), 0, stream, q, kv,
                     page_table, n_tokens, pages, indices, heads, topk, scale_log2,
                     (int32_t)chunks, (int32_t)chunk, scores, block_max);
  DSA_CHECK_LAUNCH("sparse MLA scores");
  const int64_t groups = (rows * (heads / 64) + 7) / 8;
  hipLaunchKernelGGL((p.dv == 64 ? mla_values<kFp8, 64> : mla_values<kFp8, 128>),
                     dim3((unsigned)(groups * 8 * (kVDim / p.dv))), dim3(kValueThreads), 0, stream,
                     kv, page_table, n_tokens, pages, indices, rows, heads, topk, scale_log2,
                     scores, block_max, out);
  DSA_CHECK_LAUNCH("sparse MLA values");
  return kOk;
}

template <bool kFp8>
int launch(const void* q_, int64_t rows, int64_t heads, const void* kv_, const int32_t* page_table,
           int64_t n_tokens, int64_t pages, const int32_t* indices, int64_t topk, float scale,
           void* out_, void* workspace, int64_t workspace_bytes, hipStream_t stream) {
  const uint16_t* q = static_cast<const uint16_t*>(q_);
  const uint8_t* kv = static_cast<const uint8_t*>(kv_);
  uint16_t* out = static_cast<uint16_t*>(out_);
  const float scale_log2 = scale * 1.4426950408889634f;
  MlaPlan p = mla_plan(rows, heads, topk);
  // The running max is taken on raw scores times scale_log2: an empty
  // block's -inf stays -inf (and the split form may skip it) only for
  // positive scales.
  if (workspace == nullptr || !(scale_log2 > 0.0f)) p = MlaPlan{rows, 0, 0, 0, 0};
  if (p.split_rows > 0) {
    DSA_CHECK_ARG(reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && workspace_bytes >= p.bytes,
                  "sparse MLA workspace too small or misaligned");
  }
  if (p.wide_rows > 0) {
    hipLaunchKernelGGL(sparse_mla_fwd<kFp8>,
                       dim3((unsigned)((p.wide_rows + 7) / 8 * 8 * (heads / kHeadsPerGroup))),
                       dim3(kThreads), 0, stream, q, kv, page_table, n_tokens, pages, indices,
                       p.wide_rows, heads, topk, scale_log2, out);
    DSA_CHECK_LAUNCH("sparse MLA");
  }
  if (p.split_rows > 0)
    return launch_split<kFp8>(p, q + p.wide_rows * heads * kQkDim, heads, kv, page_table, n_tokens,
                              pages, indices + p.wide_rows * topk, topk, scale_log2,
                              out + p.wide_rows * heads * kVDim, static_cast<float*>(workspace),
                              stream);
  return kOk;
}

int check_common(const void* q, int64_t rows, int64_t heads, const int32_t* indices, int64_t topk,
                 float scale, void* out) {
  DSA_CHECK_ARG(rows >= 0 && topk >= 1, "invalid sparse MLA shape");
  DSA_CHECK_ARG(topk <= kMaxSelected, "sparse MLA supports at most 4096 selected tokens per row");
  DSA_CHECK_ARG(heads > 0 && heads % kHeadsPerGroup == 0 && heads / kHeadsPerGroup < 65536,
                "heads must be a positive multiple of 64");
  DSA_CHECK_ARG(__builtin_isfinite(scale), "scale must be finite");
  DSA_CHECK_ARG(rows < 0x7FFFFFFF, "too many query rows");
  if (rows == 0) return kOk;
  DSA_CHECK_ARG(q && indices && out, "null pointer");
  DSA_CHECK_ARG(reinterpret_cast<uintptr_t>(q) % 16 == 0 && reinterpret_cast<uintptr_t>(out) % kOutAlign == 0,
                "q must be 16-byte and out 8-byte aligned");
  return kOk;
}

}  // namespace
}  // namespace dsa

extern "C" int dsa_sparse_mla_workspace_bytes(int64_t rows, int64_t heads, int64_t topk,
                                              int64_t* bytes) {
  using namespace dsa;
  DSA_CHECK_ARG(bytes != nullptr, "null pointer");
  // (Shapes the operators refuse need none.)
  *bytes = 0;
  if (rows <= 0 || rows >= 0x7FFFFFFF || heads <= 0 || heads % kHeadsPerGroup) return kOk;
  *bytes = mla_plan(rows, heads, topk).bytes;
  return kOk;
}

extern "C" int dsa_sparse_mla_bf16_ws(const void* q, int64_t rows, int64_t heads, const void* kv,
                                      int64_t kv_rows, const int32_t* indices, int64_t topk,
                                      float scale, void* out, void* workspace,
                                      int64_t workspace_bytes, hipStream_t stream) {
  using namespace dsa;
  int status = check_common(q, rows, heads, indices, topk, scale, out);
  if (status != kOk || rows == 0) return status;
  DSA_CHECK_ARG(kv_rows >= 1 && kv_rows < 0x7FFFFFFF, "KV row count must be in [1, 2^31)");
  DSA_CHECK_ARG(kv != nullptr, "null kv");
  DSA_CHECK_ARG(reinterpret_cast<uintptr_t>(kv) % 16 == 0, "kv must be 16-byte aligned");
  return launch<false>(q, rows, heads, kv, nullptr, kv_rows, 0, indices, topk, scale, out,
                       workspace, workspace_bytes, stream);
}

extern "C" int dsa_sparse_mla_bf16(const void* q, int64_t rows, int64_t heads, const void* kv,
                                   int64_t kv_rows, const int32_t* indices, int64_t topk,
                                   float scale, void* out, hipStream_t stream) {
  return dsa_sparse_mla_bf16_ws(q, rows, heads, kv, kv_rows, indices, topk, scale, out, nullptr, 0,
                                stream);
}

extern "C" int dsa_sparse_mla_fp8_paged_ws(const void* q, int64_t rows, int64_t heads,
                                           const void* cache, int64_t pages,
                                           const int32_t* page_table, int64_t n_tokens,
                                           const int32_t* indices, int64_t topk, float scale,
                                           void* out, void* workspace, int64_t workspace_bytes,
                                           hipStream_t stream) {
  using namespace dsa;
  int status = check_common(q, rows, heads, indices, topk, scale, out);
  if (status != kOk || rows == 0) return status;
  DSA_CHECK_ARG(pages >= 1 && n_tokens >= 1 && n_tokens < 0x7FFFFFFF,
                "need a nonempty cache and 1 <= n_tokens < 2^31");
  DSA_CHECK_ARG(pages * kPageTokens < 0x7FFFFFFF, "cache rows must fit int32");
  DSA_CHECK_ARG(cache && page_table, "null cache or page table");
  DSA_CHECK_ARG(reinterpret_cast<uintptr_t>(cache) % 16 == 0, "cache must be 16-byte aligned");
  return launch<true>(q, rows, heads, cache, page_table, n_tokens, pages, indices, topk, scale,
                      out, workspace, workspace_bytes, stream);
}

extern "C" int dsa_sparse_mla_fp8_paged(const void* q, int64_t rows, int64_t heads,
                                        const void* cache, int64_t pages,
                                        const int32_t* page_table, int64_t n_tokens,
                                        const int32_t* indices, int64_t topk, float scale,
                                        void* out, hipStream_t stream) {
  return dsa_sparse_mla_fp8_paged_ws(q, rows, heads, cache, pages, page_table, n_tokens, indices,
                                     topk, scale, out, nullptr, 0, stream);
}
