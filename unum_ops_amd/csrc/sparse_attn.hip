// Stage-2 sparse attention over the block table's KV slots, on gfx950.
//
// For token t and kv head h (G = 16 query heads per kv head, D = 128), the
// keys are the entries (t, h, 64k + o) of get_block_table's output
// (src/unum_ops/sparse_kernel_extension/get_table_torch.py:4-44,
// get_table_triton.py:6-67): entry p = topk_idx[h, t, k]*64 + o (wrapping
// int32) is attended when 0 <= p < seqlen_q[b] and p < token_pos_in_bs[t]
// (b = token_to_bs[t] in [0, B)), and its KV row is the slot
// Hkv * block_table[b, min(p, L-1)] + h -- row `slot` of the cache viewed as
// [-1, D], i.e. token slot block_table[b, p], head h of a [num_blocks,
// block_size, Hkv, D] cache -- or, given a precomputed slot table, that
// table's entry.  Rows outside the cache are not attended.  Then
//   out[t, h*16 + i] = softmax_j(scale * q[t, h*16+i] . K[row_j]) @ V[rows]
// (0 when no entry is attended).  The reference's consumer of the table is an
// NPU paged-attention operator (test/test_pa.py:48-71); this is its
// arithmetic on the slots the table lists.
//
// One wave walks the 64-key blocks of a (t, h) row (or a share of them, see
// sparse_attn_kernel) in halves of 32 keys.  What bounds the walk is how the
// K and V rows reach the matrix core's operand layouts: gathered straight into
// them (16 rows x 64 bytes an instruction) they come at 17 bytes a clock and
// CU, whatever the caches hold -- 1.83 ms for 4096 tokens of 2 x 64 blocks,
// also when every token takes the same blocks -- while whole 256-byte rows
// come at up to 59 from the L2.  So every row is moved whole, by buffer- or
// global-to-LDS loads, into a 16 KiB slot of the wave (32 K rows, 32 V rows),
// and read back as operands:
//   * a row's 16-byte chunk c lies at chunk c ^ sa_swz(key) of its 256 bytes,
//     so that neither the K operand's reads (one chunk of 16 keys) nor the
//     transposing reads of V (two chunks of 8 keys) meet in a bank;
//   * the slot's operands are all read into registers at once (64 VGPRs), and
//     the next half's loads start into the same slot before the arithmetic:
//     the slot waits for memory nearly all the time, and eight waves a CU
//     (two a SIMD) keep 128 KiB in flight;
//   * the loads are issued from inline assembly, their waits counted here:
//     the compiler would wait for all of them before any read of the slot.
//     The block's 64 table entries come the same way, one block ahead, into
//     two 256-byte slots, so the loop holds no load that the compiler counts;
//   * lane l computes the row address of key 4(l%16) + l/16, and a load's
//     lanes get theirs by a DPP row broadcast in the address addition.
// Per half:
//   * S^T = K Q^T on v_mfma_f32_16x16x32_bf16 (keys as M, heads as N), so a
//     lane holds four keys of a tile for one head: the online-softmax state
//     (max, sum) is one head per lane and needs no transposes;
//   * the scale's sign goes into the queries, its magnitude into the
//     exponents' fma, so the max runs over raw scores for any scale;
//   * P^T, as it stands in the accumulator layout, is the B operand of
//     v_mfma_f32_16x16x32_bf16 for O^T += V^T P^T (key slot 8g + j of a half
//     is key 4g + j%4 of tile j/4), taken as two bf16 terms (P to about
//     2^-15);
//   * the running max moves only when a half's max exceeds it by more than
//     8 (log2 units), so the O^T rescale is rare; exponentials stay <= 2^8.
//     It starts at the lowest float, not at -inf, so a half of -inf scores
//     adds zeros; a sum that is still zero at the end of a row that attended
//     a key is a softmax over -inf alone: NaN, where a row that attended
//     nothing is 0.
#include <type_traits>

#include "common.h"

namespace unum {
namespace {

constexpr float kSaLog2e = 1.4426950408889634f;
constexpr int kSaD = 128;          // head dim
constexpr int kSaG = 16;           // query heads per kv head
// Stages in flight per wave of the gather calibration.
constexpr int kSaRing = 3;
// LDS of a workgroup of the gather calibration (one wave): eight waves a CU.
constexpr int kSaLdsBytes = 20 * 1024;
// The attention kernel's LDS per wave: the K and V rows of half a block, and
// the table entries of two blocks.
constexpr int kSaHalfKeys = 32;
constexpr int kSaHalfBytes = kSaHalfKeys * kSaD * 2;   // K (or V) rows of half a block
constexpr int kSaTabBytes = 64 * 4;
constexpr int kSaWaveLds = 2 * kSaHalfBytes + 2 * kSaTabBytes;
// A workgroup of one wave takes an eighth of a CU's LDS, more than it uses: a
// ninth wave would make one SIMD's waves slower than the others', the waves
// would drift apart along their rows, and blocks that several rows attend
// would be fetched into the L2 again (4096 tokens, neighbours' selections a
// quarter alike: 941 us with eight waves a CU, 1361 us with nine).
constexpr int kSaOneWaveLds = 20 * 1024;
static_assert(kSaOneWaveLds >= kSaWaveLds, "a wave's slots");
// Waves that share a row where rows are few (see the launch).
constexpr int kSaSplit = 4;
constexpr int kSaMaxBlocks = 64;   // K <= 64 (one block id per lane)
constexpr float kSaRescale = 8.f;  // lazy-rescale threshold (log2 units)

// 256 zero bytes: the K and V "row" of every entry that is not attended, so
// each stage issues the same loads (masked keys then score 0 and carry P = 0
// against a V of zeros); also the table "entries" of a stage past the last.
__device__ __align__(256) uint32_t sa_zero_row[64];

struct SaArgs {
  const __bf16* q;
  int64_t q_st, q_sh;
  const char* kc;
  const char* vc;
  int64_t row_bytes;   // bytes between consecutive cache rows
  int64_t n_rows;      // rows of the cache viewed as [-1, D]
  const int32_t* idx;
  int64_t i_sh, i_st, i_sk;
  const int32_t* bt;   // [B, L] (fused slots), or null
  int64_t bt_sb;
  const int32_t* slots;  // [T, Hkv, K*64] slot table, or null
  const int32_t* tok_bs;
  const int32_t* pos;
  const int32_t* slen;
  int32_t pos_n, slen_n;
  void* out;           // [T, Hkv*16, 128] contiguous (u32 [T, Hkv, 64] for the gather calibration)
  int32_t T, Hkv, K, B, L;
  float c;             // softmax scale * log2(e)
  uint32_t records;    // bytes of a cache (0 past 4 GiB, where whole addresses are used)
  int32_t gshift;      // log2 of the tokens of a group (see sa_row)
};

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 sa_lds_i16x4;

// Max / sum of v over the lanes l and l^16 (l^32): v_permlane16_swap
// (v_permlane32_swap) with v in both operands returns each lane's value and
// its partner's, one in each result.
__device__ __forceinline__ float sa_max_x16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sa_max_x32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sa_sum_x16(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float sa_sum_x32(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The selection of one (t, h): lane k holds block id k (-1 past K), the
// position limit min(seqlen_q[b], token_pos_in_bs[t]) (0 when t has no
// sequence), and the base of the table the rows come from -- the slot
// table's (t, h) row, or block_table's row b.
struct SaSel {
  int32_t lane_id;
  int32_t lim;
  int32_t h;
  const int32_t* tab;
};

// The live stages: bit k of mq set when quarter q of block k (positions
// p0 .. p0+15, p0 = id*64 + 16q wrapping int32) can hold an attended entry,
// i.e. p0 lies in [0, lim).  p0 is a multiple of 16, so p0 >= 0 puts every
// position of the quarter in [0, 2^31) and p0 < 0 puts none there.  Four
// scalar words, not an array, so that no index into them is a runtime value.
struct SaStages {
  uint64_t m0, m1, m2, m3;
};

__device__ __forceinline__ SaStages sa_live(const SaSel& sel) {
  const uint32_t base = static_cast<uint32_t>(sel.lane_id) * 64u;
  auto live = [&](uint32_t q) {
    const int32_t p0 = static_cast<int32_t>(base + 16u * q);
    return p0 >= 0 && p0 < sel.lim;
  };
  return SaStages{__ballot(live(0)), __ballot(live(1)), __ballot(live(2)), __ballot(live(3))};
}

// The next live stage, 4k + q, in ascending order (-1 if none); clears it.
__device__ __forceinline__ int sa_pop(SaStages& m) {
  const uint64_t any = m.m0 | m.m1 | m.m2 | m.m3;
  if (any == 0) return -1;
  const int k = __builtin_ctzll(any);
  const uint64_t bit = 1ull << k;
  if (m.m0 & bit) { m.m0 &= ~bit; return 4 * k; }
  if (m.m1 & bit) { m.m1 &= ~bit; return 4 * k + 1; }
  if (m.m2 & bit) { m.m2 &= ~bit; return 4 * k + 2; }
  m.m3 &= ~bit;
  return 4 * k + 3;
}

// The (t, h) selection of this workgroup: block ids one per lane (one load,
// complete before the ring's loads are issued), the limit and the table row.
template <bool kTable>
__device__ __forceinline__ SaSel sa_select(const SaArgs& a, int t, int h) {
  const int lane = threadIdx.x & (kWave - 1);
  SaSel sel;
  sel.h = h;
  sel.lim = 0;
  sel.tab = nullptr;
  const int32_t b = a.tok_bs[t];
  if (b >= 0 && b < a.B) {
    const int32_t sl = a.slen[a.slen_n == 1 ? 0 : b];
    const int32_t ps = a.pos[a.pos_n == 1 ? 0 : t];
    sel.lim = sl < ps ? sl : ps;  // <= 0: nothing is attended
    sel.tab = kTable ? a.slots + (static_cast<int64_t>(t) * a.Hkv + h) * (static_cast<int64_t>(a.K) * 64)
                     : a.bt + static_cast<int64_t>(b) * a.bt_sb;
  }
  const int32_t* idx_t = a.idx + static_cast<int64_t>(h) * a.i_sh + static_cast<int64_t>(t) * a.i_st;
  sel.lane_id = lane < a.K && sel.tab != nullptr ? idx_t[static_cast<int64_t>(lane) * a.i_sk] : -1;
  return sel;
}

template <typename OutT>
__device__ __forceinline__ void sa_store4(OutT* p, f32x4 v);
template <>
__device__ __forceinline__ void sa_store4<float>(float* p, f32x4 v) {
  *reinterpret_cast<f32x4*>(p) = v;
}
template <>
__device__ __forceinline__ void sa_store4<uint16_t>(uint16_t* p, f32x4 v) {
  const uint32_t lo = f32_to_bf16_bits(v.x) | (static_cast<uint32_t>(f32_to_bf16_bits(v.y)) << 16);
  const uint32_t hi = f32_to_bf16_bits(v.z) | (static_cast<uint32_t>(f32_to_bf16_bits(v.w)) << 16);
  *reinterpret_cast<uint2*>(p) = make_uint2(lo, hi);
}

// 16-byte chunk c of a row in LDS lies at chunk c ^ sa_swz(key).  A K operand
// read takes chunk c of keys 0-3 and 12-15 and chunk c ^ 1 of keys 4-11 in one
// service (lds_b128_free), so the values of either eight keys are four pairs
// {2i, 2i + 1}; those of keys 0-7, and of 8-15, lie in different pairs, so the
// aligned chunk pairs that the transposing reads of V take from eight keys are
// distinct too.  (Keys 0-7 even, 8-15 odd, in order, met twice on every K
// read: a third of the LDS's active cycles.)
__host__ __device__ constexpr int sa_swz(int key) {
  return (((key & 7) ^ (4 * ((key >> 3) & 1))) << 1) | ((key >> 3) & 1);
}
constexpr bool sa_lds_free() {
  struct K {
    constexpr int operator()(int lane) const { return 16 * (lane & 15) + ((lane >> 4) ^ sa_swz(lane & 15)); }
  };
  if (!lds_b128_free(K{})) return false;
  for (int g = 0; g < 4; g += 2) {  // V: 32 lanes, eight keys, a chunk pair of each
    uint32_t pairs = 0;
    for (int key = 4 * g; key < 4 * g + 8; ++key) pairs |= 1u << (sa_swz(key) >> 1);
    if (pairs != 0xFFu) return false;
  }
  return true;
}
static_assert(sa_lds_free(), "K and V operand reads meet no LDS bank twice");

typedef __attribute__((address_space(3))) void* sa_lds_void;
__device__ __forceinline__ uint32_t sa_lds_at(const void* p) {
  return __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>((sa_lds_void)p)));
}

// The rows of a block: this lane's key, 4(l%16) + l/16 of its 64 (so that a
// DPP row broadcast from lane i gives each 16 lanes key 4i + l/16), and which
// lanes' keys are attended.  Below 4 GiB a row is a byte offset into both
// caches, and one that is not attended lies past their end: the buffer range
// check gives zeros.  Larger caches take whole addresses, the zero row's for
// a key that is not attended.
template <bool kWide>
struct SaRowAt;
template <>
struct SaRowAt<false> {
  uint32_t off;
  uint64_t ok;
};
template <>
struct SaRowAt<true> {
  uint64_t k, v;
  uint64_t ok;
};
constexpr uint32_t kSaNoRow = 0xFFFFFF00u;  // + 256 bytes does not wrap

struct SaMem {
  __amdgpu_buffer_rsrc_t kr, vr;
};

// Eight loads of 1 KiB (four rows each) into LDS at m0, m0 + 1024, ...  A
// write of M0 needs one wait state before an LDS load reads it.
#define UNUM_SA_LOADS(FIRST, NEXT)                                                       \
  "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\t" FIRST                            \
  NEXT("%3") NEXT("%4") NEXT("%5") NEXT("%6") NEXT("%7") NEXT("%8") NEXT("%9")           \
  "s_mov_b32 m0, %0"
#define UNUM_SA_STEP "s_add_u32 m0, m0, 0x400\n\ts_nop 0\n\t"
__device__ __forceinline__ void sa_load8(uint32_t m0, const uint32_t (&o)[8], __amdgpu_buffer_rsrc_t r) {
  int saved;
#define UNUM_SA_NEXT(V) UNUM_SA_STEP "buffer_load_dwordx4 " V ", %10, 0 offen lds\n\t"
  asm volatile(UNUM_SA_LOADS("buffer_load_dwordx4 %2, %10, 0 offen lds\n\t", UNUM_SA_NEXT)
               : "=&s"(saved)
               : "s"(m0), "v"(o[0]), "v"(o[1]), "v"(o[2]), "v"(o[3]), "v"(o[4]), "v"(o[5]), "v"(o[6]),
                 "v"(o[7]), "s"(r)
               : "memory", "scc");
#undef UNUM_SA_NEXT
}
__device__ __forceinline__ void sa_load8(uint32_t m0, const uint64_t (&p)[8]) {
  int saved;
#define UNUM_SA_NEXT(V) UNUM_SA_STEP "global_load_lds_dwordx4 " V ", off\n\t"
  asm volatile(UNUM_SA_LOADS("global_load_lds_dwordx4 %2, off\n\t", UNUM_SA_NEXT)
               : "=&s"(saved)
               : "s"(m0), "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]),
                 "v"(p[7])
               : "memory", "scc");
#undef UNUM_SA_NEXT
}

template <int kLane>
__device__ __forceinline__ uint32_t sa_row_bcast(uint32_t v) {  // DPP row_newbcast
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x150 + kLane, 0xF, 0xF, false));
}
template <int kLane>
__device__ __forceinline__ uint64_t sa_row_bcast(uint64_t v) {
  return static_cast<uint64_t>(sa_row_bcast<kLane>(static_cast<uint32_t>(v))) |
         (static_cast<uint64_t>(sa_row_bcast<kLane>(static_cast<uint32_t>(v >> 32))) << 32);
}

// The loads of half kHalf of a block: K rows to `slot`, V rows after them,
// load j moving keys 4j .. 4j+3 of the half (lanes 16r .. 16r+15: key 4j + r,
// its chunks in swizzled order; `col` holds the byte of a lane's chunk, which
// depends on j%4).  16 vector-memory operations.
template <int kHalf, bool kWide>
__device__ __forceinline__ void sa_fetch(const SaMem& mem, const SaRowAt<kWide>& at, const uint32_t (&col)[4],
                                         uint32_t slot) {
  auto rows = [&](auto v) {
    struct { decltype(v) x[8]; } o;
    o.x[0] = sa_row_bcast<8 * kHalf + 0>(v) + col[0];
    o.x[1] = sa_row_bcast<8 * kHalf + 1>(v) + col[1];
    o.x[2] = sa_row_bcast<8 * kHalf + 2>(v) + col[2];
    o.x[3] = sa_row_bcast<8 * kHalf + 3>(v) + col[3];
    o.x[4] = sa_row_bcast<8 * kHalf + 4>(v) + col[0];
    o.x[5] = sa_row_bcast<8 * kHalf + 5>(v) + col[1];
    o.x[6] = sa_row_bcast<8 * kHalf + 6>(v) + col[2];
    o.x[7] = sa_row_bcast<8 * kHalf + 7>(v) + col[3];
    return o;
  };
  if constexpr (kWide) {
    sa_load8(slot, rows(at.k).x);
    sa_load8(slot + kSaHalfBytes, rows(at.v).x);
  } else {
    const auto o = rows(at.off);
    sa_load8(slot, o.x, mem.kr);
    sa_load8(slot + kSaHalfBytes, o.x, mem.vr);
  }
}

// A block to attend: its id, where its table entries are (the slot table's
// run of it, or block_table's row), the position limit, and which of the
// wave's rows attend it (bit r; 0: no block left).
struct SaBlock {
  int32_t id;
  const int32_t* run;
  int32_t lim;
  uint32_t rows;
};

// Position of entry o of a block, wrapping int32 as the block table's (an id
// past 2^25 can wrap to a live position: the product is unsigned).
__device__ __forceinline__ int32_t sa_pos(int32_t id, int o) {
  return static_cast<int32_t>(static_cast<uint32_t>(id) * 64u + static_cast<uint32_t>(o));
}

// The load of a block's table entries into `slot`, lane l's own key's entry
// to word l: the slot table's, or block_table[b, min(p, L-1)]; zeros past the
// last block.  One vector-memory operation, always issued.
template <bool kTable>
__device__ __forceinline__ void sa_table(const SaArgs& a, const SaBlock& blk, uint32_t slot) {
  const int lane = threadIdx.x & (kWave - 1);
  const int kk = 4 * (lane & 15) + (lane >> 4);
  const int32_t* p;
  if (blk.rows == 0) {
    p = reinterpret_cast<const int32_t*>(sa_zero_row) + kk;
  } else if constexpr (kTable) {
    p = blk.run + kk;
  } else {
    const int32_t pos = sa_pos(blk.id, kk);  // the block is live: >= 0
    p = blk.run + (pos < a.L - 1 ? pos : a.L - 1);
  }
  int saved;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, off\n\ts_mov_b32 m0, %0"
               : "=&s"(saved)
               : "s"(slot), "v"(p)
               : "memory");
}

// The rows that a block's entries name (`tv`: this lane's key's).
template <bool kTable, bool kWide>
__device__ __forceinline__ SaRowAt<kWide> sa_rows(const SaArgs& a, const SaBlock& blk, int h, int32_t tv) {
  const int lane = threadIdx.x & (kWave - 1);
  const int32_t pos = sa_pos(blk.id, 4 * (lane & 15) + (lane >> 4));
  const uint32_t r = kTable ? static_cast<uint32_t>(tv)
                            : static_cast<uint32_t>(a.Hkv) * static_cast<uint32_t>(tv) + static_cast<uint32_t>(h);
  const bool ok = pos < blk.lim && r < static_cast<uint32_t>(a.n_rows);  // n_rows < 2^31: r >= 0 too
  SaRowAt<kWide> at;
  at.ok = __ballot(ok);
  if constexpr (kWide) {
    const uint64_t off = static_cast<uint64_t>(r) * static_cast<uint64_t>(a.row_bytes);
    const uint64_t zero = reinterpret_cast<uint64_t>(sa_zero_row);
    at.k = ok ? reinterpret_cast<uint64_t>(a.kc) + off : zero;
    at.v = ok ? reinterpret_cast<uint64_t>(a.vc) + off : zero;
  } else {
    at.off = ok ? r * static_cast<uint32_t>(a.row_bytes) : kSaNoRow;
  }
  return at;
}

template <int N>
__device__ __forceinline__ void sa_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

// The token (the first of kRows) and head of this workgroup.  Workgroup i runs
// on XCD i%8, and each XCD has an L2 of its own: groups of 2^gshift consecutive
// workgroups of a head go to one XCD, so that the rows that neighbouring tokens
// both attend (those of one sequence, to begin with) are fetched into one L2,
// and groups are dealt in turn, so that the XCDs get equal work also where
// contexts grow along t.  The grid is rows of 2^kSaGridShift workgroups: one
// dimension holds less than 2^32 threads, 2^24 four-wave workgroups.
constexpr int kSaGridShift = 20;
template <int kRows>
__device__ __forceinline__ bool sa_row(const SaArgs& a, int& t, int& h) {
  const uint32_t id = (blockIdx.y << kSaGridShift) + blockIdx.x;
  const uint32_t j = id >> 3;
  const uint32_t group = ((j >> a.gshift) << 3) + (id & 7);
  const uint32_t units = (static_cast<uint32_t>(a.T) + kRows - 1) / kRows;
  const uint32_t per_head = (units + (1u << a.gshift) - 1) >> a.gshift;
  h = static_cast<int>(group / per_head);
  t = kRows *
      static_cast<int>(((group - static_cast<uint32_t>(h) * per_head) << a.gshift) + (j & ((1u << a.gshift) - 1)));
  return h < a.Hkv && t < a.T;
}

// kSplit waves share a row, or (kSplit = 1) a wave takes kRows rows, two
// consecutive tokens of a head.  The two walk their blocks in one order by
// id, and a block that both attend whole is moved once for both: the L1
// delivers 64 bytes a clock, which moving every block for every token fills
// (TA busy 91 % of the cycles where all tokens take the same blocks), and
// twice the rows at once on a CU find more of their blocks in the L2.
template <typename OutT, bool kTable, bool kWide, int kSplit, int kRows>
__global__ __launch_bounds__(kWave* kSplit, 2) void sparse_attn_kernel(SaArgs a) {
  static_assert(kSplit == 1 || kRows == 1, "shared rows are single");
  static_assert(kRows == 1 || !kTable, "slot tables name rows per token: nothing to merge by");
  __shared__ __align__(1024) char lds[kSplit == 1 ? kSaOneWaveLds : kSplit * kSaWaveLds];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = kSplit == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  char* const slot = lds + wave * kSaWaveLds;
  char* const tabs = slot + 2 * kSaHalfBytes;
  int t, h;
  if (!sa_row<kRows>(a, t, h)) return;  // the whole workgroup
  const int rows = kRows == 2 && t + 1 < a.T ? 2 : 1;
  SaSel sel[kRows];
  sel[0] = sa_select<kTable>(a, t, h);
  if constexpr (kRows == 2) {
    sel[1] = sa_select<kTable>(a, t + rows - 1, h);
    if (rows == 1) sel[1].lim = 0;  // no second token: it attends nothing
  }

  // Query fragments, the B operand of S^T = K Q^T: lane (head n, g) holds
  // q[t, 16h + n, 32cc + 8g .. +8].
  bf16x8 qf[kRows][4];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const __bf16* qp = a.q + static_cast<int64_t>(i == 0 ? t : t + rows - 1) * a.q_st +
                       static_cast<int64_t>(kSaG * h + (lane & 15)) * a.q_sh + 8 * (lane >> 4);
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) qf[i][cc] = *reinterpret_cast<const bf16x8*>(qp + 32 * cc);
  }
  // A negative scale flips the queries' signs (exact).
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const uint32_t flip = a.c < 0.f ? 0x80008000u : 0u;
  const float c = fabsf(a.c);
  // The compiler's own loads (ids, queries) complete here, before the loads
  // counted below.
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) {
      qf[i][cc] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, qf[i][cc]) ^ flip);
      asm volatile("" : : "v"(qf[i][cc]));
    }
    asm volatile("" : : "v"(sel[i].lane_id));
  }
  sa_wait<0>();

  // The live blocks: first position in [0, lim).  A block's positions are 64
  // from a multiple of 64 (wrapping int32), so the first one's sign is all
  // of theirs.  Wave w of a split row takes the blocks k = w mod kSplit (ids
  // that select nothing come first: contiguous shares would be uneven).
  uint64_t live[kRows];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int32_t p0 = sa_pos(sel[i].lane_id, 0);
    live[i] = __ballot(p0 >= 0 && p0 < sel[i].lim);
  }
  if constexpr (kSplit > 1) {
    static_assert(kSplit == 4, "stripes of four waves");
    live[0] &= 0x1111111111111111ull << wave;
  }
  auto at_block = [&](const SaSel& s, int k, uint32_t who) {
    return SaBlock{__builtin_amdgcn_readlane(s.lane_id, k), kTable ? s.tab + 64 * k : s.tab, s.lim, who};
  };
  auto pop = [&]() __attribute__((always_inline)) -> SaBlock {
    if constexpr (kRows == 1) {
      if (live[0] == 0) return SaBlock{0, nullptr, 0, 0};
      const int k = __builtin_ctzll(live[0]);
      live[0] &= live[0] - 1;
      return at_block(sel[0], k, 1);
    } else {
      // The lists' next blocks: the lower id, or both when they are one block
      // of one sequence that both tokens attend whole.  (Ids in any order and
      // repeated ids are fine: each is taken once, in some order.)
      if (live[0] == 0 && live[1] == 0) return SaBlock{0, nullptr, 0, 0};
      const bool same = sel[0].tab == sel[1].tab;
      const int k0 = live[0] != 0 ? __builtin_ctzll(live[0]) : 0, k1 = live[1] != 0 ? __builtin_ctzll(live[1]) : 0;
      const int32_t id0 = __builtin_amdgcn_readlane(sel[0].lane_id, k0);
      const int32_t id1 = __builtin_amdgcn_readlane(sel[1].lane_id, k1);
      const bool first = live[0] != 0 && (live[1] == 0 || !same || id0 <= id1);
      const int32_t least = sel[0].lim < sel[1].lim ? sel[0].lim : sel[1].lim;
      const bool both = first && live[1] != 0 && same && id0 == id1 && sa_pos(id0, 63) < least;
      if (first) live[0] &= live[0] - 1;
      if (!first || both) live[1] &= live[1] - 1;
      return first ? at_block(sel[0], k0, both ? 3 : 1) : at_block(sel[1], k1, 2);
    }
  };

  // Per-lane constants of the loads and of the operand reads.
  const int g = lane >> 4;
  const int s = lane & 15;
  uint32_t col[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) col[i] = 16u * static_cast<uint32_t>(s ^ sa_swz(4 * i + g));
  int koff[4];  // chunk 4cc + g of key s
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) koff[cc] = 256 * s + 16 * ((4 * cc + g) ^ sa_swz(s));
  // V^T: dims 16dt + 4(s%4) .. +3 of key 4g + s/4
  const int vkey = 4 * g + (s >> 2);
  const int voff = 256 * vkey + 16 * (((s >> 1) & 1) ^ sa_swz(vkey)) + 8 * (s & 1);  // ^ 32 dt

  float m_run[kRows];  // running max of this lane's head's scaled scores
  float l_run[kRows];  // sum of exp2 against it over this lane's keys
  f32x4 o[kRows][8];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    m_run[i] = -3.402823466e38f;
    l_run[i] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) o[i][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  bf16x8 kf[2][4];   // K of the half: tile u, chunk step cc
  i16x4 vf[8][2];    // V^T of the half: 16-dim tile dt, key tile u
  auto read = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
      for (int u = 0; u < 2; ++u) kf[u][cc] = *reinterpret_cast<const bf16x8*>(slot + koff[cc] + 4096 * u);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        vf[dt][u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (sa_lds_i16x4*)(sa_lds_void)(slot + (voff ^ (32 * dt)) + kSaHalfBytes + 4096 * u));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  // `ok`: the half's attended keys, bit 16r + 4u + g for key 4g + r of tile u.
  auto compute_row = [&](auto row, uint64_t ok) __attribute__((always_inline)) {
    constexpr int kR = row.value;
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int cc = 0; cc < 4; ++cc)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[u][cc], qf[kR][cc], acc[u], 0, 0, 0);
    float x[8] = {acc[0].x, acc[0].y, acc[0].z, acc[0].w, acc[1].x, acc[1].y, acc[1].z, acc[1].w};
    const bool whole = ok == 0x00FF00FF00FF00FFull;  // wave-uniform
    const uint64_t mine = ok >> g;
    auto attended = [&](int i) { return ((mine >> (16 * (i & 3) + 4 * (i >> 2))) & 1) != 0; };
    if (!whole) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = attended(i) ? x[i] : -INFINITY;
    }
    float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
    mx = sa_max_x32(sa_max_x16(mx)) * c;
    if (__ballot(mx > m_run[kR] + kSaRescale) != 0) {
      const float m_new = fmaxf(m_run[kR], mx);
      const float alpha = __builtin_amdgcn_exp2f(m_run[kR] - m_new);  // 0 the first time
      l_run[kR] *= alpha;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        o[kR][dt].x *= alpha;
        o[kR][dt].y *= alpha;
        o[kR][dt].z *= alpha;
        o[kR][dt].w *= alpha;
      }
      m_run[kR] = m_new;
    }
    float p[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = __builtin_amdgcn_exp2f(fmaf(x[i], c, -m_run[kR]));
    if (!whole) {  // by the mask: a scale of zero times -inf is no -inf
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = attended(i) ? p[i] : 0.f;
    }
    l_run[kR] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    // P^T as two bf16 terms: hi = P truncated to bf16, lo = the exact residual
    // P - hi truncated to bf16, so hi + lo carries P to about 2^-15 (one bf16
    // P alone, 2^-9, left the numerator off the fp32 sum l_run[kR] by up to 0.2 %
    // of the attended values' magnitude).  A byte permute packs two values'
    // upper halves into one dword.
    uint32_t hi[8], lo[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      hi[i] = __float_as_uint(p[i]);
      lo[i] = __float_as_uint(p[i] - __uint_as_float(hi[i] & 0xffff0000u));
    }
    u32x4 ph, pl;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ph[i] = __builtin_amdgcn_perm(hi[2 * i + 1], hi[2 * i], 0x07060302u);
      pl[i] = __builtin_amdgcn_perm(lo[2 * i + 1], lo[2 * i], 0x07060302u);
    }
    // O^T += V^T P^T, one 16-dim tile at a time
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      o[kR][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, __builtin_shufflevector(vf[dt][0], vf[dt][1], 0, 1, 2, 3, 4, 5, 6, 7)),
          __builtin_bit_cast(bf16x8, ph), o[kR][dt], 0, 0, 0);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
      o[kR][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, __builtin_shufflevector(vf[dt][0], vf[dt][1], 0, 1, 2, 3, 4, 5, 6, 7)),
          __builtin_bit_cast(bf16x8, pl), o[kR][dt], 0, 0, 0);
  };
  uint32_t seen = 0;  // the rows that attended a key (wave-uniform)
  auto compute = [&](uint64_t ok, uint32_t who) __attribute__((always_inline)) {
    if (ok == 0) return;
    seen |= who;
    if (kRows == 1 || (who & 1)) compute_row(std::integral_constant<int, 0>{}, ok);
    if constexpr (kRows == 2) {
      if (who & 2) compute_row(std::integral_constant<int, 1>{}, ok);
    }
  };

  SaBlock b0 = pop();
  if (b0.rows != 0) {
    SaMem mem;
    mem.kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.kc), 0, a.records, 0x00020000);
    mem.vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(a.vc), 0, a.records, 0x00020000);
    const uint32_t slot_at = sa_lds_at(slot);
    const uint32_t tab_at = sa_lds_at(tabs);
    const int32_t* const tab = reinterpret_cast<const int32_t*>(tabs) + lane;
    constexpr uint64_t kHalfMask = 0x00FF00FF00FF00FFull;
    SaBlock b1 = pop();
    sa_table<kTable>(a, b0, tab_at);
    sa_table<kTable>(a, b1, tab_at + kSaTabBytes);
    sa_wait<1>();
    SaRowAt<kWide> at = sa_rows<kTable, kWide>(a, b0, h, tab[0]);
    sa_fetch<0>(mem, at, col, slot_at);
    int par = 1;  // the table slot of block b1
    while (true) {
      const uint64_t ok = at.ok;
      const uint32_t who = b0.rows;
      const SaBlock b2 = pop();
      sa_wait<0>();  // this half, and block b1's entries
      read();
      sa_fetch<1>(mem, at, col, slot_at);
      if (b1.rows != 0) at = sa_rows<kTable, kWide>(a, b1, h, tab[64 * par]);
      sa_table<kTable>(a, b2, tab_at + kSaTabBytes * (par ^ 1));
      compute(ok & kHalfMask, who);
      sa_wait<1>();  // this half; block b2's entries may still be on their way
      read();
      if (b1.rows != 0) sa_fetch<0>(mem, at, col, slot_at);
      compute((ok >> 8) & kHalfMask, who);
      if (b1.rows == 0) break;
      b0 = b1;
      b1 = b2;
      par ^= 1;
    }
    sa_wait<0>();  // no load may still write LDS when it is released or reused
  }

  OutT* const orow = static_cast<OutT*>(a.out) +
                     (static_cast<int64_t>(t) * a.Hkv * kSaG + kSaG * h + s) * kSaD + 4 * g;
  if constexpr (kSplit == 1) {
    // normalise and store: lane (head n, g) holds dims 16dt + 4g + r
#pragma unroll
    for (int i = 0; i < kRows; ++i) {
      if (i >= rows) break;
      const float l_tot = sa_sum_x32(sa_sum_x16(l_run[i]));
      const float inv = l_tot > 0.f ? 1.f / l_tot : ((seen >> i) & 1) ? NAN : 0.f;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt)
        sa_store4<OutT>(orow + i * static_cast<int64_t>(a.Hkv) * kSaG * kSaD + 16 * dt, o[i][dt] * inv);
    }
  } else {
    const float l_tot = sa_sum_x32(sa_sum_x16(l_run[0]));
    // Each wave leaves (max, sum) per head and its O^T in its slot -- a max of
    // -inf when it attended nothing; then wave w combines dim tiles w,
    // w + kSplit, ... of all of them.
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<f32x4*>(slot + 1024 * dt + 16 * lane) = o[0][dt];
    if (g == 0)
      *reinterpret_cast<float2*>(slot + 8192 + 8 * s) = make_float2(seen != 0 ? m_run[0] : -INFINITY, l_tot);
    __syncthreads();
    float m[kSplit], l = 0.f, top = -3.402823466e38f;
    bool any = false;
#pragma unroll
    for (int w = 0; w < kSplit; ++w) {
      const float2 ml = *reinterpret_cast<const float2*>(lds + w * kSaWaveLds + 8192 + 8 * s);
      m[w] = ml.x;
      any |= ml.x != -INFINITY;
      top = fmaxf(top, ml.x);
    }
#pragma unroll
    for (int w = 0; w < kSplit; ++w) {
      m[w] = __builtin_amdgcn_exp2f(m[w] - top);
      l += m[w] * (*reinterpret_cast<const float2*>(lds + w * kSaWaveLds + 8192 + 8 * s)).y;
    }
    const float inv = l > 0.f ? 1.f / l : any ? NAN : 0.f;
    for (int dt = wave; dt < 8; dt += kSplit) {
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < kSplit; ++w)
        v += *reinterpret_cast<const f32x4*>(lds + w * kSaWaveLds + 1024 * dt + 16 * lane) * m[w];
      sa_store4<OutT>(orow + 16 * dt, v * inv);
    }
  }
}

// Calibration of the gather rate (a measurement tool, not part of the
// attention): the same live stages, table entries and row checks, with every
// attended K and V row read once, coalesced -- lane l = 16r + s reads the
// 16-byte chunk s of the rows of keys 4r + i (i < 4), so 16 lanes read one
// 256-byte row -- kRing stages in flight, and no arithmetic but an XOR of
// the gathered words into a checksum, written per (t, h, lane) to a u32
// [T, Hkv, 64] output.  Its time is what moving every block for every token
// costs a selection; the attention kernel moves a block that two neighbouring
// tokens share once, and runs below it where selections overlap (neighbours
// 24 % alike: this 1122 us, the attention 705 us).
struct SaRows {
  i32x4 k[4];
  i32x4 v[4];
};

// Table entries of keys 4r + i of stage sg (r = lane/16).
template <bool kTable>
__device__ __forceinline__ void sa_co_table(const SaArgs& a, const SaSel& sel, int sg, int32_t (&tv)[4]) {
  const int lane = threadIdx.x & (kWave - 1);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int o = 4 * (lane >> 4) + i;  // entry of the quarter
    const int32_t* p;
    if (sg < 0) {
      p = reinterpret_cast<const int32_t*>(sa_zero_row);
    } else if constexpr (kTable) {
      p = sel.tab + 16 * sg + o;
    } else {
      const int32_t id = __builtin_amdgcn_readlane(sel.lane_id, sg >> 2);
      int32_t pc = static_cast<int32_t>(static_cast<uint32_t>(id) * 64u + static_cast<uint32_t>(16 * (sg & 3) + o));
      pc = pc < 0 ? 0 : (pc > a.L - 1 ? a.L - 1 : pc);
      p = sel.tab + pc;
    }
    tv[i] = *p;
  }
}

template <bool kTable>
__device__ __forceinline__ void sa_co_issue(const SaArgs& a, const SaSel& sel, int sg,
                                            const int32_t (&tv)[4], SaRows& st) {
  const int lane = threadIdx.x & (kWave - 1);
  const uint64_t col = static_cast<uint64_t>(16 * (lane & 15));
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int32_t row = -1;
    if (sg >= 0) {
      const int32_t id = __builtin_amdgcn_readlane(sel.lane_id, sg >> 2);
      const int32_t p = static_cast<int32_t>(static_cast<uint32_t>(id) * 64u +
                                             static_cast<uint32_t>(16 * (sg & 3) + 4 * (lane >> 4) + i));
      const int32_t r = kTable ? tv[i]
                               : static_cast<int32_t>(static_cast<uint32_t>(a.Hkv) * static_cast<uint32_t>(tv[i]) +
                                                      static_cast<uint32_t>(sel.h));
      row = p < sel.lim && r >= 0 && r < a.n_rows ? r : -1;
    }
    const char *kp, *vp;
    if (row >= 0) {
      const uint64_t off = static_cast<uint64_t>(row) * static_cast<uint64_t>(a.row_bytes) + col;
      kp = a.kc + off;
      vp = a.vc + off;
    } else {
      kp = vp = reinterpret_cast<const char*>(sa_zero_row) + col;
    }
    st.k[i] = *reinterpret_cast<const i32x4*>(kp);
    st.v[i] = *reinterpret_cast<const i32x4*>(vp);
  }
}

template <bool kTable, int kRing>
__global__ __launch_bounds__(kWave) void sparse_gather_kernel(SaArgs a) {
  const int lane = threadIdx.x;
  const int t = blockIdx.x, h = blockIdx.y;
  const SaSel sel = sa_select<kTable>(a, t, h);
  asm volatile("" : : "v"(sel.lane_id));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  SaStages stages = sa_live(sel);
  uint32_t x = 0;
  SaRows r[kRing];
  int sr[kRing], st[kRing];
  int32_t tv[kRing][4];
#pragma unroll
  for (int j = 0; j < kRing; ++j) {
    st[j] = sa_pop(stages);
    sa_co_table<kTable>(a, sel, st[j], tv[j]);
  }
#pragma unroll
  for (int j = 0; j < kRing; ++j) {
    sr[j] = st[j];
    sa_co_issue<kTable>(a, sel, sr[j], tv[j], r[j]);
    st[j] = sa_pop(stages);
    sa_co_table<kTable>(a, sel, st[j], tv[j]);
  }
  for (bool more = true; more;) {
#pragma unroll
    for (int j = 0; j < kRing; ++j) {
      if (more && sr[j] >= 0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const i32x4 kv = r[j].k[i] ^ r[j].v[i];
          x ^= static_cast<uint32_t>(kv.x ^ kv.y ^ kv.z ^ kv.w);
        }
        sr[j] = st[j];
        sa_co_issue<kTable>(a, sel, sr[j], tv[j], r[j]);
        st[j] = sa_pop(stages);
        sa_co_table<kTable>(a, sel, st[j], tv[j]);
      } else {
        more = false;
      }
    }
  }
  static_cast<uint32_t*>(a.out)[(static_cast<int64_t>(t) * a.Hkv + h) * kWave + lane] = x;
}

}  // namespace
}  // namespace unum

namespace unum {
namespace {

// Validation and argument block shared by the attention entry point and the
// gather calibration (q, out and the scale are set by the caller).
int sa_args(SaArgs& a, const char* op, const void* key_cache, const void* value_cache,
            int64_t kv_row_stride, int64_t n_rows, const int32_t* topk_idx, int64_t topk_stride_h,
            int64_t topk_stride_t, int64_t topk_stride_k, const int32_t* block_table,
            int64_t bt_stride_b, const int32_t* slots, const int32_t* token_to_bs,
            const int32_t* token_pos_in_bs, int64_t pos_numel, const int32_t* seqlen_q,
            int64_t seqlen_numel, int64_t T, int64_t Hkv, int64_t K, int64_t B, int64_t L) {
  UNUM_REQUIRE(K <= kSaMaxBlocks, "%s: at most %d blocks per token (K=%lld)", op, kSaMaxBlocks,
               (long long)K);
  UNUM_REQUIRE(key_cache && value_cache && topk_idx && token_to_bs && token_pos_in_bs && seqlen_q,
               "%s: null pointer", op);
  UNUM_REQUIRE(slots || (block_table && B >= 1 && L >= 1),
               "%s: a block table (B, L >= 1) or a slot table is required", op);
  UNUM_REQUIRE(pos_numel == 1 || pos_numel == T, "%s: token_pos_in_bs has %lld entries (T=%lld)",
               op, (long long)pos_numel, (long long)T);
  UNUM_REQUIRE(seqlen_numel == 1 || seqlen_numel >= B, "%s: seqlen_q has %lld entries (B=%lld)", op,
               (long long)seqlen_numel, (long long)B);
  UNUM_REQUIRE(n_rows >= 0 && kv_row_stride >= kSaD && (kv_row_stride % 8) == 0,
               "%s: cache rows must be D elements or more apart, in multiples of 8 (stride %lld)",
               op, (long long)kv_row_stride);
  UNUM_REQUIRE((reinterpret_cast<uintptr_t>(key_cache) & 15) == 0 &&
                   (reinterpret_cast<uintptr_t>(value_cache) & 15) == 0,
               "%s: the caches must be 16-byte aligned", op);
  UNUM_REQUIRE(T <= INT32_MAX && Hkv <= 65535 && n_rows <= INT32_MAX && B <= INT32_MAX &&
                   L <= INT32_MAX,
               "%s: size exceeds the kernel's index range", op);
  a.kc = static_cast<const char*>(key_cache);
  a.vc = static_cast<const char*>(value_cache);
  a.row_bytes = kv_row_stride * 2;
  a.n_rows = n_rows;
  a.idx = topk_idx;
  a.i_sh = topk_stride_h;
  a.i_st = topk_stride_t;
  a.i_sk = topk_stride_k;
  a.bt = block_table;
  a.bt_sb = bt_stride_b;
  a.slots = slots;
  a.tok_bs = token_to_bs;
  a.pos = token_pos_in_bs;
  a.slen = seqlen_q;
  a.pos_n = static_cast<int32_t>(pos_numel);
  a.slen_n = static_cast<int32_t>(seqlen_numel == 1 ? 1 : 2);
  a.T = static_cast<int32_t>(T);
  a.Hkv = static_cast<int32_t>(Hkv);
  a.K = static_cast<int32_t>(K);
  a.B = static_cast<int32_t>(B);
  a.L = static_cast<int32_t>(L);
  return UNUM_OK;
}

}  // namespace
}  // namespace unum

extern "C" int unum_sparse_paged_attention(
    const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* key_cache,
    const void* value_cache, int64_t kv_row_stride, int64_t n_rows, const int32_t* topk_idx,
    int64_t topk_stride_h, int64_t topk_stride_t, int64_t topk_stride_k,
    const int32_t* block_table, int64_t bt_stride_b, const int32_t* slots,
    const int32_t* token_to_bs, const int32_t* token_pos_in_bs, int64_t pos_numel,
    const int32_t* seqlen_q, int64_t seqlen_numel, void* out, int32_t out_dtype, int64_t T,
    int64_t Hq, int64_t Hkv, int64_t D, int64_t K, int64_t B, int64_t L, float scale,
    void* stream) {
  using namespace unum;
  clear_error();
  const char* op = "sparse_paged_attention";
  UNUM_REQUIRE(T >= 0 && Hq > 0 && Hkv > 0 && D > 0 && K >= 0 && B >= 0 && L >= 0,
               "%s: bad sizes (T=%lld Hq=%lld Hkv=%lld D=%lld K=%lld B=%lld L=%lld)", op,
               (long long)T, (long long)Hq, (long long)Hkv, (long long)D, (long long)K,
               (long long)B, (long long)L);
  if (T == 0) return UNUM_OK;
  if (Hq != kSaG * Hkv || D != kSaD)
    UNUM_FAIL(UNUM_ERR_UNSUPPORTED, "%s: needs 16 query heads per kv head and D = 128 (got Hq=%lld, "
              "Hkv=%lld, D=%lld)", op, (long long)Hq, (long long)Hkv, (long long)D);
  UNUM_REQUIRE(q && out, "%s: null pointer", op);
  UNUM_REQUIRE((reinterpret_cast<uintptr_t>(q) & 15) == 0 && (q_stride_t % 8) == 0 &&
                   (q_stride_h % 8) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0,
               "%s: q and out must be 16-byte aligned (q strides multiples of 8)", op);
  UNUM_REQUIRE(out_dtype == UNUM_DTYPE_BF16 || out_dtype == UNUM_DTYPE_F32,
               "%s: unsupported out dtype %d", op, out_dtype);
  SaArgs a{};
  const int st = sa_args(a, op, key_cache, value_cache, kv_row_stride, n_rows, topk_idx,
                         topk_stride_h, topk_stride_t, topk_stride_k, block_table, bt_stride_b,
                         slots, token_to_bs, token_pos_in_bs, pos_numel, seqlen_q, seqlen_numel,
                         T, Hkv, K, B, L);
  if (st != UNUM_OK) return st;
  a.q = static_cast<const __bf16*>(q);
  a.q_st = q_stride_t;
  a.q_sh = q_stride_h;
  a.out = out;
  a.c = scale * kSaLog2e;
  const int64_t bytes = n_rows > 0 ? (n_rows - 1) * a.row_bytes + 2 * kSaD : 0;
  const bool wide = bytes > static_cast<int64_t>(kSaNoRow);
  a.records = wide ? 0u : static_cast<uint32_t>(bytes);
  const int64_t rows = T * Hkv;
  // Whole rows, one a wave, need four waves a SIMD's worth of them and rows
  // that are alike; else four waves share a row.  Measured, whole / shared:
  // 64 sequences x 1 token 96 / 49 us, x 8 tokens 231 / 202, x 16 tokens
  // 420 / 318 (fewer rows at once keep a sequence's blocks in the L2); one
  // sequence x 512 tokens 105 / 103, x 1024 193 / 205, x 2048 363 / 403.  At
  // most one token a sequence, no row meets another's blocks in the L2 and
  // sharing a row only costs its combination: 512 sequences x 2 blocks
  // 15.6 / 18.2, x 64 blocks 358 / 366; 2048 x 2 blocks 50.6 / 59.9.  (B, the
  // table's rows, stands for the sequences of the batch: they are counted on
  // the device only.)
  const bool whole = rows >= 1024 && (T >= 64 * B || T <= B);
  // Two rows a wave where that still fills the chip (eight waves a CU).
  // Measured, one row a wave / two, neighbours' selections 6, 24 and 67 %
  // alike: 4096 tokens of 2 heads 1738 / 1564, 925 / 722 and 664 / 564 us,
  // 2048 tokens 687 / 573, 373 / 344 and 344 / 284, 1024 tokens (a wave a
  // SIMD) 322 / 299, 192 / 208 and 173 / 184.
  const bool pairs = whole && T > B && !slots && rows >= 4096;
  const int64_t units = pairs ? (T + 1) / 2 : T;  // workgroups of a head
  a.gshift = 0;
  while (a.gshift < 4 && ((units * Hkv) >> a.gshift) >= 128) ++a.gshift;
  const int64_t groups = ((units + (int64_t{1} << a.gshift) - 1) >> a.gshift) * Hkv;
  const int64_t wgs = ((groups + 7) / 8) << (a.gshift + 3);
  UNUM_REQUIRE(wgs <= INT32_MAX, "%s: size exceeds the kernel's index range (%lld tokens x %lld kv heads)",
               op, (long long)T, (long long)Hkv);
  constexpr int64_t kGridRow = int64_t{1} << kSaGridShift;
  const dim3 grid(static_cast<unsigned>(wgs < kGridRow ? wgs : kGridRow),
                  static_cast<unsigned>((wgs + kGridRow - 1) / kGridRow));
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto launch = [&](auto o, auto tab, auto w) {
    using OutT = decltype(o);
    if (pairs)  // never with a slot table
      hipLaunchKernelGGL((sparse_attn_kernel<OutT, false, w.value, 1, 2>), grid, dim3(kWave), 0, s, a);
    else if (whole)
      hipLaunchKernelGGL((sparse_attn_kernel<OutT, tab.value, w.value, 1, 1>), grid, dim3(kWave), 0, s, a);
    else
      hipLaunchKernelGGL((sparse_attn_kernel<OutT, tab.value, w.value, kSaSplit, 1>), grid, dim3(kWave * kSaSplit), 0,
                         s, a);
  };
  auto by_table = [&](auto o, auto w) {
    if (slots)
      launch(o, std::true_type{}, w);
    else
      launch(o, std::false_type{}, w);
  };
  auto by_width = [&](auto o) {
    if (wide)
      by_table(o, std::true_type{});
    else
      by_table(o, std::false_type{});
  };
  if (out_dtype == UNUM_DTYPE_BF16)
    by_width(uint16_t{});
  else
    by_width(float{});
  return check_launch(op);
}

extern "C" int unum_sparse_gather_calibrate(
    const void* key_cache, const void* value_cache, int64_t kv_row_stride, int64_t n_rows,
    const int32_t* topk_idx, int64_t topk_stride_h, int64_t topk_stride_t, int64_t topk_stride_k,
    const int32_t* block_table, int64_t bt_stride_b, const int32_t* slots,
    const int32_t* token_to_bs, const int32_t* token_pos_in_bs, int64_t pos_numel,
    const int32_t* seqlen_q, int64_t seqlen_numel, uint32_t* out, int64_t T, int64_t Hkv,
    int64_t K, int64_t B, int64_t L, void* stream) {
  using namespace unum;
  clear_error();
  const char* op = "sparse_gather_calibrate";
  UNUM_REQUIRE(T >= 0 && Hkv > 0 && K >= 0 && B >= 0 && L >= 0,
               "%s: bad sizes (T=%lld Hkv=%lld K=%lld B=%lld L=%lld)", op, (long long)T,
               (long long)Hkv, (long long)K, (long long)B, (long long)L);
  if (T == 0) return UNUM_OK;
  UNUM_REQUIRE(out, "%s: null pointer", op);
  SaArgs a{};
  const int st = sa_args(a, op, key_cache, value_cache, kv_row_stride, n_rows, topk_idx,
                         topk_stride_h, topk_stride_t, topk_stride_k, block_table, bt_stride_b,
                         slots, token_to_bs, token_pos_in_bs, pos_numel, seqlen_q, seqlen_numel,
                         T, Hkv, K, B, L);
  if (st != UNUM_OK) return st;
  a.out = out;
  const dim3 grid(static_cast<unsigned>(T), static_cast<unsigned>(Hkv));
  hipStream_t s = static_cast<hipStream_t>(stream);
  // eight waves per CU, as the attention kernel
  if (slots)
    hipLaunchKernelGGL((sparse_gather_kernel<true, kSaRing>), grid, dim3(kWave), kSaLdsBytes, s, a);
  else
    hipLaunchKernelGGL((sparse_gather_kernel<false, kSaRing>), grid, dim3(kWave), kSaLdsBytes, s, a);
  return check_launch(op);
}
