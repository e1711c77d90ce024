// Split-KV decode kernels for gfx950: one new query token per sequence over
// padded (left or right), unpadded, packed or paged K/V, bf16 / fp16 (paged
// pools also fp8), head_dim a multiple of 8 up to 256, 64 x 64 tiles,
// grouped-query attention with all q heads of a kv head sharing the
// look-up-table row.  The step is HBM-bound (every attended K/V byte is read
// exactly once, for all q heads of the group together), so the design goal is
// bytes in flight, not FLOPs:
//
//   work unit = one wave = consecutive half blocks (32 keys) of the row of (sequence, kv
//               head); the number of units of a row and the even split of its half
//               blocks follow from its length on the device, so waves stream
//               similar amounts of K/V whatever the sequence lengths are;
//   workgroup = kDecodeWaves consecutive units of one row (workgroups beyond a
//               row's unit count exit at once; a row that needs several
//               workgroups is cut into a whole number of them, so that none
//               holds LDS and wave slots for idle waves);
//   wave      = per half block: computes S^T = K Q^T (the q heads of the group are the MFMA
//               columns), softmax, O^T += V^T P^T with LDS transpose reads,
//               keeping a running (max, sum, O) in registers;
//   epilogue  = the waves of a workgroup merge their results through LDS.  A row
//               whose units all sit in one workgroup is written as O / LSE;
//               otherwise the workgroup leaves one fp32 partial (O unnormalised,
//               max, sum) per q head in the caller's workspace, and the workgroup
//               that arrives last merges the row's partials (arrive_last).
// A wave works on half blocks (32 keys): 2 x 8.5 KB of private LDS tiles and
// the next half block prefetched into registers, so 8 waves are resident per
// CU (2 per SIMD, <= 256 VGPRs each): one wave's loads overlap the other's
// multiplies on the same SIMD.  (Head dims above 128: 256-wide tiles, 2 x 33 KB per wave, one
// workgroup of four waves per CU and one wave per SIMD.)
#include <algorithm>
#include <atomic>
#include <chrono>
#include <type_traits>

#include "common.h"
#include "device_common.h"
#include "mfma_common.h"

namespace dk {

constexpr int kDecodeWaves = 4;  // units (waves) per workgroup

// Upper bound on the entries of one table row: the caller's hint when given,
// else the number of column blocks.
static int decode_max_row_entries(const FwdParams &p) {
  return p.csr.max_row_entries > 0 ? p.csr.max_row_entries : p.csr.num_rows;
}

// Half blocks (32 keys) per work unit (one wave).  With enough rows (sequences x kv heads) to fill the
// machine, a row is cut into as many units as a workgroup has waves, so that it is finished
// inside one workgroup; with few rows, into more units (about 1024 waves in total, down to a half block
// each: the reads of a wave then leave in one round).  At most 16 blocks (the paged path keeps a
// unit's page numbers in the lanes of one register).  Measured: 1 sequence of 1000 keys (8 kv heads of
// 16 blocks), 64 workgroups of half blocks, 8 us from the first workgroup's start to the last one's
// end (4.3 us to the last key, 1 us merge inside the workgroups, 0.8 us to publish and count, 1.5 us last
// merge), against 12 us + 4 us for units of two blocks and a merge kernel; 32 sequences (256 rows):
// 1024 waves 38.6 us, 1536 42.1, 2048 41.2, 3072 45.5.
static int decode_unit_halves(const FwdParams &p) {
  const int rows = p.seqs.batch * p.Hkv;
  const int units_per_row = std::max(kDecodeWaves, cdiv(1024, rows > 0 ? rows : 1));
  return std::min(32, std::max(1, cdiv(2 * decode_max_row_entries(p), units_per_row)));
}

// Units a row of n half blocks is cut into: as many as the unit size asks for, and at least
// the waves of one workgroup (one half block each at worst), so that every wave of the workgroup that
// finishes a row streams a share of it.  A row that needs more than one workgroup gets a whole
// number of them: a workgroup with a single busy wave would hold the LDS and the wave slots of
// four.
__host__ __device__ inline int decode_row_units(int n, int unit_halves, int waves) {
  const int by_size = (n + unit_halves - 1) / unit_halves;
  const int by_waves = n < waves ? n : waves;
  const int units = by_size > by_waves ? by_size : by_waves;
  return units > waves ? (units + waves - 1) / waves * waves : units;
}

// Which workgroup of a row arrives last is counted in a slot of the caller's workspace that nobody has
// cleared.  A slot in use holds (launch number, arrivals); every workgroup first makes sure of that
// (open_slot: it replaces whatever else it read there, and if that fails another workgroup has done
// so), long before it arrives.  Launch numbers are 56 bits from a random start, so what the memory
// happens to hold is not taken for one; the workgroup that arrives last clears the slot, so that a
// captured launch, whose number is the same on every replay, starts afresh each time.  Arriving is
// then one atomic addition (as a compare-and-swap loop, eight workgroups took 3 - 6 us), and nobody
// ever waits for another workgroup.
//
// The addition releases the workgroup's partial (which its waves have written and waited for ahead of
// a barrier) and acquires those of the workgroups that arrived before: the chain of additions orders
// every partial before the reads of the last one, on whichever die it sits.  A step over one sequence
// of 1000 keys: 7.9 us, 7.8 without the ordering; 8.6 with one more acquire in each of the last
// workgroup's waves, which the barrier behind the addition makes redundant.
using slot_t = unsigned long long;
__device__ __forceinline__ void open_slot(slot_t *slot, slot_t seen, slot_t launch) {
  if ((seen >> 8) != launch)
    __hip_atomic_compare_exchange_strong(slot, &seen, launch << 8, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool arrive_last(slot_t *slot, int n) {
  const slot_t before = __hip_atomic_fetch_add(slot, 1, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
  if ((int)(before & 255) + 1 != n) return false;
  __hip_atomic_store(slot, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

template <int D>
struct DecSmem {  // per wave: one 32-key half block of K and of V, plus q of the group
  static constexpr int kStride = D * 2 + 16;   // bytes per row
  static constexpr int kHalf = 32 * kStride;   // one half-block tile
  // followed by q of the group's heads, row-major: ratio * D * 2 bytes
  static int wave_bytes(int ratio) { return 2 * kHalf + ratio * D * 2; }
};

// workspace layout, where rows are cut over several workgroups: [batch][Hq][max_groups + 1][D + 2] floats,
// a partial (O[D] unnormalised, max, sum) per workgroup of the row; the last place of a kv group's first
// head holds the row's arrival slot

// Eight OCP e4m3 bytes -> eight elements of T.  Exact (e4m3 has 3 mantissa bits), so bf16 is
// the upper half of the fp32 value and fp16 needs no rounding mode: one convert and one pack per
// two elements.
template <typename T>
__device__ __forceinline__ uint32_t pack2_exact(float a, float b);
template <>
__device__ __forceinline__ uint32_t pack2_exact<bf16_t>(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);  // hi16(b) : hi16(a)
}
template <>
__device__ __forceinline__ uint32_t pack2_exact<f16_t>(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(a, b));
}
template <typename T>
__device__ __forceinline__ uint4 fp8x8_to(uint2 w) {
  typedef float float2_ __attribute__((ext_vector_type(2)));
  const float2_ a = __builtin_amdgcn_cvt_pk_f32_fp8((int)w.x, false), b = __builtin_amdgcn_cvt_pk_f32_fp8((int)w.x, true);
  const float2_ c = __builtin_amdgcn_cvt_pk_f32_fp8((int)w.y, false), d = __builtin_amdgcn_cvt_pk_f32_fp8((int)w.y, true);
  return make_uint4(pack2_exact<T>(a[0], a[1]), pack2_exact<T>(b[0], b[1]), pack2_exact<T>(c[0], c[1]),
                    pack2_exact<T>(d[0], d[1]));
}

// Sequence that the workgroups of grid.z = place take when the sequences are handed out by length: the `first` longest
// ones in ascending order, then the others in descending order (lengths to within a 32nd of the longest one or finer;
// equal ones in the batch's order).  At most kRankedSequences sequences, all lanes active.  Every lane loads the geometry
// of its sequences, so the lengths cost no round trip beyond the workgroup's own; the length at a rank is found bit by bit
// from the lanes' votes (64 keys to a block: six votes, 0.3 us of a step).
constexpr int kRankedSequences = 128;
__device__ __forceinline__ SeqInfo sequence_by_length(const SeqView &s, int place, int first, int causal) {
  const int rank = place < first ? first - 1 - place : place;
  const int lane = threadIdx.x & 63;
  const bool two = s.batch > 64;  // sequences a lane
  const SeqInfo lo = load_seq_lane(s, min(lane, s.batch - 1), causal);
  SeqInfo hi = lo;
  if (two) hi = load_seq_lane(s, min(lane + 64, s.batch - 1), causal);
  // length bits that are left out: six remain (of the longest sequence that is there: the extent of the key dimension is the
  // capacity of a cache or block table, or the tokens of all packed sequences together)
  const int drop = max(0, 26 - __clz(wave_max(max(lo.k_len, hi.k_len)) | 1));
  auto key = [&](const SeqInfo &t, int i) { return i < s.batch ? (t.q_len > 0 ? t.k_len >> drop : 0) : -1; };
  const int key_lo = key(lo, lane), key_hi = key(hi, lane + 64);
  auto votes = [&](int at) { return __popcll(__ballot(key_lo >= at)) + (two ? __popcll(__ballot(key_hi >= at)) : 0); };
  int len = 0;  // largest length that more than `rank` sequences reach
  for (int at = 32; at > 0; at >>= 1)
    if (votes(len + at) > rank) len += at;
  int n = rank - votes(len + 1);  // among those of that length
  const unsigned long long same_lo = __ballot(key_lo == len), same_hi = __ballot(key_hi == len);
  const bool upper = n >= __popcll(same_lo);
  if (upper) n -= __popcll(same_lo);
  const unsigned long long same = upper ? same_hi : same_lo, below = (1ull << lane) - 1;
  const int owner = __ffsll(__ballot(((same >> lane) & 1) && __popcll(same & below) == n)) - 1;
  auto from_owner = [&](int a, int b) { return __builtin_amdgcn_readlane(upper ? b : a, owner); };
  SeqInfo r;
  r.b = owner + (upper ? 64 : 0);
  r.q_start = from_owner(lo.q_start, hi.q_start), r.q_len = from_owner(lo.q_len, hi.q_len);
  r.k_start = from_owner(lo.k_start, hi.k_start), r.k_len = from_owner(lo.k_len, hi.k_len);
  r.past = from_owner(lo.past, hi.past);
  return r;
}

// KV8 (with PAGED): the K/V pools hold fp8 bytes, converted to T on the way into LDS.
// W waves per workgroup = W consecutive units of one row.
// BY_LENGTH: sequences handed out by length (decode_first_by_length); an instantiation of its own, as the code alone, jumped
// over, cost the smallest steps 0.15 of 8 us.
template <typename T, int D, bool PAD, bool SUB, bool PAGED, bool KV8, int W, bool BY_LENGTH>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2, D == 256 ? 1 : 2))) void decode_partial_kernel(
    const FwdParams p, float *ws, int unit_halves, int max_groups, slot_t launch, int first_by_length) {
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  using S = DecSmem<D>;
  constexpr int KS = D / 16, DT = D / 32, CPR = D / 8;
  // SUB: table entries are (column, bit mask over the pattern blocks inside the 64 x 64 tile)
  constexpr int EW = SUB ? 2 : 1;  // ints per table entry
  extern __shared__ __align__(16) char smem_all[];

  const int kvh = blockIdx.y;
  SeqInfo sq;
  if constexpr (BY_LENGTH)
    sq = sequence_by_length(p.seqs, blockIdx.z, first_by_length, p.causal);
  else
    sq = load_seq(p.seqs, blockIdx.z, p.causal);
  const int b = sq.b;
  if (sq.q_len <= 0) return;
  const int ratio = __builtin_amdgcn_readfirstlane(p.Hq / p.Hkv);  // integer division runs on the VALU
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wave_bytes = 2 * S::kHalf + ratio * D * 2;
  char *smem = smem_all + wave * wave_bytes;  // this wave's private tiles and q copy
  const int m = lane & 31, g = lane >> 5;  // m = q head inside the group (MFMA column)
  const int pos = sq.past;                 // absolute position of the single query token
  const int rb = pos / 64;
  const int h0 = kvh * ratio;
  const int lh = lut_head(p.csr, h0, p.Hq, p.Hkv);
  // table reads go through the scalar unit (wave-uniform addresses, no vector-memory wait)
  int row0 = 0, row1 = 0;
  if (sq.k_len > 0 && rb < p.csr.num_rows)
    scalar_load2(p.csr.ptr + lh * p.csr.ptr_sh + rb, p.csr.ptr + lh * p.csr.ptr_sh + rb + 1, row0, row1);
  // the row's half blocks are split evenly over as many units as the unit size asks for
  const int n_half = 2 * (row1 - row0);
  // never more than the host sized the grid and the workspace for: a row longer than the caller's
  // max_row_entries hint said is still cut into max_groups * W units, each with a larger share
  const int u_cnt = min(decode_row_units(n_half, unit_halves, W), max_groups * W);
  if ((int)blockIdx.x * W >= u_cnt && blockIdx.x > 0) return;  // nothing for this workgroup
  const int groups = (u_cnt + W - 1) / W;  // workgroups of this row (a row without entries is written too: O = 0, LSE = -inf)
  const int per = u_cnt > 0 ? (n_half + u_cnt - 1) / u_cnt : 0;
  const int unit = blockIdx.x * W + wave;
  const int hb0 = min(unit * per, n_half), hb1 = min(hb0 + per, n_half);  // (units beyond u_cnt: empty)
  const int e0 = row0 + (hb0 >> 1);  // table entry of the first half block
  const int e1 = row0 + ((hb1 + 1) >> 1);
  const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
  // SUB: the query's row of pattern blocks inside its tile selects f of the entry's f x f mask
  // bits; half block hb & 1 holds key parts [hb & 1, hb & 1 + 1) * f / 2 of them
  const int lb = SUB ? (p.csr.sub_block == 16 ? 4 : 5) : 6, f = 64 >> lb;
  const int row_shift = ((pos & 63) >> lb) * f;
  auto half_bits = [&](int bits, int hb) { return (bits >> (row_shift + (hb & 1) * (f >> 1))) & ((1 << (f >> 1)) - 1); };
  // contiguous K/V: the sequence's first key; paged K/V: the pools (pages are added per half block)
  static_assert(!KV8 || PAGED, "fp8 K/V comes through the paged entry");
  using KV = typename std::conditional<KV8, uint8_t, T>::type;  // element type of the K/V memory
  const KV *kbase = (const KV *)p.k.ptr + kvh * p.k.sh + (PAGED ? 0 : sq.b * p.k.sb + (int64_t)sq.k_start * p.k.st);
  const KV *vbase = (const KV *)p.v.ptr + kvh * p.v.sh + (PAGED ? 0 : sq.b * p.v.sb + (int64_t)sq.k_start * p.v.st);
  // K/V bytes are read once per step: non-temporal loads keep them from displacing each other in
  // the memory-side cache (measured 44.6 -> 40.5 us per step on 32 sequences of 1K-8K tokens)
  auto load8 = [](const KV *src) -> uint4 {  // 8 head dims starting at src, as T
    if constexpr (KV8) {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      const u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(src));
      return fp8x8_to<T>(make_uint2(w[0], w[1]));
    } else {
      typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src));
      return make_uint4(w[0], w[1], w[2], w[3]);
    }
  };

  // PAGED: page numbers of the whole unit in one vector load, four lanes per table entry (a
  // 64-key block spans at most four pages of >= 16 tokens): lane 4 j + s holds the page of keys
  // [s, s + 1) * page_size of entry e0 + j (pages of >= 64 tokens: s = 0 only).  Entries of the
  // page table beyond the sequence's last token are never read; a negative entry inside the
  // sequence (a caller's mistake: such slots mark unused pages) is read as page 0 rather than
  // as an address before the pool.
  // A unit of more than 16 entries (one of 16 whole blocks that starts at a second half, or any when the
  // caller's max_row_entries hint understated the row) reloads the register every 16 entries.
  int my_page = 0;
  auto load_pages = [&](int j0) {  // pages of entries e0 + j0 .. e0 + j0 + 15
    int pg = 0;
    const int j = j0 + (lane >> 2), s = lane & 3;
    const int ps = 1 << p.paged.page_shift;
    if (j < e1 - e0) {
      const int col = cols[(e0 + j) * EW];
      const int tok = col * 64 + (ps < 64 ? s * ps : 0);
      if (col >= 0 && tok < sq.k_len && (s == 0 || s * ps < 64))
        pg = max(p.paged.table[b * p.paged.table_sb + (tok >> p.paged.page_shift)], 0);
    }
    return pg;
  };
  if constexpr (PAGED) my_page = load_pages(0);

  // half block hb, counted from the first half of entry e0: keys cols[e0 + hb/2] * 64 + 32 * (hb & 1) + [0, 32)
  constexpr int HCH = 32 * CPR / 64;  // 16-byte chunks per lane per half tile
  uint4 kreg[HCH], vreg[HCH];
  auto prefetch = [&](int hb, int col, int bits) {
    const int key0 = col * 64 + (hb & 1) * 32;
    if constexpr (PAGED)
      if (hb > 0 && (hb & 31) == 0) my_page = load_pages(hb >> 1);
    if (SUB && half_bits(bits, hb) == 0) return;  // no attended key in this half: neither read nor used
    // element offset of row r of the half block from kbase / vbase
    int pg_lo = 0, pg_hi = 0, in_page0 = 0;
    if constexpr (PAGED) {
      // the half block's 32 keys lie in one page, or in two pages of 16
      const int psl = p.paged.page_shift, half = hb & 1;
      const int s_lo = psl < 6 ? (half * 32) >> psl : 0, s_hi = psl < 6 ? (half * 32 + 16) >> psl : 0;
      // (lane-indexed reads: the compiler may route the lane number through M0.  Nothing in this
      // file writes M0 behind its back - the LDS DMA helpers of mfma_common.h, which do, are not
      // used by the decode kernels.)
      pg_lo = __builtin_amdgcn_readlane(my_page, (((hb >> 1) & 15) * 4 + s_lo) & 63);
      pg_hi = __builtin_amdgcn_readlane(my_page, (((hb >> 1) & 15) * 4 + s_hi) & 63);
      in_page0 = key0 & ((1 << psl) - 1);
    }
    auto k_off = [&](int r) -> int64_t {
      if constexpr (PAGED) {
        const int in_page = (in_page0 + r) & ((1 << p.paged.page_shift) - 1);
        return (int64_t)(r < 16 ? pg_lo : pg_hi) * p.paged.k_page_stride + (int64_t)in_page * p.k.st;
      } else {
        return (int64_t)(key0 + r) * p.k.st;
      }
    };
    auto v_off = [&](int r) -> int64_t {
      if constexpr (PAGED) {
        const int in_page = (in_page0 + r) & ((1 << p.paged.page_shift) - 1);
        return (int64_t)(r < 16 ? pg_lo : pg_hi) * p.paged.v_page_stride + (int64_t)in_page * p.v.st;
      } else {
        return (int64_t)(key0 + r) * p.v.st;
      }
    };
    if (!PAD && col >= 0 && key0 + 32 <= sq.k_len) {  // whole half inside the sequence: no guards
#pragma unroll
      for (int c = 0; c < HCH; ++c) {
        const int idx = lane + c * 64;
        const int r = idx / CPR, ch = idx % CPR;
        kreg[c] = load8(kbase + k_off(r) + ch * 8);
        vreg[c] = load8(vbase + v_off(r) + ch * 8);
      }
    } else {  // rows beyond the sequence and (PAD) head dims beyond p.D read as zeros
#pragma unroll
      for (int c = 0; c < HCH; ++c) {
        const int idx = lane + c * 64;
        const int r = idx / CPR, ch = idx % CPR;
        kreg[c] = vreg[c] = make_uint4(0, 0, 0, 0);
        if (col >= 0 && key0 + r < sq.k_len && (!PAD || ch * 8 < p.D)) {
          kreg[c] = load8(kbase + k_off(r) + ch * 8);
          vreg[c] = load8(vbase + v_off(r) + ch * 8);
        }
      }
    }
  };
  // the first K/V request goes out before anything else touches memory
  int col_cur = 0, bits_cur = 0;
  const int first = hb0 & 1, nhalf = first + hb1 - hb0;
  if (first < nhalf) {  // (an even split can leave the last units of a row without half blocks: neutral partials)
    if constexpr (SUB)
      scalar_load2(cols + e0 * EW, cols + e0 * EW + 1, col_cur, bits_cur);
    else
      col_cur = scalar_load(cols + e0);
    prefetch(first, col_cur, bits_cur);
  }

  // behind it, for rows of several workgroups, the arrival slot
  slot_t *const slot = reinterpret_cast<slot_t *>(ws + (((int64_t)b * p.Hq + h0 + 1) * (max_groups + 1) - 1) * (D + 2));
  slot_t slot_seen = 0;
  if (groups > 1 && threadIdx.x == 0) slot_seen = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

  // q of the group's heads -> LDS (row min(m, ratio-1) feeds MFMA column m;
  // columns >= ratio are duplicates whose results are never stored)
  char *ks_ = smem, *vs_ = smem + S::kHalf, *qs_ = smem + 2 * S::kHalf;
  {
    const int hh = lane / CPR, ch = lane % CPR;  // 64 lanes cover 64 / CPR heads per pass
    for (int h = hh; h < ratio; h += 64 / CPR) {
      const T *qp = (const T *)p.q.ptr + sq.b * p.q.sb + (int64_t)(h0 + h) * p.q.sh + (int64_t)sq.q_start * p.q.st;
      uint4 w = make_uint4(0, 0, 0, 0);
      if (!PAD || ch * 8 < p.D) w = *reinterpret_cast<const uint4 *>(qp + ch * 8);
      *reinterpret_cast<uint4 *>(qs_ + h * D * 2 + ch * 16) = w;
    }
  }
  if (groups > 1 && threadIdx.x == 0) open_slot(slot, slot_seen, launch);
  const int q_read = (m < ratio ? m : ratio - 1) * D * 2 + g * 16;

  floatx16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const int k_read = m * S::kStride + g * 16;
  const int i16 = lane & 15, dgrp = (lane >> 4) & 1;
  const int v_read = (4 * g + (i16 >> 2)) * S::kStride + (16 * dgrp + 4 * (i16 & 3)) * 2;

  for (int hb = first; hb < nhalf; ++hb) {
    const int col = col_cur;
    const int hbits = SUB ? half_bits(bits_cur, hb) : 1;
    const int key0 = col * 64 + (hb & 1) * 32;
    // table entry of the next half block (the next block after an odd half)
    if ((hb & 1) && hb + 1 < nhalf) {
      const int32_t *ent = cols + (e0 + ((hb + 1) >> 1)) * EW;
      if constexpr (SUB)
        scalar_load2(ent, ent + 1, col_cur, bits_cur);
      else
        col_cur = scalar_load(ent);
    }
    // The tiles are private to this wave and LDS operations of one wave
    // execute in order, so the previous half block's reads are done; only the
    // compiler must not reorder across these points (a memory fence would
    // also drain the global prefetch issued next).
    asm volatile("" ::: "memory");
    if (hbits != 0) {  // (a half without attended keys was not read)
#pragma unroll
      for (int c = 0; c < HCH; ++c) {
        const int idx = lane + c * 64;
        const int r = idx / CPR, ch = idx % CPR;
        *reinterpret_cast<uint4 *>(ks_ + r * S::kStride + ch * 16) = kreg[c];
        *reinterpret_cast<uint4 *>(vs_ + r * S::kStride + ch * 16) = vreg[c];
      }
    }
    asm volatile("" ::: "memory");
    if (hb + 1 < nhalf) prefetch(hb + 1, col_cur, bits_cur);
    if (hbits == 0 || col < 0 || key0 >= sq.k_len || (p.causal && key0 > pos)) continue;

    floatx16 sacc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
    {
      vec8 a[KS], qb[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        a[ks] = lds_read8<vec8>(ks_ + k_read + ks * 32);
        qb[ks] = lds_read8<vec8>(qs_ + q_read + ks * 32);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) sacc = M::mma(a[ks], qb[ks], sacc);
    }
    const bool need_mask = (key0 + 31 >= sq.k_len) || (p.causal && key0 + 31 > pos);
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float sv = sacc[r] * p.scale_log2;
      if constexpr (SUB) {
        // key 8 (r / 4) + 4 g + r % 4 of the half: the last two terms stay inside a part of >= 16 keys
        if (!((hbits >> (((r >> 2) * 8) >> lb)) & 1)) sv = -INFINITY;
      }
      if (need_mask) {
        const int key = key0 + (r >> 2) * 8 + g * 4 + (r & 3);
        if (key >= sq.k_len || (p.causal && key > pos)) sv = -INFINITY;
      }
      sacc[r] = sv;
      mx = fmaxf(mx, sv);
    }
    mx = fmaxf(mx, xor32(mx));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float alpha = fast_exp2(m_run - m_use);
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pv = fast_exp2(sacc[r] - m_use);
      sacc[r] = pv;
      psum += pv;
    }
    psum += xor32(psum);
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float pf[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) pf[i] = sacc[t * 8 + i];
      const vec8 pb = M::pack(pf);
      const char *vrow = vs_ + v_read + t * 16 * S::kStride;
      vec8 a[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) a[dt] = lds_read_tr8<vec8>(vrow + dt * 64, vrow + 8 * S::kStride + dt * 64);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] = M::mma(a[dt], pb, oacc[dt]);
    }
  }

  // ---- result of this unit: lanes (m < ratio) hold head h0 + m ----
  // rows [head][D + 2] floats (O unnormalised, max, sum) in this wave's own tile area (its tiles are
  // dead by now)
  if (m < ratio) {
    float *dst = reinterpret_cast<float *>(smem) + m * (D + 2);
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *reinterpret_cast<float4 *>(dst + dt * 32 + r4 * 8 + g * 4) =
            make_float4(oacc[dt][r4 * 4], oacc[dt][r4 * 4 + 1], oacc[dt][r4 * 4 + 2], oacc[dt][r4 * 4 + 3]);
    if (g == 0) {
      dst[D] = m_run;
      dst[D + 1] = l_run;
    }
  }
  __syncthreads();
  // heads of the group are dealt to the waves; lane l owns dims l D/64 .. of its head
  constexpr int PER = D / 64;
  auto store_row = [&](int h, const float (&o)[PER], float mmax, float l) {
    const float inv = l > 0.f ? (p.paged.table ? p.paged.out_scale : 1.f) / l : 0.f;  // (includes the V scale)
    T *op = (T *)p.o.ptr + sq.b * p.o.sb + (int64_t)(h0 + h) * p.o.sh + (int64_t)sq.q_start * p.o.st;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (!PAD || lane * PER + i < p.D) op[lane * PER + i] = from_float<T>(o[i] * inv);
    if (p.lse.ptr && lane == 0)
      p.lse.ptr[sq.b * p.lse.sb + (h0 + h) * p.lse.sh + (int64_t)sq.q_start * p.lse.st] =
          l > 0.f ? (mmax + log2f(l)) * kLn2 : -INFINITY;
  };
  for (int h = wave; h < ratio; h += W) {
    float mv[W], lv[W], ov[W][PER];
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const float *row = reinterpret_cast<const float *>(smem_all + u * wave_bytes) + h * (D + 2);
      mv[u] = row[D];
      lv[u] = row[D + 1];
#pragma unroll
      for (int i = 0; i < PER; ++i) ov[u][i] = row[lane * PER + i];
    }
    float mmax = mv[0];
#pragma unroll
    for (int u = 1; u < W; ++u) mmax = fmaxf(mmax, mv[u]);
    const float muse = mmax == -INFINITY ? 0.f : mmax;
    float l = 0.f, o[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) o[i] = 0.f;
#pragma unroll
    for (int u = 0; u < W; ++u) {
      const float sc = fast_exp2(mv[u] - muse);  // a wave without half blocks has max = -inf: weight 0
      l += sc * lv[u];
#pragma unroll
      for (int i = 0; i < PER; ++i) o[i] += sc * ov[u][i];
    }
    if (groups <= 1) {
      store_row(h, o, mmax, l);
    } else {  // write-through stores: the row's other workgroups may sit on another die
      float *dst = ws + (((int64_t)b * p.Hq + h0 + h) * (max_groups + 1) + blockIdx.x) * (D + 2);
#pragma unroll
      for (int i = 0; i < PER; ++i) __hip_atomic_store(dst + lane * PER + i, o[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (lane < 2) __hip_atomic_store(dst + D + lane, lane ? l : mmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (groups <= 1) return;
  // each wave's part of the partial has reached memory before the barrier (a barrier orders the waves'
  // stores for their own compute unit; the addition behind it publishes them to the other dies)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  int *flag = reinterpret_cast<int *>(smem_all + wave_bytes - ratio * D * 2);  // wave 0's q copy: dead as well
  if (threadIdx.x == 0) *flag = arrive_last(slot, groups);
  __syncthreads();
  if (!*flag) return;
  constexpr int MAXU = 8;  // partials merged per pass: their loads leave together
  for (int h = wave; h < ratio; h += W) {
    const float *src = ws + ((int64_t)b * p.Hq + h0 + h) * (max_groups + 1) * (D + 2);
    float mmax = -INFINITY, l = 0.f, o[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) o[i] = 0.f;
    for (int s0 = 0; s0 < groups; s0 += MAXU) {
      float mv[MAXU], lv[MAXU], ov[MAXU][PER];
#pragma unroll
      for (int s = 0; s < MAXU; ++s) {
        const float *row = src + min(s0 + s, groups - 1) * (D + 2);
        mv[s] = __hip_atomic_load(row + D, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lv[s] = __hip_atomic_load(row + D + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int i = 0; i < PER; ++i) ov[s][i] = __hip_atomic_load(row + lane * PER + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      float mnew = mmax;
#pragma unroll
      for (int s = 0; s < MAXU; ++s) mnew = fmaxf(mnew, mv[s]);
      const float muse = mnew == -INFINITY ? 0.f : mnew;
      const float alpha = fast_exp2(mmax - muse);  // exp2(-inf) = 0 on the first pass
      l *= alpha;
#pragma unroll
      for (int i = 0; i < PER; ++i) o[i] *= alpha;
#pragma unroll
      for (int s = 0; s < MAXU; ++s) {
        const float sc = s0 + s < groups ? fast_exp2(mv[s] - muse) : 0.f;
        l += sc * lv[s];
#pragma unroll
        for (int i = 0; i < PER; ++i) o[i] += sc * ov[s][i];
      }
      mmax = mnew;
    }
    store_row(h, o, mmax, l);
  }
}

// Workgroups of the longest row.  (At most 255: an arrival slot counts in eight bits; longer rows
// are cut into larger units.)
static int decode_max_groups(const FwdParams &p) {
  return std::min(255, cdiv(decode_row_units(2 * decode_max_row_entries(p), decode_unit_halves(p), kDecodeWaves), kDecodeWaves));
}

// Numbers of the launches of this process (arrive_last): 56 bits, never 0.
static slot_t next_launch_number() {
  static std::atomic<slot_t> next{(uintptr_t)&next * 0x9E3779B97F4A7C15ull ^
                                (slot_t)std::chrono::system_clock::now().time_since_epoch().count()};
  slot_t n;
  do {
    n = (next.fetch_add(1, std::memory_order_relaxed) * 0xD1342543DE82EF95ull) >> 8;  // (an odd factor: 2^64 distinct products)
  } while (n == 0);
  return n;
}

bool decode_supported(const FwdParams &p, int dtype) {
  const int ratio = p.Hq / p.Hkv;
  const bool shared_row = p.csr.num_heads == 1 || (p.csr.num_heads == p.Hkv && p.Hkv != p.Hq) || ratio == 1 ||
                          (p.csr.num_heads == p.Hq && p.csr.group % ratio == 0);
  const int width = mfma_tile_width(p.D);
  const int lds = kDecodeWaves * (2 * 32 * (width * 2 + 16) + ratio * width * 2);  // DecSmem<width>::wave_bytes
  return (dtype == DK_BF16 || dtype == DK_F16) && mfma_head_dim_ok(p.D) && lds <= 160 * 1024 && p.csr.block_rows == 64 &&
         p.csr.block_cols == 64 && p.vec_ok &&
         (p.csr.entry_width == 1 || p.csr.sub_block != 0) &&
         (p.seqs.packed ? (p.seqs.packed & 2) != 0 : p.seqs.max_q_len == 1) && ratio <= 32 && shared_row && p.causal &&
         !p.seqs.zero_outside;  // (rows without a query are cleared by the prefill kernels only)
}

// Rows of one workgroup each use none of it; one place per q head then stands for "these arguments run the
// decode kernels" (dk_fwd_workspace_bytes).  With two, steps over many rows of a single block no longer
// fitted the fixed scratch of dk_fwd_noalloc (tests/test_decode_scratch.py).
size_t decode_workspace_bytes(const FwdParams &p) {
  const int groups = decode_max_groups(p), places = groups > 1 ? groups + 1 : 1;
  return (size_t)p.seqs.batch * p.Hq * places * (mfma_tile_width(p.D) + 2) * sizeof(float);
}

// Sequences whose workgroups go to empty compute units when the sequences are handed out by length, 0: they are handed out
// in the batch's order (nothing to gain while every workgroup has a compute unit of its own).  Beyond 256 workgroups
// the first compute units get a second one, and the chip's rate is only reached while all of them stream: the first round takes
// the longest sequences, shortest of them first, so that the second one, longest first, adds the most to the units that
// have the least.  Order of the batch / by length, us: 8 kv heads of 128, 48 sequences of 256 - 6000 tokens, paged 54.1 / 47.1;
// 36 of up to 11000 34.9 / 31.0, 62 of 2900 31.7 / 29.8, 41 of 330 11.1 / 11.0; 12 kv heads, 28 of 5900 42.7 / 33.2; 16 of
// 256, 23 of 1850 75.9 / 64.8.  Beyond four rounds the queue evens the sequences out and every round pays for the votes: 936
// workgroups 57.3 / 56.1, 1104 133.0 / 133.3, 1856 195.9 / 197.1, 3040 of 256 dims 204.7 / 209.9.  fp8 pools are bound by the
// conversions of a wave rather than by the memory, and few second workgroups gain nothing: 288 workgroups 26.3 / 27.0 and 22.5 / 22.6,
// 328 19.0 / 19.4, 352 32.4 / 29.2, 408 25.3 / 24.3, 480 44.5 / 41.8.
// The votes and a longest sequence that starts later than in the batch's order cost half a microsecond to two, which steps of
// little work get back only if the work of their sequences differs: rows that grow with the sequence (at least half
// as many blocks as the longest one has) do, rows that end in a window and few columns are all alike.  Sweep of 337
// steps of 10 - 180 us, order of the batch / by length, on average: 256 dims (one workgroup per compute unit) 1.09; from 320 KB of K/V
// for a workgroup of the longest row (blocks x dims >= 1280) 1.08; growing rows from 96 KB, up to three workgroups a row, 1.04 (four, 10
// sequences of 1286, 96 dims: 20.8 / 23.2 us); the others 0.99, between 0.86 (22 sequences of 4495, 96 dims, 16.1 / 18.6) and 1.11.
static int decode_first_by_length(const FwdParams &p, int groups) {
  constexpr int kUnits = 256;
  const int per_sequence = p.Hkv * groups;
  const bool ranked = (p.seqs.given & 12) && p.seqs.batch > 1 && p.seqs.batch <= kRankedSequences;
  const int64_t workgroups = (int64_t)per_sequence * p.seqs.batch;
  const int64_t from = p.paged.table && p.paged.kv_fp8 ? kUnits + 80 : kUnits;
  if (!ranked || workgroups <= from || workgroups > 4 * kUnits) return 0;
  const int entries = decode_max_row_entries(p);
  const int64_t work = (int64_t)entries * p.D / groups;
  const bool growing = (int64_t)2 * entries >= std::min(cdiv(p.seqs.max_k_len, 64), p.csr.num_rows);
  if (mfma_tile_width(p.D) < 256 && work < (growing && groups <= 3 ? 384 : 1280)) return 0;
  return std::min(p.seqs.batch, std::max(1, kUnits / per_sequence));
}

template <typename T, int D, bool PAD, bool SUB, bool PAGED, bool KV8 = false>
static int launch_decode_td(const FwdParams &p, float *ws, hipStream_t stream) {
  constexpr int W = kDecodeWaves;
  const int smem = W * DecSmem<D>::wave_bytes(p.Hq / p.Hkv);
  const int groups = std::max(1, decode_max_groups(p));
  DK_REQUIRE(smem <= 160 * 1024, "decode workgroup needs %d bytes of LDS", smem);
  const dim3 grid(groups, p.Hkv, p.seqs.batch), block(64 * W);
  const int first = decode_first_by_length(p, groups);
  DK_NOTE_KERNEL(first > 0 ? "decode_partial_kernel, sequences by length" : "decode_partial_kernel");
  if (first > 0) {
    DK_ALLOW_DYNAMIC_LDS((decode_partial_kernel<T, D, PAD, SUB, PAGED, KV8, W, true>), smem);
    hipLaunchKernelGGL((decode_partial_kernel<T, D, PAD, SUB, PAGED, KV8, W, true>), grid, block, smem, stream, p, ws,
                       decode_unit_halves(p), groups, next_launch_number(), first);
  } else {
    DK_ALLOW_DYNAMIC_LDS((decode_partial_kernel<T, D, PAD, SUB, PAGED, KV8, W, false>), smem);
    hipLaunchKernelGGL((decode_partial_kernel<T, D, PAD, SUB, PAGED, KV8, W, false>), grid, block, smem, stream, p, ws,
                       decode_unit_halves(p), groups, next_launch_number(), 0);
  }
  DK_HIP_CHECK(hipGetLastError());
  return DK_OK;
}

template <typename T, bool PAGED>
static int launch_decode_tp(const FwdParams &p, float *ws, hipStream_t stream) {
  if (p.D > 128)  // 256-wide tiles (always the zero-padding instantiation), one wave per SIMD
    return p.csr.sub_block ? launch_decode_td<T, 256, true, true, PAGED>(p, ws, stream)
                           : launch_decode_td<T, 256, true, false, PAGED>(p, ws, stream);
  if (p.csr.sub_block) {  // entries carry a bit mask over the pattern's 16- or 32-token blocks
    if (p.D == 128) return launch_decode_td<T, 128, false, true, PAGED>(p, ws, stream);
    if (p.D == 64) return launch_decode_td<T, 64, false, true, PAGED>(p, ws, stream);
    return p.D > 64 ? launch_decode_td<T, 128, true, true, PAGED>(p, ws, stream)
                    : launch_decode_td<T, 64, true, true, PAGED>(p, ws, stream);
  }
  if (p.D == 128) return launch_decode_td<T, 128, false, false, PAGED>(p, ws, stream);
  if (p.D == 64) return launch_decode_td<T, 64, false, false, PAGED>(p, ws, stream);
  return p.D > 64 ? launch_decode_td<T, 128, true, false, PAGED>(p, ws, stream)
                  : launch_decode_td<T, 64, true, false, PAGED>(p, ws, stream);
}

// head dims below the tile width (64 or 128) run the zero-padded instantiation; K/V come from the
// tensors themselves or, with a page table, from page pools
template <typename T>
static int launch_decode_t(const FwdParams &p, float *ws, hipStream_t stream) {
  if (p.paged.table && p.paged.kv_fp8) {  // fp8 pools: plain tiles only
    if (p.csr.sub_block || (p.D != 64 && p.D != 128))
      return fail(DK_ERR_UNSUPPORTED, "fp8 K/V needs head_dim 64 or 128 and pattern blocks of at least 64");
    return p.D == 128 ? launch_decode_td<T, 128, false, false, true, true>(p, ws, stream)
                      : launch_decode_td<T, 64, false, false, true, true>(p, ws, stream);
  }
  return p.paged.table ? launch_decode_tp<T, true>(p, ws, stream) : launch_decode_tp<T, false>(p, ws, stream);
}

int launch_decode(const FwdParams &p, int dtype, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  DK_REQUIRE(workspace && workspace_bytes >= decode_workspace_bytes(p), "decode workspace too small");
  DK_REQUIRE(((uintptr_t)workspace % 16) == 0, "decode workspace must be 16-byte aligned");
  float *ws = (float *)workspace;
  return dtype == DK_BF16 ? launch_decode_t<bf16_t>(p, ws, stream) : launch_decode_t<f16_t>(p, ws, stream);
}

}  // namespace dk
