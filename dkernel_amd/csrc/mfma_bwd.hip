// MFMA backward kernels for gfx950: bf16 / fp16, head dims up to 256 (tiles of 64, 128 or
// 256 columns), 64 x 64 blocks, equal-length unpadded sequences.  Two passes, no atomics:
//
//   dQ pass    (CSR rows)    workgroup = 64 q rows x one q head, 4 waves = 2 row
//              halves x 2 key halves (2 waves per SIMD; the key halves are
//              summed through LDS at the end).  Per listed K/V block:
//              S^T = K Q^T, dP^T = V dO^T (lane = q row, registers = keys, so
//              lse / delta are per-lane scalars), dS^T = P^T (dP^T - delta),
//              dQ^T += K^T dS^T with dS^T fed from registers as the B operand
//              and K^T from LDS transpose reads.  The pass also computes
//              delta = rowsum(O * dO) - dLSE of its rows and leaves it in
//              memory for the dK/dV pass, which therefore runs second.
//   dK/dV pass (CSC columns) workgroup = 64 keys x one kv head (the q heads of
//              a GQA group are looped inside), 4 waves, two workgroups per
//              CU (three at 64 head dims).  A listed q block is worked on in two steps of 32 q rows;
//              each 32 x 32 quadrant (q rows of the step x key half) has an S
//              wave (S = Q K^T, P, dV^T += dO^T P; K fragments in registers)
//              and a dP wave (dP = dO V^T, dS = P (dP - delta), dK^T += Q^T dS;
//              V fragments in registers).  P / dS feed the second products
//              from registers, dO^T / Q^T come from LDS transpose reads.
//              Every wave owns the whole accumulator of one matrix for its 32
//              keys, so nothing is summed across waves at the end.
//
// Tiles are copied HBM -> LDS asynchronously (LDS DMA, no staging registers)
// into rings of stages, in the swizzled row-major layout of mfma_common.h.
#include <climits>

#include "bwd_scratch.h"
#include "common.h"
#include "device_common.h"
#include "mfma_common.h"

namespace dk {

template <int V>
struct IntConst {  // compile-time integer passed to a generic lambda
  static constexpr int value = V;
};

template <bool V>
struct BoolConst {
  static constexpr bool value = V;
};


// ---------------------------------------------------------------------------
// dQ pass
// ---------------------------------------------------------------------------
template <typename T, int D, bool PAD, bool SUB>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2, D == 64 ? 3 : D == 256 ? 1 : 2))) void mfma_dq_kernel(const BwdParams p,
                                                                                                   int tiles_y) {
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  using TL = Tile<D>;
  constexpr int NT = 256;
  constexpr int KS = D / 16, DT = D / 32;
  constexpr int STAGE = 2 * TL::kBytes;
  // SUB: table entries are (column, bit mask over the pattern blocks inside the 64 x 64 tile)
  constexpr int EW = SUB ? 2 : 1;  // ints per table entry
  extern __shared__ __align__(16) char smem[];

  const SeqInfo sq = load_seq(p.seqs, blockIdx.z, p.causal);
  const int h = grid_head(p.csr);
  int tile = tiles_y - 1 - (int)blockIdx.y;  // longest rows first (of a causal pattern)
  if (p.csr.order)  // the table's own order, longest rows first (the grid then covers every row of it)
    tile = scalar_load(p.csr.order + lut_head(p.csr, h, p.Hq, p.Hkv) * p.csr.order_sh + blockIdx.y) - sq.past / 64;
  if (tile < 0 || tile >= seq_row_blocks(sq, 64)) return;
  const int rb = sq.past / 64 + tile;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rh = wave & 1, kh = wave >> 1;  // q-row half, key half
  const int kvh = __builtin_amdgcn_readfirstlane(h / (p.Hq / p.Hkv));  // integer division runs on the VALU
  const int m = lane & 31, g = lane >> 5;
  const int row0 = rb * 64 + rh * 32;
  const int pos = row0 + m;
  const int qi = pos - sq.past;
  const bool row_ok = qi >= 0 && qi < sq.q_len;
  if constexpr (PAD) {  // the slots of the head dims beyond p.D stay zero for the whole kernel
    zero_tiles<NT>(smem, 2 * STAGE, tid);
    __syncthreads();
  }

  // Row data.  Q and dO of the 64 rows come in as two tiles by LDS DMA, into the second K/V stage
  // (free until the loop's first step requests the second block), and the waves take their
  // fragments from there: whole cache lines, fetched once for both key halves.  Loaded straight
  // into the fragment layout (lane = row), every load instruction touches 32 rows with 32 bytes
  // each - 96 such loads per workgroup kept the memory pipeline busy for a fifth of a short
  // row's time.  O is only needed for delta = rowsum(O * dO) - dLSE: each thread loads four
  // 16-byte chunks of it, consecutive lanes along a row, multiplies them with the dO chunks in
  // LDS and the lanes of a row add up.
  constexpr int CPR = D / 8;  // 16-byte chunks per row
  __shared__ float delta_rows[64];
  float lse_raw = -INFINITY, dlse_raw = 0.f;
  uint4 oreg[64 * CPR / NT];
  {
    const int qi0 = rb * 64 - sq.past;  // query index of the tile's first row
    TileLoader<D, NT, PAD> qload, doload;
    qload.init(tid, p.q.st, p.D);
    doload.init(tid, p.dout.st, p.D);
    const T *qb = (const T *)p.q.ptr + sq.b * p.q.sb + h * p.q.sh + (int64_t)qi0 * p.q.st;
    const T *dob = (const T *)p.dout.ptr + sq.b * p.dout.sb + h * p.dout.sh + (int64_t)qi0 * p.dout.st;
    qload.issue(reinterpret_cast<const char *>(qb), -qi0, sq.q_len - qi0, smem + STAGE);
    doload.issue(reinterpret_cast<const char *>(dob), -qi0, sq.q_len - qi0, smem + STAGE + TL::kBytes);
    const T *ob = (const T *)p.o.ptr + sq.b * p.o.sb + h * p.o.sh + (int64_t)qi0 * p.o.st;
#pragma unroll
    for (int j = 0; j < 64 * CPR / NT; ++j) {
      const int r = tid / CPR + j * (NT / CPR), ch = tid % CPR;
      oreg[j] = make_uint4(0, 0, 0, 0);
      if (qi0 + r >= 0 && qi0 + r < sq.q_len && (!PAD || ch * 8 < p.D))
        oreg[j] = *reinterpret_cast<const uint4 *>(ob + (int64_t)r * p.o.st + ch * 8);
    }
    if (row_ok) {
      lse_raw = p.lse.ptr[sq.b * p.lse.sb + h * p.lse.sh + (int64_t)qi * p.lse.st];
      if (p.dlse.ptr) dlse_raw = p.dlse.ptr[sq.b * p.dlse.sb + h * p.dlse.sh + (int64_t)qi * p.dlse.st];
    }
  }

  const int lh = lut_head(p.csr, h, p.Hq, p.Hkv);
  // table reads go through the scalar unit: a vector load would have to be waited for with
  // vmcnt(0), i.e. together with every tile copy in flight
  int e0 = 0, e1 = 0;
  if (rb < p.csr.num_rows) {
    scalar_load2(p.csr.ptr + lh * p.csr.ptr_sh + rb, p.csr.ptr + lh * p.csr.ptr_sh + rb + 1, e0, e1);
  }
  const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
  const T *kbase = (const T *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh;
  const T *vbase = (const T *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh;

  TileLoader<D, NT, PAD> kload, vload;
  kload.init(tid, p.k.st, p.D);
  vload.init(tid, p.v.st, p.D);
  // blocks whose first key lies in [0, k_full_span) hold 64 keys of the sequence
  const uint32_t k_full_span = sq.k_len >= 64 ? (uint32_t)(sq.k_len - 64) + 1u : 0u;
  const uint32_t k_row_bytes = (uint32_t)p.k.st * 2u, v_row_bytes = (uint32_t)p.v.st * 2u;
  auto issue = [&](int col, int stage) {  // asynchronous copy of K/V block `col` into `stage`
    const int key0 = col * 64;
    char *ks = smem + stage * STAGE;
    // (not at the 256-wide tile: the extra scalar state pushes those kernels into scratch spills)
    if (D <= 128 && (uint32_t)key0 < k_full_span) {  // main path (one scalar compare; a padding entry is negative)
      kload.issue_full(row_address(reinterpret_cast<const char *>(kbase), key0, k_row_bytes), ks);
      vload.issue_full(row_address(reinterpret_cast<const char *>(vbase), key0, v_row_bytes), ks + TL::kBytes);
      return;
    }
    const int valid = col < 0 ? 0 : sq.k_len - key0;
    kload.issue(reinterpret_cast<const char *>(kbase + (int64_t)key0 * p.k.st), 0, valid, ks);
    vload.issue(reinterpret_cast<const char *>(vbase + (int64_t)key0 * p.v.st), 0, valid, ks + TL::kBytes);
  };
  // operand read addresses inside this wave's key half (row kh*32 + m, chunk 2ks+g swizzled;
  // transpose-read pairs) for a tile at offset 0: full pointers, and the stage is a compile-time
  // constant of the loop body, so that stage and k-step offsets are instruction immediates
  using OA = OperandAddress<D>;
  typename OA::type rd[KS], tr[DT][2];
  {
    int tro[DT][2];
    transposed_offsets<D>(lane, tro);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) rd[ks] = OA::make(smem, TL::off(kh * 32 + m, 2 * ks + g));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      tr[dt][0] = OA::make(smem, kh * 32 * TL::kRowBytes + tro[dt][0]);
      tr[dt][1] = OA::make(smem, kh * 32 * TL::kRowBytes + tro[dt][1]);
    }
  }

  floatx16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

  // Table entries: block e in col_cur (scalar register); block e + 1 is requested one block
  // early as a vector load (col_pending) and first used behind the next tile wait, so that no
  // table read ever stalls the loop.
  int col_cur = e0 < e1 ? scalar_load(cols + e0 * EW) : 0;
  int col_pending = e0 + 1 < e1 ? cols[(e0 + 1) * EW] : 0;
  int bits_cur = 0, bits_pending = 0;  // SUB: the entry's mask, carried like the column
  if constexpr (SUB) {
    bits_cur = e0 < e1 ? scalar_load(cols + e0 * EW + 1) : 0;
    bits_pending = e0 + 1 < e1 ? cols[(e0 + 1) * EW + 1] : 0;
  }
  if (e0 < e1) issue(col_cur, 0);  // the first tiles are on their way while the row data is fetched

  // Q and dO fragments, lse in the log2 domain, and delta = rowsum(O * dO) - dLSE, which this
  // kernel computes itself and also leaves in p.delta for the dK/dV pass that follows
  wait_tile_loads();
  __syncthreads();  // the Q and dO tiles (and the first K/V tiles) are visible
  vec8 qf[KS], dof[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = lds_read8<vec8>(smem + STAGE + TL::off(rh * 32 + m, 2 * ks + g));
    dof[ks] = lds_read8<vec8>(smem + STAGE + TL::kBytes + TL::off(rh * 32 + m, 2 * ks + g));
  }
#pragma unroll
  for (int j = 0; j < 64 * CPR / NT; ++j) {
    const int r = tid / CPR + j * (NT / CPR), ch = tid % CPR;
    const uint4 dow = *reinterpret_cast<const uint4 *>(smem + STAGE + TL::kBytes + TL::off(r, ch));
    float d = dot8<T>(oreg[j], dow, 0.f);
#pragma unroll
    for (int off = CPR / 2; off > 0; off >>= 1) d += __shfl_xor(d, off);
    if (ch == 0) delta_rows[r] = d;
  }
  __syncthreads();  // the row sums are there; every wave has its fragments: the second stage is free
  float lse2 = INFINITY, delta = 0.f;
  if (row_ok) {
    lse2 = lse_raw == -INFINITY ? INFINITY : lse_raw * kLog2e;
    delta = delta_rows[rh * 32 + m] - dlse_raw;
    if (kh == 0 && g == 0) p.delta[((int64_t)sq.b * p.Hq + h) * p.seqs.max_q_len + qi] = delta;
  }

  auto block_step = [&](int e, auto stage_tag) {
    constexpr int stage = decltype(stage_tag)::value;
    const int col = col_cur;
    const int bits = bits_cur;
    wait_tile_loads();
    __syncthreads();  // tile e is visible; every wave is done with the other stage
    const int col_next = __builtin_amdgcn_readfirstlane(col_pending);  // landed before the tile did
    if constexpr (SUB) bits_cur = __builtin_amdgcn_readfirstlane(bits_pending);
    if (e + 2 < e1) {
      col_pending = cols[(e + 2) * EW];
      if constexpr (SUB) bits_pending = cols[(e + 2) * EW + 1];
    }
    if (e + 1 < e1) issue(col_next, stage ^ 1);
    col_cur = col_next;
    const int key0 = col * 64 + kh * 32;  // first key of this wave's half
    if (col < 0 || key0 >= sq.k_len || (p.causal && key0 > row0 + 31)) return;
    const int quad = SUB ? tile_quadrants(bits, p.csr.sub_block) >> (8 * rh + 4 * kh) & 15 : 15;
    if (SUB && quad == 0) return;  // nothing attended (wave-uniform)
    constexpr int ks_ = stage * STAGE, vs_ = ks_ + TL::kBytes;  // byte offsets of this stage's K and V tiles

    floatx16 s, dp;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
    // batches of operand reads, then the multiplies (the scheduler barriers keep
    // the compiler from sinking each read next to its MFMA)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      vec8 ka[KS / 2];
#pragma unroll
      for (int i = 0; i < KS / 2; ++i) ka[i] = lds_operand<vec8>(rd[half * (KS / 2) + i] + ks_);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KS / 2; ++i) s = M::mma(ka[i], qf[half * (KS / 2) + i], s);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      vec8 va[KS / 2];
#pragma unroll
      for (int i = 0; i < KS / 2; ++i) va[i] = lds_operand<vec8>(rd[half * (KS / 2) + i] + vs_);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KS / 2; ++i) dp = M::mma(va[i], dof[half * (KS / 2) + i], dp);
    }
    // K^T operands of the dQ product do not depend on dS: fetch them now
    vec8 kt[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) kt[dt] = lds_operand_tr<vec8>(tr[dt][0] + ks_, tr[dt][1] + ks_);

    const bool need_mask = (key0 + 31 >= sq.k_len) || (p.causal && key0 + 31 > row0);
    const int lim = p.causal ? min(pos, sq.k_len - 1) : sq.k_len - 1;  // last visible key of this row
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(fmaf(s[r], p.scale_log2, -lse2));
    if (need_mask) {  // wave-uniform: only the diagonal block and the last, partial one pay for masks
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = key0 + (r >> 2) * 8 + g * 4 + (r & 3);
        s[r] = key > lim ? 0.f : s[r];
      }
    }
    if constexpr (SUB) {
      if (quad != 15) {  // wave-uniform: blocks of 16, the quadrant is not attended as a whole
        const int row_bits = quad >> (2 * (m >> 4));
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = ((row_bits >> (r >> 3)) & 1) ? s[r] : 0.f;
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= dp[r] - delta;  // dS^T without sm_scale (applied once at the end)
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float f[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = s[t * 8 + i];
      const vec8 dsb = M::pack(f);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        acc[dt] = M::mma(kt[dt], dsb, acc[dt]);
        if (t == 0)  // refill with the second k-step's operand as soon as the register is free
          kt[dt] = lds_operand_tr<vec8>(tr[dt][0] + ks_ + 16 * TL::kRowBytes, tr[dt][1] + ks_ + 16 * TL::kRowBytes);
      }
    }
  };
  for (int e = e0; e < e1; e += 2) {
    block_step(e, IntConst<0>{});
    if (e + 1 < e1) block_step(e + 1, IntConst<1>{});
  }

  // Sum the two key halves.  Each wave finishes half of the head dims of its rows: it hands the
  // d-tiles of the other half to its partner through LDS and adds the partner's share to its own,
  // so that conversions and stores are spread over all four waves.
  __syncthreads();
  float *red = reinterpret_cast<float *>(smem);
  static_assert(DT % 2 == 0, "two halves of the d-tiles");
#pragma unroll
  for (int i = 0; i < DT / 2; ++i) {
    // (kh is wave-uniform but not a compile-time constant: the accumulator is picked by a
    // select between two fixed registers, never by a run-time index)
    const int dt = (1 - kh) * (DT / 2) + i;  // a d-tile of the partner's half
#pragma unroll
    for (int r = 0; r < 16; ++r)
      red[((rh * DT + dt) * 16 + r) * 64 + lane] = kh == 0 ? acc[DT / 2 + i][r] : acc[i][r];
  }
  __syncthreads();
  // From the 128-wide tile on the finished rows go through a 64-row tile behind the exchange
  // area and leave as whole rows with the non-temporal hint (16 rows per wave): -1 % of the
  // backward at head_dim 128, -1.5 % at 192 / 256.  At the 64-wide tile the direct 8-byte
  // stores of the accumulator layout measure 0.5 % faster and stay.
  constexpr bool kStagedStores = D >= 128;
  char *const out_tile = smem + 2 * DT * 16 * 64 * (int)sizeof(float);
  static_assert(2 * DT * 16 * 64 * (int)sizeof(float) + TL::kBytes <= 2 * STAGE, "exchange area and output tile fit the stages");
  if constexpr (!kStagedStores) {
    if (!row_ok) return;
  }
  int lane_late = lane;  // opaque copy: the tile addresses below are computed here, not before the loop
  asm volatile("" : "+v"(lane_late));
  const int m_late = lane_late & 31, g_late = lane_late >> 5;
  T *dqp = (T *)p.dq.ptr + sq.b * p.dq.sb + h * p.dq.sh + (int64_t)qi * p.dq.st;
#pragma unroll
  for (int i = 0; i < DT / 2; ++i) {
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      float f4[4];
      const int dt = kh * (DT / 2) + i;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = r4 * 4 + j;
        const float own = kh == 0 ? acc[i][r] : acc[DT / 2 + i][r];
        f4[j] = (own + red[((rh * DT + dt) * 16 + r) * 64 + lane]) * p.sm_scale;
      }
      const uint2 o4 = pack4<T>(f4[0], f4[1], f4[2], f4[3]);
      // registers 4*r4 .. 4*r4+3 are dims 32dt + 8r4 + 4g + {0..3}
      if constexpr (kStagedStores)
        *reinterpret_cast<uint2 *>(out_tile + TL::off(rh * 32 + m_late, dt * 4 + r4) + g_late * 8) = o4;
      else if (!PAD || dt * 32 + r4 * 8 + g * 4 < p.D)
        *reinterpret_cast<uint2 *>(dqp + dt * 32 + r4 * 8 + g * 4) = o4;
    }
  }
  if constexpr (kStagedStores) {
    __syncthreads();
    const int qi0 = rb * 64 + wave * 16 - sq.past;  // query index of this wave's first row
    T *dq_row0 = (T *)p.dq.ptr + sq.b * p.dq.sb + h * p.dq.sh + (int64_t)qi0 * p.dq.st;
    store_staged_rows<T, D, PAD, 16>(out_tile + wave * 16 * TL::kRowBytes, dq_row0, p.dq.st, lane, -qi0, sq.q_len - qi0, p.D);
  }
}

// ---------------------------------------------------------------------------
// dQ pass, two q tiles per workgroup (tiles of 64 and 128 head dims)
// ---------------------------------------------------------------------------
// One workgroup = table rows 2u and 2u + 1 of one q head (128 q rows), 4 waves: wave = 32 q rows
// of one of the two rows, against all 64 keys of a block (two 32-key halves one after the other,
// in the same registers).  The workgroup walks the union of its two table rows, merged on the
// fly from the two sorted rows, and copies every K / V tile once for both: neighbouring rows of
// the local window share 15 of 16 columns and every vertical column, so the tile traffic from
// the L2 into LDS (what the one-tile kernel spent a quarter of its time on) is halved; a wave
// skips the blocks its own row does not hold.  Every wave owns the finished dQ of its rows:
// nothing is summed across waves at the end.
// CUT: launches that cut long pairs into segments; an instantiation of its own, as its prologue, jumped over, and the fifty
// scalars it spills took launches that cut nothing 4 - 8 % longer (16 heads of 128, 2 x 3108 tokens 76.3 / 79.6 us, 32 heads, 2 x 1932
// 58.4 / 63.2).
template <typename T, int D, bool PAD, bool SUB, bool CUT, int KD = D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, D == 64 ? 3 : 2))) void mfma_dq_pair_kernel(const BwdParams p,
                                                                                                      int pairs_y) {
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  using TL = Tile<D>;
  constexpr int NT = 256;
  constexpr int KS = KD / 16, DT = KD / 32;
  constexpr int STAGE = 2 * TL::kBytes;
  constexpr int EW = SUB ? 2 : 1;  // ints per table entry
  extern __shared__ __align__(16) char smem[];

  const SeqInfo sq = load_seq(p.seqs, blockIdx.z, p.causal);
  if (sq.q_len <= 0) return;
  const int first_rb = sq.past / 64, last_rb = (sq.past + sq.q_len - 1) / 64;
  const int h = grid_head(p.csr);
  int u = (first_rb >> 1) + pairs_y - 1 - (int)blockIdx.y;  // longest rows first (of a causal pattern)
  int place = blockIdx.y, seg = 0;  // (long pairs cut into segments: with the table's own order only)
  if constexpr (CUT) find_segment(p.seg, blockIdx.y, place, seg);
  if (p.csr.pair_order)  // the table's own order, longest pairs first (the grid then covers every pair of it)
    u = scalar_load(p.csr.pair_order + lut_head(p.csr, h, p.Hq, p.Hkv) * p.csr.order_sh + place);
  if (u > (last_rb >> 1) || u < (first_rb >> 1)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ts = wave >> 1, rh = wave & 1;  // which of the two table rows, which half of its 64 q rows
  const int ra = 2 * u, rb = ra + ts;
  const int kvh = __builtin_amdgcn_readfirstlane(h / (p.Hq / p.Hkv));  // integer division runs on the VALU
  const int m = lane & 31, g = lane >> 5;
  const int row0 = rb * 64 + rh * 32;
  const int pos = row0 + m;
  const int qi = pos - sq.past;
  const bool row_ok = qi >= 0 && qi < sq.q_len;  // (a table row without queries of this sequence: false everywhere)
  // the two table rows: entries [e0, emid) are row 2u, [emid, e1) row 2u + 1 (consecutive rows
  // follow each other in the table); a row without queries of this sequence contributes nothing
  auto table_rows = [&](int lh, int &e0, int &emid, int &e1) __attribute__((always_inline)) {
    const int32_t *rp = p.csr.ptr + lh * p.csr.ptr_sh;
    if (ra < p.csr.num_rows) scalar_load_row_pair(rp, ra, p.csr.num_rows, e0, emid, e1);
    if (ra < first_rb) e0 = emid;
    if (ra + 1 > last_rb) e1 = emid;
  };
  // CUT: this workgroup's entries [part[0], part[1]) and [part[2], part[3]) of the two rows, and the place of its partial sum
  // (part[4], -1: it takes both rows whole), kept in LDS until they are used.  No barrier stands between a wave's store and
  // its reads: that is sound only as long as every wave stores each place once and all waves the same value.
  __shared__ int part[5];
  if constexpr (CUT) {
    const int lh = lut_head(p.csr, h, p.Hq, p.Hkv);
    int e0 = 0, emid = 0, e1 = 0;
    table_rows(lh, e0, emid, e1);
    const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
    int a0 = e0, a1 = emid, b0 = emid, b1 = e1, slot = -1;
    if (place < p.seg.n[1]) {
      const int segments = planned_segments(p.seg, place, (e1 - e0 + 1) / 2);
      if (seg >= segments) return;
      if (segments > 1) {
        slot = seg * p.seg.n[1] + place;
        // an even share of the longer row's entries, and what the other row lists between their columns
        const bool first_longer = emid - e0 >= e1 - emid;
        const int l0 = first_longer ? e0 : emid, len = first_longer ? emid - e0 : e1 - emid;
        const int s0 = __builtin_amdgcn_readfirstlane(len * seg / segments), s1 = __builtin_amdgcn_readfirstlane(len * (seg + 1) / segments);
        const int o0 = first_longer ? emid : e0, o1 = first_longer ? e1 : emid;
        int p0 = o0, p1 = o1;
        if (seg > 0) p0 = entry_lower_bound<EW>(cols, o0, o1, scalar_load(cols + (l0 + s0) * EW));
        if (seg + 1 < segments) p1 = entry_lower_bound<EW>(cols, p0, o1, scalar_load(cols + (l0 + s1) * EW));
        a0 = first_longer ? l0 + s0 : p0, a1 = first_longer ? l0 + s1 : p1;
        b0 = first_longer ? p0 : l0 + s0, b1 = first_longer ? p1 : l0 + s1;
      }
    }
    part[0] = a0, part[1] = a1, part[2] = b0, part[3] = b1, part[4] = slot;
  }

  if (PAD && p.D < KD) {  // the slots of the head dims beyond p.D stay zero for the whole kernel
    zero_tiles<NT>(smem, 2 * STAGE, tid);
    __syncthreads();
  }

  // Row data: Q and dO of the 128 rows come in as four tiles by LDS DMA (stage 0: first table
  // row, stage 1: second), O as 16-byte chunks along the rows, multiplied with the dO chunks in
  // LDS for delta = rowsum(O * dO) - dLSE.  The first K / V request has to wait until every wave
  // has taken its fragments out of the stages.
  constexpr int CPR = D / 8;  // 16-byte chunks per row
  constexpr int OCH = 128 * CPR / NT;
  __shared__ float delta_rows[128];
  float lse_raw = -INFINITY, dlse_raw = 0.f;
  uint4 oreg[OCH];
  {
    TileLoader<D, NT, PAD> qload, doload;
    qload.init(tid, p.q.st, p.D);
    doload.init(tid, p.dout.st, p.D);
    const int qi0 = ra * 64 - sq.past;  // query index of the first of the 128 rows (may be negative)
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const int q0 = qi0 + t2 * 64;
      const T *qb = (const T *)p.q.ptr + sq.b * p.q.sb + h * p.q.sh + (int64_t)q0 * p.q.st;
      const T *dob = (const T *)p.dout.ptr + sq.b * p.dout.sb + h * p.dout.sh + (int64_t)q0 * p.dout.st;
      qload.issue(reinterpret_cast<const char *>(qb), -q0, sq.q_len - q0, smem + t2 * STAGE);
      doload.issue(reinterpret_cast<const char *>(dob), -q0, sq.q_len - q0, smem + t2 * STAGE + TL::kBytes);
    }
    const T *ob = (const T *)p.o.ptr + sq.b * p.o.sb + h * p.o.sh + (int64_t)qi0 * p.o.st;
#pragma unroll
    for (int j = 0; j < OCH; ++j) {
      const int r = tid / CPR + j * (NT / CPR), ch = tid % CPR;
      oreg[j] = make_uint4(0, 0, 0, 0);
      if (qi0 + r >= 0 && qi0 + r < sq.q_len && (!PAD || ch * 8 < p.D))
        oreg[j] = *reinterpret_cast<const uint4 *>(ob + (int64_t)r * p.o.st + ch * 8);
    }
    if (row_ok) {
      lse_raw = p.lse.ptr[sq.b * p.lse.sb + h * p.lse.sh + (int64_t)qi * p.lse.st];
      if (p.dlse.ptr) dlse_raw = p.dlse.ptr[sq.b * p.dlse.sb + h * p.dlse.sh + (int64_t)qi * p.dlse.st];
    }
  }

  const int lh = lut_head(p.csr, h, p.Hq, p.Hkv);
  int e0 = 0, emid = 0, e1 = 0;
  if constexpr (!CUT) table_rows(lh, e0, emid, e1);
  const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
  const T *kbase = (const T *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh;
  const T *vbase = (const T *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh;

  TileLoader<D, NT, PAD> kload, vload;
  kload.init(tid, p.k.st, p.D);
  vload.init(tid, p.v.st, p.D);
  // blocks whose first key lies in [0, k_full_span) hold 64 keys of the sequence
  const uint32_t k_full_span = sq.k_len >= 64 ? (uint32_t)(sq.k_len - 64) + 1u : 0u;
  const uint32_t k_row_bytes = (uint32_t)p.k.st * 2u, v_row_bytes = (uint32_t)p.v.st * 2u;
  auto issue = [&](int col, int stage) {  // asynchronous copy of K/V block `col` into `stage`
    const int key0 = col * 64;
    char *ks = smem + stage * STAGE;
    if ((uint32_t)key0 < k_full_span) {  // main path (one scalar compare; a padding entry is negative)
      kload.issue_full(row_address(reinterpret_cast<const char *>(kbase), key0, k_row_bytes), ks);
      vload.issue_full(row_address(reinterpret_cast<const char *>(vbase), key0, v_row_bytes), ks + TL::kBytes);
      return;
    }
    const int valid = col < 0 ? 0 : sq.k_len - key0;
    kload.issue(reinterpret_cast<const char *>(kbase + (int64_t)key0 * p.k.st), 0, valid, ks);
    vload.issue(reinterpret_cast<const char *>(vbase + (int64_t)key0 * p.v.st), 0, valid, ks + TL::kBytes);
  };
  // operand read addresses for a tile at offset 0: row m of a 32-key half, chunk 2ks+g swizzled;
  // transpose-read pairs of d-tile dt.  Stage, key half and k-step offsets are immediates.
  using OA = OperandAddress<D>;
  typename OA::type rd[KS], tr[DT][2];
  {
    int tro[DT][2];
    transposed_offsets<D>(lane, tro);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) rd[ks] = OA::make(smem, TL::off(m, 2 * ks + g));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) tr[dt][0] = OA::make(smem, tro[dt][0]), tr[dt][1] = OA::make(smem, tro[dt][1]);
  }

  floatx16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

  // The union of the two rows in column order: head_a / head_b are the next unconsumed entries
  // (scalar), pend_a / pend_b the entries after them (vector loads, first used behind a tile
  // wait, so that no table read stalls the loop); flg_cur says which rows hold the current column.
  constexpr int kEnd = 0x7fffffff;
  int a_pos = e0, b_pos = emid, a_end = emid, b_end = e1;
  if constexpr (CUT) {
    a_pos = __builtin_amdgcn_readfirstlane(part[0]), b_pos = __builtin_amdgcn_readfirstlane(part[2]);
    a_end = __builtin_amdgcn_readfirstlane(part[1]), b_end = __builtin_amdgcn_readfirstlane(part[3]);
  }
  int head_a = kEnd, head_b = kEnd, pend_a = 0, pend_b = 0;
  int hbits_a = 0, hbits_b = 0, pbits_a = 0, pbits_b = 0;  // SUB: the entries' masks, carried like the columns
  scalar_load_heads<EW>(cols, a_pos, a_end, b_pos, b_end, head_a, head_b, hbits_a, hbits_b);
  if (a_pos + 1 < a_end) pend_a = cols[(a_pos + 1) * EW];
  if (b_pos + 1 < b_end) pend_b = cols[(b_pos + 1) * EW];
  if constexpr (SUB) {
    if (a_pos + 1 < a_end) pbits_a = cols[(a_pos + 1) * EW + 1];
    if (b_pos + 1 < b_end) pbits_b = cols[(b_pos + 1) * EW + 1];
  }
  int col_cur = min(head_a, head_b);
  int flg_cur = (head_a == col_cur ? 1 : 0) | (head_b == col_cur ? 2 : 0);
  int bits_cur = ts ? hbits_b : hbits_a;  // mask of the current column in this wave's row (if it holds it)

  // Q and dO fragments, lse in the log2 domain, and delta = rowsum(O * dO) - dLSE, which this
  // kernel computes itself and also leaves in p.delta for the dK/dV pass that follows
  wait_tile_loads();
  __syncthreads();  // the Q and dO tiles are visible
  vec8 qf[KS], dof[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    qf[ks] = lds_read8<vec8>(smem + ts * STAGE + TL::off(rh * 32 + m, 2 * ks + g));
    dof[ks] = lds_read8<vec8>(smem + ts * STAGE + TL::kBytes + TL::off(rh * 32 + m, 2 * ks + g));
  }
#pragma unroll
  for (int j = 0; j < OCH; ++j) {
    const int r = tid / CPR + j * (NT / CPR), ch = tid % CPR;
    const uint4 dow = *reinterpret_cast<const uint4 *>(smem + (r >> 6) * STAGE + TL::kBytes + TL::off(r & 63, ch));
    float d = !PAD || ch * 8 < p.D ? dot8<T>(oreg[j], dow, 0.f) : 0.f;  // (those slots may hold anything)
#pragma unroll
    for (int off = CPR / 2; off > 0; off >>= 1) d += __shfl_xor(d, off);
    if (ch == 0) delta_rows[r] = d;
  }
  __syncthreads();  // the row sums are there; every wave has its fragments: both stages are free
  if (col_cur != kEnd) issue(col_cur, 0);
  float lse2 = INFINITY, delta = 0.f;
  if (row_ok) {
    lse2 = lse_raw == -INFINITY ? INFINITY : lse_raw * kLog2e;
    delta = delta_rows[ts * 64 + rh * 32 + m] - dlse_raw;
    if (g == 0 && (!CUT || part[4] < p.seg.n[1])) p.delta[((int64_t)sq.b * p.Hq + h) * p.seqs.max_q_len + qi] = delta;
  }

  auto block_step = [&](auto stage_tag) {
    constexpr int stage = decltype(stage_tag)::value;
    const int col = col_cur;
    const int flg = flg_cur;
    const int bits = bits_cur;
    wait_tile_loads();
    __syncthreads();  // the tile is visible; every wave is done with the other stage
    // All four values that may be needed are read ahead of the requests for the ones after them: read behind such a
    // request the compiler waits for it (vmcnt(0): a round trip to the L2 in every block, ahead of the next tile's request).
    const int next_a = __builtin_amdgcn_readfirstlane(pend_a), next_b = __builtin_amdgcn_readfirstlane(pend_b);
    int nbits_a = 0, nbits_b = 0;
    if constexpr (SUB) nbits_a = __builtin_amdgcn_readfirstlane(pbits_a), nbits_b = __builtin_amdgcn_readfirstlane(pbits_b);
    if (flg & 1) {
      ++a_pos;
      head_a = a_pos < a_end ? next_a : kEnd;
      hbits_a = nbits_a;
      if (a_pos + 1 < a_end) {
        pend_a = cols[(a_pos + 1) * EW];
        if constexpr (SUB) pbits_a = cols[(a_pos + 1) * EW + 1];
      }
    }
    if (flg & 2) {
      ++b_pos;
      head_b = b_pos < b_end ? next_b : kEnd;
      hbits_b = nbits_b;
      if (b_pos + 1 < b_end) {
        pend_b = cols[(b_pos + 1) * EW];
        if constexpr (SUB) pbits_b = cols[(b_pos + 1) * EW + 1];
      }
    }
    const int col_next = min(head_a, head_b);
    flg_cur = (head_a == col_next ? 1 : 0) | (head_b == col_next ? 2 : 0);
    if constexpr (SUB) bits_cur = ts ? hbits_b : hbits_a;
    if (col_next != kEnd) issue(col_next, stage ^ 1);
    col_cur = col_next;
    if (!((flg >> ts) & 1)) return;  // not in this wave's row
    if (col < 0) return;
    constexpr int ks_ = stage * STAGE, vs_ = ks_ + TL::kBytes;  // byte offsets of this stage's K and V tiles

#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {  // the two 32-key halves of the block
      const int key0 = col * 64 + kh * 32;
      if (key0 >= sq.k_len || (p.causal && key0 > row0 + 31)) continue;  // nothing visible (wave-uniform)
      const int quad = SUB ? tile_quadrants(bits, p.csr.sub_block) >> (8 * rh + 4 * kh) & 15 : 15;
      if (SUB && quad == 0) continue;  // nothing attended
      constexpr int kRow32 = 32 * TL::kRowBytes;
      floatx16 s, dp;
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.f;
      // batches of operand reads, then the multiplies (the scheduler barriers keep
      // the compiler from sinking each read next to its MFMA)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        vec8 ka[KS / 2];
#pragma unroll
        for (int i = 0; i < KS / 2; ++i) ka[i] = lds_operand<vec8>(rd[half * (KS / 2) + i] + ks_ + kh * kRow32);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KS / 2; ++i) s = M::mma(ka[i], qf[half * (KS / 2) + i], s);
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        vec8 va[KS / 2];
#pragma unroll
        for (int i = 0; i < KS / 2; ++i) va[i] = lds_operand<vec8>(rd[half * (KS / 2) + i] + vs_ + kh * kRow32);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < KS / 2; ++i) {
          dp = M::mma(va[i], dof[half * (KS / 2) + i], dp);
          // the probabilities only wait for S: their exponentials stand between the multiplies of dP
          if (half == 1) {
#pragma unroll
            for (int r = i * 32 / KS; r < (i + 1) * 32 / KS; ++r) s[r] = fast_exp2(fmaf(s[r], p.scale_log2, -lse2));
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      // K^T operands of the dQ product do not depend on dS: all of them are fetched now, behind the multiplies (with the
      // exponentials between those: training, 4 x 2048 tokens, 32 / 8 heads 580 -> 576 us)
      vec8 kt[2][DT];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
          kt[t][dt] = lds_operand_tr<vec8>(tr[dt][0] + ks_ + kh * kRow32 + t * 16 * TL::kRowBytes, tr[dt][1] + ks_ + kh * kRow32 + t * 16 * TL::kRowBytes);

      const bool need_mask = (key0 + 31 >= sq.k_len) || (p.causal && key0 + 31 > row0);
      const int lim = p.causal ? min(pos, sq.k_len - 1) : sq.k_len - 1;  // last visible key of this row
      if (need_mask) {  // wave-uniform: only the diagonal block and the last, partial one pay for masks
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = key0 + (r >> 2) * 8 + g * 4 + (r & 3);
          s[r] = key > lim ? 0.f : s[r];
        }
      }
      if constexpr (SUB) {
        if (quad != 15) {  // wave-uniform: blocks of 16, the quadrant is not attended as a whole
          const int row_bits = quad >> (2 * (m >> 4));
#pragma unroll
          for (int r = 0; r < 16; ++r) s[r] = ((row_bits >> (r >> 3)) & 1) ? s[r] : 0.f;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] *= dp[r] - delta;  // dS^T without sm_scale (applied once at the end)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = s[t * 8 + i];
        const vec8 dsb = M::pack(f);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[dt] = M::mma(kt[t][dt], dsb, acc[dt]);
      }
    }
  };
  while (col_cur != kEnd) {
    block_step(IntConst<0>{});
    if (col_cur == kEnd) break;
    block_step(IntConst<1>{});
  }

  int slot_end = -1;
  if constexpr (CUT) slot_end = __builtin_amdgcn_readfirstlane(part[4]);
  if (CUT && slot_end >= 0) {  // fp32 partial sum, unscaled
    int late = lane;  // (opaque: the addresses are computed here, not kept through the loop)
    asm volatile("" : "+v"(late));
    float *outp = p.seg.partial + ((((int64_t)sq.b * p.Hq + h) * p.seg.slots + slot_end) * 128 + wave * 32 + (late & 31)) * p.D + (late >> 5) * 4;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        if (!PAD || dt * 32 + r4 * 8 + (late >> 5) * 4 < p.D)
          *reinterpret_cast<float4 *>(outp + dt * 32 + r4 * 8) =
              make_float4(acc[dt][r4 * 4], acc[dt][r4 * 4 + 1], acc[dt][r4 * 4 + 2], acc[dt][r4 * 4 + 3]);
    return;
  }
  // every wave holds the finished dQ^T of its 32 rows
  __syncthreads();  // the K / V stages are free: each wave stages its tile in 32 rows of them
  {
    const int qi0 = row0 - sq.past;  // may be negative or beyond q_len: those rows are skipped
    T *dq_row0 = (T *)p.dq.ptr + sq.b * p.dq.sb + h * p.dq.sh + (int64_t)qi0 * p.dq.st;
    store_tile_rows<T, D, PAD>(smem + wave * 32 * TL::kRowBytes, acc, p.sm_scale, dq_row0, p.dq.st, lane, -qi0,
                               sq.q_len - qi0, p.D);
  }
}

// ---------------------------------------------------------------------------
// dK / dV pass
// ---------------------------------------------------------------------------
// One workgroup = one 64-key column block of one kv head, 4 waves, two workgroups per CU (three at 64 head dims; the
// start-up and close-down of one column then overlap with the other workgroup's loop, and the
// two workgroups' barriers are independent).  A listed q block is worked on in two steps of 32
// q rows; in each step the two 32 x 32 (q rows x keys) quadrants are each shared by a pair of
// waves:
//   the S wave:   S = Q K^T, P = exp(S - lse), dV^T += dO^T P     (K fragments and dV in registers)
//   the dP wave:  dP = dO V^T, dS = P (dP - delta), dK^T += Q^T dS (V fragments and dK in registers)
// so that each wave holds the accumulators of one matrix for 32 keys and fits in the 256
// registers of two waves per SIMD.  P goes from the S wave to the dP wave through LDS in fp32,
// exactly as computed.  The dP wave finishes a step one iteration late (after the next step's
// barrier has published P), so one barrier per step is enough: Q tiles and the lse / delta
// vectors live one iteration longer than dO tiles (rings of 4 and 3 stages of 32-row tiles), and
// tile loads run two steps ahead.
//
// Two in-order waves per SIMD: what a wave issues between its multiplies is what the pass waits for, more than LDS or HBM.
// Hence the loop takes a block's two steps in one iteration (P buffers and the second half's Q places are immediates),
// operand addresses are moved on in place, everything that only the change of heads or a partial tile needs is computed
// there from opaque copies, and the multiplies of one step stand next to the exponentials of the next: the S wave leaves
// the second half of dV to the following step, the dP wave forms dP of its step before dS of the one before.  Scalar
// instructions per step and wave 113 -> 60, vector ones next to the 16 multiplies 85 -> 77, matrix pipe 40 -> 46 % busy.
// This pass, us, both sides traced twice in turn: 32 heads of 128 x 8192 tokens 412 / 415 -> 388 / 386, 4 x 2048, 32 / 8 heads
// 293 / 288 -> 265 / 264, 4 x 3000 tokens of 12 heads of 64 with global blocks of 32 101 / 97 -> 94 / 95, 3000 tokens of
// 16 heads of 256 122 / 123 -> 113 / 114.
template <int D>
struct DkdvSmem {
  using TL = Tile<D>;
  static constexpr int kRows = 32;                            // q rows per step
  static constexpr int kTile = kRows * TL::kRowBytes;         // one 32-row tile
  static constexpr int kQStages = 4, kDoStages = 3, kAhead = 2;
  static constexpr int kQ = 0;                                // Q ring
  static constexpr int kDo = kQ + kQStages * kTile;           // dO ring
  static constexpr int kVec = kDo + kDoStages * kTile;        // per Q stage: lse[32], delta[32]
  static constexpr int kX = kVec + kQStages * 256;            // P exchange: [pair 2][buffer 2][16][64] floats
  static constexpr int kBytes = kX + 2 * 2 * 4096;
};

// At the 64-wide tile a step is eight multiplies per wave against the same barrier, waits and scalar work as at the
// 128-wide one, so a third workgroup per CU (45 KB of LDS and 152 - 154 registers each) fills what two leave idle: training,
// 64 dims, two / three workgroups, us: 32 heads x 8192 tokens 558 / 523, 4 x 3000 tokens of 12 heads with global blocks of
// 32 334 / 310.
template <typename T, int D, bool PAD, bool SUB, int KD = D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2, D == 64 ? 3 : D == 256 ? 1 : 2))) void mfma_dkdv_kernel(const BwdParams p, int head_split) {
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  using TL = Tile<D>;
  using S = DkdvSmem<D>;
  constexpr int NT = 256;
  constexpr int KS = KD / 16, DT = KD / 32;
  using Loader = TileLoader<D, NT, PAD, S::kRows>;
  constexpr int LPT = 2 * Loader::kChunks + 1;  // load instructions per wave per step
  // SUB: steps without an attended block are left out, and a pair of waves without a bit in its quadrant sits the
  // step out (not at the 256-wide tile and the zero-padded 128 dims: slower, and one register too many).  Blocks of
  // 32, local 16, vertical 8, 16 heads x 8000 tokens, forward and backward: 555 -> 473 us with the two other kernels.
  constexpr bool kIdle = SUB && (D == 64 || (D == 128 && (!PAD || KD < D)));
  // SUB: table entries are (row block, bit mask over the pattern blocks inside the 64 x 64 tile)
  constexpr int EW = SUB ? 2 : 1;  // ints per table entry
  extern __shared__ __align__(16) char smem[];

  const SeqInfo sq = load_seq(p.seqs, blockIdx.z, p.causal);
  // head_split: one workgroup per q head instead of per kv head; p.dk / p.dv then describe
  // per-q-head partial buffers that a second kernel sums over each kv group
  const int ratio = __builtin_amdgcn_readfirstlane(p.Hq / p.Hkv);  // integer division runs on the VALU
  const int out_head = grid_head(p.csc);
  const int kvh = head_split ? __builtin_amdgcn_readfirstlane(out_head / ratio) : out_head;
  const int gq_base = head_split ? out_head - kvh * ratio : 0, heads = head_split ? 1 : ratio;
  // Columns are handed out longest first when the table says in which order: the hardware deals
  // workgroups to its shader engines round-robin and in order, so long columns that recur with a
  // period pile up on a few engines otherwise.
  int place, seg;  // (long columns are cut into segments in that order, where a workgroup takes one q head)
  find_segment(p.seg, blockIdx.y, place, seg);
  int cb = place;
  if (p.csc.order)  // (the grid then covers every column of the table)
    cb = scalar_load(p.csc.order + lut_head(p.csc, kvh * ratio + gq_base, p.Hq, p.Hkv) * p.csc.order_sh + place);
  if (cb * 64 >= sq.k_len) return;
  // of a cut column: the entries of each q head, the part of all heads' entries that is this workgroup's, and the
  // place of its sums (-1: not cut)
  __shared__ int part[5];
  int gq_first = gq_base, gq_end = gq_base + heads;
  if (p.seg.entries) {
    int e0, len, lo, hi;
    const int segments = column_part<EW>(p, lut_head(p.csc, kvh * ratio + gq_base, p.Hq, p.Hkv), cb, place, seg, heads, sq, e0, len, lo, hi);
    if (seg >= segments) return;
    part[0] = e0, part[1] = len, part[2] = lo, part[3] = hi, part[4] = segments > 1 ? seg * p.seg.n[1] + place : -1;
    if (segments > 1 && heads > 1)  // (then len > 0)
      gq_first = __builtin_amdgcn_readfirstlane(lo / len), gq_end = __builtin_amdgcn_readfirstlane((hi + len - 1) / len);
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nh = wave & 1;  // key half; also the index of the (S wave, dP wave) pair
  const bool dp_wave = wave >= 2;
  const int n = lane & 31, g = lane >> 5;
  const int key = cb * 64 + nh * 32 + n;
  const bool key_ok = key < sq.k_len;

  Loader qload, doload;
  qload.init(tid, p.q.st, p.D);
  doload.init(tid, p.dout.st, p.D);
  if (PAD && p.D < KD) {  // the slots of the head dims beyond p.D stay zero in every stage
    zero_tiles<NT>(smem, S::kBytes, tid);
    __syncthreads();
  }
  // K fragments (S wave) or V fragments (dP wave): B operand of the first product.  Up to the
  // 128-wide tile the K and V tiles of the column come in by LDS DMA (whole cache lines; K into
  // the two Q stages that the first two steps do not use, V into the P exchange area) and the
  // waves take their fragments from there behind the first tile wait.  Loaded straight into the
  // fragment layout (lane = key), every load instruction touches 32 rows with 32 bytes each:
  // measured 8 % of the pass on columns of 16 blocks.  (At the 256-wide tile the V tile does not
  // fit the exchange area: direct loads.)
  constexpr bool kKvTiles = D <= 128;
  char *const k_tile = smem + S::kQ + 2 * S::kTile, *const v_tile = smem + S::kX;
  vec8 kvf[KS];
  if constexpr (kKvTiles) {
    static_assert(!kKvTiles || (2 * S::kTile == TL::kBytes && 2 * 2 * 4096 >= TL::kBytes), "a 64-row tile fits either place");
    TileLoader<D, NT, PAD> kload, vload;
    kload.init(tid, p.k.st, p.D);
    vload.init(tid, p.v.st, p.D);
    const T *kb = (const T *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh + (int64_t)cb * 64 * p.k.st;
    const T *vb = (const T *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh + (int64_t)cb * 64 * p.v.st;
    kload.issue(reinterpret_cast<const char *>(kb), 0, sq.k_len - cb * 64, k_tile);
    vload.issue(reinterpret_cast<const char *>(vb), 0, sq.k_len - cb * 64, v_tile);
  } else {
    const T *src = dp_wave ? (const T *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh + (int64_t)key * p.v.st
                           : (const T *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh + (int64_t)key * p.k.st;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 a = make_uint4(0, 0, 0, 0);
      if (key_ok && (!PAD || ks * 16 + g * 8 < p.D)) a = *reinterpret_cast<const uint4 *>(src + ks * 16 + g * 8);
      kvf[ks] = as_vec8<vec8>(a);
    }
    // The fragments pass through an empty asm statement: the compiler then waits for their
    // loads here, once.  Left to itself it waits at their first use inside the loop, in every
    // iteration, with vmcnt(0) -- which also waits for the tile copies in flight (issued from
    // inline assembly, so unknown to its counter bookkeeping) and undoes the prefetch.
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) asm volatile("" : "+v"(kvf[ks]));
  }
  floatx16 acc[DT];  // dV^T (S wave) or dK^T (dP wave): d x keys, summed over every q row of the column
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

  // operand read addresses inside a 32-row tile at offset 0; each role moves its copy of them on with the rings (below), so
  // that row offsets, and the half of a block, are instruction immediates
  using OA = OperandAddress<D>;
  typename OA::type rd[KS], tr[DT][2];
  {
    int tro[DT][2];
    transposed_offsets<D>(lane, tro);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) rd[ks] = OA::make(smem, TL::off(n, 2 * ks + g));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) tr[dt][0] = OA::make(smem, tro[dt][0]), tr[dt][1] = OA::make(smem, tro[dt][1]);
  }
  const uint32_t xbuf = opaque_lds_address(lds_address(smem) + S::kX + nh * 8192 + lane * 16);  // this pair's two P buffers
  const uint32_t vecs = opaque_lds_address(lds_address(smem) + S::kVec + g * 16);               // lse and delta of a Q stage

  // tiles whose first query index lies in [0, full_span) hold 32 queries
  const uint32_t full_span = sq.q_len >= S::kRows ? (uint32_t)(sq.q_len - S::kRows) + 1u : 0u;
  const uint32_t q_row_bytes = (uint32_t)p.q.st * 2u, do_row_bytes = (uint32_t)p.dout.st * 2u;
  // The q heads of the column form one stream of steps: behind a head's last entry the requests go on with the next
  // head's first one, so that a head costs no start-up of its own.  gq: head of the next request; [ent, ent_end): its
  // entries still to come.
  int gq = gq_first - 1, ent = 0, ent_end = 0;
  const int32_t *rows = nullptr;
  const char *qbase = nullptr, *dobase = nullptr;
  // lanes 0 .. 31: lse of the first 32 queries, lanes 32 .. 63: their delta; bytes from one query to the next
  const char *vec = nullptr;
  const int64_t vec_step = lane >= 32 ? (int64_t)sizeof(float) : p.lse.st * (int64_t)sizeof(float);
  auto next_head = [&]() __attribute__((always_inline)) {  // on to the next head that has entries, if there is one
    while (ent >= ent_end && gq + 1 < gq_end) {
      ++gq;
      const auto *a = late_arguments<BwdParams>();
      const int h = kvh * ratio + gq;
      const int tables = a->csc.num_heads, lh = tables == 1 ? 0 : tables == a->Hq ? h : kvh;
      rows = a->csc.idx + lh * a->csc.idx_sh;
      if (a->seg.entries) {  // (every wave has written the same values)
        const int first = __builtin_amdgcn_readfirstlane(part[0]), len = __builtin_amdgcn_readfirstlane(part[1]);
        const int before = (gq - gq_base) * len;  // entries of the heads before this one
        ent = first + max(__builtin_amdgcn_readfirstlane(part[2]) - before, 0);
        ent_end = first + min(__builtin_amdgcn_readfirstlane(part[3]) - before, len);
      } else {
        const int32_t *ptr = a->csc.ptr + lh * a->csc.ptr_sh + cb;
        if (cb < a->csc.num_rows) scalar_load2(ptr, ptr + 1, ent, ent_end);
        if (a->trim) ent_end = entry_lower_bound<EW>(rows, ent, ent_end, (sq.past + sq.q_len + 63) / 64);
      }
      qbase = reinterpret_cast<const char *>((const T *)a->q.ptr + sq.b * a->q.sb + h * a->q.sh);
      dobase = reinterpret_cast<const char *>((const T *)a->dout.ptr + sq.b * a->dout.sb + h * a->dout.sh);
      const float *lsebase = a->lse.ptr + sq.b * a->lse.sb + h * a->lse.sh;
      const float *deltabase = a->delta + ((int64_t)sq.b * a->Hq + h) * a->seqs.max_q_len;
      vec = reinterpret_cast<const char *>(lane >= 32 ? deltabase : lsebase) + (lane & 31) * vec_step;
    }
  };

  // asynchronous copy of 32-row q tile `tile`: Q and dO rows and the 32 lse / 32 delta
  // values (lanes 0..31 copy lse, lanes 32..63 delta; every wave copies the same
  // values, so that every wave issues the same number of load instructions).  Returns false
  // when rows had to be zero-filled, i.e. when the per-wave load count is not LPT.
  const uint32_t lds0 = lds_address(smem);
  auto issue = [&](int tile, int q_at, int do_at) __attribute__((always_inline)) -> bool {
    const int qi0 = tile * 32 - sq.past;  // query index of the tile's first row
    // main path: a listed block whose 32 rows all are queries (one scalar compare: a padding
    // entry, tile < 0, gives a negative qi0)
    if ((uint32_t)qi0 < full_span) {
      qload.issue_full_at(row_address(qbase, qi0, q_row_bytes), lds0 + q_at);
      doload.issue_full_at(row_address(dobase, qi0, do_row_bytes), lds0 + do_at);
      lds_dma4_lane(vec + (uint64_t)(uint32_t)qi0 * (uint64_t)vec_step, lds0 + S::kVec + q_at / (S::kTile / 256));
      return true;
    }
    char *const q_dst = smem + q_at, *const do_dst = smem + do_at, *const dst = smem + S::kVec + q_at / (S::kTile / 256);
    // Rows before the first query (qi < 0, when k is longer than q) and beyond the last are zero-filled.  Rare: everything
    // is computed here from opaque copies, or it would be held in registers through the loop, for each of its steps.
    int late = tid;
    asm volatile("" : "+v"(late));
    const auto *a = late_arguments<BwdParams>();
    Loader ql, dol;
    ql.init(late, a->q.st, a->D);
    dol.init(late, a->dout.st, a->D);
    const int lo = tile < 0 ? S::kRows : -qi0, hi = sq.q_len - qi0;
    const bool full = ql.issue(qbase + (int64_t)qi0 * q_row_bytes, lo, hi, q_dst);
    dol.issue(dobase + (int64_t)qi0 * do_row_bytes, lo, hi, do_dst);
    const char *src = vec + (int64_t)qi0 * vec_step;
    if (full) {
      lds_dma4_lane(src, lds_address(dst));
    } else if (wave == 0) {
      // rows outside the sequence: lse = +inf makes their probabilities 0
      const int row = late & 31;
      float x = late & 32 ? 0.f : INFINITY;
      if (row >= lo && row < hi) x = *reinterpret_cast<const float *>(src);
      reinterpret_cast<float *>(dst)[late & 63] = x;
    }
    return full;
  };

  // second half of the dP wave's work on a step (whose P the S wave published before the
  // last barrier): dS = P (dP - delta), dK^T += Q^T dS
  // (ta: operand addresses of its Q tile)
  auto finish_dk = [&](const auto &ta, int row_off, int qs_, int x_, const floatx16 &dp) __attribute__((always_inline)) {
    const uint32_t x = xbuf + x_, delta_s = vecs + qs_ / (S::kTile / 256) + 128;
    float ds[16];
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const floatx4 p4 = lds_read8_at<floatx4>(x + r4 * 1024);
      const floatx4 d4 = lds_read8_at<floatx4>(delta_s + r4 * 32);
      ds[r4 * 4 + 0] = p4.x * (dp[r4 * 4 + 0] - d4.x);  // without sm_scale
      ds[r4 * 4 + 1] = p4.y * (dp[r4 * 4 + 1] - d4.y);
      ds[r4 * 4 + 2] = p4.z * (dp[r4 * 4 + 2] - d4.z);
      ds[r4 * 4 + 3] = p4.w * (dp[r4 * 4 + 3] - d4.w);
    }
#pragma unroll
    for (int t2 = 0; t2 < 2; ++t2) {
      const vec8 dsb = M::pack(ds + t2 * 8);
      const int rowoff = t2 * 16 * TL::kRowBytes;
      vec8 qt[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) qt[dt] = lds_operand_tr<vec8>(ta[dt][0] + (row_off + rowoff), ta[dt][1] + (row_off + rowoff));
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[dt] = M::mma(qt[dt], dsb, acc[dt]);
    }
  };

  // The loop is instantiated once per role (not branched inside), so that the accumulators
  // are not merged through a join every iteration.
  auto run_column = [&](auto role_tag) __attribute__((always_inline)) {
  constexpr bool kDp = decltype(role_tag)::value;
  // A step is the number of its 32-row q tile; SUB: << 8 | the masks of its two quadrants, 4 bits each (steps
  // without an attended block are left out).  Without SUB steps come in pairs, the halves of a listed block.
  constexpr int kNone = INT_MAX;
  bool exact = true;  // every wave has issued exactly LPT load instructions per outstanding step
  static_assert(S::kAhead == 2 && S::kQStages == 4 && S::kDoStages == 3, "two steps in flight ahead of the one that is worked on");
  int left = 0, bits_next = 0, rb_next = 0;  // SUB: halves of block rb_next still to come
  // Requests the next step into place q_dst of the Q ring and do_dst of the dO ring (HALF 1: the second half of the block
  // whose first half, `before`, was requested last).
  auto request = [&](auto half_tag, int before, int q_dst, int do_dst) __attribute__((always_inline)) -> int {
    constexpr int kHalf = decltype(half_tag)::value;
    int step = kNone;
    if constexpr (SUB) {
      if (left == 0) {
        if (__builtin_expect(ent >= ent_end, 0)) next_head();
        if (ent < ent_end) {
          scalar_load2(rows + ent * EW, rows + ent * EW + 1, rb_next, bits_next);
          ++ent;
          bits_next = tile_quadrants(bits_next, p.csc.sub_block);
          // A listed tile without an attended block is no step where every quadrant of a step is multiplied: a product with
          // its rows could be 0 * inf.  (Elsewhere all waves sit the step out: the loop costs the steps of other tables, 4 x 3000
          // tokens of 12 heads of 64 with global blocks of 32, training 242.7 -> 246.0 us.)
          if constexpr (!kIdle) {
            while (__builtin_expect(bits_next == 0, 0)) {
              if (ent >= ent_end) next_head();
              if (ent >= ent_end) break;
              scalar_load2(rows + ent * EW, rows + ent * EW + 1, rb_next, bits_next);
              ++ent;
              bits_next = tile_quadrants(bits_next, p.csc.sub_block);
            }
          }
          left = ((bits_next & 255) != 0 ? 1 : 0) | ((bits_next >> 8) != 0 ? 2 : 0);
          if (kIdle && left == 0) left = 1;
        }
      }
      if (left != 0) {
        const int half = left & 1 ? 0 : 1;
        left &= left - 1;
        step = (rb_next * 2 + half) << 8 | (bits_next >> (8 * half) & 255);
      }
    } else if constexpr (kHalf == 0) {
      if (__builtin_expect(ent >= ent_end, 0)) next_head();
      if (ent < ent_end) {
        step = scalar_load(rows + ent) * 2;
        ++ent;
      }
    } else {
      if (before != kNone) step = before + 1;
    }
    if (step != kNone)
      exact = issue(SUB ? step >> 8 : step, q_dst, do_dst) && exact;
    return step;
  };
  static_assert(S::kQ == 0, "Q ring places are offsets");
  int do_0 = S::kDo, do_1 = S::kDo + S::kTile, do_2 = S::kDo + 2 * S::kTile;  // dO ring places of this step and the next two
  next_head();
  int cur = request(IntConst<0>{}, kNone, 0, do_0);
  int nxt = request(IntConst<1>{}, cur, S::kTile, do_1);
  if constexpr (kKvTiles) {
    // the K / V tiles are older than the requests above: everything has landed behind this wait
    wait_tile_loads();
    __syncthreads();
    const char *src = dp_wave ? v_tile : k_tile;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) kvf[ks] = lds_read8<vec8>(src + TL::off(nh * 32 + n, 2 * ks + g));
    // (the loop's first barrier comes before anything is copied over the two tiles: step 2's Q
    // tile is requested behind it, and the S waves write P behind it)
  }
  floatx16 dp_prev;
  int quad = 15, quad_prev = 15;  // SUB: masks of this wave's quadrant of steps t and t - 1 (0: both waves of the pair idle)
  int q_ring = 0;                 // Q ring place of this step (without SUB: of the block's first one)
  int x_ring = 0;                 // SUB: the P buffer of this step
  bool first = true;              // no step before this one
  // Operand addresses of the tiles that are read now, moved on with the rings.  S wave: rows of Q, columns of dO; dP wave:
  // rows of dO, columns of Q of the step before.  (Without SUB those of Q move once a block, its halves are immediates.)
  typename OA::type ra[KS], ta[DT][2];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) ra[ks] = rd[ks] + (kDp ? (int)S::kDo : 0);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 2; ++j) ta[dt][j] = tr[dt][j] + (kDp ? SUB ? 3 * S::kTile : 2 * S::kTile : (int)S::kDo);
  auto move_rows = [&](int by) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) ra[ks] += by;
  };
  auto move_cols = [&](int by) __attribute__((always_inline)) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) ta[dt][0] += by, ta[dt][1] += by;
  };
  // (not where steps are left out: the guards cost registers, 64 dims then lose their third workgroup, 241 -> 265 us)
  constexpr bool kLag = !kDp && !kIdle;
  constexpr bool kProductFirst = !kIdle;  // dP of a step ahead of dS of the one before
  vec8 lag_dot[DT], lag_pb;  // dO^T and P of the second half of the step before
  if constexpr (kLag) {
#pragma unroll
    for (int i = 0; i < 8; ++i) lag_pb[i] = 0;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) lag_dot[dt] = lag_pb;
  }
  auto finish_dv = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) acc[dt] = M::mma(lag_dot[dt], lag_pb, acc[dt]);
  };
  auto work = [&](auto half_tag) __attribute__((always_inline)) {
    constexpr int kHalf = decltype(half_tag)::value;  // (SUB: 0)
    if (nxt != kNone && exact)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPT) : "memory");
    else
      wait_tile_loads();
    __syncthreads();  // this step is visible, so is P of the step before; the stages of the step before that are free
    const int step = cur, cdo = do_0;
    const int qs_ = q_ring + kHalf * S::kTile, x_ = SUB ? x_ring : kHalf * 4096;
    // the Q place of the step before, and its P buffer
    const int pq = SUB ? (q_ring - S::kTile) & (3 * S::kTile) : kHalf ? q_ring : (q_ring ^ 2 * S::kTile) + S::kTile;
    cur = nxt;
    nxt = request(half_tag, cur, SUB || kHalf == 0 ? qs_ ^ 2 * S::kTile : (q_ring ^ 2 * S::kTile) + S::kTile, do_2);
    do_0 = do_1, do_1 = do_2, do_2 = cdo;
    if constexpr (SUB) quad = (step >> (4 * nh)) & 15;
    if constexpr (!kDp) {
      if (!kIdle || quad != 0) {
        const int pos0 = (SUB ? step >> 8 : step) * 32;  // first q position of this step
        // S = Q K^T : rows = 32 q positions, cols = 32 keys
        floatx16 sc;
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = 0.f;
        {
          vec8 qa[KS];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) qa[ks] = lds_operand<vec8>(ra[ks] + kHalf * S::kTile);
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) sc = M::mma(qa[ks], kvf[ks], sc);
        }
        if constexpr (kLag) finish_dv();
        // first dO^T operands do not depend on P
        vec8 dot[DT];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) dot[dt] = lds_operand_tr<vec8>(ta[dt][0], ta[dt][1]);
        // P = exp2(S scale - lse log2e).  Rows outside the sequence arrive with lse = +inf
        // (P = 0).  A row that saw no key has lse = -inf, but then every one of its entries
        // here is masked by causality and the select below discards the infinite value, so no
        // conversion is needed.  Masks are applied only in steps that need them (the diagonal
        // block and the last, partial column block): wave-uniform choice between two loops.
        const bool edge = (p.causal && (cb * 64 + nh * 32 + 31 > pos0)) || cb * 64 + 63 >= sq.k_len;
        // last visible q-row offset test: key is visible to row pos iff key <= pos
        const int kcmp = key_ok ? (p.causal ? key - pos0 : INT_MIN) : INT_MAX;  // masked iff kcmp > row offset
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
          // registers 4*r4 .. +3 are q rows 8*r4 + 4g + {0..3} of the step
          const floatx4 l4 = lds_read8_at<floatx4>(vecs + qs_ / (S::kTile / 256) + r4 * 32);
          const float lr[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            sc[r4 * 4 + i] = fast_exp2(fmaf(sc[r4 * 4 + i], p.scale_log2, -lr[i] * kLog2e));
        }
        if (edge) {
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[r] = kcmp > (r >> 2) * 8 + g * 4 + (r & 3) ? 0.f : sc[r];
        }
        if constexpr (SUB) {
          if (quad != 15) {  // wave-uniform: blocks of 16, the quadrant is not attended as a whole
            const int key_bits = quad >> (n >> 4);
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[r] = ((key_bits >> (2 * (r >> 3))) & 1) ? sc[r] : 0.f;
          }
        }
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          lds_write16_at(xbuf + x_ + r4 * 1024, floatx4{sc[r4 * 4], sc[r4 * 4 + 1], sc[r4 * 4 + 2], sc[r4 * 4 + 3]});
        // dV^T += dO^T P
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
          float pf[8];
#pragma unroll
          for (int i = 0; i < 8; ++i) pf[i] = sc[t2 * 8 + i];
          const vec8 pb = M::pack(pf);
          if (t2 == 1 && kLag) {
            lag_pb = pb;
            continue;
          }
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) {
            acc[dt] = M::mma(dot[dt], pb, acc[dt]);
            if (t2 == 0) {
              const int rowoff = 16 * TL::kRowBytes;
              (kLag ? lag_dot[dt] : dot[dt]) = lds_operand_tr<vec8>(ta[dt][0] + rowoff, ta[dt][1] + rowoff);
            }
          }
        }
      }
    } else {
      auto product = [&](floatx16 &dp) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) dp[r] = 0.f;
        if (!kIdle || quad != 0) {
          vec8 da[KS];
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) da[ks] = lds_operand<vec8>(ra[ks]);
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) dp = M::mma(da[ks], kvf[ks], dp);
        }
      };
      floatx16 dp;
      if constexpr (kProductFirst) product(dp);
      if (!first && (!kIdle || quad_prev != 0)) finish_dk(ta, SUB || kHalf ? 0 : S::kTile, pq, x_ ^ 4096, dp_prev);
      if (SUB || kHalf == 0) move_cols(qs_ - (SUB ? pq : pq - S::kTile));
      if constexpr (kProductFirst)
        dp_prev = dp;
      else
        product(dp_prev);
    }
    if constexpr (SUB) quad_prev = quad;
    first = false;
    if constexpr (kDp)
      move_rows(do_0 - cdo);
    else
      move_cols(do_0 - cdo);
  };
  while (cur != kNone) {
    work(IntConst<0>{});
    if constexpr (SUB) {
      const int next = (q_ring + S::kTile) & (3 * S::kTile);
      if constexpr (!kDp) move_rows(next - q_ring);
      q_ring = next, x_ring ^= 4096;
    } else {
      work(IntConst<1>{});
      const int next = q_ring ^ 2 * S::kTile;
      if constexpr (!kDp) move_rows(next - q_ring);
      q_ring = next;
    }
  }
  __syncthreads();  // P of the last step is visible
  if constexpr (kLag) finish_dv();
  if constexpr (kDp) {
    const int pq = SUB ? (q_ring - S::kTile) & (3 * S::kTile) : (q_ring ^ 2 * S::kTile) + S::kTile;
    if (!first && (!kIdle || quad_prev != 0)) finish_dk(ta, SUB ? 0 : S::kTile, pq, SUB ? x_ring ^ 4096 : 4096, dp_prev);
  }
  };
  if (dp_wave)
    run_column(BoolConst<true>{});
  else
    run_column(BoolConst<false>{});

  // every wave holds the finished dV^T (S wave) or dK^T (dP wave) of its 32 keys
  const auto *a = late_arguments<BwdParams>();
  const auto &outv = dp_wave ? a->dk : a->dv;
  const float out_scale = dp_wave ? a->sm_scale : 1.f;
  const int slot = a->seg.entries ? __builtin_amdgcn_readfirstlane(part[4]) : -1;
  if (head_split || slot >= 0) {  // fp32 partial of this q head, or of this segment
    if (!key_ok) return;
    float *outp;
    if (slot >= 0)
      outp = a->seg.partial + ((((int64_t)sq.b * gridDim.x + out_head) * a->seg.slots + slot) * 128 + (dp_wave ? 0 : 64) + nh * 32 + n) * p.D;
    else
      outp = (float *)outv.ptr + sq.b * outv.sb + out_head * outv.sh + (int64_t)key * outv.st;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        float4 o4;
        o4.x = acc[dt][r4 * 4 + 0] * out_scale;
        o4.y = acc[dt][r4 * 4 + 1] * out_scale;
        o4.z = acc[dt][r4 * 4 + 2] * out_scale;
        o4.w = acc[dt][r4 * 4 + 3] * out_scale;
        if (!PAD || dt * 32 + r4 * 8 + g * 4 < p.D) *reinterpret_cast<float4 *>(outp + dt * 32 + r4 * 8 + g * 4) = o4;
      }
    return;
  }
  if constexpr (D >= 128) {
    // each wave stages its 32 keys x D in one stage of the Q ring and writes whole rows (as in
    // the dQ pass: from the 128-wide tile on)
    __syncthreads();  // the dP waves have finished their last step (it reads the Q ring)
    const int key0 = cb * 64 + nh * 32;
    T *out_row0 = (T *)outv.ptr + sq.b * outv.sb + out_head * outv.sh + (int64_t)key0 * outv.st;
    store_tile_rows<T, D, PAD>(smem + S::kQ + wave * S::kTile, acc, out_scale, out_row0, outv.st, lane, 0, sq.k_len - key0, p.D);
  } else {
    if (!key_ok) return;
    T *outp = (T *)outv.ptr + sq.b * outv.sb + out_head * outv.sh + (int64_t)key * outv.st;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        if (!PAD || dt * 32 + r4 * 8 + g * 4 < p.D)
          *reinterpret_cast<uint2 *>(outp + dt * 32 + r4 * 8 + g * 4) =
              pack4<T>(acc[dt][r4 * 4] * out_scale, acc[dt][r4 * 4 + 1] * out_scale, acc[dt][r4 * 4 + 2] * out_scale,
                       acc[dt][r4 * 4 + 3] * out_scale);
      }
  }
}

// Explicit instantiations: with only the implicit ones the fp16 host stubs of
// these kernels are not emitted by this compiler version.
// (256-wide tiles: the zero-padding instantiations only; they also take head_dim 256 itself)
template __global__ void mfma_dq_kernel<bf16_t, 256, true, false>(const BwdParams, int);
template __global__ void mfma_dq_kernel<bf16_t, 256, true, true>(const BwdParams, int);
template __global__ void mfma_dq_kernel<f16_t, 256, true, false>(const BwdParams, int);
template __global__ void mfma_dq_kernel<f16_t, 256, true, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 256, true, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 256, true, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 256, true, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 256, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, false, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, false, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, false, false, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, false, true, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, false, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, false, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, true, false, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 128, true, true, true, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, false, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, false, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, true, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, true, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, false, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, false, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, true, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<bf16_t, 64, true, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, false, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, false, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, false, false, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, false, true, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, false, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, false, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, true, false, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 128, true, true, true, 96>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, false, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, false, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, true, false, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, true, false, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, false, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, false, true, true>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, true, true, false>(const BwdParams, int);
template __global__ void mfma_dq_pair_kernel<f16_t, 64, true, true, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 128, false, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 128, true, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 128, true, false, 96>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 128, false, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 128, true, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 128, true, true, 96>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 64, false, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 64, true, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 64, false, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<bf16_t, 64, true, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 128, false, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 128, true, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 128, true, false, 96>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 128, false, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 128, true, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 128, true, true, 96>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 64, false, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 64, true, false>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 64, false, true>(const BwdParams, int);
template __global__ void mfma_dkdv_kernel<f16_t, 64, true, true>(const BwdParams, int);

// Sum of the per-q-head dK / dV partials over each kv group (head_split mode).  One thread
// per 8 head dims of one (batch, kv head, key): blockIdx.y = 0 sums dK, 1 sums dV.
// part: fp32 [batch][Hq][keys][D] contiguous.
template <typename T>
__global__ __launch_bounds__(256) void dkdv_group_sum_kernel(const float *part_k, const float *part_v, TensorView dk,
                                                             TensorView dv, int batch, int Hq, int Hkv, int keys,
                                                             int D) {
  const int cpr = D / 8;
  const int64_t total = (int64_t)batch * Hkv * keys * cpr;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int ch = (int)(i % cpr);
  const int key = (int)((i / cpr) % keys);
  const int kvh = (int)((i / ((int64_t)cpr * keys)) % Hkv);
  const int b = (int)(i / ((int64_t)cpr * keys * Hkv));
  const int ratio = Hq / Hkv;
  const float *part = blockIdx.y ? part_v : part_k;
  const TensorView &out = blockIdx.y ? dv : dk;
  float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
  const float *src = part + (((int64_t)b * Hq + kvh * ratio) * keys + key) * D + ch * 8;
  for (int gq = 0; gq < ratio; ++gq) {
    const float4 a = *reinterpret_cast<const float4 *>(src + (int64_t)gq * keys * D);
    const float4 c = *reinterpret_cast<const float4 *>(src + (int64_t)gq * keys * D + 4);
    lo.x += a.x, lo.y += a.y, lo.z += a.z, lo.w += a.w;
    hi.x += c.x, hi.y += c.y, hi.z += c.z, hi.w += c.w;
  }
  T o8[8] = {from_float<T>(lo.x), from_float<T>(lo.y), from_float<T>(lo.z), from_float<T>(lo.w),
             from_float<T>(hi.x), from_float<T>(hi.y), from_float<T>(hi.z), from_float<T>(hi.w)};
  uint4 *dst = reinterpret_cast<uint4 *>((T *)out.ptr + b * out.sb + kvh * out.sh + (int64_t)key * out.st + ch * 8);
#pragma unroll
  for (int i = 0; i < (int)sizeof(T) / 2; ++i) dst[i] = reinterpret_cast<const uint4 *>(o8)[i];
}

// Sums of the segments of long rows and columns: eight workgroups per (place in the order, head, batch) add the partial sums
// of a row's segments in their order.  A slot has room for 128 rows of D floats: 128 q rows (dQ of a pair of rows), 64 q
// rows (dQ of a row), or 64 keys of dK and the same 64 of dV.  Bound: latency of a launch over few bytes (64 KB per
// segment at 128 dims).
constexpr int kSumParts = 8;  // workgroups per row: one or two 16-byte pieces of every segment per thread
template <typename TO>
__global__ __launch_bounds__(256) void segment_sum_kernel(const LutView lut, const SegView seg, SegRows what, TensorView a, TensorView b,
                                                          int Hq, int Hkv, int ratio, int D, float scale, int tokens,
                                                          int past, int trim_rows, int entry_width) {
  const int place = blockIdx.x / kSumParts, share = blockIdx.x % kSumParts, head = blockIdx.y;  // ratio: q heads per `head`
  const int h = head * ratio;  // a q head that the table head of this row serves
  const int lh = lut_head(lut, h, Hq, Hkv);
  const bool pairs = what == SegRows::kQueryPairs, queries = what != SegRows::kKeys;
  const int row = (pairs ? lut.pair_order : lut.order)[lh * lut.order_sh + place];
  const int32_t *ptr = lut.ptr + lh * lut.ptr_sh;
  int len;
  if (pairs) {
    // (as the dQ kernel counts: a row without queries contributes nothing)
    const int first_rb = past / 64, last_rb = (past + tokens - 1) / 64, ra = 2 * row;
    if (row > (last_rb >> 1) || row < (first_rb >> 1)) return;
    int e0 = ptr[ra], mid = ptr[ra + 1], e1 = mid;
    if (ra + 1 < lut.num_rows) e1 = ptr[ra + 2];
    if (ra < first_rb) e0 = mid;
    if (ra + 1 > last_rb) e1 = mid;
    len = (e1 - e0 + 1) / 2;
  } else {
    if (row * 64 >= tokens + (queries ? past : 0)) return;
    int e0 = ptr[row], e1 = ptr[row + 1];
    if (trim_rows > 0) {
      const int32_t *idx = lut.idx + lh * lut.idx_sh;
      int lo = e0, hi = e1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (idx[mid * entry_width] < trim_rows)
          lo = mid + 1;
        else
          hi = mid;
      }
      e1 = lo;
    }
    len = (e1 - e0) * ratio;  // (1 for queries)
  }
  const int segments = planned_segments(seg, place, len);
  if (segments < 2) return;
  const float *src = seg.partial + (((int64_t)blockIdx.z * gridDim.y + head) * seg.slots + place) * 128 * D;
  const int64_t step = (int64_t)seg.n[1] * 128 * D;
  const int pieces = D / 4, rows = (what == SegRows::kQueries ? 64 : 128) / kSumParts;
  for (int j = threadIdx.x; j < rows * pieces; j += 256) {
    const int i = share * rows * pieces + j, r = i / pieces, c = i % pieces;
    const int t = pairs ? row * 128 + r - past : queries ? row * 64 + r - past : row * 64 + (r & 63);
    if (t < 0 || t >= tokens) continue;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < segments; s0 += 4) {
      float4 w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = *reinterpret_cast<const float4 *>(src + min(s0 + k, segments - 1) * step + (int64_t)i * 4);
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (s0 + k < segments) v.x += w[k].x, v.y += w[k].y, v.z += w[k].z, v.w += w[k].w;
    }
    const TensorView &out = queries || r < 64 ? a : b;
    TO *dst = (TO *)out.ptr + blockIdx.z * out.sb + head * out.sh + (int64_t)t * out.st + c * 4;
    if constexpr (sizeof(TO) == 4)
      *reinterpret_cast<float4 *>(dst) = make_float4(v.x * scale, v.y * scale, v.z * scale, v.w * scale);
    else
      *reinterpret_cast<uint2 *>(dst) = pack4<TO>(v.x * scale, v.y * scale, v.z * scale, v.w * scale);
  }
}

template <typename TO>
static int launch_segment_sum_t(const LutView &lut, const SegView &seg, SegRows what, const TensorView &a, const TensorView &b, int heads,
                                const BwdParams &p, float scale, int tokens, int past, hipStream_t stream) {
  DK_NOTE_KERNEL("segment_sum_kernel");
  hipLaunchKernelGGL((segment_sum_kernel<TO>), dim3(seg.n[1] * kSumParts, heads, p.seqs.batch), dim3(256), 0, stream, lut, seg, what, a, b,
                     p.Hq, p.Hkv, p.Hq / heads, p.D, scale, tokens, past, p.trim ? (past + p.seqs.max_q_len + 63) / 64 : 0,
                     lut.entry_width);
  DK_HIP_CHECK(hipGetLastError());
  return DK_OK;
}
int launch_segment_sum(const LutView &lut, const SegView &seg, SegRows what, const TensorView &a, const TensorView &b, int dtype, int heads,
                       const BwdParams &p, float scale, int tokens, int past, hipStream_t stream) {
  switch (dtype) {
    case DK_BF16: return launch_segment_sum_t<bf16_t>(lut, seg, what, a, b, heads, p, scale, tokens, past, stream);
    case DK_F16: return launch_segment_sum_t<f16_t>(lut, seg, what, a, b, heads, p, scale, tokens, past, stream);
    default: return launch_segment_sum_t<float>(lut, seg, what, a, b, heads, p, scale, tokens, past, stream);
  }
}

template <typename T>
static int launch_group_sum_t(const BwdParams &p, const float *part_k, const float *part_v, hipStream_t stream) {
  const int keys = p.seqs.max_k_len;
  const int64_t total = (int64_t)p.seqs.batch * p.Hkv * keys * (p.D / 8);
  DK_NOTE_KERNEL("dkdv_group_sum_kernel");
  hipLaunchKernelGGL((dkdv_group_sum_kernel<T>), dim3((unsigned)cdiv64(total, 256), 2), dim3(256), 0, stream, part_k, part_v,
                     p.dk, p.dv, p.seqs.batch, p.Hq, p.Hkv, keys, p.D);
  DK_HIP_CHECK(hipGetLastError());
  return DK_OK;
}

int launch_dkdv_group_sum(const BwdParams &p, int dtype, const float *part_k, const float *part_v, hipStream_t stream) {
  switch (dtype) {
    case DK_BF16: return launch_group_sum_t<bf16_t>(p, part_k, part_v, stream);
    case DK_F16: return launch_group_sum_t<f16_t>(p, part_k, part_v, stream);
    default: return launch_group_sum_t<float>(p, part_k, part_v, stream);
  }
}

// Scratch for the head-split dK/dV pass: fp32 per-q-head partials of dK and dV (16-bit partials
// would round each head's share before the sum).  Zero when the pass would not be split (one
// q head per kv head).
size_t bwd_group_bytes(const BwdParams &p) {
  if (p.Hq == p.Hkv) return 0;
  const size_t need = 2 * (size_t)p.seqs.batch * p.Hq * p.seqs.max_k_len * p.D * sizeof(float);
  // beyond 4 GiB of partials (large batches) the pass keeps its in-workgroup loop over the group:
  // there are enough columns to balance then, and the scratch would rival the tensors themselves
  return need <= ((size_t)4 << 30) ? need : 0;
}

static BwdScratch mfma_bwd_scratch(const BwdParams &p, bool walk) {
  const int width = mfma_tile_width(p.D), per_cu = width == 64 ? 3 : width == 128 ? 2 : 1;
  return plan_bwd_scratch(p, bwd_group_bytes(p), width == 256 ? 0 : 256 * per_cu, true, 256 * per_cu, walk ? kWalkFrom : -1, kLeastGain);
}
size_t mfma_bwd_workspace_bytes(const BwdParams &p) { return mfma_bwd_scratch(p, true).bytes; }

bool mfma_bwd_supported(const BwdParams &p, int dtype) {
  return (dtype == DK_BF16 || dtype == DK_F16) && mfma_head_dim_ok(p.D) && p.csr.block_rows == 64 &&
         p.csr.block_cols == 64 && p.csr.sub_block == p.csc.sub_block &&
         (p.csr.sub_block != 0 || (p.csr.entry_width == 1 && p.csc.entry_width == 1)) &&
         p.csc.block_rows == 64 && p.csc.block_cols == 64 &&
         p.vec_ok && mfma_row_bytes_ok(p.q) && mfma_row_bytes_ok(p.k) && mfma_row_bytes_ok(p.v) &&
         mfma_row_bytes_ok(p.dout);
}

template <typename T, int D, bool PAD, bool SUB, int KD = D>
static int launch_bwd_td(const BwdParams &p, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  const SeqView &s = p.seqs;
  constexpr int smem_dq = 2 * 2 * Tile<D>::kBytes;
  constexpr int smem_dkdv = DkdvSmem<D>::kBytes;
  DK_ALLOW_DYNAMIC_LDS((mfma_dkdv_kernel<T, D, PAD, SUB, KD>), smem_dkdv);
  const int past = p.causal ? s.max_k_len - s.max_q_len : 0;
  const int tiles = (past + s.max_q_len - 1) / 64 - past / 64 + 1;
  DK_REQUIRE(tiles <= 65535 && cdiv(s.max_k_len, 64) <= 65535 && p.csc.num_rows <= 65535 &&
                 (!(p.csr.order || p.csr.pair_order) || p.csr.num_rows <= 65535),
             "sequence too long for one launch");
  const BwdScratch scratch = usable_bwd_scratch([&](bool walk) { return mfma_bwd_scratch(p, walk); }, workspace, workspace_bytes);
  // dQ first: it also writes delta, which the dK/dV pass reads
  if constexpr (D <= 128) {  // two table rows per workgroup
    int pairs = (((past + s.max_q_len - 1) / 64) >> 1) - ((past / 64) >> 1) + 1;
    if (p.csr.pair_order) pairs = (p.csr.num_rows + 1) / 2;  // handed out in the table's order: all of them
    BwdParams pq = p;
    if (p.csr.pair_order && segment_items(scratch.dq, pairs) <= 65535) pq.seg = scratch.dq;
    const int items = (int)segment_items(pq.seg, pairs);
    pq.csr.rot = head_rotation(p.csr, p.Hq, items);  // (uneven heads: dealt to the queues in rotation)
    DK_NOTE_KERNEL(pq.csr.rot ? "mfma_dq_pair_kernel, heads in rotation" : "mfma_dq_pair_kernel");
    if (pq.seg.entries) {
      DK_ALLOW_DYNAMIC_LDS((mfma_dq_pair_kernel<T, D, PAD, SUB, true, KD>), smem_dq);
      hipLaunchKernelGGL((mfma_dq_pair_kernel<T, D, PAD, SUB, true, KD>), dim3(p.Hq, items, s.batch), dim3(256), smem_dq, stream, pq, pairs);
    } else {
      DK_ALLOW_DYNAMIC_LDS((mfma_dq_pair_kernel<T, D, PAD, SUB, false, KD>), smem_dq);
      hipLaunchKernelGGL((mfma_dq_pair_kernel<T, D, PAD, SUB, false, KD>), dim3(p.Hq, items, s.batch), dim3(256), smem_dq, stream, pq, pairs);
    }
    DK_HIP_CHECK(hipGetLastError());
    if (pq.seg.entries) {
      const int dtype = std::is_same<T, bf16_t>::value ? DK_BF16 : DK_F16;
      if (int rc = launch_segment_sum(p.csr, pq.seg, SegRows::kQueryPairs, p.dq, p.dq, dtype, p.Hq, p, p.sm_scale, s.max_q_len, past, stream)) return rc;
    }
  } else {
    DK_ALLOW_DYNAMIC_LDS((mfma_dq_kernel<T, D, PAD, SUB>), smem_dq);
    const int rows = p.csr.order ? p.csr.num_rows : tiles;  // handed out in the table's order: all of them
    BwdParams pq = p;
    pq.csr.rot = head_rotation(p.csr, p.Hq, rows);
    DK_NOTE_KERNEL(pq.csr.rot ? "mfma_dq_kernel, heads in rotation" : "mfma_dq_kernel");
    hipLaunchKernelGGL((mfma_dq_kernel<T, D, PAD, SUB>), dim3(p.Hq, rows, s.batch), dim3(256), smem_dq, stream, pq, rows);
  }
  DK_HIP_CHECK(hipGetLastError());
  // With several q heads per kv head a workgroup walks a column for all of them, long columns in segments, or, where
  // walk_groups() says so, the pass runs one workgroup per q head into per-head partials and a bandwidth-bound kernel sums
  // each group.  (Without lengths to cut by, the longest column - a vertical one near the start: every later q block, times
  // the group's size - alone would outlast the average CU's share of the whole pass.)
  const bool per_q_head = scratch.group > 0;
  // The table's longest-first order is taken unless the heads along grid.x are a multiple of the
  // 32 (XCD, shader engine) queues that the hardware deals workgroups to in turn: then every queue
  // serves whole heads, long columns and short ones alike, and the ascending order keeps
  // neighbouring columns - which share most of their Q / dO tiles - together in time (1.7 %
  // faster on the 32-head benchmark; with 8 or 16 heads the order is worth 20 - 40 %).
  BwdParams po = p;
  po.trim = p.csc.row_lengths && p.csr.num_rows > tiles + past / 64;  // (tables with lengths list their entries in order)
  if (p.csc.order && segment_items(scratch.kv, p.csc.num_rows) <= 65535) po.seg = scratch.kv;
  if (((per_q_head ? p.Hq : p.Hkv) % 32) == 0 && !po.seg.entries) po.csc.order = nullptr;
  // with a hand-out order the grid covers every column of the table (those beyond the keys exit at once)
  const int cblocks = po.csc.order ? (int)segment_items(po.seg, p.csc.num_rows) : cdiv(s.max_k_len, 64);
  po.csc.rot = head_rotation(p.csc, per_q_head ? p.Hq : p.Hkv, cblocks);
  if (per_q_head) {
    BwdParams pp = po;
    const int64_t keys = s.max_k_len;
    float *part_k = (float *)workspace, *part_v = part_k + (int64_t)s.batch * p.Hq * keys * p.D;
    pp.dk = TensorView{part_k, p.Hq * keys * p.D, keys * p.D, p.D};
    pp.dv = TensorView{part_v, p.Hq * keys * p.D, keys * p.D, p.D};
    DK_NOTE_KERNEL(pp.csc.rot ? "mfma_dkdv_kernel (one workgroup per q head), heads in rotation"
                              : "mfma_dkdv_kernel (one workgroup per q head)");
    hipLaunchKernelGGL((mfma_dkdv_kernel<T, D, PAD, SUB, KD>), dim3(p.Hq, cblocks, s.batch), dim3(256), smem_dkdv, stream, pp, 1);
    DK_HIP_CHECK(hipGetLastError());
    if (pp.seg.entries)
      if (int rc = launch_segment_sum(p.csc, pp.seg, SegRows::kKeys, pp.dk, pp.dv, DK_F32, p.Hq, po, 1.f, s.max_k_len, past, stream)) return rc;
    return launch_group_sum_t<T>(p, part_k, part_v, stream);
  }
  DK_NOTE_KERNEL(po.csc.rot ? "mfma_dkdv_kernel, heads in rotation" : "mfma_dkdv_kernel");
  hipLaunchKernelGGL((mfma_dkdv_kernel<T, D, PAD, SUB, KD>), dim3(p.Hkv, cblocks, s.batch), dim3(256), smem_dkdv, stream, po, 0);
  DK_HIP_CHECK(hipGetLastError());
  if (po.seg.entries) {
    const int dtype = std::is_same<T, bf16_t>::value ? DK_BF16 : DK_F16;
    return launch_segment_sum(p.csc, po.seg, SegRows::kKeys, p.dk, p.dv, dtype, p.Hkv, po, 1.f, s.max_k_len, past, stream);
  }
  return DK_OK;
}

// head dims below the tile width (64 or 128) run the zero-padded instantiation, those of 72 - 96 with 96 of the 128
// dims multiplied (as in the forward; training, 96 dims, 2 x 3000 tokens, 32 / 8 heads: 516 -> 460 us)
template <typename T>
static int launch_bwd_t(const BwdParams &p, void *ws, size_t ws_bytes, hipStream_t stream) {
  if (p.D > 128)  // 256-wide tiles, one wave per SIMD
    return p.csr.sub_block ? launch_bwd_td<T, 256, true, true>(p, ws, ws_bytes, stream)
                           : launch_bwd_td<T, 256, true, false>(p, ws, ws_bytes, stream);
  if (p.csr.sub_block) {  // entries carry a bit mask over the pattern's 16- or 32-token blocks
    if (p.D == 128) return launch_bwd_td<T, 128, false, true>(p, ws, ws_bytes, stream);
    if (p.D == 64) return launch_bwd_td<T, 64, false, true>(p, ws, ws_bytes, stream);
    if (p.D > 64 && p.D <= 96) return launch_bwd_td<T, 128, true, true, 96>(p, ws, ws_bytes, stream);
    return p.D > 64 ? launch_bwd_td<T, 128, true, true>(p, ws, ws_bytes, stream)
                    : launch_bwd_td<T, 64, true, true>(p, ws, ws_bytes, stream);
  }
  if (p.D == 128) return launch_bwd_td<T, 128, false, false>(p, ws, ws_bytes, stream);
  if (p.D == 64) return launch_bwd_td<T, 64, false, false>(p, ws, ws_bytes, stream);
  if (p.D > 64 && p.D <= 96) return launch_bwd_td<T, 128, true, false, 96>(p, ws, ws_bytes, stream);
  return p.D > 64 ? launch_bwd_td<T, 128, true, false>(p, ws, ws_bytes, stream)
                  : launch_bwd_td<T, 64, true, false>(p, ws, ws_bytes, stream);
}

int launch_mfma_bwd(const BwdParams &p, int dtype, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  return dtype == DK_BF16 ? launch_bwd_t<bf16_t>(p, workspace, workspace_bytes, stream)
                          : launch_bwd_t<f16_t>(p, workspace, workspace_bytes, stream);
}

}  // namespace dk
