// fp32 inputs on the matrix cores of gfx950: v_mfma_f32_32x32x2_f32, head dims up to 128 (multiples
// of 4, zero-padded on chip to 64, 96 or 128), 64 x 64 tiles with one int per table entry.  Forward
// (fixed, padded, packed and single-token sequences, LSE) and backward (dQ over CSR rows, dK/dV over
// CSC columns; delta = rowsum(O * dO) - dLSE by a small kernel ahead of them).  fp32 products with
// fp32 accumulation: results agree with the generic fp32-FMA kernels to rounding.
//
//   D(32x32) += A(32x2) * B(2x32):  A operand, lane l: row l%32, k = l/32 (one float)
//                                   B operand, lane l: col l%32, k = l/32
//                                   accumulator, lane l, register r: col l%32, row 8(r/4) + 4(l/32) + r%4
//
// The contraction index of a product may be walked in any order as long as A and B agree, so:
//  * products over head dims (S = K Q^T, dP = V dO^T, ...) give lane (x, g) the dims KD/2 g + s in
//    step s: a lane's operands of KD/2 steps are consecutive floats (16-byte reads);
//  * products over keys or q rows (O^T += V^T P^T, dQ^T += K^T dS^T, dV^T += dO^T P, dK^T += Q^T dS)
//    take step r = the pair of rows that accumulator register r of the two half-waves stands for,
//    8(r/4) + r%4 and 8(r/4) + 4 + r%4: the second operand is then the lane's own register r of
//    the S / P / dS accumulator, with no exchange between lanes, and the first one a 4-byte LDS read
//    per lane, 32 consecutive floats of one tile row per half-wave.
//
// Work split: a workgroup of four waves takes one 64 x 64 block at a time and each wave one of its
// 32 x 32 quadrants (row half x key half), so that a block's four products run on the four SIMDs at
// once and the waves' partial results (over the key halves, or the q-row halves in the dK/dV pass)
// are added through LDS once, at the end.  An instruction of this shape occupies the matrix pipe for
// 64 cycles, so one wave per SIMD covers its own LDS reads, exponentials and bookkeeping; tiles are
// copied HBM -> LDS asynchronously (LDS DMA) into two stages, the next block's while the current one
// is multiplied.  Bound: fp32 MFMA (a large fp32 product of the vendor library: 153 TFLOP/s).  Measured
// forward / backward, us: 1 x 8192 tokens, 32 heads of 64 dims, local 16, vert 8: 906 / 2765 = 101 / 82
// TFLOP/s (two waves of 32 x 64 quadrants over a single stage: 1114 / 3836); 8 heads x 1024 tokens of 64
// dims: 26 / 126 (52 / 262); 16 heads x 2000 tokens of 128 dims, local 8, vert 4: 128 / 430 (fp32-FMA
// kernels of generic_*.hip: 474 / 3189; backward with every column whole: 491, the longest one's time).
#include <type_traits>

#include "bwd_scratch.h"
#include "common.h"
#include "device_common.h"
#include "mfma_common.h"

namespace dk {

size_t bwd_group_bytes(const BwdParams &p);
int launch_segment_sum(const LutView &lut, const SegView &seg, SegRows what, const TensorView &a, const TensorView &b, int dtype, int heads,
                       const BwdParams &p, float scale, int tokens, int past, hipStream_t stream);
int launch_dkdv_group_sum(const BwdParams &p, int dtype, const float *part_k, const float *part_v, hipStream_t stream);

namespace f32 {

constexpr int NT = 256;  // threads: four waves

__device__ __forceinline__ floatx16 mma(float a, float b, floatx16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// KD: head dims multiplied (64, 96 or 128); tiles are 64 rows of W = 64 or 128 floats in the
// swizzled layout of a 16-bit tile of twice the width (mfma_common.h).  PAD: the tensors hold fewer
// head dims than KD (the others are zeros in LDS) or than W (never read).
template <int KD, bool PAD>
struct Shape {
  static constexpr int W = KD <= 64 ? 64 : 128;
  using TL = Tile<2 * W>;
  using Loader = TileLoader<2 * W, NT, PAD>;
  static constexpr int HD = KD / 2;   // head dims per lane of a product over head dims
  static constexpr int DT = KD / 32;  // 32-dim tiles of a result
  static constexpr int kTile = TL::kBytes;
  static constexpr int kStage = 2 * kTile;  // two tiles: K and V, or Q and dO
  static constexpr int kSmem = 2 * kStage;
};

// Result of dot_dims: above 64 dims the last chain is left to be added where the sum is read, so that
// nobody waits for the matrix core in between.
template <int KD>
struct DimSum {
  floatx16 sum, last;
  __device__ __forceinline__ float operator[](int r) const { return sum[r] + last[r]; }
};
template <>
struct DimSum<64> {
  floatx16 sum;
  __device__ __forceinline__ float operator[](int r) const { return sum[r]; }
};

// X Y^T (32 x 32) over the head dims: rows = rows row0 .. row0 + 31 of tile `xt` (row0 a multiple of
// 32), columns = the lanes' own rows of Y, yf[s] = dim HD g + s of that row.
//
// Above 64 dims the sum is built from chains of 32 dims (one batch of operand reads each), added on the
// vector unit while the matrix core multiplies the next one.  Relative error of the output against 64
// bits, 300 tokens of 128 dims: one chain of 128 roundings 3.1e-7, chains of 32 1.7e-7, the fp32-FMA
// kernels (four chains of 32) 2.0e-7; dQ 4.6e-7, 3.5e-7, 3.6e-7.  Price: 16 heads x 2000 tokens
// of 128 dims, forward 126 -> 128 us, forward and backward 608 -> 621.
template <int KD, bool PAD>
__device__ __forceinline__ DimSum<KD> dot_dims(const char *xt, int row0, const float (&yf)[KD / 2], int lane) {
  using S = Shape<KD, PAD>;
  constexpr int CH = S::HD / 4, B = 4;  // 16-byte chunks per lane, read in batches ahead of their multiplies
  static_assert(CH % B == 0, "whole batches");
  constexpr int RUN = KD <= 64 ? CH / B : 1;  // batches per chain
  // (opaque: the read addresses - a few XORs per 64-cycle multiply - are computed here; hoisted out of
  // the caller's loop they would occupy registers throughout)
  asm volatile("" : "+v"(lane));
  const int m = lane & 31, g = lane >> 5;
  const char *row = xt + (row0 + m) * S::TL::kRowBytes;
  const int swz = S::TL::swz(m);
  float4 x[2][B];
#pragma unroll
  for (int i = 0; i < B; ++i) x[0][i] = *reinterpret_cast<const float4 *>(row + (((g * CH + i) ^ swz) << 4));
  floatx16 chain[2], sum;  // the chain in work and the finished one before it; their sum
#pragma unroll
  for (int b = 0; b < CH / B; ++b) {
    if (b + 1 < CH / B) {
#pragma unroll
      for (int i = 0; i < B; ++i)
        x[(b + 1) & 1][i] = *reinterpret_cast<const float4 *>(row + (((g * CH + (b + 1) * B + i) ^ swz) << 4));
    }
    __builtin_amdgcn_sched_barrier(0);
    floatx16 &acc = chain[(b / RUN) & 1];
    if (b % RUN == 0) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const float4 w = x[b & 1][i];
      acc = mma(w.x, yf[(b * B + i) * 4], acc);
      acc = mma(w.y, yf[(b * B + i) * 4 + 1], acc);
      acc = mma(w.z, yf[(b * B + i) * 4 + 2], acc);
      acc = mma(w.w, yf[(b * B + i) * 4 + 3], acc);
      if (RUN == 1 && b > 0 && i == 0) {  // (the chain before has long left the matrix core)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = b == 1 ? chain[0][r] : sum[r] + chain[(b - 1) & 1][r];
        asm volatile("" : "+v"(sum));  // (here, not sunk behind the last chain with all of them alive)
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  if constexpr (RUN > 1)
    return {chain[0]};
  else
    return {sum, chain[(CH / B - 1) & 1]};
}

// acc[dt](32 dims x 32 columns) += T^T(dims x rows) * W(rows x columns) over the 32 rows row0 .. row0 + 31 of
// tile `t`: step r takes rows 8(r/4) + r%4 (+4 in the upper half-wave), w[r] is the lane's own
// accumulator register r of W^T's product (column = lane % 32).
template <int KD, bool PAD>
__device__ __forceinline__ void dot_rows(const char *t, int row0, const floatx16 &w, int lane, floatx16 (&acc)[KD / 32]) {
  using S = Shape<KD, PAD>;
  constexpr int DT = S::DT, B = 2;  // steps per batch of operand reads
  asm volatile("" : "+v"(lane));  // as in dot_dims
  const int g = lane >> 5, m = lane & 31;
  const char *base = t + row0 * S::TL::kRowBytes + (m & 3) * 4;
  auto read = [&](int r, int dt) {
    const int row = (r >> 2) * 8 + g * 4 + (r & 3);
    return *reinterpret_cast<const float *>(base + S::TL::off(row, dt * 8 + (m >> 2)));
  };
  float a[2][B][DT];
#pragma unroll
  for (int i = 0; i < B; ++i)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) a[0][i][dt] = read(i, dt);
#pragma unroll
  for (int b = 0; b < 16 / B; ++b) {
    if (b + 1 < 16 / B) {
#pragma unroll
      for (int i = 0; i < B; ++i)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) a[(b + 1) & 1][i][dt] = read((b + 1) * B + i, dt);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < B; ++i)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[dt] = mma(a[b & 1][i][dt], w[b * B + i], acc[dt]);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// consecutive floats of a row (dims HD g ..) as one lane's operands; zeros when !ok or beyond d
template <int HD>
__device__ __forceinline__ void load_frag(const float *row, bool ok, int g, int d, float (&f)[HD]) {
#pragma unroll
  for (int c = 0; c < HD / 4; ++c) {
    float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
    if (ok && g * HD + c * 4 < d) w = *reinterpret_cast<const float4 *>(row + g * HD + c * 4);
    f[c * 4] = w.x, f[c * 4 + 1] = w.y, f[c * 4 + 2] = w.z, f[c * 4 + 3] = w.w;
  }
}

// Addition of two waves' accumulators through LDS.  Each wave of a pair keeps half of the 32-dim
// tiles (wave 0 the first half, wave 1 the second and the middle one of an odd count): it hands the
// others over and adds the partner's share, scaled by `own` / `other`, to its own.  `buf`: DT * 4 KB
// per pair.  Between give and take: a barrier.  (`second` is wave-uniform but not a compile-time
// constant: accumulators are picked by selects between values in fixed registers - picked by a
// branch they end up in scratch memory.)
__device__ __forceinline__ void give_tile(const float (&v)[16], float *buf, int dt, int lane) {
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4)
    *reinterpret_cast<float4 *>(buf + ((dt * 4 + r4) * 64 + lane) * 4) =
        make_float4(v[r4 * 4], v[r4 * 4 + 1], v[r4 * 4 + 2], v[r4 * 4 + 3]);
}
template <int DT>
__device__ __forceinline__ void give_half(const floatx16 (&acc)[DT], bool second, float *buf, int lane) {
  constexpr int N = DT / 2;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = second ? acc[i][r] : acc[DT - N + i][r];
    give_tile(v, buf, second ? i : DT - N + i, lane);
  }
  if (DT % 2 && !second) {
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = acc[N][r];
    give_tile(v, buf, N, lane);
  }
}
// ... and the finished half of the row goes to memory (dims 32 dt + 8 r4 + 4 g + {0..3})
__device__ __forceinline__ void take_tile(const float (&v)[16], const float *buf, int dt, int lane, float own, float other,
                                          float *row, bool ok, int d) {
#pragma unroll
  for (int r4 = 0; r4 < 4; ++r4) {
    const float4 p = *reinterpret_cast<const float4 *>(buf + ((dt * 4 + r4) * 64 + lane) * 4);
    const int d0 = dt * 32 + r4 * 8 + (lane >> 5) * 4;
    if (ok && d0 < d)
      *reinterpret_cast<float4 *>(row + d0) = make_float4(v[r4 * 4] * own + p.x * other, v[r4 * 4 + 1] * own + p.y * other,
                                                          v[r4 * 4 + 2] * own + p.z * other, v[r4 * 4 + 3] * own + p.w * other);
  }
}
template <int DT>
__device__ __forceinline__ void take_half_and_store(const floatx16 (&acc)[DT], bool second, const float *buf, int lane,
                                                    float own, float other, float *row, bool ok, int d) {
  constexpr int N = DT / 2;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = second ? acc[DT - N + i][r] : acc[i][r];
    take_tile(v, buf, second ? DT - N + i : i, lane, own, other, row, ok, d);
  }
  if (DT % 2 && second) {
    float v[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) v[r] = acc[N][r];
    take_tile(v, buf, N, lane, own, other, row, ok, d);
  }
}

template <int DT>
__device__ __forceinline__ void clear(floatx16 (&acc)[DT]) {
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;
}

template <int V>
struct Stage {  // compile-time stage passed to a generic lambda
  static constexpr int value = V;
};

// ---------------------------------------------------------------------------
// forward: workgroup = 64 q rows of one head; wave = 32 rows x 32 keys of every block, with its own
// running maximum and sum (the two key halves of a row are merged at the end)
// ---------------------------------------------------------------------------
template <int KD, bool PAD>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(KD <= 64 ? 2 : 1, KD <= 64 ? 2 : 1))) void fwd_kernel(
    const FwdParams p, int tiles_y) {
  using S = Shape<KD, PAD>;
  extern __shared__ __align__(16) char smem[];
  SeqInfo sq;
  int tile;
  bool has_rows;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (p.csr.order && !p.seqs.packed) {  // the table's own order, longest rows first (the grid covers every row of it)
    sq = load_seq(p.seqs, blockIdx.z, p.causal);
    tile = scalar_load(p.csr.order + lut_head(p.csr, grid_head(p.csr), p.Hq, p.Hkv) * p.csr.order_sh + blockIdx.y) - sq.past / 64;
    has_rows = tile >= 0 && tile < seq_row_blocks(sq, 64);
  } else {
    has_rows = resolve_tile(p.seqs, p.causal, 64, 1, tiles_y - 1 - (int)blockIdx.y, blockIdx.z, sq, tile);
  }
  if (p.seqs.packed && p.seqs.zero_outside && blockIdx.y == 0) lse_outside_packed(p.seqs, p.lse, grid_head(p.csr), 1, tid, NT);
  if (p.seqs.zero_outside && !p.seqs.packed)
    zero_rows_outside<float>(p.seqs, sq, blockIdx.y, tiles_y, p.o, p.lse, grid_head(p.csr), 1, p.D, p.vec_ok, tid, NT);
  if (!has_rows) return;
  const int rb = sq.past / 64 + tile;
  const int rh = wave & 1, kh = wave >> 1;  // row half, key half
  const int h = grid_head(p.csr), kvh = __builtin_amdgcn_readfirstlane(h / (p.Hq / p.Hkv));
  const int m = lane & 31, g = lane >> 5;
  const int row0 = rb * 64 + rh * 32;
  const int pos = row0 + m, qi = pos - sq.past;
  const bool row_ok = qi >= 0 && qi < sq.q_len;
  if constexpr (PAD) {  // the slots of the head dims beyond p.D stay zero for the whole kernel
    zero_tiles<NT>(smem, S::kSmem, tid);
    __syncthreads();
  }

  const int lh = lut_head(p.csr, h, p.Hq, p.Hkv);
  int e0 = 0, e1 = 0;
  if (rb < p.csr.num_rows)
    scalar_load2(p.csr.ptr + lh * p.csr.ptr_sh + rb, p.csr.ptr + lh * p.csr.ptr_sh + rb + 1, e0, e1);
  const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
  const float *kbase = (const float *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh + (int64_t)sq.k_start * p.k.st;
  const float *vbase = (const float *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh + (int64_t)sq.k_start * p.v.st;
  typename S::Loader kload, vload;
  kload.init(tid, 2 * p.k.st, 2 * p.D);
  vload.init(tid, 2 * p.v.st, 2 * p.D);
  auto issue = [&](int col, int stage) {
    const int key0 = col * 64, valid = col < 0 ? 0 : sq.k_len - key0;
    kload.issue(reinterpret_cast<const char *>(kbase + (int64_t)key0 * p.k.st), 0, valid, smem + stage * S::kStage);
    vload.issue(reinterpret_cast<const char *>(vbase + (int64_t)key0 * p.v.st), 0, valid, smem + stage * S::kStage + S::kTile);
  };
  int col_cur = 0, col_pending = 0;  // the block in work and (requested one block early) the one after it
  if (e0 < e1) {
    col_cur = scalar_load(cols + e0);
    issue(col_cur, 0);
    col_pending = e0 + 1 < e1 ? cols[e0 + 1] : 0;
  }
  float qf[S::HD];
  load_frag<S::HD>((const float *)p.q.ptr + sq.b * p.q.sb + h * p.q.sh + (int64_t)(sq.q_start + qi) * p.q.st, row_ok, g, p.D, qf);

  floatx16 oacc[S::DT];
  clear(oacc);
  float m_run = -INFINITY, l_run = 0.f;  // running maximum (log2 domain) and this lane's share of the row sum
  const int lim = p.causal ? min(pos, sq.k_len - 1) : sq.k_len - 1;  // last visible key of this row

  auto block_step = [&](int e, auto stage_tag) {
    constexpr int stage = decltype(stage_tag)::value;
    const int col = col_cur;
    wait_tile_loads();
    __syncthreads();  // the block's tiles are visible; every wave is done with the other stage
    col_cur = __builtin_amdgcn_readfirstlane(col_pending);
    if (e + 2 < e1) col_pending = cols[e + 2];
    if (e + 1 < e1) issue(col_cur, stage ^ 1);
    const int key0 = col * 64 + kh * 32;  // first key of this wave's half
    if (col < 0 || key0 >= sq.k_len || (p.causal && key0 > row0 + 31)) return;  // nothing visible (wave-uniform)
    const char *ks = smem + stage * S::kStage, *vs = ks + S::kTile;
    // S^T = K Q^T: lane = q row, registers = keys 8(r/4) + 4g + r%4 of the half
    const DimSum<KD> dots = dot_dims<KD, PAD>(ks, kh * 32, qf, lane);
    floatx16 s;
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = key0 + (r >> 2) * 8 + g * 4 + (r & 3);
      s[r] = key > lim || !row_ok ? -INFINITY : dots[r] * p.scale_log2;
      mx = fmaxf(mx, s[r]);
    }
    mx = max_with_other_half(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(s[r] - m_use);
      psum += s[r];
    }
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {  // wave-uniform: some row's maximum has moved
      const float alpha = fast_exp2(m_run - m_use);  // exp2(-inf) = 0 before the first visible key
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < S::DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
      m_run = m_new;
    }
    l_run += psum;
    dot_rows<KD, PAD>(vs, kh * 32, s, lane, oacc);  // O^T += V^T P^T
  };
  for (int e = e0; e < e1; e += 2) {
    block_step(e, Stage<0>{});
    if (e + 1 < e1) block_step(e + 1, Stage<1>{});
  }
  l_run += xor32(l_run);

  // ---- merge of the two key halves of a row: maxima and sums, then the accumulators by halves ----
  __syncthreads();  // the tiles are free
  float *ml = reinterpret_cast<float *>(smem + 2 * S::DT * 4096);  // behind the exchange areas of the two pairs
  float *buf = reinterpret_cast<float *>(smem) + rh * S::DT * 1024;
  if (g == 0) {
    ml[(wave * 2) * 32 + m] = m_run;
    ml[(wave * 2 + 1) * 32 + m] = l_run;
  }
  give_half<S::DT>(oacc, kh == 1, buf, lane);
  __syncthreads();
  const int mate = wave ^ 2;
  const float m_o = ml[(mate * 2) * 32 + m], l_o = ml[(mate * 2 + 1) * 32 + m];
  const float m_all = fmaxf(m_run, m_o), m_ref = m_all == -INFINITY ? 0.f : m_all;
  const float a_own = fast_exp2(m_run - m_ref), a_other = fast_exp2(m_o - m_ref);
  const float l_all = l_run * a_own + l_o * a_other;
  const float inv = l_all > 0.f ? 1.f / l_all : 0.f;
  float *orow = (float *)p.o.ptr + sq.b * p.o.sb + h * p.o.sh + (int64_t)(sq.q_start + qi) * p.o.st;
  take_half_and_store<S::DT>(oacc, kh == 1, buf, lane, a_own * inv, a_other * inv, orow, row_ok, p.D);
  if (row_ok && p.lse.ptr && g == 0 && kh == 0)
    p.lse.ptr[sq.b * p.lse.sb + h * p.lse.sh + (int64_t)(sq.q_start + qi) * p.lse.st] =
        l_all > 0.f ? (m_all + log2f(l_all)) * kLn2 : -INFINITY;
}

// ---------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------
// delta = rowsum(O * dO) - dLSE: one thread per 16-byte piece of a row, PIECES pieces per row
template <int PIECES>
__global__ __launch_bounds__(256) void delta_kernel(const BwdParams p) {
  const int r = threadIdx.x / PIECES, ch = threadIdx.x % PIECES;
  const int qi = blockIdx.x * (256 / PIECES) + r, h = blockIdx.y, b = blockIdx.z;
  const bool ok = qi < p.seqs.max_q_len;
  float d = 0.f;
  if (ok && ch * 4 < p.D) {
    const float4 o = *reinterpret_cast<const float4 *>((const float *)p.o.ptr + b * p.o.sb + h * p.o.sh + (int64_t)qi * p.o.st + ch * 4);
    const float4 g = *reinterpret_cast<const float4 *>((const float *)p.dout.ptr + b * p.dout.sb + h * p.dout.sh + (int64_t)qi * p.dout.st + ch * 4);
    d = o.x * g.x + o.y * g.y + o.z * g.z + o.w * g.w;
  }
#pragma unroll
  for (int off = PIECES / 2; off > 0; off >>= 1) d += __shfl_xor(d, off);
  if (ok && ch == 0) {
    if (p.dlse.ptr) d -= p.dlse.ptr[b * p.dlse.sb + h * p.dlse.sh + (int64_t)qi * p.dlse.st];
    p.delta[((int64_t)b * p.Hq + h) * p.seqs.max_q_len + qi] = d;
  }
}

// dQ: workgroup = 64 q rows of one head; wave = 32 rows x 32 keys of every listed block: S^T = K Q^T,
// dP^T = V dO^T (lane = q row: lse and delta are per-lane scalars), dS^T = P^T (dP^T - delta),
// dQ^T += K^T dS^T; the two key halves are added at the end.  CUT: launches that cut long rows into segments, as in the 16-bit
// pass (in one instantiation with them launches that cut nothing spilled forty scalars more).
template <int KD, bool PAD, bool CUT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(KD <= 64 ? 2 : 1, KD <= 64 ? 2 : 1))) void dq_kernel(
    const BwdParams p, int tiles_y) {
  using S = Shape<KD, PAD>;
  extern __shared__ __align__(16) char smem[];
  const SeqInfo sq = load_seq(p.seqs, blockIdx.z, p.causal);
  const int h = grid_head(p.csr), kvh = __builtin_amdgcn_readfirstlane(h / (p.Hq / p.Hkv));
  int tile = tiles_y - 1 - (int)blockIdx.y;
  int place = blockIdx.y, seg = 0, segments = 1;  // (long rows are cut into segments: with the table's own order only)
  if constexpr (CUT) find_segment(p.seg, blockIdx.y, place, seg);
  if (p.csr.order)
    tile = scalar_load(p.csr.order + lut_head(p.csr, h, p.Hq, p.Hkv) * p.csr.order_sh + place) - sq.past / 64;
  if (tile < 0 || tile >= seq_row_blocks(sq, 64)) return;
  const int rb = sq.past / 64 + tile;
  const int lh = lut_head(p.csr, h, p.Hq, p.Hkv);
  int e0 = 0, e1 = 0;
  auto table_row = [&]() __attribute__((always_inline)) {
    if (rb < p.csr.num_rows)
      scalar_load2(p.csr.ptr + lh * p.csr.ptr_sh + rb, p.csr.ptr + lh * p.csr.ptr_sh + rb + 1, e0, e1);
  };
  if constexpr (CUT) {
    table_row();
    if (place < p.seg.n[1]) {
      const int len = e1 - e0;
      segments = planned_segments(p.seg, place, len);
      if (seg >= segments) return;
      e1 = e0 + __builtin_amdgcn_readfirstlane(len * (seg + 1) / segments);
      e0 += __builtin_amdgcn_readfirstlane(len * seg / segments);
    }
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rh = wave & 1, kh = wave >> 1;
  const int m = lane & 31, g = lane >> 5;
  const int row0 = rb * 64 + rh * 32;
  const int pos = row0 + m, qi = pos - sq.past;
  const bool row_ok = qi >= 0 && qi < sq.q_len;
  if constexpr (PAD) {
    zero_tiles<NT>(smem, S::kSmem, tid);
    __syncthreads();
  }

  if constexpr (!CUT) table_row();
  const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
  const float *kbase = (const float *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh;
  const float *vbase = (const float *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh;
  typename S::Loader kload, vload;
  kload.init(tid, 2 * p.k.st, 2 * p.D);
  vload.init(tid, 2 * p.v.st, 2 * p.D);
  auto issue = [&](int col, int stage) {
    const int key0 = col * 64, valid = col < 0 ? 0 : sq.k_len - key0;
    kload.issue(reinterpret_cast<const char *>(kbase + (int64_t)key0 * p.k.st), 0, valid, smem + stage * S::kStage);
    vload.issue(reinterpret_cast<const char *>(vbase + (int64_t)key0 * p.v.st), 0, valid, smem + stage * S::kStage + S::kTile);
  };
  int col_cur = 0, col_pending = 0;
  if (e0 < e1) {
    col_cur = scalar_load(cols + e0);
    issue(col_cur, 0);
    col_pending = e0 + 1 < e1 ? cols[e0 + 1] : 0;
  }
  float qf[S::HD], dof[S::HD];
  load_frag<S::HD>((const float *)p.q.ptr + sq.b * p.q.sb + h * p.q.sh + (int64_t)qi * p.q.st, row_ok, g, p.D, qf);
  load_frag<S::HD>((const float *)p.dout.ptr + sq.b * p.dout.sb + h * p.dout.sh + (int64_t)qi * p.dout.st, row_ok, g, p.D, dof);
  float lse2 = INFINITY, delta = 0.f;  // a row outside the sequence: P = exp2(. - inf) = 0
  if (row_ok) {
    const float lse = p.lse.ptr[sq.b * p.lse.sb + h * p.lse.sh + (int64_t)qi * p.lse.st];
    lse2 = lse == -INFINITY ? INFINITY : lse * kLog2e;
    delta = p.delta[((int64_t)sq.b * p.Hq + h) * p.seqs.max_q_len + qi];
  }
  floatx16 acc[S::DT];
  clear(acc);
  const int lim = p.causal ? min(pos, sq.k_len - 1) : sq.k_len - 1;

  auto block_step = [&](int e, auto stage_tag) {
    constexpr int stage = decltype(stage_tag)::value;
    const int col = col_cur;
    wait_tile_loads();
    __syncthreads();
    col_cur = __builtin_amdgcn_readfirstlane(col_pending);
    if (e + 2 < e1) col_pending = cols[e + 2];
    if (e + 1 < e1) issue(col_cur, stage ^ 1);
    const int key0 = col * 64 + kh * 32;
    if (col < 0 || key0 >= sq.k_len || (p.causal && key0 > row0 + 31)) return;
    const char *ks = smem + stage * S::kStage, *vs = ks + S::kTile;
    const DimSum<KD> dots = dot_dims<KD, PAD>(ks, kh * 32, qf, lane), dp = dot_dims<KD, PAD>(vs, kh * 32, dof, lane);
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = key0 + (r >> 2) * 8 + g * 4 + (r & 3);
      const float pr = key > lim ? 0.f : fast_exp2(fmaf(dots[r], p.scale_log2, -lse2));
      s[r] = pr * (dp[r] - delta);  // dS^T without sm_scale (applied once at the end)
    }
    dot_rows<KD, PAD>(ks, kh * 32, s, lane, acc);
  };
  for (int e = e0; e < e1; e += 2) {
    block_step(e, Stage<0>{});
    if (e + 1 < e1) block_step(e + 1, Stage<1>{});
  }
  __syncthreads();
  float *buf = reinterpret_cast<float *>(smem) + rh * S::DT * 1024;
  give_half<S::DT>(acc, kh == 1, buf, lane);
  __syncthreads();
  float *row = (float *)p.dq.ptr + sq.b * p.dq.sb + h * p.dq.sh + (int64_t)qi * p.dq.st;
  if (CUT && segments > 1)
    row = p.seg.partial + ((((int64_t)sq.b * p.Hq + h) * p.seg.slots + seg * p.seg.n[1] + place) * 128 + rh * 32 + m) * p.D;
  const float scale = CUT && segments > 1 ? 1.f : p.sm_scale;
  take_half_and_store<S::DT>(acc, kh == 1, buf, lane, scale, scale, row, row_ok, p.D);
}

// dK / dV: workgroup = 64 keys of one kv head (the q heads of its group one after the other) or of
// one q head (head_split: p.dk / p.dv then describe per-q-head partial buffers); wave = 32 keys, with
// their K and V rows in registers, x 32 q rows of every listed block: S = Q K^T, dP = dO V^T (lane =
// key, registers = q rows), P = exp(S - lse), dS = P (dP - delta), dV^T += dO^T P, dK^T += Q^T dS; the
// two q-row halves are added at the end.  Every CSC entry is tested against the sequence length.
template <int KD, bool PAD>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(KD <= 64 ? 2 : 1, KD <= 64 ? 2 : 1))) void dkdv_kernel(
    const BwdParams p, int head_split) {
  using S = Shape<KD, PAD>;
  extern __shared__ __align__(16) char smem[];
  float *const vecs = reinterpret_cast<float *>(smem + S::kSmem);  // per stage: lse[64] (log2 domain), delta[64]
  const SeqInfo sq = load_seq(p.seqs, blockIdx.z, p.causal);
  const int ratio = __builtin_amdgcn_readfirstlane(p.Hq / p.Hkv);
  const int out_head = grid_head(p.csc);
  const int kvh = head_split ? __builtin_amdgcn_readfirstlane(out_head / ratio) : out_head;
  const int gq_base = head_split ? out_head - kvh * ratio : 0, heads = head_split ? 1 : ratio;
  // longest columns first when the table gives the order, long ones in segments (as in the 16-bit pass)
  int place, seg;
  find_segment(p.seg, blockIdx.y, place, seg);
  int cb = place;
  if (p.csc.order)
    cb = scalar_load(p.csc.order + lut_head(p.csc, kvh * ratio + gq_base, p.Hq, p.Hkv) * p.csc.order_sh + place);
  if (cb * 64 >= sq.k_len) return;
  // of a cut column: the entries of each q head, the part of all heads' entries that is this workgroup's, and the
  // place of its sums (-1: not cut)
  __shared__ int part[5];
  if (p.seg.entries) {
    int e0, len, lo, hi;
    const int segments = column_part<1>(p, lut_head(p.csc, kvh * ratio + gq_base, p.Hq, p.Hkv), cb, place, seg, heads, sq, e0, len, lo, hi);
    if (seg >= segments) return;
    part[0] = e0, part[1] = len, part[2] = lo, part[3] = hi, part[4] = segments > 1 ? seg * p.seg.n[1] + place : -1;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nh = wave & 1, qh = wave >> 1;  // key half, q-row half
  const int n = lane & 31, g = lane >> 5;
  const int key0 = cb * 64 + nh * 32, key = key0 + n;
  const bool key_ok = key < sq.k_len;
  if constexpr (PAD) {
    zero_tiles<NT>(smem, S::kSmem, tid);
    __syncthreads();
  }
  float kf[S::HD], vf[S::HD];
  load_frag<S::HD>((const float *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh + (int64_t)key * p.k.st, key_ok, g, p.D, kf);
  load_frag<S::HD>((const float *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh + (int64_t)key * p.v.st, key_ok, g, p.D, vf);
  floatx16 dk[S::DT], dv[S::DT];
  clear(dk);
  clear(dv);
  typename S::Loader qload, doload;
  qload.init(tid, 2 * p.q.st, 2 * p.D);
  doload.init(tid, 2 * p.dout.st, 2 * p.D);

  // (the end is worked out again on every turn: one scalar less to keep)
  for (int gq = gq_base; gq < (head_split ? gq_base + 1 : p.Hq / p.Hkv); ++gq) {
    const int h = kvh * ratio + gq;
    const int lh = lut_head(p.csc, h, p.Hq, p.Hkv);
    int e0 = 0, e1 = 0;
    if (cb < p.csc.num_rows)
      scalar_load2(p.csc.ptr + lh * p.csc.ptr_sh + cb, p.csc.ptr + lh * p.csc.ptr_sh + cb + 1, e0, e1);
    const int32_t *rows = p.csc.idx + lh * p.csc.idx_sh;
    if (p.seg.entries) {  // (every wave has written the same values)
      const int first = __builtin_amdgcn_readfirstlane(part[0]), len = __builtin_amdgcn_readfirstlane(part[1]);
      const int before = (gq - gq_base) * len;  // entries of the heads before this one
      e0 = first + max(__builtin_amdgcn_readfirstlane(part[2]) - before, 0);
      e1 = first + min(__builtin_amdgcn_readfirstlane(part[3]) - before, len);
    }
    const float *qbase = (const float *)p.q.ptr + sq.b * p.q.sb + h * p.q.sh;
    const float *dobase = (const float *)p.dout.ptr + sq.b * p.dout.sb + h * p.dout.sh;
    const float *lsebase = p.lse.ptr + sq.b * p.lse.sb + h * p.lse.sh;
    const float *deltabase = p.delta + ((int64_t)sq.b * p.Hq + h) * p.seqs.max_q_len;
    float vec = 0.f;  // this thread's lse (threads 0..63) or delta (64..127) of the block that was requested last
    auto issue = [&](int rbq, int stage) {
      const int qi0 = rbq * 64 - sq.past;  // query index of the block's first row
      const int lo = rbq < 0 ? 64 : -qi0, hi = sq.q_len - qi0;
      qload.issue(reinterpret_cast<const char *>(qbase + (int64_t)qi0 * p.q.st), lo, hi, smem + stage * S::kStage);
      doload.issue(reinterpret_cast<const char *>(dobase + (int64_t)qi0 * p.dout.st), lo, hi, smem + stage * S::kStage + S::kTile);
      const int r = tid & 63;
      const bool ok = r >= lo && r < hi;
      if (tid < 64)
        vec = ok ? lsebase[(int64_t)(qi0 + r) * p.lse.st] : -INFINITY;
      else if (tid < 128)
        vec = ok ? deltabase[qi0 + r] : 0.f;
    };
    int rb_cur = 0, rb_pending = 0;
    if (e0 < e1) {
      rb_cur = scalar_load(rows + e0);
      issue(rb_cur, 0);
      rb_pending = e0 + 1 < e1 ? rows[e0 + 1] : 0;
    }
    auto block_step = [&](int e, auto stage_tag) {
      constexpr int stage = decltype(stage_tag)::value;
      const int rbq = rb_cur;
      wait_tile_loads();
      // (+inf where there is no row or the row saw no key: P = 0)
      if (tid < 64)
        vecs[stage * 128 + tid] = vec == -INFINITY ? INFINITY : vec * kLog2e;
      else if (tid < 128)
        vecs[stage * 128 + tid] = vec;
      __syncthreads();
      rb_cur = __builtin_amdgcn_readfirstlane(rb_pending);
      if (e + 2 < e1) rb_pending = rows[e + 2];
      if (e + 1 < e1) issue(rb_cur, stage ^ 1);
      const int pos0 = rbq * 64 + qh * 32;  // first q position of this wave's half
      if (rbq < 0 || (p.causal && key0 > pos0 + 31)) return;  // nothing visible (wave-uniform)
      const char *qs = smem + stage * S::kStage, *dos = qs + S::kTile;
      const float *lse_s = vecs + stage * 128 + qh * 32, *delta_s = lse_s + 64;
      // rows = q (tile), columns = keys (registers)
      const DimSum<KD> dots = dot_dims<KD, PAD>(qs, qh * 32, kf, lane), dps = dot_dims<KD, PAD>(dos, qh * 32, vf, lane);
      floatx16 s, ds;
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const float4 l4 = *reinterpret_cast<const float4 *>(lse_s + r4 * 8 + g * 4);
        const float4 d4 = *reinterpret_cast<const float4 *>(delta_s + r4 * 8 + g * 4);
        const float lr[4] = {l4.x, l4.y, l4.z, l4.w}, dr[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = r4 * 4 + i;
          const bool vis = key_ok && (!p.causal || key <= pos0 + r4 * 8 + g * 4 + i);
          s[r] = vis ? fast_exp2(fmaf(dots[r], p.scale_log2, -lr[i])) : 0.f;
          ds[r] = s[r] * (dps[r] - dr[i]);  // dS without sm_scale (applied once at the end)
        }
      }
      dot_rows<KD, PAD>(dos, qh * 32, s, lane, dv);
      dot_rows<KD, PAD>(qs, qh * 32, ds, lane, dk);
    };
    for (int e = e0; e < e1; e += 2) {
      block_step(e, Stage<0>{});
      if (e + 1 < e1) block_step(e + 1, Stage<1>{});
    }
    __syncthreads();  // every wave is done with the tiles before the next head (or the sums below) reuses them
  }
  // dK and dV one after the other through the same exchange areas
  float *buf = reinterpret_cast<float *>(smem) + nh * S::DT * 1024;
  float *buf2 = buf + 2 * S::DT * 1024;
  give_half<S::DT>(dk, qh == 1, buf, lane);
  give_half<S::DT>(dv, qh == 1, buf2, lane);
  __syncthreads();
  float *dkp = (float *)p.dk.ptr + sq.b * p.dk.sb + out_head * p.dk.sh + (int64_t)key * p.dk.st;
  float *dvp = (float *)p.dv.ptr + sq.b * p.dv.sb + out_head * p.dv.sh + (int64_t)key * p.dv.st;
  const int slot = p.seg.entries ? __builtin_amdgcn_readfirstlane(part[4]) : -1;
  if (slot >= 0) {
    dkp = p.seg.partial + ((((int64_t)sq.b * gridDim.x + out_head) * p.seg.slots + slot) * 128 + nh * 32 + n) * p.D;
    dvp = dkp + 64 * p.D;
  }
  take_half_and_store<S::DT>(dk, qh == 1, buf, lane, p.sm_scale, p.sm_scale, dkp, key_ok, p.D);
  take_half_and_store<S::DT>(dv, qh == 1, buf2, lane, 1.f, 1.f, dvp, key_ok, p.D);
}

static bool lut_ok(const LutView &l) {
  return l.block_rows == 64 && l.block_cols == 64 && l.entry_width == 1 && l.sub_block == 0;
}
static bool dims_ok(int d, bool wide) { return d % 4 == 0 && (wide ? d > 64 && d <= 128 : d >= 4 && d <= 64); }
// the tile copies keep a tile's byte offsets in 32 bits
static bool rows_ok(const TensorView &t) { return t.st >= 0 && t.st < (int64_t(1) << 23); }

template <int KD, bool PAD>
static int launch_fwd(const FwdParams &p, int tiles, hipStream_t stream) {
  constexpr int smem = Shape<KD, PAD>::kSmem;
  DK_ALLOW_DYNAMIC_LDS((fwd_kernel<KD, PAD>), smem);
  hipLaunchKernelGGL((fwd_kernel<KD, PAD>), dim3(p.Hq, tiles, p.seqs.packed ? 1 : p.seqs.batch), dim3(NT), smem, stream, p, tiles);
  DK_HIP_CHECK(hipGetLastError());
  return DK_OK;
}

template <int KD, bool PAD>
static int launch_dq(const BwdParams &p, int rows, hipStream_t stream) {
  constexpr int smem = Shape<KD, PAD>::kSmem;
  if (p.seg.entries) {
    DK_ALLOW_DYNAMIC_LDS((dq_kernel<KD, PAD, true>), smem);
    hipLaunchKernelGGL((dq_kernel<KD, PAD, true>), dim3(p.Hq, rows, p.seqs.batch), dim3(NT), smem, stream, p, rows);
  } else {
    DK_ALLOW_DYNAMIC_LDS((dq_kernel<KD, PAD, false>), smem);
    hipLaunchKernelGGL((dq_kernel<KD, PAD, false>), dim3(p.Hq, rows, p.seqs.batch), dim3(NT), smem, stream, p, rows);
  }
  DK_HIP_CHECK(hipGetLastError());
  return DK_OK;
}

template <int KD, bool PAD>
static int launch_dkdv(const BwdParams &p, int columns, int heads, hipStream_t stream) {
  constexpr int smem = Shape<KD, PAD>::kSmem + 2 * 128 * (int)sizeof(float);
  DK_ALLOW_DYNAMIC_LDS((dkdv_kernel<KD, PAD>), smem);
  hipLaunchKernelGGL((dkdv_kernel<KD, PAD>), dim3(heads, columns, p.seqs.batch), dim3(NT), smem, stream, p, heads != p.Hkv);
  DK_HIP_CHECK(hipGetLastError());
  return DK_OK;
}

// head dims multiplied: the multiple of 32 from 64 on that holds the tensors' own
#define DK_BY_HEAD_DIM(launch, D, ...)                                                                  \
  ((D) == 64 ? launch<64, false>(__VA_ARGS__) : (D) < 64 ? launch<64, true>(__VA_ARGS__)                \
   : (D) <= 96 ? launch<96, true>(__VA_ARGS__) : (D) < 128 ? launch<128, true>(__VA_ARGS__) : launch<128, false>(__VA_ARGS__))

}  // namespace f32

bool mfma_f32_fwd_supported(const FwdParams &p, int dtype, bool wide) {
  return dtype == DK_F32 && f32::dims_ok(p.D, wide) && p.vec_ok && f32::lut_ok(p.csr) && f32::rows_ok(p.k) && f32::rows_ok(p.v);
}

bool mfma_f32_bwd_supported(const BwdParams &p, int dtype, bool wide) {
  return dtype == DK_F32 && f32::dims_ok(p.D, wide) && p.vec_ok && f32::lut_ok(p.csr) && f32::lut_ok(p.csc) &&
         f32::rows_ok(p.q) && f32::rows_ok(p.k) && f32::rows_ok(p.v) && f32::rows_ok(p.dout);
}

int launch_mfma_f32_fwd(const FwdParams &p, hipStream_t stream) {
  const SeqView &s = p.seqs;
  int tiles;
  if (s.packed)
    tiles = cdiv(s.max_q_len, 64) + 2 * s.batch;  // as for the 16-bit forward: an upper bound over all sequences
  else if (s.given)
    tiles = cdiv(s.max_q_len, 64) + 1;
  else {
    const int past = p.causal ? s.max_k_len - s.max_q_len : 0;
    tiles = (past + s.max_q_len - 1) / 64 - past / 64 + 1;
  }
  if (p.csr.order && !s.packed) tiles = p.csr.num_rows;  // handed out in the table's order: all of them
  DK_REQUIRE(tiles <= 65535, "too many q tiles for one launch (%d)", tiles);
  FwdParams pr = p;
  pr.csr.rot = head_rotation(p.csr, p.Hq, tiles);  // (uneven heads: dealt to the queues in rotation)
  DK_NOTE_KERNEL(pr.csr.rot ? "f32::fwd_kernel, heads in rotation" : "f32::fwd_kernel");
  using namespace f32;
  return DK_BY_HEAD_DIM(launch_fwd, p.D, pr, tiles, stream);
}

// Scratch of the backward.  Head dims up to 64: a workgroup of the dK/dV pass walks whole groups of q heads, long columns
// cut into segments (16 / 4 heads of 64, 2000 tokens, training: 904 us uncut, 407 cut; 4000 tokens 1833 / 821; 3 x 1000,
// 24 / 8 753 / 565).  Above, one workgroup per q head into partials that are summed is the faster one at every size (a
// step takes four times the 16-bit kernel's time, the partials as long as there: 4 x 2000, 32 / 8 heads of 128, 5064 us against
// 5684; 2 x 2000, 24 / 8 of 96, 1599 / 1662), unless the partials would not fit.
static BwdScratch mfma_f32_bwd_scratch(const BwdParams &p, bool walk) {
  const int slots = 256 * (p.D <= 64 ? 2 : 1);
  return plan_bwd_scratch(p, p.D > 64 && p.D % 8 == 0 ? bwd_group_bytes(p) : 0, slots, false, slots, walk ? INFINITY : -1, -1);
}
size_t mfma_f32_bwd_workspace_bytes(const BwdParams &p) { return mfma_f32_bwd_scratch(p, true).bytes; }

int launch_mfma_f32_bwd(const BwdParams &p, void *workspace, size_t workspace_bytes, hipStream_t stream) {
  const SeqView &s = p.seqs;
  const int past = p.causal ? s.max_k_len - s.max_q_len : 0;
  const int tiles = (past + s.max_q_len - 1) / 64 - past / 64 + 1;
  const int cblocks = cdiv(s.max_k_len, 64);
  DK_REQUIRE(tiles <= 65535 && cblocks <= 65535, "sequence too long for one launch");
  DK_NOTE_KERNEL("f32::delta_kernel");
  if (p.D <= 64)
    hipLaunchKernelGGL(f32::delta_kernel<16>, dim3(cdiv(s.max_q_len, 16), p.Hq, s.batch), dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(f32::delta_kernel<32>, dim3(cdiv(s.max_q_len, 8), p.Hq, s.batch), dim3(256), 0, stream, p);
  DK_HIP_CHECK(hipGetLastError());
  DK_REQUIRE(!p.csr.order || p.csr.num_rows <= 65535, "sequence too long for one launch");
  const BwdScratch scratch = usable_bwd_scratch([&](bool walk) { return mfma_f32_bwd_scratch(p, walk); }, workspace, workspace_bytes);
  BwdParams pq = p;
  if (p.csr.order && segment_items(scratch.dq, p.csr.num_rows) <= 65535) pq.seg = scratch.dq;
  // handed out in the table's order: all of them
  const int rows = p.csr.order ? (int)segment_items(pq.seg, p.csr.num_rows) : tiles;
  pq.csr.rot = head_rotation(p.csr, p.Hq, rows);
  DK_NOTE_KERNEL(pq.csr.rot ? "f32::dq_kernel, heads in rotation" : "f32::dq_kernel");
  using namespace f32;
  if (int rc = DK_BY_HEAD_DIM(launch_dq, p.D, pq, rows, stream)) return rc;
  if (pq.seg.entries)
    if (int rc = launch_segment_sum(p.csr, pq.seg, SegRows::kQueries, p.dq, p.dq, DK_F32, p.Hq, p, p.sm_scale, s.max_q_len, past, stream)) return rc;
  // Several q heads per kv head: one workgroup per q head into fp32 partials of its own and a sum over
  // each group, as in the 16-bit pass (one workgroup walking the whole group makes the longest column
  // outlast the rest of the launch).
  const bool per_q_head = scratch.group > 0;
  const int heads = per_q_head ? p.Hq : p.Hkv;
  BwdParams po = p;  // the order only where heads do not line up with the hardware's 32 workgroup queues
  po.trim = p.csc.row_lengths && p.csr.num_rows > tiles + past / 64;  // (as in the 16-bit pass)
  if (p.csc.order && segment_items(scratch.kv, p.csc.num_rows) <= 65535) po.seg = scratch.kv;
  if (heads % 32 == 0 && !po.seg.entries) po.csc.order = nullptr;
  DK_REQUIRE(p.csc.num_rows <= 65535, "sequence too long for one launch");
  const int columns = po.csc.order ? (int)segment_items(po.seg, p.csc.num_rows) : cblocks;
  po.csc.rot = head_rotation(p.csc, heads, columns);
  float *part_k = (float *)workspace, *part_v = part_k + (int64_t)s.batch * p.Hq * s.max_k_len * p.D;
  if (per_q_head) {
    po.dk = TensorView{part_k, (int64_t)p.Hq * s.max_k_len * p.D, (int64_t)s.max_k_len * p.D, p.D};
    po.dv = TensorView{part_v, (int64_t)p.Hq * s.max_k_len * p.D, (int64_t)s.max_k_len * p.D, p.D};
  }
  DK_NOTE_KERNEL(po.csc.rot ? "f32::dkdv_kernel, heads in rotation" : "f32::dkdv_kernel");
  if (int rc = DK_BY_HEAD_DIM(launch_dkdv, p.D, po, columns, heads, stream)) return rc;
  if (po.seg.entries)
    if (int rc = launch_segment_sum(p.csc, po.seg, SegRows::kKeys, po.dk, po.dv, DK_F32, heads, po, 1.f, s.max_k_len, past, stream)) return rc;
  return per_q_head ? launch_dkdv_group_sum(p, DK_F32, part_k, part_v, stream) : DK_OK;
}

}  // namespace dk
