// Forward kernel for launches too small to fill the chip (short prompts, few heads): the block loop of
// a row is split over the waves of a workgroup instead of running through the whole row in each of them.
//
//   workgroup = 32 q rows of one head, 4 waves; wave = every fourth half block (32 keys) of the row,
//               with its own running maximum, sum and O.  The waves share nothing until the end, so
//               there is no barrier in the loop: each keeps private LDS tiles (K and V of a half block,
//               rows padded by 16 bytes) and fetches the next half block into registers while it
//               multiplies, as the decode kernel does.  The four results are merged through LDS, eight
//               threads per row, and leave as whole rows.
//
// Bound: latency (three dependent reads, one round trip to the first keys, the merge).  K/V tiles are
// fetched once per 32 rows and head, which only a small launch can afford.  The rule that chooses it is
// in mfma_fwd.hip (split_pays).
#pragma once

#include "device_common.h"
#include "mfma_common.h"

namespace dk {

constexpr int kSplitWaves = 4;

template <int D>
struct SplitSmem {  // per wave
  static constexpr int kStride = D * 2 + 16;  // bytes per tile row
  static constexpr int kHalf = 32 * kStride;  // one 32-key tile
  static constexpr int kWave = 2 * kHalf;     // K and V; in the end 32 rows of (O[D], max, sum, pad) floats
  static constexpr int kRow = D + 4;          // floats per row of a result
  static_assert(32 * kRow * 4 <= kWave, "a wave's result fits its tiles");
  static constexpr int kBytes = kSplitWaves * kWave;
};

template <typename T, int D, bool PAD, bool SUB, int KD = D>
__global__ __launch_bounds__(64 * kSplitWaves) __attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : 2, D == 64 ? 3 : D == 256 ? 1 : 2))) void mfma_fwd_split_kernel(
    const FwdParams p, int tiles_y) {
  using M = Mma<T>;
  using vec8 = typename M::vec8;
  using S = SplitSmem<D>;
  constexpr int W = kSplitWaves, NT = 64 * W;
  constexpr int KS = KD / 16, DT = KD / 32, CPR = D / 8;
  constexpr int EW = SUB ? 2 : 1;  // ints per table entry
  extern __shared__ __align__(16) char smem_all[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = grid_head(p.csr);
  if (p.seqs.packed && p.seqs.zero_outside && blockIdx.y == 0) lse_outside_packed(p.seqs, p.lse, h, 1, tid, NT);
  SeqInfo sq;
  int tile;
  if (!resolve_tile(p.seqs, p.causal, 32, 1, tiles_y - 1 - (int)blockIdx.y, blockIdx.z, sq, tile)) {
    if (p.seqs.zero_outside && !p.seqs.packed)
      zero_rows_outside<T>(p.seqs, sq, blockIdx.y, tiles_y, p.o, p.lse, h, 1, p.D, p.vec_ok, tid, NT);
    return;
  }
  const int row0 = (sq.past / 32 + tile) * 32;  // first absolute position
  const int rb = row0 / 64;
  const int kvh = __builtin_amdgcn_readfirstlane(h / (p.Hq / p.Hkv));
  const int m = lane & 31, g = lane >> 5;
  const int pos = row0 + m, qi = pos - sq.past;
  const bool row_ok = qi >= 0 && qi < sq.q_len;
  const int lh = lut_head(p.csr, h, p.Hq, p.Hkv);
  int e0 = 0, e1 = 0;
  if (rb < p.csr.num_rows)
    scalar_load2(p.csr.ptr + lh * p.csr.ptr_sh + rb, p.csr.ptr + lh * p.csr.ptr_sh + rb + 1, e0, e1);
  const int32_t *cols = p.csr.idx + lh * p.csr.idx_sh;
  const T *kbase = (const T *)p.k.ptr + sq.b * p.k.sb + kvh * p.k.sh + (int64_t)sq.k_start * p.k.st;
  const T *vbase = (const T *)p.v.ptr + sq.b * p.v.sb + kvh * p.v.sh + (int64_t)sq.k_start * p.v.st;
  char *const smem = smem_all + wave * S::kWave, *const ks_ = smem, *const vs_ = smem + S::kHalf;

  constexpr int HCH = 32 * CPR / 64;  // 16-byte chunks per lane per half tile
  uint4 kreg[HCH], vreg[HCH];
  auto prefetch = [&](int hb, int col) {  // half block hb of the row: keys col * 64 + 32 * (hb & 1) + [0, 32)
    const int key0 = col * 64 + (hb & 1) * 32;
    const bool whole = !PAD && col >= 0 && key0 + 32 <= sq.k_len;
#pragma unroll
    for (int c = 0; c < HCH; ++c) {
      const int r = (lane + c * 64) / CPR, ch = (lane + c * 64) % CPR;
      kreg[c] = vreg[c] = make_uint4(0, 0, 0, 0);  // rows beyond the sequence, head dims beyond p.D
      if (whole || (col >= 0 && key0 + r < sq.k_len && (!PAD || ch * 8 < p.D))) {
        kreg[c] = *reinterpret_cast<const uint4 *>(kbase + (int64_t)(key0 + r) * p.k.st + ch * 8);
        vreg[c] = *reinterpret_cast<const uint4 *>(vbase + (int64_t)(key0 + r) * p.v.st + ch * 8);
      }
    }
  };
  const int nhalf = 2 * (e1 - e0);
  int col_cur = 0, bits_cur = 0;
  auto entry = [&](int hb) {
    const int32_t *ent = cols + (e0 + (hb >> 1)) * EW;
    if constexpr (SUB)
      scalar_load2(ent, ent + 1, col_cur, bits_cur);
    else
      col_cur = scalar_load(ent);
  };
  if (wave < nhalf) {
    entry(wave);
    prefetch(wave, col_cur);
  }
  vec8 qf[KS];
  {
    const T *qp = (const T *)p.q.ptr + sq.b * p.q.sb + h * p.q.sh + (int64_t)(sq.q_start + qi) * p.q.st;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 w = make_uint4(0, 0, 0, 0);
      if (row_ok && (!PAD || ks * 16 + g * 8 < p.D)) w = *reinterpret_cast<const uint4 *>(qp + ks * 16 + g * 8);
      qf[ks] = as_vec8<vec8>(w);
    }
  }
  floatx16 oacc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;
  const int lim = p.causal ? min(pos, sq.k_len - 1) : sq.k_len - 1;  // last visible key of this row
  const int k_read = m * S::kStride + g * 16;
  const int i16 = lane & 15, dgrp = (lane >> 4) & 1;
  const int v_read = (4 * g + (i16 >> 2)) * S::kStride + (16 * dgrp + 4 * (i16 & 3)) * 2;

  for (int hb = wave; hb < nhalf; hb += W) {
    const int col = col_cur, bits = bits_cur;
    const int key0 = col * 64 + (hb & 1) * 32;
    // (the tiles are this wave's own and its LDS operations execute in order; only the compiler must
    // not reorder across these points)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int c = 0; c < HCH; ++c) {
      const int r = (lane + c * 64) / CPR, ch = (lane + c * 64) % CPR;
      *reinterpret_cast<uint4 *>(ks_ + r * S::kStride + ch * 16) = kreg[c];
      *reinterpret_cast<uint4 *>(vs_ + r * S::kStride + ch * 16) = vreg[c];
    }
    asm volatile("" ::: "memory");
    if (hb + W < nhalf) {
      entry(hb + W);
      prefetch(hb + W, col_cur);
    }
    if (col < 0 || key0 >= sq.k_len || (p.causal && key0 > row0 + 31)) continue;  // nothing visible (wave-uniform)
    // S^T = K Q^T: lane = q row, registers = keys 8 (r / 4) + 4 g + r % 4 of the half block
    floatx16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
    {
      vec8 a[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) a[ks] = lds_read8<vec8>(ks_ + k_read + ks * 32);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = M::mma(a[ks], qf[ks], s);
    }
    if constexpr (SUB) {
      // pattern blocks of the tile that this row does not attend: bit (row part) * f + (key part)
      const int lb = p.csr.sub_block == 16 ? 4 : 5, f = 64 >> lb;
      const int row_bits = bits >> (((pos & 63) >> lb) * f);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key_part = ((hb & 1) * 32 + (r >> 2) * 8) >> lb;  // the last terms stay inside a part of >= 16 keys
        s[r] = ((row_bits >> key_part) & 1) ? s[r] : -INFINITY;
      }
    }
    if (key0 + 31 >= sq.k_len || (p.causal && key0 + 31 > row0)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = key0 + (r >> 2) * 8 + g * 4 + (r & 3) > lim ? -INFINITY : s[r];
    }
    float mx = max_of(s);
    mx = max_with_other_half(mx) * p.scale_log2;  // scale > 0: max commutes with it
    const float m_new = fmaxf(m_run, mx);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    if (__builtin_amdgcn_ballot_w64(m_new > m_run) != 0) {  // wave-uniform: some row's maximum has moved
      const float alpha = fast_exp2(m_run - m_use);
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
      m_run = m_new;
    }
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], p.scale_log2, -m_use));
      psum += s[r];
    }
    l_run += psum;  // this lane's share of the row sum
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float pf[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) pf[i] = s[t * 8 + i];
      const vec8 pb = M::pack(pf);
      const char *vrow = vs_ + v_read + t * 16 * S::kStride;
      vec8 a[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) a[dt] = lds_read_tr8<vec8>(vrow + dt * 64, vrow + 8 * S::kStride + dt * 64);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) oacc[dt] = M::mma(a[dt], pb, oacc[dt]);
    }
  }
  l_run += xor32(l_run);

  // ---- merge: each wave leaves its 32 rows (O unnormalised, max, sum) in its own tiles ----
  {
    float *row = reinterpret_cast<float *>(smem) + m * S::kRow;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4)
        *reinterpret_cast<float4 *>(row + dt * 32 + r4 * 8 + g * 4) =
            make_float4(oacc[dt][r4 * 4], oacc[dt][r4 * 4 + 1], oacc[dt][r4 * 4 + 2], oacc[dt][r4 * 4 + 3]);
    if (g == 0) *reinterpret_cast<float2 *>(row + D) = make_float2(m_run, l_run);
  }
  __syncthreads();
  const int r = tid / 8, part = tid % 8;  // eight threads per row: chunks part, part + 8, ... of eight dims
  const int qr = row0 + r - sq.past;
  float mv[W], lv[W];
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const float2 ml = *reinterpret_cast<const float2 *>(reinterpret_cast<const float *>(smem_all + u * S::kWave) + r * S::kRow + D);
    mv[u] = ml.x, lv[u] = ml.y;
  }
  float mmax = mv[0], l = 0.f;
#pragma unroll
  for (int u = 1; u < W; ++u) mmax = fmaxf(mmax, mv[u]);
  const float muse = mmax == -INFINITY ? 0.f : mmax;
#pragma unroll
  for (int u = 0; u < W; ++u) {
    mv[u] = fast_exp2(mv[u] - muse);  // a wave that saw no key: weight 0
    l += mv[u] * lv[u];
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (qr >= 0 && qr < sq.q_len) {
    T *op = (T *)p.o.ptr + sq.b * p.o.sb + h * p.o.sh + (int64_t)(sq.q_start + qr) * p.o.st;
#pragma unroll
    for (int c = 0; c < CPR / 8; ++c) {
      const int ch = part + c * 8;
      float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < W; ++u) {
        const float *src = reinterpret_cast<const float *>(smem_all + u * S::kWave) + r * S::kRow + ch * 8;
        const float4 a = *reinterpret_cast<const float4 *>(src), b = *reinterpret_cast<const float4 *>(src + 4);
        o[0] += mv[u] * a.x, o[1] += mv[u] * a.y, o[2] += mv[u] * a.z, o[3] += mv[u] * a.w;
        o[4] += mv[u] * b.x, o[5] += mv[u] * b.y, o[6] += mv[u] * b.z, o[7] += mv[u] * b.w;
      }
      const uint2 lo = pack4<T>(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv), hi = pack4<T>(o[4] * inv, o[5] * inv, o[6] * inv, o[7] * inv);
      if (!PAD || ch * 8 < p.D) *reinterpret_cast<uint4 *>(op + ch * 8) = make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
    if (p.lse.ptr && part == 0)
      p.lse.ptr[sq.b * p.lse.sb + h * p.lse.sh + (int64_t)(sq.q_start + qr) * p.lse.st] =
          l > 0.f ? (mmax + log2f(l)) * kLn2 : -INFINITY;
  }
  if (p.seqs.zero_outside && !p.seqs.packed)
    zero_rows_outside<T>(p.seqs, sq, blockIdx.y, tiles_y, p.o, p.lse, h, 1, p.D, p.vec_ok, tid, NT);
}

}  // namespace dk
