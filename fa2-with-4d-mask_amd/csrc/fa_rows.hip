// Forward of a few query rows against many keys on gfx950 (MI355X): decoding
// (one new token per sequence) and short chunks, where the 256-row blocks of
// fa_fwd.hip would leave most of their rows empty and most CUs without a
// workgroup.  Restates the maths of the reference's TileLang forward
// (python/fa2.py:22-139), as fa_fwd.hip does.
//
//   fwd_rows_kernel     the rows of every head of a kv-head's group (row
//                       r = tq G + g) in blocks of 32, the key axis cut into
//                       a.ns ranges: one workgroup of 4 waves per (32 packed
//                       rows, key range, kv-head, batch).  Each wave walks every
//                       fourth 32-key tile of the range with its own running
//                       maximum, sum and O^T, merged through LDS at the end.
//   fwd_combine_kernel  joins the key ranges' partial results (also those of
//                       the key-split launches of fa_fwd.hip).
//
// What bounds it: reading K and V once.  A wave holds one whole tile of K and
// of V in flight (16 KB at head dim 128) while it works on the one before, two
// workgroups per CU (head dim 256: one), so about 128 KB per CU are on the way at any
// time.  K rows
// go straight from memory into MFMA operand registers (S^T = K Q^T reads a K
// row per lane); only V takes the way through LDS, in a region of each wave's
// own (no barrier in the loop), for the transpose reads of O^T += V^T P^T.
//
// A mask is read as the caller gives it, one byte per (row, key) -- these
// launches read each byte once, so there is nothing to gain from the prepared
// bit form and its three launches -- and tiles of which no row keeps a key are
// skipped before their K and V are loaded.  (Not so tiles whose scores are all
// -inf: their keys are kept, and a NaN or Inf in K or V reaches O as it does in
// fa_fwd.hip.)
//
// Measured (bf16, Hq 32, Hk 8, D 128): one row against 16384 keys 15 us + 5 for
// the combine (67 MB of K and V; 330 us in fwd_kernel, 32 workgroups); a batch of
// 16, 3001 keys, left padding up to half: 31 + 4 us (253 + 16 for the prepared
// mask before), the live 155 MB at 5.0 TB/s.
#include "fa_common.h"
#include "fa_kernels.h"

namespace fa {
namespace {

constexpr int kRKeys = 32;    // keys per tile
constexpr int kRWaves = 4;
constexpr int kRScan = 32;    // tiles of a wave whose liveness is looked at together

// chunk swizzle of the V tile's rows: the transpose reads (4 rows x 4 chunks)
// hit distinct banks
template <int D> __device__ __forceinline__ int swz_rv(int r) {
  return D == 64 ? (((r >> 1) & 1) << 2) : ((r & 3) << 2);
}

// The products as fp32 values: otherwise the 16-bit rounding of O may be taken
// from the unrounded product (v_fma_mix) and its residual from the rounded one,
// an ulp apart at a tie.
__device__ __forceinline__ void hold(f32x4& x, f32x4& y) { asm volatile("" : "+v"(x), "+v"(y)); }

template <typename T, int D, bool MASK, bool SCORE>
__global__ __launch_bounds__(kRWaves * 64, D == 256 ? 1 : 2) void fwd_rows_kernel(const FwdArgs a) {
  using V8 = typename Vec8<T>::type;
  constexpr int DS = D / 16, NB = D / 32, CH = D / 8, ROWB = 2 * D;
  constexpr int VT = kRKeys * ROWB;          // bytes of one V tile
  constexpr int U = kRKeys * CH / 64;        // 16-byte V chunks per lane
  constexpr int OS = D + 4;                  // merge stride (floats)
  // with a mask or a score P enters O in two 16-bit parts, as in fa_fwd.hip
  constexpr bool PREC = MASK || SCORE;
  constexpr int KEEPB = MASK ? kRScan * 256 : 0;   // keep words of a wave's scanned tiles
  constexpr int WORK = kRWaves * (VT + KEEPB), MERGE = kRWaves * 32 * OS * 4;
  __shared__ __attribute__((aligned(1024))) char smem[WORK > MERGE ? WORK : MERGE];
  __shared__ float sml[kRWaves][2][32];      // running maximum and sum per wave and row

  // ---- which (batch, kv-head, key range, row block) ---------------------------
  // Row blocks of a range next to each other, then the ranges of a kv-head:
  // with the XCD remap an XCD's L2 serves the row blocks that share K and V.
  const int R = a.Tq * a.G;
  const int nrb = (R + 31) / 32;
  const int W = xcd_remap(blockIdx.x, a.B * a.Hk * a.ns * nrb);
  const int rb = W % nrb, W1 = W / nrb;
  const int sp = W1 % a.ns, bk = W1 / a.ns;
  const int b = bk / a.Hk, kvh = bk - b * a.Hk;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hf = lane >> 5;
  const int Tk = a.Tk;
  const int r = min(rb * 32 + l32, R - 1);   // this lane's packed row (rows past R repeat the last)
  const int tq = r / a.G, h = kvh * a.G + (r - tq * a.G);
  const float c2 = a.scale_log2;

  // Q fragment (B of S^T): lane holds Q[row][16 ds + 8 hf .. +7]
  V8 qf[DS];
  {
    const uint32_t neg = a.qsign < 0.f ? 0x80008000u : 0u;
    const T* src = (const T*)a.q + b * a.qsb + h * a.qsh + (int64_t)tq * a.qst + hf * 8;
    u32x4 x[DS];
    load_row(x, src, a.Dv);
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) qf[ds] = as_vec8<T>(only_cols(x[ds], ds, a.Dv, neg));
  }
  // (head dim 256: in AGPRs, which MFMA reads as well, to keep them out of the
  // 256 VGPRs of the loop)
  if constexpr (D == 256) {
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) asm volatile("" : "+a"(qf[ds]));
  }
  const T* __restrict__ kp = (const T*)a.k + b * a.ksb + kvh * a.ksh;
  const T* __restrict__ vp = (const T*)a.v + b * a.vsb + kvh * a.vsh;
  const uint8_t* mrow = MASK ? a.mask + b * a.msb + h * a.msh + (int64_t)tq * a.msq : nullptr;
  const float* srow = SCORE ? a.score + b * a.ssb + h * a.ssh + (int64_t)tq * a.ssq : nullptr;
  const int lim = a.causal ? min(Tk, tq + 1) : Tk;   // keys [0, lim) of this lane's row

  // ---- key tiles of the workgroup and of this wave ------------------------------
  const int nt = ((a.causal ? min(Tk, a.Tq) : Tk) + kRKeys - 1) / kRKeys;
  const int t_lo = (int)((int64_t)nt * sp / a.ns), t_hi = (int)((int64_t)nt * (sp + 1) / a.ns);
  const int t_w = t_lo + wave;
  const int n_w = t_w < t_hi ? (t_hi - t_w + kRWaves - 1) / kRWaves : 0;   // tiles t_w + 4 i

  // ---- loads ---------------------------------------------------------------------
  u32x4 kf[DS], vr[U];
  uint32_t goff_v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int idx = lane + u * 64;
    goff_v[u] = 8 * (idx % CH) < a.Dv ? (uint32_t)((idx / CH) * a.vst * 2) + (uint32_t)((idx % CH) * 16) : kNoRec;
  }
  const uint32_t goff_k = (uint32_t)(l32 * a.kst * 2) + (uint32_t)(hf * 16);
  // rows of tile t through a buffer from its first key; keys past Tk (and a
  // tile that is not there) read zeros
  auto tile_rs = [&](const T* base, int64_t st, int t, bool valid) __attribute__((always_inline)) {
    const int rows = min(Tk - t * kRKeys, kRKeys);
    const bool ok = valid && rows > 0;
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (ok ? (int64_t)t * kRKeys * st : 0)), (short)0,
                                             ok ? (int)((int64_t)(rows - 1) * st * 2 + 2 * a.Dv) : 0, 0x00020000);
  };
  auto load_k = [&](int t, bool valid) __attribute__((always_inline)) {
    const auto rs = tile_rs(kp, a.kst, t, valid);
#pragma unroll
    for (int ds = 0; ds < DS; ++ds) kf[ds] = __builtin_amdgcn_raw_buffer_load_b128(rs, goff_k + 32 * ds, 16 * ds < a.Dv ? 0 : kNoRec, 0);
  };
  auto load_v = [&](int t, bool valid) __attribute__((always_inline)) {
    const auto rs = tile_rs(vp, a.vst, t, valid);
#pragma unroll
    for (int u = 0; u < U; ++u) vr[u] = __builtin_amdgcn_raw_buffer_load_b128(rs, goff_v[u], 0, 0);
  };
  // scores of tile t at this lane's row (entry 4 gi + e: key 32 t + 8 gi +
  // 4 hf + e); keys past Tk read key Tk - 1 (dropped below)
  auto load_score = [&](int t, f32x16& x) __attribute__((always_inline)) {
    if ((t + 1) * kRKeys <= Tk) {
#pragma unroll
      for (int gi = 0; gi < 4; ++gi) {
        struct __attribute__((packed, aligned(4))) F4 { float v[4]; };
        const F4 y = *(const F4*)(srow + t * kRKeys + gi * 8 + hf * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[gi * 4 + e] = y.v[e];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = srow[min(t * kRKeys + 8 * (i >> 2) + 4 * hf + (i & 3), Tk - 1)];
    }
  };
  // keep bits of tile t at this lane's row (bit 8 gi + e <-> entry 4 gi + e)
  auto load_keep = [&](int t) __attribute__((always_inline)) -> uint32_t {
    uint32_t w = 0;
    const int k0 = t * kRKeys + 4 * hf;
    if (a.mask4 && (t + 1) * kRKeys <= Tk) {   // rows 4-byte aligned: four keys per load
      uint32_t x[4];
#pragma unroll
      for (int gi = 0; gi < 4; ++gi) x[gi] = *(const uint32_t*)(mrow + k0 + 8 * gi);
#pragma unroll
      for (int gi = 0; gi < 4; ++gi)
#pragma unroll
        for (int e = 0; e < 4; ++e) w |= ((x[gi] >> (8 * e)) & 0xffu) != 0 ? 1u << (8 * gi + e) : 0u;
    } else {
      uint8_t x[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = mrow[min(k0 + 8 * (i >> 2) + (i & 3), Tk - 1)];
#pragma unroll
      for (int i = 0; i < 16; ++i) w |= x[i] != 0 ? 1u << (8 * (i >> 2) + (i & 3)) : 0u;
    }
    return w;
  };
  // the first lim keys of the row, as keep bits of the tile at k0
  auto in_row = [&](int k0) __attribute__((always_inline)) -> uint32_t {
    const int n = lim - (k0 + 4 * hf);
    return n >= 32 ? ~0u : (n <= 0 ? 0u : (1u << n) - 1u);
  };

  f32x16 oacc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) oacc[nb] = f32x16{};
  float m_run = kNegInf, l_run = 0.f;
  float m_lift = kNegInf;   // what a tile's maximum has to exceed to move m_run (with a score)
  const int tr_row = 4 * hf + ((lane >> 2) & 3);
  const int tr_col = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  char* vt = smem + wave * VT;
  uint32_t* keep = (uint32_t*)(smem + kRWaves * VT + wave * KEEPB);

  for (int ic = 0; ic < n_w; ic += kRScan) {
    // ---- live tiles among the next kRScan of this wave --------------------------
    const int cnt = min(kRScan, n_w - ic);
    uint32_t live = cnt == 32 ? ~0u : (1u << cnt) - 1u;
    if constexpr (MASK) {
      live = 0;
#pragma unroll 2
      for (int i = 0; i < cnt; ++i) {
        const int t = t_w + kRWaves * (ic + i);
        const uint32_t w = in_row(t * kRKeys) & load_keep(t);
        keep[i * 64 + lane] = w;
        live |= wave_any(w != 0) ? 1u << i : 0u;
      }
    }
    if (live == 0) continue;

    // ---- the tiles: K(next) and V(next) are loaded while this one is worked on ----
    f32x16 sc = f32x16{};
    int i = __builtin_ctz(live);
    live &= live - 1;
    load_k(t_w + kRWaves * (ic + i), true);
    if constexpr (SCORE) load_score(t_w + kRWaves * (ic + i), sc);
    load_v(t_w + kRWaves * (ic + i), true);
    for (;;) {
      const int k0 = (t_w + kRWaves * (ic + i)) * kRKeys;
      const bool more = live != 0;
      const int i_nx = more ? __builtin_ctz(live) : i;
      const int t_nx = t_w + kRWaves * (ic + i_nx);
      live &= live - 1;
      f32x16 s;
      if constexpr (SCORE) {
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = a.qsign < 0.f ? -sc[j] : sc[j];
      } else {
        s = f32x16{};
      }
#pragma unroll
      for (int ds = 0; ds < DS; ++ds) s = mfma32(as_vec8<T>(kf[ds]), qf[ds], s);
      load_k(t_nx, more);
      if constexpr (SCORE) load_score(t_nx, sc);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int idx = lane + u * 64, rr = idx / CH, c = idx % CH;
        lds_write16(vt + rr * ROWB + ((c ^ swz_rv<D>(rr)) * 16), vr[u]);
      }
      load_v(t_nx, more);
      // dropped entries to -inf (kept ones to 0 with scale 0)
      if (MASK || a.zero_scale || a.causal || k0 + kRKeys > Tk) {
        uint32_t w = in_row(k0);
        if constexpr (MASK) w &= keep[i * 64 + lane];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const bool kept = (w >> (8 * (j >> 2) + (j & 3))) & 1u;
          s[j] = kept ? (a.zero_scale ? 0.f : s[j]) : kNegInf;
        }
      }
      // running maximum: the first kept tile's, then raised in whole steps (the
      // rounded P then does not depend on which tile raised it, as in fa_fwd.hip)
      float mx = s[0];
#pragma unroll
      for (int j = 1; j < 16; ++j) mx = fmaxf(mx, s[j]);
      mx = half_max(mx);
      const float mc = mx * c2;
      float mneg = m_run == kNegInf ? 0.f : -m_run;
      if (wave_any(mc > (SCORE ? m_lift : m_run))) {   // (-inf for rows of far_max(): with every tile)
        const float m_new = m_run == kNegInf ? mc : raise_max(m_run, mc);
        const float alpha = m_run == kNegInf ? 0.f : exp2_fast(m_run - m_new);
        l_run *= alpha;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) oacc[nb] *= alpha;
        m_run = m_new;
        mneg = m_run == kNegInf ? 0.f : -m_run;
        if constexpr (SCORE) {
          m_lift = far_max(m_run) ? kNegInf : m_run;
          const bool far = far_max(m_run) && mx > kNegInf;
          const float sub = far ? mx : 0.f;
#pragma unroll
          for (int j = 0; j < 16; ++j) s[j] -= sub;
          if (far) mneg = mc - m_run;
        }
      }
      V8 pk[2], pkl[PREC ? 2 : 1];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[e] = exp2_fast(fmaf(s[8 * c + e], c2, mneg));
          l_run += p[e];
        }
        pk[c] = pack8<T>(p[0], p[1], p[2], p[3], p[4], p[5], p[6], p[7]);
        if constexpr (PREC) {
          float q[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) q[e] = p[e] - (float)(T)p[e];
          pkl[c] = pack8<T>(q[0], q[1], q[2], q[3], q[4], q[5], q[6], q[7]);
        }
      }
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int row = 16 * c + tr_row;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int col = nb * 32 + tr_col;
          const char* p = vt + row * ROWB + (((col >> 3) ^ swz_rv<D>(row)) * 16) + (col & 7) * 2;
          const V8 va = cat_tr<T>(lds_read_tr(p), lds_read_tr(p + 8 * ROWB));
          oacc[nb] = mfma32(va, pk[c], oacc[nb]);
          if constexpr (PREC) oacc[nb] = mfma32(va, pkl[c], oacc[nb]);
        }
      }
      if (!more) break;
      i = i_nx;
    }
  }

  // ---- merge the waves -----------------------------------------------------------
  const float l_tot = half_sum(l_run);
  if (hf == 0) {
    sml[wave][0][l32] = m_run;
    sml[wave][1][l32] = l_tot;
  }
  __syncthreads();   // also: every wave is done with its V tile and keep words
  auto merged_max = [&](int row) __attribute__((always_inline)) -> float {
    return fmaxf(fmaxf(sml[0][0][row], sml[1][0][row]), fmaxf(sml[2][0][row], sml[3][0][row]));
  };
  auto weight = [&](float m, float mm) __attribute__((always_inline)) -> float {
    return m == kNegInf ? 0.f : exp2_fast(m - mm);
  };
  {
    const float w = weight(m_run, merged_max(l32));
    float* st = (float*)smem + (wave * 32 + l32) * OS;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int gi = 0; gi < 4; ++gi) {
        f32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = oacc[nb][gi * 4 + e] * w;
        *(f32x4*)(st + nb * 32 + gi * 8 + hf * 4) = x;
      }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 32 * CH / (kRWaves * 64); ++u) {
    const int idx = tid + u * kRWaves * 64, row = idx / CH, c = idx % CH;
    const int rr = rb * 32 + row;
    if (rr >= R) continue;
    const int q_ = rr / a.G, h_ = kvh * a.G + (rr - q_ * a.G);
    const int64_t ri = ((int64_t)b * a.Hq + h_) * a.Tq + q_;
    const float mm = merged_max(row);
    float l = 0.f;
    f32x4 x0 = f32x4{}, x1 = f32x4{};
#pragma unroll
    for (int w = 0; w < kRWaves; ++w) {
      l += sml[w][1][row] * weight(sml[w][0][row], mm);
      const float* st = (const float*)smem + (w * 32 + row) * OS + c * 8;
      x0 += *(const f32x4*)st;
      x1 += *(const f32x4*)(st + 4);
    }
    if (a.ns > 1) {
      const int64_t pr = (int64_t)sp * a.B * a.Hq * a.Tq + ri;
      float* po = a.part_o + pr * D + c * 8;
      *(f32x4*)po = x0;
      *(f32x4*)(po + 4) = x1;
      if (c == 0) {
        a.part_ml[2 * pr] = mm;
        a.part_ml[2 * pr + 1] = l;
      }
    } else {
      if (8 * c >= a.Dv) continue;
      const float inv = 1.0f / l;
      x0 *= inv;
      x1 *= inv;
      hold(x0, x1);
      const V8 o = pack8<T>(x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]);
      gstore16((T*)a.o + b * a.osb + h_ * a.osh + (int64_t)q_ * a.ost + c * 8, as_u32x4<T>(o));
      if (PREC && a.olo) {
        const V8 lo = pack8<T>(x0[0] - (float)o[0], x0[1] - (float)o[1], x0[2] - (float)o[2], x0[3] - (float)o[3],
                               x1[0] - (float)o[4], x1[1] - (float)o[5], x1[2] - (float)o[6], x1[3] - (float)o[7]);
        gstore16((T*)a.olo + b * a.olsb + h_ * a.olsh + (int64_t)q_ * a.olst + c * 8, as_u32x4<T>(lo));
      }
      if (c == 0) a.lse[ri] = l > 0.f ? mm + log2_fast(l) : kPosInf;
    }
  }
}

// ---------------------------------------------------------------------------
// O and LSE from the partial results of a.ns key ranges
// ---------------------------------------------------------------------------
// LPR lanes of a wave per row and NW waves: lane i < ns of them holds range i's
// maximum and sum; D / 8 lanes share the row's columns, and the NW LPR / (D / 8)
// groups of those the ranges, summed over the groups at the end (fixed order:
// deterministic).  Few ranges: LPR = D / 8, several rows per wave, each lane
// reading all of its ranges; up to 64 (decoding: few rows): a workgroup per row,
// whose waves take a quarter of the ranges each (64 ranges of 32 rows: 4.6 us, 9.1
// with a wave per row).  Bound by the latency and the
// per-CU rate of reading the partials, which the launch before left in L2.
template <typename T, int D, int LPR, int NW>
__global__ __launch_bounds__(256) void fwd_combine_kernel(const FwdArgs a) {
  using V8 = typename Vec8<T>::type;
  static_assert(NW == 1 || (NW == 4 && LPR == 64), "waves of one row");
  constexpr int CH = D / 8, NG = NW * LPR / CH, RPB = 256 / (NW * LPR);
  const int lane = threadIdx.x % LPR, c = lane % CH;
  const int grp = (NW == 1 ? 0 : (int)(threadIdx.x / 64) * (LPR / CH)) + lane / CH;
  const int64_t rows = (int64_t)a.B * a.Hq * a.Tq;
  const int64_t rb = (int64_t)blockIdx.x * RPB + (NW == 1 ? threadIdx.x / LPR : 0);
  const int64_t ri = min_i64(rb, rows - 1);
  const bool mine = rb < rows;
  const int q = (int)(ri % a.Tq);
  const int64_t bh = ri / a.Tq;
  const int b = (int)(bh / a.Hq), h = (int)(bh - (int64_t)b * a.Hq);
  float m = kNegInf, l = 0.f;
  if (lane < a.ns) {
    m = a.part_ml[2 * (lane * rows + ri)];
    l = a.part_ml[2 * (lane * rows + ri) + 1];
  }
  float mm = m;
#pragma unroll
  for (int d = 1; d < LPR; d <<= 1) mm = fmaxf(mm, __shfl_xor(mm, d));
  const float w = m == kNegInf ? 0.f : exp2_fast(m - mm);
  float lt = l * w;
#pragma unroll
  for (int d = 1; d < LPR; d <<= 1) lt += __shfl_xor(lt, d);
  f32x4 x0 = f32x4{}, x1 = f32x4{};
  // (a lane's loads all in flight: one load latency)
#pragma unroll 8
  for (int i = grp; i < (a.ns + NG - 1) / NG * NG; i += NG) {
    const float wi = __shfl(w, i, LPR);   // ranges past ns have weight 0
    const float* p = a.part_o + ((int64_t)min(i, a.ns - 1) * rows + ri) * D + c * 8;
    const f32x4 y0 = *(const f32x4*)p, y1 = *(const f32x4*)(p + 4);
    if (i < a.ns) {
      x0 += y0 * wi;
      x1 += y1 * wi;
    }
  }
#pragma unroll
  for (int d = CH; d < LPR; d <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x0[e] += __shfl_xor(x0[e], d);
      x1[e] += __shfl_xor(x1[e], d);
    }
  if constexpr (NW > 1) {   // lane c of each wave holds the wave's sum
    __shared__ f32x4 part[NW][CH][2];
    const int w = threadIdx.x / 64;
    if (lane < CH) {
      part[w][c][0] = x0;
      part[w][c][1] = x1;
    }
    __syncthreads();
    x0 = part[0][c][0];
    x1 = part[0][c][1];
#pragma unroll
    for (int i = 1; i < NW; ++i) {
      x0 += part[i][c][0];
      x1 += part[i][c][1];
    }
  }
  if (grp != 0 || !mine || 8 * c >= a.Dv) return;
  const float inv = 1.0f / lt;
  x0 *= inv;
  x1 *= inv;
  hold(x0, x1);
  const V8 o = pack8<T>(x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]);
  gstore16((T*)a.o + b * a.osb + h * a.osh + (int64_t)q * a.ost + c * 8, as_u32x4<T>(o));
  if (a.olo) {
    const V8 lo = pack8<T>(x0[0] - (float)o[0], x0[1] - (float)o[1], x0[2] - (float)o[2], x0[3] - (float)o[3],
                           x1[0] - (float)o[4], x1[1] - (float)o[5], x1[2] - (float)o[6], x1[3] - (float)o[7]);
    gstore16((T*)a.olo + b * a.olsb + h * a.olsh + (int64_t)q * a.olst + c * 8, as_u32x4<T>(lo));
  }
  if (c == 0) a.lse[ri] = lt > 0.f ? mm + log2_fast(lt) : kPosInf;
}

template <typename T, int D>
hipError_t launch_rows_t(const FwdArgs& a, hipStream_t s) {
  const int nrb = (a.Tq * a.G + 31) / 32;
  const dim3 grid((unsigned)(a.B * a.Hk * a.ns * nrb)), block(kRWaves * 64);
  const bool m = a.mask != nullptr, sc = a.score != nullptr;
  if (m && sc) hipLaunchKernelGGL((fwd_rows_kernel<T, D, true, true>), grid, block, 0, s, a);
  else if (m) hipLaunchKernelGGL((fwd_rows_kernel<T, D, true, false>), grid, block, 0, s, a);
  else if (sc) hipLaunchKernelGGL((fwd_rows_kernel<T, D, false, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((fwd_rows_kernel<T, D, false, false>), grid, block, 0, s, a);
  return hipGetLastError();
}

template <typename T, int D>
hipError_t launch_combine_t(const FwdArgs& a, hipStream_t s) {
  const int64_t rows = (int64_t)a.B * a.Hq * a.Tq;
  if (a.ns <= 8) {   // D / 8 >= 8 lanes per row
    constexpr int RPB = 256 / (D / 8);
    hipLaunchKernelGGL((fwd_combine_kernel<T, D, D / 8, 1>), dim3((unsigned)((rows + RPB - 1) / RPB)), dim3(256), 0, s, a);
  } else {
    hipLaunchKernelGGL((fwd_combine_kernel<T, D, 64, 4>), dim3((unsigned)rows), dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t launch_rows_d(const FwdArgs& a, int D, hipStream_t s) {
  if (D == 64) return launch_rows_t<T, 64>(a, s);
  if (D == 128) return launch_rows_t<T, 128>(a, s);
  if (D == 256) return launch_rows_t<T, 256>(a, s);
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_combine_d(const FwdArgs& a, int D, hipStream_t s) {
  if (D == 64) return launch_combine_t<T, 64>(a, s);
  if (D == 128) return launch_combine_t<T, 128>(a, s);
  if (D == 256) return launch_combine_t<T, 256>(a, s);
  return hipErrorInvalidValue;
}

}  // namespace

int fwd_rows_keys() { return kRKeys; }

hipError_t launch_fwd_rows(const FwdArgs& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_rows_d<bf16>(a, D, s) : launch_rows_d<f16>(a, D, s);
}

hipError_t launch_fwd_combine(const FwdArgs& a, int D, int dtype, hipStream_t s) {
  return dtype == 0 ? launch_combine_d<bf16>(a, D, s) : launch_combine_d<f16>(a, D, s);
}

}  // namespace fa
