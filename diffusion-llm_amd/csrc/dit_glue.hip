// dit_glue.hip - the elementwise work around attention in a DiT block, fused.
//
// ln_modulate_kernel: modulate(LN(x), shift, scale) of DiTBlock.forward
//   (model/modules.py:537-568) with the weight-only LayerNorm
//   (model/modules.py:243-288) and modulate (model/modules.py:778-788), one
//   read of x and one write of the result instead of ~8 eager ops:
//     mean, var (correction 0) of the fp32-upcast row; inv = rsqrt(var + eps);
//     y = (w * (x - mean)) * inv in fp32, cast back to x's dtype;
//     out = y * (1 + scale) + shift: 1 + scale in the vectors' dtype (a
//     Python scalar does not promote), the product and the sum in the
//     promoted dtype of y and the vectors (bf16 if both are bf16, every op
//     rounded, as eager bf16 tensor ops; fp32 otherwise), optionally rounded
//     to bf16 for the next matmul (what autocast does at its input).
//   FUSED: of the updated residual row x + gate * y, which is stored too.
//   Bound by HBM: a row is read once into registers (d_model <= 4096), its sums
//   are reduced with DPP and permlane swaps. Dtypes are template arguments and
//   every load and store of a wave is one contiguous piece (4-element chunks: 1
//   KB of fp32, 512 B of bf16); with 8-element chunks and run-time dtypes a
//   fp32 load spanned twice its bytes, a bf16 one was issued twice, half the
//   lanes of a 768-wide row were idle and every row reloaded its vectors (6 KB
//   against the row's own 4.5). 8 x 2048 x 768, fp32 x, bf16 result: 17.2 ->
//   12.9 us (5.9 TB/s); FUSED 37.6 -> 31.1 us (4.9 TB/s); bf16 x: 16.7 -> 11.8
//   and 29.3 -> 23.4 us; 4096 x 2048 fp32: 15.9 -> 12.4 and 26.4 -> 23.5 us. Two
//   waves to a row above 2048 features: see ln_modulate_kernel.
// gate_residual_kernel: x + gate * y (the residual updates of
//   DiTBlock.forward, :560-566): gate * y in the promoted dtype of gate and y,
//   then the add in the promoted dtype of x and that product; bit-exact with
//   the eager ops. out may alias x.
#include <algorithm>

#include "bd3_device.h"
#include "bd3_launch.h"
#include "bd3_mask.h"

namespace bd3 {
namespace {

__device__ __forceinline__ float rbf(float f) { return (float)(__bf16)f; }  // round to bf16 (RNE)

// 8 consecutive elements starting at p (16-byte aligned for bf16, 32 for
// fp32) as raw bits: two 16-byte loads, the second of the same 16 bytes when
// the elements are bf16, so the pair is issued without a branch on the dtype.
struct Raw8 {
  u32x4 lo, hi;
};

__device__ __forceinline__ Raw8 ld_raw8(const void* p, int fp32) {
  Raw8 r;
  r.lo = ld16(p);
  r.hi = ld16(static_cast<const char*>(p) + (fp32 ? 16 : 0));
  return r;
}

__device__ __forceinline__ void unpack8(const Raw8& r, int fp32, float (&v)[8]) {
  float f[8], b[8];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    // (element values first: __builtin_bit_cast of a vector element lvalue
    // reads element 0 with this compiler)
    const uint32_t l = r.lo[k], h = r.hi[k];
    f[k] = __uint_as_float(l);
    f[4 + k] = __uint_as_float(h);
    b[2 * k] = __uint_as_float(l << 16);
    b[2 * k + 1] = __uint_as_float(l & 0xffff0000u);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = fp32 ? f[e] : b[e];
}

__device__ __forceinline__ void store8(void* p, int fp32, const float (&v)[8]) {
  if (fp32) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
    *(reinterpret_cast<f32x4*>(p) + 1) = f32x4{v[4], v[5], v[6], v[7]};
  } else {
    *reinterpret_cast<bf16x8*>(p) = to_bf16x8(v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7]);
  }
}

__device__ __forceinline__ const char* elem(const void* base, int fp32, int64_t i) {
  return static_cast<const char*>(base) + i * (fp32 ? 4 : 2);
}

// 4 consecutive elements as loaded: fp32 (16 bytes) or bf16 (8 bytes).
template <bool F32>
struct Raw4;
template <>
struct Raw4<true> {
  u32x4 v;
  __device__ __forceinline__ void load(const void* p) { v = ld16(p); }
  __device__ __forceinline__ void get(float (&f)[4]) const {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = v[k];
      f[k] = __uint_as_float(w);
    }
  }
};
template <>
struct Raw4<false> {
  u32x2 v;
  __device__ __forceinline__ void load(const void* p) { v = *static_cast<const u32x2*>(p); }
  __device__ __forceinline__ void get(float (&f)[4]) const {
    const uint32_t l = v[0], h = v[1];
    f[0] = __uint_as_float(l << 16);
    f[1] = __uint_as_float(l & 0xffff0000u);
    f[2] = __uint_as_float(h << 16);
    f[3] = __uint_as_float(h & 0xffff0000u);
  }
};

__device__ __forceinline__ void store4(void* p, bool fp32, const float (&v)[4]) {
  if (fp32)
    *static_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
  else
    *static_cast<bf16x4*>(p) = to_bf16x4(v[0], v[1], v[2], v[3]);
}

// modulate(LN(row), shift, scale), with FUSED of the updated residual row
// x + gate * y (gate_residual_kernel's dtypes and roundings), which is stored
// too: one launch and one read of the residual instead of two of each
// (DiTBlock.forward, model/modules.py:560-566 then the next sublayer's
// :537-568). out_x may alias x (a wave has read its chunks of the row before it
// writes them, and no other wave uses them).
//
// A wave owns `a.wave_rows` consecutive rows; lane l holds the 4-element chunks
// l, l + 64, ... of a row, so every load and store of a wave is one contiguous
// piece. CH: chunks per lane. Rows of up to 4 chunks per lane keep the gain, 1 +
// scale and shift (and the gate) in registers from row to row and request the
// next row before they work on the current one; longer rows load them per row.
// XF / MF / YF: x, the vectors, y in fp32.
//
// PAIR: rows of more than 2048, two waves (a 128-thread workgroup) to a row,
// each with every other run of 64 chunks, and the sums exchanged through LDS:
// 126-228 VGPRs, two to four waves per SIMD. One wave a row would hold up to 16
// chunks per lane (246-256 VGPRs and up to 184 AGPRs, one or two waves per SIMD).
// us with one -> two waves, bf16 result, x / vectors: 16384 x 2304 bf16 / fp32 76.8
// -> 37.5, bf16 / bf16 FUSED 136.9 -> 76.7; 16384 x 4096 fp32 / bf16 87.0 -> 82.5,
// FUSED 182 -> 152, bf16 / bf16 FUSED 176 -> 110; 1024 x 4096 fp32 / bf16 8.4 (8.4),
// FUSED 14.3 -> 13.4.
template <int CH, bool XF, bool MF, bool YF, bool FUSED, bool PAIR>
__global__ __launch_bounds__(PAIR ? 128 : 256) void ln_modulate_kernel(GlueArgs a) {
#pragma clang fp contract(off)  // separate products and sums, as the eager ops
  static_assert(!PAIR || CH > 4, "shorter rows keep their vectors");
  constexpr int kStep = PAIR ? 128 : 64;  // chunks between a lane's chunks
  constexpr bool KEEP = CH <= 4;
  constexpr bool kGyBf16 = !MF && !YF;
  constexpr bool kRowF32 = FUSED ? XF || MF || YF : XF;  // dtype of the row that is normalised
  constexpr bool kModBf16 = !kRowF32 && !MF;             // modulate in bf16 iff the row and the vectors are
  const int lane = PAIR ? wi_x() : wi_x() & 63;  // in the row
  const int wave = PAIR ? wg_x() : wave_uniform((int)(wg_x() * (a.wg_threads >> 6) + (wi_x() >> 6)));
  // unsigned: the last workgroup's waves may start past 2^31 (at most 2^25 + 3 waves of 64 rows)
  const uint32_t first = (uint32_t)a.row0 + (uint32_t)wave * (uint32_t)a.wave_rows;
  if (first >= (uint32_t)a.rows) return;
  const int r0 = (int)first, r1 = r0 + imin(a.wave_rows, a.rows - r0);
  const int nch = a.d >> 2;
  const float d_inv = (float)a.d;
  int col[CH];  // first element of the lane's chunk k (lanes past the row repeat its last chunk)
#pragma unroll
  for (int k = 0; k < CH; ++k) col[k] = 4 * imin(lane + kStep * k, nch - 1);

  auto x_row = [&](int b, int s) { return elem(a.x, XF, (int64_t)b * a.sx_b + (int64_t)s * a.sx_s); };
  auto y_row = [&](int b, int s) { return elem(a.y, YF, (int64_t)b * a.sy_b + (int64_t)s * a.sy_s); };
  Raw4<XF> xr[CH];
  Raw4<YF> yr[FUSED ? CH : 1];
  auto load_row = [&](int b, int s) {
    const char* xp = x_row(b, s);
#pragma unroll
    for (int k = 0; k < CH; ++k) xr[k].load(xp + col[k] * (XF ? 4 : 2));
    if constexpr (FUSED) {
      const char* yp = y_row(b, s);
#pragma unroll
      for (int k = 0; k < CH; ++k) yr[k].load(yp + col[k] * (YF ? 4 : 2));
    }
  };
  int b = r0 / a.seq, s = r0 - b * a.seq;
  load_row(b, s);

  // gain; 1 + scale (rounded to the vectors' dtype: a Python scalar does not promote); shift; gate
  constexpr int KV = KEEP ? CH : 1;
  float w[KV][4], t[KV][4], sh[KV][4];
  Raw4<MF> gate[FUSED && KEEP ? CH : 1];
  auto load_w = [&](int k, float (&f)[4]) {
    if (a.w_fp32) {
      Raw4<true> r;
      r.load(elem(a.weight, 1, col[k]));
      r.get(f);
    } else {
      Raw4<false> r;
      r.load(elem(a.weight, 0, col[k]));
      r.get(f);
    }
  };
  auto one_plus = [&](const Raw4<MF>& r, float (&f)[4]) {
    r.get(f);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = MF ? 1.f + f[e] : rbf(1.f + f[e]);
  };
  auto load_vectors = [&](int bb) {
    Raw4<MF> rt[KV], rs[KV];
#pragma unroll
    for (int k = 0; k < KV; ++k) {
      rt[k].load(elem(a.scale, MF, (int64_t)bb * a.sm_b + col[k]));
      rs[k].load(elem(a.shift, MF, (int64_t)bb * a.sm_b + col[k]));
      if constexpr (FUSED) gate[k].load(elem(a.gate, MF, (int64_t)bb * a.sm_b + col[k]));
    }
#pragma unroll
    for (int k = 0; k < KV; ++k) {
      one_plus(rt[k], t[k]);
      rs[k].get(sh[k]);
    }
  };
  // Rows of more than 4 chunks: requested with the row, decoded where they are
  // used. The gain's dtype is a run-time flag: two 8-byte loads (the same 8
  // bytes twice for bf16) instead of a branch that would wait for its load.
  constexpr int RV = KEEP ? 1 : CH;
  Raw4<MF> vt[RV], vs[RV], vg[FUSED ? RV : 1];
  u32x2 wlo[RV], whi[RV];
  if constexpr (KEEP) {
#pragma unroll
    for (int k = 0; k < CH; ++k) load_w(k, w[k]);
    load_vectors(b);
  } else {
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      if constexpr (FUSED) vg[k].load(elem(a.gate, MF, (int64_t)b * a.sm_b + col[k]));
      const char* wp = elem(a.weight, a.w_fp32, col[k]);
      wlo[k] = *reinterpret_cast<const u32x2*>(wp);
      whi[k] = *reinterpret_cast<const u32x2*>(wp + (a.w_fp32 ? 8 : 0));
      vt[k].load(elem(a.scale, MF, (int64_t)b * a.sm_b + col[k]));
      vs[k].load(elem(a.shift, MF, (int64_t)b * a.sm_b + col[k]));
    }
  }
  // Sum over the row's lanes. PAIR: of the two waves' sums, an LDS slot for each
  // and for each of the row's two sums.
  __shared__ float part[2][2];
  auto row_sum = [&](float v, int use) {
    v = wave_sum(v);
    if constexpr (PAIR) {
      const int half = (int)wi_x() >> 6;
      if ((wi_x() & 63) == 0) part[use][half] = v;
      __syncthreads();
      v += part[use][half ^ 1];
    }
    return v;
  };

  for (int row = r0;;) {
    // the row's values (zero past its end); with FUSED the updated residual, stored
    float v[CH][4];
    if constexpr (FUSED) {
      char* xo = const_cast<char*>(elem(a.out_x, kRowF32, (int64_t)b * a.sxo_b + (int64_t)s * a.sxo_s));
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        float xv[4], yv[4], gv[4];
        xr[k].get(xv);
        yr[k].get(yv);
        if constexpr (KEEP) {
          gate[k].get(gv);
        } else {
          vg[k].get(gv);
        }
        const bool in = lane + kStep * k < nch;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float gy = gv[e] * yv[e];
          if (kGyBf16) gy = rbf(gy);
          const float o = xv[e] + gy;
          v[k][e] = in ? (kRowF32 ? o : rbf(o)) : 0.f;
        }
        if (in) store4(xo + (int64_t)col[k] * (kRowF32 ? 4 : 2), kRowF32, v[k]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < CH; ++k) {
        xr[k].get(v[k]);
        const bool in = lane + kStep * k < nch;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[k][e] = in ? v[k][e] : 0.f;
      }
    }
    const int nrow = row + 1;
    int nb = b, ns = s + 1;
    if (ns == a.seq) {
      ns = 0;
      ++nb;
    }
    if constexpr (KEEP)
      if (nrow < r1) load_row(nb, ns);

    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < CH; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) sum += v[k][e];
    const float mean = row_sum(sum, 0) / d_inv;
    float sq = 0.f;
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      const bool in = lane + kStep * k < nch;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[k][e] -= mean;
        const float dd = v[k][e] * v[k][e];
        sq += in ? dd : 0.f;
      }
    }
    const float inv = rsqrtf(row_sum(sq, 1) / d_inv + a.eps);
    char* outr = const_cast<char*>(elem(a.out, a.out_fp32, (int64_t)b * a.so_b + (int64_t)s * a.so_s));
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      float wk[4], tk[4], shk[4], o[4];
      if constexpr (!KEEP) {
        float wb[4];
        Raw4<false>{wlo[k]}.get(wb);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t f = e < 2 ? wlo[k][e] : whi[k][e - 2];
          wk[e] = a.w_fp32 ? __uint_as_float(f) : wb[e];
        }
        one_plus(vt[k], tk);
        vs[k].get(shk);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float y = ((KEEP ? w[KEEP ? k : 0][e] : wk[e]) * v[k][e]) * inv;
        if (!kRowF32) y = rbf(y);  // .to(original dtype)
        const float te = KEEP ? t[KEEP ? k : 0][e] : tk[e], se = KEEP ? sh[KEEP ? k : 0][e] : shk[e];
        o[e] = kModBf16 ? rbf(rbf(y * te) + se) : y * te + se;
      }
      if (lane + kStep * k < nch) store4(outr + (int64_t)col[k] * (a.out_fp32 ? 4 : 2), a.out_fp32, o);
    }
    if (!KEEP || nrow >= r1) break;
    if constexpr (KEEP)
      if (nb != b) load_vectors(nb);
    row = nrow;
    b = nb;
    s = ns;
  }
}

// x + gate * y with an fp32 residual (the result is fp32): 4 elements per
// thread, so each load of x (16 bytes per lane) covers one contiguous 1 KB
// per wave, where 8-element chunks (two 16-byte halves 32 bytes apart per
// lane) split every load across twice the span. GF / YF: gate / y in fp32.
// Measured at 8 x 2048 x 768: 25.8 -> 23.3 us, bit-identical.
template <bool GF, bool YF>
__global__ __launch_bounds__(256) void gate_residual_f32_kernel(GlueArgs a) {
#pragma clang fp contract(off)  // gate * y rounded before the add, as the eager ops
  const int64_t e = (int64_t)wg_x() * 256 + wi_x();  // one 4-element chunk
  const int nch = a.d >> 2;
  if (e >= (int64_t)a.rows * nch) return;
  const int row = (int)(e / nch), c = (int)(e - (int64_t)row * nch);
  const int b = row / a.seq, s = row - b * a.seq;
  Raw4<true> xr;
  Raw4<GF> gr;
  Raw4<YF> yr;
  xr.load(static_cast<const float*>(a.x) + (int64_t)b * a.sx_b + (int64_t)s * a.sx_s + 4 * c);
  gr.load(elem(a.shift, GF, (int64_t)b * a.sm_b + 4 * c));  // gate
  yr.load(elem(a.y, YF, (int64_t)b * a.sy_b + (int64_t)s * a.sy_s + 4 * c));
  float x[4], g[4], y[4];
  xr.get(x);
  gr.get(g);
  yr.get(y);
  const bool gy_bf16 = !GF && !YF;
  f32x4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    float gy = g[k] * y[k];
    if (gy_bf16) gy = rbf(gy);
    o[k] = x[k] + gy;
  }
  *reinterpret_cast<f32x4*>(static_cast<float*>(a.out) + (int64_t)b * a.so_b + (int64_t)s * a.so_s + 4 * c) = o;
}

__global__ __launch_bounds__(256) void gate_residual_kernel(GlueArgs a) {
#pragma clang fp contract(off)  // gate * y rounded before the add, as the eager ops
  const int64_t e = (int64_t)wg_x() * 256 + wi_x();  // one 8-element chunk
  const int nch = a.d >> 3;
  if (e >= (int64_t)a.rows * nch) return;
  const int row = (int)(e / nch), c = (int)(e - (int64_t)row * nch);
  const int b = row / a.seq, s = row - b * a.seq;
  const Raw8 xr = ld_raw8(elem(a.x, a.x_fp32, (int64_t)b * a.sx_b + (int64_t)s * a.sx_s + 8 * c), a.x_fp32);
  const Raw8 gr = ld_raw8(elem(a.shift, a.m_fp32, (int64_t)b * a.sm_b + 8 * c), a.m_fp32);  // gate
  const Raw8 yr = ld_raw8(elem(a.y, a.y_fp32, (int64_t)b * a.sy_b + (int64_t)s * a.sy_s + 8 * c), a.y_fp32);
  float x[8], g[8], y[8], o[8];
  unpack8(xr, a.x_fp32, x);
  unpack8(gr, a.m_fp32, g);
  unpack8(yr, a.y_fp32, y);
  const bool gy_bf16 = !a.m_fp32 && !a.y_fp32;
  const bool out_bf16 = !a.x_fp32 && gy_bf16;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    float gy = g[k] * y[k];
    if (gy_bf16) gy = rbf(gy);
    o[k] = x[k] + gy;  // rounded to bf16 by the store when both are bf16
  }
  store8(const_cast<char*>(elem(a.out, !out_bf16, (int64_t)b * a.so_b + (int64_t)s * a.so_s + 8 * c)), !out_bf16, o);
}

}  // namespace

namespace {
bool glue_pair(int d) { return d > 2048; }  // two waves to a row
// 4-element chunks of a row per lane.
int glue_chunks(int d) { return (d / 4 + (glue_pair(d) ? 127 : 63)) / (glue_pair(d) ? 128 : 64); }
}  // namespace

// Rows per wave: enough waves to keep 8 per SIMD (8192 over 1024 SIMDs), then
// up to 8 rows each, so that the vectors are loaded once for them and the
// next row is on its way. 8 x 2048 rows x 768 (fp32 residual): fused 31.1 us at
// 2 rows a wave, 32.5 at 4, 34.4 at 8, 31.9 at 1; alone 12.9 / 12.8 / 13.6 /
// 13.8. Few rows take one-wave workgroups, which spread over all CUs. A launch
// holds fewer than 2^32 threads: very many short rows take more than 8 a wave,
// longer ones go out in launches of 2^24.
GlueGrid glue_grid(int rows, int d) {
  GlueGrid g;
  const bool several = glue_chunks(d) <= 4;
  g.rows = several ? rows : imin(rows, 1 << 24);
  g.wave_rows = several ? imax(imin(imax(rows / 8192, 1), 8), (int)(((int64_t)rows + (1 << 25) - 1) >> 25)) : 1;
  const int64_t waves = ((int64_t)g.rows + g.wave_rows - 1) / g.wave_rows;
  g.threads = glue_pair(d) ? 128 : waves <= 1024 ? 64 : 256;
  const int64_t per = glue_pair(d) ? 1 : g.threads / 64;  // waves (pairs of them) per workgroup
  g.workgroups = (unsigned)((waves + per - 1) / per);
  return g;
}

namespace {

template <int CH, bool FUSED, bool PAIR = false>
void launch_rows_ch(const GlueArgs& a, dim3 grid, dim3 block, hipStream_t stream) {
#define BD3_ROWS(XF, MF, YF) hipLaunchKernelGGL((ln_modulate_kernel<CH, XF, MF, YF, FUSED, PAIR>), grid, block, 0, stream, a)
  const int t = (a.x_fp32 ? 4 : 0) | (a.m_fp32 ? 2 : 0) | (FUSED && a.y_fp32 ? 1 : 0);
  switch (t) {
    case 0: BD3_ROWS(false, false, false); break;
    case 2: BD3_ROWS(false, true, false); break;
    case 4: BD3_ROWS(true, false, false); break;
    case 6: BD3_ROWS(true, true, false); break;
    default:
      if constexpr (FUSED) {
        if (t == 1) BD3_ROWS(false, false, true);
        if (t == 3) BD3_ROWS(false, true, true);
        if (t == 5) BD3_ROWS(true, false, true);
        if (t == 7) BD3_ROWS(true, true, true);
      }
  }
#undef BD3_ROWS
}

template <bool FUSED>
hipError_t launch_rows(GlueArgs a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  const int ch = glue_chunks(a.d);
  if (ch > 8) return hipErrorInvalidValue;  // d_model > 4096: rejected by the C ABI
  const GlueGrid g = glue_grid(a.rows, a.d);
  a.wave_rows = g.wave_rows;
  a.wg_threads = g.threads;
  const dim3 block(g.threads), grid(g.workgroups);
  const int rows = a.rows;
  for (int64_t r = 0; r < rows; r += g.rows) {
    a.row0 = (int)r;
    a.rows = (int)std::min<int64_t>(rows, r + g.rows);  // the launch's end
    if (glue_pair(a.d))
      ch <= 6 ? launch_rows_ch<6, FUSED, true>(a, grid, block, stream)
              : launch_rows_ch<8, FUSED, true>(a, grid, block, stream);
    else if (ch <= 1)
      launch_rows_ch<1, FUSED>(a, grid, block, stream);
    else if (ch <= 2)
      launch_rows_ch<2, FUSED>(a, grid, block, stream);
    else if (ch <= 3)
      launch_rows_ch<3, FUSED>(a, grid, block, stream);
    else if (ch <= 4)
      launch_rows_ch<4, FUSED>(a, grid, block, stream);
    else if (ch <= 6)
      launch_rows_ch<6, FUSED>(a, grid, block, stream);
    else
      launch_rows_ch<8, FUSED>(a, grid, block, stream);
  }
  return hipGetLastError();
}

}  // namespace

hipError_t launch_ln_modulate(const GlueArgs& a, hipStream_t stream) { return launch_rows<false>(a, stream); }

hipError_t launch_gate_residual_ln_modulate(const GlueArgs& a, hipStream_t stream) {
  return launch_rows<true>(a, stream);
}

hipError_t launch_gate_residual(const GlueArgs& a, hipStream_t stream) {
  if (a.x_fp32) {  // fp32 residual and result: 4-element chunks
    const int64_t n4 = (int64_t)a.rows * (a.d >> 2);
    if (n4 == 0) return hipSuccess;
    const dim3 grid((unsigned)((n4 + 255) / 256));
    if (a.m_fp32 && a.y_fp32)
      hipLaunchKernelGGL((gate_residual_f32_kernel<true, true>), grid, dim3(256), 0, stream, a);
    else if (a.m_fp32)
      hipLaunchKernelGGL((gate_residual_f32_kernel<true, false>), grid, dim3(256), 0, stream, a);
    else if (a.y_fp32)
      hipLaunchKernelGGL((gate_residual_f32_kernel<false, true>), grid, dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((gate_residual_f32_kernel<false, false>), grid, dim3(256), 0, stream, a);
    return hipGetLastError();
  }
  const int64_t n = (int64_t)a.rows * (a.d >> 3);
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(gate_residual_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

}  // namespace bd3
