// subs_sample.hip - one ancestral denoising step of BD3-LM sampling, fused:
// SUBS parameterization + categorical draw + carry-over of unmasked tokens.
//
// Counterpart of subs_parameterization (model/subs.py:11-43) followed by the
// sampler's update (sample/sampler.py:110-122) and sample_categorical
// (sample/sampler.py:11-34), for rows whose token is [MASK] (the others keep
// their token, which is what torch.where(block != mask, block, new) does):
//   x_i   = logits_i + bias_i            (bias = NEG_INF = -1e6 at [MASK], in the logits dtype)
//   lp_i  = (x_i - max x) - log(sum_j exp(x_j - max x))   (model/modules.py:791-799)
//   q_i   = double(exp(lp_i)) * (1 - s/t),  q_mask = s/t
//   new   = argmax_i q_i / (EPS - log(u_i + EPS)),  u_i ~ U[0, 1) in float64, EPS = 1e-10
// in the dtypes the reference runs under bf16 autocast: for bf16 logits the
// bias add and the shift x - max are bf16 ops (rounded), exp / sum / log and
// the final subtraction are fp32; for fp32 logits everything up to q is
// fp32. q, the noise and the ratio are float64, as in the reference.
// The uniforms come either from the caller (u, float64 per element: the
// reference's torch.rand_like draw, for exact reproduction) or from the
// counter-based Philox4x32-10 generator (Salmon, Moraes, Dror, Shaw,
// "Parallel random numbers: as easy as 1, 2, 3", SC'11), keyed by a 64-bit
// seed with the 64-bit element-pair index and a 64-bit offset as counter, so
// no noise tensor is materialised.
//
// subs_scan_kernel: a workgroup takes a row's maximum (16-byte loads; the row is
//   in L2 for all but the first of its workgroups), then reads its slice of the
//   row ONCE: the fp32 sum of exponentials and, in the same pass, the candidates
//   for the draw. With e_i = exp(x_i - max) and g_i = EPS - log(u_i + EPS) the
//   winner maximises q_i / g_i, i.e. e_i / g_i up to the row's normaliser, so
//   no element needs the sum first: fp32 bounds of e_i / g_i against a running
//   lower bound of the best one leave a few candidates per row, and only those
//   take the float64 logarithm and division, once the sum is known. Every bound
//   errs towards keeping an element, so the token is the one the full
//   evaluation gives.
//   Up to kSubsSpreadRows rows, 512 workgroups (two per CU) are dealt out over
//   the masked rows and cut each into up to 16 slices; above, or without a
//   workspace, one workgroup does a whole row.
// subs_finish_kernel (spread calls): one workgroup per row adds the slices'
//   sums and evaluates their candidates.
//
// Bound by the instructions per element (~37, Philox's ten rounds per element
// pair about half of them), not by reading the logits. Against one 1024-thread
// workgroup per row with three passes over an LDS copy of it (131 KB, so one
// per CU) and the float64 path inside the last pass, per call at 50258 bf16
// logits: 16 masked rows 57 -> 12.3 us (scan 7.7, finish 3.8), 256 rows half of
// them masked 58.7 -> 20.1, all masked 58.7 -> 27.0; a block with no masked row
// left 3-4 -> 5 us (the second launch: the host does not know the tokens). 1024 workgroups instead of
// 512 take 26.4 and 32.3 us for the last two (every slice reads its whole row
// for the maximum), 256 take 21.6 and 28.4; a slice per workgroup in grid order
// instead of dealing the masked rows out took 31.1 us for the half-masked ones.
// Logits must be finite (the token drawn for a row with NaN / inf logits is
// unspecified).
#include "bd3_device.h"
#include "bd3_launch.h"

namespace bd3 {
namespace {

constexpr int kSubsThreads = 1024;
constexpr float kNegInf = -1e6f;   // model/subs.py:8
constexpr double kEps = 1e-10;     // sample/sampler.py:8

__device__ __forceinline__ float bf16_round(float f) {
  return (float)(__bf16)f;  // round to nearest even
}

// Philox4x32-10 block: counter c, key k (Random123's philox4x32, 10 rounds).
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
    // one three-input xor each (v_bitop3_b32; the compiler emits two)
    const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c[1], k0, 0x96);
    const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c[3], k1, 0x96);
    c[0] = n0;
    c[1] = (uint32_t)p1;
    c[2] = n2;
    c[3] = (uint32_t)p0;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
}

// 53-bit uniform in [0, 1) from 64 random bits.
__device__ __forceinline__ double u53(uint32_t lo, uint32_t hi) {
  const uint64_t v = ((uint64_t)hi << 32) | lo;
  return (double)(v >> 11) * 0x1.0p-53;
}

template <typename T>
__device__ __forceinline__ float load_logit(const T* p, int i);
template <>
__device__ __forceinline__ float load_logit<uint16_t>(const uint16_t* p, int i) {
  return __builtin_bit_cast(float, (uint32_t)p[i] << 16);
}
template <>
__device__ __forceinline__ float load_logit<float>(const float* p, int i) {
  return p[i];
}

// x_i: the logit l of element i plus the [MASK] bias, rounded to the logits dtype.
template <typename T>
__device__ __forceinline__ float biased(float l, int i, int mask_index) {
  if (i != mask_index) return l;
  if constexpr (sizeof(T) == 2) {
    return bf16_round(l + bf16_round(kNegInf));
  } else {
    return l + kNegInf;
  }
}

template <typename T>
__device__ __forceinline__ float shifted(float x, float m) {
  if constexpr (sizeof(T) == 2) {
    return bf16_round(x - m);
  } else {
    return x - m;
  }
}

__device__ __forceinline__ float block_max(float v, float* red) {
  v = wave_max(v);
  const int w = wi_x() >> 6;
  if ((wi_x() & 63) == 0) red[w] = v;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int i = 1; i < kSubsThreads / 64; ++i) r = fmaxf(r, red[i]);
  __syncthreads();
  return r;
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int w = wi_x() >> 6;
  if ((wi_x() & 63) == 0) red[w] = v;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int i = 1; i < kSubsThreads / 64; ++i) r += red[i];
  __syncthreads();
  return r;
}

// (value, index) argmax, first index on ties (torch.argmax). The ratios are
// finite and non-negative for finite logits: q >= 0 and the noise term
// EPS - log(u + EPS) > 0 for every u in [0, 1).
__device__ __forceinline__ bool better(double v, int i, double bv, int bi) {
  return v > bv || (v == bv && i < bi);
}

// Uniform of element e = row * vocab + i: the caller's, or word pair (0, 1)
// (e even) or (2, 3) (e odd) of Philox block e / 2.
__device__ __forceinline__ void philox_pair(const SubsArgs& a, uint64_t pair, uint32_t (&c)[4]) {
  c[0] = (uint32_t)pair;
  c[1] = (uint32_t)(pair >> 32);
  c[2] = (uint32_t)a.offset;
  c[3] = (uint32_t)(a.offset >> 32);
  philox4x32_10(c, (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
}

__device__ __forceinline__ double uniform_of(const SubsArgs& a, uint64_t e) {
  if (a.u != nullptr) return a.u[e];
  uint32_t c[4];
  philox_pair(a, e >> 1, c);
  return (e & 1) ? u53(c[2], c[3]) : u53(c[0], c[1]);
}

// q_i / (EPS - log(u_i + EPS)) of element i, the reference's arithmetic.
template <typename T>
__device__ double exact_ratio(const SubsArgs& a, const T* lp, uint64_t base, int i, float m, float lse) {
  double q = a.keep;  // s / t
  if (i != a.mask_index) {
    const float l = shifted<T>(load_logit<T>(lp, i), m) - lse;
    q = (double)expf(l) * (1.0 - a.keep);
  }
  return q / (kEps - log(uniform_of(a, base + i) + kEps));
}

// exp(d) for d <= 0: 2^(d log2 e) with the product's rounding error put back
// (first order), as accurate as expf without its range reduction. Below
// exp(-87) it is 0 or a flushed denormal; the clamp keeps d - ph finite.
__device__ __forceinline__ float exp_neg(float d) {
  d = fmaxf(d, -200.f);
  const float ph = d * kLog2e;
  const float pl = fmaf(d, 1.925963033500e-8f, fmaf(d, kLog2e, -ph));  // log2(e) - fp32(log2(e))
  const float e = fast_exp2(ph);
  return fmaf(e, pl * kLn2, e);
}

// Largest biased logit of the row, over the workgroup: 16-byte loads of the
// aligned middle, single elements before and after it. A 32-bit word holding
// two bf16 values orders as its upper one (the lower one only adds mantissa
// bits), so the upper values need no unpacking until the end.
template <typename T>
__device__ float row_max(const SubsArgs& a, const T* lp, float* red) {
  constexpr int E = 16 / sizeof(T);  // elements per load
  const int V = a.vocab, tid = wi_x();
  const int mis = (int)(reinterpret_cast<uintptr_t>(lp) & 15) / (int)sizeof(T);
  const int head = min((E - mis) % E, V);
  const int nb = (V - head) / E, tail0 = head + nb * E;
  const int mask = a.mask_index;
  const int bm = mask >= head && mask < tail0 ? (mask - head) / E : -1;  // the load that holds [MASK]
  float m = -INFINITY, mh = -INFINITY;
  if (tid < head) m = biased<T>(load_logit<T>(lp, tid), tid, mask);
  if (tid < V - tail0) m = fmaxf(m, biased<T>(load_logit<T>(lp, tail0 + tid), tail0 + tid, mask));
  if (tid >= 64 && tid < 64 + E && bm >= 0) {  // that load's elements one by one
    const int i = head + E * bm + tid - 64;
    m = fmaxf(m, biased<T>(load_logit<T>(lp, i), i, mask));
  }
  constexpr int U = 4;  // loads in flight
  for (int k0 = tid; k0 < nb; k0 += U * kSubsThreads) {
    u32x4 w[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      int k = min(k0 + j * kSubsThreads, nb - 1);
      if (k == bm) k = k > 0 ? 0 : nb - 1;  // another one in its place (itself if there is none)
      w[j] = ld16(lp + head + E * k);
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
      if (nb == 1 && bm == 0) break;
      float x[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint32_t v = w[j][c];
        x[c] = __uint_as_float(v);
      }
      mh = fmaxf(fmaxf(mh, x[0]), x[1]);
      mh = fmaxf(fmaxf(mh, x[2]), x[3]);
      if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = __uint_as_float(__float_as_uint(x[c]) << 16);
        m = fmaxf(fmaxf(m, x[0]), x[1]);
        m = fmaxf(fmaxf(m, x[2]), x[3]);
      }
    }
  }
  if constexpr (sizeof(T) == 2) mh = __uint_as_float(__float_as_uint(mh) & 0xffff0000u);
  return block_max(fmaxf(m, mh), red);
}

// Pruning bounds. For u below kUNear, g = EPS - log(u + EPS) is estimated from
// v_log_f32 (absolute error below 1e-6 there, relative error below 1e-4);
// nearer to 1, 1 - u <= g <= EPS + 1.0012 (1 - u), used while 1 - u > 1e-6 (the
// rounding of u + EPS in float64 stays far below). kRel covers those errors
// and the fp32 rounding of e.
constexpr float kUNear = 0.999f;
constexpr float kRel = 3e-4f;
// 1 / (EPS - log(EPS)), the least ratio e / g of the row's largest logit (e = 1).
constexpr float kLeastRatio = 0.0433f;
constexpr int kCand = 4096;      // candidates a workgroup can hold
constexpr int kSliceCand = 61;   // candidates a slice can hand over

// One slice's result (512 bytes of workspace).
struct SubsSlice {
  float m, sum, least;  // row maximum, the slice's sum of exponentials, lower bound of the best e / g
  int count;            // candidates, or -1: too many, evaluate the whole row
  int slices;           // slices of the row
  int pad;
  int index[kSliceCand];
  float most[kSliceCand];  // upper bound of the candidate's e / g
};
static_assert(sizeof(SubsSlice) == kSubsSliceBytes, "the workspace holds one SubsSlice per row and slice");

struct Best {
  double v;
  int i;
};

// Argmax over the workgroup (first index on ties); the result is valid in thread 0.
template <int NT>
__device__ __forceinline__ Best block_argmax(Best b, double* bval, int* bidx) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double ov = __shfl_xor(b.v, o, 64);
    const int oi = __shfl_xor(b.i, o, 64);
    if (better(ov, oi, b.v, b.i)) b = {ov, oi};
  }
  const int w = wi_x() >> 6;
  if ((wi_x() & 63) == 0) {
    bval[w] = b.v;
    bidx[w] = b.i;
  }
  __syncthreads();
  if (wi_x() == 0)
    for (int k = 1; k < NT / 64; ++k)
      if (better(bval[k], bidx[k], b.v, b.i)) b = {bval[k], bidx[k]};
  return b;
}

// Elements i and i + 1 of a row, both inside it; `wide`: one load of both.
template <typename T>
__device__ __forceinline__ void load_two(const T* p, bool wide, float& x0, float& x1) {
  if (!wide) {
    x0 = load_logit<T>(p, 0);
    x1 = load_logit<T>(p, 1);
  } else if constexpr (sizeof(T) == 2) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(p);
    x0 = __uint_as_float(w << 16);
    x1 = __uint_as_float(w & 0xffff0000u);
  } else {
    const float2 w = *reinterpret_cast<const float2*>(p);
    x0 = w.x;
    x1 = w.y;
  }
}

// The row a workgroup of the spread grid (a.spread) works on, its slice and
// the slices per row. Only masked rows have work, so the grid's workgroups
// are dealt out over them: rank % 8 of a row keeps its slices on one XCD (the
// row is read once into that L2). -1: nothing to do.
struct RowSlice {
  int row, slice, slices;
};
__device__ __forceinline__ RowSlice spread_rows(const SubsArgs& a, uint64_t* masks) {
  const int tid = wi_x();
  const int groups = (a.rows + 63) >> 6;  // of 64 rows, one ballot each
  for (int g = tid >> 6; g < groups; g += kSubsThreads / 64) {
    const int r = 64 * g + (tid & 63);
    const uint64_t b = __ballot(r < a.rows && a.xt[min(r, a.rows - 1)] == a.mask_index);
    if ((tid & 63) == 0) masks[g] = b;
  }
  __syncthreads();
  int active = 0;
  for (int g = 0; g < groups; ++g) active += __popcll(masks[g]);
  const int padded = max(8, (active + 7) & ~7);
  RowSlice r;
  r.slices = max(1, min(a.slices, a.spread / padded));
  r.slice = wg_x() / padded;
  int rank = wg_x() - r.slice * padded;
  r.row = -1;
  if (rank >= active || r.slice >= r.slices) return r;
  int g = 0;
  for (int n = __popcll(masks[0]); rank >= n; n = __popcll(masks[g])) {
    rank -= n;
    ++g;
  }
  // the row whose bit has `rank` set bits below it
  const uint64_t b = masks[g];
  const int below = __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0));
  const uint64_t hit = __ballot(((b >> (tid & 63)) & 1) != 0 && below == rank);
  r.row = wave_uniform(64 * g + __ffsll((unsigned long long)hit) - 1);
  return r;
}

template <typename T, bool GIVEN>
__global__ __launch_bounds__(kSubsThreads, 8) void subs_scan_kernel(SubsArgs a) {
  __shared__ float red[kSubsThreads / 64];
  __shared__ double bval[kSubsThreads / 64];
  __shared__ int bidx[kSubsThreads / 64];
  __shared__ uint64_t masks[kSubsSpreadRows / 64];
  __shared__ int c_index[kCand];
  __shared__ float c_most[kCand];
  __shared__ int c_count;
  __shared__ int c_least;  // bits of a non-negative float: ordered as integers
  constexpr int NT = kSubsThreads;
  const int tid = wi_x();
  RowSlice rs = {wg_x(), 0, 1};
  if (a.spread) {
    rs = spread_rows(a, masks);
    if (rs.row < 0) return;
  } else if (const int64_t xt = a.xt[rs.row]; xt != a.mask_index) {  // carry-over: an unmasked token stays
    if (tid == 0) a.out[rs.row] = xt;
    return;
  }
  const int row = rs.row, slice = rs.slice;
  const T* lp = static_cast<const T*>(a.logits) + (int64_t)row * a.ld;
  const int V = a.vocab;
  const uint64_t base = (uint64_t)row * (uint64_t)V;
  const float m = row_max<T>(a, lp, red);
  const float xm = biased<T>(load_logit<T>(lp, a.mask_index), a.mask_index, a.mask_index);
  // The largest logit is a real token's (always, unless [MASK]'s own exceeds
  // the others by the bias): its ratio is at least kLeastRatio. Otherwise no
  // bound holds (every e may underflow) and the whole row is evaluated.
  const bool bounded = m > xm;
  if (tid == 0) {
    c_count = 0;
    c_least = __float_as_int(bounded ? kLeastRatio : 0.f);
  }
  __syncthreads();

  float sum = 0.f;
  // Element i's exponential e into the sum and, if its ratio may be the
  // best, into the candidates. uf: u rounded to fp32 or at most 2^-32 below
  // it; om: 1 - u the same way.
  auto element = [&](int i, float x, float uf, float om, float least) {
    const float e = exp_neg(shifted<T>(x, m));
    sum += e;
    // 3.4e-10: EPS and the 2^-32 that uf may lie below u
    const float g = fmaf(__builtin_amdgcn_logf(uf + 3.4e-10f), -kLn2 * (1.f - kRel), -2e-6f);
    if (e < least * g) return;
    float g_lo, g_hi;  // closer bounds of EPS - log(u + EPS)
    if (uf < kUNear) {
      g_lo = -kLn2 * (1.f - kRel) * __builtin_amdgcn_logf(fmaf(uf, 1.000001f, 3.4e-10f));
      g_hi = -kLn2 * (1.f + kRel) * __builtin_amdgcn_logf(fmaf(uf, 0.999999f, 1e-10f)) + 1e-10f;
    } else {
      g_lo = om > 1e-6f ? om * (1.f - kRel) : 0.f;
      g_hi = 3.5e-10f + om * (1.0012f + kRel);  // EPS and the 2^-32 that om may lie below 1 - u
    }
    if (e < least * g_lo) return;
    const int at = atomicAdd(&c_count, 1);
    if (at < kCand) {
      c_index[at] = i;
      c_most[at] = g_lo > 0.f ? e / g_lo : INFINITY;
    }
    if (i != a.mask_index) atomicMax(&c_least, __float_as_int(e / g_hi * (1.f - kRel)));
  };

  // The row's elements in the pairs that share a Philox block (2q, 2q + 1 of
  // the flattened (rows, vocab) index); a pair that hangs over an end of the
  // row leaves one element, taken alone by slice 0.
  const uint64_t first = base >> 1;
  const int off = (int)(base & 1);  // pair q holds elements 2q - off and 2q - off + 1
  const int q0 = off, q1 = (V + off) >> 1;
  const int per = (q1 - q0 + rs.slices - 1) / rs.slices;
  const int qe = min(q1, q0 + (slice + 1) * per);
  const bool wide = (reinterpret_cast<uintptr_t>(lp - off) & (2 * sizeof(T) - 1)) == 0;
  const int qm = (a.mask_index + off) >> 1, hm = (a.mask_index + off) & 1;
  if (slice == 0 && tid < 2) {
    const int i = tid == 0 ? 0 : V - 1;
    if (tid == 0 ? off == 1 : ((V + off) & 1) == 1) {
      const double u = uniform_of(a, base + i);
      element(i, i == a.mask_index ? xm : load_logit<T>(lp, i), (float)u, (float)(1.0 - u),
              bounded ? kLeastRatio : 0.f);
    }
  }
  for (int q = q0 + slice * per + tid; q < qe; q += NT) {
    const int i0 = 2 * q - off;
    float x0, x1;
    load_two<T>(lp + i0, wide, x0, x1);
    const float least = __int_as_float(__hip_atomic_load(&c_least, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    float uf[2], om[2];
    if constexpr (GIVEN) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double u = a.u[base + (uint64_t)(i0 + h)];
        uf[h] = (float)u;
        om[h] = (float)(1.0 - u);
      }
    } else {
      uint32_t c[4];
      philox_pair(a, first + (uint64_t)q, c);
      // u from its high word
      uf[0] = (float)c[1] * 0x1.0p-32f;
      uf[1] = (float)c[3] * 0x1.0p-32f;
      om[0] = (float)(~c[1]) * 0x1.0p-32f;
      om[1] = (float)(~c[3]) * 0x1.0p-32f;
    }
    if (q == qm) (hm ? x1 : x0) = xm;
    element(i0, x0, uf[0], om[0], least);
    element(i0 + 1, x1, uf[1], om[1], least);
  }
  sum = block_sum(sum, red);  // also orders the candidates before their use
  const int count = bounded ? c_count : kCand + 1;
  const float least = __int_as_float(c_least);

  if (a.spread) {
    SubsSlice* out = static_cast<SubsSlice*>(a.ws) + (int64_t)row * a.slices + slice;
    __shared__ int n_kept;
    if (tid == 0) n_kept = 0;
    __syncthreads();
    if (count <= kCand)
      for (int k = tid; k < count; k += NT)
        if (c_most[k] >= least) {
          const int at = atomicAdd(&n_kept, 1);
          if (at < kSliceCand) {
            out->index[at] = c_index[k];
            out->most[at] = c_most[k];
          }
        }
    __syncthreads();
    if (tid == 0) {
      out->m = m;
      out->sum = sum;
      out->least = least;
      out->count = count <= kCand && n_kept <= kSliceCand ? n_kept : -1;
      out->slices = rs.slices;
    }
    return;
  }
  const float lse = logf(sum);
  Best b = {-INFINITY, 0x7fffffff};
  auto consider = [&](int i) {
    const double r = exact_ratio<T>(a, lp, base, i, m, lse);
    if (better(r, i, b.v, b.i)) b = {r, i};
  };
  if (count > kCand) {
    for (int i = tid; i < V; i += NT) consider(i);
  } else {
    for (int k = tid; k < count; k += NT)
      if (c_most[k] >= least) consider(c_index[k]);
    if (tid == 0) consider(a.mask_index);
  }
  b = block_argmax<NT>(b, bval, bidx);
  if (tid == 0) a.out[row] = b.i;
}

constexpr int kFinishThreads = 256;

template <typename T>
__global__ __launch_bounds__(kFinishThreads) void subs_finish_kernel(SubsArgs a) {
  __shared__ double bval[kFinishThreads / 64];
  __shared__ int bidx[kFinishThreads / 64];
  const int tid = wi_x();
  const int row = wg_x();
  const SubsSlice* sl = static_cast<const SubsSlice*>(a.ws) + (int64_t)row * a.slices;
  // Lane s of every wave reads slice s's results (at most 64 slices; those
  // past the row's own count hold anything and are dropped).
  const int lane = tid & 63;
  const SubsSlice& mine = sl[min(lane, a.slices - 1)];
  const float s_sum = mine.sum, s_least = mine.least, m = sl->m;
  const int s_count = mine.count, slices = sl->slices;
  const int64_t xt = a.xt[row];
  if (xt != a.mask_index) {  // carry-over: an unmasked token stays
    if (tid == 0) a.out[row] = xt;
    return;
  }
  const T* lp = static_cast<const T*>(a.logits) + (int64_t)row * a.ld;
  const uint64_t base = (uint64_t)row * (uint64_t)a.vocab;
  const bool in = lane < slices;
  const float lse = logf(wave_sum(in ? s_sum : 0.f));
  const float least = wave_max(in ? s_least : 0.f);
  Best b = {-INFINITY, 0x7fffffff};
  auto consider = [&](int i) {
    const double r = exact_ratio<T>(a, lp, base, i, m, lse);
    if (better(r, i, b.v, b.i)) b = {r, i};
  };
  if (__ballot(in && s_count < 0) != 0) {
    for (int i = tid; i < a.vocab; i += kFinishThreads) consider(i);
  } else {
    // wave w takes slices w, w + 4, ...; wave 0's last lane [MASK]
    for (int s = tid >> 6; s < slices; s += kFinishThreads / 64) {
      const int n = __shfl(s_count, s, 64);
      int i = -1;
      if (lane < n && sl[s].most[lane] >= least) i = sl[s].index[lane];
      if (s == 0 && lane == 63) i = a.mask_index;
      if (i >= 0) consider(i);
    }
  }
  b = block_argmax<kFinishThreads>(b, bval, bidx);
  if (tid == 0) a.out[row] = b.i;
}

template <typename T>
hipError_t launch_subs(const SubsArgs& a, hipStream_t stream) {
  const dim3 grid(a.spread ? a.spread : a.rows);
  if (a.u != nullptr)
    hipLaunchKernelGGL((subs_scan_kernel<T, true>), grid, dim3(kSubsThreads), 0, stream, a);
  else
    hipLaunchKernelGGL((subs_scan_kernel<T, false>), grid, dim3(kSubsThreads), 0, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !a.spread) return e;
  hipLaunchKernelGGL((subs_finish_kernel<T>), dim3(a.rows), dim3(kFinishThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_subs_sample(const SubsArgs& a, hipStream_t stream) {
  if (a.rows == 0) return hipSuccess;
  return a.fp32 ? launch_subs<float>(a, stream) : launch_subs<uint16_t>(a, stream);
}

}  // namespace bd3
