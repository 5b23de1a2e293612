// Scaled convolutions (tbf16/conv.py of the reference): a bf16 convolution runs
// as an fp16 one on inputs scaled by exact powers of two -- one exponent per
// sample for the input (a convolution mixes positions, so rows cannot be scaled
// separately) and one per output channel for the weight -- and the scales are
// undone in an epilogue that writes bf16. tbf16_conv2d runs 2-D convolutions whole
// (an implicit GEMM, gemm.hip's ksplit_kernel); for the others (1-D, 3-D, groups, small
// ones) the fp16 convolution is MIOpen's, called by the Python layer between the
// input and epilogue passes here.
//
// Memory layout: a sample is n = C * prod(spatial) elements stored back to back
// (contiguous NC... or channels-last, both keep the batch outermost), so the
// input passes run over B * n elements in memory order and find the sample as
// index / n. The passes of this file are HBM-bound streams of 16-byte vectors; the
// implicit GEMM that they feed is bound by its products.
#include <algorithm>

#include "abi_util.h"
#include "common.h"

namespace tbf16 {
int launch_conv_gemm(bool channels_last, const uint16_t* x16, const uint16_t* wp, int64_t B, int64_t O, int64_t P, int64_t K,
                     const float* w_sinv, const uint16_t* bias, const ConvShape& c, const int32_t* exps, uint16_t* y,
                     hipStream_t st);
}  // namespace tbf16

namespace {
using namespace tbf16;

constexpr int kThreads = 256;
// Elements of one sample per block of the input passes (a multiple of 8).
constexpr int64_t kChunk = 8192;

__device__ __forceinline__ uint32_t mag_max2(uint32_t w, uint32_t m) {
  return max(m, max(w & 0x7FFFu, (w >> 16) & 0x7FFFu));
}

// Largest bf16 magnitude as its bit pattern. An unsigned max of |x| bits orders
// finite values as their magnitudes, puts inf above them and every NaN pattern
// above inf, so one NaN makes the maximum NaN, as torch's max-norm does.
__device__ __forceinline__ uint32_t mag_max8(uint4 v, uint32_t m) {
  return mag_max2(v.w, mag_max2(v.z, mag_max2(v.y, mag_max2(v.x, m))));
}

// Exponent of the per-sample scale (conv.py:28-31,49-50): frexp(amax) - t, with
// all-zero and NaN samples taken as amax = 1 (torch.where(amax > 0, amax, 1)) and
// inf giving frexp's 0.
__device__ __forceinline__ int sample_exp(uint32_t m, int t) {
  if (m == 0u || m > 0x7F80u) return 1 - t;
  return frexp_exp(__uint_as_float(m << 16)) - t;
}

__device__ __forceinline__ uint32_t block_max_u32(uint32_t m) {
  __shared__ uint32_t red[kThreads / kWave];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, kWave));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  uint32_t r = red[0];
#pragma unroll
  for (int w = 1; w < kThreads / kWave; ++w) r = max(r, red[w]);
  return r;
}

// Elements [lo, hi) of x: scalar reads for the unaligned ends, 16-byte vectors
// (x is 16-byte aligned at element 0, so vectors sit at multiples of 8
// elements) with four loads in flight per lane for the rest. f(v, vec) takes
// each vector with its index, g(i) each scalar element.
template <typename FV, typename FS>
__device__ __forceinline__ void for_run(int64_t lo, int64_t hi, FV f, FS g) {
  const int64_t vlo = (lo + 7) >> 3, vhi = hi >> 3;
  if (vlo >= vhi) {
    for (int64_t i = lo + threadIdx.x; i < hi; i += kThreads) g(i);
    return;
  }
  for (int64_t i = lo + threadIdx.x; i < vlo * 8; i += kThreads) g(i);
  for (int64_t i = vhi * 8 + threadIdx.x; i < hi; i += kThreads) g(i);
  int64_t v = vlo + threadIdx.x;
  for (; v + 3 * kThreads < vhi; v += 4 * kThreads) f(v, 4);
  for (; v < vhi; v += kThreads) f(v, 1);
}

// Block b * nch + c reduces elements [c * kChunk, (c + 1) * kChunk) of sample b
// into partial[b * nch + c].
__device__ __forceinline__ void sample_amax_block(const uint16_t* __restrict__ x, int64_t n, int nch,
                                                  uint32_t* __restrict__ partial) {
  const int64_t b = blockIdx.x / nch;
  const int64_t c = blockIdx.x - b * nch;
  const int64_t lo = b * n + c * kChunk;
  const int64_t hi = std::min(b * n + n, lo + kChunk);
  const uint4* xv = reinterpret_cast<const uint4*>(x);
  uint32_t m = 0u;
  for_run(
      lo, hi,
      [&](int64_t v, int cnt) {
        if (cnt == 4) {
          const uint4 a0 = xv[v], a1 = xv[v + kThreads], a2 = xv[v + 2 * kThreads], a3 = xv[v + 3 * kThreads];
          m = mag_max8(a3, mag_max8(a2, mag_max8(a1, mag_max8(a0, m))));
        } else {
          m = mag_max8(xv[v], m);
        }
      },
      [&](int64_t i) { m = max(m, x[i] & 0x7FFFu); });
  m = block_max_u32(m);
  if (threadIdx.x == 0) partial[blockIdx.x] = m;
}

__global__ __launch_bounds__(kThreads) void sample_amax_kernel(const uint16_t* __restrict__ x, int64_t n, int nch,
                                                               uint32_t* __restrict__ partial) {
  sample_amax_block(x, n, nch, partial);
}

// ---- implicit convolution: its two operands -------------------------------------------
// MIOpen's fp16 convolution of 512 channels at 128 x 128 wrote the input out nine times
// (57 us) for a GEMM of 72 us, between a cast pass (7 us), an epilogue (6 us) and a copy
// of the bias. Here the cast pass writes the input once, channels last with its zero
// padding and channels padded to 64, and the GEMM reads each tap straight from it: 151 ->
// 86 us a call (contiguous), 175 -> 88 (channels last).
// The first launch also takes the samples' maxima and lays the weight out as
// [channel][tap][Cp] (its (O, C, KH, KW) rows have the taps innermost).
__global__ __launch_bounds__(kThreads) void conv_scan_kernel(const uint16_t* __restrict__ x, int64_t n, int nch,
                                                             uint32_t* __restrict__ partial, unsigned amax_blocks,
                                                             const uint16_t* __restrict__ w, int64_t O, int C, int T,
                                                             int Cp, uint16_t* __restrict__ wp) {
  if (blockIdx.x < amax_blocks) {
    sample_amax_block(x, n, nch, partial);
    return;
  }
  // one thread per 8 channels of one tap, taps varying fastest: a wave's reads of one
  // channel cover neighbouring taps and channels
  const int64_t i = (int64_t)(blockIdx.x - amax_blocks) * kThreads + threadIdx.x;
  const int c8 = Cp >> 3;
  if (i >= O * c8 * T) return;
  const int tap = (int)(i % T), c = (int)(i / T % c8) * 8;
  const int64_t o = i / T / c8;
  uint16_t v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = c + e < C ? w[(o * C + c + e) * T + tap] : (uint16_t)0;
  __builtin_memcpy(wp + (o * T + tap) * Cp + c, v, 16);
}

// Block (64 padded columns, padded row, image x 64-channel chunk): x16 = fp16(x 2^-e) of its
// pixels and channels, zeros in the padding. CL: x is channels last (C % 8 == 0); else its
// 64 x 64 (channel, pixel) square is turned over in LDS.
template <bool CL>
__global__ __launch_bounds__(kThreads) void conv_pack_kernel(const uint16_t* __restrict__ x, int C, int H, int W, int ph,
                                                             int pw, int Hp, int Wp, int Cp, int nch,
                                                             const uint32_t* __restrict__ partial, int t,
                                                             int32_t* __restrict__ exps, uint16_t* __restrict__ y) {
  __shared__ __align__(16) uint16_t tile[CL ? 1 : 64][72];  // [pixel][channel], padded against bank conflicts
  const int chunks = Cp >> 6;
  const int64_t b = blockIdx.z / chunks;
  const int c0 = (int)(blockIdx.z % chunks) * 64, w0 = (int)blockIdx.x * 64, hp = (int)blockIdx.y;
  const int h = hp - ph;
  const bool row_in = h >= 0 && h < H;
  uint16_t* const yrow = y + ((b * Hp + hp) * Wp) * (int64_t)Cp + c0;
  // the raw values first: they are in flight while the sample's exponent is derived
  uint4 vec[2];       // CL: pixel i / 8, channels 8 (i % 8) .. + 7 for i = thread + 256 j
  uint32_t pair[8];   // else pixels 2 (thread % 32), + 1 of channel thread / 32 + 8 j
  if constexpr (CL) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = threadIdx.x + j * kThreads, w = w0 + (i >> 3) - pw, c = (i & 7) * 8;
      vec[j] = make_uint4(0, 0, 0, 0);
      if (row_in && w >= 0 && w < W && c0 + c < C) vec[j] = ldg16(x + ((b * H + h) * (int64_t)W + w) * C + c0 + c);
    }
  } else {
    const int w = w0 + 2 * (threadIdx.x & 31) - pw;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = c0 + (threadIdx.x >> 5) + 8 * j;
      pair[j] = 0u;
      if (row_in && c < C) {
        const uint16_t* const src = x + ((b * C + c) * (int64_t)H + h) * W + w;
        if (w >= 0 && w + 1 < W) __builtin_memcpy(&pair[j], src, 4);
        else if (w >= 0 && w < W) pair[j] = src[0];
        else if (w + 1 >= 0 && w + 1 < W) pair[j] = (uint32_t)src[1] << 16;
      }
    }
  }
  uint32_t m = 0u;
  for (int i = threadIdx.x; i < nch; i += kThreads) m = max(m, partial[b * nch + i]);
  const int e = sample_exp(block_max_u32(m), t);
  if (blockIdx.x == 0 && blockIdx.y == 0 && c0 == 0 && threadIdx.x == 0) exps[b] = e;
  const float s = ldexp1(-e);
  if constexpr (CL) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = threadIdx.x + j * kThreads, px = w0 + (i >> 3);
      if (px < Wp) stg16(yrow + (int64_t)px * Cp + (i & 7) * 8, cvt_bf16x8_f16x8(vec[j], s));
    }
  } else {
    const int px = 2 * (threadIdx.x & 31);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int c = (threadIdx.x >> 5) + 8 * j;
      const uint32_t v = cvt_bf16x2_f16x2(pair[j], s);
      tile[px][c] = (uint16_t)v;
      tile[px + 1][c] = (uint16_t)(v >> 16);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int i = threadIdx.x + j * kThreads, p = i >> 3, c = (i & 7) * 8;
      if (w0 + p < Wp) stg16(yrow + (int64_t)(w0 + p) * Cp + c, *reinterpret_cast<const uint4*>(&tile[p][c]));
    }
  }
}

// Block b * nch + c: the exponent of sample b from its nch partial maxima, then
// x16 = fp16(x * 2^-e) for the same elements the max pass block covered
// (conv.py:51-54: torch.mul of bf16 by the fp32 scale ldexp(1, -e), written to
// fp16: one RNE rounding of the fp32 product). The scale is ldexp(1, -e) in
// fp32, so -e >= 128 gives inf exactly as the reference does.
__global__ __launch_bounds__(kThreads) void sample_cast_kernel(const uint16_t* __restrict__ x, int64_t n, int nch,
                                                               const uint32_t* __restrict__ partial, int t,
                                                               int32_t* __restrict__ exps,
                                                               uint16_t* __restrict__ y) {
  const int64_t b = blockIdx.x / nch;
  const int64_t c = blockIdx.x - b * nch;
  uint32_t m = 0u;
  for (int i = threadIdx.x; i < nch; i += kThreads) m = max(m, partial[b * nch + i]);
  const int e = sample_exp(block_max_u32(m), t);
  if (c == 0 && threadIdx.x == 0) exps[b] = e;
  const float s = ldexp1(-e);
  const int64_t lo = b * n + c * kChunk;
  const int64_t hi = std::min(b * n + n, lo + kChunk);
  const uint4* xv = reinterpret_cast<const uint4*>(x);
  uint4* yv = reinterpret_cast<uint4*>(y);
  for_run(
      lo, hi,
      [&](int64_t v, int cnt) {
        if (cnt == 4) {
          const uint4 a0 = xv[v], a1 = xv[v + kThreads], a2 = xv[v + 2 * kThreads], a3 = xv[v + 3 * kThreads];
          yv[v] = cvt_bf16x8_f16x8(a0, s);
          yv[v + kThreads] = cvt_bf16x8_f16x8(a1, s);
          yv[v + 2 * kThreads] = cvt_bf16x8_f16x8(a2, s);
          yv[v + 3 * kThreads] = cvt_bf16x8_f16x8(a3, s);
        } else {
          yv[v] = cvt_bf16x8_f16x8(xv[v], s);
        }
      },
      [&](int64_t i) { y[i] = __builtin_bit_cast(uint16_t, (_Float16)(__uint_as_float((uint32_t)x[i] << 16) * s)); });
}

// out = bf16(y * (2^exps[b] * ws[o]) [+ bias[o]]) in fp32 (conv.py:56-60): the
// scale is the fp32 product of the two powers of two, y * scale is exact unless
// it leaves fp32's normal range, the bias add rounds once to fp32 and the result
// once more to bf16, as torch's mul / addcmul into a bf16 tensor do.
// CL = 0: (B, O, P) layout, CL = 1: (B, P, O).
template <bool BIAS>
__device__ __forceinline__ float epi_elem(float v, float sc, float bias) {
  return BIAS ? fmaf(v, sc, bias) : v * sc;
}

// ALIGNED: every 16-byte vector lies in one (b, o) row (CL = 0, P % 8 == 0) or
// covers 8 channels of one pixel starting at a multiple of 8 (CL = 1, O % 8 == 0,
// ws and bias 16-byte aligned), so the scales are found once per vector.
template <bool CL, bool BIAS, bool ALIGNED>
__global__ __launch_bounds__(kThreads) void conv_epilogue_kernel(const uint16_t* __restrict__ y, int64_t O, int64_t P,
                                                                 int64_t total, const int32_t* __restrict__ exps,
                                                                 const float* __restrict__ ws,
                                                                 const float* __restrict__ bias,
                                                                 uint16_t* __restrict__ out) {
  const int64_t nv = total >> 3;
  for (int64_t v = (int64_t)blockIdx.x * kThreads + threadIdx.x; v < nv; v += (int64_t)gridDim.x * kThreads) {
    const int64_t i0 = v * 8;
    const uint4 in = reinterpret_cast<const uint4*>(y)[v];
    const uint32_t w[4] = {in.x, in.y, in.z, in.w};
    float r[8];
    if constexpr (ALIGNED && !CL) {
      const int64_t row = i0 / P, b = row / O, o = row - b * O;
      const float sc = ldexp1(exps[b]) * ws[o], bs = BIAS ? bias[o] : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) r[k] = epi_elem<BIAS>((k & 1) ? f16_hi(w[k >> 1]) : f16_lo(w[k >> 1]), sc, bs);
    } else if constexpr (ALIGNED) {
      const int64_t q = i0 / O, o = i0 - q * O, b = q / P;
      const float eb = ldexp1(exps[b]);
      const float4 w0 = *reinterpret_cast<const float4*>(ws + o), w1 = *reinterpret_cast<const float4*>(ws + o + 4);
      float4 b0 = make_float4(0.f, 0.f, 0.f, 0.f), b1 = b0;
      if constexpr (BIAS) {
        b0 = *reinterpret_cast<const float4*>(bias + o);
        b1 = *reinterpret_cast<const float4*>(bias + o + 4);
      }
      const float wk[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
      const float bk[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
#pragma unroll
      for (int k = 0; k < 8; ++k)
        r[k] = epi_elem<BIAS>((k & 1) ? f16_hi(w[k >> 1]) : f16_lo(w[k >> 1]), eb * wk[k], bk[k]);
    } else if constexpr (!CL) {
      // elements run along P within one (b, o) row; a row change is rare
      int64_t row = i0 / P, p = i0 - row * P;
      int64_t b = row / O, o = row - b * O;
      float sc = ldexp1(exps[b]) * ws[o], bs = BIAS ? bias[o] : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        r[k] = epi_elem<BIAS>((k & 1) ? f16_hi(w[k >> 1]) : f16_lo(w[k >> 1]), sc, bs);
        if (k < 7 && ++p == P) {
          p = 0;
          if (++o == O) o = 0, ++b;
          sc = ldexp1(exps[b]) * ws[o];
          if (BIAS) bs = bias[o];
        }
      }
    } else {
      // elements run along O within one pixel
      const int64_t q = i0 / O;
      int64_t o = i0 - q * O;
      int64_t b = q / P, pix = q - b * P;
      float eb = ldexp1(exps[b]);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        r[k] = epi_elem<BIAS>((k & 1) ? f16_hi(w[k >> 1]) : f16_lo(w[k >> 1]), eb * ws[o], BIAS ? bias[o] : 0.f);
        if (k < 7 && ++o == O) {
          o = 0;
          if (++pix == P) pix = 0, ++b, eb = ldexp1(exps[b]);
        }
      }
    }
    reinterpret_cast<uint4*>(out)[v] =
        make_uint4(pack_bf16(r[0], r[1]), pack_bf16(r[2], r[3]), pack_bf16(r[4], r[5]), pack_bf16(r[6], r[7]));
  }
  if (blockIdx.x == 0) {
    for (int64_t i = nv * 8 + threadIdx.x; i < total; i += kThreads) {
      int64_t b, o;
      if constexpr (!CL) {
        const int64_t row = i / P;
        b = row / O;
        o = row - b * O;
      } else {
        o = i % O;
        b = i / O / P;
      }
      const float val = (float)__builtin_bit_cast(_Float16, y[i]);
      const float rr = epi_elem<BIAS>(val, ldexp1(exps[b]) * ws[o], BIAS ? bias[o] : 0.f);
      out[i] = __builtin_bit_cast(uint16_t, (__bf16)rr);
    }
  }
}

int64_t amax_chunks(int64_t n) { return std::max<int64_t>(1, cdiv(n, kChunk)); }

unsigned stream_blocks(int64_t nv) { return (unsigned)std::max<int64_t>(1, std::min<int64_t>(cdiv(nv, kThreads), 4096)); }

}  // namespace

extern "C" size_t tbf16_conv_input_ws_bytes(int64_t B, int64_t n) {
  if (B <= 0 || n <= 0) return 0;
  return align_up((size_t)(B * amax_chunks(n)) * sizeof(uint32_t), 256);
}

extern "C" int tbf16_conv_input(const void* x, int64_t B, int64_t n, int t, int32_t* exps, void* x16, void* ws,
                                int64_t ws_bytes, void* stream) {
  TB_CHECK(B >= 0 && n >= 0, "conv_input: negative size");
  if (B == 0) return 0;
  TB_CHECK(x && exps && x16, "conv_input: null pointer");
  TB_CHECK(aligned16(x) && aligned16(x16), "conv_input: x and x16 must be 16-byte aligned");
  TB_CHECK(n > 0, "conv_input: empty samples are handled by the caller");
  const int64_t nch = amax_chunks(n);
  TB_CHECK(B * nch <= 0x7FFFFFFF, "conv_input: tensor too large");
  TB_CHECK(ws && ws_bytes >= (int64_t)tbf16_conv_input_ws_bytes(B, n), "conv_input: workspace too small");
  hipStream_t st = as_stream(stream);
  sample_amax_kernel<<<(unsigned)(B * nch), kThreads, 0, st>>>((const uint16_t*)x, n, (int)nch, (uint32_t*)ws);
  TB_LAUNCH_CHECK("conv_input (max)");
  sample_cast_kernel<<<(unsigned)(B * nch), kThreads, 0, st>>>((const uint16_t*)x, n, (int)nch, (const uint32_t*)ws,
                                                               t, exps, (uint16_t*)x16);
  TB_LAUNCH_CHECK("conv_input (cast)");
  return 0;
}

extern "C" int tbf16_conv_epilogue(const void* y16, int64_t B, int64_t O, int64_t P, int channels_last,
                                   const int32_t* exps, const float* ws, const float* bias, void* out, void* stream) {
  TB_CHECK(B >= 0 && O >= 0 && P >= 0, "conv_epilogue: negative size");
  const int64_t total = B * O * P;
  if (total == 0) return 0;
  TB_CHECK(y16 && exps && ws && out, "conv_epilogue: null pointer");
  TB_CHECK(aligned16(y16) && aligned16(out), "conv_epilogue: y16 and out must be 16-byte aligned");
  hipStream_t st = as_stream(stream);
  const unsigned blocks = stream_blocks(total >> 3);
  const bool aligned = channels_last ? (O % 8 == 0 && aligned16(ws) && (!bias || aligned16(bias))) : P % 8 == 0;
#define LAUNCH(CL, BI, AL)                                                                                    \
  conv_epilogue_kernel<CL, BI, AL><<<blocks, kThreads, 0, st>>>((const uint16_t*)y16, O, P, total, exps, ws, bias, \
                                                                (uint16_t*)out)
#define LAUNCH2(CL, BI) \
  if (aligned) LAUNCH(CL, BI, true); else LAUNCH(CL, BI, false)
  if (channels_last) {
    if (bias) { LAUNCH2(true, true); } else { LAUNCH2(true, false); }
  } else {
    if (bias) { LAUNCH2(false, true); } else { LAUNCH2(false, false); }
  }
#undef LAUNCH2
#undef LAUNCH
  TB_LAUNCH_CHECK("conv_epilogue");
  return 0;
}

namespace {
struct Conv2dPlan {
  ConvShape c;
  int64_t B, O, P, K, nch;
  size_t exps, wp, x16, total;
};
// 0, or an error with its reason set: sizes the kernels' 32-bit offsets do not reach
int conv2d_plan(int64_t B, int64_t C, int64_t H, int64_t W, int64_t O, int64_t KH, int64_t KW, const int64_t* stride,
                const int64_t* pad, const int64_t* dilation, Conv2dPlan& p) {
  TB_CHECK(B > 0 && C > 0 && H > 0 && W > 0 && O > 0 && KH > 0 && KW > 0, "conv2d: empty");
  TB_CHECK(stride && pad && dilation && stride[0] > 0 && stride[1] > 0 && pad[0] >= 0 && pad[1] >= 0 && dilation[0] > 0 &&
               dilation[1] > 0,
           "conv2d: bad stride, padding or dilation");
  ConvShape& c = p.c;
  c.Hp = H + 2 * pad[0];
  c.Wp = W + 2 * pad[1];
  c.Cp = cdiv(C, 64) * 64;
  c.KH = KH; c.KW = KW;
  c.sh = stride[0]; c.sw = stride[1];
  c.dh = dilation[0]; c.dw = dilation[1];
  const int64_t eh = (KH - 1) * c.dh + 1, ew = (KW - 1) * c.dw + 1;
  TB_CHECK(c.Hp >= eh && c.Wp >= ew, "conv2d: the kernel is larger than the padded input");
  const int64_t Ho = (c.Hp - eh) / c.sh + 1;
  c.Wo = (c.Wp - ew) / c.sw + 1;
  p.B = B; p.O = O;
  p.P = Ho * c.Wo;
  p.K = KH * KW * c.Cp;
  p.nch = amax_chunks(C * H * W);
  TB_CHECK(c.Hp * c.Wp * c.Cp < (int64_t)1 << 30 && p.K < (int64_t)1 << 22 && O < (int64_t)1 << 31 && B < 65536 &&
               c.Hp < 65536 && B * (c.Cp / 64) < 65536 && B * p.nch < (int64_t)1 << 30 && O * p.K < (int64_t)1 << 33,
           "conv2d: tensor too large");
  p.exps = align_up((size_t)(B * p.nch) * 4, 256);
  p.wp = p.exps + align_up((size_t)B * 4, 256);
  p.x16 = p.wp + align_up((size_t)O * (size_t)p.K * 2, 256);
  p.total = p.x16 + align_up((size_t)B * (size_t)(c.Hp * c.Wp * c.Cp) * 2, 256);
  return 0;
}
}  // namespace

extern "C" size_t tbf16_conv2d_ws_bytes(int64_t B, int64_t C, int64_t H, int64_t W, int64_t O, int64_t KH, int64_t KW,
                                        const int64_t* stride, const int64_t* pad, const int64_t* dilation) {
  Conv2dPlan p;
  return conv2d_plan(B, C, H, W, O, KH, KW, stride, pad, dilation, p) ? 0 : p.total;
}

extern "C" int tbf16_conv2d(const void* x, int64_t B, int64_t C, int64_t H, int64_t W, int channels_last, int t,
                            const void* w16, int64_t O, int64_t Cw, int64_t KH, int64_t KW, const int64_t* stride,
                            const int64_t* pad, const int64_t* dilation, const float* w_sinv, const void* bias, void* y,
                            void* ws, int64_t ws_bytes, void* stream) {
  TB_CHECK(Cw == C, "conv2d: the input has %lld channels, the weight %lld", (long long)C, (long long)Cw);
  Conv2dPlan p;
  if (int rc = conv2d_plan(B, C, H, W, O, KH, KW, stride, pad, dilation, p)) return rc;
  TB_CHECK(x && w16 && w_sinv && y && aligned16(x) && aligned16(y), "conv2d: null or misaligned pointer");
  TB_CHECK(!channels_last || C % 8 == 0, "conv2d: channels-last input needs channels in multiples of 8");
  TB_CHECK(ws && aligned16(ws) && ws_bytes >= (int64_t)p.total, "conv2d: workspace too small");
  hipStream_t st = as_stream(stream);
  uint8_t* const base = static_cast<uint8_t*>(ws);
  uint32_t* const partial = reinterpret_cast<uint32_t*>(base);
  int32_t* const exps = reinterpret_cast<int32_t*>(base + p.exps);
  uint16_t* const wp = reinterpret_cast<uint16_t*>(base + p.wp);
  uint16_t* const x16 = reinterpret_cast<uint16_t*>(base + p.x16);
  const ConvShape& c = p.c;
  const unsigned amax_blocks = (unsigned)(B * p.nch);
  const int64_t wblocks = cdiv(O * (c.Cp / 8) * KH * KW, kThreads);
  conv_scan_kernel<<<(unsigned)(amax_blocks + wblocks), kThreads, 0, st>>>((const uint16_t*)x, C * H * W, (int)p.nch, partial,
                                                                            amax_blocks, (const uint16_t*)w16, O, (int)C,
                                                                            (int)(KH * KW), (int)c.Cp, wp);
  TB_LAUNCH_CHECK("conv2d/scan");
  const dim3 grid((unsigned)cdiv(c.Wp, 64), (unsigned)c.Hp, (unsigned)(B * (c.Cp / 64)));
#define PACK(CL)                                                                                                       \
  conv_pack_kernel<CL><<<grid, kThreads, 0, st>>>((const uint16_t*)x, (int)C, (int)H, (int)W, (int)pad[0], (int)pad[1], \
                                                  (int)c.Hp, (int)c.Wp, (int)c.Cp, (int)p.nch, partial, t, exps, x16)
  if (channels_last) PACK(true);
  else PACK(false);
#undef PACK
  TB_LAUNCH_CHECK("conv2d/pack");
  return launch_conv_gemm(channels_last != 0, x16, wp, B, O, p.P, p.K, w_sinv, (const uint16_t*)bias, c, exps,
                          (uint16_t*)y, st);
}
