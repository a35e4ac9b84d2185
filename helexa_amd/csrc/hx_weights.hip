// Weight preparation on the device: GGUF quantiser (the ISQ step), dequantiser,
// repack of GGUF rows into the kernels' planar layouts; plus the decoder-layer
// RMSNorm and residual add.
//
// Reference: quantize_parallel / quantize_blocks
// (crates/neuron/src/harness/tp/isq.rs:39-113): f32 rows, last dim tiled by the
// block size, blocks independent, each quantised by candle's from_float block
// rule (restated below); Qwen3_5RmsNorm
// (crates/neuron/src/harness/arch/qwen3_5/rmsnorm.rs:67-80).
#include "hx_internal.h"

namespace hx {

int64_t gguf_block_elems(int fmt) {
  switch (fmt) {
    case HX_F32: case HX_F16: case HX_BF16: return 1;
    case HX_Q8_0: return 32;
    case HX_Q4_K: case HX_Q6_K: return 256;
    default: return 0;
  }
}

int64_t gguf_block_bytes(int fmt) {
  switch (fmt) {
    case HX_F32: return 4;
    case HX_F16: case HX_BF16: return 2;
    case HX_Q8_0: return 34;
    case HX_Q4_K: return 144;
    case HX_Q6_K: return 210;
    default: return 0;
  }
}

HX_DEV void st_u16(uint8_t* p, uint16_t v) {
  p[0] = (uint8_t)(v & 0xff);
  p[1] = (uint8_t)(v >> 8);
}
HX_DEV uint16_t ld_u16(const uint8_t* p) { return (uint16_t)(p[0] | (p[1] << 8)); }

// ---------------------------------------------------------------- quantiser
// The block rules of candle's GgmlType::from_float, which quantize_parallel
// calls per block (isq.rs:98, 104-112; isq.rs:1-19 and 123-161 hold it
// byte-identical to candle's QTensor::quantize). candle's k_quants port of
// ggml's first k_quants.c reference quantisers, restated from the published
// algorithms: every float operation in the published order (no contraction),
// so the bytes equal the CPU restatement's.
//
// The published sums run in order over a sub-block (32 elements of a Q4_K
// superblock, 16 of a Q6_K one) and the sub-blocks are independent until the
// superblock's scale maxima, so a thread takes one sub-block, held in
// registers, and the maxima are reductions over 8 or 16 neighbouring lanes.
// Rows come in and blocks go out through LDS, so that global memory sees whole
// 16-byte accesses in address order. Q4_K and Q6_K are bound by VALU issue (the
// refit rounds: about 13 instructions an element a round). Measured for
// 64 x 512 x 2048 weights against one thread per block, which read its block
// from global memory element by element and kept the codes in scratch: Q4_K
// 2,677 -> 177 us, Q6_K 828 -> 307 us, Q8_0 209 -> 75 us (4.5 TB/s), BF16
// 137 -> 74 us.

// clampi(nearest(v), 0, hi) of the published rule, as a float: nearest is
// f32::round (half away from zero) and a saturating cast (NaN -> 0). Clamping
// first changes nothing (both bounds are whole) and leaves 0 <= c <= hi, where
// trunc(c + pred(0.5)) is roundf(c) (round_away, hx_quant.h).
HX_DEV float code_pos(float v, float hi) {
  return __builtin_truncf(__builtin_amdgcn_fmed3f(v, 0.0f, hi) + 0.49999997f);   // med3 of a NaN: the least of the others
}
// clampi(nearest(v), lo, hi) for |lo|, |hi| <= 128, as a float without -0
HX_DEV float code_sym(float v, float lo, float hi) {
  const float c = fminf(fmaxf(v == v ? v : 0.0f, lo), hi);
  return __builtin_truncf(c + __builtin_copysignf(0.49999997f, c)) + 0.0f;
}
// nearest(v) as a whole
HX_DEV int rs_nearest(float v) {
  const float r = roundf(v);
  if (r != r) return 0;
  if (r >= 2147483648.0f) return 2147483647;
  if (r < -2147483648.0f) return -2147483647 - 1;
  return (int)r;
}

// max over aligned groups of 8 lanes: quad_perm xor 1, xor 2, then the mirrored
// lane of the group (the other quad); every lane of the wave takes part
HX_DEV float max8(float v) {
  v = fmaxf(v, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0xB1, 0xf, 0xf, true)));
  v = fmaxf(v, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x4E, 0xf, 0xf, true)));
  return fmaxf(v, __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x141, 0xf, 0xf, true)));
}

// the workgroup's 256 SB floats from src (n of them valid, the rest zero) into
// LDS, sub-blocks of SB at a pitch of SB + 4 (16-byte reads and writes of
// neighbouring sub-blocks then fall on different banks); rows need not be
// 16-byte aligned
template <int SB>
HX_DEV void qz_stage_in(const float* src, int64_t n, float* in) {
  const bool al = ((uintptr_t)src & 15) == 0;
#pragma unroll
  for (int i = 0; i < SB / 4; i++) {
    const int q = 4 * ((int)threadIdx.x + 256 * i);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (q < n) {   // n is a multiple of 4
      if (al) v = *(const float4*)(src + q);
      else v = make_float4(src[q], src[q + 1], src[q + 2], src[q + 3]);
    }
    *(float4*)(in + (q / SB) * (SB + 4) + q % SB) = v;
  }
}
// n bytes from LDS (16-byte aligned) to dst (any alignment), by the workgroup
HX_DEV void qz_stage_out(const uint8_t* out, int n, uint8_t* dst) {
  if (((uintptr_t)dst & 15) == 0) {
    for (int i = 16 * (int)threadIdx.x; i + 16 <= n; i += 16 * 256) *(uint4*)(dst + i) = *(const uint4*)(out + i);
    const int i = (n & ~15) + (int)threadIdx.x;
    if (i < n) dst[i] = out[i];
  } else {
    for (int i = threadIdx.x; i < n; i += 256) dst[i] = out[i];
  }
}

// make_qkx1_quants(nmax = 15, ntry = 5, x[32]) -> (scale, -min): codes
// clamp(round((x - min) / scale), 0, nmax) alternated with the least-squares
// scale and the mean-residual min (<= 0), from min = min(0, min x) and
// scale = (max - min) / nmax, until the codes stop changing or ntry rounds.
// Codes and the sum of their squares (at most 7,200) are whole floats.
HX_DEV void make_qkx1(const float (&x)[32], float& scale_out, float& min_out) {
  float mn = x[0], mx = x[0];
#pragma unroll
  for (int i = 1; i < 32; i++) {
    const float v = x[i];
    mn = v < mn ? v : mn;
    mx = v > mx ? v : mx;
  }
  scale_out = 0.0f;
  min_out = 0.0f;
  if (mx == mn) return;
  if (mn > 0.0f) mn = 0.0f;
  float iscale = 15.0f / (mx - mn);
  float scale = 1.0f / iscale;
  float L[32];
#pragma unroll
  for (int i = 0; i < 32; i++) L[i] = 0.0f;
  for (int t = 0; t < 5; t++) {
    float sumlx = 0.0f, suml2 = 0.0f;
    bool changed = false;
#pragma unroll
    for (int i = 0; i < 32; i++) {
      const float y = x[i] - mn, l = code_pos(iscale * y, 15.0f);
      changed |= l != L[i];
      L[i] = l;
      sumlx += y * l;
      suml2 = __builtin_fmaf(l, l, suml2);
    }
    scale = sumlx / suml2;
    float sum = -0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) sum += x[i] - scale * L[i];
    mn = sum / 32.0f;
    if (mn > 0.0f) mn = 0.0f;
    iscale = 1.0f / scale;
    if (!changed) break;
  }
  scale_out = scale;
  min_out = -mn;
}

// Q4_K (BlockQ4K::from_float): make_qkx1_quants(15, 5) per 32 elements; scales
// and mins to 6 bits against their maxima; codes re-fitted with the stored
// ones. Workgroup: 32 superblocks, lane group of 8 = superblock, thread =
// sub-block.
__global__ __launch_bounds__(256) void k_quantize_q4k(const float* src, int64_t nblocks, uint8_t* dst) {
  __shared__ __attribute__((aligned(16))) float in[256 * 36];
  __shared__ __attribute__((aligned(16))) uint8_t out[32 * 144];
  const int64_t b0 = (int64_t)blockIdx.x * 32;
  const int nb = (int)(nblocks - b0 < 32 ? nblocks - b0 : 32);
  qz_stage_in<32>(src + b0 * 256, (int64_t)nb * 256, in);
  __syncthreads();
  const int j = threadIdx.x & 7;
  float x[32];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float4 v = *(const float4*)(in + threadIdx.x * 36 + 4 * i);
    x[4 * i] = v.x; x[4 * i + 1] = v.y; x[4 * i + 2] = v.z; x[4 * i + 3] = v.w;
  }
  float scale, mins;
  make_qkx1(x, scale, mins);
  const float max_scale = fmaxf(max8(scale), 0.0f), max_min = fmaxf(max8(mins), 0.0f);
  const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
  const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
  const int a = rs_nearest(inv_scale * scale), m = rs_nearest(inv_min * mins);
  const uint32_t ls = (uint8_t)(a < 63 ? a : 63), lm = (uint8_t)(m < 63 ? m : 63);
  // the partner sub-block (j ^ 4) shares this one's scale bytes: j < 4 stores
  // s[j], s[j + 4] and s[j + 8]
  const uint32_t ps = (uint32_t)__shfl_xor((int)ls, 4), pm = (uint32_t)__shfl_xor((int)lm, 4);
  const uint32_t s_lo = j < 4 ? ls : ps, s_hi = j < 4 ? ps : ls, m_lo = j < 4 ? lm : pm, m_hi = j < 4 ? pm : lm;
  const uint32_t s0 = (uint8_t)(s_lo | ((s_hi >> 4) << 6)), s1 = (uint8_t)(m_lo | ((m_hi >> 4) << 6));
  const uint32_t s2 = (s_hi & 0xF) | ((m_hi & 0xF) << 4);
  const uint32_t sc = j < 4 ? s0 & 63 : (s2 & 0xF) | ((s0 >> 6) << 4);
  const uint32_t mq = j < 4 ? s1 & 63 : (s2 >> 4) | ((s1 >> 6) << 4);
  const uint16_t dh = f32_to_f16(max_scale / 63.0f), mh = f32_to_f16(max_min / 63.0f);
  uint8_t* ob = out + (threadIdx.x >> 3) * 144;
  if (j == 0) *(uint32_t*)ob = (uint32_t)dh | ((uint32_t)mh << 16);
  if (j < 4) {
    ob[4 + j] = (uint8_t)s0;
    ob[8 + j] = (uint8_t)s1;
    ob[12 + j] = (uint8_t)s2;
  }
  const float dd = f16_to_f32(dh) * (float)(int)sc, dm = f16_to_f32(mh) * (float)(int)mq;
  uint32_t w[8];   // codes, one per byte
#pragma unroll
  for (int i = 0; i < 8; i++) {
    uint32_t v = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) v |= (uint32_t)code_pos((x[4 * i + q] + dm) / dd, 15.0f) << (8 * q);
    w[i] = dd == 0.0f ? 0u : v;
  }
  // 64-element group c = j / 2: low nibbles of the even lane's codes, high of
  // the odd lane's; the even lane writes qs words 0..3, the odd one 4..7
  const bool odd = j & 1;
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(odd ? w[i] : w[4 + i]), 0xB1, 0xf, 0xf, true);
    o[i] = odd ? got | (w[4 + i] << 4) : w[i] | (got << 4);
  }
  *(uint4*)(ob + 16 + 32 * (j >> 1) + (odd ? 16 : 0)) = make_uint4(o[0], o[1], o[2], o[3]);
  __syncthreads();
  qz_stage_out(out, nb * 144, dst + b0 * 144);
}

// make_qx_quants(n = 16, nmax = 32, x, L, rmse_type = 1), weights x^2: codes
// from the largest-|x| element, up to 3 rounds re-deriving them from the
// least-squares scale while the weighted fit improves, up to 5 rounds of
// single-code moves that improve it. Returns the scale; L holds the codes
// (whole floats in [-32, 31]); zero: every x is zero, whose stored code is 0.
HX_DEV float make_qx(const float (&x)[16], float (&L)[16], bool& zero) {
  float max = 0.0f, amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const float ax = fabsf(x[i]);
    if (ax > amax) {
      amax = ax;
      max = x[i];
    }
  }
#pragma unroll
  for (int i = 0; i < 16; i++) L[i] = 0.0f;
  zero = amax == 0.0f;
  if (zero) return 0.0f;
  const float iscale = -32.0f / max;
  float sumlx = 0.0f, suml2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const float l = code_sym(iscale * x[i], -32.0f, 31.0f), w = x[i] * x[i];
    L[i] = l;
    sumlx += w * x[i] * l;
    suml2 += w * l * l;
  }
  float scale = sumlx / suml2;
  float best = scale * sumlx;
  for (int t = 0; t < 3; t++) {
    const float is = 1.0f / scale;
    float slx = 0.0f, sl2 = 0.0f, N[16];
    bool changed = false;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float l = code_sym(is * x[i], -32.0f, 31.0f), w = x[i] * x[i];
      N[i] = l;
      changed |= l != L[i];
      slx += w * x[i] * l;
      sl2 += w * l * l;
    }
    if (!changed || sl2 == 0.0f || slx * slx <= best * sl2) break;
#pragma unroll
    for (int i = 0; i < 16; i++) L[i] = N[i];
    sumlx = slx;
    suml2 = sl2;
    scale = sumlx / suml2;
    best = scale * sumlx;
  }
  for (int t = 0; t < 5; t++) {
    bool moved = false;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const float w = x[i] * x[i], l = L[i];
      float slx = sumlx - w * x[i] * l;
      if (slx > 0.0f) {
        float sl2 = suml2 - w * l * l;
        const float nl = code_sym(x[i] * sl2 / slx, -32.0f, 31.0f);
        if (nl != l) {
          slx += w * x[i] * nl;
          sl2 += w * nl * nl;
          if (sl2 > 0.0f && slx * slx * suml2 > sumlx * sumlx * sl2) {
            L[i] = nl;
            sumlx = slx;
            suml2 = sl2;
            scale = sumlx / suml2;
            moved = true;
          }
        }
      }
    }
    if (!moved) break;
  }
  return scale;
}

// Q6_K (BlockQ6K::from_float): make_qx_quants(16, 32, rmse 1) per 16 elements;
// scales to int8 against -128 / (largest-|.| scale, the first of equals); codes
// re-fitted to [-32, 31]. Workgroup: 16 superblocks, lane group of 16 =
// superblock, thread = sub-block; the codes meet in LDS, one per byte, and are
// packed four at a time.
__global__ __launch_bounds__(256) void k_quantize_q6k(const float* src, int64_t nblocks, uint8_t* dst) {
  __shared__ __attribute__((aligned(16))) float in[256 * 20];
  __shared__ __attribute__((aligned(16))) uint8_t code[16 * 256];
  __shared__ __attribute__((aligned(16))) uint8_t out[16 * 210];
  const int64_t b0 = (int64_t)blockIdx.x * 16;
  const int nb = (int)(nblocks - b0 < 16 ? nblocks - b0 : 16);
  qz_stage_in<16>(src + b0 * 256, (int64_t)nb * 256, in);
  __syncthreads();
  const int j = threadIdx.x & 15, sb = threadIdx.x >> 4;
  float x[16], L[16];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float4 v = *(const float4*)(in + threadIdx.x * 20 + 4 * i);
    x[4 * i] = v.x; x[4 * i + 1] = v.y; x[4 * i + 2] = v.z; x[4 * i + 3] = v.w;
  }
  bool zero;
  const float sc = make_qx(x, L, zero);
  // the first scale of largest magnitude (a NaN never is): of two lane groups
  // whose maxima tie, the lower one's
  float ma = fabsf(sc) > 0.0f ? fabsf(sc) : 0.0f, max_scale = fabsf(sc) > 0.0f ? sc : 0.0f;
#pragma unroll
  for (int s = 1; s < 16; s <<= 1) {
    const float oa = __shfl_xor(ma, s), ov = __shfl_xor(max_scale, s);
    const bool take = (threadIdx.x & s) ? oa >= ma : oa > ma;
    ma = take ? oa : ma;
    max_scale = take ? ov : max_scale;
  }
  const float iscale = -128.0f / max_scale;
  const uint16_t dh = f32_to_f16(1.0f / iscale);
  const int v = rs_nearest(iscale * sc);
  const int8_t ysc = (int8_t)(uint8_t)(v < 127 ? v : 127);
  const float dj = f16_to_f32(dh) * (float)ysc;
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    w[i] = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float keep = zero ? 0.0f : L[4 * i + q] + 32.0f;
      const float l = dj == 0.0f ? keep : code_sym(x[4 * i + q] / dj, -32.0f, 31.0f) + 32.0f;
      w[i] |= (uint32_t)l << (8 * q);
    }
  }
  *(uint4*)(code + 16 * threadIdx.x) = make_uint4(w[0], w[1], w[2], w[3]);
  uint8_t* ob = out + sb * 210;
  ob[192 + j] = (uint8_t)ysc;
  if (j == 0) *(uint16_t*)(ob + 208) = dh;
  __syncthreads();
  // 48 packed words a superblock: ql words 0..31 (half n = word / 16, quarters
  // q and q + 2 of it with q = word % 16 / 8), then qh words 32..47
  for (int i = threadIdx.x; i < 16 * 48; i += 256) {
    const int s = i / 48, o = i % 48;
    const uint32_t* c = (const uint32_t*)(code + 256 * s);   // 32 words a half, 8 a quarter
    uint32_t p;
    if (o < 32) {
      const int h = 32 * (o >> 4) + (o & 15);
      p = (c[h] & 0x0F0F0F0Fu) | ((c[h + 16] & 0x0F0F0F0Fu) << 4);
    } else {
      const int h = 32 * ((o - 32) >> 3) + (o & 7);
      p = ((c[h] >> 4) & 0x03030303u) | (((c[h + 8] >> 4) & 0x03030303u) << 2) |
          (((c[h + 16] >> 4) & 0x03030303u) << 4) | (((c[h + 24] >> 4) & 0x03030303u) << 6);
    }
    uint16_t* q = (uint16_t*)(out + s * 210 + 4 * o);
    q[0] = (uint16_t)p;
    q[1] = (uint16_t)(p >> 16);
  }
  __syncthreads();
  qz_stage_out(out, nb * 210, dst + b0 * 210);
}

// Q8_0 (BlockQ8_0::from_float): d = amax / 127, q = (i8)round(x * (1 / d))
// (saturating, NaN -> 0). Bound by HBM; workgroup: 128 blocks, a block's 32
// elements in 8 lanes.
__global__ __launch_bounds__(256) void k_quantize_q8_0(const float* src, int64_t nblocks, uint8_t* dst) {
  __shared__ __attribute__((aligned(16))) uint8_t out[128 * 34];
  const int64_t b0 = (int64_t)blockIdx.x * 128;
  const int nb = (int)(nblocks - b0 < 128 ? nblocks - b0 : 128);
  const float* s = src + b0 * 32;
  const bool al = ((uintptr_t)s & 15) == 0;
  float4 v[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int q = 4 * ((int)threadIdx.x + 256 * i);
    v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (q < nb * 32) {
      if (al) v[i] = *(const float4*)(s + q);
      else v[i] = make_float4(s[q], s[q + 1], s[q + 2], s[q + 3]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const float x[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
    const float amax = max8(fmaxf(fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), fabsf(x[2])), fabsf(x[3])));
    const float d = fmaxf(amax, 0.0f) / 127.0f;   // all NaN: the published running maximum starts at 0
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) w |= ((uint32_t)(int)code_sym(x[j] * id, -128.0f, 127.0f) & 0xffu) << (8 * j);
    const int p = (int)threadIdx.x + 256 * i;
    uint16_t* o = (uint16_t*)(out + (p >> 3) * 34);
    if ((p & 7) == 0) o[0] = f32_to_f16(d);
    o[1 + 2 * (p & 7)] = (uint16_t)w;
    o[2 + 2 * (p & 7)] = (uint16_t)(w >> 16);
  }
  __syncthreads();
  qz_stage_out(out, nb * 34, dst + b0 * 34);
}

// f32 -> bf16 / f16, eight elements a thread where both sides are 16-byte
// aligned, else (and for the last n % 8) one by one
template <int FMT>
__global__ __launch_bounds__(256) void k_round_f32(const float* src, int64_t n, uint8_t* dst) {
  auto cv = [](float f) -> uint32_t { return FMT == HX_BF16 ? f32_to_bf16(f) : f32_to_f16(f); };
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i + 8 <= n && (((uintptr_t)src | (uintptr_t)dst) & 15) == 0) {
    const float4 a = *(const float4*)(src + i), b = *(const float4*)(src + i + 4);
    *(uint4*)(dst + 2 * i) = make_uint4(cv(a.x) | (cv(a.y) << 16), cv(a.z) | (cv(a.w) << 16), cv(b.x) | (cv(b.y) << 16),
                                        cv(b.z) | (cv(b.w) << 16));
  } else {
    for (int64_t k = i; k < n && k < i + 8; k++) st_u16(dst + 2 * k, (uint16_t)cv(src[k]));
  }
}

// ---------------------------------------------------------------- dequantiser
template <int FMT>
__global__ __launch_bounds__(256) void k_dequantize(const uint8_t* src, int64_t nblocks, float* dst) {
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= nblocks) return;
  if (FMT == HX_Q8_0) {
    const uint8_t* p = src + b * 34;
    float d = f16_to_f32(ld_u16(p));
    for (int j = 0; j < 32; j++) dst[b * 32 + j] = d * (float)(int8_t)p[2 + j];
  } else if (FMT == HX_Q4_K) {
    const uint8_t* p = src + b * 144;
    float d = f16_to_f32(ld_u16(p)), dmin = f16_to_f32(ld_u16(p + 2));
    const uint8_t* s = p + 4;
    for (int c = 0; c < 4; c++) {
      int sc[2], m[2];
      for (int h = 0; h < 2; h++) {
        int j = 2 * c + h;
        if (j < 4) {
          sc[h] = s[j] & 63;
          m[h] = s[j + 4] & 63;
        } else {
          sc[h] = (s[j + 4] & 0xF) | ((s[j - 4] >> 6) << 4);
          m[h] = (s[j + 4] >> 4) | ((s[j] >> 6) << 4);
        }
      }
      float d0 = d * (float)sc[0], m0 = dmin * (float)m[0], d1 = d * (float)sc[1], m1 = dmin * (float)m[1];
      for (int l = 0; l < 32; l++) {
        uint8_t q = p[16 + 32 * c + l];
        dst[b * 256 + 64 * c + l] = d0 * (float)(q & 0xF) - m0;
        dst[b * 256 + 64 * c + 32 + l] = d1 * (float)(q >> 4) - m1;
      }
    }
  } else if (FMT == HX_Q6_K) {
    const uint8_t* p = src + b * 210;
    const uint8_t* ql = p;
    const uint8_t* qh = p + 128;
    const int8_t* sc = (const int8_t*)(p + 192);
    float d = f16_to_f32(ld_u16(p + 208));
    for (int n = 0; n < 2; n++)
      for (int l = 0; l < 32; l++) {
        int is = l / 16;
        int q1 = (int)((ql[64 * n + l] & 0xF) | (((qh[32 * n + l] >> 0) & 3) << 4)) - 32;
        int q2 = (int)((ql[64 * n + l + 32] & 0xF) | (((qh[32 * n + l] >> 2) & 3) << 4)) - 32;
        int q3 = (int)((ql[64 * n + l] >> 4) | (((qh[32 * n + l] >> 4) & 3) << 4)) - 32;
        int q4 = (int)((ql[64 * n + l + 32] >> 4) | (((qh[32 * n + l] >> 6) & 3) << 4)) - 32;
        float* y = dst + b * 256 + 128 * n;
        y[l] = d * (float)sc[8 * n + is] * (float)q1;
        y[l + 32] = d * (float)sc[8 * n + is + 2] * (float)q2;
        y[l + 64] = d * (float)sc[8 * n + is + 4] * (float)q3;
        y[l + 96] = d * (float)sc[8 * n + is + 6] * (float)q4;
      }
  } else if (FMT == HX_BF16) {
    dst[b] = bf16_to_f32(ld_u16(src + 2 * b));
  } else if (FMT == HX_F16) {
    dst[b] = f16_to_f32(ld_u16(src + 2 * b));
  } else if (FMT == HX_F32) {
    dst[b] = ((const float*)src)[b];
  }
}

// ---------------------------------------------------------------- repack
// one thread per GGUF block of one [rows][K] matrix in a stack of `count`
__global__ __launch_bounds__(256) void k_repack_q8_0(const uint8_t* src, int64_t count, int64_t rows, int64_t K,
                                                     uint8_t* dst, int64_t dst_stride) {
  const int64_t nb_row = K / 32, nb_mat = rows * nb_row;
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= count * nb_mat) return;
  const int64_t m = b / nb_mat, r = (b % nb_mat) / nb_row, j = b % nb_row;
  const uint8_t* s = src + b * 34;
  uint8_t* mat = dst + m * dst_stride;
  uint8_t* qs = mat + r * K + j * 32;
  for (int i = 0; i < 32; i++) qs[i] = s[2 + i];
  uint8_t* d = mat + rows * K + (r * nb_row + j) * 2;
  d[0] = s[0];
  d[1] = s[1];
}

__global__ __launch_bounds__(256) void k_repack_q6_k(const uint8_t* src, int64_t count, int64_t rows, int64_t K,
                                                     uint8_t* dst, int64_t dst_stride) {
  const int64_t nb_row = K / 256, nb_mat = rows * nb_row;
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= count * nb_mat) return;
  const int64_t m = b / nb_mat, r = (b % nb_mat) / nb_row, j = b % nb_row;
  const uint8_t* s = src + b * 210;
  uint8_t* mat = dst + m * dst_stride;
  const int R = (int)rows, KK = (int)K, row = (int)r, o = (int)j;
  uint8_t* d = mat + rows * (K / 2 + K / 4 + K / 16) + (r * nb_row + j) * 2;
  // planes in the stored layout of q6k_at (pieces of 32, 32 and 16 bytes)
  for (int p = 0; p < 4; p++) {
    uint8_t* ql = (uint8_t*)q6k_ql(mat, R, KK, row, 128 * o + 32 * p);
    for (int i = 0; i < 32; i++) ql[i] = s[32 * p + i];
  }
  for (int p = 0; p < 2; p++) {
    uint8_t* qh = (uint8_t*)q6k_qh(mat, R, KK, row, 64 * o + 32 * p);
    for (int i = 0; i < 32; i++) qh[i] = s[128 + 32 * p + i];
  }
  uint8_t* sc = (uint8_t*)q6k_sc(mat, R, KK, row, 16 * o);
  for (int i = 0; i < 16; i++) sc[i] = s[192 + i];
  d[0] = s[208];
  d[1] = s[209];
}

// GGUF Q4_K rows -> the stored layout of q4k_sb: one thread per superblock
__global__ __launch_bounds__(256) void k_repack_q4_k(const uint8_t* src, int64_t count, int64_t rows, int64_t K,
                                                     uint8_t* dst, int64_t dst_stride) {
  const int64_t nb_row = K / 256, nb_mat = rows * nb_row;
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (b >= count * nb_mat) return;
  const int64_t m = b / nb_mat, r = (b % nb_mat) / nb_row, j = b % nb_row;
  const uint8_t* s = src + b * 144;   // the caller's rows: any alignment
  uint8_t* d = (uint8_t*)q4k_sb(dst + m * dst_stride, (int)rows, (int)K, (int)r, (int)j);
  for (int i = 0; i < 144; i++) d[i] = s[i];
}

hipError_t launch_quantize(int fmt, const float* src, int64_t rows, int64_t cols, void* dst, hipStream_t s) {
  const int64_t nb = rows * (cols / gguf_block_elems(fmt));
  auto grid = [&](int per) { return dim3((unsigned)((nb + per - 1) / per)); };   // blocks a workgroup takes
  uint8_t* d = (uint8_t*)dst;
  switch (fmt) {
    case HX_Q8_0: hipLaunchKernelGGL(k_quantize_q8_0, grid(128), dim3(256), 0, s, src, nb, d); break;
    case HX_Q4_K: hipLaunchKernelGGL(k_quantize_q4k, grid(32), dim3(256), 0, s, src, nb, d); break;
    case HX_Q6_K: hipLaunchKernelGGL(k_quantize_q6k, grid(16), dim3(256), 0, s, src, nb, d); break;
    case HX_BF16: hipLaunchKernelGGL(k_round_f32<HX_BF16>, grid(2048), dim3(256), 0, s, src, nb, d); break;
    case HX_F16: hipLaunchKernelGGL(k_round_f32<HX_F16>, grid(2048), dim3(256), 0, s, src, nb, d); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_dequantize(int fmt, const void* src, int64_t rows, int64_t cols, float* dst, hipStream_t s) {
  const int64_t nb = rows * (cols / gguf_block_elems(fmt));
  const dim3 grid((unsigned)((nb + 255) / 256));
  const uint8_t* p = (const uint8_t*)src;
  switch (fmt) {
    case HX_Q8_0: hipLaunchKernelGGL(k_dequantize<HX_Q8_0>, grid, dim3(256), 0, s, p, nb, dst); break;
    case HX_Q4_K: hipLaunchKernelGGL(k_dequantize<HX_Q4_K>, grid, dim3(256), 0, s, p, nb, dst); break;
    case HX_Q6_K: hipLaunchKernelGGL(k_dequantize<HX_Q6_K>, grid, dim3(256), 0, s, p, nb, dst); break;
    case HX_BF16: hipLaunchKernelGGL(k_dequantize<HX_BF16>, grid, dim3(256), 0, s, p, nb, dst); break;
    case HX_F16: hipLaunchKernelGGL(k_dequantize<HX_F16>, grid, dim3(256), 0, s, p, nb, dst); break;
    case HX_F32: hipLaunchKernelGGL(k_dequantize<HX_F32>, grid, dim3(256), 0, s, p, nb, dst); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_repack(int fmt, const void* src, int64_t count, int64_t rows, int64_t K, void* dst,
                         int64_t dst_stride, hipStream_t s) {
  const uint8_t* p = (const uint8_t*)src;
  uint8_t* d = (uint8_t*)dst;
  if (fmt == HX_Q8_0) {
    const int64_t nb = count * rows * (K / 32);
    hipLaunchKernelGGL(k_repack_q8_0, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, s, p, count, rows, K, d,
                       dst_stride);
  } else if (fmt == HX_Q6_K) {
    const int64_t nb = count * rows * (K / 256);
    hipLaunchKernelGGL(k_repack_q6_k, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, s, p, count, rows, K, d,
                       dst_stride);
  } else if (fmt == HX_Q4_K) {
    const int64_t nb = count * rows * (K / 256);
    hipLaunchKernelGGL(k_repack_q4_k, dim3((unsigned)((nb + 255) / 256)), dim3(256), 0, s, p, count, rows, K, d,
                       dst_stride);
  } else {
    const int64_t packed = rows * (K / gguf_block_elems(fmt)) * gguf_block_bytes(fmt);
    return hipMemcpy2DAsync(d, dst_stride, p, packed, packed, count, hipMemcpyDeviceToDevice, s);
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------- RMSNorm
// one block per token; f32 sum of squares (per-thread strided, then a fixed
// tree), y = x * rsqrt(mean + eps) * (1 + w) rounded to the activation dtype.
// Bound by latency: the token's (and the weight's) elements, NV a thread, are
// loaded together and the token's kept in registers (element by element in a
// loop, twice: 7.7 us for 27 tokens of 2048, 8.3 for 512, against 6.6 and 7).
template <int NV>
__global__ __launch_bounds__(256) void k_rmsnorm(const void* x, bool bf, int H, const float* w, float eps, void* y) {
  __shared__ float red[128];
  const int64_t t = blockIdx.x;
  const int tid = threadIdx.x;
  float v[NV], wv[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) {   // elements past the end: 0, which adds nothing
    const int i = tid + 256 * j;
    v[j] = i < H ? ld_act(x, t * H + i, bf) : 0.f;
    wv[j] = i < H ? w[i] : 0.f;
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; j++) ss = __builtin_fmaf(v[j], v[j], ss);
  // tree over 256: 128, 64 across waves, 32 .. 1 inside wave 0
  if (tid >= 128) red[tid - 128] = ss;
  __syncthreads();
  if (tid < 128) ss += red[tid];
  __syncthreads();
  if (tid >= 64 && tid < 128) red[tid - 64] = ss;
  __syncthreads();
  if (tid < 64) {
    ss += red[tid];
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) ss += __shfl_down(ss, off, 64);
    if (tid == 0) red[64] = ss;
  }
  __syncthreads();
  const float inv = 1.0f / sqrtf(red[64] / (float)H + eps);
#pragma unroll
  for (int j = 0; j < NV; j++) {
    const int i = tid + 256 * j;
    if (i >= H) break;
    const float o = v[j] * inv * (1.0f + wv[j]);
    if (bf) ((uint16_t*)y)[t * H + i] = f32_to_bf16(o);
    else ((float*)y)[t * H + i] = o;
  }
}

// any H, element by element; same arithmetic
__global__ __launch_bounds__(256) void k_rmsnorm_loop(const void* x, bool bf, int64_t H, const float* w, float eps,
                                                      void* y) {
  __shared__ float red[256];
  const int64_t t = blockIdx.x;
  float ss = 0.f;
  for (int64_t i = threadIdx.x; i < H; i += 256) {
    float v = ld_act(x, t * H + i, bf);
    ss = __builtin_fmaf(v, v, ss);
  }
  red[threadIdx.x] = ss;
  __syncthreads();
  for (int off = 128; off >= 1; off >>= 1) {
    if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
    __syncthreads();
  }
  const float inv = 1.0f / sqrtf(red[0] / (float)H + eps);
  for (int64_t i = threadIdx.x; i < H; i += 256) {
    float v = ld_act(x, t * H + i, bf) * inv * (1.0f + w[i]);
    if (bf) ((uint16_t*)y)[t * H + i] = f32_to_bf16(v);
    else ((float*)y)[t * H + i] = v;
  }
}

__global__ __launch_bounds__(256) void k_residual_add(void* x, const void* y, bool bf, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  if (bf) {
    uint16_t* px = (uint16_t*)x;
    px[i] = f32_to_bf16(bf16_to_f32(px[i]) + bf16_to_f32(((const uint16_t*)y)[i]));
  } else {
    ((float*)x)[i] += ((const float*)y)[i];
  }
}

hipError_t launch_rmsnorm(const void* x, bool xbf, int64_t T, int64_t H, const float* w, float eps, void* y,
                          hipStream_t s) {
  const dim3 g((unsigned)T);
  // as many registers as the row needs; longer rows than 4096 loop
  if (H <= 1024) hipLaunchKernelGGL(k_rmsnorm<4>, g, dim3(256), 0, s, x, xbf, (int)H, w, eps, y);
  else if (H <= 2048) hipLaunchKernelGGL(k_rmsnorm<8>, g, dim3(256), 0, s, x, xbf, (int)H, w, eps, y);
  else if (H <= 4096) hipLaunchKernelGGL(k_rmsnorm<16>, g, dim3(256), 0, s, x, xbf, (int)H, w, eps, y);
  else hipLaunchKernelGGL(k_rmsnorm_loop, g, dim3(256), 0, s, x, xbf, H, w, eps, y);
  return hipGetLastError();
}

hipError_t launch_residual_add(void* x, const void* y, bool bf, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_residual_add, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, y, bf, n);
  return hipGetLastError();
}

}  // namespace hx
