// Expert kernels: SwiGLU gate/up GEMV, down GEMV with the weighted combine
// (every shape outside the fast decode and prefill MFMA kernels). For GGUF
// weights the expert calls of m <= 64 rows read the f32 d q of the Q8 codes
// of their tokens (k_xq_f32) and of their rows of h (k_hq_f32, in place),
// the reference's quantised arm up to f32 rounding; larger calls compute
// exactly in f32 (the reference's f16 arm within f16 operand rounding).
//
// Reference: Qwen3_5MLP::forward (crates/neuron/src/harness/arch/qwen3_5/mlp.rs:54-60),
// the scatter loop of Module::forward (moe.rs:177-195: experts ascending,
// then the sigmoid-gated shared expert) and the fused path's weighted down
// GEMM + sum over k (crates/neuron/src/harness/tp/tp_qwen3_5.rs:1192-1225).
//
// Work is described by the slot list the dispatch wrote: slot u = (expert e,
// start position in the permuted order, token count); the shared expert is
// the last slot with e == E, start F and all T tokens. SwiGLU activations of
// slot u's j-th token live in row start+j of hbuf (shared: row F+t).
#include "hx_internal.h"

namespace hx {

// load n (multiple of 8, 8-aligned offset) activations as f32
HX_DEV void load_run(const void* base, bool bf, int64_t off, float* out, int n) {
  if (bf) {
    const uint4* p = (const uint4*)((const uint16_t*)base + off);
    for (int v = 0; v < n / 8; v++) {
      uint4 q = p[v];
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        out[8 * v + 2 * j] = __uint_as_float(w[j] << 16);
        out[8 * v + 2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
      }
    }
  } else {
    const float4* p = (const float4*)((const float*)base + off);
    for (int v = 0; v < n / 4; v++) {
      float4 q = p[v];
      out[4 * v] = q.x; out[4 * v + 1] = q.y; out[4 * v + 2] = q.z; out[4 * v + 3] = q.w;
    }
  }
}

// the CH activations of chunk c of a row, in chunk order
template <int FMT>
HX_DEV void load_chunk_x(const void* row, bool bf, int c, float* xv) {
  using CK = Chunk<FMT>;
#pragma unroll
  for (int r = 0; r < CK::CH / CK::RUN; r++) load_run(row, bf, CK::pos(c, r * CK::RUN), xv + r * CK::RUN, CK::RUN);
}

// ----------------------------------------------------------------------------
// gate/up + SwiGLU. grid = (row blocks, slots). Each wave owns NRG row groups of
// RG = 64 / LPR rows; lane ll of a row group owns chunks ll + LPR * ci.
// ----------------------------------------------------------------------------
template <int FMT, int LPR, int CPL, int NTOK, int NRG>
__global__ __launch_bounds__(256) void k_gate_up(ExpertArgs a) {
  using CK = Chunk<FMT>;
  constexpr int CH = CK::CH, RG = 64 / LPR, NS = CK::NSUM > 0 ? CK::NSUM : 1;
  // the slot's first tokens' entries are read together with the weights: one round
  // trip less
  const int u = blockIdx.y;
  const int e = a.slots[3 * u], start = a.slots[3 * u + 1], count = a.slots[3 * u + 2];
  if (u >= a.counts[0]) return;
  const bool sh = e == a.E;
  const uint8_t* G = sh ? a.sgate.base : a.gate.mat(e);
  const uint8_t* U = sh ? a.sup.base : a.up.mat(e);
  const int rows = sh ? a.Is : a.I;
  const int K = a.H, nch = K / CH;
  const int lane = lane_id(), wave = threadIdx.x >> 6, rg = lane / LPR, ll = lane % LPR;
  const int row_base = (blockIdx.x * 4 + wave) * (RG * NRG);
  if (row_base >= rows) return;
  // GGUF weights, a call of m <= HX_QUANT_M rows: the reference quantises the
  // tokens to the vec_dot type (MaybeQuantLinear, tp_linear.rs:120-137); they
  // come as the f32 d q of their codes (k_xq_f32)
  const bool qa = a.xq32 && count <= HX_QUANT_M;

  // the entries of the first tokens (scalar loads), then the weights: every load
  // of the wave is in flight before any math
  int ent[NTOK];
#pragma unroll
  for (int tok = 0; tok < NTOK; tok++) ent[tok] = sh ? min(tok, count - 1) : a.perm[start + min(tok, count - 1)];
  typename CK::Raw rgt[NRG][CPL], rup[NRG][CPL];
#pragma unroll
  for (int g = 0; g < NRG; g++) {
    const int row = row_base + g * RG + rg;
#pragma unroll
    for (int ci = 0; ci < CPL; ci++) {
      const int c = ll + LPR * ci;
      if (row < rows && c < nch) {
        CK::load(G, rows, K, row, c, rgt[g][ci]);
        CK::load(U, rows, K, row, c, rup[g][ci]);
      }
    }
  }
  for (int tg = 0; tg < count; tg += NTOK) {
    float xv[NTOK][CPL][CH], xs[NTOK][CPL][NS];
    int hrow[NTOK];
#pragma unroll
    for (int tok = 0; tok < NTOK; tok++) {
      const int j = tg + tok < count ? tg + tok : count - 1;
      const int t = sh ? j : (tg == 0 ? ent[tok] : a.perm[start + j]) / a.k;
      hrow[tok] = sh ? a.F + j : start + j;
      const bool xb = a.xbf && !qa;
      const void* xr = qa ? (const void*)(a.xq32 + (int64_t)t * K)
                          : xb ? (const void*)((const uint16_t*)a.x + (int64_t)t * K)
                               : (const void*)((const float*)a.x + (int64_t)t * K);
#pragma unroll
      for (int ci = 0; ci < CPL; ci++) {
        const int c = ll + LPR * ci;
        if (c < nch) {
          load_chunk_x<FMT>(xr, xb, c, xv[tok][ci]);
          CK::sums(xv[tok][ci], xs[tok][ci]);
        }
      }
    }
#pragma unroll
    for (int g = 0; g < NRG; g++) {
      const int row = row_base + g * RG + rg;
#pragma unroll
      for (int tok = 0; tok < NTOK; tok++) {
        float pg = 0.f, pu = 0.f;
#pragma unroll
        for (int ci = 0; ci < CPL; ci++) {
          const int c = ll + LPR * ci;
          if (row < rows && c < nch) {
            pg += CK::dot(rgt[g][ci], xv[tok][ci], xs[tok][ci]);
            pu += CK::dot(rup[g][ci], xv[tok][ci], xs[tok][ci]);
          }
        }
        pg = wave_sum<LPR>(pg);
        pu = wave_sum<LPR>(pu);
        if (ll == 0 && row < rows && tg + tok < count) {
          float h = siluf_(pg) * pu;
          a.hbuf[(int64_t)hrow[tok] * a.hstride + row] = h;
          if (a.hbf) a.hbf[(int64_t)hrow[tok] * a.hstride + row] = f32_to_bf16(h);
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------
// decode down projection + combine. Block = RG output rows (one wave-row-group);
// its 4 waves split the rows of h in dispatch order (the routed rows by expert,
// then the shared expert's), whose token, weight and expert come from the decode
// plan; contrib[hr][r] collects weight * (down_e row . h) in LDS and each token's
// output sums its rows in that order (experts ascending, then the shared
// expert), as moe.rs:178-194 does. Bound by latency at the sizes that come here:
// plan, then weights and rows of h together (by slot list, permutation and
// routing weights in turn, the rows of h behind the weights: 8.0 us for 4 tokens
// of the 256-wide f32 block, 7.4 so; 54 -> 47 us a forward of 2 bf16 tokens).
// ----------------------------------------------------------------------------
template <int FMT, int LPR, int CPL, int SPW>
__global__ __launch_bounds__(256) void k_down_combine(ExpertArgs a) {
  using CK = Chunk<FMT>;
  constexpr int CH = CK::CH, RG = 64 / LPR, NS = CK::NSUM > 0 ? CK::NSUM : 1;
  constexpr bool HPRE = CPL * CH <= 16;   // rows of h short enough to be held beside the weights
  extern __shared__ float contrib[];
  const int T = a.T, NH = a.F + T, nr = a.F + (a.Is > 0 ? T : 0);   // plan stride; rows of h in use
  int* stok = (int*)(contrib + nr * RG);
  const int32_t* plan = a.plan + 4 + 4 * a.max_slots;   // tokens, weights, experts of the rows
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int rg = lane / LPR, ll = lane % LPR;
  const int n0 = blockIdx.x * RG, row = n0 + rg;
  for (int i = threadIdx.x; i < nr; i += 256) stok[i] = plan[i];
  for (int hb = wave; hb < nr; hb += 4 * SPW) {
    typename CK::Raw raw[SPW][CPL];
    float wgt[SPW], hv[SPW][HPRE ? CPL * CH : 1];
    int Ks[SPW];
#pragma unroll
    for (int s = 0; s < SPW; s++) {
      const int hr = min(hb + 4 * s, nr - 1), e = plan[2 * NH + hr];
      const bool sh = e == a.E;
      wgt[s] = __int_as_float(plan[NH + hr]);
      Ks[s] = sh ? a.Is : a.I;
      const uint8_t* W = sh ? a.sdown.base : a.down.mat(e);
#pragma unroll
      for (int ci = 0; ci < CPL; ci++) {
        const int c = ll + LPR * ci;
        if (hb + 4 * s < nr && row < a.H && c < Ks[s] / CH) {
          CK::load(W, a.H, Ks[s], row, c, raw[s][ci]);
          if constexpr (HPRE) load_chunk_x<FMT>(a.hbuf + (int64_t)hr * a.hstride, false, c, hv[s] + CH * ci);
        }
      }
    }
#pragma unroll
    for (int s = 0; s < SPW; s++) {
      const int hr = hb + 4 * s;
      if (hr >= nr) break;
      float p = 0.f;
#pragma unroll
      for (int ci = 0; ci < CPL; ci++) {
        const int c = ll + LPR * ci;
        if (row < a.H && c < Ks[s] / CH) {
          float xv[CH], xs[NS];
          if constexpr (HPRE) {
#pragma unroll
            for (int j = 0; j < CH; j++) xv[j] = hv[s][CH * ci + j];
          } else {
            load_chunk_x<FMT>(a.hbuf + (int64_t)hr * a.hstride, false, c, xv);
          }
          CK::sums(xv, xs);
          p += CK::dot(raw[s][ci], xv, xs);
        }
      }
      p = wave_sum<LPR>(p);
      if (ll == 0) contrib[hr * RG + rg] = wgt[s] * p;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < T * RG; i += 256) {
    const int t = i / RG, r = i % RG;
    if (n0 + r >= a.H) continue;
    float y = 0.f;
    for (int hr = 0; hr < nr; hr++) y += stok[hr] == t ? contrib[hr * RG + r] : 0.f;
    const int64_t o = (int64_t)t * a.H + n0 + r;
    if (a.xbf) ((uint16_t*)a.y)[o] = f32_to_bf16(y);
    else ((float*)a.y)[o] = y;
  }
}

// ----------------------------------------------------------------------------
// prefill fallback down projection: obuf[hrow][n] = w * (down_e row n . h[hrow])
// grid = (row blocks, slots)
// ----------------------------------------------------------------------------
template <int FMT, int LPR, int CPL, int NTOK, int NRG>
__global__ __launch_bounds__(256) void k_down_rows(ExpertArgs a) {
  using CK = Chunk<FMT>;
  constexpr int CH = CK::CH, RG = 64 / LPR, NS = CK::NSUM > 0 ? CK::NSUM : 1;
  const int u = blockIdx.y;
  if (u >= a.counts[0]) return;
  const int e = a.slots[3 * u], start = a.slots[3 * u + 1], count = a.slots[3 * u + 2];
  const bool sh = e == a.E;
  const uint8_t* W = sh ? a.sdown.base : a.down.mat(e);
  const int K = sh ? a.Is : a.I, nch = K / CH, rows = a.H;
  const int lane = lane_id(), wave = threadIdx.x >> 6, rg = lane / LPR, ll = lane % LPR;
  const int row_base = (blockIdx.x * 4 + wave) * (RG * NRG);
  if (row_base >= rows) return;
  typename CK::Raw raw[NRG][CPL];
#pragma unroll
  for (int g = 0; g < NRG; g++) {
    const int row = row_base + g * RG + rg;
#pragma unroll
    for (int ci = 0; ci < CPL; ci++) {
      const int c = ll + LPR * ci;
      if (row < rows && c < nch) CK::load(W, rows, K, row, c, raw[g][ci]);
    }
  }
  for (int tg = 0; tg < count; tg += NTOK) {
    float xv[NTOK][CPL][CH], xs[NTOK][CPL][NS], wgt[NTOK];
    int hrow[NTOK];
#pragma unroll
    for (int tok = 0; tok < NTOK; tok++) {
      const int j = tg + tok < count ? tg + tok : count - 1;
      hrow[tok] = sh ? a.F + j : start + j;
      wgt[tok] = sh ? a.sgw[j] : a.topk_w[a.perm[start + j]];
#pragma unroll
      for (int ci = 0; ci < CPL; ci++) {
        const int c = ll + LPR * ci;
        if (c < nch) {
          load_chunk_x<FMT>(a.hbuf + (int64_t)hrow[tok] * a.hstride, false, c, xv[tok][ci]);
          CK::sums(xv[tok][ci], xs[tok][ci]);
        }
      }
    }
#pragma unroll
    for (int g = 0; g < NRG; g++) {
      const int row = row_base + g * RG + rg;
#pragma unroll
      for (int tok = 0; tok < NTOK; tok++) {
        float p = 0.f;
#pragma unroll
        for (int ci = 0; ci < CPL; ci++) {
          const int c = ll + LPR * ci;
          if (row < rows && c < nch) p += CK::dot(raw[g][ci], xv[tok][ci], xs[tok][ci]);
        }
        p = wave_sum<LPR>(p);
        if (ll == 0 && row < rows && tg + tok < count) {
          const int64_t o = (int64_t)hrow[tok] * a.H + row;
          if (a.xbf) ((uint16_t*)a.obuf)[o] = f32_to_bf16(wgt[tok] * p);
          else ((float*)a.obuf)[o] = wgt[tok] * p;
        }
      }
    }
  }
}

// ----------------------------------------------------------------------------
// combine: y[t] = sum of the token's k weighted expert rows in ascending expert
// order (= ascending permuted position), then the shared expert's row.
// Grid (T, ceil(H / 2048)): a block serves one token and up to 2048 outputs,
// 8 per thread. Wave 0 sorts the token's k positions once (rank of each among
// the k, into LDS); every thread then issues all k + 1 row loads together.
// ----------------------------------------------------------------------------
// RES (the decoder's residual stream, a.resid): y is not written, resid[t]
// becomes resid[t] + y[t], y rounded to the activation dtype first (a kernel of
// its own for that addition took 4.9 us at 27 tokens, 5.2 us at 512).
// (the bound of 8 workgroups per CU holds it to 64 registers, so the T
// workgroups of a prefill are all resident at once instead of in two rounds;
// the residual's element takes one more step of registers)
template <bool RES>
__global__ __launch_bounds__(256, RES ? 7 : 8) void k_combine(ExpertArgs a) {
  __shared__ int spos[HX_MAX_TOPK + 1];
  const int t = blockIdx.x, k = a.k;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const int p = lane < k ? a.inv[(int64_t)t * k + lane] : 0x7fffffff;
    int rank = 0;
    for (int j = 0; j < k; j++) rank += __builtin_amdgcn_readlane(p, j) < p;
    if (lane < k) spos[rank] = p;
    if (lane == 0) spos[k] = a.F + t;   // the shared expert's row (used when Is > 0)
  }
  __syncthreads();
  const int n0 = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (n0 >= a.H) return;
  const int nrows = k + (a.Is > 0 ? 1 : 0);
  // the shared expert's row (row k) scaled here when the down GEMM stored it
  // unweighted; the routed rows are multiplied by 1 (exact)
  const float shs = a.shared_raw && a.Is > 0 ? a.sgw[t] : 1.f;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (a.xbf) {
    uint4 rx = make_uint4(0u, 0u, 0u, 0u);
    if (RES) rx = *(const uint4*)(a.resid + (int64_t)t * a.H + n0);
    // rows loaded B at a time without branches: indices past the last row are
    // clamped to it and their values masked to +0 (adding +0 changes nothing)
    constexpr int B = 12;
    for (int j0 = 0; j0 < nrows; j0 += B) {
      uint4 q[B];
#pragma unroll
      for (int j = 0; j < B; j++) {
        const int r = spos[min(j0 + j, nrows - 1)];
        q[j] = *(const uint4*)((const uint16_t*)a.obuf + (int64_t)r * a.H + n0);
      }
#pragma unroll
      for (int j = 0; j < B; j++) {
        const uint32_t m = j0 + j < nrows ? 0xffffffffu : 0u;
        const uint32_t w[4] = {q[j].x & m, q[j].y & m, q[j].z & m, q[j].w & m};
        const float sc = j0 + j == k ? shs : 1.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          acc[2 * i] += __uint_as_float(w[i] << 16) * sc;
          acc[2 * i + 1] += __uint_as_float(w[i] & 0xffff0000u) * sc;
        }
      }
    }
    uint4 o;
    o.x = f32_to_bf16(acc[0]) | ((uint32_t)f32_to_bf16(acc[1]) << 16);
    o.y = f32_to_bf16(acc[2]) | ((uint32_t)f32_to_bf16(acc[3]) << 16);
    o.z = f32_to_bf16(acc[4]) | ((uint32_t)f32_to_bf16(acc[5]) << 16);
    o.w = f32_to_bf16(acc[6]) | ((uint32_t)f32_to_bf16(acc[7]) << 16);
    if (RES) {
      auto add = [](uint32_t r, uint32_t y) {
        const uint32_t lo = f32_to_bf16(__uint_as_float(r << 16) + __uint_as_float(y << 16));
        return lo | ((uint32_t)f32_to_bf16(__uint_as_float(r & 0xffff0000u) + __uint_as_float(y & 0xffff0000u)) << 16);
      };
      *(uint4*)(a.resid + (int64_t)t * a.H + n0) =
          make_uint4(add(rx.x, o.x), add(rx.y, o.y), add(rx.z, o.z), add(rx.w, o.w));
    } else {
      *(uint4*)((uint16_t*)a.y + (int64_t)t * a.H + n0) = o;
    }
  } else {
    for (int j = 0; j < nrows; j++) {
      const float4* q = (const float4*)((const float*)a.obuf + (int64_t)spos[j] * a.H + n0);
      const float4 u = q[0], v = q[1];
      const float sc = j == k ? shs : 1.f;
      acc[0] += u.x * sc; acc[1] += u.y * sc; acc[2] += u.z * sc; acc[3] += u.w * sc;
      acc[4] += v.x * sc; acc[5] += v.y * sc; acc[6] += v.z * sc; acc[7] += v.w * sc;
    }
    float* base = RES ? (float*)a.resid : (float*)a.y;
    float4* p = (float4*)(base + (int64_t)t * a.H + n0);
    if (RES) {
      const float4 u = p[0], v = p[1];
      p[0] = make_float4(u.x + acc[0], u.y + acc[1], u.z + acc[2], u.w + acc[3]);
      p[1] = make_float4(v.x + acc[4], v.y + acc[5], v.z + acc[6], v.w + acc[7]);
    } else {
      p[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
      p[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
    }
  }
}

// ----------------------------------------------------------------------------
// launchers: pick LPR / CPL from K and the chunk size
// ----------------------------------------------------------------------------
template <int FMT>
static int chunks_per_row(int K) { return K / Chunk<FMT>::CH; }

// chunks per row -> (lanes per row, chunks per lane); rows longer than 512
// chunks are rejected when the block is created
#define HX_LPR_CASES(MACRO, NCH)                       \
  if ((NCH) > 512) { return hipErrorInvalidValue; }    \
  else if ((NCH) > 256) { MACRO(64, 8); }              \
  else if ((NCH) > 128) { MACRO(64, 4); }              \
  else if ((NCH) > 64) { MACRO(64, 2); }               \
  else if ((NCH) > 32) { MACRO(64, 1); }               \
  else if ((NCH) > 16) { MACRO(32, 1); }               \
  else if ((NCH) > 8) { MACRO(16, 1); }                \
  else { MACRO(8, 1); }

template <int FMT>
static hipError_t gate_up_fmt(const ExpertArgs& a, bool decode, hipStream_t s) {
  const int nch = chunks_per_row<FMT>(a.H);
  const int maxrows = a.I > a.Is ? a.I : a.Is;
  const int nslot = a.max_slots;
#define GU(LPR, CPL)                                                                          \
  {                                                                                           \
    constexpr int RG = 64 / LPR, NRG = (CPL >= 2 ? 1 : 2);                                    \
    dim3 grid((maxrows + 4 * RG * NRG - 1) / (4 * RG * NRG), nslot);                          \
    if (decode && a.T == 1)                                                                   \
      hipLaunchKernelGGL((k_gate_up<FMT, LPR, CPL, 1, NRG>), grid, dim3(256), 0, s, a);       \
    else                                                                                      \
      hipLaunchKernelGGL((k_gate_up<FMT, LPR, CPL, 2, NRG>), grid, dim3(256), 0, s, a);       \
  }
  HX_LPR_CASES(GU, nch)
#undef GU
  return hipGetLastError();
}

template <int FMT>
static hipError_t down_combine_fmt(const ExpertArgs& a, hipStream_t s) {
  const int K = a.I > a.Is ? a.I : a.Is;
  const int nch = chunks_per_row<FMT>(K);
#define DC(LPR, CPL)                                                                            \
  {                                                                                             \
    constexpr int RG = 64 / LPR;                                                                \
    size_t lds = (size_t)(a.F + a.T) * (RG + 1) * sizeof(float);                                \
    hipLaunchKernelGGL((k_down_combine<FMT, LPR, CPL, 4>), dim3((a.H + RG - 1) / RG), dim3(256), \
                       lds, s, a);                                                              \
  }
  HX_LPR_CASES(DC, nch)
#undef DC
  return hipGetLastError();
}

template <int FMT>
static hipError_t down_rows_fmt(const ExpertArgs& a, hipStream_t s) {
  const int K = a.I > a.Is ? a.I : a.Is;
  const int nch = chunks_per_row<FMT>(K);
#define DR(LPR, CPL)                                                                          \
  {                                                                                           \
    constexpr int RG = 64 / LPR, NRG = (CPL >= 2 ? 1 : 2);                                    \
    dim3 grid((a.H + 4 * RG * NRG - 1) / (4 * RG * NRG), a.max_slots);                        \
    hipLaunchKernelGGL((k_down_rows<FMT, LPR, CPL, 2, NRG>), grid, dim3(256), 0, s, a);       \
  }
  HX_LPR_CASES(DR, nch)
#undef DR
  return hipGetLastError();
}

hipError_t launch_gate_up_gemv(const ExpertArgs& a, hipStream_t s) {
  switch (a.gate.fmt) {
    case HX_F32: return gate_up_fmt<HX_F32>(a, true, s);
    case HX_BF16: return gate_up_fmt<HX_BF16>(a, true, s);
    case HX_Q8_0: return gate_up_fmt<HX_Q8_0>(a, true, s);
    case HX_Q4_K: return gate_up_fmt<HX_Q4_K>(a, true, s);
    case HX_Q6_K: return gate_up_fmt<HX_Q6_K>(a, true, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gate_up_prefill(const ExpertArgs& a, hipStream_t s) {
  switch (a.gate.fmt) {
    case HX_F32: return gate_up_fmt<HX_F32>(a, false, s);
    case HX_BF16: return gate_up_fmt<HX_BF16>(a, false, s);
    case HX_Q8_0: return gate_up_fmt<HX_Q8_0>(a, false, s);
    case HX_Q4_K: return gate_up_fmt<HX_Q4_K>(a, false, s);
    case HX_Q6_K: return gate_up_fmt<HX_Q6_K>(a, false, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_down_gemv_combine(const ExpertArgs& a, hipStream_t s) {
  switch (a.down.fmt) {
    case HX_F32: return down_combine_fmt<HX_F32>(a, s);
    case HX_BF16: return down_combine_fmt<HX_BF16>(a, s);
    case HX_Q8_0: return down_combine_fmt<HX_Q8_0>(a, s);
    case HX_Q4_K: return down_combine_fmt<HX_Q4_K>(a, s);
    case HX_Q6_K: return down_combine_fmt<HX_Q6_K>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_down_prefill(const ExpertArgs& a, hipStream_t s) {
  switch (a.down.fmt) {
    case HX_F32: return down_rows_fmt<HX_F32>(a, s);
    case HX_BF16: return down_rows_fmt<HX_BF16>(a, s);
    case HX_Q8_0: return down_rows_fmt<HX_Q8_0>(a, s);
    case HX_Q4_K: return down_rows_fmt<HX_Q4_K>(a, s);
    case HX_Q6_K: return down_rows_fmt<HX_Q6_K>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_combine(const ExpertArgs& a, hipStream_t s) {
  // H % 8 == 0 holds for every block this library creates with a combine step
  const dim3 g((unsigned)a.T, (unsigned)((a.H / 8 + 255) / 256));
  if (a.resid) hx_launch(k_combine<true>, g, dim3(256), 0, s, a);
  else hx_launch(k_combine<false>, g, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace hx
