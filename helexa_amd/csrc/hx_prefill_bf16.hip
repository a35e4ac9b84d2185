// Prefill grouped GEMMs on the matrix cores for unquantised checkpoints (bf16
// activations, bf16 experts).
//
// Reference: the plain Linear arm of MaybeQuantLinear inside the fused MoE path
// (crates/neuron/src/harness/tp/tp_linear.rs:107-118,
// crates/neuron/src/harness/tp/tp_qwen3_5.rs:1192-1225): three grouped GEMMs
// over expert-sorted rows, the routing weights folded into the down GEMM.
//
// Work unit: one M tile of the dispatch list (<= 64 permuted rows of one
// expert, or of the shared expert) x one N tile, as in hx_prefill.hip. Products
// of bf16 pairs are exact and summed in f32 by v_mfma_f32_16x16x32_bf16 (lane l
// holds A[l%16][8(l/16)+i], B[8(l/16)+i][l%16] and D rows 4(l/16)+i of column
// l%16). h = silu(g) u is an f32 value and stays one: it is cut into three bf16
// parts (8 significant bits each, by truncation, so hi + mid + lo == h), and the
// down GEMM multiplies all three, the smallest first.
//
// A prompt of a few hundred tokens gives most experts a handful of rows, so the
// launches are bound by streaming the weights (6.3 MB an expert at the 80B-A3B
// widths) from HBM. A weight element is used by one wave only, so each wave
// loads its MFMA operands from global memory straight into registers, one
// chunk ahead; LDS holds just the rows all waves share (double buffered, one
// barrier a chunk, which leaves the weight loads in flight). Tiles run only the
// 16-row sub-tiles they use. Measured at 301 skewed tokens, 80B-A3B layer (1.05
// GB of gate / up and 0.52 GB of down rows touched): gate/up 1,210 -> 211 us
// (5.0 TB/s), down 588 -> 119 us (4.4 TB/s), against the GEMV kernels of
// hx_experts.hip, which multiply two tokens a pass on the vector units.
#include "hx_prefill_dev.h"
#include <type_traits>

namespace hx {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

HX_DEV u32x4_t ld16(const void* p) { return *(const u32x4_t*)p; }
HX_DEV bf16x8_t bfrag(u32x4_t v) { return __builtin_bit_cast(bf16x8_t, v); }
HX_DEV bf16x8_t bfrag(const uint16_t* p) { return bfrag(ld16(p)); }
HX_DEV f32x4_t mfma_bf16(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
template <int V>
using ic = std::integral_constant<int, V>;

// f32 -> bf16 parts hi, mid, lo with hi + mid + lo == v (each step truncates, so
// the remainder is exact); inf and NaN go whole into hi. A part that comes out
// zero where v is not is the smallest bf16 of v's sign, 2^-133, instead: times an
// infinite weight each part then gives the infinity that v gives, where a zero
// gives NaN. What it adds to v is below half an f32 step from |v| = 2^-108 on.
HX_DEV void split3(float v, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const uint32_t u = __float_as_uint(v);
  const bool fin = (u & 0x7f800000u) != 0x7f800000u;
  const float r = fin ? v - __uint_as_float(u & 0xffff0000u) : 0.f;
  const uint32_t ur = __float_as_uint(r), ul = __float_as_uint(r - __uint_as_float(ur & 0xffff0000u));
  const uint32_t least = v == 0.f ? u >> 16 : ((u >> 16) & 0x8000u) | 1u;
  auto part = [&](uint32_t w) { return w & 0x7fff0000u ? w >> 16 : least; };
  hi = v == v ? part(u) : 0x7fc0u;
  mid = part(ur);
  lo = part(ul);
}

// the M tile of a workgroup. SM (up to HX_DECODE_MAX_T tokens): slot `tile` of the
// decode plan, at most 8 rows; else the dispatch list's tile
template <bool SM>
HX_DEV bool bf_tile(const ExpertArgs& a, int tile, int& e, int& p0, int& rows) {
  if constexpr (SM) {
    const int4 rec = *(const int4*)(a.plan + 4 + 4 * min(tile, a.max_slots - 1));
    const int n = a.plan[0];
    e = rec.x;
    p0 = rec.y;
    rows = rec.z;
    return tile < n;
  } else {
    int mc;
    return get_tile<HX_TILES_ALL>(a, tile, e, p0, rows, mc);
  }
}

// the three planes of h: two in hbuf's bytes, one in hbf, rows of hstride
HX_DEV uint16_t* h_plane(const ExpertArgs& a, int p) {
  return p < 2 ? (uint16_t*)a.hbuf + (int64_t)p * (a.F + a.T) * a.hstride : a.hbf;
}

// ---------------------------------------------------------------- gate/up
// 64 rows x (64 gate + 64 up columns); wave w owns columns 16 w .. + 15 of both.
// K chunk 128: rows at a pitch of 136 in LDS (the 16 lanes of a fragment read
// fall on different banks); per wave and chunk 8 weight loads of 16 bytes a lane,
// each a 64-byte run of 16 weight rows.
constexpr int BG_K = 128, BG_LD = BG_K + 8;
constexpr int BG_OP = 68;   // pitch of the f32 tile of h (aliases the rows)

template <int MT, int LR>   // LR: rows an LDS buffer holds
HX_DEV void bf_gate_up_main(const ExpertArgs& a, uint16_t* As, const uint8_t* G, const uint8_t* U, int rows, int p0,
                            int n0, bool sh) {
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, l16 = lane & 15, kq = lane >> 4;
  const int K = a.H, nk = K / BG_K;   // even
  // uniform bases and 32-bit lane offsets
  const uint8_t* bp[2] = {G + (int64_t)n0 * K * 2, U + (int64_t)n0 * K * 2};
  const uint32_t bo = (uint32_t)((16 * wave + l16) * K + 8 * kq) * 2;
  const int r0 = tid >> 4, seg = tid & 15;   // A piece i: row r0 + 16 i, elements 8 seg ..
  // the rows' entries are read ahead of the first weight loads and used behind them
  int src[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) {
    const int p = p0 + min(r0 + 16 * i, rows - 1);   // padding rows repeat the last row
    src[i] = sh ? p : a.perm[p];
  }
  __builtin_amdgcn_sched_barrier(0);
  const uint16_t* ap[MT];
  u32x4_t ar[MT], b[2][2][4];
  auto load_a = [&](int kc) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; i++) ar[i] = ld16(ap[i] + kc * BG_K);
  };
  auto load_b = [&](int kc, auto buf) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
      for (int s = 0; s < 4; s++) b[decltype(buf)::value][m][s] = ld16(bp[m] + kc * (2 * BG_K) + (bo + 64 * s));
  };
  auto store_a = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; i++) *(u32x4_t*)(As + (buf * LR + r0 + 16 * i) * BG_LD + 8 * seg) = ar[i];
  };
  f32x4_t acc[2][MT];
#pragma unroll
  for (int m = 0; m < 2; m++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[m][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  load_b(0, ic<0>{});
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < MT; i++) ap[i] = (const uint16_t*)a.x + (int64_t)(sh ? src[i] - a.F : src[i] / a.k) * K + 8 * seg;
  load_a(0);
  store_a(0);
  lds_barrier();
  auto step = [&](int kc, auto par, auto more) __attribute__((always_inline)) {
    constexpr int P = decltype(par)::value;
    if constexpr (decltype(more)::value) {   // the rows first: waiting for them then leaves the weights in flight
      load_a(kc + 1);
      load_b(kc + 1, ic<1 - P>{});
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
      for (int i = 0; i < MT; i++) {
        const bf16x8_t av = bfrag(As + (P * LR + 16 * i + l16) * BG_LD + 32 * s + 8 * kq);
#pragma unroll
        for (int m = 0; m < 2; m++) acc[m][i] = mfma_bf16(av, bfrag(b[P][m][s]), acc[m][i]);
      }
      if constexpr (MT >= 3) __builtin_amdgcn_sched_barrier(0);   // fewer row fragments held: no spills
    }
    if constexpr (decltype(more)::value) store_a(1 - P);
    lds_barrier();
  };
  for (int kc = 0; kc < nk - 2; kc += 2) {
    step(kc, ic<0>{}, ic<1>{});
    step(kc + 1, ic<1>{}, ic<1>{});
  }
  step(nk - 2, ic<0>{}, ic<1>{});
  step(nk - 1, ic<1>{}, ic<0>{});
  // h in f32 through LDS (the rows are done with), out as three bf16 planes,
  // eight columns a thread
  float* ot = (float*)As;
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int q = 0; q < 4; q++)
      ot[(16 * i + 4 * kq + q) * BG_OP + 16 * wave + l16] = siluf_(acc[0][i][q]) * acc[1][i][q];
  lds_barrier();
  const int c8 = 8 * (tid & 7);
#pragma unroll
  for (int m = tid >> 3; m < 16 * MT; m += 32) {
    if (m >= rows) break;
    const float4 u = *(const float4*)(ot + m * BG_OP + c8), v = *(const float4*)(ot + m * BG_OP + c8 + 4);
    const float f[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    uint32_t w[3][8];
#pragma unroll
    for (int j = 0; j < 8; j++) split3(f[j], w[0][j], w[1][j], w[2][j]);
#pragma unroll
    for (int p = 0; p < 3; p++)
      *(uint4*)(h_plane(a, p) + (int64_t)(p0 + m) * a.hstride + n0 + c8) =
          make_uint4(w[p][0] | (w[p][1] << 16), w[p][2] | (w[p][3] << 16), w[p][4] | (w[p][5] << 16),
                     w[p][6] | (w[p][7] << 16));
  }
}

// grid (I / 64, tiles rounded up to 8), mapped by xcd_tile
template <bool SM>
__global__ __launch_bounds__(256, SM ? 4 : 3) void k_gate_up_bf16(ExpertArgs a) {
  constexpr int LR = SM ? 16 : PM;
  __shared__ __attribute__((aligned(16))) uint16_t As[2 * LR * BG_LD];
  static_assert(sizeof(float) * LR * BG_OP <= sizeof(As), "the tile of h fits the rows' LDS");
  int nt, tile, e, p0, rows;
  xcd_tile(nt, tile);
  if (!bf_tile<SM>(a, tile, e, p0, rows)) return;
  const bool sh = e == a.E;
  const uint8_t* G = sh ? a.sgate.base : a.gate.mat(e);
  const uint8_t* U = sh ? a.sup.base : a.up.mat(e);
  const int n0 = nt * 64;
  if constexpr (SM) {
    bf_gate_up_main<1, LR>(a, As, G, U, rows, p0, n0, sh);
  } else {
    switch ((rows + 15) >> 4) {   // uniform over the workgroup
      case 1: bf_gate_up_main<1, LR>(a, As, G, U, rows, p0, n0, sh); break;
      case 2: bf_gate_up_main<2, LR>(a, As, G, U, rows, p0, n0, sh); break;
      case 3: bf_gate_up_main<3, LR>(a, As, G, U, rows, p0, n0, sh); break;
      default: bf_gate_up_main<4, LR>(a, As, G, U, rows, p0, n0, sh); break;
    }
  }
}

// ---------------------------------------------------------------- down
// 64 rows of h x 128 output columns; wave w owns columns 32 w .. + 31 (two
// fragments). K chunk 64: the three planes of the rows in LDS, the 16-byte
// pieces of row r at slot piece ^ (r / 2 % 8) (rows are 128 bytes apart, so
// without it every other row meets the same banks); the weights come 128 K at
// a time. Rows are scaled by their routing weight by position and written as
// bf16 to the per-assignment rows; SM (up to 8 tokens) as f32 ones, which
// k_combine_few sums: the decode step's output is rounded once.
constexpr int BD_K = 64;
template <bool SM>
struct Bd {
  static constexpr int PLANE = (SM ? 32 : PM) * BD_K, STAGE = 3 * PLANE;
};
constexpr int BD_OP = 136;    // pitch of the bf16 output tile (aliases the rows)
constexpr int BD_OPF = 132;   // of the f32 one

template <int MT, bool SM>
HX_DEV void bf_down_main(const ExpertArgs& a, uint16_t* As, float* rws, const uint8_t* W, int K, int rows, int p0, int n0,
                         float rw) {
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, l16 = lane & 15, kq = lane >> 4;
  constexpr int NA = (MT + 1) / 2;   // rounds of 32 rows
  constexpr int BD_PLANE = Bd<SM>::PLANE, BD_STAGE = Bd<SM>::STAGE;
  const int nc = K / 128;            // even
  const uint8_t* bp = W + (int64_t)n0 * K * 2;
  const uint32_t bo = (uint32_t)((32 * wave + l16) * K + 8 * kq) * 2, bj = (uint32_t)(16 * K) * 2;
  const int r0 = tid >> 3, pc = tid & 7;
  uint32_t ao[NA];
#pragma unroll
  for (int i = 0; i < NA; i++) ao[i] = (uint32_t)(min(r0 + 32 * i, rows - 1) * a.hstride + 8 * pc);
  const int64_t h0 = (int64_t)p0 * a.hstride;
  const uint16_t* hp[3] = {h_plane(a, 0) + h0, h_plane(a, 1) + h0, h_plane(a, 2) + h0};
  u32x4_t ar[3][NA], b[2][2][4];
  auto load_a = [&](int hc) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int i = 0; i < NA; i++) ar[p][i] = ld16(hp[p] + hc * BD_K + ao[i]);
  };
  auto store_a = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 3; p++)
#pragma unroll
      for (int i = 0; i < NA; i++) {
        const int r = r0 + 32 * i;
        *(u32x4_t*)(As + buf * BD_STAGE + p * BD_PLANE + r * BD_K + 8 * (pc ^ ((r >> 1) & 7))) = ar[p][i];
      }
  };
  auto load_b = [&](int c, auto buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int s = 0; s < 4; s++) b[decltype(buf)::value][j][s] = ld16(bp + c * 256 + (bo + j * bj + 64 * s));
  };
  f32x4_t acc[2][MT];
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  load_a(0);
  load_b(0, ic<0>{});
  store_a(0);
  lds_barrier();
  // half chunk HF of weight chunk c (its weights in buffer P); last: no chunk follows
  auto step = [&](int c, auto half, auto buf, auto last) __attribute__((always_inline)) {
    constexpr int HF = decltype(half)::value, P = decltype(buf)::value;
    constexpr bool more = HF == 0 || !decltype(last)::value;
    if constexpr (more) load_a(2 * c + HF + 1);
    if constexpr (HF == 0 && !decltype(last)::value) load_b(c + 1, ic<1 - P>{});
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int i = 0; i < MT; i++) {
        const int r = 16 * i + l16;
        const uint16_t* at = As + HF * BD_STAGE + r * BD_K + 8 * ((4 * s + kq) ^ ((r >> 1) & 7));
        const bf16x8_t a0 = bfrag(at), a1 = bfrag(at + BD_PLANE), a2 = bfrag(at + 2 * BD_PLANE);
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j][i] = mfma_bf16(a2, bfrag(b[P][j][2 * HF + s]), acc[j][i]);
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j][i] = mfma_bf16(a1, bfrag(b[P][j][2 * HF + s]), acc[j][i]);
#pragma unroll
        for (int j = 0; j < 2; j++) acc[j][i] = mfma_bf16(a0, bfrag(b[P][j][2 * HF + s]), acc[j][i]);
      }
      if constexpr (MT >= 3) __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (more) store_a(1 - HF);
    lds_barrier();
  };
  for (int c = 0; c < nc - 2; c += 2) {
    step(c, ic<0>{}, ic<0>{}, ic<0>{});
    step(c, ic<1>{}, ic<0>{}, ic<0>{});
    step(c + 1, ic<0>{}, ic<1>{}, ic<0>{});
    step(c + 1, ic<1>{}, ic<1>{}, ic<0>{});
  }
  step(nc - 2, ic<0>{}, ic<0>{}, ic<0>{});
  step(nc - 2, ic<1>{}, ic<0>{}, ic<0>{});
  step(nc - 1, ic<0>{}, ic<1>{}, ic<1>{});
  step(nc - 1, ic<1>{}, ic<1>{}, ic<1>{});
  if (tid < PM) rws[tid] = rw;
  lds_barrier();
  if constexpr (SM) {
    float* of = (float*)As;
    const f32x4_t w = *(const f32x4_t*)(rws + 4 * kq);
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int j = 0; j < 2; j++) of[(4 * kq + q) * BD_OPF + 32 * wave + 16 * j + l16] = w[q] * acc[j][0][q];
    lds_barrier();
    const int m = tid >> 5, c4 = 4 * (tid & 31);   // rows 0 .. 7: a slot has no more
    if (m < rows)
      *(float4*)((float*)a.obuf + (int64_t)(p0 + m) * a.H + n0 + c4) = *(const float4*)(of + m * BD_OPF + c4);
    return;
  }
  uint16_t* ot = As;
#pragma unroll
  for (int i = 0; i < MT; i++) {
    const f32x4_t w = *(const f32x4_t*)(rws + 16 * i + 4 * kq);
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int j = 0; j < 2; j++)
        ot[(16 * i + 4 * kq + q) * BD_OP + 32 * wave + 16 * j + l16] = f32_to_bf16(w[q] * acc[j][i][q]);
  }
  lds_barrier();
  const int c8 = 8 * (tid & 15);
#pragma unroll
  for (int i = 0, m = tid >> 4; i < MT; i++, m += 16)
    if (m < rows)
      *(uint4*)((uint16_t*)a.obuf + (int64_t)(p0 + m) * a.H + n0 + c8) = *(const uint4*)(ot + m * BD_OP + c8);
}

// grid (H / 128, tiles rounded up to 8), mapped by xcd_tile
template <bool SM>
__global__ __launch_bounds__(256, SM ? 4 : 3) void k_down_bf16(ExpertArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t As[2 * Bd<SM>::STAGE];
  __shared__ __attribute__((aligned(16))) float rws[PM];
  static_assert(PM * BD_OP <= 2 * Bd<false>::STAGE && 16 * BD_OPF * 2 <= 2 * Bd<true>::STAGE,
                "the output tile fits the rows' LDS");
  int nt, tile, e, p0, rows;
  xcd_tile(nt, tile);
  if (!bf_tile<SM>(a, tile, e, p0, rows)) return;
  const bool sh = e == a.E;
  const uint8_t* W = sh ? a.sdown.base : a.down.mat(e);
  const int K = sh ? a.Is : a.I, n0 = nt * 128;
  // a row's routing weight, used by the epilogue
  const float rw = threadIdx.x < PM ? a.wpos[p0 + min((int)threadIdx.x, rows - 1)] : 0.f;
  if constexpr (SM) {
    bf_down_main<1, SM>(a, As, rws, W, K, rows, p0, n0, rw);
  } else {
    switch ((rows + 15) >> 4) {   // uniform over the workgroup
      case 1: bf_down_main<1, SM>(a, As, rws, W, K, rows, p0, n0, rw); break;
      case 2: bf_down_main<2, SM>(a, As, rws, W, K, rows, p0, n0, rw); break;
      case 3: bf_down_main<3, SM>(a, As, rws, W, K, rows, p0, n0, rw); break;
      default: bf_down_main<4, SM>(a, As, rws, W, K, rows, p0, n0, rw); break;
    }
  }
}

// ---------------------------------------------------------------- combine, up to 8 tokens
// y[t] = the sum of token t's f32 rows in dispatch order (experts ascending, then
// the shared expert), rounded once. Bound by latency: grid (T, H / 1024), four
// outputs a thread, all its row loads together. RES as k_combine.
template <bool RES>
__global__ __launch_bounds__(256) void k_combine_few(ExpertArgs a) {
  __shared__ int spos[HX_MAX_TOPK + 1];
  const int t = blockIdx.x, k = a.k, tid = threadIdx.x;
  if (tid < 64) {
    const int p = tid < k ? a.inv[t * k + tid] : 0x7fffffff;
    int rank = 0;
    for (int j = 0; j < k; j++) rank += __builtin_amdgcn_readlane(p, j) < p;
    if (tid < k) spos[rank] = p;
    if (tid == 0) spos[k] = a.F + t;
  }
  const int n0 = (blockIdx.y * 256 + tid) * 4;
  const bool in = n0 < a.H;
  const int64_t o = (int64_t)t * a.H + (in ? n0 : 0);
  uint2 rx = make_uint2(0u, 0u);
  if (RES) rx = *(const uint2*)(a.resid + o);
  __syncthreads();
  if (!in) return;
  const int nrows = k + (a.Is > 0 ? 1 : 0);
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  constexpr int B = 12;
  for (int j0 = 0; j0 < nrows; j0 += B) {
    float4 q[B];
#pragma unroll
    for (int j = 0; j < B; j++)   // past the last row: the last one again, not added
      q[j] = *(const float4*)((const float*)a.obuf + (int64_t)spos[min(j0 + j, nrows - 1)] * a.H + n0);
#pragma unroll
    for (int j = 0; j < B; j++) {
      const bool use = j0 + j < nrows;
      acc[0] += use ? q[j].x : 0.f;
      acc[1] += use ? q[j].y : 0.f;
      acc[2] += use ? q[j].z : 0.f;
      acc[3] += use ? q[j].w : 0.f;
    }
  }
  uint32_t y[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    y[i] = f32_to_bf16(acc[i]);
    const uint32_t w = i < 2 ? rx.x : rx.y;
    if (RES) y[i] = f32_to_bf16(__uint_as_float(i & 1 ? w & 0xffff0000u : w << 16) + __uint_as_float(y[i] << 16));
  }
  uint16_t* out = (RES ? a.resid : (uint16_t*)a.y) + o;
  if (((uintptr_t)out & 7) == 0) {
    *(uint2*)out = make_uint2(y[0] | (y[1] << 16), y[2] | (y[3] << 16));
  } else {   // an output at any element, as the vector kernels take it
#pragma unroll
    for (int i = 0; i < 4; i++) out[i] = (uint16_t)y[i];
  }
}

// ---------------------------------------------------------------- launchers
// every prefill call of the widths the chunks (two of 128 K an iteration) and
// column tiles divide; other widths take the GEMV kernels (from 9 tokens on the
// MFMA kernels are the faster: 9 tokens 114 against 138 us, 301 tokens 365
// against 1,856 us, 2048 tokens 777 against 12,660 us a forward of the 80B-A3B
// layer; fewer tokens: few_bf16_ok). So do calls of more M tiles than a launch's
// grid takes (from about 378,000 tokens of that layer on): the GEMV kernels' grids
// do not grow with the tokens.
bool prefill_bf16_ok(const ExpertArgs& a) {
  return a.max_tiles <= HX_MAX_GRID_Y && a.xbf && a.gate.fmt == HX_BF16 && a.down.fmt == HX_BF16 && a.H % 256 == 0 && a.I % 256 == 0 &&
         (a.Is == 0 || a.Is == a.I);
}

// A workgroup's K loop is a chain of round trips however few slots there are
// (about 25 us over both launches), which the decode GEMVs' short workgroups do
// not have. Forward, GEMV against this: 128 experts of 256, hidden 2048, top-8: 4
// tokens 44.2 / 45.7 us, 5 52.4 / 49.2, 8 67.0 / 56.3; 128 of 768, top-6: 3
// 51.9 / 58.3, 5 77.6 / 65.8, 8 105.0 / 74.0; 64 of 256, hidden 1024, top-4: 5
// (20 assignments) 25.6 / 28.3, 6 28.7 / 29.8, 8 33.6 / 31.4; 80B-A3B layer: 2
// 47.1 / 47.0, 3 69.8 / 58.4, 4 84.0 / 80.2, 5 101.8 / 90.2, 8 146.3 / 125.6. The
// line is where the smaller of these layers gain (five tokens, 30 assignments); the
// widest would gain from 3 tokens on, which a rule on tokens alone gives up.
bool few_bf16_ok(const ExpertArgs& a, int64_t T) {
  return T >= 5 && T <= HX_DECODE_MAX_T && T * a.k >= 30 && prefill_bf16_ok(a);
}

hipError_t launch_gate_up_bf16(const ExpertArgs& a, hipStream_t s) {
  if (a.T <= HX_DECODE_MAX_T)
    hx_launch(k_gate_up_bf16<true>, dim3(a.I / 64, (a.max_slots + 7) / 8 * 8), dim3(256), 0, s, a);
  else hx_launch(k_gate_up_bf16<false>, dim3(a.I / 64, (a.max_tiles + 7) / 8 * 8), dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_down_bf16(const ExpertArgs& a, hipStream_t s) {
  if (a.T <= HX_DECODE_MAX_T)
    hx_launch(k_down_bf16<true>, dim3(a.H / 128, (a.max_slots + 7) / 8 * 8), dim3(256), 0, s, a);
  else hx_launch(k_down_bf16<false>, dim3(a.H / 128, (a.max_tiles + 7) / 8 * 8), dim3(256), 0, s, a);
  return hipGetLastError();
}
hipError_t launch_combine_few(const ExpertArgs& a, hipStream_t s) {
  const dim3 g((unsigned)a.T, (unsigned)((a.H + 1023) / 1024));
  if (a.resid) hx_launch(k_combine_few<true>, g, dim3(256), 0, s, a);
  else hx_launch(k_combine_few<false>, g, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace hx
