// Prefill grouped GEMMs whose weights go from global memory straight into the
// registers of the wave that multiplies them (bf16 activations, Q8_0 experts).
//
// Reference: as hx_prefill.hip, whose work units, arms (m <= HX_QUANT_M rows:
// the f16 d q of the activations' codes; more: f16 activations, products
// rounded to f16) and element order along K ((0, 2, 1, 3) in every group of 4)
// these kernels share.
//
// A weight is used by one wave only (wave w of a workgroup owns its columns for
// all 64 rows of the tile), so staging it in LDS buys nothing: each lane loads
// 16 bytes of codes of its column's row per 64 K and dequantises them into its
// MFMA operands, one K chunk of 128 ahead. LDS holds the activation rows, which
// all four waves read: two buffers of 64 x 128 f16, filled through registers a
// chunk ahead, one barrier a chunk that leaves the weight loads in flight.
//
// Tiles run only the 16-row sub-tiles they use. What a workgroup needs before
// its first chunk goes out in one chain of two loads (tile record, then the row
// indices; weights and scales beside the latter), and the routing weights of the
// epilogue are read at the start. Bound by the rate at which weights come
// through the fabric (loads alone: 0.9 of the gate/up time at 512 tokens).
// Measured (80B-A3B layer, Q8_0, skewed tokens) against both operands
// dequantised into LDS by all threads: gate/up 27 tokens 118 -> 98 us, 512
// tokens 161 -> 136 (4.6 TB/s), 2048 297 -> 235; down 61 -> 49, 83 -> 71, 168 -> 133.
// Four fragments a wave for tiles of at most 32 rows (half the workgroups, twice
// the bytes each) were slower: 512 tokens gate/up 154 us, and 185 when the idle
// workgroups were those of odd column blocks, which all fall to the same two of
// an XCD's four shader engines.
//
// MFMA (v_mfma_f32_16x16x32_f16: lane l holds A[l%16][8(l/16)+i],
// B[8(l/16)+i][l%16], D rows 4(l/16)+i of column l%16): step s of a chunk takes
// elements 32 s .. + 31, as in hx_prefill.hip, so that the partial sums, and with
// them every output bit, are those of the kernels that dequantise into LDS.
// Summing in the order in which the lanes' 16 bytes lie, without the exchange of
// FragQ8::order, moved one output in 250 of a 512-token call by one bf16 step, for
// 0.4 to 0.7 % of the time (512 tokens 252.0 us, 253.8 with it; 2048 445.7, 447.4);
// 8-byte loads in place of the exchange took 314 and 573 us.
#include "hx_prefill_dev.h"
#include "hx_quant.h"
#include <type_traits>

namespace hx {

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
template <int V>
using ic = std::integral_constant<int, V>;

#define HX_HD __host__ __device__
constexpr int PD_K = 128, PD_LD = PD_K + 8;   // K chunk; LDS row pitch (16 rows of a fragment: different banks)

HX_DEV u32x4_t ld16(const void* p) { return *(const u32x4_t*)p; }
// buffer loads: a uniform base (with its extent, past which reads give 0), a
// 32-bit lane offset kept for the whole kernel and a uniform offset that moves
// with the chunk: no 64-bit address registers a stream
HX_DEV __amdgpu_buffer_rsrc_t rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00027000);
}
HX_DEV u32x4_t buf16(__amdgpu_buffer_rsrc_t r, uint32_t lane_off, uint32_t off) {
  return __builtin_amdgcn_raw_buffer_load_b128(r, lane_off, off, 0);
}
HX_DEV h2_t h2(uint32_t v) { return __builtin_bit_cast(h2_t, v); }
HX_DEV uint32_t u32(h2_t v) { return __builtin_bit_cast(uint32_t, v); }
// position of element i of a row in the swizzled storage order
HX_DEV int swz(int i) { return (i & ~3) | ((i & 1) << 1) | ((i >> 1) & 1); }

// ---------------------------------------------------------------- Q8_0
// planar rows: K int8 codes, then the scale plane [rows][K / 32] f16. A lane
// loads two runs of 16 codes a chunk: run u is piece m of elements 64 u .. + 63,
// m = kq with its two bits exchanged, so that lane groups 2 j and 2 j + 1 hold
// what either needs of steps 2 u and 2 u + 1 (order). The scales of the tile's 128 weight
// rows are copied into LDS first, whole rows at a time: read chunk by chunk, 8
// bytes of each row, every load touched 16 cache lines that were gone before
// the next chunk's (2048 tokens of the 80B-A3B layer: gate/up 284 us, 215 us
// without those loads).
struct FragQ8 {
  struct Raw {
    u32x4_t q[2];
  };
  static constexpr int AUX_PAD = 8;   // bytes after a row's scales: 16 rows on different banks
  // K columns whose scales are in LDS at a time, and the LDS bytes of one
  // weight row's (at most 136, so that three workgroups fit a CU at any K)
  static constexpr int WIN = 2048;
  HX_HD static int aux_row(int K) { return (K < WIN ? K : WIN) / 16 + AUX_PAD; }
  __amdgpu_buffer_rsrc_t q;   // the matrix from the tile's first row on
  uint32_t qo;                // this lane's row
  uint32_t sc;                // byte in aux of this lane's row's scales
  // a weight row's scales in the plane behind a matrix of R rows
  HX_DEV static const uint8_t* aux_src(const uint8_t* mat, int R, int K, int row) {
    return mat + (int64_t)R * K + (int64_t)row * (K / 16);
  }
  // the scales of columns k0 .. k0 + kw - 1 of NR of the tile's weight rows into
  // LDS: 256 / NR threads a row (src: aux_src of this thread's, slot: its place
  // in aux), all their 16-byte pieces in flight together, the store behind them
  template <int NR>
  struct Aux {
    static constexpr int TPR = 256 / NR, NP = WIN / 256 / TPR;
    u32x4_t v[NP];
    HX_DEV void load(const uint8_t* src, int k0, int kw) {
#pragma unroll
      for (int i = 0; i < NP; i++)
        v[i] = ld16(src + k0 / 16 + 16 * min(TPR * i + (int)threadIdx.x % TPR, kw / 256 - 1));
    }
    HX_DEV void store(int K, int kw, uint8_t* aux) const {
#pragma unroll
      for (int i = 0; i < NP; i++) {
        const int p = TPR * i + (int)threadIdx.x % TPR;
        if (p < kw / 256) {   // rows are 8-byte aligned
          u32x2_t* o = (u32x2_t*)(aux + ((int)threadIdx.x / TPR) * aux_row(K) + 16 * p);
          o[0] = u32x2_t{v[i].x, v[i].y};
          o[1] = u32x2_t{v[i].z, v[i].w};
        }
      }
    }
  };
  // rows row0 .. of a matrix; this lane's is row0 + r, its scales row ar of aux
  HX_DEV void init(const uint8_t* mat, int K, int row0, int r, int kq, int ar) {
    q = rsrc(mat + (int64_t)row0 * K, (uint32_t)(128 * K));   // at most 128 rows of a tile
    qo = (uint32_t)(r * K + 16 * ((kq >> 1) | ((kq & 1) << 1)));
    sc = (uint32_t)(ar * aux_row(K));
  }
  HX_DEV void load(int kc, Raw& w) const {
    w.q[0] = buf16(q, qo, (uint32_t)(kc * PD_K));
    w.q[1] = buf16(q, qo + 64, (uint32_t)(kc * PD_K));
  }
  // run u as loaded -> its codes + 128, words 0, 1: elements 64 u + 8 kq .. + 7 (step 2 u), words
  // 2, 3: 64 u + 32 + 8 kq .. (step 2 u + 1). permlane16_swap exchanges lane
  // groups 1 and 3 of its first operand with 0 and 2 of its second.
  HX_DEV static u32x4_t order(const Raw& w, int u) {
    const u32x4_t c = w.q[u] ^ 0x80808080u;
    const auto a = __builtin_amdgcn_permlane16_swap(c.x, c.z, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(c.y, c.w, false, false);
    return u32x4_t{a[0], b[0], a[1], b[1]};
  }
  // the scales of chunk kc of the window, a half a step
  HX_DEV u32x2_t scales(int kc, const uint8_t* aux) const { return *(const u32x2_t*)(aux + sc + 8 * kc); }
  // MFMA operand of step s: (1024 + 128 + code) as f16 by the 0x64 byte, minus
  // 1152 (exact), times the scale (one rounding)
  HX_DEV static f16x8_t frag(u32x4_t run, int s, u32x2_t scales) {
    const _Float16 sv = h2(scales[s >> 1])[s & 1];
    const h2_t sc2 = {sv, sv}, off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const uint32_t u = run[2 * (s & 1) + j];
      o[2 * j] = u32((h2(__builtin_amdgcn_perm(u, 0x64646464u, 0x00060004u)) + off) * sc2);
      o[2 * j + 1] = u32((h2(__builtin_amdgcn_perm(u, 0x64646464u, 0x00070005u)) + off) * sc2);
    }
    return __builtin_bit_cast(f16x8_t, u32x4_t{o[0], o[1], o[2], o[3]});
  }
};

// ---------------------------------------------------------------- the K loop
// LDS of a tile of MT sub-tiles: the rows' two buffers, then the scales of its
// 128 weight rows; a launch takes the largest tile's
constexpr int PD_NF = 2;   // column fragments a wave takes
HX_HD constexpr int pd_rows_bytes(int MT) { return 2 * 16 * MT * PD_LD * 2; }
template <class F>
static int pd_lds(int K) { return pd_rows_bytes(4) + 64 * PD_NF * F::aux_row(K); }

// acc[f][i] = 16 rows (sub-tile i) x this wave's 16 columns of fragment f, over
// K columns. rows(ap): the sources of this thread's pieces of the rows' chunk 0
// (thread t moves 16 bytes t % 16 of rows t / 16 + 16 i), called once the first
// weight loads are on their way; asrc: F::aux_src of this thread's weight row.
template <class F, int MT, class Rows>
HX_DEV void pd_gemm(uint8_t* lds, const F (&w)[PD_NF], int K, const uint8_t* asrc, Rows rows,
                    f32x4_t (&acc)[PD_NF][MT]) {
  constexpr int NF = PD_NF;
  const int tid = threadIdx.x, lane = lane_id(), l16 = lane & 15, kq = lane >> 4;
  const int r0 = tid >> 4, seg = tid & 15;
  uint16_t* As = (uint16_t*)lds;
  uint8_t* aux = lds + pd_rows_bytes(MT);
  const uint16_t* ap[MT];
  u32x4_t ar[MT];
  typename F::Raw b[2][NF];
#pragma unroll
  for (int f = 0; f < NF; f++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[f][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += F::WIN) {   // a window of scales at a time
    const int kw = min(F::WIN, K - k0), nk = kw / PD_K, kb = k0 / PD_K;
    auto load_a = [&](int kc) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < MT; i++) ar[i] = ld16(ap[i] + (kb + kc) * PD_K);
    };
    auto store_a = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < MT; i++) *(u32x4_t*)(As + (buf * 16 * MT + r0 + 16 * i) * PD_LD + 8 * seg) = ar[i];
    };
    auto load_b = [&](int kc, auto buf) __attribute__((always_inline)) {
#pragma unroll
      for (int f = 0; f < NF; f++) w[f].load(kb + kc, b[decltype(buf)::value][f]);
    };
    // (the last window's LDS reads ended at the loop's last barrier)
    load_b(0, ic<0>{});
    typename F::template Aux<64 * NF> av;
    av.load(asrc, k0, kw);
    __builtin_amdgcn_sched_barrier(0);
    if (k0 == 0) rows(ap);
    load_a(0);
    av.store(K, kw, aux);
    store_a(0);
    lds_barrier();
    auto step = [&](int kc, auto par) __attribute__((always_inline)) {
      constexpr int P = decltype(par)::value;
      if (kc + 1 < nk) {   // the rows first: waiting for them then leaves the weights in flight
        load_a(kc + 1);
        load_b(kc + 1, ic<1 - P>{});
      }
      __builtin_amdgcn_sched_barrier(0);
      u32x2_t sv[NF];
      u32x4_t run[NF];   // not back into b: its next loads would be waited for here
#pragma unroll
      for (int f = 0; f < NF; f++) sv[f] = w[f].scales(kc, aux);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        f16x8_t bf[NF];
        if (s % 2 == 0) {
#pragma unroll
          for (int f = 0; f < NF; f++) run[f] = F::order(b[P][f], s / 2);
        }
#pragma unroll
        for (int f = 0; f < NF; f++) bf[f] = F::frag(run[f], s, sv[f]);
#pragma unroll
        for (int i = 0; i < MT; i++) {
          const f16x8_t a =
              __builtin_bit_cast(f16x8_t, ld16(As + (P * 16 * MT + 16 * i + l16) * PD_LD + 32 * s + 8 * kq));
#pragma unroll
          for (int f = 0; f < NF; f++) acc[f][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bf[f], acc[f][i], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);   // one step's operands at a time: without it they spill
      }
      if (kc + 1 < nk) store_a(1 - P);
      lds_barrier();
    };
    for (int kc = 0; kc < nk; kc += 2) {   // nk is even
      step(kc, ic<0>{});
      step(kc + 1, ic<1>{});
    }
  }
}

// ---------------------------------------------------------------- gate/up
// 64 rows x (64 gate + 64 up columns), wave w owning columns 16 w .. + 15 of
// both (fragment 0: gate, 1: up)
template <class F, int MT>
HX_DEV void pd_gate_up(const ExpertArgs& a, uint8_t* lds, const uint8_t* G, const uint8_t* U, int I, int rows, int p0,
                       int nt, bool sh, bool qa) {
  constexpr int NC = 64;        // gate (and up) columns of the tile
  constexpr int OP = NC + 4;    // pitch of the f32 tile of h (aliases the LDS)
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, l16 = lane & 15, kq = lane >> 4;
  const int K = a.H, n0 = nt * NC;
  const uint16_t* X = qa ? a.xq : a.xh;
  // the rows' entries: read ahead of the first weight loads, used behind them
  int src[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) {
    const int p = p0 + min((tid >> 4) + 16 * i, rows - 1);   // padding rows repeat the last row
    src[i] = sh ? p : a.perm[p];
  }
  __builtin_amdgcn_sched_barrier(0);
  const int c = 16 * wave + l16;
  F w[PD_NF];
  w[0].init(G, K, n0, c, kq, c);
  w[1].init(U, K, n0, c, kq, NC + c);
  const uint8_t* asrc = F::aux_src(tid < 2 * NC ? G : U, I, K, n0 + (tid / 2) % NC);   // two threads a row
  f32x4_t acc[PD_NF][MT];
  pd_gemm<F, MT>(lds, w, K, asrc, [&](const uint16_t* (&ap)[MT]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; i++) ap[i] = X + (int64_t)(sh ? src[i] - a.F : src[i] / a.k) * K + 8 * (tid & 15);
  }, acc);
  // h through LDS, out 16 bytes a thread in the swizzled order: quantised arm
  // the f16 d q of its codes where the down weights are Q8_0 too (the tile
  // holds whole blocks of 32 columns; a kernel of its own with h in f32 out and
  // in again took 5 to 8 us), f32 in natural order for k_hq_fq where they are
  // not; else gate and up rounded to f16 and h in f16
  float* ot = (float*)lds;
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float g = acc[0][i][q], u = acc[1][i][q];
      // the product rounded once in either arm: through an f32 first, one in
      // 3,000 f16 values of h came out one step off
      float h;
      if (qa) h = siluf_(g) * u;
      else h = (float)(_Float16)(siluf_((float)(_Float16)g) * (float)(_Float16)u);
      ot[(16 * i + 4 * kq + q) * OP + c] = h;
    }
  lds_barrier();
  if (qa && a.down.fmt != HX_Q8_0) {
    const int c4 = 4 * (tid & 15);
#pragma unroll
    for (int i = 0, m = tid >> 4; i < MT; i++, m += 16)
      if (m < rows) *(float4*)(a.hbuf + (int64_t)(p0 + m) * a.hstride + n0 + c4) = *(const float4*)(ot + m * OP + c4);
    return;
  }
  const int c8 = 8 * (tid & 7);
#pragma unroll
  for (int m = tid >> 3; m < 16 * MT; m += 32) {   // 16 MT rows: whole waves, which quant_group needs
    const float4 u = *(const float4*)(ot + m * OP + c8), v = *(const float4*)(ot + m * OP + c8 + 4);
    const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
    float q[8], d;
    quant_group<HX_Q8_0>(x, q, d);
    _Float16 h[8];
#pragma unroll
    for (int j = 0; j < 8; j++) h[j] = qa ? fq_f16(q[j], d) : (_Float16)x[j];
    if (m < rows)
      *(u32x4_t*)(a.hbf + (int64_t)(p0 + m) * a.hstride + n0 + c8) =
          u32x4_t{u32(h2_t{h[0], h[2]}), u32(h2_t{h[1], h[3]}), u32(h2_t{h[4], h[6]}), u32(h2_t{h[5], h[7]})};
  }
}

// grid (I / 64, tiles rounded up to 8), mapped by xcd_tile; LDS pd_lds(H)
template <class F, int TS>
__global__ __launch_bounds__(256, 3) void k_gate_up_direct(ExpertArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  static_assert(4 * 16 * (64 + 4) <= pd_rows_bytes(1), "the tile of h fits the rows' LDS");
  int nt, tile, e, p0, rows, mc;
  xcd_tile(nt, tile);
  if (!get_tile<TS>(a, tile, e, p0, rows, mc)) return;
  const bool sh = e == a.E, qa = mc <= HX_QUANT_M;
  const uint8_t* G = sh ? a.sgate.base : a.gate.mat(e);
  const uint8_t* U = sh ? a.sup.base : a.up.mat(e);
  const int I = sh ? a.Is : a.I;
  switch ((rows + 15) >> 4) {   // uniform over the workgroup
    case 1: pd_gate_up<F, 1>(a, lds, G, U, I, rows, p0, nt, sh, qa); break;
    case 2: pd_gate_up<F, 2>(a, lds, G, U, I, rows, p0, nt, sh, qa); break;
    case 3: pd_gate_up<F, 3>(a, lds, G, U, I, rows, p0, nt, sh, qa); break;
    default: pd_gate_up<F, 4>(a, lds, G, U, I, rows, p0, nt, sh, qa); break;
  }
}

// ---------------------------------------------------------------- down
// 64 rows of h x 128 output columns, wave w owning columns 32 w .. + 31 (two
// fragments). Rows are scaled by their routing weight by position (f16 arm: the
// products rounded to f16 first) and written as bf16 to the per-assignment rows.
template <class F, int MT>
HX_DEV void pd_down(const ExpertArgs& a, uint8_t* lds, float* rws, const uint8_t* W, int K, int rows, int p0, int nt,
                    float rw, bool fa) {
  constexpr int NC = 128, OP = NC + 8;   // columns of the tile; pitch of the bf16 output tile (aliases the LDS)
  const int tid = threadIdx.x, lane = lane_id(), wave = tid >> 6, l16 = lane & 15, kq = lane >> 4;
  const int n0 = nt * NC, c = 32 * wave + l16;
  F w[PD_NF];
  w[0].init(W, K, n0, c, kq, c);
  w[1].init(W, K, n0, c + 16, kq, c + 16);
  f32x4_t acc[PD_NF][MT];
  pd_gemm<F, MT>(lds, w, K, F::aux_src(W, a.H, K, n0 + tid / 2),
                 [&](const uint16_t* (&ap)[MT]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < MT; i++)
      ap[i] = a.hbf + (int64_t)(p0 + min((tid >> 4) + 16 * i, rows - 1)) * a.hstride + 8 * (tid & 15);
  }, acc);
  if (tid < PM) rws[tid] = rw;
  lds_barrier();
  uint16_t* ot = (uint16_t*)lds;
#pragma unroll
  for (int i = 0; i < MT; i++) {
    const f32x4_t w4 = *(const f32x4_t*)(rws + 16 * i + 4 * kq);
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int f = 0; f < PD_NF; f++) {
        const float v = fa ? (float)(_Float16)acc[f][i][q] : acc[f][i][q];
        ot[(16 * i + 4 * kq + q) * OP + c + 16 * f] = f32_to_bf16(w4[q] * v);
      }
  }
  lds_barrier();
  const int c8 = 8 * (tid & 15);
#pragma unroll
  for (int i = 0, m = tid >> 4; i < MT; i++, m += 16)
    if (m < rows)
      *(u32x4_t*)((uint16_t*)a.obuf + (int64_t)(p0 + m) * a.H + n0 + c8) = ld16(ot + m * OP + c8);
}

// grid (H / 128, tiles rounded up to 8), mapped by xcd_tile; LDS pd_lds(I)
template <class F, int TS>
__global__ __launch_bounds__(256, 3) void k_down_direct(ExpertArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __shared__ __attribute__((aligned(16))) float rws[PM];
  static_assert(2 * 16 * (128 + 8) <= pd_rows_bytes(1), "the output tile fits the rows' LDS");
  int nt, tile, e, p0, rows, mc;
  xcd_tile(nt, tile);
  if (!get_tile<TS>(a, tile, e, p0, rows, mc)) return;
  const bool sh = e == a.E, fa = mc > HX_QUANT_M;
  const uint8_t* W = sh ? a.sdown.base : a.down.mat(e);
  const int K = sh ? a.Is : a.I;
  // a row's routing weight (the sigmoid gate of a shared row left to the combine: 1), used by the epilogue
  const float rw = threadIdx.x >= PM ? 0.f : sh && a.shared_raw ? 1.f : a.wpos[p0 + min((int)threadIdx.x, rows - 1)];
  switch ((rows + 15) >> 4) {   // uniform over the workgroup
    case 1: pd_down<F, 1>(a, lds, rws, W, K, rows, p0, nt, rw, fa); break;
    case 2: pd_down<F, 2>(a, lds, rws, W, K, rows, p0, nt, rw, fa); break;
    case 3: pd_down<F, 3>(a, lds, rws, W, K, rows, p0, nt, rw, fa); break;
    default: pd_down<F, 4>(a, lds, rws, W, K, rows, p0, nt, rw, fa); break;
  }
}

// ---------------------------------------------------------------- launchers
template <class F, int TS>
static void pd_launch(bool down, dim3 grid, const ExpertArgs& a, hipStream_t s) {
  if (down) hx_launch(k_down_direct<F, TS>, grid, dim3(256), pd_lds<F>(a.I), s, a);   // Is is I (or 0)
  else hx_launch(k_gate_up_direct<F, TS>, grid, dim3(256), pd_lds<F>(a.H), s, a);
}
template <class F>
static hipError_t pd_launch_ts(bool down, dim3 grid, const ExpertArgs& a, hipStream_t s) {
  switch (a.tsel) {
    case HX_TILES_ROUTED: pd_launch<F, HX_TILES_ROUTED>(down, grid, a, s); break;
    case HX_TILES_SHARED: pd_launch<F, HX_TILES_SHARED>(down, grid, a, s); break;
    default: pd_launch<F, HX_TILES_ALL>(down, grid, a, s); break;
  }
  return hipGetLastError();
}

hipError_t launch_gate_up_q8(const ExpertArgs& a, dim3 grid, hipStream_t s) {
  return pd_launch_ts<FragQ8>(false, grid, a, s);
}
hipError_t launch_down_q8(const ExpertArgs& a, dim3 grid, hipStream_t s) {
  return pd_launch_ts<FragQ8>(true, grid, a, s);
}

}  // namespace hx
