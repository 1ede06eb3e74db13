// Grouped GEMMs: one launch over many [N][K] weight blocks.
//
//  * experts (GG_UP / GG_DOWN): a row tile belongs to one expert (table built
//    on the device by moe_group, moe.hip, so a captured graph follows the
//    routing); the token rows are gathered while they are staged to LDS, the
//    up projection's epilogue applies the clamped gated activation, the down
//    projection's epilogue the routing weight, writing choice k of token t to
//    slab[k][t] -- the same slabs the next norm folds into the residual for
//    split-K projections (norm.hip), so combining costs no launch.  A shared
//    expert of other sizes is one more group of the same launch.
//  * heads (GG_BATCH): per-head projections into and out of the latent space
//    of latent attention (attention_latent.hip).
//
// bf16: MFMA 16x16x32, tiles staged HBM -> LDS by 16-byte LDS-DMA into a ring
// of k-steps (the scheme of gemm_ring in gemm.hip), 4 waves as 2 x 2.  Decode is bound by the
// stream of the experts' weights, prompts by the matrix cores; both lose what a block waits
// before its first loads, so W starts without the routing, and the routing weights of a down
// tile arrive under its products.  32 experts of 2048 x 1024 and a shared one of 2048, 4 a
// token: 64 tokens up 58 -> 46 us (6.1 TB/s), down 37 -> 33; 16000 tokens down 587 -> 504.
// fp32, for models served in it: two fp16 terms of every value on fp16 MFMAs, or three bf16 ones; where few rows
// leave the stream of the weights as the bound, MFMA 16x16x4 on fp32 operands with the bf16
// kernel's staging; VALU tiles with fused multiply-adds where K has no whole steps of 32 or a
// row starts off 16 bytes.
//
// A few tokens (single-stream decode): weight streaming instead of tiles, one
// wave per output column and (token, choice), no sorting by expert; the down
// projection sums a token's experts in the wave and adds into the residual.
#include "common.h"
#include "moe_params.h"

#include <type_traits>

namespace lsd {

namespace gg {
constexpr int BK = 64;
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void gbl_cvoid;

// Where one row tile's operands are.
struct Tile {
  const void* A; const void* W; void* out;
  long lda, ldw, ldo;
  int N, K, rows, row0;   // rows of the tile (<= TM) and its first row
  int n0;
  int group;              // expert / head whose weight block this is (shared expert: 0)
  float limit;
  bool routed, live;
};

// Logical workgroup -> (row tile, column tile): groups of `gr` row tiles walk the
// columns together, so a weight panel is re-read from L2 by its neighbours.  With
// few rows the group is the whole table: an XCD then takes a range of columns of
// every expert, and the unused end of the table costs all XCDs the same.
template <int MODE, int TM, int TN>
__device__ __forceinline__ Tile locate(const GgParams& p) {
  Tile t{};
  t.live = true;
  if constexpr (MODE == GG_UP || MODE == GG_DOWN) {
    // the shared expert's tiles first; shared and routed tiles are each spread over
    // all XCDs on their own (their K loops differ in length)
    const int tiles_s = (p.T + TM - 1) / TM, ntn_s = p.Ns > 0 ? (p.Ns + TN - 1) / TN : 0;
    const int grs = p.gr_s, shared = (tiles_s + grs - 1) / grs * grs * ntn_s;
    int bid = blockIdx.x;
    if (bid < shared) {
      bid = xcd_remap(bid, shared);
      const int gi = bid / (grs * ntn_s), rem = bid % (grs * ntn_s);
      const int tile = gi * grs + rem % grs;
      if (tile >= tiles_s) { t.live = false; return t; }
      t.A = p.As; t.lda = p.ldas; t.W = p.Ws; t.ldw = p.ldws; t.out = p.outs; t.ldo = p.ldos;
      t.N = p.Ns; t.K = p.Ks; t.row0 = tile * TM; t.rows = min(TM, p.T - tile * TM);
      t.n0 = (rem / grs) * TN;
      t.limit = p.limit_s;
      t.routed = false;
      return t;
    }
    const int gr = p.gr, ntn = (p.N + TN - 1) / TN;
    bid = xcd_remap(bid - shared, gridDim.x - shared);
    const int gi = bid / (gr * ntn), rem = bid % (gr * ntn);
    const int tile = gi * gr + rem % gr;
    if (tile >= p.n_tiles) { t.live = false; return t; }
    const int e = p.tiles[4 * tile], s0 = p.tiles[4 * tile + 1], n = p.tiles[4 * tile + 2];
    if (n == 0) { t.live = false; return t; }
    t.A = p.A; t.lda = p.lda; t.W = p.W; t.ldw = p.ldw; t.out = p.out; t.ldo = p.ldo;
    t.N = p.N; t.K = p.K; t.rows = n; t.row0 = s0;
    t.n0 = (rem / gr) * TN;
    t.group = e;
    t.limit = p.limit;
    t.routed = true;
    return t;
  } else {
    const int ntm = (p.M + TM - 1) / TM, ntn = (p.N + TN - 1) / TN;
    const int bid = xcd_remap(blockIdx.x, gridDim.x);
    const int g = bid / (ntm * ntn), rem = bid % (ntm * ntn);
    const int tm = rem % ntm;
    t.A = p.A; t.lda = p.lda; t.W = p.W; t.ldw = p.ldw; t.out = p.out; t.ldo = p.ldo;
    t.N = p.N; t.K = p.K; t.row0 = tm * TM; t.rows = min(TM, p.M - tm * TM);
    t.n0 = (rem / ntm) * TN;
    t.group = g;
    t.routed = true;
    return t;
  }
}

// Advance the operands to the tile's group (the element type is known here).
template <int MODE, typename T>
__device__ __forceinline__ void resolve(const GgParams& p, Tile& t) {
  const long g = t.group;
  if (t.routed) t.W = static_cast<const T*>(t.W) + g * p.w_gs;
  if constexpr (MODE == GG_BATCH) t.out = static_cast<T*>(t.out) + g * p.o_gs;
  if constexpr (MODE == GG_F32 || MODE == GG_ADD) t.out = static_cast<float*>(t.out) + g * p.o_gs;
  if constexpr (MODE != GG_UP && MODE != GG_DOWN) t.A = static_cast<const T*>(t.A) + g * p.a_gs;
}

// Source row of tile row i (clamped to a valid one).
template <int MODE>
__device__ __forceinline__ long a_row(const GgParams& p, const Tile& t, int i) {
  const int r = t.row0 + min(i, t.rows - 1);
  if constexpr (MODE == GG_UP) return t.routed ? p.perm[r] / p.top : r;
  return r;
}

// g = min(gate, limit), u = clamp(up, +-limit): g sigmoid(alpha g) (u + one).  SiLU
// gates have limit = infinity, alpha = 1 and one = 0.
__device__ __forceinline__ float glu_fast(float g, float u, float limit, float alpha, float one) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * alpha * g)) * (u + one);
}
__device__ __forceinline__ float glu_exact(float g, float u, float limit, float alpha, float one) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g / (1.f + expf(-alpha * g)) * (u + one);
}
__device__ __forceinline__ float sigmoid_fast(float z) {
  return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}
}  // namespace gg

template <int MODE, int TM, int TN, int SLOTS, int AUX = 0>
__global__ __launch_bounds__(256) void group_gemm_kernel(GgParams p) {
  using namespace gg;
  constexpr int MI = TM / 32, JT = TN / 32;  // 16 x 16 tiles per wave (2 x 2 waves)
  constexpr int A_BYTES = TM * BK * 2, SLOT_BYTES = (TM + TN) * BK * 2;
  constexpr int LPS = TM / 32 + TN / 32;     // LDS-DMA instructions per thread per k-step
  constexpr int LPA = TM / 32, D = SLOTS - 1;
  constexpr int CLD = TN + 4;
  constexpr int SMEM = SLOTS * SLOT_BYTES > TM * CLD * 4 ? SLOTS * SLOT_BYTES : TM * CLD * 4;
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  __shared__ int s_row[MODE == GG_DOWN ? TM : 1];   // GG_DOWN: slab row and weight of the tile's rows
  __shared__ float s_wt[MODE == GG_DOWN ? TM : 1];

  Tile t = locate<MODE, TM, TN>(p);
  if (!t.live) return;
  resolve<MODE, bf16>(p, t);
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const int wm = w >> 1, wn = w & 1, r = lane & 15, g = lane >> 4;

  // The ring is filled as early as each operand's addresses are known: W first, A behind the
  // row numbers it is gathered by.  Loads into registers between them only make the counted
  // waits below wait for more.
  const int KT = t.K / BK;
// Few rows: each column tile starts its sums at another k (512 bytes on), so that the blocks
  // under way do not all stand at the same place of rows that lie powers of two apart
  const int rot = MODE == GG_UP && TM == 32 ? t.n0 / TN * 4 % KT : 0;
  auto at_k = [&](int kt) { return (kt + rot >= KT ? kt + rot - KT : kt + rot) * BK; };
  const bf16* ap[TM / 32];
  const bf16* wp[TN / 32];
  long arow[TM / 32];
#pragma unroll
  for (int q = 0; q < TM / 32; ++q) arow[q] = a_row<MODE>(p, t, (w * (TM / 32) + q) * 8 + (lane >> 3));
  int ent = 0;  // GG_DOWN: the tile's row threadIdx.x
  if constexpr (MODE == GG_DOWN) {
    ent = t.row0 + min((int)threadIdx.x % TM, t.rows - 1);
    if (t.routed) ent = p.perm[ent];
  }
  // per-lane source addresses of this wave's LDS-DMA rows (16-byte chunks
  // XOR-swizzled on the source side, as in gemm.hip stage_tile)
#pragma unroll
  for (int q = 0; q < TN / 32; ++q) {
    const int row = (w * (TN / 32) + q) * 8 + (lane >> 3);
    wp[q] = static_cast<const bf16*>(t.W) + (long)min(t.n0 + row, t.N - 1) * t.ldw +
            (((lane & 7) ^ ((row >> 1) & 7)) << 3);
  }
  auto issue_w = [&](int kt, int slot) {
    char* b = smem + slot * SLOT_BYTES;
#pragma unroll
    for (int q = 0; q < TN / 32; ++q)
      __builtin_amdgcn_global_load_lds((gbl_cvoid*)(wp[q] + at_k(kt)),
                                       (lds_void*)(b + A_BYTES + (w * (TN / 32) + q) * 1024), 16, 0, AUX);
  };
  auto issue_a = [&](int kt, int slot) {
    char* b = smem + slot * SLOT_BYTES;
#pragma unroll
    for (int q = 0; q < TM / 32; ++q)
      __builtin_amdgcn_global_load_lds((gbl_cvoid*)(ap[q] + at_k(kt)), (lds_void*)(b + (w * (TM / 32) + q) * 1024), 16,
                                       0, 0);
  };
  auto frag = [&](const char* tile, int row, int chunk) {
    return *reinterpret_cast<const bf16x8*>(tile + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4));
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < KT) issue_w(d, d);
#pragma unroll
  for (int q = 0; q < TM / 32; ++q) {
    const int row = (w * (TM / 32) + q) * 8 + (lane >> 3);
    ap[q] = static_cast<const bf16*>(t.A) + arow[q] * t.lda + (((lane & 7) ^ ((row >> 1) & 7)) << 3);
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < KT) issue_a(d, d);
  float wt_row = 1.f;
  if constexpr (MODE == GG_DOWN) {
    if (t.routed) wt_row = p.wts[ent];
    else if (p.wts_s) wt_row = p.wts_s[ent];
  }
  f32x4 acc[MI][JT];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  int slot = 0, kt = 0;
  auto step = [&]() {
    const char* ta = smem + slot * SLOT_BYTES;
    const char* tw = ta + A_BYTES;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 af[MI], wf[JT];
#pragma unroll
      for (int i = 0; i < MI; ++i) af[i] = frag(ta, wm * 16 * MI + i * 16 + r, kk * 4 + g);
#pragma unroll
      for (int j = 0; j < JT; ++j) wf[j] = frag(tw, wn * (TN / 2) + j * 16 + r, kk * 4 + g);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < JT; ++j) acc[i][j] = mfma16(af[i], wf[j], acc[i][j]);
    }
    slot = slot == SLOTS - 1 ? 0 : slot + 1;
  };
  auto turn = [&](bool more) {
    __builtin_amdgcn_s_barrier();  // every wave's part of k-step kt has landed; step kt - 1 is read
    if (more) {
      issue_a(kt + D, slot == 0 ? SLOTS - 1 : slot - 1);
      issue_w(kt + D, slot == 0 ? SLOTS - 1 : slot - 1);
    }
    step();
    ++kt;
  };
  if constexpr (D == 1) {
    while (kt < KT) {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
      turn(kt + 1 < KT);
    }
  } else {
    // The first waits: behind A of k-step kt are A of the filled steps after it and all of the
    // steps issued since
    count_down<D - 1>([&](auto ic) {
      constexpr int d = decltype(ic)::v + 1;  // filled steps after kt
      if (kt + D < KT) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPA * d + LPS * (D - 1 - d)));
        turn(true);
      }
    });
    while (kt + D < KT) {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPS * (D - 1)));
      turn(true);
    }
    count_down<D>([&](auto ic) {  // the last D steps, nothing left to issue
      constexpr int d = decltype(ic)::v;
      if (KT - 1 - kt == d) {
        if (KT >= 2 * D) __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPS * d));
        else __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPA * d));  // filled ones: A alone is behind
        turn(false);
      }
    });
  }
  if constexpr (MODE == GG_DOWN) {
    if (threadIdx.x < TM) {
      s_row[threadIdx.x] = t.routed ? (ent % p.top) * p.T + ent / p.top : ent;  // < top * T, checked on the host to fit
      s_wt[threadIdx.x] = wt_row;
    }
  }
  __syncthreads();

  // epilogue through LDS: row-contiguous 16-byte stores
  float* ct = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < JT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        ct[(wm * 16 * MI + i * 16 + 4 * g + q) * CLD + wn * (TN / 2) + j * 16 + r] = acc[i][j][q];
  __syncthreads();
  constexpr int CPR = TN / 8;
  for (int c = threadIdx.x; c < TM * CPR; c += 256) {
    const int row = c / CPR, ch = c % CPR, n = t.n0 + ch * 8;
    if (row >= t.rows || n >= t.N) continue;
    const float* src = ct + row * CLD + ch * 8;
    const int m = t.row0 + row;
    if constexpr (MODE == GG_UP) {
      // gate and up rows interleaved in 16-row blocks: [gate16 | up16]
      if ((ch & 3) >= 2) continue;
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f2bf(glu_fast(src[e], src[16 + e], t.limit, p.alpha, p.up_one));
      st8(static_cast<bf16*>(t.out) + (long)m * t.ldo + (n >> 5) * 16 + (n & 15), o);
    } else if constexpr (MODE == GG_DOWN) {
      const long orow = s_row[row];
      const float wt = s_wt[row];
      if (p.slab_bf16) {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf(src[e] * wt);
        st8(static_cast<bf16*>(t.out) + orow * t.ldo + n, o);
      } else {
        f32x4* o = reinterpret_cast<f32x4*>(static_cast<float*>(t.out) + orow * t.ldo + n);
        o[0] = f32x4{src[0] * wt, src[1] * wt, src[2] * wt, src[3] * wt};
        o[1] = f32x4{src[4] * wt, src[5] * wt, src[6] * wt, src[7] * wt};
      }
    } else {
      bf16x8 o;
      if (p.gate) {
        const float* gt = p.gate + m * p.ldg + t.group * p.o_gs + n;
        const f32x4 ga = *reinterpret_cast<const f32x4*>(gt), gb = *reinterpret_cast<const f32x4*>(gt + 4);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf(src[e] * sigmoid_fast(e < 4 ? ga[e & 3] : gb[e & 3]));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f2bf(src[e]);
      }
      st8(static_cast<bf16*>(t.out) + (long)m * t.ldo + n, o);
    }
  }
}

// Results of a tile from its fp32 image in LDS, rows of TN + 4.
template <int MODE, int TM, int TN, int NT = 256>
__device__ __forceinline__ void f32_epilogue(const GgParams& p, const gg::Tile& t, const float* ct) {
  using namespace gg;
  constexpr int CLD = TN + 4;
  constexpr int CPR = TN / 4;
  // 16-byte stores (16 heads of 565 x 512 x 128 22.3 -> 20.2 us), or single ones into rows of any width
  const bool whole = (t.N | (int)t.ldo) % 4 == 0 && reinterpret_cast<uintptr_t>(t.out) % 16 == 0;
  for (int c = threadIdx.x; c < min(TM, t.rows) * CPR; c += NT) {
    const int row = c / CPR, ch = (c % CPR) * 4, n = t.n0 + ch, m = t.row0 + row;
    if (n >= t.N) continue;
    const float* src = ct + row * CLD + ch;
    f32x4 v = *reinterpret_cast<const f32x4*>(src);
    if constexpr (MODE == GG_UP) {  // gate and up rows in 16-row blocks; N % 32 == 0
      if (ch & 16) continue;
      const f32x4 u = *reinterpret_cast<const f32x4*>(src + 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = glu_exact(v[e], u[e], t.limit, p.alpha, p.up_one);
      *reinterpret_cast<f32x4*>(static_cast<float*>(t.out) + (long)m * t.ldo + (n >> 5) * 16 + (n & 15)) = v;
      continue;
    }
    long orow = m;
    float wt = 1.f;
    if constexpr (MODE == GG_DOWN) {
      if (t.routed) {
        const int ent = p.perm[m];
        wt = p.wts[ent];
        orow = (long)(ent % p.top) * p.T + ent / p.top;
      } else if (p.wts_s) {
        wt = p.wts_s[m];
      }
    }
    float* o = static_cast<float*>(t.out) + orow * t.ldo + n;
    if (whole) {
      if constexpr (MODE == GG_DOWN) v *= wt;
      else if constexpr (MODE == GG_ADD) v += *reinterpret_cast<const f32x4*>(o);
      else if constexpr (MODE == GG_F32)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float gt = p.gate ? 1.f / (1.f + expf(-p.gate[m * p.ldg + t.group * p.o_gs + n + e])) : 1.f;
          v[e] = (v[e] + (p.bias ? p.bias[n + e] : 0.f)) * gt;
        }
      *reinterpret_cast<f32x4*>(o) = v;
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // single stores: rows of any width
      if (n + e >= t.N) break;
      if constexpr (MODE == GG_DOWN) o[e] = v[e] * wt;
      else if constexpr (MODE == GG_ADD) o[e] += v[e];
      else if constexpr (MODE == GG_F32) {
        const float gt = p.gate ? 1.f / (1.f + expf(-p.gate[m * p.ldg + t.group * p.o_gs + n + e])) : 1.f;
        o[e] = (v[e] + (p.bias ? p.bias[n + e] : 0.f)) * gt;
      }
      else o[e] = v[e];
    }
  }
}

// fp32: 16 MT x 64 tiles, 32-deep k-steps (128-byte rows, the bf16 kernel's staging and swizzle);
// wave w owns 16 columns of all rows and leaves out the 16-row tiles that hold none, so an
// expert's last rows cost what they are.  A lane's 16-byte fragment feeds four MFMA 16x16x4,
// whose k-slot g stands for k = 4 g + j in both operands.
// For few rows, bound by the latency and the stream of the weights.
// ADDR64: 64-bit addresses, for few rows and for those that 32 bits do not reach (gg_f32).
template <int MODE, int MT, bool ADDR64>
__global__ __launch_bounds__(256, MT == 2 ? 4 : 3) void group_gemm_f32_mfma_kernel(GgParams p) {
  using namespace gg;
  constexpr int TM = 16 * MT, TN = 64, BKF = 32, SLOTS = 3;
  constexpr int A_BYTES = TM * 128, SLOT_BYTES = (TM + TN) * 128, LPS = TM / 32 + TN / 32, CLD = TN + 4;
  constexpr int SMEM = SLOTS * SLOT_BYTES > TM * CLD * 4 ? SLOTS * SLOT_BYTES : TM * CLD * 4;
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  Tile t = locate<MODE, TM, TN>(p);
  if (!t.live) return;
  resolve<MODE, float>(p, t);
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int live = __builtin_amdgcn_readfirstlane((t.rows + 15) / 16);

  // bytes of rows from the tile's first one, of gathered ones from the first of all
  typedef std::conditional_t<ADDR64, long, unsigned> Off;
  const long r0 = MODE == GG_UP && t.routed ? 0 : t.row0;
  const float* ab = static_cast<const float*>(t.A) + r0 * t.lda;
  const float* wb = static_cast<const float*>(t.W) + (long)t.n0 * t.ldw;
  Off ao[TM / 32], wo[TN / 32];
#pragma unroll
  for (int q = 0; q < TM / 32; ++q) {
    const int row = (w * (TM / 32) + q) * 8 + (lane >> 3);
    ao[q] = (Off)((a_row<MODE>(p, t, row) - r0) * t.lda * 4) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int q = 0; q < TN / 32; ++q) {
    const int row = (w * (TN / 32) + q) * 8 + (lane >> 3);
    wo[q] = (Off)(min(row, t.N - 1 - t.n0) * t.ldw * 4) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
  }
  auto dma = [&](const float* base, char* to, Off off, int k) {
    if constexpr (ADDR64)
      __builtin_amdgcn_global_load_lds((gbl_cvoid*)(reinterpret_cast<const char*>(base) + off + k), (lds_void*)to, 16, 0, 0);
    else
      lds_dma16(base, to, off, k);
  };
  auto issue = [&](int kt, int slot) {
    char* b = smem + slot * SLOT_BYTES;
#pragma unroll
    for (int q = 0; q < TM / 32; ++q) dma(ab, b + (w * (TM / 32) + q) * 1024, ao[q], kt * BKF * 4);
#pragma unroll
    for (int q = 0; q < TN / 32; ++q) dma(wb, b + A_BYTES + (w * (TN / 32) + q) * 1024, wo[q], kt * BKF * 4);
  };
  auto frag = [&](const char* tile, int row, int chunk) {
    return *reinterpret_cast<const f32x4*>(tile + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4));
  };
  f32x4 acc[2][MT];  // halves of the sums: a chain half as long rounds less
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[0][i] = acc[1][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));  // the routing loads are done before loads are counted
  const int KT = t.K / BKF;
#pragma unroll
  for (int d = 0; d < SLOTS; ++d)
    if (d < KT) issue(d, d);
  // k-step kt has landed for all waves, whose reads of the one before are done
  auto landed = [&](int kt) {
    constexpr int NO_LDS = ~0xf00;  // and no LDS read under way
    const int later = min(SLOTS - 1 - (kt > 0), KT - 1 - kt);
    if (later == 2) __builtin_amdgcn_s_waitcnt(vmcnt_imm(2 * LPS) & NO_LDS);
    else if (later == 1) __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPS) & NO_LDS);
    else __builtin_amdgcn_s_waitcnt(vmcnt_imm(0) & NO_LDS);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // L: row tiles that hold rows (a branch per tile would keep the fragments' loads apart).
  // Half a step's fragments are read while the other half is multiplied
  auto steps = [&](auto L) {
    f32x4 wf[2], af[2][L];
    auto read = [&](int slot, int kk) {
      const char* ta = smem + slot * SLOT_BYTES;
      wf[kk] = frag(ta + A_BYTES, w * 16 + r, kk * 4 + g);
#pragma unroll
      for (int i = 0; i < L; ++i) af[kk][i] = frag(ta, i * 16 + r, kk * 4 + g);
      __builtin_amdgcn_sched_barrier(0);
    };
    auto products = [&](int kk) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < L; ++i)
          acc[kk][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[kk][i][e], wf[kk][e], acc[kk][i], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    };
    landed(0);
    read(0, 0);
    int slot = 0;
    for (int kt = 0; kt < KT; ++kt) {
      read(slot, 1);
      products(0);
      const int next = slot == SLOTS - 1 ? 0 : slot + 1;
      if (kt + 1 < KT) {
        landed(kt + 1);
        if (kt + SLOTS < KT) issue(kt + SLOTS, slot);
        read(next, 0);
      }
      products(1);
      slot = next;
    }
  };
  if constexpr (MT == 4) {
    if (live == 4) steps(std::integral_constant<int, 4>{});
    else if (live == 3) steps(std::integral_constant<int, 3>{});
  }
  if (live == 2) steps(std::integral_constant<int, 2>{});
  else if (live == 1) steps(std::integral_constant<int, 1>{});
  __syncthreads();
  float* ct = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) ct[(i * 16 + 4 * g + q) * CLD + w * 16 + r] = acc[0][i][q] + acc[1][i][q];
  __syncthreads();
  f32_epilogue<MODE, TM, TN>(p, t, ct);
}

// ---------------------------------------------------------------------------
// fp32 on the 16-bit matrix cores
// ---------------------------------------------------------------------------
// x = hi + mid + lo, each bf16: of 24 bits the first two, rounded to nearest, leave rests of 16 and 8
// bits, so nothing is lost from 2^-110 on (below, lo is subnormal).  big: the largest |x|.  (Dot products with
// (-1, 0) and (0, -1) would unpack and subtract at once, but keep the MFMAs of other waves waiting.)
struct Split {
  bf16x4 t[3];
};
__device__ __forceinline__ Split split3(f32x4 x, float& big) {
  big = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), big);
  big = fmaxf(fmaxf(fabsf(x[2]), fabsf(x[3])), big);
  Split s;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bf16x2 a = pack2(x[0], x[1]), b = pack2(x[2], x[3]);
    s.t[i] = __builtin_shufflevector(a, b, 0, 1, 2, 3);
    if (i == 2) break;
    const unsigned ua = __builtin_bit_cast(unsigned, a), ub = __builtin_bit_cast(unsigned, b);
    x[0] -= __builtin_bit_cast(float, ua << 16);
    x[1] -= __builtin_bit_cast(float, ua & 0xffff0000u);
    x[2] -= __builtin_bit_cast(float, ub << 16);
    x[3] -= __builtin_bit_cast(float, ub & 0xffff0000u);
  }
  return s;
}

// The parts' images of a tile are whole in LDS: their sum, and the results.  WAVES a part.
template <int MODE, int TM, int TN, int WAVES, int WK>
__device__ __forceinline__ void parts_out(const GgParams& p, const gg::Tile& t, float* ct) {
  constexpr int IMAGE = TM * (TN + 4);
  __syncthreads();
  if constexpr (WK > 1) {
    for (int c = threadIdx.x; c < IMAGE / 4; c += 64 * WAVES * WK) {
      f32x4* o = reinterpret_cast<f32x4*>(ct) + c;
#pragma unroll
      for (int i = 1; i < WK; ++i) *o += o[i * (IMAGE / 4)];
    }
    __syncthreads();
  }
  f32_epilogue<MODE, TM, TN, 64 * WAVES * WK>(p, t, ct);
}

// What follows the products on three terms, S the tile's sums.  Terms behind bf16's numbers are lost: of an operand, 2^-134 at
// most.  Where that may count the tile is computed again by fp32 MFMAs, in the order of the kernel above: an operand of 2^56 or
// more (outside), a sum that is not finite, one below 2^-40.  Zeros among these stand where all of their column are and its first
// weights too, as padding's; looking through all of a column's weights took 10 to 50 us of a launch with padding.
template <int MODE, int MT, int WN, int WK>
__device__ __forceinline__ void split_tail(const GgParams& p, const gg::Tile& t, char* smem, f32x4 (&S)[MT], int first, int T, bool outside) {
  using namespace gg;
  constexpr int TM = 16 * MT, TN = 16 * WN, BKF = 32, CLD = TN + 4, IMAGE = TM * CLD;
  constexpr bool WHOLE = MODE == GG_F32 || MODE == GG_ADD;
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int w = wave % WN, part = wave / WN;
  const int live = __builtin_amdgcn_readfirstlane((t.rows + 15) / 16);
  const float* wp = static_cast<const float*>(t.W) + (long)min(t.n0 + w * 16 + r, t.N - 1) * t.ldw + first * BKF + 4 * g;
  bool exact = outside;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v = fabsf(S[i][q]);
      exact |= !(v >= 0x1p-40f && v < INFINITY) && (WHOLE || i < live);
    }
  exact = __syncthreads_or(exact);
  if (exact) {  // for zeros alone only where the column has other sums, or W values in the part's first k-step
    int zero = 0, other = 0, some = outside;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float v = fabsf(S[i][q]);
        zero |= v == 0.f && (WHOLE || i < live);
        other |= v > 0.f;
        some |= !(v < INFINITY) || (v < 0x1p-40f && v > 0.f);
      }
    zero |= __shfl_xor(zero, 16);
    zero |= __shfl_xor(zero, 32);
    if (zero && T > 0) {
      const f32x4 u = *reinterpret_cast<const f32x4*>(wp), v = *reinterpret_cast<const f32x4*>(wp + 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) other |= u[e] != 0.f || v[e] != 0.f;
    }
    exact = __syncthreads_or(some || (zero && other));
  }
  if (exact) {
#pragma unroll 1
    for (int i = 0; i < live; ++i) {
      const float* a = static_cast<const float*>(t.A) + a_row<MODE>(p, t, i * 16 + r) * t.lda + first * BKF + 4 * g;
      f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
      for (int k = 0; k < T * BKF; k += BKF)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x4 av = *reinterpret_cast<const f32x4*>(a + k + 16 * h), wv = *reinterpret_cast<const f32x4*>(wp + k + 16 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) s[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], wv[e], s[h], 0, 0, 0);
        }
#pragma unroll
      for (int h = 0; h < MT; ++h)
        if (h == i) S[h] = s[0] + s[1];
    }
  }
  float* ct = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) ct[part * IMAGE + (i * 16 + 4 * g + q) * CLD + w * 16 + r] = S[i][q];
  parts_out<MODE, TM, TN, WN, WK>(p, t, ct);
}

// 16 MT x 16 WN tiles, 32-deep k-steps, WK parts of the k-steps on WN waves each, summed in LDS.
// Of the nine products of two split operands the six largest are summed (the others are below 2^-26 of
// it), hi hi apart from the rest, whose sums round at 2^-8 of theirs.  A goes through registers into three
// LDS planes, split once a block; W, whose columns no two waves share, straight into fragments.
// Slot g of a fragment's k stands for 4 g + (0..3) and 16 + 4 g + (0..3), in both operands.
// Off 64 bits by half and less of what fp32 MFMAs are, whose sums round every four products: K = 2048
// 2.7e-7 and 5.7e-7 of the result, parts of K 1.3e-7 and 1.9e-7; K = 5632 4.7e-7 and 9.5e-7; SiLU of two
// 4.2e-7 and 8.5e-7.
// Bound by the matrix cores (six MFMAs at sixteen times the fp32 rate) and the splitting beside them
// (22 issue cycles a value, which a tile's rows and columns share), and by what a k-step waits for: hence
// parts of K where blocks are few, and 16 columns a wave, so that four waves share a SIMD (32 columns,
// two waves: experts below 282 and 133 us).  Against fp32 MFMAs: 565 x 2048 x 2048 59 -> 43 us, 565 x 2560 x
// 2048 63 -> 49, 100 x 2048 x 2048 29 -> 23, 1000 x 11264 x 2048 390 -> 286; 2260 rows over 32 experts of
// 2048 x 1024 and 565 through a shared one of 2048 up 325 -> 244, down 152 -> 121.  Splitting W a k-step
// ahead, beside the MFMAs, gives nothing: MFMAs and splitting take turns to issue.
// (A maximum of W's values beside the one of both took 20 % of the products.)
template <int MODE, int MT, int WN, int WK, int D>
__global__ __launch_bounds__(64 * WN * WK, WN == 8 ? 4 : 1) void group_gemm_f32_split_kernel(GgParams p) {
  using namespace gg;
  constexpr int TM = 16 * MT, TN = 16 * WN, BKF = 32, CLD = TN + 4, PLANE = TM * 64, SLOT = 3 * PLANE;
  constexpr int RA = 8 * WN, QA = (TM + RA - 1) / RA;  // rows of A that a part's threads bring at a time
  constexpr int IMAGE = TM * CLD, SMEM = WK * (2 * SLOT > IMAGE * 4 ? 2 * SLOT : IMAGE * 4);
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  Tile t = locate<MODE, TM, TN>(p);
  if (!t.live) return;
  resolve<MODE, float>(p, t);
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int w = wave % WN, part = wave / WN, tid = threadIdx.x % (64 * WN);
  const int live = __builtin_amdgcn_readfirstlane((t.rows + 15) / 16);
  // this part's k-steps; the first part has as many as any
  const int KT = t.K / BKF, most = (KT + WK - 1) / WK, first = part * most, T = max(0, min(most, KT - first));
  // A: thread i has four k's of rows i / 8, i / 8 + RA ..; W: this lane's column of each 16
  const int ar = tid >> 3, ac = tid & 7;
  const float* ap[QA];
#pragma unroll
  for (int q = 0; q < QA; ++q)
    ap[q] = static_cast<const float*>(t.A) + a_row<MODE>(p, t, ar + RA * q) * t.lda + first * BKF + 4 * ac;
  const float* wp = static_cast<const float*>(t.W) + (long)min(t.n0 + w * 16 + r, t.N - 1) * t.ldw + first * BKF + 4 * g;
  auto at = [&](int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 1) & 3)) << 4); };  // in a plane

  f32x4 acc[2][MT];  // hi hi, the others
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[0][i] = acc[1][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  float big = 0.f;
  f32x4 ra[D][QA], rw[D][2];
  auto load = [&](int kt, f32x4 (&a)[QA], f32x4 (&b)[2]) {  // (behind the last k-step: that one again)
    const long k = (long)min(kt, T - 1) * BKF;
#pragma unroll
    for (int q = 0; q < QA; ++q) a[q] = *reinterpret_cast<const f32x4*>(ap[q] + k);
    b[0] = *reinterpret_cast<const f32x4*>(wp + k);
    b[1] = *reinterpret_cast<const f32x4*>(wp + k + 16);
  };
  char* const slots = smem + part * 2 * SLOT;
  auto put_a = [&](int slot, const f32x4 (&a)[QA]) {  // chunk g: k's 4 g and 16 + 4 g
    char* b = slots + slot * SLOT;
#pragma unroll
    for (int q = 0; q < QA; ++q) {
      if (TM % RA && q == QA - 1 && ar + RA * q >= TM) break;
      const Split s = split3(a[q], big);
#pragma unroll
      for (int i = 0; i < 3; ++i)
        st4(reinterpret_cast<bf16*>(b + i * PLANE + at(ar + RA * q, ac & 3) + (ac >> 2) * 8), s.t[i]);
    }
  };
  auto steps = [&](auto L) {
    bf16x8 wf[3];
    auto step = [&](int kt, int set) {
      __syncthreads();  // A of k-step kt is in its slot, the other one's reads are done
      if (WK > 1 && kt >= T) return;
      const char* b = slots + (kt & 1) * SLOT;
      const Split x = split3(rw[set][0], big), y = split3(rw[set][1], big);
#pragma unroll
      for (int c = 0; c < 3; ++c) wf[c] = __builtin_shufflevector(x.t[c], y.t[c], 0, 1, 2, 3, 4, 5, 6, 7);
      load(kt + D, ra[set], rw[set]);
#pragma unroll
      for (int i0 = 0; i0 < L; i0 += 2) {  // two tiles at a time: independent chains
        constexpr int ca[6] = {0, 0, 1, 1, 0, 2}, cw[6] = {0, 1, 0, 1, 2, 0};
        bf16x8 af[2][3];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int i = i0; i < min((int)L, i0 + 2); ++i)
            af[i - i0][c] = *reinterpret_cast<const bf16x8*>(b + c * PLANE + at(i * 16 + r, g));
#pragma unroll
        for (int c = 0; c < 6; ++c)
#pragma unroll
          for (int i = i0; i < min((int)L, i0 + 2); ++i)
            acc[c > 0][i] = mfma16(af[i - i0][ca[c]], wf[cw[c]], acc[c > 0][i]);
      }
      put_a(~kt & 1, ra[(set + 1) % D]);
    };
    int kt = 0;
    for (; kt + D <= most; kt += D)
#pragma unroll
      for (int d = 0; d < D; ++d) step(kt + d, d);
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
      if (kt + d < most) step(kt + d, d);
  };
  if (WK == 1 || T > 0) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, ra[d], rw[d]);
    put_a(0, ra[0]);
  }
  count_down<MT>([&](auto ic) {
    constexpr int l = decltype(ic)::v + 1;
    if (MODE == GG_UP || MODE == GG_DOWN ? live == l : l == MT) steps(std::integral_constant<int, l>{});
  });
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[0][i] += acc[1][i];
  split_tail<MODE, MT, WN, WK>(p, t, smem, acc[0], first, T, big >= 0x1p56f);
}

// Long sums, on two fp16 terms: scale x = hi + lo / 2048, both rounded to nearest: off by up to 2^-24 of x or, below
// 2^-12 / scale, 2^-36 / scale, hi infinite from 65520 / scale on.  most: the largest |x|.
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
constexpr float LO = 2048.f, SCALE_A = 4.f, SCALE_W = 256.f;
__device__ __forceinline__ void split2(f32x4 x, float scale, f16x4& hi, f16x4& lo, float& most) {
  most = fmaxf(fmaxf(fabsf(x[0]), fabsf(x[1])), most);
  most = fmaxf(fmaxf(fabsf(x[2]), fabsf(x[3])), most);
#pragma unroll
  for (int e = 0; e < 4; ++e) hi[e] = (_Float16)__builtin_fmaf(x[e], scale, 0.f);
  asm("" : "+v"(hi));  // (pairs as they are: otherwise every second one is converted again for its rest)
#pragma unroll
  for (int e = 0; e < 4; ++e) lo[e] = (_Float16)__builtin_fmaf(__builtin_fmaf(x[e], scale, -(float)hi[e]), LO, 0.f);
}

template <int N, class F>
__device__ __forceinline__ void count_up(F f) {  // f(0) .. f(N - 1)
  if constexpr (N > 0) {
    count_up<N - 1>(f);
    f(Int<N - 1>{});
  }
}

// Sums of one 16 x 16 tile by fp32 MFMAs, in eight chains, or they would be further off than three bf16 terms' (two chains 7.9e-7 of
// the result, K = 2048, eight 4.0e-7, three terms 4.05e-7); a, w: this lane's row and column at its k's.  AHEAD k-steps' loads are
// on their way.
__device__ __forceinline__ f32x4 fp32_sums(const float* a, const float* w, int steps) {
  constexpr int AHEAD = 4;
  f32x4 s[2][4] = {}, av[AHEAD][2], wv[AHEAD][2];
  auto load = [&](int k, int at) {  // (behind the last one that one again)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      av[at][h] = *reinterpret_cast<const f32x4*>(a + min(k, steps - 1) * 32 + 16 * h);
      wv[at][h] = *reinterpret_cast<const f32x4*>(w + min(k, steps - 1) * 32 + 16 * h);
    }
  };
  auto add = [&](int at) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int h = 0; h < 2; ++h) s[h][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[at][h][e], wv[at][h][e], s[h][e], 0, 0, 0);
  };
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) load(k, k);
  int k0 = 0;
#pragma unroll 1
  for (; k0 + AHEAD <= steps; k0 += AHEAD)  // (whole groups: a way out between would have every load waited for)
#pragma unroll
    for (int k = 0; k < AHEAD; ++k) {
      add(k);
      __builtin_amdgcn_sched_barrier(0);
      load(k0 + k + AHEAD, k);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
  for (int k = 0; k < AHEAD - 1; ++k)
    if (k0 + k < steps) add(k);
  return ((s[0][0] + s[0][1]) + (s[0][2] + s[0][3])) + ((s[1][0] + s[1][1]) + (s[1][2] + s[1][3]));
}

// Sums of n products, n a multiple of 4, of a row and of C columns by a wave.
template <int C>
__device__ __forceinline__ void fp32_row(const float* a, const float* const (&w)[C], int n, float (&out)[C]) {
  const int at = 4 * lane_id();
  f32x4 s[C] = {};
#pragma unroll 4
  for (int k = 0; k < n; k += 256)
    if (k + at < n) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(a + k + at);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const f32x4 y = *reinterpret_cast<const f32x4*>(w[c] + k + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[c][e] = __builtin_fmaf(x[e], y[e], s[c][e]);
      }
    }
#pragma unroll
  for (int c = 0; c < C; ++c) out[c] = wave_sum((s[c][0] + s[c][1]) + (s[c][2] + s[c][3]));
}

// 16 MT WM x 16 NT WN tiles with half of the kernel above's products: hi hi, in two chains, and hi lo + lo hi.  A value takes 4
// operations to split instead of 6, which go on for the next k-step between this one's MFMAs; PF k-steps are loaded ahead of that.
// The two chains make up for what the terms leave out: off 64 bits by (before) K = 1024 1.65e-7 (1.94e-7) of the result, K = 2048
// 2.2e-7 (2.7e-7), in two parts 1.73e-7 (1.94e-7), in three 1.49e-7 (1.50e-7), K = 5632 3.5e-7 (4.7e-7), SiLU of two, K = 2048
// 3.4e-7 (4.3e-7); with one chain 2.2e-7 at K = 1024.  Shorter ones are left to the kernel above: K = 544 1.38e-7 (1.30e-7).
// Not so where sums round less than the terms: rows without negative values, K = 1024 1.7e-7 (1.4e-7), K = 2048 2.2e-7 (2.15e-7), in
// three parts 1.5e-7 (1.2e-7), K = 5632 3.5e-7 (3.9e-7); columns of 2 % of the weights, K = 2048 1.1e-7 (0.5e-7); a lone product 2^-23 at most (none).
// Bound by what a CU takes in.  W goes through LDS like A, in whole lines: loaded straight into fragments (16 rows of 64 bytes
// an instruction), 1000 x 11264 x 2048 on 64 x 128 took 230 us, without the splitting 216, without the MFMAs 200, without both 203,
// without loads behind the first ones 136; through LDS 208 to 225, and 176 on 128 x 128.  Waves of 32 x 32 read least from LDS.
// Against the kernel above: 500 x 1985 x 2048 40.3 -> 31.3 us, 565 x 2048 41.2 -> 31.5, 961 x 2048 58.3 -> 45.6, 565 x 4160 75 -> 48,
// 1000 x 11264 258 -> 176, 565 x 2624 51 -> 43; 2260 rows over 32 experts of 2048 x 1024 and 565 through a shared one of 2048 up
// 259 -> 201, down 126 -> 106, 5600 and 1400 rows 452 -> 356 and 245 -> 190.  For experts 96 rows a tile, the few rows behind
// a full one with it, were behind, with their registers at two waves a SIMD (up 472, down 240 with the most rows).
//
// The terms leave out at most 3 2^-24 of the sizes of the products, and 2^-38 and half as much again a product with a small value of
// A, 2^-44 with one of W: of K products 1.5 K (2^-38 of the column's largest weight + 2^-44 of the row's largest value).  Of a sum
// of 2^-13 of the one and 2^-19 of the other and more that is 3 K / 4 of its 2^-24.
// Where the sizes of a sum's two chains are together less than that it is computed again from the operands, and where it is not
// finite: by itself where a 16 x 16 tile has such sums in up to ROWS rows, by fp32 MFMAs where in more.  (By the size of the sum
// alone, every tenth tile of normal operands would have one, 3 us of a launch.)  A row or a column of zeros has zeros.
// Before that a tile with a value of 16376 in A or 256 in W is summed once more with powers of two for scales that hold its
// largest values, up to 2^60; what is small beside them is lost sooner, and the line above moves with it.  Not one of experts, whose
// registers are all taken (down products of 700 rows 80 -> 87 us, others up to 2 % faster and slower with the code for it).
// 961 x 2048 x 2048, us: normal operands 47 (three bf16 terms 58), a value of 20000 79 (58), one in every tenth row 87, in every
// row 81 (58; by fp32 MFMAs alone 272); rows of 2^-8 48.
template <int MODE, int WM, int MT, int WN, int NT, int WK, int PF, int OCC>
__global__ __launch_bounds__(64 * WM * WN * WK, OCC) void group_gemm_f32_half_kernel(GgParams p) {
  using namespace gg;
  constexpr int TM = 16 * MT * WM, TN = 16 * NT * WN, BKF = 32, CLD = TN + 4, PLANE = (TM + TN) * 64, SLOT = 2 * PLANE;
  constexpr int RQ = 8 * WM * WN, QA = (TM + RQ - 1) / RQ, QW = TN / RQ;  // rows that a part's threads bring at a time
  constexpr int IMAGE = TM * CLD, SMEM = WK * (2 * SLOT > IMAGE * 4 ? 2 * SLOT : IMAGE * 4);
  static_assert(TN % RQ == 0, "whole passes over W");
  __shared__ __attribute__((aligned(16))) char smem[SMEM];
  __shared__ float wmax[WK * TN];
  __shared__ __attribute__((aligned(16))) float amax[WK * TM];
  Tile t = locate<MODE, TM, TN>(p);
  if (!t.live) return;
  resolve<MODE, float>(p, t);
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int wn = wave % WN, wm = wave / WN % WM, part = wave / (WN * WM), tid = threadIdx.x % (64 * WM * WN);
  const int live = __builtin_amdgcn_readfirstlane((t.rows + 15) / 16) - wm * MT;  // of this wave's tiles
  // this part's k-steps; the first part has as many as any
  const int KT = t.K / BKF, most = (KT + WK - 1) / WK, first = part * most, T = max(0, min(most, KT - first));
  constexpr int UNITS = QW + QA;
  f32x4 acc[3][MT][NT];  // hi hi of even and of odd k-steps, 2048 times the others
  // All products with these scales; whether a value is beyond the terms'.  (mine: the thread, as addresses of its own: kept in
  // registers for another pass, they would have the loops' spilled)
  auto products = [&](float sa, float sw, int mine) {
    const int lane = mine & 63, r = lane & 15, g = lane >> 4;
    // thread i brings four k's of rows i / 8, i / 8 + RQ .. of W and of A: whole lines
    const int row = mine >> 3, ac = mine & 7;
    const float* src[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; ++u)
      src[u] = (u < QW ? static_cast<const float*>(t.W) + (long)min(t.n0 + row + RQ * u, t.N - 1) * t.ldw
                       : static_cast<const float*>(t.A) + a_row<MODE>(p, t, row + RQ * (u - QW)) * t.lda) + first * BKF + 4 * ac;
    auto at = [&](int row, int chunk) { return row * 64 + ((chunk ^ ((row >> 1) & 3)) << 4); };  // in a plane: W's rows, A's

#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[c][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int from = (MODE == GG_UP || MODE == GG_DOWN) && p.turn && T > 0 ? (t.n0 / TN * 11 + t.group * 7) % T : 0;
    float largest[UNITS] = {};
    f32x4 raw[PF][UNITS];
    char* const slots = smem + part * 2 * SLOT;
    auto load = [&](int u, int kt, int ring) {  // (behind the last k-step: that one again)
      const int k = min(kt, T - 1) + from;
      raw[ring][u] = *reinterpret_cast<const f32x4*>(src[u] + (long)(k >= T ? k - T : k) * BKF);
    };
    char* const put = slots + at(row, ac & 3) + (ac >> 2) * 8;  // chunk g: k's 4 g and 16 + 4 g (RQ rows on: the same chunk)
    auto part_up = [&](int u, int ring, int slot) {
      if (TM % RQ && u == UNITS - 1 && row + RQ * (QA - 1) >= TM) return;
      f16x4 hi, lo;
      split2(raw[ring][u], u < QW ? sw : sa, hi, lo, largest[u]);
      char* b = put + slot * SLOT + (u < QW ? RQ * u : TN + RQ * (u - QW)) * 64;
      *reinterpret_cast<u32x2*>(b) = __builtin_bit_cast(u32x2, hi);
      *reinterpret_cast<u32x2*>(b + PLANE) = __builtin_bit_cast(u32x2, lo);
    };
    auto steps = [&](auto L) {
      auto step = [&](int kt, auto unroll) {
        constexpr int U = decltype(unroll)::v, S = U & 1, R = (U + 1) % PF, GROUPS = L < 2 ? 1 : (L + 1) / 2;
        __syncthreads();  // k-step kt is in its slot, the other one's reads are done
        if (WK > 1 && kt >= T) return;
        const char* b = slots + S * SLOT;
        f16x8 wf[NT][2];
        if constexpr (L > 0) {
#pragma unroll
          for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int c = 0; c < 2; ++c) wf[j][c] = *reinterpret_cast<const f16x8*>(b + c * PLANE + at((wn * NT + j) * 16 + r, g));
        }
#pragma unroll
        for (int i0 = 0; i0 < 2 * GROUPS; i0 += 2) {
          f16x8 af[2][2];
#pragma unroll
          for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int i = i0; i < min((int)L, i0 + 2); ++i)
              af[i - i0][c] = *reinterpret_cast<const f16x8*>(b + c * PLANE + at(TN + (wm * MT + i) * 16 + r, g));
#pragma unroll
          for (int u = i0 / 2 * UNITS / GROUPS; u < (i0 / 2 + 1) * UNITS / GROUPS; ++u) {
            part_up(u, R, S ^ 1);
            load(u, kt + 1 + PF, R);
          }
#pragma unroll
          for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = i0; i < min((int)L, i0 + 2); ++i)
#pragma unroll
              for (int j = 0; j < NT; ++j) {
                f32x4& s = acc[c ? 2 : S][i][j];
                s = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[i - i0][c >> 1], wf[j][c & 1], s, 0, 0, 0);
              }
        }
        // an MFMA, a part of the splitting, and so on; a pair of tiles' reads in front of its first
        if constexpr (L > 0) {
          __builtin_amdgcn_sched_group_barrier(0x100, 2 * NT, 0);
#pragma unroll
          for (int i = 0; i < 3 * L * NT; ++i) {
            if (i % (6 * NT) == 0) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, (UNITS * 16 + 3 * L * NT - 1) / (3 * L * NT), 0);
          }
        }
      };
      int kt = 0;
      for (; kt + 2 <= most; kt += 2) count_up<2>([&](auto u) { step(kt + decltype(u)::v, u); });
      if (kt < most) step(kt, Int<0>{});
    };
    if (WK == 1 || T > 0) {
#pragma unroll
      for (int d = 0; d < PF; ++d)
#pragma unroll
        for (int u = 0; u < UNITS; ++u) load(u, d, d);
#pragma unroll
      for (int u = 0; u < UNITS; ++u) {
        part_up(u, 0, 0);
        load(u, PF, 0);
      }
    }
    if constexpr (MODE == GG_UP || MODE == GG_DOWN) {
      count_up<MT + 1>([&](auto ic) {
        constexpr int l = decltype(ic)::v;
        if (min(max(live, 0), MT) == l) steps(std::integral_constant<int, l>{});
      });
    } else {
      steps(std::integral_constant<int, MT>{});
    }
    bool over = false;
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {  // of a row's eight threads
      float& m = largest[u];
#pragma unroll
      for (int d = 1; d < 8; d *= 2) m = fmaxf(m, __shfl_xor(m, d));
      over |= !(m * (u < QW ? sw : sa) < 65504.f);
      const int at = row + RQ * (u < QW ? u : u - QW);
      if (ac == 0 && u < QW) wmax[part * TN + at] = m;
      if (ac == 0 && u >= QW && at < TM) amax[part * TM + at] = m;
    }
    return __syncthreads_or(over);  // (and every wave has read its last k-step)
  };
  float ua = 1.f / SCALE_A, uw = 1.f / SCALE_W;  // of the products' sums (powers of two)
  if (products(SCALE_A, SCALE_W, tid) && MODE != GG_UP && MODE != GG_DOWN) {  // once more with scales that hold the largest values
    float most_a = 0.f, most_w = 0.f;
    for (int c = lane; c < WK * TM; c += 64) most_a = fmaxf(most_a, amax[c]);
    for (int c = lane; c < WK * TN; c += 64) most_w = fmaxf(most_w, wmax[c]);
    most_a = wave_max(most_a);
    most_w = wave_max(most_w);
    if (most_a < 0x1p60f && most_w < 0x1p60f) {
      auto fit = [](float most, float unit) {  // most / unit below 2^15, or as it was
        const float to = __builtin_bit_cast(float, (__builtin_bit_cast(unsigned, most) >> 23) - 14 << 23);
        return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, most < 65504.f * unit ? unit : to)));
      };
      ua = fit(most_a, ua);
      uw = fit(most_w, uw);
      int mine = tid;
      asm volatile("" : "+v"(mine));
      products(1.f / ua, 1.f / uw, mine);
    }
  }
  constexpr int ROWS = 3;
  float* const ct = reinterpret_cast<float*>(smem) + part * IMAGE;
  const float unit = ua * uw;
  float least = INFINITY, odd = 0.f, line = 0x1p-24f * unit;  // of this lane's sums: the smallest size; zero where all are finite; the line's most
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const f32x4 av = *reinterpret_cast<const f32x4*>(amax + part * TM + (wm * MT + i) * 16 + 4 * g);
    line = fmaxf(fmaxf(fmaxf(av[0], av[1]), fmaxf(av[2], av[3])) * (uw * 0x1p-10f), line);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      line = fmaxf(wmax[part * TN + (wn * NT + j) * 16 + r] * (ua * 0x1p-10f), line);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float c0 = acc[0][i][j][q], c1 = acc[1][i][j][q], s = (c0 + c1 + acc[2][i][j][q] * (1.f / LO)) * unit;
        least = fminf(least, fabsf(c0) + fabsf(c1));
        odd = __builtin_fmaf(s, 0.f, odd);
        ct[((wm * MT + i) * 16 + 4 * g + q) * CLD + (wn * NT + j) * 16 + r] = acc[2][i][j][q] = s;
      }
    }
  }
  unsigned again = 0;  // row 4 g + q of tile (i, j), column r: bit (i NT + j) 4 + q where it is computed again
  if (__ballot(least * unit < line || odd != 0.f) != 0) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const f32x4 av = *reinterpret_cast<const f32x4*>(amax + part * TM + (wm * MT + i) * 16 + 4 * g);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const float wv = wmax[part * TN + (wn * NT + j) * 16 + r];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const bool few = (fabsf(acc[0][i][j][q]) + fabsf(acc[1][i][j][q])) * unit < fmaxf((wv * ua + av[q] * uw) * 0x1p-11f, 0x1p-24f * unit);
          const bool out = (wm * MT + i) * 16 + 4 * g + q < t.rows && t.n0 + (wn * NT + j) * 16 + r < t.N;
          again |= (unsigned)(out && ((few && wv > 0.f && av[q] > 0.f) || !(fabsf(acc[2][i][j][q]) < INFINITY))) << ((i * NT + j) * 4 + q);
        }
      }
    }
  }
  if (__ballot(again != 0) != 0 && T > 0) {
    const float* const A = static_cast<const float*>(t.A) + first * BKF;
    const float* const W = static_cast<const float*>(t.W) + first * BKF;
#pragma unroll 1
    for (int f = 0; f < MT * NT; ++f) {
      const int r0 = (wm * MT + f / NT) * 16, c0 = (wn * NT + f % NT) * 16;
      unsigned long long row[4];  // columns to be summed, of 16 bits for each of the rows q, 4 + q, 8 + q, 12 + q
      int rows = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        row[q] = __ballot(again >> (4 * f + q) & 1);
#pragma unroll
        for (int h = 0; h < 64; h += 16) rows += (row[q] >> h & 0xffff) != 0;
      }
      if (rows > ROWS) {
        const f32x4 s = fp32_sums(A + a_row<MODE>(p, t, r0 + r) * t.lda + 4 * g, W + (long)min(t.n0 + c0 + r, t.N - 1) * t.ldw + 4 * g, T);
#pragma unroll
        for (int q = 0; q < 4; ++q) ct[(r0 + 4 * g + q) * CLD + c0 + r] = s[q];
        continue;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll 1
        while (row[q]) {  // a column, or four of a row, the last ones the same
          const int h = __builtin_ctzll(row[q]) >> 4, at = r0 + 4 * h + q;
          const float* ar = A + a_row<MODE>(p, t, at) * t.lda;
          auto some = [&](auto count) {
            constexpr int C = decltype(count)::v;
            int col[C];
            const float* w[C];
            float s[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
              const unsigned left = row[q] >> 16 * h & 0xffff;
              col[c] = left ? __builtin_ctz(left) : col[0];
              if (left) row[q] &= row[q] - 1;
              w[c] = W + (long)(t.n0 + c0 + col[c]) * t.ldw;
            }
            fp32_row<C>(ar, w, T * BKF, s);
            if (lane == 0)
#pragma unroll
              for (int c = 0; c < C; ++c) ct[at * CLD + c0 + col[c]] = s[c];
          };
          if (__builtin_popcountll(row[q] >> 16 * h & 0xffff) > 1) some(Int<4>{});
          else some(Int<1>{});
        }
    }
  }
  parts_out<MODE, TM, TN, WM * WN, WK>(p, t, reinterpret_cast<float*>(smem));
}

// Rows without whole k-steps of 32 or off 16 bytes: 64 x 64 tiles, 4 x 4 outputs per thread, 16-deep k-steps.
template <int MODE>
__global__ __launch_bounds__(256) void group_gemm_f32_kernel(GgParams p) {
  using namespace gg;
  constexpr int TM = 64, TN = 64, KS = 16;
  __shared__ float as[KS][TM + 4];
  __shared__ float ws[KS][TN + 4];
  Tile t = locate<MODE, TM, TN>(p);
  if (!t.live) return;
  resolve<MODE, float>(p, t);
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  // loads: thread -> row tid / 4, four k at (tid % 4) * 4
  const int lr = threadIdx.x >> 2, lk = (threadIdx.x & 3) * 4;
  const float* ap = static_cast<const float*>(t.A) + a_row<MODE>(p, t, lr) * t.lda + lk;
  const float* wp = static_cast<const float*>(t.W) + (long)min(t.n0 + lr, t.N - 1) * t.ldw + lk;
  float acc[4][4] = {};
  for (int k0 = 0; k0 < t.K; k0 += KS) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(ap + k0);
    const f32x4 w = *reinterpret_cast<const f32x4*>(wp + k0);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      as[lk + j][lr] = a[j];
      ws[lk + j][lr] = w[j];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KS; ++k) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        av[i] = as[k][ty * 4 + i];
        // columns tx + 16 j: a gate column's up column (16 to the right in an
        // interleaved 32-row block) belongs to the same thread
        wv[i] = ws[k][tx + 16 * i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = ty * 4 + i;
    if (row >= t.rows) continue;
    const int m = t.row0 + row;
    if constexpr (MODE == GG_UP) {
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const int n = t.n0 + tx + 16 * j;
        if (n < t.N)
          static_cast<float*>(t.out)[(long)m * t.ldo + (n >> 5) * 16 + (n & 15)] =
              glu_exact(acc[i][j], acc[i][j + 1], t.limit, p.alpha, p.up_one);
      }
      continue;
    }
    long orow = m;
    float wt = 1.f;
    if constexpr (MODE == GG_DOWN) {
      if (t.routed) {
        const int ent = p.perm[m];
        wt = p.wts[ent];
        orow = (long)(ent % p.top) * p.T + ent / p.top;
      } else if (p.wts_s) {
        wt = p.wts_s[m];
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = t.n0 + tx + 16 * j;
      if (n >= t.N) continue;
      float* o = static_cast<float*>(t.out) + orow * t.ldo + n;
      if constexpr (MODE == GG_DOWN) *o = acc[i][j] * wt;
      else if constexpr (MODE == GG_ADD) *o += acc[i][j];
      else if constexpr (MODE == GG_F32) {
        const float gt = p.gate ? 1.f / (1.f + expf(-p.gate[m * p.ldg + t.group * p.o_gs + n])) : 1.f;
        *o = (acc[i][j] + (p.bias ? p.bias[n] : 0.f)) * gt;
      }
      else *o = acc[i][j];
    }
  }
}

// ---------------------------------------------------------------------------
// A few tokens: every (token, choice) streams its expert's weight rows
// ---------------------------------------------------------------------------
// One wave computes C gated columns of one (token, expert): 2 C weight rows,
// all lanes on consecutive 16-byte chunks.  Blocks of the shared expert first.
template <int C>
__global__ __launch_bounds__(256) void moe_gemv_up_kernel(MoeGemvParams p) {
  const int lane = lane_id(), w = threadIdx.x >> 6;
  const int nb_s = (p.Fs + 4 * C - 1) / (4 * C), nb = (p.F + 4 * C - 1) / (4 * C);
  int bid = blockIdx.x;
  const bf16 *W, *A;
  bf16* out;
  float limit;
  int F, c0;
  if (bid < nb_s * p.T) {
    const int t = bid / nb_s;
    c0 = (bid % nb_s) * 4 * C;
    A = static_cast<const bf16*>(p.h) + (long)t * p.K;
    W = static_cast<const bf16*>(p.ws);
    out = static_cast<bf16*>(p.mids) + (long)t * p.Fs;
    F = p.Fs;
    limit = p.limit_s;
  } else {
    bid -= nb_s * p.T;
    const int ent = bid / nb;
    c0 = (bid % nb) * 4 * C;
    A = static_cast<const bf16*>(p.h) + (long)(ent / p.top) * p.K;
    W = static_cast<const bf16*>(p.w) + (long)p.ids[ent] * 2 * p.F * p.K;
    out = static_cast<bf16*>(p.mid) + (long)ent * p.F;
    F = p.F;
    limit = p.limit;
  }
  c0 += w * C;
  if (c0 >= F) return;  // wave-uniform, no barriers
  const bf16* wr[2 * C];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int c = min(c0 + j, F - 1);
    wr[2 * j] = W + (long)((c >> 4) * 32 + (c & 15)) * p.K;
    wr[2 * j + 1] = wr[2 * j] + 16L * p.K;
  }
  float acc[2 * C] = {};
#pragma unroll 4
  for (int k = lane * 8; k < p.K; k += 512) {
    const bf16x8 a = ld8(A + k);
#pragma unroll
    for (int j = 0; j < 2 * C; ++j) acc[j] = dot8(a, ld8(wr[j] + k), acc[j]);
  }
#pragma unroll
  for (int j = 0; j < 2 * C; ++j) acc[j] = wave_sum(acc[j]);
#pragma unroll
  for (int j = 0; j < C; ++j)
    if (lane == j && c0 + j < F) out[c0 + j] = f2bf(gg::glu_fast(acc[2 * j], acc[2 * j + 1], limit, p.alpha, p.up_one));
}

// One wave: one column of one token's residual += all its experts.
__global__ __launch_bounds__(256) void moe_gemv_down_kernel(MoeGemvParams p) {
  const int lane = lane_id(), t = blockIdx.y;
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= p.K) return;  // K: the residual's width here
  const int ck = (p.F + 511) / 512, cs = (p.Fs + 511) / 512;
  float* x = p.x + (long)t * p.K + n;
  const float x0 = p.add ? *x : 0.f;
  float acc = 0.f;
  const int items = p.top * ck;
#pragma unroll 8
  for (int i = 0; i < items; ++i) {
    const int k = i / ck, c = (i % ck) * 512 + lane * 8;
    const int ent = t * p.top + k, cc = min(c, p.F - 8);
    const bf16x8 a = ld8(static_cast<const bf16*>(p.mid) + (long)ent * p.F + cc);
    const bf16x8 v = ld8(static_cast<const bf16*>(p.w) + ((long)p.ids[ent] * p.K + n) * p.F + cc);
    const float d = dot8(a, v, 0.f) * p.wts[ent];
    acc += c < p.F ? d : 0.f;
  }
#pragma unroll 4
  for (int i = 0; i < cs; ++i) {
    const int c = i * 512 + lane * 8, cc = min(c, p.Fs - 8);
    const bf16x8 a = ld8(static_cast<const bf16*>(p.mids) + (long)t * p.Fs + cc);
    const bf16x8 v = ld8(static_cast<const bf16*>(p.ws) + (long)n * p.Fs + cc);
    const float d = dot8(a, v, 0.f) * (p.wts_s ? p.wts_s[t] : 1.f);
    acc += c < p.Fs ? d : 0.f;
  }
  acc = wave_sum(acc);
  if (lane == 0) *x = x0 + acc;
}

}  // namespace lsd

using namespace lsd;

static long gg_blocks(const GgParams& p, int mode, int tm, int tn) {
  if (mode == GG_UP || mode == GG_DOWN) {
    long b = (long)((p.n_tiles + p.gr - 1) / p.gr) * p.gr * ((p.N + tn - 1) / tn);
    if (p.Ns > 0) b += (long)(((p.T + tm - 1) / tm + p.gr_s - 1) / p.gr_s) * p.gr_s * ((p.Ns + tn - 1) / tn);
    return b;
  }
  return (long)((p.M + tm - 1) / tm) * ((p.N + tn - 1) / tn) * p.groups;
}

template <int MODE, int TM, int TN, int SLOTS, int AUX = 0>
static hipError_t gg_on(const GgParams& p, hipStream_t st) {
  const long blocks = gg_blocks(p, MODE, TM, TN);
  if (blocks) hipLaunchKernelGGL((group_gemm_kernel<MODE, TM, TN, SLOTS, AUX>), dim3((unsigned)blocks), dim3(256), 0, st, p);
  return hipGetLastError();
}

template <int MODE>
static hipError_t gg_launch(const GgParams& p, int tm, hipStream_t st) {
  switch (tm) {
    // decode: the experts' weights pass once, so non-temporally (2048 x 2048 up, 64 tokens of 4
    // in 32 experts 54 -> 49 us); the heads' do for every row tile
    case 32: return gg_on<MODE, 32, 64, 4, MODE == GG_BATCH ? 0 : 2>(p, st);
    case 64: return gg_on<MODE, 64, 128, 3>(p, st);
    case 128: return gg_on<MODE, 128, 128, 2>(p, st);
    default: return hipErrorInvalidValue;
  }
}

// tm: row-tile rows (32 / 64 / 128; the expert modes' table must use the same)
extern "C" hipError_t lsd_group_gemm(const GgParams* p, int mode, int tm, hipStream_t st) {
  switch (mode) {
    case GG_BATCH: return gg_launch<GG_BATCH>(*p, tm, st);
    case GG_UP: return gg_launch<GG_UP>(*p, tm, st);
    case GG_DOWN: return gg_launch<GG_DOWN>(*p, tm, st);
    default: return hipErrorInvalidValue;
  }
}

template <int MODE, int MT>
static hipError_t gg_f32_on(const GgParams& p, bool addr64, hipStream_t st) {
  const long blocks = gg_blocks(p, MODE, 16 * MT, 64);
  const dim3 grid((unsigned)blocks), block(256);
  if (blocks && addr64) hipLaunchKernelGGL((group_gemm_f32_mfma_kernel<MODE, MT, true>), grid, block, 0, st, p);
  else if (blocks) hipLaunchKernelGGL((group_gemm_f32_mfma_kernel<MODE, MT, false>), grid, block, 0, st, p);
  return hipGetLastError();
}

template <int MODE, int MT, int WN, int WK, int D>
static hipError_t gg_split_on(const GgParams& p, hipStream_t st) {
  const long blocks = gg_blocks(p, MODE, 16 * MT, 16 * WN);
  if (blocks)
    hipLaunchKernelGGL((group_gemm_f32_split_kernel<MODE, MT, WN, WK, D>), dim3((unsigned)blocks), dim3(64 * WN * WK), 0, st, p);
  return hipGetLastError();
}

template <int MODE, int WM, int MT, int WN, int NT, int WK, int PF, int OCC>
static hipError_t gg_half_on(const GgParams& p, hipStream_t st) {
  const long blocks = gg_blocks(p, MODE, 16 * MT * WM, 16 * NT * WN);
  if (blocks)
    hipLaunchKernelGGL((group_gemm_f32_half_kernel<MODE, WM, MT, WN, NT, WK, PF, OCC>), dim3((unsigned)blocks),
                       dim3(64 * WM * WN * WK), 0, st, p);
  return hipGetLastError();
}

// The split kernels' tiles: what their blocks take in rounds of 256, in us at K = 2048 (fixed part, a round), as
// measured over 100 .. 1500 rows of 2048 .. 11264 columns.  565 rows of 2048 columns: 48 x 64 47.3 us, 64 x 64 52.0,
// 80 x 64 43.3, 48 x 128 47.7; 300 of 2048 48 x 64 in two parts of K 33.7, in four 29.0; 565 of 4160
// 48 x 128 86, 80 x 128 100, 96 x 128 73; 1000 of 2048 64 x 64 67.7, 64 x 128 61.0; of 4160 80 x 128 117, 96 x 128
// 128; of 11264 64 x 128 306, 80 x 128 299, 96 x 128 286.
// For every K: of 329 sizes with K from 544 to 8192 the tiles so chosen take 0.54 to 1.02 of the fp32 MFMAs' times.
struct SplitTile {
  int rows, cols, parts, fixed, round;
};
static const SplitTile SPLIT_TILES[] = {{32, 64, 4, 1, 21}, {48, 64, 4, 1, 27}, {64, 64, 2, 4, 28}, {80, 64, 3, 0, 41},
                                        {48, 128, 1, 2, 42}, {64, 128, 1, 4, 48}, {80, 128, 1, 0, 59}, {96, 128, 1, 0, 70}};
// Two fp16 terms: K of 1024 and more, of which a part has 682 (the kernel has both errors), in no fewer parts than three
// terms would take (sums of 1024 in one part are 1.7e-7 off, in three on three terms 1.1e-7), where that is ahead: 100 rows
// of 2048 on 64 x 64 27.2 us, on three terms and 32 x 64 22.8.  48 x 128 never is: 565 rows of 2560 44.8, on 64 x 128 39.8.
static const SplitTile HALF_TILES[] = {{64, 64, 2, 6, 22}, {80, 64, 3, 3, 29}, {64, 128, 1, 8, 34}, {96, 128, 1, 0, 49}, {128, 128, 1, 0, 57}};
static bool half_terms(int K, int parts) { return K >= 1024 && K >= 682 * parts; }
static int split_tile(const GgParams& p) {  // of SPLIT_TILES, or behind them
  int best = 0;
  long least = 0;
  for (int i = 0, parts = 0; i < 13; ++i) {
    const SplitTile& t = i < 8 ? SPLIT_TILES[i] : HALF_TILES[i - 8];
    if (i == 8) parts = SPLIT_TILES[best].parts;
    if (i >= 8 && (t.parts < parts || !half_terms(p.K, t.parts))) continue;
    const long cost = t.fixed + (gg_blocks(p, GG_F32, t.rows, t.cols) + 255) / 256 * t.round;
    if (i == 0 || cost < least) best = i, least = cost;
  }
  return best;
}

// Products on split operands: experts from 18 rows a tile of the table on (2048 x 1024, 4 of 32 experts:
// 300 tokens, 24 rows, up 185 us either way, down 93; 200, 18 rows, 161 -> 149, 78 -> 68; 160, 15 rows, 139
// and 160, 71 and 77; 2 of 16 of 1024 x 512: 200, 18 rows, 38 -> 31), short K from 28 (1024 x 512, 4 of 32: 200 tokens,
// 18 rows, K = 128 10.8 and 14.2, 256 15.7 and 19.0, 384 24.0 either way, 512 28.1 and 26.6; 565, 34 rows, 128 18.7
// and 15.9), where the fp32 tiles, half as wide, are one a CU and more (2 of 8, 200 tokens, 224 tiles: K = 128 7.1 and
// 9.9, 512 14.4 and 17.6, 1536 35.5 and 41.4; 2 of 8 of 256 x 128, 1000 tokens, 9.2 and 11.9; 2 of 8 of 2048 x 1024, 120
// tokens, 256 tiles, 67 and 51).
// Others with more than 16 rows, unless the few are
// bound by the weights' stream (20 rows of 32000 x 2048 42 us and 50, of 16384 31.1 and 27.5) or K is short for the
// splitting to hide (565 rows of 2048, K = 256 12.2 and 12.8, 512 19.2 and 17.9; of 4096, K = 512 31.4 and 32.9;
// 100 rows of 2048, K = 512 10.6 and 11.1, 2048 28.7 and 22.9), up to 768 where the fp32 tiles fill the chip once (24 rows:
// K = 640, N = 6144 11.3 and 11.0, 11264 12.1 and 13.3, 16000 12.5 and 13.5, K = 768, N = 11264 13.4 either way;
// 40 rows of 8192, K = 544 10.7 and 11.1, of 11264 13.5 and 13.0).
static bool on_split(const GgParams& p, bool routed) {
  if (routed) {
    const long rows = (long)p.T * p.top, experts = p.n_tiles - rows / 64;
    // fp32 tiles that hold rows, about: half a tile an expert beside whole ones
    long tiles = max(experts, rows / 64 + experts / 2) * ((p.N + 63) / 64);
    if (p.Ns > 0) tiles += (p.T + 63L) / 64 * ((p.Ns + 63) / 64);
    return tiles >= 256 && rows >= (p.K >= 384 ? 18L : 28L) * p.n_tiles;
  }
  const long tiles = gg_blocks(p, GG_F32, 32, 64);
  if (p.K <= 512 || p.M <= 16 || (p.M <= 32 && tiles > 256)) return false;
  return p.K >= 768 || tiles > 256 || tiles <= (p.M <= 32 ? 96 : 192);
}

// Whether each column tile of experts on two terms starts its sums at another k than its neighbours and than the next expert: blocks
// under way together otherwise stand at the same place of rows of W that lie whole 4 KB apart.  Up to 96 rows an expert, whose
// W is read about once; long sums only where all blocks start at once.  us with, without, 32 experts, 4 a token:
//   2048 x 1024 (K = 2048 up, 1024 down)   200 tokens 106 115, 58 70   300 110 120, 61 73   500 150 160, 84 91   700 169 168, 89 94
//   2048 x 2048   200 204 203, 106 120   500 268 277, 153 167   4096 x 1024 (more blocks)   240 209 205, 115 132   400 222 213, 125 144
//   16 experts, 2 a token, 4096 x 1024, one round   200 127 147, 58 72   500 151 157, 83 88
// 175 rows an expert 2048 x 1024 368 and 362, 190 and 189; other strides, 2048 x 1088, 8 experts of 2560 x 2560, 1600 x 1600, 300 to
// 1400 tokens: 1 to 3 % slower so.
static bool moe_turned(const GgParams& p) {
  const long rows = (long)p.T * p.top, experts = p.n_tiles - rows / 64;
  if (p.K % 1024 != 0 || rows > 96 * experts) return false;
  return p.K <= 2048 || experts * ((p.N + 127) / 128) + (p.Ns > 0 ? (p.T + 63L) / 64 * ((p.Ns + 127) / 128) : 0) <= 256;
}

// Whether experts' products are on split operands (tests)
extern "C" int lsd_moe_on_split(int T, int top, int n_tiles, int N, int Ns, int K) {
  GgParams p{};
  p.T = T, p.top = top, p.n_tiles = n_tiles, p.N = N, p.Ns = Ns, p.K = K;
  return on_split(p, true);
}

extern "C" int lsd_moe_turned(int T, int top, int n_tiles, int N, int Ns, int K) {
  GgParams p{};
  p.T = T, p.top = top, p.n_tiles = n_tiles, p.N = N, p.Ns = Ns, p.K = K;
  return moe_turned(p);
}

template <int MODE>
static hipError_t gg_f32(const GgParams& p, hipStream_t st) {
  // the tiles' loads take whole 16 bytes and k-steps of 32
  auto at = [](const void* x) { return reinterpret_cast<uintptr_t>(x); };
  if (p.K % 32 || (p.Ns > 0 && p.Ks % 32) || (at(p.A) | at(p.W) | at(p.As) | at(p.Ws)) % 16) {
    const long blocks = gg_blocks(p, MODE, 64, 64);
    if (blocks) hipLaunchKernelGGL((group_gemm_f32_kernel<MODE>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    return hipGetLastError();
  }
  if (on_split(p, MODE == GG_UP || MODE == GG_DOWN)) {
    if constexpr (MODE == GG_F32 || MODE == GG_ADD) {
      switch (split_tile(p)) {
        case 0: return gg_split_on<MODE, 2, 4, 4, 2>(p, st);
        case 1: return gg_split_on<MODE, 3, 4, 4, 2>(p, st);
        case 2: return gg_split_on<MODE, 4, 4, 2, 2>(p, st);
        case 3: return gg_split_on<MODE, 5, 4, 3, 2>(p, st);
        case 4: return gg_split_on<MODE, 3, 8, 1, 3>(p, st);
        case 6: return gg_split_on<MODE, 5, 8, 1, 2>(p, st);
        case 7: return gg_split_on<MODE, 6, 8, 1, 2>(p, st);
        case 8: return gg_half_on<MODE, 2, 2, 2, 2, 2, 1, 4>(p, st);
        case 9: return gg_half_on<MODE, 1, 5, 4, 1, 3, 1, 3>(p, st);
        case 10: return gg_half_on<MODE, 2, 2, 4, 2, 1, 1, 4>(p, st);
        case 11: return gg_half_on<MODE, 2, 3, 4, 2, 1, 2, 2>(p, st);
        case 12: return gg_half_on<MODE, 2, 4, 4, 2, 1, 2, 2>(p, st);
      }
    } else if (half_terms(min(p.K, p.Ns > 0 ? p.Ks : p.K), 1)) {
      GgParams q = p;
      q.turn = moe_turned(p);
      return gg_half_on<MODE, 2, 2, 4, 2, 1, 2, 4>(q, st);
    }
    return gg_split_on<MODE, 4, 8, 1, 3>(p, st);
  }
  // The others count bytes from a tile's first row, or from the first of the rows it gathers, in 32 bits
  // where those hold them (524288 tokens of 2048 are 4 GB)
  auto out = [](long rows, long ld, int K) { return (rows * ld + K) * 4 >= 1L << 32; };
  const bool far = out(MODE == GG_UP ? p.T : 64, p.lda, p.K) || out(64, p.ldw, p.K) ||
                   (p.Ns > 0 && (out(64, p.ldas, p.Ks) || out(64, p.ldws, p.Ks)));
  // Up to 16 rows are bound by the latency of their loads, which is less with 64-bit addresses (8 rows
  // of 2048 x 2048 19.3 us, with offsets of 32 bits 21.2; of 1408 x 4704 40.8 and 45.7; but 32 rows of
  // 2048 x 2048 28.3 and 27.4.  Experts, 2 of 32 and a shared one of 2048, 1024 columns down: 8
  // tokens 18.9 and 21.6; 4 of 32 of 2048 x 1024 up: 11 tokens 99.7 and 107; 4 of 16 of 1024 x 512 up,
  // the other way, 16.5 and 15.7).
  const bool addr64 = far || (MODE == GG_UP || MODE == GG_DOWN ? p.T : p.M) <= 16;
  if constexpr (MODE == GG_F32 || MODE == GG_ADD) {
    // half tiles where the fullest CU gets less work of them (N = 2048, K = 512: 565 rows 19 us)
    auto rounds = [&](int tm) { return (gg_blocks(p, MODE, tm, 64) + 255) / 256; };
    if (rounds(32) < 2 * rounds(64)) return gg_f32_on<MODE, 2>(p, addr64, st);
  }
  return gg_f32_on<MODE, 4>(p, addr64, st);
}

// Rows and columns of the tiles of M x N fp32 results of K products (0: few), and parts of K (tests)
extern "C" void lsd_group_gemm_split_tile(int M, int N, int K, int* tile) {
  GgParams p{};
  p.M = M, p.N = N, p.K = K, p.groups = 1;
  const int i = split_tile(p);
  const SplitTile& t = i < 8 ? SPLIT_TILES[i] : HALF_TILES[i - 8];
  tile[0] = t.rows, tile[1] = t.cols, tile[2] = t.parts;
}

// fp32 kernels: 64-row tiles
extern "C" hipError_t lsd_group_gemm_f32(const GgParams* p, int mode, hipStream_t st) {
  switch (mode) {
    case GG_UP: return gg_f32<GG_UP>(*p, st);
    case GG_DOWN: return gg_f32<GG_DOWN>(*p, st);
    case GG_F32: return gg_f32<GG_F32>(*p, st);
    case GG_ADD: return gg_f32<GG_ADD>(*p, st);
    default: return hipErrorInvalidValue;
  }
}

// up: K input columns, F / Fs gated columns; down: K residual columns
extern "C" hipError_t lsd_moe_gemv_up(const MoeGemvParams* p, hipStream_t st) {
  constexpr int C = 2;
  const long nb = (long)((p->Fs + 4 * C - 1) / (4 * C)) * p->T + (long)((p->F + 4 * C - 1) / (4 * C)) * p->T * p->top;
  hipLaunchKernelGGL((moe_gemv_up_kernel<C>), dim3((unsigned)nb), dim3(256), 0, st, *p);
  return hipGetLastError();
}

extern "C" hipError_t lsd_moe_gemv_down(const MoeGemvParams* p, hipStream_t st) {
  hipLaunchKernelGGL(moe_gemv_down_kernel, dim3((p->K + 3) / 4, p->T), dim3(256), 0, st, *p);
  return hipGetLastError();
}
