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
// fp32, for models served in it: MFMA 16x16x4 on fp32 operands, the same staging; VALU tiles
// with fused multiply-adds where K has no whole steps of 32 or a row starts off 16 bytes.
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

// fp32: 16 MT x 64 tiles, 32-deep k-steps (128-byte rows, the bf16 kernel's staging and swizzle);
// wave w owns 16 columns of all rows and leaves out the 16-row tiles that hold none, so an
// expert's last rows cost what they are.  A lane's 16-byte fragment feeds four MFMA 16x16x4,
// whose k-slot g stands for k = 4 g + j in both operands.
// Bound by the matrix cores, whose fp32 rate is a sixteenth of bf16's (154 TF/s), and, where
// experts have some tens of rows, by their weights.  64 x 128 tiles were no faster.
// Loads by lds_dma16 (global_load_lds before): 2260 rows over 32 experts of 2048 x 1024 and
// 565 through a shared one of 2048 up 325 -> 295 us, down 169 -> 160; 565 x 2048 x 2048 63 -> 54;
// 8192 x 8192 x 2048 118 -> 133 TF/s.
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
  constexpr int CPR = TN / 4;
  for (int c = threadIdx.x; c < min(TM, t.rows) * CPR; c += 256) {
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

template <int MODE>
static hipError_t gg_f32(const GgParams& p, hipStream_t st) {
  // the tiles' loads take whole 16 bytes and k-steps of 32
  auto at = [](const void* x) { return reinterpret_cast<uintptr_t>(x); };
  if (p.K % 32 || (p.Ns > 0 && p.Ks % 32) || (at(p.A) | at(p.W) | at(p.As) | at(p.Ws)) % 16) {
    const long blocks = gg_blocks(p, MODE, 64, 64);
    if (blocks) hipLaunchKernelGGL((group_gemm_f32_kernel<MODE>), dim3((unsigned)blocks), dim3(256), 0, st, p);
    return hipGetLastError();
  }
  // and count bytes from a tile's first row, or from the first of the rows it gathers, in 32 bits
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
    // half tiles where the fullest CU gets less work of them (N = K = 2048: 565 rows 67 against
    // 80 us, 200 rows 32 against 46); at the same work the whole ones (1000 rows 84 against 91)
    auto rounds = [&](int tm) { return (gg_blocks(p, MODE, tm, 64) + 255) / 256; };
    if (rounds(32) < 2 * rounds(64)) return gg_f32_on<MODE, 2>(p, addr64, st);
  }
  return gg_f32_on<MODE, 4>(p, addr64, st);
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
