// Decode GEMM of 9 .. 256 rows:  C[M,N] = A[M,K] . W[N,K]^T  (+ epilogue)
//
// What bounds it is the stream of W out of HBM, which is read once, and the rate at which
// a CU takes LDS-DMA in (about 50 GB/s: W and A together).  So:
//  * W and A go to LDS by 16-byte LDS-DMA in whole 128-byte lines.  Fragments loaded
//    straight to registers touch 16 rows x 64 bytes per instruction and stop at 4.2 TB/s with
//    16 rows, 3.4 with 40 (28672 x 4096); this kernel reaches 5.3 with both.
//  * a ring as deep as two blocks per CU allow (80 KB): 4 to 7 k-steps in flight per block.
//    With two, W arrives at half the rate.  Wide tiles of up to 64 rows load W non-temporally
//    (28672 x 4096 at 40 rows 49.5 -> 44.0 us, 4096 x 14336 23.0 -> 21.3); narrow ones, whose
//    weights are small, and more rows are 0 to 20 % slower that way.
//  * rows of W that lie powers of two apart: blocks that walk through K together stand at the same place of
//    all of them, and where they all start at once W arrives at 4.9 to 5.5 TB/s.  Each column tile then starts its sums
//    elsewhere (deep_turn): 16384 x 4096 of 24 rows 25.9 -> 21.9 us, 32000 x 2048 26.3 -> 23.5, 11264 x 2048 11.2 -> 10.6.
//  * a block holds all of up to 64 rows; more are also divided among blocks beside each other,
//    which find W in L2, where that brings a CU fewer bytes.  Its width (128 to 16 columns)
//    follows from the columns: narrow outputs take narrow tiles, whose waves split the k-step's
//    32-wide parts among them (WK) and are summed through LDS.  No K splits over blocks, no
//    tickets and no workspace, except where the caller takes the partial sums as slabs.
//
// Alone, cold weights, before (split-K with the weights in registers; 128 x 64 ring) -> now:
//   28672 x 4096 gate/up, 40 rows   65.9 -> 37.8 us     4096 x 14336 slabs, 40 rows  28.8 -> 21.3
//   6144 x 4096 QKV, 40 rows        18.7 -> 14.4        4096 x 4096 slabs, 40 rows   15.0 -> 8.7
//   6144 x 2048, 24 rows            12.2 -> 7.6         2624 x 2048 fp32, 64 rows    13.1 -> 7.5
//   11264 x 2048 gate/up, 96 rows   19.8 -> 16.8        4800 x 1600 QKV, 128 rows    13.6 -> 9.4
#include "gemm_epilogue.h"

namespace lsd {

namespace {
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void gbl_cvoid;
constexpr int NT_LOAD = 2;  // cache policy of an LDS-DMA: non-temporal
}  // namespace

// WM x WN waves of MTW x NTW 16 x 16 tiles, times WK waves on different 32-wide parts of a
// k-step of BK; SLOTS k-steps in LDS; AUX: cache policy of W; ONE: a block holds all rows (a row
// block found at run time, by a division, costs 0.3 us a launch: 40 rows of GPT-2 XL 2274 -> 2211 us
// a step without).
// turn: a column tile starts its sums at another k than its neighbours.
template <int WM, int WN, int WK, int MTW, int NTW, int BK, int SLOTS, int AUX, int EPI, bool ONE>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_deep_kernel(GemmParams p, int tiles_n, int row_blocks, int turn) {
  constexpr int WAVES = WM * WN * WK, BM = 16 * WM * MTW, BN = 16 * WN * NTW;
  constexpr int RB = BK * 2, CPR = RB / 16, RPI = 64 / CPR;  // bytes and 16-byte chunks of a row, rows per instruction
  constexpr int A_BYTES = BM * RB, SLOT = (BM + BN) * RB;
  constexpr int IA = BM / RPI, IW = BN / RPI;                // LDS-DMA instructions of a k-step
  constexpr int LA = (IA + WAVES - 1) / WAVES, LW = (IW + WAVES - 1) / WAVES, LPS = LA + LW, D = SLOTS - 1;
  constexpr int CLD = BN + 4, CT = WK * BM * CLD * 4;
  static_assert(LPS * D <= 63, "the wait counter holds 63 loads");
  static_assert(BK / 32 % WK == 0 && BM % RPI == 0 && BN % RPI == 0, "tile sizes");
  __shared__ __attribute__((aligned(16))) char smem[SLOTS * SLOT > CT ? SLOTS * SLOT : CT];
  const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wk = w % WK, wn = (w / WK) % WN, wm = w / (WK * WN);
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int nb = ONE ? bid : bid / row_blocks, m0 = ONE ? 0 : (bid - nb * row_blocks) * BM;  // (row blocks side by side share W)
  const int split = nb / tiles_n, n0 = (nb - split * tiles_n) * BN;
  const int KT = p.K / BK;
  const int kb = (int)((long)KT * split / p.splits), ke = (int)((long)KT * (split + 1) / p.splits);

  // per-lane source addresses; 16-byte chunks XOR-swizzled on the source side.  Where the
  // instructions do not divide among the waves, the last one is issued again: every wave
  // counts the same number of loads, and the copy writes the same bytes.
  auto swz = [](int row) { return BK == 64 ? (row >> 1) & 7 : row & 15; };
  const bf16* srca[LA];
  const bf16* srcw[LW];
  int dsta[LA], dstw[LW];
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int ins = min(w + q * WAVES, IA - 1), row = ins * RPI + lane / CPR;
    dsta[q] = ins * 1024;
    srca[q] = p.A + (long)min(m0 + row, p.M - 1) * p.lda + (((lane % CPR) ^ swz(row)) << 3);
  }
#pragma unroll
  for (int q = 0; q < LW; ++q) {
    const int ins = min(w + q * WAVES, IW - 1), row = ins * RPI + lane / CPR;
    dstw[q] = A_BYTES + ins * 1024;
    srcw[q] = p.W + (long)min(n0 + row, p.N - 1) * p.ldw + (((lane % CPR) ^ swz(row)) << 3);
  }
  const int from = (nb * 5 & 31) & turn;  // (turn: 31, of at least 32 k-steps, or 0)
  auto issue = [&](int kt, int slot) {
    kt += from;
    kt = kt >= KT ? kt - KT : kt;
#pragma unroll
    for (int q = 0; q < LW; ++q)
      __builtin_amdgcn_global_load_lds((gbl_cvoid*)(srcw[q] + (long)kt * BK), (lds_void*)(smem + slot * SLOT + dstw[q]),
                                       16, 0, AUX);
#pragma unroll
    for (int q = 0; q < LA; ++q)
      __builtin_amdgcn_global_load_lds((gbl_cvoid*)(srca[q] + (long)kt * BK), (lds_void*)(smem + slot * SLOT + dsta[q]),
                                       16, 0, 0);
  };
  f32x4 acc[MTW][NTW];
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto frag = [&](const char* t, int row, int chunk) {
    return *reinterpret_cast<const bf16x8*>(t + row * RB + ((chunk ^ swz(row)) << 4));
  };
  int slot = 0;
  auto step = [&]() {
    const char* t = smem + slot * SLOT;
#pragma unroll
    for (int kk = 0; kk < BK / 32; kk += WK) {
      bf16x8 af[MTW], wf[NTW];
#pragma unroll
      for (int i = 0; i < MTW; ++i) af[i] = frag(t, (wm * MTW + i) * 16 + r, (kk + wk) * 4 + g);
#pragma unroll
      for (int j = 0; j < NTW; ++j) wf[j] = frag(t + A_BYTES, (wn * NTW + j) * 16 + r, (kk + wk) * 4 + g);
#pragma unroll
      for (int i = 0; i < MTW; ++i)
#pragma unroll
        for (int j = 0; j < NTW; ++j) acc[i][j] = mfma16(af[i], wf[j], acc[i][j]);
    }
    slot = slot == SLOTS - 1 ? 0 : slot + 1;
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (kb + d < ke) issue(kb + d, d);
  int kt = kb;
  for (; kt + D < ke; ++kt) {
    __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPS * (D - 1)));  // this wave's part of k-step kt has landed
    __builtin_amdgcn_s_barrier();                          // ... and every wave's; step kt - 1 is read
    issue(kt + D, slot == 0 ? SLOTS - 1 : slot - 1);
    step();
  }
  count_down<D>([&](auto ic) {  // the last D steps, nothing left to issue
    constexpr int d = decltype(ic)::v;
    if (ke - 1 - kt == d) {
      __builtin_amdgcn_s_waitcnt(vmcnt_imm(LPS * d));
      __builtin_amdgcn_s_barrier();
      step();
      ++kt;
    }
  });
  __syncthreads();

  // epilogue through LDS: the WK parts summed, row-contiguous 16-byte stores
  float* ct = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i = 0; i < MTW; ++i)
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        ct[(wk * BM + (wm * MTW + i) * 16 + 4 * g + q) * CLD + (wn * NTW + j) * 16 + r] = acc[i][j][q];
  __syncthreads();
  auto eight = [&](const float* s, float* v) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] = s[e];
#pragma unroll
      for (int h = 1; h < WK; ++h) v[e] += s[h * BM * CLD + e];
    }
  };
  for (int c = threadIdx.x; c < BM * (BN / 8); c += 64 * WAVES) {
    const int row = c / (BN / 8), ch = c % (BN / 8), m = m0 + row, n = n0 + ch * 8;
    if (m >= p.M || n >= p.N) continue;
    const float* s = ct + row * CLD + ch * 8;
    float v[8];
    eight(s, v);
    if constexpr (EPI == EPI_SILU_MUL) {
      if ((ch & 3) >= 2) continue;  // up columns: 16 to the right of their gates
      float u[8];
      eight(s + 16, u);
      const bf16x8 o = gated8(v, u, p.glu, p.act_scale);
      st8(reinterpret_cast<bf16*>(p.out) + (long)m * p.ldo + (n >> 5) * 16 + (n & 15), o);
    } else {
      epilogue8<EPI>(p, m, n, v, split);
    }
  }
}

// A block's rows and columns.  A CU takes in its blocks' rows of W and A at one rate, so the
// shape with the least of ceil(blocks / CUs) (columns + rows) is the fastest one: measured at 64 rows,
// 4800 x 1600 on 75 blocks of 64 columns 11.9 us, on 150 of 32 8.8; 2624 x 2048 on 82 of 32 8.8,
// on 164 of 16 7.5; 8512 x 2048 on 133 of 64 13.0, on 266 of 32 15.6.
struct DeepShape {
  int rows, cols;
};
// All rows in a block (up to 128; more are two blocks side by side): whether a call is taken at all
// goes by these.
static int deep_rows(int M) {
  return M > 192 ? 128 : M > 128 ? 96 : M > 96 ? 128 : M > 64 ? 96 : (M + 15) / 16 * 16;
}
static int deep_cols(int M, int N, int K, int splits, int epi) {
  const int rows = deep_rows(M), mbs = (M + rows - 1) / rows;
  int best = 0;
  long least = 0;
  for (int bn = 64; bn >= 16; bn /= 2) {
    if (bn == 16 && (M > 64 || epi == EPI_SILU_MUL || K % 128 != 0 || K / 128 < splits)) break;
    const long blocks = (long)((N + bn - 1) / bn) * splits * mbs, cost = (blocks + 255) / 256 * (bn + rows);
    if (best == 0 || cost < least) { best = bn; least = cost; }
  }
  return best;
}
// More than 64 rows also in blocks of fewer rows, whose neighbours find W in L2 (48 x 96 only up to two
// of them: 140 rows of 11264 x 2048 24.2 us, so 25.4).  All rows in a block -> here:
//   96 rows   3072 x 2048 12.3 -> 8.9 (48 x 32), 6464 13.2 -> 11.7 (48 x 64), 8512 14.9 -> 13.4 (48 x 80)
//   128 rows  4800 x 1600 11.8 -> 9.4 (48 x 64), 6144 x 4096 24.9 -> 21.9 (48 x 80)
//   256 rows  4800 x 1600 14.1 -> 11.9 (64 x 80), 11264 x 2048 gate/up 30.8 -> 27.3 (64 x 96)
// and over 176 products of 50 to 256 rows 7 % on average.  Each of these shapes adds up K as the
// ones that hold all rows do, so the bits are the same, where column tiles all start at the first k.  (32 x 32 for 49 to 64 rows, 2624 x 2048 8.3 -> 7.6
// us, does not: it halves the k-steps among two waves where 16 columns had four, and a router
// behind it decided close calls otherwise; with four waves it is no faster.)  Behind, by 0.2 us, 768 x 3072 in 8 slabs of
// 128 rows (4.7 us).
// Beside another lane's launches the chip is full either way and what blocks take in together counts,
// a fifth more with 64 x 80 at 256 rows than with 128 x 64.  GPT-2 XL in two lanes, all rows in a block
// against here, tokens a second: 256 rows a lane 52.6 and 51.9 thousand, 200 48.5 and 48.6, 160 44.9 and
// 44.2, 144 43.4 and 43.8, 128 40.0 and 41.4, 96 36.7 and 37.0.
// Up to 128 rows also 128 columns, which take in A half as often (us on 64 columns -> 128, both where deep_turn lets them start
// elsewhere): 28672 x 4096, 16 / 32 / 48 / 64 rows 38.7 39.8 42.6 47.1 -> 36.2 36.8 37.8 39.1; 32000 x 2048, 48 rows 24.9 -> 24.1, 96
// 33.6 -> 28.8, 128 36.3 -> 30.5; 128256 x 4096, 48 rows 190 -> 174; 50304 x 1600, 48 rows 36.1 -> 32.2; but 40960 x 1600, where they
// cost more, 27.5 and 30.0.
static DeepShape deep_shape(int M, int N, int K, int splits, int epi, int lanes) {
  DeepShape best{deep_rows(M), deep_cols(M, N, K, splits, epi)};
  if (M >= 160 && lanes > 1) return best;
  auto cost = [&](DeepShape s) {
    const long blocks = (long)((N + s.cols - 1) / s.cols) * splits * ((M + s.rows - 1) / s.rows);
    return (blocks + 255) / 256 * (s.rows + s.cols);
  };
  long least = cost(best);
  auto offer = [&](DeepShape s) {
    if (epi == EPI_SILU_MUL && s.cols % 32 != 0) return;
    if (cost(s) < least) { best = s; least = cost(s); }
  };
  if (M <= 128 && (epi == EPI_SILU_MUL || epi == EPI_F32 || epi == EPI_BF16 || epi == EPI_GELU)) offer({best.rows, 128});
  if (M <= 64) return best;
  for (int cols : {32, 64, 80, 96})
    if (cols < 96 || M <= 96) offer({48, cols});
  for (int cols : {64, 80, 96}) offer({64, cols});
  return best;
}

// Column tiles start at places of K of their own where W's rows lie whole 4 KB apart and all blocks start at once: two a CU
// (96 x 128 and 128 x 128 ones, one a CU, are never more than 256: lsd_gemm_deep_ok).  Later ones are out of step by themselves (128256 x 4096, 48 rows of 128 columns 174 us, turned 190), as are rows of other
// strides (K = 1600, 768: up to 4 % slower turned), and 32 columns gain too little (6144 x 4096 14.3 and 14.9).
static bool deep_turn(int splits, int K, long ldw, long blocks, int cols) {
  return splits == 1 && K >= 2048 && K % 2048 == 0 && ldw % 2048 == 0 && cols >= 64 && blocks <= 512;
}

template <int EPI>
static hipError_t deep_launch(const GemmParams& p, hipStream_t st) {
  const DeepShape s = deep_shape(p.M, p.N, p.K, p.splits, EPI, p.lanes);
  const int tn = (p.N + s.cols - 1) / s.cols, mbs = (p.M + s.rows - 1) / s.rows;
  const int turn = deep_turn(p.splits, p.K, p.ldw, (long)tn * mbs, s.cols) ? 31 : 0;
#define LSD_DEEP_K(ONE, ROWS, COLS, WM, WN, WK, BK, SLOTS, AUX)                                                       \
  if (s.rows == ROWS && s.cols == COLS) {                                                                             \
    hipLaunchKernelGGL((gemm_deep_kernel<WM, WN, WK, ROWS / (16 * WM), COLS / (16 * WN), BK, SLOTS, AUX, EPI, ONE>),  \
                       dim3((unsigned)(tn * p.splits * mbs)), dim3(64 * WM * WN * WK), 0, st, p, tn, mbs, turn);            \
    return hipGetLastError();                                                                                         \
  }
  // slots: two blocks per CU, of 96 and 128 rows by 128 columns one
  if (mbs == 1) {
    LSD_DEEP_K(true, 48, 64, 1, 4, 1, 64, 5, NT_LOAD)
    LSD_DEEP_K(true, 48, 32, 1, 2, 2, 64, 8, 0)
    if constexpr (EPI != EPI_SILU_MUL) {
      LSD_DEEP_K(true, 48, 16, 1, 1, 4, 128, 5, 0)
    }
    if constexpr (EPI == EPI_SILU_MUL || EPI == EPI_F32 || EPI == EPI_BF16 || EPI == EPI_GELU) {
      LSD_DEEP_K(true, 16, 128, 1, 4, 1, 64, 3, NT_LOAD)
      LSD_DEEP_K(true, 32, 128, 1, 4, 1, 64, 3, NT_LOAD)
      LSD_DEEP_K(true, 48, 128, 1, 4, 1, 64, 3, NT_LOAD)
      LSD_DEEP_K(true, 64, 128, 1, 4, 1, 64, 3, NT_LOAD)
      LSD_DEEP_K(true, 96, 128, 2, 4, 1, 64, 4, 0)
      LSD_DEEP_K(true, 128, 128, 2, 4, 1, 64, 4, 0)
    }
    LSD_DEEP_K(true, 16, 64, 1, 4, 1, 64, 8, NT_LOAD)
    LSD_DEEP_K(true, 32, 64, 1, 4, 1, 64, 6, NT_LOAD)
    LSD_DEEP_K(true, 64, 64, 1, 4, 1, 64, 5, NT_LOAD)
    LSD_DEEP_K(true, 16, 32, 1, 2, 2, 64, 8, 0)
    LSD_DEEP_K(true, 32, 32, 1, 2, 2, 64, 8, 0)
    LSD_DEEP_K(true, 64, 32, 1, 2, 2, 64, 6, 0)
    if constexpr (EPI != EPI_SILU_MUL) {
      LSD_DEEP_K(true, 16, 16, 1, 1, 4, 128, 8, 0)
      LSD_DEEP_K(true, 32, 16, 1, 1, 4, 128, 6, 0)
      LSD_DEEP_K(true, 64, 16, 1, 1, 4, 128, 4, 0)
    }
    // (as many blocks of half the rows and 64 columns take in less than 96 x 32 or 128 x 32, except
    // where rounding up the columns of each slab makes them a round more)
    LSD_DEEP_K(true, 96, 64, 2, 2, 2, 64, 4, 0)
    if constexpr (EPI == EPI_SLAB) {
      LSD_DEEP_K(true, 96, 32, 2, 2, 2, 64, 5, 0)
    }
    LSD_DEEP_K(true, 128, 64, 2, 2, 2, 64, 3, 0)
    return hipErrorInvalidValue;
  }
  LSD_DEEP_K(false, 48, 32, 1, 2, 2, 64, 8, 0)
  LSD_DEEP_K(false, 48, 64, 1, 4, 2, 64, 5, 0)
  LSD_DEEP_K(false, 64, 64, 4, 1, 2, 64, 5, 0)
  if constexpr (EPI != EPI_SILU_MUL) {
    LSD_DEEP_K(false, 48, 80, 3, 1, 2, 64, 5, 0)
    LSD_DEEP_K(false, 64, 80, 4, 1, 2, 64, 4, 0)
  }
  LSD_DEEP_K(false, 48, 96, 3, 2, 2, 64, 4, 0)
  LSD_DEEP_K(false, 64, 96, 2, 2, 2, 64, 4, 0)
  LSD_DEEP_K(false, 96, 64, 2, 2, 2, 64, 4, 0)
  LSD_DEEP_K(false, 96, 32, 2, 2, 2, 64, 5, 0)
  LSD_DEEP_K(false, 128, 64, 2, 2, 2, 64, 3, 0)
  LSD_DEEP_K(false, 128, 32, 2, 2, 2, 64, 4, 0)
#undef LSD_DEEP_K
  return hipErrorInvalidValue;
}

}  // namespace lsd

using namespace lsd;

// 1 .. 256 rows, whole k-steps; gate / up pairs lie in one tile.  splits > 1 only as slabs:
// the other epilogues run unsplit, whatever the caller asked for.  More than 48 rows only up to
// two blocks a CU (49 .. 64 rows two and a half): behind that the 128 x 128 tiles, which read A half
// as often, are as fast or faster.  Vocabulary-wide, deep ring in blocks of 64 columns against those tiles (deep_shape has what 128
// columns give up to 48 rows; more rows have not been timed on them where they are not taken):
//   50304 x 1600  64 rows 40.3 against 37.0 us, 96 50 against 41, 128 56 against 44 (48 rows 38 and 37)
//   128256 x 4096  64 rows 220 against 203, 128 260 against 208 (40 rows both 190)
//   40960 x 1600  64 rows 31.5 against 35, 80 36 against 37, 128 44 against 42
// More than 128 rows are two row blocks: whole steps of 48 layers of 1600, 160 sequences
// 4472 -> 4117 us, 256 5426 -> 5326; 12 layers of 2048, 140 sequences 1285 -> 1198; not with more
// blocks: 4096 x 14336 at 256 rows in 8 slabs, 1024 of them, 47.5 -> 57.2 us.
extern "C" int lsd_gemm_deep_ok(int M, int N, int K, int epi, int splits) {
  if (M < 1 || M > 256 || K < 64 || K % 64 != 0 || N % (epi == EPI_SILU_MUL ? 32 : 16) != 0) return 0;
  if (epi != EPI_SLAB) splits = 1;
  if (splits < 1 || splits > K / 64) return 0;
  if (M <= 48) return 1;
  const int bn = deep_cols(M, N, K, splits, epi);
  return (long)((N + bn - 1) / bn) * splits * (M > 128 ? 2 : 1) <= (M > 64 ? 512 : 640);
}

// rows * 1024 + columns of a block, for a call that is taken
extern "C" int lsd_gemm_deep_shape(int M, int N, int K, int epi, int splits, int lanes) {
  const DeepShape s = deep_shape(M, N, K, epi == EPI_SLAB ? splits : 1, epi, lanes);
  return s.rows * 1024 + s.cols;
}

// Whether its column tiles start at places of K of their own (tests)
extern "C" int lsd_gemm_deep_turned(int M, int N, int K, long ldw, int epi, int splits) {
  const DeepShape s = deep_shape(M, N, K, splits, epi, 1);
  return deep_turn(splits, K, ldw, (long)((N + s.cols - 1) / s.cols) * ((M + s.rows - 1) / s.rows), s.cols);
}

extern "C" hipError_t lsd_gemm_deep(const GemmParams* p, int epi, hipStream_t st) {
  if (!lsd_gemm_deep_ok(p->M, p->N, p->K, epi, p->splits)) return hipErrorInvalidValue;
  GemmParams q = *p;
  if (epi != EPI_SLAB) q.splits = 1;
  switch (epi) {
#define LSD_DEEP(E) \
  case E: return deep_launch<E>(q, st);
    LSD_DEEP(EPI_BF16)
    LSD_DEEP(EPI_GELU)
    LSD_DEEP(EPI_SILU_MUL)
    LSD_DEEP(EPI_F32)
    LSD_DEEP(EPI_RESID)
    LSD_DEEP(EPI_QKV)
    LSD_DEEP(EPI_SLAB)
#undef LSD_DEEP
    default: return hipErrorInvalidValue;
  }
}
