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
//  * a block holds all rows (up to 128; more are two blocks beside each other, the second of
//    which finds W in L2), so W is read once, and its width (64, 32 or 16 columns) follows
//    from the columns: narrow outputs take narrow tiles, whose waves split the k-step's
//    32-wide parts among them (WK) and are summed through LDS.  No K splits over blocks, no
//    tickets and no workspace, except where the caller takes the partial sums as slabs.
//
// Alone, cold weights, before (split-K with the weights in registers; 128 x 64 ring) -> now:
//   28672 x 4096 gate/up, 40 rows   65.9 -> 44.0 us     4096 x 14336 slabs, 40 rows  28.8 -> 21.3
//   6144 x 4096 QKV, 40 rows        18.7 -> 14.4        4096 x 4096 slabs, 40 rows   15.0 -> 8.7
//   6144 x 2048, 24 rows            12.2 -> 7.6         2624 x 2048 fp32, 64 rows    13.1 -> 7.5
//   11264 x 2048 gate/up, 96 rows   19.8 -> 17.7        4800 x 1600 QKV, 128 rows    13.6 -> 12.0
#include "gemm_epilogue.h"

namespace lsd {

namespace {
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) const void gbl_cvoid;
constexpr int NT_LOAD = 2;  // cache policy of an LDS-DMA: non-temporal
}  // namespace

// WM x WN waves of MTW x NTW 16 x 16 tiles, times WK waves on different 32-wide parts of a
// k-step of BK; SLOTS k-steps in LDS; AUX: cache policy of W; TWO: two row blocks.
template <int WM, int WN, int WK, int MTW, int NTW, int BK, int SLOTS, int AUX, int EPI, bool TWO = false>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_deep_kernel(GemmParams p, int tiles_n) {
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
  const int m0 = TWO ? (bid & 1) * BM : 0, nb = TWO ? bid >> 1 : bid;  // (row blocks side by side share W)
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
  auto issue = [&](int kt, int slot) {
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
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = f2bf(gated(v[e], u[e], p.glu, p.act_scale));
      st8(reinterpret_cast<bf16*>(p.out) + (long)m * p.ldo + (n >> 5) * 16 + (n & 15), o);
    } else {
      epilogue8<EPI>(p, m, n, v, split);
    }
  }
}

// Columns of a block.  A CU takes in its blocks' rows of W and A at one rate, so the width with
// the least of ceil(blocks / CUs) (columns + rows) is the fastest one: measured at 64 rows,
// 4800 x 1600 on 75 blocks of 64 columns 11.9 us, on 150 of 32 8.8; 2624 x 2048 on 82 of 32 8.8,
// on 164 of 16 7.5; 8512 x 2048 on 133 of 64 13.0, on 266 of 32 15.6.
static int deep_rows(int M) {  // of a block
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

template <int EPI, int MT>
static hipError_t deep_rows64(const GemmParams& p, int bn, hipStream_t st) {
  // slots: two blocks per CU
  constexpr int S64 = MT == 1 ? 8 : MT == 2 ? 6 : 5, S32 = MT == 4 ? 6 : 8, S16 = MT == 1 ? 8 : MT == 2 ? 6 : MT == 3 ? 5 : 4;
  const int tn = (p.N + bn - 1) / bn;
  const dim3 grid((unsigned)(tn * p.splits)), block(256);
  if (bn == 64)
    hipLaunchKernelGGL((gemm_deep_kernel<1, 4, 1, MT, 1, 64, S64, NT_LOAD, EPI>), grid, block, 0, st, p, tn);
  else if (bn == 32)
    hipLaunchKernelGGL((gemm_deep_kernel<1, 2, 2, MT, 1, 64, S32, 0, EPI>), grid, block, 0, st, p, tn);
  else if constexpr (EPI != EPI_SILU_MUL)
    hipLaunchKernelGGL((gemm_deep_kernel<1, 1, 4, MT, 1, 128, S16, 0, EPI>), grid, block, 0, st, p, tn);
  return hipGetLastError();
}

template <int EPI, int MTW, bool TWO>
static hipError_t deep_rows128(const GemmParams& p, int bn, hipStream_t st) {
  const int tn = (p.N + bn - 1) / bn;
  const dim3 grid((unsigned)(tn * p.splits * (TWO ? 2 : 1))), block(512);
  if (bn == 64)
    hipLaunchKernelGGL((gemm_deep_kernel<2, 2, 2, MTW, 2, 64, MTW == 3 ? 4 : 3, 0, EPI, TWO>), grid, block, 0, st, p, tn);
  else
    hipLaunchKernelGGL((gemm_deep_kernel<2, 2, 2, MTW, 1, 64, MTW == 3 ? 5 : 4, 0, EPI, TWO>), grid, block, 0, st, p, tn);
  return hipGetLastError();
}

template <int EPI>
static hipError_t deep_launch(const GemmParams& p, hipStream_t st) {
  const int bn = deep_cols(p.M, p.N, p.K, p.splits, EPI);
  if (p.M <= 16) return deep_rows64<EPI, 1>(p, bn, st);
  if (p.M <= 32) return deep_rows64<EPI, 2>(p, bn, st);
  if (p.M <= 48) return deep_rows64<EPI, 3>(p, bn, st);
  if (p.M <= 64) return deep_rows64<EPI, 4>(p, bn, st);
  if (p.M <= 96) return deep_rows128<EPI, 3, false>(p, bn, st);
  if (p.M <= 128) return deep_rows128<EPI, 4, false>(p, bn, st);
  return p.M <= 192 ? deep_rows128<EPI, 3, true>(p, bn, st) : deep_rows128<EPI, 4, true>(p, bn, st);
}

}  // namespace lsd

using namespace lsd;

// 1 .. 256 rows, whole k-steps; gate / up pairs lie in one tile.  splits > 1 only as slabs:
// the other epilogues run unsplit, whatever the caller asked for.  More than 48 rows only up to
// two blocks a CU (49 .. 64 rows two and a half): behind that the 128 x 128 tiles, which read A half
// as often, are as fast or faster.  Vocabulary-wide, deep ring against those tiles:
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
