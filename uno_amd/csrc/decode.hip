// Few-row products of decode and draft blocks.
//
// A draft block of the two-pass decoder runs every linear layer on B x L rows (128 for 8 sequences
// of 16 rows): the product is a stream of the weight matrix past a small activation tile. The
// training GEMMs tile M and N and give each workgroup the whole K walk; at 128 rows that leaves
// a few dozen workgroups for a 4096-wide output and most of the chip idle. Here every workgroup
// owns one output tile of up to 128 rows and a contiguous range of the K tiles, so the grid is
// (output tiles) x (K ranges) and fills all CUs while each weight element is still read once.
//
// The gated LoRA update y += (m (.) x A^T) (s B)^T rides along: the rows of A are extra output
// columns of the same product (they share the activation stream), and the kernel that adds the K
// ranges' fp32 partial sums (in range order, so the result does not depend on which workgroup
// finished first) also forms the hidden h = bf16(m (.) x A^T) of its rows and applies the rank-r
// update and the epilogue. With one K range and no LoRA the product kernel writes C itself.
#include "common.h"
#include "../../include/unok.h"

#include <type_traits>

namespace {

// RB_K is the unit K ranges are made of, RB_W the waves of a workgroup; RB_D tiles are in flight and
// RB_P activation fragments are read ahead.
constexpr int RB_K = 128, RB_W = 4, RB_D = 3, RB_P = 6;

struct RowsGemm {
  const bf16_t* A; int64_t lda;      // [M, K] activations
  const bf16_t* B; int64_t ldb;      // [N, K] weight
  const bf16_t* LA; int64_t ldla;    // [R, K] LoRA A rows: output columns N .. N + R of the product
  int M, N, K, R;
  int splits;                        // K ranges
  float* ws; int64_t ldw;            // [splits][M][ldw = N + R] fp32 partial sums (split path)
  bf16_t* C; int64_t ldc;            // direct path output
  const bf16_t* Res; int64_t ldres;  // direct path residual
};

// 16 bytes from global memory straight into LDS: lane l writes lds_wave_base + 16 l.
__device__ __forceinline__ void dma16(const void* g, bf16_t* lds_wave_base) {
  __builtin_amdgcn_global_load_lds(g, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}

// s_waitcnt vmcnt(N) through the builtin (expcnt and lgkmcnt left at their maxima), so that the
// compiler's own wait placement knows the loads it covers have completed.
template <int N> __device__ __forceinline__ void rows_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

// Grid: one workgroup per (K range, output column tile, output row tile), row tiles fastest so
// that the row tiles of one weight tile run on the same XCD. Column tiles past N cover the LoRA A
// rows. Wave w owns output columns 16 CW w + [0, 16 CW) of the tile for all 16 TM rows, as CW x TM
// accumulators of 16x16x32 MFMAs whose first operand (16 weight rows x 32 k) it loads straight from
// global memory into registers, RB_D K tiles ahead; consecutive loads take the two 64-byte halves
// of the rows' 128-byte lines, so a load touches 16 lines for 64 bytes each (a 32x32x16 operand
// touches 64 lines for 16 bytes). The 16 TM x BK activation tile, which all waves read, goes to LDS
// by direct-to-LDS loads. Rows beyond M and columns beyond N (R) are clamped to the last valid row
// and never stored. At most 64 KB of LDS and 256 registers leave room for two workgroups per CU, so
// one multiplies while the other waits.
//
// Bound by HBM: each weight is read once. TM follows the row count, so a block of one sequence (16
// rows) multiplies one row tile, and CW the weight (rows_narrow). Measured with cold weights, with
// the reduction below, against 128 x 128 tiles of 32x32x16 MFMAs for every row count: 16 rows, 4096
// -> 6144 30 -> 18.7 us, 4096 -> 24576 68 -> 49 us, 12288 -> 4096 40 -> 31 us, 4096 -> 151936 282 ->
// 231 us (5.4 TB/s); 128 rows 37 -> 29, 84 -> 83, 47 -> 44 and 319 -> 302 us, where LDS reads and the
// activation tiles' own traffic take their share (deeper K tiles and 8-wave workgroups gain nothing).
template <int TM, int CW, bool DIRECT>
__global__ __launch_bounds__(RB_W * 64, 2) void gemm_nt_rows_kernel(const RowsGemm p) {
  constexpr int BM = 16 * TM, NW = RB_W, BN = 16 * CW * NW, BK = TM == 8 ? 64 : 128, D = RB_D, AS = RB_D + 1;
  constexpr int KS = BK / 32;                       // MFMA k-steps per tile
  constexpr int ACH = BK / 8;                       // 16-byte chunks per activation row
  constexpr int A_RPI = 64 / ACH;                   // activation rows per direct-to-LDS load
  constexpr int A_INS = BM / (A_RPI * NW);        // direct-to-LDS loads per wave and tile
  constexpr int W_INS = CW * KS;                    // weight loads per lane and tile
  constexpr int LPT = A_INS + W_INS;
  static_assert(A_INS >= 1 && (D - 1) * LPT < 64, "tile shape");
  extern __shared__ __attribute__((aligned(16))) bf16_t smem[];

  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int nM = (p.M + BM - 1) / BM, nNm = (p.N + BN - 1) / BN;
  const int nN = nNm + (p.LA ? (p.R + BN - 1) / BN : 0);
  const int lin = xcd_remap(blockIdx.x, nM * nN * p.splits);
  const int tm = lin % nM, tn = (lin / nM) % nN, split = lin / (nM * nN);
  const int m0 = tm * BM;
  const bool lora_tile = tn >= nNm;
  // this tile's columns: weight rows n0 .. of B, or LoRA A rows n0 .. of LA (output columns N + n0 ..)
  const int n0 = (lora_tile ? tn - nNm : tn) * BN;
  const int ncols = lora_tile ? p.R : p.N;

  const int nku = p.K / RB_K;
  const int kb = (int)((int64_t)split * nku / p.splits) * (RB_K / BK);
  const int ke = (int)((int64_t)(split + 1) * nku / p.splits) * (RB_K / BK);

  const int lr = lane & 15, lg = lane >> 4;
  const int64_t ldw = lora_tile ? p.ldla : p.ldb;
  const bf16_t* wbase = (lora_tile ? p.LA : p.B) + lg * 8;
  const bf16_t* wrow[CW];
#pragma unroll
  for (int j = 0; j < CW; ++j) wrow[j] = wbase + (int64_t)min(n0 + (wid * CW + j) * 16 + lr, ncols - 1) * ldw;

  // the activation row r's 16-byte chunk c sits in slot c ^ swz(r): the 16 rows one fragment read
  // covers hit 16 different 16-byte groups of the 256-byte bank row
  auto swz = [](int r) { return BK == 64 ? (r >> 1) & 7 : r & 15; };
  const int arow_in = lane / ACH, aslot = lane % ACH;
  auto issue_a = [&](int t, int stage) {
    bf16_t* as = smem + stage * BM * BK;
    const int kk = t * BK;
#pragma unroll
    for (int i = 0; i < A_INS; ++i) {
      const int r = (i * NW + wid) * A_RPI + arow_in;
      const int gm = min(m0 + r, p.M - 1);
      dma16(p.A + (int64_t)gm * p.lda + kk + ((aslot ^ swz(r)) << 3), as + (i * NW + wid) * A_RPI * BK);
    }
  };
  auto issue_w = [&](int t, bf16x8_t (&w)[W_INS]) {
    const int kk = t * BK;
#pragma unroll
    for (int j = 0; j < CW; ++j)
#pragma unroll
      for (int s = 0; s < KS; ++s) w[j * KS + s] = *(const bf16x8_t*)(wrow[j] + kk + s * 32);
  };

  f32x4_t acc[CW][TM];
#pragma unroll
  for (int j = 0; j < CW; ++j)
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[j][i][e] = 0.f;

  // A uniform pipeline over RB_D + 1 weight register sets. Step t waits for tile t, passes the
  // barrier, issues the weight loads of tile t + RB_D, multiplies tile t and then issues the
  // activation loads of tile t + RB_D (past the end: the range's last tile again, into a free
  // stage and set). RB_D weight tiles stay in flight during the multiply, and each wait leaves
  // exactly the RB_D - 1 younger tile groups outstanding. (Activation loads issued before the
  // multiply would make the compiler wait for them before its LDS reads.) The loop runs whole groups
  // of four steps; the last n % 4 tiles, in flight already, are waited for in full: the counted wait
  // would not hold there, because loads that no later step reads are not emitted.
  const int n = ke - kb;
  if (n > 0) {
    bf16x8_t w0[W_INS], w1[W_INS], w2[W_INS], w3[W_INS];
    // (the empty statements keep the three tiles' loads in order, as the counted waits need)
    issue_w(kb, w0);
    issue_a(kb, 0);
    asm volatile("" ::: "memory");
    issue_w(kb + min(1, n - 1), w1);
    issue_a(kb + min(1, n - 1), 1);
    asm volatile("" ::: "memory");
    issue_w(kb + min(2, n - 1), w2);
    issue_a(kb + min(2, n - 1), 2);
    auto multiply = [&](int t, const bf16x8_t (&w)[W_INS]) {
      const bf16_t* as = smem + (t % AS) * BM * BK;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        bf16x8_t a[TM];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int r = i * 16 + lr;
          a[i] = *(const bf16x8_t*)&as[r * BK + (((s * 4 + lg) ^ swz(r)) << 3)];
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < CW; ++j)
            acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j * KS + s], a[i], acc[j][i], 0, 0, 0);
      }
      // fragment reads run RB_P ahead of the multiplies that use them
      constexpr int NR = KS * TM, P = NR < RB_P ? NR : RB_P;
      __builtin_amdgcn_sched_group_barrier(SG_DS_READ, P, 0);
#pragma unroll
      for (int i = 0; i < NR - P; ++i) {
        __builtin_amdgcn_sched_group_barrier(SG_MFMA, CW, 0);
        __builtin_amdgcn_sched_group_barrier(SG_DS_READ, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, CW * P, 0);
    };
    auto step = [&](int t, bf16x8_t (&w)[W_INS], bf16x8_t (&wnext)[W_INS]) {
      rows_wait_vm<(D - 1) * LPT>();
      // each wave waited for its own loads of tile t; after the barrier the tile is in LDS and
      // every wave is past tile t - 1, whose stage the activation refill below reuses
      asm volatile("s_barrier" ::: "memory");
      const int tnext = kb + min(t + D, n - 1);
      issue_w(tnext, wnext);
      __builtin_amdgcn_sched_barrier(0);
      multiply(t, w);
      __builtin_amdgcn_sched_barrier(0);
      issue_a(tnext, (t + D) % AS);
    };
    int t = 0;
    for (; t + 4 <= n; t += 4) {
      step(t, w0, w3);
      step(t + 1, w1, w0);
      step(t + 2, w2, w1);
      step(t + 3, w3, w2);
    }
    rows_wait_vm<0>();
    asm volatile("s_barrier" ::: "memory");
    if (t < n) multiply(t, w0);
    if (t + 1 < n) multiply(t + 1, w1);
    if (t + 2 < n) multiply(t + 2, w2);
  }

  // acc[j][i] of lane l: C[row 16 i + l % 16][cols 16 CW w + 16 j + 4 (l / 16) + 0..3]; N and R are
  // multiples of 4, so the four columns exist together.
#pragma unroll
  for (int j = 0; j < CW; ++j) {
    const int col = n0 + (wid * CW + j) * 16 + lg * 4;
    if (col >= ncols) continue;
    const int64_t wcol = lora_tile ? (int64_t)p.N + col : col;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = m0 + i * 16 + lr;
      if (row >= p.M) continue;
      if constexpr (DIRECT) {
        f32x4_t v = acc[j][i];
        if (p.Res) {
          const uint2 u = *(const uint2*)(p.Res + (int64_t)row * p.ldres + col);
          v[0] += __uint_as_float(u.x << 16); v[1] += __uint_as_float(u.x & 0xffff0000u);
          v[2] += __uint_as_float(u.y << 16); v[3] += __uint_as_float(u.y & 0xffff0000u);
        }
        *(uint2*)(p.C + (int64_t)row * p.ldc + col) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      } else {
        *(f32x4_t*)(p.ws + ((int64_t)split * p.M + row) * p.ldw + wcol) = acc[j][i];
      }
    }
  }
}

// ---------------------------------------------------------------------------------------
// Reduction with the rank-r LoRA update and the epilogue. Workgroup tile: 16 rows x 64 columns
// (EPI 0) or 16 rows x 64 SwiGLU features, i.e. 64 gate and the 64 matching up columns (EPI 1);
// wave w takes columns 16 w + [0, 16) of them.
//   1. every lane starts the loads of its own partials (row l % 16, columns 4 (l / 16) + 0..3 of the
//      wave's) and of its (s B) fragments, so that their latency passes behind step 2;
//   2. h = bf16(m (.) sum of the LoRA-column partials, in range order) of the tile's rows, the hidden
//      columns that its segments read, into LDS;
//   3. the rank-r update h (s B)^T with 16x16x32 MFMAs, whose result lies in exactly the lanes of
//      step 1, then the partials in range order, the update and the residual, rounded once:
// EPI 0: C[M, N]   = bf16(sum + u + Res);
// EPI 1: C[M, N/2] = bf16(silu(g) * u), g = bf16(gate column value), u = bf16(up column value)
//        (the [gate | up] product rounded to bf16 and then the SwiGLU of unok_swiglu_fwd).
// Segment boundaries are multiples of 16, so each wave's 16 columns read one segment of h.
// Bound by latency: one pass of loads, one barrier.
// ---------------------------------------------------------------------------------------
constexpr int RR_ROWS = 16, RR_COLS = 64, RR_HMAX = 512;

struct RowsReduce {
  const float* ws; int64_t ldw; int splits;
  int M, N, R;
  const bf16_t* LB; int64_t ldlb; int r;   // [N, r] (s B); null: no LoRA
  int nseg; int seg_end[4]; int seg_col[4];
  const uint8_t* gate;
  const bf16_t* Res; int64_t ldres;
  bf16_t* C; int64_t ldc;
};

__device__ __forceinline__ int red_seg_col(const RowsReduce& p, int n) {
  int c = p.seg_col[0];
  if (p.nseg > 1 && n >= p.seg_end[0]) c = p.seg_col[1];
  if (p.nseg > 2 && n >= p.seg_end[1]) c = p.seg_col[2];
  if (p.nseg > 3 && n >= p.seg_end[2]) c = p.seg_col[3];
  return c;
}

// Sum of the ranges' partials at src (range stride `plane` floats), in range order; the first eight
// ranges' values are in v already.
__device__ __forceinline__ f32x4_t sum_ranges(const float* src, int64_t plane, int splits, const f32x4_t (&v)[8]) {
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < 8; ++q)
    if (q < splits) acc += v[q];
  for (int k0 = 8; k0 < splits; k0 += 8) {
    f32x4_t w[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (k0 + q < splits) w[q] = *(const f32x4_t*)(src + (k0 + q) * plane);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (k0 + q < splits) acc += w[q];
  }
  return acc;
}

template <int EPI>
__global__ __launch_bounds__(256) void rows_reduce_kernel(const RowsReduce p) {
  constexpr int NH = EPI == 1 ? 2 : 1;             // column groups per lane: (gate, up) or one
  __shared__ __attribute__((aligned(16))) bf16_t Hs[RR_ROWS * (RR_HMAX + 40)];
  const bool lora = p.LB != nullptr;
  const int nout = EPI == 1 ? p.N / 2 : p.N;
  const int ctiles = (nout + RR_COLS - 1) / RR_COLS;
  const int r0 = (blockIdx.x / ctiles) * RR_ROWS;
  const int c0 = (blockIdx.x % ctiles) * RR_COLS;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int lr = lane & 15, lg = lane >> 4;
  const int64_t plane = (int64_t)p.M * p.ldw;

  // 1. own partials (clamped to existing rows and columns)
  const int cbase = c0 + wid * 16 + lg * 4;
  const int row = r0 + lr, lrow = min(row, p.M - 1);
  const float* src[NH];
  f32x4_t v[NH][8];
#pragma unroll
  for (int h = 0; h < NH; ++h) {
    src[h] = p.ws + (int64_t)lrow * p.ldw + min(cbase, nout - 4) + h * nout;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (q < p.splits) v[h][q] = *(const f32x4_t*)(src[h] + q * plane);
  }
  uint2 rv = make_uint2(0, 0);
  if (EPI == 0 && p.Res) rv = *(const uint2*)(p.Res + (int64_t)lrow * p.ldres + min(cbase, nout - 4));
  f32x4_t u[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) u[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (lora) {
    const int wcol = min(c0 + wid * 16, nout - 1);   // first column of the wave's 16
    uint4 lb[NH][4];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const bf16_t* lrow_b = p.LB + (int64_t)(min(c0 + wid * 16 + lr, nout - 1) + h * nout) * p.ldlb;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        const int k = kk * 32 + 8 * lg;
        lb[h][kk] = k < p.r ? *(const uint4*)(lrow_b + k) : make_uint4(0, 0, 0, 0);
      }
    }
    // 2. the hidden columns [h0, h1) that this tile's segments read
    int h0 = p.R, h1 = 0;
#pragma unroll
    for (int t = 0; t < RR_COLS / 16; ++t)
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int c = red_seg_col(p, min(c0 + t * 16, nout - 1) + h * nout);
        h0 = min(h0, c);
        h1 = max(h1, c + p.r);
      }
    h0 &= ~7;
    const int hw4 = (h1 - h0 + 3) / 4;             // columns in fours (R is a multiple of 8)
    const int hld = ((h1 - h0 + 31) & ~31) + 40;   // bf16 row stride: a zero tail of 32 or more, rows spread over banks
    for (int i = tid; i < RR_ROWS * hw4; i += 256) {
      const int rr = i / hw4, j = (i % hw4) * 4;
      const int hrow = min(r0 + rr, p.M - 1);
      const float* hs = p.ws + (int64_t)hrow * p.ldw + p.N + h0 + j;
      f32x4_t x[8];
#pragma unroll
      for (int q = 0; q < 8; ++q)
        if (q < p.splits) x[q] = *(const f32x4_t*)(hs + q * plane);
      const f32x4_t a = sum_ranges(hs, plane, p.splits, x);
      const bool on = p.gate == nullptr || p.gate[hrow] != 0;
      *(uint2*)(Hs + rr * hld + j) = on ? make_uint2(pack2_bf16(a[0], a[1]), pack2_bf16(a[2], a[3])) : make_uint2(0, 0);
    }
    for (int i = tid; i < RR_ROWS * 16; i += 256) *(uint32_t*)(Hs + (i / 16) * hld + hw4 * 4 + (i % 16) * 2) = 0;
    __syncthreads();
    // 3. lane l supplies (s B) of column l % 16 and h of row l % 16 at k = 32 kk + 8 (l / 16) + [0, 8);
    // D element e of lane l is row l % 16, column 4 (l / 16) + e
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const bf16_t* hrow = Hs + lr * hld + red_seg_col(p, wcol + h * nout) - h0;
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        if (kk * 32 >= p.r) break;
        const bf16x8_t hv = *(const bf16x8_t*)(hrow + kk * 32 + 8 * lg);
        u[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, lb[h][kk]), hv, u[h], 0, 0, 0);
      }
    }
  }

  if (cbase >= nout || row >= p.M) return;
  float o[4];
  if constexpr (EPI == 0) {
    f32x4_t a = sum_ranges(src[0], plane, p.splits, v[0]) + u[0];
    if (p.Res) {
      a[0] += __uint_as_float(rv.x << 16); a[1] += __uint_as_float(rv.x & 0xffff0000u);
      a[2] += __uint_as_float(rv.y << 16); a[3] += __uint_as_float(rv.y & 0xffff0000u);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = a[c];
  } else {
    const f32x4_t a = sum_ranges(src[0], plane, p.splits, v[0]) + u[0];
    const f32x4_t b = sum_ranges(src[NH - 1], plane, p.splits, v[NH - 1]) + u[NH - 1];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float g = Elem<bf16_t>::round(a[c]);
      const float w = Elem<bf16_t>::round(b[c]);
      o[c] = g * sigmoidf_(g) * w;
    }
  }
  *(uint2*)(p.C + (int64_t)row * p.ldc + cbase) = make_uint2(pack2_bf16(o[0], o[1]), pack2_bf16(o[2], o[3]));
}

// Row tile of the product in 16-row units.
int rows_tm(int M) { return M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8; }

// Column tile: 64 columns (one MFMA column per wave) put twice the workgroups in flight, 128 read the
// activation tile half as often. With few rows the activations are small next to the weights; with
// more, 64 columns pay only while the weight is small enough for the launch, not the traffic, to
// bound it (64 against 128 columns: 16 rows 4096 -> 24576 49 / 58 us; 32 rows 53 / 57, and 4096 ->
// 151936 245 / 240; 128 rows 4096 -> 4096 21 / 23 us, 12288 -> 4096 47 / 44 us).
bool rows_narrow(int M, int N, int K) {
  return M <= 16 || (int64_t)N * K <= (M <= 32 ? 1ll << 27 : 1ll << 25);
}

int64_t rows_tiles(int M, int N, int K, int R) {
  const int bm = rows_tm(M) * 16, bn = rows_narrow(M, N, K) ? 16 * RB_W : 32 * RB_W;
  return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn + (R + bn - 1) / bn);
}

template <bool DIRECT>
void launch_rows(const RowsGemm& p, unsigned nb, hipStream_t st) {
  auto go = [&](auto tm, auto cw) {
    constexpr int TM = decltype(tm)::value, CW = decltype(cw)::value;
    constexpr size_t lds = (size_t)(RB_D + 1) * 16 * TM * (TM == 8 ? 64 : 128) * sizeof(bf16_t);
    UNOK_SET_LDS_ONCE((gemm_nt_rows_kernel<TM, CW, DIRECT>), lds);
    hipLaunchKernelGGL((gemm_nt_rows_kernel<TM, CW, DIRECT>), dim3(nb), dim3(RB_W * 64), lds, st, p);
  };
  auto by_width = [&](auto tm) {
    if (rows_narrow(p.M, p.N, p.K)) go(tm, std::integral_constant<int, 1>{});
    else if constexpr (decltype(tm)::value > 1) go(tm, std::integral_constant<int, 2>{});
  };
  switch (rows_tm(p.M)) {
    case 1: by_width(std::integral_constant<int, 1>{}); break;
    case 2: by_width(std::integral_constant<int, 2>{}); break;
    case 4: by_width(std::integral_constant<int, 4>{}); break;
    default: by_width(std::integral_constant<int, 8>{});
  }
}

// K ranges for an M x N product (plus R LoRA columns) of nk K tiles: the count that minimises the
// critical path in tile steps (rounds of 256 workgroups times the K tiles of the longest range plus
// two for the pipeline fill), the partial-sum traffic (written and read once, priced at half a
// weight tile step per 32 KB per CU because it stays in the on-chip caches for these sizes) and the
// reduction's serial loads (a quarter step per range). A round counts one workgroup per CU although
// two fit: the weight stream is the bound, and the second shares it rather than adding to it. Over
// 70 products (5 to 256 rows, widths 2048 and 4096, LoRA, SwiGLU and heads, cold weights) the count
// is the best of 12 measured in 54 and at most 7% behind in the others: 16 rows 4096 -> 6144 two
// ranges 20.6 us, the best (five) 19.8; 128 rows 2048 -> 2048 six 16.0, three 15.1; 12288 -> 4096
// seven 42.7 against 160.8 in one.
int rows_auto_splits(int M, int N, int K, int R, bool need_ws) {
  const int64_t tiles = rows_tiles(M, N, K, R);
  const int nk = K >= RB_K ? K / RB_K : 1;
  int best = 1;
  double best_t = 1e30;
  const int smax = nk < 64 ? nk : 64;
  for (int s = 1; s <= smax; ++s) {
    const int64_t wgs = tiles * s;
    const double waves = (double)((wgs + 255) / 256);
    const double steps = waves * (double)((nk + s - 1) / s + 2) + 0.25 * s;
    const double part = (s > 1 || need_ws) ? 0.5 * (double)s * M * (N + R) * 8.0 / (256.0 * 32768.0) : 0.0;
    const double t = steps + part;
    if (t < best_t - 1e-9) { best_t = t; best = s; }
  }
  return best;
}

bool rows_needs_ws(int epilogue, int R, int splits) { return splits > 1 || epilogue != 0 || R > 0; }

// ---------------------------------------------------------------------------------------
// Attention of a draft block over the KV cache, in three kernels per layer:
//   prep     q/k RMSNorm + RoPE of the fused qkv rows (the arithmetic of unok_qknorm_rope_fwd),
//            the block's K and V rows into the caches at (b, kv head, length_b + t), and the
//            queries into the decode layout: the queries of one (sequence, K/V head) pair, rep q
//            heads x L rows, are the first rep * L of 128 rows (row 128 pair + L (h % rep) + t),
//            the rest zero;
//   attn     unok_attn_fwd_split over S key ranges of each pair's cache rows;
//   combine  the S partial rows of each query merged by their log-sum-exp weights and written to
//            the attention output [B * L, nq * D] at (b * L + t, head h).
// ---------------------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void decode_prep_kernel(const bf16_t* __restrict__ qkv, int64_t ld,
                                                          const bf16_t* __restrict__ wq, const bf16_t* __restrict__ wk,
                                                          const int64_t* __restrict__ lengths,
                                                          const float* __restrict__ inv_freq, float eps,
                                                          bf16_t* __restrict__ kc, bf16_t* __restrict__ vc,
                                                          int max_len, bf16_t* __restrict__ qd, int B, int L, int nq,
                                                          int nk) {
  constexpr int LPH = D / 8, HALF = D / 2;          // lanes per head row, 8 elements per lane
  const int lane = threadIdx.x & 63;
  const int64_t item = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPH;
  const int sub = lane % LPH, c0 = sub * 8;
  const int M = B * L, nh = nq + 2 * nk, rep = nq / nk;
  const int64_t heads = (int64_t)M * nh;
  const int pad = 128 - rep * L;
  if (item >= heads) {
    // zero padding rows of the decode query layout
    const int64_t z = item - heads;
    if (z >= (int64_t)B * nk * pad) return;
    const int64_t row = (z / pad) * 128 + rep * L + z % pad;
    *(uint4*)(qd + row * D + c0) = make_uint4(0, 0, 0, 0);
    return;
  }
  const int m = (int)(item / nh), hd = (int)(item % nh);
  const int b = m / L, t = m % L;
  const int64_t len = lengths[b];
  float x[8];
  {
    const uint4 u = *(const uint4*)(qkv + (int64_t)m * ld + (int64_t)hd * D + c0);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) { x[2 * i] = __uint_as_float(w[i] << 16); x[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u); }
  }
  bf16_t* dst;
  if (hd < nq + nk) {
    const bool isq = hd < nq;
    const bf16_t* wn = isq ? wq : wk;
    if (wn != nullptr) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) ss += x[e] * x[e];
#pragma unroll
      for (int o = LPH / 2; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      const float r = rsqrtf(ss / (float)D + eps);
      const uint4 u = *(const uint4*)(wn + c0);
      const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w0 = __uint_as_float(w[i] << 16), w1 = __uint_as_float(w[i] & 0xffff0000u);
        x[2 * i] = x[2 * i] * r * w0;
        x[2 * i + 1] = x[2 * i + 1] * r * w1;
      }
    }
    const float p = (float)(len + t);
    const int j0 = c0 % HALF;
    const float sgn = c0 < HALF ? -1.f : 1.f;
    float out[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float sv, cv;
      sincosf(p * inv_freq[j0 + e], &sv, &cv);
      const float y = __shfl_xor(x[e], LPH / 2, 64);   // partner element i +- d/2
      out[e] = x[e] * cv + sgn * y * sv;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = out[e];
    if (isq) {
      const int kv = hd / rep, rr = hd % rep;
      dst = qd + ((int64_t)(b * nk + kv) * 128 + rr * L + t) * D;
    } else {
      if (len + t >= max_len) return;
      dst = kc + ((int64_t)(b * nk + hd - nq) * max_len + len + t) * D;
    }
  } else {
    if (len + t >= max_len) return;
    dst = vc + ((int64_t)(b * nk + hd - nq - nk) * max_len + len + t) * D;
  }
  *(uint4*)(dst + c0) = make_uint4(pack2_bf16(x[0], x[1]), pack2_bf16(x[2], x[3]), pack2_bf16(x[4], x[5]),
                                   pack2_bf16(x[6], x[7]));
}

// Row maps of a draft block's attention from the committed lengths, one thread per (range, decode
// row): range s of the S key ranges of a query row holds keys [s c, (s + 1) c) of its causal prefix
// (c = committed length / S), the last range the rest; padding rows have empty ranges and dst -1.
__global__ __launch_bounds__(256) void decode_maps_kernel(const int64_t* __restrict__ lengths, int L, int nq, int nk,
                                                          int max_len, int S, int QR, int4* __restrict__ ivs,
                                                          int32_t* __restrict__ dst) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= S * QR) return;
  const int s = i / QR, q = i % QR, pair = q / 128, slot = q % 128, rep = nq / nk;
  const bool valid = slot < rep * L;
  const int t = slot % L;
  const int64_t len = lengths[pair / nk], seen = len + t + 1, c = len / S;
  const int64_t start = (int64_t)pair * max_len;
  const int64_t lo = s * c, hi = s == S - 1 ? seen : min((s + 1) * c, seen);
  ivs[2 * i] = make_int4((int)(start + (valid ? lo : 0)), (int)(start + (valid ? max(hi, lo) : 0)), 0, 0);
  ivs[2 * i + 1] = make_int4(0, 0, 0, 0);
  if (s == 0) dst[q] = valid ? ((pair / nk) * L + t) * nq + (pair % nk) * rep + slot / L : -1;
}

// O[dst[i]] = sum_s 2^(lse_s - m) O_s[i] / sum_s 2^(lse_s - m) over the S partial rows s * QR + i
// (lse in log2 units, m their maximum; a range without keys has lse = -inf and weight 0); rows
// with dst[i] < 0 are skipped.
template <int D>
__global__ __launch_bounds__(256) void attn_split_combine_kernel(const bf16_t* __restrict__ op, int64_t ldp,
                                                                 const float* __restrict__ lse,
                                                                 const int32_t* __restrict__ dst, int QR, int S,
                                                                 bf16_t* __restrict__ out, int64_t ldo) {
  constexpr int LPR = D / 8;
  const int64_t item = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  if (item >= QR) return;
  const int i = (int)item, c0 = (threadIdx.x % LPR) * 8;
  const int d = dst[i];
  if (d < 0) return;
  // eight ranges' rows in flight at a time; the ranges are few, so their weights are read twice
  float m = -INFINITY;
  for (int s0 = 0; s0 < S; s0 += 8) {
    float l[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) l[q] = s0 + q < S ? lse[(int64_t)(s0 + q) * QR + i] : -INFINITY;
#pragma unroll
    for (int q = 0; q < 8; ++q) m = fmaxf(m, l[q]);
  }
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float wsum = 0.f;
  if (m != -INFINITY) {
    for (int s0 = 0; s0 < S; s0 += 8) {
      float l[8];
      uint4 u[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int64_t r = (int64_t)min(s0 + q, S - 1) * QR + i;
        l[q] = s0 + q < S ? lse[r] : -INFINITY;
        u[q] = *(const uint4*)(op + r * ldp + c0);
      }
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        if (l[q] == -INFINITY) continue;
        const float w = exp2f(l[q] - m);
        wsum += w;
        const uint32_t v[4] = {u[q].x, u[q].y, u[q].z, u[q].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          acc[2 * k] += w * __uint_as_float(v[k] << 16);
          acc[2 * k + 1] += w * __uint_as_float(v[k] & 0xffff0000u);
        }
      }
    }
  }
  const float inv = wsum > 0.f ? 1.f / wsum : 0.f;
  *(uint4*)(out + (int64_t)d * ldo + c0) =
      make_uint4(pack2_bf16(acc[0] * inv, acc[1] * inv), pack2_bf16(acc[2] * inv, acc[3] * inv),
                 pack2_bf16(acc[4] * inv, acc[5] * inv), pack2_bf16(acc[6] * inv, acc[7] * inv));
}

}  // namespace

// Workspace bytes of unok_gemm_nt_rows for this shape (R = 0 without LoRA; splits <= 0: the
// automatic count).
UNOK_EXPORT int64_t unok_gemm_nt_rows_workspace(int M, int N, int K, int R, int epilogue, int splits) {
  if (M <= 0 || N <= 0 || K <= 0 || R < 0) return 0;
  const int s = splits > 0 ? splits : rows_auto_splits(M, N, K, R, epilogue != 0 || R > 0);
  if (!rows_needs_ws(epilogue, R, s)) return 0;
  return (int64_t)s * M * (N + R) * (int64_t)sizeof(float);
}

UNOK_EXPORT int unok_gemm_nt_rows(int M, int N, int K, const void* A, int64_t lda, const void* B, int64_t ldb,
                                  const void* LA, int64_t ldla, int R, const void* LB, int64_t ldlb, int r,
                                  int nseg, const int* seg_end, const int* seg_col,
                                  void* C, int64_t ldc, const void* Res, int64_t ldres, const uint8_t* gate,
                                  int epilogue, int splits, void* workspace, int64_t ws_bytes, void* stream) {
  UNOK_REQUIRE(M >= 0 && N >= 0 && K >= 0, UNOK_EINVAL, "gemm_nt_rows: negative size M=%d N=%d K=%d", M, N, K);
  if (M == 0 || N == 0) return 0;
  UNOK_REQUIRE(epilogue == 0 || epilogue == 1, UNOK_EINVAL, "gemm_nt_rows: epilogue %d is not 0 or 1", epilogue);
  UNOK_REQUIRE(K > 0 && K % RB_K == 0, UNOK_EINVAL, "gemm_nt_rows: K=%d must be a positive multiple of 128", K);
  UNOK_REQUIRE(lda % 8 == 0 && ldb % 8 == 0 && ((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0, UNOK_EALIGN,
               "gemm_nt_rows: lda=%lld ldb=%lld must be multiples of 8 and A/B 16-byte aligned", (long long)lda,
               (long long)ldb);
  UNOK_REQUIRE(N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C & 7) == 0, UNOK_EALIGN,
               "gemm_nt_rows: N=%d and ldc=%lld must be multiples of 4 and C 8-byte aligned", N, (long long)ldc);
  UNOK_REQUIRE(epilogue == 0 || N % 32 == 0, UNOK_EINVAL, "gemm_nt_rows: the SwiGLU epilogue needs N=%d a multiple of 32",
               N);
  UNOK_REQUIRE(epilogue == 0 || Res == nullptr, UNOK_EINVAL, "gemm_nt_rows: the SwiGLU epilogue takes no residual");
  UNOK_REQUIRE(Res == nullptr || (ldres % 4 == 0 && ((uintptr_t)Res & 7) == 0), UNOK_EALIGN,
               "gemm_nt_rows: ldres=%lld must be a multiple of 4 and Res 8-byte aligned", (long long)ldres);
  const bool lora = LA != nullptr;
  RowsReduce q{};
  q.nseg = 1;
  for (int i = 0; i < 4; ++i) { q.seg_end[i] = N; q.seg_col[i] = 0; }
  if (lora) {
    UNOK_REQUIRE(R > 0 && R <= 512 && R % 8 == 0 && LB != nullptr && r > 0 && r <= 128 && r % 8 == 0, UNOK_EINVAL,
                 "gemm_nt_rows: LoRA needs 0 < R <= 512 A rows (a multiple of 8) and a rank 0 < r <= 128 "
                 "(a multiple of 8), got R=%d r=%d", R, r);
    UNOK_REQUIRE(ldla % 8 == 0 && ((uintptr_t)LA & 15) == 0 && ldlb % 8 == 0 && ((uintptr_t)LB & 15) == 0,
                 UNOK_EALIGN, "gemm_nt_rows: ldla=%lld ldlb=%lld must be multiples of 8 and LA/LB 16-byte aligned",
                 (long long)ldla, (long long)ldlb);
    if (nseg > 0) {
      UNOK_REQUIRE(nseg <= 4 && seg_end && seg_col, UNOK_EINVAL, "gemm_nt_rows: at most 4 segments");
      q.nseg = nseg;
      for (int i = 0; i < nseg; ++i) {
        q.seg_end[i] = seg_end[i];
        q.seg_col[i] = seg_col[i];
        UNOK_REQUIRE(seg_col[i] >= 0 && seg_col[i] % 8 == 0 && seg_col[i] + r <= R, UNOK_EINVAL,
                     "gemm_nt_rows: segment %d reads LoRA hidden columns %d..%d of %d (start a multiple of 8)", i, seg_col[i],
                     seg_col[i] + r, R);
        UNOK_REQUIRE(i + 1 == nseg || seg_end[i] % 16 == 0, UNOK_EINVAL,
                     "gemm_nt_rows: segment end %d not a multiple of 16", seg_end[i]);
      }
      UNOK_REQUIRE(seg_end[nseg - 1] == N, UNOK_EINVAL, "gemm_nt_rows: last segment must end at N");
    } else {
      UNOK_REQUIRE(r <= R, UNOK_EINVAL, "gemm_nt_rows: rank %d exceeds the %d LoRA A rows", r, R);
    }
  } else {
    R = 0;
  }
  const int nk = K / RB_K;
  const int s = splits > 0 ? splits : rows_auto_splits(M, N, K, R, epilogue != 0 || lora);
  UNOK_REQUIRE(s <= nk, UNOK_EINVAL, "gemm_nt_rows: %d K ranges for %d K tiles", s, nk);

  RowsGemm p{};
  p.A = (const bf16_t*)A; p.lda = lda;
  p.B = (const bf16_t*)B; p.ldb = ldb;
  p.LA = lora ? (const bf16_t*)LA : nullptr; p.ldla = ldla;
  p.M = M; p.N = N; p.K = K; p.R = R;
  p.splits = s;
  const int64_t nb = rows_tiles(M, N, K, R) * s;
  UNOK_REQUIRE(nb < (1ll << 31), UNOK_EINVAL, "gemm_nt_rows: grid too large");
  hipStream_t st = (hipStream_t)stream;
  if (!rows_needs_ws(epilogue, R, s)) {
    p.C = (bf16_t*)C; p.ldc = ldc; p.Res = (const bf16_t*)Res; p.ldres = ldres;
    launch_rows<true>(p, (unsigned)nb, st);
    return unok::check_launch("gemm_nt_rows");
  }
  const int64_t need = (int64_t)s * M * (N + R) * (int64_t)sizeof(float);
  UNOK_REQUIRE(workspace != nullptr && ws_bytes >= need && ((uintptr_t)workspace & 15) == 0, UNOK_EINVAL,
               "gemm_nt_rows: workspace of %lld bytes (16-byte aligned) required, got %lld", (long long)need,
               (long long)ws_bytes);
  p.ws = (float*)workspace; p.ldw = N + R;
  launch_rows<false>(p, (unsigned)nb, st);
  int rc = unok::check_launch("gemm_nt_rows");
  if (rc) return rc;

  q.ws = (const float*)workspace; q.ldw = N + R; q.splits = s;
  q.M = M; q.N = N; q.R = R;
  q.LB = lora ? (const bf16_t*)LB : nullptr; q.ldlb = ldlb; q.r = lora ? r : 0;
  q.gate = gate;
  q.Res = (const bf16_t*)Res; q.ldres = ldres;
  q.C = (bf16_t*)C; q.ldc = ldc;
  const int nout = epilogue == 1 ? N / 2 : N;
  const int64_t blocks = (int64_t)((M + RR_ROWS - 1) / RR_ROWS) * ((nout + RR_COLS - 1) / RR_COLS);
  if (epilogue == 0)
    hipLaunchKernelGGL((rows_reduce_kernel<0>), dim3((unsigned)blocks), dim3(256), 0, st, q);
  else
    hipLaunchKernelGGL((rows_reduce_kernel<1>), dim3((unsigned)blocks), dim3(256), 0, st, q);
  return unok::check_launch("gemm_nt_rows_reduce");
}

// q/k norm + RoPE of a draft block's fused qkv rows, its K/V rows into the caches and its queries
// into the decode layout (see decode_prep_kernel). bf16; D in {64, 128}; wq / wk null: no q/k norm.
UNOK_EXPORT int unok_decode_prep(int B, int L, int nq, int nk, int D, const void* qkv, int64_t ld, const void* wq,
                                 const void* wk, const int64_t* lengths, const float* inv_freq, float eps, void* kc,
                                 void* vc, int max_len, void* qd, void* stream) {
  UNOK_REQUIRE(B >= 0 && L >= 0 && nq > 0 && nk > 0 && nq % nk == 0, UNOK_EINVAL,
               "decode_prep: B=%d L=%d nq=%d nk=%d", B, L, nq, nk);
  if (B == 0 || L == 0) return 0;
  UNOK_REQUIRE(D == 64 || D == 128, UNOK_EINVAL, "decode_prep: head dim %d not in {64,128}", D);
  UNOK_REQUIRE((nq / nk) * L <= 128, UNOK_EINVAL, "decode_prep: %d q heads x %d rows exceed 128 rows per K/V head",
               nq / nk, L);
  UNOK_REQUIRE(ld % 8 == 0 && ((uintptr_t)qkv & 15) == 0 && ((uintptr_t)kc & 15) == 0 && ((uintptr_t)vc & 15) == 0 &&
                   ((uintptr_t)qd & 15) == 0 && (wq == nullptr || ((uintptr_t)wq & 15) == 0) &&
                   (wk == nullptr || ((uintptr_t)wk & 15) == 0),
               UNOK_EALIGN, "decode_prep: rows must be 16-byte aligned");
  const int64_t heads = (int64_t)B * L * (nq + 2 * nk);
  const int64_t pads = (int64_t)B * nk * (128 - (nq / nk) * L);
  const int lph = D / 8;
  const int64_t blocks = ((heads + pads) * lph + 255) / 256;
  hipStream_t st = (hipStream_t)stream;
  if (D == 128)
    hipLaunchKernelGGL((decode_prep_kernel<128>), dim3((unsigned)blocks), dim3(256), 0, st, (const bf16_t*)qkv, ld,
                       (const bf16_t*)wq, (const bf16_t*)wk, lengths, inv_freq, eps, (bf16_t*)kc, (bf16_t*)vc, max_len,
                       (bf16_t*)qd, B, L, nq, nk);
  else
    hipLaunchKernelGGL((decode_prep_kernel<64>), dim3((unsigned)blocks), dim3(256), 0, st, (const bf16_t*)qkv, ld,
                       (const bf16_t*)wq, (const bf16_t*)wk, lengths, inv_freq, eps, (bf16_t*)kc, (bf16_t*)vc, max_len,
                       (bf16_t*)qd, B, L, nq, nk);
  return unok::check_launch("decode_prep");
}

// Merge of the S partial rows of split-key attention (see attn_split_combine_kernel). bf16.
UNOK_EXPORT int unok_attn_split_combine(int QR, int S, int D, const void* opart, int64_t ldp, const float* lse,
                                        const int32_t* dst, void* out, int64_t ldo, void* stream) {
  UNOK_REQUIRE(QR >= 0 && S >= 1, UNOK_EINVAL, "attn_split_combine: QR=%d S=%d", QR, S);
  if (QR == 0) return 0;
  UNOK_REQUIRE(D == 64 || D == 128, UNOK_EINVAL, "attn_split_combine: head dim %d not in {64,128}", D);
  UNOK_REQUIRE(ldp % 8 == 0 && ldo % 8 == 0 && ((uintptr_t)opart & 15) == 0 && ((uintptr_t)out & 15) == 0, UNOK_EALIGN,
               "attn_split_combine: rows must be 16-byte aligned");
  const int64_t blocks = ((int64_t)QR * (D / 8) + 255) / 256;
  hipStream_t st = (hipStream_t)stream;
  if (D == 128)
    hipLaunchKernelGGL((attn_split_combine_kernel<128>), dim3((unsigned)blocks), dim3(256), 0, st,
                       (const bf16_t*)opart, ldp, lse, dst, QR, S, (bf16_t*)out, ldo);
  else
    hipLaunchKernelGGL((attn_split_combine_kernel<64>), dim3((unsigned)blocks), dim3(256), 0, st,
                       (const bf16_t*)opart, ldp, lse, dst, QR, S, (bf16_t*)out, ldo);
  return unok::check_launch("attn_split_combine");
}

// Key intervals (ivs, [S * QR, 8] int32) and output rows (dst, [QR] int32) of a draft block's split-key
// attention, QR = 128 B nk decode rows (see decode_maps_kernel).
UNOK_EXPORT int unok_decode_maps(int B, int L, int nq, int nk, int max_len, int S, const int64_t* lengths, int32_t* ivs,
                                 int32_t* dst, void* stream) {
  UNOK_REQUIRE(B >= 0 && L >= 0 && nq > 0 && nk > 0 && nq % nk == 0 && S >= 1 && max_len >= 0, UNOK_EINVAL,
               "decode_maps: B=%d L=%d nq=%d nk=%d S=%d max_len=%d", B, L, nq, nk, S, max_len);
  if (B == 0 || L == 0) return 0;
  const int64_t rows = (int64_t)B * nk * 128 * S;
  UNOK_REQUIRE((nq / nk) * L <= 128 && rows < (1ll << 30) && (int64_t)B * nk * max_len < (1ll << 31) &&
                   (int64_t)B * L * nq < (1ll << 31),
               UNOK_EINVAL, "decode_maps: B=%d L=%d max_len=%d S=%d exceed the row layout", B, L, max_len, S);
  UNOK_REQUIRE(((uintptr_t)ivs & 15) == 0, UNOK_EALIGN, "decode_maps: ivs must be 16-byte aligned");
  hipLaunchKernelGGL(decode_maps_kernel, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, (hipStream_t)stream, lengths,
                     L, nq, nk, max_len, S, B * nk * 128, (int4*)ivs, dst);
  return unok::check_launch("decode_maps");
}

// ---------------------------------------------------------------------------------------
// One decoder layer of a draft block: its 13 kernels in order, launched from here. A layer of a small
// model runs for less time than the nine calls take that make them one by one from Python.
// ---------------------------------------------------------------------------------------
namespace {

struct DraftBuffers {
  int64_t x, qkv, qd, op, lse, o, h1, s, ws, bytes;
};

DraftBuffers draft_buffers(const unok_draft_layer_args& a) {
  const int64_t M = (int64_t)a.B * a.L, q = (int64_t)a.nq * a.D, kv = (int64_t)a.nk * a.D;
  const int64_t QR = (int64_t)a.B * a.nk * 128;
  DraftBuffers b;
  int64_t at = 0;
  auto take = [&](int64_t n) { const int64_t p = at; at += (n + 255) / 256 * 256; return p; };
  b.x = take(M * a.H * 2);
  b.qkv = take(M * (q + 2 * kv) * 2);
  b.qd = take(QR * a.D * 2);
  b.op = take(QR * a.S * a.D * 2);
  b.lse = take(QR * a.S * 4);
  b.o = take(M * q * 2);
  b.h1 = take(M * a.H * 2);
  b.s = take(M * a.F * 2);
  const int64_t need[4] = {unok_gemm_nt_rows_workspace((int)M, (int)(q + 2 * kv), a.H, 3 * a.r, 0, 0),
                           unok_gemm_nt_rows_workspace((int)M, a.H, (int)q, a.r, 0, 0),
                           unok_gemm_nt_rows_workspace((int)M, 2 * a.F, a.H, 2 * a.r, 1, 0),
                           unok_gemm_nt_rows_workspace((int)M, a.H, a.F, a.r, 0, 0)};
  int64_t most = 0;
  for (int64_t n : need) most = n > most ? n : most;
  b.ws = take(most);
  b.bytes = at;
  return b;
}

int draft_sizes_ok(const unok_draft_layer_args* a) {
  UNOK_REQUIRE(a != nullptr && a->B >= 0 && a->L >= 0 && a->nq > 0 && a->nk > 0 && a->nq % a->nk == 0 && a->H > 0 &&
                   a->F > 0 && a->r > 0 && a->S >= 1 && (a->D == 64 || a->D == 128) &&
                   (int64_t)a->B * a->L < (1 << 24) && (int64_t)a->nq * a->D < (1 << 24) && a->F < (1 << 24),
               UNOK_EINVAL, "draft_layer: bad sizes");
  return 0;
}

}  // namespace

UNOK_EXPORT int64_t unok_draft_layer_scratch(const unok_draft_layer_args* a) {
  if (draft_sizes_ok(a)) return -1;
  return draft_buffers(*a).bytes;
}

UNOK_EXPORT int unok_draft_layer(const unok_draft_layer_args* a, void* stream) {
  int rc = draft_sizes_ok(a);
  if (rc || a->B == 0 || a->L == 0) return rc;
  for (const void* q : {a->ln_in, a->ln_post, a->w_qkv, a->a_qkv, a->b_qkv, a->w_o, a->a_o, a->b_o, a->w_gu, a->a_gu, a->b_gu,
                        a->w_d, a->a_d, a->b_d, (const void*)a->kc, (const void*)a->vc, (const void*)a->lengths,
                        (const void*)a->inv_freq, (const void*)a->gate, (const void*)a->ivs, (const void*)a->dst, a->h,
                        (const void*)a->h_out})
    UNOK_REQUIRE(q != nullptr, UNOK_EINVAL, "draft_layer: null operand");
  UNOK_REQUIRE(a->h != a->h_out, UNOK_EINVAL, "draft_layer: h and h_out may not overlap");
  const DraftBuffers b = draft_buffers(*a);
  UNOK_REQUIRE(a->scratch != nullptr && a->scratch_bytes >= b.bytes && ((uintptr_t)a->scratch & 255) == 0, UNOK_EINVAL,
               "draft_layer: scratch of %lld bytes (256-byte aligned) required, got %lld", (long long)b.bytes,
               (long long)a->scratch_bytes);
  const int M = a->B * a->L, q = a->nq * a->D, kv = a->nk * a->D, H = a->H, F = a->F, r = a->r, QR = a->B * a->nk * 128;
  char* base = (char*)a->scratch;
  void *x = base + b.x, *qkv = base + b.qkv, *qd = base + b.qd, *op = base + b.op, *o = base + b.o, *h1 = base + b.h1,
       *s = base + b.s, *ws = base + b.ws;
  float* lse = (float*)(base + b.lse);
  const int64_t ws_bytes = b.bytes - b.ws;
  const int qkv_end[3] = {q, q + kv, q + 2 * kv}, qkv_col[3] = {0, r, 2 * r};
  const int gu_end[2] = {F, 2 * F}, gu_col[2] = {0, r};
  auto linear = [&](const void* in, int K, const void* w, const void* la, const void* lb, int N, int nseg, const int* end,
                    const int* col, const void* res, int epi, void* out) {
    return unok_gemm_nt_rows(M, N, K, in, K, w, K, la, K, (nseg ? nseg : 1) * r, lb, r, r, nseg, end, col, out,
                             epi ? N / 2 : N, res, N, a->gate, epi, 0, ws, ws_bytes, stream);
  };
  if ((rc = unok_rmsnorm_fwd(UNOK_BF16, M, H, a->h, H, a->ln_in, x, H, nullptr, a->eps, stream))) return rc;
  if ((rc = linear(x, H, a->w_qkv, a->a_qkv, a->b_qkv, q + 2 * kv, 3, qkv_end, qkv_col, nullptr, 0, qkv))) return rc;
  if ((rc = unok_decode_prep(a->B, a->L, a->nq, a->nk, a->D, qkv, q + 2 * kv, a->q_norm, a->k_norm, a->lengths,
                             a->inv_freq, a->eps, a->kc, a->vc, a->max_len, qd, stream)))
    return rc;
  if ((rc = unok_attn_fwd_split(QR, a->S, a->D, qd, a->D, a->kc, a->D, a->vc, a->D, a->ivs, op, a->D, lse, a->scale, stream)))
    return rc;
  if ((rc = unok_attn_split_combine(QR, a->S, a->D, op, a->D, lse, a->dst, o, a->D, stream))) return rc;
  if ((rc = linear(o, q, a->w_o, a->a_o, a->b_o, H, 0, nullptr, nullptr, a->h, 0, h1))) return rc;
  if ((rc = unok_rmsnorm_fwd(UNOK_BF16, M, H, h1, H, a->ln_post, x, H, nullptr, a->eps, stream))) return rc;
  if ((rc = linear(x, H, a->w_gu, a->a_gu, a->b_gu, 2 * F, 2, gu_end, gu_col, nullptr, 1, s))) return rc;
  return linear(s, F, a->w_d, a->a_d, a->b_d, H, 0, nullptr, nullptr, h1, 0, a->h_out);
}
