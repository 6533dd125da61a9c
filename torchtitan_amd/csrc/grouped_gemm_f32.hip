// fp32 grouped GEMMs for the MoE experts in fp32 on MI355X (gfx950).
//
// The reference's readability path _run_experts_for_loop
// (torchtitan/models/common/moe.py:24-50) multiplies each expert's token
// segment in the input dtype: for fp32 models every product and sum is fp32.
// These kernels do the same arithmetic for all experts in one launch per GEMM,
// on v_mfma_f32_16x16x4f32 (fp32 operands, fp32 accumulation), with the
// SwiGLU of :41-43 and its autograd fused into the epilogues:
//   gate_up  g = x w1^T, u = x w3^T, h = silu(g) * u        (fp32 each)
//   down     y = h w2^T
//   bwd_dgu  dh = dy w2; du = dh * silu(g); dg = silu'(g) * (dh * u)
//   bwd_dx   dx = dg w1 + du w3
//   bwd_dw   out[e] = a_e^T b_e over expert e's rows (dw1, dw3, dw2)
//
// Tiles: 64 x 64 outputs, 32 of k per LDS stage, two stages (one in dW of few rows); eight
// waves per workgroup in the row modes, four in dW. What bounds fp32 is the matrix cores (a 16 x 16 x 4 MFMA
// takes 32 clocks; 154 TFLOP/s measured over a large product) and, at few tiles, how
// evenly 64 x 64 tiles fall on the CUs, so the rest has to stay out of their way:
// operands go to LDS by direct-to-LDS copies (16 bytes a lane, no staging registers or
// LDS stores), and every LDS read is one 8- or 16-byte read that feeds two or four MFMAs.
// Which k a lane group supplies to an MFMA is free as long as both operands agree: step
// (h, j) takes k = 16 h + 4 g + j from lane group g = lane / 16, so that
//  * a k-contiguous operand (rows of 128 bytes, 16-byte chunk c of row r at c ^ (r & 7))
//    gives a lane the operands of four steps in one 16-byte read of its row;
//  * a k-major operand (32 k-rows of 64 columns, chunk c of k-row k at
//    c ^ 8 ((k >> 2) & 1)) gives a lane two neighbouring columns of its k, which go to two
//    MFMA tiles: tile q holds columns 2 i + q, and a lane's results over the tiles are
//    contiguous in the output row.
// All of these reads are free of bank conflicts.
// Measured (us, against scalar LDS reads of register-staged 16-deep tiles, four waves) at
// 8192 rows of 8 experts, dim 256, hidden 512 | 16384 rows, 512, 1024: gate_up 59 -> 56 |
// 329 -> 319, down 37 -> 33 | 187 -> 166, dgu 40 -> 37 | 222 -> 184, dx 67 -> 64 | 354 ->
// 344, the three dW (one launch, before three) 157 -> 82 | 765 -> 542. Without copies and
// stores gate_up still takes 43 | 264 us: the MFMAs at the clock they leave. Three stages
// measured the same as two.
// Row-grouped modes map workgroups to (expert, 64-row tile) from a scan of the counts,
// so no host sync or padding is needed; surplus workgroups exit.
#include "common.h"

namespace moe {
namespace f32g {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
#define LDSP __attribute__((address_space(3)))

constexpr int kMaxE = 1024;
constexpr int BM = 64, BN = 64, BK = 32;
constexpr int kTile = 64 * BK;  // floats of one operand's stage (8 KB)

enum Mode : int { kGateUp = 0, kDown = 1, kDgu = 2, kDx = 3 };

struct Params {
  const int64_t* counts;
  int64_t R;
  int E;
  int N, K;        // N output columns, K contraction (dx: of each half)
  const float* a;  // row operand [R, K]
  const float* a2; // second row operand (dx: du)
  const float* b;  // NT: [E, N, K]; NN: [E, K, N]
  const float* b2; // second weight (gate_up: w3; dx: w3)
  const float* g;  // dgu: saved g, u [R, N]
  const float* u;
  float* o0;
  float* o1;
  float* o2;
};

__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }

__device__ const float4 kZeroChunk[4] = {};  // source of the k-rows past a segment

// global accesses of four floats: any tensor of floats, 16-byte aligned or not
typedef f32x4_t f32x4_u __attribute__((aligned(4)));

// lane i's 16 bytes at g land at LDS byte address lds + 16 i: a direct-to-LDS copy, or,
// where an operand is not 16-byte aligned, through registers
template <bool ALIGNED>
__device__ __forceinline__ void copy16(const float* g, uint32_t lds) {
  if constexpr (ALIGNED)
    asm volatile("global_load_lds_dwordx4 %0, off" :: "v"(g), "{m0}"(lds) : "memory");
  else
    *(LDSP f32x4_t*)(size_t)(lds + 16 * (threadIdx.x & 63)) = *(const f32x4_u*)g;
}
__device__ __forceinline__ uint32_t lds_addr(float* p) { return (uint32_t)(size_t)((LDSP float*)p); }

// Expert segments: rows [start, start + count) clamped to R.
struct Seg { int start, count; };

// This lane's experts 4 t .. 4 t + 3 of the counts (t = threadIdx.x) with their starts,
// counts cut where they run past R.
__device__ __forceinline__ void scan_counts(const int64_t* counts, int64_t R, int E, int* s_tmp, int (&st)[4],
                                            int (&cnt)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ee = threadIdx.x * 4 + i;
    const int64_t c = ee < E ? counts[ee] : 0;
    cnt[i] = c < 0 ? 0 : (int)(c > R ? R : c);
  }
  block_exclusive_scan4(cnt, st, s_tmp);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t room = R - st[i];
    cnt[i] = room <= 0 ? 0 : (cnt[i] > room ? (int)room : cnt[i]);
  }
}

// This workgroup's tile: the expert, its 64 rows mt and 64 columns nt of the ntn; e = -1
// where there is none. Workgroup b runs on XCD b % 8, and each XCD takes an eighth of the
// tiles, neighbouring ones (they share an operand in its L2): of the tiles that the counts
// make, not of the grid, which is sized for every row and the worst raggedness. An order over
// the grid left XCDs idle: with 8192 of 65536 rows in use (8 experts, dim 512, hidden 1024)
// every tile was on one, gate_up 1154 us, now 193; with all of 8192 rows in use (dim 256,
// hidden 512) the surplus was all on one, forward 92 -> 77 us, backward 163 -> 140.
// Every thread of the block must call it.
__device__ __forceinline__ void find_tile(const Params& p, int ntn, int* s_tmp, int* s_out, int& e, Seg& seg, int& mt,
                                          int& nt) {
  int cnt[4], st[4], tiles[4], tst[4];
  scan_counts(p.counts, p.R, p.E, s_tmp, st, cnt);
#pragma unroll
  for (int i = 0; i < 4; ++i) tiles[i] = (cnt[i] + BM - 1) / BM;
  const int total = block_exclusive_scan4(tiles, tst, s_tmp);
  const int b = workgroup(), eighth = (total * ntn + 7) / 8, t = (b & 7) * eighth + (b >> 3);
  const int bx = (b >> 3) < eighth ? t / ntn : total;
  nt = t % ntn;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ee = threadIdx.x * 4 + i;
    if (ee < p.E && bx >= tst[i] && bx < tst[i] + tiles[i]) {
      s_out[0] = ee;
      s_out[1] = st[i];
      s_out[2] = cnt[i];
      s_out[3] = tst[i];
    }
  }
  if (bx >= total && threadIdx.x == 0) s_out[0] = -1;
  __syncthreads();
  e = s_out[0];
  seg.start = s_out[1];
  seg.count = s_out[2];
  mt = bx - s_out[3];
}

// dW: start and count of expert e's rows, cut where they run past R. Every wave adds up the
// counts before e by itself (each sum cut at R: none wraps), without barriers: where an expert
// has few rows a workgroup is little more than this, two copies and its stores.
__device__ __forceinline__ Seg find_segment(const int64_t* counts, int64_t R, int e, int lane) {
  const uint32_t most = (uint32_t)R;
  auto cut = [&](int64_t c) { return c < 0 ? 0u : (c > R ? most : (uint32_t)c); };
  uint32_t start = 0;
  for (int base = 0; base < e; base += 256) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ee = base + 4 * lane + i;
      if (ee < e) start = min(start + cut(counts[ee]), most);
    }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) start = min(start + (uint32_t)__shfl_xor((int)start, off), most);
  start = __builtin_amdgcn_readfirstlane(start);
  return Seg{(int)start, (int)min(cut(counts[e]), most - start)};
}

// A stage of an operand is eight 1 KB pieces (8 rows, or 4 k-rows): in the row modes a wave
// copies one, in dW two.
// k-contiguous: lane -> row 8 c + lane / 8, 16-byte chunk (lane & 7) ^ (row & 7)
__device__ __forceinline__ int row_of(int c, int lane) { return 8 * c + (lane >> 3); }
__device__ __forceinline__ int row_chunk(int lane) { return (lane & 7) ^ ((lane >> 3) & 7); }
// k-major: lane -> k-row 4 c + lane / 16, chunk (lane & 15) ^ 8 ((k >> 2) & 1), k >> 2 == c
__device__ __forceinline__ int krow_of(int c, int lane) { return 4 * c + (lane >> 4); }
__device__ __forceinline__ int krow_chunk(int c, int lane) { return (lane & 15) ^ ((c & 1) << 3); }

// chunk h of a k-contiguous tile's row: steps (h, 0 .. 3) of lane group g
__device__ __forceinline__ f32x4_t read_row(const float* tile, int row, int g, int h) {
  return *(const f32x4_t*)(tile + row * BK + (((g + 4 * h) ^ (row & 7)) << 2));
}
// step (h, j) of a k-major tile: columns 32 w + 2 (lane & 15), + 1
__device__ __forceinline__ f32x2_t read_col2(const float* tile, int lane, int w, int h, int j) {
  const int g = lane >> 4, k = 16 * h + 4 * g + j;
  const int c = 8 * w + ((lane & 15) >> 1);
  return *(const f32x2_t*)(tile + k * 64 + ((c ^ ((g & 1) << 3)) << 2) + 2 * (lane & 1));
}

// Row-grouped modes: 64 rows of one expert x 64 output columns, eight waves of 16 x 32. The
// weights are k-contiguous in gate_up and down, k-major in dgu and dx.
template <int MODE, bool ALIGNED>
__global__ __launch_bounds__(512, MODE == kGateUp ? 6 : 8) void rows_kernel(Params p) {
  constexpr bool kTwoB = MODE == kGateUp;                 // two weights into two accumulator sets
  constexpr bool kNT = MODE == kGateUp || MODE == kDown;  // weights [E, N, K]; else [E, K, N]
  constexpr int TN = 2, NB = kTwoB ? 2 : 1;
  __shared__ __attribute__((aligned(1024))) float sA[2][kTile];
  __shared__ __attribute__((aligned(1024))) float sB[2][NB][kTile];
  __shared__ int s_tmp[8];
  __shared__ int s_out[4];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int e, mt, nt;
  Seg seg;
  find_tile(p, p.N / BN, s_tmp, s_out, e, seg, mt, nt);
  const int n0 = nt * BN;
  if (e < 0) return;  // past the last tile
  const int64_t row0 = (int64_t)seg.start + (int64_t)mt * BM;
  const int nrows = min(BM, seg.count - mt * BM);
  const int wm = w >> 1, wn = w & 1;
  const int g = lane >> 4, li = lane & 15;

  // this lane's copy sources: rows past the segment re-read its last row (their results
  // are not stored)
  const float *srcA, *srcB[NB];
  srcA = p.a + (row0 + min(row_of(w, lane), nrows - 1)) * p.K + row_chunk(lane) * 4;
#pragma unroll
  for (int q = 0; q < NB; ++q) {
    const float* base = (q ? p.b2 : p.b) + (int64_t)e * p.N * p.K;
    srcB[q] = kNT ? base + (int64_t)(n0 + row_of(w, lane)) * p.K + row_chunk(lane) * 4
                  : base + (int64_t)krow_of(w, lane) * p.N + n0 + krow_chunk(w, lane) * 4;
  }
  const int64_t stepB = kNT ? BK : (int64_t)BK * p.N;
  const int nk = p.K / BK, nkt = MODE == kDx ? 2 * nk : nk;
  // dx: the second half of the k-steps runs over du and w3
  const int64_t jumpA = MODE == kDx ? p.a2 - p.a : 0, jumpB = MODE == kDx ? p.b2 - p.b : 0;
  auto issue = [&](int kt, int s) {
    const bool half = MODE == kDx && kt >= nk;
    const int kk = half ? kt - nk : kt;
    copy16<ALIGNED>(srcA + (half ? jumpA : 0) + kk * BK, lds_addr(sA[s] + w * 256));
#pragma unroll
    for (int q = 0; q < NB; ++q)
      copy16<ALIGNED>(srcB[q] + (half ? jumpB : 0) + kk * stepB, lds_addr(sB[s][q] + w * 256));
  };

  f32x4_t acc[NB][TN];
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[q][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  issue(0, 0);
  for (int kt = 0; kt < nkt; ++kt) {
    const int s = kt & 1;
    // the stage has landed in every wave, and every wave is done with the other buffer
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + 1 < nkt) issue(kt + 1, s ^ 1);
    const float* cA = sA[s];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4_t av = read_row(cA, 16 * wm + li, g, h);
      if constexpr (kNT) {
        f32x4_t bv[NB][TN];
#pragma unroll
        for (int q = 0; q < NB; ++q)
#pragma unroll
          for (int j = 0; j < TN; ++j) bv[q][j] = read_row(sB[s][q], 32 * wn + 16 * j + li, g, h);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int q = 0; q < NB; ++q)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[q][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[q][j][v], av[v], acc[q][j], 0, 0, 0);
      } else {
        f32x2_t bv[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) bv[v] = read_col2(sB[s][0], lane, wn, h, v);
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[v][j], av[v], acc[0][j], 0, 0, 0);
      }
    }
  }

  // epilogue: a lane holds row li of the wave's 16 and, as 16-byte pieces, columns
  // 16 j + 4 g .. + 3 (gate_up, down) or 8 g + 4 j .. + 3 (dgu, dx) of its 32
  const int lr = 16 * wm + li;
  if (lr >= nrows) return;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t o = (row0 + lr) * p.N + n0 + 32 * wn + (kNT ? 16 * j + 4 * g : 8 * g + 4 * j);
    f32x4_t c;
    if constexpr (kNT) c = acc[0][j];
    else c = f32x4_t{acc[0][0][2 * j], acc[0][1][2 * j], acc[0][0][2 * j + 1], acc[0][1][2 * j + 1]};
    {
      if constexpr (MODE == kGateUp) {
        const f32x4_t uu = acc[NB - 1][j];
        f32x4_t hh;
#pragma unroll
        for (int v = 0; v < 4; ++v) hh[v] = silu_f(c[v]) * uu[v];
        *(f32x4_u*)(p.o0 + o) = c;
        *(f32x4_u*)(p.o1 + o) = uu;
        *(f32x4_u*)(p.o2 + o) = hh;
      } else if constexpr (MODE == kDgu) {
        const f32x4_t gg = *(const f32x4_u*)(p.g + o), uu = *(const f32x4_u*)(p.u + o);
        f32x4_t dg, du;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float sig = 1.0f / (1.0f + expf(-gg[v]));
          du[v] = c[v] * silu_f(gg[v]);                                         // dh * silu(g)
          dg[v] = (c[v] * uu[v]) * (sig * (1.0f + gg[v] * (1.0f - sig)));       // silu'(g) (dh u)
        }
        *(f32x4_u*)(p.o1 + o) = du;
        *(f32x4_u*)(p.o0 + o) = dg;
      } else {
        *(f32x4_u*)(p.o0 + o) = c;
      }
    }
  }
}

// Weight gradients: out[e][m][n] = sum over expert e's rows r of a[r][m] b[r][n], up to
// three products per launch (each alone has too few tiles to fill the chip at the sizes
// this path is used at). Waves: 32 x 32 each.
// NS stages. One where experts have few rows (launch_dw): such a workgroup waits for its one
// stage and writes its tile, and with half the LDS eight of them share a CU instead of five;
// its last stage is copied and multiplied only up to 16 rows where it has no more (the test
// costs the long loop of two stages 2 to 5 %).
struct DwJob {
  const float* a;  // [R, M]
  const float* b;  // [R, N]
  float* out;      // [E, M, N]
  int M, N;
};
struct DwParams {
  const int64_t* counts;
  int64_t R;
  int E;
  int per_e;  // tiles of one expert, the same in every job: M N / 64^2
  int tiles;  // of all jobs
  DwJob job[3];
};

template <bool ALIGNED, int NS>
__global__ __launch_bounds__(256, 4) void dw_kernel(DwParams p) {
  __shared__ __attribute__((aligned(1024))) float sA[NS][kTile];
  __shared__ __attribute__((aligned(1024))) float sB[NS][kTile];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Workgroup b runs on XCD b % 8. Every XCD takes an eighth of each (job, expert)'s tiles,
  // neighbouring ones: whole experts per XCD would share more in its L2 but leave XCDs
  // idle where the experts' row counts differ. The jobs start at experts a third apart:
  // a CU's workgroups, a chip apart in the grid, would otherwise all belong to the same
  // heavy expert.
  const int q = p.per_e % 8 == 0 ? p.per_e >> 3 : 0, b = workgroup();
  if (b >= p.tiles) return;
  const int group = q ? (b >> 3) / q : b / p.per_e;
  const int t = q ? (b & 7) * q + (b >> 3) % q : b % p.per_e;
  const int ji = group / p.E, e = (group + ji * ((p.E + 2) / 3)) % p.E;
  const DwJob job = ji == 0 ? p.job[0] : (ji == 1 ? p.job[1] : p.job[2]);
  const int M = job.M, N = job.N, ntn = N / BN;
  const int m0 = (t / ntn) * BM, n0 = (t % ntn) * BN;
  const Seg seg = find_segment(p.counts, p.R, e, lane);
  const int wm = w >> 1, wn = w & 1, g = lane >> 4, li = lane & 15;
  const float* A = job.a + (int64_t)seg.start * M + m0;
  const float* B = job.b + (int64_t)seg.start * N + n0;
  auto issue = [&](int k0, int s) {
    if (NS == 1 && w >= 2 && k0 + BK / 2 >= seg.count) return;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int cc = 2 * w + c, k = k0 + krow_of(cc, lane), col = krow_chunk(cc, lane) * 4;
      const bool in = k < seg.count;
      copy16<ALIGNED>(in ? A + (int64_t)k * M + col : (const float*)kZeroChunk, lds_addr(sA[s] + cc * 256));
      copy16<ALIGNED>(in ? B + (int64_t)k * N + col : (const float*)kZeroChunk, lds_addr(sB[s] + cc * 256));
    }
  };
  f32x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (seg.count > 0) issue(0, 0);
  for (int k0 = 0, s = 0; k0 < seg.count; k0 += BK, s ^= NS - 1) {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (NS == 2 && k0 + BK < seg.count) issue(k0 + BK, s ^ 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (NS == 1 && h == 1 && k0 + BK / 2 >= seg.count) break;
      f32x2_t av[4], bv[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        av[j] = read_col2(sA[s], lane, wm, h, j);
        bv[j] = read_col2(sB[s], lane, wn, h, j);
      }
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[s4][j], av[s4][i], acc[i][j], 0, 0, 0);
    }
    if (NS == 1 && k0 + BK < seg.count) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has read the stage
      issue(k0 + BK, 0);
    }
  }
  // m-tile i holds rows 32 wm + 2 li + i; a lane's columns are 32 wn + 8 g .. + 7, two 16-byte
  // pieces. The lanes of a row exchange them so that each store writes 64 whole bytes of 16 rows
  // (lane group g pieces g and 4 + g).
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float* o = job.out + ((int64_t)e * M + m0 + 32 * wm + 2 * li + i) * N + n0 + 32 * wn + 4 * g;
    f32x4_t lo, hi;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i][v & 1][v >> 1]),
                                                      __float_as_uint(acc[i][v & 1][2 + (v >> 1)]), false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(x[0], x[1], false, false);
      lo[v] = __uint_as_float(y[0]);
      hi[v] = __uint_as_float(y[1]);
    }
    *(f32x4_u*)o = lo;
    *(f32x4_u*)(o + 16) = hi;
  }
}

// Zeroes the rows from sum(counts) on of up to four [R, cols] tensors, 16 bytes a lane from
// each tensor's first 16-byte boundary on. Mostly there are none and the launch only reads the
// counts (2 us, where clearing the whole tensors first took 42 us of a 370 us pass at 8192
// rows, dim 256, hidden 512). Where a buffer is mostly unused it is bound by its stores: one
// block per CU writes 939 MB (65472 rows past the counts, dim 512, hidden 1024) in 148 us (390
// with 4-byte stores of 64 blocks), 6.3 TB/s; the forward there takes 239 us, 262 where
// whole tensors were cleared first. 512 and more blocks are slower (270 to 285).
struct ZeroParams {
  const int64_t* counts;
  int64_t R;
  int E;
  float* t[4];
  int64_t cols[4];
};
__global__ __launch_bounds__(256) void zero_rest_kernel(ZeroParams p) {
  // in 64 bits: counts that are all past R sum up to E R, which would wrap an int and put the
  // first cleared row before the tensor
  __shared__ int64_t s_sum[4];
  int64_t total = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int ee = threadIdx.x * 4 + i;
    const int64_t c = ee < p.E ? p.counts[ee] : 0;
    total += c < 0 ? 0 : (c > p.R ? p.R : c);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = total;
  __syncthreads();
  total = s_sum[0] + s_sum[1] + s_sum[2] + s_sum[3];
  if (total >= p.R) return;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (p.cols[q] == 0) continue;
    float* rest = p.t[q] + total * p.cols[q];
    const int64_t n = (p.R - total) * p.cols[q];
    const int64_t head = min(n, (int64_t)((16 - ((uintptr_t)rest & 15)) & 15) / 4), n4 = (n - head) / 4;
    if (t < head) rest[t] = 0.f;
    for (int64_t i = t; i < n4; i += step) *(f32x4_t*)(rest + head + 4 * i) = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (t < n - head - 4 * n4) rest[head + 4 * n4 + t] = 0.f;
  }
}

inline bool dims_ok(int64_t R, int E, int a, int b) {
  return R >= 0 && E >= 1 && E <= kMaxE && a >= 64 && b >= 64 && a % 64 == 0 && b % 64 == 0;
}

inline bool aligned16(const void* a, const void* b, const void* c, const void* d) {
  return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c | (uintptr_t)d) & 15) == 0;
}

template <int MODE>
int launch_rows(const Params& p, hipStream_t stream) {
  if (p.R == 0) return kOk;
  // >= sum over experts of ceil(count / 64), times the column tiles; whole eighths (find_tile)
  const int64_t gx = (p.R + BM - 1) / BM + p.E, grid = (gx * (p.N / BN) + 7) / 8 * 8;
  if (grid > kMaxGrid) return kErrUnsupportedShape;
  const dim3 blocks = sliced(grid), threads(512);
  if (aligned16(p.a, p.a2, p.b, p.b2)) hipLaunchKernelGGL((rows_kernel<MODE, true>), blocks, threads, 0, stream, p);
  else hipLaunchKernelGGL((rows_kernel<MODE, false>), blocks, threads, 0, stream, p);
  return launch_status();
}

int launch_dw(DwParams& p, int jobs, hipStream_t stream) {
  const int64_t per_e = (int64_t)(p.job[0].M / BM) * (p.job[0].N / BN), grid = per_e * p.E * jobs;
  if (grid > kMaxGrid) return kErrUnsupportedShape;
  p.per_e = (int)per_e;
  p.tiles = (int)grid;
  bool aligned = true;
  for (int j = 0; j < jobs; ++j) aligned = aligned && aligned16(p.job[j].a, p.job[j].b, nullptr, nullptr);
  // up to 64 rows per expert, two stages or fewer. All three weights, us, against three launches
  // of 16-row stages, with two stages | with one: 64 experts of 1024 / 704, backward of 250 rows
  // 348 -> 369 | 330, of 1000 with 300 in use 340 -> 376 | 334, 1000 in use 412 -> 387 | 352;
  // past the line two stages win where the chip is not full: 8 experts of 256 / 512, 1000 rows
  // 57 | 59, 8000 rows 195 | 209
  const bool few = p.R <= 64 * (int64_t)p.E;
  auto* kernel = aligned ? (few ? dw_kernel<true, 1> : dw_kernel<true, 2>)
                         : (few ? dw_kernel<false, 1> : dw_kernel<false, 2>);
  hipLaunchKernelGGL(kernel, sliced(grid), dim3(256), 0, stream, p);
  return launch_status();
}

}  // namespace f32g
}  // namespace moe

using namespace moe;
using namespace moe::f32g;

MOE_API int moe_grouped_gemm_f32_gate_up(const float* x, const float* w1, const float* w3, const int64_t* counts,
                                         int64_t n_rows, int32_t n_experts, int32_t dim, int32_t hidden, float* g,
                                         float* u, float* h, hipStream_t stream) {
  if (!dims_ok(n_rows, n_experts, dim, hidden)) return kErrInvalidArgument;
  if (n_rows > 0 && (!x || !w1 || !w3 || !counts || !g || !u || !h)) return kErrInvalidArgument;
  Params p{};
  p.counts = counts; p.R = n_rows; p.E = n_experts; p.N = hidden; p.K = dim;
  p.a = x; p.b = w1; p.b2 = w3; p.o0 = g; p.o1 = u; p.o2 = h;
  return launch_rows<kGateUp>(p, stream);
}

MOE_API int moe_grouped_gemm_f32_down(const float* h, const float* w2, const int64_t* counts, int64_t n_rows,
                                      int32_t n_experts, int32_t dim, int32_t hidden, float* y, hipStream_t stream) {
  if (!dims_ok(n_rows, n_experts, dim, hidden)) return kErrInvalidArgument;
  if (n_rows > 0 && (!h || !w2 || !counts || !y)) return kErrInvalidArgument;
  Params p{};
  p.counts = counts; p.R = n_rows; p.E = n_experts; p.N = dim; p.K = hidden;
  p.a = h; p.b = w2; p.o0 = y;
  return launch_rows<kDown>(p, stream);
}

MOE_API int moe_grouped_gemm_f32_bwd_dgu(const float* dy, const float* w2, const float* g, const float* u,
                                         const int64_t* counts, int64_t n_rows, int32_t n_experts, int32_t dim,
                                         int32_t hidden, float* dg, float* du, hipStream_t stream) {
  if (!dims_ok(n_rows, n_experts, dim, hidden)) return kErrInvalidArgument;
  if (n_rows > 0 && (!dy || !w2 || !g || !u || !counts || !dg || !du)) return kErrInvalidArgument;
  Params p{};
  p.counts = counts; p.R = n_rows; p.E = n_experts; p.N = hidden; p.K = dim;
  p.a = dy; p.b = w2; p.g = g; p.u = u; p.o0 = dg; p.o1 = du;
  return launch_rows<kDgu>(p, stream);
}

MOE_API int moe_grouped_gemm_f32_bwd_dx(const float* dg, const float* du, const float* w1, const float* w3,
                                        const int64_t* counts, int64_t n_rows, int32_t n_experts, int32_t dim,
                                        int32_t hidden, float* dx, hipStream_t stream) {
  if (!dims_ok(n_rows, n_experts, dim, hidden)) return kErrInvalidArgument;
  if (n_rows > 0 && (!dg || !du || !w1 || !w3 || !counts || !dx)) return kErrInvalidArgument;
  Params p{};
  p.counts = counts; p.R = n_rows; p.E = n_experts; p.N = dim; p.K = hidden;
  p.a = dg; p.a2 = du; p.b = w1; p.b2 = w3; p.o0 = dx;
  return launch_rows<kDx>(p, stream);
}

MOE_API int moe_grouped_gemm_f32_bwd_dw(const float* a, const float* b, const int64_t* counts, int64_t n_rows,
                                        int32_t n_experts, int32_t m, int32_t n, float* out, hipStream_t stream) {
  if (!dims_ok(n_rows, n_experts, m, n)) return kErrInvalidArgument;
  if (!counts || !out || (n_rows > 0 && (!a || !b))) return kErrInvalidArgument;
  DwParams p{};
  p.counts = counts; p.R = n_rows; p.E = n_experts;
  p.job[0] = DwJob{a, b, out, m, n};
  return launch_dw(p, 1, stream);
}

MOE_API int moe_grouped_gemm_f32_bwd_dw_all(const float* dg, const float* du, const float* dy, const float* x,
                                            const float* h, const int64_t* counts, int64_t n_rows, int32_t n_experts,
                                            int32_t dim, int32_t hidden, float* dw1, float* dw3, float* dw2,
                                            hipStream_t stream) {
  if (!dims_ok(n_rows, n_experts, dim, hidden)) return kErrInvalidArgument;
  if (!counts || !dw1 || !dw2 || !dw3 || (n_rows > 0 && (!dg || !du || !dy || !x || !h))) return kErrInvalidArgument;
  DwParams p{};
  p.counts = counts; p.R = n_rows; p.E = n_experts;
  p.job[0] = DwJob{dg, x, dw1, hidden, dim};
  p.job[1] = DwJob{du, x, dw3, hidden, dim};
  p.job[2] = DwJob{dy, h, dw2, dim, hidden};
  return launch_dw(p, 3, stream);
}

MOE_API int moe_zero_rows_past_f32(const int64_t* counts, int64_t n_rows, int32_t n_experts, float* t0, int64_t cols0,
                                   float* t1, int64_t cols1, float* t2, int64_t cols2, float* t3, int64_t cols3,
                                   hipStream_t stream) {
  if (n_rows < 0 || n_experts < 1 || n_experts > kMaxE || !counts) return kErrInvalidArgument;
  if (cols0 < 0 || cols1 < 0 || cols2 < 0 || cols3 < 0) return kErrInvalidArgument;
  if (n_rows == 0) return kOk;  // (empty tensors have null pointers)
  if ((cols0 && !t0) || (cols1 && !t1) || (cols2 && !t2) || (cols3 && !t3)) return kErrInvalidArgument;
  const ZeroParams p{counts, n_rows, n_experts, {t0, t1, t2, t3}, {cols0, cols1, cols2, cols3}};
  hipLaunchKernelGGL(zero_rest_kernel, dim3(256), dim3(256), 0, stream, p);
  return launch_status();
}
