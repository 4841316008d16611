// fp32 nearest codeword per row, for the offline multi-exit additive
// coordinate refinement (src/jointkv/nested_vq.py:178-215 `_nearest_indices`
// as called at nested_vq.py:690-692): states [H,N,D], tables [H,K,D], both
// fp32 and not deployed to fp16, distance (|x|^2 + |c|^2) - 2 x.c, the lowest
// index on ties (torch.argmin's rule).
//
// D = 128 (a head) runs on the fp32 matrix instructions below; other
// dimensions on nearest_f32_kernel.
//
// nearest_f32_kernel: one 256-thread block takes 64 rows of one head and walks the head's table
// in 64-codeword tiles.  Rows and codewords are staged in LDS with a row
// pitch of D rounded up to 4 plus 4 floats, so the 16 codeword rows a wave
// reads at one k fall in distinct banks.  Thread (r, c) of the 16 x 16 grid
// accumulates x.c for rows 4r..4r+3 and codewords 4c..4c+3 of the tile with
// float4 LDS reads and keeps each row's best (distance, index); the 16
// threads that share a row then reduce over lane shuffles.
#include <algorithm>

#include "jkv_common.h"

namespace jkv {

static const int kNrRows = 64;
static const int kNrCodes = 64;
static const int kNrMaxD = 128;
static const int kNrPitch = kNrMaxD + 4;

struct NearestArgs {
  const float* states;  // [H][N][D]
  const float* tables;  // [H][K][D]
  int64_t* indices;     // [H][N]
  int64_t H, N, D, K;
};

__global__ __launch_bounds__(256) void nearest_f32_kernel(NearestArgs a) {
  __shared__ __align__(16) float xs[kNrRows * kNrPitch];
  __shared__ __align__(16) float cs[kNrCodes * kNrPitch];
  __shared__ float s_xx[kNrRows];
  __shared__ float s_cc[kNrCodes];

  const int tid = threadIdx.x;
  const int64_t h = blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * kNrRows;
  const int D = (int)a.D;
  const int DP = (D + 3) & ~3;
  const int64_t nrows = min((int64_t)kNrRows, a.N - row0);

  // rows of this block, zero padded to DP and to 64 rows
  const float* xsrc = a.states + (h * a.N + row0) * a.D;
  for (int i = tid; i < kNrRows * DP; i += 256) {
    const int r = i / DP, k = i - r * DP;
    xs[r * kNrPitch + k] = (r < nrows && k < D) ? xsrc[(int64_t)r * D + k] : 0.f;
  }
  __syncthreads();
  if (tid < kNrRows) {
    // |x|^2 in dimension order
    float acc = 0.f;
    for (int k = 0; k < D; ++k) acc = fmaf(xs[tid * kNrPitch + k], xs[tid * kNrPitch + k], acc);
    s_xx[tid] = acc;
  }

  const int tr = tid >> 4;  // rows 4tr..4tr+3
  const int tc = tid & 15;  // codewords 4tc..4tc+3 of a tile
  float best[4];
  int bidx[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    best[i] = __builtin_huge_valf();
    bidx[i] = 0;
  }
  const float* csrc_head = a.tables + h * a.K * a.D;
  for (int64_t c0 = 0; c0 < a.K; c0 += kNrCodes) {
    const int64_t ncodes = min((int64_t)kNrCodes, a.K - c0);
    __syncthreads();  // the previous tile's readers are done
    const float* csrc = csrc_head + c0 * a.D;
    for (int i = tid; i < kNrCodes * DP; i += 256) {
      const int r = i / DP, k = i - r * DP;
      cs[r * kNrPitch + k] = (r < ncodes && k < D) ? csrc[(int64_t)r * D + k] : 0.f;
    }
    __syncthreads();
    if (tid < kNrCodes) {
      float acc = 0.f;
      for (int k = 0; k < D; ++k) acc = fmaf(cs[tid * kNrPitch + k], cs[tid * kNrPitch + k], acc);
      s_cc[tid] = acc;
    }
    float dot[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) dot[i][j] = 0.f;
    const float* xrow = &xs[(4 * tr) * kNrPitch];
    const float* crow = &cs[(4 * tc) * kNrPitch];
    for (int k = 0; k < DP; k += 4) {
      float4 xv[4], cv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xv[i] = *(const float4*)(xrow + i * kNrPitch + k);
        cv[i] = *(const float4*)(crow + i * kNrPitch + k);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float t = dot[i][j];
          t = fmaf(xv[i].x, cv[j].x, t);
          t = fmaf(xv[i].y, cv[j].y, t);
          t = fmaf(xv[i].z, cv[j].z, t);
          t = fmaf(xv[i].w, cv[j].w, t);
          dot[i][j] = t;
        }
    }
    __syncthreads();  // s_cc of this tile is written
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * tc + j;
      if (c < ncodes) {
        const float cc = s_cc[c];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float dist = (s_xx[4 * tr + i] + cc) - 2.f * dot[i][j];
          // codewords arrive in increasing index order per thread: strict <
          // keeps the first of equal distances
          if (dist < best[i]) {
            best[i] = dist;
            bidx[i] = (int)(c0 + c);
          }
        }
      }
    }
  }
  // the 16 lanes of one row group hold disjoint codeword sets: reduce with
  // the lower index winning ties
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float ob = __shfl_xor(best[i], off, 16);
      const int oi = __shfl_xor(bidx[i], off, 16);
      if (ob < best[i] || (ob == best[i] && oi < bidx[i])) {
        best[i] = ob;
        bidx[i] = oi;
      }
    }
  }
  if (tc == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * tr + i;
      if (r < nrows) a.indices[h * a.N + row0 + r] = bidx[i];
    }
  }
}


// D = 128 and K <= 256: x.c on v_mfma_f32_32x32x2_f32 (fp32 products and
// sums).  A 512-thread block holds the head's whole table in LDS, staged
// once; each of its eight waves keeps 32 rows in registers as the B operand
// and takes every SPLIT-th 32-codeword chunk, so a block covers 256 / SPLIT
// rows.  Two chunks accumulate side by side.  The contraction's order is
// free as long as A and B share it: lane half h takes dims 8m + 4h .. +3 of
// step group m, so one 16-byte LDS read feeds four products.
//
// Bound: the fp32 matrix rate (64 cycles per product, 2 waves per SIMD); LDS
// reads are 4 bytes per cycle and SIMD.  [8,8192,128] against 256 codewords:
// 186 us on nearest_f32_kernel (23 TFLOP/s, bound by its LDS reads),
// 41 us here (27 us of products; the rows' load leads, and the distances fold
// while both waves of a SIMD wait).
// Pitch 132 floats puts eight consecutive codewords' 16-byte pieces in
// distinct banks.
static const int kNmThreads = 512;
static const int kNmCodes = 256;
static const int kNmPitch = 132;
static const int kNmLdsBytes = (kNmCodes * kNmPitch + kNmCodes) * 4;

template <int SPLIT>
__global__ __launch_bounds__(kNmThreads) void nearest_mfma_kernel(NearestArgs a) {
  static_assert(SPLIT == 1 || SPLIT == 2 || SPLIT == 4 || SPLIT == 8, "waves per row tile");
  extern __shared__ __align__(16) float nm_lds[];
  float* cs = nm_lds;                       // [256][132]
  float* s_cc = nm_lds + kNmCodes * kNmPitch;  // |c|^2, +inf past K
  __shared__ float s_best[8][32];
  __shared__ int s_idx[8][32];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, hf = lane >> 5;
  const int K = (int)a.K;
  const int chunks = (K + 31) >> 5;
  const int64_t h = blockIdx.y;
  constexpr int kTiles = 8 / SPLIT;  // 32-row tiles per block
  const int tile = wave / SPLIT, part = wave % SPLIT;
  const int64_t row = ((int64_t)blockIdx.x * kTiles + tile) * 32 + j;
  const int64_t at = row < a.N ? row : a.N - 1;  // rows past N repeat the last

  // the table in halves of four chunks (zero rows past K), 16 bytes per thread
  // and load, eight in flight: the first ahead of the rows, the second behind
  // them
  const float4* csrc = (const float4*)(a.tables + h * a.K * 128);
  float4 piece[8];
  auto fetch = [&](int part_of) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int i = 4096 * part_of + kNmThreads * q + tid;
      piece[q] = (float4){0.f, 0.f, 0.f, 0.f};
      if ((i >> 5) < K) piece[q] = csrc[i];
    }
  };
  auto put = [&](int part_of) {
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int i = 4096 * part_of + kNmThreads * q + tid;
      *(float4*)(cs + (i >> 5) * kNmPitch + 4 * (i & 31)) = piece[q];
    }
  };
  // |c|^2 of codewords from .. from + n (+inf past K)
  auto norms = [&](int from, int n) {
    if (tid >= n) return;
    float acc = __builtin_inff();
    if (from + tid < K) {
      acc = 0.f;
      const float* c = cs + (from + tid) * kNmPitch;
#pragma unroll 8
      for (int q = 0; q < 128; q += 4) {
        const float4 v = *(const float4*)(c + q);
        acc = fmaf(v.x, v.x, acc);
        acc = fmaf(v.y, v.y, acc);
        acc = fmaf(v.z, v.z, acc);
        acc = fmaf(v.w, v.w, acc);
      }
    }
    s_cc[from + tid] = acc;
  };
  fetch(0);
  // this lane's half of its row: dims 8m + 4 hf .. +3
  const float4* xsrc = (const float4*)(a.states + (h * a.N + at) * 128) + hf;
  float4 x[16];
#pragma unroll
  for (int m = 0; m < 16; ++m) x[m] = xsrc[2 * m];
  put(0);
  // up to two waves to a row tile, each wave's pairs of chunks lie within the
  // halves: the second half's loads fly during the first half's products
  // ([8,8192] 47.2 -> 45.5 us per launch, [8,1500] 17.5 -> 16.2 against one
  // staging loop, 16 loads one after the other, ahead of everything)
  constexpr bool kHalves = SPLIT <= 2;
  const bool second = chunks > 4;
  if (second) fetch(1);
  if (!kHalves && second) put(1);
  __syncthreads();
  norms(0, kHalves ? 128 : 256);
  float xx = 0.f;
#pragma unroll
  for (int m = 0; m < 16; ++m) {
    xx = fmaf(x[m].x, x[m].x, xx);
    xx = fmaf(x[m].y, x[m].y, xx);
    xx = fmaf(x[m].z, x[m].z, xx);
    xx = fmaf(x[m].w, x[m].w, xx);
  }
  xx += __shfl_xor(xx, 32, 64);
  __syncthreads();

  float best = __builtin_inff();
  int bidx = 0;
  // chunks c0, c0 + SPLIT, ... below end: two at a time
  auto search = [&](int c0, int end) {
    for (; c0 < end; c0 += 2 * SPLIT) {
      const int c1 = c0 + SPLIT;
      const bool two = c1 < chunks;
      const float* ap0 = cs + (32 * c0 + j) * kNmPitch + 4 * hf;
      const float* ap1 = two ? cs + (32 * c1 + j) * kNmPitch + 4 * hf : ap0;
      float16v acc0 = {}, acc1 = {};
#pragma unroll
      for (int m = 0; m < 16; ++m) {
        const float4 a0 = *(const float4*)(ap0 + 8 * m);
        const float4 a1 = *(const float4*)(ap1 + 8 * m);
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.x, x[m].x, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.x, x[m].x, acc1, 0, 0, 0);
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.y, x[m].y, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.y, x[m].y, acc1, 0, 0, 0);
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.z, x[m].z, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.z, x[m].z, acc1, 0, 0, 0);
        acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(a0.w, x[m].w, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(a1.w, x[m].w, acc1, 0, 0, 0);
      }
      // element el of lane (hf, j) is codeword 8 (el / 4) + 4 hf + el % 4 of the
      // chunk: indices rise within the lane, so strict < keeps the first of
      // equal distances
      auto fold = [&](int c, const float16v& acc) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int k0 = 32 * c + 8 * q + 4 * hf;
          const float4 cc = *(const float4*)(s_cc + k0);
          const float cv[4] = {cc.x, cc.y, cc.z, cc.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float dist = (xx + cv[e]) - 2.f * acc[4 * q + e];
            if (dist < best) {
              best = dist;
              bidx = k0 + e;
            }
          }
        }
      };
      fold(c0, acc0);
      if (two) fold(c1, acc1);
    }
  };
  if constexpr (kHalves) {
    search(part, min(chunks, 4));
    if (second) {
      put(1);
      __syncthreads();
      norms(128, 128);
      __syncthreads();
      search(4 + part, chunks);
    }
  } else {
    search(part, chunks);
  }
  // the other lane half holds the row's other codewords; the lower index wins ties
  {
    const float ob = __shfl_xor(best, 32, 64);
    const int oi = __shfl_xor(bidx, 32, 64);
    if (ob < best || (ob == best && oi < bidx)) {
      best = ob;
      bidx = oi;
    }
  }
  if constexpr (SPLIT > 1) {
    if (hf == 0) {
      s_best[wave][j] = best;
      s_idx[wave][j] = bidx;
    }
    __syncthreads();
    if (part != 0) return;
#pragma unroll
    for (int q = 1; q < SPLIT; ++q) {
      const float ob = s_best[wave + q][j];
      const int oi = s_idx[wave + q][j];
      if (ob < best || (ob == best && oi < bidx)) {
        best = ob;
        bidx = oi;
      }
    }
  }
  if (hf == 0 && row < a.N) a.indices[h * a.N + row] = bidx;
}

// The split with the least estimated time: rounds of 256 one-per-CU blocks,
// each its share of the eight chunks plus about a tenth of the whole search
// for its staging: [8,N,128] with N = 1,500 takes 16 waves'-worth of chunks in
// parallel at SPLIT 4 where SPLIT 1 would leave 200 CUs idle.
// Few codewords leave waves without a chunk, which costs little: [8,8192] 14
// us with 4 to 64 words, 24 with 128, 42 with 256 (nearest_f32_kernel 54, 66,
// 112, 186); [8,300] against 16 10 and 23.
static int nearest_split(int64_t H, int64_t N) {
  int best = 1;
  double least = 0.0;
  for (int split = 1; split <= 8; split *= 2) {
    const double rounds = (double)ceil_div(H * ceil_div(N, (int64_t)(256 / split)), 256);
    const double t = rounds * (1.0 / split + 0.1);
    if (split == 1 || t < least) {
      best = split;
      least = t;
    }
  }
  return best;
}

template <int SPLIT>
static int launch_nearest_mfma(const NearestArgs& a, hipStream_t stream) {
  const dim3 grid((uint32_t)ceil_div(a.N, (int64_t)(256 / SPLIT)), (uint32_t)a.H);
  hipLaunchKernelGGL(nearest_mfma_kernel<SPLIT>, grid, dim3(kNmThreads), kNmLdsBytes, stream, a);
  JKV_CHECK_LAUNCH();
  return JKV_OK;
}

// The M nearest codewords of every row, nearest first (equal distances in
// index order), optionally skipping one index per row (`excluded`, [H][N]):
// `_nearest_topk_indices` (nested_vq.py:218-260), the shortlist search of the
// block refinement.  Same tiles as above; each thread keeps a sorted list of
// M per row, and one thread per row merges the 16 lists from LDS.
template <int M>
__global__ __launch_bounds__(256) void nearest_topk_f32_kernel(NearestArgs a, const int64_t* excluded) {
  __shared__ __align__(16) float xs[kNrRows * kNrPitch];
  __shared__ __align__(16) float cs[kNrCodes * kNrPitch];
  __shared__ float s_xx[kNrRows];
  __shared__ float s_cc[kNrCodes];
  __shared__ float cand_d[kNrRows][16 * M];
  __shared__ int cand_i[kNrRows][16 * M];

  const int tid = threadIdx.x;
  const int64_t h = blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * kNrRows;
  const int D = (int)a.D;
  const int DP = (D + 3) & ~3;
  const int64_t nrows = min((int64_t)kNrRows, a.N - row0);

  const float* xsrc = a.states + (h * a.N + row0) * a.D;
  for (int i = tid; i < kNrRows * DP; i += 256) {
    const int r = i / DP, k = i - r * DP;
    xs[r * kNrPitch + k] = (r < nrows && k < D) ? xsrc[(int64_t)r * D + k] : 0.f;
  }
  __syncthreads();
  if (tid < kNrRows) {
    float acc = 0.f;
    for (int k = 0; k < D; ++k) acc = fmaf(xs[tid * kNrPitch + k], xs[tid * kNrPitch + k], acc);
    s_xx[tid] = acc;
  }

  const int tr = tid >> 4;
  const int tc = tid & 15;
  int ex[4];
  float bd[4][M];
  int bi[4][M];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * tr + i;
    ex[i] = (excluded != nullptr && r < nrows) ? (int)excluded[h * a.N + row0 + r] : -1;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      bd[i][m] = __builtin_huge_valf();
      bi[i][m] = -1;
    }
  }
  const float* csrc_head = a.tables + h * a.K * a.D;
  for (int64_t c0 = 0; c0 < a.K; c0 += kNrCodes) {
    const int64_t ncodes = min((int64_t)kNrCodes, a.K - c0);
    __syncthreads();
    const float* csrc = csrc_head + c0 * a.D;
    for (int i = tid; i < kNrCodes * DP; i += 256) {
      const int r = i / DP, k = i - r * DP;
      cs[r * kNrPitch + k] = (r < ncodes && k < D) ? csrc[(int64_t)r * D + k] : 0.f;
    }
    __syncthreads();
    if (tid < kNrCodes) {
      float acc = 0.f;
      for (int k = 0; k < D; ++k) acc = fmaf(cs[tid * kNrPitch + k], cs[tid * kNrPitch + k], acc);
      s_cc[tid] = acc;
    }
    float dot[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) dot[i][j] = 0.f;
    const float* xrow = &xs[(4 * tr) * kNrPitch];
    const float* crow = &cs[(4 * tc) * kNrPitch];
    for (int k = 0; k < DP; k += 4) {
      float4 xv[4], cv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xv[i] = *(const float4*)(xrow + i * kNrPitch + k);
        cv[i] = *(const float4*)(crow + i * kNrPitch + k);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float t = dot[i][j];
          t = fmaf(xv[i].x, cv[j].x, t);
          t = fmaf(xv[i].y, cv[j].y, t);
          t = fmaf(xv[i].z, cv[j].z, t);
          t = fmaf(xv[i].w, cv[j].w, t);
          dot[i][j] = t;
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = 4 * tc + j;
      if (c < ncodes) {
        const float cc = s_cc[c];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float dd = (s_xx[4 * tr + i] + cc) - 2.f * dot[i][j];
          int ii = (int)(c0 + c);
          if (ii != ex[i] && dd < bd[i][M - 1]) {
            // insertion into the sorted list: strict < keeps equal
            // distances in arrival (index) order
#pragma unroll
            for (int m = 0; m < M; ++m) {
              if (dd < bd[i][m]) {
                const float td = bd[i][m];
                const int ti = bi[i][m];
                bd[i][m] = dd;
                bi[i][m] = ii;
                dd = td;
                ii = ti;
              }
            }
          }
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      cand_d[4 * tr + i][tc * M + m] = bd[i][m];
      cand_i[4 * tr + i][tc * M + m] = bi[i][m];
    }
  __syncthreads();
  if (tid < nrows) {
    int64_t* out = a.indices + (h * a.N + row0 + tid) * M;
    for (int m = 0; m < M; ++m) {
      float best = __builtin_huge_valf();
      int bidx = 0x7fffffff, pos = -1;
      for (int q = 0; q < 16 * M; ++q) {
        const int id = cand_i[tid][q];
        const float d = cand_d[tid][q];
        if (id >= 0 && (pos < 0 || d < best || (d == best && id < bidx))) {
          best = d;
          bidx = id;
          pos = q;
        }
      }
      out[m] = pos >= 0 ? bidx : 0;
      if (pos >= 0) cand_i[tid][pos] = -1;
    }
  }
}

}  // namespace jkv

extern "C" int jkv_nearest_f32(const float* states, int64_t H, int64_t N, int64_t D,
                               const float* tables, int64_t K, int64_t* indices,
                               jkv_stream_t stream_) {
  using namespace jkv;
  hipStream_t stream = (hipStream_t)stream_;
  JKV_CHECK_ARG(H > 0 && N >= 0 && K > 0, "invalid nearest-codeword geometry");
  JKV_CHECK_ARG(D > 0 && D <= kNrMaxD, "nearest-codeword dimension must lie in 1..%d (got %lld)",
                kNrMaxD, (long long)D);
  JKV_CHECK_ARG(H <= 65535, "at most 65535 heads per call (got %lld)", (long long)H);
  JKV_CHECK_ARG(K < ((int64_t)1 << 31), "nearest-codeword size too large");
  // one 256-thread block per 64 rows: the grid's x extent counts work items
  JKV_CHECK_ARG(ceil_div(N, (int64_t)kNrRows) * 256 < ((int64_t)1 << 32),
                "at most %lld rows per head (got %lld)", (long long)(kNrRows * ((((int64_t)1 << 32) - 1) / 256)),
                (long long)N);
  if (N == 0) return JKV_OK;
  JKV_CHECK_ARG(states && tables && indices, "null buffer");
  NearestArgs a = {states, tables, indices, H, N, D, K};
  // whole heads against 8-bit stages, 16-byte rows: the matrix kernel (its
  // grid counts 512-thread blocks of 32 rows at least)
  if (D == 128 && K <= kNmCodes && (((uintptr_t)states | (uintptr_t)tables) % 16) == 0 &&
      ceil_div(N, (int64_t)32) * kNmThreads < ((int64_t)1 << 32)) {
    switch (nearest_split(H, N)) {
      case 1: return launch_nearest_mfma<1>(a, stream);
      case 2: return launch_nearest_mfma<2>(a, stream);
      case 4: return launch_nearest_mfma<4>(a, stream);
      default: return launch_nearest_mfma<8>(a, stream);
    }
  }
  dim3 grid((uint32_t)ceil_div(N, (int64_t)kNrRows), (uint32_t)H);
  hipLaunchKernelGGL(nearest_f32_kernel, grid, dim3(256), 0, stream, a);
  JKV_CHECK_LAUNCH();
  return JKV_OK;
}

extern "C" int jkv_nearest_topk_f32(const float* states, int64_t H, int64_t N, int64_t D,
                                    const float* tables, int64_t K, int64_t M,
                                    const int64_t* excluded, int64_t* indices,
                                    jkv_stream_t stream_) {
  using namespace jkv;
  hipStream_t stream = (hipStream_t)stream_;
  JKV_CHECK_ARG(H > 0 && N >= 0 && K > 0, "invalid nearest-codeword geometry");
  JKV_CHECK_ARG(D > 0 && D <= kNrMaxD, "nearest-codeword dimension must lie in 1..%d (got %lld)",
                kNrMaxD, (long long)D);
  JKV_CHECK_ARG(M >= 1 && M <= 8, "top-k candidate count must lie in 1..8 (got %lld)", (long long)M);
  JKV_CHECK_ARG(M < K, "top-k candidate count must lie in [1, cardinality)");
  JKV_CHECK_ARG(H <= 65535, "at most 65535 heads per call (got %lld)", (long long)H);
  JKV_CHECK_ARG(K < ((int64_t)1 << 31), "nearest-codeword size too large");
  // one 256-thread block per 64 rows: the grid's x extent counts work items
  JKV_CHECK_ARG(ceil_div(N, (int64_t)kNrRows) * 256 < ((int64_t)1 << 32),
                "at most %lld rows per head (got %lld)", (long long)(kNrRows * ((((int64_t)1 << 32) - 1) / 256)),
                (long long)N);
  if (N == 0) return JKV_OK;
  JKV_CHECK_ARG(states && tables && indices, "null buffer");
  NearestArgs a = {states, tables, indices, H, N, D, K};
  dim3 grid((uint32_t)ceil_div(N, (int64_t)kNrRows), (uint32_t)H);
  switch (M) {
#define JKV_TOPK_CASE(m) \
  case m: hipLaunchKernelGGL(nearest_topk_f32_kernel<m>, grid, dim3(256), 0, stream, a, excluded); break;
    JKV_TOPK_CASE(1) JKV_TOPK_CASE(2) JKV_TOPK_CASE(3) JKV_TOPK_CASE(4)
    JKV_TOPK_CASE(5) JKV_TOPK_CASE(6) JKV_TOPK_CASE(7) JKV_TOPK_CASE(8)
#undef JKV_TOPK_CASE
  }
  JKV_CHECK_LAUNCH();
  return JKV_OK;
}
