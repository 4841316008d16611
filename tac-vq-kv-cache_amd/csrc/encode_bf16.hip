// Grouped residual-VQ / grouped-CQ encode of bf16 states on MFMA for gfx950:
// group dimension d in {4, 8}, K = 256 codewords, S in {1, 2} stages, no
// whitener (closed_loop_vq.py:52-76,343-409; cq_tac.py:64-113), with the
// 32-bit distances of the one-row-per-thread kernel these shapes ran on.
//
// Scores.  The row's constant |r|^2 leaves the argmin alone, so a stage takes
// the largest a_i = r.c_i - |c_i|^2/2.  Per (problem, stage) the codewords
// are scaled by a power of two that brings their largest element into
// [16, 32) (never down), which is exact and keeps fp16's subnormal step far
// below the codewords; the residual r (fp32) is scaled alike and split into
// r_hi + r_lo (two fp16 words).  A bf16 x needs r_hi alone in stage 1 (8
// significant bits); stage 2 takes both.  The half norm rides in the product
// as three fp16 words against (-2^10, -1, -2^-11), i.e. with fp32's bits.
// v_mfma_f32_32x32x16_f16, 32 codewords x 32 rows, two row tiles per wave:
//   d = 8, stage 1   [c | n] . [x | -]            one product per tile
//   d = 8, stage 2   [c | c] . [r_hi | r_lo]      plus [. | n] . [0 | -], the
//                    same for both tiles, as their common accumulator start
//   d = 4            [c c | n] . [r_hi r_lo | -]  one product per tile
// Products are exact and sums fp32.
//
// Argmin, to the codes of the one-row-per-thread kernel.  The planes are in
// "MFMA order" (slot 32c + i of chunk c holds codeword 128 h(i) + 16c +
// el(i)), so a lane half sees codewords 128h..128h+127 in index order.  Per
// chunk and tile a lane folds each run of 8 scores ("octet") to its maximum
// and keeps the two largest and the first one's octet, all 32 bits.  The
// winning octet's 8 codewords get that kernel's own distance (|r|^2 + |c|^2)
// - 2 r.c, operation for operation (scaling by a power of two changes no
// rounding), and the first of the smallest is taken.  Where the second octet
// comes within 2^-18 (|r|^2 + max |c|^2) of the first, above the worst that
// the roundings of two scores can sum to (split 2^-23, sixteen fp32 adds
// 2^-20, the other kernel's sums 2^-21, each of |r|^2 + |c|^2 and for two
// octets), the row takes a scan of all 256 codewords with those operations
// instead (a few rows in 10^5).  So do
// rows that the fp16 words cannot carry (a residual 2,000 times the largest
// codeword or more, infinities, NaN) and problems with codewords beyond
// |c|^2 = 1e8 or not finite.
//
// Bound: VALU issue of the argmin, as in encode_grouped.hip (16 fold
// operations per 16 scores here).  [2,8,2047,128], 16 groups, two stages,
// both exits: 866 us one row per thread, 27 us here, the same outputs.  The
// scan works a row at a time with four codewords per lane: a lane scanning
// all 256 for its own row held its workgroup up by ~45 us.
#include "encode_args.h"

namespace jkv {

namespace {

typedef uint16_t ushort8 __attribute__((ext_vector_type(8)));
typedef uint16_t ushort4v __attribute__((ext_vector_type(4)));

// codeword index -> its slot in the MFMA-ordered planes
__device__ __forceinline__ int wide_slot(int k) {
  const int h = k >> 7, c = (k >> 4) & 7, el = k & 15;
  return 32 * c + 8 * (el >> 2) + 4 * h + (el & 3);
}

// lanes 32-63 of p trade places with lanes 0-31 of q, dword by dword
__device__ __forceinline__ void wide_swap(half8& p, half8& q) {
  uint4 a = __builtin_bit_cast(uint4, p);
  uint4 b = __builtin_bit_cast(uint4, q);
  auto r0 = __builtin_amdgcn_permlane32_swap(a.x, b.x, false, false);
  auto r1 = __builtin_amdgcn_permlane32_swap(a.y, b.y, false, false);
  auto r2 = __builtin_amdgcn_permlane32_swap(a.z, b.z, false, false);
  auto r3 = __builtin_amdgcn_permlane32_swap(a.w, b.w, false, false);
  a = uint4{(uint32_t)r0[0], (uint32_t)r1[0], (uint32_t)r2[0], (uint32_t)r3[0]};
  b = uint4{(uint32_t)r0[1], (uint32_t)r1[1], (uint32_t)r2[1], (uint32_t)r3[1]};
  p = __builtin_bit_cast(half8, a);
  q = __builtin_bit_cast(half8, b);
}

// maximum of v over this lane's 16-lane row, in every lane of the row
__device__ __forceinline__ uint32_t wide_row_max(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x140, 0xF, 0xF, false));
  return v;
}

__device__ __forceinline__ float bf16_to_f32(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }

// round to nearest even, NaN kept quiet (Elem<JKV_BF16>::store's rounding)
__device__ __forceinline__ uint16_t f32_to_bf16(float v) {
  const uint32_t u = __float_as_uint(v);
  uint32_t r = (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
  if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) r = (u >> 16) | 0x40u;
  return (uint16_t)r;
}

// the largest of three scores (v_maximum3_f32; a NaN score stays and loses
// every later comparison)
__device__ __forceinline__ float wide_max3(float a, float b, float c) {
  return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}

static const int kWideRowsPerWave = 64;
static const int kWideRowsPerIter = 4 * kWideRowsPerWave;
// scaled residuals above this (or NaN) leave the fp16 words
static const float kWideMaxScaled = 60000.f;

struct WideArgs {
  EncodeArgs e;
  void* recon_depth[2];
  int64_t rows_per_wg, n_chunks;
};

}  // namespace

template <int D, int S>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void rvq_encode_bf16(WideArgs m) {
  static_assert(D == 4 || D == 8, "group dimension 4 or 8");
  static_assert(S == 1 || S == 2, "one or two stages");
  const EncodeArgs& a = m.e;
  __shared__ half8 tab_c[S][256];               // scaled codewords, MFMA order (d = 4: [c, c])
  __shared__ half8 tab_n[S][256];               // half norms as three fp16 words, MFMA order
  __shared__ __align__(16) float nrm[S][256];   // scaled |c|^2/2, index order
  __shared__ uint32_t s_max[S][2][16];          // largest |element| and |c|^2 of each 16-lane row of the staging threads

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h32 = lane >> 5, j32 = lane & 31;

  // logical block: group fastest, then row chunk, then head, so that the
  // groups of one row range share its rows' lines (counts fit 32 bits:
  // host-checked)
  const uint32_t L = xcd_remap(blockIdx.x, gridDim.x);
  const uint32_t G32 = (uint32_t)a.G, nch = (uint32_t)m.n_chunks;
  const bool active = L < (uint32_t)(a.H * a.G) * nch;
  const uint32_t Lg = active ? L / G32 : 0u;
  const uint32_t g = active ? L - Lg * G32 : 0u;
  const uint32_t h = Lg / nch;
  const uint32_t chunk = Lg - h * nch;
  const uint32_t p = h * G32 + g;

  // ---- the fp16-deployed codebooks: thread tid takes codeword tid ----
  half_t cw[S][D];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const float* src = a.tables + ((int64_t)(p * S + s) * 256 + tid) * D;
    float mx = 0.f, nc = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      cw[s][i] = (half_t)src[i];
      const float v = (float)cw[s][i];
      mx = fmaxf(mx, fabsf(v));
      nc = fmaf(v, v, nc);
    }
    // non-negative floats order like their bits, infinities and NaN last (a
    // NaN element shows in the norm)
    const uint32_t me = wide_row_max(__float_as_uint(mx)), mn = wide_row_max(__float_as_uint(nc));
    if ((tid & 15) == 0) {
      s_max[s][0][tid >> 4] = me;
      s_max[s][1][tid >> 4] = mn;
    }
  }
  __syncthreads();
  float scale[S], unscale[S], nmax[S];  // nmax: largest scaled |c|^2 / 2
  bool p_ok = true;  // every stage's codewords fit the fp16 words
#pragma unroll
  for (int s = 0; s < S; ++s) {
    uint32_t me = 0u, mn = 0u;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      me = max(me, s_max[s][0][q]);
      mn = max(mn, s_max[s][1][q]);
    }
    p_ok = p_ok && mn <= __float_as_uint(1e8f);
    // largest element in [2^e, 2^(e+1)): scale 2^(4-e), at least 1
    const int e = (int)(me >> 23) - 127;
    const int up = (me == 0u || e >= 4) ? 0 : 4 - e;  // e >= -24: up <= 28
    scale[s] = __uint_as_float((uint32_t)(127 + up) << 23);
    unscale[s] = __uint_as_float((uint32_t)(127 - up) << 23);
    nmax[s] = 0.5f * __uint_as_float(mn) * scale[s] * scale[s];
  }
  const int slot = wide_slot(tid);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    half8 c;
    float nc = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      c[i] = (half_t)((float)cw[s][i % D] * scale[s]);  // exact
      if (i < D) nc = fmaf((float)c[i], (float)c[i], nc);
    }
    const float n = 0.5f * nc;
    const half_t w1 = (half_t)(n * 0x1p-10f);
    const float rest = n - (float)w1 * 0x1p10f;
    const half_t w2 = (half_t)rest;
    const half_t w3 = (half_t)((rest - (float)w2) * 0x1p11f);
    const half_t zero = (half_t)0.f;
    tab_c[s][slot] = c;
    tab_n[s][slot] = half8{w1, w2, w3, zero, zero, zero, zero, zero};
    nrm[s][tid] = n;
  }
  __syncthreads();
  if (!active) return;

  // ---- rows (rows, strides and offsets fit 32 bits: host-checked) ----
  const uint32_t rows = (uint32_t)(a.B * a.T), T32 = (uint32_t)a.T;
  const uint32_t r_begin = chunk * (uint32_t)m.rows_per_wg;
  const uint32_t r_end = min(r_begin + (uint32_t)m.rows_per_wg, rows);
  const uint16_t* states = (const uint16_t*)a.states;
  const uint32_t Dfull = G32 * D;
  const uint32_t head_x = h * (uint32_t)a.sh + g * D;
  const uint32_t head_c = h * (uint32_t)a.ch + g * S;
  const uint32_t out_bstride = (uint32_t)a.H * T32 * Dfull;
  const uint32_t head_o = h * T32 * Dfull + g * D;
  // this lane's row: its batch entry and token (a row past the range reads
  // the range's first)
  auto split_row = [&](uint32_t at, uint32_t* rb, uint32_t* rt) -> bool {
    const uint32_t row = at + (uint32_t)lane;
    const bool valid = row < r_end;
    const uint32_t rw = valid ? row : r_begin;
    *rb = rw / T32;
    *rt = rw - *rb * T32;
    return valid;
  };
  auto load_x = [&](uint32_t at) -> ushort8 {
    uint32_t rb, rt;
    split_row(at, &rb, &rt);
    const uint16_t* src = states + (rb * (uint32_t)a.sb + head_x + rt * (uint32_t)a.st);
    if constexpr (D == 8) return *(const ushort8*)src;
    const ushort4v v = *(const ushort4v*)src;
    return ushort8{v[0], v[1], v[2], v[3], 0, 0, 0, 0};
  };

  const half_t zh = (half_t)0.f;
  const half8 zero8 = half8{};
  // B words against the norm plane
  const half8 nb = half8{(half_t)-0x1p10f, (half_t)-1.f, (half_t)-0x1p-11f, zh, zh, zh, zh, zh};
  const half8 nb_only = h32 ? nb : zero8;

  // One stage's search of 8 chunks of 32 codewords x 2 row tiles.  LO: the
  // d = 8 product with r_lo, its norms from a product of their own.  Returns
  // the octet (h << 4 | o) of this lane's row and how far its score lies
  // above every other octet's.
  auto search = [&](int s, auto lo_tag, const half8 (&b)[2], float* lead) -> int {
    constexpr bool LO = decltype(lo_tag)::value;
    const half8* ap = (!LO && h32 ? &tab_n[s][0] : &tab_c[s][0]) + j32;
    const half8* np = &tab_n[s][0] + j32;
    const float16v zero16 = {};
    float best[2] = {-__builtin_inff(), -__builtin_inff()};
    float next[2] = {-__builtin_inff(), -__builtin_inff()};  // second largest octet
    int oct[2] = {0, 0};
    float16v acc[2][2];
    half8 af = ap[0], nf = LO ? np[0] : zero8;
    // chunk c's products into acc[c & 1]
    auto product = [&](int buf) {
      float16v start = zero16;
      if constexpr (LO) start = __builtin_amdgcn_mfma_f32_32x32x16_f16(nf, nb_only, zero16, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < 2; ++t) acc[buf][t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, b[t], start, 0, 0, 0);
    };
    product(0);
    af = ap[32];
    if constexpr (LO) nf = np[32];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int cur = c & 1;
      // the next chunk's products run while this one's scores are folded
      if (c + 1 < 8) product(cur ^ 1);
      if (c + 2 < 8) {
        af = ap[32 * (c + 2)];
        if constexpr (LO) nf = np[32 * (c + 2)];
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const float16v v = acc[cur][t];
#pragma unroll
        for (int o = 0; o < 2; ++o) {
          float mx = wide_max3(v[8 * o], v[8 * o + 1], v[8 * o + 2]);
          mx = wide_max3(mx, v[8 * o + 3], v[8 * o + 4]);
          mx = wide_max3(mx, v[8 * o + 5], v[8 * o + 6]);
          mx = __builtin_elementwise_maximum(mx, v[8 * o + 7]);
          next[t] = __builtin_amdgcn_fmed3f(mx, best[t], next[t]);
          if (mx > best[t]) {
            best[t] = mx;
            oct[t] = 2 * c + o;
          }
        }
        // pin the running maximum, so the compiler does not keep every
        // accumulator of the stage live
        asm volatile("" : "+v"(best[t]), "+v"(next[t]), "+v"(oct[t]));
      }
      // issue order: one tile's product of chunk c + 1, then the 16 fold
      // operations of one tile of chunk c
      if (c + 1 < 8) __builtin_amdgcn_sched_group_barrier(0x008, LO ? 2 : 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
      if (c + 1 < 8) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    // row `lane` is tile lane/32: both halves' (score, octet), the lower
    // codewords (half 0) on ties
    auto ps = __builtin_amdgcn_permlane32_swap(__float_as_uint(best[0]), __float_as_uint(best[1]), false, false);
    auto po = __builtin_amdgcn_permlane32_swap((uint32_t)oct[0], (uint32_t)oct[1], false, false);
    auto pn = __builtin_amdgcn_permlane32_swap(__float_as_uint(next[0]), __float_as_uint(next[1]), false, false);
    const float s0 = __uint_as_float((uint32_t)ps[0]), s1 = __uint_as_float((uint32_t)ps[1]);
    const float n0 = __uint_as_float((uint32_t)pn[0]), n1 = __uint_as_float((uint32_t)pn[1]);
    *lead = fmaxf(s0, s1) - fmaxf(fminf(s0, s1), fmaxf(n0, n1));
    return s1 > s0 ? 16 | (int)po[1] : (int)po[0];
  };

  // the scaled codeword plane word of codeword k
  auto word = [&](int s, int k) -> half8 { return tab_c[s][wide_slot(k)]; };

  // the fp32 distances of the row's winning octet: its first best codeword
  auto rescore = [&](int s, int oct, const float (&rs)[D], float rr) -> int {
    const int ibase = 8 * oct;  // 128 h + 8 o
    const int pbase = wide_slot(ibase);
    const float4 n0 = *(const float4*)&nrm[s][ibase];
    const float4 n1 = *(const float4*)&nrm[s][ibase + 4];
    const float nv[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
    float best = __builtin_inff();
    int at = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const half8 c = tab_c[s][pbase + 8 * (e >> 2) + (e & 3)];
      float dot = 0.f;
#pragma unroll
      for (int i = 0; i < D; ++i) dot = fmaf(rs[i], (float)c[i], dot);
      const float dist = (rr + 2.0f * nv[e]) - 2.0f * dot;
      if (dist < best) {
        best = dist;
        at = e;
      }
    }
    return ibase + at;
  };

  // every codeword for the row of lane `from`, with the operations of the
  // one-row-per-thread kernel, four codewords per lane: the first of the
  // smallest distances (0 where none is below infinity), in every lane
  auto scan = [&](int s, const float (&r)[D], int from) -> int {
    float q[D], rr = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      q[i] = __shfl(r[i], from, 64);
      rr = fmaf(q[i], q[i], rr);
    }
    const float* src = a.tables + (int64_t)(p * S + s) * 256 * D;
    float best = __builtin_inff();
    int bk = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = 64 * u + lane;
      float cc = 0.f, dot = 0.f;
#pragma unroll
      for (int i = 0; i < D; ++i) {
        const float c = deploy16(src[k * D + i]);
        cc = fmaf(c, c, cc);
        dot = fmaf(q[i], c, dot);
      }
      const float dist = (rr + cc) - 2.0f * dot;
      if (dist < best) {
        best = dist;
        bk = k;
      }
    }
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const float ob = __shfl_xor(best, off, 64);
      const int ok = __shfl_xor(bk, off, 64);
      if (ob < best || (ob == best && ok < bk)) {
        best = ob;
        bk = ok;
      }
    }
    return best < __builtin_inff() ? bk : 0;
  };

  // one stage for this lane's residual r: its code
  auto stage = [&](int s, auto first_tag, const float (&r)[D]) -> int {
    constexpr bool kFirst = decltype(first_tag)::value;
    constexpr bool kLo = D == 8 && !kFirst;
    float rs[D];
    bool ok = p_ok;
    half8 hi = zero8, lo = zero8;
#pragma unroll
    for (int i = 0; i < D; ++i) {
      rs[i] = r[i] * scale[s];
      ok = ok && fabsf(rs[i]) <= kWideMaxScaled;  // (false for NaN)
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const float v = ok ? rs[i] : 0.f;
      const half_t vh = (half_t)v;
      hi[i] = vh;
      const half_t vl = (half_t)(v - (float)vh);
      if constexpr (D == 4) {
        hi[4 + i] = vl;
      } else {
        lo[i] = vl;
      }
    }
    half8 b[2];
    b[0] = hi;
    b[1] = kLo ? lo : nb;
    wide_swap(b[0], b[1]);
    float rr = 0.f;
#pragma unroll
    for (int i = 0; i < D; ++i) rr = fmaf(rs[i], rs[i], rr);
    float lead;
    const int oct = search(s, std::integral_constant<bool, kLo>{}, b, &lead);
    int code = rescore(s, oct, rs, rr);
    // (false for NaN leads)
    const bool clear = ok && lead > (rr + 2.0f * nmax[s]) * 0x1p-18f;
    for (uint64_t todo = __ballot(!clear); todo != 0; todo &= todo - 1) {
      const int from = __builtin_ctzll(todo);
      const int k = scan(s, r, from);
      if (lane == from) code = k;
    }
    return code;
  };

  ushort8 x16 = {};
  uint32_t base = r_begin + (uint32_t)wave * kWideRowsPerWave;
  if (base < r_end) x16 = load_x(base);
  for (; base < r_end; base += kWideRowsPerIter) {
    uint32_t rb, rt;
    const bool valid = split_row(base, &rb, &rt);
    const uint32_t co = rb * (uint32_t)a.cb + head_c + rt * (uint32_t)a.ct;
    const uint32_t oo = rb * out_bstride + head_o + rt * Dfull;
    float r[D], dec[D];
#pragma unroll
    for (int i = 0; i < D; ++i) r[i] = bf16_to_f32(x16[i]);
    // the next slab's row loads during this one's search
    if (base + kWideRowsPerIter < r_end) x16 = load_x(base + kWideRowsPerIter);

    uint32_t code = 0u;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      int k;
      if (s == 0) {
        k = stage(0, std::true_type{}, r);
      } else {
        k = stage(s, std::false_type{}, r);
      }
      code |= (uint32_t)k << (8 * s);
      const half8 c = word(s, k);
#pragma unroll
      for (int i = 0; i < D; ++i) {
        const float cv = p_ok ? (float)c[i] * unscale[s] : deploy16(a.tables[((int64_t)(p * S + s) * 256 + k) * D + i]);
        r[i] -= cv;
        dec[i] = s == 0 ? 0.f + cv : dec[i] + cv;  // the fp32 stage sum
      }
      void* out = m.recon_depth[s];
      if (out != nullptr && valid) {
        uint16_t* op = (uint16_t*)out + oo;
        if constexpr (D == 8) {
          ushort8 v;
#pragma unroll
          for (int i = 0; i < 8; ++i) v[i] = f32_to_bf16(dec[i]);
          *(ushort8*)op = v;
        } else {
          ushort4v v;
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = f32_to_bf16(dec[i]);
          *(ushort4v*)op = v;
        }
      }
    }
    if (valid) {
      uint8_t* cp = a.codes + co;
      if constexpr (S == 1) {
        cp[0] = (uint8_t)code;
      } else {
        *(uint16_t*)cp = (uint16_t)code;
      }
    }
  }
}

template <int D, int S>
static int launch_bf16_t(const EncodeArgs& e, hipStream_t stream) {
  WideArgs m = {};
  m.e = e;
  for (int i = 0; i < e.n_exits; ++i) m.recon_depth[e.exit_depth[i] - 1] = e.recon[i];
  const int64_t rows = e.B * e.T, P = e.H * e.G;
  // rows per workgroup: amortise the codebook staging while the launch still
  // has three workgroups per CU
  int64_t rpw = 4096;
  while (rpw > kWideRowsPerIter && P * ceil_div(rows, rpw) < 256 * 3) rpw >>= 1;
  m.rows_per_wg = rpw;
  m.n_chunks = ceil_div(rows, rpw);
  int64_t nblocks = P * m.n_chunks;
  if (nblocks > 8) nblocks = ceil_div(nblocks, 8) * 8;  // xcd_remap needs a multiple of 8
  JKV_CHECK_ARG(nblocks < (int64_t)1 << 31, "grid too large");
  hipLaunchKernelGGL((rvq_encode_bf16<D, S>), dim3((uint32_t)nblocks), dim3(256), 0, stream, m);
  JKV_CHECK_LAUNCH();
  return JKV_OK;
}

int launch_bf16(const EncodeArgs& e, hipStream_t stream) {
  if (e.d == 8) return e.S == 1 ? launch_bf16_t<8, 1>(e, stream) : launch_bf16_t<8, 2>(e, stream);
  return e.S == 1 ? launch_bf16_t<4, 1>(e, stream) : launch_bf16_t<4, 2>(e, stream);
}

}  // namespace jkv
