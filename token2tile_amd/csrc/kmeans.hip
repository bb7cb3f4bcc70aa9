// S2: warm-started k-means maintenance, and the init_state helpers
// (fast_assign, Lloyd iterations, centroid updates), for gfx950.
//
// Pipeline of one maintenance call (all deterministic):
//   prep centroids -> assign (MFMA distances + argmin, and the label histogram
//   of the work-group's rows) -> stable counting sort of the labels (column
//   scans, ballot-ranked scatter) -> per-cluster sums in sorted row order
//   (exact int64 fixed point for query clusters; sequential fp32 for key
//   clusters, which also writes the cluster-ordered V) -> value statistics
//   (lam, sumv).
#include "t2t_common.h"

#define KM_R 32            // rank of the projected space
#define AS_CHUNK 256       // centroids staged per LDS chunk in assign
#define KM_MAXC 4096

static inline int pad32(int c) { return (c + 31) & ~31; }

// ---------------------------------------------------------------------------
// fast_assign, general form (D = 64 and 128).  Transposed MFMA product: centroids on the row
// axis (A), tokens on the column axis (B), so a lane owns one token and 16
// centroids per 32-centroid block, visited in ascending index order:
// d2 = |x|^2 + (cn2 - 2 x.c); key = (bits(d2) & ~m) | c, the smallest key wins.
// ---------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void fast_assign_kernel(const uint16_t* __restrict__ X,
                                                          const uint16_t* __restrict__ cen,
                                                          int32_t* __restrict__ labels, int N,
                                                          int C, int ibits) {
  constexpr int KS = D / 16;
  __shared__ __attribute__((aligned(16))) uint16_t sC[AS_CHUNK * D];
  __shared__ float sN[AS_CHUNK];
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int jl = lane & 31, hh = lane >> 5;
  const int row = blockIdx.x * 128 + wave * 32 + jl;
  const bool ok = row < N;
  const uint16_t* xh = X + (size_t)h * N * D;
  u32x4 bx[KS];
  float xsq = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    bx[s] = u32x4{0u, 0u, 0u, 0u};
    if (ok) bx[s] = *(const u32x4*)(xh + (size_t)row * D + 16 * s + 8 * hh);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float a = h2f((uint16_t)(bx[s][t] & 0xffff)), b = h2f((uint16_t)(bx[s][t] >> 16));
      xsq += a * a + b * b;
    }
  }
  xsq = half_sum(xsq);
  const uint16_t* ch = cen + (size_t)h * C * D;
  const int Cp = (C + 31) & ~31;
  int bkey = 0x7fffffff;
  const int kmask = -(1 << ibits);
  for (int c0 = 0; c0 < Cp; c0 += AS_CHUNK) {
    const int nc = (Cp - c0) < AS_CHUNK ? (Cp - c0) : AS_CHUNK;
    __syncthreads();
    // stage the chunk (padding = 0) and the squared norms in fp32, summed
    // sequentially over the dims (each square is exact)
    for (int i = tid; i < nc * D / 8; i += 256) {
      const int ci = c0 + (i * 8) / D;
      u32x4 v = {0u, 0u, 0u, 0u};
      if (ci < C) v = ((const u32x4*)(ch + (size_t)c0 * D))[i];
      ((u32x4*)sC)[i] = v;
    }
    for (int i = tid; i < nc; i += 256) {
      const int ci = c0 + i;
      float s = 0.f;
      if (ci < C) {
        const uint16_t* cp = ch + (size_t)ci * D;
        for (int d = 0; d < D; ++d) {
          const float v = h2f(cp[d]);
          s = s + v * v;
        }
      }
      sN[i] = (ci < C) ? s : __builtin_inff();
    }
    __syncthreads();
    for (int cb = 0; cb < nc / 32; ++cb) {
      f32x16 acc = zero16();
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4 av = *(const u32x4*)(sC + (cb * 32 + jl) * D + 16 * s + 8 * hh);
        acc = Mfma<F16T>::run(av, bx[s], acc);
      }
#pragma unroll
      for (int a = 0; a < 16; ++a) {
        const int ci = c0 + cb * 32 + 8 * (a / 4) + 4 * hh + (a % 4);
        const float cn2 = sN[cb * 32 + 8 * (a / 4) + 4 * hh + (a % 4)];
        const float d2 = xsq + (cn2 - 2.0f * acc[a]);
        int key = (__builtin_bit_cast(int, d2) & kmask) | ci;
        if (ci >= C) key = 0x7fffffff;
        bkey = key < bkey ? key : bkey;
      }
    }
  }
  const int ok2 = (int)half_partner((uint32_t)bkey);
  bkey = ok2 < bkey ? ok2 : bkey;
  if (ok && hh == 0) labels[(size_t)h * N + row] = bkey & ((1 << ibits) - 1);
}

// ---------------------------------------------------------------------------
// fast_assign at D = 32, the rank of the projected space: the labels of
// fast_assign_kernel, bit for bit (same operands, same fp32 operations, same
// keys), in the loop shape of assign_km_kernel: eight waves of RB 32-row
// blocks, so a centroid fragment read from LDS feeds RB MFMA chains, and the
// centroids staged 512 at a time with their norms.
//
// The general form is bound by its VALU work, 3.5 operations per distance
// against two MFMAs per 1024.  Here a block of 16 distances costs its 16
// fused multiply-adds and a min tree; fp32 addition is monotone, so the least
// distance is |x|^2 + the least (|c|^2 - 2 x.c), and when that is not
// negative and its key's distance part is above the running key's, no key of
// the block can win.  Only other blocks (and any with a NaN, which the tree
// hands on) build their 16 keys.
//
// guess (optional): a label per row, any value.  The distance to that
// centroid, summed here, plus 2^-15 of the sum of its terms' magnitudes is
// above the MFMA's (33 terms in any order round under 2^-18 of that sum, the
// two additions under 2^-22), so the running key may start at the largest key
// of that distance: the guessed centroid's own key is not above it.
// order (optional): a permutation of the rows, the order they are taken in.
// Sorted by the guesses, the 32 rows of a block all stop at the same one or two
// of the centroid blocks; in row order nearly half of the blocks stop some row.
// Measured at 40 x 75600 rows, 2048 centroids: 1.2 ms in the general form, 0.81
// without a guess, 0.54 with guess and order; 8 x 32760 113 -> 78 us.
// ---------------------------------------------------------------------------
#define FA_WAVES 8
#define FA_CHUNK 512
template <int RB>
__global__ __launch_bounds__(FA_WAVES * 64) void fast_assign32_kernel(
    const uint16_t* __restrict__ X, const uint16_t* __restrict__ cen, int32_t* labels, int N, int C,
    int ibits, const int32_t* guess, const int32_t* __restrict__ order) {
  constexpr int D = 32;
  __shared__ __attribute__((aligned(16))) uint16_t sC[FA_CHUNK * D];
  __shared__ __attribute__((aligned(16))) float sN[FA_CHUNK];
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int jl = lane & 31, hh = lane >> 5;
  const int Cp = (C + 31) & ~31;
  const int kmask = -(1 << ibits);
  const uint16_t* xh = X + (size_t)h * N * D;
  const uint16_t* ch = cen + (size_t)h * C * D;
  const int rbase = blockIdx.x * (FA_WAVES * 32 * RB) + wave * 32 * RB + jl;
  u32x4 bx[RB][2];
  float xsq[RB];
  int best[RB];
  auto row_of = [&](int pos) { return order && pos < N ? order[(size_t)h * N + pos] : pos; };
#pragma unroll
  for (int k = 0; k < RB; ++k) {
    const int row = row_of(rbase + 32 * k);
    const bool ok = row < N;
    float xs = 0.f;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bx[k][s] = u32x4{0u, 0u, 0u, 0u};
      if (ok) bx[k][s] = *(const u32x4*)(xh + (size_t)row * D + 16 * s + 8 * hh);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const float a = h2f((uint16_t)(bx[k][s][t] & 0xffff)), b = h2f((uint16_t)(bx[k][s][t] >> 16));
        xs += a * a + b * b;
      }
    }
    xsq[k] = half_sum(xs);
    best[k] = 0x7fffffff;
    const int g = (ok && guess) ? guess[(size_t)h * N + row] : -1;
    const bool have = g >= 0 && g < C;
    float part = 0.f, mag = 0.f, cn = 0.f;
    if (have) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4 cv = *(const u32x4*)(ch + (size_t)g * D + 16 * s + 8 * hh);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float x = h2f((uint16_t)(bx[k][s][t] >> (16 * e)));
            const float cc = h2f((uint16_t)(cv[t] >> (16 * e)));
            part = fmaf(x, cc, part);
            mag = fmaf(fabsf(x), fabsf(cc), mag);
            cn = fmaf(cc, cc, cn);
          }
      }
    }
    part = half_sum(part);
    mag = half_sum(mag);
    cn = half_sum(cn);
    const float ub = xsq[k] + (cn - 2.0f * part) + 0x1p-15f * (xsq[k] + cn + 2.0f * mag) + 0x1p-120f;
    if (have && ub >= 0.f && ub < 0x1p126f) best[k] = __builtin_bit_cast(int, ub) | ~kmask;
  }
  auto mn = [](float a, float b) { return __builtin_elementwise_minimum(a, b); };
  for (int c0 = 0; c0 < Cp; c0 += FA_CHUNK) {
    const int nc = Cp - c0 < FA_CHUNK ? Cp - c0 : FA_CHUNK;
    if (c0 > 0) __syncthreads();  // every wave is done with the previous chunk
    // a thread stages one centroid (16-byte chunk c of row r at c ^ ((r >> 2) & 3))
    // and sums its norm over the dims in order; padding: zeros, norm inf
    if (tid < nc) {
      const bool in = c0 + tid < C;
      const u32x4* cp = (const u32x4*)(ch + (size_t)(c0 + (in ? tid : 0)) * D);
      float sum = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const u32x4 v = in ? cp[c] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float a = h2f((uint16_t)(v[t] & 0xffff)), b = h2f((uint16_t)(v[t] >> 16));
          sum = sum + a * a;
          sum = sum + b * b;
        }
        ((u32x4*)sC)[tid * 4 + (c ^ ((tid >> 2) & 3))] = v;
      }
      sN[tid] = in ? sum : __builtin_inff();
    }
    __syncthreads();
    for (int cb = 0; cb < nc / 32; ++cb) {
      const int r = cb * 32 + jl;
      const bool part = c0 + cb * 32 + 32 > C;  // wave-uniform: the block holds padding
      const u32x4* crow = (const u32x4*)sC + r * 4;
      const u32x4 a0 = crow[(0 + hh) ^ ((r >> 2) & 3)];
      const u32x4 a1 = crow[(2 + hh) ^ ((r >> 2) & 3)];
      f32x4 cn[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) cn[q] = *(const f32x4*)(sN + cb * 32 + 8 * q + 4 * hh);
#pragma unroll
      for (int k = 0; k < RB; ++k) {
        f32x16 acc = Mfma<F16T>::run(a0, bx[k][0], zero16());
        acc = Mfma<F16T>::run(a1, bx[k][1], acc);
        float t[16];
#pragma unroll
        for (int a = 0; a < 16; ++a) t[a] = cn[a / 4][a % 4] - 2.0f * acc[a];
        float t8[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) t8[i] = mn(t[2 * i], t[2 * i + 1]);
        const float d2 =
            xsq[k] + mn(mn(mn(t8[0], t8[1]), mn(t8[2], t8[3])), mn(mn(t8[4], t8[5]), mn(t8[6], t8[7])));
        const bool skip = d2 >= 0.f && (__builtin_bit_cast(int, d2) & kmask) > (best[k] & kmask);
        if (__ballot(!skip) != 0ull) {  // wave-uniform
          // the index bits below 32 first, the block's base (a multiple of 32)
          // once at the end: both lie under the mask, so the order is the same
          int kb = 0x7fffffff;
          if (part) {
            asm volatile("" ::: "memory");  // a branch of its own, not selects
#pragma unroll
            for (int a = 0; a < 16; ++a) {
              const int key = (__builtin_bit_cast(int, xsq[k] + t[a]) & kmask) | (8 * (a / 4) + (a % 4));
              const bool pad = c0 + cb * 32 + 4 * hh + 8 * (a / 4) + (a % 4) >= C;
              kb = !pad && key < kb ? key : kb;
            }
          } else {
#pragma unroll
            for (int a = 0; a < 16; ++a) {
              const int key = (__builtin_bit_cast(int, xsq[k] + t[a]) & kmask) | (8 * (a / 4) + (a % 4));
              kb = key < kb ? key : kb;
            }
          }
          kb |= c0 + cb * 32 + 4 * hh;
          best[k] = kb < best[k] ? kb : best[k];
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < RB; ++k) {
    const int o = (int)half_partner((uint32_t)best[k]);
    const int b = o < best[k] ? o : best[k];
    const int row = row_of(rbase + 32 * k);
    if (row < N && hh == 0) labels[(size_t)h * N + row] = b & ~kmask;
  }
}

// Row blocks per wave (LDS reads per distance fall with them): four while the
// launch still has four work-groups per CU, fewer when it would not fill the
// chip.
static void launch_fast_assign32(const void* x, const void* c, int32_t* labels, int H, int N, int C,
                                 int ibits, const int32_t* guess, const int32_t* order,
                                 hipStream_t st) {
#define FA_LAUNCH(RB)                                                                            \
  hipLaunchKernelGGL(fast_assign32_kernel<RB>, dim3(cdiv(N, FA_WAVES * 32 * RB), H),             \
                     dim3(FA_WAVES * 64), 0, st, (const uint16_t*)x, (const uint16_t*)c, labels, \
                     N, C, ibits, guess, order)
  if ((long long)H * cdiv(N, FA_WAVES * 128) >= 1024)
    FA_LAUNCH(4);
  else if ((long long)H * cdiv(N, FA_WAVES * 64) >= 512)
    FA_LAUNCH(2);
  else
    FA_LAUNCH(1);
#undef FA_LAUNCH
}

// ---------------------------------------------------------------------------
// k-means assignment at rank 32: d = |c|^2 + x.(-2c),
// argmin, ties to the lowest index.  One work-group per 256 RB rows: RB 32-row
// blocks per wave, so every centroid fragment and norm read from LDS feeds RB
// MFMA chains, and CS groups of eight waves that share the rows and take the
// centroid blocks in turn (below).  The centroids (-2c and |c|^2 from
// cen_prep_kernel) are staged in chunks of CMAX rows (34 KB at 512: four
// work-groups of eight waves per CU, two of sixteen).
// Centroid row r keeps its 16-byte chunk c at c ^ ((r >> 2) & 3), so the 32
// rows a fragment read touches fall on distinct banks.
//
// Pruning bound from a guess: the row's previous label (the label buffer's
// old contents, any value; used only when it names a centroid).  Its distance,
// summed here in fp32, plus a bound on the rounding of that sum and of the
// MFMA's own (33 terms in any order: under 2^-18 of the sum of their
// magnitudes each; 2^-16 is taken) is strictly above the MFMA distance of the
// guessed centroid, so starting the running minimum there changes no label:
// the result is still the first centroid, in visiting order, at the minimum
// MFMA distance.  A block then costs a min tree and one compare; only a block
// whose minimum improves on some lane's running minimum looks for its lowest
// index at that value.
//
// The work-group's rows are one chunk of the counting sort: once the labels
// are known, their histogram is taken in the LDS of the centroids and written
// beside them.  RB, the row blocks per wave (km_rb), sets the chunk, 256 RB
// rows.  One launch serves up to two row sets (blockIdx.z): the key pass and
// the first query pass do not depend on each other.
// ---------------------------------------------------------------------------
#define AK_WAVES 8
#define AK_CHUNK 512
struct AssignArgs {
  const uint16_t* X;       // [H, N, 32]
  const uint16_t* cprep;   // [H, C, 32] -2c
  const float* cnorm;      // [H, C]
  int32_t* labels;         // [H, N]
  const int32_t* guess;    // [H, N] or null; may be labels itself
  int32_t* chist;          // [H, chunks, C]
  int C, pin_begin, pin_label;
};
// CS groups of AK_WAVES waves take the centroid blocks of the same rows in turn
// (two where the launch leaves CUs idle: 2 x 4096 rows, 64 work-groups, 26 us in
// one group, 21 in two).
template <int RB, int CS>
__global__ __launch_bounds__(AK_WAVES * 64 * CS) void assign_km_kernel(AssignArgs g0, AssignArgs g1,
                                                                       int N) {
  constexpr int CMAX = AK_CHUNK, AK_RB = RB;
  const AssignArgs& ga = blockIdx.z ? g1 : g0;
  const uint16_t* __restrict__ X = ga.X;
  const uint16_t* __restrict__ cprep = ga.cprep;
  const float* __restrict__ cnorm = ga.cnorm;
  int32_t* labels = ga.labels;
  const int32_t* guess = ga.guess;
  const int C = ga.C, pin_begin = ga.pin_begin, pin_label = ga.pin_label;
  constexpr int D = 32;
  __shared__ __attribute__((aligned(16))) uint16_t sC[CMAX * D];
  __shared__ __attribute__((aligned(16))) float sN[CMAX];
  const int h = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) % AK_WAVES;
  const int cg = CS > 1 ? __builtin_amdgcn_readfirstlane(tid >> 6) / AK_WAVES : 0;
  const int jl = lane & 31, hh = lane >> 5;
  const int Cp = (C + 31) & ~31;
  const uint16_t* xh = X + (size_t)h * N * D;
  const int rbase = blockIdx.x * (AK_WAVES * 32 * AK_RB) + wave * 32 * AK_RB + jl;
  u32x4 bx[AK_RB][2];
  float best[AK_RB];
  int bidx[AK_RB];
#pragma unroll
  for (int k = 0; k < AK_RB; ++k) {
    const int row = rbase + 32 * k;
    const bool ok = row < N;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bx[k][s] = u32x4{0u, 0u, 0u, 0u};
      if (ok) bx[k][s] = *(const u32x4*)(xh + (size_t)row * D + 16 * s + 8 * hh);
    }
    // pruning bound from the row's previous label
    best[k] = __builtin_inff();
    bidx[k] = 0;
    const int g = (ok && guess) ? guess[(size_t)h * N + row] : -1;
    const bool have = g >= 0 && g < C;
    float part = 0.f, mag = 0.f;
    if (have) {
      const uint16_t* cg = cprep + ((size_t)h * C + g) * D;
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4 cv = *(const u32x4*)(cg + 16 * s + 8 * hh);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float x0 = h2f((uint16_t)(bx[k][s][t] & 0xffff)), c0 = h2f((uint16_t)(cv[t] & 0xffff));
          const float x1 = h2f((uint16_t)(bx[k][s][t] >> 16)), c1 = h2f((uint16_t)(cv[t] >> 16));
          part = fmaf(x0, c0, part);
          part = fmaf(x1, c1, part);
          mag = fmaf(fabsf(x0), fabsf(c0), mag);
          mag = fmaf(fabsf(x1), fabsf(c1), mag);
        }
      }
    }
    const float opart = __builtin_bit_cast(float, half_partner(__builtin_bit_cast(uint32_t, part)));
    const float omag = __builtin_bit_cast(float, half_partner(__builtin_bit_cast(uint32_t, mag)));
    if (have) {
      const float cn = cnorm[(size_t)h * C + g];
      const float d = cn + (hh ? opart + part : part + opart);
      const float sz = fabsf(cn) + (hh ? omag + mag : mag + omag);
      best[k] = d + 0x1p-16f * sz + 0x1p-126f;
      bidx[k] = g;
    }
  }
  auto mn = [](float a, float b) { return __builtin_elementwise_minimum(a, b); };
  const u32x4* cph = (const u32x4*)(cprep + (size_t)h * C * D);
  for (int c0 = 0; c0 < Cp; c0 += CMAX) {
  const int nc = Cp - c0 < CMAX ? Cp - c0 : CMAX;
  if (c0 > 0) __syncthreads();  // every wave is done with the previous chunk
  for (int i = tid; i < nc * 4; i += AK_WAVES * 64 * CS) {
    const int r = i >> 2, c = i & 3;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (c0 + r < C) v = cph[(size_t)c0 * 4 + i];
    ((u32x4*)sC)[r * 4 + (c ^ ((r >> 2) & 3))] = v;
  }
  for (int i = tid; i < nc; i += AK_WAVES * 64 * CS)
    sN[i] = c0 + i < C ? cnorm[(size_t)h * C + c0 + i] : __builtin_inff();
  __syncthreads();
  for (int cb = cg; cb < nc / 32; cb += CS) {
    const int r = cb * 32 + jl;
    const u32x4* crow = (const u32x4*)sC + r * 4;
    const u32x4 a0 = crow[(0 + hh) ^ ((r >> 2) & 3)];
    const u32x4 a1 = crow[(2 + hh) ^ ((r >> 2) & 3)];
    f32x16 init;
#pragma unroll
    for (int gq = 0; gq < 4; ++gq) {
      const float4 nv = *(const float4*)(sN + cb * 32 + 8 * gq + 4 * hh);
      init[4 * gq + 0] = nv.x;
      init[4 * gq + 1] = nv.y;
      init[4 * gq + 2] = nv.z;
      init[4 * gq + 3] = nv.w;
    }
#pragma unroll
    for (int k = 0; k < AK_RB; ++k) {
      f32x16 acc = Mfma<F16T>::run(a0, bx[k][0], init);
      acc = Mfma<F16T>::run(a1, bx[k][1], acc);
      float t8[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) t8[i] = mn(acc[2 * i], acc[2 * i + 1]);
      const float bmin = mn(mn(mn(t8[0], t8[1]), mn(t8[2], t8[3])), mn(mn(t8[4], t8[5]), mn(t8[6], t8[7])));
      if (__ballot(bmin < best[k]) != 0ull) {
        if (bmin < best[k]) {
          int ia = 15;
#pragma unroll
          for (int a = 14; a >= 0; --a) ia = acc[a] == bmin ? a : ia;
          best[k] = bmin;
          bidx[k] = c0 + cb * 32 + 8 * (ia >> 2) + 4 * hh + (ia & 3);
        }
      }
    }
  }
  }
  int lab[AK_RB];
#pragma unroll
  for (int k = 0; k < AK_RB; ++k) {
    const float ob = __builtin_bit_cast(float, half_partner(__builtin_bit_cast(uint32_t, best[k])));
    const int oi = (int)half_partner((uint32_t)bidx[k]);
    lab[k] = bidx[k];
    if (ob < best[k] || (ob == best[k] && oi < bidx[k])) {
      lab[k] = oi;
      best[k] = ob;
    }
  }
  if constexpr (CS > 1) {
    // the other group's best of each row, ties to the lower index
    static_assert(CS == 2 && CMAX * 4 >= AK_WAVES * 32 * AK_RB * 4, "the values fit");
    int* sI = (int*)sC;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < AK_RB; ++k)
      if (cg == 1 && hh == 0) {
        sN[(wave * AK_RB + k) * 32 + jl] = best[k];
        sI[(wave * AK_RB + k) * 32 + jl] = lab[k];
      }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < AK_RB; ++k)
      if (cg == 0) {
        const float ob = sN[(wave * AK_RB + k) * 32 + jl];
        const int oi = sI[(wave * AK_RB + k) * 32 + jl];
        if (ob < best[k] || (ob == best[k] && oi < lab[k])) lab[k] = oi;
      }
  }
  const bool owner = cg == 0 && hh == 0;
#pragma unroll
  for (int k = 0; k < AK_RB; ++k) {
    const int row = rbase + 32 * k;
    lab[k] = row >= pin_begin ? pin_label : lab[k];
    if (row < N && owner) labels[(size_t)h * N + row] = lab[k];
  }
  // the chunk's label histogram, in the LDS of the centroids
  static_assert(CMAX * D * 2 >= KM_MAXC * 4, "the histogram fits the centroid chunk");
  int* hist = (int*)sC;
  __syncthreads();
  for (int i = tid; i < C; i += AK_WAVES * 64 * CS) hist[i] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < AK_RB; ++k)
    if (rbase + 32 * k < N && owner) atomicAdd(&hist[lab[k]], 1);
  __syncthreads();
  int32_t* ho = ga.chist + ((size_t)h * gridDim.x + blockIdx.x) * C;
  for (int i = tid; i < C; i += AK_WAVES * 64 * CS) ho[i] = hist[i];
}

// ---------------------------------------------------------------------------
// stable counting sort of labels -> counts, cbase (exclusive scan), perm, over
// chunks of 256 RB rows.  Like the assignment, each kernel takes up to two
// label sets in one launch (blockIdx.z).  Rows whose label is not in [0, C) are
// in no cluster: not counted, and perm ends before them.
// ---------------------------------------------------------------------------
struct SortArgs {
  const int32_t* lab;  // [H, N]
  int32_t* chist;      // [H, chunks, C]
  int32_t* counts;     // [H, C]
  int32_t* cbase;      // [H, C]
  int32_t* perm;       // [H, N]
  int C;
};

__global__ __launch_bounds__(256) void sort_hist_kernel(const int32_t* __restrict__ lab,
                                                        int32_t* __restrict__ chist, int N, int C,
                                                        int rows) {
  __shared__ int hist[KM_MAXC];
  const int h = blockIdx.y, k = blockIdx.x, tid = threadIdx.x;
  for (int i = tid; i < C; i += 256) hist[i] = 0;
  __syncthreads();
  const int r0 = k * rows;
  const int r1 = (r0 + rows) < N ? (r0 + rows) : N;
  for (int r = r0 + tid; r < r1; r += 256) {
    const int c = lab[(size_t)h * N + r];
    if ((unsigned)c < (unsigned)C) atomicAdd(&hist[c], 1);
  }
  __syncthreads();
  int32_t* out = chist + ((size_t)h * gridDim.x + k) * C;
  for (int i = tid; i < C; i += 256) out[i] = hist[i];
}

// chunk-local start offsets: chist[h, k, c] <- sum of chist[h, k', c] over
// k' < k, and counts[h, c] <- the column total.  One work-group per 64
// clusters, lane = cluster, a quarter of the chunks per wave: the quarters'
// totals are taken first (their chunks read 16 at a time, all in flight
// together), so the latency is a few memory round trips, not one per chunk.
#define SCAN_GRP 16
__global__ __launch_bounds__(256) void sort_colscan_kernel(SortArgs g0, SortArgs g1, int nChunk) {
  __shared__ int tot[4][64];
  const SortArgs& g = blockIdx.z ? g1 : g0;
  const int C = g.C;
  const int h = blockIdx.y, l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = blockIdx.x * 64 + l;
  const bool in = c < C;
  int32_t* col = g.chist + (size_t)h * nChunk * C + (in ? c : 0);
  const int per = (nChunk + 3) / 4;
  const int ka = w * per, kb = ka + per < nChunk ? ka + per : nChunk;
  int v[SCAN_GRP];
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < SCAN_GRP; ++i) v[i] = in && k0 + i < kb ? col[(size_t)(k0 + i) * C] : 0;
  };
  int sum = 0;
  for (int k0 = ka; k0 < kb; k0 += SCAN_GRP) {
    load(k0);
#pragma unroll
    for (int i = 0; i < SCAN_GRP; ++i) sum += v[i];
  }
  tot[w][l] = sum;
  __syncthreads();
  int run = 0;
  for (int i = 0; i < w; ++i) run += tot[i][l];
  if (in && w == 3) g.counts[(size_t)h * C + c] = run + sum;
  for (int k0 = ka; k0 < kb; k0 += SCAN_GRP) {
    if (per > SCAN_GRP) load(k0);  // else the only group is still held
#pragma unroll
    for (int i = 0; i < SCAN_GRP; ++i) {
      if (in && k0 + i < kb) col[(size_t)(k0 + i) * C] = run;
      run += v[i];
    }
  }
}

__device__ inline void wave_sync_km() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One work-group of four waves per chunk, 64 RB consecutive rows per wave;
// rows of equal label keep their order (each wave's own histogram gives the
// waves' starts, ballot ranking the rows of a wave).  A cluster's start in the
// permutation is the exclusive scan of the counts over clusters (formed here;
// the first chunk's work-group writes it to cbase) plus the chunk-local
// offset.  With one wave per 1024-row chunk its 16 dependent ranking steps took
// 9-20 us of every sort of a small call, and the scan was a launch of its own.
template <int RB>
__global__ __launch_bounds__(256) void sort_scatter_kernel(SortArgs g0, SortArgs g1, int N,
                                                           int nChunk) {
  extern __shared__ int cc[];  // [4][C]
  __shared__ int wsum[4];
  const SortArgs& g = blockIdx.z ? g1 : g0;
  const int C = g.C;
  const int h = blockIdx.y, k = blockIdx.x, tid = threadIdx.x, l = tid & 63, w = tid >> 6;
  const int r0 = k * 256 * RB + w * 64 * RB;
  int* mine = cc + w * C;
  int labs[RB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int row = r0 + 64 * i + l;
    labs[i] = row < N ? g.lab[(size_t)h * N + row] : -1;
    if ((unsigned)labs[i] >= (unsigned)C) labs[i] = -1;  // in no cluster
  }
  for (int c = l; c < C; c += 64) mine[c] = 0;
  wave_sync_km();
#pragma unroll
  for (int i = 0; i < RB; ++i)
    if (labs[i] >= 0) atomicAdd(&mine[labs[i]], 1);
  // exclusive scan of the head's counts: thread tid owns clusters per tid ..
  const int per = (C + 255) / 256;
  const int32_t* cnt = g.counts + (size_t)h * C;
  int loc = 0;
  for (int i = 0; i < per; ++i)
    if (tid * per + i < C) loc += cnt[tid * per + i];
  const int inc = wave_incl_scan(loc);
  if (l == 63) wsum[w] = inc;
  __syncthreads();
  int run = inc - loc;
  for (int i = 0; i < w; ++i) run += wsum[i];
  const int32_t* off = g.chist + ((size_t)h * nChunk + k) * C;
  for (int i = 0; i < per; ++i) {
    const int c = tid * per + i;
    if (c < C) {
      if (k == 0) g.cbase[(size_t)h * C + c] = run;
      int start = run + off[c];
      run += cnt[c];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = cc[j * C + c];
        cc[j * C + c] = start;
        start += t;
      }
    }
  }
  __syncthreads();
  int lbits = 1;
  while ((1 << lbits) < C) ++lbits;
  const unsigned long long lt = (1ull << l) - 1ull;
#pragma unroll
  for (int i = 0; i < RB; ++i) {
    const int row = r0 + 64 * i + l;
    if (r0 + 64 * i >= N) break;  // wave-uniform
    const int c = labs[i];
    const bool valid = c >= 0;
    unsigned long long peers = __ballot(valid);
    for (int b = 0; b < lbits; ++b) {
      const unsigned long long bb = __ballot((c >> b) & 1);
      peers &= ((c >> b) & 1) ? bb : ~bb;
    }
    const int rank = __popcll(peers & lt);
    const int leader = (int)__ffsll((long long)peers) - 1;
    int base = 0;
    if (valid && l == leader) {
      base = mine[c];
      mine[c] = base + __popcll(peers);
    }
    base = __shfl(base, leader < 0 ? 0 : leader, 64);
    if (valid) g.perm[(size_t)h * N + base + rank] = row;
    wave_sync_km();
  }
}

// cbase[h, c] = exclusive scan of counts[h, :] over clusters
__global__ __launch_bounds__(1024) void cbase_kernel(const int32_t* __restrict__ counts,
                                                     int32_t* __restrict__ cbase, int C) {
  __shared__ int wsum[16];
  const int h = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int per = (C + 1023) / 1024;
  int loc = 0;
  for (int i = 0; i < per; ++i) {
    const int c = tid * per + i;
    if (c < C) loc += counts[(size_t)h * C + c];
  }
  const int inc = wave_incl_scan(loc);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  int run = inc - loc;
  for (int i = 0; i < w; ++i) run += wsum[i];
  for (int i = 0; i < per; ++i) {
    const int c = tid * per + i;
    if (c < C) {
      cbase[(size_t)h * C + c] = run;
      run += counts[(size_t)h * C + c];
    }
  }
}

// Row blocks per wave of the assignment, and so the rows of a sort chunk
// (256 RB): four where the launch still has four work-groups per CU, else
// fewer, down to one.  At four throughout, 2 x 4096 rows gave the assignment 8
// work-groups (both query passes and the key pass 70 us; 30 at one) and 5 x
// 75600 gave it 370 of unequal share (172 us; 137 at two).
static int km_rb(int H, int N) {
  if ((long long)H * cdiv(N, 1024) >= 1024) return 4;
  return (long long)H * cdiv(N, 512) >= 512 ? 2 : 1;
}
static int km_chunks(int H, int N) { return cdiv(N, 256 * km_rb(H, N)); }
// Chunks of all heads that a workspace holds.  H km_chunks falls where km_rb
// steps up; a workspace sized for the longest call has to serve the shorter ones
// (and fewer heads), so its size must not: one row block has at most 2 x 511
// chunks, two at most 2 x 1023.
static size_t km_chunk_cap(int H, int N) {
  const size_t one = (size_t)H * cdiv(N, 256), four = (size_t)H * cdiv(N, 1024);
  const size_t most = four > 2046 ? four : 2046;
  return one < most ? one : most;
}

// the sort proper, from the chunk histograms; sets: 1 or 2
static int run_scatter(const SortArgs& a, const SortArgs& b, int sets, int H, int N, hipStream_t st) {
  const int nChunk = km_chunks(H, N);
  const int C = sets == 2 && b.C > a.C ? b.C : a.C;
  hipLaunchKernelGGL(sort_colscan_kernel, dim3(cdiv(C, 64), H, sets), dim3(256), 0, st, a, b, nChunk);
  const dim3 g(nChunk, H, sets);
  const size_t lds = (size_t)4 * C * sizeof(int);
  switch (km_rb(H, N)) {
    case 4: hipLaunchKernelGGL(sort_scatter_kernel<4>, g, dim3(256), lds, st, a, b, N, nChunk); break;
    case 2: hipLaunchKernelGGL(sort_scatter_kernel<2>, g, dim3(256), lds, st, a, b, N, nChunk); break;
    default: hipLaunchKernelGGL(sort_scatter_kernel<1>, g, dim3(256), lds, st, a, b, N, nChunk);
  }
  return t2t_check_launch("counting sort");
}

static int run_sort(const int32_t* lab, int32_t* counts, int32_t* cbase, int32_t* perm,
                    int32_t* chist, int H, int N, int C, hipStream_t st) {
  const int rows = 256 * km_rb(H, N);
  hipLaunchKernelGGL(sort_hist_kernel, dim3(cdiv(N, rows), H), dim3(256), 0, st, lab, chist, N, C, rows);
  const SortArgs a{lab, chist, counts, cbase, perm, C};
  return run_scatter(a, a, 1, H, N, st);
}

// ---------------------------------------------------------------------------
// per-cluster integer sums in sorted order -> fp16 means (one wave/cluster)
//   MODE 0: rne(x * 32768) sums, mean = fp16(f32(S) / (32768 * f32(n)))
//   MODE 1: rne(x * 2^20) sums, mean = fp16(f32(f64(S) / 2^20 / f64(n)))
// empty clusters keep `old`.
// ---------------------------------------------------------------------------
// WPC waves share a cluster (their sums are exact integers, so the split does
// not change the result): four when the clusters alone would leave the chip
// nearly empty and a wave walking its cluster 64 rows at a time is the whole
// launch's time.  cprep / cnorm (optional): -2 mean and its squared norm, as
// cen_prep_kernel gives them, for the next assignment.
template <int MODE, int WPC>
__global__ __launch_bounds__(256) void fixed_mean_kernel(
    const uint16_t* __restrict__ X, const int32_t* __restrict__ perm,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ cbase,
    const uint16_t* __restrict__ old, uint16_t* __restrict__ out, uint16_t* __restrict__ cprep,
    float* __restrict__ cnorm, int N, int C) {
  __shared__ long long part[WPC > 1 ? WPC : 1][32];
  const int h = blockIdx.y;
  const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int c = WPC > 1 ? blockIdx.x : blockIdx.x * 4 + w;
  if (c >= C) return;
  const int n = counts[(size_t)h * C + c];
  const int b = cbase[(size_t)h * C + c];
  // lane l sums dims 4 (l % 8) .. + 3 of rows i with i % 8 = l / 8: the
  // cluster's row indices are read 64 at a time (one coalesced load, the next
  // one's in flight) and broadcast, so eight independent row loads are in
  // flight per lane.  The sums are exact integers, so their order does not
  // change the result.
  const int dq = l & 7, rg = l >> 3;
  const float scale = MODE == 0 ? 32768.0f : 1048576.0f;
  long long S[4] = {0, 0, 0, 0};
  const int32_t* ph = perm + (size_t)h * N + b;
  const uint16_t* xh = X + (size_t)h * N * KM_R + 4 * dq;
  const int first = WPC > 1 ? 64 * w : 0;
  int nxt = first + l < n ? ph[first + l] : -1;
  for (int i0 = first; i0 < n; i0 += 64 * WPC) {
    const int myrow = nxt;
    nxt = i0 + 64 * WPC + l < n ? ph[i0 + 64 * WPC + l] : -1;
    u32x2 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int row = __shfl(myrow, 8 * j + rg, 64);
      v[j] = row >= 0 ? *(const u32x2*)(xh + (size_t)row * KM_R) : u32x2{0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint16_t x = (uint16_t)(v[j][e >> 1] >> (16 * (e & 1)));
        S[e] += (long long)rintf(h2f(x) * scale);
      }
  }
  // sum over the eight row groups (lane bits 3..5), then over the waves
#pragma unroll
  for (int m = 8; m < 64; m <<= 1)
#pragma unroll
    for (int e = 0; e < 4; ++e) S[e] += __shfl_xor(S[e], m, 64);
  if constexpr (WPC > 1) {
    if (rg == 0)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[w][4 * dq + e] = S[e];
    __syncthreads();
    if (w > 0) return;
#pragma unroll
    for (int i = 1; i < WPC; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) S[e] += part[i][4 * dq + e];
  }
  float mv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const size_t o = ((size_t)h * C + c) * KM_R + 4 * dq + e;
    uint16_t v;
    if (n == 0) {
      v = old[o];
    } else if (MODE == 0) {
      v = f2h(opaque((float)S[e] / (32768.0f * (float)n)));
    } else {
      const double m = ((double)S[e] / 1048576.0) / (double)n;
      v = f2h(opaque((float)m));
    }
    mv[e] = h2f(v);
    if (rg == 0) {
      out[o] = v;
      if (cprep) cprep[o] = f2h(-2.0f * mv[e]);
    }
  }
  if (cnorm) {  // dims in order: dim 4 i + e is lane i's mv[e]
    float s = 0.f;
#pragma unroll
    for (int d = 0; d < KM_R; ++d) {
      const float v = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mv[d & 3]), d >> 2));
      s = s + v * v;
    }
    if (l == 0) cnorm[(size_t)h * C + c] = s;
  }
}

template <int MODE>
static void launch_fixed_mean(const void* X, const int32_t* perm, const int32_t* counts,
                              const int32_t* cbase, const void* old, void* out, uint16_t* cprep,
                              float* cnorm, int H, int N, int C, hipStream_t st) {
  if ((long long)H * C < 4096)
    hipLaunchKernelGGL((fixed_mean_kernel<MODE, 4>), dim3(C, H), dim3(256), 0, st, (const uint16_t*)X,
                       perm, counts, cbase, (const uint16_t*)old, (uint16_t*)out, cprep, cnorm, N, C);
  else
    hipLaunchKernelGGL((fixed_mean_kernel<MODE, 1>), dim3(cdiv(C, 4), H), dim3(256), 0, st,
                       (const uint16_t*)X, perm, counts, cbase, (const uint16_t*)old, (uint16_t*)out,
                       cprep, cnorm, N, C);
}

// ---------------------------------------------------------------------------
// key side: per cluster, sequential fp32 sums of KU (lanes 0..31, one dim
// each) and V (two dims per lane) in sorted row order; V_sorted rows; ck2.
// perm == nullptr: rows are already cluster ordered (V_sorted input).
// ---------------------------------------------------------------------------
// MEAN: vsum and ck2 hold the cluster's means of V (over max(n, 1)) and KU (the
// fused_update_vstats outputs), and cmax is not written; or, where ck16 is given,
// ck16 and V_sorted hold those means in 16 bits (fp16, and V's type).
#define KG_UNR 16
template <typename T, bool MEAN>
__global__ __launch_bounds__(256) void key_gather_kernel(
    const uint16_t* __restrict__ KU, const uint16_t* __restrict__ V,
    const int32_t* __restrict__ perm, const int32_t* __restrict__ counts,
    const int32_t* __restrict__ cbase, const uint16_t* __restrict__ ck0, float* __restrict__ ck2,
    uint16_t* __restrict__ V_sorted, float* __restrict__ vsum, float* __restrict__ cmax, int N,
    int C, long long svh, long long svn, uint16_t* __restrict__ ck16, uint16_t* __restrict__ cks,
    float scale) {
  const int h = blockIdx.y;
  const int l = threadIdx.x & 63;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= C) return;
  const int n = counts[(size_t)h * C + c];
  const int b = cbase[(size_t)h * C + c];
  const int32_t* ph = perm ? perm + (size_t)h * N + b : nullptr;
  const uint16_t* kh = KU ? KU + (size_t)h * N * KM_R : nullptr;
  // V row n of head h at V + h svh + n svn (elements; svn even)
  const uint32_t* vh = (const uint32_t*)(V + (size_t)h * svh);
  const size_t vrow = (size_t)(svn >> 1);
  uint32_t* vsh = !MEAN && V_sorted ? (uint32_t*)(V_sorted + (size_t)h * N * 128) : nullptr;
  // lanes 0..15 also sum the projected key rows, dims 2 l and 2 l + 1 (one
  // 4-byte load per row; each dim still sums its rows in order)
  float ax0 = 0.f, ax1 = 0.f, v0 = 0.f, v1 = 0.f;
  const uint32_t* kh32 = (const uint32_t*)kh;
  // The cluster's row indices are read 64 at a time (one coalesced load) and
  // taken lane by lane as wave-uniform values, so each row's loads address
  // from a scalar base.  Rows go in chunks of KG_UNR, software pipelined:
  // chunk i + 1's loads are in flight while chunk i is stored and summed.
  // Every load is unconditional (rows past the block repeat its last row and
  // are not consumed), so the memory-counter waits can count on them.
  auto run = [&](auto KS) {
    constexpr bool ks = decltype(KS)::value;
    int nxt = (l < n) ? (ph ? ph[l] : b + l) : 0;
    for (int i0 = 0; i0 < n; i0 += 64) {
      const int myrow = nxt;
      nxt = (i0 + 64 + l < n) ? (ph ? ph[i0 + 64 + l] : b + i0 + 64 + l) : 0;
      const int m = n - i0 < 64 ? n - i0 : 64;
      uint32_t va[2][KG_UNR], xa[2][KG_UNR];
      auto load = [&](int i, uint32_t (&vv)[KG_UNR], uint32_t (&xv)[KG_UNR]) {
#pragma unroll
        for (int u = 0; u < KG_UNR; ++u) {
          const int rw = __builtin_amdgcn_readlane(myrow, i + u < m ? i + u : m - 1);
          vv[u] = __builtin_nontemporal_load(&vh[(size_t)rw * vrow + l]);
          if constexpr (ks) xv[u] = kh32[(size_t)rw * (KM_R / 2) + (l & 15)];
        }
      };
      auto consume = [&](int i, const uint32_t (&vv)[KG_UNR], const uint32_t (&xv)[KG_UNR]) {
#pragma unroll
        for (int u = 0; u < KG_UNR; ++u) {
          if (i + u >= m) break;
          if (vsh) vsh[(size_t)(b + i0 + i + u) * 64 + l] = vv[u];
          v0 += T::to_f((uint16_t)(vv[u] & 0xffff));
          v1 += T::to_f((uint16_t)(vv[u] >> 16));
          if constexpr (ks) {
            ax0 += h2f((uint16_t)(xv[u] & 0xffff));
            ax1 += h2f((uint16_t)(xv[u] >> 16));
          }
        }
      };
      load(0, va[0], xa[0]);
      for (int i = 0; i < m; i += 2 * KG_UNR) {
        load(i + KG_UNR, va[1], xa[1]);
        consume(i, va[0], xa[0]);
        if (i + KG_UNR >= m) break;
        if (i + 2 * KG_UNR < m) load(i + 2 * KG_UNR, va[0], xa[0]);
        consume(i + KG_UNR, va[1], xa[1]);
      }
    }
  };
  if (kh32)
    run(std::true_type{});
  else
    run(std::false_type{});
  const size_t vi = ((size_t)h * C + c) * 128 + 2 * l;
  if constexpr (MEAN) {
    const float d = n ? (float)n : 1.0f;
    const float w0 = opaque(v0 / d), w1 = opaque(v1 / d);
    if (ck16) {
      *(uint32_t*)(V_sorted + vi) = (uint32_t)T::from_f(w0) | ((uint32_t)T::from_f(w1) << 16);
    } else {
      vsum[vi] = w0;
      vsum[vi + 1] = w1;
    }
  } else {
    float* vo = vsum + vi;
    vo[0] = v0;
    vo[1] = v1;
    // the cluster's largest |value sum|, for the per-head scale lam
    const float mx = wave_max(fmaxf(fabsf(v0), fabsf(v1)));
    if (l == 0) cmax[(size_t)h * C + c] = mx;
  }
  if ((ck2 || (MEAN && ck16)) && l < 16) {
    const size_t o = ((size_t)h * C + c) * KM_R + 2 * l;
    const float m0 = opaque(n ? ax0 / (float)n : h2f(ck0[o]));
    const float m1 = opaque(n ? ax1 / (float)n : h2f(ck0[o + 1]));
    if (ck2) {
      ck2[o] = m0;
      ck2[o + 1] = m1;
    }
    if (ck16) {  // the finalised centroids as well (centroid_finalize_kernel)
      *(uint32_t*)(ck16 + o) = (uint32_t)f2h(m0) | ((uint32_t)f2h(m1) << 16);
      if constexpr (!MEAN)
        *(uint32_t*)(cks + o) =
            (uint32_t)f2h(opaque(m0 * scale)) | ((uint32_t)f2h(opaque(m1 * scale)) << 16);
    }
  }
}

// lam = max(1, max|vsum| / 32768); sumv = fp16(vsum * (1 / lam)).  The grid
// spans every head's 128 C values (VS_PER per thread): each block reduces the
// head's C per-cluster maxima (cmax, written by key_gather_kernel) to lam
// itself, so the head needs no single-block pass over all of vsum.
#define VS_PER 8
__global__ __launch_bounds__(1024) void vstats_kernel(const float* __restrict__ vsum,
                                                      const float* __restrict__ cmax,
                                                      uint16_t* __restrict__ sumv,
                                                      float* __restrict__ lam, int C) {
  __shared__ float red[16];
  const int h = blockIdx.y, tid = threadIdx.x;
  const float* ch = cmax + (size_t)h * C;
  float mx = 0.f;
  for (int i = tid; i < C; i += 1024) mx = fmaxf(mx, ch[i]);
  mx = wave_max(mx);
  if ((tid & 63) == 0) red[tid >> 6] = mx;
  __syncthreads();
  mx = 0.f;
  for (int i = 0; i < 16; ++i) mx = fmaxf(mx, red[i]);
  const float lm = fmaxf(1.0f, mx / 32768.0f);
  const float inv = 1.0f / lm;
  if (blockIdx.x == 0 && tid == 0) lam[h] = lm;
  const size_t CE = (size_t)C * 128;
  const size_t i0 = ((size_t)blockIdx.x * 1024 + tid) * VS_PER;
  const float* vh = vsum + (size_t)h * CE;
  uint16_t* sh = sumv + (size_t)h * CE;
  if (i0 + VS_PER <= CE) {  // CE is a multiple of 128: every group is whole
    const f32x4 a = *(const f32x4*)(vh + i0), b = *(const f32x4*)(vh + i0 + 4);
    u32x4 o;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      o[e] = (uint32_t)f2h(opaque(a[2 * e] * inv)) | ((uint32_t)f2h(opaque(a[2 * e + 1] * inv)) << 16);
      o[2 + e] = (uint32_t)f2h(opaque(b[2 * e] * inv)) | ((uint32_t)f2h(opaque(b[2 * e + 1] * inv)) << 16);
    }
    *(u32x4*)(sh + i0) = o;
  }
}
static void launch_vstats(const float* vsum, const float* cmax, void* sumv, float* lam, int H,
                          int C, const T2tCentroidOut& co, hipStream_t st) {
  if (co.tiles) {  // with the tile image that holds the same sums
    t2t_launch_vstats_tiles(vsum, cmax, co.cks, sumv, lam, co.tiles, H, st);
    return;
  }
  hipLaunchKernelGGL(vstats_kernel, dim3(cdiv(C * 128, 1024 * VS_PER), H), dim3(1024), 0, st,
                     vsum, cmax, (uint16_t*)sumv, lam, C);
}

// ---------------------------------------------------------------------------
// host entry points
// ---------------------------------------------------------------------------
struct KmmWs {
  int32_t* qlab1;
  uint16_t* cq1;
  int32_t* perm1;
  int32_t* counts1;
  int32_t* cbase1;
  int32_t* cbaseq;
  int32_t* cbasek;
  int32_t* chistq;
  int32_t* chistk;
  float* vsum;
  float* cmax;
  uint16_t* cprepq;  // -2c of the query centroids of the assignment in flight
  float* cnormq;     // and their squared norms
  uint16_t* cprepk;  // the same of the key centroids
  float* cnormk;
  size_t total;
};

static KmmWs kmm_layout(int H, int N, int CQ, int CK, void* base) {
  WsCarver w(base);
  KmmWs k;
  const size_t chunks = km_chunk_cap(H, N);
  k.qlab1 = w.take<int32_t>((size_t)H * N);
  k.cq1 = w.take<uint16_t>((size_t)H * CQ * KM_R);
  k.perm1 = w.take<int32_t>((size_t)H * N);
  k.counts1 = w.take<int32_t>((size_t)H * CQ);
  k.cbase1 = w.take<int32_t>((size_t)H * CQ);
  k.cbaseq = w.take<int32_t>((size_t)H * CQ);
  k.cbasek = w.take<int32_t>((size_t)H * CK);
  k.chistq = w.take<int32_t>(chunks * CQ);
  k.chistk = w.take<int32_t>(chunks * CK);
  k.vsum = w.take<float>((size_t)H * CK * 128);
  k.cmax = w.take<float>((size_t)H * CK);
  k.cprepq = w.take<uint16_t>((size_t)H * CQ * KM_R);
  k.cnormq = w.take<float>((size_t)H * CQ);
  k.cprepk = w.take<uint16_t>((size_t)H * CK * KM_R);
  k.cnormk = w.take<float>((size_t)H * CK);
  k.total = w.off;
  return k;
}

extern "C" size_t t2t_kmm_ws_bytes(int H, int N, int CQ, int CK) {
  return kmm_layout(H, N, CQ, CK, nullptr).total;
}

// -2c (exact in fp16) and the fp32 squared norm of every centroid, summed
// sequentially over the dims (each square is exact): the operands of
// assign_km_kernel, for the query (blockIdx.z 0) and key centroids
__global__ __launch_bounds__(256) void cen_prep_kernel(
    const uint16_t* __restrict__ cenq, uint16_t* __restrict__ cprepq, float* __restrict__ cnormq,
    int CQ, const uint16_t* __restrict__ cenk, uint16_t* __restrict__ cprepk,
    float* __restrict__ cnormk, int CK) {
  const uint16_t* cen = blockIdx.z ? cenk : cenq;
  const int C = blockIdx.z ? CK : CQ;
  const int h = blockIdx.y, ci = blockIdx.x * 256 + threadIdx.x;
  if (ci >= C) return;
  const u32x4* cp = (const u32x4*)(cen + ((size_t)h * C + ci) * KM_R);
  u32x4* op = (u32x4*)((blockIdx.z ? cprepk : cprepq) + ((size_t)h * C + ci) * KM_R);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32x4 v = cp[i];
    u32x4 o;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float a = h2f((uint16_t)(v[t] & 0xffff)), b = h2f((uint16_t)(v[t] >> 16));
      s = s + a * a;
      s = s + b * b;
      o[t] = (uint32_t)f2h(-2.0f * a) | ((uint32_t)f2h(-2.0f * b) << 16);
    }
    op[i] = o;
  }
  (blockIdx.z ? cnormk : cnormq)[(size_t)h * C + ci] = s;
}

// sets: 1 or 2 row sets in one launch
static int launch_assign_km(const AssignArgs& a, const AssignArgs& b, int sets, int H, int N,
                            hipStream_t st) {
  const dim3 g(km_chunks(H, N), H, sets);
  switch (km_rb(H, N)) {
    case 4: hipLaunchKernelGGL((assign_km_kernel<4, 1>), g, dim3(AK_WAVES * 64), 0, st, a, b, N); break;
    case 2: hipLaunchKernelGGL((assign_km_kernel<2, 1>), g, dim3(AK_WAVES * 64), 0, st, a, b, N); break;
    default:
      if ((long long)g.x * H * sets <= 256)
        hipLaunchKernelGGL((assign_km_kernel<1, 2>), g, dim3(AK_WAVES * 128), 0, st, a, b, N);
      else
        hipLaunchKernelGGL((assign_km_kernel<1, 1>), g, dim3(AK_WAVES * 64), 0, st, a, b, N);
  }
  return t2t_check_launch("assign");
}

template <typename T>
static void launch_key_gather(const void* KU, const void* V, const int32_t* perm,
                              const int32_t* counts, const int32_t* cbase, const void* ck0,
                              float* ck2, void* V_sorted, float* vsum, float* cmax, int H, int N,
                              int C, long long svh, long long svn, const T2tCentroidOut& co,
                              hipStream_t st) {
  hipLaunchKernelGGL((key_gather_kernel<T, false>), dim3(cdiv(C, 4), H), dim3(256), 0, st,
                     (const uint16_t*)KU, (const uint16_t*)V, perm, counts, cbase,
                     (const uint16_t*)ck0, ck2, (uint16_t*)V_sorted, vsum, cmax, N, C, svh, svn,
                     (uint16_t*)co.ck16, (uint16_t*)co.cks, co.scale);
}

#define KM_CHECK(x)            \
  do {                         \
    int _rc = (x);             \
    if (_rc) return _rc;       \
  } while (0)

static int kmm_impl(const void* QU, const void* KU, const void* V, int v_dtype,
                    const void* cq0, const void* ck0, int32_t* qlab, void* cq2, int32_t* klab,
                    float* ck2, int32_t* qcounts, int32_t* qperm, int32_t* kcounts,
                    int32_t* kperm, void* V_sorted, void* sumv, float* lam, int H, int N, int CQ,
                    int CK, int pin_tail, void* ws, size_t ws_bytes, long long svh,
                    long long svn, const T2tCentroidOut& co, void* stream) {
  T2T_REQUIRE(!co.tiles || CK == 2048, "kmm_run: the tile image holds 2048 clusters, not %d", CK);
  T2T_REQUIRE(QU && KU && V && cq0 && ck0 && qlab && cq2 && klab && ck2 && qcounts && qperm &&
                  kcounts && kperm && sumv && lam,
              "kmm_run: null pointer");  // V_sorted may be NULL: not written
  T2T_REQUIRE(v_dtype == T2T_F16 || v_dtype == T2T_BF16, "kmm_run: dtype %d", v_dtype);
  T2T_REQUIRE(H > 0 && N > 0, "kmm_run: H=%d N=%d", H, N);
  T2T_REQUIRE(CQ >= 1 && CQ <= KM_MAXC && CK >= 1 && CK <= KM_MAXC,
              "kmm_run: CQ=%d CK=%d must be in [1, %d]", CQ, CK, KM_MAXC);
  T2T_REQUIRE(pin_tail >= 0 && pin_tail <= N, "kmm_run: pin_tail must be in [0, N]");
  T2T_REQUIRE(svn >= 128 && svn % 8 == 0 && svh >= 0 && svh % 8 == 0,
              "kmm_run: V strides (%lld, %lld) must be multiples of 8, row stride >= 128", svh, svn);
  const KmmWs need = kmm_layout(H, N, CQ, CK, nullptr);
  if (!ws || ws_bytes < need.total) {
    t2t_set_error("kmm_run: workspace %zu < %zu bytes", ws_bytes, need.total);
    return T2T_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  KmmWs w = kmm_layout(H, N, CQ, CK, ws);
  const int nores = N + 1;  // no pinned rows
  // The key pass does not depend on the query passes, so it shares the
  // launches of the first one.  The label buffers' previous contents (the
  // caller's labels of the last call, or anything) are warm-start guesses:
  // pass 1 starts from qlab, pass 2 from pass 1's labels, the key pass from klab
  hipLaunchKernelGGL(cen_prep_kernel, dim3(cdiv(CQ > CK ? CQ : CK, 256), H, 2), dim3(256), 0, st,
                     (const uint16_t*)cq0, w.cprepq, w.cnormq, CQ, (const uint16_t*)ck0, w.cprepk,
                     w.cnormk, CK);
  const AssignArgs ak{(const uint16_t*)KU, w.cprepk, w.cnormk, klab, klab, w.chistk, CK,
                      pin_tail > 0 ? N - pin_tail : nores, CK - 1};
  const AssignArgs aq1{(const uint16_t*)QU, w.cprepq, w.cnormq, w.qlab1, qlab, w.chistq, CQ, nores, 0};
  KM_CHECK(launch_assign_km(ak, aq1, 2, H, N, st));
  const SortArgs sk{klab, w.chistk, kcounts, w.cbasek, kperm, CK};
  const SortArgs sq1{w.qlab1, w.chistq, w.counts1, w.cbase1, w.perm1, CQ};
  KM_CHECK(run_scatter(sk, sq1, 2, H, N, st));
  launch_fixed_mean<0>(QU, w.perm1, w.counts1, w.cbase1, cq0, w.cq1, w.cprepq, w.cnormq, H, N, CQ, st);
  T2T_LAUNCH_CHECK("qmean 1");
  // query pass 2
  const AssignArgs aq2{(const uint16_t*)QU, w.cprepq, w.cnormq, qlab, w.qlab1, w.chistq, CQ, nores, 0};
  KM_CHECK(launch_assign_km(aq2, aq2, 1, H, N, st));
  const SortArgs sq2{qlab, w.chistq, qcounts, w.cbaseq, qperm, CQ};
  KM_CHECK(run_scatter(sq2, sq2, 1, H, N, st));
  launch_fixed_mean<0>(QU, qperm, qcounts, w.cbaseq, w.cq1, cq2, nullptr, nullptr, H, N, CQ, st);
  T2T_LAUNCH_CHECK("qmean 2");
  // key sums and value statistics
  if (v_dtype == T2T_F16)
    launch_key_gather<F16T>(KU, V, kperm, kcounts, w.cbasek, ck0, ck2, V_sorted, w.vsum, w.cmax, H, N, CK,
                            svh, svn, co, st);
  else
    launch_key_gather<BF16T>(KU, V, kperm, kcounts, w.cbasek, ck0, ck2, V_sorted, w.vsum, w.cmax, H, N, CK,
                             svh, svn, co, st);
  T2T_LAUNCH_CHECK("key gather");
  launch_vstats(w.vsum, w.cmax, sumv, lam, H, CK, co, st);
  T2T_LAUNCH_CHECK("vstats");
  return T2T_OK;
}

extern "C" int t2t_kmm_run(const void* QU, const void* KU, const void* V, int v_dtype,
                           const void* cq0, const void* ck0, int32_t* qlab, void* cq2,
                           int32_t* klab, float* ck2, int32_t* qcounts, int32_t* qperm,
                           int32_t* kcounts, int32_t* kperm, void* V_sorted, void* sumv,
                           float* lam, int H, int N, int CQ, int CK, int pin_tail, void* ws,
                           size_t ws_bytes, void* stream) {
  return kmm_impl(QU, KU, V, v_dtype, cq0, ck0, qlab, cq2, klab, ck2, qcounts, qperm, kcounts,
                  kperm, V_sorted, sumv, lam, H, N, CQ, CK, pin_tail, ws, ws_bytes,
                  (long long)N * 128, 128, T2tCentroidOut{}, stream);
}

extern "C" int t2t_kmm_run_strided(const void* QU, const void* KU, const void* V, int v_dtype,
                                   long long v_head_stride, long long v_row_stride,
                                   const void* cq0, const void* ck0, int32_t* qlab, void* cq2,
                                   int32_t* klab, float* ck2, int32_t* qcounts, int32_t* qperm,
                                   int32_t* kcounts, int32_t* kperm, void* V_sorted, void* sumv,
                                   float* lam, int H, int N, int CQ, int CK, int pin_tail,
                                   void* ws, size_t ws_bytes, void* stream) {
  return kmm_impl(QU, KU, V, v_dtype, cq0, ck0, qlab, cq2, klab, ck2, qcounts, qperm, kcounts,
                  kperm, V_sorted, sumv, lam, H, N, CQ, CK, pin_tail, ws, ws_bytes, v_head_stride,
                  v_row_stride, T2tCentroidOut{}, stream);
}

int t2t_kmm_run_out(const void* QU, const void* KU, const void* V, int v_dtype, long long svh,
                    long long svn, const void* cq0, const void* ck0, int32_t* qlab, void* cq2,
                    int32_t* klab, float* ck2, int32_t* qcounts, int32_t* qperm, int32_t* kcounts,
                    int32_t* kperm, void* V_sorted, void* sumv, float* lam, int H, int N, int CQ, int CK,
                    int pin_tail, void* ws, size_t ws_bytes, const T2tCentroidOut& co, void* stream) {
  return kmm_impl(QU, KU, V, v_dtype, cq0, ck0, qlab, cq2, klab, ck2, qcounts, qperm, kcounts, kperm,
                  V_sorted, sumv, lam, H, N, CQ, CK, pin_tail, ws, ws_bytes, svh, svn, co, stream);
}

// ---- value statistics of a reuse call ----
struct VWs {
  int32_t* cbase;
  float* vsum;
  float* cmax;
  size_t total;
};
static VWs vws_layout(int H, int CK, void* base) {
  WsCarver w(base);
  VWs v;
  v.cbase = w.take<int32_t>((size_t)H * CK);
  v.vsum = w.take<float>((size_t)H * CK * 128);
  v.cmax = w.take<float>((size_t)H * CK);
  v.total = w.off;
  return v;
}

extern "C" size_t t2t_vstats_ws_bytes(int H, int N, int CK) {
  (void)N;
  return vws_layout(H, CK, nullptr).total;
}

static int vstats_common(const void* V, int v_dtype, const int32_t* kperm, const int32_t* kcounts,
                         void* V_sorted, void* sumv, float* lam, int H, int N, int CK, void* ws,
                         size_t ws_bytes, long long svh, long long svn, const T2tCentroidOut& co,
                         hipStream_t st) {
  T2T_REQUIRE(!co.tiles || (CK == 2048 && co.cks), "vstats: the tile image holds 2048 clusters");
  T2T_REQUIRE(V && kcounts && sumv && lam, "vstats: null pointer");
  T2T_REQUIRE(v_dtype == T2T_F16 || v_dtype == T2T_BF16, "vstats: dtype %d", v_dtype);
  T2T_REQUIRE(H > 0 && N > 0 && CK >= 1 && CK <= KM_MAXC, "vstats: H=%d N=%d CK=%d", H, N, CK);
  T2T_REQUIRE(svn >= 128 && svn % 8 == 0 && svh >= 0 && svh % 8 == 0,
              "vstats: V strides (%lld, %lld) must be multiples of 8, row stride >= 128", svh, svn);
  const size_t need = vws_layout(H, CK, nullptr).total;
  if (!ws || ws_bytes < need) {
    t2t_set_error("vstats: workspace %zu < %zu bytes", ws_bytes, need);
    return T2T_ERR_WORKSPACE;
  }
  VWs w = vws_layout(H, CK, ws);
  hipLaunchKernelGGL(cbase_kernel, dim3(H), dim3(1024), 0, st, kcounts, w.cbase, CK);
  if (v_dtype == T2T_F16)
    launch_key_gather<F16T>(nullptr, V, kperm, kcounts, w.cbase, nullptr, nullptr, V_sorted,
                            w.vsum, w.cmax, H, N, CK, svh, svn, T2tCentroidOut{}, st);
  else
    launch_key_gather<BF16T>(nullptr, V, kperm, kcounts, w.cbase, nullptr, nullptr, V_sorted,
                             w.vsum, w.cmax, H, N, CK, svh, svn, T2tCentroidOut{}, st);
  launch_vstats(w.vsum, w.cmax, sumv, lam, H, CK, co, st);
  T2T_LAUNCH_CHECK("vstats");
  return T2T_OK;
}

extern "C" int t2t_kmm_run_vstats_gather(const void* V, int v_dtype, const int32_t* kperm,
                                         const int32_t* kcounts, void* V_sorted, void* sumv,
                                         float* lam, int H, int N, int CK, void* ws,
                                         size_t ws_bytes, void* stream) {
  T2T_REQUIRE(kperm, "vstats_gather: null kperm");  // V_sorted may be NULL: not written
  return vstats_common(V, v_dtype, kperm, kcounts, V_sorted, sumv, lam, H, N, CK, ws, ws_bytes,
                       (long long)N * 128, 128, T2tCentroidOut{}, (hipStream_t)stream);
}

extern "C" int t2t_kmm_run_vstats_gather_strided(const void* V, int v_dtype,
                                                 long long v_head_stride, long long v_row_stride,
                                                 const int32_t* kperm, const int32_t* kcounts,
                                                 void* V_sorted, void* sumv, float* lam, int H,
                                                 int N, int CK, void* ws, size_t ws_bytes,
                                                 void* stream) {
  T2T_REQUIRE(kperm, "vstats_gather: null kperm");  // V_sorted may be NULL: not written
  return vstats_common(V, v_dtype, kperm, kcounts, V_sorted, sumv, lam, H, N, CK, ws, ws_bytes,
                       v_head_stride, v_row_stride, T2tCentroidOut{}, (hipStream_t)stream);
}

int t2t_vstats_gather_out(const void* V, int v_dtype, long long svh, long long svn,
                          const int32_t* kperm, const int32_t* kcounts, void* V_sorted, void* sumv,
                          float* lam, int H, int N, int CK, void* ws, size_t ws_bytes,
                          const T2tCentroidOut& co, void* stream) {
  T2T_REQUIRE(kperm, "vstats_gather: null kperm");
  return vstats_common(V, v_dtype, kperm, kcounts, V_sorted, sumv, lam, H, N, CK, ws, ws_bytes, svh, svn,
                       co, (hipStream_t)stream);
}

extern "C" int t2t_kmm_run_vstats(const void* V_sorted, int v_dtype, const int32_t* kcounts,
                                  void* sumv, float* lam, int H, int N, int CK, void* ws,
                                  size_t ws_bytes, void* stream) {
  return vstats_common(V_sorted, v_dtype, nullptr, kcounts, nullptr, sumv, lam, H, N, CK, ws,
                       ws_bytes, (long long)N * 128, 128, T2tCentroidOut{}, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------
// init_state helpers
// ---------------------------------------------------------------------------
extern "C" int t2t_fast_assign(const void* x, const void* c, int32_t* labels, int H, int N, int C,
                               int D, void* stream) {
  T2T_REQUIRE(x && c && labels, "fast_assign: null pointer");
  T2T_REQUIRE(H > 0 && N > 0 && C >= 1 && C <= KM_MAXC, "fast_assign: H=%d N=%d C=%d", H, N, C);
  T2T_REQUIRE(D == 32 || D == 64 || D == 128, "fast_assign: D=%d not in {32, 64, 128}", D);
  hipStream_t st = (hipStream_t)stream;
  int ibits = 1;
  while ((1 << ibits) < C) ++ibits;
  const dim3 g(cdiv(N, 128), H);
  if (D == 32)
    launch_fast_assign32(x, c, labels, H, N, C, ibits, nullptr, nullptr, st);
  else if (D == 64)
    hipLaunchKernelGGL((fast_assign_kernel<64>), g, dim3(256), 0, st, (const uint16_t*)x,
                       (const uint16_t*)c, labels, N, C, ibits);
  else
    hipLaunchKernelGGL((fast_assign_kernel<128>), g, dim3(256), 0, st, (const uint16_t*)x,
                       (const uint16_t*)c, labels, N, C, ibits);
  T2T_LAUNCH_CHECK("fast_assign");
  return T2T_OK;
}

struct DetWs {
  int32_t* perm;
  int32_t* cbase;
  int32_t* chist;
  size_t total;
};
static DetWs det_layout(int H, int N, int C, void* base) {
  WsCarver w(base);
  DetWs d;
  d.perm = w.take<int32_t>((size_t)H * N);
  d.cbase = w.take<int32_t>((size_t)H * C);
  d.chist = w.take<int32_t>(km_chunk_cap(H, N) * C);
  d.total = w.off;
  return d;
}

extern "C" size_t t2t_det_update_ws_bytes(int H, int N, int C) {
  return det_layout(H, N, C, nullptr).total;
}

// ---------------------------------------------------------------------------
// fp32 centroid means (the reference's fused_update_vstats without values):
// 16 lanes per cluster, two dims each, sum its rows in sorted order, fp32 and
// sequential per dim; an empty cluster keeps fp32(old).  The cluster's row
// indices are read 16 at a time and passed around within the 16 lanes, so
// each lane has 16 row loads in flight.  (One wave per cluster, its half idle
// and waiting on every row before the next, took 318 us on average over the
// 512 and 2048 cluster calls at 40 x 75600 rows.)  out16: fp16 means instead.
// With values, key_gather_kernel<T, true> sums both.
// ---------------------------------------------------------------------------
#define SM_UNR 16
__global__ __launch_bounds__(256) void seg_mean_kernel(
    const uint16_t* __restrict__ X, const int32_t* __restrict__ perm,
    const int32_t* __restrict__ counts, const int32_t* __restrict__ cbase,
    const uint16_t* old, float* __restrict__ cent, uint16_t* out16, int N, int C) {
  const int h = blockIdx.y;
  const int l = threadIdx.x & 15, q0 = threadIdx.x & 48;
  const int c = blockIdx.x * 16 + (threadIdx.x >> 4);
  const bool in = c < C;
  const int n = in ? counts[(size_t)h * C + c] : 0;
  const int32_t* ph = perm + (size_t)h * N + (in ? cbase[(size_t)h * C + c] : 0);
  const uint32_t* xh = (const uint32_t*)(X + (size_t)h * N * KM_R) + l;
  float ax0 = 0.f, ax1 = 0.f;
  int nxt = l < n ? ph[l] : 0;
  // the wave runs to its longest cluster; a finished one loads row 0 unused
  for (int i0 = 0; __ballot(i0 < n) != 0ull; i0 += SM_UNR) {
    const int my = nxt;
    nxt = i0 + SM_UNR + l < n ? ph[i0 + SM_UNR + l] : 0;
    uint32_t v[SM_UNR];
#pragma unroll
    for (int u = 0; u < SM_UNR; ++u)
      v[u] = xh[(size_t)__shfl(my, q0 + u, 64) * (KM_R / 2)];
#pragma unroll
    for (int u = 0; u < SM_UNR; ++u)
      if (i0 + u < n) {
        ax0 += h2f((uint16_t)(v[u] & 0xffff));
        ax1 += h2f((uint16_t)(v[u] >> 16));
      }
  }
  if (!in) return;
  const size_t o = ((size_t)h * C + c) * KM_R + 2 * l;
  const float m0 = n ? ax0 / (float)n : h2f(old[o]), m1 = n ? ax1 / (float)n : h2f(old[o + 1]);
  if (out16) {
    *(uint32_t*)(out16 + o) = (uint32_t)f2h(opaque(m0)) | ((uint32_t)f2h(opaque(m1)) << 16);
  } else {
    cent[o] = m0;
    cent[o + 1] = m1;
  }
}

// cent / vmean in fp32, or cent16 / vmean16 in fp16 and v's type
static int update_impl(const void* x, const int32_t* labels, const void* old, const void* v,
                       int v_dtype, float* cent, void* cent16, int32_t* counts, float* vmean,
                       void* vmean16, int H, int N, int C, int D, void* ws, size_t ws_bytes,
                       void* stream) {
  T2T_REQUIRE(x && labels && old && (cent || cent16) && counts, "fused_update_vstats: null pointer");
  T2T_REQUIRE(!v || vmean || vmean16, "fused_update_vstats: v given without vmean");
  T2T_REQUIRE(!v || v_dtype == T2T_F16 || v_dtype == T2T_BF16, "fused_update_vstats: dtype %d",
              v_dtype);
  T2T_REQUIRE(H > 0 && N > 0 && C >= 1 && C <= KM_MAXC, "fused_update_vstats: H=%d N=%d C=%d", H,
              N, C);
  T2T_REQUIRE(D == KM_R, "fused_update_vstats: D=%d (built for %d)", D, KM_R);
  const size_t need = det_layout(H, N, C, nullptr).total;
  if (!ws || ws_bytes < need) {
    t2t_set_error("fused_update_vstats: workspace %zu < %zu bytes", ws_bytes, need);
    return T2T_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  DetWs w = det_layout(H, N, C, ws);
  KM_CHECK(run_sort(labels, counts, w.cbase, w.perm, w.chist, H, N, C, st));
  const long long vs = (long long)N * 128;
#define UP_LAUNCH(T)                                                                              \
  hipLaunchKernelGGL((key_gather_kernel<T, true>), dim3(cdiv(C, 4), H), dim3(256), 0, st,         \
                     (const uint16_t*)x, (const uint16_t*)v, w.perm, counts, w.cbase,             \
                     (const uint16_t*)old, cent, (uint16_t*)vmean16, vmean, (float*)nullptr, N, C, \
                     vs, 128ll, (uint16_t*)cent16, (uint16_t*)nullptr, 0.f)
  if (!v)
    hipLaunchKernelGGL(seg_mean_kernel, dim3(cdiv(C, 16), H), dim3(256), 0, st, (const uint16_t*)x,
                       w.perm, counts, w.cbase, (const uint16_t*)old, cent, (uint16_t*)cent16, N, C);
  else if (v_dtype == T2T_BF16)
    UP_LAUNCH(BF16T);
  else
    UP_LAUNCH(F16T);
#undef UP_LAUNCH
  T2T_LAUNCH_CHECK("fused_update_vstats");
  return T2T_OK;
}

extern "C" int t2t_fused_update_vstats(const void* x, const int32_t* labels, const void* old,
                                       const void* v, int v_dtype, float* cent, int32_t* counts,
                                       float* vmean, int H, int N, int C, int D, void* ws,
                                       size_t ws_bytes, void* stream) {
  return update_impl(x, labels, old, v, v_dtype, cent, nullptr, counts, vmean, nullptr, H, N, C, D, ws,
                     ws_bytes, stream);
}

extern "C" int t2t_fused_update_vstats16(const void* x, const int32_t* labels, const void* old,
                                         const void* v, int v_dtype, void* cent16, int32_t* counts,
                                         void* vmean16, int H, int N, int C, int D, void* ws,
                                         size_t ws_bytes, void* stream) {
  return update_impl(x, labels, old, v, v_dtype, nullptr, cent16, counts, nullptr, vmean16, H, N, C, D,
                     ws, ws_bytes, stream);
}

// ---- warm Lloyd iterations (init_state) ----
struct LloydWs {
  int32_t* labels;
  int32_t* counts;
  DetWs sort;
  size_t total;
};
static LloydWs lloyd_layout(int H, int N, int C, void* base) {
  WsCarver w(base);
  LloydWs l;
  l.labels = w.take<int32_t>((size_t)H * N);
  l.counts = w.take<int32_t>((size_t)H * C);
  l.sort = det_layout(H, N, C, base ? (char*)base + w.off : nullptr);
  l.total = w.off + l.sort.total;
  return l;
}

extern "C" size_t t2t_lloyd_ws_bytes(int H, int N, int C) {
  return lloyd_layout(H, N, C, nullptr).total;
}

extern "C" int t2t_lloyd(const void* x, void* cen, int iters, int H, int N, int C, int D, void* ws,
                         size_t ws_bytes, void* stream) {
  T2T_REQUIRE(x && cen, "lloyd: null pointer");
  T2T_REQUIRE(H > 0 && N > 0 && C >= 1 && C <= KM_MAXC && iters >= 0, "lloyd: H=%d N=%d C=%d iters=%d",
              H, N, C, iters);
  T2T_REQUIRE(D == KM_R, "lloyd: D=%d (built for %d)", D, KM_R);
  const size_t need = t2t_lloyd_ws_bytes(H, N, C);
  if (!ws || ws_bytes < need) {
    t2t_set_error("lloyd: workspace %zu < %zu bytes", ws_bytes, need);
    return T2T_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  LloydWs w = lloyd_layout(H, N, C, ws);
  int ibits = 1;
  while ((1 << ibits) < C) ++ibits;
  for (int i = 0; i < iters; ++i) {
    // an iteration's labels start from the previous one's, rows in their order
    launch_fast_assign32(x, cen, w.labels, H, N, C, ibits, i ? w.labels : nullptr,
                         i ? w.sort.perm : nullptr, st);
    KM_CHECK(run_sort(w.labels, w.counts, w.sort.cbase, w.sort.perm, w.sort.chist, H, N, C, st));
    // in place: a cluster's old centroid is read by its own lanes alone
    hipLaunchKernelGGL(seg_mean_kernel, dim3(cdiv(C, 16), H), dim3(256), 0, st, (const uint16_t*)x,
                       w.sort.perm, w.counts, w.sort.cbase, (const uint16_t*)cen, (float*)nullptr,
                       (uint16_t*)cen, N, C);
  }
  T2T_LAUNCH_CHECK("lloyd");
  return T2T_OK;
}

extern "C" int t2t_det_centroid_update(const void* x, const int32_t* labels, const void* old,
                                       void* out, int32_t* counts, int H, int N, int C, int D,
                                       void* ws, size_t ws_bytes, void* stream) {
  T2T_REQUIRE(x && labels && old && out && counts, "det_update: null pointer");
  T2T_REQUIRE(H > 0 && N > 0 && C >= 1 && C <= KM_MAXC, "det_update: H=%d N=%d C=%d", H, N, C);
  T2T_REQUIRE(D == KM_R, "det_update: D=%d (built for %d)", D, KM_R);
  const size_t need = det_layout(H, N, C, nullptr).total;
  if (!ws || ws_bytes < need) {
    t2t_set_error("det_update: workspace %zu < %zu bytes", ws_bytes, need);
    return T2T_ERR_WORKSPACE;
  }
  hipStream_t st = (hipStream_t)stream;
  DetWs w = det_layout(H, N, C, ws);
  KM_CHECK(run_sort(labels, counts, w.cbase, w.perm, w.chist, H, N, C, st));
  launch_fixed_mean<1>(x, w.perm, counts, w.cbase, old, out, nullptr, nullptr, H, N, C, st);
  T2T_LAUNCH_CHECK("det_update");
  return T2T_OK;
}
