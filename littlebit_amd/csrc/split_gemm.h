// Split GEMM path: fp32 activations, more rows than the decode path takes at
// its best.  Included by littlebit_amd.hip inside its anonymous namespace.
//
//   sg_scale_kernel   A_s[m, k] = g_s[k] * input[m, k] per branch s, as bf16
//                     hi and lo = bf16(v - hi)
//   sg_latent_kernel  T_s[m, r] = l_s[r] * sum_k sV_s[r, k] * A_s[m, k], as hi / lo
//   sg_expand_kernel  y[m, n] = bias[n] + sum_b h_b[n] * sum_r sU_b[n, r] * T_b[m, r]
// and, where the k range of a stage's tiles is cut into parts so that enough
// blocks run side by side, a kernel that sums the parts' fp32 tiles in part
// order (sg_reduce_t_kernel, sg_reduce_y_kernel): every call repeats bit for
// bit.
//
// A and T rows interleave the two planes per sign word: 32 hi values then
// the 32 lo values of the same k, 128 bytes.  One k-step is one sign word per
// column: a 128-byte row segment holds both planes' operands of it, so a
// +-1 operand expanded from the word feeds the hi and the lo MFMA, and the
// stage ring is that of a 64-k step of plain bf16.
//
// What bounds it: the MFMAs, two per product.  At M = 1024 gate and up of the
// Llama-2 target (4096 -> 2 x 11008, ranks 298 + 2686) run 369 GFLOP of them
// in 328 us, 1.13 PFLOP/s, where an 8192^3 bf16 library product reaches 1.19
// on the same card; a call of few tiles is bound by its chain of steps (M =
// 300, 4096 -> 4096, ranks 205 + 1843: 48 us, 0.42 PFLOP/s).  128-row tiles
// with a 64-k step of two separate planes (128 KB of LDS ring, one wave per
// SIMD, and two accumulator sets) took 506 us and 94 us; here a block needs
// 16 KB or 32 KB of LDS and at most 128 registers, so four waves per SIMD
// hide each other's LDS reads, barriers and expansions.  A stage of four
// steps per barrier for the 32-row tiles measured no faster (M = 300 stage 2
// 21.0 -> 23.3 us: three blocks per CU instead of seven).

struct SgSeg {         // stage-1 operands of one branch
  const uint32_t* V;   // [R, KW]
  const uint32_t* Vt;  // the same words tiled (tile_v_kernel), or null
  const float* g;      // [K]
  const float* l;      // [R]
  int R;
  int RP;              // R rounded up to 128 (32 * 4 * groups of words)
  int tcol;            // first latent column of the segment in a T row
  int nt0;             // first column tile of the segment
  int64_t abase;       // offset of the segment's [M][lda] block in a
};

struct SgProj {        // stage-2 operands of one projection
  const uint32_t* U[2];
  const float* h[2];
  const float* bias;
  const float* res;    // [M, N] fp32 added to y, or null (may alias y)
  void* y;
  int RW[2];           // words per U row
  int ng[2];           // groups of 4 words, ceil(RW / 4)
  int tcol;            // latent column of branch 0 (branch 1's follow its padding)
  int nb;
  int N;
  int nt0;             // first column tile of the projection
};

struct SgParams {
  SgSeg seg[kMaxSeg];
  SgProj proj[kMaxProj];
  int nseg, nproj;
  int M, K, KW;
  int lda;             // elements per A row, 64 * KW
  int ldt;             // elements per T row, 2 * sum of RP
  int xvec;            // x (x1, rms weight) rows and every g allow 16-byte loads
  int xmode;           // LBK_INPUT_*
  const void* x;
  const void* x1;
  const float* nw;
  float eps;
  uint16_t* a;
  uint16_t* t;
  float* part;         // stage 1's parts of the k range: [parts][M][ldt / 2] fp32
  int parts;           // 1: tiles store T themselves
  int NT;              // column tiles over all segments / projections
};

// One 8-k chunk of one row per thread, every segment of the call: the input
// is read (and its transform applied) once, not once per segment.  Bound by
// its stores, 4 bytes per element and segment: q/k/v of two branches at M =
// 700, K = 4096 writes 69 MB (a block per row and segment took 32 us; this
// about 15).
// grid = (M, ceil(32 KW / (8 * 256))).
template <typename XT>
__global__ __launch_bounds__(kBlock) void sg_scale_kernel(SgParams p) {
  const int m = int(blockIdx.x), tid = int(threadIdx.x);
  const XT* __restrict__ xr = static_cast<const XT*>(p.x) + int64_t(m) * p.K;
  const XT* __restrict__ ur = p.x1 ? static_cast<const XT*>(p.x1) + int64_t(m) * p.K : xr;
  float rsm = 1.f;
  if (p.xmode == LBK_INPUT_RMSNORM) {
    __shared__ float rs[1];
    __shared__ float rscratch[kBlock / 64];
    if (p.xvec) {
      float part[1] = {0.f};
      for (int k = 8 * tid; k < p.K; k += 8 * kBlock) {
        float v[8];
        load8(xr + k, v);
#pragma unroll
        for (int i = 0; i < 8; ++i) part[0] += v[i] * v[i];
      }
      rms_finish<1, kBlock>(part, p.K, p.eps, rs, rscratch, tid);
    } else {
      rms_scales<XT, 1, kBlock>(xr, 1, p.K, p.eps, rs, rscratch, tid);
    }
    rsm = rs[0];
  }
  const int k = 8 * (int(blockIdx.y) * kBlock + tid);
  if (k >= 32 * p.KW) return;
  float v[8];
  const bool vec = p.xvec && k + 8 <= p.K;
  if (vec) {
    load8(xr + k, v);
    if (p.xmode == LBK_INPUT_RMSNORM) {
      float wv[8];
      load8(p.nw + k, wv);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] *= wv[i] * rsm;
    } else if (p.xmode == LBK_INPUT_SILU_MUL) {
      float uv[8];
      load8(ur + k, uv);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = silu_f(v[i]) * uv[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float e = 0.f;
      if (k + i < p.K) {
        e = to_f32(xr[k + i]);
        if (p.xmode == LBK_INPUT_RMSNORM) e *= p.nw[k + i] * rsm;
        else if (p.xmode == LBK_INPUT_SILU_MUL) e = silu_f(e) * to_f32(ur[k + i]);
      }
      v[i] = e;
    }
  }
  uint16_t* __restrict__ out = p.a + int64_t(m) * p.lda + (k >> 5) * 64 + (k & 31);
  for (int s = 0; s < p.nseg; ++s) {
    const float* __restrict__ g = p.seg[s].g;
    float a[8];
    if (vec) {
      load8(g + k, a);
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] *= v[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] = k + i < p.K ? v[i] * g[k + i] : 0.f;
    }
    u32x4 h, l;
    split8(a, h, l);
    uint16_t* o = out + p.seg[s].abase;
    *reinterpret_cast<u32x4*>(o) = h;
    *reinterpret_cast<u32x4*>(o + 32) = l;
  }
}

// acc[i][j] += A[m0 + 32 i + .., both planes of steps s0 .. s1) . S[.., c + 32 j + ..]
// A: rows of interleaved 128-byte steps, `src` the lane's DMA sources of step
// s0; words(g) loads the lane's columns' sign words of steps 4 g .. 4 g + 3
// (s0 a multiple of 4); boundary(g) runs before group g's MFMAs.
//
// The block's tile is 32 MI rows x 128 NJ columns, wave w of 4 taking
// columns 32 NJ w ..: a column's words are expanded by one wave only, into
// registers, straight from registers (no LDS), one 16-byte load per column
// and 4 steps.  A tiles go from global memory straight to LDS through a ring
// of 4 stages issued 3 steps ahead; 16-byte chunk c of row r is stored at
// chunk c ^ swz(r), swz(r) = (r ^ (r >> 3)) & 7 (no bank conflicts).  Vector
// loads complete in issue order, and each step issues the same loads on
// every path (clamped addresses): W = a group's word loads, F = a fill,
//   W0 F0 F1 F2 | step 0: W1 F3 | step 1: F4 | step 2: F5 | step 3: F6 | ...
// so before step ks (q = ks % 4) F(ks) has landed once at most 2 fills, and
// for q = 1, 2 also the next group's words, are outstanding.
template <int MI, int NJ, typename WordsFn, typename BoundaryFn>
__device__ __forceinline__ void sg_mainloop(const uint16_t* const (&src)[MI], int n, int g0, WordsFn&& words,
                                            BoundaryFn&& boundary, const uint32_t (&kone)[NJ],
                                            f32x16 (&acc)[MI][NJ], int tid) {
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  typedef __attribute__((address_space(1))) void* glb_ptr_t;
  constexpr int TILE = 32 * MI * 64;  // elements per stage
  __shared__ __attribute__((aligned(16))) uint16_t st0[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t st1[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t st2[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t st3[TILE];
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  uint32_t kmask = 0x80008000u;
  asm volatile("" : "+v"(kmask));
  // element offset of 16-byte chunk c of the lane's row in subtile 0; rows 32 i
  // + lr swizzle by swz(lr) ^ (4 i & 7), so subtile 1 reads chunk c ^ 4's place
  const int swz = (lr ^ (lr >> 3)) & 7;
  int off[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) off[c] = lr * 64 + (((2 * c + lh) ^ swz) << 3);
  auto fill = [&](int f, uint16_t* st) {
    const int64_t at = int64_t(min(f, n - 1)) * 64;
#pragma unroll
    for (int j = 0; j < MI; ++j)
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(src[j] + at), (lds_ptr_t)(st + (wave * MI + j) * 512), 16, 0, 0);
  };
  u32x4 wc[NJ], wn[NJ];
  auto compute = [&](const uint16_t* a, int q) {
    uint32_t w[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) w[j] = wc[j][q] >> (8 * lh);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 b[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) b[j] = signs_to_bf16x8(w[j], 2 * s, kmask, kone[j]);
#pragma unroll
      for (int pl = 0; pl < 2; ++pl)
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          // chunk 2 s + lh of plane pl: off[2 pl + s], planes swapped in odd subtiles
          const bf16x8 f = *reinterpret_cast<const bf16x8*>(a + 2048 * i + off[2 * (pl ^ (i & 1)) + s]);
#pragma unroll
          for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, b[j], acc[i][j], 0, 0, 0);
        }
    }
  };
  auto arrive = [&](auto newer) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(decltype(newer)::value));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  typedef std::integral_constant<int, 2 * MI> Fills;
  typedef std::integral_constant<int, 2 * MI + NJ> FillsWords;
  // pins the words' first use to their group: hoisted past a barrier it
  // would wait for every load in flight
  auto group = [&](int ks, const uint16_t* cur, uint16_t* nxt) {
    arrive(Fills{});
#pragma unroll
    for (int j = 0; j < NJ; ++j) wn[j] = words(g0 + (ks >> 2) + 1, j);
    fill(ks + 3, nxt);
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(wc[j]));
    boundary(g0 + (ks >> 2), wc);
    compute(cur, 0);
  };
#pragma unroll
  for (int j = 0; j < NJ; ++j) wc[j] = words(g0, j);
  __builtin_amdgcn_sched_barrier(0);
  fill(0, st0);
  __builtin_amdgcn_sched_barrier(0);
  fill(1, st1);
  __builtin_amdgcn_sched_barrier(0);
  fill(2, st2);
  __builtin_amdgcn_sched_barrier(0);
  int ks = 0;
  for (; ks + 4 <= n; ks += 4) {
    group(ks, st0, st3);
    arrive(FillsWords{});
    fill(ks + 4, st0);
    compute(st1, 1);
    arrive(FillsWords{});
    fill(ks + 5, st1);
    compute(st2, 2);
    arrive(Fills{});
    fill(ks + 6, st2);
    compute(st3, 3);
#pragma unroll
    for (int j = 0; j < NJ; ++j) wc[j] = wn[j];
  }
  if (ks < n) group(ks, st0, st3);
  if (ks + 1 < n) {
    arrive(FillsWords{});
    fill(ks + 4, st0);
    compute(st1, 1);
  }
  if (ks + 2 < n) {
    arrive(FillsWords{});
    compute(st2, 2);
  }
  // no DMA may be in flight when the block's LDS is given back
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
  asm volatile("" ::: "memory");
}

// The lane's DMA sources of a tile's rows (rows past M repeat row M - 1).
template <int MI>
__device__ __forceinline__ void sg_sources(const uint16_t* (&src)[MI], const uint16_t* A, int64_t lda, int M, int m0,
                                           int tid) {
#pragma unroll
  for (int j = 0; j < MI; ++j) {
    const int slot = ((tid >> 6) * MI + j) * 64 + (tid & 63);
    const int row = slot >> 3, c = (slot & 7) ^ ((row ^ (row >> 3)) & 7);
    src[j] = A + int64_t(min(m0 + row, M - 1)) * lda + 8 * c;
  }
}

// Words [at, at + 4) of a matrix of `total` words.  The load is moved back
// where it would pass the matrix's end; sg_shift_words then moves the words
// to their places (needed only for a row's last group).  A matrix of fewer
// than 4 words is read word by word.
__device__ __forceinline__ u32x4 sg_load_words(const uint32_t* W, int64_t at, int64_t total) {
  typedef u32x4 __attribute__((aligned(4))) u32x4u;
  if (total < 4)
    return u32x4{W[min(at, total - 1)], W[min(at + 1, total - 1)], W[min(at + 2, total - 1)], W[min(at + 3, total - 1)]};
  return *reinterpret_cast<const u32x4u*>(W + min(at, total - 4));
}
__device__ __forceinline__ u32x4 sg_shift_words(u32x4 w, int64_t at, int64_t total) {
  const int sh = total < 4 ? 0 : int(max(int64_t(0), at - (total - 4)));
  if (sh == 1) w = u32x4{w[1], w[2], w[3], 0u};
  if (sh == 2) w = u32x4{w[2], w[3], 0u, 0u};
  if (sh >= 3) w = u32x4{w[3], 0u, 0u, 0u};
  return w;
}

// Block -> (row tile, part, column tile): XCD x runs one contiguous range of
// row-tile-major order, so the blocks that read the same rows of A (or T)
// share an L2.
struct SgTile {
  int mt, part, nt;
};
__device__ __forceinline__ SgTile sg_tile(const SgParams& p) {
  const int L = xcd_contiguous_block(int(blockIdx.x), int(gridDim.x));
  SgTile t;
  t.nt = L % p.NT;
  const int mp = L / p.NT;
  t.part = mp % p.parts;
  t.mt = mp / p.parts;
  return t;
}

// Stage 1.  grid = row tiles * parts * column tiles.
template <int MI>
__global__ __launch_bounds__(kBlock, 4) void sg_latent_kernel(SgParams p) {
  constexpr int NJ = 1;
  const int tid = int(threadIdx.x), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const SgTile tl = sg_tile(p);
  int si = 0;
#pragma unroll
  for (int i = 1; i < kMaxSeg; ++i) si += (i < p.nseg && tl.nt >= p.seg[i].nt0) ? 1 : 0;
  const SgSeg& G = p.seg[__builtin_amdgcn_readfirstlane(si)];
  const int m0 = tl.mt * (32 * MI);
  const int c0 = (tl.nt - G.nt0) * (128 * NJ) + 32 * NJ * wave;  // the wave's first latent row
  const int ngr = (p.KW + 3) >> 2;
  const int ga = tl.part * ngr / p.parts, gb = (tl.part + 1) * ngr / p.parts;
  const int n = min(4 * gb, p.KW) - 4 * ga;
  const uint16_t* src[MI];
  sg_sources<MI>(src, p.a + G.abase + int64_t(ga) * 256, p.lda, p.M, m0, tid);
  const int64_t total = int64_t(G.R) * p.KW;
  int col[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) col[j] = min(c0 + 32 * j + lr, G.R - 1);
  auto words = [&](int g, int j) {
    const int gc = min(g, gb - 1);
    if (G.Vt) return *reinterpret_cast<const u32x4*>(G.Vt + ((int64_t(col[j] >> 4) * ngr + gc) * 16 + (col[j] & 15)) * 4);
    return sg_load_words(G.V, int64_t(col[j]) * p.KW + 4 * gc, total);
  };
  auto boundary = [&](int g, u32x4 (&w)[NJ]) {
    if (!G.Vt && 4 * g + 4 > p.KW) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[j] = sg_shift_words(w[j], int64_t(col[j]) * p.KW + 4 * g, total);
    }
  };
  f32x16 acc[MI][NJ];
  uint32_t kone[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    kone[j] = 0x3F803F80u;
    asm volatile("" : "+v"(kone[j]));
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[i][j] = f32x16{};
  }
  sg_mainloop<MI, NJ>(src, n, ga, words, boundary, kone, acc, tid);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int r = c0 + 32 * j + lr;
    if (r >= G.RP) continue;
    const bool live = r < G.R;  // columns R <= r < RP of T are zero
    const float lv = live ? G.l[r] : 0.f;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int m = m0 + 32 * i + 8 * (q >> 2) + 4 * lh + (q & 3);
        if (m >= p.M) continue;
        if (p.parts > 1) {
          p.part[(int64_t(tl.part) * p.M + m) * (p.ldt >> 1) + G.tcol + r] = acc[i][j][q];
        } else {
          uint16_t h, l;
          split1(live ? lv * acc[i][j][q] : 0.f, h, l);
          uint16_t* o = p.t + int64_t(m) * p.ldt + 2 * G.tcol + (r >> 5) * 64 + (r & 31);
          o[0] = h;
          o[32] = l;
        }
      }
  }
}

// T from stage 1's parts, summed in part order.  One thread per 4 columns.
__global__ __launch_bounds__(kBlock) void sg_reduce_t_kernel(SgParams p) {
  const int cols = p.ldt >> 1;
  const int64_t i = (int64_t(blockIdx.x) * kBlock + threadIdx.x) * 4;
  if (i >= int64_t(p.M) * cols) return;
  const int m = int(i / cols), c = int(i - int64_t(m) * cols);
  int si = 0;
#pragma unroll
  for (int s = 1; s < kMaxSeg; ++s) si += (s < p.nseg && c >= p.seg[s].tcol) ? 1 : 0;
  const SgSeg& G = p.seg[si];
  const int r = c - G.tcol;
  const int64_t ps = int64_t(p.M) * cols;
  f32x4 s = *reinterpret_cast<const f32x4*>(p.part + i);
  for (int q = 1; q < p.parts; ++q) s += *reinterpret_cast<const f32x4*>(p.part + i + q * ps);
  uint32_t hi[2], lo[2];
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = r + e < G.R ? s[e] * G.l[r + e] : 0.f;
  split_pairs<4>(v, hi, lo);
  uint16_t* o = p.t + int64_t(m) * p.ldt + 2 * G.tcol + (r >> 5) * 64 + (r & 31);
  *reinterpret_cast<u32x2*>(o) = u32x2{hi[0], hi[1]};
  *reinterpret_cast<u32x2*>(o + 32) = u32x2{lo[0], lo[1]};
}

// Stage 2.  grid = row tiles * column tiles (p.parts 1).  A projection's
// steps are branch 0's words, padded to whole groups of 4 (the T columns
// there are zero, whatever bits the words hold), then branch 1's: one
// pipeline through both.  One accumulator set: after branch 0 each column's
// S0 is scaled by r = (h0 / h1) 2^-e in fp32 and branch 1 is added with the
// operand +-2^-e (exact in bf16), e = max(0, exponent of h0 / h1): acc = 2^-e
// (h0 S0 + h1 S1) / h1 stays within a factor 2 of the larger term, and y = (h1
// 2^e) acc.  Where h1 is zero, or h0 / h1 past 2^126, branch 1 adds nothing.
template <typename YT, int MI, int NJ>
__global__ __launch_bounds__(kBlock, 4) void sg_expand_kernel(SgParams p) {
  const int tid = int(threadIdx.x), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const SgTile tl = sg_tile(p);
  int pi = 0;
#pragma unroll
  for (int i = 1; i < kMaxProj; ++i) pi += (i < p.nproj && tl.nt >= p.proj[i].nt0) ? 1 : 0;
  const SgProj& P = p.proj[__builtin_amdgcn_readfirstlane(pi)];
  const int m0 = tl.mt * (32 * MI);
  const int c0 = (tl.nt - P.nt0) * (128 * NJ) + 32 * NJ * wave;
  const int ng0 = P.ng[0];
  const int ngr = P.nb > 1 ? ng0 + P.ng[1] : ng0;
  const int steps = P.nb > 1 ? 4 * ng0 + P.RW[1] : P.RW[0];
  const uint16_t* src[MI];
  sg_sources<MI>(src, p.t + 2 * P.tcol, p.ldt, p.M, m0, tid);
  int col[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) col[j] = min(c0 + 32 * j + lr, P.N - 1);
  auto words = [&](int g, int j) {
    const int gc = min(g, ngr - 1);
    const int b = gc >= ng0 ? 1 : 0, gl = gc - (b ? ng0 : 0);
    const int64_t rw = b ? P.RW[1] : P.RW[0];
    return sg_load_words(b ? P.U[1] : P.U[0], int64_t(col[j]) * rw + 4 * gl, int64_t(P.N) * rw);
  };
  f32x16 acc[MI][NJ];
  uint32_t kone[NJ];
  float f[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    kone[j] = 0x3F803F80u;
    asm volatile("" : "+v"(kone[j]));
    f[j] = P.h[0][col[j]];
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[i][j] = f32x16{};
  }
  auto boundary = [&](int g, u32x4 (&w)[NJ]) {
    const int b = g >= ng0 ? 1 : 0, gl = g - (b ? ng0 : 0);
    const int rw = b ? P.RW[1] : P.RW[0];
    if (4 * gl + 4 > rw) {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        w[j] = sg_shift_words(w[j], int64_t(col[j]) * rw + 4 * gl, int64_t(P.N) * rw);
    }
    if (g == ng0) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const float h1 = P.h[1][col[j]], ratio = f[j] / h1;
        const int e = max(0, int((__float_as_uint(ratio) >> 23) & 0xffu) - 127);
        if (h1 != 0.f && e <= 126) {
          const float r = ldexpf(ratio, -e);
#pragma unroll
          for (int i = 0; i < MI; ++i) acc[i][j] *= r;
          f[j] = ldexpf(h1, e);
          kone[j] = (0x3F80u - (uint32_t(e) << 7)) * 0x10001u;
        } else {
          kone[j] = 0u;
          if (h1 != h1) f[j] = h1;
        }
      }
    }
  };
  sg_mainloop<MI, NJ>(src, steps, 0, words, boundary, kone, acc, tid);
  YT* __restrict__ y = static_cast<YT*>(P.y);
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int nn = c0 + 32 * j + lr;
    if (nn >= P.N) continue;
    const float bn = P.bias ? P.bias[nn] : 0.f;
    const float* res = P.res;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int m = m0 + 32 * i + 8 * (q >> 2) + 4 * lh + (q & 3);
        if (m >= p.M) continue;
        const size_t o = size_t(m) * P.N + nn;
        store_out(y, o, f[j] * acc[i][j][q] + bn + (res ? res[o] : 0.f));
      }
  }
}
