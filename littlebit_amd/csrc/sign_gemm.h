// GEMM path: more rows than the decode path takes.  Included by
// littlebit_amd.hip inside its anonymous namespace.
//
//   sg_scale_kernel   A_s[m, k] = g_s[k] * input[m, k] per branch s, where the
//                     input cannot be read as it is
//   sg_latent_kernel  T_s[m, r] = l_s[r] * sum_k sV_s[r, k] * A_s[m, k]
//   sg_reduce_t_kernel  T from the fp32 tiles of the parts, in part order, where
//                     stage 1's k range is cut into parts so that enough blocks
//                     run side by side (every call repeats bit for bit)
//   sg_expand_kernel  y[m, n] = bias[n] + sum_b h_b[n] * sum_r sU_b[n, r] * T_b[m, r]
//
// SPLIT (fp32 activations): A and T as bf16 hi and lo = bf16(v - hi), both
// through the MFMAs, so products keep ~2^-17 relative error.  Rows interleave
// the planes per sign word, 32 hi values then the 32 lo values of the same k,
// 128 bytes.  One k-step is one sign word per column: a 128-byte row segment
// holds both planes' operands of it, and a +-1 operand expanded from the word
// feeds the hi and the lo MFMA.  Without (bf16 activations) one plane, the
// precision of the reference's bf16 forward (littlebit.py:116-121); a 128-byte
// step is 64 k, two words.  bf16 rows of whole steps are read as they are (GB),
// with g, rounded to bf16, in the B operand.
//
// What bounds it: the MFMAs of large calls.  fp32, M = 1024, gate and up of the
// Llama-2 target (4096 -> 2 x 11008, ranks 298 + 2686): 369 GFLOP (two MFMAs per
// product) in 328 us, 1.13 PFLOP/s, where an 8192^3 bf16 library product reaches
// 1.19 on the same card.  bf16, M = 2048, the Llama-3 gate (4096 -> 14336, ranks
// 318 + 2867): 240 GFLOP in 240 us, 1.00 PFLOP/s (9 VALU per expanded operand
// and 2 MFMAs).  A call of few tiles is bound by its chain of steps (fp32, M =
// 300, 4096 -> 4096, ranks 205 + 1843: 48 us, 0.42 PFLOP/s): stage 2's 67 steps
// take 23 us and stage 1's 43 take 17, about 800 cycles each, of which 340 are
// the step itself without any memory access; what the rest waits for is not
// shown (the compiler's wait for all loads in every group of four steps, for the
// words that two forms of load merge into, is 0.7 us of the 48).  128-row tiles with 64 KB (bf16) or 128 KB
// (fp32, separate planes, two accumulator sets) of LDS ring, two and one waves
// per SIMD, took 506, 255 and 94 us for the three, and 43 us against 19 for a
// bf16 draft projection of rank 205 at M = 300; here a block needs 16 or 32 KB
// of LDS and at most 128 registers, so four waves per SIMD hide each other's LDS
// reads, barriers and expansions (where stage 1 of a bf16 call has tiles for a
// little more than three of those blocks per CU over a long K, 128-row tiles of 64
// KB, two blocks per CU, are the faster ones: figures at sg_plan).  A stage of four steps per barrier for the
// 32-row tiles measured no faster (fp32, M = 300, stage 2: 21.0 -> 23.3 us,
// three blocks per CU instead of seven).

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
  int lda;             // elements per A row: 64 KW split, else K rounded up to 64 (K of x itself)
  int ldt;             // elements per T row: tcols, twice that split
  int tcols;           // latent columns of a row, the sum of RP
  int xvec;            // x (x1, rms weight) rows and every g allow 16-byte loads
  int xmode;           // LBK_INPUT_*
  const void* x;
  const void* x1;
  const float* nw;
  float eps;
  uint16_t* a;
  uint16_t* t;
  float* part;         // stage 1's parts of the k range: [parts][M][tcols] fp32
  int parts;           // 1: tiles store T themselves
  int NT;              // column tiles over all segments / projections
};

// One 8-k chunk of one row per thread, every segment of the call: the input
// is read (and its transform applied) once, not once per segment.  Bound by
// its stores, 4 bytes per element and segment: q/k/v of two branches at M =
// 700, K = 4096 writes 69 MB (a block per row and segment took 32 us; this
// about 15).
// grid = (M, ceil(32 KW / (8 * 256))).
template <typename XT, bool SPLIT>
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
  if (k >= (SPLIT ? 32 * p.KW : p.lda)) return;
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
  uint16_t* __restrict__ out = p.a + int64_t(m) * p.lda + (SPLIT ? (k >> 5) * 64 + (k & 31) : k);
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
    if constexpr (SPLIT) *reinterpret_cast<u32x4*>(o + 32) = l;
  }
}

// acc[.][i][j] += A[m0 + 32 i + .., steps 0 .. n) . S[.., c + 32 j + ..], the
// lo plane's products into acc[NP - 1] (NP 2: a set of sums for each plane)
// A: rows of 128-byte steps, `src` the lane's DMA sources of step 0; words(g)
// loads the lane's columns' sign words of group g0 + g (4 words: 4 steps of
// one word with SPLIT, 2 steps of two without); boundary(g) runs before group
// g's MFMAs.  GB: the B operand is +-g[k] (gk = g of step 0).
//
// The block's tile is 32 MI rows x 128 NJ columns, wave w of 4 taking
// columns 32 NJ w ..: a column's words are expanded by one wave only, into
// registers, straight from registers (no LDS), one 16-byte load per column
// and group.  A tiles go from global memory straight to LDS through a ring
// of 4 stages issued 3 steps ahead; 16-byte chunk c of row r is stored at
// chunk c ^ swz(r), swz(r) = (r ^ (r >> 3)) & 7 (no bank conflicts).  Vector
// loads complete in issue order, and each step of the ring issues the same
// loads on every path (clamped addresses): W = a group's word loads, F = a fill,
//   SPLIT: W0 F0 F1 F2 | step 0: W1 F3 | step 1: F4 | step 2: F5 | step 3: F6 | ...
//   else:  W0 F0 W1 F1 F2 | step 0: W2 F3 | step 1: F4 | step 2: W3 F5 | step 3: F6 | ...
// so before step ks F(ks) has landed once at most 2 fills and the words
// issued since are outstanding (SPLIT: those of steps ks % 4 = 1, 2; else of
// every step).  With GB each F is led by a load of the 64 g values of the
// step after it, lane k's; they go to one of two LDS buffers as bf16 when
// that F is waited for (all of a part's g in LDS cost the 64-row tiles their
// fourth block per CU: 816 tiles of 4096 columns 85 us, with the buffers 66).
template <bool SPLIT, bool GB, int MI, int NJ, int NP, typename WordsFn, typename BoundaryFn>
__device__ __forceinline__ void sg_mainloop(const uint16_t* const (&src)[MI], int n, int g0, WordsFn&& words,
                                            BoundaryFn&& boundary, const uint32_t (&kone)[NJ],
                                            f32x16 (&acc)[NP][MI][NJ], int tid, const float* __restrict__ gk = nullptr) {
  static_assert(!(SPLIT && GB), "split planes carry g themselves");
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  typedef __attribute__((address_space(1))) void* glb_ptr_t;
  constexpr int TILE = 32 * MI * 64;  // elements per stage
  constexpr int GPI = SPLIT ? 1 : 2;  // groups of words per 4 steps
  __shared__ __attribute__((aligned(16))) uint16_t st0[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t st1[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t st2[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t st3[TILE];
  __shared__ __attribute__((aligned(16))) uint16_t gs[2][GB ? 64 : 1];
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  uint32_t kmask = 0x80008000u;
  asm volatile("" : "+v"(kmask));
  // element offset of 16-byte chunk 2 c + lh of the lane's row in subtile 0; rows
  // 32 i + lr swizzle by swz(lr) ^ (4 i & 7), so odd subtiles read chunk ^ 4's place
  const int swz = (lr ^ (lr >> 3)) & 7;
  int off[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) off[c] = lr * 64 + (((2 * c + lh) ^ swz) << 3);
  auto g_at = [&](int f) { return GB ? gk[64 * min(f, n - 1) + lane] : 0.f; };
  // the empty asm pins the value's first use to its step (see the words below)
  auto put_g = [&](int f, float v) {
    if constexpr (GB) {
      asm volatile("" : "+v"(v));
      if (wave == 0) gs[f & 1][lane] = f32_to_bf16(v);
    }
  };
  float gr[4];  // g of step f + 1, loaded with fill(f), at f % 4
  auto fill = [&](int f, uint16_t* st, float& gn) {
    gn = g_at(f + 1);
    const int64_t at = int64_t(min(f, n - 1)) * 64;
#pragma unroll
    for (int j = 0; j < MI; ++j)
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(src[j] + at), (lds_ptr_t)(st + (wave * MI + j) * 512), 16, 0, 0);
  };
  u32x4 wc[GPI][NJ], wn[GPI][NJ];
  auto compute = [&](const uint16_t* a, int ks, int q) {
    if constexpr (SPLIT) {
      uint32_t w[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[j] = wc[0][j][q] >> (8 * lh);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        bf16x8 b[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = signs_to_bf16x8(w[j], 2 * s, kmask, kone[j]);
#pragma unroll
        for (int pl = 0; pl < 2; ++pl)
#pragma unroll
          for (int i = 0; i < MI; ++i) {
            const bf16x8 f = *reinterpret_cast<const bf16x8*>(a + 2048 * i + off[(2 * pl + s) ^ (2 * (i & 1))]);
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              acc[pl % NP][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, b[j], acc[pl % NP][i][j], 0, 0, 0);
          }
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        u32x4 gv = {};
        if constexpr (GB) gv = *reinterpret_cast<const u32x4*>(&gs[ks & 1][16 * s + 8 * lh]);
        bf16x8 b[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const uint32_t w = wc[q >> 1][j][2 * (q & 1) + (s >> 1)] >> (8 * lh);
          b[j] = GB ? signs_times_bf16x8(w, 2 * (s & 1), kmask, gv) : signs_to_bf16x8(w, 2 * (s & 1), kmask, kone[j]);
        }
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const bf16x8 f = *reinterpret_cast<const bf16x8*>(a + 2048 * i + off[s ^ (2 * (i & 1))]);
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            acc[0][i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f, b[j], acc[0][i][j], 0, 0, 0);
        }
      }
    }
  };
  auto load_words = [&](int g, u32x4 (&w)[NJ]) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) w[j] = words(g0 + g, j);
  };
  // step ks = 4 it + q on stage `cur`, refilling `nxt` (the stage of step ks - 1).
  // TAIL: one of the last n % 4 steps, which loads nothing (no step is left to
  // read it, and the compiler drops a load that nobody reads, so it could not be
  // counted on): F(ks) has landed once at most the fills of the 2 - q later
  // steps are outstanding.
  auto step = [&](auto qc, auto tailc, int ks, const uint16_t* cur, uint16_t* nxt) {
    constexpr int q = decltype(qc)::value;
    constexpr bool TAIL = decltype(tailc)::value;
    constexpr int newer =
        TAIL ? (2 - q) * MI : 2 * (MI + (GB ? 1 : 0)) + (SPLIT ? (q == 1 || q == 2 ? NJ : 0) : NJ);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(newer));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    constexpr bool first = SPLIT ? q == 0 : (q & 1) == 0;  // the first step of a group
    constexpr int h = SPLIT ? 0 : q >> 1;
    const int g = (ks >> 2) * GPI + h;
    if constexpr (first && !TAIL) load_words(g + GPI, wn[h]);
    if constexpr (!TAIL || q < 2) put_g(ks + 1, gr[q]);
    if constexpr (!TAIL) fill(ks + 3, nxt, gr[(q + 3) & 3]);
    if constexpr (first) {
      // pins the words' first use to their group: hoisted past a barrier it
      // would wait for every load in flight
#pragma unroll
      for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(wc[h][j]));
      boundary(g0 + g, wc[h]);
    }
    compute(cur, ks, q);
  };
  constexpr std::integral_constant<int, 0> q0{};
  constexpr std::integral_constant<int, 1> q1{};
  constexpr std::integral_constant<int, 2> q2{};
  constexpr std::integral_constant<int, 3> q3{};
  put_g(0, g_at(0));
  load_words(0, wc[0]);
  __builtin_amdgcn_sched_barrier(0);
  fill(0, st0, gr[0]);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (!SPLIT) {
    load_words(1, wc[1]);
    __builtin_amdgcn_sched_barrier(0);
  }
  fill(1, st1, gr[1]);
  __builtin_amdgcn_sched_barrier(0);
  fill(2, st2, gr[2]);
  __builtin_amdgcn_sched_barrier(0);
  int ks = 0;
  for (; ks + 4 <= n; ks += 4) {
    step(q0, std::false_type{}, ks, st0, st3);
    step(q1, std::false_type{}, ks + 1, st1, st0);
    step(q2, std::false_type{}, ks + 2, st2, st1);
    step(q3, std::false_type{}, ks + 3, st3, st2);
#pragma unroll
    for (int h = 0; h < GPI; ++h)
#pragma unroll
      for (int j = 0; j < NJ; ++j) wc[h][j] = wn[h][j];
  }
  if (ks < n) step(q0, std::true_type{}, ks, st0, st3);
  if (ks + 1 < n) step(q1, std::true_type{}, ks + 1, st1, st0);
  if (ks + 2 < n) step(q2, std::true_type{}, ks + 2, st2, st1);
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

// Stage 1.  grid = row tiles * parts * column tiles.  SPLIT sums the planes
// apart and adds the two sums at the end: half the roundings at the sums' full
// size (4096 -> 4096, ranks 205 + 1843, M = 300: error against 64 bits 3.490e-6
// -> 3.482e-6 of the result's norm; 1,024 rows 3.502e-6 -> 3.477e-6), no slower
// (layer of 700 rows 818 -> 810 us).
template <bool SPLIT, bool GB, int MI>
__global__ __launch_bounds__(kBlock, MI == 4 ? 2 : 4) void sg_latent_kernel(SgParams p) {
  constexpr int NJ = 1;
  constexpr int WPS = SPLIT ? 1 : 2;  // sign words per step
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
  const int n = (min(4 * gb, p.KW) - 4 * ga + WPS - 1) / WPS;
  const uint16_t* src[MI];
  sg_sources<MI>(src, p.a + G.abase + int64_t(ga) * (256 / WPS), p.lda, p.M, m0, tid);
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
  constexpr int NP = SPLIT ? 2 : 1;
  f32x16 acc[NP][MI][NJ];
  uint32_t kone[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    kone[j] = 0x3F803F80u;
    asm volatile("" : "+v"(kone[j]));
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int u = 0; u < NP; ++u) acc[u][i][j] = f32x16{};
  }
  sg_mainloop<SPLIT, GB, MI, NJ, NP>(src, n, ga, words, boundary, kone, acc, tid, GB ? G.g + 128 * ga : nullptr);
  if constexpr (NP == 2) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[0][i][j] += acc[1][i][j];
  }
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
          p.part[(int64_t(tl.part) * p.M + m) * p.tcols + G.tcol + r] = acc[0][i][j][q];
          continue;
        }
        const float v = live ? lv * acc[0][i][j][q] : 0.f;
        if constexpr (SPLIT) {
          uint16_t h, l;
          split1(v, h, l);
          uint16_t* o = p.t + int64_t(m) * p.ldt + 2 * G.tcol + (r >> 5) * 64 + (r & 31);
          o[0] = h;
          o[32] = l;
        } else {
          p.t[int64_t(m) * p.ldt + G.tcol + r] = f32_to_bf16(v);
        }
      }
  }
}

// T from stage 1's parts, summed in part order.  One thread per 4 columns.
template <bool SPLIT>
__global__ __launch_bounds__(kBlock) void sg_reduce_t_kernel(SgParams p) {
  const int cols = p.tcols;
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
  if constexpr (SPLIT) {
    uint16_t* o = p.t + int64_t(m) * p.ldt + 2 * G.tcol + (r >> 5) * 64 + (r & 31);
    *reinterpret_cast<u32x2*>(o) = u32x2{hi[0], hi[1]};
    *reinterpret_cast<u32x2*>(o + 32) = u32x2{lo[0], lo[1]};
  } else {
    *reinterpret_cast<u32x2*>(p.t + int64_t(m) * p.ldt + c) = u32x2{hi[0], hi[1]};
  }
}

// Stage 2.  grid = row tiles * column tiles (p.parts 1).  A projection's
// steps are branch 0's words, padded to whole groups of 4 (the T columns
// there are zero, whatever bits the words hold), then branch 1's: one
// pipeline through both.  Branch 0 is the one of the larger rank: the other's
// few products are the ones rounded at the size of the whole sum (error
// against 64 bits at the shape above 3.482e-6, 3.492e-6 in the other order and
// 3.480e-6 with a call per branch).  One accumulator set: after branch 0 each column's
// S0 is scaled by r = (h0 / h1) 2^-e in fp32 and branch 1 is added with the
// operand +-2^-e (exact in bf16), e = max(0, exponent of h0 / h1): acc = 2^-e
// (h0 S0 + h1 S1) / h1 stays within a factor 2 of the larger term, and y = (h1
// 2^e) acc.  Where h1 is zero, or h0 / h1 past 2^126, branch 1 adds nothing.
template <typename YT, bool SPLIT, int MI, int NJ>
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
  const int nw = P.nb > 1 ? 4 * ng0 + P.RW[1] : P.RW[0];
  const int steps = SPLIT ? nw : (nw + 1) / 2;
  const uint16_t* src[MI];
  sg_sources<MI>(src, p.t + (SPLIT ? 2 : 1) * P.tcol, p.ldt, p.M, m0, tid);
  int col[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) col[j] = min(c0 + 32 * j + lr, P.N - 1);
  auto words = [&](int g, int j) {
    const int gc = min(g, ngr - 1);
    const int b = gc >= ng0 ? 1 : 0, gl = gc - (b ? ng0 : 0);
    const int64_t rw = b ? P.RW[1] : P.RW[0];
    return sg_load_words(b ? P.U[1] : P.U[0], int64_t(col[j]) * rw + 4 * gl, int64_t(P.N) * rw);
  };
  f32x16 acc[1][MI][NJ];
  uint32_t kone[NJ];
  float f[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    kone[j] = 0x3F803F80u;
    asm volatile("" : "+v"(kone[j]));
    f[j] = P.h[0][col[j]];
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[0][i][j] = f32x16{};
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
          for (int i = 0; i < MI; ++i) acc[0][i][j] *= r;
          f[j] = ldexpf(h1, e);
          kone[j] = (0x3F80u - (uint32_t(e) << 7)) * 0x10001u;
        } else {
          kone[j] = 0u;
          if (h1 != h1) f[j] = h1;
        }
      }
    }
  };
  sg_mainloop<SPLIT, false, MI, NJ, 1>(src, steps, 0, words, boundary, kone, acc, tid);
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
        store_out(y, o, f[j] * acc[0][i][j][q] + bn + (res ? res[o] : 0.f));
      }
  }
}
