// Attention of N new tokens at positions start .. start+N-1 over the cache and
// themselves, causal or with a tree mask (a new token sees every cached position
// and the new tokens its mask row marks, itself included when the row says so),
// fp32 throughout on v_mfma_f32_32x32x2_f32.  The reference runs its batch
// forward token by token (patches/littlebit_cpu_optimized.cpp:1846-2079) and its
// tree verification through the model's attention with the tree mask
// (tree_utils.py:72-214).  Included by littlebit_amd.hip inside its anonymous
// namespace.
//
// A block takes 32 query rows of one kv head (rows = token-major (token, head
// of the group) pairs, so a tile's rows see nearly the same positions and the
// heads of a group share the keys and values) and a chunk of the positions in
// tiles of 32; its 4 waves take the chunk's tiles w, w + 4, ..: every wave has the
// same work whatever the causal range, and the longest blocks are dispatched
// first.  The waves' (o, max, sum) meet in LDS at the end: the output itself
// (prompts, one chunk), or one partial per (head, chunk, token) for
// attn_batch_combine_kernel (BATCH).
//
// Per tile a wave forms S^T = K Q^T and O^T += V^T P^T: S^T's C layout (lane
// = query, registers = positions 8 a + 4 half + b) is the B operand of the
// second product register by register, so P never moves between lanes, and
// a query's max, sum and rescale are per-lane scalars (its two half-lanes
// meet in one swap).  K tiles go straight to the wave's own LDS (16-byte chunk
// c of row r at chunk c ^ r: no bank conflicts), issued as soon as the tile
// before has been read, so they arrive under the second product; V rows go
// to registers, issued before the first product, which covers them.  No
// barrier in the loop.
//
// Prompts are bound by the fp32 MFMAs (a large fp32 library product reaches 154
// TFLOP/s on this card), short ones by the last blocks of a grid that fills the
// chip about twice: 1,024 tokens of 32 heads x 128 in 108 us (80 TFLOP/s),
// after 3,000 cached positions 488 us (121), 2,048 tokens of 32 query / 8 kv
// heads 300 us (115).  The products, mask, softmax and copies as library
// calls over the [heads, n, positions] scores took about 480 us for the
// first.  Batches wait for loads and for the tiles a wave has in turn (each 2 x
// 64 MFMAs, about 3.5 us): 33 tokens of 32 heads x 128 after 1,000 positions
// 25.6 us (attn_batch_kernel 27.0), of 8 kv heads 21.3 (26.9); 64 tokens after
// 2,000 40.1 (57.8); figures on both sides of the line at attn_rows_chunks.
struct AttnRowsParams {
  const float* q;  // [N][heads * HD], unscaled
  const float* k;  // [N][kv_heads * HD] new keys
  const float* v;  // [N][kv_heads * HD] new values
  float* kc;       // [kv_heads][max_seq][HD]
  float* vc;
  const uint8_t* tree;       // BATCH: [N][N], row i marks the new tokens token i sees; null: causal
  float* part;               // BATCH: [heads][chunks][N][HD + 2], o, max, sum
  float* out;                // [N][heads * HD]
  const int64_t* start_ptr;  // start read on the device when set (graph replay), else `start`
  int64_t start;
  int N, heads, kvh, rep, max_seq, ntile, chunks;
  float scale;
};

// NS is the number of sums over the dims that make a score.  1: one chunk,
// causal, two blocks per CU.  More (BATCH): a tree mask, chunks and a device
// start may be given; the grid is a block per CU, so registers are free, and
// each tile's weighted values have sums of their own too.  At 1,000 positions
// the rounding error falls from 4.1e-7 of the result's norm to 2.3e-7 (NS 4);
// with 8 sums it is 2.1e-7 for 1 us more.
template <int HD, int NS>
__global__ __launch_bounds__(256, NS > 1 ? 1 : 2) void attn_rows_kernel(AttnRowsParams p) {
  constexpr bool BATCH = NS > 1;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  typedef __attribute__((address_space(1))) void* glb_ptr_t;
  constexpr int NC = HD / 32;  // 32-dim tiles of O^T; lane rows hold dims NC * row ..
  constexpr int CH = HD / 4;   // 16-byte chunks per row
  typedef float vecf __attribute__((ext_vector_type(NC)));
  __shared__ __attribute__((aligned(16))) float kt[4][32 * HD];
  __shared__ float sm[4][32], sl[4][32];
  const int tid = int(threadIdx.x), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const int g = int(blockIdx.x) % p.kvh;  // heads spread over the XCDs, a head's blocks on one
  const int chunk = BATCH ? int(blockIdx.x) / p.kvh % p.chunks : 0;
  const int tile = p.ntile - 1 - int(blockIdx.x) / p.kvh / (BATCH ? p.chunks : 1);
  const int64_t start64 = BATCH && p.start_ptr ? *p.start_ptr : p.start;
  if (start64 < 0 || start64 + p.N > p.max_seq) return;  // nothing read or stored (the combine writes zeros)
  const int start = int(start64);
  // this block's share of the new keys and values goes to the cache; new
  // positions are read from k and v, so nobody waits for it
  if (chunk == 0) {
    const int t0 = int(int64_t(tile) * p.N / p.ntile), t1 = int(int64_t(tile + 1) * p.N / p.ntile);
    for (int e = tid; e < (t1 - t0) * CH; e += 256) {
      const int tok = t0 + e / CH, c = 4 * (e % CH);
      const int64_t src = (int64_t(tok) * p.kvh + g) * HD + c;
      const int64_t dst = (int64_t(g) * p.max_seq + start + tok) * HD + c;
      *reinterpret_cast<float4*>(p.kc + dst) = *reinterpret_cast<const float4*>(p.k + src);
      *reinterpret_cast<float4*>(p.vc + dst) = *reinterpret_cast<const float4*>(p.v + src);
    }
  }
  const int rows = p.N * p.rep, row0 = tile * 32;
  const int row = min(row0 + lr, rows - 1);
  const int tok = row / p.rep;             // the lane's query; it sees positions <= start + tok
  const int first = start + row0 / p.rep;  // the tile's first query's last
  // tiles of the cache (the last may be partial), then of the new positions:
  // no tile reads from both
  const int seen = BATCH && p.tree ? p.N : min(row0 + 31, rows - 1) / p.rep + 1;  // new positions the tile's queries see
  const int Tc = (start + 31) >> 5;
  const int Ta = Tc + ((seen + 31) >> 5);
  // the chunk: an even share of the positions there are (the grid may be sized for a later start)
  const int tpc = BATCH ? 4 * ((((Tc + ((p.N + 31) >> 5) + 3) >> 2) + p.chunks - 1) / p.chunks) : 0;
  const int T = BATCH ? min(Ta, (chunk + 1) * tpc) : Ta, ta = chunk * tpc + wave;
  const float qs = p.scale * 1.44269504088896340736f;  // log2(e): the weights are powers of two
  f32x4 qf[HD / 8];
  {
    const float* qp = p.q + (int64_t(tok) * p.heads + g * p.rep + row % p.rep) * HD + 4 * lh;
#pragma unroll
    for (int i = 0; i < HD / 8; ++i) qf[i] = qs * *reinterpret_cast<const f32x4*>(qp + 8 * i);
  }
  float* const mine = kt[wave];
  // Rows of tile t: n valid rows from a uniform base; each load is a uniform
  // row address plus the lane's own offset.  A partial tile repeats its last row.
  struct Rows {
    const float *k, *v;
    int stride, n, pos;
  };
  auto rows_of = [&](int t) {
    Rows x;
    if (t < Tc) {
      const int64_t at = (int64_t(g) * p.max_seq + 32 * t) * HD;
      x.k = p.kc + at;
      x.v = p.vc + at;
      x.stride = HD;
      x.pos = 32 * t;
      x.n = min(32, start - 32 * t);
    } else {
      const int r = 32 * (t - Tc);
      const int64_t at = (int64_t(r) * p.kvh + g) * HD;
      x.k = p.k + at;
      x.v = p.v + at;
      x.stride = p.kvh * HD;
      x.pos = start + r;
      x.n = min(32, seen - r);
    }
    return x;
  };
  constexpr int RPI = 64 / CH;  // rows per DMA instruction
  // The lane's offsets are formed where they are used (the empty asm keeps
  // them from being hoisted: 16 registers each, which spill).
  const int fr = lane / CH, fc = lane % CH;
  auto fill = [&](const Rows& x) {
    uint32_t c0 = uint32_t(fc ^ fr) * 16u;  // chunk (RPI j + fr) ^ fc: RPI j has no bit of fr
    asm volatile("" : "+v"(c0));
    const char* base = reinterpret_cast<const char*>(x.k);
    if (x.n == 32) {
      const uint32_t row = uint32_t(fr * x.stride) * 4u;
#pragma unroll
      for (int j = 0; j < CH / 2; ++j)
        __builtin_amdgcn_global_load_lds(
            (glb_ptr_t)(base + int64_t(RPI * j) * x.stride * 4 + (row + (c0 ^ (uint32_t((RPI * j) & (CH - 1)) * 16u)))),
            (lds_ptr_t)(mine + 256 * j), 16, 0, 0);
    } else {
      int f = fr;
      asm volatile("" : "+v"(f));
#pragma unroll
      for (int j = 0; j < CH / 2; ++j)
        __builtin_amdgcn_global_load_lds(
            (glb_ptr_t)(base + (uint32_t(min(RPI * j + f, x.n - 1) * x.stride) * 4u +
                                (c0 ^ (uint32_t((RPI * j) & (CH - 1)) * 16u)))),
            (lds_ptr_t)(mine + 256 * j), 16, 0, 0);
    }
  };
  f32x16 o[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) o[c] = f32x16{};
  float m = -INFINITY, l = 0.f;
  Rows x = rows_of(ta);
  if (ta < T) fill(x);
  for (int t = ta; t < T; t += 4) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));  // the K tile has landed
    asm volatile("" ::: "memory");
    vecf vv[16];
    const char* vbase = reinterpret_cast<const char*>(x.v);
    if (x.n == 32) {
      const uint32_t off = uint32_t(4 * lh * x.stride + NC * lr) * 4u;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        vv[i] = *reinterpret_cast<const vecf*>(vbase + int64_t(8 * (i >> 2) + (i & 3)) * x.stride * 4 + off);
    } else {
      int h4 = 4 * lh;
      asm volatile("" : "+v"(h4));
#pragma unroll
      for (int i = 0; i < 16; ++i)
        vv[i] = *reinterpret_cast<const vecf*>(
            vbase + uint32_t(min(8 * (i >> 2) + h4 + (i & 3), x.n - 1) * x.stride + NC * lr) * 4u);
    }
    __builtin_amdgcn_sched_barrier(0);
    f32x16 sc[NS];
#pragma unroll
    for (int u = 0; u < NS; ++u) sc[u] = f32x16{};
    uint32_t k0 = uint32_t(lr * HD + (((lh ^ lr) & (CH - 1)) << 2)) * 4u;  // chunk (2 i + lh) ^ lr of row lr
    asm volatile("" : "+v"(k0));
    auto kread = [&](int i) {
      return *reinterpret_cast<const f32x4*>(reinterpret_cast<const char*>(mine) + (k0 ^ uint32_t(32 * i)));
    };
    f32x4 kf = kread(0);
#pragma unroll
    for (int i = 0; i < HD / 8; ++i) {
      const f32x4 kn = kread(i + 1 < HD / 8 ? i + 1 : i);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sc[i % NS] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[e], qf[i][e], sc[i % NS], 0, 0, 0);
      kf = kn;
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(63));  // every read of the tile is done
    asm volatile("" ::: "memory");
    const int pos0 = x.pos, n = x.n;
    // on every path, so that the wait for V counts these loads as newer (after
    // the last tile the same tile again, unused)
    x = rows_of(t + 4 < T ? t + 4 : t);
    fill(x);
#pragma unroll
    for (int d = NS / 2; d > 0; d /= 2)
#pragma unroll
      for (int u = 0; u < d; ++u) sc[u] += sc[u + d];
    f32x16& s = sc[0];
    float mx = -INFINITY;
    if (BATCH && p.tree && pos0 >= start) {
      const uint8_t* tr = p.tree + int64_t(tok) * p.N + (pos0 - start);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int r = 8 * (i >> 2) + 4 * lh + (i & 3);
        if (r >= n || tr[min(r, n - 1)] == 0) s[i] = -INFINITY;
      }
    } else if (n < 32 || pos0 + 31 > first) {  // a tile that some query does not see whole
      int last = min(n - 1, start + tok - pos0) - 4 * lh;  // the lane's query sees its rows up to here
      asm volatile("" : "+v"(last));
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (8 * (i >> 2) + (i & 3) > last) s[i] = -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
    mx = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32)));
    const float base = mx == -INFINITY ? 0.f : mx;  // nothing seen so far: every weight is 0
    const float corr = __builtin_amdgcn_exp2f(m - base);
    m = mx;
    float sum[4] = {};
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      s[i] = __builtin_amdgcn_exp2f(s[i] - base);
      sum[i & 3] += s[i];
    }
    l = l * corr + ((sum[0] + sum[1]) + (sum[2] + sum[3]));
    if constexpr (BATCH) {
      f32x16 a[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) a[c] = f32x16{};
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) a[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[i][c], s[i], a[c], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < NC; ++c) o[c] = o[c] * corr + a[c];
    } else {
      if (__any(corr != 1.f)) {
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c] *= corr;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) o[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[i][c], s[i], o[c], 0, 0, 0);
    }
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));
  asm volatile("" ::: "memory");
  // O^T of the wave into its tile's LDS as [query][dims], vector r of a row at r ^ query
  l += __shfl_xor(l, 32);
  if (lh == 0) {
    sm[wave][lr] = m;
    sl[wave][lr] = l;
  }
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    vecf x;
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c] = o[c][q];
    const int r = 8 * (q >> 2) + 4 * lh + (q & 3);
    *reinterpret_cast<vecf*>(mine + lr * HD + NC * (r ^ lr)) = x;
  }
  __syncthreads();
  const int qr = tid >> 3;
  if (row0 + qr >= rows) return;
  float M = fmaxf(fmaxf(sm[0][qr], sm[1][qr]), fmaxf(sm[2][qr], sm[3][qr]));
  float w[4], L = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    w[i] = sm[i][qr] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sm[i][qr] - M);
    L += w[i] * sl[i][qr];
  }
  const int qtok = (row0 + qr) / p.rep, head = g * p.rep + (row0 + qr) % p.rep;
  typedef vecf __attribute__((aligned(4))) vecu;
  float* op = BATCH ? p.part + ((int64_t(head) * p.chunks + chunk) * p.N + qtok) * (HD + 2)
                     : p.out + (int64_t(qtok) * p.heads + head) * HD;
  const float inv = BATCH ? 1.f : 1.f / L;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int r = 4 * (tid & 7) + u;
    vecf x = {};
#pragma unroll
    for (int i = 0; i < 4; ++i) x += w[i] * *reinterpret_cast<const vecf*>(kt[i] + qr * HD + NC * (r ^ qr));
    *reinterpret_cast<vecu*>(op + NC * r) = x * inv;
  }
  if (BATCH && (tid & 7) == 0) {
    op[HD] = M * 0.69314718055994530942f;  // natural exponents in the partials
    op[HD + 1] = L;
  }
}
