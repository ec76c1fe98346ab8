// The two scans of the chunk backward for bfloat16 inputs (included by
// chunk_bwd.hip after chunk_bwd_bf16.hpp, whose operand reads it uses): the
// state at every chunk start, forward, and the adjoint at every chunk end,
// reverse (the notation is chunk_bwd.hip's).
//
// A workgroup takes 16 NW value columns of one (role, sequence, value head):
// NW waves compute, each 16 columns with the whole chain of a chunk in its
// registers (an accumulator tile is the next product's B operand as it
// stands, see chunk_bwd_bf16.hpp), so a step has no exchange between waves and
// one barrier. NW more waves load: they hold the next chunk's rows in
// registers, write them to the LDS buffer that the step before has left, and
// start on the chunk after.
//
//   state    X = V - Gamma K S,  U = T beta X,  S <- gamma_C S + K^T E U
//   adjoint  dU = M^T dO + E K dS',  dX = beta T^T dU,
//            dS <- gamma_C dS' + (scale Gamma Q)^T dO - (Gamma K)^T dX
//
// What bounds it: the states themselves, 2 x 64 KiB a chunk and value head at
// K = V = 128 written in float32 for the gradient kernel, then the fill of LDS
// from L2 (about 25 bytes a clock and CU). So the reverse scan takes M^T (64 x
// 64, as a bf16 pair), Q and dO and forms the two products with dO itself:
// they were records of the local kernel's (dU0 and J, 96 KiB in float32 a
// chunk and head, written once and read once).

// ---------------------------------------------------------------------------
// Per (chunk, value head): T = (I + A)^-1 and M^T as bf16 pairs, c, beta.
// Wave w holds token rows 16 w .. of q as operands (no LDS), so four
// workgroups share a CU; the inverse's serial rows are what it waits for.
// ---------------------------------------------------------------------------
template <int K>
constexpr size_t local_bf16_lds() {
  return sizeof(u16) * BC * (K + 8) + sizeof(float) * (BC * LC + 2 * BC + 3 * 256);
}

template <int K>
__global__ __launch_bounds__(BNT) void bwd_local_bf16_kernel(BwdParams p) {
  constexpr int LK = K + 8;
  extern __shared__ __align__(16) float lds[];
  PBGDN_POISON_LDS(lds, local_bf16_lds<K>());
  PBGDN_POISON_SYNC();
  u16 *sk = reinterpret_cast<u16 *>(lds);
  float *sa = reinterpret_cast<float *>(sk + BC * LK), *sc = sa + BC * LC, *sbeta = sc + BC, *sr = sbeta + BC;
  u16 *mh = reinterpret_cast<u16 *>(sa);  // M^T, a pair of rows of LC, in sa's bytes once T is out
  const int h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const Lane ln{lane & 15, lane >> 4};
  const int hk = h / (p.Hv / p.Hk);
  if (p.cu_seqlens) zero_uncovered<u16>(p, blockIdx.x, h);
  BwdSeq seq;
  int i;
  if (!chunk_of(p, blockIdx.x, blockIdx.z, seq, i)) return;
  const int t0 = i * BC;
  const long r = rec(p, seq, h, i);
  bh8_t qf[K / 32];
  {
    RawRows<u16, K> rk;
    rk.load(p.k, seq, t0, p.Hk, hk, K);
    const int t = t0 + 16 * wave + ln.c;
    const u16 *row = static_cast<const u16 *>(p.q) + ((seq.bos + min(t, seq.len - 1)) * p.Hk + hk) * K + 8 * ln.g;
#pragma unroll
    for (int kb = 0; kb < K / 32; ++kb) qf[kb] = *reinterpret_cast<const bh8_t *>(row + 32 * kb);
    if (wave == 0) {  // inclusive cumulative sum of g over the chunk (zero past T)
      const int tt = t0 + lane;
      float x = tt < seq.len ? p.g[(seq.bos + tt) * p.Hv + h] : 0.f;
      const float bt = tt < seq.len ? load_elem(p.beta, (seq.bos + tt) * p.Hv + h, p.beta_dtype) : 0.f;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
      }
      sc[lane] = x;
      sbeta[lane] = bt;
      p.ws_c[r * BC + lane] = x;
      p.ws_beta[r * BC + lane] = bt;
    }
    rk.put(sk, LK);
  }
  __syncthreads();
  // A = strict_lower(beta_t (K K^T) o D), rows 16w .. of this wave; M^T's
  // columns 16w .. : M^T[s][t] = scale (k_s . q_t) e^(c_t - c_s), t >= s, and
  // 0 for the tokens past the sequence
  float4_t mt[4];
  {
    const int t = 16 * wave + ln.c;
    const bool in = t0 + t < seq.len;
#pragma unroll
    for (int tc = 0; tc < 4; ++tc) {
      float4_t kk = zero4(), kq = zero4();
#pragma unroll
      for (int kb = 0; kb < K / 32; ++kb) {
        const bh8_t kr = ln.rows16(sk, LK, 16 * tc, kb);
        kk = mfma_bf16(ln.rows16(sk, LK, 16 * wave, kb), kr, kk);
        kq = mfma_bf16(kr, qf[kb], kq);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int ta = 16 * wave + 4 * ln.g + e, sa2 = 16 * tc + ln.c;
        sa[ta * LC + sa2] = ta > sa2 ? sbeta[ta] * kk[e] * expf(sc[ta] - sc[sa2]) : 0.f;
        const int s2 = 16 * tc + 4 * ln.g + e;
        mt[tc][e] = in && t >= s2 ? p.scale * kq[e] * expf(sc[t] - sc[s2]) : 0.f;
      }
    }
  }
  __syncthreads();
  invert_unit_lower(sa, sr);
  auto out = [&](float *ws, int half, int piece) -> uint4 & {
    return reinterpret_cast<uint4 *>(ws + r * BC * BC)[half * 512 + piece];
  };
#pragma unroll
  for (int m = 0; m < 2; ++m) {  // T
    const int e = tid + BNT * m;
    const float *x = &sa[(e >> 3) * LC + 8 * (e & 7)];
    v2u32_t h0, l0, h1, l1;
    split_bf16(ld4(x), h0, l0);
    split_bf16(ld4(x + 4), h1, l1);
    out(p.ws_T, 0, e) = uint4{h0[0], h0[1], h1[0], h1[1]};
    out(p.ws_T, 1, e) = uint4{l0[0], l0[1], l1[0], l1[1]};
  }
  __syncthreads();
#pragma unroll
  for (int tc = 0; tc < 4; ++tc) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      put_pair1(mh, BC * LC, (16 * tc + 4 * ln.g + e) * LC + 16 * wave + ln.c, mt[tc][e]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 4; ++m) {  // M^T
    const int half = m >> 1, e = tid + BNT * (m & 1);
    const u16 *x = mh + (half * BC + (e >> 3)) * LC + 8 * (e & 7);
    const v2u32_t a = *reinterpret_cast<const v2u32_t *>(x), b = *reinterpret_cast<const v2u32_t *>(x + 4);
    out(p.ws_M, half, e) = uint4{a[0], a[1], b[0], b[1]};
  }
}

// ---------------------------------------------------------------------------
// The scans.
// ---------------------------------------------------------------------------
template <int K, int NW>
struct Scan16 {
  static constexpr int NT = 128 * NW, LOADERS = 64 * NW;
  static constexpr int LK = K + 8, LB = BC + 8, LC16 = 16 * NW + 8;  // row strides (elements)
  static constexpr int PAIR = 2 * BC * LB;
  // one buffer: K rows, the T pair, the V or dO columns, the vectors e^c,
  // e^(c_last - c), beta; the adjoint's also Q rows and the M^T pair
  static constexpr int OFF_T = BC * LK, OFF_X = OFF_T + PAIR, OFF_VEC = OFF_X + BC * LC16;
  static constexpr int OFF_Q = OFF_VEC + 2 * 4 * BC, OFF_M = OFF_Q + BC * LK, BUF = OFF_M + PAIR;
  static constexpr size_t BYTES = 2 * sizeof(u16) * BUF;
  static_assert(OFF_VEC % 8 == 0 && OFF_Q % 8 == 0 && BUF % 8 == 0, "16-byte pieces");
};

// One chunk's inputs in the registers of the loading waves (thread tid of
// 64 NW). Rows past the sequence's end are clamped into it and zeroed.
template <int K, int NW, bool ADJ>
struct ScanLoad {
  using L = Scan16<K, NW>;
  static constexpr int N = L::LOADERS, KP = BC * K / 8 / N, TP = 768 / N, XP = BC * 2 * NW / N;
  uint4 k[KP], t[TP], x[XP], q[ADJ ? KP : 1], m[ADJ ? TP : 1];
  float cv, bv, last;

  // Piece e of a triangular pair: [half][row][8 pieces], without the quadrant
  // that holds zeros only (T: rows < 32 of columns >= 32; M^T: the other one).
  __device__ static __forceinline__ void tri(int e, bool upper, int &half, int &row, int &part) {
    half = e >= 384;
    const int f = half ? e - 384 : e;
    if (f < 128) {
      row = (f >> 2) + (upper ? 32 : 0);
      part = (f & 3) + (upper ? 4 : 0);
    } else {
      row = ((f - 128) >> 3) + (upper ? 0 : 32);
      part = f & 7;
    }
  }

  __device__ __forceinline__ void load(const BwdParams &p, const BwdSeq &seq, int h, int hk, int i, int v0, int tid) {
    const int t0 = i * BC;
    const long r = rec(p, seq, h, i);
    const uint4 *wt = reinterpret_cast<const uint4 *>(p.ws_T + r * BC * BC);
    const uint4 *wm = reinterpret_cast<const uint4 *>(p.ws_M + r * BC * BC);
    const u16 *src = static_cast<const u16 *>(ADJ ? p.dout : p.v);
    auto row_of = [&](int row) { return seq.bos + min(t0 + row, seq.len - 1); };
#pragma unroll
    for (int a = 0; a < KP; ++a) {
      const int e = tid + N * a, row = e / (K / 8), part = e % (K / 8);
      const long off = (row_of(row) * p.Hk + hk) * K + part * 8;
      const bool in = t0 + row < seq.len;
      const uint4 y = *reinterpret_cast<const uint4 *>(static_cast<const u16 *>(p.k) + off);
      k[a] = in ? y : uint4{0u, 0u, 0u, 0u};
      if constexpr (ADJ) {
        const uint4 z = *reinterpret_cast<const uint4 *>(static_cast<const u16 *>(p.q) + off);
        q[a] = in ? z : uint4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int a = 0; a < TP; ++a) {
      int half, row, part;
      tri(tid + N * a, false, half, row, part);
      t[a] = wt[half * 512 + row * 8 + part];
      if constexpr (ADJ) {
        tri(tid + N * a, true, half, row, part);
        m[a] = wm[half * 512 + row * 8 + part];
      }
    }
#pragma unroll
    for (int a = 0; a < XP; ++a) {
      const int e = tid + N * a, row = e / (2 * NW), part = e % (2 * NW);
      const uint4 y = *reinterpret_cast<const uint4 *>(src + (row_of(row) * p.Hv + h) * p.V + v0 + part * 8);
      x[a] = t0 + row < seq.len ? y : uint4{0u, 0u, 0u, 0u};
    }
    cv = p.ws_c[r * BC + (tid & 63)];
    bv = p.ws_beta[r * BC + (tid & 63)];
    last = p.ws_c[r * BC + BC - 1];
  }

  __device__ __forceinline__ void store(u16 *buf, int tid) const {
#pragma unroll
    for (int a = 0; a < KP; ++a) {
      const int e = tid + N * a, row = e / (K / 8), part = e % (K / 8);
      *reinterpret_cast<uint4 *>(buf + row * L::LK + part * 8) = k[a];
      if constexpr (ADJ) *reinterpret_cast<uint4 *>(buf + L::OFF_Q + row * L::LK + part * 8) = q[a];
    }
#pragma unroll
    for (int a = 0; a < TP; ++a) {
      int half, row, part;
      tri(tid + N * a, false, half, row, part);
      *reinterpret_cast<uint4 *>(buf + L::OFF_T + (half * BC + row) * L::LB + part * 8) = t[a];
      if constexpr (ADJ) {
        tri(tid + N * a, true, half, row, part);
        *reinterpret_cast<uint4 *>(buf + L::OFF_M + (half * BC + row) * L::LB + part * 8) = m[a];
      }
    }
#pragma unroll
    for (int a = 0; a < XP; ++a) {
      const int e = tid + N * a, row = e / (2 * NW), part = e % (2 * NW);
      *reinterpret_cast<uint4 *>(buf + L::OFF_X + row * L::LC16 + part * 8) = x[a];
    }
    if (tid < BC) {
      float *vec = reinterpret_cast<float *>(buf + L::OFF_VEC);
      vec[tid] = expf(cv);
      vec[BC + tid] = expf(last - cv);
      vec[2 * BC + tid] = bv;
    }
  }
};

// Chunk i's step on a wave's 16 columns: s is the state (or adjoint) before it
// and after it.
template <int K, int NW, bool ADJ>
__device__ __forceinline__ void scan16_step(const BwdParams &p, const u16 *buf, const Lane &ln, int col,
                                            float4_t (&s)[K / 16]) {
  using L = Scan16<K, NW>;
  constexpr int KT = K / 16, KB = K / 32, LK = L::LK, LB = L::LB, CC = BC * LB;
  const u16 *sk = buf, *tp = buf + L::OFF_T, *sx = buf + L::OFF_X;
  const float *sgam = reinterpret_cast<const float *>(buf + L::OFF_VEC), *se = sgam + BC, *sbeta = se + BC;
  v2u32_t sh[KT], sl[KT];
#pragma unroll
  for (int m = 0; m < KT; ++m) split_bf16(s[m], sh[m], sl[m]);
  float4_t y[4];  // K S
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) y[rt] = zero4();
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const bh8_t bh = frag_pair(sh[2 * kb], sh[2 * kb + 1]), bl = frag_pair(sl[2 * kb], sl[2 * kb + 1]);
    bh8_t a[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) a[rt] = ln.rows(sk, LK, 16 * rt, kb);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) y[rt] = mfma_bf16(a[rt], bh, y[rt]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) y[rt] = mfma_bf16(a[rt], bl, y[rt]);
  }
  v2u32_t xh[4], xl[4];  // beta X, or dU
  v2u32_t oh[4], ol[4];  // scale Gamma dO
  if constexpr (!ADJ) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      const int o = 16 * rt + 4 * ln.g;
      const float4_t x = bf16x4_float(ln.tr(sx + 16 * rt * L::LC16, L::LC16, col)) - ld4(&sgam[o]) * y[rt];
      split_bf16(x * ld4(&sbeta[o]), xh[rt], xl[rt]);
    }
  } else {
    const u16 *mt = buf + L::OFF_M;
    bh8_t dof[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) dof[kb] = ln.cols(sx, L::LC16, kb, col);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) y[rt] *= ld4(&se[16 * rt + 4 * ln.g]);
#pragma unroll
    for (int kb = 1; kb >= 0; --kb) {  // t >= s
#pragma unroll
      for (int rt = 0; rt < 2 * kb + 2; ++rt) y[rt] = mfma_bf16(ln.rows(mt, LB, 16 * rt, kb), dof[kb], y[rt]);
#pragma unroll
      for (int rt = 0; rt < 2 * kb + 2; ++rt) y[rt] = mfma_bf16(ln.rows(mt + CC, LB, 16 * rt, kb), dof[kb], y[rt]);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      split_bf16(y[rt], xh[rt], xl[rt]);
      const float4_t d = bf16x4_float(ln.tr(sx + 16 * rt * L::LC16, L::LC16, col));
      split_bf16(d * (ld4(&sgam[16 * rt + 4 * ln.g]) * p.scale), oh[rt], ol[rt]);
    }
  }
  // U = T (beta X), s <= t; or dX / beta = T^T dU, t >= s
  float4_t z[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) z[rt] = zero4();
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const bh8_t bh = frag_pair(xh[2 * kb], xh[2 * kb + 1]), bl = frag_pair(xl[2 * kb], xl[2 * kb + 1]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      if (ADJ ? kb < (rt >> 1) : kb > (rt >> 1)) continue;
      const bh8_t th = ADJ ? ln.cols(tp, LB, kb, 16 * rt) : ln.rows(tp, LB, 16 * rt, kb);
      const bh8_t tl = ADJ ? ln.cols(tp + CC, LB, kb, 16 * rt) : ln.rows(tp + CC, LB, 16 * rt, kb);
      z[rt] = mfma_bf16(th, bh, z[rt]);
      z[rt] = mfma_bf16(th, bl, z[rt]);
      z[rt] = mfma_bf16(tl, bh, z[rt]);
    }
  }
  const float gam_c = sgam[BC - 1];
  v2u32_t zh[4], zl[4];  // E U, or -Gamma dX
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) {
    const int o = 16 * rt + 4 * ln.g;
    split_bf16(ADJ ? z[rt] * (-(ld4(&sgam[o]) * ld4(&sbeta[o]))) : z[rt] * ld4(&se[o]), zh[rt], zl[rt]);
  }
#pragma unroll
  for (int m = 0; m < KT; ++m) s[m] *= gam_c;
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const bh8_t bh = frag_pair(zh[2 * kb], zh[2 * kb + 1]), bl = frag_pair(zl[2 * kb], zl[2 * kb + 1]);
#pragma unroll
    for (int m0 = 0; m0 < KT; m0 += 4) {
      bh8_t a[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = ln.cols(sk, LK, kb, 16 * (m0 + m));
#pragma unroll
      for (int m = 0; m < 4; ++m) s[m0 + m] = mfma_bf16(a[m], bh, s[m0 + m]);
#pragma unroll
      for (int m = 0; m < 4; ++m) s[m0 + m] = mfma_bf16(a[m], bl, s[m0 + m]);
    }
    if constexpr (ADJ) {
      const u16 *sq = buf + L::OFF_Q;
      const bh8_t ch = frag_pair(oh[2 * kb], oh[2 * kb + 1]), cl = frag_pair(ol[2 * kb], ol[2 * kb + 1]);
#pragma unroll
      for (int m0 = 0; m0 < KT; m0 += 4) {
        bh8_t a[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) a[m] = ln.cols(sq, LK, kb, 16 * (m0 + m));
#pragma unroll
        for (int m = 0; m < 4; ++m) s[m0 + m] = mfma_bf16(a[m], ch, s[m0 + m]);
#pragma unroll
        for (int m = 0; m < 4; ++m) s[m0 + m] = mfma_bf16(a[m], cl, s[m0 + m]);
      }
    }
  }
}

template <int K, int NW, bool ADJ>
__device__ __forceinline__ void scan16_pass(const BwdParams &p, u16 *lds, int n, int h, int v0) {
  using L = Scan16<K, NW>;
  constexpr int KT = K / 16;
  const BwdSeq seq = seq_of(p, n);
  const int hk = h / (p.Hv / p.Hk);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  auto chunk = [&](int j) { return ADJ ? seq.n - 1 - j : j; };  // the chunk of step j
  if (wave >= NW) {
    const int tid = threadIdx.x - 64 * NW;
    ScanLoad<K, NW, ADJ> in;
    if (seq.n > 0) {
      in.load(p, seq, h, hk, chunk(0), v0, tid);
      in.store(lds, tid);
      if (seq.n > 1) in.load(p, seq, h, hk, chunk(1), v0, tid);
    }
    for (int j = 0; j < seq.n; ++j) {
      __syncthreads();  // step j's buffer is written, step j - 1's is free
      if (j + 1 < seq.n) in.store(lds + ((j + 1) & 1) * L::BUF, tid);
      if (j + 2 < seq.n) in.load(p, seq, h, hk, chunk(j + 2), v0, tid);
    }
    return;
  }
  const int lane = threadIdx.x & 63;
  const Lane ln{lane & 15, lane >> 4};
  const int v = v0 + 16 * wave;
  const long kv = (static_cast<long>(n) * p.Hv + h) * K * p.V + v + ln.c;
  const float *start = ADJ ? p.dht : p.h0;
  float4_t s[KT];
#pragma unroll
  for (int m = 0; m < KT; ++m) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[m][e] = start ? start[kv + static_cast<long>(16 * m + 4 * ln.g + e) * p.V] : 0.f;
  }
  for (int j = 0; j < seq.n; ++j) {
    float4_t *ws = reinterpret_cast<float4_t *>((ADJ ? p.ws_dS : p.ws_S) + rec(p, seq, h, chunk(j)) * K * p.V) +
                   (v >> 4) * KT * 64 + lane;
#pragma unroll
    for (int m = 0; m < KT; ++m) ws[64 * m] = s[m];
    __syncthreads();
    scan16_step<K, NW, ADJ>(p, lds + (j & 1) * L::BUF, ln, 16 * wave, s);
  }
  if (ADJ && p.dh0) {
#pragma unroll
    for (int m = 0; m < KT; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) p.dh0[kv + static_cast<long>(16 * m + 4 * ln.g + e) * p.V] = s[m][e];
    }
  }
}

// Both roles in one launch, the adjoint (the longer step) first. The column
// groups and value heads of a key head read the same K and Q rows: one XCD.
template <int K, int NW>
__global__ __launch_bounds__(128 * NW) __attribute__((amdgpu_waves_per_eu(NW / 2, NW / 2)))
void bwd_scans_bf16_kernel(BwdParams p) {
  extern __shared__ __align__(16) float lds[];
  PBGDN_POISON_LDS(lds, (Scan16<K, NW>::BYTES));
  PBGDN_POISON_SYNC();
  const int cols = p.V / (16 * NW), group = p.Hv / p.Hk, keys = p.num_seqs * p.Hk;
  int key, member;
  xcd_group(blockIdx.x, 2 * keys, group * cols, p.xcds, key, member);
  const bool adjoint = key < keys;
  if (!adjoint) key -= keys;
  const int n = key / p.Hk, h = (key % p.Hk) * group + member / cols, v0 = (member % cols) * 16 * NW;
  u16 *buf = reinterpret_cast<u16 *>(lds);
  if (adjoint) {
    scan16_pass<K, NW, true>(p, buf, n, h, v0);
  } else {
    scan16_pass<K, NW, false>(p, buf, n, h, v0);
  }
}
