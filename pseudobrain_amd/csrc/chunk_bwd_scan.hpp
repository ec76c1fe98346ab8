// The two scans of the chunk backward for bfloat16 inputs (included by
// chunk_bwd.hip after chunk_bwd_bf16.hpp, whose operand reads it uses): the
// state at every chunk start, forward, and the adjoint at every chunk end,
// reverse (the notation is chunk_bwd.hip's).
//
// A workgroup takes 16 NW value columns of one (role, sequence, value head):
// NW waves compute, each 16 columns with the whole chain of a chunk in its
// registers (an accumulator tile is the next product's B operand as it
// stands, see chunk_bwd_bf16.hpp), so a step has no exchange between waves and
// one barrier. Four more waves load: they hold the next two chunks' rows in
// registers and write each to the LDS buffer that the step before has left.
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
// chunk and head, written once and read once). At 1 x 32,768 tokens of 32 heads
// 1.59 (four barriers a step, 16 columns a workgroup) -> 1.34 ms, the chain of a
// step and its traffic 1.1 ms each by themselves; at 4 x 2,048 437 -> 233 us.

// ---------------------------------------------------------------------------
// Per (chunk, value head): T = (I + A)^-1 and M^T as bf16 pairs, c, beta.
// Wave w holds token rows 16 w .. of q as operands (no LDS), so four
// workgroups share a CU. 0.70 (with dU0 and J) -> 0.25 ms at 1 x 32,768 tokens
// of 32 heads, 0.6 GB written; the inverse's serial rows are what it waits for.
// ---------------------------------------------------------------------------
template <int K>
constexpr size_t local_bf16_lds() {
  return sizeof(u16) * BC * K + sizeof(float) * (BC * LC + 2 * BC + 3 * 256);
}

template <int K>
__global__ __launch_bounds__(BNT) void bwd_local_bf16_kernel(BwdParams p) {
  extern __shared__ __align__(16) float lds[];
  PBGDN_POISON_LDS(lds, local_bf16_lds<K>());
  PBGDN_POISON_SYNC();
  u16 *sk = reinterpret_cast<u16 *>(lds);
  float *sa = reinterpret_cast<float *>(sk + BC * K), *sc = sa + BC * LC, *sbeta = sc + BC, *sr = sbeta + BC;
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
    RowsAhead<K, BNT> rk;
    rk.load(tid, static_cast<const u16 *>(p.k) + ((seq.bos + t0) * p.Hk + hk) * K, p.Hk * K, seq.len - t0);
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
    rk.put(tid, sk, seq.len - t0);
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
        const bh8_t kr = ln.rows16<K>(sk, 16 * tc, kb);
        kk = mfma_bf16(ln.rows16<K>(sk, 16 * wave, kb), kr, kk);
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
  static constexpr int LOADERS = 256, NT = 64 * NW + LOADERS;
  static constexpr int COLS = 16 * NW, PAIR = 2 * BC * BC;
  // one buffer: K rows, the T pair, the V or dO columns, four vectors (e^c,
  // e^(c_last - c), beta; the adjoint's scale e^c, e^(c_last - c), -beta e^c;
  // e^c_last last); the adjoint's also Q rows and the M^T pair
  static constexpr int OFF_T = BC * K, OFF_X = OFF_T + PAIR, OFF_VEC = OFF_X + BC * COLS;
  static constexpr int OFF_Q = OFF_VEC + 2 * 4 * BC, OFF_M = OFF_Q + BC * K, BUF = OFF_M + PAIR;
  static constexpr size_t BYTES = 2 * sizeof(u16) * BUF;
  static_assert(OFF_VEC % 8 == 0 && OFF_Q % 8 == 0 && BUF % 8 == 0, "16-byte pieces");
};

// One chunk's inputs in the registers of the loading waves (thread tid of
// LOADERS). Rows past the sequence's end are clamped into it by the loads and
// zeroed by the stores.
template <int K, int NW, bool ADJ>
struct ScanLoad {
  using L = Scan16<K, NW>;
  static constexpr int N = L::LOADERS, KP = BC * K / 8 / N, TP = 768 / N, XP = BC * 2 * NW / N;
  uint4 k[KP], t[TP], x[XP], q[ADJ ? KP : 1], m[ADJ ? TP : 1];
  float cv, bv, last;
  int left;  // tokens from the chunk's first to the sequence's end

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

  // Uniform bases and 32-bit lane offsets (a chunk's rows of all heads are
  // under 2^31 bytes: 64 rows, at most 65,535 heads of 128 elements).
  __device__ __forceinline__ void load(const BwdParams &p, const BwdSeq &seq, int h, int hk, int i, int v0, int tid) {
    const int t0 = i * BC;
    left = seq.len - t0;
    const int top = min(left, BC) - 1;
    const long r = rec(p, seq, h, i), row0 = seq.bos + t0;
    const u16 *kb = static_cast<const u16 *>(p.k) + (row0 * p.Hk + hk) * K;
    const u16 *qb = static_cast<const u16 *>(p.q) + (row0 * p.Hk + hk) * K;
    const u16 *xb = static_cast<const u16 *>(ADJ ? p.dout : p.v) + (row0 * p.Hv + h) * p.V + v0;
    const uint4 *wt = reinterpret_cast<const uint4 *>(p.ws_T + r * BC * BC);
    const uint4 *wm = reinterpret_cast<const uint4 *>(p.ws_M + r * BC * BC);
    const uint32_t kstride = p.Hk * K, xstride = p.Hv * p.V;
#pragma unroll
    for (int a = 0; a < KP; ++a) {
      const int e = tid + N * a;
      const uint32_t off = min(e / (K / 8), top) * kstride + (e % (K / 8)) * 8;
      k[a] = *reinterpret_cast<const uint4 *>(kb + off);
      if constexpr (ADJ) q[a] = *reinterpret_cast<const uint4 *>(qb + off);
    }
#pragma unroll
    for (int a = 0; a < TP; ++a) {
      int half, row, part;
      tri(tid + N * a, false, half, row, part);
      t[a] = wt[static_cast<uint32_t>(half * 512 + row * 8 + part)];
      if constexpr (ADJ) {
        tri(tid + N * a, true, half, row, part);
        m[a] = wm[static_cast<uint32_t>(half * 512 + row * 8 + part)];
      }
    }
#pragma unroll
    for (int a = 0; a < XP; ++a) {
      const int e = tid + N * a;
      const uint32_t off = min(e / (2 * NW), top) * xstride + (e % (2 * NW)) * 8;
      x[a] = *reinterpret_cast<const uint4 *>(xb + off);
    }
    cv = p.ws_c[r * BC + (tid & 63)];
    bv = p.ws_beta[r * BC + (tid & 63)];
    last = p.ws_c[r * BC + BC - 1];
  }

  __device__ __forceinline__ void store(u16 *buf, int tid, float scale) {
    if (left < BC) {
      const uint4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int a = 0; a < KP; ++a) {
        if ((tid + N * a) / (K / 8) < left) continue;
        k[a] = zero;
        if constexpr (ADJ) q[a] = zero;
      }
#pragma unroll
      for (int a = 0; a < XP; ++a) {
        if ((tid + N * a) / (2 * NW) >= left) x[a] = zero;
      }
    }
#pragma unroll
    for (int a = 0; a < KP; ++a) {
      const int e = tid + N * a, row = e / (K / 8), part = e % (K / 8);
      *reinterpret_cast<uint4 *>(buf + unit_at<K>(row, part)) = k[a];
      if constexpr (ADJ) *reinterpret_cast<uint4 *>(buf + L::OFF_Q + unit_at<K>(row, part)) = q[a];
    }
#pragma unroll
    for (int a = 0; a < TP; ++a) {
      int half, row, part;
      tri(tid + N * a, false, half, row, part);
      *reinterpret_cast<uint4 *>(buf + L::OFF_T + unit_at<BC>(half * BC + row, part)) = t[a];
      if constexpr (ADJ) {
        tri(tid + N * a, true, half, row, part);
        *reinterpret_cast<uint4 *>(buf + L::OFF_M + unit_at<BC>(half * BC + row, part)) = m[a];
      }
    }
#pragma unroll
    for (int a = 0; a < XP; ++a) {
      const int e = tid + N * a, row = e / (2 * NW), part = e % (2 * NW);
      *reinterpret_cast<uint4 *>(buf + L::OFF_X + unit_at<L::COLS>(row, part)) = x[a];
    }
    if (tid < BC) {
      float *vec = reinterpret_cast<float *>(buf + L::OFF_VEC);
      const float gam = expf(cv);
      vec[tid] = ADJ ? scale * gam : gam;
      vec[BC + tid] = expf(last - cv);
      vec[2 * BC + tid] = ADJ ? -gam * bv : bv;
      if (tid == BC - 1) vec[4 * BC - 1] = gam;
    }
  }
};

// A step's order is written out: the LDS reads of a product are issued before
// the products (and the splits) that precede it, which hide their latency. The
// compiler left to itself reads each fragment just before its use (some sixty
// exposed waits a step: 1,681 us of scans at 1 x 32,768 tokens of 32 heads).
// Key tiles' operands of the contraction over tokens 32 kb ..
template <int KT>
__device__ __forceinline__ void read_cols(const Lane &ln, const u16 *m, int kb, bh8_t (&a)[KT]) {
#pragma unroll
  for (int t = 0; t < KT; ++t) a[t] = ln.cols<16 * KT>(m, kb, 16 * t);
}

// s += the operands times a pair.
template <int KT>
__device__ __forceinline__ void add_products(float4_t (&s)[KT], const bh8_t (&a)[KT], bh8_t bh, bh8_t bl) {
#pragma unroll
  for (int t = 0; t < KT; ++t) s[t] = mfma_bf16(a[t], bh, s[t]);
#pragma unroll
  for (int t = 0; t < KT; ++t) s[t] = mfma_bf16(a[t], bl, s[t]);
}

// Chunk i's step on a wave's 16 columns: s is the state (or adjoint) before it
// and after it.
template <int K, int NW, bool ADJ>
__device__ __forceinline__ void scan16_step(const u16 *buf, const Lane &ln, int col, float4_t (&s)[K / 16]) {
  using L = Scan16<K, NW>;
  constexpr int KT = K / 16, KB = K / 32, W = L::COLS, CC = BC * BC;
  const u16 *sk = buf, *tp = buf + L::OFF_T, *sx = buf + L::OFF_X;
  const float *vec = reinterpret_cast<const float *>(buf + L::OFF_VEC) + 4 * ln.g;
  // ---- K S
  bh8_t ka[KB][4];
#pragma unroll
  for (int kb = 0; kb < KB / 2; ++kb) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) ka[kb][rt] = ln.rows<K>(sk, 16 * rt, kb);
  }
  keep_order();
  v2u32_t sh[KT], sl[KT];
#pragma unroll
  for (int m = 0; m < KT; ++m) split_bf16(s[m], sh[m], sl[m]);
  keep_order();
#pragma unroll
  for (int kb = KB / 2; kb < KB; ++kb) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) ka[kb][rt] = ln.rows<K>(sk, 16 * rt, kb);
  }
  keep_order();
  float4_t y[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) y[rt] = zero4();
  auto ks = [&](int kb) {
    const bh8_t bh = frag_pair(sh[2 * kb], sh[2 * kb + 1]), bl = frag_pair(sl[2 * kb], sl[2 * kb + 1]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) y[rt] = mfma_bf16(ka[kb][rt], bh, y[rt]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) y[rt] = mfma_bf16(ka[kb][rt], bl, y[rt]);
  };
#pragma unroll
  for (int kb = 0; kb < KB / 2; ++kb) ks(kb);
  keep_order();
  // T's operands (the triangle): fragment (rt, kb) of U's rows or dX's columns
  bh8_t th[4][2], tl[4][2];
  auto used = [](int rt, int kb) { return ADJ ? kb >= (rt >> 1) : kb <= (rt >> 1); };
  auto read_t = [&] {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        if (!used(rt, kb)) continue;
        th[rt][kb] = ADJ ? ln.cols<BC>(tp, kb, 16 * rt) : ln.rows<BC>(tp, 16 * rt, kb);
        tl[rt][kb] = ADJ ? ln.cols<BC>(tp + CC, kb, 16 * rt) : ln.rows<BC>(tp + CC, 16 * rt, kb);
      }
    }
  };
  v2u32_t xh[4], xl[4];  // beta X, or dU
  v2u32_t oh[4], ol[4];  // scale Gamma dO
  bw_i16x4_t xr[4];      // V's or dO's rows
  float4_t w0[4], w1[4];
  if constexpr (!ADJ) {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      xr[rt] = ln.tr<W>(sx, 16 * rt, col);
      w0[rt] = ld4(vec + 16 * rt);           // e^c
      w1[rt] = ld4(vec + 2 * BC + 16 * rt);  // beta
    }
    read_t();
    keep_order();
#pragma unroll
    for (int kb = KB / 2; kb < KB; ++kb) ks(kb);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      split_bf16((bf16x4_float(xr[rt]) - w0[rt] * y[rt]) * w1[rt], xh[rt], xl[rt]);
    }
  } else {
    const u16 *mt = buf + L::OFF_M;
    bh8_t mh[4][2], ml[4][2], dof[2];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) w0[rt] = ld4(vec + BC + 16 * rt);  // e^(c_last - c)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) xr[rt] = ln.tr<W>(sx, 16 * rt, col);
#pragma unroll
    for (int kb = 1; kb >= 0; --kb) {
#pragma unroll
      for (int rt = 0; rt < 2 * kb + 2; ++rt) {  // t >= s
        mh[rt][kb] = ln.rows<BC>(mt, 16 * rt, kb);
        ml[rt][kb] = ln.rows<BC>(mt + CC, 16 * rt, kb);
      }
    }
    keep_order();
#pragma unroll
    for (int kb = KB / 2; kb < KB; ++kb) ks(kb);
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      dof[kb] = frag_pair(__builtin_bit_cast(v2u32_t, xr[2 * kb]), __builtin_bit_cast(v2u32_t, xr[2 * kb + 1]));
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) y[rt] *= w0[rt];
    keep_order();
    read_t();
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) w1[rt] = ld4(vec + 16 * rt);  // scale e^c
    keep_order();
#pragma unroll
    for (int kb = 1; kb >= 0; --kb) {
#pragma unroll
      for (int rt = 0; rt < 2 * kb + 2; ++rt) y[rt] = mfma_bf16(mh[rt][kb], dof[kb], y[rt]);
#pragma unroll
      for (int rt = 0; rt < 2 * kb + 2; ++rt) y[rt] = mfma_bf16(ml[rt][kb], dof[kb], y[rt]);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) split_bf16(bf16x4_float(xr[rt]) * w1[rt], oh[rt], ol[rt]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) split_bf16(y[rt], xh[rt], xl[rt]);
  }
  keep_order();
  // ---- U = T (beta X), s <= t; or dX / beta = T^T dU, t >= s
  bh8_t a0[KT], a1[KT];
  read_cols(ln, ADJ ? buf + L::OFF_Q : sk, 0, a0);
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) w0[rt] = ld4(vec + (ADJ ? 2 : 1) * BC + 16 * rt);  // -beta e^c, or e^(c_last - c)
  const float gam_c = vec[4 * BC - 1 - 4 * ln.g];
  keep_order();
  float4_t z[4];
#pragma unroll
  for (int rt = 0; rt < 4; ++rt) z[rt] = zero4();
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    const bh8_t bh = frag_pair(xh[2 * kb], xh[2 * kb + 1]), bl = frag_pair(xl[2 * kb], xl[2 * kb + 1]);
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      if (used(rt, kb)) z[rt] = mfma_bf16(th[rt][kb], bh, z[rt]);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      if (used(rt, kb)) z[rt] = mfma_bf16(th[rt][kb], bl, z[rt]);
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      if (used(rt, kb)) z[rt] = mfma_bf16(tl[rt][kb], bh, z[rt]);
    }
  }
#pragma unroll
  for (int m = 0; m < KT; ++m) s[m] *= gam_c;
  keep_order();
  read_cols(ln, ADJ ? buf + L::OFF_Q : sk, 1, a1);
  keep_order();
  v2u32_t zh[4], zl[4];  // E U, or -Gamma dX
  if constexpr (ADJ) {  // Q's products fill the splits' place in the chain
    add_products(s, a0, frag_pair(oh[0], oh[1]), frag_pair(ol[0], ol[1]));
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) split_bf16(z[rt] * w0[rt], zh[rt], zl[rt]);
    keep_order();
    read_cols(ln, sk, 0, a0);
    keep_order();
    add_products(s, a1, frag_pair(oh[2], oh[3]), frag_pair(ol[2], ol[3]));
    keep_order();
    read_cols(ln, sk, 1, a1);
    keep_order();
  } else {
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) split_bf16(z[rt] * w0[rt], zh[rt], zl[rt]);
  }
  add_products(s, a0, frag_pair(zh[0], zh[1]), frag_pair(zl[0], zl[1]));
  add_products(s, a1, frag_pair(zh[2], zh[3]), frag_pair(zl[2], zl[3]));
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
    // Two chunks in flight: a step's loads have two steps to arrive (one step
    // was too short: the fill of 68 KiB came after the loads' latency, 3.3 us
    // a step).
    ScanLoad<K, NW, ADJ> even, odd;
    auto load = [&](ScanLoad<K, NW, ADJ> &in, int j) { in.load(p, seq, h, hk, chunk(min(j, seq.n - 1)), v0, tid); };
    u16 *buf1 = lds + L::BUF;
    if (seq.n > 0) {
      load(even, 0);
      load(odd, 1);
      even.store(lds, tid, p.scale);
      load(even, 2);
    }
    for (int j = 0; j < seq.n; j += 2) {
      __syncthreads();  // step j's buffer is written, step j - 1's is free
      odd.store(buf1, tid, p.scale);
      load(odd, j + 3);
      if (j + 1 == seq.n) break;
      __syncthreads();
      even.store(lds, tid, p.scale);
      load(even, j + 4);
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
    scan16_step<K, NW, ADJ>(lds + (j & 1) * L::BUF, ln, 16 * wave, s);
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
__global__ __launch_bounds__(64 * NW + 256) __attribute__((amdgpu_waves_per_eu(2, 2)))
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
