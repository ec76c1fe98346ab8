// The gradient kernel of the chunk backward for bfloat16 inputs (included by
// chunk_bwd.hip, whose notation and helpers it uses).
//
// A workgroup of V / 16 waves takes items (chunk, key head) in turn, and of
// each the value heads of the key head, so dq and dk are summed over them in
// registers. For each value head:
//
//   chain    wave w holds the 16 value columns 16 w .. of the start state S
//            and the end adjoint dS' in registers and forms its columns of
//            X = V - Gamma K S, U = T beta X, dU = M^T dO + E K dS' and
//            dX = beta T^T dU with no barrier: an accumulator tile is the B
//            operand of the next product as it stands, once the contraction
//            slots of the A operand are numbered to match (below).
//   stages   the contractions over the value columns need every wave's
//            columns: X, dU, then U, dX and the states pass through LDS as
//            transposed bf16 high / low halves, one pair at a time, and the
//            waves share out the output tiles:
//            dTb = dU X^T, dM = dO U^T (64 x 64), dK1 = U dS'^T,
//            dK2 = dX S^T, dQ0 = dO S^T (64 x K).
//   C x C    the gradient through M, T and A, and the sums for dg and dbeta.
//
// The decay sums sum_v (K dS' o U)_t and sum_v (K S o dX)_t are formed in the
// chain, where all four are in float32: as sums over the keys of K o dK1 and K o
// dK2, whose products take U and dX as bf16 pairs, they left dg with 1.2 times
// its error against 64 bits (geometric mean of 22 calls; up to 1.9), and the
// kernel 1% slower. sum_v (Q S o dO)_t does come from the keys
// (sum_k (Q o dQ0)_t): dO is exact in bf16 there.
// LDS: 135 KiB at K = V = 128, so one workgroup a CU, eight waves.
//
// 3.55 (16-column tiles in turn, with the reduction) -> 1.57 ms at 1 x 32,768
// tokens of 32 heads, 0.47 ms at 4 x 2,048 (kernel trace). A head takes about
// 60,000 cycles (the medians of 32 heads): inputs into LDS 1,700, chain 9,200,
// stages 19,200 (ten barriers), row scales 1,600, C x C matrices and sums 9,500,
// last products and the issue of the next head's loads 9,500 (6,200 to 19,400),
// dg and, after the last head, the output 6,000 (2,000 to 17,700). LDS is
// active in 36% of the CU's busy cycles, a quarter of it bank conflicts.
//
// Contraction slots: the B operand of a 32-row step kb made of two
// accumulator tiles holds, in lane (c, g), rows 32 kb + 4 g + j (j < 4) and
// 32 kb + 16 + 4 g + j - 4 of column c; A operands are read in that order (two
// 8-byte pieces of a row, or two transposing reads).

// LDS arrays are row-major without padding, W elements a row, the 16-byte units
// of row r swizzled: unit u stands at u ^ unit_swz<W>(r). 32 lanes of a
// transposing read take 32 bytes of 8 rows, 32 lanes of a row read 16 bytes of
// 16 rows, and either way the 16 units differ modulo 256 bytes. (With rows
// padded by 16 bytes the transposing reads conflicted two ways, with 32 the row
// reads.) Conflicts fell from 46% to 25% of the gradient kernel's LDS cycles and
// from 42% to 32% of the scans' (4 x 2,048 tokens); what is left was not taken
// apart (row reads that the compiler pairs, and the writes, are not covered).
template <int W>
__device__ __forceinline__ constexpr int unit_swz(int r) {
  static_assert(W == 128 || W == 64 || W == 32, "row widths");
  return W == 128 ? 2 * (r & 7) + ((r >> 3) & 1)
         : W == 64 ? 2 * ((r >> 1) & 3) + ((r >> 3) & 1)
                   : 2 * ((r >> 2) & 1);  // (transposing reads only)
}
// Offset of 16-byte unit u of row r.
template <int W>
__device__ __forceinline__ constexpr int unit_at(int r, int u) {
  return r * W + 8 * (u ^ unit_swz<W>(r));
}

// The operand reads of one lane (c, g); row0, col0 multiples of 16, kb steps of
// 32. A struct rather than functions of threadIdx.x, so that a kernel can make
// its lane opaque to the compiler where addresses and comparisons must not be
// kept across a loop.
struct Lane {
  int c, g;

  // Element (row0 + c, col0 + 4 g): four of a row, 8 bytes.
  template <int W>
  __device__ __forceinline__ int four(int row0, int col0) const {
    return row0 * W + ((unit_at<W>(c, g >> 1) + 4 * (g & 1)) ^ col0);
  }
  // Four rows row0 + 4 g .. of column col0 + c (ds_read_tr16).
  template <int W>
  __device__ __forceinline__ bw_i16x4_t tr(const u16 *m, int row0, int col0) const {
    const int at = (unit_at<W>(4 * g + (c >> 2), (c >> 1) & 1) + 4 * (c & 1)) ^ col0;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) bw_i16x4_t *)(m + row0 * W + at));
  }
  // Rows row0 + c as the operand of step kb.
  template <int W>
  __device__ __forceinline__ bh8_t rows(const u16 *m, int row0, int kb) const {
    const v2u32_t x = *reinterpret_cast<const v2u32_t *>(m + four<W>(row0, 32 * kb));
    const v2u32_t y = *reinterpret_cast<const v2u32_t *>(m + four<W>(row0, 32 * kb + 16));
    return __builtin_bit_cast(bh8_t, v4u32_t{x[0], x[1], y[0], y[1]});
  }
  // The same with the slots in order (both operands read this way).
  template <int W>
  __device__ __forceinline__ bh8_t rows16(const u16 *m, int row0, int kb) const {
    return *reinterpret_cast<const bh8_t *>(m + row0 * W + (unit_at<W>(c, g) ^ (32 * kb)));
  }
  // Columns col0 + c, contraction over the array's rows 32 kb ..
  template <int W>
  __device__ __forceinline__ bh8_t cols(const u16 *m, int kb, int col0) const {
    const bw_i16x4_t x = tr<W>(m, 32 * kb, col0), y = tr<W>(m, 32 * kb + 16, col0);
    return __builtin_bit_cast(bh8_t, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
  }
  // Rows a0 .. of a times rows b0 .. of b, over KD columns.
  template <int KD>
  __device__ __forceinline__ float4_t rows_rows(const u16 *a, const u16 *b, int a0, int b0) const {
    float4_t acc = zero4();
#pragma unroll
    for (int kb = 0; kb < KD / 32; ++kb) acc = mfma_bf16(rows16<KD>(a, a0, kb), rows16<KD>(b, b0, kb), acc);
    return acc;
  }
};

__device__ __forceinline__ bh8_t frag_pair(v2u32_t x, v2u32_t y) {
  return __builtin_bit_cast(bh8_t, v4u32_t{x[0], x[1], y[0], y[1]});
}

// Four bf16 (a transposing read's result) as float.
__device__ __forceinline__ float4_t bf16x4_float(bw_i16x4_t x) {
  const v2u32_t w = __builtin_bit_cast(v2u32_t, x);
  return float4_t{__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16),
                  __uint_as_float(w[1] & 0xffff0000u)};
}

// No instruction crosses this point: bounds how far the compiler moves reads.
__device__ __forceinline__ void keep_order() { __builtin_amdgcn_sched_barrier(0); }

template <int K, int V>
struct GradLds {
  static constexpr int NW = V / 16, NT = 64 * NW, COLS = NW / 2;  // waves; wave pairs
  static constexpr int CC = BC * BC;                              // one 64 x 64 half
  static constexpr int TV = V * BC;                               // one V x 64 half
  // the shared area: M^T pair and V rows (chain); X^T and dU^T pairs; the U^T
  // or dX^T pair and one state half; four C x C pairs
  static constexpr int USED = 4 * TV > 2 * TV + V * K ? 4 * TV : 2 * TV + V * K,
                       AREA = USED > 8 * CC ? USED : 8 * CC;
  static_assert(2 * CC + BC * V <= AREA && 2 * TV + V * K <= AREA, "the area's uses");
  static constexpr int FLOATS = 4 * BC + 3 * COLS * BC + NW * BC + 4 * BC + 16;
  static constexpr size_t BYTES = sizeof(u16) * (2 * BC * K + BC * V + 2 * CC + AREA) + sizeof(float) * FLOATS;
};

// Rows 0 .. 63 from a uniform base (the chunk's first row) in registers, to be
// put into LDS later: rows past `left` are clamped into the sequence by the
// loads and zeroed by the put, so nothing waits for the loads before that.
template <int W, int NT>
struct RowsAhead {
  static constexpr int PPR = W / 8, PER = BC * PPR / NT;
  v4u32_t raw[PER];

  __device__ __forceinline__ void load(int tid, const u16 *base, uint32_t stride, int left) {
    const int top = min(left, BC) - 1;
#pragma unroll
    for (int m = 0; m < PER; ++m) {
      const int e = tid + NT * m;
      const uint32_t off = static_cast<uint32_t>(min(e / PPR, top)) * stride + (e % PPR) * 8;
      raw[m] = *reinterpret_cast<const v4u32_t *>(base + off);
    }
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int m = 0; m < PER; ++m) raw[m] = v4u32_t{0u, 0u, 0u, 0u};
  }
  __device__ __forceinline__ void put(int tid, u16 *dst, int left) {
    if (left < BC) {
#pragma unroll
      for (int m = 0; m < PER; ++m) {
        if ((tid + NT * m) / PPR >= left) raw[m] = v4u32_t{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int m = 0; m < PER; ++m) {
      const int e = tid + NT * m;
      *reinterpret_cast<v4u32_t *>(dst + unit_at<W>(e / PPR, e % PPR)) = raw[m];
    }
  }
};

// Four elements of an output row; one by one (narrow) where the outputs are not
// 8-byte aligned.
__device__ __forceinline__ void store_four(u16 *at, v2u32_t x, bool narrow) {
  if (!narrow) {
    *reinterpret_cast<v2u32_t *>(at) = x;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) at[e] = static_cast<u16>(x[e >> 1] >> (16 * (e & 1)));
}

// A gradient workgroup's place in its items (chunk, group of value heads).
struct GradItem {
  BwdSeq seq;
  int i, block;   // the chunk; the value heads block * heads ..
  unsigned item;  // the item's index
};
// The first item at or after `item` (in steps of `step`) that holds a chunk.
__device__ __forceinline__ bool grad_item(const BwdParams &p, unsigned item, unsigned step, unsigned items,
                                          unsigned chunks, unsigned blocks, GradItem &it) {
  for (; item < items; item += step) {
    const unsigned rest = item / chunks;
    if (!chunk_of(p, item % chunks, rest / blocks, it.seq, it.i)) continue;
    it.block = rest % blocks;
    it.item = item;
    return true;
  }
  return false;
}

template <int K, int V>
__global__ __launch_bounds__(4 * V) void bwd_grad_bf16_kernel(BwdParams p, int heads) {
  using L = GradLds<K, V>;
  constexpr int NW = L::NW, NT = L::NT, COLS = L::COLS, CC = L::CC, TV = L::TV;
  constexpr int KT = K / 16, KB = K / 32, VB = V / 32;
  constexpr int KTW = KT / COLS, CTW = 4 / COLS;  // key tiles, C x C column tiles of a wave
  extern __shared__ __align__(16) float lds[];
  PBGDN_POISON_LDS(lds, L::BYTES);
  PBGDN_POISON_SYNC();
  const int group = p.Hv / p.Hk;
  const unsigned chunks = p.cu_seqlens ? p.records : p.n, blocks = p.Hv / heads, items = chunks * blocks * p.B;
  GradItem it, next;
  if (!grad_item(p, blockIdx.x, gridDim.x, items, chunks, blocks, it)) return;
  // A head's inputs, in registers from the stages of the head before: a CU
  // holds one workgroup, so loads issued at a head's start were waited for in
  // full (16,000 to 60,000 cycles of a head's 60,000 to 100,000).
  float4_t sf[KT], df[KT];
  v4u32_t rt[BC * BC / 4 / NT], rm[BC * BC / 4 / NT];  // the T and M^T pairs: 1,024 pieces of 16 bytes each
  RowsAhead<V, NT> rv, rd;
  RowsAhead<K, NT> rq, rk;
  float cv, bv, last;
  auto load_adjoint = [&](const GradItem &at, int h, int tid) {
    const float4_t *wd = reinterpret_cast<const float4_t *>(p.ws_dS + rec(p, at.seq, h, at.i) * K * V) +
                         __builtin_amdgcn_readfirstlane(tid >> 6) * KT * 64;
#pragma unroll
    for (int m = 0; m < KT; ++m) df[m] = wd[static_cast<uint32_t>(64 * m + (tid & 63))];
  };
  auto load_state = [&](const GradItem &at, int h, int tid) {
    const float4_t *ws = reinterpret_cast<const float4_t *>(p.ws_S + rec(p, at.seq, h, at.i) * K * V) +
                         __builtin_amdgcn_readfirstlane(tid >> 6) * KT * 64;
#pragma unroll
    for (int m = 0; m < KT; ++m) sf[m] = ws[static_cast<uint32_t>(64 * m + (tid & 63))];
  };
  auto load_rest = [&](const GradItem &at, int h, bool keys, int tid) {
    const long r = rec(p, at.seq, h, at.i), row0 = at.seq.bos + at.i * BC;
    const int left = at.seq.len - at.i * BC;
    const v4u32_t *wt = reinterpret_cast<const v4u32_t *>(p.ws_T + r * BC * BC);
    const v4u32_t *wm = reinterpret_cast<const v4u32_t *>(p.ws_M + r * BC * BC);
#pragma unroll
    for (int m = 0; m < BC * BC / 4 / NT; ++m) rt[m] = wt[static_cast<uint32_t>(tid + NT * m)];
#pragma unroll
    for (int m = 0; m < BC * BC / 4 / NT; ++m) rm[m] = wm[static_cast<uint32_t>(tid + NT * m)];
    rv.load(tid, static_cast<const u16 *>(p.v) + (row0 * p.Hv + h) * V, p.Hv * V, left);
    rd.load(tid, static_cast<const u16 *>(p.dout) + (row0 * p.Hv + h) * V, p.Hv * V, left);
    if (keys) {
      rq.load(tid, static_cast<const u16 *>(p.q) + (row0 * p.Hk + h / group) * K, p.Hk * K, left);
      rk.load(tid, static_cast<const u16 *>(p.k) + (row0 * p.Hk + h / group) * K, p.Hk * K, left);
    } else {  // (a value on every path: see the call)
      rq.clear();
      rk.clear();
    }
    cv = p.ws_c[r * BC + (tid & 63)];
    bv = p.ws_beta[r * BC + (tid & 63)];
    last = p.ws_c[r * BC + BC - 1];
  };
  load_adjoint(it, it.block * heads, threadIdx.x);
  load_state(it, it.block * heads, threadIdx.x);
  load_rest(it, it.block * heads, true, threadIdx.x);
  float4_t tq[KTW][2], tk[KTW][2];
#pragma unroll
  for (int m = 0; m < KTW; ++m) {
#pragma unroll
    for (int a = 0; a < 2; ++a) tq[m][a] = tk[m][a] = zero4();
  }
  int hh = 0;  // the value head of the item's group
  bool more = true;
  for (bool first = true; more; first = false) {
    // The LDS base and the thread index are made opaque for each head: the
    // compiler otherwise keeps every phase's addresses and comparisons in
    // registers across the loop (212 spilled registers a lane).
    int base = 0, tid = threadIdx.x;
    asm volatile("" : "+s"(base), "+v"(tid));
    const int lane = tid & 63, c = lane & 15, g4 = lane >> 4;
    Lane L4{c, g4};
    // makes the operand addresses of the phase before unknown to the compiler,
    // which would keep them in registers for the next
    auto renew = [&] { asm volatile("" : "+v"(L4.c), "+v"(L4.g)); };
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), v0 = 16 * wave;
    const int rp = wave & 1, cp = wave >> 1;  // row tiles 2 rp, 2 rp + 1; column (key) tiles of pair cp
    u16 *sq = reinterpret_cast<u16 *>(lds + base), *sk = sq + BC * K, *sdo = sk + BC * K, *tp = sdo + BC * V,
        *area = tp + 2 * CC;
    float *sc = reinterpret_cast<float *>(area + L::AREA), *sgam = sc + BC, *se = sgam + BC, *sbeta = se + BC;
    // partial sums: rows by wave pair (dc, dbeta, dgamma's part of Q S) and by
    // wave (the chain's decay sums), columns by wave parity
    float *prc = sbeta + BC, *prb = prc + COLS * BC, *pdg = prb + COLS * BC, *pch = pdg + COLS * BC;
    float *pcc = pch + NW * BC, *pcb = pcc + 2 * BC, *sred = pcb + 2 * BC;
    const int h = it.block * heads + hh, t0 = it.i * BC, left = it.seq.len - t0;  // the chunk's tokens: left, if under BC
    const long row0 = it.seq.bos + t0;
    // ---- this head's inputs into LDS
    u16 *mt = area, *sv = area + 2 * CC;
    if (!first) __syncthreads();  // the previous head's readers of LDS are done
    if (hh == 0) {
      rq.put(tid, sq, left);
      rk.put(tid, sk, left);
    }
    rd.put(tid, sdo, left);
    rv.put(tid, sv, left);
#pragma unroll
    for (int m = 0; m < BC * BC / 4 / NT; ++m) {
      const int e = tid + NT * m;  // half e / 512, row (e / 8) & 63
      *reinterpret_cast<v4u32_t *>(tp + unit_at<BC>(e >> 3, e & 7)) = rt[m];
      *reinterpret_cast<v4u32_t *>(mt + unit_at<BC>(e >> 3, e & 7)) = rm[m];
    }
    if (tid < BC) {
      sc[tid] = cv;
      sgam[tid] = expf(cv);
      se[tid] = expf(last - cv);
      sbeta[tid] = bv;
    }
    __syncthreads();
    // ---- chain: this wave's 16 value columns
    float dgc = 0.f;
    v2u32_t sh[KT], sl[KT], dh[KT], dl[KT];
#pragma unroll
    for (int m = 0; m < KT; ++m) {
#pragma unroll
      for (int e = 0; e < 4; ++e) dgc += sf[m][e] * df[m][e];
      split_bf16(sf[m], sh[m], sl[m]);
      split_bf16(df[m], dh[m], dl[m]);
    }
    keep_order();
    float4_t x[4], du[4], ekd[4];  // X; E K dS' + M^T dO, and E K dS' alone
    v2u32_t bxh[4], bxl[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      float4_t ks = zero4(), kd = zero4();
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const bh8_t a = L4.rows<K>(sk, 16 * rt, kb);
        ks = mfma_bf16(a, frag_pair(sh[2 * kb], sh[2 * kb + 1]), ks);
        kd = mfma_bf16(a, frag_pair(dh[2 * kb], dh[2 * kb + 1]), kd);
        ks = mfma_bf16(a, frag_pair(sl[2 * kb], sl[2 * kb + 1]), ks);
        kd = mfma_bf16(a, frag_pair(dl[2 * kb], dl[2 * kb + 1]), kd);
      }
      const int o = 16 * rt + 4 * g4;
      x[rt] = bf16x4_float(L4.tr<V>(sv, 16 * rt, v0)) - ld4(&sgam[o]) * ks;
      split_bf16(x[rt] * ld4(&sbeta[o]), bxh[rt], bxl[rt]);
      du[rt] = ekd[rt] = ld4(&se[o]) * kd;
      keep_order();
    }
    // The chain's decay sums, over this wave's columns: to d/dc of token t
    // -(E K dS' o U + Gamma K S o dX), with V - X for Gamma K S (no registers for
    // it); to that of the last one gamma_C S . dS' and all of E K dS' o U.
    dgc *= sgam[BC - 1];
    float4_t dch = zero4();  // element rt: token 16 rt + 4 g + (c & 3), over the columns of four lanes
    auto add_rows = [&](float4_t y, int rt) {  // four sums over four lanes, one left in each
      const bool odd = c & 1, upper = c & 2;
      const float y01 = (odd ? y[1] : y[0]) + dpp_mov<0xb1>(odd ? y[0] : y[1]);
      const float y23 = (odd ? y[3] : y[2]) + dpp_mov<0xb1>(odd ? y[2] : y[3]);
      dch[rt] += (upper ? y23 : y01) + dpp_mov<0x4e>(upper ? y01 : y23);
    };
    v2u32_t duh[4], dul[4];
    {
      bh8_t dof[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) dof[kb] = L4.cols<V>(sdo, kb, v0);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
#pragma unroll
        for (int kb = rt >> 1; kb < 2; ++kb) {  // t >= s
          du[rt] = mfma_bf16(L4.rows<BC>(mt, 16 * rt, kb), dof[kb], du[rt]);
          du[rt] = mfma_bf16(L4.rows<BC>(mt + CC, 16 * rt, kb), dof[kb], du[rt]);
        }
        split_bf16(du[rt], duh[rt], dul[rt]);
      }
    }
    v2u32_t xh[4], xl[4], dxh[4], dxl[4], uh[4], ul[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
      float4_t dx = zero4(), u = zero4();
#pragma unroll
      for (int kb = 0; kb <= rt >> 1; ++kb) {  // U = T (beta X), s <= t
        const bh8_t th = L4.rows<BC>(tp, 16 * rt, kb), tl = L4.rows<BC>(tp + CC, 16 * rt, kb);
        const bh8_t bh = frag_pair(bxh[2 * kb], bxh[2 * kb + 1]), bl = frag_pair(bxl[2 * kb], bxl[2 * kb + 1]);
        u = mfma_bf16(th, bh, u);
        u = mfma_bf16(th, bl, u);
        u = mfma_bf16(tl, bh, u);
      }
#pragma unroll
      for (int kb = rt >> 1; kb < 2; ++kb) {  // dX = beta T^T dU, t >= s
        const bh8_t th = L4.cols<BC>(tp, kb, 16 * rt), tl = L4.cols<BC>(tp + CC, kb, 16 * rt);
        const bh8_t bh = frag_pair(duh[2 * kb], duh[2 * kb + 1]), bl = frag_pair(dul[2 * kb], dul[2 * kb + 1]);
        dx = mfma_bf16(th, bh, dx);
        dx = mfma_bf16(th, bl, dx);
        dx = mfma_bf16(tl, bh, dx);
      }
      dx *= ld4(&sbeta[16 * rt + 4 * g4]);
      const float4_t eu = ekd[rt] * u;
      dgc += (eu[0] + eu[1]) + (eu[2] + eu[3]);
      add_rows(eu + (bf16x4_float(L4.tr<V>(sv, 16 * rt, v0)) - x[rt]) * dx, rt);
      split_bf16(u, uh[rt], ul[rt]);
      split_bf16(x[rt], xh[rt], xl[rt]);
      split_bf16(dx, dxh[rt], dxl[rt]);
      keep_order();
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {  // over the other lanes of the row: rotations by 8 and 4
      dch[rt] += dpp_mov<0x128>(dch[rt]);
      dch[rt] += dpp_mov<0x124>(dch[rt]);
    }
    pch[wave * BC + 16 * (c >> 2) + 4 * g4 + (c & 3)] =
        c < 8 ? (c < 4 ? dch[0] : dch[1]) : (c < 12 ? dch[2] : dch[3]);
    dgc = wave_sum(dgc);
    if (lane == 0) sred[wave] = dgc;
    renew();
    // ---- contractions over the value columns
    u16 *a0 = area, *a1 = area + 2 * TV;
    auto publish = [&](u16 *m, const v2u32_t (&hi)[4], const v2u32_t (&lo)[4]) {  // [V][64] transposed pair
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        *reinterpret_cast<v2u32_t *>(m + L4.four<BC>(v0, 16 * rt)) = hi[rt];
        *reinterpret_cast<v2u32_t *>(m + TV + L4.four<BC>(v0, 16 * rt)) = lo[rt];
      }
    };
    auto publish_state = [&](const v2u32_t (&x)[KT]) {  // [V][K] transposed half
#pragma unroll
      for (int m = 0; m < KT; ++m) *reinterpret_cast<v2u32_t *>(a1 + L4.four<K>(v0, 16 * m)) = x[m];
    };
    float4_t dtb[CTW][2], dm[CTW][2], dk1[KTW][2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int m = 0; m < CTW; ++m) dtb[m][a] = dm[m][a] = zero4();
#pragma unroll
      for (int m = 0; m < KTW; ++m) dk1[m][a] = zero4();
    }
    __syncthreads();
    publish(a0, xh, xl);
    publish(a1, duh, dul);
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {  // dTb = dU X^T
      bh8_t ah[2], al[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        ah[a] = L4.cols<BC>(a1, kb, 32 * rp + 16 * a);
        al[a] = L4.cols<BC>(a1 + TV, kb, 32 * rp + 16 * a);
      }
#pragma unroll
      for (int m = 0; m < CTW; ++m) {
        const bh8_t bh = L4.cols<BC>(a0, kb, 16 * (CTW * cp + m)), bl = L4.cols<BC>(a0 + TV, kb, 16 * (CTW * cp + m));
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          dtb[m][a] = mfma_bf16(ah[a], bh, dtb[m][a]);
          dtb[m][a] = mfma_bf16(ah[a], bl, dtb[m][a]);
          dtb[m][a] = mfma_bf16(al[a], bh, dtb[m][a]);
        }
      }
    }
    __syncthreads();
    renew();
    publish(a0, uh, ul);
    publish_state(dh);
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {  // dM = dO U^T; dK1 = U dS'^T, the high half of dS'
      bh8_t od[2], ah[2], al[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        od[a] = L4.rows<V>(sdo, 32 * rp + 16 * a, kb);
        ah[a] = L4.cols<BC>(a0, kb, 32 * rp + 16 * a);
        al[a] = L4.cols<BC>(a0 + TV, kb, 32 * rp + 16 * a);
      }
#pragma unroll
      for (int m = 0; m < CTW; ++m) {
        const bh8_t bh = L4.cols<BC>(a0, kb, 16 * (CTW * cp + m)), bl = L4.cols<BC>(a0 + TV, kb, 16 * (CTW * cp + m));
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          dm[m][a] = mfma_bf16(od[a], bh, dm[m][a]);
          dm[m][a] = mfma_bf16(od[a], bl, dm[m][a]);
        }
      }
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
        const bh8_t b = L4.cols<K>(a1, kb, 16 * (KTW * cp + m));
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          dk1[m][a] = mfma_bf16(ah[a], b, dk1[m][a]);
          dk1[m][a] = mfma_bf16(al[a], b, dk1[m][a]);
        }
      }
    }
    __syncthreads();
    renew();
    publish_state(dl);
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {  // dK1: the low half of dS'
      const bh8_t a_0 = L4.cols<BC>(a0, kb, 32 * rp), a_1 = L4.cols<BC>(a0, kb, 32 * rp + 16);
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
        const bh8_t b = L4.cols<K>(a1, kb, 16 * (KTW * cp + m));
        dk1[m][0] = mfma_bf16(a_0, b, dk1[m][0]);
        dk1[m][1] = mfma_bf16(a_1, b, dk1[m][1]);
      }
    }
    renew();
    // dK1's row scale
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const float4_t e4 = ld4(&se[32 * rp + 16 * a + 4 * g4]);
#pragma unroll
      for (int m = 0; m < KTW; ++m) tk[m][a] += e4 * dk1[m][a];
    }
    __syncthreads();
    renew();
    publish(a0, dxh, dxl);
    publish_state(sh);
    {  // dv = dX, rounded (its high half): this wave's columns, four a lane and token
      u16 *dv = static_cast<u16 *>(p.dv) + (row0 * p.Hv + h) * V + v0;
      const uint32_t stride = p.Hv * V;
#pragma unroll
      for (int rt = 0; rt < 4; ++rt) {
        const v2u32_t x = __builtin_bit_cast(v2u32_t, L4.tr<BC>(a0, v0, 16 * rt));
        if (16 * rt + c < left) store_four(dv + (16 * rt + c) * stride + 4 * g4, x, p.narrow);
      }
    }
    __syncthreads();
    float4_t dk2[KTW][2], dq0[KTW][2];
#pragma unroll
    for (int m = 0; m < KTW; ++m) {
#pragma unroll
      for (int a = 0; a < 2; ++a) dk2[m][a] = dq0[m][a] = zero4();
    }
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {  // dK2 = dX S^T, dQ0 = dO S^T, the high half of S
      bh8_t od[2], ah[2], al[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        od[a] = L4.rows<V>(sdo, 32 * rp + 16 * a, kb);
        ah[a] = L4.cols<BC>(a0, kb, 32 * rp + 16 * a);
        al[a] = L4.cols<BC>(a0 + TV, kb, 32 * rp + 16 * a);
      }
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
        const bh8_t b = L4.cols<K>(a1, kb, 16 * (KTW * cp + m));
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          dk2[m][a] = mfma_bf16(ah[a], b, dk2[m][a]);
          dq0[m][a] = mfma_bf16(od[a], b, dq0[m][a]);
          dk2[m][a] = mfma_bf16(al[a], b, dk2[m][a]);
        }
      }
    }
    __syncthreads();
    renew();
    publish_state(sl);
    __syncthreads();
#pragma unroll
    for (int kb = 0; kb < VB; ++kb) {  // the low half of S
      bh8_t od[2], ah[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        od[a] = L4.rows<V>(sdo, 32 * rp + 16 * a, kb);
        ah[a] = L4.cols<BC>(a0, kb, 32 * rp + 16 * a);
      }
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
        const bh8_t b = L4.cols<K>(a1, kb, 16 * (KTW * cp + m));
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          dk2[m][a] = mfma_bf16(ah[a], b, dk2[m][a]);
          dq0[m][a] = mfma_bf16(od[a], b, dq0[m][a]);
        }
      }
    }
    renew();
    // ---- the other row scales, and Q S's part of the decay sums over the keys
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int o = 32 * rp + 16 * a + 4 * g4;
      const float4_t gam = ld4(&sgam[o]);
      float4_t dgam = zero4();
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
        const int col = 16 * (KTW * cp + m);
        dgam += p.scale * (bf16x4_float(L4.tr<K>(sq, 32 * rp + 16 * a, col)) * dq0[m][a]);
        tq[m][a] += dq0[m][a] * (gam * p.scale);
        tk[m][a] -= gam * dk2[m][a];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = group_sum(dgam[e], 16);
        if (c == 0) pdg[cp * BC + o + e] = x;
      }
    }
    __syncthreads();  // the stages' readers are done: the area now holds the C x C pairs
    renew();
    // The C x C matrices as transposed pairs [column][row]: a lane's four rows
    // of a column are one 8-byte write a half.
    u16 *b1t = area, *b2t = b1t + 2 * CC, *b3t = b2t + 2 * CC, *b4t = b3t + 2 * CC;
    auto put_t = [&](u16 *m, int row0, int col0, float4_t x) {
      v2u32_t hi, lo;
      split_bf16(x, hi, lo);
      u16 *at = m + L4.four<BC>(col0, row0);
      *reinterpret_cast<v2u32_t *>(at) = hi;
      *reinterpret_cast<v2u32_t *>(at + CC) = lo;
    };
    // dM o Mt into b1 (and its dc terms); dT = dTb diag(beta) into b2 (and dbeta)
    float4_t rc[2], rb[2], dec[CTW][2];  // row sums; D = e^(c_t - c_s)
    float cc[CTW], cb[CTW];
#pragma unroll
    for (int m = 0; m < CTW; ++m) cc[m] = cb[m] = 0.f;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int row0 = 32 * rp + 16 * a;
      const float4_t ct = ld4(&sc[row0 + 4 * g4]);
      rc[a] = rb[a] = zero4();
#pragma unroll
      for (int m = 0; m < CTW; ++m) {
        const int col0 = 16 * (CTW * cp + m), s2 = col0 + c, above = s2 - row0 - 4 * g4;  // e >= above: t >= s
        const float cs = sc[s2], bs = sbeta[s2];
        const float4_t qk = L4.rows_rows<K>(sq, sk, row0, col0);
        const bw_i16x4_t thi = L4.tr<BC>(tp, row0, col0), tlo = L4.tr<BC>(tp + CC, row0, col0);
        const float4_t tv = bf16x4_float(thi) + bf16x4_float(tlo);
#pragma unroll
        for (int e = 0; e < 4; ++e) dec[m][a][e] = expf(ct[e] - cs);
        float4_t dmd = dm[m][a] * (dec[m][a] * p.scale);
#pragma unroll
        for (int e = 0; e < 4; ++e) dmd[e] = e >= above ? dmd[e] : 0.f;
        const float4_t dcr = dmd * qk, dbr = dtb[m][a] * tv;
        put_t(b1t, row0, col0, dmd);
        put_t(b2t, row0, col0, dtb[m][a] * bs);
        rc[a] += dcr;
        cc[m] -= (dcr[0] + dcr[1]) + (dcr[2] + dcr[3]);
        cb[m] += (dbr[0] + dbr[1]) + (dbr[2] + dbr[3]);
      }
    }
    __syncthreads();
    renew();
    // W = T^T dT
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int m = 0; m < CTW; ++m) {
        const int row0 = 32 * rp + 16 * a, col0 = 16 * (CTW * cp + m);
        float4_t w = zero4();
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const bh8_t th = L4.cols<BC>(tp, kb, row0), tl = L4.cols<BC>(tp + CC, kb, row0);
          const bh8_t bh = L4.rows<BC>(b2t, col0, kb), bl = L4.rows<BC>(b2t + CC, col0, kb);
          w = mfma_bf16(th, bh, w);
          w = mfma_bf16(th, bl, w);
          w = mfma_bf16(tl, bh, w);
        }
        put_t(b4t, row0, col0, w);
      }
    }
    __syncthreads();
    renew();
    // dA = -W T^T (strict lower): H = dA beta_t D into b3; dbeta, dc terms
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const float4_t bt = ld4(&sbeta[32 * rp + 16 * a + 4 * g4]);
#pragma unroll
      for (int m = 0; m < CTW; ++m) {
        const int row0 = 32 * rp + 16 * a, col0 = 16 * (CTW * cp + m), above = col0 + c - row0 - 4 * g4;
        float4_t da = zero4();
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const bh8_t wh = L4.cols<BC>(b4t, kb, row0), wl = L4.cols<BC>(b4t + CC, kb, row0);
          const bh8_t th = L4.rows<BC>(tp, col0, kb), tl = L4.rows<BC>(tp + CC, col0, kb);
          da = mfma_bf16(wh, th, da);
          da = mfma_bf16(wh, tl, da);
          da = mfma_bf16(wl, th, da);
        }
        const float4_t gk = L4.rows_rows<K>(sk, sk, row0, col0);
        float4_t dad = dec[m][a] * -da;  // dA o D, t > s
#pragma unroll
        for (int e = 0; e < 4; ++e) dad[e] = e > above ? dad[e] : 0.f;
        const float4_t b = dad * gk, bb = b * bt;
        put_t(b3t, row0, col0, dad * bt);
        rb[a] += b;
        rc[a] += bb;
        cc[m] -= (bb[0] + bb[1]) + (bb[2] + bb[3]);
      }
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = group_sum(rc[a][e], 16), y = group_sum(rb[a][e], 16);
        if (c == 0) {
          prc[cp * BC + 32 * rp + 16 * a + 4 * g4 + e] = x;
          prb[cp * BC + 32 * rp + 16 * a + 4 * g4 + e] = y;
        }
      }
    }
#pragma unroll
    for (int m = 0; m < CTW; ++m) {
      const float x = add_xor32(add_xor16(cc[m])), y = add_xor32(add_xor16(cb[m]));
      if (g4 == 0) {
        pcc[rp * BC + 16 * (CTW * cp + m) + c] = x;
        pcb[rp * BC + 16 * (CTW * cp + m) + c] = y;
      }
    }
    __syncthreads();
    // The next head's inputs (the same head's again if it is the last: a load
    // left out on one path would keep the old values alive to the end of the
    // loop on every path), loaded during the last products. Earlier they do not
    // fit into the registers: issued among the stages they were spilled as they
    // arrived.
    const bool last_head = hh + 1 == heads;
    next = it;
    if (last_head) more = grad_item(p, it.item + gridDim.x, gridDim.x, items, chunks, blocks, next);
    if (!more) next = it;
    const int nh = next.block * heads + (last_head ? 0 : hh + 1);
    renew();
    // dQ += (dM o Mt) K;  dK += (dM o Mt)^T Q + H K + H^T K
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      keep_order();
      bh8_t kf[KTW], qf[KTW];
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
        kf[m] = L4.cols<K>(sk, kb, 16 * (KTW * cp + m));
        qf[m] = L4.cols<K>(sq, kb, 16 * (KTW * cp + m));
      }
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        // (spread over the products, which go on while the CU takes the loads)
        if (kb == 0 && a == 0) load_adjoint(next, nh, tid);
        if (kb == 0 && a == 1) load_state(next, nh, tid);
        if (kb == 1 && a == 0) load_rest(next, nh, last_head, tid);
        keep_order();
        const int row0 = 32 * rp + 16 * a;
        auto product = [&](float4_t (&x)[KTW][2], bh8_t hi, bh8_t lo, const bh8_t (&b)[KTW]) {
#pragma unroll
          for (int m = 0; m < KTW; ++m) x[m][a] = mfma_bf16(hi, b[m], x[m][a]);
#pragma unroll
          for (int m = 0; m < KTW; ++m) x[m][a] = mfma_bf16(lo, b[m], x[m][a]);
        };
        product(tq, L4.cols<BC>(b1t, kb, row0), L4.cols<BC>(b1t + CC, kb, row0), kf);
        product(tk, L4.rows<BC>(b1t, row0, kb), L4.rows<BC>(b1t + CC, row0, kb), qf);
        product(tk, L4.cols<BC>(b3t, kb, row0), L4.cols<BC>(b3t + CC, kb, row0), kf);
        product(tk, L4.rows<BC>(b3t, row0, kb), L4.rows<BC>(b3t + CC, row0, kb), kf);
        keep_order();
      }
    }
    if (wave == 0) {  // dc -> dg = reverse cumulative sum within the chunk
      const int t = lane;
      float dct = pcc[t] + pcc[BC + t], dbt = pcb[t] + pcb[BC + t], dgam = 0.f, dch = 0.f, gc = 0.f;
#pragma unroll
      for (int m = 0; m < COLS; ++m) {
        dct += prc[m * BC + t];
        dbt += prb[m * BC + t];
        dgam += pdg[m * BC + t];
      }
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        dch += pch[w * BC + t];
        gc += sred[w];
      }
      float dcv = dct + dgam * sgam[t] - dch;
      if (t == BC - 1) dcv += gc;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const float y = __shfl_down(dcv, off, 64);
        if (lane + off < 64) dcv += y;
      }
      if (t < left) {
        const long o = (row0 + t) * p.Hv + h;
        p.dg[o] = dcv;
        store_elem(p.dbeta, o, p.beta_dtype, dbt);
      }
    }
    if (last_head) {
      // dq, dk: summed over the key head's value heads, or (one head an item of
      // several) per value head in float32 for the reduction kernel
      if (heads == group) {
        // each tile through LDS, transposed (this wave writes and reads it), for
        // pieces of four keys a lane and token
        __syncthreads();  // this head's readers of sq and sk are done
        const long base = (row0 * p.Hk + h / group) * K;
        const uint32_t stride = p.Hk * K;
        u16 *buf = sq + wave * 16 * BC;
        auto out = [&](void *dst, const float4_t (&x)[KTW][2]) {
#pragma unroll
          for (int m = 0; m < KTW; ++m) {
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              *reinterpret_cast<v2u32_t *>(buf + L4.four<BC>(0, 16 * a)) =
                  __builtin_bit_cast(v2u32_t, __builtin_convertvector(x[m][a], bf16x4_t));
            }
#pragma unroll
            for (int a = 0; a < 2; ++a) {
              const v2u32_t y = __builtin_bit_cast(v2u32_t, L4.tr<BC>(buf, 0, 16 * a));
              const int t = 32 * rp + 16 * a + c;
              u16 *row = static_cast<u16 *>(dst) + base + 16 * (KTW * cp + m);
              if (t < left) store_four(row + t * stride + 4 * g4, y, p.narrow);
            }
          }
        };
        out(p.dq, tq);
        out(p.dk, tk);
      } else {
        const long base = (row0 * p.Hv + h) * K;
#pragma unroll
        for (int m = 0; m < KTW; ++m) {
#pragma unroll
          for (int a = 0; a < 2; ++a) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int t = 32 * rp + 16 * a + 4 * g4 + e, kk = 16 * (KTW * cp + m) + c;
              if (t >= left) continue;
              const uint32_t off = t * static_cast<uint32_t>(p.Hv * K) + kk;
              (p.ws_dq + base)[off] = tq[m][a][e];
              (p.ws_dk + base)[off] = tk[m][a][e];
            }
          }
        }
      }
#pragma unroll
      for (int m = 0; m < KTW; ++m) {
#pragma unroll
        for (int a = 0; a < 2; ++a) tq[m][a] = tk[m][a] = zero4();
      }
    }
    it = next;
    hh = last_head ? 0 : hh + 1;
  }
}
