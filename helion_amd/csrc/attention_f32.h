// fp32 attention on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32:
// exact fp32 products, fp32 accumulation), head_dim 64 and 128.  Included by
// attention.hip, whose argument structs, tile layout and DMA it uses.
//
// Bound: the matrix pipe.  32 x 32 x 2 takes 64 cycles of a SIMD for 4096
// FLOP (157 TFLOP/s on the card at 2.4 GHz, 153 reached by a large library
// product here), so one 32 x 32 block of scores costs D / 2 such
// instructions per product against about 16 * 6 VALU instructions: a plain
// two-stage tile loop with two wavefronts per SIMD keeps the pipe busy.
//
// Tile and split: a workgroup owns 64 rows of one (batch, head) (128 in the
// head_dim 128 forward) -- query rows in the forward and dQ, kv rows in dK/dV
// -- and SH wavefronts share each 32-row block, taking the 32-row parts of
// every streamed step in turn; their partial results meet in LDS once, at the
// end, in a fixed order.  A small batch of medium sequences (the usual fp32
// call) leaves few row tiles, and causal ones of unequal length; short work
// items balance best.  SH is 2 (64-row steps; two workgroups of four
// wavefronts a CU at head_dim 64; at head_dim 128 eight wavefronts in the
// forward and four, at 230 to 330 registers a lane, in the backward), or 4
// where that leaves compute units idle (128-row steps, head_dim 64).
//
// Operands: a lane's own row (l32 = lane & 31) lives in registers as 16-byte
// granules, elements 8 st + 4 g + j (g = lane >> 5); a tile's rows come from
// LDS by 16-byte reads of the same granules, four matrix instructions per
// read (instruction j multiplies elements 8 st + j and 8 st + 4 + j).  The
// second products take S (or dS) straight from the accumulators: register r
// holds rows 8 (r >> 2) + 4 g + (r & 3) of the tile block, so instruction r
// contracts those two rows and its other operand is one 4-byte LDS read per
// 32 columns of the same row-major tile.  Nothing is transposed and no
// score leaves the registers.
//
// Measured at [4, 12, 1024, 64] causal, forward and backward: 300 us a pass
// against 9500 us on the SIMT kernels (77 + 111 + 143 us of kernels in the
// profiler against 2820 + 3374 + 3394), 86 to 93 TFLOP/s each on the blocks
// they compute; error against float64 6.5e-7 against 8.0e-7.  At head_dim 128,
// forward / backward alone against SIMT, causal: [4, 12, 1024] 136 / 470 us
// against 4530 / 8760, [1, 32, 1024] 135 / 292 against 3370 / 6040, [2, 16,
// 700] 93 / 184 against 1760 / 3090, [8, 12, 128] 25 / 52 against 254 / 470.
//
// Numerics: every product, sum and weight is fp32; p = 2^((s * scale - m)
// log2 e) with the difference formed before the conversion to log2 units, so
// its error is that of exp(s * scale - m).
//
// Masked pairs of a partly masked 32 x 32 block are multiplied too, with a
// weight of zero, and zero times an infinite or NaN element of the other
// operand is NaN.  So where there are masked pairs, rows whose sums end in any
// NaN are taken again with the SIMT code, which visits the visible pairs
// only: what a hidden row holds never reaches the result.  The forward does so
// for an infinite sum too: its weights reach 2^8 (lazy rescaling) where those
// of the SIMT code reach 1, so values of 1e36 may overflow in its sums alone.
// (A reference point that follows every row's maximum would do without, and
// costs the forward 2 to 3%.)  It costs the forward under 1% and the backward
// 1 to 3% ([4, 12, 1024, 64] 235 -> 241 us: other registers in the main loop); a
// call all of whose rows are NaN takes four times what the SIMT kernels did,
// one wavefront going through its 32 rows.

// Per-lane byte offsets into a BTile of D fp32 (2 D 16-bit) columns: row
// granule 2 i + g of row l32 (i < 8; a granule 16 columns of 16 bytes on is
// 256 bytes on), and column l32's dword of rows 4 g + .. for the four values
// that the low key bits take (the rest of the swizzle is compile-time).
template <int D>
struct F32Offs {
  typedef BTile<2 * D> P;
  uint32_t row[8], col[4];
  __device__ __forceinline__ void init() {
    const int lane = threadIdx.x & 63, l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int i = 0; i < 8; ++i) row[i] = (uint32_t)P::off(l32, 2 * i + g);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      col[i] = (uint32_t)(4 * g * P::RB + ((((l32 >> 2) ^ g) ^ (2 * i)) << 4) + (l32 & 3) * 4);
  }
  // elements 8 st + 4 g + {0..3} of row l32 of the 32-row block at `blk`
  __device__ __forceinline__ float4 rd_row(const char* blk, int st) const {
    return *reinterpret_cast<const float4*>(blk + row[st & 7] + (st >> 3) * 256);
  }
  // element 32 mt + l32 of row 8 (r >> 2) + 4 g + (r & 3) of the block
  __device__ __forceinline__ float rd_col(const char* blk, int r, int mt) const {
    const int kk = ((r & 3) << 2) | (2 * ((r >> 2) & 1));
    return *reinterpret_cast<const float*>(blk + col[(kk & 7) >> 1] +
                                           (8 * (r >> 2) + (r & 3)) * P::RB +
                                           (((8 * mt) ^ (kk & 8)) << 4));
  }
};

__device__ __forceinline__ f32x16 mma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float at4(const float4& v, int j) {
  return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w;
}

// acc += X Y^T over D: X the 32 tile rows at `blk`, Y this lane's row (registers).
template <int D>
__device__ __forceinline__ f32x16 f32_rows(const F32Offs<D>& of, const char* blk,
                                           const float4 (&y)[D / 8], f32x16 acc) {
  constexpr int KQ = D / 8, AHEAD = 3;  // reads in flight ahead of their use
  float4 x[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) x[i] = of.rd_row(blk, i);
#pragma unroll
  for (int st = 0; st < KQ; ++st) {
    const float4 c = x[st % AHEAD];
    if (st + AHEAD < KQ) x[st % AHEAD] = of.rd_row(blk, st + AHEAD);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = mma_f32(at4(c, j), at4(y[st], j), acc);
  }
  return acc;
}

// out[mt] += X^T P over the 32 rows at `blk` (out: columns of X by this lane's row).
template <int D>
__device__ __forceinline__ void f32_cols(const F32Offs<D>& of, const char* blk, const f32x16& p,
                                         f32x16 (&out)[D / 32]) {
  constexpr int MT = D / 32, AHEAD = 4;
  float x[AHEAD][MT];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) x[i][mt] = of.rd_col(blk, i, mt);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      out[mt] = mma_f32(x[r % AHEAD][mt], p[r], out[mt]);
      if (r + AHEAD < 16) x[r % AHEAD][mt] = of.rd_col(blk, r + AHEAD, mt);
    }
  }
}

// This lane's row of D floats (zero when the row does not exist).
template <int D>
__device__ __forceinline__ void f32_load_row(float4 (&y)[D / 8], const float* p, bool valid, int g) {
#pragma unroll
  for (int st = 0; st < D / 8; ++st)
    y[st] = valid ? *reinterpret_cast<const float4*>(p + 8 * st + 4 * g)
                  : make_float4(0.f, 0.f, 0.f, 0.f);
}

template <int D>
__device__ __forceinline__ void f32_store_row(float* p, const f32x16 (&v)[D / 32], float sc, int g) {
#pragma unroll
  for (int mt = 0; mt < D / 32; ++mt)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      store4<float>(p + 32 * mt + 8 * rr + 4 * g, v[mt][4 * rr] * sc, v[mt][4 * rr + 1] * sc,
                    v[mt][4 * rr + 2] * sc, v[mt][4 * rr + 3] * sc);
}

// TILES pairs of 64-row fp32 tiles (rows r0.. of x and of y) by DMA, the
// 16-bit tiles' engine on rows of 2 D halves.
template <int D, int WAVES>
struct F32Dma {
  typedef BTile<2 * D> P;
  BtDma<bf16_t, 2 * D, WAVES, true> dma;
  __device__ __forceinline__ void init(int64_t sx, int64_t sy) { dma.init(2 * sx, 2 * sy); }
  template <int TILES>
  __device__ __forceinline__ void issue(char* dst, const float* x, int64_t sx, const float* y,
                                        int64_t sy, int r0, int n_rows) const {
#pragma unroll
    for (int i = 0; i < TILES; ++i)
      if (i == 0 || r0 + 64 * i < n_rows)
        dma.issue(dst + i * 2 * P::BYTES, (const bf16_t*)x, 2 * sx, (const bf16_t*)y, 2 * sy,
                  r0 + 64 * i, n_rows);
  }
  // byte offset of the i-th of SH 32-row blocks of x
  template <int SH>
  static __device__ __forceinline__ int rows_at(int i) {
    if constexpr (SH == 2) return 32 * i * P::RB;
    else return (i >> 1) * 2 * P::BYTES + (i & 1) * 32 * P::RB;
  }
};

template <int MT>
__device__ __forceinline__ bool f32_all_finite(const f32x16 (&v)[MT]) {
  float z = 0.f;  // NaN once an infinity or a NaN has been multiplied by 0
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 16; ++r) z = fmaf(v[mt][r], 0.f, z);
  return z == 0.f;
}

template <int MT>
__device__ __forceinline__ bool f32_any_nan(const f32x16 (&v)[MT]) {
  bool nan = false;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 16; ++r) nan |= v[mt][r] != v[mt][r];
  return nan;
}

// The wavefront's rows (bit l32) of which a lane says so.
__device__ __forceinline__ uint32_t f32_rows_where(bool x) {
  const uint64_t m = __builtin_amdgcn_ballot_w64(x);
  return (uint32_t)m | (uint32_t)(m >> 32);
}

// Row blocks of 32 per workgroup; SH wavefronts (2 or 4) share each.
template <int D> constexpr int f32_fwd_blocks() { return D == 128 ? 4 : 2; }
constexpr int kF32BwdBlocks = 2;
// workgroups per compute unit that the kernels are compiled for
template <int D> constexpr int f32_groups(int waves) { return D == 64 && waves <= 4 ? 2 : 1; }

template <int D, int SH>
__global__ void __launch_bounds__(64 * SH * f32_fwd_blocks<D>(), f32_groups<D>(SH * f32_fwd_blocks<D>()))
attn_fwd_f32(FwdArgs a) {
  constexpr int QB = f32_fwd_blocks<D>(), WAVES = SH * QB, MT = D / 32;
  constexpr int BM = 32 * QB, BK = 32 * SH;  // rows, keys per step
  typedef BTile<2 * D> P;
  constexpr int PART = QB * 64 * (16 * MT + 2);
  constexpr int STAGE = SH * P::BYTES;  // K, V of every 64 keys
  static_assert((SH - 1) * PART * 4 <= 2 * STAGE, "merge buffer");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int l32 = lane & 31, g = lane >> 5;
  const int qb = wave % QB, half = wave / QB;
  int bh, rank;
  lpt_item(xcd_remap(blockIdx.x, gridDim.x), gridDim.x, a.B * a.H, a.n_tiles, a.causal, a.B * a.H,
           bh, rank);
  const int q0 = (a.n_tiles - 1 - rank) * BM;  // rank 0: the most kv tiles
  const int b = bh / a.H, h = bh % a.H, hk = h / (a.H / a.Hkv);
  const float* kp = (const float*)a.k + b * a.sk_b + hk * a.sk_h;
  const float* vp = (const float*)a.v + b * a.sv_b + hk * a.sv_h;
  const int qw0 = q0 + 32 * qb, qrow = qw0 + l32;
  const bool qvalid = qrow < a.Tq;

  float4 qf[D / 8];
  f32_load_row<D>(qf, (const float*)a.q + b * a.sq_b + h * a.sq_h + (int64_t)qrow * a.sq_s, qvalid, g);
  F32Offs<D> of;
  of.init();
  f32x16 o[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) o[mt] = zero16();
  float m = -INFINITY, nm = 0.f, l = 0.f;  // nm: -m, 0 while m is -inf

  const int kv_end = a.causal ? min(a.Tkv, min(q0 + BM, a.Tq)) : a.Tkv;
  const int n_kv = (int)cdiv(kv_end, BK);
  F32Dma<D, WAVES> dma;
  dma.init(a.sk_s, a.sv_s);
  if (n_kv > 0) dma.template issue<SH / 2>(smem, kp, a.sk_s, vp, a.sv_s, 0, a.Tkv);
  for (int it = 0; it < n_kv; ++it) {
    wait_vmcnt<0>();
    __syncthreads();
    if (it + 1 < n_kv)
      dma.template issue<SH / 2>(smem + ((it + 1) & 1) * STAGE, kp, a.sk_s, vp, a.sv_s, BK * (it + 1), a.Tkv);
    const int kb = BK * it + 32 * half;  // this wavefront's 32 keys
    if (qw0 >= a.Tq || kb >= a.Tkv || (a.causal && kb > qw0 + 31)) continue;
    const char* Ks = smem + (it & 1) * STAGE + F32Dma<D, WAVES>::template rows_at<SH>(half);
    const char* Vs = Ks + P::BYTES;
    f32x16 s = f32_rows<D>(of, Ks, qf, zero16());
    if (kb + 32 > a.Tkv || (a.causal && kb + 31 > qw0))
      mask_above(s, (a.causal ? min(a.Tkv - 1, qrow) : a.Tkv - 1) - kb - 4 * g);
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = xor32_max(mx) * a.scale;
    // lazy rescaling as in attn_fwd_v2: m moves when a row's max exceeds it
    // by more than 5.5 (every p <= 2^8)
    if (__builtin_amdgcn_ballot_w64(mx > m + 5.5f) != 0) {
      const float m_new = fmaxf(m, mx);
      const float alpha = m_new == -INFINITY ? 1.f : fast_exp2((m - m_new) * kLog2e);
      m = m_new;
      nm = m == -INFINITY ? 0.f : -m;
      l *= alpha;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[mt][r] *= alpha;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], a.scale, nm) * kLog2e);
      l += s[r];
    }
    f32_cols<D>(of, Vs, s, o);
  }
  l += __shfl_xor(l, 32, 64);

  // the other wavefronts' (m, l, o) into LDS, merged by the first
  float* part = reinterpret_cast<float*>(smem) + qb * 64 * (16 * MT + 2) + lane;
  __syncthreads();
  if (half > 0) {
    float* out = part + (half - 1) * PART;
    out[0] = m;
    out[64] = l;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) out[64 * (2 + 16 * mt + r)] = o[mt][r];
  }
  __syncthreads();
  if (half == 0) {
#pragma unroll
    for (int i = 0; i < SH - 1; ++i, part += PART) {
      const float m1 = part[0], mm = fmaxf(m, m1);
      const float w0 = m == -INFINITY ? 0.f : fast_exp2((m - mm) * kLog2e);
      const float w1 = m1 == -INFINITY ? 0.f : fast_exp2((m1 - mm) * kLog2e);
      m = mm;
      l = l * w0 + part[64] * w1;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[mt][r] = o[mt][r] * w0 + part[64 * (2 + 16 * mt + r)] * w1;
    }
  }
  uint32_t redo = f32_rows_where(half == 0 && qvalid && !f32_all_finite(o));
  const bool again = (redo >> l32) & 1;
  for (; redo != 0; redo &= redo - 1)
    simt_fwd_row<float, D / 64>(a, D, (int64_t)bh * a.Tq + qw0 + __builtin_ctz(redo));
  if (half > 0 || !qvalid || again) return;
  // no visible key: zeros; visible keys whose scores are all -inf: NaN, as exp(-inf + inf)
  const float inv = l > 0.f ? 1.0f / l : (n_kv > 0 ? __builtin_nanf("") : 0.f);
  f32_store_row<D>((float*)a.o + b * a.so_b + h * a.so_h + (int64_t)qrow * a.so_s, o, inv, g);
  if (g == 0)
    a.lse[(int64_t)bh * a.Tq + qrow] = l > 0.f || n_kv == 0 ? m + logf(l) : __builtin_nanf("");
}

// Sum of the accumulators of the SH wavefronts of a row block, in order: the
// others hand theirs to the first through LDS (PART floats apart).
template <int MT, int SH, int PART>
__device__ __forceinline__ void f32_merge(float* part, f32x16 (&v)[MT], int half) {
  __syncthreads();
  if (half > 0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[(half - 1) * PART + 64 * (16 * mt + r)] = v[mt][r];
  }
  __syncthreads();
  if (half == 0) {
#pragma unroll
    for (int i = 0; i < SH - 1; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) v[mt][r] += part[i * PART + 64 * (16 * mt + r)];
  }
}

// dQ, and delta = rowsum(dO * O) for the dK/dV kernel: S^T = K Q^T and
// dP^T = V dO^T from row reads, dQ^T += K^T dS^T.
template <int D, int SH>
__global__ void __launch_bounds__(64 * SH * kF32BwdBlocks, f32_groups<D>(SH * kF32BwdBlocks))
attn_bwd_dq_f32(BwdArgs a) {
  constexpr int QB = kF32BwdBlocks, WAVES = SH * QB, MT = D / 32;
  constexpr int BM = 32 * QB, BK = 32 * SH;
  typedef BTile<2 * D> P;
  constexpr int PART = QB * 64 * 16 * MT;
  constexpr int STAGE = SH * P::BYTES;  // K, V of every 64 keys
  static_assert((SH - 1) * PART * 4 <= 2 * STAGE, "merge buffer");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int l32 = lane & 31, g = lane >> 5;
  const int qb = wave % QB, half = wave / QB;
  int bh, rank;
  lpt_item(xcd_remap(blockIdx.x, gridDim.x), gridDim.x, a.B * a.H, a.n_tiles, a.causal, a.B * a.H,
           bh, rank);
  const int q0 = (a.n_tiles - 1 - rank) * BM;
  const int b = bh / a.H, h = bh % a.H, hk = h / (a.H / a.Hkv);
  const float* kp = (const float*)a.k + b * a.sk_b + hk * a.sk_h;
  const float* vp = (const float*)a.v + b * a.sv_b + hk * a.sv_h;
  const int qw0 = q0 + 32 * qb, qrow = qw0 + l32;
  const bool qvalid = qrow < a.Tq;

  float4 qf[D / 8], df[D / 8];
  f32_load_row<D>(qf, (const float*)a.q + b * a.sq_b + h * a.sq_h + (int64_t)qrow * a.sq_s, qvalid, g);
  f32_load_row<D>(df, (const float*)a.dout + b * a.sdo_b + h * a.sdo_h + (int64_t)qrow * a.sdo_s,
                  qvalid, g);
  const float lse = qvalid ? a.lse[(int64_t)bh * a.Tq + qrow] : INFINITY;
  float dl = 0.f;
  if (qvalid) {
    const float* orow = (const float*)a.o + b * a.so_b + h * a.so_h + (int64_t)qrow * a.so_s;
#pragma unroll
    for (int st = 0; st < D / 8; ++st) {
      const float4 of = *reinterpret_cast<const float4*>(orow + 8 * st + 4 * g);
      dl += (df[st].x * of.x + df[st].y * of.y) + (df[st].z * of.z + df[st].w * of.w);
    }
  }
  dl += __shfl_xor(dl, 32, 64);
  if (qvalid && g == 0 && half == 0) a.delta[(int64_t)bh * a.Tq + qrow] = dl;

  F32Offs<D> of;
  of.init();
  f32x16 dq[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) dq[mt] = zero16();
  const int kv_end = a.causal ? min(a.Tkv, min(q0 + BM, a.Tq)) : a.Tkv;
  const int n_kv = (int)cdiv(kv_end, BK);
  F32Dma<D, WAVES> dma;
  dma.init(a.sk_s, a.sv_s);
  if (n_kv > 0) dma.template issue<SH / 2>(smem, kp, a.sk_s, vp, a.sv_s, 0, a.Tkv);
  for (int it = 0; it < n_kv; ++it) {
    wait_vmcnt<0>();
    __syncthreads();
    if (it + 1 < n_kv)
      dma.template issue<SH / 2>(smem + ((it + 1) & 1) * STAGE, kp, a.sk_s, vp, a.sv_s, BK * (it + 1), a.Tkv);
    const int kb = BK * it + 32 * half;
    if (qw0 >= a.Tq || kb >= a.Tkv || (a.causal && kb > qw0 + 31)) continue;
    const char* Ks = smem + (it & 1) * STAGE + F32Dma<D, WAVES>::template rows_at<SH>(half);
    const char* Vs = Ks + P::BYTES;
    f32x16 s = f32_rows<D>(of, Ks, qf, zero16());
    const f32x16 dp = f32_rows<D>(of, Vs, df, zero16());
    if (kb + 32 > a.Tkv || (a.causal && kb + 31 > qw0))
      mask_above(s, (a.causal ? min(a.Tkv - 1, qrow) : a.Tkv - 1) - kb - 4 * g);
#pragma unroll
    for (int r = 0; r < 16; ++r)
      s[r] = fast_exp2(fmaf(s[r], a.scale, -lse) * kLog2e) * (dp[r] - dl);
    f32_cols<D>(of, Ks, s, dq);
  }
  f32_merge<MT, SH, PART>(reinterpret_cast<float*>(smem) + qb * 64 * 16 * MT + lane, dq, half);
  uint32_t redo =
      a.causal || a.Tkv % 32 != 0 ? f32_rows_where(half == 0 && qvalid && f32_any_nan(dq)) : 0;
  if (half == 0 && qvalid && !((redo >> l32) & 1))
    f32_store_row<D>((float*)a.dq + b * a.sdq_b + h * a.sdq_h + (int64_t)qrow * a.sdq_s, dq, a.scale, g);
  for (; redo != 0; redo &= redo - 1)  // reads the delta stored above, before f32_merge's barriers
    simt_dq_row<float, D / 64>(a, D, (int64_t)bh * a.Tq + qw0 + __builtin_ctz(redo));
}

// dK and dV: a lane owns one kv row, the query tiles of every head of its
// group stream by: S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS.
template <int D, int SH>
__global__ void __launch_bounds__(64 * SH * kF32BwdBlocks, f32_groups<D>(SH * kF32BwdBlocks))
attn_bwd_dkdv_f32(BwdArgs a) {
  constexpr int KB = kF32BwdBlocks, WAVES = SH * KB, MT = D / 32;
  constexpr int BN = 32 * KB, BQ = 32 * SH;  // kv rows, query rows per step
  typedef BTile<2 * D> P;
  constexpr int PART = KB * 64 * 16 * MT;
  // Q and dO of every 64 query rows, then lse and delta (BQ floats each)
  constexpr int STAGE = SH * P::BYTES + SH * 256;
  static_assert((SH - 1) * PART * 4 <= 2 * STAGE && WAVES >= SH, "merge buffer");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

  const int lane = threadIdx.x & 63, wave = wave_id();
  const int l32 = lane & 31, g = lane >> 5;
  const int blk = wave % KB, half = wave / KB;
  int bhk, kt;  // kt = 0 sees the most queries
  lpt_item(xcd_remap(blockIdx.x, gridDim.x), gridDim.x, a.B * a.Hkv, a.n_tiles, a.causal,
           a.B * a.Hkv, bhk, kt);
  const int b = bhk / a.Hkv, hk = bhk % a.Hkv, group = a.H / a.Hkv;
  const int kv0 = kt * BN, kvb = kv0 + 32 * blk, kvw = kvb + l32;
  const bool kvvalid = kvw < a.Tkv;

  const int q_begin = a.causal ? kv0 : 0;  // top-left causal: rows < kv0 see none
  const int n_q = a.Tq > q_begin ? (int)cdiv(a.Tq - q_begin, BQ) : 0;
  const int n_steps = n_q * group;
  f32x16 dk[MT], dv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) dk[mt] = dv[mt] = zero16();
  float* dkr = (float*)a.dk + b * a.sdk_b + hk * a.sdk_h + (int64_t)kvw * a.sdk_s;
  float* dvr = (float*)a.dv + b * a.sdv_b + hk * a.sdv_h + (int64_t)kvw * a.sdv_s;
  if (n_steps == 0) {  // no query sees these rows
    if (half == 0 && kvvalid) {
      f32_store_row<D>(dkr, dk, 1.f, g);
      f32_store_row<D>(dvr, dv, 1.f, g);
    }
    return;
  }

  float4 kf[D / 8], vf[D / 8];
  f32_load_row<D>(kf, (const float*)a.k + b * a.sk_b + hk * a.sk_h + (int64_t)kvw * a.sk_s, kvvalid, g);
  f32_load_row<D>(vf, (const float*)a.v + b * a.sv_b + hk * a.sv_h + (int64_t)kvw * a.sv_s, kvvalid, g);
  F32Offs<D> of;
  of.init();
  F32Dma<D, WAVES> dma;
  dma.init(a.sq_s, a.sdo_s);
  auto issue = [&](int hq, int q0, char* stage) {
    dma.template issue<SH / 2>(stage, (const float*)a.q + b * a.sq_b + hq * a.sq_h, a.sq_s,
                               (const float*)a.dout + b * a.sdo_b + hq * a.sdo_h, a.sdo_s, q0, a.Tq);
    // wavefront 2 i: lse of 64-row tile i, 2 i + 1: delta
    const int64_t row = ((int64_t)b * a.H + hq) * a.Tq + min(q0 + 64 * (wave >> 1) + lane, a.Tq - 1);
    if (wave < SH)
      dma4((wave & 1 ? a.delta : a.lse) + row,
           __builtin_amdgcn_readfirstlane(
               lds_addr<true>(stage + SH * P::BYTES + (wave & 1) * SH * 128 + (wave >> 1) * 256)));
  };
  // (head, tile) of the current step and of the one being fetched
  int hq = hk * group, qi = 0, hq_n = hq, qi_n = 0;
  issue(hq, q_begin, smem);
  for (int step = 0; step < n_steps; ++step) {
    wait_vmcnt<0>();
    __syncthreads();
    hq = hq_n;
    qi = qi_n;
    if (++qi_n == n_q) {
      qi_n = 0;
      ++hq_n;
    }
    if (step + 1 < n_steps) issue(hq_n, q_begin + BQ * qi_n, smem + ((step + 1) & 1) * STAGE);
    const int qb = q_begin + BQ * qi + 32 * half;  // this wavefront's 32 query rows
    if (kvb >= a.Tkv || qb >= a.Tq || (a.causal && qb + 31 < kvb)) continue;
    const char* stage = smem + (step & 1) * STAGE;
    const char* Qs = stage + F32Dma<D, WAVES>::template rows_at<SH>(half);
    const char* dOs = Qs + P::BYTES;
    const float* lse_s = reinterpret_cast<const float*>(stage + SH * P::BYTES) + 32 * half + 4 * g;
    f32x16 s = f32_rows<D>(of, Qs, kf, zero16());
    f32x16 dp = f32_rows<D>(of, dOs, vf, zero16());
    if ((a.causal && qb < kvb + 31) || qb + 32 > a.Tq)
      mask_outside(s, a.causal ? kvw - qb - 4 * g : -64, a.Tq - qb - 4 * g);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const float4 L = *reinterpret_cast<const float4*>(lse_s + 8 * rr);
      const float4 Dl = *reinterpret_cast<const float4*>(lse_s + BQ + 8 * rr);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r = 4 * rr + j;
        s[r] = fast_exp2(fmaf(s[r], a.scale, -at4(L, j)) * kLog2e);
        dp[r] = s[r] * (dp[r] - at4(Dl, j));
      }
    }
    f32_cols<D>(of, dOs, s, dv);
    f32_cols<D>(of, Qs, dp, dk);
  }
  float* part = reinterpret_cast<float*>(smem) + blk * 64 * 16 * MT + lane;
  f32_merge<MT, SH, PART>(part, dk, half);
  f32_merge<MT, SH, PART>(part, dv, half);
  uint32_t redo = a.causal || a.Tq % 32 != 0
                      ? f32_rows_where(half == 0 && kvvalid && (f32_any_nan(dk) || f32_any_nan(dv)))
                      : 0;
  if (half == 0 && kvvalid && !((redo >> l32) & 1)) {
    f32_store_row<D>(dkr, dk, a.scale, g);
    f32_store_row<D>(dvr, dv, 1.f, g);
  }
  for (; redo != 0; redo &= redo - 1)
    simt_dkdv_row<float, D / 64>(a, D, (int64_t)bhk * a.Tkv + kvb + __builtin_ctz(redo));
}

// Whether four wavefronts share a row block (head_dim 64): `blocks` of 64
// rows that leave compute units idle, or under the causal mask at most two of
// them a compute unit, whose longest sweeps set the time.  Forward and
// backward, two -> four wavefronts a block: [1, 32, 1024] 240 -> 206 us,
// [2, 16, 700] 155 -> 129, [1, 16, 2048] 453 -> 362, against [4, 12, 1024]
// 288 -> 326, [16, 12, 300] 154 -> 201 and, without a mask, [2, 12, 1024]
// 309 -> 340: a compute unit then runs one workgroup whose wavefronts meet
// at every barrier instead of two that cover each other.
bool f32_share4(int64_t D, bool causal, int64_t blocks) {
  return D == 64 && blocks <= (causal ? 2 : 1) * (int64_t)cu_count();
}

// Whether the query rows (forward, dQ) stay on the SIMT kernels: a 32 x 32
// block costs the matrix kernels the same however few of its pairs exist,
// and a workgroup fills a compute unit (half of one at head_dim 64), while the
// SIMT kernels take one wavefront a row and one key after the other.  So they
// win where a row sees at most `few` keys, and where a few rows and keys of
// very many heads make many workgroups of little work.  Measured, SIMT ->
// matrix, forward, us:
//   keys    causal [8, 8] x 64 heads, 64: 7.7 -> 14.2, [13, 13] x 512 11.5 ->
//     14.3, [14, 14] x 2048, 128: 63 -> 72, against [16, 16] x 64, 128: 12 -> 10
//   heads, no mask  head_dim 128: 1 x 64 keys x 4096 heads 113 -> 203, x 2048 83 -> 104,
//     x 1024 85 -> 54; 2 x 128 x 4096 270 -> 338; 4 x 64 x 2048 106 -> 104;
//     head_dim 64: 1 x 32 x 4096 32 -> 55, 1 x 64 x 4096 59 -> 57, x 2048 53 -> 31
bool f32_rows_simt(int64_t D, bool causal, int64_t heads, int64_t Tq, int64_t Tkv, int64_t few) {
  const int64_t keys = causal ? std::min(Tq, Tkv) : Tkv;  // of a row, at most
  int64_t per = D == 64 ? 64 : heads >= 8 * (int64_t)cu_count() ? 16 : 32;
  if (keys <= 16) per = D == 64 ? 32 : 16;
  return keys <= few || Tq * keys <= heads / per;
}
constexpr int64_t kF32FewFwd = 13;
// Backward: keys of a row (dQ), query rows of a head (dK/dV; whatever the
// group: the matrix kernel takes a step of 64 rows per head).  [16, 16] x 8
// heads at 128: 24.6 -> 29 us for both, [18, 18] 27 -> 30, [20, 20] x 64 32 -> 30;
// at 64 [16, 16] 18.5 -> 20, [18, 18] 20 -> 20
template <int D> constexpr int64_t f32_few_bwd() { return D == 128 ? 18 : 16; }

template <int D>
int fwd_f32(const FwdArgs& a, hipStream_t st) {
  if (f32_rows_simt(D, a.causal, (int64_t)a.B * a.H, a.Tq, a.Tkv, kF32FewFwd)) {
    attn_fwd_simt<float, D / 64><<<(unsigned)((int64_t)a.B * a.H * a.Tq), 64, 0, st>>>(a, D);
    return check_launch("attention forward (simt)");
  }
  FwdArgs x = a;
  constexpr int QB = f32_fwd_blocks<D>();
  x.n_tiles = (int)cdiv(a.Tq, 32 * QB);
  const int64_t blocks = (int64_t)x.n_tiles * a.B * a.H;
  if constexpr (D == 64) {
    if (f32_share4(D, a.causal, blocks)) {
      attn_fwd_f32<D, 4><<<(unsigned)blocks, 256 * QB, 0, st>>>(x);
      return check_launch("attention forward (fp32)");
    }
  }
  attn_fwd_f32<D, 2><<<(unsigned)blocks, 128 * QB, 0, st>>>(x);
  return check_launch("attention forward (fp32)");
}

// dQ first: it also computes delta, which the dK/dV kernel reads.
template <int D>
int bwd_f32(const BwdArgs& a, hipStream_t st) {
  constexpr int RB = kF32BwdBlocks;
  BwdArgs x = a;
  x.n_tiles = (int)cdiv(a.Tq, 32 * RB);
  const int64_t q_blocks = (int64_t)x.n_tiles * a.B * a.H;
  if (f32_rows_simt(D, a.causal, (int64_t)a.B * a.H, a.Tq, a.Tkv, f32_few_bwd<D>())) {
    const int64_t rows = (int64_t)a.B * a.H * a.Tq;
    attn_bwd_delta<float><<<(unsigned)cdiv(rows, 4), 256, 0, st>>>(a, D);
    if (int e = check_launch("attention backward (delta)")) return e;
    attn_bwd_dq_simt<float, D / 64><<<(unsigned)rows, 64, 0, st>>>(a, D);
  } else if (f32_share4(D, a.causal, q_blocks)) {
    if constexpr (D == 64) attn_bwd_dq_f32<D, 4><<<(unsigned)q_blocks, 256 * RB, 0, st>>>(x);
  } else {
    attn_bwd_dq_f32<D, 2><<<(unsigned)q_blocks, 128 * RB, 0, st>>>(x);
  }
  if (int e = check_launch("attention backward (dq, fp32)")) return e;
  x.n_tiles = (int)cdiv(a.Tkv, 32 * RB);
  const int64_t kv_blocks = (int64_t)x.n_tiles * a.B * a.Hkv;
  if (a.Tq <= f32_few_bwd<D>()) {
    const int64_t kv_rows = (int64_t)a.B * a.Hkv * a.Tkv;
    attn_bwd_dkdv_simt<float, D / 64><<<(unsigned)kv_rows, 64, 0, st>>>(a, D);
  } else if (f32_share4(D, a.causal, kv_blocks)) {
    if constexpr (D == 64) attn_bwd_dkdv_f32<D, 4><<<(unsigned)kv_blocks, 256 * RB, 0, st>>>(x);
  } else {
    attn_bwd_dkdv_f32<D, 2><<<(unsigned)kv_blocks, 128 * RB, 0, st>>>(x);
  }
  return check_launch("attention backward (dk/dv, fp32)");
}
