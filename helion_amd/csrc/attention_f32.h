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
// Tile and split: a workgroup owns 32 * RBLK rows of one (batch, head) --
// query rows in the forward and dQ, kv rows in dK/dV -- and TWO wavefronts
// share each 32-row block, taking the two 32-row halves of every streamed
// 64-row tile; their partial results meet in LDS once, at the end, in a
// fixed order.  A small batch of medium sequences (the usual fp32 call)
// leaves few row tiles: 64-row tiles whose sweep is split over four
// wavefronts keep every SIMD of a compute unit on the same short work item,
// which balances causal sweeps better than 128-row tiles would.
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
// Measured at [4, 12, 1024, 64] causal, forward and backward: 289 us a pass
// against 9520 us on the SIMT kernels (78 + 110 + 139 us of kernels in the
// profiler against 2820 + 3374 + 3394), 87 to 99 TFLOP/s each on the blocks
// they compute; error against float64 6.5e-7 against 8.0e-7.
//
// Numerics: every product, sum and weight is fp32; p = 2^((s * scale - m)
// log2 e) with the difference formed before the conversion to log2 units, so
// its error is that of exp(s * scale - m).

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

// Two 64-row fp32 tiles by DMA (the 16-bit tiles' engine on rows of 2 D halves).
template <int D, int WAVES>
struct F32Dma {
  BtDma<bf16_t, 2 * D, WAVES> dma;
  __device__ __forceinline__ void init(int64_t sx, int64_t sy) { dma.init(2 * sx, 2 * sy); }
  __device__ __forceinline__ void issue(char* dst, const float* x, int64_t sx, const float* y,
                                        int64_t sy, int r0, int n_rows) const {
    dma.issue(dst, (const bf16_t*)x, 2 * sx, (const bf16_t*)y, 2 * sy, r0, n_rows);
  }
};

// 32-row blocks per workgroup: the forward at head_dim 128 runs four (eight
// wavefronts, two per SIMD beside its 128 KB of LDS); the backward kernels
// at head_dim 128 hold 230 to 330 registers a lane and run one wavefront per
// SIMD; everything at head_dim 64 runs two workgroups of four per CU.
template <int D> constexpr int f32_fwd_blocks() { return D == 128 ? 4 : 2; }
constexpr int kF32BwdBlocks = 2;

template <int D>
__global__ void __launch_bounds__(128 * f32_fwd_blocks<D>(), D == 128 ? 1 : 2)
attn_fwd_f32(FwdArgs a) {
  constexpr int QB = f32_fwd_blocks<D>(), WAVES = 2 * QB, MT = D / 32, BM = 32 * QB;
  typedef BTile<2 * D> P;
  constexpr int STAGE = 2 * P::BYTES;  // K, V
  static_assert(QB * 64 * (16 * MT + 2) * 4 <= 2 * STAGE, "merge buffer");
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

  const int kv_end = a.causal ? min(a.Tkv, q0 + BM) : a.Tkv;
  const int n_kv = (int)cdiv(kv_end, 64);
  F32Dma<D, WAVES> dma;
  dma.init(a.sk_s, a.sv_s);
  if (n_kv > 0) dma.issue(smem, kp, a.sk_s, vp, a.sv_s, 0, a.Tkv);
  for (int it = 0; it < n_kv; ++it) {
    wait_vmcnt<0>();
    __syncthreads();
    if (it + 1 < n_kv)
      dma.issue(smem + ((it + 1) & 1) * STAGE, kp, a.sk_s, vp, a.sv_s, 64 * (it + 1), a.Tkv);
    const int kb = 64 * it + 32 * half;  // this wavefront's 32 keys
    if (kb >= a.Tkv || (a.causal && kb > qw0 + 31)) continue;
    const char* Ks = smem + (it & 1) * STAGE + 32 * half * P::RB;
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

  // the second half's (m, l, o) into LDS, merged by the first
  float* part = reinterpret_cast<float*>(smem) + qb * 64 * (16 * MT + 2) + lane;
  __syncthreads();
  if (half == 1) {
    part[0] = m;
    part[64] = l;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[64 * (2 + 16 * mt + r)] = o[mt][r];
  }
  __syncthreads();
  if (half == 1 || !qvalid) return;
  const float m1 = part[0], mt_ = fmaxf(m, m1);
  const float w0 = m == -INFINITY ? 0.f : fast_exp2((m - mt_) * kLog2e);
  const float w1 = m1 == -INFINITY ? 0.f : fast_exp2((m1 - mt_) * kLog2e);
  l = l * w0 + part[64] * w1;
  // no visible key: zeros; visible keys whose scores are all -inf: NaN, as exp(-inf + inf)
  const float inv = l > 0.f ? 1.0f / l : (n_kv > 0 ? __builtin_nanf("") : 0.f);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[mt][r] = o[mt][r] * w0 + part[64 * (2 + 16 * mt + r)] * w1;
  f32_store_row<D>((float*)a.o + b * a.so_b + h * a.so_h + (int64_t)qrow * a.so_s, o, inv, g);
  if (g == 0)
    a.lse[(int64_t)bh * a.Tq + qrow] = l > 0.f || n_kv == 0 ? mt_ + logf(l) : __builtin_nanf("");
}

// Sum of the two halves' accumulators: half 1 hands its over through LDS.
template <int MT>
__device__ __forceinline__ void f32_merge(float* part, f32x16 (&v)[MT], int half) {
  __syncthreads();
  if (half == 1) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) part[64 * (16 * mt + r)] = v[mt][r];
  }
  __syncthreads();
  if (half == 0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) v[mt][r] += part[64 * (16 * mt + r)];
  }
}

// dQ, and delta = rowsum(dO * O) for the dK/dV kernel: S^T = K Q^T and
// dP^T = V dO^T from row reads, dQ^T += K^T dS^T.
template <int D>
__global__ void __launch_bounds__(128 * kF32BwdBlocks, D == 128 ? 1 : 2)
attn_bwd_dq_f32(BwdArgs a) {
  constexpr int QB = kF32BwdBlocks, WAVES = 2 * QB, MT = D / 32, BM = 32 * QB;
  typedef BTile<2 * D> P;
  constexpr int STAGE = 2 * P::BYTES;  // K, V
  static_assert(QB * 64 * 16 * MT * 4 <= 2 * STAGE, "merge buffer");
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
  const int kv_end = a.causal ? min(a.Tkv, q0 + BM) : a.Tkv;
  const int n_kv = (int)cdiv(kv_end, 64);
  F32Dma<D, WAVES> dma;
  dma.init(a.sk_s, a.sv_s);
  if (n_kv > 0) dma.issue(smem, kp, a.sk_s, vp, a.sv_s, 0, a.Tkv);
  for (int it = 0; it < n_kv; ++it) {
    wait_vmcnt<0>();
    __syncthreads();
    if (it + 1 < n_kv)
      dma.issue(smem + ((it + 1) & 1) * STAGE, kp, a.sk_s, vp, a.sv_s, 64 * (it + 1), a.Tkv);
    const int kb = 64 * it + 32 * half;
    if (kb >= a.Tkv || (a.causal && kb > qw0 + 31)) continue;
    const char* Ks = smem + (it & 1) * STAGE + 32 * half * P::RB;
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
  f32_merge<MT>(reinterpret_cast<float*>(smem) + qb * 64 * 16 * MT + lane, dq, half);
  if (half == 0 && qvalid)
    f32_store_row<D>((float*)a.dq + b * a.sdq_b + h * a.sdq_h + (int64_t)qrow * a.sdq_s, dq, a.scale, g);
}

// dK and dV: a lane owns one kv row, the query tiles of every head of its
// group stream by: S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS.
template <int D>
__global__ void __launch_bounds__(128 * kF32BwdBlocks, D == 128 ? 1 : 2)
attn_bwd_dkdv_f32(BwdArgs a) {
  constexpr int KB = kF32BwdBlocks, WAVES = 2 * KB, MT = D / 32, BN = 32 * KB;
  typedef BTile<2 * D> P;
  constexpr int STAGE = 2 * P::BYTES + 512;  // Q, dO, lse[64], delta[64]
  static_assert(KB * 64 * 16 * MT * 4 <= 2 * STAGE && WAVES >= 2, "merge buffer");
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

  float4 kf[D / 8], vf[D / 8];
  f32_load_row<D>(kf, (const float*)a.k + b * a.sk_b + hk * a.sk_h + (int64_t)kvw * a.sk_s, kvvalid, g);
  f32_load_row<D>(vf, (const float*)a.v + b * a.sv_b + hk * a.sv_h + (int64_t)kvw * a.sv_s, kvvalid, g);
  F32Offs<D> of;
  of.init();
  f32x16 dk[MT], dv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) dk[mt] = dv[mt] = zero16();

  const int q_begin = a.causal ? kv0 : 0;  // top-left causal: rows < kv0 see none
  const int n_q = a.Tq > q_begin ? (int)cdiv(a.Tq - q_begin, 64) : 0;
  const int n_steps = n_q * group;
  F32Dma<D, WAVES> dma;
  dma.init(a.sq_s, a.sdo_s);
  auto issue = [&](int hq, int q0, char* stage) {
    dma.issue(stage, (const float*)a.q + b * a.sq_b + hq * a.sq_h, a.sq_s,
              (const float*)a.dout + b * a.sdo_b + hq * a.sdo_h, a.sdo_s, q0, a.Tq);
    const int64_t row = ((int64_t)b * a.H + hq) * a.Tq + min(q0 + lane, a.Tq - 1);
    if (wave == 0) dma4(a.lse + row, __builtin_amdgcn_readfirstlane(lds_addr(stage + 2 * P::BYTES)));
    if (wave == 1)
      dma4(a.delta + row, __builtin_amdgcn_readfirstlane(lds_addr(stage + 2 * P::BYTES + 256)));
  };
  // (head, tile) of the current step and of the one being fetched
  int hq = hk * group, qi = 0, hq_n = hq, qi_n = 0;
  if (n_steps > 0) issue(hq, q_begin, smem);
  for (int step = 0; step < n_steps; ++step) {
    wait_vmcnt<0>();
    __syncthreads();
    hq = hq_n;
    qi = qi_n;
    if (++qi_n == n_q) {
      qi_n = 0;
      ++hq_n;
    }
    if (step + 1 < n_steps) issue(hq_n, q_begin + 64 * qi_n, smem + ((step + 1) & 1) * STAGE);
    const int qb = q_begin + 64 * qi + 32 * half;  // this wavefront's 32 query rows
    if (qb >= a.Tq || (a.causal && qb + 31 < kvb)) continue;
    const char* stage = smem + (step & 1) * STAGE;
    const char* Qs = stage + 32 * half * P::RB;
    const char* dOs = Qs + P::BYTES;
    const float* lse_s = reinterpret_cast<const float*>(stage + 2 * P::BYTES) + 32 * half + 4 * g;
    f32x16 s = f32_rows<D>(of, Qs, kf, zero16());
    f32x16 dp = f32_rows<D>(of, dOs, vf, zero16());
    if ((a.causal && qb < kvb + 31) || qb + 32 > a.Tq)
      mask_outside(s, a.causal ? kvw - qb - 4 * g : -64, a.Tq - qb - 4 * g);
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const float4 L = *reinterpret_cast<const float4*>(lse_s + 8 * rr);
      const float4 Dl = *reinterpret_cast<const float4*>(lse_s + 64 + 8 * rr);
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
  f32_merge<MT>(part, dk, half);
  f32_merge<MT>(part, dv, half);
  if (half == 0 && kvvalid) {
    f32_store_row<D>((float*)a.dk + b * a.sdk_b + hk * a.sdk_h + (int64_t)kvw * a.sdk_s, dk, a.scale, g);
    f32_store_row<D>((float*)a.dv + b * a.sdv_b + hk * a.sdv_h + (int64_t)kvw * a.sdv_s, dv, 1.f, g);
  }
}

template <int D>
int fwd_f32(const FwdArgs& a, hipStream_t st) {
  FwdArgs x = a;
  constexpr int QB = f32_fwd_blocks<D>();
  x.n_tiles = (int)cdiv(a.Tq, 32 * QB);
  const int64_t blocks = (int64_t)x.n_tiles * a.B * a.H;
  attn_fwd_f32<D><<<(unsigned)blocks, 128 * QB, 0, st>>>(x);
  return check_launch("attention forward (fp32)");
}

// dQ first: it also computes delta, which the dK/dV kernel reads.
template <int D>
int bwd_f32(const BwdArgs& a, hipStream_t st) {
  BwdArgs x = a;
  x.n_tiles = (int)cdiv(a.Tq, 32 * kF32BwdBlocks);
  const int64_t q_blocks = (int64_t)x.n_tiles * a.B * a.H;
  attn_bwd_dq_f32<D><<<(unsigned)q_blocks, 128 * kF32BwdBlocks, 0, st>>>(x);
  if (int e = check_launch("attention backward (dq, fp32)")) return e;
  x.n_tiles = (int)cdiv(a.Tkv, 32 * kF32BwdBlocks);
  const int64_t kv_blocks = (int64_t)x.n_tiles * a.B * a.Hkv;
  attn_bwd_dkdv_f32<D><<<(unsigned)kv_blocks, 128 * kF32BwdBlocks, 0, st>>>(x);
  return check_launch("attention backward (dk/dv, fp32)");
}
