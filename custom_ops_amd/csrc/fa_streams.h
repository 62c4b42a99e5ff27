// fa_streams.h — the key-stream kernels, for grids too small for the tile
// kernels. Included by fa_fwd.hip inside namespace mi355fa.
//
// A workgroup serves 32·RG query rows of one (batch, KV head) with RG·KG
// waves: KG key groups, each of RG waves that share the group's K/V tiles
// (32 rows per wave). Key group k runs its own stream of 32-key tiles; at the
// end the groups merge their (O, m, l) through LDS, in fp32.
//  * The rows are the flattened (q-head of the group, query) pairs of the KV
//    head, so a GQA decode step (Sq = 1) fills one 32-row block with all its
//    heads and reads K and V once.
//  * Tile t belongs to stream t mod (splits·KG): the live tiles of a causal,
//    window or padding mask spread evenly over the streams.
//  * The mask runs ahead of K and V: when they are issued the tile's mask has
//    landed, and a tile whose mask is all -inf (for the group's rows) is not
//    loaded.
//  * Masks whose rows are not 16-byte aligned come by LDS DMA too, as the
//    aligned 16-byte blocks that hold each row's 32 entries (5 of them); a
//    lane then reads its entries at its row's offset.

constexpr int kTS = 32;   // keys per tile

// One wave's 32 query rows: Q, O, the running max and sum, and the products.
template <int D, bool BF16> struct StreamRows {
  typedef typename Elt<BF16>::v8 V8;
  static constexpr int KD = D / 16, DB = D / 32, UPR = D / 8;
  V8 qreg[KD];
  f32x16 oacc[DB];
  float m_run, mlog2, l_run, c2, inv_scale, slack_u;
  uint32_t k_rd[KD], v_rd[DB];
  V8 msel[BF16 ? 2 : 1];

  __device__ __forceinline__ void init(float scale, int lane) {
    const int l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int i = 0; i < DB; ++i) oacc[i] = f32x16{};
    m_run = -INFINITY;
    mlog2 = l_run = 0.f;
    c2 = scale * kLog2e;
    inv_scale = 1.f / scale;
    slack_u = kRescaleSlack / scale;
#pragma unroll
    for (int kd = 0; kd < KD; ++kd) k_rd[kd] = (uint32_t)(l32 * UPR + ((2 * kd + g) ^ (l32 % UPR))) * 16u;
    const int s16 = lane & 15, grp = lane >> 4, row = 16 * g + s16 / 4;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int d = 32 * db + 16 * (grp & 1) + 4 * (s16 & 3);
      v_rd[db] = (uint32_t)(row * D * 2 + (((d / 8) ^ v_swz<D>(row)) * 16) + (d % 8) * 2);
    }
    if constexpr (BF16) {   // the mask MFMA's A operand (see Attn::MMF)
      const uint32_t sb = (uint32_t)bitcast<uint16_t>((__bf16)inv_scale);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int e = key_perm(l32) - 16 * c - 8 * g;
        u32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = (e == 2 * j) ? sb : (e == 2 * j + 1) ? (sb << 16) : 0u;
        msel[c] = bitcast<V8>(w);
      }
    }
  }

  // u = mask·(1/scale) + K·Qᵀ of one 32-key tile
  __device__ __forceinline__ f32x16 scores(const u32x4 (&mask)[2], const uint8_t* sK) {
    // all K reads at once (two in flight, as the compiler would order them,
    // leave the matrix core waiting for the LDS)
    V8 a[KD];
#pragma unroll
    for (int kd = 0; kd < KD; ++kd) a[kd] = bitcast<V8>(*reinterpret_cast<const u32x4*>(sK + k_rd[kd]));
    __builtin_amdgcn_sched_barrier(0);
    f32x16 s;
    if constexpr (BF16) {
      typedef unsigned short us2 __attribute__((ext_vector_type(2)));
      const us2 lim = {0xff7fu, 0xff7fu};   // -max_bf16 (-inf would make NaN on the matrix core)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        u32x4 x = mask[c];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          x[j] = bitcast<uint32_t>(__builtin_elementwise_min(bitcast<us2>(x[j]), lim));
        s = Elt<BF16>::mfma(msel[c], bitcast<V8>(x), c == 0 ? f32x16{} : s);
      }
    } else {
      const f32x16 mk = mask_to_f32<BF16>(mask[0], mask[1]);
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = mk[e] * inv_scale;
    }
#pragma unroll
    for (int kd = 0; kd < KD; ++kd) s = Elt<BF16>::mfma(a[kd], qreg[kd], s);
    return s;
  }

  // keys from sk - n·32 on are past Sk; then the running max (moved, and O and
  // l rescaled, only when it grew by more than the slack). Returns whether any
  // row of the wave has a key above -inf in the tile (NaN counts).
  __device__ __forceinline__ bool rescale(f32x16& s, int left, int g) {
    if (left < kTS) {
#pragma unroll
      for (int e = 0; e < 16; ++e) s[e] = (g * 16 + e < left) ? s[e] : -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int e = 1; e < 16; ++e) mx = fmaxf(mx, s[e]);
    mx = xhalf_max(mx);
    const bool some = __builtin_amdgcn_ballot_w64(!(mx == -INFINITY)) != 0;
    const bool need = mx > m_run + slack_u;
    if (__builtin_amdgcn_ballot_w64(need)) {
      const float alpha = need ? __builtin_amdgcn_exp2f((m_run - mx) * c2) : 1.f;
      m_run = need ? mx : m_run;
      mlog2 = (m_run == -INFINITY) ? 0.f : m_run * c2;
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
    }
    return some;
  }

  // P = exp2(u·c2 − m·c2) of 8 of the lane's keys, rounded; l += Σ P
  __device__ __forceinline__ V8 probs(const f32x16& s, int j) {
    f32x8 pf;
#pragma unroll
    for (int e = 0; e < 8; ++e) pf[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j * 8 + e], c2, -mlog2));
    const V8 r = __builtin_convertvector(pf, V8);
    l_run = psum8<BF16>(r, l_run);
    return r;
  }

  // Oᵀ += Vᵀ·Pᵀ
  __device__ __forceinline__ void pv(const V8 (&pj)[2], const uint8_t* sV) {
    V8 a[2 * DB];
#pragma unroll
    for (int i = 0; i < 2 * DB; ++i) {
      const int j = i / DB, db = i % DB;
      const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(sV + v_rd[db] + j * 8 * D * 2));
      const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(sV + v_rd[db] + j * 8 * D * 2 + 4 * D * 2));
      a[i] = bitcast<V8>(__builtin_shufflevector(v0, v1, 0, 1, 2, 3, 4, 5, 6, 7));
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * DB; ++i) oacc[i % DB] = Elt<BF16>::mfma(a[i], pj[i / DB], oacc[i % DB]);
  }
};

// One wave's mask tiles (32 rows x 32 keys) through its own LDS buffer.
// Aligned rows (AL): 4 units of 16 bytes per row, unit c of row r at slot
// c ^ (r / 4) % 4 (the 16 rows of a b128 read phase, at a 64-byte pitch, then
// cover all 64 banks once). Unaligned rows: the 5 aligned blocks that hold the
// row's 64 bytes, at an 80-byte pitch; a lane reads 5 words from its row's
// word offset and shifts by the odd entry, if any. The offset is the same for
// every tile (64 bytes apart).
template <bool BF16, bool AL> struct StreamMask {
  static constexpr int kUnits = AL ? 4 : 5;
  static constexpr int kLoads = AL ? 2 : 3;               // DMA instructions per tile
  static constexpr int kBytes = kLoads * 1024;            // LDS bytes per tile buffer
  static constexpr uint32_t kNegPair = BF16 ? 0xff80ff80u : 0xfc00fc00u;
  const char* base;      // the batch's mask, down to a 16-byte boundary
  uint32_t bytes;        // from there to the end, up to a 16-byte boundary
  uint32_t off[kLoads], rd[2], odd;

  // rowof(i): mask row of the wave's row i; chunk c of a lane's operand: keys
  // 16c + 8g (bf16, the mask MFMA's B operand) or 16g + 8c (fp16, its own keys)
  template <class F>
  __device__ __forceinline__ void init(const KParams& p, int b, int lane, const F& rowof) {
    const uintptr_t a = reinterpret_cast<uintptr_t>(p.mask + (int64_t)b * p.m_bs);
    const uint32_t lead = AL ? 0u : (uint32_t)(a & 15u);
    base = reinterpret_cast<const char*>(a - lead);
    bytes = (uint32_t)p.msq * (uint32_t)p.m_rs * 2u + lead;
    if (!AL) bytes = (bytes + 15u) & ~15u;
    const int l32 = lane & 31, g = lane >> 5;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int u = i * 64 + lane, r = AL ? u / 4 : min(u / 5, 31);
      const int c = AL ? (u % 4) ^ ((r >> 2) & 3) : u % 5;
      const uint32_t start = lead + (uint32_t)rowof(r) * (uint32_t)p.m_rs * 2u;
      // the last instruction's lanes past unit 159: outside the buffer
      off[i] = (AL || u < 160) ? (start & ~15u) + (uint32_t)c * 16u : 0xfffffff0u;
    }
    const uint32_t start = lead + (uint32_t)rowof(l32) * (uint32_t)p.m_rs * 2u;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int u = BF16 ? 2 * c + g : 2 * g + c;
      rd[c] = AL ? (uint32_t)(l32 * 64 + ((u ^ ((l32 >> 2) & 3)) * 16))
                 : (uint32_t)(l32 * 80 + u * 16) + (start & 12u);
    }
    odd = start & 2u;
  }
  // Tile n by DMA to LDS; past the last tile the same number of loads, from
  // an empty buffer.
  __device__ __forceinline__ void issue(int n, int ntile, uint32_t lds) const {
    const uint32_t sh = (uint32_t)n * kTS * 2u;
    const i32x4 r = make_rsrc_words(base + (n < ntile ? sh : 0u), n < ntile ? bytes - sh : 0u);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) bload16_lds(r, lds + (uint32_t)(i * 1024), off[i]);
  }
  __device__ __forceinline__ void read(u32x4 (&w)[2], const uint8_t* buf) const {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if constexpr (AL) {
        w[c] = *reinterpret_cast<const u32x4*>(buf + rd[c]);
      } else {
        uint32_t x[5];
#pragma unroll
        for (int j = 0; j < 5; ++j) x[j] = *reinterpret_cast<const uint32_t*>(buf + rd[c] + 4 * j);
#pragma unroll
        for (int j = 0; j < 4; ++j) w[c][j] = __builtin_amdgcn_alignbyte(x[j + 1], x[j], odd);
      }
    }
  }
  // Entries past Sk in the last tile (left: keys from its first to Sk) are
  // anything at all: the caller's pad columns, the next row, what out-of-range
  // DMA lanes left in the LDS. They become -inf, so that they neither meet a zero
  // of the selector as +inf or NaN nor make a tile live whose own keys are all
  // blocked.
  static __device__ __forceinline__ void clip(u32x4 (&w)[2], int left, int g) {
    if (__builtin_expect((uint32_t)(left - 1) < (uint32_t)(kTS - 1), 0)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int e = (BF16 ? 16 * (i / 4) + 8 * g : 16 * g + 8 * (i / 4)) + 2 * (i % 4);
        const uint32_t keep = e + 1 < left ? ~0u : (e < left ? 0xffffu : 0u);
        w[i / 4][i % 4] = (w[i / 4][i % 4] & keep) | (kNegPair & ~keep);
      }
    }
  }
  // whether the wave's rows hold an entry that is not -inf
  static __device__ __forceinline__ bool any(const u32x4 (&w)[2]) {
    // all entries are -inf exactly when their AND and their OR are (comparing
    // word by word would chain 8 scalar mask operations)
    uint32_t x = w[0][0], y = w[0][0];
#pragma unroll
    for (int i = 1; i < 8; ++i) { x &= w[i / 4][i % 4]; y |= w[i / 4][i % 4]; }
    return __builtin_amdgcn_ballot_w64(((x ^ kNegPair) | (y ^ kNegPair)) != 0u) != 0;
  }
};

// this wave's LDS reads have returned (a DMA may overwrite what they read)
__device__ __forceinline__ void wait_lds() {
  __builtin_amdgcn_s_waitcnt(15 | (7 << 4) | (0 << 8) | (3 << 14));
  __atomic_signal_fence(__ATOMIC_SEQ_CST);
}

// A workgroup's place: batch, KV head, split, and its block of 32·RG of the KV
// head's flattened rows (row r: head hk·ratio + r / Sq, query r % Sq; lanes
// past the last row repeat it and store nothing)
struct StreamIdx {
  int b, hk, split, row0, rows, h0, sq;
  template <int RG, class P> __device__ __forceinline__ static StreamIdx of(P p) {
    StreamIdx x;
    int t = xcd_remap(blockIdx.x, p->total);
    x.row0 = (t % p->num_m) * (32 * RG);   // row blocks fastest: they share K and V
    t /= p->num_m;
    x.split = t % p->num_splits;
    t /= p->num_splits;
    const int nhk = p->h / p->ratio;
    x.hk = t % nhk;
    x.b = t / nhk;
    x.rows = p->ratio * p->sq;
    x.h0 = x.hk * p->ratio;
    x.sq = p->sq;
    return x;
  }
  __device__ __forceinline__ void row(int r, int& h, int& m) const {
    const int f = min(r, rows - 1), j = f / sq;
    h = h0 + j;
    m = f - j * sq;
  }
};

// Merge of the KG key groups' (O, m, l): every wave's O registers (16 bytes
// per lane and quad of 4 registers, free of bank conflicts) and (m, l) go
// through LDS, and wave (rg, kg) sums quads kg·kPer .. of the groups' waves
// rg. Every wave has left its LDS stages and has no DMA in flight.
template <int D, bool BF16, int RG, int KG>
__device__ __forceinline__ void stream_merge(const StreamRows<D, BF16>& a, uint8_t* smem, int rg, int kg, int lane) {
  constexpr int kQuads = D / 8, kPer = kQuads / KG;
  static_assert(kPer >= 1, "at least one quad per wave");
  const int l32 = lane & 31, g = lane >> 5;
  float* const sml = reinterpret_cast<float*>(smem + RG * KG * kQuads * 1024);   // [kg][rg][m, l][32 rows]
  const float l_all = xhalf_sum(a.l_run);
#pragma unroll
  for (int j = 0; j < kQuads; ++j) {
    f32x4 x;
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = a.oacc[j / 4][(j % 4) * 4 + e];
    *reinterpret_cast<f32x4*>(smem + (((kg * RG + rg) * kQuads + j) * 64 + lane) * 16) = x;
  }
  sml[((kg * RG + rg) * 2 + g) * 32 + l32] = g == 0 ? a.m_run : l_all;
  wg_barrier();
  float mw[KG], mx = -INFINITY;
#pragma unroll
  for (int w = 0; w < KG; ++w) {
    mw[w] = sml[(w * RG + rg) * 64 + l32];
    mx = fmaxf(mx, mw[w]);
  }
  const float mxc = (mx == -INFINITY) ? 0.f : mx;
  float l = 0.f;
#pragma unroll
  for (int w = 0; w < KG; ++w) {
    mw[w] = __builtin_amdgcn_exp2f((mw[w] - mxc) * a.c2);   // 0 for a group that saw no key of the row
    l = __builtin_fmaf(mw[w], sml[(w * RG + rg) * 64 + 32 + l32], l);
  }
  const float inv = (l == 0.f || l != l) ? 1.f : 1.f / l;
  f32x4 out[kPer];
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    f32x4 acc = {};
#pragma unroll
    for (int w = 0; w < KG; ++w)
      acc += mw[w] * *reinterpret_cast<const f32x4*>(smem + (((w * RG + rg) * kQuads + kg * kPer + j) * 64 + lane) * 16);
    out[j] = acc * inv;
  }
  const kernarg_ptr p = reload_params();
  const StreamIdx ix = StreamIdx::of<RG>(p);
  int h, m;
  const int r = ix.row0 + rg * 32 + l32;
  ix.row(r, h, m);
  const bool in = r < ix.rows;
  // quad j holds d = 8j + 4g .. +3 of the lane's row
  if (p->num_splits > 1) {   // the split's partial: fp32, with its LSE
    const int64_t prow = (((int64_t)ix.split * p->b + ix.b) * p->h + h) * p->sq + m;
    float* dst = reinterpret_cast<float*>(p->o_part) + prow * D + kg * kPer * 8 + g * 4;
#pragma unroll
    for (int j = 0; j < kPer; ++j)
      if (in) *reinterpret_cast<f32x4*>(dst + j * 8) = out[j];
    if (kg == 0 && g == 0 && in)
      p->lse_part[prow] = (l == 0.f || l != l) ? -INFINITY
                         : __builtin_fmaf(mx, p->scale, __builtin_amdgcn_logf(l) * 0.69314718f);
    return;
  }
  typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
  typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
  auto half = [&](int j) {
    if constexpr (BF16) return bitcast<u32x2>(__builtin_convertvector(out[j], bf16x4));
    else return bitcast<u32x2>(__builtin_convertvector(out[j], f16x4));
  };
  uint16_t* dst = p->o + (int64_t)ix.b * p->o_bs + (int64_t)h * p->o_hs + (int64_t)m * p->o_rs;
  // two quads exchanged with the lane 32 apart make a 16-byte chunk per lane
  // (chunk j below, j + 1 above)
  if constexpr (kPer >= 2) {
#pragma unroll
    for (int j = 0; j < kPer; j += 2) {
      const u32x2 lo = half(j), hi = half(j + 1);
      const auto s0 = __builtin_amdgcn_permlane32_swap(lo[0], hi[0], false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(lo[1], hi[1], false, false);
      if (in) *reinterpret_cast<u32x4*>(dst + (kg * kPer + j + g) * 8) = u32x4{s0[0], s1[0], s0[1], s1[1]};
    }
  } else {
    if (in) *reinterpret_cast<u32x2*>(dst + kg * 8 + g * 4) = half(0);
  }
}

// RG = 1: every wave is a key group of its own, with its own waits and no
// barrier in the loop. K(t + 1) leaves when QK(t) has read the K stage,
// V(t + 1) when PV(t) has read the V stage; with KG streams per workgroup that
// keeps K and V tiles of all of them in flight.
template <int D, bool BF16, bool AL, int KG>
__global__ __launch_bounds__(64 * KG) __attribute__((amdgpu_waves_per_eu(2, 2)))
void fa_fwd_kernel_ks(const KParams p) {
  typedef StreamRows<D, BF16> R;
  typedef StreamMask<BF16, AL> M;
  typedef typename R::V8 V8;
  constexpr int kLoads = D / 16, kKV = kTS * D * 2;    // DMA instructions and bytes of a K (or V) tile
  // aligned rows: a second mask buffer, so that the first two masks leave
  // together (unaligned ones would not leave room for two workgroups per CU)
  constexpr int MB = AL ? 2 : 1;
  constexpr int kWaveBytes = 2 * kKV + MB * M::kBytes;
  constexpr int kMerge = KG * (D / 8) * 1024 + KG * 256;
  constexpr int kLds = KG * kWaveBytes > kMerge ? KG * kWaveBytes : kMerge;
  __shared__ __align__(16) uint8_t smem[kLds];

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const StreamIdx ix = StreamIdx::of<1>(&p);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)smem;
  uint8_t* const sK = smem + wave * kWaveBytes;     // [K | V | mask]
  uint8_t* const sV = sK + kKV;
  uint8_t* const sM = sV + kKV;
  const uint32_t ldsK = lds0 + (uint32_t)(wave * kWaveBytes), ldsV = ldsK + kKV, ldsM = ldsV + kKV;

  const int stride = p.num_splits * KG, ntile = (p.sk + kTS - 1) / kTS;
  const int first = ix.split * KG + wave;
  const int cnt = first < ntile ? (ntile - first + stride - 1) / stride : 0;

  R a;
  a.init(p.scale, lane);
  if (cnt > 0) {
    int qh, qm;
    ix.row(ix.row0 + l32, qh, qm);
    M mk;
    mk.init(p, ix.b, lane, [&](int i) {
      int h, m;
      ix.row(ix.row0 + i, h, m);
      return m;
    });
    mk.issue(first, ntile, ldsM);
    if constexpr (MB == 2) mk.issue(first + stride, ntile, ldsM + M::kBytes);
    {
      const uint16_t* qp = p.q + (int64_t)ix.b * p.q_bs + (int64_t)qh * p.q_hs + (int64_t)qm * p.q_rs + g * 8;
#pragma unroll
      for (int kd = 0; kd < R::KD; ++kd) a.qreg[kd] = bitcast<V8>(*reinterpret_cast<const u32x4*>(qp + kd * 16));
    }
    const char* kbase = reinterpret_cast<const char*>(p.k + (int64_t)ix.b * p.k_bs + (int64_t)ix.hk * p.k_hs);
    const char* vbase = reinterpret_cast<const char*>(p.v + (int64_t)ix.b * p.v_bs + (int64_t)ix.hk * p.v_hs);
    const uint32_t kbytes = (uint32_t)p.sk * p.k_rs * 2u, vbytes = (uint32_t)p.sk * p.v_rs * 2u;
    uint32_t k_off[kLoads], v_off[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int u = i * 64 + lane, r = u / R::UPR, slot = u % R::UPR;
      k_off[i] = (uint32_t)(key_perm(r) * p.k_rs + (slot ^ (r % R::UPR)) * 8) * 2u;
      v_off[i] = (uint32_t)(r * p.v_rs + (slot ^ v_swz<D>(r)) * 8) * 2u;
    }
    auto issue = [&](const char* base, uint32_t bytes, int rs, int n, uint32_t lds, const uint32_t (&off)[kLoads]) {
      const uint32_t sh = (uint32_t)n * kTS * (uint32_t)rs * 2u;
      const i32x4 r = make_rsrc_words(base + sh, bytes - sh);
      if (p.kv_nt) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) bload16_lds<true>(r, lds + (uint32_t)(i * 1024), off[i]);
      } else {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) bload16_lds<false>(r, lds + (uint32_t)(i * 1024), off[i]);
      }
    };
    auto issue_k = [&](int n) { issue(kbase, kbytes, p.k_rs, n, ldsK, k_off); };
    auto issue_v = [&](int n) { issue(vbase, vbytes, p.v_rs, n, ldsV, v_off); };

    // V rows that the last tile's DMA leaves unwritten must hold finite values
    // (their P is exactly 0)
    auto clear = [&](uint8_t* st) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        *reinterpret_cast<u32x4*>(st + i * 1024 + lane * 16) = u32x4{0u, 0u, 0u, 0u};
      wait_lds();
    };
    if (p.sk % kTS != 0) clear(sV);
    // The first tile's K and V are loaded whatever its mask holds. With one
    // buffer the second tile's mask leaves when the first's has been read.
    // Where it is all -inf they are cleared: NaN in them (rows of a cache that
    // nobody has written) would reach the tile's scores, and by way of the V stage
    // the last tile's missing rows. ([2,8,512,512] d = 64
    // 8.03 -> 8.20 µs, [1,8,100,200] 7.65 -> 7.86; decided in the loop 8.35 and 7.94.)
    issue_k(first);
    issue_v(first);
    u32x4 mraw[2], mnext[2];
    // Everything: Q too. (The compiler would otherwise wait for Q before each
    // iteration's first products, and with it for every DMA in flight.)
    wait_vmcnt<0>();
    mk.read(mraw, sM);
    wait_lds();
    M::clip(mraw, p.sk - first * kTS, g);
    if constexpr (MB == 1) mk.issue(first + stride, ntile, ldsM);
    if (__builtin_expect(!M::any(mraw), 0)) {
      clear(sK);
      clear(sV);
    }

    bool live = true;
    for (int i = 0; i < cnt; ++i) {
      const int n = first + i * stride;
      // in flight, oldest first: K(n) and V(n) if live, with mask(n + stride)
      // before K(n) (first tile, one buffer: behind V(n))
      if (live && (MB == 2 || i > 0)) wait_vmcnt<kLoads>();
      else wait_vmcnt<0>();
      mk.read(mnext, sM + ((i + 1) % MB) * M::kBytes);
      wait_lds();   // with one buffer the next DMA goes where this was read
      M::clip(mnext, p.sk - (n + stride) * kTS, g);
      const bool live_next = M::any(mnext) && i + 1 < cnt;
      mk.issue(n + 2 * stride, ntile, ldsM + (uint32_t)((i % MB) * M::kBytes));
      if (live) {
        f32x16 s = a.scores(mraw, sK);
        wait_lds();
        if (live_next) issue_k(n + stride);
        const bool some = a.rescale(s, p.sk - n * kTS, g);
        V8 pj[2];
        if (some) {
#pragma unroll
          for (int j = 0; j < 2; ++j) pj[j] = a.probs(s, j);
        }
        // V(n): older than mask(n + 2 stride) and K(n + stride)
        if (live_next) wait_vmcnt<M::kLoads + kLoads>();
        else wait_vmcnt<M::kLoads>();
        if (some) a.pv(pj, sV);
        wait_lds();
        if (live_next) issue_v(n + stride);
      } else if (live_next) {
        issue_k(n + stride);
        issue_v(n + stride);
      }
      live = live_next;
#pragma unroll
      for (int c = 0; c < 2; ++c) mraw[c] = mnext[c];
    }
  }
  wait_vmcnt<0>();
  wg_barrier();
  stream_merge<D, BF16, 1, KG>(a, smem, 0, wave, lane);
}

