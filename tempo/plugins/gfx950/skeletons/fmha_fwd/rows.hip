// fmha_rows -- attention forward for few query rows (Sq * H / Hkv <= 32: a decode step), and the
// merge of key ranges that several workgroups computed.  Semantics and lane maps are
// fmha_fwd/kernel.hip's, whose helpers this file uses.
//
// k_fmha_rows.  All packed rows of one (batch, KV head) fit the 32 columns of one MFMA, so there
// is nothing to share between waves but the rows: each wave streams key blocks of its own (block
// lo + wave, + 4, ...) and keeps its own running max, sum and O; the four are merged through LDS
// at the end.  What bounds it is HBM: every key and value is read once, by one workgroup, and
// the matrix work of a wave's 32-key block (0.45 us at D = 256) is a tenth of the time the CU's
// share of the HBM rate takes to bring its four waves' blocks (128 KiB at 28 GB/s).  So the layout
// serves the stream only:
//   * a wave's K and V blocks have one LDS slot each (128 KiB per workgroup at D = 256, 64 KiB
//     and two workgroups per CU at D = 128).  K(next) is copied as soon as the scores have read
//     K, V(next) as soon as P.V has read V, so at least half of the LDS is always in flight;
//     copies retire in order, so one counted wait exposes K or V alone.
//   * no workgroup barrier inside the loop: the waves drift apart and their copies interleave.
//   * the key range is cut into `chunk` blocks per workgroup (grid = ranges x KV heads x
//     batch), so that a batch of a few sequences fills the 256 CUs; each range's unnormalised O,
//     reference and sum go to the workspace in fp32 and k_fmha_combine merges them.
//   * the copies carry the nontemporal policy, for K and V pass once (us, cached -> nontemporal, 16
//     heads, 8 KV heads, D = 256: 8 sequences x 4099 keys 53 -> 47.5, 32 x 4096 174 -> 153; 32
//     heads, D = 128, 32 x 2048 54 -> 45).
// Measured (us; before: a 128-row tile of k_fmha_fwd per query head), the same heads: 8 x 4099
// 149 -> 47.5 (5.7 TB/s); 32 x 4096 345 -> 153 (7.0 TB/s); 1 x 32768 1084 -> 54; 1 x 512 21 -> 12;
// 32 heads, D = 128, 32 x 2048 196 -> 45.
namespace fmha {

template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, D == 128 ? 2 : 1) void k_fmha_rows(
    const _Float16* __restrict__ Q, const _Float16* __restrict__ Kg,
    const _Float16* __restrict__ Vg, _Float16* __restrict__ O, float* __restrict__ LSE, int B,
    int H, int Hkv, int Sq, int Sk, float scale_log2, long q_sb, long q_ss, long q_sh, long k_sb,
    long k_ss, long k_sh, long v_sb, long v_ss, long v_sh, long o_sb, long o_ss, long o_sh,
    int chunk, float* __restrict__ part, float* __restrict__ part_ml) {
  constexpr int KB = 32, WAVES = 4;
  constexpr int DS = D / 16, DB = D / 32, DCH = D / 8;
  constexpr int RB = D * 2;
  constexpr int ROWS_PER_KB = 1024 / RB;
  constexpr int BLK = KB / ROWS_PER_KB;  // copies (1 KiB each) of one operand's block
  constexpr int TILE_B = KB * RB;
  __shared__ __attribute__((aligned(1024))) char ks[WAVES * TILE_B];
  __shared__ __attribute__((aligned(1024))) char vs[WAVES * TILE_B];
  __shared__ float wm[WAVES][32], wl[WAVES][32];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane >> 5, l32 = lane & 31;
  const int G = H / Hkv, R = Sq * G, per = Hkv * B;
  const int sp = blockIdx.x / per, hb = blockIdx.x % per;
  const int hk = hb % Hkv, b = hb / Hkv;
  const int off = Sk - Sq;
  const int nkt = fmha_tile_blocks<CAUSAL>(0, R, R, G, Sq, Sk);
  const int lo = sp * chunk, hi = min(nkt, lo + chunk);

  const int row = min(l32, R - 1), qi = row / G;
  const _Float16* Qp = Q + b * q_sb + (long)(hk * G + row % G) * q_sh + (long)qi * q_ss;
  f16x8 qf[DS];
#pragma unroll
  for (int st = 0; st < DS; ++st) qf[st] = *reinterpret_cast<const f16x8*>(Qp + 16 * st + 8 * hl);

  const char* Kp = reinterpret_cast<const char*>(Kg + b * k_sb + (long)hk * k_sh);
  const char* Vp = reinterpret_cast<const char*>(Vg + b * v_sb + (long)hk * v_sh);
  char* const kw = ks + wave * TILE_B;
  char* const vw = vs + wave * TILE_B;

  // copies: instruction i of a block fills its rows [i, i + 1) * ROWS_PER_KB; the chunk swizzle
  // has period 16 rows, so lane offsets repeat every 16 / ROWS_PER_KB instructions
  const int rin = lane / DCH, phys = lane % DCH;
  constexpr int PER = 16 / ROWS_PER_KB;
  int crow[PER], ccol[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    crow[i] = i * ROWS_PER_KB + rin;
    ccol[i] = (phys ^ fmha_swz(crow[i])) * 16;
  }
  // rows past Sk re-read row Sk-1; the buffer starts at the block's first row and ends with row
  // Sk-1 (host: 32 rows x stride x 2 < 2^31)
  auto copy_block = [&](const char* base, long ss, char* dst, int kb) {
    const int j0 = kb * KB;
    const char* blk = base + (long)j0 * ss * 2;
    const long span = (long)(Sk - 1 - j0) * ss * 2 + D * 2;
    const unsigned nrec = span < 0xFFFFFFFFL ? (unsigned)span : 0xFFFFFFFFu;
    const int lastr = Sk - 1 - j0;
#pragma unroll
    for (int i = 0; i < BLK; ++i) {
      const int rr = min(crow[i % PER] + (i / PER) * 16, lastr);
      fmha_buf_lds16<2>(blk, nrec, dst + i * 1024, (unsigned)(rr * (int)ss * 2 + ccol[i % PER]));
    }
  };

  const int kkey = fmha_swz(l32);
  int koff[8];
#pragma unroll
  for (int s7 = 0; s7 < 8; ++s7) koff[s7] = l32 * RB + (((2 * s7) | hl) ^ kkey) * 16;
  const int tg = lane >> 4, tj = lane & 15;
  const int tk = 4 * (tg >> 1) + (tj >> 2);
  const int cd = 2 * (tg & 1) + ((tj & 3) >> 1);
  const int half = 8 * (tj & 1);
  int voff0[4], voff1[4];
#pragma unroll
  for (int p4 = 0; p4 < 4; ++p4) {
    voff0[p4] = tk * RB + (((p4 << 2) | cd) ^ fmha_swz(tk)) * 16 + half;
    voff1[p4] = (tk + 8) * RB + (((p4 << 2) | cd) ^ fmha_swz(tk + 8)) * 16 + half;
  }

  f32x16 acc_o[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc_o[i][v] = 0.f;
  float m_run = -__builtin_inff(), l_run = 0.f;

  int kb = lo + wave;
  if (kb < hi) {
    copy_block(Kp, k_ss, kw, kb);
    copy_block(Vp, v_ss, vw, kb);
  }
  auto block = [&](auto morec) {  // block kb; more: copies of block kb + WAVES follow its reads
    constexpr bool more = decltype(morec)::value;
    asm volatile("" ::: "memory");
    fmha_wait_vm<BLK>();  // K is in (V's copies, issued after it, may still fly)
    asm volatile("" ::: "memory");
    f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
    for (int st = 0; st < DS; ++st) {
      const f16x8 kf = *reinterpret_cast<const f16x8*>(kw + koff[st & 7] + (st >> 3) * 256);
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[st], s, 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // K has been read: its slot is free
    if constexpr (more) copy_block(Kp, k_ss, kw, kb + WAVES);
    const int j0 = kb * KB;
    if (j0 + KB > Sk || (CAUSAL && j0 + KB - 1 > off)) {
      const int lim = (CAUSAL ? min(Sk - 1, qi + off) : Sk - 1) - j0 - 4 * hl;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = (8 * (r >> 2) + (r & 3)) > lim ? -__builtin_inff() : s[r];
    }
    float mx = -__builtin_inff();
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    const float mxs = fmha_max_halves(mx) * scale_log2;
    if (__builtin_amdgcn_ballot_w64(!(mxs - m_run <= FMHA_TAU)) != 0) {
      const float m_new = fmaxf(m_run, mxs);
      const float alpha =
          (m_new == -__builtin_inff()) ? 1.f : __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
      m_run = m_new;
#pragma unroll
      for (int i = 0; i < DB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc_o[i][r] *= alpha;
    }
    const float m_use = (m_run == -__builtin_inff()) ? 0.f : m_run;
    f16x8 p[2];
    float psum = 0.f;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float pv = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], scale_log2, -m_use));
      psum += pv;
      p[e >> 3][e & 7] = (_Float16)pv;
    }
    l_run += fmha_sum_halves(psum);
    asm volatile("" ::: "memory");
    fmha_wait_vm<more ? BLK : 0>();  // V is in (K(next) may still fly)
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < DS; ++i) {
      const int tt = i / DB, db = i % DB;
      const u32x2 a = fmha_tr_read(vw + voff0[db & 3] + 16 * tt * RB + (db >> 2) * 256);
      const u32x2 c = fmha_tr_read(vw + voff1[db & 3] + 16 * tt * RB + (db >> 2) * 256);
      const u32x4 vv = {a[0], a[1], c[0], c[1]};
      acc_o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(vv), p[tt], acc_o[db], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // V has been read
    if constexpr (more) copy_block(Vp, v_ss, vw, kb + WAVES);
  };
  for (; kb + WAVES < hi; kb += WAVES) block(IC<1>{});
  if (kb < hi) block(IC<0>{});

  // merge of the four waves: a common reference, then O and l summed in wave order.  Wave w's
  // scaled O is a [32][D] fp32 image (16-byte chunk c of row r at c ^ r) in the K and V slots.
  if (hl == 0) wm[wave][l32] = m_run;
  __syncthreads();
  const float m = fmaxf(fmaxf(wm[0][l32], wm[1][l32]), fmaxf(wm[2][l32], wm[3][l32]));
  const float w = __builtin_amdgcn_exp2f(m_run - ((m == -__builtin_inff()) ? 0.f : m));
  if (hl == 0) wl[wave][l32] = l_run * w;
  constexpr int IMG = 32 * D * 4;
  static_assert(2 * IMG == WAVES * TILE_B, "two images per operand's slots");
  char* const img = (wave < 2 ? ks : vs) + (wave & 1) * IMG;
  if (l32 < R) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 o = {acc_o[db][4 * g + 0] * w, acc_o[db][4 * g + 1] * w,
                         acc_o[db][4 * g + 2] * w, acc_o[db][4 * g + 3] * w};
        *reinterpret_cast<f32x4*>(img + l32 * D * 4 + (((db * 8 + 2 * g + hl) ^ l32) * 16)) = o;
      }
  }
  __syncthreads();
  const bool split = nkt > chunk;
  const long RT = (long)per * R;
  for (int t = tid; t < R * (D / 4); t += 256) {
    const int r = t / (D / 4), c = t % (D / 4);
    const int at = r * D * 4 + ((c ^ r) * 16);
    const f32x4 o0 = *reinterpret_cast<const f32x4*>(ks + at);
    const f32x4 o1 = *reinterpret_cast<const f32x4*>(ks + IMG + at);
    const f32x4 o2 = *reinterpret_cast<const f32x4*>(vs + at);
    const f32x4 o3 = *reinterpret_cast<const f32x4*>(vs + IMG + at);
    const f32x4 o = ((o0 + o1) + o2) + o3;
    const float l = ((wl[0][r] + wl[1][r]) + wl[2][r]) + wl[3][r];
    if (split) {
      const long pr = (long)sp * RT + (long)hb * R + r;
      *reinterpret_cast<f32x4*>(part + pr * D + 4 * c) = o;
      if (c == 0) {
        part_ml[pr * 2] = fmaxf(fmaxf(wm[0][r], wm[1][r]), fmaxf(wm[2][r], wm[3][r]));
        part_ml[pr * 2 + 1] = l;
      }
      continue;
    }
    const float inv = l > 0.f ? 1.f / l : 0.f;
    const int h = hk * G + r % G, i = r / G;
    f16x4 y;
    y[0] = (_Float16)(o[0] * inv);
    y[1] = (_Float16)(o[1] * inv);
    y[2] = (_Float16)(o[2] * inv);
    y[3] = (_Float16)(o[3] * inv);
    *reinterpret_cast<f16x4*>(O + b * o_sb + (long)i * o_ss + (long)h * o_sh + 4 * c) = y;
    if (LSE && c == 0) {
      const float mr = fmaxf(fmaxf(wm[0][r], wm[1][r]), fmaxf(wm[2][r], wm[3][r]));
      LSE[((long)b * H + h) * Sq + i] =
          l > 0.f ? mr * 0.6931471805599453f + __logf(l) : -__builtin_inff();
    }
  }
}

// k_fmha_combine -- merges the key ranges of one packed row: one wave per row, lane l holds D / 64
// consecutive d.  With references m_s, sums l_s and unnormalised O_s: O = sum 2^(m_s - m) O_s /
// sum 2^(m_s - m) l_s, m = max m_s, in range order.  Rows of a tile that one workgroup finished
// alone (at most `chunk` key blocks) are skipped: their O is already written.  At most 64 ranges.
// Bound by its launch and by the partial results' bytes (2 x ranges x rows x D x 4 at ~4.5 TB/s).
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256) void k_fmha_combine(const float* __restrict__ part,
                                                      const float* __restrict__ part_ml,
                                                      _Float16* __restrict__ O,
                                                      float* __restrict__ LSE, int B, int H,
                                                      int Hkv, int Sq, int Sk, int rows, int chunk,
                                                      long o_sb, long o_ss, long o_sh) {
  constexpr int E = D / 64;
  typedef float fe __attribute__((ext_vector_type(E)));
  typedef _Float16 he __attribute__((ext_vector_type(E)));
  const int lane = threadIdx.x & 63;
  const int G = H / Hkv, R = Sq * G;
  const long RT = (long)B * Hkv * R;
  const long row = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (row >= RT) return;
  const int r = (int)(row % R), hb = (int)(row / R);
  const int nkt = fmha_tile_blocks<CAUSAL>(r / rows * rows, rows, R, G, Sq, Sk);
  if (nkt <= chunk) return;
  const int n = (nkt + chunk - 1) / chunk;
  float ml = -__builtin_inff(), ll = 0.f;  // lane s: range s
  if (lane < n) {
    ml = part_ml[(lane * RT + row) * 2];
    ll = part_ml[(lane * RT + row) * 2 + 1];
  }
  float m = ml;
#pragma unroll
  for (int x = 32; x > 0; x >>= 1) m = fmaxf(m, __shfl_xor(m, x));
  const float w = __builtin_amdgcn_exp2f(ml - ((m == -__builtin_inff()) ? 0.f : m));
  const float* p = part + row * D + lane * E;
  fe o;
#pragma unroll
  for (int e = 0; e < E; ++e) o[e] = 0.f;
  float l = 0.f;
  constexpr int U = 8;  // ranges in flight
  for (int s = 0; s < n; s += U) {
    fe v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)
      v[u] = *reinterpret_cast<const fe*>(p + (long)min(s + u, n - 1) * RT * D);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= n) break;
      const float ws = __shfl(w, s + u);
      l += ws * __shfl(ll, s + u);
#pragma unroll
      for (int e = 0; e < E; ++e) o[e] += ws * v[u][e];
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int hk = hb % Hkv, b = hb / Hkv, i = r / G, h = hk * G + r % G;
  he y;
#pragma unroll
  for (int e = 0; e < E; ++e) y[e] = (_Float16)(o[e] * inv);
  *reinterpret_cast<he*>(O + b * o_sb + (long)i * o_ss + (long)h * o_sh + lane * E) = y;
  if (LSE && lane == 0)
    LSE[((long)b * H + h) * Sq + i] =
        l > 0.f ? m * 0.6931471805599453f + __logf(l) : -__builtin_inff();
}

}  // namespace fmha
