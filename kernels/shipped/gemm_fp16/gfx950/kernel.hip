// kernel.hip -- FROZEN copy of the gfx950 skeletons for the gemm_fp16 delivery.
// Generated by tempo/plugins/gfx950/ship.py from: common/cdna4.h, gemm_mfma/kernel.hip, gemm_mfma/ilv.hip, gemv_stream/kernel.hip, common/splitk_host.h.
// Do not edit: change the skeleton, then re-run the freeze step.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace tempo {
namespace gen {

// ===== common/cdna4.h =====
// cdna4.h -- device vocabulary shared by the gfx950 skeletons (CDNA4, wave64, MFMA).
//
// The skeleton sources carry no namespace of their own: the freeze step that writes a shipped
// kernel file (kernels/shipped/<op>/gfx950/kernel.hip) and the plugin's render() wrap them in
// the op's namespace, so two shipped ops linked into one library never share a symbol.
//
// MFMA lane maps used below (wave64):
//   32x32x16 f16: operand lane l carries row (l % 32) and the 8 k-values of k-group (l / 32);
//                 result lane l carries column (l % 32), rows 8*(v/4) + 4*(l/32) + (v%4), v<16.
//   16x16x32 f16: operand lane l carries row (l % 16) and the 8 k-values of k-group (l / 16);
//                 result lane l carries column (l % 16), rows 4*(l/16) + v, v<4.
// The k-group -> k assignment only has to be the same for both operands (a sum over k does not
// care about its order), so the skeletons may permute k freely as long as A and B agree.  The
// row/column maps of the result are what the epilogue depends on; the plugin's tensor section
// declares them and an on-GPU bijection probe checks them.

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// compile-time integer tag (lets a generic lambda take a constant register-buffer index)
template <int V>
struct IC {
  static constexpr int value = V;
};

template <int MS>
struct Mfma;

template <>
struct Mfma<32> {
  typedef f32x16 acc_t;
  static constexpr int KSTEP = 16;  // k per instruction
  static constexpr int NACC = 16;   // result floats per lane
  static constexpr int GROUPS = 4;  // result row groups of 4 consecutive rows
  static constexpr int GROUP_STRIDE = 8;
  __device__ __forceinline__ static acc_t run(const f16x8& a, const f16x8& b, const acc_t& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

template <>
struct Mfma<16> {
  typedef f32x4 acc_t;
  static constexpr int KSTEP = 32;
  static constexpr int NACC = 4;
  static constexpr int GROUPS = 1;
  static constexpr int GROUP_STRIDE = 16;
  __device__ __forceinline__ static acc_t run(const f16x8& a, const f16x8& b, const acc_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Result row of value v for lane l (see the map above).
template <int MS>
__device__ __forceinline__ int mfma_out_row(int lane, int g, int e) {
  return g * Mfma<MS>::GROUP_STRIDE + 4 * (lane / MS) + e;
}

// ------------------------------------------------------------------------------------------
// Bit-exact dequantisation in registers.
//
// Weight formats (op-level "fmt"):
//   1  int8, symmetric, one fp16 scale per output channel:   W = fp16_rn(q * s)
//   2  uint8, asymmetric, fp16 scale + uint8 zero-point per (row, 128-group): W = fp16_rn((q-z)*s)
//
// The integer q (or q - z) is built as an fp16 without rounding: the bit pattern 0x64XX is the
// fp16 value 1024 + XX for a byte XX, and subtracting 1024 + z (also exact) leaves q - z exactly
// (|q - z| <= 255 < 2048, where fp16 spacing is 1).  The scale multiply is one IEEE fp16 multiply,
// which is correctly rounded (RNE) -- and since q*s is exact in fp32 (8 x 11 significant bits),
// fp16_rn(fp16 q * fp16 s) == fp16_rn(float(q) * float(s)), the closed form of the formats.
// No q*s - z*s folding: that would round twice.
// ------------------------------------------------------------------------------------------

// Four bytes of w -> four fp16 values 1024 + byte, as two packed halves pairs.
__device__ __forceinline__ void bytes_to_magic(uint32_t w, uint32_t& lo, uint32_t& hi) {
  // v_perm_b32 selector: bytes 0..3 come from the second operand (w), 4..7 from the first.
  lo = __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u);  // [b1 | 0x64, b0 | 0x64] -> halves
  hi = __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u);
}

__device__ __forceinline__ f16x2 as_h2(uint32_t u) { return __builtin_bit_cast(f16x2, u); }
__device__ __forceinline__ uint32_t as_u32(f16x2 h) { return __builtin_bit_cast(uint32_t, h); }

// 8 weight bytes (two dwords) -> 8 dequantised fp16 values.  `bias` is 1024 + zero-point
// (uint8 formats) or 1152 (int8 after the sign flip), `s` the fp16 scale, both broadcast.
__device__ __forceinline__ f16x8 dequant8(uint32_t w0, uint32_t w1, _Float16 bias, _Float16 s) {
  uint32_t p0, p1, p2, p3;
  bytes_to_magic(w0, p0, p1);
  bytes_to_magic(w1, p2, p3);
  const f16x2 b2 = {bias, bias};
  const f16x2 s2 = {s, s};
  const f16x2 d0 = (as_h2(p0) - b2) * s2;
  const f16x2 d1 = (as_h2(p1) - b2) * s2;
  const f16x2 d2 = (as_h2(p2) - b2) * s2;
  const f16x2 d3 = (as_h2(p3) - b2) * s2;
  f16x8 r;
  r[0] = d0[0]; r[1] = d0[1]; r[2] = d1[0]; r[3] = d1[1];
  r[4] = d2[0]; r[5] = d2[1]; r[6] = d3[0]; r[7] = d3[1];
  return r;
}

// int8 (two's complement) bytes: flip the sign bit so byte = q + 128, then bias = 1152.
__device__ __forceinline__ f16x8 dequant8_i8(uint32_t w0, uint32_t w1, _Float16 s) {
  return dequant8(w0 ^ 0x80808080u, w1 ^ 0x80808080u, (_Float16)1152.0f, s);
}

__device__ __forceinline__ f16x8 dequant8_u8(uint32_t w0, uint32_t w1, uint8_t z, _Float16 s) {
  return dequant8(w0, w1, (_Float16)(1024.0f + (float)z), s);
}

// The lane index recomputed from the exec-mask bit count (mbcnt), for epilogues: a value derived
// from threadIdx.x and kept across a register-full main loop gets spilled; this one is rebuilt
// where it is needed.
__device__ __forceinline__ int lane_id() {
  return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
}

__device__ __forceinline__ f16x8 as_f16x8(const u32x4& u) { return __builtin_bit_cast(f16x8, u); }
__device__ __forceinline__ u32x4 as_u32x4(const f16x8& h) { return __builtin_bit_cast(u32x4, h); }

// Fused gate/up epilogue: silu(g) * u on the fp16-rounded GEMM results, i.e. exactly what the
// unfused chain (two fp16 GEMM outputs, then silu and a product) sees, in fp32, one rounding to
// fp16 at the end.  silu(x) = x / (1 + e^-x); e^-x by the hardware exponential.
__device__ __forceinline__ _Float16 silu_mul_f16(float g, float u) {
  const float gh = (float)(_Float16)g;
  const float uh = (float)(_Float16)u;
  return (_Float16)(gh / (1.0f + __expf(-gh)) * uh);
}

// ===== gemm_mfma/kernel.hip =====
// gemm_mfma -- tiled C[M,N] = A[M,K] . B[N,K]^T on CDNA4 matrix cores (gfx950).
//
// Semantics follow the reference's naive kernel (kernels/naive/gemm_fp16.cu:60-68): fp16
// operands, fp32 accumulation, one RNE rounding to fp16 per output.  The order of the k
// summation differs (MFMA dot products), which is why parity is a relL2 gate, not bit equality.
//
// Template axes (the plugin's search space, tempo/plugins/gfx950/space.py):
//   BM, BN   macro tile of C per workgroup
//   BK       k extent of one LDS stage (the LDS holds two stages: double buffer)
//   WM, WN   waves along M and N (workgroup = WM*WN*64 lanes); wave tile (BM/WM) x (BN/WN)
//   MS       MFMA shape: 32 -> v_mfma_f32_32x32x16_f16, 16 -> v_mfma_f32_16x16x32_f16
//   SWZ      LDS chunk swizzle: 0 none, 1 chunk ^ (row % CPR), 2 chunk ^ ((row/2) % CPR)
//   GROUP    raster group height in tiles (L2 reuse); 0 = row-major tile order
//   XCD      1 = remap block ids so each of the 8 XCDs owns a contiguous run of tiles
//   BFMT     B operand format: 0 fp16, 1 int8 + per-row fp16 scale, 2 uint8 + per-(row,group)
//            fp16 scale and uint8 zero-point.  Formats 1 and 2 dequantise while staging the
//            B tile into LDS (once per workgroup, not once per wave), bit-exact with the
//            closed forms in cdna4.h.
//
// Layout in registers: the MFMA "A" operand is fed from B rows (n) and the "B" operand from A
// rows (m), so each lane's result values are 4 consecutive n of one m -- the epilogue writes
// 8-byte runs of C instead of 2-byte scatters.
//
// LDS layout: per stage, A tile [BM][BK] and B tile [BN][BK] fp16, k contiguous, 16-byte chunks
// swizzled by row so the 16-byte MFMA feed reads (one row per lane) spread over the banks.
//
// Requirements checked by the launcher (applicable()): N % BN == 0, K % BK == 0, 16-byte
// aligned rows; M is predicated (rows past M are loaded from row M-1 and never stored).

// LDS chunk swizzle: the 16-byte chunk c of tile row `row` is stored at chunk c ^ f(row).
// SWZ 1: f = (row / rows-per-128B) % CPR -- spreads 8 consecutive rows over 32 banks.
// SWZ 2: f = (row / rows-per-256B) % CPR -- spreads 16 consecutive rows over 64 banks.
template <int BK, int SWZ>
__device__ __forceinline__ int lds_chunk(int row, int chunk) {
  constexpr int CPR = BK / 8;  // 16-byte chunks per row
  constexpr int ROW_BYTES = BK * 2;
  if constexpr (SWZ == 1) {
    constexpr int R128 = ROW_BYTES >= 128 ? 1 : 128 / ROW_BYTES;
    return chunk ^ ((row / R128) & (CPR - 1));
  } else if constexpr (SWZ == 2) {
    constexpr int R256 = ROW_BYTES >= 256 ? 1 : 256 / ROW_BYTES;
    return chunk ^ ((row / R256) & (CPR - 1));
  } else {
    return chunk;
  }
}

// Tile order: block id -> (tile_m, tile_n).
template <int GROUP, int XCD>
__device__ __forceinline__ void tile_of(int bid, int nm, int nn, int& tm, int& tn) {
  const int total = nm * nn;
  if constexpr (XCD) {
    // Workgroups are handed to the 8 XCDs round-robin (bid % 8).  Give XCD x the contiguous
    // run [x*total/8, (x+1)*total/8) of the tile order so its concurrent tiles share panels in
    // that XCD's own L2.
    if ((total & 7) == 0) bid = (bid & 7) * (total >> 3) + (bid >> 3);
  }
  if constexpr (GROUP > 0) {
    const int per = GROUP * nn;
    const int g = bid / per;
    const int first = g * GROUP;
    const int gs = min(GROUP, nm - first);
    const int r = bid - g * per;
    tm = first + r % gs;
    tn = r / gs;
  } else {
    tm = bid / nn;
    tn = bid - tm * nn;
  }
}

// Split-K tile order: block id -> (tile_m, tile_n, split).  The XCD remap runs over all
// tiles x ksplit workgroups, then the order is split-major: the workgroups an XCD holds at once
// share k ranges, i.e. the same activation panel slices, in that XCD's L2.
template <int GROUP, int XCD>
__device__ __forceinline__ void split_tile_of(int bid, int nm, int nn, int ksplit, int& tm, int& tn,
                                              int& sk) {
  const int tiles = nm * nn;
  if constexpr (XCD) {
    const int total = tiles * ksplit;
    if ((total & 7) == 0) bid = (bid & 7) * (total >> 3) + (bid >> 3);
  }
  sk = bid / tiles;
  tile_of<GROUP, 0>(bid - sk * tiles, nm, nn, tm, tn);
}

// acc += src[0], src[per], ... src[(U - 1) per], in that order, all loaded first.
template <int U>
__device__ __forceinline__ void add_splits(f32x4& acc, const float* src, long per) {
  f32x4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const f32x4*>(src + u * per);
#pragma unroll
  for (int u = 0; u < U; ++u) acc += v[u];
}

// Split-K reduction: C[m][n] = fp16_rn(ws[0][m][n] + ws[1][m][n] + ... + ws[S-1][m][n]), the
// partial sums added in the fixed order s = 0 .. S-1 in fp32 (deterministic), one rounding to
// fp16.  ws is [S][M][N] fp32 (rows of N), N % 4 == 0; each thread takes 4 consecutive n.  A pure
// streaming read bound by its latency: the loads of UNROLL <= S splits are all issued before their
// adds, and the host takes UNROLL = S up to 8, so that no split's load waits for another's; past 8
// they go in eights, then four, two, one of what remains (us, the whole call, eights whose
// last one re-reads the last split -> this: (64, 3584, 11008) uint8, 9 splits, 23.1 -> 22.5; (48,
// 512, 13824) fp16, 27 splits, 11.0 -> 10.2).
// (A template so that every translation unit that includes this file may instantiate it.)
template <int UNROLL = 8>
__global__ __launch_bounds__(256) void k_splitk_reduce(const float* __restrict__ ws, int S, int M,
                                                       int N, _Float16* __restrict__ C, int ldc) {
  const long per = (long)M * N;
  const long i4 = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i4 >= per) return;
  const int m = (int)(i4 / N), n = (int)(i4 - (long)m * N);
  const float* src = ws + i4;
  f32x4 v[UNROLL];
#pragma unroll
  for (int u = 0; u < UNROLL; ++u) v[u] = *reinterpret_cast<const f32x4*>(src + u * per);
  f32x4 acc = v[0];
#pragma unroll
  for (int u = 1; u < UNROLL; ++u) acc += v[u];
  if constexpr (UNROLL == 8) {  // S > 8
    int s = 8;
    for (; s + 8 <= S; s += 8) add_splits<8>(acc, src + s * per, per);
    if ((S - s) & 4) {
      add_splits<4>(acc, src + s * per, per);
      s += 4;
    }
    if ((S - s) & 2) {
      add_splits<2>(acc, src + s * per, per);
      s += 2;
    }
    if ((S - s) & 1) add_splits<1>(acc, src + s * per, per);
  }
  f16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (_Float16)acc[e];
  *reinterpret_cast<f16x4*>(C + (long)m * ldc + n) = o;
}

// Split-K reduction of the fused gate/up product: ws is [S][M][2N] fp32, gate columns then up
// columns; C[m][n] = fp16_rn(silu(g) * u) of the two sums rounded to fp16, each added in split
// order as above (the tiles' own epilogue sees the same rounded pair).
template <int UNROLL>
__global__ __launch_bounds__(256) void k_splitk_reduce_gu(const float* __restrict__ ws, int S,
                                                          int M, int N, _Float16* __restrict__ C,
                                                          int ldc) {
  const long per = 2 * (long)M * N;
  const long i4 = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i4 >= (long)M * N) return;
  const int m = (int)(i4 / N), n = (int)(i4 - (long)m * N);
  const float* src = ws + (long)m * 2 * N + n;
  f32x4 g, u;
  for (int s = 0; s < S; s += UNROLL) {
    f32x4 vg[UNROLL], vu[UNROLL];
#pragma unroll
    for (int x = 0; x < UNROLL; ++x) {
      const float* p = src + min(s + x, S - 1) * per;
      vg[x] = *reinterpret_cast<const f32x4*>(p);
      vu[x] = *reinterpret_cast<const f32x4*>(p + N);
    }
#pragma unroll
    for (int x = 0; x < UNROLL; ++x)
      if (s + x == 0) {
        g = vg[0];
        u = vu[0];
      } else if (s + x < S) {
        g += vg[x];
        u += vu[x];
      }
  }
  f16x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = silu_mul_f16(g[e], u[e]);
  *reinterpret_cast<f16x4*>(C + (long)m * ldc + n) = o;
}

template <int BM, int BN, int BK, int WM, int WN, int MS, int SWZ, int GROUP, int XCD, int BFMT>
struct GemmCfg {
  static constexpr int THREADS = WM * WN * 64;
  static constexpr int CPR = BK / 8;
  static constexpr int WTM = BM / WM;  // wave tile rows (m)
  static constexpr int WTN = BN / WN;  // wave tile cols (n)
  static constexpr int TM = WTM / MS;  // MFMA blocks per wave along m
  static constexpr int TN = WTN / MS;
  static constexpr int KS = BK / Mfma<MS>::KSTEP;  // MFMA k-steps per stage
  static constexpr int A_IT = BM * CPR / THREADS;  // 16-byte A chunks per thread per stage
  static constexpr int B_IT = BN * CPR / THREADS;
  static constexpr int LDS_BYTES = 2 * (BM + BN) * BK * 2;
  static_assert(BK % Mfma<MS>::KSTEP == 0, "BK must hold whole MFMA k-steps");
  static_assert(WTM % MS == 0 && WTN % MS == 0, "wave tile must hold whole MFMA blocks");
  static_assert((BM * CPR) % THREADS == 0 && (BN * CPR) % THREADS == 0, "tile/thread split");
  static_assert(CPR == 4 || CPR == 8, "BK of 32 or 64");
};

// Raw B chunk as loaded from global memory: 16 bytes of fp16, or 8 bytes of int8/uint8.
template <int BFMT>
struct BRaw;
template <>
struct BRaw<0> { u32x4 v; };
template <>
struct BRaw<1> { u32x2 v; };
template <>
struct BRaw<2> { u32x2 v; };

template <int BM, int BN, int BK, int WM, int WN, int MS, int SWZ, int GROUP, int XCD, int BFMT>
__global__ __launch_bounds__(WM * WN * 64, 1) void k_gemm(
    const _Float16* __restrict__ A, const void* __restrict__ Bv,
    const _Float16* __restrict__ scale, const uint8_t* __restrict__ zero,
    _Float16* __restrict__ C, int M, int N, int K, int lda, int ldb, int ldc, int group) {
  using Cfg = GemmCfg<BM, BN, BK, WM, WN, MS, SWZ, GROUP, XCD, BFMT>;
  using MF = Mfma<MS>;
  constexpr int T = Cfg::THREADS, CPR = Cfg::CPR;
  constexpr int TM = Cfg::TM, TN = Cfg::TN;

  __shared__ __attribute__((aligned(16))) _Float16 smem[2 * (BM + BN) * BK];
  _Float16* const sA = smem;                 // [2][BM][BK]
  _Float16* const sB = smem + 2 * BM * BK;   // [2][BN][BK]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / WN, wn = wave % WN;

  const int nm = (M + BM - 1) / BM, nn = N / BN;
  int tmi, tni;
  tile_of<GROUP, XCD>(blockIdx.x, nm, nn, tmi, tni);
  const int m0 = tmi * BM, n0 = tni * BN;

  // ---- global -> register staging -------------------------------------------------------
  const u32x4* gA[Cfg::A_IT];
  int sAoff[Cfg::A_IT];
#pragma unroll
  for (int i = 0; i < Cfg::A_IT; ++i) {
    const int q = tid + i * T, r = q / CPR, c = q % CPR;
    const int gm = min(m0 + r, M - 1);
    gA[i] = reinterpret_cast<const u32x4*>(A + (long)gm * lda + c * 8);
    sAoff[i] = r * BK + lds_chunk<BK, SWZ>(r, c) * 8;
  }
  int sBoff[Cfg::B_IT];
  long gBoff[Cfg::B_IT];  // element offset of the chunk's row start + k
  int bRow[Cfg::B_IT], bC[Cfg::B_IT];
#pragma unroll
  for (int i = 0; i < Cfg::B_IT; ++i) {
    const int q = tid + i * T, r = q / CPR, c = q % CPR;
    bRow[i] = n0 + r;
    bC[i] = c;
    gBoff[i] = (long)(n0 + r) * ldb + c * 8;
    sBoff[i] = r * BK + lds_chunk<BK, SWZ>(r, c) * 8;
  }
  _Float16 rowScale[Cfg::B_IT];
  if constexpr (BFMT == 1) {
#pragma unroll
    for (int i = 0; i < Cfg::B_IT; ++i) rowScale[i] = scale[bRow[i]];
  }

  u32x4 ra[Cfg::A_IT];
  BRaw<BFMT> rb[Cfg::B_IT];

  auto load_stage = [&](int k0) {
#pragma unroll
    for (int i = 0; i < Cfg::A_IT; ++i) ra[i] = gA[i][k0 / 8];
#pragma unroll
    for (int i = 0; i < Cfg::B_IT; ++i) {
      if constexpr (BFMT == 0)
        rb[i].v = *reinterpret_cast<const u32x4*>(
            reinterpret_cast<const _Float16*>(Bv) + gBoff[i] + k0);
      else
        rb[i].v = *reinterpret_cast<const u32x2*>(
            reinterpret_cast<const uint8_t*>(Bv) + gBoff[i] + k0);
    }
  };
  auto store_stage = [&](int buf, int k0) {
    _Float16* a = sA + buf * BM * BK;
    _Float16* b = sB + buf * BN * BK;
#pragma unroll
    for (int i = 0; i < Cfg::A_IT; ++i) *reinterpret_cast<u32x4*>(a + sAoff[i]) = ra[i];
#pragma unroll
    for (int i = 0; i < Cfg::B_IT; ++i) {
      u32x4 v;
      if constexpr (BFMT == 0) {
        v = rb[i].v;
      } else if constexpr (BFMT == 1) {
        v = as_u32x4(dequant8_i8(rb[i].v[0], rb[i].v[1], rowScale[i]));
      } else {
        const int k = k0 + bC[i] * 8;
        const long gi = (long)bRow[i] * (K / group) + k / group;
        v = as_u32x4(dequant8_u8(rb[i].v[0], rb[i].v[1], zero[gi], scale[gi]));
      }
      *reinterpret_cast<u32x4*>(b + sBoff[i]) = v;
    }
  };

  typename MF::acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < MF::NACC; ++v) acc[i][j][v] = 0.f;

  // fragment read offsets (row part) inside one stage
  const int fr = lane % MS;
  const int fk = lane / MS;  // k-group of this lane
  int aRow[TM], bRowF[TN];
#pragma unroll
  for (int i = 0; i < TM; ++i) aRow[i] = wm * Cfg::WTM + i * MS + fr;
#pragma unroll
  for (int j = 0; j < TN; ++j) bRowF[j] = wn * Cfg::WTN + j * MS + fr;

  const int NT = K / BK;
  load_stage(0);
  store_stage(0, 0);
  __syncthreads();

  for (int kt = 0; kt < NT; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < NT) load_stage((kt + 1) * BK);
    const _Float16* a = sA + cur * BM * BK;
    const _Float16* b = sB + cur * BN * BK;
#pragma unroll
    for (int ks = 0; ks < Cfg::KS; ++ks) {
      const int chunk = ks * (64 / MS) + fk;
      f16x8 fa[TM], fb[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[i] = *reinterpret_cast<const f16x8*>(a + aRow[i] * BK +
                                                lds_chunk<BK, SWZ>(aRow[i], chunk) * 8);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[j] = *reinterpret_cast<const f16x8*>(b + bRowF[j] * BK +
                                                lds_chunk<BK, SWZ>(bRowF[j], chunk) * 8);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = MF::run(fb[j], fa[i], acc[i][j]);
    }
    if (kt + 1 < NT) store_stage(cur ^ 1, (kt + 1) * BK);
    __syncthreads();
  }

  // ---- epilogue: each lane owns 4 consecutive n of one m per result group ----------------
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + wm * Cfg::WTM + i * MS + (lane % MS);
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int g = 0; g < MF::GROUPS; ++g) {
        const int n = n0 + wn * Cfg::WTN + j * MS + mfma_out_row<MS>(lane, g, 0);
        f16x4 o;
        o[0] = (_Float16)acc[i][j][4 * g + 0];
        o[1] = (_Float16)acc[i][j][4 * g + 1];
        o[2] = (_Float16)acc[i][j][4 * g + 2];
        o[3] = (_Float16)acc[i][j][4 * g + 3];
        *reinterpret_cast<f16x4*>(C + (long)m * ldc + n) = o;
      }
    }
  }
}

// ============================================================================================
// k_gemm_dma -- fp16 B only.  Same tile, swizzle and epilogue as k_gemm, but the global -> LDS
// copy is the gfx950 LDS-DMA load (global_load_lds_dwordx4): data goes straight from L2 into
// LDS without passing through registers, the copy costs one instruction per 1 KiB per wave, and
// STAGES-1 k-tiles are in flight while one is computed.
//
// One DMA instruction fills a contiguous 1 KiB of LDS, lane l writing bytes [16l, 16l+16).  The
// swizzle is therefore applied on the GLOBAL side: lane l fetches the chunk that belongs at LDS
// slot l.  Waits are explicit (s_waitcnt vmcnt(N) for this wave's own copies, then s_barrier
// for everyone's); the compiler does not order LDS reads after LDS-DMA writes by itself.
// ============================================================================================
typedef __attribute__((address_space(3))) void lds_void_t;

// s_waitcnt vmcnt(N) lgkmcnt(0).  gfx9 encoding: vmcnt[3:0] bits 3:0, expcnt bits 6:4,
// lgkmcnt bits 11:8, vmcnt[5:4] bits 15:14.
template <int N>
__device__ __forceinline__ void s_wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
}

// 16-byte-per-lane buffer load into LDS: lane l's 16 bytes at byte offset voff + soff of the
// raw buffer [base, base + nrec) land at lds + 16 l.  (A helper function rather than inline in
// the kernel's lambdas: inside a lambda of a kernel template the host pass drops the kernel's
// launch stub.)
__device__ __forceinline__ void buf_lds16(const void* base, int nrec, void* lds, int voff, int soff) {
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, nrec, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 16, voff, soff, 0, 0);
}
// The same with 1- or 2-byte lanes (zero-points, scales); such lanes land 4 bytes apart in LDS.
template <int SIZE>
__device__ __forceinline__ void buf_lds_n(const void* base, int nrec, void* lds, int voff, int soff) {
  static_assert(SIZE == 1 || SIZE == 2, "byte or half lanes");
  const __amdgpu_buffer_rsrc_t r =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, nrec, 0x00020000);
  if constexpr (SIZE == 1)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 1, voff, soff, 0, 0);
  else
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)lds, 2, voff, soff, 0, 0);
}

// XT = 1 pipelines across k-tile boundaries: the wait + barrier for tile kt+1, the DMA issue of
// tile kt+STAGES and the first fragment reads of tile kt+1 all happen BEFORE the last MFMA group
// of tile kt, so the matrix cores have work while the workgroup synchronises.  The prologue then
// fills all STAGES buffers.  XT = 0 keeps the plain loop (wait + barrier at the top of a tile).
// MINB = workgroups the compiler must leave room for on one CU (register budget 512 / waves per
// SIMD); 2 lets two small-tile workgroups share a CU, so one computes while the other waits.
// MS = MFMA shape (32: v_mfma_f32_32x32x16_f16, 16: v_mfma_f32_16x16x32_f16).
template <int BM, int BN, int BK, int WM, int WN, int STAGES, int SWZ, int GROUP, int XCD,
          int XT = 0, int MINB = 1, int MS = 32>
__global__ __launch_bounds__(WM * WN * 64, MINB) void k_gemm_dma(
    const _Float16* __restrict__ A, const _Float16* __restrict__ B, _Float16* __restrict__ C,
    int M, int N, int K, int lda, int ldb, int ldc) {
  using MF = Mfma<MS>;
  constexpr int NW = WM * WN;
  constexpr int CPR = BK / 8;
  constexpr int RPB = 1024 / (BK * 2);  // tile rows per 1 KiB DMA block
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / MS, TN = WTN / MS;
  constexpr int KS = BK / MF::KSTEP;
  constexpr int A_BLK = BM / RPB / NW;  // DMA instructions per wave per stage
  constexpr int B_BLK = BN / RPB / NW;
  constexpr int L = A_BLK + B_BLK;
  constexpr int STAGE_ELEMS = (BM + BN) * BK;
  static_assert(BM % (RPB * NW) == 0 && BN % (RPB * NW) == 0, "DMA blocks per wave");
  static_assert(STAGES >= 2 && (STAGES - 2 + XT) * L < 64, "stages / vmcnt range");
  static_assert(WTM % MS == 0 && WTN % MS == 0 && BK % MF::KSTEP == 0, "tile shape");

  __shared__ __attribute__((aligned(1024))) _Float16 smem[STAGES * STAGE_ELEMS];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;

  const int nm = (M + BM - 1) / BM, nn = N / BN;
  int tmi, tni;
  tile_of<GROUP, XCD>(blockIdx.x, nm, nn, tmi, tni);
  const int m0 = tmi * BM, n0 = tni * BN;

  // per-lane global sources: DMA block i of this wave = tile block (i*NW + wave)
  const _Float16* srcA[A_BLK];
  const _Float16* srcB[B_BLK];
  {
    const int rin = lane / CPR, phys = lane % CPR;
#pragma unroll
    for (int i = 0; i < A_BLK; ++i) {
      const int row = (i * NW + wave) * RPB + rin;
      const int c = lds_chunk<BK, SWZ>(row, phys);  // involution: logical chunk of slot `phys`
      srcA[i] = A + (long)min(m0 + row, M - 1) * lda + c * 8;
    }
#pragma unroll
    for (int i = 0; i < B_BLK; ++i) {
      const int row = (i * NW + wave) * RPB + rin;
      const int c = lds_chunk<BK, SWZ>(row, phys);
      srcB[i] = B + (long)(n0 + row) * ldb + c * 8;
    }
  }
  auto issue = [&](int kt) {
    const int st = kt % STAGES;
    _Float16* sa = smem + st * STAGE_ELEMS;
    _Float16* sb = sa + BM * BK;
    const int k0 = kt * BK;
#pragma unroll
    for (int i = 0; i < A_BLK; ++i)
      __builtin_amdgcn_global_load_lds((void*)(srcA[i] + k0),
                                       (lds_void_t*)(sa + (i * NW + wave) * RPB * BK), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < B_BLK; ++i)
      __builtin_amdgcn_global_load_lds((void*)(srcB[i] + k0),
                                       (lds_void_t*)(sb + (i * NW + wave) * RPB * BK), 16, 0, 0);
  };

  typename MF::acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < MF::NACC; ++v) acc[i][j][v] = 0.f;

  const int fr = lane % MS, fk = lane / MS;
  int aOff[TM], bOff[TN];  // row offsets (elements) of this lane's fragment rows
#pragma unroll
  for (int i = 0; i < TM; ++i) aOff[i] = (wm * WTM + i * MS + fr);
#pragma unroll
  for (int j = 0; j < TN; ++j) bOff[j] = (wn * WTN + j * MS + fr);

  const int NT = K / BK;
  if constexpr (XT) {
    f16x8 fa[2][TM], fb[2][TN];
    auto read = [&](auto bufc, const _Float16* a, int ks) {
      constexpr int bb = decltype(bufc)::value;
      const _Float16* b = a + BM * BK;
      const int chunk = ks * (64 / MS) + fk;
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[bb][i] = *reinterpret_cast<const f16x8*>(a + aOff[i] * BK +
                                                    lds_chunk<BK, SWZ>(aOff[i], chunk) * 8);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[bb][j] = *reinterpret_cast<const f16x8*>(b + bOff[j] * BK +
                                                    lds_chunk<BK, SWZ>(bOff[j], chunk) * 8);
    };
    auto mma = [&](auto bufc) {
      constexpr int bb = decltype(bufc)::value;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = MF::run(fb[bb][j], fa[bb][i], acc[i][j]);
    };
    static_assert(KS % 2 == 0, "fragment buffers alternate; a tile holds an even k-step count");
    // prologue: every buffer gets a tile; wait for tile 0 (tiles 1..STAGES-1 stay in flight)
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < NT) issue(s);
    asm volatile("" ::: "memory");
    if (NT >= STAGES) s_wait_vm<(STAGES - 1) * L>();
    else s_wait_vm<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(IC<0>{}, smem, 0);
    __builtin_amdgcn_sched_barrier(0);
    for (int kt = 0; kt < NT; ++kt) {
      const _Float16* a = smem + (kt % STAGES) * STAGE_ELEMS;
#pragma unroll
      for (int ks = 0; ks < KS - 2; ks += 2) {
        read(IC<1>{}, a, ks + 1);
        mma(IC<0>{});
        __builtin_amdgcn_sched_barrier(0);
        read(IC<0>{}, a, ks + 2);
        mma(IC<1>{});
        __builtin_amdgcn_sched_barrier(0);
      }
      read(IC<1>{}, a, KS - 1);
      mma(IC<0>{});
      __builtin_amdgcn_sched_barrier(0);
      if (kt + 1 < NT) {
        // Tile kt+1 has landed for this wave (tiles up to kt+STAGES-1 may still be in flight)
        // and this wave's reads of tile kt are complete (lgkmcnt 0) ...
        asm volatile("" ::: "memory");
        if (kt + STAGES < NT) s_wait_vm<(STAGES - 2) * L>();
        else s_wait_vm<0>();
        // ... and everyone's: tile kt+1 is readable and buffer kt % STAGES is free.
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (kt + STAGES < NT) issue(kt + STAGES);
        read(IC<0>{}, smem + ((kt + 1) % STAGES) * STAGE_ELEMS, 0);
      }
      mma(IC<1>{});
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < NT) issue(s);

  for (int kt = 0; kt < NT; ++kt) {
    // this wave's copies of tile kt have landed (later tiles may still be in flight) ...
    asm volatile("" ::: "memory");  // compiler-only fence: no LDS access crosses the barrier
    if (kt + STAGES - 2 < NT) s_wait_vm<(STAGES - 2) * L>();
    else s_wait_vm<0>();
    // ... and everyone's have; everyone is also done reading the buffer about to be refilled
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (kt + STAGES - 1 < NT) issue(kt + STAGES - 1);

    const _Float16* a = smem + (kt % STAGES) * STAGE_ELEMS;
    const _Float16* b = a + BM * BK;
    f16x8 fa[2][TM], fb[2][TN];
    auto read = [&](auto bufc, int ks) {
      constexpr int bb = decltype(bufc)::value;
      const int chunk = ks * (64 / MS) + fk;
#pragma unroll
      for (int i = 0; i < TM; ++i)
        fa[bb][i] = *reinterpret_cast<const f16x8*>(a + aOff[i] * BK +
                                                    lds_chunk<BK, SWZ>(aOff[i], chunk) * 8);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[bb][j] = *reinterpret_cast<const f16x8*>(b + bOff[j] * BK +
                                                    lds_chunk<BK, SWZ>(bOff[j], chunk) * 8);
    };
    auto mma = [&](auto bufc) {
      constexpr int bb = decltype(bufc)::value;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = MF::run(fb[bb][j], fa[bb][i], acc[i][j]);
    };
    // Fragment double buffer: the reads of step ks+1 are issued before the 16 MFMAs of step ks
    // and the scheduler is not allowed to sink them (sched_barrier), so LDS latency hides
    // under the matrix-core work instead of stalling every few MFMAs.
    read(IC<0>{}, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ks += 2) {
      if (ks + 1 < KS) read(IC<1>{}, ks + 1);
      mma(IC<0>{});
      __builtin_amdgcn_sched_barrier(0);
      if (ks + 2 < KS) read(IC<0>{}, ks + 2);
      if (ks + 1 < KS) mma(IC<1>{});
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  }

  // ---- epilogue: each lane owns 4 consecutive n of one m per result group ----------------
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + wm * WTM + i * MS + (lane % MS);
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
#pragma unroll
      for (int g = 0; g < MF::GROUPS; ++g) {
        const int n = n0 + wn * WTN + j * MS + mfma_out_row<MS>(lane, g, 0);
        f16x4 o;
        o[0] = (_Float16)acc[i][j][4 * g + 0];
        o[1] = (_Float16)acc[i][j][4 * g + 1];
        o[2] = (_Float16)acc[i][j][4 * g + 2];
        o[3] = (_Float16)acc[i][j][4 * g + 3];
        *reinterpret_cast<f16x4*>(C + (long)m * ldc + n) = o;
      }
    }
  }
}

// ===== gemm_mfma/ilv.hip =====
// gemm_mfma/ilv.hip -- the interleaved prefill GEMM (fp16 x fp16).  Uses the tile machinery of
// gemm_mfma/kernel.hip (lds_chunk, tile_of, s_wait_vm, buf_lds16), which must come first.
// ============================================================================================
// k_gemm_ilv -- fp16 B only, prefill: one wave per SIMD, large wave tiles, and a main loop that
// is software-pipelined by hand ("interleaved").
//
// Each wave owns a (BM/WM) x (BN/WN) tile of C (128 x 128 for the shipped 256 x 256 / 4-wave
// row: 256 fp32 accumulators per lane, all in AGPRs), so every fragment byte read from LDS feeds
// twice the MFMAs it does in a 64 x 64 wave tile: LDS traffic per flop is halved, which is what
// the power-limited matrix cores of this part spend their budget on besides the MFMAs.
//
// Substep = 32 k (one v_mfma_f32_16x16x32_f16 per 16 x 16 block of the wave tile).  A substep
// issues its TM*TN MFMAs on the fragments read during the previous substep, and between them
// (in CH chunks fenced by sched_barrier) the LDS reads of the next substep's fragments -- in the
// first RSP chunks, so they have landed long before they are needed -- and, in the substep that
// holds the tile barrier, the LDS-DMA copies that refill the stage the barrier has just freed.
// One barrier per k-tile; no MFMA ever waits on an LDS read issued in the same substep.
//
// Stage of tile t = t % STAGES.  The barrier of tile t (in its last substep) is passed once
// every wave has finished reading tile t (lgkmcnt 0) and its own copies of tile t+1 have landed
// (vmcnt); after it tile t+1 is readable by all and stage t % STAGES is refilled with tile
// t + STAGES.  Past the last tile the refill re-copies tile NT-1 into a stage nobody reads again
// and the last substep reads fragments it does not use: the loop body stays one straight-line
// region, so the interleave holds from the first tile to the last.  Those copies are younger
// than every copy a later wait counts, so the vmcnt arithmetic is unchanged, and the kernel
// drains them (vmcnt 0) before the epilogue, so no copy lands after the workgroup has left.
//
// Copies are buffer loads with an LDS destination (buffer_load_dwordx4 ... lds): the resource
// descriptor (SGPRs) points at this tile's A or B panel, each copy's per-lane byte offset is a
// loop constant and the k offset goes in the scalar offset, so a copy costs no vector address
// arithmetic (the 64-bit per-copy address adds of the global form took VALU issue slots next to
// the MFMAs).
//
// Epilogue: where the C tile fits the stages (and a C row is a power of two of at least 256
// bytes), it goes through LDS (free by then) -- fp16 values written in the MFMA layout into a
// row-major image whose 16-byte chunks are XOR-swizzled by row, read back as whole rows and
// written out with 16-byte nontemporal stores, eight lanes per 128-byte line.  Stored straight
// from the MFMA layout, each row gets 32-byte pieces per instruction, and those partial-line
// writes took twice as long (8 us against 4 us per 256 x 256 tile).
//
// Requirements (applicable() + the ladder): N % BN == 0, K % 64 == 0 (an even number of
// substeps), 16-byte aligned rows of A and B, C and ldc 8-byte aligned, panel byte offsets below
// 2^31 (BM*lda*2, BN*ldb*2).  M is predicated: A rows past M-1 are re-read from row M-1 and
// never stored.
//
// SPLIT = 1 (split-K): the grid is tiles x ksplit workgroups (split_tile_of); workgroup split sk
// takes the k-tiles [sk*kper, min((sk+1)*kper, K/BK)), kper = ceil((K/BK) / ksplit) -- the host
// picks ksplit so that no split is empty -- and writes its fp32 partial tile straight from the
// accumulators to ws[sk][M][N] (16 bytes per lane and block); k_splitk_reduce then adds the
// splits in order and rounds once.  Narrow-N, long-K shapes get enough workgroups this way.
//
// EPI = 1 (fused gate/up, prefill): C[M][N] = silu(A.B[0..N)^T) * (A.B[N..2N)^T), B holding the
// gate rows then the up rows (2N rows, N the output width).  A workgroup covers BN/2 output
// columns: its B tile is BN/2 gate rows followed by the BN/2 matching up rows (two panels, the
// copy blocks of each half a compile-time set), so the gate and up results of one output sit
// in the same C tile image in LDS, BN/2 columns apart; the epilogue reads both halves back and
// writes fp16_rn(silu(g) * u) of the fp16-rounded g and u (silu_mul_f16).  No split-K.
//
// Build: this kernel is compiled with -mllvm -amdgpu-sched-strategy=iterative-minreg (its own
// translation unit).  The default pre-RA scheduler reorders the 256 accumulator chains of a
// 128 x 128 wave tile such that the register allocator no longer keeps each accumulator in one
// AGPR tuple, and the loop fills with v_accvgpr_read/write/mov copies.
// ============================================================================================
template <int BM, int BN, int BK, int WM, int WN, int STAGES, int GROUP, int XCD, int RSP,
          int SPLIT = 0, int EPI = 0>
__global__ __launch_bounds__(WM * WN * 64, 1) void k_gemm_ilv(
    const _Float16* __restrict__ A, const _Float16* __restrict__ B, _Float16* __restrict__ C,
    int M, int N, int K, int lda, int ldb, int ldc, float* __restrict__ ws, int ksplit, int up) {
  using MF = Mfma<16>;
  constexpr int SWZ = 2;
  constexpr int NW = WM * WN;
  constexpr int CPR = BK / 8;                 // 16-byte chunks per tile row
  constexpr int RPB = 1024 / (BK * 2);        // tile rows per 1 KiB copy block
  constexpr int R256 = BK * 2 >= 256 ? 1 : 256 / (BK * 2);  // rows per SWZ 2 key step
  constexpr int WTM = BM / WM, WTN = BN / WN;
  constexpr int TM = WTM / 16, TN = WTN / 16;
  constexpr int KS = BK / 32;                 // substeps per k-tile
  constexpr int A_BLK = BM / RPB / NW, B_BLK = BN / RPB / NW;
  constexpr int L = A_BLK + B_BLK;            // copies per wave per k-tile
  constexpr int STAGE = (BM + BN) * BK;
  constexpr int NMF = TM * TN, NR = TM + TN;  // MFMAs and fragment reads per substep
  constexpr int CH = NR > L ? NR : L;
  constexpr int RSPAN = RSP > 0 && RSP < CH ? RSP : CH;
  static_assert(BM % (RPB * NW) == 0 && BN % (RPB * NW) == 0, "copy blocks per wave");
  static_assert(STAGES >= 2 && (STAGES - 1) * L < 64, "stages / vmcnt range");
  // EPI: the gate half of the B tile is its first HB copy blocks of every wave
  constexpr int HB = (BN / 2) / (NW * RPB);
  static_assert(!EPI || (SPLIT == 0 && (BN / 2) % (NW * RPB) == 0), "gate/up: whole copy blocks");
  static_assert(WTM % 16 == 0 && WTN % 16 == 0 && (KS == 1 || KS == 2), "tile shape");
  // rows 16 apart (fragment blocks) and NW*RPB apart (copy blocks) share the swizzle key, so
  // one per-lane offset serves every block of an operand
  static_assert((16 / R256) % CPR == 0 && (NW * RPB / R256) % CPR == 0, "swizzle periods");

  __shared__ __attribute__((aligned(1024))) _Float16 smem[STAGES * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;

  constexpr int BNO = EPI ? BN / 2 : BN;  // output columns per tile
  const int nm = (M + BM - 1) / BM, nn = N / BNO;
  int tmi, tni, sk = 0;
  if constexpr (SPLIT)
    split_tile_of<GROUP, XCD>(blockIdx.x, nm, nn, ksplit, tmi, tni, sk);
  else
    tile_of<GROUP, XCD>(blockIdx.x, nm, nn, tmi, tni);
  const int m0 = tmi * BM, n0 = tni * BNO;
  // k-tiles of this workgroup: [kbase, kbase + NT)
  const int NTALL = K / BK;
  const int kper = SPLIT ? (NTALL + ksplit - 1) / ksplit : NTALL;
  const int kbase = sk * kper;
  const int NT = min(kper, NTALL - kbase);

  // Copy d of this wave fills 1 KiB block (ib*NW + wave) of the A (d < A_BLK) or B tile; lane l
  // fetches the 16-byte chunk that belongs at LDS slot l (the swizzle is an involution).  The
  // buffers start at the tile's panels; A rows past M-1 are clamped to row M-1.
  const int crow = wave * RPB + lane / CPR;                       // tile row of block ib = 0
  const int cchunk = lds_chunk<BK, SWZ>(crow, lane % CPR) * 8;    // element offset in the row
  const _Float16* panelA = A + (long)m0 * lda;
  const _Float16* panelB = B + (long)n0 * ldb;
  // EPI: the up half of the B tile starts at row up + n0 (up = the full output width; a launch
  // over some of the output columns has B offset to its first gate row)
  const _Float16* panelU = B + (long)(up + n0) * ldb;
  const int nrecA = min(M - m0, BM) * lda * 2, nrecB = (EPI ? BN / 2 : BN) * ldb * 2;
  int voff[L];
#pragma unroll
  for (int d = 0; d < L; ++d) {
    const bool isA = d < A_BLK;
    const int ib = isA ? d : d - A_BLK;
    const int r = crow + ib * NW * RPB;
    const int rb = EPI && !isA && ib >= HB ? r - BN / 2 : r;  // row inside its B panel
    voff[d] = isA ? (min(r, M - 1 - m0) * lda + cchunk) * 2 : (rb * ldb + cchunk) * 2;
  }
  auto dma = [&](int kt, int ksrc, int d) {
    const bool isA = d < A_BLK;
    const int ib = isA ? d : d - A_BLK;
    _Float16* dst = smem + (kt % STAGES) * STAGE + (isA ? 0 : BM * BK) + (ib * NW + wave) * RPB * BK;
    const _Float16* pan = isA ? panelA : (EPI && ib >= HB ? panelU : panelB);
    buf_lds16(pan, isA ? nrecA : nrecB, dst, voff[d], (kbase + ksrc) * BK * 2);
  };

  typename MF::acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[i][j][v] = 0.f;

  const int fr = lane % 16, fk = lane / 16;
  int aOff[KS], bOff[KS];  // fragment offsets (elements) inside a stage, per substep
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int ra = wm * WTM + fr, rb = wn * WTN + fr;
    aOff[ks] = ra * BK + lds_chunk<BK, SWZ>(ra, ks * 4 + fk) * 8;
    bOff[ks] = BM * BK + rb * BK + lds_chunk<BK, SWZ>(rb, ks * 4 + fk) * 8;
  }

  f16x8 fa[2][TM], fb[2][TN];
  // One substep on fragment buffer bb: read the next substep (tile rkt, substep rks) into bb^1,
  // refill (DMA) the stage of tile dkt with k-tile dsrc, and run the MFMAs on bb.
  auto substep = [&](auto bufc, auto dmac, int rkt, int rks, int dkt, int dsrc) {
    constexpr int bb = decltype(bufc)::value;
    constexpr bool DMA = decltype(dmac)::value;
    const _Float16* s = smem + (rkt % STAGES) * STAGE;
#pragma unroll
    for (int q = 0; q < CH; ++q) {
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        if (r * RSPAN / NR != q) continue;
        if (r < TM)
          fa[bb ^ 1][r] = *reinterpret_cast<const f16x8*>(s + aOff[rks] + r * 16 * BK);
        else
          fb[bb ^ 1][r - TM] = *reinterpret_cast<const f16x8*>(s + bOff[rks] + (r - TM) * 16 * BK);
      }
      if constexpr (DMA) {
#pragma unroll
        for (int d = 0; d < L; ++d)
          if (d * CH / L == q) dma(dkt, dsrc, d);
      }
#pragma unroll
      for (int t = q * NMF / CH; t < (q + 1) * NMF / CH; ++t)
        acc[t / TN][t % TN] = MF::run(fb[bb][t % TN], fa[bb][t / TN], acc[t / TN][t % TN]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  const int NU = NT * KS;  // substeps (even: K % 64 == 0)
  auto step = [&](auto bufc, auto barc, int u) {
    constexpr bool BAR = decltype(barc)::value;
    const int kt = KS == 1 ? u : u >> 1;
    asm volatile("" ::: "memory");
    if constexpr (BAR) {
      // this wave's reads of tile kt are done and its copies of tile kt+1 have landed ...
      s_wait_vm<(STAGES - 2) * L>();
      // ... and everyone's: tile kt+1 is readable, stage kt % STAGES is free
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      substep(bufc, IC<true>{}, kt + 1, 0, kt + STAGES, min(kt + STAGES, NT - 1));
    } else {
      // this substep's fragments were read in the first chunks of the previous one: the wait
      // is free, and placing it here keeps the compiler from waiting after this substep's
      // first reads instead
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
      asm volatile("" ::: "memory");
      substep(bufc, IC<false>{}, kt, 1, 0, 0);
    }
  };

  // prologue: every stage in flight, tile 0 landed and visible, its first fragments read
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
#pragma unroll
    for (int d = 0; d < L; ++d) dma(s, min(s, NT - 1), d);
  asm volatile("" ::: "memory");
  s_wait_vm<(STAGES - 1) * L>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < TM; ++i) fa[0][i] = *reinterpret_cast<const f16x8*>(smem + aOff[0] + i * 16 * BK);
#pragma unroll
  for (int j = 0; j < TN; ++j) fb[0][j] = *reinterpret_cast<const f16x8*>(smem + bOff[0] + j * 16 * BK);
  __builtin_amdgcn_sched_barrier(0);

  for (int u = 0; u < NU; u += 2) {
    step(IC<0>{}, IC<KS == 1>{}, u);
    step(IC<1>{}, IC<true>{}, u + 1);
  }
  s_wait_vm<0>();  // the refills past the end land before the workgroup's LDS is released

  if constexpr (SPLIT) {
    // fp32 partial tile of split sk: each lane's 4 consecutive n of one m per block, 16 bytes
    float* part = ws + (long)sk * M * N;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wm * WTM + i * 16 + fr;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j)
        *reinterpret_cast<f32x4*>(part + (long)m * N + n0 + wn * WTN + j * 16 + 4 * fk) = acc[i][j];
    }
    return;
  }

  // ---- epilogue ------------------------------------------------------------------------------
  // Rows are written out in 16-byte pieces when C and ldc allow it, else in 8-byte halves.
  const bool c16 = ((reinterpret_cast<uintptr_t>(C) | (uintptr_t)ldc * 2) & 15) == 0;
  auto store16 = [&](_Float16* dst, const u32x4& v) {
    if (c16) {
      __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(dst));
    } else {
      __builtin_nontemporal_store(u32x2{v[0], v[1]}, reinterpret_cast<u32x2*>(dst));
      __builtin_nontemporal_store(u32x2{v[2], v[3]}, reinterpret_cast<u32x2*>(dst + 4));
    }
  };
  constexpr int RB = BN * 2;                  // bytes per C row
  constexpr int CPRW = RB / 16;               // 16-byte chunks per C row
  constexpr bool LDS_EPI = BM * BN <= STAGES * STAGE && CPRW >= 16 && (CPRW & (CPRW - 1)) == 0 &&
                           (NW * 64) % CPRW == 0;
  static_assert(!EPI || LDS_EPI, "gate/up: the epilogue pairs the halves through LDS");
  if constexpr (LDS_EPI) {
    // The C tile through LDS (the stages are free by then): a row-major fp16 image whose 16-byte
    // chunk c of row r sits at chunk c ^ (r % 16), so the 16 rows of an MFMA block write to 16
    // distinct bank groups and a row's chunks read back conflict-free; then whole rows out.
    constexpr int RPP = NW * 64 / CPRW;       // C rows per pass of the whole workgroup
    __syncthreads();                          // every wave is done with the stages
    uint8_t* cs = reinterpret_cast<uint8_t*>(smem);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int r = wm * WTM + i * 16 + fr;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int cb = (wn * WTN + j * 16 + 4 * fk) * 2;  // byte offset of the lane's 4 values
        f16x4 o;
        o[0] = (_Float16)acc[i][j][0];
        o[1] = (_Float16)acc[i][j][1];
        o[2] = (_Float16)acc[i][j][2];
        o[3] = (_Float16)acc[i][j][3];
        *reinterpret_cast<f16x4*>(cs + r * RB + (((cb >> 4) ^ (r & 15)) << 4) + (cb & 15)) = o;
      }
    }
    __syncthreads();
    if constexpr (EPI) {
      // output row r, chunk c (8 columns): gate chunk c, up chunk c + CPRW/2 of image row r
      constexpr int CPO = CPRW / 2, RPO = NW * 64 / CPO;
#pragma unroll 4
      for (int p = 0; p < BM / RPO; ++p) {
        const int r = p * RPO + tid / CPO, c = tid % CPO;
        const f16x8 g = as_f16x8(*reinterpret_cast<const u32x4*>(cs + r * RB + ((c ^ (r & 15)) << 4)));
        const f16x8 u =
            as_f16x8(*reinterpret_cast<const u32x4*>(cs + r * RB + (((c + CPO) ^ (r & 15)) << 4)));
        f16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = silu_mul_f16((float)g[e], (float)u[e]);
        if (m0 + r < M) store16(C + (long)(m0 + r) * ldc + n0 + c * 8, __builtin_bit_cast(u32x4, o));
      }
      return;
    }
#pragma unroll 4
    for (int p = 0; p < BM / RPP; ++p) {
      const int r = p * RPP + tid / CPRW, c = tid % CPRW;
      const u32x4 v = *reinterpret_cast<const u32x4*>(cs + r * RB + ((c ^ (r & 15)) << 4));
      if (m0 + r < M) store16(C + (long)(m0 + r) * ldc + n0 + c * 8, v);
    }
  } else {
    // straight from the MFMA layout: each lane owns 4 consecutive n of one m per block
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wm * WTM + i * 16 + fr;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn * WTN + j * 16 + 4 * fk;
        f16x4 o;
        o[0] = (_Float16)acc[i][j][0];
        o[1] = (_Float16)acc[i][j][1];
        o[2] = (_Float16)acc[i][j][2];
        o[3] = (_Float16)acc[i][j][3];
        *reinterpret_cast<f16x4*>(C + (long)m * ldc + n) = o;
      }
    }
  }
}

// ===== gemv_stream/kernel.hip =====
// gemv_stream -- the small-M (decode) regime of C[M,N] = A[M,K] . deq(B)[N,K]^T on gfx950.
//
// At M <= 32 the operation is bound by reading B once from HBM (2MNK flops against NK or 2NK
// bytes).  The kernel therefore streams B exactly once with 16-byte loads, dequantises in
// registers (formats 1 and 2, bit-exact closed forms in cdna4.h) and feeds the values straight
// into v_mfma_f32_16x16x32_f16 -- the weight rows are the MFMA "A" operand (16 rows per
// instruction), the activation rows the "B" operand (16 columns, padded past M).  The matrix
// cores are >20x over-provisioned here; what they save is the VALU time a dot-product path
// would spend on 2MNK multiply-adds, leaving the VALU to the dequantisation alone.
//
// One workgroup = one slab of 16*R weight rows; its S waves split K into S contiguous chunks
// (S = blockDim.x / 64).  At the end the waves add their partial sums through LDS in wave order
// 0..S-1 (deterministic) and wave 0 writes fp16 C.  No global workspace and no cross-workgroup
// synchronisation: on this part an agent-scope fence is an L2 write-back + invalidate of the
// whole XCD, which per-wave split-K reductions through global memory would pay every time.
//
// Template axes: MB (16-column blocks of M: M <= 16*MB), R (row groups per wave; each activation
// fragment feeds R row groups, so activation traffic is 1/R of the one-group-per-wave form), U
// (k-steps of 64 per pipeline stage), BFMT (0 fp16, 1 int8 + row scale, 2 uint8 + group scale
// and zero-point with group 128: the stage's scales and zero-points for its 64*U/128 groups
// arrive with one small load each, in flight together with the weights).
//
// EPI (fused gate/up epilogue): 0 = plain C = A.B^T.  1 = C[m][n] = silu(G[m][n]) * U[m][n] with
// G = A . B[0..N)^T and U = A . B[up..up+N)^T (B holds 2N rows: the gate rows, then the up rows;
// scales and zero-points follow the B rows).  Each wave then carries 2R row groups, the gate
// groups of its slab and the matching up groups, so the two results of one output meet in the
// same lane and the epilogue combines them in registers (k_stream).  k_stream_sh pairs its slab
// waves instead: half of them stream gate slabs, half the matching up slabs, and the up results
// reach their gate partners through LDS before the epilogue.
//
// k order inside one 64-step: lane (row r = l%16, kgroup g = l/16) owns the 16 consecutive
// k-values [16g, 16g+16) of its row; the first MFMA takes elements 0..7, the second 8..15.
// The activation fragment uses the same map, so each product pairs equal k.

struct StreamArgs {
  const _Float16* A;   // [M][lda]
  const void* B;       // [N][ldb] fp16 / int8 / uint8
  const _Float16* scale;
  const uint8_t* zero;
  _Float16* C;         // [M][ldc]
  int M, N, K, lda, ldb, ldc;
  int S;               // waves per workgroup = k chunks per slab
  int chunk;           // k per chunk (multiple of 64*U; K is a multiple of 64*U too)
  int group;           // k per scale group (fmt 2)
  int up;              // EPI = 1: row offset of the "up" half of B (= N, the output width)
  int nbig = 0;        // k_stream_line with TL = 1: workgroups of SN slabs (the rest: tails)
  int ks = 1;          // k_stream_line: k slices across workgroups (grid = workgroups x ks)
  int kspan = 0;       // ks > 1: k per slice (whole 128-k steps)
  float* part = nullptr;  // ks > 1: fp32 partial sums [ks][M][N], summed by k_splitk_reduce
  int mtiles = 1;      // k_stream_line: row tiles of mrows rows each across workgroups
  int mrows = 0;       // (mtiles > 1) rows per tile, 16 MB
};

// Group-wise metadata of one stage for one lane's row (fmt 2, group 128): GPS = 64*U/128 groups.
template <int GPS>
struct GMeta;
template <>
struct GMeta<1> { uint8_t z; uint16_t s; };
template <>
struct GMeta<2> { uint16_t z; uint32_t s; };
template <>
struct GMeta<4> { uint32_t z; u32x2 s; };

template <int GPS>
__device__ __forceinline__ void gmeta_load(GMeta<GPS>& g, const uint8_t* z, const _Float16* s) {
  if constexpr (GPS == 1) {
    g.z = *z;
    g.s = *reinterpret_cast<const uint16_t*>(s);
  } else if constexpr (GPS == 2) {
    g.z = *reinterpret_cast<const uint16_t*>(z);
    g.s = *reinterpret_cast<const uint32_t*>(s);
  } else {
    g.z = *reinterpret_cast<const uint32_t*>(z);
    g.s = *reinterpret_cast<const u32x2*>(s);
  }
}

template <int GPS>
__device__ __forceinline__ void gmeta_get(const GMeta<GPS>& g, int i, uint8_t& z, _Float16& s) {
  if constexpr (GPS == 1) {
    z = g.z;
    s = __builtin_bit_cast(_Float16, g.s);
  } else if constexpr (GPS == 2) {
    z = (uint8_t)(g.z >> (8 * i));
    s = __builtin_bit_cast(_Float16, (uint16_t)(g.s >> (16 * i)));
  } else {
    z = (uint8_t)(g.z >> (8 * i));
    s = __builtin_bit_cast(_Float16, (uint16_t)(g.s[i >> 1] >> (16 * (i & 1))));
  }
}

template <int BFMT>
struct WRaw;  // per lane, per row group, per 64-step: the 16 k-values of its row
template <>
struct WRaw<0> { u32x4 v[2]; };  // 32 bytes fp16
template <>
struct WRaw<1> { u32x4 v; };     // 16 bytes int8
template <>
struct WRaw<2> { u32x4 v; };     // 16 bytes uint8

// ---- result: lane holds C[m = b*16 + r16][n = nbase + r*16 + 4*kg + v], v = 0..3 ------------
// (EPI: the gate result in acc[r], the up result of the same outputs in acc[r + R])
template <int MB, int R, int EPI, int RR>
__device__ __forceinline__ void stream_store(const StreamArgs& p, const f32x4 (&acc)[RR][MB],
                                             int nbase, int r16, int kg) {
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int m = b * 16 + r16;
    if (m >= p.M) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = nbase + r * 16 + 4 * kg;
      f16x4 o;
#pragma unroll
      for (int v = 0; v < 4; ++v)
        o[v] = EPI ? silu_mul_f16(acc[r][b][v], acc[r + R][b][v]) : (_Float16)acc[r][b][v];
      *reinterpret_cast<f16x4*>(p.C + (long)m * p.ldc + n) = o;
    }
  }
}

// ks > 1: the fp32 partial sums of k slice `ksi` go to part[ksi][m][n] (same lane map), to be
// added in slice order by k_splitk_reduce.
template <int MB, int R, int RR>
__device__ __forceinline__ void stream_store_part(const StreamArgs& p, const f32x4 (&acc)[RR][MB],
                                                  int nbase, int r16, int kg, int ksi) {
  float* dst = p.part + (long)ksi * p.M * p.N;
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int m = b * 16 + r16;
    if (m >= p.M) continue;
#pragma unroll
    for (int r = 0; r < R; ++r)
      *reinterpret_cast<f32x4*>(dst + (long)m * p.N + nbase + r * 16 + 4 * kg) = acc[r][b];
  }
}

// ALDS = 1: the workgroup first copies A[0..M)[0..K) into LDS (row stride 2K+16 bytes, so the 16
// rows of one fragment read land in 16 distinct bank groups) and the k-loop reads activation
// fragments from there -- one weight load per k-step instead of one weight + two activation
// loads, and for M = 1 the 16 lanes of a k-group read one address (an LDS broadcast).  Chosen by
// the launcher when M*(2K+16) bytes fit its LDS budget.
template <int MB, int R, int U, int BFMT, int ALDS = 0, int EPI = 0>
__global__ __launch_bounds__(512) void k_stream(StreamArgs p) {
  constexpr int RR = EPI ? 2 * R : R;  // row groups per wave
  extern __shared__ __attribute__((aligned(16))) uint8_t dsm_s[];
  const long arow_bytes = 2L * p.K + 16;
  const long act_bytes = ALDS ? (long)p.M * arow_bytes : 0;
  f32x4* red = reinterpret_cast<f32x4*>(dsm_s + act_bytes);  // [S][RR*MB][64] partials
  const int lane = threadIdx.x & 63;
  const int split = threadIdx.x >> 6;
  const int slab = blockIdx.x;
  const int kbeg = min(p.K, split * p.chunk);
  const int kend = min(p.K, kbeg + p.chunk);

  const int r16 = lane & 15;  // row within a 16-row group / column within a 16-col block
  const int kg = lane >> 4;   // k-group 0..3
  const int nbase = slab * 16 * R;

  // weight row pointers
  // row groups of this wave: gate groups 0..R-1, then (EPI) the matching up groups
  auto row_of = [&](int r) -> long {
    return (EPI && r >= R ? (long)p.up + nbase + (r - R) * 16 : (long)nbase + r * 16) + r16;
  };
  const uint8_t* wrow[RR];
  _Float16 rscale[RR];
#pragma unroll
  for (int r = 0; r < RR; ++r) {
    const long n = row_of(r);
    constexpr int EB = BFMT == 0 ? 2 : 1;
    wrow[r] = reinterpret_cast<const uint8_t*>(p.B) + (n * p.ldb + 16 * kg) * EB;
    if constexpr (BFMT == 1) rscale[r] = p.scale[n];
  }
  // activation row pointers (rows past M read row M-1; their results are never stored)
  const _Float16* arow[MB];
  const uint8_t* alds[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int m = min(b * 16 + r16, p.M - 1);
    arow[b] = p.A + (long)m * p.lda + 16 * kg;
    alds[b] = dsm_s + m * arow_bytes + 32 * kg;
  }
  if constexpr (ALDS) {
    const int cpr = p.K / 8;  // 16-byte chunks per activation row
    for (int i = threadIdx.x; i < p.M * cpr; i += blockDim.x) {
      const int m = i / cpr, c = i - m * cpr;
      *reinterpret_cast<u32x4*>(dsm_s + m * arow_bytes + c * 16) =
          *reinterpret_cast<const u32x4*>(p.A + (long)m * p.lda + c * 8);
    }
    __syncthreads();
  }

  f32x4 acc[RR][MB], acc2[RR][MB];
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc2[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  WRaw<BFMT> w[2][U][RR];
  u32x4 a[2][U][MB][ALDS ? 1 : 2];
  constexpr int GPS = (64 * U) / 128 > 0 ? (64 * U) / 128 : 1;  // groups per stage (fmt 2)
  GMeta<GPS> gm[2][RR];
  const long gstride = BFMT == 2 ? (long)(p.K / 128) : 0;  // groups per weight row

  // Every stage is whole: K and the chunk are multiples of 64*U (checked by the launcher), so
  // the loads carry no predicate and the compiler can wait for exactly the stage it consumes.
  auto issue = [&](auto bufc, int k0) {
    constexpr int buf = decltype(bufc)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 64 * u;
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        if constexpr (BFMT == 0) {
          const u32x4* q = reinterpret_cast<const u32x4*>(wrow[r] + (long)k * 2);
          w[buf][u][r].v[0] = q[0];
          w[buf][u][r].v[1] = q[1];
        } else {
          w[buf][u][r].v = *reinterpret_cast<const u32x4*>(wrow[r] + k);
        }
      }
      if constexpr (BFMT == 2) {
        if (u == 0) {
#pragma unroll
          for (int r = 0; r < RR; ++r) {
            const long gi = row_of(r) * gstride + k0 / 128;
            gmeta_load<GPS>(gm[buf][r], p.zero + gi, p.scale + gi);
          }
        }
      }
      if constexpr (!ALDS) {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          const u32x4* q = reinterpret_cast<const u32x4*>(arow[b] + k);
          a[buf][u][b][0] = q[0];
          a[buf][u][b][1] = q[1];
        }
      }
    }
  };

  // two independent accumulator chains per (row group, column block): consecutive MFMAs never
  // wait on each other's result
  auto compute = [&](auto bufc, int k0) {
    constexpr int buf = decltype(bufc)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        f16x8 w0, w1;
        if constexpr (BFMT == 0) {
          w0 = as_f16x8(w[buf][u][r].v[0]);
          w1 = as_f16x8(w[buf][u][r].v[1]);
        } else if constexpr (BFMT == 1) {
          const u32x4 q = w[buf][u][r].v;
          w0 = dequant8_i8(q[0], q[1], rscale[r]);
          w1 = dequant8_i8(q[2], q[3], rscale[r]);
        } else {
          const u32x4 q = w[buf][u][r].v;
          uint8_t z;
          _Float16 s;
          gmeta_get<GPS>(gm[buf][r], (64 * u) / 128, z, s);
          w0 = dequant8_u8(q[0], q[1], z, s);
          w1 = dequant8_u8(q[2], q[3], z, s);
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          u32x4 a0, a1;
          if constexpr (ALDS) {
            const uint8_t* q = alds[b] + (long)(k0 + 64 * u) * 2;
            a0 = *reinterpret_cast<const u32x4*>(q);
            a1 = *reinterpret_cast<const u32x4*>(q + 16);
          } else {
            a0 = a[buf][u][b][0];
            a1 = a[buf][u][b][1];
          }
          acc[r][b] = Mfma<16>::run(w0, as_f16x8(a0), acc[r][b]);
          acc2[r][b] = Mfma<16>::run(w1, as_f16x8(a1), acc2[r][b]);
        }
      }
    }
  };

  // two-stage register pipeline: loads of stage s+1 are in flight while stage s computes.
  // Unrolled by two so every register-array index is a compile-time constant, and the steady
  // state always issues before it computes (tail peeled), so the wait before each compute is
  // "all but the stage just issued" on every path into it.
  constexpr int STEP = 64 * U;
  int k0 = kbeg;
  int n = (kend - kbeg) / STEP;  // whole stages in this chunk (0 for a wave past K)
  if (n > 0) issue(IC<0>{}, k0);
  while (n >= 3) {
    issue(IC<1>{}, k0 + STEP);
    compute(IC<0>{}, k0);
    issue(IC<0>{}, k0 + 2 * STEP);
    compute(IC<1>{}, k0 + STEP);
    k0 += 2 * STEP;
    n -= 2;
  }
  if (n == 2) {
    issue(IC<1>{}, k0 + STEP);
    compute(IC<0>{}, k0);
    compute(IC<1>{}, k0 + STEP);
  } else if (n == 1) {
    compute(IC<0>{}, k0);
  }
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[r][b] += acc2[r][b];

  // ---- result: lane holds C[m = b*16 + r16][n = nbase + r*16 + 4*kg + v], v = 0..3 ----------
  if (p.S > 1) {
    // partials of every wave through LDS; summed in wave order by wave 0
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int b = 0; b < MB; ++b) red[(split * RR * MB + r * MB + b) * 64 + lane] = acc[r][b];
    __syncthreads();
    if (split != 0) return;
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        f32x4 t = red[(r * MB + b) * 64 + lane];
        for (int w = 1; w < p.S; ++w) {
          const f32x4 v = red[(w * RR * MB + r * MB + b) * 64 + lane];
          t[0] += v[0]; t[1] += v[1]; t[2] += v[2]; t[3] += v[3];
        }
        acc[r][b] = t;
      }
  }
  stream_store<MB, R, EPI>(p, acc, nbase, r16, kg);
}

// Debug/verification entry: dequantise a [rows x cols] tile of B starting at (n0, k0) with the
// same device functions the GEMM feeds use, writing fp16 [rows][cols].  cols % 8 == 0.
template <int BFMT>
__global__ void k_dequant_tile(StreamArgs p, int n0, int k0, int rows, int cols, _Float16* out) {
  const int per_row = cols / 8;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * per_row) return;
  const int r = idx / per_row, c8 = idx - r * per_row;
  const long n = n0 + r;
  const long k = k0 + c8 * 8;
  f16x8 v;
  if constexpr (BFMT == 1) {
    const u32x2 q = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint8_t*>(p.B) +
                                                    n * p.ldb + k);
    v = dequant8_i8(q[0], q[1], p.scale[n]);
  } else {
    const u32x2 q = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint8_t*>(p.B) +
                                                    n * p.ldb + k);
    const long gi = n * (p.K / p.group) + k / p.group;
    v = dequant8_u8(q[0], q[1], p.zero[gi], p.scale[gi]);
  }
  *reinterpret_cast<f16x8*>(out + (long)r * cols + c8 * 8) = v;
}

// ============================================================================================
// k_stream_dma -- same operation, work split and reduction as k_stream, but everything a k-step
// consumes travels HBM/L2 -> LDS with the gfx950 LDS-DMA load (global_load_lds_dwordx4) into a
// PRIVATE ring of D k-steps per wave: R*(1|2) KiB of weights and 2*MB KiB of activation
// fragments per step.  Bytes in flight cost no registers, and because every k-step issues the
// same instructions, one constant wait -- s_waitcnt vmcnt((D-1) * per-step count) -- is exactly
// "step j has landed" (vmcnt retires in issue order, so a shorter-distance load of any kind
// would cap the depth of the weight prefetch; that is why the activations ride the ring too).
//
// Per wave, iteration j:  wait for step j;  ds_read slot j % D -> registers;  lgkmcnt(0);
// DMA step j+D into slot j % D (past the chunk's end the index clamps to the last step: a
// redundant L2 hit that keeps the count constant);  dequantise + MFMA.
//
// DMA lane map: lane l fetches the 16 bytes of the operand fragment it will consume (row
// l % 16, k-group l / 16), LDS-DMA stores lane l's 16 bytes at byte 16*l of the 1 KiB block,
// and lane l reads back exactly those bytes: the ring is a latency buffer, not a shuffle.
// fmt 2 scale/zero-points of the wave's whole chunk are staged in LDS once, before the loop.
// ============================================================================================
typedef __attribute__((address_space(3))) void lds_void_stream_t;

template <int N>
__device__ __forceinline__ void s_wait_vm_stream() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

template <int MB, int R, int D, int BFMT>
struct StreamDma {
  static constexpr int WB = BFMT == 0 ? 2 : 1;  // weight bytes per element
  static constexpr int LD = R * WB;              // weight DMA instructions (1 KiB) per step
  static constexpr int LA = 2 * MB;              // activation DMA instructions per step
  static constexpr int SLOT = (LD + LA) * 1024;  // ring slot bytes
  static constexpr int WAIT = (D - 1) * (LD + LA);
  static constexpr int META_GROUPS = 64;         // fmt 2: groups staged per wave (chunk <= 8192 k)
  static constexpr int META = BFMT == 2 ? R * 16 * META_GROUPS * 3 : 0;  // z (1 B) + s (2 B)
  static constexpr int WAVE_BYTES = D * SLOT + META;
  static_assert(WAIT < 64, "ring too deep for vmcnt");
  static constexpr size_t lds(int S) {
    return (size_t)S * WAVE_BYTES + (S > 1 ? (size_t)S * R * MB * 64 * 16 : 0);
  }
};

template <int MB, int R, int D, int BFMT>
__global__ __launch_bounds__(512) void k_stream_dma(StreamArgs p) {
  using SD = StreamDma<MB, R, D, BFMT>;
  constexpr int WB = SD::WB, LD = SD::LD, SLOT = SD::SLOT;
  extern __shared__ __attribute__((aligned(1024))) uint8_t dsm[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slab = blockIdx.x;
  uint8_t* ring = dsm + (size_t)wave * SD::WAVE_BYTES;
  uint8_t* meta = ring + D * SLOT;  // fmt 2: [R*16 rows][64 groups] z, then s
  f32x4* red = reinterpret_cast<f32x4*>(dsm + (size_t)p.S * SD::WAVE_BYTES);

  const int kbeg = min(p.K, wave * p.chunk);
  const int kend = min(p.K, kbeg + p.chunk);
  const int n = (kend - kbeg) / 64;  // k-steps of this wave (>= 1 by construction of S)
  const int r16 = lane & 15, kg = lane >> 4;
  const int nbase = slab * 16 * R;

  const uint8_t* wsrc[R];
  _Float16 rscale[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const long row = nbase + r * 16 + r16;
    wsrc[r] = reinterpret_cast<const uint8_t*>(p.B) + (row * p.ldb + kbeg + 16 * kg) * WB;
    if constexpr (BFMT == 1) rscale[r] = p.scale[row];
  }
  const _Float16* asrc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) asrc[b] = p.A + (long)min(b * 16 + r16, p.M - 1) * p.lda + kbeg + 16 * kg;

  if constexpr (BFMT == 2) {
    // stage this wave's scale/zero-points: R*16 rows x G groups (G = chunk/128 <= 64)
    const int g0 = kbeg / 128, G = (kend - 1) / 128 - g0 + 1;  // groups the chunk touches
    const long gstride = p.K / 128;
    for (int i = lane; i < R * 16 * G; i += 64) {
      const int row = i / G, g = i - row * G;
      const long gi = (long)(nbase + row) * gstride + g0 + g;
      meta[row * SD::META_GROUPS + g] = p.zero[gi];
      reinterpret_cast<_Float16*>(meta + R * 16 * SD::META_GROUPS)[row * SD::META_GROUPS + g] = p.scale[gi];
    }
    __builtin_amdgcn_s_waitcnt(0);  // staged before any DMA is counted
  }

  f32x4 acc[R][MB];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto dma = [&](int j) {  // step j (clamped) -> ring slot j % D
    const int jj = min(j, n - 1);
    uint8_t* slot = ring + (j % D) * SLOT;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int h = 0; h < WB; ++h)
        __builtin_amdgcn_global_load_lds((void*)(wsrc[r] + (long)jj * 64 * WB + 16 * h),
                                         (lds_void_stream_t*)(slot + (r * WB + h) * 1024), 16, 0, 0);
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        __builtin_amdgcn_global_load_lds((void*)(asrc[b] + jj * 64 + 8 * h),
                                         (lds_void_stream_t*)(slot + (LD + 2 * b + h) * 1024), 16, 0, 0);
  };

  for (int j = 0; j < D; ++j) dma(j);
  for (int j = 0; j < n; ++j) {
    asm volatile("" ::: "memory");
    s_wait_vm_stream<SD::WAIT>();  // step j has landed
    asm volatile("" ::: "memory");
    const uint8_t* slot = ring + (j % D) * SLOT;
    u32x4 w[R][WB], av[MB][2];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int h = 0; h < WB; ++h)
        w[r][h] = *reinterpret_cast<const u32x4*>(slot + (r * WB + h) * 1024 + 16 * lane);
#pragma unroll
    for (int b = 0; b < MB; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        av[b][h] = *reinterpret_cast<const u32x4*>(slot + (LD + 2 * b + h) * 1024 + 16 * lane);
    uint8_t zc[R];
    _Float16 sc[R];
    if constexpr (BFMT == 2) {
      const int g = (kbeg + j * 64) / 128 - kbeg / 128;  // group of this step in the stage
#pragma unroll
      for (int r = 0; r < R; ++r) {
        zc[r] = meta[(r * 16 + r16) * SD::META_GROUPS + g];
        sc[r] = reinterpret_cast<const _Float16*>(meta + R * 16 * SD::META_GROUPS)[(r * 16 + r16) * SD::META_GROUPS + g];
      }
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): operands are in registers, slot is free
    asm volatile("" ::: "memory");
    dma(j + D);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      f16x8 w0, w1;
      if constexpr (BFMT == 0) {
        w0 = as_f16x8(w[r][0]);
        w1 = as_f16x8(w[r][1]);
      } else if constexpr (BFMT == 1) {
        w0 = dequant8_i8(w[r][0][0], w[r][0][1], rscale[r]);
        w1 = dequant8_i8(w[r][0][2], w[r][0][3], rscale[r]);
      } else {
        w0 = dequant8_u8(w[r][0][0], w[r][0][1], zc[r], sc[r]);
        w1 = dequant8_u8(w[r][0][2], w[r][0][3], zc[r], sc[r]);
      }
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        acc[r][b] = Mfma<16>::run(w0, as_f16x8(av[b][0]), acc[r][b]);
        acc[r][b] = Mfma<16>::run(w1, as_f16x8(av[b][1]), acc[r][b]);
      }
    }
    (void)zc;
    (void)sc;
  }
  __builtin_amdgcn_s_waitcnt(0);  // no LDS-DMA write may outlive this workgroup's LDS
  asm volatile("" ::: "memory");

  if (p.S > 1) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int b = 0; b < MB; ++b) red[(wave * R * MB + r * MB + b) * 64 + lane] = acc[r][b];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        f32x4 t = red[(r * MB + b) * 64 + lane];
        for (int w = 1; w < p.S; ++w) {
          const f32x4 v = red[(w * R * MB + r * MB + b) * 64 + lane];
          t[0] += v[0]; t[1] += v[1]; t[2] += v[2]; t[3] += v[3];
        }
        acc[r][b] = t;
      }
  }
#pragma unroll
  for (int b = 0; b < MB; ++b) {
    const int m = b * 16 + r16;
    if (m >= p.M) continue;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int nn = nbase + r * 16 + 4 * kg;
      f16x4 o;
      o[0] = (_Float16)acc[r][b][0];
      o[1] = (_Float16)acc[r][b][1];
      o[2] = (_Float16)acc[r][b][2];
      o[3] = (_Float16)acc[r][b][3];
      *reinterpret_cast<f16x4*>(p.C + (long)m * p.ldc + nn) = o;
    }
  }
}

template <int MB, int R, int D, int BFMT>
constexpr size_t stream_dma_lds(int S) {
  return StreamDma<MB, R, D, BFMT>::lds(S);
}

// Streaming-read probe: each wave streams its share of `bytes` through a private LDS-DMA ring
// of D KiB (no compute) and folds one dword per step into an output, so nothing is optimised
// away.  Measures the read bandwidth this part sustains with the ring discipline.
template <int D>
__global__ __launch_bounds__(256) void k_read_probe(const uint8_t* src, long bytes_per_wave,
                                                    unsigned* out) {
  __shared__ __attribute__((aligned(1024))) uint8_t ring_all[4 * D * 1024];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const long gw = (long)blockIdx.x * 4 + wave;
  uint8_t* ring = ring_all + wave * D * 1024;
  const uint8_t* base = src + gw * bytes_per_wave + 16 * lane;
  const int n = (int)(bytes_per_wave / 1024);
  unsigned accum = 0;
  auto dma = [&](int j) {
    const int jj = min(j, n - 1);
    __builtin_amdgcn_global_load_lds((void*)(base + (long)jj * 1024),
                                     (lds_void_stream_t*)(ring + (j % D) * 1024), 16, 0, 0);
  };
  for (int j = 0; j < D; ++j) dma(j);
  for (int j = 0; j < n; ++j) {
    asm volatile("" ::: "memory");
    s_wait_vm_stream<D - 1>();
    asm volatile("" ::: "memory");
    accum += *reinterpret_cast<const unsigned*>(ring + (j % D) * 1024 + 16 * lane);
    __builtin_amdgcn_s_waitcnt(0xc07f);
    asm volatile("" ::: "memory");
    dma(j + D);
  }
  __builtin_amdgcn_s_waitcnt(0);
  asm volatile("" ::: "memory");
  if (accum == 0x9e3779b9u) out[0] = accum;  // practically never; keeps the reads alive
}

// ============================================================================================
// k_stream_sh -- the decode kernel with the activations SHARED between waves.
//
// k_stream re-reads the whole activation block A[0..M)[k-chunk] from L2 in every workgroup (one
// workgroup = one slab of 16R weight rows), so at M = 16..32 the activation traffic equals or
// exceeds the weight traffic and, measured, caps the kernel well below the M = 1 rate (the same
// kernel with all activation rows aliased to one reaches the M = 1 rate).  Here one workgroup
// holds SN slabs x SK k-chunks of waves (wave w: slab group w % SN, k-chunk w / SN).  The SN waves
// of one k-chunk walk the same k-steps, so each stage of activations (16*MB rows x 64U k) is
// brought global -> LDS ONCE by LDS-DMA (the SN waves split the copy) into a two-slot ring of that
// k-chunk, and read from there by all SN waves: activation traffic drops by SN.  Weights stay in
// the register pipeline of k_stream (stage s+1 in flight while stage s computes), dequantised in
// registers, MFMA 16x16x32 as before; the SK partial sums of a slab are added through LDS in
// k-chunk order (deterministic) and written by the chunk-0 wave.
//
// Per iteration s (all waves of the workgroup in step): wait until this wave's copies for stage s
// have landed and its LDS reads of stage s-1 are done; s_barrier (everyone's copies for stage s
// landed, everyone done with slot (s+1) % 2); issue the weight loads of stage s+1 and the
// activation copy of stage s+1 into slot (s+1) % 2; compute stage s.
//
// LDS activation stage: [16*MB rows][64U k] fp16, 16-byte chunk c of row r stored at chunk
// c ^ (r % 16), so the 16 rows of one fragment read hit 16 distinct bank groups.  Rows >= M are
// copies of row M-1 (never stored to C).
// Requirements (launcher): N % (16*R*SN) == 0, the stage count K / (64U) divisible by SK, and
// (2*MB*U) % SN == 0 (whole 1 KiB copy blocks per wave).
// ============================================================================================
template <int N>
__device__ __forceinline__ void s_wait_vm_lgkm0() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
}

template <int MB, int U>
struct StreamSh {
  static constexpr int RB = 128 * U;                // bytes per activation row per stage
  static constexpr int STAGE = 16 * MB * RB;        // bytes per activation stage
  static constexpr int NBLK = STAGE / 1024;         // 1 KiB copy blocks per stage
  static constexpr size_t lds(int SN, int SK, int R) {
    return (size_t)SK * 2 * STAGE + (SK > 1 ? (size_t)SN * SK * R * MB * 64 * 16 : 0);
  }
};

// TPB: the launch bound (512 or 1024 lanes; 1024 caps a lane at 128 registers)
template <int MB, int R, int U, int BFMT, int SN, int TPB = 512, int EPI = 0>
__global__ __launch_bounds__(TPB) void k_stream_sh(StreamArgs p) {
  // EPI = 1 pairs the slab waves instead of widening them: of the SN slab waves of a workgroup
  // the first SN/2 take gate slabs and the last SN/2 the matching up slabs, so a wave carries R
  // row groups exactly as in the plain kernel; after the k reduction each up wave hands its
  // result to its gate partner through LDS.
  constexpr int RR = R;
  static_assert(!EPI || SN % 2 == 0, "the fused gate/up pairing needs an even SN");
  constexpr int SPW = EPI ? SN / 2 : SN;  // output slabs per workgroup
  using SS = StreamSh<MB, U>;
  constexpr int RB = SS::RB, STAGE = SS::STAGE, NBLK = SS::NBLK;
  static_assert(NBLK % SN == 0, "activation copy blocks split evenly over the slab waves");
  static_assert(U >= 2, "a stage row must hold at least 16 chunks for the swizzle");
  constexpr int BW = NBLK / SN;  // copy blocks per wave per stage
  extern __shared__ __attribute__((aligned(1024))) uint8_t dsh[];
  const int SK = p.S;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ng = wave % SN, kgrp = wave / SN;
  uint8_t* ring = dsh + (size_t)kgrp * 2 * STAGE;
  f32x4* red = reinterpret_cast<f32x4*>(dsh + (size_t)SK * 2 * STAGE);

  const int r16 = lane & 15;
  const int kg = lane >> 4;
  const bool upw = EPI && ng >= SPW;  // an up wave (EPI)
  const int slab = blockIdx.x * SPW + (upw ? ng - SPW : ng);
  const int nbase = slab * 16 * R;  // output rows of this wave's slab
  const int kbeg = kgrp * p.chunk;
  constexpr int STEP = 64 * U;
  const int nst = p.chunk / STEP;  // identical for every k-chunk (launcher)

  // row groups of this wave: gate groups 0..R-1, then (EPI) the matching up groups
  auto row_of = [&](int r) -> long { return (upw ? (long)p.up : 0L) + nbase + r * 16 + r16; };
  const uint8_t* wrow[RR];
  _Float16 rscale[RR];
#pragma unroll
  for (int r = 0; r < RR; ++r) {
    const long n = row_of(r);
    constexpr int EB = BFMT == 0 ? 2 : 1;
    wrow[r] = reinterpret_cast<const uint8_t*>(p.B) + (n * p.ldb + 16 * kg) * EB;
    if constexpr (BFMT == 1) rscale[r] = p.scale[n];
  }

  // activation copy: block i of this wave = stage block (i*SN + ng); lane -> (row, phys chunk)
  long asrc[BW];
#pragma unroll
  for (int i = 0; i < BW; ++i) {
    const int off = (i * SN + ng) * 1024 + 16 * lane;
    const int row = off / RB, phys = (off % RB) / 16;
    const int logical = phys ^ (row & 15);
    asrc[i] = (long)min(row, p.M - 1) * p.lda + 8 * logical;
  }
  auto copy_act = [&](int s) {
    uint8_t* dst = ring + (s & 1) * STAGE;
    const _Float16* base = p.A + kbeg + s * STEP;
#pragma unroll
    for (int i = 0; i < BW; ++i)
      __builtin_amdgcn_global_load_lds((void*)(base + asrc[i]),
                                       (lds_void_stream_t*)(dst + (i * SN + ng) * 1024), 16, 0, 0);
  };
  // fragment read offsets: row b*16 + r16, chunks 8u + 2kg (+1) XOR r16; (8u + 2kg) ^ r16 only
  // touches bits 0..3, so two variants by u & 1, plus 16 chunks per two k-steps
  int aoff0[2], aoff1[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    aoff0[q] = r16 * RB + ((8 * q + 2 * kg) ^ r16) * 16;
    aoff1[q] = r16 * RB + ((8 * q + 2 * kg + 1) ^ r16) * 16;
  }

  f32x4 acc[RR][MB], acc2[RR][MB];
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc2[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  WRaw<BFMT> w[2][U][RR];
  constexpr int GPS = (64 * U) / 128 > 0 ? (64 * U) / 128 : 1;
  GMeta<GPS> gm[2][RR];
  const long gstride = BFMT == 2 ? (long)(p.K / 128) : 0;

  auto issue_w = [&](auto bufc, int k0) {
    constexpr int buf = decltype(bufc)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 64 * u;
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        if constexpr (BFMT == 0) {
          const u32x4* q = reinterpret_cast<const u32x4*>(wrow[r] + (long)k * 2);
          w[buf][u][r].v[0] = q[0];
          w[buf][u][r].v[1] = q[1];
        } else {
          w[buf][u][r].v = *reinterpret_cast<const u32x4*>(wrow[r] + k);
        }
      }
    }
    if constexpr (BFMT == 2) {
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        const long gi = row_of(r) * gstride + k0 / 128;
        gmeta_load<GPS>(gm[buf][r], p.zero + gi, p.scale + gi);
      }
    }
  };

  auto compute = [&](auto bufc, int s) {
    constexpr int buf = decltype(bufc)::value;
    const uint8_t* a = ring + (s & 1) * STAGE;
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        f16x8 w0, w1;
        if constexpr (BFMT == 0) {
          w0 = as_f16x8(w[buf][u][r].v[0]);
          w1 = as_f16x8(w[buf][u][r].v[1]);
        } else if constexpr (BFMT == 1) {
          const u32x4 q = w[buf][u][r].v;
          w0 = dequant8_i8(q[0], q[1], rscale[r]);
          w1 = dequant8_i8(q[2], q[3], rscale[r]);
        } else {
          const u32x4 q = w[buf][u][r].v;
          uint8_t z;
          _Float16 sc;
          gmeta_get<GPS>(gm[buf][r], (64 * u) / 128, z, sc);
          w0 = dequant8_u8(q[0], q[1], z, sc);
          w1 = dequant8_u8(q[2], q[3], z, sc);
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          const uint8_t* rowp = a + b * 16 * RB + (u >> 1) * 256;
          const u32x4 a0 = *reinterpret_cast<const u32x4*>(rowp + aoff0[u & 1]);
          const u32x4 a1 = *reinterpret_cast<const u32x4*>(rowp + aoff1[u & 1]);
          acc[r][b] = Mfma<16>::run(w0, as_f16x8(a0), acc[r][b]);
          acc2[r][b] = Mfma<16>::run(w1, as_f16x8(a1), acc2[r][b]);
        }
      }
    }
  };

  // one pipeline step: (top) stage s landed for everyone; issue stage s+1; compute stage s
  auto step = [&](auto bufc, int s) {
    constexpr int buf = decltype(bufc)::value;
    asm volatile("" ::: "memory");
    s_wait_vm_lgkm0<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + 1 < nst) {
      issue_w(IC<buf ^ 1>{}, kbeg + (s + 1) * STEP);
      copy_act(s + 1);
    }
    compute(bufc, s);
  };

  if (nst > 0) {
    issue_w(IC<0>{}, kbeg);
    copy_act(0);
  }
  int s = 0;
  for (; s + 1 < nst; s += 2) {
    step(IC<0>{}, s);
    step(IC<1>{}, s + 1);
  }
  if (s < nst) step(IC<0>{}, s);

#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int b = 0; b < MB; ++b) acc[r][b] += acc2[r][b];

  if (SK > 1) {
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int b = 0; b < MB; ++b) red[(wave * RR * MB + r * MB + b) * 64 + lane] = acc[r][b];
    __syncthreads();
    if (kgrp == 0) {
#pragma unroll
      for (int r = 0; r < RR; ++r)
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          f32x4 t = acc[r][b];
          for (int g = 1; g < SK; ++g) {
            const f32x4 v = red[((g * SN + ng) * RR * MB + r * MB + b) * 64 + lane];
            t[0] += v[0]; t[1] += v[1]; t[2] += v[2]; t[3] += v[3];
          }
          acc[r][b] = t;
        }
    }
  }
  if constexpr (EPI) {
    // every wave is past its last ring read (barrier), so ring memory carries the up results
    f32x4* xb = reinterpret_cast<f32x4*>(dsh);
    if (SK == 1) __syncthreads();
    if (kgrp == 0 && upw) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < MB; ++b) xb[(((ng - SPW) * R + r) * MB + b) * 64 + lane] = acc[r][b];
    }
    __syncthreads();
    if (kgrp != 0 || upw) return;
    f32x4 both[2 * R][MB];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int b = 0; b < MB; ++b) {
        both[r][b] = acc[r][b];
        both[R + r][b] = xb[((ng * R + r) * MB + b) * 64 + lane];
      }
    stream_store<MB, R, 1>(p, both, nbase, r16, kg);
  } else {
    if (kgrp != 0) return;
    stream_store<MB, R, 0>(p, acc, nbase, r16, kg);
  }
}

// ============================================================================================
// k_stream_line -- the decode kernel whose weight stream travels in whole 128-byte lines.
//
// A 16-byte weight fragment in the MFMA operand layout (row l % 16, k-group l / 16) puts only
// 64 bytes of each row into one load instruction: every 128-byte line of the weights is touched
// by two instructions, and the streaming rate stays near 6 TB/s.  Here the weights go HBM -> LDS
// by LDS-DMA (global_load_lds_dwordx4) with the nontemporal cache policy, and each copy
// instruction fetches 8 rows x 128 bytes -- lane l takes 16 bytes of row l / 8 -- so every line
// is fetched whole by one instruction, never cached, and the stream runs at about 7 TB/s.  The
// fragments are read back from LDS in the MFMA layout; which 16-byte chunk a lane fetches is
// chosen so the LDS image is swizzled (chunk c of row r stored at chunk c ^ ((r / 2) % 8)) and
// those reads are free of bank conflicts.
//
// Each wave owns a PRIVATE ring of D steps (no barrier inside the loop).  A step is 128 k of
// RR row groups (16 weight rows each): EB lines per row (EB = 1 byte per weight for int8/uint8,
// 2 for fp16), plus the activations of those 128 k: for MB = 0 (M = 1) the 256-byte slice of
// row 0 by one dword copy, read back by broadcast; for MB = 1 or 2 (M <= 16 or 32) the 16*MB
// rows x 256 bytes (rows past M re-read row M-1), chunk c of row m stored at chunk c ^ (m % 16).
// Every step issues the same copies, so one constant wait -- vmcnt((D-1) * copies per step) --
// is exactly "step j has landed"; the copies past the chunk's end re-fetch its last step into a
// slot nobody reads, and the kernel drains them before the LDS is reused.
//
// Work split: one workgroup = SN slabs of 16*R weight rows x S k chunks (whole steps); wave w
// takes slab w % SN and chunk w / SN.  The S partial sums of a slab are added through LDS in
// chunk order and written by its chunk-0 wave, as k_stream does.  With ks > 1 (plain epilogue)
// the grid holds ks workgroups per slab group, workgroup b taking k slice b % ks of kspan k; the
// S chunks split that slice, and the slice's sum goes to the fp32 partials (k_splitk_reduce adds
// the slices in order) -- so a slab count that is not a multiple of the CU count still spreads
// evenly over the part.
// SN = 1: every wave also owns its activation ring (no barrier in the loop).  SN > 1: the SN
// waves of one k chunk walk the same steps and SHARE one activation ring -- each issues LA/SN of
// the copies of a step -- so the activation traffic drops by SN; one workgroup barrier per step
// orders them: at iteration j every wave has its own copies of step j landed (vmcnt), then the
// barrier makes all of step j readable and guarantees that every wave has finished reading step
// j-1.  The shared ring has D+1 slots, one more than the weight rings, so the slot of step j-1 is
// the one step j+D goes into: each iteration issues the weights and the activations of the same
// step, and the constant wait leaves D-1 whole steps of weights in flight, as with SN = 1.  All
// chunks then hold the same number of steps (the launcher's split), so every wave passes the same
// barriers.
// k order of a step: lane (row l % 16, kgroup g = l / 16) takes k [64h + 16g, 64h + 16g + 16) of
// each half h = 0, 1 -- the activation fragments use the same map.
// fmt 2: the zero-point and scale of (row, group) are staged in the wave's LDS before the loop
// (one group = one step).  EPI = 1 (fused gate/up, output width p.N, up rows from p.up): with
// SN = 1 each wave carries the gate row groups of its slab and the matching up row groups,
// combined in registers as in k_stream; with SN >= 2 the slab waves pair up -- waves sg < SN/2
// stream gate slabs, the others the matching up slabs (same activation ring) -- and each up
// result reaches its gate partner through LDS before the epilogue.
// Requirements (launcher): K % 128 == 0, the chunk a multiple of 128, N % (16 R SNO) == 0 with
// SNO the output slabs per workgroup (SN, or SN/2 when paired).
// ============================================================================================
template <int MB, int R, int D, int BFMT, int EPI = 0, int SN = 1>
struct StreamLine {
  // EPI with SN >= 2 pairs the slab waves (gate, up); with SN = 1 each wave carries both
  static constexpr bool PAIRED = EPI && SN >= 2;
  static_assert(!PAIRED || SN % 2 == 0, "paired gate/up slab waves");
  static constexpr int SNO = PAIRED ? SN / 2 : SN;       // output slabs per workgroup
  static constexpr int RR = EPI && !PAIRED ? 2 * R : R;  // row groups per wave
  static constexpr int EB = BFMT == 0 ? 2 : 1;           // bytes per weight
  static constexpr int MBE = MB > 0 ? MB : 1;            // 16-column blocks of the result
  static constexpr int WSLOT = RR * EB * 2048;           // weight bytes per step
  static constexpr int ASLOT = MB > 0 ? MB * 16 * 256 : 256;  // activation bytes per step
  // activation copies per step: MB > 0: 4 per 16 rows (1 KiB each), split over the SN slab
  // waves; MB = 0: every wave copies the whole 256-byte slice (one dword per lane) into the same
  // slot -- identical bytes, so the copies of different waves may land in any order -- which
  // keeps one copy per wave and step, whatever SN is
  static constexpr int LA = MB > 0 ? 4 * MB : SN;
  static constexpr int LAW = LA / SN;                    // ... issued by each wave
  static constexpr int L = 2 * RR * EB + LAW;            // copies per step per wave
  static constexpr int WAIT = (D - 1) * L;
  static constexpr int DA = SN > 1 ? D + 1 : D;          // slots of the shared activation ring
  static_assert(SN >= 1 && LA % SN == 0, "activation copies split evenly over the slab waves");
  static_assert(D >= 2 && (D - 1) * L < 64, "ring depth / vmcnt range");
  // LDS of one wave: D weight slots (+ its own activation ring when SN = 1) + (fmt 2) the staged
  // zero-points and scales of G groups; one shared activation ring per k chunk when SN > 1
  static constexpr size_t wave_bytes(int G) {
    return ((size_t)D * (WSLOT + (SN == 1 ? ASLOT : 0)) +
            (BFMT == 2 ? ((size_t)RR * 16 * G * 3 + 15) / 16 * 16 : 0) + 1023) / 1024 * 1024;
  }
  static constexpr size_t act_bytes() { return SN > 1 ? ((size_t)DA * ASLOT + 1023) / 1024 * 1024 : 0; }
  // S > 1: the k chunks' partial sums ([S][SN][RR][MBE] x 1 KiB) are reduced through LDS; they
  // reuse the rings (all waves are past their loops then) except in the paired epilogue, whose
  // up-to-gate exchange uses the start of the LDS after the reduction
  static constexpr size_t red_bytes(int S) { return (size_t)S * SN * RR * MBE * 1024; }
  static constexpr size_t lds(int S, int G) {
    const size_t rings = (size_t)S * (SN * wave_bytes(G) + act_bytes());
    if (S <= 1) return rings;
    return PAIRED ? rings + red_bytes(S) : (rings > red_bytes(S) ? rings : red_bytes(S));
  }
};

__device__ __forceinline__ int line_key(int row16) { return (row16 >> 1) & 7; }

// The body of k_stream_line for the workgroup that covers slab group `wgi` (SNO output slabs).
template <int MB, int R, int D, int BFMT, int EPI, int SN>
__device__ __forceinline__ void line_body(const StreamArgs& p, int G, int wgi, int ksi,
                                          uint8_t* dsm) {
  using SL = StreamLine<MB, R, D, BFMT, EPI, SN>;
  constexpr int RR = SL::RR, EB = SL::EB, MBE = SL::MBE, WSLOT = SL::WSLOT, ASLOT = SL::ASLOT;
  constexpr int WSTRIDE = SN == 1 ? WSLOT + ASLOT : WSLOT;  // bytes per ring slot of a wave
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sg = wave % SN, kc = wave / SN;  // slab of the workgroup, k chunk
  const size_t wbytes = SL::wave_bytes(G);
  uint8_t* group = dsm + kc * (SN * wbytes + SL::act_bytes());  // k chunk's LDS
  uint8_t* ring = group + SL::act_bytes() + sg * wbytes;         // this wave's weight ring
  // activation slot of step j: inside the wave's own ring slot (SN = 1) or the shared ring
  auto aslot = [&](int j) -> uint8_t* {
    return SN == 1 ? ring + (j % D) * WSTRIDE + WSLOT : group + (j % SL::DA) * ASLOT;
  };
  uint8_t* meta_z = ring + D * WSTRIDE;                                  // fmt 2: [RR*16][G]
  _Float16* meta_s = reinterpret_cast<_Float16*>(meta_z + (RR * 16 * G + 1) / 2 * 2);
  const int S = p.S;  // k chunks
  f32x4* red = reinterpret_cast<f32x4*>(SL::PAIRED ? dsm + S * (SN * wbytes + SL::act_bytes())
                                                   : dsm);

  const int k0 = ksi * p.kspan, k1 = ksi * p.kspan + (p.ks > 1 ? p.kspan : p.K);  // k slice
  const int kbeg = min(k1, k0 + kc * p.chunk);
  const int kend = min(k1, kbeg + p.chunk);
  const int n = (kend - kbeg) / 128;  // steps of this wave (>= 1; equal in all chunks if SN > 1)
  const int r16 = lane & 15, kg = lane >> 4;
  constexpr bool PAIRED = SL::PAIRED;
  const bool upw = PAIRED && sg >= SN / 2;                         // paired: an up wave
  const int nbase = (wgi * SL::SNO + (PAIRED ? sg % (SN / 2) : sg)) * 16 * R;
  auto row_of = [&](int r) -> long {  // first row of row group r
    if constexpr (PAIRED) return (upw ? (long)p.up : 0L) + nbase + r * 16;
    return EPI && r >= R ? (long)p.up + nbase + (r - R) * 16 : (long)nbase + r * 16;
  };

  // weight copy (r, h, i) fills rows 8i .. 8i+7 of row group r with line h of the step; lane l
  // takes slot l: row 8i + l/8, physical chunk l%8, i.e. logical chunk (l%8) ^ key(row)
  const uint8_t* wsrc[RR][2];
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int rr = 8 * i + lane / 8;
      const int c = (lane % 8) ^ line_key(rr);
      wsrc[r][i] = reinterpret_cast<const uint8_t*>(p.B) + ((row_of(r) + rr) * p.ldb + kbeg) * EB + c * 16;
    }
  // activation copies: MB = 0 -> lane l takes bytes [4l, 4l+4) of row 0's 256-byte slice (every
  // wave the whole slice); MB > 0 -> copy t fills rows 4t .. 4t+3, lane l the physical chunk l%16
  // of row 4t + l/16, and this wave issues copies t = sg + SN*u, u < LAW.
  const uint8_t* asrc[SL::LAW];
#pragma unroll
  for (int u = 0; u < SL::LAW; ++u) {
    const int t = sg + SN * u;
    if constexpr (MB == 0) {
      asrc[u] = reinterpret_cast<const uint8_t*>(p.A) + 2L * kbeg + 4 * lane;
    } else {
      const int m = 4 * t + lane / 16;
      const int c = (lane % 16) ^ (m & 15);
      asrc[u] = reinterpret_cast<const uint8_t*>(p.A + (long)min(m, p.M - 1) * p.lda) + 2L * kbeg + c * 16;
    }
  }
  auto dma_w = [&](int j) {
    const int jj = min(j, n - 1);
    uint8_t* slot = ring + (j % D) * WSTRIDE;
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int h = 0; h < EB; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          void* src = (void*)(wsrc[r][i] + (long)jj * 128 * EB + 128 * h);
          lds_void_stream_t* dst = (lds_void_stream_t*)(slot + (r * EB + h) * 2048 + i * 1024);
          // the weights stream through once (nontemporal: not kept in the caches), except with
          // row tiles, whose workgroups on one XCD read the same weight rows from its L2
          if (p.mtiles > 1)
            __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
          else
            __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 2 /* nt */);
        }
  };
  auto dma_a = [&](int j) {
    const int jj = min(j, n - 1);
    uint8_t* slot = aslot(j);
#pragma unroll
    for (int u = 0; u < SL::LAW; ++u) {
      if constexpr (MB == 0)
        __builtin_amdgcn_global_load_lds((void*)(asrc[u] + jj * 256),
                                         (lds_void_stream_t*)slot, 4, 0, 0);
      else
        __builtin_amdgcn_global_load_lds((void*)(asrc[u] + jj * 256),
                                         (lds_void_stream_t*)(slot + (sg + SN * u) * 1024), 16, 0, 0);
    }
  };

  _Float16 rscale[RR];
  if constexpr (BFMT == 1) {
#pragma unroll
    for (int r = 0; r < RR; ++r) rscale[r] = p.scale[row_of(r) + r16];
  }
  // prologue: copy units in the loop's order -- weights of step j, then its activations
  for (int j = 0; j < D; ++j) {
    dma_w(j);
    dma_a(j);
  }
  if constexpr (BFMT == 2) {  // this wave's zero-points and scales, one group per step
    // entry i of [RR*16 rows][n groups] is lane i % 64's, batches of 8 per lane: the loads of a
    // batch are in flight together before the LDS stores wait on them.  Each lane steps its
    // (row, group) by 64 entries with the wave-uniform quotient and remainder of 64 / n (one
    // division per wave, not one per entry: per-entry divisions cost 10-20% of a fmt 2 decode
    // launch)
    const long gstride = p.K / 128;
    const int g0 = kbeg / 128;
    const int nn = max(n, 1);
    const int tot = RR * 16 * n;
    const int q64 = 64 / nn, r64 = 64 - q64 * nn;
    int row0 = lane / nn, col0 = lane - row0 * nn;
    for (int i0 = lane; i0 < tot; i0 += 64 * 8) {
      uint8_t zz[8];
      _Float16 ss[8];
      int row = row0, g = col0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (i0 + 64 * u < tot) {
          const long gi = (row_of(row / 16) + row % 16) * gstride + g0 + g;
          zz[u] = p.zero[gi];
          ss[u] = p.scale[gi];
        }
        g += r64;
        row += q64;
        if (g >= nn) {
          g -= nn;
          ++row;
        }
      }
      row = row0;
      g = col0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        if (i0 + 64 * u < tot) {
          meta_z[row * G + g] = zz[u];
          meta_s[row * G + g] = ss[u];
        }
        g += r64;
        row += q64;
        if (g >= nn) {
          g -= nn;
          ++row;
        }
      }
      row0 = row;
      col0 = g;
    }
  }
  __builtin_amdgcn_s_waitcnt(0);  // prologue copies landed, scales and metadata loaded
  if constexpr (SN > 1) __syncthreads();

  f32x4 acc[RR][MBE], acc2[RR][MBE];
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int b = 0; b < MBE; ++b) {
      acc[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
      acc2[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
  const int key = line_key(r16);

  // fragments of half h of step j (weights of every row group, activations of every block)
  auto read_w = [&](const uint8_t* slot, int r, int h, u32x4 (&w)[2]) {
    if constexpr (BFMT == 0) {
#pragma unroll
      for (int q = 0; q < 2; ++q)
        w[q] = *reinterpret_cast<const u32x4*>(slot + (r * 2 + h) * 2048 + r16 * 128 +
                                               (((2 * kg + q) ^ key) * 16));
    } else {
      w[0] = *reinterpret_cast<const u32x4*>(slot + r * 2048 + r16 * 128 + (((4 * h + kg) ^ key) * 16));
    }
  };
  auto read_a = [&](const uint8_t* as, int b, int h, u32x4 (&a)[2]) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int c = 8 * h + 2 * kg + q;  // 16-byte chunk of the 256-byte activation slice
      if constexpr (MB == 0)
        a[q] = *reinterpret_cast<const u32x4*>(as + c * 16);
      else
        a[q] = *reinterpret_cast<const u32x4*>(as + (16 * b + r16) * 256 + ((c ^ r16) * 16));
    }
  };
  auto dequant = [&](const u32x4 (&w)[2], int r, uint8_t z, _Float16 sc, f16x8& w0, f16x8& w1) {
    if constexpr (BFMT == 0) {
      w0 = as_f16x8(w[0]);
      w1 = as_f16x8(w[1]);
    } else if constexpr (BFMT == 1) {
      w0 = dequant8_i8(w[0][0], w[0][1], rscale[r]);
      w1 = dequant8_i8(w[0][2], w[0][3], rscale[r]);
    } else {
      w0 = dequant8_u8(w[0][0], w[0][1], z, sc);
      w1 = dequant8_u8(w[0][2], w[0][3], z, sc);
    }
  };

  for (int j = 0; j < n; ++j) {
    asm volatile("" ::: "memory");
    s_wait_vm_stream<SL::WAIT>();  // this wave's copies of step j have landed
    if constexpr (SN > 1) __builtin_amdgcn_s_barrier();  // ... and everyone's
    asm volatile("" ::: "memory");
    const uint8_t* slot = ring + (j % D) * WSTRIDE;
    const uint8_t* as = aslot(j);
    uint8_t z[RR];
    _Float16 sc[RR];
    if constexpr (BFMT == 2) {
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        z[r] = meta_z[(16 * r + r16) * G + j];
        sc[r] = meta_s[(16 * r + r16) * G + j];
      }
    }
    // early reads hold a whole step's fragments (8 RR EB + 16 MBE VGPRs) beside the
    // accumulators (8 RR MBE): within 80 of them the kernel stays inside its register budget
    // (the fp16 form with two row groups and two activation blocks, 96, spilled)
    if constexpr (MB <= 2 && 8 * RR * EB + 16 * MBE + 8 * RR * MBE <= 80) {
      // early reads: every fragment of the step into registers, then the slot is refilled while
      // the MFMAs run
      u32x4 w[RR][2][2], a[MBE][2][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int b = 0; b < MBE; ++b) read_a(as, b, h, a[b][h]);
#pragma unroll
        for (int r = 0; r < RR; ++r) read_w(slot, r, h, w[r][h]);
      }
      // the fences keep the matrix work below the copies: left to itself the scheduler moves
      // MFMAs and dequantisation between the reads, each read then waits on its own and the
      // next step's copies go out only after all of them
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): slot j is read, it may be refilled
      asm volatile("" ::: "memory");
      dma_w(j + D);
      dma_a(j + D);  // SN > 1: slot (j-1) % (D+1), free since the barrier
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < RR; ++r) {
          f16x8 w0, w1;
          dequant(w[r][h], r, z[r], sc[r], w0, w1);
#pragma unroll
          for (int b = 0; b < MBE; ++b) {
            acc[r][b] = Mfma<16>::run(w0, as_f16x8(a[b][h][0]), acc[r][b]);
            acc2[r][b] = Mfma<16>::run(w1, as_f16x8(a[b][h][1]), acc2[r][b]);
          }
        }
    } else {
      // late reads (many activation blocks or row groups): half by half, fragments read just
      // before their MFMAs; the slot is refilled once both halves are done
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 w[RR][2];
#pragma unroll
        for (int r = 0; r < RR; ++r) read_w(slot, r, h, w[r]);
        f16x8 w0[RR], w1[RR];
#pragma unroll
        for (int r = 0; r < RR; ++r) dequant(w[r], r, z[r], sc[r], w0[r], w1[r]);
#pragma unroll
        for (int b = 0; b < MBE; ++b) {
          u32x4 a[2];
          read_a(as, b, h, a);
#pragma unroll
          for (int r = 0; r < RR; ++r) {
            acc[r][b] = Mfma<16>::run(w0[r], as_f16x8(a[0]), acc[r][b]);
            acc2[r][b] = Mfma<16>::run(w1[r], as_f16x8(a[1]), acc2[r][b]);
          }
        }
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): slot j is read, it may be refilled
      asm volatile("" ::: "memory");
      dma_w(j + D);
      dma_a(j + D);
    }
  }
  s_wait_vm_stream<0>();  // the copies past the end land before the LDS is reused
#pragma unroll
  for (int r = 0; r < RR; ++r)
#pragma unroll
    for (int b = 0; b < MBE; ++b) acc[r][b] += acc2[r][b];

  if (S > 1) {  // partial sums of the S k chunks of each slab, added in chunk order
    if constexpr (!PAIRED) __syncthreads();  // every wave is past its ring reads: reuse them
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int b = 0; b < MBE; ++b) red[((wave * RR + r) * MBE + b) * 64 + lane] = acc[r][b];
    __syncthreads();
    if (kc != 0) return;
#pragma unroll
    for (int r = 0; r < RR; ++r)
#pragma unroll
      for (int b = 0; b < MBE; ++b) {
        f32x4 t = red[((sg * RR + r) * MBE + b) * 64 + lane];
        for (int c = 1; c < S; ++c) {
          const f32x4 v = red[(((c * SN + sg) * RR + r) * MBE + b) * 64 + lane];
          t[0] += v[0]; t[1] += v[1]; t[2] += v[2]; t[3] += v[3];
        }
        acc[r][b] = t;
      }
  }
  if constexpr (PAIRED) {
    // every wave is past its last ring read (vmcnt 0 above; the barrier below or the reduction's)
    // so ring memory of chunk 0 carries the up results to their gate partners
    f32x4* xb = reinterpret_cast<f32x4*>(dsm);
    if (S == 1) __syncthreads();
    if (upw) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < MBE; ++b) xb[(((sg - SN / 2) * R + r) * MBE + b) * 64 + lane] = acc[r][b];
    }
    __syncthreads();
    if (upw) return;
    f32x4 both[2 * R][MBE];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int b = 0; b < MBE; ++b) {
        both[r][b] = acc[r][b];
        both[R + r][b] = xb[((sg * R + r) * MBE + b) * 64 + lane];
      }
    stream_store<MBE, R, 1>(p, both, nbase, r16, kg);
  } else if (EPI == 0 && p.ks > 1) {
    stream_store_part<MBE, R>(p, acc, nbase, r16, kg, ksi);
  } else {
    stream_store<MBE, R, EPI>(p, acc, nbase, r16, kg);
  }
}

// TL = 1 (SN > 1, one k chunk): the grid is p.nbig workgroups of SN slab waves -- a whole number
// of them per CU -- followed by one workgroup per remaining output slab, in which wave 0 streams
// that slab over the whole K with its own activation ring (the body with SN = 1; for the fused
// gate/up, EPI = 1, waves 0 and 1 stream its gate and up rows as a pair on a shared activation
// ring, the body with SN = 2) and the other waves leave at once.  (A single tail wave carrying
// both gate and up streamed twice the bytes of the other waves and set the launch's end: the
// M = 32 gate/up row lost 4-7 % to the unfused chain with it.)  A grid of whole rounds plus at
// most one such tail per CU keeps the slabs per
// CU within one of each other; with workgroups of SN slabs alone, a partial last round puts
// 2 SN slabs on some CUs and SN on others (N = 34816, SN = 4: 8 or 12).
template <int MB, int R, int D, int BFMT, int EPI = 0, int SN = 1, int TPB = 1024, int TL = 0>
__global__ __launch_bounds__(TPB) void k_stream_line(StreamArgs p, int G) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t dsm[];
  if constexpr (TL) {
    static_assert(SN > 1, "tail workgroups: a shared activation ring in the whole rounds");
    constexpr int SNO = StreamLine<MB, R, D, BFMT, EPI, SN>::SNO;  // output slabs per workgroup
    // tail workgroups: one output slab each, on one wave, or (gate/up) on a pair of waves, gate
    // and up, so that a tail wave streams as many weight rows as a wave of the whole rounds.
    // The other waves of the block leave at once; the pair's barriers wait only for the waves
    // still running.
    constexpr int TSN = EPI ? 2 : 1;
    const int wgi = blockIdx.x;
    if (wgi >= p.nbig) {
      if (threadIdx.x >= 64 * TSN) return;
      line_body<MB, R, D, BFMT, EPI, TSN>(p, G, p.nbig * SNO + (wgi - p.nbig), 0, dsm);
      return;
    }
  }
  if (p.mtiles > 1) {
    // row tiles (one k slice): workgroup b takes row tile mi of slab group sgi, the row tiles of
    // one slab group on one XCD (workgroups go to the 8 XCDs round robin) so their weight rows
    // stream from HBM into that XCD's L2 once
    const int b = blockIdx.x, groups = (int)gridDim.x / p.mtiles;
    int mi, sgi;
    if (groups % 8 == 0) {
      const int j = b / 8;
      mi = j % p.mtiles;
      sgi = (j / p.mtiles) * 8 + b % 8;
    } else {
      mi = b % p.mtiles;
      sgi = b / p.mtiles;
    }
    StreamArgs q = p;
    q.A = p.A + (long)mi * p.mrows * p.lda;
    q.C = p.C + (long)mi * p.mrows * p.ldc;
    q.M = min(p.mrows, p.M - mi * p.mrows);
    line_body<MB, R, D, BFMT, EPI, SN>(q, G, sgi, 0, dsm);
    return;
  }
  const int wgi = p.ks > 1 ? (int)blockIdx.x / p.ks : (int)blockIdx.x;
  line_body<MB, R, D, BFMT, EPI, SN>(p, G, wgi, (int)blockIdx.x - wgi * p.ks, dsm);
}

// ===== common/splitk_host.h =====
// common/splitk_host.h -- host side of the split-K launches, frozen into each delivery's
// kernel.hip after the kernels (it names k_splitk_reduce): the workspace a split-K row needs,
// where it comes from, and how many splits a row takes.
//
// A split-K row adds fp32 partial sums of its k ranges, [splits][M][N], in a workspace and reduces
// them with k_splitk_reduce on the same stream.  The workspace is either memory the caller hands
// over, or the delivery's pool: one buffer per (device, stream), allocated on first use and grown
// when a larger shape needs it, so calls on different streams stay independent.  A call is two
// kernels, and a stream orders kernels, not calls: the pool's buffer is leased, locked from before
// the first is enqueued until after the second, so that no other thread's partial sums land
// between them.

// Workspace of a split-K row.  `ptr`/`bytes`: device memory the caller hands over (may be
// null / 0), `shared` where calls on other streams take the same memory; `pool`: the row may take
// the delivery's per-(device, stream) pool instead; `need`: when set, the row only reports the
// bytes it needs (0 for rows without a workspace) and launches nothing.
struct Workspace {
  void* ptr = nullptr;
  size_t bytes = 0;
  bool pool = false;
  bool shared = false;
  size_t* need = nullptr;
};

// The workspace of one call, from workspace_for() until the call's last kernel is enqueued.  ptr is
// null where none could be had; `held` locks a pool buffer (nothing for the caller's memory).
struct Lease {
  float* ptr = nullptr;
  std::unique_lock<std::mutex> held;
};

// The pool: one buffer per (device, stream), grown on demand.  A buffer that a larger shape
// outgrows is retired, not freed: work already queued on the stream or a graph captured earlier
// may still use it, so it stays allocated until the process ends.  Sizes are whole powers of two
// from 1 MiB, so the retired buffers of a stream together stay below its current one.  Growing
// needs hipMalloc, which a stream under graph capture cannot take: there the pool returns
// hipErrorStreamCaptureUnsupported and the caller hands over its workspace instead (launch_with,
// or the C ABI's *_launch_ws entry points).  (The frozen file's preamble includes <map>, <mutex>,
// <utility> and <vector>.)
struct PoolBuffer {
  std::mutex busy;
  void* ptr = nullptr;
  size_t bytes = 0;
  std::vector<void*> retired;
};
inline Lease pool_lease(hipStream_t s, size_t bytes, hipError_t* err) {
  static std::mutex mu;
  static std::map<std::pair<int, hipStream_t>, PoolBuffer> pool;  // nodes keep their address
  Lease l;
  int dev = 0;
  if ((*err = hipGetDevice(&dev)) != hipSuccess) return l;
  PoolBuffer* e = nullptr;
  {
    std::lock_guard<std::mutex> lock(mu);
    e = &pool[std::make_pair(dev, s)];
  }
  std::unique_lock<std::mutex> held(e->busy);
  if (e->bytes < bytes) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if ((*err = hipStreamIsCapturing(s, &cs)) != hipSuccess) return l;
    if (cs != hipStreamCaptureStatusNone) {
      *err = hipErrorStreamCaptureUnsupported;
      return l;
    }
    size_t size = (size_t)1 << 20;
    while (size < bytes) size *= 2;
    // another stream's capture, which would forbid this thread's hipMalloc, is none of its concern
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    if ((*err = hipThreadExchangeStreamCaptureMode(&mode)) != hipSuccess) return l;
    void* q = nullptr;
    const hipError_t got = hipMalloc(&q, size);
    *err = hipThreadExchangeStreamCaptureMode(&mode);
    if (got != hipSuccess) {
      (void)hipGetLastError();  // the caller may go on without a workspace
      *err = hipErrorOutOfMemory;
      return l;
    }
    if (e->ptr) e->retired.push_back(e->ptr);
    e->ptr = q;
    e->bytes = size;
  }
  l.ptr = static_cast<float*>(e->ptr);
  l.held = std::move(held);
  return l;
}

// The workspace of a split-K launch: the caller's if it is large enough, else the pool's when the
// row may take it.  Null with *err set otherwise (hipErrorOutOfMemory: the caller's buffer is
// too small and no pool was allowed).
inline Lease workspace_for(const Workspace& w, size_t bytes, hipStream_t s, hipError_t* err) {
  *err = hipSuccess;
  if (w.pool && !(w.ptr && w.bytes >= bytes)) return pool_lease(s, bytes, err);
  Lease l;
  if (w.ptr && w.bytes >= bytes)
    l.ptr = static_cast<float*>(w.ptr);
  else
    *err = hipErrorOutOfMemory;
  return l;
}

// The workspace of a split that a row only gains by: its own path needs `own` bytes.  Where that is
// none, the call takes no memory that work on another stream may be using -- a `shared` workspace,
// the pool of a stream under capture (its graph may be replayed on any stream), the pool under
// hipStreamPerThread (one handle, a stream per thread) -- so that calls which need nothing share
// nothing.
inline Lease workspace_to_gain(const Workspace& w, size_t bytes, size_t own, hipStream_t s,
                               hipError_t* err) {
  if (own == 0) {
    const bool given = w.ptr && w.bytes >= bytes;
    bool refuse = given ? w.shared : w.pool && s == hipStreamPerThread;
    if (!given && w.pool && !refuse) {
      hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
      if (hipStreamIsCapturing(s, &cs) != hipSuccess) {
        (void)hipGetLastError();  // the caller goes on without a workspace
        refuse = true;
      }
      refuse = refuse || cs != hipStreamCaptureStatusNone;
    }
    if (refuse) {
      *err = hipErrorOutOfMemory;
      return Lease{};
    }
  }
  return workspace_for(w, bytes, s, err);
}

// Split count of a split-K row: the most splits such that tiles x splits stays within `slots`
// workgroups (one round of the part: a split count that spills into a second round makes every
// split of that round wait for it), each split keeping at least `minkt` k-tiles, and no split
// empty.  1 = no split.
inline int split_count(int tiles, int ktiles, int slots, int minkt) {
  if (slots <= 0 || minkt <= 0 || 2 * tiles > slots) return 1;
  int sp = slots / tiles;
  if (sp > ktiles / minkt) sp = ktiles / minkt;
  if (sp <= 1) return 1;
  const int per = (ktiles + sp - 1) / sp;
  return (ktiles + per - 1) / per;
}

// A plan picks, for one shape, the tile of the interleaved kernel and the split count with the
// least estimated time.  A table serves the rows up to m_max: microseconds per 1000 k of one round
// of a tile (one workgroup on each of the 256 CUs; per weight format), and what a round, a split
// (its second kernel) and a MB of partial sums (written and read) add.  The figures are fits to
// measured grids (100 .. 2200 workgroups; N = 1024 .. 34816, K = 2560 .. 17408) and order the
// alternatives only.  As times they are low: over random shapes at M > 64 with the weights from HBM
// splits take 1.16 times as long (median of 2054; 1.00 to 1.34 at the 5th and 95th percentile),
// unsplit tiles 1.09 times (of 2675; 0.91 to 1.67, the latter at short K) -- (200, 15360, 3840) fp16
// 42 us for 34, (2048, 2 x 17408, 5120) int8 620 for 501 -- for a round's rate depends on the clock
// under load and, below M = 256, on the HBM.
struct TileDims {
  int bm, bn, bk;
  bool splits;  // instantiated with split-K (the 256 x 256 tiles spill with it)
};
struct TileRate {
  int tile;
  double us[2];
};
struct PlanTable {
  int m_max;
  double round, split, mb;
  double weights;  // the least a million weights take (HBM), whatever the tile
  int n;
  TileRate rate[6];
};
struct TilePlan {
  int tile, splits;  // tile -1: none fits
  double us;
};
constexpr size_t kPlanWorkspace = (size_t)32 << 20;  // the allocation-free entry point's scratch

// The table of M rows (the last one has no bound).
inline const PlanTable& plan_table(const PlanTable* tabs, int M) {
  while (M > tabs->m_max) ++tabs;
  return *tabs;
}
inline double tile_us(const PlanTable& t, double rate, int bm, int bn, int bk, int M, int N, int K,
                      int splits) {
  const int ktiles = K / bk, per = (ktiles + splits - 1) / splits;
  const long wgs = (long)((M + bm - 1) / bm) * (N / bn) * splits;
  const double rounds = (double)((wgs + 255) / 256), hbm = t.weights * 1e-6 * N * K;
  double us = rounds * per * bk * rate * 1e-3;
  us = (us > hbm ? us : hbm) + rounds * t.round;
  return splits == 1 ? us : us + t.split + t.mb * 8e-6 * splits * M * N;
}
inline TilePlan plan_tiles(const TileDims* dims, const PlanTable* tabs, int f, int M, int N, int K,
                           bool split) {
  const PlanTable& t = plan_table(tabs, M);
  TilePlan best = {-1, 1, 0};
  for (int i = 0; i < t.n; ++i) {
    const TileDims& d = dims[t.rate[i].tile];
    if (N % d.bn || K % d.bk) continue;
    const int ktiles = K / d.bk;
    const long tiles = (long)((M + d.bm - 1) / d.bm) * (N / d.bn);
    for (int sp = 1; sp <= (split && d.splits ? 16 : 1); ++sp) {
      const int per = (ktiles + sp - 1) / sp;
      if (sp > 1 && (per * d.bk < 256 || tiles * sp > 512 ||
                     (size_t)sp * M * N * sizeof(float) > kPlanWorkspace))
        break;
      if ((ktiles + per - 1) / per != sp) continue;  // a split would be empty
      const double us = tile_us(t, t.rate[i].us[f], d.bm, d.bn, d.bk, M, N, K, sp);
      if (best.tile < 0 || us < best.us) best = {t.rate[i].tile, sp, us};
    }
  }
  return best;
}

// Launch of the split-K reduction: C = fp16_rn(sum over the splits of ws), in split order.
template <int UNROLL>
inline void run_reduce(const float* ws, int splits, int M, int N, _Float16* C, int ldc,
                       hipStream_t s) {
  const long work = (long)M * N / 4;
  hipLaunchKernelGGL(k_splitk_reduce<UNROLL>, dim3((unsigned)((work + 255) / 256)), dim3(256), 0, s,
                     ws, splits, M, N, C, ldc);
}
inline hipError_t launch_reduce(const float* ws, int splits, int M, int N, _Float16* C, int ldc,
                                hipStream_t s) {
  switch (splits) {  // every split's load in flight at once
    case 2: run_reduce<2>(ws, splits, M, N, C, ldc, s); break;
    case 3: run_reduce<3>(ws, splits, M, N, C, ldc, s); break;
    case 4: run_reduce<4>(ws, splits, M, N, C, ldc, s); break;
    case 5: run_reduce<5>(ws, splits, M, N, C, ldc, s); break;
    case 6: run_reduce<6>(ws, splits, M, N, C, ldc, s); break;
    case 7: run_reduce<7>(ws, splits, M, N, C, ldc, s); break;
    case 1: run_reduce<1>(ws, splits, M, N, C, ldc, s); break;
    default: run_reduce<8>(ws, splits, M, N, C, ldc, s);
  }
  return hipGetLastError();
}

// The same for the fused gate/up product: ws holds [S][M][2N] sums, the gate columns then the up
// columns.
inline hipError_t launch_reduce_gu(const float* ws, int splits, int M, int N, _Float16* C, int ldc,
                                   hipStream_t s) {
  const long work = (long)M * N / 4;
  const dim3 grid((unsigned)((work + 255) / 256)), blk(256);
  if (splits <= 2)
    hipLaunchKernelGGL(k_splitk_reduce_gu<2>, grid, blk, 0, s, ws, splits, M, N, C, ldc);
  else
    hipLaunchKernelGGL(k_splitk_reduce_gu<4>, grid, blk, 0, s, ws, splits, M, N, C, ldc);
  return hipGetLastError();
}

}  // namespace gen
}  // namespace tempo
