// okq_gemm_f32.hip -- prefill dequant-GEMM for f32 activations with the
// weights dequantised in registers: Y[M,N] = X[M,K] W[N,K]^T (+bias), Q4_K,
// Q5_K, Q6_K and Q8_0, one or several matrices that read the same X.  bf16
// activations (one fp16 plane: kTwo false) take it where their own kernels
// do not pay: Q6_K grids too small for gemm_wide_q6k_kernel's tiles (us per
// call, against weights staged through LDS: 64 x 4096 -> 14336 80 -> 34, 300 x
// 4096 -> 14336 185 -> 100, 128 x 14336 -> 4096 61 -> 48, 33 x 4096 -> 4096 24
// -> 22), and Q4_K / Q5_K tensors within 256 rows of 4 GiB (elsewhere the
// kernels of okq_gemm_wide.hip and okq_gemm_pair.hip are faster: 128 x 4096 ->
// 1024 15.6 against 19.4).
//
// Numerics.  A = the pre-pass's row-scaled activations as two fp16 planes,
// x = hi + lo to 2^-22; B = the integer part of the weight, exact in fp16
// (Q4_K / Q5_K: sc * q; Q8_0: q; Q6_K: sc * (q - 32) as B1 = its fp16
// rounding and the exact remainder B2 in {-1, 0, 1}).  Both planes are
// contracted with B (Q6_K: hi with B1 and B2, lo with B1: lo * B2 is below
// 2^-22 of the product), so every product is exact and only f32 sums round;
// d is applied in f32 per super-block (Q8_0: per block of 32), with the
// Q4_K / Q5_K min term dmin * sum_j m_j xsum_j from one more MFMA.
//
// Per call, against a kernel that staged dequantised weights in LDS
// (us): 512 x 4096 -> 14336 Q4_K 219 -> 123, Q5_K 244 -> 136, Q6_K 306 -> 168,
// Q8_0 219 -> 152; 2048 x 14336 -> 4096 Q4_K 767 -> 450, Q6_K 1007 -> 602;
// 64 x 14336 -> 4096 Q4_K 58 -> 34; 33 x 4096 -> 4096 Q4_K 24 -> 20.
//
// What bounds it: the MFMAs, two per weight fragment and row block (Q6_K
// three) where bf16 activations need one, at the rate that the power budget
// leaves them.  So a weight is dequantised once for both planes, by the one
// wave that owns its column, and only the activations pass through LDS.
//
// Layout: one 8-wave workgroup per CU on a 128 x 256 tile; wave w owns
// columns 32w .. 32w+31 for all 128 rows (four 32x32x16 MFMA blocks).  A
// stage is half a super-block (128 K): 64 KB of activations (both planes) and
// 2 KB of per-32 sums, double-buffered in LDS by buffer-to-LDS copies one
// stage ahead; a super-block per stage would not fit twice.  The 16-byte
// chunk c of row r sits at chunk c ^ (r & 15).  A step (8 per stage, 16 K)
// contracts the hi fragments while the lo ones are read, then the lo
// fragments while the next step's hi ones are read and its weights
// dequantised: as many fragment registers as for one plane.
//   * K order inside a stage: MFMA step s, lane group g = lane / 32.
//     Q4_K / Q5_K: k = 64 g + 8 s + [0, 8) (lane group g reads the 32 qs bytes
//     of one chunk, low nibbles at steps 0-3).  Q6_K / Q8_0: k = 32 (s / 2) +
//     16 g + 8 (s & 1) + [0, 8) (a step stays inside one Q8_0 block and one
//     Q6_K scale).
#include "okq_device.h"
#include "okq_internal.h"

namespace okq {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f16x __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef __attribute__((address_space(3))) void *LdsPtr;

constexpr int kMaxM = 128;           // rows of the taller tile
constexpr int kFN = 256;             // tile columns (8 waves x 32)
constexpr int kPlane = kMaxM * 128;  // halves of one plane of a stage

__device__ __forceinline__ Rsrc make_rsrc(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}

// Activation stages: two buffers of [2 planes][128 rows][128 halves] and
// [128 rows][4 (hi, lo) per-32 sums]; distinct objects, so that the fragment
// reads of one do not wait for the loads into the other.
__shared__ __attribute__((aligned(16))) _Float16 fA0[2 * kPlane];
__shared__ __attribute__((aligned(16))) _Float16 fA1[2 * kPlane];
__shared__ __attribute__((aligned(16))) _Float16 fX0[kMaxM * 8];
__shared__ __attribute__((aligned(16))) _Float16 fX1[kMaxM * 8];
__shared__ __attribute__((aligned(16))) float fR[kMaxM];  // the tile's row scales for the epilogue

__device__ __forceinline__ h2 pk_fma(uint32_t spread, h2 m, h2 o) {
  return __builtin_elementwise_fma(__builtin_bit_cast(h2, spread), m, o);
}
__device__ __forceinline__ h2 splat(float v) {
  const _Float16 h = (_Float16)v;
  return h2{h, h};
}
__device__ __forceinline__ h8 join(h2 a, h2 b, h2 c, h2 d) { return h8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]}; }

// A lane's weights of one stage as loaded (Raw) and as the steps use them
// (Cur), per format.
template <int kType>
struct Raw;
template <int kType>
struct Cur;
template <>
struct Raw<kQ4_K> {
  u32x4 hd, q0, q1;
};
template <>
struct Cur<kQ4_K> {
  uint32_t q[8];
  h2 sc[2], off[2];  // low and high nibble planes
  h2 m;              // their mins (6-bit integers)
  float d, dmin;
};
template <>
struct Raw<kQ5_K> {
  u32x4 hd, q0, q1, r0, r1;
};
template <>
struct Cur<kQ5_K> : Cur<kQ4_K> {
  uint32_t hc[4];  // fifth bits: of bytes 8j .. 8j+3 in the low nibbles, 8j+4 .. 8j+7 in the high (bit = nibble plane)
};
template <>
struct Raw<kQ6_K> {
  u32x4 a, b, h;             // ql, ql + 32 and qh windows of 16 bytes
  uint32_t a4, b4, h4;       // their fifth dwords
  u32x3 s;
  uint32_t d;
};
template <>
struct Cur<kQ6_K> {
  uint32_t a[4], b[4], h[4];
  h2 sc[4];  // of quarters 0..3
  float d;
};
template <>
struct Raw<kQ8_0> {
  u32x4 v0, v1, v2, v3;
  uint32_t v4;
};
template <>
struct Cur<kQ8_0> {
  uint32_t q[4][4];
  uint32_t d01, d23;
};

}  // namespace

template <int kType, int kNB, bool kTwo>
__device__ __forceinline__ void f32_body(const _Float16 *__restrict__ xhi, const _Float16 *__restrict__ xlo,
                                         const h2 *__restrict__ xsum, const float *__restrict__ rscale, int M, int K,
                                         const PrefillMats &mats) {
  constexpr bool kMins = kType == kQ4_K || kType == kQ5_K;
  constexpr bool kPerBlock = kType == kQ8_0;  // d changes every 32 K
  constexpr bool kLow = kType == kQ6_K;       // a second weight plane
  constexpr uint32_t kSB = (uint32_t)sb_bytes_of(kType);
  constexpr int kFM = 32 * kNB;        // tile rows
  constexpr int kRW = kFM / 8;         // rows each wave copies
  constexpr int kCP = kRW / 4;         // its copy instructions per plane and stage (4 rows each)
  constexpr int kPieces = kTwo ? 2 * kCP : kCP;

  // Workgroup b runs on XCD b % 8; each matrix's (slice, tile) jobs are cut
  // into eight contiguous ranges, so every XCD holds its share of every
  // matrix, in the matrices' order.  Tiles go in groups of up to 8 M-tiles
  // (okq_gemm_wide.hip).
  const int b = (int)blockIdx.x;
  const int xcd = b % 8, xi = b / 8;
  const int x1 = sarg(mats.mat[1].px0), x2 = sarg(mats.mat[2].px0), x3 = sarg(mats.mat[3].px0);
  const int mi = (int)(xi >= x1) + (int)(xi >= x2) + (int)(xi >= x3);
  const PrefillMat &mt = mats.mat[mi];
  const uint8_t *const W = sarg(mt.w);
  const int N = sarg(mt.n), tiles = sarg(mt.tiles), ksplit = sarg(mt.ksplit);
  const int jobs = tiles * ksplit;
  const int job = xcd * sarg(mt.pxn) + xi - sarg(mt.px0);
  if (job >= jobs) return;
  const int z = job / tiles, tile = job % tiles;
  const int tiles_m = (M + kFM - 1) / kFM, tiles_n = tiles / tiles_m;
  const int grp = tile / (8 * tiles_n), rg = tile % (8 * tiles_n);
  const int gm = tiles_m - 8 * grp < 8 ? tiles_m - 8 * grp : 8;
  const int m0 = (8 * grp + rg % gm) * kFM;
  const int n0 = (rg / gm) * kFN;

  const int tid = (int)threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, cl = lane & 31;
  const int nsb_all = K >> 8;
  const int sb0 = (int)((int64_t)z * nsb_all / ksplit);
  const int nst = 2 * ((int)((int64_t)(z + 1) * nsb_all / ksplit) - sb0);  // stages (half super-blocks)
  const uint32_t row_bytes = (uint32_t)nsb_all * kSB;
  const uint32_t K2 = (uint32_t)K * 2u;

  const Rsrc rs_h = make_rsrc(xhi, (uint32_t)((size_t)M * K * 2));
  const Rsrc rs_l = make_rsrc(xlo, (uint32_t)((size_t)M * K * 2));
  const Rsrc rs_s = make_rsrc(xsum, (uint32_t)((size_t)M * (K / 32) * 4));
  const Rsrc rs_w = make_rsrc(W, (uint32_t)((size_t)N * row_bytes));

  // Activation copy of stage st: wave w moves rows kRW w .. kRW w + kRW - 1 of
  // both planes, four rows (1 KB) per instruction; lane L of instruction t
  // writes chunk L & 15 of row kRW w + 4t + L/16, which holds the row's logical
  // chunk (L & 15) ^ (row & 15).  Rows past M read past the planes: zeros.
  // The sums: lane L of wave w takes the 16 bytes of row 64 (w & 1) + L
  // (or, with 64 rows, L; the other waves repeat them, so that every wave
  // issues the same loads per stage).
  const uint32_t a_row = (uint32_t)(m0 + kRW * wave + (lane >> 4)) * K2;
  const int s_row = 64 * (wave % ((kFM + 63) / 64));
  const uint32_t s_off = (uint32_t)(m0 + s_row + lane) * (uint32_t)(K / 32) * 4u;
  auto copy_piece = [&](int t, int st, _Float16 *bufA) {
    const uint32_t kb = (uint32_t)(sb0 * 256 + st * 128);  // first K of the stage
    const int p = t / kCP, u = t % kCP;  // plane, instruction
    const uint32_t off = a_row + 16u * ((uint32_t)(lane & 15) ^ ((uint32_t)(kRW * wave + 4 * u + (lane >> 4)) & 15u));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(p == 0 ? rs_h : rs_l, (LdsPtr)(bufA + p * kPlane + (kRW * wave + 4 * u) * 128),
                                             16, off, (int)((uint32_t)u * 4u * K2 + kb * 2u), 0, 0);
  };
  auto copy_sums = [&](int st, _Float16 *bufX) {
    const uint32_t kb = (uint32_t)(sb0 * 256 + st * 128);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_s, (LdsPtr)(bufX + s_row * 8), 16, s_off, (int)(kb / 8u), 0, 0);
  };

  // This lane's weight column n0 + 32w + cl (columns past N take the last
  // one's weights: their outputs are not stored).
  const int col = n0 + 32 * wave + cl;
  const uint32_t w_col = (uint32_t)(col < N ? col : N - 1) * row_bytes;
  Raw<kType> raw;
  Cur<kType> cur;
  auto ldw = [&](uint32_t voff, uint32_t soff) { return __builtin_amdgcn_raw_buffer_load_b128(rs_w, voff, (int)soff, 0); };
  auto ldw1 = [&](uint32_t voff, uint32_t soff) { return __builtin_amdgcn_raw_buffer_load_b32(rs_w, voff, (int)soff, 0); };
  auto ld_raw = [&](int st) {
    const uint32_t so = (uint32_t)(sb0 + (st >> 1)) * kSB, h = (uint32_t)(st & 1);
    if constexpr (kMins) {
      const uint32_t vq = w_col + (kType == kQ5_K ? 48u : 16u) + 32u * (uint32_t)g;
      raw.hd = ldw(w_col, so);
      raw.q0 = ldw(vq, so + 64u * h);
      raw.q1 = ldw(vq + 16u, so + 64u * h);
      if constexpr (kType == kQ5_K) {
        raw.r0 = ldw(w_col + 16u, so);
        raw.r1 = ldw(w_col + 32u, so);
      }
    } else if constexpr (kType == kQ6_K) {
      // super-blocks are 210 bytes: dword windows starting r = 0 or 2 bytes early
      const uint32_t base = w_col + so, a = base & ~3u;
      const uint32_t gq = 64u * h + 16u * (uint32_t)g, gh = 128u + 32u * h + 16u * (uint32_t)g;
      raw.a = ldw(a + gq, 0);
      raw.a4 = ldw1(a + gq + 16u, 0);
      raw.b = ldw(a + gq + 32u, 0);
      raw.b4 = ldw1(a + gq + 48u, 0);
      raw.h = ldw(a + gh, 0);
      raw.h4 = ldw1(a + gh + 16u, 0);
      raw.s = __builtin_amdgcn_raw_buffer_load_b96(rs_w, a + 192u + 8u * h, 0, 0);
      raw.d = __builtin_amdgcn_raw_buffer_load_b16(rs_w, base + 208u, 0, 0);
    } else {
      // blocks 2g and 2g + 1 of the stage whole (68 bytes)
      const uint32_t v = w_col + 68u * (uint32_t)g, s2 = so + 136u * h;
      raw.v0 = ldw(v, s2);
      raw.v1 = ldw(v + 16u, s2);
      raw.v2 = ldw(v + 32u, s2);
      raw.v3 = ldw(v + 48u, s2);
      raw.v4 = ldw1(v + 64u, s2);
    }
  };
  // raw (of stage st) -> cur
  auto prepare = [&](int st, const int h) {
    if constexpr (kMins) {
      const uint32_t q[8] = {raw.q0.x, raw.q0.y, raw.q0.z, raw.q0.w, raw.q1.x, raw.q1.y, raw.q1.z, raw.q1.w};
#pragma unroll
      for (int i = 0; i < 8; ++i) cur.q[i] = q[i];
      const uint32_t j0 = 4u * (uint32_t)h + 2u * (uint32_t)g;  // sub-block of the low nibble plane
      cur.dmin = f16_bits_hw(raw.hd.x >> 16);
      cur.d = f16_bits_hw(raw.hd.x & 0xffffu);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        // low planes take (sc, -1024 sc) on 0x6400 | q = 1024 + q; high
        // planes, masked in place (1024 + 16 q), (sc / 16, -64 sc)
        uint32_t sc, mv;
        q4k_scale_min_sel(j0 + (uint32_t)u, raw.hd.y, raw.hd.z, raw.hd.w, sc, mv);
        const float f = (float)sc;
        cur.sc[u] = splat(u ? f * 0.0625f : f);
        cur.off[u] = splat(u ? -64.0f * f : -1024.0f * f);
        cur.m[u] = (_Float16)(float)mv;
      }
      if constexpr (kType == kQ5_K) {
        // bits 2g, 2g + 1 (half 0) or 4 + 2g, 5 + 2g (half 1) of every byte
        const uint32_t sh = 4u * (uint32_t)h + 2u * (uint32_t)g;
        const uint32_t r[8] = {raw.r0.x, raw.r0.y, raw.r0.z, raw.r0.w, raw.r1.x, raw.r1.y, raw.r1.z, raw.r1.w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          cur.hc[j] = ((r[2 * j] >> sh) & 0x03030303u) | (((r[2 * j + 1] >> sh) & 0x03030303u) << 4);
      }
    } else if constexpr (kType == kQ6_K) {
      const uint32_t r = (w_col + (uint32_t)(sb0 + (st >> 1)) * kSB) & 3u;
      auto fit = [&](const u32x4 &w, uint32_t w4, uint32_t o[4]) {
        o[0] = realign(w.y, w.x, r);
        o[1] = realign(w.z, w.y, r);
        o[2] = realign(w.w, w.z, r);
        o[3] = realign(w4, w.w, r);
      };
      fit(raw.a, raw.a4, cur.a);
      fit(raw.b, raw.b4, cur.b);
      fit(raw.h, raw.h4, cur.h);
      // this lane group's scales: bytes g + 2t of the half's 8
      const uint32_t s0 = realign(raw.s.y, raw.s.x, r) >> (8 * g), s1 = realign(raw.s.z, raw.s.y, r) >> (8 * g);
      cur.sc[0] = splat((float)(int8_t)s0);
      cur.sc[1] = splat((float)(int8_t)(s0 >> 16));
      cur.sc[2] = splat((float)(int8_t)s1);
      cur.sc[3] = splat((float)(int8_t)(s1 >> 16));
      cur.d = f16_bits_hw(raw.d & 0xffffu);
    } else {
      // the lane groups trade halves, so that each holds its 16 q bytes of
      // all four blocks (okq_gemm_q8.hip)
      const uint32_t w[17] = {raw.v0.x, raw.v0.y, raw.v0.z, raw.v0.w, raw.v1.x, raw.v1.y, raw.v1.z, raw.v1.w, raw.v2.x,
                              raw.v2.y, raw.v2.z, raw.v2.w, raw.v3.x, raw.v3.y, raw.v3.z, raw.v3.w, raw.v4};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const auto a = __builtin_amdgcn_permlane32_swap(realign(w[k + 1], w[k], 2u), realign(w[k + 5], w[k + 4], 2u),
                                                        false, false);
        cur.q[0][k] = a[0] ^ 0x80808080u;
        cur.q[2][k] = a[1] ^ 0x80808080u;
        const auto c = __builtin_amdgcn_permlane32_swap(w[9 + k], w[13 + k], false, false);
        cur.q[1][k] = c[0] ^ 0x80808080u;
        cur.q[3][k] = c[1] ^ 0x80808080u;
      }
      const uint32_t dd = __builtin_amdgcn_perm(w[8], w[0], 0x07060100u);
      const auto d = __builtin_amdgcn_permlane32_swap(dd, dd, false, false);
      cur.d01 = d[0];
      cur.d23 = d[1];
    }
  };

  // B fragment(s) of step s
  auto dequant = [&](int s, h8 &b1, h8 &b2) {
    if constexpr (kMins) {
      const uint32_t d0 = cur.q[2 * (s & 3)], d1 = cur.q[2 * (s & 3) + 1];
      const bool hi = (s >> 2) != 0;
      const uint32_t mask = hi ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
      uint32_t n0v = d0 & mask, n1v = d1 & mask;
      uint32_t e0 = 0x64646464u, e1 = 0x64646464u;
      uint32_t s00 = 0x04010400u, s01 = 0x04030402u;
      if constexpr (kType == kQ5_K) {
        // the fifth bit: bit 4 of the byte on low planes (1024 + q5), the
        // exponent byte on high planes (1024 + 256 h + 16 q4 = 1024 + 16 q5)
        const uint32_t bit = (uint32_t)(s >> 2), c = cur.hc[s & 3];
        const uint32_t h0 = (c >> bit) & 0x01010101u, h1 = (c >> (bit + 4u)) & 0x01010101u;
        if (hi) {
          e0 |= h0;
          e1 |= h1;
          s00 = 0x05010400u;
          s01 = 0x07030602u;
        } else {
          n0v |= h0 << 4;
          n1v |= h1 << 4;
        }
      }
      const h2 sc = cur.sc[s >> 2], off = cur.off[s >> 2];
      b1 = join(pk_fma(__builtin_amdgcn_perm(e0, n0v, s00), sc, off), pk_fma(__builtin_amdgcn_perm(e0, n0v, s01), sc, off),
                pk_fma(__builtin_amdgcn_perm(e1, n1v, s00), sc, off), pk_fma(__builtin_amdgcn_perm(e1, n1v, s01), sc, off));
    } else if constexpr (kType == kQ6_K) {
      const int t = s >> 1, e = 2 * (s & 1);
      const uint32_t q0 = (t & 1) ? cur.b[e] : cur.a[e], q1 = (t & 1) ? cur.b[e + 1] : cur.a[e + 1];
      const uint32_t n0v = ((t >> 1) ? q0 : q0 << 4) & 0xF0F0F0F0u, n1v = ((t >> 1) ? q1 : q1 << 4) & 0xF0F0F0F0u;
      const uint32_t e0 = 0x64646464u | ((cur.h[e] >> (2 * t)) & 0x03030303u);
      const uint32_t e1 = 0x64646464u | ((cur.h[e + 1] >> (2 * t)) & 0x03030303u);
      // (1024 + 16 q) / 16 - 96 = q - 32, exact; B1 its product with sc
      // rounded to fp16, B2 the exact remainder
      const h2 c16 = splat(0.0625f), c96 = splat(-96.0f), sc = cur.sc[t];
      const h2 v0 = pk_fma(__builtin_amdgcn_perm(e0, n0v, 0x05010400u), c16, c96);
      const h2 v1 = pk_fma(__builtin_amdgcn_perm(e0, n0v, 0x07030602u), c16, c96);
      const h2 v2 = pk_fma(__builtin_amdgcn_perm(e1, n1v, 0x05010400u), c16, c96);
      const h2 v3 = pk_fma(__builtin_amdgcn_perm(e1, n1v, 0x07030602u), c16, c96);
      const h2 p0 = v0 * sc, p1 = v1 * sc, p2 = v2 * sc, p3 = v3 * sc;
      b1 = join(p0, p1, p2, p3);
      b2 = join(__builtin_elementwise_fma(v0, sc, -p0), __builtin_elementwise_fma(v1, sc, -p1),
                __builtin_elementwise_fma(v2, sc, -p2), __builtin_elementwise_fma(v3, sc, -p3));
    } else {
      // 0x6400 | (q + 128) = 1152 + q, minus 1152
      const uint32_t w0 = cur.q[s >> 1][2 * (s & 1)], w1 = cur.q[s >> 1][2 * (s & 1) + 1];
      const h2 c = splat(-1152.0f);
      b1 = join(__builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04010400u)) + c,
                __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w0, 0x04030402u)) + c,
                __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04010400u)) + c,
                __builtin_bit_cast(h2, __builtin_amdgcn_perm(0x64646464u, w1, 0x04030402u)) + c);
    }
  };

  f16x acc[kNB], accs[kNB];
  u32x2 xs0[kNB];  // Q4_K / Q5_K: the first half's sums and mins, until the super-block folds
  h2 m0s;
  const f16x zero = {};
#pragma unroll
  for (int i = 0; i < kNB; ++i) acc[i] = zero;

  // A fragment of row block i at MFMA step s: row 32 i + cl, logical chunk c
  // (Q4_K / Q5_K: 8 g + s; otherwise 4 (s / 2) + 2 g + (s & 1)), stored at
  // chunk c ^ (cl & 15); the lane's part is opaque, so that the compiler keeps
  // one XOR per step instead of a register per step
  int a_lane = kMins ? cl * 256 + 128 * (g ^ ((cl >> 3) & 1)) : cl * 256, a_x = kMins ? cl & 7 : (2 * g) ^ (cl & 15);
  asm volatile("" : "+v"(a_lane), "+v"(a_x));
  auto a_addr = [&](int s) { return a_lane + 16 * ((kMins ? s : 4 * (s >> 1) + (s & 1)) ^ a_x); };
  auto a_at = [&](const _Float16 *bufA, int addr, int i) {
    return *reinterpret_cast<const h8 *>(reinterpret_cast<const char *>(bufA) + addr + 8192 * i);
  };

  // One stage (half h of a super-block, weights in cur) from (bufA, bufX),
  // stage st_next's activations copied into (nbufA, nbufX) meanwhile, one
  // copy instruction per step (the sums with the last).
  auto contract = [&](const _Float16 *bufA, const _Float16 *bufX, const int h, int st_next, _Float16 *nbufA,
                      _Float16 *nbufX) {
    h8 ah[kNB], al[kNB], b1, b2, n1, n2;
    float dj[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kPerBlock) {
      dj[0] = f16_bits_hw(cur.d01 & 0xffffu), dj[1] = f16_bits_hw(cur.d01 >> 16);
      dj[2] = f16_bits_hw(cur.d23 & 0xffffu), dj[3] = f16_bits_hw(cur.d23 >> 16);
    }
    auto fold = [&](int i, float d) {
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = __builtin_fmaf(d, accs[i][e], acc[i][e]);
    };
#pragma unroll
    for (int i = 0; i < kNB; ++i) ah[i] = a_at(bufA, a_addr(0), i);
    dequant(0, b1, b2);
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      if (kTwo || s < 7) {  // one plane: al takes the next step's fragments
        const int ad = a_addr(kTwo ? s : s + 1);
#pragma unroll
        for (int i = 0; i < kNB; ++i) al[i] = a_at(kTwo ? bufA + kPlane : bufA, ad, i);
      }
      if (s < kPieces) copy_piece(s, st_next, nbufA);
      if (kMins && s == 7) copy_sums(st_next, nbufX);
      __builtin_amdgcn_sched_barrier(0);  // the lo reads issue ahead of the hi MFMAs
      const bool restart = kPerBlock ? (s & 1) == 0 : (h == 0 && s == 0);
#pragma unroll
      for (int i = 0; i < kNB; ++i) {
        if (kPerBlock && restart && s > 0) fold(i, dj[(s >> 1) - 1]);
        accs[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], b1, restart ? zero : accs[i], 0, 0, 0);
      }
      if constexpr (kLow) {
#pragma unroll
        for (int i = 0; i < kNB; ++i) accs[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah[i], b2, accs[i], 0, 0, 0);
      }
      if constexpr (kTwo) {
        if (s < 7) {
          const int ad = a_addr(s + 1);
#pragma unroll
          for (int i = 0; i < kNB; ++i) ah[i] = a_at(bufA, ad, i);
        }
        __builtin_amdgcn_sched_barrier(0);  // and the next hi reads ahead of the lo MFMAs
#pragma unroll
        for (int i = 0; i < kNB; ++i) accs[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al[i], b1, accs[i], 0, 0, 0);
      } else if (s < 7) {
#pragma unroll
        for (int i = 0; i < kNB; ++i) ah[i] = al[i];
      }
      if (s < 7) {
        dequant(s + 1, n1, n2);
        b1 = n1;
        b2 = n2;
      }
    }
    if constexpr (kMins) {
      // this half's share of the min term: the (hi, lo) sums of the lane
      // group's two sub-blocks and their mins
      u32x2 xs[kNB];
#pragma unroll
      for (int i = 0; i < kNB; ++i) xs[i] = *reinterpret_cast<const u32x2 *>(bufX + (32 * i + cl) * 8 + 4 * g);
      if (h == 0) {
#pragma unroll
        for (int i = 0; i < kNB; ++i) xs0[i] = xs[i];
        m0s = cur.m;
      } else {
        // acc += d * accs - dmin * t with t = sum_j m_j xsum_j of the
        // super-block, formed apart: the two parts mostly cancel (q is
        // unsigned), so acc itself never takes either alone
        const h8 mb = h8{m0s[0], m0s[0], m0s[1], m0s[1], cur.m[0], cur.m[0], cur.m[1], cur.m[1]};
        const float d = cur.d, dmin = cur.dmin;
        f16x t[kNB];
#pragma unroll
        for (int i = 0; i < kNB; ++i)
          t[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              __builtin_bit_cast(h8, u32x4{xs0[i].x, xs0[i].y, xs[i].x, xs[i].y}), mb, zero, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < kNB; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float v = dmin * t[i][e];
            acc[i][e] += __builtin_fmaf(d, accs[i][e], -v);
          }
      }
    } else if constexpr (kPerBlock) {
#pragma unroll
      for (int i = 0; i < kNB; ++i) fold(i, dj[3]);
    } else if (h == 1) {
      const float d = cur.d;
#pragma unroll
      for (int i = 0; i < kNB; ++i) fold(i, d);
    }
  };

  // Pipeline: stage st reads buffer st & 1 while stage st + 1's weights go
  // into the raw registers (first) and its activations into the other buffer.
  // Every stage issues the same loads (past the last one they reload it: idle
  // buffer, dead registers), so the compiler's load counts stay exact; the
  // copy is last, so the wait for every load before the stage's one barrier
  // is the wait for it.
  const int last = nst - 1;
  auto clamp_st = [&](int st) { return st < last ? st : last; };
#pragma unroll
  for (int t = 0; t < kPieces; ++t) copy_piece(t, 0, fA0);
  if constexpr (kMins) copy_sums(0, fX0);
  if (tid < kFM) fR[tid] = m0 + tid < M ? rscale[m0 + tid] : 0.0f;
  ld_raw(0);
  __builtin_amdgcn_s_waitcnt(0);  // vmcnt(0) expcnt(0) lgkmcnt(0)
  prepare(0, 0);
  __syncthreads();
  constexpr int kWaitAll = 0x0070;  // vmcnt(0) expcnt(7) lgkmcnt(0), gfx9 encoding
  const int rows = M - m0 < kFM ? M - m0 : kFM;
  // rows whose scale is NaN (computed by the pre-pass), tested by every lane
  // of the wave before any lane leaves for a column past N
  const bool flagged =
      __builtin_amdgcn_ballot_w64(__builtin_isnan(fR[lane]) || (kFM > 64 && __builtin_isnan(fR[kFM - 64 + lane]))) != 0;
  // Q8_0 folds every 32 K: over a long K the folds' roundings would exceed
  // those of the MFMA sums they stand for (2048 rows x 14336 x 4096: 3.9e-7
  // from float64, 2.4e-7 for exact d * q planes in three MFMAs), so after every
  // kSegment stages the sums so far wait in the output (or partial) and a new
  // segment starts from zero: 2.1e-7, and 516 -> 554 us (825 with the planes).
  constexpr int kSegment = 28;
  float *const dst0 = (ksplit > 1 ? sarg(mt.part) + (size_t)z * M * N : sarg(mt.y)) + (size_t)m0 * N + col;
  // this lane's sums plus those parked (add), parked again (keep) or taken;
  // outside the stage loop and without branches, or the sums would spill
  auto parked = [&](bool add, bool keep) {
    // the tile's rows and columns through a range-checked descriptor: rows
    // past M end past it, columns past N and rows that the pre-pass wrote are
    // sent there.  (The lane's offset is opaque: hoisted out of the stage loop,
    // the 64 addresses would spill.)
    const Rsrc rs_y = make_rsrc(dst0 - col, (uint32_t)((size_t)rows * N * 4));
    uint32_t off = (uint32_t)(4 * g * N + col) * 4u;
    asm volatile("" : "+v"(off));
#pragma unroll
    for (int i = 0; i < kNB; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4 sc = *reinterpret_cast<const float4 *>(fR + 32 * i + 8 * j + 4 * g);
        const float sv[4] = {sc.x, sc.y, sc.z, sc.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int e = 4 * j + q;
          const bool out = col >= N || __builtin_isnan(sv[q]);
          const uint32_t o = out ? 0xFFFFFFF0u : off + (uint32_t)((32 * i + 8 * j + q) * N) * 4u;
          const float v =
              acc[i][e] + as_f32((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_y, add ? o : 0xFFFFFFF0u, 0, 0));
          __builtin_amdgcn_raw_buffer_store_b32(as_u32(v), rs_y, keep ? o : 0xFFFFFFF0u, 0, 0);
          acc[i][e] = keep ? 0.0f : v;
        }
        if (j & 1) __builtin_amdgcn_sched_barrier(0);  // 8 values in flight
      }
  };
  auto run = [&](int st, int end) {
    for (; st < end; st += 2) {
      ld_raw(st + 1);
      __builtin_amdgcn_sched_barrier(0);  // the prefetch issues first
      contract(fA0, fX0, 0, st + 1, fA1, fX1);
      prepare(st + 1, 1);
      __builtin_amdgcn_s_waitcnt(kWaitAll);
      __builtin_amdgcn_s_barrier();
      const int nx = st + 2 < nst ? st + 2 : last - 1;  // an even stage: the half that prepare assumes
      ld_raw(nx);
      __builtin_amdgcn_sched_barrier(0);
      contract(fA1, fX1, 1, clamp_st(st + 2), fA0, fX0);
      prepare(nx, 0);
      __builtin_amdgcn_s_waitcnt(kWaitAll);
      __builtin_amdgcn_s_barrier();
    }
  };
  if constexpr (kPerBlock) {
    for (int st = 0;; st += kSegment) {
      const bool done = st + kSegment >= nst;
      run(st, done ? nst : st + kSegment);
      if (nst <= kSegment) break;
      parked(st > 0, !done);
      if (done) break;
    }
  } else {
    run(0, nst);
  }

  // epilogue: lane (cl, g) holds rows 8 (e / 4) + 4 g + e % 4 of column cl
  // of each 32 x 32 block; split K stores the raw partial sums, otherwise the
  // row scale (from LDS) and the bias are applied.  A whole tile stores
  // without per-value row tests.
  if (col >= N) return;
  if (ksplit > 1) {
    float *dst = dst0;
    auto store = [&](bool guard) {
#pragma unroll
      for (int i = 0; i < kNB; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = 32 * i + 8 * (e >> 2) + 4 * g + (e & 3);
          if (!guard || r < rows) dst[(size_t)r * N] = acc[i][e];
        }
    };
    if (rows == kFM) {
      store(false);
    } else {
      store(true);
    }
    return;
  }
  const float *const bias = sarg(mt.bias);
  const float bv = bias ? bias[col] : 0.0f;
  float *dst = dst0;
  auto store = [&](bool guard, bool skip) {
#pragma unroll
    for (int i = 0; i < kNB; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int r0 = 32 * i + 8 * j + 4 * g;
        const float4 rs = *reinterpret_cast<const float4 *>(fR + r0);
        const float rv[4] = {rs.x, rs.y, rs.z, rs.w};
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if ((!guard || r0 + q < rows) && (!skip || !__builtin_isnan(rv[q])))
            dst[(size_t)(r0 + q) * N] = acc[i][4 * j + q] * rv[q] + bv;
      }
  };
  if (flagged) {
    store(true, true);
  } else if (rows == kFM) {
    store(false, false);
  } else {
    store(true, false);
  }
}

// Tiles of 32 kNB rows (a row's result does not depend on the height).
template <int kType, int kNB, bool kTwo>
__global__ __launch_bounds__(512) void gemm_f32_kernel(const _Float16 *__restrict__ xhi, const _Float16 *__restrict__ xlo,
                                                       const h2 *__restrict__ xsum, const float *__restrict__ rscale,
                                                       int M, int K, PrefillMats mats) {
  f32_body<kType, kNB, kTwo>(xhi, xlo, xsum, rscale, M, K, mats);
}

// Tile height in 32-row blocks: a stage of 2, 3 or 4 blocks takes about 0.6,
// 0.8 and 1 of the full tile's time (what does not scale is the weights'
// dequantisation and the loads), so the height of least total.
static int tile_blocks(int64_t M) {
  const int64_t c4 = 10 * ((M + 127) / 128), c3 = 8 * ((M + 95) / 96), c2 = 6 * ((M + 63) / 64);
  return c4 <= c3 && c4 <= c2 ? 4 : c3 <= c2 ? 3 : 2;
}
static int tile_rows(int64_t M) { return 32 * tile_blocks(M); }
int gemm_f32_blocks(int64_t M) { return tile_blocks(M); }
int gemm_f32_tiles(int64_t M, int64_t N) { return (int)(((M + tile_rows(M) - 1) / tile_rows(M)) * ((N + kFN - 1) / kFN)); }

hipError_t launch_gemm_f32(int type, const _Float16 *xhi, const _Float16 *xlo, const void *xsum, const float *rscale,
                           int64_t M, int64_t K, PrefillMats &mats, int count, hipStream_t s) {
  if (K % 256 != 0 || count < 1 || count > kPrefillMats) return hipErrorInvalidValue;
  int px = 0;
  for (int i = 0; i < kPrefillMats; ++i) {
    PrefillMat &m = mats.mat[i];
    if (i >= count) {
      m.px0 = INT32_MAX;
      continue;
    }
    if (m.ksplit < 1 || m.ksplit > K / 256) return hipErrorInvalidValue;
    m.tiles = gemm_f32_tiles(M, m.n);
    m.px0 = px;
    m.pxn = (m.tiles * m.ksplit + 7) / 8;
    px += m.pxn;
  }
  const dim3 grid((unsigned)(px * 8)), block(512);
  const h2 *sums = static_cast<const h2 *>(xsum);
  const int nb = tile_blocks(M);
#define OKQ_F32_NB(TYPE_, TWO_)                                                                                         \
  if (nb == 2)                                                                                                          \
    launch_timed(gemm_f32_kernel<TYPE_, 2, TWO_>, grid, block, 0u, s, xhi, xlo, sums, rscale, (int)M, (int)K, mats);     \
  else if (nb == 3)                                                                                                     \
    launch_timed(gemm_f32_kernel<TYPE_, 3, TWO_>, grid, block, 0u, s, xhi, xlo, sums, rscale, (int)M, (int)K, mats);     \
  else                                                                                                                  \
    launch_timed(gemm_f32_kernel<TYPE_, 4, TWO_>, grid, block, 0u, s, xhi, xlo, sums, rscale, (int)M, (int)K, mats)
#define OKQ_F32(TYPE_)          \
  if (xlo) {                    \
    OKQ_F32_NB(TYPE_, true);    \
  } else {                      \
    OKQ_F32_NB(TYPE_, false);   \
  }
  if (type == kQ4_K) {
    OKQ_F32(kQ4_K)
  } else if (type == kQ5_K) {
    OKQ_F32(kQ5_K)
  } else if (type == kQ6_K) {
    OKQ_F32(kQ6_K)
  } else if (xlo) {  // bf16 Q8_0: okq_gemm_q8.hip
    OKQ_F32_NB(kQ8_0, true);
  } else {
    return hipErrorInvalidValue;
  }
#undef OKQ_F32_NB
#undef OKQ_F32
  return hipGetLastError();
}

}  // namespace okq
