// fp32 GEMMs and scans on the bf16 matrix cores of gfx950.
//
// An fp32 value is the sum of three bf16 values, x = x1 + x2 + x3 (8 + 8 + 8
// significant bits: x1 and x2 rounded to nearest, so |x2| <= 2^-8 |x| and |x3|
// <= 2^-17 |x|, either sign; exact above 2^-109, below it x3 is a bf16 subnormal,
// off by at most 2^-133), and a product a b is taken as the six partial products
// a1 b1, a1 b2, a2 b1, a2 b2, a1 b3, a3 b1, exact in the fp32 accumulators of
// v_mfma_f32_16x16x32_bf16 (which keeps subnormal operands); the three
// left out are below 2^-24 + 2^-34 of |a b|, of either sign.  The signs matter:
// an MFMA drops bits of products far below its accumulator, and with x1
// truncated (x2 of x's sign) a sum of 4096 positive products lost 3.6e-6 of its
// value, 5.3e-7 with x1 rounded and 8.5e-7 on the native fp32 MFMA.  An MFMA
// sums 32 k at once where the native fp32 MFMA sums 2, so a long dot product
// rounds fewer times than it does there: error relative to the sum of |a b|,
// normal operands, K = 64, 1024, 4096: 1.8e-8, 2.4e-8, 2.5e-8 against 2.8e-8.
// Six bf16 products per fp32 one: 2500 / 6 = 417 TFLOP/s against the fp32
// units' 157.  Measured against the native fp32 MFMA (32x32x2) kernels this
// replaces: 170 against 110 TFLOP/s in the GEMMs; 1000 tokens, hidden 1000,
// teacher hidden 1200, vocabulary 30001: 2.44 -> 1.49 ms a step, gradients off
// float64 by 6.4e-7 of their norm against 9e-7; 512 x 256 x 4096: 504 -> 128 us
// of kernels.  All eight products down to 2^-34 take 1.70 ms for the former at
// the same error.  The matrix cores are busy 56% of the cycles at 1.94 GHz (the
// socket's power limit).
//
// Operands without such a split (infinities, values that round past the bf16
// range) and sums of at most 16 products, where six roundings are more than the
// sum's own (one product: 3.4e-8 of it against 2.5e-8): the tile is done over on
// the native fp32 MFMA before it is written out.  The loaders keep the largest
// magnitude they split (under 1% of the first call above); looking at it in
// every K step took 7% of that call and multiplying single steps natively there
// 9% (loads issued later, registers).
//
// Workgroup: WA x 2 waves, wave tile (16 MB) squared, K steps of 32.  An
// operand's K step goes global -> registers (the step after next's loads are
// in flight during this one's MFMAs) -> split once per workgroup -> three
// bf16 planes in one of two LDS stages, from where each wave reads its
// fragments (16 bytes per lane) as the 16-bit kernels do.  One barrier per
// step: of the two waves on a SIMD one multiplies this step and then splits
// the next, the other splits first, so a SIMD's vector and matrix units are
// both busy.  K-contiguous and MN-contiguous operands differ only in the
// loader: the latter transposes 4 x 4 values in registers on its way into
// LDS, so no operand needs a transposed copy in memory.
//
// MB = 4, WA = 4: 256 x 128 tiles, 8 waves, 144 KiB of LDS, one workgroup to a
// CU.  MB = 2, WA = 2: 64 x 64 tiles, 4 waves, 48 KiB, three to a CU, for
// problems whose large tiles would leave CUs idle.
//
// LDS plane: 64 bytes (32 k) per row, four rows per 256-byte bank line.  Row
// r, x = (r / 4) % 4, sits in slot (r ^ x) % 4 of its line and its 16-byte
// chunk c at c ^ f(x) ^ 2 ((r / 16) % 2), f = 0, 2, 3, 1.  A fragment read
// serves lanes 0-3, 12-15, 20-23 and 24-27 (and so on) at a time: rows 0-3 and
// 12-15 of one chunk with rows 4-7 and 8-11 of the next, distinct positions
// for this f (c ^ x put two of the four on the same banks: 4 more cycles per
// read).  A transposed write's 8 row quads x 4 k quads and a K-contiguous
// write's 4 rows x 8 k quads cover the line as well.
#pragma once
#include "kernels.hpp"

namespace orda {

constexpr int kS3Step = 32;  // K elements per step

template <int MB_, int WA_>
struct S3Cfg {
  static constexpr int MB = MB_, WA = WA_;
  static constexpr int kThreads = WA * 128;
  static constexpr int kRowsA = 16 * MB * WA, kRowsB = 32 * MB;
  static constexpr int kStage = (kRowsA + kRowsB) * 192;  // three planes of 64 bytes per row
  static constexpr int kLds = 2 * kStage + 16;  // and the marks
};
using S3Big = S3Cfg<4, 4>;
using S3Small = S3Cfg<2, 2>;

__device__ __forceinline__ uint32_t s3_addr(int row, int chunk) {
  const int x = (row >> 2) & 3;
  const int f = (((x ^ (x >> 1)) & 1) << 1) | (x >> 1);
  return (uint32_t)((row >> 2) * 256 + (((row & 3) ^ x) << 6) + ((chunk ^ f ^ (((row >> 4) & 1) << 1)) << 4));
}

// Largest magnitude that rounds to a finite bf16 value (0x7f7f7fff).
constexpr float kS3Max = 3.39617746e38f;
constexpr int kS3Short = 16;  // sums of at most this many products are native

// Four k values of one row to its three planes (8 bytes each, PL bytes apart)
// at `d`, the row's s3_addr plus 8 (k quad % 2) in the operand's first plane.
template <int PL>
__device__ __forceinline__ void s3_put(char* d, float x0, float x1, float x2, float x3) {
  float r[4], q[4];
  const uint2 p1 = make_uint2(pack2<bf16>(x0, x1), pack2<bf16>(x2, x3));
  r[0] = x0 - __uint_as_float(p1.x << 16);
  r[1] = x1 - __uint_as_float(p1.x & 0xffff0000u);
  r[2] = x2 - __uint_as_float(p1.y << 16);
  r[3] = x3 - __uint_as_float(p1.y & 0xffff0000u);
  const uint2 p2 = make_uint2(pack2<bf16>(r[0], r[1]), pack2<bf16>(r[2], r[3]));
  q[0] = r[0] - __uint_as_float(p2.x << 16);
  q[1] = r[1] - __uint_as_float(p2.x & 0xffff0000u);
  q[2] = r[2] - __uint_as_float(p2.y << 16);
  q[3] = r[3] - __uint_as_float(p2.y & 0xffff0000u);
  const uint2 p3 = make_uint2(
      __builtin_amdgcn_perm(__float_as_uint(q[1]), __float_as_uint(q[0]), 0x07060302u),
      __builtin_amdgcn_perm(__float_as_uint(q[3]), __float_as_uint(q[2]), 0x07060302u));
  *reinterpret_cast<uint2*>(d) = p1;
  *reinterpret_cast<uint2*>(d + PL) = p2;
  *reinterpret_cast<uint2*>(d + 2 * PL) = p3;
}

__device__ __forceinline__ float4 s3_load(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  const u4v_t v = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0);
  return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}
// All but 16 of the 2^32 bytes that a resource can address: 256 K-major rows of
// 2^22 values (the largest hidden size) stay below kS3Oob.
constexpr uint32_t kS3Oob = 0xfffffff0u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t s3_rsrc(const float* p) { return uniform_rsrc(p, kS3Oob); }

// (a NaN counts as nothing: its products are NaN on any path)
__device__ __forceinline__ float s3_largest(float m, const float4& x) {
  m = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), m);
  return fmaxf(fmaxf(fabsf(x.z), fabsf(x.w)), m);
}

// K-contiguous operand of R rows (NT threads): piece i of a thread is row
// NT / 8 i + tid / 8, k 4 (tid % 8) .. + 3.  Rows past `rows` and k past
// `krem` (a multiple of 4) read zero.  Pieces [I0, I1) of NP only: the tied
// scan keeps student and teacher rows in the two halves of B.
template <int R, int NT, int NP = R * 8 / NT>
struct S3K {
  static constexpr int kStride = NT / 8;
  float4 v[NP];
  template <int I0, int I1>
  __device__ __forceinline__ void load(const float* p, int64_t ld, int64_t rows, int64_t krem) {
    const int r = threadIdx.x >> 3, kq = threadIdx.x & 7;
    const auto rs = s3_rsrc(p);
#pragma unroll
    for (int i = I0; i < I1; ++i) {
      const int row = r + kStride * (i - I0);
      const bool ok = row < rows && kq * 4 < krem;
      v[i] = s3_load(rs, ok ? (uint32_t)row * (uint32_t)(ld * 4) + (uint32_t)(kq * 16) : kS3Oob);
    }
  }
  __device__ __forceinline__ void store(char* op) const {
    // (kStride, a multiple of 32, rows on is kStride / 4 bank lines on, at the
    // same slot and swizzle)
    const int r = threadIdx.x >> 3, kq = threadIdx.x & 7;
    char* d = op + s3_addr(r, kq >> 1) + (kq & 1) * 8;
#pragma unroll
    for (int i = 0; i < NP; ++i) s3_put<R * 64>(d + i * kStride * 64, v[i].x, v[i].y, v[i].z, v[i].w);
  }
  __device__ __forceinline__ float largest(float m) const {
#pragma unroll
    for (int i = 0; i < NP; ++i) m = s3_largest(m, v[i]);
    return m;
  }
};

// MN-contiguous operand of R rows (element (row, k) at p[k ld + row]): a
// thread takes 4 rows x 4 k; wave w rows 32 w .. + 31 (w < R / 32).  Rows past
// `cols` (read in fours: a quad whose first row is valid is readable) and k
// past krem read zero.
template <int R>
struct S3M {
  float4 v[4] = {};  // (zero in the waves that load nothing)
  __device__ __forceinline__ void load(const float* p, int64_t ld, int64_t cols, int64_t krem) {
    const int lane = threadIdx.x & 63, w = wave_id();
    if (w >= R / 32) return;
    const int m0 = w * 32 + (lane & 7) * 4, k0 = (lane >> 3) * 4;
    const auto rs = s3_rsrc(p);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool ok = m0 < cols && k0 + j < krem;
      v[j] = s3_load(rs, ok ? (uint32_t)(k0 + j) * (uint32_t)(ld * 4) + (uint32_t)(m0 * 4) : kS3Oob);
    }
  }
  __device__ __forceinline__ void store(char* op) const {
    const int lane = threadIdx.x & 63, w = wave_id();
    if (w >= R / 32) return;
    const int m0 = w * 32 + (lane & 7) * 4, kq = lane >> 3;
    const uint32_t a = s3_addr(m0, kq >> 1) + (uint32_t)((kq & 1) * 8);  // (row m0 + i: slot bits ^ i)
    s3_put<R * 64>(op + a, v[0].x, v[1].x, v[2].x, v[3].x);
    s3_put<R * 64>(op + (a ^ 64u), v[0].y, v[1].y, v[2].y, v[3].y);
    s3_put<R * 64>(op + (a ^ 128u), v[0].z, v[1].z, v[2].z, v[3].z);
    s3_put<R * 64>(op + (a ^ 192u), v[0].w, v[1].w, v[2].w, v[3].w);
  }
  __device__ __forceinline__ float largest(float m) const {
#pragma unroll
    for (int j = 0; j < 4; ++j) m = s3_largest(m, v[j]);
    return m;
  }
};

template <int MB>
using S3Acc = f32x4[MB][MB];

template <int MB>
__device__ __forceinline__ void s3_zero(S3Acc<MB>& acc) {
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// One K step of a wave: A rows 16 mb on from opA (the wave's first row), B
// rows brow(nb) on from opB, blocks nb in [J0, J1).  The wave's first row is a
// multiple of 32 and a block's of 16, so a fragment's address is one of two
// lane offsets (even and odd blocks) plus a constant.  Smallest products
// first.  SWAP: B x A^T.
template <class C, int J0, int J1, bool SWAP, class BRow>
__device__ __forceinline__ void s3_mul(S3Acc<C::MB>& acc, const char* opA, const char* opB, const BRow& brow) {
  constexpr int MB = C::MB;
  const int lane = threadIdx.x & 63;
  const uint32_t fo = s3_addr(lane & 15, lane >> 4);
  auto frag = [&](const char* op, int row0, int plane, int pl) __attribute__((always_inline)) {
    return *reinterpret_cast<const bf16x8*>(op + ((row0 & 16) ? fo ^ 32u : fo) + plane * pl + row0 * 64);
  };
  bf16x8 b[3][MB];
#pragma unroll
  for (int p = 0; p < 3; ++p)
#pragma unroll
    for (int nb = J0; nb < J1; ++nb) b[p][nb] = frag(opB, brow(nb), p, C::kRowsB * 64);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    bf16x8 a[3];
#pragma unroll
    for (int p = 0; p < 3; ++p) a[p] = frag(opA, mb * 16, p, C::kRowsA * 64);
    constexpr int pa[6] = {0, 2, 1, 0, 1, 0}, pb[6] = {2, 0, 1, 1, 0, 0};
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int nb = J0; nb < J1; ++nb) {
        f32x4& c = acc[mb][nb];
        if constexpr (SWAP) c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[pb[t]][nb], a[pa[t]], c, 0, 0, 0);
        else c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[pa[t]], b[pb[t]][nb], c, 0, 0, 0);
      }
  }
}

// The workgroup's marks, behind the second stage: mark i % 2 holds the last of
// its tiles i, counted from 1, with a value past kS3Max.  A thread marks tile i
// as it splits the tile's last step, a step before that is multiplied, and the
// mark is read when it has been: a barrier lies between, and one more before
// tile i + 2 writes there.
struct S3Marks {
  int* mark;
  float big = 0.f;
  __device__ __forceinline__ explicit S3Marks(char* p) : mark(reinterpret_cast<int*>(p)) {
    if (threadIdx.x < 2) mark[threadIdx.x] = 0;
    stage_barrier();
  }
  __device__ __forceinline__ void last_put(int tile) {
    if (big > kS3Max) mark[tile & 1] = tile + 1;
    big = 0.f;
  }
  __device__ __forceinline__ bool met(int tile) const {
    return __builtin_amdgcn_readfirstlane(mark[tile & 1]) == tile + 1;
  }
};

// The kernel's argument (its first), read where it is used: the rarely taken
// code below would keep a dozen of its fields in SGPRs through the K loop.
template <class P>
__device__ __forceinline__ const __attribute__((address_space(4))) P* s3_args() {
  uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return (const __attribute__((address_space(4))) P*)p;
}

// A wave's accumulators (blocks nb in [J0, J1)) += the products of k in [k0, k1)
// on the native fp32 MFMA (16x16x4): av(mb, k) and bv(nb, k) are the operands'
// values of the lane's row (lane % 16 of a block), from memory, zero outside it.
template <class C, int J0, int J1, bool SWAP, class AV, class BV>
__device__ __forceinline__ void s3_native(S3Acc<C::MB>& acc, int64_t k0, int64_t k1, const AV& av, const BV& bv) {
  const int kl = opaque_lane() >> 4;
#pragma unroll 1
  for (; k0 < k1; k0 += 4) {
    const int64_t k = k0 + kl;
    float b[C::MB];
#pragma unroll
    for (int nb = J0; nb < J1; ++nb) b[nb] = k < k1 ? bv(nb, k) : 0.f;
#pragma unroll
    for (int mb = 0; mb < C::MB; ++mb) {
      const float a = k < k1 ? av(mb, k) : 0.f;
#pragma unroll
      for (int nb = J0; nb < J1; ++nb) {
        f32x4& c = acc[mb][nb];
        if constexpr (SWAP) c = __builtin_amdgcn_mfma_f32_16x16x4f32(b[nb], a, c, 0, 0, 0);
        else c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b[nb], c, 0, 0, 0);
      }
    }
  }
}

// The K loop over `total` steps: put(stage) splits the loaded step into a
// stage, fetch(s) loads step s into registers, mul(s, stage) multiplies step
// s.  done(s) runs after step s's mul (a scan's epilogue).
template <class C, class Fetch, class Put, class Mul, class Done>
__device__ __forceinline__ void s3_loop(char* lds, int total, const Fetch& fetch, const Put& put, const Mul& mul,
                                        const Done& done) {
  if (total <= 0) return;
  const bool split_first = wave_id() >= C::WA;
  fetch(0);
  put(lds);
  if (total > 1) fetch(1);
  stage_barrier();
  for (int s = 0; s < total; ++s) {
    char* cur = lds + (s & 1) * C::kStage;
    char* nxt = lds + ((s & 1) ^ 1) * C::kStage;
    if (!split_first) mul(s, cur);
    if (s + 1 < total) {
      put(nxt);
      if (s + 2 < total) fetch(s + 2);
    }
    if (split_first) mul(s, cur);
    done(s);
    stage_barrier();
  }
}

// ------------------------------------------------------------------- GEMM
// C[M x N] (GEMM_STORE, GEMM_ACC_T: C +=, GEMM_SPLIT: split s's K range
// [s k_per_split, ...) to C32 + s split_stride, GEMM_ACC: C32 +=) A B^T, fp32.  A K-major or
// MN-major; B K-major (one segment), or MN-major, for a K-major A in up to two
// K segments as k_gemm2 (rows [0, b_kseg) from B, the first b_kval0 valid, the
// rest from B1).  Persistent: workgroup b (in XCD order) runs work items b, b +
// grid, ... (split-major, tiles banded as k_gemm2) as one step sequence, the
// next tile's loads in flight while this one is written out.  ldc a multiple of 4, C 16-byte aligned, and N a multiple of 4 or
// C's columns padded to one.
template <class C, int LA, int LB, int MODE>
__global__ __launch_bounds__(C::kThreads, C::MB == 4 ? 2 : 3) void k_gemm_s3(GemmParams P) {
  constexpr int MB = C::MB, RA = C::kRowsA, RB = C::kRowsB;
  __shared__ __attribute__((aligned(16))) char lds[C::kLds];
  const int tiles = P.tiles_m * P.tiles_n, total = tiles * P.splits;
  const int b0 = xcd_order(blockIdx.x, gridDim.x), grid = gridDim.x;
  const int nt = b0 < total ? (total - 1 - b0) / grid + 1 : 0;
  struct Tile {
    int split;
    int64_t m0, n0;
  };
  auto tile_of = [&](int i) {
    const int t_all = b0 + i * grid;
    Tile x;
    x.split = t_all / tiles;
    const int t = t_all - x.split * tiles;
    constexpr int G = 8;
    const int band = t / (G * P.tiles_n), first_m = band * G;
    const int gm = min(P.tiles_m - first_m, G), rem = t % (G * P.tiles_n);
    x.m0 = (int64_t)(first_m + rem % gm) * RA;
    x.n0 = (int64_t)(rem / gm) * RB;
    return x;
  };
  const float* A = static_cast<const float*>(P.A);
  const float* B = static_cast<const float*>(P.B);
  const float* B1 = static_cast<const float*>(P.B1);
  // steps of a tile's first segment and all its steps (a short last split's
  // run past its end and read zeros)
  const int64_t len0 = P.B1 ? P.b_kseg : P.k_per_split;
  const int s0 = (int)((len0 + kS3Step - 1) / kS3Step);
  const int steps = s0 + (P.B1 ? (int)((P.K - len0 + kS3Step - 1) / kS3Step) : 0);
  typename std::conditional<LA == KMAJ, S3K<RA, C::kThreads>, S3M<RA>>::type la;
  typename std::conditional<LB == KMAJ, S3K<RB, C::kThreads>, S3M<RB>>::type lb;
  int fi = 0, fs = 0;  // tile and step of the next fetch
  Tile f = tile_of(0);
  auto fetch = [&](int) __attribute__((always_inline)) {
    const bool second = fs >= s0;
    const int64_t kb = (int64_t)f.split * P.k_per_split;
    const int64_t k0 = (int64_t)(second ? fs - s0 : fs) * kS3Step;  // inside the segment
    const int64_t ka = second ? len0 + k0 : k0;                     // inside A's K range
    const int64_t end = min<int64_t>(P.K - kb, second ? P.K : len0);
    if constexpr (LA == KMAJ) la.template load<0, RA * 8 / C::kThreads>(A + f.m0 * P.lda + kb + ka, P.lda, P.M - f.m0, end - ka);
    else la.load(A + (kb + ka) * P.lda + f.m0, P.lda, P.M - f.m0, end - ka);
    if constexpr (LB == KMAJ) lb.template load<0, RB * 8 / C::kThreads>(B + f.n0 * P.ldb + kb + k0, P.ldb, P.N - f.n0, end - k0);
    else if (second) lb.load(B1 + k0 * P.ldb1 + f.n0, P.ldb1, P.N - f.n0, P.b_kval1 - k0);
    else lb.load(B + (kb + k0) * P.ldb + f.n0, P.ldb, P.N - f.n0, min<int64_t>(P.b_kval0 - kb, len0) - k0);
    if (++fs == steps) {
      fs = 0;
      if (++fi < nt) f = tile_of(fi);
    }
  };
  S3Marks marks(lds + 2 * C::kStage);
  int pi = 0, ps = 0;  // tile and step being split
  auto put = [&](char* st) __attribute__((always_inline)) {
    la.store(st);
    lb.store(st + RA * 192);
    marks.big = lb.largest(la.largest(marks.big));
    if (++ps == steps) {
      ps = 0;
      marks.last_put(pi++);
    }
  };
  const int w = wave_id(), wm = w >> 1, wn = w & 1;
  S3Acc<MB> acc;
  s3_zero<MB>(acc);
  auto mul = [&](int, const char* st) __attribute__((always_inline)) {
    s3_mul<C, 0, MB, true>(acc, st + wm * (16 * MB * 64), st + RA * 192 + wn * (16 * MB * 64), [](int nb) { return nb * 16; });
  };
  int mi = 0, ms = 0;  // tile and step being multiplied
  auto done = [&](int) __attribute__((always_inline)) {
    if (++ms < steps) return;
    ms = 0;
    const Tile x = tile_of(mi++);
    const int ol = opaque_lane();
    if (P.K <= kS3Short || marks.met(mi - 1)) {
      s3_zero<MB>(acc);
      const auto* q = s3_args<GemmParams>();
      const float* a = static_cast<const float*>(q->A);
      const float* b = static_cast<const float*>(q->B);
      const float* b1 = static_cast<const float*>(q->B1);
      const int64_t kb = (int64_t)x.split * q->k_per_split, seg = b1 ? q->b_kseg : q->K;
      const int64_t m = x.m0 + wm * 16 * MB + (ol & 15), n = x.n0 + wn * 16 * MB + (ol & 15);
      auto av = [&](int mb, int64_t k) {
        const int64_t r = m + mb * 16;
        return r < q->M ? a[LA == KMAJ ? r * q->lda + k : k * q->lda + r] : 0.f;
      };
      auto bv = [&](int nb, int64_t k) {
        const int64_t c = n + nb * 16;
        if (c >= q->N) return 0.f;
        if (LB == KMAJ) return b[c * q->ldb + k];
        if (k >= seg) return k - seg < q->b_kval1 ? b1[(k - seg) * q->ldb1 + c] : 0.f;
        return k < q->b_kval0 ? b[k * q->ldb + c] : 0.f;
      };
      s3_native<C, 0, MB, true>(acc, kb, min<int64_t>(q->K, b1 ? q->K : kb + q->k_per_split), av, bv);
    }
    const int mlim = (int)min<int64_t>(P.M - x.m0, RA), nlim = (int)min<int64_t>(P.N - x.n0, RB);
    float* D = (MODE == GEMM_SPLIT || MODE == GEMM_ACC ? P.C32 + x.split * P.split_stride : static_cast<float*>(P.C)) + x.m0 * P.ldc + x.n0;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = wm * 16 * MB + mb * 16 + (ol & 15);
#pragma unroll
      for (int nb = 0; nb < MB; ++nb) {
        const int n = wn * 16 * MB + nb * 16 + 4 * (ol >> 4);
        if (m < mlim && n < nlim) {
          float4* p = reinterpret_cast<float4*>(D + (int64_t)m * P.ldc + n);
          float4 o = make_float4(acc[mb][nb][0], acc[mb][nb][1], acc[mb][nb][2], acc[mb][nb][3]);
          if constexpr (MODE == GEMM_ACC_T || MODE == GEMM_ACC) {
            const float4 c = *p;
            o = make_float4(c.x + o.x, c.y + o.y, c.z + o.z, c.w + o.w);
          }
          *p = o;
        }
      }
    }
    s3_zero<MB>(acc);
  };
  s3_loop<C>(lds, nt * steps, fetch, put, mul, done);
}

// ------------------------------------------------------------------- scan
// 256 vocabulary rows x 128 columns of B.  ALONE: 128 student tokens, 4 per
// lane (teacher logits, if any, from memory).  TIED: 64 tokens, student rows
// in columns 0-63 and teacher rows of the same tokens in 64-127 (2 per lane,
// both logits of a token in the lane).  SEP (without STORE; with it the
// teacher's GEMM fills L first and ALONE reads it back, both fp32): the same
// columns, W x student rows and then W_t x teacher rows into their own halves.
struct Layout16x4 {
  static constexpr int kMB = 4, kR = 4;
  __device__ static constexpr int row(int mb, int r) { return mb * 16 + r; }
};
struct S3PairAP {
  using Lay = Layout16x4;
  const S3Acc<4>& a;
  int j;
  __device__ __forceinline__ float s(int mb, int r) const { return a[mb][j][r]; }
  __device__ __forceinline__ float t(int mb, int r) const { return a[mb][j + 2][r]; }
};
struct S3MemAP {
  using Lay = Layout16x4;
  const S3Acc<4>& a;
  int j;
  const float (&x)[4][4];
  __device__ __forceinline__ float s(int mb, int r) const { return a[mb][j][r]; }
  __device__ __forceinline__ float t(int mb, int r) const { return x[mb][r]; }
};
template <> struct GuardMasked<S3PairAP> : std::true_type {};
template <> struct GuardMasked<S3MemAP> : std::true_type {};
template <> struct GuardMaskedLin<S3PairAP> : std::true_type {};
template <> struct GuardMaskedLin<S3MemAP> : std::true_type {};
template <> struct GuardStudent<S3PairAP> : std::true_type {};
template <> struct GuardStudent<S3MemAP> : std::true_type {};

// The lane's token's teacher logits at its rows of the tile, from [N x V]
// memory or L's teacher columns (rows past V: unused).
__device__ __forceinline__ void s3_teacher(float (&x)[4][4], const FusedParams& P, int64_t t, int64_t v) {
  const bool tok = t < P.N;
  if (P.tsrc == TSRC_L) {
    const float* L = static_cast<const float*>(P.Lout) + v * P.ldL + P.tcolL + t;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int e = 0; e < 4; ++e) x[mb][e] = tok && v + mb * 16 + e < P.V ? L[(mb * 16 + e) * P.ldL] : 0.f;
    return;
  }
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) {
    const int64_t vb = v + mb * 16, off = t * P.V + vb;
    if (P.lt_dtype == DT_F32 && P.V % 4 == 0 && reinterpret_cast<uintptr_t>(P.Lt) % 16 == 0) {
      float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
      if (tok && vb < P.V) f = *reinterpret_cast<const float4*>(static_cast<const float*>(P.Lt) + off);
      x[mb][0] = f.x; x[mb][1] = f.y; x[mb][2] = f.z; x[mb][3] = f.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = tok && vb + e < P.V;
        if (P.lt_dtype == DT_F32) x[mb][e] = ok ? static_cast<const float*>(P.Lt)[off + e] : 0.f;
        else if (P.lt_dtype == DT_BF16) x[mb][e] = ok ? (float)static_cast<const bf16*>(P.Lt)[off + e] : 0.f;
        else x[mb][e] = ok ? (float)static_cast<const f16*>(P.Lt)[off + e] : 0.f;
      }
    }
  }
}

enum S3Teacher { S3_ALONE = 0, S3_TIED = 1, S3_SEP = 2 };
template <int SV, bool STORE, int TS>
__global__ __launch_bounds__(S3Big::kThreads, 2) void k_scan_s3(FusedParams P) {
  static_assert(TS != S3_SEP || !STORE, "stored: the teacher's GEMM runs on its own");
  using C = S3Big;
  constexpr int MB = 4, RA = C::kRowsA;
  constexpr bool PAIR = TS != S3_ALONE;
  constexpr int NJ = PAIR ? 2 : 4, kTok = PAIR ? 64 : 128;
  constexpr bool kPhase1 = sv_phase1(SV);
  __shared__ __attribute__((aligned(16))) char lds[C::kLds];
  const int lane = threadIdx.x & 63;
  const int w = wave_id(), wm = w >> 1, wn = w & 1;
  int tt, vr;
  grouped_tile<4>(xcd_order(blockIdx.x, gridDim.x), P.n_ttiles, P.n_vranges, tt, vr);
  const int64_t t0 = (int64_t)tt * kTok;
  const int vt0 = vr * P.tiles_per_range;
  const int ntiles = min(vt0 + P.tiles_per_range, P.n_vtiles) - vt0;
  // column of block nb within the wave's columns (from wcol, of either half);
  // the lane's token j: student in block j, teacher (PAIR) in block j + 2
  auto brow = [](int nb) { return PAIR ? (nb >> 1) * 64 + (nb & 1) * 16 : nb * 16; };
  const int wcol = wn * (PAIR ? 32 : 64);
  auto tok = [&](int j) { return t0 + wcol + j * 16 + (lane & 15); };

  RowState st[NJ];
  float lse_sT[NJ], lse_tT[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    state_init_fam(st[j], kPhase1 ? FAM_NONE : P.fam);
    lse_sT[j] = lse_tT[j] = 0.f;
    if (kPhase1 && tok(j) < P.N) {
      lse_sT[j] = P.rowp[1 * P.N + tok(j)];
      lse_tT[j] = P.rowp[3 * P.N + tok(j)];
    }
  }
  const float* W = static_cast<const float*>(P.W);
  const float* Wt = static_cast<const float*>(P.Wt);
  const float* hs = static_cast<const float*>(P.hs) + t0 * P.H;
  const float* ht = PAIR ? static_cast<const float*>(P.ht) + t0 * P.Ht : nullptr;
  const int64_t brows = P.N - t0;
  const int s0 = (int)((P.H + kS3Step - 1) / kS3Step);
  const int steps = s0 + (TS == S3_SEP ? (int)((P.Ht + kS3Step - 1) / kS3Step) : 0);  // per tile
  S3K<RA, C::kThreads> la;
  S3K<C::kRowsB, C::kThreads, TS == S3_SEP ? 1 : 2> lb;  // (SEP: the live half)
  int fv = vt0, fs = 0;  // tile and step of the next fetch (one call per step, in order)
  auto fetch = [&](int) __attribute__((always_inline)) {
    const int64_t v0 = (int64_t)fv * 256;
    if (TS != S3_SEP || fs < s0) {
      const int64_t k0 = (int64_t)fs * kS3Step;
      la.template load<0, 4>(W + v0 * P.H + k0, P.H, P.V - v0, P.H - k0);
      lb.template load<0, PAIR ? 1 : 2>(hs + k0, P.H, brows, P.H - k0);
      if constexpr (TS == S3_TIED) lb.template load<1, 2>(ht + k0, P.H, brows, P.H - k0);
    } else {
      const int64_t k0 = (int64_t)(fs - s0) * kS3Step;
      la.template load<0, 4>(Wt + v0 * P.Ht + k0, P.Ht, P.V - v0, P.Ht - k0);
      lb.template load<0, 1>(ht + k0, P.Ht, brows, P.Ht - k0);
    }
    if (++fs == steps) {
      fs = 0;
      ++fv;
    }
  };
  S3Marks marks(lds + 2 * C::kStage);
  int ps = 0, pv = 0;  // step and tile being split
  auto put = [&](char* sg) __attribute__((always_inline)) {
    la.store(sg);
    lb.store(sg + RA * 192 + (TS == S3_SEP && ps >= s0 ? 64 * 64 : 0));
    marks.big = lb.largest(la.largest(marks.big));
    if (++ps == steps) {
      ps = 0;
      marks.last_put(pv++);
    }
  };
  S3Acc<MB> acc;
  s3_zero<MB>(acc);
  int ms = 0, mv = vt0;  // step and tile being multiplied
  auto mul = [&](int, const char* sg) __attribute__((always_inline)) {
    const char* a = sg + wm * (16 * MB * 64);
    const char* b = sg + RA * 192 + wcol * 64;
    if (TS != S3_SEP || ms < s0) s3_mul<C, 0, TS == S3_SEP ? 2 : 4, false>(acc, a, b, brow);
    else s3_mul<C, 2, 4, false>(acc, a, b, brow);
  };
  auto done = [&](int) __attribute__((always_inline)) {
    if (++ms < steps) return;
    const int64_t v0 = (int64_t)mv * 256;
    ms = 0;
    ++mv;
    const int64_t vlimit = P.V - v0;
    const int ol = opaque_lane();  // (the epilogue's addresses stay out of the K loop's registers)
    const int vlane0 = wm * 64 + 4 * (ol >> 4);
    if (P.H <= kS3Short || (TS == S3_SEP && P.Ht <= kS3Short) || marks.met(mv - 1 - vt0)) {
      s3_zero<MB>(acc);
      const auto* q = s3_args<FusedParams>();
      auto rows = [&](const void* p, int64_t ld) {
        return [=](int mb, int64_t k) {
          const int64_t v = v0 + wm * 64 + mb * 16 + (ol & 15);
          return v < q->V ? static_cast<const float*>(p)[v * ld + k] : 0.f;
        };
      };
      auto cols = [&](const void* p, int64_t ld) {
        return [=](int nb, int64_t k) {
          const int64_t t = t0 + wcol + (PAIR ? nb & 1 : nb) * 16 + (ol & 15);
          return t < q->N ? static_cast<const float*>(p)[t * ld + k] : 0.f;
        };
      };
      s3_native<C, 0, PAIR ? 2 : 4, false>(acc, 0, q->H, rows(q->W, q->H), cols(q->hs, q->H));
      if constexpr (TS == S3_TIED) s3_native<C, 2, 4, false>(acc, 0, q->H, rows(q->W, q->H), cols(q->ht, q->H));
      if constexpr (TS == S3_SEP) s3_native<C, 2, 4, false>(acc, 0, q->Ht, rows(q->Wt, q->Ht), cols(q->ht, q->Ht));
    }
    if constexpr (STORE) {
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        const bool teacher = PAIR && nb >= 2;
        if (teacher && !P.store_t) break;
        const int64_t t = t0 + wcol + (teacher ? nb - 2 : nb) * 16 + (ol & 15);
        float* d = static_cast<float*>(P.Lout) + (v0 + vlane0) * P.ldL + t + (teacher ? P.tcolL : 0);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (t < P.N && vlane0 + mb * 16 + e < vlimit) d[e * P.ldL] = acc[mb][nb][e];
          d += 16 * P.ldL;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    static_for<0, NJ>([&](auto J) {
      constexpr int j = decltype(J)::value;
      if constexpr (PAIR) {
        scan_variant<SV>(st[j], S3PairAP{acc, j}, vlane0, vlimit, vlimit >= 256, lse_sT[j], lse_tT[j], P);
      } else {
        float x[4][4] = {};
        if (P.tsrc != TSRC_NONE) {
          s3_teacher(x, P, tok(j), v0 + vlane0);
          if constexpr (STORE) {
            if (P.tsrc == TSRC_MEM && P.store_t && tok(j) < P.N) {
              float* d = static_cast<float*>(P.Lout) + (v0 + vlane0) * P.ldL + P.tcolL + tok(j);
#pragma unroll
              for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                  if (vlane0 + mb * 16 + e < vlimit) d[e * P.ldL] = x[mb][e];
                d += 16 * P.ldL;
              }
            }
          }
        }
        scan_variant<SV>(st[j], S3MemAP{acc, j, x}, vlane0, vlimit, vlimit >= 256, lse_sT[j], lse_tT[j], P);
      }
    });
    s3_zero<MB>(acc);
  };
  s3_loop<C>(lds, ntiles * steps, fetch, put, mul, done);

  // combine lanes l ^ 16 and l ^ 32, then the four waves sharing the tokens
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    RowState o = shfl_state(st[j], 16);
    merge_any<kPhase1>(st[j], o, P);
    o = shfl_state(st[j], 32);
    merge_any<kPhase1>(st[j], o, P);
  }
  __syncthreads();
  float* xch = reinterpret_cast<float*>(lds);  // [wm - 1][wn][j][kNStat][16]
  auto at = [&](int m, int j) { return xch + (((m * 2 + wn) * NJ + j) * kNStat) * 16 + lane; };
  if (wm > 0 && lane < 16) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float* d = at(wm - 1, j);
      const float* sv = reinterpret_cast<const float*>(&st[j]);
#pragma unroll
      for (int f = 0; f < kNStat; ++f) d[f * 16] = sv[f];
    }
  }
  __syncthreads();
  if (wm == 0 && lane < 16) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      for (int m = 0; m < C::WA - 1; ++m) {
        RowState o;
        float* od = reinterpret_cast<float*>(&o);
        const float* sv = at(m, j);
#pragma unroll
        for (int f = 0; f < kNStat; ++f) od[f] = sv[f * 16];
        merge_any<kPhase1>(st[j], o, P);
      }
      if (tok(j) < P.N) {
        float* dst = P.partial + (int64_t)vr * kNStat * P.N + tok(j);
        const float* v = reinterpret_cast<const float*>(&st[j]);
#pragma unroll
        for (int f = 0; f < kNStat; ++f) dst[(int64_t)f * P.N] = v[f];
      }
    }
  }
}

}  // namespace orda
