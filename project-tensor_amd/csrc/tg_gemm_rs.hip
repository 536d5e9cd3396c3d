// Register-staged GEMM on the 16-bit matrix cores:
//   C[z] = alpha * op(A[z]) @ op(B[z]) + beta * C[z] (+ bias)
// (reference: Tensor.__matmul__ and its closure, _core.py:999-1068), for fp32 operands.
//
// fp32 products.  Every fp32 operand element is split into three bf16 terms,
//   x = h + m + l,  h = bf16(x), m = bf16(x - h), l = bf16(x - h - m),
// round-to-nearest each (Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial
// Intelligence Datatype For Higher-Precision Computations", ARITH 2019).  24 significand bits
// fall into 8 + 8 + 8, so the split is exact.
// Of the nine products of two split operands the six with weight >= 2^-16 are kept,
//   hh + hm + mh + mm + hl + lh,
// accumulated in fp32; the three that are dropped (a term is at most 2^-8 of the one before
// it) are together at most 2^-24 of the product, and of either sign.  Six bf16 MFMAs
// (v_mfma_f32_32x32x16_bf16) replace eight fp32 ones (v_mfma_f32_32x32x2_f32) of twice the
// issue time each.
// Both operands are multiplied by 2^24 before they are split, and the sums by 2^-48 at the
// end: every fp32 number is a multiple of 2^-149, so every term of its split is one of
// 2^-125, a normal bf16 number, and the split is exact for subnormal operands too.  What
// that leaves to catch is overflow: a block that ends with a non-finite accumulator (an
// infinite or NaN operand, one of 2^104 or more, or a sum of 2^80 or more) computes its tile
// again on the fp32 matrix cores, operands unstaged: 8192x4096x1024 with an infinity in every
// row block 1430 us, 360 without.  (Unscaled, an operand below 2^-102 had to be redone the
// same way, and softmax outputs 71 below their row's maximum are such operands.)
//
// Block: WGM x WGN waves, each SM*32 x SN*32 of C.  k-tiles of 32 are loaded into
// registers (16-byte loads at element alignment), split, and written to LDS as three
// bf16 planes in the operand's own orientation ([row][32 k], or [k][columns] read back by
// ds_read_b64_tr_b16), double-buffered with one barrier per tile: while tile t is
// multiplied, tile t + 1 is split and stored and tile t + 2 is in flight.
// 16-byte chunks of a plane row are XOR-swizzled by the row, so reads and writes are free
// of bank conflicts.
#include "tg_gemm_rs.h"

#include <algorithm>
#include <cmath>

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short v4i16 __attribute__((ext_vector_type(4)));
#define TG_LDS_RS __attribute__((address_space(3)))

constexpr int BK = 32;
constexpr int kScaleExp = 24;  // operands are scaled by 2^kScaleExp
constexpr float kScale = 1 << kScaleExp;
constexpr int kTurn = 2 * BK;  // k extent of one partial sum

// Four floats at 4-byte alignment (a global load takes any dword address).
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

// XOR key of row r for rows of CH 16-byte chunks: the 16 (or, for 64-byte rows, 4 times
// 4) rows that a read instruction's bank cycle covers get distinct chunk positions.
template <int CH> __device__ __forceinline__ int rs_key(int r) {
  if (CH == 4) return (r >> 2) & 3;
  if (CH == 8) {
    const int x = (r >> 1) & 7;
    return ((x & 1) << 2) | (x >> 1);
  }
  return ((r & 3) << 2) | ((r >> 2) & 3);
}

// One operand's tile: EXT rows (m or n) by 32 k.  KC: contiguous along k in memory.
template <bool KC, int EXT, int NT>
struct RsOp {
  static constexpr int CH = KC ? BK / 8 : EXT / 8;    // 8-element chunks per stored row
  static constexpr int NCH = EXT * BK / 8 / NT;       // chunks per thread
  static constexpr int PLANE = EXT * BK * 2;          // bytes of one bf16 plane
  static_assert(NCH >= 1 && EXT * BK / 8 % NT == 0, "tile must split evenly over the threads");
  float v[NCH][8];
  const float* p[NCH];
  int64_t step;  // elements from one k-tile to the next
  int64_t lim;   // columns (m or n) of the matrix from the block's first one
  // g: the matrix; x0: the block's first row (m or n); xlim: rows of the matrix.
  __device__ __forceinline__ void init(const float* g, int64_t ld, int64_t x0, int64_t xlim) {
    lim = xlim - x0;
    step = KC ? BK : BK * ld;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int u = threadIdx.x + i * NT, r = u / CH, c = u % CH;
      if (KC) {
        // rows past the matrix read its last row: they only feed C entries never stored
        const int64_t row = r < lim ? x0 + r : xlim - 1;
        p[i] = g + row * ld + c * 8;
      } else {
        p[i] = g + r * ld + x0 + c * 8;
      }
    }
  }
  // Load the tile at p and advance.  kleft: k extent left from the tile's first k.
  // edge (uniform): some element lies past K or, for !KC, past the last column; those
  // read as zero.
  __device__ __forceinline__ void load(bool edge, int64_t kleft) {
    if (!edge) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const f32x4_u a = *reinterpret_cast<const f32x4_u*>(p[i]);
        const f32x4_u b = *reinterpret_cast<const f32x4_u*>(p[i] + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[i][e] = a[e];
          v[i][4 + e] = b[e];
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int u = threadIdx.x + i * NT, r = u / CH, c = u % CH;
        // valid elements of this chunk
        int64_t n = KC ? kleft - c * 8 : (r < kleft ? lim - c * 8 : 0);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = e < n ? p[i][e] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < NCH; ++i) p[i] += step;
  }
  // Split the held chunks, times `by` (+-kScale), into the three planes at lds.
  __device__ __forceinline__ void store(char* lds, float by) const {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int u = threadIdx.x + i * NT, r = u / CH, c = u % CH;
      const int off = r * CH * 16 + ((c ^ rs_key<CH>(r)) << 4);
      uint4 q[3];
      unsigned* qh = reinterpret_cast<unsigned*>(&q[0]);
      unsigned* qm = reinterpret_cast<unsigned*>(&q[1]);
      unsigned* ql = reinterpret_cast<unsigned*>(&q[2]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x0 = v[i][2 * e] * by, x1 = v[i][2 * e + 1] * by;
        const unsigned h = __builtin_bit_cast(unsigned, bf16x2{(__bf16)x0, (__bf16)x1});
        const float r0 = x0 - __builtin_bit_cast(float, h << 16);
        const float r1 = x1 - __builtin_bit_cast(float, h & 0xffff0000u);
        const unsigned m = __builtin_bit_cast(unsigned, bf16x2{(__bf16)r0, (__bf16)r1});
        const float s0 = r0 - __builtin_bit_cast(float, m << 16);
        const float s1 = r1 - __builtin_bit_cast(float, m & 0xffff0000u);
        qh[e] = h;
        qm[e] = m;
        ql[e] = __builtin_bit_cast(unsigned, bf16x2{(__bf16)s0, (__bf16)s1});
      }
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<uint4*>(lds + pl * PLANE + off) = q[pl];
    }
  }
};

// Fragment reader of one plane: 8 k-elements k = ks*16 + 8h + e of row/column
// wbase + 32 i + (lane % 32).
template <bool KC, int EXT, int S>
struct RsFrag {
  static constexpr int CH = KC ? BK / 8 : EXT / 8;
  int off[KC ? BK / 16 : 2 * S];
  __device__ __forceinline__ void init(int lane, int wbase) {
    const int l32 = lane & 31, h = lane >> 5;
    if (KC) {
#pragma unroll
      for (int ks = 0; ks < BK / 16; ++ks)
        off[ks] = (wbase + l32) * (BK * 2) + (((2 * ks + h) ^ rs_key<CH>(l32)) << 4);
    } else {
      const int s = lane & 15, nh = (lane >> 4) & 1;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < S; ++i) {
          const int row = 8 * h + 4 * j + (s >> 2);
          const int col = wbase + 32 * i + 16 * nh + 4 * (s & 3);
          off[j * S + i] = row * CH * 16 + (((col >> 3) ^ rs_key<CH>(row)) << 4) + (col & 7) * 2;
        }
    }
  }
  __device__ __forceinline__ bf16x8 get(const char* plane, int i, int ks) const {
    if constexpr (KC) {
      return *reinterpret_cast<const bf16x8*>(plane + i * 32 * BK * 2 + off[ks]);
    } else {
      union {
        v4i16 h[2];
        bf16x8 v;
      } u;
      const char* b = plane + ks * 16 * EXT * 2;
      u.h[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TG_LDS_RS v4i16*)(b + off[i]));
      u.h[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((TG_LDS_RS v4i16*)(b + off[S + i]));
      return u.v;
    }
  }
};

// The wave's SM x SN accumulator tiles again on the fp32 matrix cores, operands straight
// from global memory (the rare blocks whose operands the split cannot hold).
template <bool TA, bool TB, int SM, int SN>
__device__ __forceinline__ void rs_fp32_tiles(const float* __restrict__ A, int64_t lda,
                                           const float* __restrict__ B, int64_t ldb, int64_t M,
                                           int64_t N, int64_t K, int64_t m, int64_t n,
                                           f32x16 (&acc)[SM][SN]) {
  const int lane = threadIdx.x & 63, l32 = lane & 31, h = lane >> 5;
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  for (int64_t k0 = 0; k0 < K; k0 += 8) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int64_t k = k0 + 4 * h + e;
      float a[SM], b[SN];
#pragma unroll
      for (int i = 0; i < SM; ++i) {
        const int64_t row = m + 32 * i + l32;
        a[i] = (row < M && k < K) ? (TA ? A[k * lda + row] : A[row * lda + k]) : 0.f;
      }
#pragma unroll
      for (int j = 0; j < SN; ++j) {
        const int64_t col = n + 32 * j + l32;
        b[j] = (col < N && k < K) ? (TB ? B[col * ldb + k] : B[k * ldb + col]) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < SM; ++i)
#pragma unroll
        for (int j = 0; j < SN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  }
}

// How the sums are kept as exact as the fp32 matrix cores': an MFMA rounds its result once,
// and drops what of its addends lies below, which takes sums down by a little more than it
// takes them up.  Six MFMAs per 16 k into one accumulator leave an entry up to 1.2 times as
// far off as v_mfma_f32_32x32x2 does (non-negative A: 4096x4096x2048 6.7e-7 of the 2-norm,
// 5.8e-7 there), and column sums of C, a bias gradient behind it, 10 times (pairs of rows
// with opposite signs take that back for zero-mean entries only).  So every 64 k are summed
// from zero and added to a second accumulator by the vector unit, every second time with A's
// signs, and the partial sum's, turned round, so that neighbouring partial sums err to
// opposite sides: entries 1.7e-7 there, column sums at or below those of the fp32
// instructions for operands of either or of one sign.  4096x4096x2048 takes 380 us, 366 with
// one accumulator; partial sums of 128 k take 368, but leave column sums of offset operands
// 2 to 4 times as far off as the fp32 instructions at K = 512.
// STAG: the upper half of the waves multiplies before it stores.
template <bool TA, bool TB, int WGM, int WGN, int SM, int SN, bool STAG>
__global__ __launch_bounds__(64 * WGM * WGN, 2) void k_gemm_rs(
    int64_t M, int64_t N, int64_t K, int64_t ktot, float alpha, const float* __restrict__ A,
    int64_t lda, int64_t sa, const float* __restrict__ B, int64_t ldb, int64_t sb, float beta,
    float* __restrict__ C, int64_t ldc, int64_t sc, const float* __restrict__ bias, int gx,
    int tiles) {
  constexpr int NT = 64 * WGM * WGN, TBM = WGM * SM * 32, TBN = WGN * SN * 32;
  using OA = RsOp<!TA, TBM, NT>;
  using OB = RsOp<TB, TBN, NT>;
  __shared__ __attribute__((aligned(16))) char a0[3 * OA::PLANE];
  __shared__ __attribute__((aligned(16))) char b0[3 * OB::PLANE];
  __shared__ __attribute__((aligned(16))) char a1[3 * OA::PLANE];
  __shared__ __attribute__((aligned(16))) char b1[3 * OB::PLANE];
  // XCD-contiguous bands: launch index i runs on XCD i % 8, which takes tiles
  // [x*T/8, (x+1)*T/8) so that neighbouring tiles share operand rows in its L2.
  int lin = (int)blockIdx.x;
  {
    const int x = lin & 7, q = tiles >> 3, r = tiles & 7;
    lin = x * q + (x < r ? x : r) + (lin >> 3);
  }
  const int64_t m0 = (int64_t)(lin / gx) * TBM, n0 = (int64_t)(lin % gx) * TBN;
  const int64_t bz = blockIdx.z;
  A += bz * sa;
  B += bz * sb;
  C += bz * sc;
  K = K < ktot - bz * K ? K : ktot - bz * K;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave / WGN) * SM * 32, wn = (wave % WGN) * SN * 32;
  const int l32 = lane & 31, lh = lane >> 5;
  RsFrag<!TA, TBM, SM> fa;
  RsFrag<TB, TBN, SN> fb;
  fa.init(lane, wm);
  fb.init(lane, wn);
  f32x16 acc[SM][SN];
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  f32x16 sum[SM][SN];
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j) sum[i][j] = acc[i][j];
  OA oa;
  OB ob;
  oa.init(A, lda, m0, M);
  ob.init(B, ldb, n0, N);
  const bool ea = TA && m0 + TBM > M, eb = !TB && n0 + TBN > N;
  auto load = [&](int64_t k0) {
    const bool ek = k0 + BK > K;
    oa.load(ea || ek, K - k0);
    ob.load(eb || ek, K - k0);
  };
  auto mul = [&](int64_t k0, const char* as, const char* bs) {
    if (k0 % kTurn == 0 && k0 > 0) {
      // the partial sum is whole: add it (in whole vectors: element by element the compiler
      // keeps the arrays in scratch memory)
#pragma unroll
      for (int i = 0; i < SM; ++i)
#pragma unroll
        for (int j = 0; j < SN; ++j) {
          sum[i][j] = acc[i][j] - sum[i][j];
          acc[i][j] = f32x16{};
        }
    }
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      bf16x8 af[SM][3], bf[SN][3];
#pragma unroll
      for (int p = 0; p < 3; ++p) {
#pragma unroll
        for (int i = 0; i < SM; ++i) af[i][p] = fa.get(as + p * OA::PLANE, i, ks);
#pragma unroll
        for (int j = 0; j < SN; ++j) bf[j][p] = fb.get(bs + p * OB::PLANE, j, ks);
      }
      constexpr int PA[6] = {0, 0, 1, 1, 0, 2}, PB[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int i = 0; i < SM; ++i)
#pragma unroll
          for (int j = 0; j < SN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i][PA[t]], bf[j][PB[t]],
                                                                acc[i][j], 0, 0, 0);
    }
  };
  // tile t is multiplied from one buffer while tile t + 1 (in registers) is split into
  // the other and tile t + 2 is loaded
  const bool late = STAG && wave >= WGM * WGN / 2;
  auto turned = [&](int64_t k0) { return k0 / kTurn % 2 != 0; };
  auto step = [&](int64_t k0, const char* as, const char* bs, char* an, char* bn) {
    __syncthreads();
    if (late) mul(k0, as, bs);
    if (k0 + BK < K) {
      oa.store(an, turned(k0 + BK) ? -kScale : kScale);
      ob.store(bn, kScale);
      if (k0 + 2 * BK < K) load(k0 + 2 * BK);
    }
    if (!late) mul(k0, as, bs);
  };
  if (K > 0) {
    load(0);
    oa.store(a0, kScale);
    ob.store(b0, kScale);
    if (BK < K) load(BK);
    for (int64_t k0 = 0; k0 < K; k0 += 2 * BK) {
      step(k0, a0, b0, a1, b1);
      if (k0 + BK >= K) break;
      step(k0 + BK, a1, b1, a0, b0);
    }
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SN; ++j) acc[i][j] -= sum[i][j];
    // operands the split cannot hold: redo the tile on the fp32 matrix cores
    bool bad = false;
#pragma unroll
    for (int i = 0; i < SM; ++i)
#pragma unroll
      for (int j = 0; j < SN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) bad |= !(fabsf(acc[i][j][r]) <= 3.402823466e38f);
    if (__syncthreads_or(bad)) {
      rs_fp32_tiles<TA, TB, SM, SN>(A, lda, B, ldb, M, N, K, m0 + wm, n0 + wn, acc);
    } else {
      // both scales off again (one rounding where the entry is subnormal)
#pragma unroll
      for (int i = 0; i < SM; ++i)
#pragma unroll
        for (int j = 0; j < SN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            acc[i][j][r] = ldexpf(turned(K - 1) ? -acc[i][j][r] : acc[i][j][r], -2 * kScaleExp);
    }
  }
#pragma unroll
  for (int i = 0; i < SM; ++i)
#pragma unroll
    for (int j = 0; j < SN; ++j) {
      const int64_t col = n0 + wn + j * 32 + l32;
      if (col >= N) continue;
      const float bv = bias ? bias[col] : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + wm + i * 32 + (r >> 2) * 8 + lh * 4 + (r & 3);
        if (row < M) {
          float* pc = C + row * ldc + col;
          float v = alpha * acc[i][j][r] + bv;
          if (beta != 0.f) v += beta * *pc;
          *pc = v;
        }
      }
    }
}

// Small outputs: one 32 x 32 tile per workgroup, its NW wavefronts each taking 1/NW of K
// with the fp32 MFMA's fragments read straight from global memory (no operand is shared
// between wavefronts), then the partial tiles added in LDS in a fixed order.  Of every
// 8 k, lane half h multiplies k + 4h .. k + 4h + 3 in four MFMAs (the same pairing for A
// and B).
// NW: 16, or 4 where lanes read along the rows of both operands (A transposed, B plain):
// workgroups are smaller and more of them run, so a tile's sums and stores cost less.
template <bool TA, bool TB, int NW>
__global__ __launch_bounds__(64 * NW) void k_gemm_rs_small(
    int64_t M, int64_t N, int64_t K, int64_t ktot, float alpha, const float* __restrict__ A,
    int64_t lda, int64_t sa, const float* __restrict__ B, int64_t ldb, int64_t sb, float beta,
    float* __restrict__ C, int64_t ldc, int64_t sc, const float* __restrict__ bias) {
  const int64_t bz = blockIdx.z;
  A += bz * sa;
  B += bz * sb;
  C += bz * sc;
  K = K < ktot - bz * K ? K : ktot - bz * K;
  const int64_t m0 = (int64_t)blockIdx.y * 32, n0 = (int64_t)blockIdx.x * 32;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l32 = lane & 31, h = lane >> 5;
  const int64_t row = m0 + l32, col = n0 + l32;
  const int64_t per = ((K + 8 * NW - 1) / (8 * NW)) * 8;  // k per wavefront, a multiple of 8
  const int64_t kb = wave * per;
  const int64_t ke = kb + per < K ? kb + per : K;
  const bool rok = row < M, cok = col < N;
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll 4
  for (int64_t k0 = kb; k0 < ke; k0 += 8) {
    float a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t k = k0 + 4 * h + j;
      const bool kok = k < ke;
      a[j] = (rok && kok) ? (TA ? A[k * lda + row] : A[row * lda + k]) : 0.f;
      b[j] = (cok && kok) ? (TB ? B[col * ldb + k] : B[k * ldb + col]) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], acc, 0, 0, 0);
  }
  __shared__ float red[NW][16][64];
#pragma unroll
  for (int r = 0; r < 16; ++r) red[wave][r][lane] = acc[r];
  __syncthreads();
  for (int r = wave; r < 16; r += NW) {  // wave w finishes accumulator registers w, w + NW, ..
    float v = red[0][r][lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w][r][lane];
    const int64_t i = m0 + (r >> 2) * 8 + h * 4 + (r & 3);
    if (i < M && cok) {
      float o = alpha * v;
      if (bias) o += bias[col];
      float* pc = C + i * ldc + col;
      if (beta != 0.f) o += beta * *pc;
      *pc = o;
    }
  }
}

template <int WGM, int WGN, int SM, int SN, bool STAG>
int rs_launch(int ta, int tb, int64_t M, int64_t N, int64_t K, int64_t ktot, float alpha,
              const float* A, int64_t lda, int64_t sa, const float* B, int64_t ldb, int64_t sb,
              float beta, float* C, int64_t ldc, int64_t sc, int64_t batch, const float* bias,
              hipStream_t s) {
  constexpr int TBM = WGM * SM * 32, TBN = WGN * SN * 32;
  const int64_t gx = (N + TBN - 1) / TBN, gy = (M + TBM - 1) / TBM;
  if (gx * gy > INT32_MAX) {
    tg_set_error("tg_gemm: output of %lld x %lld has too many tiles", (long long)M, (long long)N);
    return TG_ERR_INVALID;
  }
  const dim3 grid((unsigned)(gx * gy), 1, (unsigned)batch);
#define TG_RS(TA_, TB_)                                                                      \
  k_gemm_rs<TA_, TB_, WGM, WGN, SM, SN, STAG><<<grid, 64 * WGM * WGN, 0, s>>>(               \
      M, N, K, ktot, alpha, A, lda, sa, B, ldb, sb, beta, C, ldc, sc, bias, (int)gx,          \
      (int)(gx * gy))
  if (!ta && !tb) TG_RS(false, false);
  else if (!ta) TG_RS(false, true);
  else if (!tb) TG_RS(true, false);
  else TG_RS(true, true);
#undef TG_RS
  return tg_check_launch("tg_gemm");
}

enum { RS_256x128 = 0, RS_128x128, RS_64x64, RS_SMALL, RS_SMALL4 };

}  // namespace

// Estimated times (us) of the kernels, from their measured time per 32-deep k-tile and
// block with every CU busy; the smallest wins.  Per k-tile: 256x128 3.2 us, 128x128
// 1.75 us (one block per CU each), 64x64 1.13 / 1.4 / 1.95 us with one / two / three
// blocks per CU; a block's start and store take 3-4 us.  The small kernel takes 0.9 us
// per 128 k plus 2.1 us for each block per CU (its operands come straight from the
// caches); with 4 waves, A transposed, 3 us and per k 0.012 plus 0.0063 for each tile per CU
// (1722x370x427: 16 us, 64x64 blocks 26; 1114x632x784 26 and 40).  A K split adds the finishing launch: 10 us, half of it
// the host's, and its traffic at 3.5 TB/s.
// (Measured against the previous kernels, us: 8192x4096x1024 727 -> 402, 1024x4096x8192
// with A transposed 1086 -> 399, 832x1664x8932 1210 -> 224, 1000^3 117 -> 37,
// 448x256x32000 867 -> 72, 33x257x784 20 -> 15.)
TgRsPlan tg_gemm_rs_plan(bool tn, int64_t M, int64_t N, int64_t K, int64_t batch,
                         bool can_split) {
  TgRsPlan best{RS_256x128, 1, K};
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return best;
  const double ncu = (double)tg_num_cus();
  const auto tiles = [&](int64_t bm, int64_t bn) {
    return (double)((M + bm - 1) / bm) * (double)((N + bn - 1) / bn) * (double)batch;
  };
  const auto rounds = [&](double blocks) { return std::ceil(blocks / ncu); };
  double tbest = 1e30;
  for (int64_t S = 1; S <= (can_split ? 32 : 1); S *= 2) {
    const int64_t kc = S == 1 ? K : ((K + S - 1) / S + 63) / 64 * 64;
    if (S > 1 && (kc < 128 || (K + kc - 1) / kc != S)) continue;
    const double kt = (double)((kc + BK - 1) / BK);
    const double fin = S > 1 ? 10.0 + (double)(S + 1) * (double)M * (double)N * 4.0 / 3.5e6 : 0.0;
    // (a split's partial sums stay within 256 MiB)
    if (S > 1 && (double)S * (double)M * (double)N * 4.0 > 268435456.0) break;
    double t[5];
    t[RS_256x128] = rounds(tiles(256, 128) * S) * (kt * 3.2 + 4.0);
    t[RS_128x128] = rounds(tiles(128, 128) * S) * (kt * 1.75 + 3.5);
    const double b64 = tiles(64, 64) * S, full = std::floor(b64 / (3 * ncu));
    const double rest = rounds(b64 - full * 3 * ncu);
    t[RS_64x64] = full * (kt * 1.95 + 3.0) +
                  (rest > 0 ? kt * (rest > 2 ? 1.95 : rest > 1 ? 1.4 : 1.13) + 3.0 : 0.0);
    t[RS_SMALL] = t[RS_SMALL4] = 1e30;
    if ((M + 31) / 32 <= 65535) {
      const double per_cu = tiles(32, 32) * S / ncu;
      t[RS_SMALL] = (double)((kc + 127) / 128) * (0.9 + 2.1 * per_cu) + 3.0;
      if (tn && S == 1) t[RS_SMALL4] = (double)kc * (0.012 + 0.0063 * std::max(per_cu, 1.0)) + 3.0;
    }
    for (int i = 0; i < 5; ++i)
      if (t[i] + fin < tbest) {
        tbest = t[i] + fin;
        best = TgRsPlan{i, S, kc};
      }
  }
  return best;
}

int tg_gemm_rs(const TgRsPlan& p, int ta, int tb, int64_t M, int64_t N, int64_t K, float alpha,
               const float* A, int64_t lda, int64_t sa, const float* B, int64_t ldb, int64_t sb,
               float beta, float* C, int64_t ldc, int64_t sc, int64_t batch, const float* bias,
               hipStream_t s) {
  const int64_t kc = p.S > 1 ? p.kc : K;
  const int64_t ktot = p.S > 1 ? K : INT64_MAX;
#define TG_RSL(...)                                                                        \
  rs_launch<__VA_ARGS__>(ta, tb, M, N, kc, ktot, alpha, A, lda, sa, B, ldb, sb, beta, C, ldc, \
                         sc, batch, bias, s)
  switch (p.shape) {
    case RS_256x128: return TG_RSL(4, 2, 2, 2, true);
    case RS_128x128: return TG_RSL(4, 2, 1, 2, true);
    case RS_64x64: return TG_RSL(2, 2, 1, 1, false);
    default: break;
  }
#undef TG_RSL
  const dim3 gs((unsigned)((N + 31) / 32), (unsigned)((M + 31) / 32), (unsigned)batch);
#define TG_SM(TA_, TB_, NW_)                                                                   \
  k_gemm_rs_small<TA_, TB_, NW_><<<gs, 64 * NW_, 0, s>>>(M, N, kc, ktot, alpha, A, lda, sa, B, ldb, \
                                                         sb, beta, C, ldc, sc, bias)
  if (p.shape == RS_SMALL4) TG_SM(true, false, 4);
  else if (!ta && !tb) TG_SM(false, false, 16);
  else if (!ta) TG_SM(false, true, 16);
  else if (!tb) TG_SM(true, false, 16);
  else TG_SM(true, true, 16);
#undef TG_SM
  return tg_check_launch("tg_gemm");
}
