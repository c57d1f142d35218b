// gemm.hip - the prefill GEMM of the Q8 arithmetic on the int8 matrix cores
// of gfx950 (one weight type per build, IHIP_ONLY_FMT_*).
//
// What it computes: y[r, o] = bias[o] + sum over groups of the exact
// TInferCpuBackend.Linear terms (backend.cpu.pas:1409-1566, 823-967) for
// quantized activation rows x (Q8_0 or Q8_K, by quantize_q8_0/_k) and weights
// in the HIP layout of layout.h - the same terms, in double, as the one-row
// GEMV of linear.hip (group_q8, group_q8k, superblock_q8k); only the order of
// the double sum over groups differs (here: group order, or with a block's KS
// waves sharing the sum, wave k the chunks of 8 groups k, k + KS, .. in order
// and then the waves' sums in wave order).
//
// Mapping to CDNA4: a wave owns one or two tiles of 32 rows x 32 outputs. Per
// 32-value group it runs v_mfma_i32_32x32x32_i8 with A = the activation codes
// of a tile's rows and B = the weight codes of its outputs, widened to int8
// (centred for Q4_0/Q5_0/Q6_K, the e2m1 table for MXFP4): the exact int32
// group dot products, 16 per lane. The scales follow: a lane owns one output
// and 16 rows. For the formats of 32 values the products dw dx of all its
// outputs come from one outer-product MFMA (v_mfma_f32_32x32x16_f16 with one
// k: two halves, the product exact in single), where reading 16 row scales a
// group from LDS cost more than the group's arithmetic; then one fused
// multiply-add in double per output. K-quants multiply the group sums by their
// integer sub-scales and form one term per super-block; Q4_K's minimum sum is
// one f16 MFMA a super-block over the code sums split 64 hi + lo. Q6_K's
// 16-value sub-blocks are two v_mfma_i32_32x32x16_i8, lane half h feeding
// values 8h..8h+7 of each: with the group's nibble order (byte j: value j,
// value j + 16) both come from bytes 8h..8h+7 of the 16-byte group.
//
// Bound by the chain LDS -> widening -> MFMA -> terms of a group and the two
// barriers of a step, which two waves a SIMD do not cover: on full chips vector
// instructions issue 45% of the time (36 to 59 per MFMA), MFMAs 9%. Measured
// against the 64 x 64 tiles with row scales in LDS that this replaces, us, the
// launch alone: Q4_K 512 rows 2048 -> 6144 47.8 -> 30.4 (424 TOP/s), 1024 rows
// 2048 -> 4096 61.9 -> 34.0 (505), Q6_K 512 rows 58.8 -> 47.2, Q8_0 51.9 -> 43.7,
// 301 rows 3072 -> 1024 35.4 -> 16.7 (the sum over 4 waves).
//
// Operand layout of both MFMAs (probed on gfx950): A lane l = row l % 32,
// B lane l = column l % 32, 16 (8) k values each, the k order free but the
// same in A and B; result register i of lane l = row 8 (i / 4) + 4 (l / 32) +
// i % 4, column l % 32.
#include "formats.h"

namespace ihip {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f_t __attribute__((ext_vector_type(16)));
typedef _Float16 v8h_t __attribute__((ext_vector_type(8)));

struct GemmArgs {
  const uint8_t* w;   // matrix, or expert 0 with items
  const uint8_t* xq;  // quantized rows [*, in + 4 G]: int8 codes, then float dx per group
  const float* bias;  // [out], [experts, out] with items, or null
  float* y;           // [*, out]
  int64_t stride;     // bytes between experts
  int32_t out, in, rows, pad;
  // grouped experts: tile row block blockIdx.y = item (expert, start, count
  // <= 64) over perm, the slots sorted by expert; slot s reads x row
  // s / x_per_slot (0: row 0) and writes y row s
  const int4* items;
  const int* perm;
  int32_t x_per_slot, pad2;
  const float* x;  // float rows [*, in] (float weights)
  // float weights, ksplit > 1: block z sums the values [z klen, (z + 1) klen)
  // and writes its double partial sums (no bias) to part [ksplit, rows, out]
  double* part;
  int32_t ksplit, klen;
};

constexpr int GBM = 64, GBN = 64;  // tile rows and outputs (float weights, f8f6f4)
constexpr int GKC = 8;             // groups per chunk: 256 values, a K-quant super-block

// the 16 codes of code dwords 0 and 1 (values 0..7 of the low half of a
// group's bytes, then of the high) as int8 in the Q8 arithmetic's value
// (centred where the format has an offset the CPU subtracts through the
// activation sum)
template <int F>
__device__ __forceinline__ v4i widen(const Raw& v)
{
  uint32_t c[4] = {code_bytes<F>(v, 0, 0), code_bytes<F>(v, 1, 0), code_bytes<F>(v, 0, 1),
                   code_bytes<F>(v, 1, 1)};
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t t = c[k];
    if constexpr (F == DT_Q4_0) {  // q - 8: the 4-bit value sign-extended after flipping bit 3
      t ^= 0x08080808u;
      t |= (t & 0x08080808u) * 0x1Eu;
    } else if constexpr (F == DT_Q5_0) {  // q - 16
      t ^= 0x10101010u;
      t |= (t & 0x10101010u) * 0x0Eu;
    } else if constexpr (F == DT_Q6_K) {  // q - 32
      t ^= 0x20202020u;
      t |= (t & 0x20202020u) * 0x06u;
    }
    c[k] = t;
  }
  return v4i{(int)c[0], (int)c[1], (int)c[2], (int)c[3]};
}

// widen() of lane half h (values 8h..8h+7 and 16+8h..16+8h+7 of the group)
template <int F>
__device__ __forceinline__ v4i b_operand(const Raw& r, int h)
{
  // the lane half's view of the group: code dwords 2h and 2h + 1 moved to
  // dwords 0 and 1, chosen by masks (values, never an index into registers)
  const uint32_t m = 0u - (uint32_t)h;
  Raw v = r;
  v.q0.x = (r.q0.x & ~m) | (r.q0.z & m);
  v.q0.y = (r.q0.y & ~m) | (r.q0.w & m);
  v.q1.x = (r.q1.x & ~m) | (r.q1.z & m);
  v.q1.y = (r.q1.y & ~m) | (r.q1.w & m);
  if constexpr (F == DT_Q5_0 || F == DT_Q5_1) v.b = r.b >> (8 * h);  // 4 bits per code dword
  if constexpr (F == DT_Q6_K) {  // 2 bits per code dword
    v.b = r.b >> (4 * h);
    v.c = r.c >> (4 * h);
  }
  return widen<F>(v);
}

// does the format need the activation code sum of a group (through the
// minimum / offset the CPU applies with it)
constexpr bool needs_xsum(int F) { return F == DT_Q4_K || F == DT_Q5_1; }

// The fields of Raw a format uses, as dwords: how a weight group sits in LDS.
template <int F>
constexpr int raw_dwords()
{
  return F == DT_Q8_0 ? 9 : (F == DT_Q4_K || F == DT_Q6_K) ? 8 : (F == DT_Q5_0 || F == DT_Q5_1) ? 6 : 5;
}

template <int F>
__device__ __forceinline__ void raw_put(uint32_t* d, int stride, const Raw& r)
{
  uint32_t v[9] = {r.q0.x, r.q0.y, r.q0.z, r.q0.w, 0, 0, 0, 0, 0};
  if constexpr (F == DT_Q8_0 || F == DT_Q4_K) {
    v[4] = r.q1.x; v[5] = r.q1.y; v[6] = r.q1.z; v[7] = r.q1.w;
    v[8] = r.a;
  } else if constexpr (F == DT_Q6_K) {
    v[4] = r.a; v[5] = r.b; v[6] = r.c; v[7] = r.d;
  } else {
    v[4] = r.a;
    v[5] = r.b;
  }
#pragma unroll
  for (int k = 0; k < raw_dwords<F>(); k++) d[k * stride] = v[k];
}

template <int F>
__device__ __forceinline__ Raw raw_get(const uint32_t* d, int stride)
{
  uint32_t v[9];
#pragma unroll
  for (int k = 0; k < raw_dwords<F>(); k++) v[k] = d[k * stride];
  Raw r{};
  r.q0 = make_uint4(v[0], v[1], v[2], v[3]);
  if constexpr (F == DT_Q8_0 || F == DT_Q4_K) {
    r.q1 = make_uint4(v[4], v[5], v[6], v[7]);
    if constexpr (F == DT_Q8_0) r.a = v[8];
  } else if constexpr (F == DT_Q6_K) {
    r.a = v[4]; r.b = v[5]; r.c = v[6]; r.d = v[7];
  } else {
    r.a = v[4];
    if constexpr (F == DT_Q5_0 || F == DT_Q5_1) r.b = v[5];
  }
  return r;
}

constexpr int G8A = 8 * 8 + 2;  // gemm8: LDS dwords per activation row

// ------------------------------------------- MXFP4 on the scaled f8f6f4 MFMA
// v_mfma_scale_f32_32x32x64_f8f6f4 with B the group's e2m1 codes as they are
// stored (no decode) and A the activation codes split q = 16 hi + lo (hi, lo
// in [-8, 8]): A's first 32 k are e4m3(16 hi) and its last 32 e4m3(lo), B's
// two 32-k blocks both the group's 32 codes, every block scale 1. Each
// product is exact (e4m3 x e2m1) and every partial sum a multiple of 1/2
// below 2^23, so the f32 result is the exact group dot sum q w over the e2m1
// values, half the doubled-table integer sum of the int8 path: the CPU's
// group sum, as exact. One instruction per 32-value group, like the int8
// MFMA, without the e2m1 -> int8 decode of the weights.
//
// Operand layout (probed on gfx950): byte j of an 8-bit operand in lane half
// h holds k = 16 h + j (j < 16) or 32 + 16 h + (j - 16); nibble j of a 4-bit
// operand in lane half h holds k = 32 h + j. The k order is free as long as A
// and B agree: B's block position p is nibble p of the 16 stored code bytes,
// value v(p) = p / 2 + 16 (p % 2) (byte j: value j low, value j + 16 high), so
// A's positions take q[v(p)]. A row's planes per group (f8_planes): for h =
// 0, 1 the 32 bytes e4m3(16 hi[v(16h + j)]) j < 16, e4m3(lo[v(16h + j)]) j
// < 16 - lane half h reads bytes 32h..32h+31 of the group.
typedef int v8i_t __attribute__((ext_vector_type(8)));

// a chunk of GKC groups of the tile in registers, from coalesced loads
struct ChunkRegs {
  Raw wr[2];      // weight groups: column t / 8 (+ 32), group t % 8
  v4u32 xc[4];    // the first half of the planes: row t / 4, groups 2 (t % 4) and 2 (t % 4) + 1
  float dx[2];    // and their scales
  v4u32 xp[4];    // the second half
};
constexpr int GSW = GKC * raw_dwords<DT_Q8_0>() + 1;  // LDS dwords per weight column (odd)

// e4m3 of an integer in [-8, 8] (times 16 when x16: the exponent + 4)
__device__ __forceinline__ uint32_t e4m3_small(int v, bool x16)
{
  const int a = v < 0 ? -v : v;
  // 0, 1 .. 8: 0x00 0x38 0x40 0x44 0x48 0x4A 0x4C 0x4E 0x50
  const uint32_t lo4 = 0x44403800u, hi4 = 0x4E4C4A48u;
  uint32_t m = a == 8 ? 0x50u : (a < 4 ? (lo4 >> (8 * a)) & 255u : (hi4 >> (8 * (a - 4))) & 255u);
  if (x16 && a) m += 0x20u;
  return v < 0 ? (m | 0x80u) : m;
}

template <int F>
__device__ __forceinline__ void chunk_load8(const GemmArgs& a, const uint8_t* wb, const Regions& rg,
                                            int col0, const int* sxr, int64_t xstride, int G, int gc,
                                            ChunkRegs& cr)
{
  const int t = threadIdx.x;
#pragma unroll
  for (int p = 0; p < 2; p++) {
    const int64_t o = min(col0 + (t >> 3) + 32 * p, a.out - 1);
    load_group<F>(wb, rg, o, G, min(gc + (t & 7), G - 1), a.in, cr.wr[p]);
  }
  const uint8_t* xr = a.xq + (int64_t)sxr[t >> 2] * xstride;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int g = min(gc + 2 * (t & 3) + k, G - 1);
    const v4u32* q = (const v4u32*)(xr + (int64_t)g * 64);
    cr.xc[2 * k] = q[0];
    cr.xc[2 * k + 1] = q[1];
    cr.xp[2 * k] = q[2];
    cr.xp[2 * k + 1] = q[3];
    cr.dx[k] = ((const float*)(xr + (int64_t)G * 64))[g];
  }
}

constexpr int GSA8 = GKC * 16 + 4;  // LDS dwords per activation row of planes

template <int F>
__device__ __forceinline__ void chunk_store8(const ChunkRegs& cr, uint32_t* sw, uint32_t* sa, double* sdx)
{
  const int t = threadIdx.x;
  constexpr int WS = GKC * raw_dwords<F>() + 1;
#pragma unroll
  for (int p = 0; p < 2; p++) raw_put<F>(sw + ((t >> 3) + 32 * p) * WS + (t & 7), GKC, cr.wr[p]);
  const int row = t >> 2;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const int j = 2 * (t & 3) + k;
    uint32_t* d = sa + row * GSA8 + j * 16;
    *(v4u32*)d = cr.xc[2 * k];
    *(v4u32*)(d + 4) = cr.xc[2 * k + 1];
    *(v4u32*)(d + 8) = cr.xp[2 * k];
    *(v4u32*)(d + 12) = cr.xp[2 * k + 1];
    sdx[j * GBM + row] = (double)cr.dx[k];
  }
}

// the MXFP4 GEMM on the f8f6f4 matrix cores: gemm's tiles, chunks and
// double scaling; A from the planes of f8_planes
__device__ __forceinline__ void gemm_mxfp4_f8(const GemmArgs& a)
{
  constexpr int F = DT_MXFP4;
  __shared__ uint32_t sw_[GBN * GSW];
  __shared__ __align__(16) uint32_t sa_[GBM * GSA8];
  __shared__ __align__(16) double sdx_[GKC * GBM];
  __shared__ int sxr[GBM], syr[GBM];
  const int t = threadIdx.x, l = t & 63, w = t >> 6, h = l >> 5;
  const int wm = w & 1, wn = w >> 1;
  const int G = a.in >> 5;
  const int64_t xstride = 68 * (int64_t)G;
  const uint8_t* wb = a.w;
  const float* bias = a.bias;
  int nrows;
  if (a.items) {
    const int4 it = a.items[blockIdx.y];
    if (it.z <= 0) return;
    wb += (int64_t)it.x * a.stride;
    if (bias) bias += (int64_t)it.x * a.out;
    nrows = min(GBM, it.z);
    if (t < GBM) {
      const int sl = a.perm[it.y + min(t, nrows - 1)];
      sxr[t] = a.x_per_slot ? sl / a.x_per_slot : 0;
      syr[t] = sl;
    }
  } else {
    const int r0 = blockIdx.y * GBM;
    nrows = min(GBM, a.rows - r0);
    if (t < GBM) sxr[t] = syr[t] = r0 + min(t, nrows - 1);
  }
  __syncthreads();
  const Regions rg = regions(F, a.out, a.in);
  const int col0 = blockIdx.x * GBN;
  const int o_real = col0 + 32 * wn + (l & 31);
  const int64_t o = min(o_real, a.out - 1);
  const int rb = 32 * wm + 4 * h;
  constexpr int WS = GKC * raw_dwords<F>() + 1;
  const uint32_t* myw = sw_ + (32 * wn + (l & 31)) * WS;
  const uint32_t* mya = sa_ + (32 * wm + (l & 31)) * GSA8 + 8 * h;
  double acc[16];
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = 0.0;
  const int nch = (G + GKC - 1) / GKC;
  ChunkRegs cr;
  chunk_load8<F>(a, wb, rg, col0, sxr, xstride, G, 0, cr);
  chunk_store8<F>(cr, sw_, sa_, sdx_);
  chunk_load8<F>(a, wb, rg, col0, sxr, xstride, G, GKC, cr);
  __syncthreads();
  for (int c = 0; c < nch; c++) {
    const int gc = c * GKC;
#pragma unroll
    for (int j = 0; j < GKC; j++) {
      const int g = gc + j;
      if (g < G) {
        const Raw r = raw_get<F>(myw + j, GKC);
        const v4u32 a0 = *(const v4u32*)(mya + j * 16), a1 = *(const v4u32*)(mya + j * 16 + 4);
        const v8i_t av = {(int)a0.x, (int)a0.y, (int)a0.z, (int)a0.w, (int)a1.x, (int)a1.y, (int)a1.z, (int)a1.w};
        const v8i_t bv = {(int)r.q0.x, (int)r.q0.y, (int)r.q0.z, (int)r.q0.w, 0, 0, 0, 0};
        const v16f_t z = {};
        // formats: A e4m3 (0), B e2m1 (4); every block scale E8M0 127 (1.0)
        const v16f_t cf = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, z, 0, 4, 0, 0x7F7F7F7F, 0,
                                                                           0x7F7F7F7F);
        const double dw = mxfp4_q8_scale(r.a);
        double2 dq[8];
#pragma unroll
        for (int q = 0; q < 8; q++) dq[q] = *(const double2*)&sdx_[j * GBM + rb + 8 * (q >> 1) + 2 * (q & 1)];
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const double2 d2 = dq[i >> 1];
          const double dx = (i & 1) ? d2.y : d2.x;
          // 2 cf: the doubled-table integer group sum of the CPU, exact
          acc[i] = __builtin_fma(2.0 * (double)cf[i], dw * dx, acc[i]);
        }
      }
    }
    __syncthreads();
    chunk_store8<F>(cr, sw_, sa_, sdx_);
    chunk_load8<F>(a, wb, rg, col0, sxr, xstride, G, gc + 2 * GKC, cr);
    __syncthreads();
  }
  if (o_real >= a.out) return;
  const double b = bias ? (double)bias[o] : 0.0;
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const int rt = rb + 8 * (i >> 2) + (i & 3);
    if (rt < nrows) {
      double v = acc[i];
      if (bias) v = b + v;
      a.y[(int64_t)syr[rt] * a.out + o] = (float)v;
    }
  }
}

// the e4m3 planes of quantized activation rows for gemm_mxfp4_f8: row r of
// xq (codes [in], then dx [G]) into row r of planes (64 bytes per group as
// above, then the same dx [G]); one thread per group
struct PlanesArgs {
  const uint8_t* xq;
  uint8_t* planes;
  int32_t rows, in;
};
__device__ __forceinline__ void f8_planes(const PlanesArgs& a)
{
  const int G = a.in >> 5;
  const int64_t gi = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int row = blockIdx.y;
  if (gi >= G) return;
  const uint8_t* src = a.xq + (int64_t)row * ((int64_t)a.in + 4 * G);
  uint8_t* dst = a.planes + (int64_t)row * 68 * G;
  const v4u32 c0 = *(const v4u32*)(src + gi * 32), c1 = *(const v4u32*)(src + gi * 32 + 16);
  const uint32_t cw[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
  uint32_t outw[16];
#pragma unroll
  for (int hh = 0; hh < 2; hh++)
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
      uint32_t whi = 0, wlo = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) {
        const int p = 16 * hh + 4 * jj + b;
        const int v = (p >> 1) + 16 * (p & 1);
        const int q = (int)(int8_t)((cw[v >> 2] >> (8 * (v & 3))) & 255u);
        const int hi = (q + 8) >> 4, lo = q - 16 * hi;
        whi |= e4m3_small(hi, true) << (8 * b);
        wlo |= e4m3_small(lo, false) << (8 * b);
      }
      outw[8 * hh + jj] = whi;
      outw[8 * hh + 4 + jj] = wlo;
    }
  v4u32* d = (v4u32*)(dst + gi * 64);
#pragma unroll
  for (int k = 0; k < 4; k++) d[k] = v4u32{outw[4 * k], outw[4 * k + 1], outw[4 * k + 2], outw[4 * k + 3]};
  ((float*)(dst + (int64_t)G * 64))[gi] = ((const float*)(src + a.in))[gi];
}

// Block shapes. A block has 4 waves; a wave owns MT tiles of 32 rows x 32
// outputs and every KS-th chunk of the sum, the 4 / KS waves across make
// 32 MT rows x 128 / KS outputs, and the KS partial sums of an output meet in
// LDS at the end.
constexpr int GSA = 68;  // LDS dwords of an activation row's chunk (64 and a 16-byte shift of banks)

// code dwords of a group, and the dwords beside them (scale, high bits)
template <int F>
constexpr int code_dwords() { return F == DT_Q8_0 ? 8 : 4; }
template <int F>
constexpr int side_dwords()
{
  return F == DT_Q4_K ? 0 : F == DT_Q6_K ? 3 : (F == DT_Q5_0 || F == DT_Q5_1) ? 2 : 1;
}
constexpr bool kquant(int F) { return F == DT_Q4_K || F == DT_Q6_K; }
// LDS dwords of a weight column's codes of a chunk: the 32 columns of a wave
// read 8 (Q8_0: 16) bytes each at one group, 2 (4) dwords a column apart
template <int F>
constexpr int col_dwords() { return F == DT_Q8_0 ? 68 : 34; }

// LDS of a block, in dwords: the regions of one step (4 wave slots of weights,
// KS chunks of activation rows), reused by the partial sums
template <int F, int MT, int KS>
struct GemmLds {
  static constexpr int A = 0;                                    // codes [KS][32 MT][GSA]
  static constexpr int B = A + KS * 32 * MT * GSA;               // codes [4][32][col_dwords]
  static constexpr int X = B + 128 * col_dwords<F>();            // side dwords [.][GKC][128]
  static constexpr int H = X + side_dwords<F>() * GKC * 128;     // K-quants: header [128][4]
  static constexpr int D = H + (F == DT_Q4_K ? 512 : F == DT_Q6_K ? 128 : 0);
  // K-quants: a double per row; else the scale's half bits per (group, row)
  static constexpr int S = D + (kquant(F) ? KS * 32 * MT * 2 : KS * GKC * 32 * MT);
  // Q4_K: the code sums as halves [KS][32 MT][16]; Q5_1: dx times the sum, doubles
  static constexpr int END = S + (F == DT_Q4_K ? KS * 32 * MT * 8 : F == DT_Q5_1 ? KS * GKC * 32 * MT * 2 : 0);
  static constexpr int RED = (KS - 1) * (4 / KS) * MT * 2048;    // partial sums, doubles
  static constexpr int DWORDS = END > RED ? END : RED;
};

// a step's operands in registers, from coalesced loads (each 8 lanes read 8
// consecutive groups of a weight row, or a row's 256 activation codes)
template <int F, int MT, int KS>
struct StepRegs {
  Raw wr[4];               // slot p: column t / 8 of wave slot p, group t % 8
  v4u32 xc[KS * MT][2];    // rows t / 8 + 32 mt, group t % 8 of chunk ks
  float dx[KS * MT];
};

template <int F, int MT, int KS>
__device__ __forceinline__ void step_load(const GemmArgs& a, const uint8_t* wb, const Regions& rg, int col0,
                                          const int* sxr, int64_t xstride, int G, int g0,
                                          StepRegs<F, MT, KS>& r)
{
  const int t = threadIdx.x;
  // groups past the last read the last one again; their scales are zero, so
  // their terms are
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const int64_t o = min(col0 + 32 * (p / KS) + (t >> 3), a.out - 1);
    const int g = g0 + GKC * (p % KS) + (t & 7);
    load_group<F, false, true>(wb, rg, o, G, min(g, G - 1), a.in, r.wr[p]);
    if (!kquant(F) && g >= G) r.wr[p].a = 0;
  }
#pragma unroll
  for (int q = 0; q < KS * MT; q++) {
    const int g = g0 + GKC * (q / MT) + (t & 7), gl = min(g, G - 1);
    const uint8_t* xr = a.xq + (int64_t)sxr[32 * (q % MT) + (t >> 3)] * xstride;
    const v4u32* c = (const v4u32*)(xr + (int64_t)gl * 32);
    r.xc[q][0] = c[0];
    r.xc[q][1] = c[1];
    r.dx[q] = ((const float*)(xr + a.in))[gl];
    if (!kquant(F) && g >= G) r.dx[q] = 0.0f;
  }
}

__device__ __forceinline__ uint32_t half_bits(float v)
{
  return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)v);
}

template <int F, int MT, int KS>
__device__ __forceinline__ void step_store(const StepRegs<F, MT, KS>& r, uint32_t* lds)
{
  using L = GemmLds<F, MT, KS>;
  const int t = threadIdx.x, g = t & 7;
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const int col = 32 * p + (t >> 3);
    uint32_t* d = lds + L::B + col * col_dwords<F>() + g * code_dwords<F>();
    const Raw& w = r.wr[p];
    if constexpr (F == DT_Q8_0) {
      *(uint4*)d = w.q0;
      *(uint4*)(d + 4) = w.q1;
    } else {
      *(uint2*)d = make_uint2(w.q0.x, w.q0.y);
      *(uint2*)(d + 2) = make_uint2(w.q0.z, w.q0.w);
    }
    uint32_t* x = lds + L::X + g * 128 + col;
    if constexpr (F == DT_Q4_K) {
      if (g < 4) lds[L::H + 4 * col + g] = w.q1.x;  // (QH: dword t % 4 of the header)
    } else if constexpr (F == DT_Q6_K) {
      x[0] = w.a;
      x[GKC * 128] = w.b;
      x[2 * GKC * 128] = w.c;
      if (g == 0) lds[L::H + col] = w.d;
    } else {
      x[0] = F == DT_MXFP4 ? half_bits((float)mxfp4_q8_scale(w.a)) : w.a;
      if constexpr (F == DT_Q5_0 || F == DT_Q5_1) x[GKC * 128] = w.b;
    }
  }
#pragma unroll
  for (int q = 0; q < KS * MT; q++) {
    const int row = 32 * (q % MT) + (t >> 3), kr = (q / MT) * 32 * MT + row;
    const v4u32 u0 = r.xc[q][0], u1 = r.xc[q][1];
    uint32_t* d = lds + L::A + kr * GSA + g * 8;
    // lane half h of the MFMA reads 16 bytes: the values its weight bytes hold
    if constexpr (F == DT_Q8_0) {
      *(v4u32*)d = u0;
      *(v4u32*)(d + 4) = u1;
    } else {
      *(v4u32*)d = v4u32{u0.x, u0.y, u1.x, u1.y};
      *(v4u32*)(d + 4) = v4u32{u0.z, u0.w, u1.z, u1.w};
    }
    if constexpr (kquant(F)) {
      if (g == 0) ((double*)(lds + L::D))[kr] = (double)r.dx[q];
    } else {
      lds[L::D + (q / MT) * GKC * 32 * MT + g * 32 * MT + row] = half_bits(r.dx[q]);
    }
    if constexpr (F == DT_Q4_K || F == DT_Q5_1) {
      int sm = 0;
      sm = sdot4((int)u0.x, 0x01010101, sm); sm = sdot4((int)u0.y, 0x01010101, sm);
      sm = sdot4((int)u0.z, 0x01010101, sm); sm = sdot4((int)u0.w, 0x01010101, sm);
      sm = sdot4((int)u1.x, 0x01010101, sm); sm = sdot4((int)u1.y, 0x01010101, sm);
      sm = sdot4((int)u1.z, 0x01010101, sm); sm = sdot4((int)u1.w, 0x01010101, sm);
      if constexpr (F == DT_Q4_K) {
        // sum = 64 hi + lo, each exact in half: lo of the 8 groups, then hi
        uint16_t* s = (uint16_t*)(lds + L::S) + kr * 16 + g;
        s[0] = (uint16_t)half_bits((float)(sm & 63));
        s[8] = (uint16_t)half_bits((float)(sm >> 6));
      } else {
        ((double*)(lds + L::S))[(q / MT) * GKC * 32 * MT + g * 32 * MT + row] = (double)r.dx[q] * (double)sm;
      }
    }
  }
}

// four bytes below 64 as two pairs of halves (1024 + b as bits, then - 1024)
__device__ __forceinline__ v8h_t bytes_half8(uint32_t b0, uint32_t b1, _Float16 times)
{
  typedef _Float16 v2h __attribute__((ext_vector_type(2)));
  const v2h off = {(_Float16)-1024.0f, (_Float16)-1024.0f}, mul = {times, times};
  v8h_t v;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t w = __builtin_amdgcn_perm(0x64646464u, k < 2 ? b0 : b1, (k & 1) ? 0x04030402u : 0x04010400u);
    const v2h h = (__builtin_bit_cast(v2h, w) + off) * mul;
    v[2 * k] = h.x;
    v[2 * k + 1] = h.y;
  }
  return v;
}

// a value the compiler may not reassociate through: it would hold the products
// of a whole super-block to sum them in another order, and spill
__device__ __forceinline__ int keep(int v)
{
  __asm__("" : "+v"(v));
  return v;
}

template <int F, int MT, int KS>
__device__ __forceinline__ void gemm_tiles(const GemmArgs& a, const uint8_t* wb, const float* bias, int nrows,
                                           const int* sxr, const int* syr, uint32_t* lds)
{
  using L = GemmLds<F, MT, KS>;
  const int t = threadIdx.x, l = t & 63, w = t >> 6, h = l >> 5, c32 = l & 31;
  const int wn = w / KS, ks = w % KS;
  const int G = a.in >> 5;
  const int64_t xstride = (int64_t)a.in + 4 * (int64_t)G;
  const Regions rg = regions(F, a.out, a.in);
  const int col0 = blockIdx.x * (128 / KS);
  // this lane's weight column and activation rows in LDS
  const int col = 32 * w + c32;
  const uint32_t* myb = lds + L::B + col * col_dwords<F>() + h * (code_dwords<F>() / 2);
  const uint32_t* mya = lds + L::A + (ks * 32 * MT + c32) * GSA + 4 * h;
  const uint32_t* myx = lds + L::X + col;
  const uint32_t lowhalf = h ? 0u : 0xffffu;

  double acc[MT][16];
  int isum[MT][16];
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      acc[m][i] = 0.0;
      isum[m][i] = 0;
    }
  const v16i zi = {};
  const v16f_t zf = {};

  // the operands of a group read from LDS
  struct Ops {
    uint2 q;         // this lane half's code bytes
    v4u32 q16;       // (Q8_0)
    uint32_t x, b, c;  // scale and high bits
    v4u32 xa[MT];    // activation codes
    uint32_t dx[MT];   // the scale of the lane's row, as half bits
  };
  struct Sums {
    v16i s, s2;   // group sums (Q6_K: of its two sub-blocks)
    v16f_t p;     // dw dx of every output (block formats of 32 values)
  };
  auto read = [&](int j) __attribute__((always_inline)) -> Ops {
    Ops r = {};
    if constexpr (F == DT_Q8_0) r.q16 = *(const v4u32*)(myb + j * 8);
    else r.q = *(const uint2*)(myb + j * 4);
    if constexpr (F != DT_Q4_K) r.x = myx[j * 128];
    if constexpr (side_dwords<F>() > 1) r.b = myx[(GKC + j) * 128];
    if constexpr (side_dwords<F>() > 2) r.c = myx[(2 * GKC + j) * 128];
#pragma unroll
    for (int m = 0; m < MT; m++) {
      r.xa[m] = *(const v4u32*)(mya + m * 32 * GSA + j * 8);
      if constexpr (!kquant(F)) r.dx[m] = lds[L::D + (ks * GKC + j) * 32 * MT + 32 * m + c32];
    }
    return r;
  };
  // the group's weight codes as int8 in the lanes' order
  auto codes = [&](const Ops& r) __attribute__((always_inline)) -> v4i {
    if constexpr (F == DT_Q8_0) {
      return __builtin_bit_cast(v4i, r.q16);
    } else {
      Raw v{};
      v.q0.x = r.q.x;
      v.q0.y = r.q.y;
      if constexpr (F == DT_Q5_0 || F == DT_Q5_1) v.b = r.b >> (8 * h);
      if constexpr (F == DT_Q6_K) {
        v.b = r.b >> (4 * h);
        v.c = r.c >> (4 * h);
      }
      return widen<F>(v);
    }
  };
  auto multiply = [&](const Ops& g, int m, const v4i& b) __attribute__((always_inline)) -> Sums {
    const v4i x = __builtin_bit_cast(v4i, g.xa[m]);
    Sums r;
    if constexpr (F == DT_Q6_K) {
      r.s = __builtin_amdgcn_mfma_i32_32x32x16_i8((long)(((uint64_t)(uint32_t)x.y << 32) | (uint32_t)x.x),
                                                  (long)(((uint64_t)(uint32_t)b.y << 32) | (uint32_t)b.x), zi, 0, 0, 0);
      r.s2 = __builtin_amdgcn_mfma_i32_32x32x16_i8((long)(((uint64_t)(uint32_t)x.w << 32) | (uint32_t)x.z),
                                                   (long)(((uint64_t)(uint32_t)b.w << 32) | (uint32_t)b.z), zi, 0, 0, 0);
    } else {
      r.s = __builtin_amdgcn_mfma_i32_32x32x32_i8(x, b, zi, 0, 0, 0);
    }
    if constexpr (!kquant(F)) {
      // dw dx of the 32 x 32 outputs as one outer product (k = 0 alone): both
      // halves, the product exact in single
      const v4u32 av = {g.dx[m] & lowhalf, 0, 0, 0}, bv = {g.x & lowhalf, 0, 0, 0};
      r.p = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h_t, av), __builtin_bit_cast(v8h_t, bv), zf,
                                                   0, 0, 0);
    }
    return r;
  };
  // Q4_K: the scales of groups 0..3 and 4..7 of the super-block, as bytes
  uint32_t sc0 = 0, sc1 = 0, hd0 = 0;
  // the terms of group j: K-quants into the super-block's integer sum, else
  // into the double sum (s dw dx is exact, one rounding per group)
  auto terms = [&](int j, int m, const Sums& r, uint32_t x) __attribute__((always_inline)) {
    if constexpr (F == DT_Q4_K) {
      const int sc = (int)(((j & 4) ? sc1 : sc0) >> (8 * (j & 3))) & 255;
#pragma unroll
      for (int i = 0; i < 16; i++) isum[m][i] = keep(isum[m][i] + __mul24(sc, r.s[i]));  // |sums| < 2^16, sc < 64
    } else if constexpr (F == DT_Q6_K) {
      const int sa = (int)(int8_t)(x & 255u), sb = (int)(int8_t)(x >> 8);
#pragma unroll
      for (int i = 0; i < 16; i++)
        isum[m][i] = keep(keep(isum[m][i] + __mul24(sa, r.s[i])) + __mul24(sb, r.s2[i]));
    } else {
#pragma unroll
      for (int i = 0; i < 16; i++) acc[m][i] = __builtin_fma((double)r.s[i], (double)r.p[i], acc[m][i]);
      if constexpr (F == DT_Q5_1) {
        const double m51 = half_to_float(x >> 16);
        const double* xs = (const double*)(lds + L::S) + (ks * GKC + j) * 32 * MT + 32 * m + 4 * h;
#pragma unroll
        for (int i = 0; i < 16; i++) acc[m][i] = __builtin_fma(m51, xs[8 * (i >> 2) + (i & 3)], acc[m][i]);
      }
    }
  };

  StepRegs<F, MT, KS> r;
  const int nch = (G + GKC - 1) / GKC, nst = (nch + KS - 1) / KS;
  step_load<F, MT, KS>(a, wb, rg, col0, sxr, xstride, G, 0, r);
  step_store<F, MT, KS>(r, lds);
  step_load<F, MT, KS>(a, wb, rg, col0, sxr, xstride, G, GKC * KS, r);
  __syncthreads();
  for (int c = 0; c < nst; c++) {
    const int ng = min(GKC, G - (c * KS + ks) * GKC);  // groups of this wave's chunk
    if constexpr (F == DT_Q4_K) {
      const uint4 hd = *(const uint4*)(lds + L::H + 4 * col);  // (scale_min_k4)
      sc0 = hd.y & 0x3f3f3f3fu;
      sc1 = (hd.w & 0x0f0f0f0fu) | ((hd.y >> 2) & 0x30303030u);
      hd0 = hd.x;
    }
    // (a chunk past the last: no terms; groups past the last in a chunk have
    // zero scales)
    if (ng > 0) {
      Ops g = read(0);
#pragma unroll
      for (int j = 0; j < GKC; j++) {
        const v4i b = codes(g);
        Sums s[MT];
#pragma unroll
        for (int m = 0; m < MT; m++) s[m] = multiply(g, m, b);
        const uint32_t x = g.x;
        // the next group's LDS reads are under way while the terms are formed
        if (j + 1 < GKC) g = read(j + 1);
#pragma unroll
        for (int m = 0; m < MT; m++) {
          terms(j, m, s[m], x);
          // (free to move them further, the scheduler would spill; Q6_K's
          // 64-row tile, at 256 registers, holds 11 in scratch even so)
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (kquant(F)) {
      // the super-block's term (rows hold whole ones): d dx isum, Q4_K
      // - dmin dx sum_j m_j bsum_j, the sum exact from one f16 MFMA over the
      // halves of the code sums (lane half 0: lo m_j, 1: hi 64 m_j)
      if (ng > 0) {
        double d, dm = 0;
        v8h_t bm;
        if constexpr (F == DT_Q4_K) {
          const uint4 hd = *(const uint4*)(lds + L::H + 4 * col);
          d = half_to_float(hd0 & 0xffffu);
          dm = -(double)half_to_float(hd0 >> 16);
          bm = bytes_half8(hd.z & 0x3f3f3f3fu, ((hd.w >> 4) & 0x0f0f0f0fu) | ((hd.z >> 2) & 0x30303030u),
                           (_Float16)(h ? 64.0f : 1.0f));
        } else {
          d = half_to_float(lds[L::H + col]);
        }
#pragma unroll
        for (int m = 0; m < MT; m++) {
          const double* xs = (const double*)(lds + L::D) + ks * 32 * MT + 32 * m + 4 * h;
          v16f_t cm;
          if constexpr (F == DT_Q4_K) {
            const v8h_t am = *(const v8h_t*)(lds + L::S + (ks * 32 * MT + 32 * m + c32) * 8 + 4 * h);
            cm = __builtin_amdgcn_mfma_f32_32x32x16_f16(am, bm, zf, 0, 0, 0);
          }
#pragma unroll
          for (int i = 0; i < 16; i++) {
            double v = d * (double)isum[m][i];
            if constexpr (F == DT_Q4_K) v = __builtin_fma(dm, (double)cm[i], v);
            acc[m][i] = __builtin_fma(xs[8 * (i >> 2) + (i & 3)], v, acc[m][i]);
            isum[m][i] = 0;
          }
        }
      }
    }
    __syncthreads();  // the step's LDS reads are done
    if (c + 1 < nst) {
      step_store<F, MT, KS>(r, lds);
      if (c + 2 < nst) step_load<F, MT, KS>(a, wb, rg, col0, sxr, xstride, G, (c + 2) * GKC * KS, r);
      __syncthreads();
    }
  }
  if constexpr (KS > 1) {
    // the partial sums of wave ks > 0 through LDS to wave ks = 0 of the column
    double* red = (double*)lds;
    if (ks > 0) {
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) red[(((wn * (KS - 1) + ks - 1) * MT + m) * 16 + i) * 64 + l] = acc[m][i];
    }
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int q = 0; q < KS - 1; q++)
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[m][i] += red[(((wn * (KS - 1) + q) * MT + m) * 16 + i) * 64 + l];
  }
  const int o = col0 + 32 * wn + c32;
  if (o >= a.out) return;
  const double b = bias ? (double)bias[o] : 0.0;
#pragma unroll
  for (int m = 0; m < MT; m++)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int rt = 32 * m + 8 * (i >> 2) + 4 * h + (i & 3);
      if (rt < nrows) {
        double v = acc[m][i];
        if (bias) v = b + v;
        a.y[(int64_t)syr[rt] * a.out + o] = (float)v;
      }
    }
}

template <int F, int MT, int KS>
__device__ __forceinline__ void gemm(const GemmArgs& a)
{
  constexpr int BM = 32 * MT;
  __shared__ __align__(16) uint32_t lds[GemmLds<F, MT, KS>::DWORDS];
  __shared__ int sxr[BM], syr[BM];
  const int t = threadIdx.x;
  const uint8_t* wb = a.w;
  const float* bias = a.bias;
  int nrows;
  if (a.items) {
    // an item of up to 64 slots: 64 / BM blocks
    constexpr int PARTS = 64 / BM;
    const int4 it = a.items[blockIdx.y / PARTS];
    const int r0 = (int)(blockIdx.y % PARTS) * BM;
    if (it.z <= r0) return;
    wb += (int64_t)it.x * a.stride;
    if (bias) bias += (int64_t)it.x * a.out;
    nrows = min(BM, it.z - r0);
    if (t < BM) {
      const int sl = a.perm[it.y + r0 + min(t, nrows - 1)];
      sxr[t] = a.x_per_slot ? sl / a.x_per_slot : 0;
      syr[t] = sl;
    }
  } else {
    const int r0 = blockIdx.y * BM;
    nrows = min(BM, a.rows - r0);
    if (t < BM) sxr[t] = syr[t] = r0 + min(t, nrows - 1);
  }
  __syncthreads();
  // an item (or a last tile) of at most 32 rows needs one tile a wave
  if constexpr (MT == 2) {
    if (nrows <= 32) {
      gemm_tiles<F, 1, KS>(a, wb, bias, nrows, sxr, syr, lds);
      return;
    }
  }
  gemm_tiles<F, MT, KS>(a, wb, bias, nrows, sxr, syr, lds);
}

// ------------------------------------------------ a small batch of rows
// gemm8: the same arithmetic for at most 8 activation rows (blockIdx.y: a
// chunk of 8 rows, or a grouped-expert item of at most 8 slots), the weights
// streamed once: a block owns 128 outputs (4 waves of 32) and walks the
// output tiles of its grid share. Per 32-value group a wave runs the MFMA of
// the big GEMM with the rows in A lanes 0..7 (lanes 8..31 zero): of its
// result registers, 0..3 hold the 8 rows x 32 outputs, one (row, output) per
// lane and register, so the scaling in double wastes no lane. The chunks of
// GKC groups (128 weight columns, 8 activation rows) are loaded coalesced
// into registers a chunk ahead, then through LDS to the lanes.
constexpr int G8N = 128;  // outputs of a block tile

struct Chunk8 {
  Raw wr[4];    // weight groups: column t / 8 + 32 p, group t % 8
  v4u32 xc[2];  // activation codes (t < 64): row t / 8, group t % 8
  float dx;
};

template <int F>
__device__ __forceinline__ void chunk8_load(const GemmArgs& a, const uint8_t* wb, const Regions& rg,
                                            int col0, const int* sxr, int64_t xstride, int G, int gc,
                                            Chunk8& cr)
{
  const int t = threadIdx.x;
  const int g = min(gc + (t & 7), G - 1);
#pragma unroll
  for (int p = 0; p < 4; p++) {
    const int64_t o = min(col0 + (t >> 3) + 32 * p, a.out - 1);
    load_group<F, true>(wb, rg, o, G, g, a.in, cr.wr[p]);
  }
  if (t < 64) {
    const uint8_t* xr = a.xq + (int64_t)sxr[t >> 3] * xstride;
    const v4u32* q = (const v4u32*)(xr + (int64_t)g * 32);
    cr.xc[0] = q[0];
    cr.xc[1] = q[1];
    cr.dx = ((const float*)(xr + a.in))[g];
  }
}

template <int F>
__device__ __forceinline__ void chunk8_store(const Chunk8& cr, uint32_t* sw, uint32_t* sa, float* sdx,
                                             int* sbs)
{
  const int t = threadIdx.x;
  constexpr int WS = GKC * raw_dwords<F>() + 1;
#pragma unroll
  for (int p = 0; p < 4; p++) raw_put<F>(sw + ((t >> 3) + 32 * p) * WS + (t & 7), GKC, cr.wr[p]);
  if (t < 64) {
    const int row = t >> 3, j = t & 7;
    uint32_t* d = sa + row * G8A + j * 8;
    *(v4u32*)d = cr.xc[0];
    *(v4u32*)(d + 4) = cr.xc[1];
    sdx[j * 8 + row] = cr.dx;
    if constexpr (needs_xsum(F)) {
      const v4u32 u0 = cr.xc[0], u1 = cr.xc[1];
      int sm = 0;
      sm = sdot4((int)u0.x, 0x01010101, sm); sm = sdot4((int)u0.y, 0x01010101, sm);
      sm = sdot4((int)u0.z, 0x01010101, sm); sm = sdot4((int)u0.w, 0x01010101, sm);
      sm = sdot4((int)u1.x, 0x01010101, sm); sm = sdot4((int)u1.y, 0x01010101, sm);
      sm = sdot4((int)u1.z, 0x01010101, sm); sm = sdot4((int)u1.w, 0x01010101, sm);
      sbs[j * 8 + row] = sm;
    }
  }
}

template <int F>
__device__ __forceinline__ void gemm8(const GemmArgs& a)
{
  constexpr int WS = GKC * raw_dwords<F>() + 1;
  __shared__ uint32_t sw_[G8N * WS];
  __shared__ __align__(16) uint32_t sa_[8 * G8A];
  __shared__ __align__(16) float sdx_[GKC * 8];
  __shared__ int sbs_[needs_xsum(F) ? GKC * 8 : 1];
  __shared__ int sxr[8], syr[8];
  const int t = threadIdx.x, l = t & 63, w = t >> 6, h = l >> 5;
  const int G = a.in >> 5;
  const int64_t xstride = (int64_t)a.in + 4 * (int64_t)G;
  const uint8_t* wb = a.w;
  const float* bias = a.bias;
  int nrows;
  if (a.items) {
    const int4 it = a.items[blockIdx.y];
    if (it.z <= 0) return;
    wb += (int64_t)it.x * a.stride;
    if (bias) bias += (int64_t)it.x * a.out;
    nrows = min(8, it.z);
    if (t < 8) {
      const int sl = a.perm[it.y + min(t, nrows - 1)];
      sxr[t] = a.x_per_slot ? sl / a.x_per_slot : 0;
      syr[t] = sl;
    }
  } else {
    const int r0 = blockIdx.y * 8;
    nrows = min(8, a.rows - r0);
    if (t < 8) sxr[t] = syr[t] = r0 + min(t, nrows - 1);
  }
  __syncthreads();
  const Regions rg = regions(F, a.out, a.in);
  const int ntiles = (a.out + G8N - 1) / G8N;
  const int nch = (G + GKC - 1) / GKC;
  // this block's (tile, chunk) steps, tile-major: step q is chunk q % nch of
  // tile blockIdx.x + (q / nch) gridDim.x
  const int mytiles = ((int)blockIdx.x < ntiles) ? (ntiles - 1 - (int)blockIdx.x) / (int)gridDim.x + 1 : 0;
  const int nsteps = mytiles * nch;
  if (nsteps == 0) return;
  const int arow = l & 31;  // A lane: row arow (rows 8.. are zero)
  const uint32_t* myw = sw_ + (32 * w + (l & 31)) * WS;
  const uint32_t* mya = sa_ + min(arow, 7) * G8A;
  auto step_at = [&](int q, int& col0, int& gc) {
    col0 = ((int)blockIdx.x + (q / nch) * (int)gridDim.x) * G8N;
    gc = (q % nch) * GKC;
  };
  double acc[4];
  int isum[4], msum[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    acc[i] = 0.0;
    isum[i] = msum[i] = 0;
  }
  Chunk8 cr;
  int col0, gc;
  step_at(0, col0, gc);
  chunk8_load<F>(a, wb, rg, col0, sxr, xstride, G, gc, cr);
  chunk8_store<F>(cr, sw_, sa_, sdx_, sbs_);
  if (nsteps > 1) {
    int c1, g1;
    step_at(1, c1, g1);
    chunk8_load<F>(a, wb, rg, c1, sxr, xstride, G, g1, cr);
  }
  __syncthreads();
  for (int q = 0; q < nsteps; q++) {
    step_at(q, col0, gc);
#pragma unroll
    for (int j = 0; j < GKC; j++) {
      const int g = gc + j;
      if (g < G) {
        const Raw r = raw_get<F>(myw + j, GKC);
        uint2 x0 = *(const uint2*)(mya + j * 8 + 2 * h);
        uint2 x1 = *(const uint2*)(mya + j * 8 + 4 + 2 * h);
        if (arow >= 8) x0 = x1 = make_uint2(0u, 0u);
        const float* sdx = sdx_ + j * 8;
        const int* sbs = sbs_ + (needs_xsum(F) ? j * 8 : 0);
        const v4i bv = b_operand<F>(r, h);
        v16i s;
        v16i s2 = {};
        if constexpr (F == DT_Q6_K) {
          const v16i z = {};
          s = __builtin_amdgcn_mfma_i32_32x32x16_i8(
              (long)(((uint64_t)x0.y << 32) | x0.x),
              (long)(((uint64_t)(uint32_t)bv.y << 32) | (uint32_t)bv.x), z, 0, 0, 0);
          s2 = __builtin_amdgcn_mfma_i32_32x32x16_i8(
              (long)(((uint64_t)x1.y << 32) | x1.x),
              (long)(((uint64_t)(uint32_t)bv.w << 32) | (uint32_t)bv.z), z, 0, 0, 0);
        } else {
          const v4i av = {(int)x0.x, (int)x0.y, (int)x1.x, (int)x1.y};
          const v16i z = {};
          s = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv, z, 0, 0, 0);
        }
        // result register i < 4 of lane l: row 4 h + i, output l % 32
        if constexpr (F == DT_Q4_K) {
          int sc, mn;
          scale_min_k4(g & 7, r.q1.y, r.q1.z, r.q1.w, sc, mn);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            isum[i] += __mul24(sc, s[i]);
            msum[i] += __mul24(mn, sbs[4 * h + i]);
          }
          if ((g & 7) == 7) {
            const double hd = half_to_float(r.q1.x & 0xffffu), hm = half_to_float(r.q1.x >> 16);
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const double dx = sdx[4 * h + i];
              acc[i] = acc[i] + ((hd * dx) * (double)isum[i] - (hm * dx) * (double)msum[i]);
              isum[i] = msum[i] = 0;
            }
          }
        } else if constexpr (F == DT_Q6_K) {
          const int sa = (int)(int8_t)(r.a & 255u), sb = (int)(int8_t)(r.a >> 8);
#pragma unroll
          for (int i = 0; i < 4; i++) isum[i] += __mul24(sa, s[i]) + __mul24(sb, s2[i]);
          if ((g & 7) == 7) {
            const double d = half_to_float(r.d);
#pragma unroll
            for (int i = 0; i < 4; i++) {
              const double dx = sdx[4 * h + i];
              acc[i] = acc[i] + (d * dx) * (double)isum[i];
              isum[i] = 0;
            }
          }
        } else if constexpr (F == DT_Q5_1) {
          const double d = half_to_float(r.a & 0xffffu), m = half_to_float(r.a >> 16);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const double dx = sdx[4 * h + i];
            const double tt = (double)s[i] * (d * dx);
            acc[i] = acc[i] + (tt + m * (dx * (double)sbs[4 * h + i]));
          }
        } else {
          double dw;
          if constexpr (F == DT_MXFP4) dw = mxfp4_q8_scale(r.a);
          else dw = half_to_float(r.a);
          const float4 d4 = *(const float4*)&sdx[4 * h];
          const double dxs[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
          for (int i = 0; i < 4; i++) acc[i] = __builtin_fma((double)s[i], dw * dxs[i], acc[i]);
        }
      }
    }
    __syncthreads();  // the chunk's LDS reads are done
    if (q + 1 < nsteps) {
      chunk8_store<F>(cr, sw_, sa_, sdx_, sbs_);
      if (q + 2 < nsteps) {
        int c2, g2;
        step_at(q + 2, c2, g2);
        chunk8_load<F>(a, wb, rg, c2, sxr, xstride, G, g2, cr);
      }
    }
    // the tile's last chunk: its outputs, then a fresh sum
    if (q % nch == nch - 1) {
      const int o = col0 + 32 * w + (l & 31);
      if (o < a.out) {
        const double b = bias ? (double)bias[o] : 0.0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const int rt = 4 * h + i;
          if (rt < nrows) {
            double v = acc[i];
            if (bias) v = b + v;
            a.y[(int64_t)syr[rt] * a.out + o] = (float)v;
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        acc[i] = 0.0;
        isum[i] = msum[i] = 0;
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------- float weights
// y[r, o] = bias[o] + sum_i x[r, i] w[o, i] for F32 / BF16 / F16 weights in
// the Q8 arithmetic of TInferCpuBackend.Linear's float branch
// (backend.cpu.pas:1548-1565): every product of a float activation and a
// float weight is exact in double, and the sum runs in double, here on the
// f64 matrix cores (v_mfma_f64_16x16x4_f64; only the order of the double sum
// differs from the CPU's). A block owns BM rows x 4096 / BM outputs, each of
// its 4 waves 32 x 32 as 2 x 2 tiles of 16 x 16; chunks of FKC values of x and
// w are loaded as 16-byte words into LDS (the next chunk's loads in flight
// while one is computed; in is a multiple of 32, so chunks are whole).
//
// A lane group's k values are a contiguous quarter of the chunk, so a lane
// reads its 8 steps of a tile row as two 16-byte LDS words. Bound by the f64
// matrix cores (a 64-cycle MFMA per 1024 products: 307 of the 714 us of 1024
// rows 2880 -> 4096 before, when the operands came by 4-byte loads and LDS
// reads; 397 now). 32 rows x 128 outputs for up to 32 rows, whose
// matrix work is half a 64-row tile's.
typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int FKC = 32;       // values of the sum per chunk
constexpr int FST = FKC + 4;  // LDS floats of a row's chunk

// N values from element i of float weights, widened
template <int F, int N>
__device__ __forceinline__ void wvals(const uint8_t* w, int64_t i, float (&v)[N])
{
  if constexpr (F == DT_F32) {
    const v4u32* p = (const v4u32*)(w + i * 4);
#pragma unroll
    for (int k = 0; k < N / 4; k++) {
      const v4u32 u = p[k];
      v[4 * k] = bits_float(u.x);
      v[4 * k + 1] = bits_float(u.y);
      v[4 * k + 2] = bits_float(u.z);
      v[4 * k + 3] = bits_float(u.w);
    }
  } else {
    const v4u32* p = (const v4u32*)(w + i * 2);
#pragma unroll
    for (int k = 0; k < N / 8; k++) {
      const v4u32 u = p[k];
      const uint32_t q[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
      for (int j = 0; j < 4; j++) {
        v[8 * k + 2 * j] = F == DT_BF16 ? bits_float(q[j] << 16) : half_to_float(q[j] & 0xffffu);
        v[8 * k + 2 * j + 1] = F == DT_BF16 ? bits_float(q[j] & 0xffff0000u) : half_to_float(q[j] >> 16);
      }
    }
  }
}

template <int F, int BM>
__device__ __forceinline__ void gemm_flt(const GemmArgs& a)
{
  constexpr int BN = 4096 / BM;
  constexpr int XT = 256 / BM, XN = FKC / XT;  // threads and values of a row's chunk
  constexpr int WT = 256 / BN, WN = FKC / WT;
  __shared__ __align__(16) float xs[2][BM][FST];
  __shared__ __align__(16) float ws[2][BN][FST];
  __shared__ int sxr[BM], syr[BM];
  const int t = threadIdx.x, l = t & 63, w = t >> 6;
  const int wm = w % (BM / 32), wn = w / (BM / 32);
  const uint8_t* wb = a.w;
  const float* bias = a.bias;
  int nrows;
  if (a.items) {
    const int4 it = a.items[blockIdx.y];
    if (it.z <= 0) return;
    wb += (int64_t)it.x * a.stride;
    if (bias) bias += (int64_t)it.x * a.out;
    nrows = min(BM, it.z);
    if (t < BM) {
      const int sl = a.perm[it.y + min(t, nrows - 1)];
      sxr[t] = a.x_per_slot ? sl / a.x_per_slot : 0;
      syr[t] = sl;
    }
  } else {
    const int r0 = blockIdx.y * BM;
    nrows = min(BM, a.rows - r0);
    if (t < BM) sxr[t] = syr[t] = r0 + min(t, nrows - 1);
  }
  __syncthreads();
  const int col0 = blockIdx.x * BN;
  // this block's values of the sum: [kb, ke)
  const int kb = a.ksplit > 1 ? (int)blockIdx.z * a.klen : 0;
  const int ke = a.ksplit > 1 ? min(a.in, kb + a.klen) : a.in;
  const int nch = (ke - kb) / FKC;  // (a split past the end: none)
  // a thread's share of a chunk
  const int xr = t / XT, xk = XN * (t % XT), wr = t / WT, wk = WN * (t % WT);
  const float* xrow = a.x + (int64_t)sxr[xr] * a.in + xk;
  const int64_t wrow = (int64_t)min(col0 + wr, a.out - 1) * a.in + wk;
  float xv[XN], wv[WN];
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < XN / 4; u++) {
      const float4 v = *(const float4*)(xrow + k0 + 4 * u);
      xv[4 * u] = v.x;
      xv[4 * u + 1] = v.y;
      xv[4 * u + 2] = v.z;
      xv[4 * u + 3] = v.w;
    }
    wvals<F, WN>(wb, wrow + k0, wv);
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < XN; u += 4) *(float4*)&xs[buf][xr][xk + u] = make_float4(xv[u], xv[u + 1], xv[u + 2], xv[u + 3]);
#pragma unroll
    for (int u = 0; u < WN; u += 4) *(float4*)&ws[buf][wr][wk + u] = make_float4(wv[u], wv[u + 1], wv[u + 2], wv[u + 3]);
  };
  v4d acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
  if (nch > 0) {
    load(kb);
    store(0);
  }
  __syncthreads();
  // operand lane mapping of v_mfma_f64_16x16x4_f64 (probed on gfx950): A
  // lane l = row l % 16, k = l / 16; B lane l = column l % 16, k = l / 16;
  // result register e of lane l = row 4 e + l / 16, column l % 16
  const int ar = l & 15, ak = l >> 4;
  for (int c = 0; c < nch; c++) {
    const int buf = c & 1;
    if (c + 1 < nch) load(kb + (c + 1) * FKC);
    const float* xp = &xs[buf][32 * wm + ar][8 * ak];
    const float* wp = &ws[buf][32 * wn + ar][8 * ak];
#pragma unroll
    for (int q = 0; q < 8; q += 4) {
      float4 av[2], bv[2];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        av[i] = *(const float4*)(xp + 16 * i * FST + q);
        bv[i] = *(const float4*)(wp + 16 * i * FST + q);
      }
#pragma unroll
      for (int u = 0; u < 4; u++) {
        double ad[2], bd[2];
#pragma unroll
        for (int i = 0; i < 2; i++) {
          ad[i] = u == 0 ? av[i].x : u == 1 ? av[i].y : u == 2 ? av[i].z : av[i].w;
          bd[i] = u == 0 ? bv[i].x : u == 1 ? bv[i].y : u == 2 ? bv[i].z : bv[i].w;
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ad[i], bd[j], acc[i][j], 0, 0, 0);
      }
    }
    // (the other buffer was last read before the barrier that ended the chunk
    // before)
    if (c + 1 < nch) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int o = col0 + 32 * wn + 16 * j + ar;
    if (o >= a.out) continue;
    const double b = bias ? (double)bias[o] : 0.0;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int rt = 32 * wm + 16 * i + 4 * e + ak;
        if (rt < nrows) {
          double v = acc[i][j][e];
          if (a.ksplit > 1) {
            a.part[((int64_t)blockIdx.z * a.rows + syr[rt]) * a.out + o] = v;
            continue;
          }
          if (bias) v = b + v;
          a.y[(int64_t)syr[rt] * a.out + o] = (float)v;
        }
      }
  }
}

}  // namespace ihip

#define IHIP_GEMM_TILES(NAME, F, MT, KS)                                                            \
  extern "C" __global__ __launch_bounds__(256, 2) void gemm_##NAME##_m##MT##k##KS(ihip::GemmArgs a) \
  {                                                                                                 \
    ihip::gemm<F, MT, KS>(a);                                                                       \
  }
// (64-row tiles share a K-quant's decode between two MFMA tiles; the formats
// of 32 values would spill in them, two doubles an output and group)
#define IHIP_GEMM_K(NAME, F)     \
  IHIP_GEMM_TILES(NAME, F, 2, 1) \
  IHIP_GEMM(NAME, F)
#define IHIP_GEMM(NAME, F)                                                                          \
  IHIP_GEMM_TILES(NAME, F, 1, 1)                                                                    \
  IHIP_GEMM_TILES(NAME, F, 1, 2)                                                                    \
  IHIP_GEMM_TILES(NAME, F, 1, 4)                                                                    \
  extern "C" __global__ __launch_bounds__(256) void gemm8_##NAME(ihip::GemmArgs a)                    \
  {                                                                                                 \
    ihip::touch_kernargs<sizeof(ihip::GemmArgs)>();                                                 \
    ihip::gemm8<F>(a);                                                                              \
  }

#define IHIP_GEMM_FLT(NAME, F)                                                               \
  extern "C" __global__ __launch_bounds__(256, 4) void gemm_##NAME##_r64(ihip::GemmArgs a) \
  {                                                                                          \
    ihip::gemm_flt<F, 64>(a);                                                                \
  }                                                                                          \
  extern "C" __global__ __launch_bounds__(256, 4) void gemm_##NAME##_r32(ihip::GemmArgs a) \
  {                                                                                          \
    ihip::gemm_flt<F, 32>(a);                                                                \
  }

#ifdef IHIP_ONLY_FMT_Q8_0
IHIP_GEMM(q8_0, ihip::DT_Q8_0)
#endif
#ifdef IHIP_ONLY_FMT_F32
IHIP_GEMM_FLT(f32, ihip::DT_F32)
#endif
#ifdef IHIP_ONLY_FMT_BF16
IHIP_GEMM_FLT(bf16, ihip::DT_BF16)
#endif
#ifdef IHIP_ONLY_FMT_F16
IHIP_GEMM_FLT(f16, ihip::DT_F16)
#endif
#ifdef IHIP_ONLY_FMT_Q4_0
IHIP_GEMM(q4_0, ihip::DT_Q4_0)
#endif
#ifdef IHIP_ONLY_FMT_MXFP4
extern "C" __global__ __launch_bounds__(256) void gemm_mxfp4_f8(ihip::GemmArgs a) { ihip::gemm_mxfp4_f8(a); }
extern "C" __global__ __launch_bounds__(256) void f8_planes(ihip::PlanesArgs a) { ihip::f8_planes(a); }
IHIP_GEMM(mxfp4, ihip::DT_MXFP4)
#endif
#ifdef IHIP_ONLY_FMT_Q5_0
IHIP_GEMM(q5_0, ihip::DT_Q5_0)
#endif
#ifdef IHIP_ONLY_FMT_Q5_1
IHIP_GEMM(q5_1, ihip::DT_Q5_1)
#endif
#ifdef IHIP_ONLY_FMT_Q4_K
IHIP_GEMM_K(q4_k, ihip::DT_Q4_K)
#endif
#ifdef IHIP_ONLY_FMT_Q6_K
IHIP_GEMM_K(q6_k, ihip::DT_Q6_K)
#endif
