// deltanet.hip - the Gated DeltaNet mixer of Qwen3.5 and the output gate of its
// full attention on gfx950: TDecoderModel.DeltaPrep (decoder.pas:2755-2855),
// TInferBackend.DeltaRule (backend.cpu.pas:1890-1972), the gated RMSNorm of
// DeltaNetBlock (decoder.pas:2740-2745) and GateBySigmoid (:2594-2610); the
// device contract of tools/cuda/deltanet.cu (dnconv, dnprep, deltarule,
// gatednorm, splitgate, gatemul).
//
// The arithmetic is the CPU's: single steps round to single, the sums are
// double (products of two singles are exact in double, so an fma is the
// CPU's add of the product). Sums over a wave are reduced in a tree, not in
// the CPU's serial order: the double results differ in the last bits, the
// single results they round to almost never.
//
// The states live on the device per DeltaNet layer: conv [channels, kw - 1]
// (the last inputs, oldest first) and S [value heads, value dim, key dim].
#include "common.h"

using namespace ihip;

// Silu (decoder.pas:2612-2623): x / (1 + exp(-x)) in double, 0 below -100
__device__ __forceinline__ float dn_silu(float x)
{
  const double d = x;
  if (d < -100) return 0.0f;
  return (float)(d / (1.0 + exp(-d)));
}

// 1 / (1 + exp(-x)) in double rounded to single, 0 below -100
__device__ __forceinline__ float dn_sigmoid(float x)
{
  const double d = x;
  if (d < -100) return 0.0f;
  return (float)(1.0 / (1.0 + exp(-d)));
}

// the largest convolution and key dimension handled (a lane keeps
// DN_MAXK / 64 values of a state column)
#define DN_MAXKW 8
#define DN_MAXK 256

struct DnConvArgs {
  float* qkv;        // [rows, channels], convolved and silu'd in place
  const float* w;    // [channels, kw]
  float* conv;       // [channels, kw - 1], moved on
  int32_t rows, channels, kw, pad;
};

// the causal depthwise convolution, one thread per channel over every row in
// order: weight kw - 1 takes the new input, weights 0.. the kept inputs
// (oldest first); then silu
extern "C" __global__ __launch_bounds__(256) void dn_conv(DnConvArgs a)
{
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c >= a.channels) return;
  const int k1 = a.kw - 1;
  float st[DN_MAXKW], w[DN_MAXKW];
#pragma unroll
  for (int j = 0; j < DN_MAXKW; j++) {
    st[j] = j < k1 ? a.conv[(int64_t)c * k1 + j] : 0.f;
    w[j] = j < a.kw ? a.w[(int64_t)c * a.kw + j] : 0.f;
  }
  float wl = w[0];
#pragma unroll
  for (int j = 1; j < DN_MAXKW; j++)
    if (j == k1) wl = w[j];
  for (int t = 0; t < a.rows; t++) {
    const int64_t i = (int64_t)t * a.channels + c;
    const float x = a.qkv[i];
    double acc = (double)wl * (double)x;
#pragma unroll
    for (int j = 0; j < DN_MAXKW; j++)
      if (j < k1) acc = __builtin_fma((double)w[j], (double)st[j], acc);
#pragma unroll
    for (int j = 0; j + 1 < DN_MAXKW; j++)
      if (j + 1 < k1) st[j] = st[j + 1];
#pragma unroll
    for (int j = 0; j < DN_MAXKW; j++)
      if (j == k1 - 1) st[j] = x;
    a.qkv[i] = dn_silu((float)acc);
  }
#pragma unroll
  for (int j = 0; j < DN_MAXKW; j++)
    if (j < k1) a.conv[(int64_t)c * k1 + j] = st[j];
}

struct DnPrepArgs {
  float* qkv;          // [rows, channels]: [q heads | k heads | v heads]
  float* beta;         // [rows, vh]: in_proj_b, becomes sigmoid(b)
  float* decay;        // [rows, vh]: in_proj_a, becomes the decay
  float* z;            // [rows, vh * dv]: becomes silu(z)
  const float* dt_bias;  // [vh]
  const float* neg_a;    // [vh]: -exp(A_log)
  int32_t kh, vh, dk, dv, channels, pad;
};

// per (item, row), one wave: a q or k head L2-normed (x / sqrt(sum x^2 +
// 1e-6), the queries also times dk^-0.5 as a single factor); a value head:
// beta = sigmoid(b), decay = exp(neg_a * softplus(a + dt_bias)) (beyond 20
// softplus is its input; below 1e-6 exp gives log1p's value e - e^2 / 2),
// silu of its z
extern "C" __global__ __launch_bounds__(64) void dn_prep(DnPrepArgs a)
{
  const int item = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
  const int i = item - 2 * a.kh;
  if (i < 0) {
    float* s = a.qkv + (int64_t)t * a.channels + (int64_t)item * a.dk;
    double acc = 0;
    for (int j = lane; j < a.dk; j += 64) {
      const double e = s[j];
      acc = __builtin_fma(e, e, acc);
    }
    acc = wave_sum(acc, 64);
    const float f = (float)(1.0 / sqrt(acc + 1e-6));
    const float scale = (float)(1.0 / sqrt((double)a.dk));
    for (int j = lane; j < a.dk; j += 64) {
      float v = s[j] * f;
      if (item < a.kh) v = v * scale;
      s[j] = v;
    }
    return;
  }
  const int64_t f = (int64_t)t * a.vh + i;
  if (lane == 0) {
    a.beta[f] = dn_sigmoid(a.beta[f]);
    const float x = a.decay[f] + a.dt_bias[i];
    float sp;
    if (x > 20) {
      sp = x;
    } else {
      const double e = exp((double)x);
      sp = e < 1e-6 ? (float)(e - e * e / 2) : (float)log(1.0 + e);
    }
    sp = a.neg_a[i] * sp;
    a.decay[f] = (float)exp((double)sp);
  }
  float* zz = a.z + f * a.dv;
  for (int j = lane; j < a.dv; j += 64) zz[j] = dn_silu(zz[j]);
}

struct DnConvPrepArgs {
  float* qkv;          // [channels]: one row, convolved, silu'd and prepared in place
  const float* w;      // [channels, kw]
  float* conv;         // [channels, kw - 1], moved on
  float* beta;         // [vh]
  float* decay;        // [vh]
  float* z;            // [vh * dv]
  const float* dt_bias;
  const float* neg_a;
  int32_t kh, vh, dk, dv, channels, kw;
};

// one row: the convolution of an item's channels and the item's DeltaPrep in
// one launch (dn_conv then dn_prep's arithmetic), one wave per item - a q or
// k head (its dk channels convolved, then L2-normed), or a value head (its dv
// channels convolved; beta, decay, silu(z))
extern "C" __global__ __launch_bounds__(64) void dn_convprep1(DnConvPrepArgs a)
{
  const int item = blockIdx.x, lane = threadIdx.x;
  const int i = item - 2 * a.kh;
  const int first = i < 0 ? item * a.dk : 2 * a.kh * a.dk + i * a.dv;
  const int cnt = i < 0 ? a.dk : a.dv;
  const int k1 = a.kw - 1;
  constexpr int NC = DN_MAXK / 64;  // channels per lane (items of up to 256)
  float y[NC];
#pragma unroll
  for (int u = 0; u < NC; u++) {
    y[u] = 0.f;
    const int cc = lane + 64 * u;
    if (cc >= cnt) continue;
    const int64_t c = first + cc;
    float st[DN_MAXKW], w[DN_MAXKW];
#pragma unroll
    for (int j = 0; j < DN_MAXKW; j++) {
      st[j] = j < k1 ? a.conv[c * k1 + j] : 0.f;
      w[j] = j < a.kw ? a.w[c * a.kw + j] : 0.f;
    }
    float wl = w[0];
#pragma unroll
    for (int j = 1; j < DN_MAXKW; j++)
      if (j == k1) wl = w[j];
    const float x = a.qkv[c];
    double acc = (double)wl * (double)x;
#pragma unroll
    for (int j = 0; j < DN_MAXKW; j++)
      if (j < k1) acc = __builtin_fma((double)w[j], (double)st[j], acc);
#pragma unroll
    for (int j = 0; j + 1 < DN_MAXKW; j++)
      if (j + 1 < k1) a.conv[c * k1 + j] = st[j + 1];
    if (k1 > 0) a.conv[c * k1 + k1 - 1] = x;
    y[u] = dn_silu((float)acc);
  }
  if (i < 0) {
    double acc = 0;
#pragma unroll
    for (int u = 0; u < NC; u++) {
      const double e = y[u];
      acc = __builtin_fma(e, e, acc);
    }
    acc = wave_sum(acc, 64);
    const float f = (float)(1.0 / sqrt(acc + 1e-6));
    const float scale = (float)(1.0 / sqrt((double)a.dk));
#pragma unroll
    for (int u = 0; u < NC; u++) {
      const int cc = lane + 64 * u;
      if (cc >= cnt) continue;
      float v = y[u] * f;
      if (item < a.kh) v = v * scale;
      a.qkv[first + cc] = v;
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < NC; u++) {
    const int cc = lane + 64 * u;
    if (cc < cnt) a.qkv[first + cc] = y[u];
  }
  if (lane == 0) {
    a.beta[i] = dn_sigmoid(a.beta[i]);
    const float x = a.decay[i] + a.dt_bias[i];
    float sp;
    if (x > 20) {
      sp = x;
    } else {
      const double e = exp((double)x);
      sp = e < 1e-6 ? (float)(e - e * e / 2) : (float)log(1.0 + e);
    }
    sp = a.neg_a[i] * sp;
    a.decay[i] = (float)exp((double)sp);
  }
  float* zz = a.z + (int64_t)i * a.dv;
  for (int j = lane; j < a.dv; j += 64) zz[j] = dn_silu(zz[j]);
}

struct DnRowsArgs {
  const float* x;      // [rows, channels]: the projected channels
  float* y;            // [rows, channels]: convolved, silu'd and prepared
  const float* w;      // [channels, kw]
  float* conv;         // [channels, kw - 1], moved on
  float* beta;         // [rows, vh]
  float* decay;        // [rows, vh]
  float* z;            // [rows, vh * dv]
  const float* dt_bias;
  const float* neg_a;
  int32_t kh, vh, dk, dv, channels, kw, rows, pad;
};

// The convolution and DeltaPrep of a prompt chunk in one launch: one wave per
// (item, row), dn_conv's and dn_prep's arithmetic. A row's convolution reads
// the kw - 1 rows before it from x, so it writes to y, and every row is
// computed on its own: (items) x (rows / 4) blocks fill the chip, where a
// thread per channel walking the rows in order (24 blocks for 6144 channels)
// waited for a load and a store per row. Bound by silu's double exp and
// division (two per channel and row in all). Qwen3.5-0.8B's layer, 512 rows of
// 6144 channels: 256 + 16 us as dn_conv and dn_prep, 33 us as this.
// The kept inputs are read by the blocks of the first rows alone; the block
// of row group 0 writes the new ones after its own reads, so no other block
// meets them half changed.
extern "C" __global__ __launch_bounds__(256) void dn_convprep(DnRowsArgs a)
{
  const int item = blockIdx.x, lane = threadIdx.x & 63;
  const int t = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int i = item - 2 * a.kh;
  const int first = i < 0 ? item * a.dk : 2 * a.kh * a.dk + i * a.dv;
  const int cnt = i < 0 ? a.dk : a.dv;
  const int k1 = a.kw - 1;
  constexpr int NC = DN_MAXK / 64;  // channels per lane (items of up to 256)
  if (t < a.rows) {
    float y[NC];
#pragma unroll
    for (int u = 0; u < NC; u++) {
      y[u] = 0.f;
      const int cc = lane + 64 * u;
      if (cc >= cnt) continue;
      const int64_t c = first + cc;
      float st[DN_MAXKW], w[DN_MAXKW];
      // input j of the row is row t - k1 + j, or a kept input before the chunk
#pragma unroll
      for (int j = 0; j < DN_MAXKW; j++) {
        const int r = t - k1 + j;
        st[j] = j > k1 ? 0.f : r >= 0 ? a.x[(int64_t)r * a.channels + c] : a.conv[c * k1 + k1 + r];
        w[j] = j <= k1 ? a.w[c * a.kw + j] : 0.f;
      }
      float wl = w[0], xl = st[0];
#pragma unroll
      for (int j = 1; j < DN_MAXKW; j++)
        if (j == k1) {
          wl = w[j];
          xl = st[j];
        }
      double acc = (double)wl * (double)xl;
#pragma unroll
      for (int j = 0; j < DN_MAXKW; j++)
        if (j < k1) acc = __builtin_fma((double)w[j], (double)st[j], acc);
      y[u] = dn_silu((float)acc);
    }
    float* yr = a.y + (int64_t)t * a.channels + first;
    if (i < 0) {
      double acc = 0;
#pragma unroll
      for (int u = 0; u < NC; u++) {
        const double e = y[u];
        acc = __builtin_fma(e, e, acc);
      }
      acc = wave_sum(acc, 64);
      const float f = (float)(1.0 / sqrt(acc + 1e-6));
      const float scale = (float)(1.0 / sqrt((double)a.dk));
#pragma unroll
      for (int u = 0; u < NC; u++) {
        const int cc = lane + 64 * u;
        if (cc >= cnt) continue;
        float v = y[u] * f;
        if (item < a.kh) v = v * scale;
        yr[cc] = v;
      }
    } else {
#pragma unroll
      for (int u = 0; u < NC; u++) {
        const int cc = lane + 64 * u;
        if (cc < cnt) yr[cc] = y[u];
      }
      const int64_t f = (int64_t)t * a.vh + i;
      if (lane == 0) {
        a.beta[f] = dn_sigmoid(a.beta[f]);
        const float x = a.decay[f] + a.dt_bias[i];
        float sp;
        if (x > 20) {
          sp = x;
        } else {
          const double e = exp((double)x);
          sp = e < 1e-6 ? (float)(e - e * e / 2) : (float)log(1.0 + e);
        }
        sp = a.neg_a[i] * sp;
        a.decay[f] = (float)exp((double)sp);
      }
      float* zz = a.z + f * a.dv;
      for (int j = lane; j < a.dv; j += 64) zz[j] = dn_silu(zz[j]);
    }
  }
  // the kept inputs moved on to the chunk's last ones
  if (blockIdx.y != 0 || k1 == 0) return;
  __syncthreads();  // rows 0 .. 3 have read the old ones
  for (int cc = threadIdx.x; cc < cnt; cc += 256) {
    const int64_t c = first + cc;
    float st[DN_MAXKW];
#pragma unroll
    for (int j = 0; j < DN_MAXKW; j++) {
      const int r = a.rows - k1 + j;
      st[j] = j >= k1 ? 0.f : r >= 0 ? a.x[(int64_t)r * a.channels + c] : a.conv[c * k1 + k1 + r];
    }
#pragma unroll
    for (int j = 0; j < DN_MAXKW; j++)
      if (j < k1) a.conv[c * k1 + j] = st[j];
  }
}

struct DnRuleArgs {
  const float* qkv;    // [rows, stride]: [q heads | k heads | v heads]
  const float* beta;   // [rows, vh]
  const float* decay;  // [rows, vh]
  float* state;        // [vh, dv, dk]
  float* y;            // [rows, vh * dv]
  int32_t rows, stride, kh, vh, dk, dv, group, pad;
};

// the delta rule over rows tokens in order: one wave per column j of a
// value head's S (block = 4 columns of one head), the column in registers
// (DN_MAXK / 64 values per lane) across every token. Per token: the column
// decayed, what it predicts for the key (a double sum), delta = (v_j -
// prediction) * beta, k * delta written in, the column read by the query.
// The next token's operands are loaded while this one is computed.
extern "C" __global__ __launch_bounds__(256) void dn_rule(DnRuleArgs a)
{
  constexpr int NV = DN_MAXK / 64;
  const int head = blockIdx.x, lane = threadIdx.x & 63;
  const int j = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (j >= a.dv) return;
  const int kd = a.kh * a.dk, vdw = a.vh * a.dv;
  const int off = ((head / a.group) % a.kh) * a.dk;
  float* col = a.state + ((int64_t)head * a.dv + j) * a.dk;
  float s[NV];
#pragma unroll
  for (int m = 0; m < NV; m++) {
    const int i = lane + 64 * m;
    s[m] = i < a.dk ? col[i] : 0.f;
  }
  // the operands of token t: q and k of the key head (lane's share), v_j,
  // the decay and beta of the head
  float q[NV], k[NV], v = 0.f, g = 0.f, b = 0.f;
  auto load = [&](int t, float (&qq)[NV], float (&kk)[NV], float& vv, float& gg, float& bb) {
    const float* r = a.qkv + (int64_t)t * a.stride;
#pragma unroll
    for (int m = 0; m < NV; m++) {
      const int i = lane + 64 * m;
      qq[m] = i < a.dk ? r[off + i] : 0.f;
      kk[m] = i < a.dk ? r[kd + off + i] : 0.f;
    }
    vv = r[2 * kd + head * a.dv + j];
    gg = a.decay[(int64_t)t * a.vh + head];
    bb = a.beta[(int64_t)t * a.vh + head];
  };
  if (a.rows > 0) load(0, q, k, v, g, b);
  for (int t = 0; t < a.rows; t++) {
    float qn[NV] = {}, kn[NV] = {}, vn = 0.f, gn = 0.f, bn = 0.f;
    if (t + 1 < a.rows) load(t + 1, qn, kn, vn, gn, bn);
    double acc = 0;
#pragma unroll
    for (int m = 0; m < NV; m++) {
      s[m] = s[m] * g;
      acc = __builtin_fma((double)s[m], (double)k[m], acc);
    }
    acc = wave_sum(acc, 64);
    const float pred = (float)acc;
    float delta = v - pred;
    delta = delta * b;
    double o = 0;
#pragma unroll
    for (int m = 0; m < NV; m++) {
      const float p = k[m] * delta;
      s[m] = s[m] + p;
      o = __builtin_fma((double)s[m], (double)q[m], o);
    }
    o = wave_sum(o, 64);
    if (lane == 0) a.y[(int64_t)t * vdw + head * a.dv + j] = (float)o;
#pragma unroll
    for (int m = 0; m < NV; m++) {
      q[m] = qn[m];
      k[m] = kn[m];
    }
    v = vn;
    g = gn;
    b = bn;
  }
#pragma unroll
  for (int m = 0; m < NV; m++) {
    const int i = lane + 64 * m;
    if (i < a.dk) col[i] = s[m];
  }
}

// The delta rule of a prompt chunk: dn_rule's arithmetic and sum order, two
// columns per wave (a column over 32 lanes, NM pairs of values each, lane L
// holding values 2L and 2L + 1 of every 64: the first level of dn_rule's wave
// sum is then inside the lane), the tokens' operands staged through LDS in
// chunks of CT, the next chunk's loads in flight while one is computed.
// Bound by a token's serial chain (the prediction's wave sum, delta, the
// column's update), which the next token's loads, one memory round trip a
// token, stretched in dn_rule: 16 heads of 128 x 128, 512 tokens, 455 us there,
// 145 us here (190 with each token's output summed on its own).
template <int NM, int CT>
__device__ __forceinline__ void dn_rule_chunks(const DnRuleArgs& a)
{
  constexpr int W = 64 * NM;         // a token's q (or k) in LDS, zeros past dk
  constexpr int PRE = CT * 2 * W / 256;
  __shared__ float sq[2][CT][2][W];  // [buffer][token][q, k]
  __shared__ float sv[2][CT][8];     // v of the block's 8 columns
  __shared__ float sg[2][CT][2];     // decay, beta
  const int t = threadIdx.x, head = blockIdx.x, L = t & 31;
  const int jl = t >> 5, j = blockIdx.y * 8 + jl;
  const int kd = a.kh * a.dk, vdw = a.vh * a.dv;
  const int off = ((head / a.group) % a.kh) * a.dk;
  float* col = a.state + ((int64_t)head * a.dv + min(j, a.dv - 1)) * a.dk;
  float s[NM][2];
#pragma unroll
  for (int m = 0; m < NM; m++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int i = 64 * m + 2 * L + e;
      s[m][e] = i < a.dk ? col[i] : 0.f;
    }
  // a thread's share of a chunk's operands, in registers until the chunk
  // before is computed
  float pre[PRE], pv = 0.f, pg = 0.f;
  auto load = [&](int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PRE; u++) {
      const int e = t + 256 * u, tok = min(t0 + e / (2 * W), a.rows - 1), i = e % W;
      const int base = (e / W) & 1 ? kd + off : off;
      pre[u] = i < a.dk ? a.qkv[(int64_t)tok * a.stride + base + i] : 0.f;
    }
    if (t < CT * 8) {
      const int tok = min(t0 + (t >> 3), a.rows - 1);
      const int c = min((int)blockIdx.y * 8 + (t & 7), a.dv - 1);
      pv = a.qkv[(int64_t)tok * a.stride + 2 * kd + (int64_t)head * a.dv + c];
    } else if (t < CT * 10) {
      const int u = t - CT * 8, tok = min(t0 + (u >> 1), a.rows - 1);
      pg = ((u & 1) ? a.beta : a.decay)[(int64_t)tok * a.vh + head];
    }
  };
  auto store = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PRE; u++) (&sq[b][0][0][0])[t + 256 * u] = pre[u];
    if (t < CT * 8) sv[b][t >> 3][t & 7] = pv;
    else if (t < CT * 10) (&sg[b][0][0])[t - CT * 8] = pg;
  };
  // one token: the state moved on, this lane's part of the output
  auto token = [&](int buf, int u) __attribute__((always_inline)) -> double {
    float q[NM][2], k[NM][2];
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const float2 qq = *(const float2*)&sq[buf][u][0][64 * m + 2 * L];
      const float2 kk = *(const float2*)&sq[buf][u][1][64 * m + 2 * L];
      q[m][0] = qq.x; q[m][1] = qq.y;
      k[m][0] = kk.x; k[m][1] = kk.y;
    }
    const float v = sv[buf][u][jl], g = sg[buf][u][0], b = sg[buf][u][1];
    double p0 = 0, p1 = 0;
#pragma unroll
    for (int m = 0; m < NM; m++) {
      s[m][0] = s[m][0] * g;
      s[m][1] = s[m][1] * g;
      p0 = __builtin_fma((double)s[m][0], (double)k[m][0], p0);
      p1 = __builtin_fma((double)s[m][1], (double)k[m][1], p1);
    }
    const float pred = (float)wave_sum(p0 + p1, 32);
    float delta = v - pred;
    delta = delta * b;
    double o0 = 0, o1 = 0;
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const float w0 = k[m][0] * delta, w1 = k[m][1] * delta;
      s[m][0] = s[m][0] + w0;
      s[m][1] = s[m][1] + w1;
      o0 = __builtin_fma((double)s[m][0], (double)q[m][0], o0);
      o1 = __builtin_fma((double)s[m][1], (double)q[m][1], o1);
    }
    return o0 + o1;
  };
  load(0);
  store(0);
  __syncthreads();
  int buf = 0;
  for (int t0 = 0; t0 < a.rows; t0 += CT, buf ^= 1) {
    if (t0 + CT < a.rows) load(t0 + CT);
    const int nt = min(CT, a.rows - t0);
    // the outputs of 8 tokens are summed over the lanes together, off the
    // chain from token to token (rows_sum8: lane bits 0, 1, 2 hold token
    // 4 b0 + 2 b1 + b2, each with wave_sum's bits)
    for (int u0 = 0; u0 < nt; u0 += 8) {
      double o[8];
      if (u0 + 8 <= nt) {
#pragma unroll
        for (int u = 0; u < 8; u++) o[u] = token(buf, u0 + u);
      } else {
#pragma unroll
        for (int u = 0; u < 8; u++) o[u] = u0 + u < nt ? token(buf, u0 + u) : 0.0;
      }
      int u;
      rows_sum8(o, 32, u);
      if (L < 8 && u0 + u < nt && j < a.dv)
        a.y[(int64_t)(t0 + u0 + u) * vdw + (int64_t)head * a.dv + j] = (float)o[0];
    }
    // the other buffer was last read before the barrier that ended the chunk
    // before this one
    if (t0 + CT < a.rows) store(buf ^ 1);
    __syncthreads();
  }
  if (j >= a.dv) return;
#pragma unroll
  for (int m = 0; m < NM; m++)
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const int i = 64 * m + 2 * L + e;
      if (i < a.dk) col[i] = s[m][e];
    }
}
extern "C" __global__ __launch_bounds__(256) void dn_rule_128(DnRuleArgs a) { dn_rule_chunks<2, 16>(a); }
extern "C" __global__ __launch_bounds__(256) void dn_rule_256(DnRuleArgs a) { dn_rule_chunks<4, 8>(a); }

struct DnNormArgs {
  float* x;        // [rows, cols]: the rule's output, normed and gated in place
  const float* w;  // [cols]
  const float* z;  // [rows, cols]: silu(z)
  double eps;
  int32_t rows, cols;
};

// the gated RMSNorm of every value head's output, one wave per row: the
// RMSNorm of TInferCpuBackend.RmsNorm (double sum, x * inv rounded to single
// before the weight), then times silu(z)
extern "C" __global__ __launch_bounds__(256) void dn_gatenorm(DnNormArgs a)
{
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= a.rows) return;
  float* x = a.x + (int64_t)row * a.cols;
  const float* z = a.z + (int64_t)row * a.cols;
  double s = 0;
  for (int c = lane; c < a.cols; c += 64) {
    const double d = x[c];
    s = __builtin_fma(d, d, s);
  }
  s = wave_sum(s, 64);
  const double inv = 1.0 / sqrt(s / (double)a.cols + a.eps);
  for (int c = lane; c < a.cols; c += 64) {
    const float n = (float)((double)x[c] * inv);
    const float y = a.w[c] * n;
    x[c] = y * z[c];
  }
}

struct GateArgs {
  const float* qg;  // split_gate: [rows * heads, 2 * hd]
  float* q;         // split_gate: [rows * heads, hd]; gate_sigmoid: the attention output
  float* g;         // [rows * heads, hd]: the gates
  int64_t n;        // rows * heads * hd
  int32_t hd, pad;
};

// the query projection of a gated attention holds per head its query, then
// its gate: apart into q and g
extern "C" __global__ __launch_bounds__(256) void split_gate(GateArgs a)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  const int64_t r = i / a.hd, c = i - r * a.hd;
  a.q[i] = a.qg[r * 2 * a.hd + c];
  a.g[i] = a.qg[r * 2 * a.hd + a.hd + c];
}

// GateBySigmoid: q[i] *= sigmoid(g[i]), the sigmoid rounded to single first
extern "C" __global__ __launch_bounds__(256) void gate_sigmoid(GateArgs a)
{
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  a.q[i] = a.q[i] * dn_sigmoid(a.g[i]);
}
