// Warm-start network on MI355X (gfx950): the C-ABI of include/fvs2d_mlp.h.
//
// Training step for a batch of M rows (M a multiple of 64), depth L hidden
// layers of width 256:
//   k_forward        cell records -> bfloat16 input rows X0[M][96] (68 used),
//                    then for every hidden layer Z = X W + b, H = GELU(Z),
//                    the activations of a row tile staying in LDS
//   k_head           y = H W + b (float32), loss, dy, dZ of the last hidden
//                    layer, output-layer weight/bias gradient partials
//   k_backward       dZ_prev = (dZ W^T) * GELU'(Z_prev) down to the first
//                    hidden layer, dZ of a row tile staying in LDS
//   k_wgrad          weight-gradient partials X^T dZ (and bias partials)
//   k_adam           sums the partials in a fixed order, Adam update, and
//                    refreshes the bfloat16 copies of the weights
// Prediction is one k_forward launch with the output layer in it.
// The matrix products run on v_mfma_f32_16x16x32_bf16.  The weight gradient
// reduces over the batch rows: each workgroup sums a contiguous slice of rows
// into one of S partial copies, the Adam kernel adds the S copies in slice
// order, so the result does not depend on scheduling (no float atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <exception>
#include <memory>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/fvs2d.h"
#include "../../include/fvs2d_mlp.h"

namespace fvs {
int set_error(int code, const std::string &msg);
}

namespace {

using u16 = unsigned short;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kW = FVS_MLP_WIDTH;
constexpr int kOut = FVS_MLP_OUT;
constexpr int kFeat = FVS_MLP_FEATURES;
constexpr int kRaw = FVS_MLP_RAW;
constexpr int kMaxDepth = 8;
constexpr int kMaxLayers = kMaxDepth + 1;
constexpr int kMaxSplit = 64;
constexpr int kBK = 32;        // reduction depth of one MFMA
constexpr int kSlabs0 = (kFeat + kBK - 1) / kBK;  // slabs of the input layer
constexpr int kIn = kBK * kSlabs0;                // its columns, padded
constexpr int kRows = 64;      // batch rows come in multiples of this

static_assert(kW == 256, "the GEMM tiling assumes width 256");

int fail(int code, const std::string &msg) { return fvs::set_error(code, msg); }
// an exception thrown by host code inside an entry point ends as an error
// code and message, never as a C++ exception crossing into the caller
int host_exception(const char *fn) {
  try {
    throw;
  } catch (const std::bad_alloc &) {
    return fail(FVS_ENOMEM, std::string(fn) + ": host memory exhausted");
  } catch (const std::exception &e) {
    return fail(FVS_ESTATE, std::string(fn) + ": " + e.what());
  } catch (...) {
    return fail(FVS_ESTATE, std::string(fn) + ": host exception");
  }
}

#define MLPC(x)                                                                           \
  do {                                                                                    \
    hipError_t e_ = (x);                                                                  \
    if (e_ != hipSuccess) return fail(FVS_EHIP, std::string(#x ": ") + hipGetErrorString(e_)); \
  } while (0)

// float -> bfloat16, round to nearest even (NaN stays NaN)
__host__ __device__ inline u16 f2bf(float x) {
  unsigned u = __builtin_bit_cast(unsigned, x);
  if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
  u += 0x7fffu + ((u >> 16) & 1u);
  return u16(u >> 16);
}
__host__ __device__ inline float bf2f(u16 h) { return __builtin_bit_cast(float, unsigned(h) << 16); }

// 1 / d for d >= 1, correctly rounded: an approximate reciprocal, one Newton
// step and one correction by the exact remainder (fused multiply-adds).  The
// general division also scales operands that could overflow or vanish, five
// instructions more; the epilogues are bound by vector instructions (91% of the
// issue cycles).  Equal to 1 / d for every float of [1, 2^60); the cap keeps the
// remainder of an infinite d finite.  65,536 rows: forward in training 118 ->
// 106 us, backward 132 -> 121.
__device__ inline float recip(float d) {
  const float c = fminf(d, 0x1p60f);
  const float r0 = __builtin_amdgcn_rcpf(c), r1 = fmaf(fmaf(-c, r0, 1.0f), r0, r0);
  return fmaf(fmaf(-c, r1, 1.0f), r1, r1);
}

// erf by Abramowitz & Stegun 7.1.26 (Hastings' rational approximation,
// |error| <= 1.5e-7): branch-free, so the 64 evaluations per thread of a GEMM
// epilogue do not split the wavefront; far below bfloat16 resolution (3.9e-3)
__device__ inline float erf_as(float x) {
  const float ax = fabsf(x);
  const float t = recip(1.0f + 0.3275911f * ax);
  const float poly = ((((1.061405429f * t - 1.453152027f) * t + 1.421413741f) * t - 0.284496736f) * t +
                      0.254829592f) * t;
  return copysignf(1.0f - poly * __expf(-ax * ax), x);
}
__device__ inline float gelu(float z) { return 0.5f * z * (1.0f + erf_as(z * 0.70710678118654752f)); }
__device__ inline float gelu_grad(float z) {
  return 0.5f * (1.0f + erf_as(z * 0.70710678118654752f)) + z * __expf(-0.5f * z * z) * 0.39894228040143268f;
}

// splitmix64 finaliser (Steele, Lea, Flood 2014): row sampling and weight init
__host__ __device__ inline unsigned long long mix64(unsigned long long z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// ---------------------------------------------------------------- features
// Base angle of the radial (kind 0) or angular (kind 1) harmonics of a cell
// record, and its sine and cosine.
struct Angle {
  double a, s, c;
};
__device__ __forceinline__ Angle base_angle(const float *__restrict__ r, int kind) {
  const double dx = double(r[0]) - 0.5, y = r[1];
  Angle t;
  if (kind == 0) {
    const double kPi = 3.14159265358979323846;
    t.a = kPi * (log1p(4.0 * sqrt(dx * dx + y * y)) / log1p(200.0));
  } else {
    t.a = atan2(y, dx);
  }
  sincos(t.a, &t.s, &t.c);
  return t;
}
// Input columns 8q..8q+7: harmonics 4(q%4)+1..+4 of the radial (q < 4) or
// angular (q < 8) base angle (one sincos of the first, then the angle-addition
// recurrence), q = 8 the four scalar channels.
constexpr int kFeatChunks = (kFeat + 7) / 8;
__device__ __forceinline__ void harmonics(const Angle &t, int q, float f[8]) {
  double sk = t.s, ck = t.c;
  if (q & 3) sincos(double(4 * (q & 3) + 1) * t.a, &sk, &ck);
  for (int h = 0; h < 4; ++h) {
    f[2 * h] = float(sk);
    f[2 * h + 1] = float(ck);
    const double sn = sk * t.c + ck * t.s, cn = ck * t.c - sk * t.s;
    sk = sn;
    ck = cn;
  }
}
__device__ __forceinline__ void scalars(const float *__restrict__ r, float f[8]) {
  f[0] = float(log1p(100.0 * double(r[2])) / log1p(5000.0));
  f[1] = float((double(r[3]) - 0.675) / 0.175);
  f[2] = float((double(r[4]) - 1.0) / 3.0);
  f[3] = float((double(r[5]) - 0.125) / 0.025);
  f[4] = f[5] = f[6] = f[7] = 0.f;
}

// the feature map alone, float32: 256 rows per workgroup, blockIdx.y the columns
__global__ __launch_bounds__(256) void k_features(int n, const float *__restrict__ raw, float *__restrict__ F32) {
  const int m = blockIdx.x * 256 + threadIdx.x, q = blockIdx.y;
  if (m >= n) return;
  const float *r = raw + long(m) * kRaw;
  float f[8];
  if (q < 8) harmonics(base_angle(r, q >> 2), q, f);
  else scalars(r, f);
  for (int c = 0; c < 8; ++c)
    if (8 * q + c < kFeat) F32[long(m) * kFeat + 8 * q + c] = f[c];
}

__device__ __forceinline__ unsigned pack2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// Sum over the 32 lanes of a half wavefront, the same in each: pairs 16 lanes
// apart, then 8, 4, 2 and 1.  From 8 on by row rotation in the vector unit
// instead of five trips through LDS: what a lane gets from the lane n further
// on is what it would get from its partner, because the sums of the steps
// before repeat every 2n lanes.
__device__ __forceinline__ float row_sum(float y) {
  y += __shfl_xor(y, 16, 64);
  auto ror = [](float x, auto ctl) __attribute__((always_inline)) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), decltype(ctl)::value, 0xf, 0xf, true));
  };
  y += ror(y, std::integral_constant<int, 0x128>());
  y += ror(y, std::integral_constant<int, 0x124>());
  y += ror(y, std::integral_constant<int, 0x122>());
  y += ror(y, std::integral_constant<int, 0x121>());
  return y;
}

// ------------------------------------------------------ forward / backward
// One launch for all layers: as one product per layer, 65,536 rows took 5 x 45
// us forward in training (Z, H written, H read back) and prediction 397 us a
// call; in this form 118 us forward, 132 us backward, and 246 us a call.
// A workgroup owns TR rows and all 256 columns of every layer: the rows' activations stay in LDS from layer to layer, and only what the
// weight gradient reads is written to HBM.  Each wavefront holds the results of
// its columns; its weights are not shared with the other wavefronts, so they go
// from L2 to registers without LDS, in the order the MFMA operand wants them
// (pack_at): one contiguous KB per load.
constexpr int kActLd = kW + 8;  // LDS row (elements): 16-byte accesses of 16 rows meet distinct banks

// Element of the packed copy of B[n][k]: per slab of 32 k and 64 columns of a
// wavefront four operand blocks of 16 columns x 32 k.  Row t of block j is
// column 32 (j / 2) + 8 (t / 4) + 4 (j % 2) + t % 4, so that a lane's results
// of blocks 2h and 2h + 1 are eight consecutive columns: activations leave as
// 16-byte vectors, four lanes to a 64-byte segment.
__host__ __device__ inline int pack_at(int n, int k) {
  const int c = n & 31, t = 4 * (c >> 3) + (c & 3), j = 2 * ((n >> 5) & 1) + ((c >> 2) & 1);
  return ((((k >> 5) * 4 + (n >> 6)) * 4 + j) * 64 + t + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

// Tile of a workgroup: TR rows, NJ operand blocks (16 NJ columns) for each of
// its 16 / NJ wavefronts, D slabs of weights in registers or in flight.  W:
// wavefronts per SIMD that the registers allow (4 (TR / 16) NJ accumulators,
// 4 D NJ weights).
template <int TR_, int NJ_, int D_, int W_>
struct Tile {
  static constexpr int TR = TR_, NJ = NJ_, D = D_, W = W_, NT = 1024 / NJ_, NR = TR_ / 16;
  static_assert(NJ == 4 || NJ == 2, "results leave as pairs of blocks");
};

// acc = rows of act (TR x 32 ns) times a wavefront's columns, slab after slab
// (Wp: the lane's place in the packed weights); the caller has loaded the first D
// slabs of b.
template <int NJ>
__device__ __forceinline__ void load_slab(const u16 *__restrict__ Wp, int s, bf16x8 (&b)[NJ]) {
#pragma unroll
  for (int j = 0; j < NJ; ++j) b[j] = *reinterpret_cast<const bf16x8 *>(Wp + (s * 16 + j) * 512);
}
template <class TL>
__device__ __forceinline__ void chain_layer(const u16 *__restrict__ act, const u16 *__restrict__ Wp, int ns, int lane,
                                            bf16x8 (&b)[TL::D][TL::NJ], f32x4 (&acc)[TL::NR][TL::NJ]) {
  const u16 *ap = act + (lane & 15) * kActLd + 8 * (lane >> 4);
#pragma unroll
  for (int i = 0; i < TL::NR; ++i)
#pragma unroll
    for (int j = 0; j < TL::NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < ns; s0 += TL::D) {
#pragma unroll
    for (int u = 0; u < TL::D; ++u) {
      const int s = s0 + u;
      if (s < ns) {
#pragma unroll
        for (int i = 0; i < TL::NR; ++i) {
          const bf16x8 a = *reinterpret_cast<const bf16x8 *>(ap + 16 * i * kActLd + kBK * s);
#pragma unroll
          for (int j = 0; j < TL::NJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[u][j], a, acc[i][j], 0, 0, 0);
        }
        if (s + TL::D < ns) load_slab<TL::NJ>(Wp, s + TL::D, b[u]);
      }
    }
  }
}

// the rows of a pass: records (and targets) given by the caller, rows from
// nvalid on zero, or with ndata > 0 drawn from a set of that many: row m takes
// record hash(seed, step, m) mod ndata
struct Rows {
  const float *raw, *tgt;
  long nvalid, ndata;
  unsigned long long seed;
  long step;
};
__device__ __forceinline__ long row_source(const Rows &R, long m) {
  if (R.ndata > 0)
    return long(mix64(R.seed ^ mix64((unsigned long long)R.step * 0x100000001ull + (unsigned long long)m)) %
                (unsigned long long)R.ndata);
  return m < R.nvalid ? m : -1;
}

// dW = A^T D reduces over the rows of the batch, so its operands want eight
// rows of one column in a lane.  The forward and backward kernels write them
// that way from LDS (pack_rows): per 32 rows and 16 columns one KB, lane by
// lane, 16 bytes each; nothing is transposed here.
__device__ __forceinline__ void pack_rows(const u16 *__restrict__ act, int rows, int cblocks, u16 *__restrict__ out,
                                          int lane, int wv, int waves) {
  const u16 *src = act + 8 * (lane >> 4) * kActLd + (lane & 15);
  for (int q = wv; q < rows / kBK * cblocks; q += waves) {
    const u16 *p = src + (q / cblocks) * kBK * kActLd + 16 * (q % cblocks);
    unsigned v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = unsigned(p[2 * e * kActLd]) | unsigned(p[(2 * e + 1) * kActLd]) << 16;
    *reinterpret_cast<uint4 *>(out + (long(q) * 64 + lane) * 8) = make_uint4(v[0], v[1], v[2], v[3]);
  }
}

struct Chain {
  int L;
  long M;
  const u16 *W[kMaxDepth];     // packed weights
  const float *bias[kMaxDepth];
  u16 *X0, *Z[kMaxDepth], *H[kMaxDepth];
  const float *Wh, *bh;        // output layer
  float *T, *Y;
};

// Features and all hidden layers of TR rows.  TRAIN: X0, Z, H and the targets
// go to HBM (X0 and H in the weight gradient's order, the last H by rows for
// k_head); otherwise only the network's output does.
template <class TL, bool TRAIN>
__global__ __launch_bounds__(TL::NT, TL::W) void k_forward(Chain c, Rows R) {
  constexpr int TR = TL::TR, NJ = TL::NJ, D = TL::D, NT = TL::NT;
  __shared__ __attribute__((aligned(16))) u16 act[TR * kActLd];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long r0 = long(blockIdx.x) * TR;
  const int lp = (wv * NJ * 64 + lane) * 8;  // the lane's place in a slab of packed weights
  bf16x8 b[D][NJ];
#pragma unroll
  for (int u = 0; u < D; ++u)
    if (u < kSlabs0) load_slab<NJ>(c.W[0] + lp, u, b[u]);
  // Consecutive lanes take the same columns of consecutive rows: a wavefront
  // evaluates one kind of feature (the kinds differ in their functions).  The
  // base angles are formed once per row and wait behind the row's input columns.
  auto angle = [&](int row, int kind) __attribute__((always_inline)) -> Angle & {
    return *reinterpret_cast<Angle *>(act + row * kActLd + kBK * kSlabs0 + kind * int(sizeof(Angle) / sizeof(u16)));
  };
  static_assert(kBK * kSlabs0 * sizeof(u16) + 2 * sizeof(Angle) <= kActLd * sizeof(u16), "room for the angles");
  for (int e = tid; e < 2 * TR; e += NT) {
    const int row = e % TR, kind = e / TR;
    const long m = r0 + row, src = m < c.M ? row_source(R, m) : -1;
    if (src >= 0) angle(row, kind) = base_angle(R.raw + src * kRaw, kind);
  }
  __syncthreads();
  for (int e = tid; e < TR * (4 * kSlabs0); e += NT) {
    const int row = e % TR, q = e / TR;
    const long m = r0 + row;
    const long src = m < c.M ? row_source(R, m) : -1;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (q < kFeatChunks && src >= 0) {
      float f[8];
      if (q < 8) harmonics(angle(row, q >> 2), q, f);
      else scalars(R.raw + src * kRaw, f);
      v = make_uint4(pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]), pack2(f[6], f[7]));
    }
    *reinterpret_cast<uint4 *>(act + row * kActLd + 8 * q) = v;
    if (TRAIN && q == 0 && m < c.M)
      *reinterpret_cast<float4 *>(c.T + m * kOut) =
          src >= 0 ? *reinterpret_cast<const float4 *>(R.tgt + src * kOut) : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  __syncthreads();
  const int rows = int(c.M - r0 < TR ? c.M - r0 : TR);
  if (TRAIN) pack_rows(act, rows, 2 * kSlabs0, c.X0 + r0 * kIn, lane, wv, NT / 64);
  f32x4 acc[TL::NR][NJ];
  for (int l = 0; l < c.L; ++l) {
    chain_layer<TL>(act, c.W[l] + lp, l == 0 ? kSlabs0 : kW / kBK, lane, b, acc);
    if (l + 1 < c.L)
#pragma unroll
      for (int u = 0; u < D; ++u) load_slab<NJ>(c.W[l + 1] + lp, u, b[u]);
    const int n0 = 16 * NJ * wv + 8 * (lane >> 4);
    float bv[NJ / 2][8];
#pragma unroll
    for (int h = 0; h < NJ / 2; ++h)
#pragma unroll
      for (int e = 0; e < 8; ++e) bv[h][e] = c.bias[l][n0 + 32 * h + e];
    __syncthreads();  // every wavefront has read the layer's input
#pragma unroll
    for (int i = 0; i < TL::NR; ++i) {
      const int row = 16 * i + (lane & 15);
#pragma unroll
      for (int h = 0; h < NJ / 2; ++h) {
        float z[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) z[e] = acc[i][2 * h + (e >> 2)][e & 3] + bv[h][e];
        const uint4 hv = make_uint4(pack2(gelu(z[0]), gelu(z[1])), pack2(gelu(z[2]), gelu(z[3])),
                                    pack2(gelu(z[4]), gelu(z[5])), pack2(gelu(z[6]), gelu(z[7])));
        *reinterpret_cast<uint4 *>(act + row * kActLd + n0 + 32 * h) = hv;
        if (TRAIN && r0 + 16 * i < c.M) {
          const long idx = (r0 + row) * kW + n0 + 32 * h;
          *reinterpret_cast<uint4 *>(c.Z[l] + idx) =
              make_uint4(pack2(z[0], z[1]), pack2(z[2], z[3]), pack2(z[4], z[5]), pack2(z[6], z[7]));
          if (l + 1 == c.L) *reinterpret_cast<uint4 *>(c.H[l] + idx) = hv;
        }
      }
    }
    __syncthreads();
    if (TRAIN && l + 1 < c.L) pack_rows(act, rows, kW / 16, c.H[l] + r0 * kW, lane, wv, NT / 64);
  }
  if (!TRAIN) {
    // the output layer, 32 lanes per row as in k_head
    const int q = tid & 31, rs = tid >> 5;
    float w[8][kOut];
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int o = 0; o < kOut; ++o) w[e][o] = c.Wh[(8 * q + e) * kOut + o];
    for (int row = rs; row < TR; row += NT / 32) {
      const uint4 hv = *reinterpret_cast<const uint4 *>(act + row * kActLd + 8 * q);
      const unsigned hw[4] = {hv.x, hv.y, hv.z, hv.w};
      float y[kOut] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float h = bf2f(u16((hw[e >> 1] >> (16 * (e & 1))) & 0xffffu));
#pragma unroll
        for (int o = 0; o < kOut; ++o) y[o] += h * w[e][o];
      }
#pragma unroll
      for (int o = 0; o < kOut; ++o) y[o] = row_sum(y[o]);
      if (q == 0 && r0 + row < R.nvalid)
        *reinterpret_cast<float4 *>(c.Y + (r0 + row) * kOut) =
            make_float4(y[0] + c.bh[0], y[1] + c.bh[1], y[2] + c.bh[2], y[3] + c.bh[3]);
    }
  }
}

// dZ of the hidden layers below the last, each in the place of its layer's Z
// (c.W: the backward operands; Z of the last layer holds its dZ by rows), all of
// them left in the weight gradient's order
template <class TL>
__global__ __launch_bounds__(TL::NT, TL::W) void k_backward(Chain c) {
  constexpr int TR = TL::TR, NJ = TL::NJ, D = TL::D, NT = TL::NT;
  __shared__ __attribute__((aligned(16))) u16 act[TR * kActLd];
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long r0 = long(blockIdx.x) * TR;
  const int lp = (wv * NJ * 64 + lane) * 8;
  bf16x8 b[D][NJ];
  if (c.L > 1)
#pragma unroll
    for (int u = 0; u < D; ++u) load_slab<NJ>(c.W[c.L - 1] + lp, u, b[u]);
  const u16 *top = c.Z[c.L - 1];
  for (int e = tid; e < TR * (kW / 8); e += NT) {
    const int row = e / (kW / 8), q = e % (kW / 8);
    *reinterpret_cast<uint4 *>(act + row * kActLd + 8 * q) =
        r0 + row < c.M ? *reinterpret_cast<const uint4 *>(top + (r0 + row) * kW + 8 * q) : make_uint4(0, 0, 0, 0);
  }
  __syncthreads();
  const int rows = int(c.M - r0 < TR ? c.M - r0 : TR);
  pack_rows(act, rows, kW / 16, c.Z[c.L - 1] + r0 * kW, lane, wv, NT / 64);
  f32x4 acc[TL::NR][NJ];
  for (int l = c.L - 1; l > 0; --l) {
    chain_layer<TL>(act, c.W[l] + lp, kW / kBK, lane, b, acc);
    if (l > 1)
#pragma unroll
      for (int u = 0; u < D; ++u) load_slab<NJ>(c.W[l - 1] + lp, u, b[u]);
    const int n0 = 16 * NJ * wv + 8 * (lane >> 4);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TL::NR; ++i) {
      const int row = 16 * i + (lane & 15);
      __builtin_amdgcn_sched_barrier(0);  // Z of few rows at a time in registers
#pragma unroll
      for (int h = 0; h < NJ / 2; ++h) {
        uint4 dv = make_uint4(0, 0, 0, 0);
        if (r0 + 16 * i < c.M) {
          const uint4 zv = *reinterpret_cast<const uint4 *>(c.Z[l - 1] + (r0 + row) * kW + n0 + 32 * h);
          const unsigned zw[4] = {zv.x, zv.y, zv.z, zv.w};
          float d[8];
#pragma unroll
          for (int e = 0; e < 8; ++e)
            d[e] = acc[i][2 * h + (e >> 2)][e & 3] * gelu_grad(bf2f(u16((zw[e >> 1] >> (16 * (e & 1))) & 0xffffu)));
          dv = make_uint4(pack2(d[0], d[1]), pack2(d[2], d[3]), pack2(d[4], d[5]), pack2(d[6], d[7]));
        }
        *reinterpret_cast<uint4 *>(act + row * kActLd + n0 + 32 * h) = dv;
      }
    }
    __syncthreads();  // all of Z is read, all of dZ in LDS
    pack_rows(act, rows, kW / 16, c.Z[l - 1] + r0 * kW, lane, wv, NT / 64);
  }
}

// ------------------------------------------------------------ weight gradient
// Row slices whose partials are kept apart (added by k_adam in their order): S
// slices of cs slabs of 32 rows; a slice's slabs are summed in ng interleaved
// groups, ((g0 + g1) + g2) + g3 with ng = 4.
struct WGrad {
  int L, S, cs, ng;
  const u16 *A[kMaxDepth], *D[kMaxDepth];
  long offW[kMaxDepth], offb[kMaxDepth], P;
  float *G;
};
constexpr int kWgThreads = 512;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(1))) const u32x4 *GlobalIn;

// Partials of dW[k][n] for 16 NB inputs k, all 256 columns n and the slabs of a
// slice, group after group.  A slab is 16 (NB + 16) KB of packed operands, read
// into two LDS buffers (every fragment is a contiguous KB) with two more slabs
// in registers on their way: the matrix cores need a quarter of the time that
// these bytes take from HBM.  Wavefront (wk, wn) holds 8 NB x 64 results of the
// group and as many of the groups before.  With Gb the first 256 threads also
// sum a column of D each (the bias gradient).  All layers of 65,536 rows: 94 us;
// as a launch per layer that transposed row-major operands into LDS, 64 inputs a
// workgroup, 185 us.
template <int NB>
__device__ __forceinline__ void wgrad_tile(const u16 *A, int astride, const u16 *D, int s0, int cs, int ng, int Kreal,
                                           float *__restrict__ GW, float *__restrict__ Gb, u16 *__restrict__ lds) {
  constexpr int NI = NB / 2, kSlab = (NB + 16) * 512;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), wk = wv >> 2, wn = wv & 3;
  const bool own_a = tid < 64 * NB;  // A's 16-byte pieces of a slab; D's are two per thread
  const GlobalIn Ap = (GlobalIn)A + (own_a ? tid : 0), Dp = (GlobalIn)D + tid;
  int at = s0, g = 0;  // the next slab to load (past the end: the last one again)
  auto load = [&](u32x4 &a, u32x4 &d0, u32x4 &d1) __attribute__((always_inline)) {
    a = Ap[long(at) * astride];
    d0 = Dp[long(at) * 1024];
    d1 = Dp[long(at) * 1024 + 512];
    if (at + ng < s0 + cs) at += ng;
    else if (g + 1 < ng) at = s0 + ++g;
  };
  auto store = [&](int buf, u32x4 a, u32x4 d0, u32x4 d1) __attribute__((always_inline)) {
    u32x4 *p = reinterpret_cast<u32x4 *>(lds + buf * kSlab) + tid;
    if (own_a) p[0] = a;
    p[64 * NB] = d0;
    p[64 * NB + 512] = d1;
  };
  f32x4 acc[NI][4], sum[NI][4];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float db = 0.f, dbs = 0.f;
  const int per = cs / ng;
  int left = per;  // slabs of the group still to add
  auto multiply = [&](const u16 *buf) __attribute__((always_inline)) {
    const u16 *As = buf + wk * NI * 512 + lane * 8, *Ds = buf + (NB + 4 * wn) * 512 + lane * 8;
    bf16x8 b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf16x8 *>(Ds + j * 512);
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const bf16x8 a = *reinterpret_cast<const bf16x8 *>(As + i * 512);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a, acc[i][j], 0, 0, 0);
    }
    if (Gb && tid < kW) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint4 v = *reinterpret_cast<const uint4 *>(buf + (NB + (tid >> 4)) * 512 + ((tid & 15) + 16 * q) * 8);
        const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) db += bf2f(u16((w[e >> 1] >> (16 * (e & 1))) & 0xffffu));
      }
    }
    if (--left == 0) {
      left = per;
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sum[i][j] = sum[i][j] + acc[i][j];
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
      dbs += db;
      db = 0.f;
    }
  };
  u32x4 x0, x1, x2, y0, y1, y2;
  load(x0, x1, x2);
  load(y0, y1, y2);
  store(0, x0, x1, x2);
  load(x0, x1, x2);
  for (int t = 0; t < cs; t += 2) {
    __syncthreads();  // slab t is in buffer 0, and buffer 1 has been read
    store(1, y0, y1, y2);
    load(y0, y1, y2);
    multiply(lds);
    if (t + 1 == cs) break;
    __syncthreads();
    store(0, x0, x1, x2);
    load(x0, x1, x2);
    multiply(lds + kSlab);
  }
  // lane l holds dW[16i + l%16][16j + 4(l/16)..+3]
  const int n0 = 64 * wn + 4 * (lane >> 4);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = 16 * (wk * NI + i) + (lane & 15);
    if (k >= Kreal) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<f32x4 *>(GW + long(k) * kW + n0 + 16 * j) = sum[i][j];
  }
  if (Gb && tid < kW) Gb[tid] = dbs;
}

// Workgroups: per slice two 128-input tiles of each layer from the last to the
// second, then the input layer's one tile.  The two tiles of a layer read the
// same D; with the slices in eights they go to one XCD (workgroups are handed to
// the eight XCDs in turn), whose L2 serves the second.
__global__ __launch_bounds__(kWgThreads, 2) void k_wgrad(WGrad g) {
  __shared__ __attribute__((aligned(16))) u16 lds[2 * 24 * 512];
  const int hidden = 2 * (g.L - 1) * g.S;
  int w = blockIdx.x;
  if (w >= hidden) {
    w -= hidden;
    wgrad_tile<2 * kSlabs0>(g.A[0], 128 * kSlabs0, g.D[0], w * g.cs, g.cs, g.ng, kFeat, g.G + long(w) * g.P + g.offW[0],
                            g.G + long(w) * g.P + g.offb[0], lds);
    return;
  }
  const int l = g.L - 1 - w / (2 * g.S);
  w %= 2 * g.S;
  const int s = g.S % 8 == 0 ? (w >> 4) * 8 + (w & 7) : w >> 1, kt = g.S % 8 == 0 ? (w >> 3) & 1 : w & 1;
  float *Gs = g.G + long(s) * g.P;
  wgrad_tile<8>(g.A[l] + kt * 8 * 512, 1024, g.D[l], s * g.cs, g.cs, g.ng, 128, Gs + g.offW[l] + kt * 128L * kW,
                kt == 0 ? Gs + g.offb[l] : nullptr, lds);
}

// largest divisor of M/32 that is at most kMaxSplit: row slices of the
// gradient reduction, each a multiple of 32 rows
int nsplit(int M) {
  const int u = M / kBK;
  for (int s = std::min(u, kMaxSplit); s >= 1; --s)
    if (u % s == 0) return s;
  return 1;
}

// ------------------------------------------------------------ output layer
constexpr int kHeadRows = 128;                 // rows per workgroup
constexpr int kHeadPart = kW * kOut + kOut;    // output-layer parameters

// Workgroup b handles rows [128b, min(128b + 128, M)), 64 or 128: y = H Wh + bh in
// float32, dy = 2 (y - t) / (nvalid * 4) for rows < nvalid (0 otherwise), the
// last hidden layer's dZ = bf16((dy Wh^T) * GELU'(Z)) in the place of Z, and this
// workgroup's partial gradients of Wh and bh (Gh[b][...]) and loss sum (lossp[b]).
// First 32 rows at a time with 32 lanes per row and 8 hidden columns per lane,
// dy to LDS; then the sums over the rows, a quarter of the threads per output,
// rows rs, rs + 8, ... in a thread.  (Both in one pass, 8 rows at a time: 4,096
// rows 30 -> 19 us, 65,536 rows 48 -> 44; bound by vector instructions.)
constexpr int kHeadThreads = 1024;
// a + b with b as it was rounded: not fused with the product it comes from
__device__ __forceinline__ float add_rounded(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}
__global__ __launch_bounds__(kHeadThreads, 4) void k_head(long M, long nvalid, float inv_no, const u16 *__restrict__ H,
                                                       u16 *Z, const float *__restrict__ Wh,
                                                       const float *__restrict__ bh, const float *__restrict__ T,
                                                       float *__restrict__ Gh, float *__restrict__ lossp) {
  __shared__ float red[4][32][8 * kOut + kOut + 1];
  __shared__ __attribute__((aligned(16))) float res[kHeadRows][kOut];  // y - t
  const int tid = threadIdx.x, q = tid & 31, lane = tid & 63, wv = (tid >> 6) & 3;
  const long mbeg = long(blockIdx.x) * kHeadRows;
  const int rows = int(M - mbeg < kHeadRows ? M - mbeg : kHeadRows);
  {
    float w[8][kOut], bo[kOut];
    for (int c = 0; c < 8; ++c)
      for (int o = 0; o < kOut; ++o) w[c][o] = Wh[(8 * q + c) * kOut + o];
    for (int o = 0; o < kOut; ++o) bo[o] = bh[o];
    for (int r0 = 0; r0 < rows; r0 += 64) {  // two rows per thread, their loads together
      uint4 h2[2], z2[2];
      float4 t2[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const long m = mbeg + r0 + 32 * u + (tid >> 5);
        h2[u] = *reinterpret_cast<const uint4 *>(H + m * kW + 8 * q);
        z2[u] = *reinterpret_cast<const uint4 *>(Z + m * kW + 8 * q);
        t2[u] = *reinterpret_cast<const float4 *>(T + m * kOut);
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int r = r0 + 32 * u + (tid >> 5);
        const long m = mbeg + r;
        const uint4 hv = h2[u], zv = z2[u];
        const float4 t4 = t2[u];
        const float tv[kOut] = {t4.x, t4.y, t4.z, t4.w};
        const unsigned hw[4] = {hv.x, hv.y, hv.z, hv.w};
        float dy[kOut];
        for (int o = 0; o < kOut; ++o) {
          float t = 0.f;
          for (int c = 0; c < 8; ++c) t += bf2f(u16((hw[c >> 1] >> (16 * (c & 1))) & 0xffffu)) * w[c][o];
          const float y = row_sum(t) + bo[o];
          const float d = m < nvalid ? y - tv[o] : 0.f;
          dy[o] = 2.f * d * inv_no;
          if (q == 0) res[r][o] = d;
        }
        const unsigned zw[4] = {zv.x, zv.y, zv.z, zv.w};
        unsigned pk[4] = {0, 0, 0, 0};
        for (int c = 0; c < 8; ++c) {
          float g = 0.f;
          for (int o = 0; o < kOut; ++o) g += dy[o] * w[c][o];
          const float z = bf2f(u16((zw[c >> 1] >> (16 * (c & 1))) & 0xffffu));
          pk[c >> 1] |= unsigned(f2bf(g * gelu_grad(z))) << (16 * (c & 1));
        }
        *reinterpret_cast<uint4 *>(Z + m * kW + 8 * q) = make_uint4(pk[0], pk[1], pk[2], pk[3]);
      }
    }
  }
  __syncthreads();
  const int rs = (tid >> 5) & 7, o = tid >> 8;
  float gw[8] = {0, 0, 0, 0, 0, 0, 0, 0}, gb = 0.f, ls = 0.f;
  for (int r0 = rs; r0 < rows; r0 += 64) {
    uint4 h8[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) h8[u] = *reinterpret_cast<const uint4 *>(H + (mbeg + r0 + 8 * u) * kW + 8 * q);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float *d = res[r0 + 8 * u];
      const unsigned hw[4] = {h8[u].x, h8[u].y, h8[u].z, h8[u].w};
      const float dy = 2.f * d[o] * inv_no;
      for (int c = 0; c < 8; ++c) gw[c] += bf2f(u16((hw[c >> 1] >> (16 * (c & 1))) & 0xffffu)) * dy;
      gb = add_rounded(gb, dy);
      if (o == 0)
        for (int e = 0; e < kOut; ++e) ls += d[e] * d[e];
    }
  }
  // rows rs and rs^1 share a wavefront: add the two halves, then the 4 row groups
  for (int c = 0; c < 8; ++c) gw[c] += __shfl_xor(gw[c], 32, 64);
  gb += __shfl_xor(gb, 32, 64);
  ls += __shfl_xor(ls, 32, 64);
  if (lane < 32) {
    for (int c = 0; c < 8; ++c) red[wv][q][c * kOut + o] = gw[c];
    red[wv][q][8 * kOut + o] = gb;
    if (o == 0) red[wv][q][8 * kOut + kOut] = ls;
  }
  __syncthreads();
  float *Gb = Gh + long(blockIdx.x) * kHeadPart;
  auto total = [&](int qq, int e) { return red[0][qq][e] + red[1][qq][e] + red[2][qq][e] + red[3][qq][e]; };
  Gb[tid] = total(tid / (8 * kOut), tid % (8 * kOut));  // columns 8 qq + c, outputs o: tid = 32 qq + 4 c + o
  if (tid < kOut) Gb[kW * kOut + tid] = total(0, 8 * kOut + tid);
  if (tid == 0) lossp[blockIdx.x] = total(0, 8 * kOut + kOut);
}
static_assert(kHeadThreads == kW * kOut, "one weight of the output layer per thread");

// Output-layer gradient: column c of the nhb partial rows, summed by 16
// groups of rows (group g takes rows g, g+16, ...) and then the 16 group
// sums in a fixed tree; the order does not depend on scheduling.
__global__ __launch_bounds__(256) void k_head_reduce(int nhb, const float *__restrict__ Gh, float *__restrict__ gh) {
  __shared__ float red[16][16];
  const int t = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int c = blockIdx.x * 16 + t;
  float s = 0.f;
  if (c < kHeadPart)
    for (int b0 = g; b0 < nhb; b0 += 128) {  // eight loads in flight
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = b0 + 16 * u < nhb ? Gh[long(b0 + 16 * u) * kHeadPart + c] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
  red[g][t] = s;
  __syncthreads();
  for (int h = 8; h >= 1; h >>= 1) {
    if (g < h) red[g][t] += red[g + h][t];
    __syncthreads();
  }
  if (g == 0 && c < kHeadPart) gh[c] = red[0][t];
}

// --------------------------------------------------------------- optimiser
struct LayerTab {
  long offW[kMaxLayers], offb[kMaxLayers];
  int in[kMaxLayers], out[kMaxLayers];
  u16 *Wt[kMaxLayers];  // packed copies (pack_at): forward operand, reduction over the inputs
  u16 *Wk[kMaxLayers];  // backward-data operand, reduction over the outputs
  int nl;
};

// mode 0: publish the bfloat16 copies only; 1: sum partials into gout;
// 2: sum partials, Adam update, publish.  Hidden-layer gradients come as
// nsplit slices of G, added in slice order; the output layer's (parameters
// from offHead on) already reduced in gh.  Workgroup 0 also reduces the nhb
// loss partials into the step's loss (lossh may be null).
__global__ __launch_bounds__(256) void k_adam(long P, int nsplit, int mode, const float *__restrict__ G,
                                              const float *__restrict__ gh, int nhb, long offHead,
                                              float *__restrict__ w, float *__restrict__ m1,
                                              float *__restrict__ m2, float lr, float b1, float b2, float eps,
                                              float bc1, float bc2, LayerTab tab, float *__restrict__ gout,
                                              const float *__restrict__ lossp, double inv_no,
                                              double *__restrict__ lossh) {
  __shared__ double lred[256];
  const long p = long(blockIdx.x) * 256 + threadIdx.x;
  if (blockIdx.x == 0 && lossh && mode != 0) {
    double s = 0.0;
    for (int k = threadIdx.x; k < nhb; k += 256) s += double(lossp[k]);
    lred[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h >= 1; h >>= 1) {
      if (int(threadIdx.x) < h) lred[threadIdx.x] += lred[threadIdx.x + h];
      __syncthreads();
    }
    if (threadIdx.x == 0) *lossh = lred[0] * inv_no;
  }
  if (p >= P) return;
  if (mode != 0) {
    float g = 0.f;
    if (p >= offHead) {
      g = gh[p - offHead];
    } else {
      // the slices' partials in flight 16 at a time, summed in slice order
      for (int k = 0; k < nsplit; k += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = k + u < nsplit ? G[long(k + u) * P + p] : 0.f;
#pragma unroll
        for (int u = 0; u < 16; ++u) g += v[u];
      }
    }
    if (gout) gout[p] = g;
    if (mode == 2) {
      const float a = b1 * m1[p] + (1.f - b1) * g;
      const float b = b2 * m2[p] + (1.f - b2) * g * g;
      m1[p] = a;
      m2[p] = b;
      w[p] -= lr * (a / bc1) / (sqrtf(b / bc2) + eps);
    }
  }
  if (mode == 1) return;
  for (int l = 0; l < tab.nl; ++l) {
    if (p >= tab.offW[l] && p < tab.offb[l]) {
      const long e = p - tab.offW[l];
      const int k = int(e / tab.out[l]), n = int(e % tab.out[l]);
      const u16 v = f2bf(w[p]);
      if (tab.Wt[l]) tab.Wt[l][pack_at(n, k)] = v;
      if (tab.Wk[l]) tab.Wk[l][pack_at(k, n)] = v;
    }
  }
}

}  // namespace

// ------------------------------------------------------------------ context
struct fvs_mlp {
  fvs_mlp_options opt{};
  int L = 0;   // hidden layers
  int M = 0;   // batch rows
  long P = 0;  // parameters
  LayerTab tab{};
  hipStream_t stream = nullptr;
  float *w = nullptr, *m1 = nullptr, *m2 = nullptr, *G = nullptr, *Gh = nullptr, *gh = nullptr,
        *lossp = nullptr, *gtmp = nullptr;
  double *lossh = nullptr;
  u16 *X0 = nullptr;
  u16 *Z[kMaxDepth] = {}, *H[kMaxDepth] = {};  // the backward pass leaves dZ in Z
  float *T = nullptr, *Y = nullptr, *F32 = nullptr;
  float *raw = nullptr, *tgt = nullptr;  // training set
  long ndata = 0;
  float *iraw = nullptr, *itgt = nullptr;  // staging of caller rows (batch rows)
  long t = 0;                              // Adam step count
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  float last_ms = 0.f;
  std::vector<void *> allocs;
  // per-launch timing
  bool profiling = false;
  std::vector<hipEvent_t> evpool;
  std::vector<int> evclass;
  int evused = 0;

  template <class T_>
  int alloc(T_ *&p, size_t n) {
    void *q = nullptr;
    MLPC(hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T_)));
    allocs.push_back(q);
    p = static_cast<T_ *>(q);
    return 0;
  }
  ~fvs_mlp() {
    for (void *q : allocs) (void)hipFree(q);
    for (hipEvent_t e : evpool) (void)hipEventDestroy(e);
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

// MC_FEAT: part of MC_FWD
enum { MC_FEAT, MC_FWD, MC_HEAD, MC_WGRAD, MC_BWD, MC_ADAM, MC_N };

struct Prof {
  fvs_mlp &m;
  bool on;
  Prof(fvs_mlp &mm, int cls) : m(mm), on(mm.profiling && mm.evused + 2 <= int(mm.evpool.size())) {
    if (!on) return;
    (void)hipEventRecord(m.evpool[m.evused], m.stream);
    m.evclass.push_back(cls);
  }
  ~Prof() {
    if (!on) return;
    (void)hipEventRecord(m.evpool[m.evused + 1], m.stream);
    m.evused += 2;
  }
};

// f(tile): the tile of a pass over M rows.  128 rows read the weights least
// often and keep the matrix cores busiest, but need two tiles for each CU (32,768
// rows, 10 training steps: 2728 us in tiles of 128, 2235 in tiles of 64); fewer
// rows go in tiles of 32, each over 8 wavefronts (4,096 rows: 1258 us, over 4
// wavefronts 1334; 16,384 rows: 1602, in tiles of 64 1775).
template <class F>
void with_tile(long M, F f) {
  if (M >= 128 * 512) f(Tile<128, 4, 2, 2>());
  else if (M >= 64 * 512) f(Tile<64, 4, 2, 3>());
  else f(Tile<32, 2, 4, 4>());
}

Chain chain_of(const fvs_mlp &m, long M, u16 *const *W) {
  Chain c{};
  c.L = m.L;
  c.M = M;
  for (int l = 0; l < m.L; ++l) {
    c.W[l] = W[l];
    c.bias[l] = m.w + m.tab.offb[l];
    c.Z[l] = m.Z[l];
    c.H[l] = m.H[l];
  }
  c.X0 = m.X0;
  c.Wh = m.w + m.tab.offW[m.L];
  c.bh = m.w + m.tab.offb[m.L];
  c.T = m.T;
  c.Y = m.Y;
  return c;
}

template <bool TRAIN>
void launch_forward(fvs_mlp &m, int M, const Rows &R) {
  Prof pf(m, MC_FWD);
  const Chain c = chain_of(m, M, m.tab.Wt);
  with_tile(M, [&](auto t) {
    using TL = decltype(t);
    hipLaunchKernelGGL((k_forward<TL, TRAIN>), dim3((M + TL::TR - 1) / TL::TR), dim3(TL::NT), 0, m.stream, c, R);
  });
}

// network output of M rows into Y
int predict_pass(fvs_mlp &m, int M, const Rows &R) {
  launch_forward<false>(m, M, R);
  MLPC(hipGetLastError());
  return 0;
}

// forward and backward over M rows: loss and weight-gradient partials
int train_pass(fvs_mlp &m, int M, const Rows &R) {
  const int L = m.L;
  launch_forward<true>(m, M, R);
  {
    Prof pf(m, MC_HEAD);
    const float inv_no = 1.0f / float(double(R.nvalid) * kOut);
    hipLaunchKernelGGL(k_head, dim3((M + kHeadRows - 1) / kHeadRows), dim3(kHeadThreads), 0, m.stream, long(M), R.nvalid,
                       inv_no, m.H[L - 1], m.Z[L - 1], m.w + m.tab.offW[L], m.w + m.tab.offb[L], m.T, m.Gh, m.lossp);
  }
  {
    Prof pf(m, MC_BWD);
    const Chain c = chain_of(m, M, m.tab.Wk);
    with_tile(M, [&](auto t) {
      using TL = decltype(t);
      hipLaunchKernelGGL((k_backward<TL>), dim3((M + TL::TR - 1) / TL::TR), dim3(TL::NT), 0, m.stream, c);
    });
  }
  {
    Prof pf(m, MC_WGRAD);
    WGrad g{};
    for (int l = 0; l < L; ++l) {
      g.A[l] = l == 0 ? m.X0 : m.H[l - 1];
      g.D[l] = m.Z[l];
      g.offW[l] = m.tab.offW[l];
      g.offb[l] = m.tab.offb[l];
    }
    g.L = L;
    g.S = nsplit(M);
    g.cs = M / kBK / g.S;
    g.ng = g.cs % 4 == 0 ? 4 : 1;
    g.G = m.G;
    g.P = m.P;
    hipLaunchKernelGGL(k_wgrad, dim3((2 * L - 1) * g.S), dim3(kWgThreads), 0, m.stream, g);
  }
  MLPC(hipGetLastError());
  return 0;
}

int launch_adam(fvs_mlp &m, int mode, int S, int nhb, double inv_no, double *lossh, float *gout) {
  Prof pf(m, MC_ADAM);
  if (mode != 0)
    hipLaunchKernelGGL(k_head_reduce, dim3((kHeadPart + 15) / 16), dim3(256), 0, m.stream, nhb, m.Gh, m.gh);
  float bc1 = 1.f, bc2 = 1.f;
  if (mode == 2) {
    m.t += 1;
    bc1 = float(1.0 - std::pow(m.opt.beta1, double(m.t)));
    bc2 = float(1.0 - std::pow(m.opt.beta2, double(m.t)));
  }
  hipLaunchKernelGGL(k_adam, dim3(unsigned((m.P + 255) / 256)), dim3(256), 0, m.stream, m.P, S, mode, m.G, m.gh,
                     nhb, m.tab.offW[m.L], m.w, m.m1, m.m2, float(m.opt.lr), float(m.opt.beta1), float(m.opt.beta2),
                     float(m.opt.eps), bc1, bc2, m.tab, gout, m.lossp, inv_no, lossh);
  MLPC(hipGetLastError());
  return 0;
}

int stage_rows(fvs_mlp &m, int n, const float *raw, const float *target) {
  MLPC(hipMemcpyAsync(m.iraw, raw, size_t(n) * kRaw * sizeof(float), hipMemcpyHostToDevice, m.stream));
  if (target)
    MLPC(hipMemcpyAsync(m.itgt, target, size_t(n) * kOut * sizeof(float), hipMemcpyHostToDevice, m.stream));
  return 0;
}

int round64(long n) { return int((n + kRows - 1) / kRows * kRows); }

}  // namespace

extern "C" {

int fvs_mlp_create(fvs_mlp **out, const fvs_mlp_options *opt) try {
  if (!out || !opt) return fail(FVS_EINVAL, "null argument");
  *out = nullptr;
  if (opt->depth < 1 || opt->depth > kMaxDepth) return fail(FVS_EINVAL, "depth must be 1..8");
  if (opt->batch < kRows || opt->batch % kRows) return fail(FVS_EINVAL, "batch must be a positive multiple of 64");
  if (!(opt->lr > 0) || !(opt->beta1 >= 0 && opt->beta1 < 1) || !(opt->beta2 >= 0 && opt->beta2 < 1) ||
      !(opt->eps > 0))
    return fail(FVS_EINVAL, "Adam parameters out of range");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(FVS_EHIP, "no HIP device");
  std::unique_ptr<fvs_mlp> holder(new fvs_mlp());  // freed on every early return or exception
  fvs_mlp *m = holder.get();
  m->opt = *opt;
  m->L = opt->depth;
  m->M = opt->batch;
  LayerTab &tb = m->tab;
  tb.nl = m->L + 1;
  long off = 0;
  for (int l = 0; l <= m->L; ++l) {
    tb.in[l] = (l == 0) ? kFeat : kW;
    tb.out[l] = (l == m->L) ? kOut : kW;
    tb.offW[l] = off;
    off += long(tb.in[l]) * tb.out[l];
    tb.offb[l] = off;
    off += tb.out[l];
  }
  m->P = off;
  if (hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking) != hipSuccess) return fail(FVS_EHIP, "stream");
  if (hipEventCreate(&m->ev0) != hipSuccess || hipEventCreate(&m->ev1) != hipSuccess)
    return fail(FVS_EHIP, "event");
  const size_t M = size_t(m->M);
  int rc = 0;
  rc = rc ? rc : m->alloc(m->w, m->P);
  rc = rc ? rc : m->alloc(m->m1, m->P);
  rc = rc ? rc : m->alloc(m->m2, m->P);
  rc = rc ? rc : m->alloc(m->gtmp, m->P);
  rc = rc ? rc : m->alloc(m->G, size_t(kMaxSplit) * m->P);
  rc = rc ? rc : m->alloc(m->Gh, (M + kHeadRows - 1) / kHeadRows * kHeadPart);
  rc = rc ? rc : m->alloc(m->gh, kHeadPart);
  rc = rc ? rc : m->alloc(m->lossp, (M + kHeadRows - 1) / kHeadRows);
  rc = rc ? rc : m->alloc(m->lossh, 1);
  rc = rc ? rc : m->alloc(m->X0, M * kIn);
  for (int l = 0; l < m->L && !rc; ++l) {
    rc = m->alloc(m->Z[l], M * kW);
    rc = rc ? rc : m->alloc(m->H[l], M * kW);
  }
  rc = rc ? rc : m->alloc(m->T, M * kOut);
  rc = rc ? rc : m->alloc(m->Y, M * kOut);
  rc = rc ? rc : m->alloc(m->F32, M * kFeat);
  rc = rc ? rc : m->alloc(m->iraw, M * kRaw);
  rc = rc ? rc : m->alloc(m->itgt, M * kOut);
  for (int l = 0; l < m->L && !rc; ++l) {
    rc = m->alloc(tb.Wt[l], size_t(kW) * (l == 0 ? kIn : kW));
    if (!rc && l > 0) rc = m->alloc(tb.Wk[l], size_t(kW) * kW);
  }
  if (rc) return rc;
  tb.Wt[m->L] = tb.Wk[m->L] = nullptr;
  tb.Wk[0] = nullptr;
  // padding input rows of the packed weights
  if (hipMemsetAsync(tb.Wt[0], 0, size_t(kW) * kIn * sizeof(u16), m->stream) != hipSuccess)
    return fail(FVS_EHIP, "memset");
  // Glorot-uniform weights from the seed, zero biases
  std::vector<float> w(m->P, 0.f);
  for (int l = 0; l <= m->L; ++l) {
    const double a = std::sqrt(6.0 / double(tb.in[l] + tb.out[l]));
    for (long e = 0; e < long(tb.in[l]) * tb.out[l]; ++e) {
      const unsigned long long r = mix64(opt->seed * 0x9E3779B97F4A7C15ull + (unsigned long long)(tb.offW[l] + e));
      const double u = double(r >> 11) * (1.0 / 9007199254740992.0);
      w[tb.offW[l] + e] = float((2.0 * u - 1.0) * a);
    }
  }
  rc = fvs_mlp_set_params(m, w.data());
  if (rc) return rc;
  *out = holder.release();
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_create");
}

int fvs_mlp_destroy(fvs_mlp *m) try {
  delete m;
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_destroy");
}

long long fvs_mlp_nparams(const fvs_mlp *m) { return m ? m->P : -1; }

int fvs_mlp_get_params(fvs_mlp *m, float *p) try {
  if (!m || !p) return fail(FVS_EINVAL, "null argument");
  MLPC(hipMemcpyAsync(p, m->w, size_t(m->P) * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  MLPC(hipStreamSynchronize(m->stream));
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_get_params");
}

int fvs_mlp_set_params(fvs_mlp *m, const float *p) try {
  if (!m || !p) return fail(FVS_EINVAL, "null argument");
  MLPC(hipMemcpyAsync(m->w, p, size_t(m->P) * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MLPC(hipMemsetAsync(m->m1, 0, size_t(m->P) * sizeof(float), m->stream));
  MLPC(hipMemsetAsync(m->m2, 0, size_t(m->P) * sizeof(float), m->stream));
  m->t = 0;
  if (int rc = launch_adam(*m, 0, 0, 0, 0.0, nullptr, nullptr)) return rc;
  MLPC(hipStreamSynchronize(m->stream));
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_set_params");
}

int fvs_mlp_features(fvs_mlp *m, int n, const float *raw, float *feat) try {
  if (!m || (n > 0 && (!raw || !feat))) return fail(FVS_EINVAL, "null argument");
  if (n < 0 || n > m->M) return fail(FVS_EINVAL, "n must be 0..batch");
  if (n == 0) return 0;
  if (int rc = stage_rows(*m, n, raw, nullptr)) return rc;
  hipLaunchKernelGGL(k_features, dim3((n + 255) / 256, kFeatChunks), dim3(256), 0, m->stream, n, m->iraw, m->F32);
  MLPC(hipGetLastError());
  MLPC(hipMemcpyAsync(feat, m->F32, size_t(n) * kFeat * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  MLPC(hipStreamSynchronize(m->stream));
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_features");
}

int fvs_mlp_set_data(fvs_mlp *m, long long n, const float *raw, const float *target) try {
  if (!m || !raw || !target) return fail(FVS_EINVAL, "null argument");
  if (n < 1) return fail(FVS_EINVAL, "empty training set");
  if (m->raw) {
    for (void *q : {static_cast<void *>(m->raw), static_cast<void *>(m->tgt)}) {
      (void)hipFree(q);
      m->allocs.erase(std::find(m->allocs.begin(), m->allocs.end(), q));
    }
    m->raw = m->tgt = nullptr;
  }
  if (int rc = m->alloc(m->raw, size_t(n) * kRaw)) return rc;
  if (int rc = m->alloc(m->tgt, size_t(n) * kOut)) return rc;
  MLPC(hipMemcpyAsync(m->raw, raw, size_t(n) * kRaw * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MLPC(hipMemcpyAsync(m->tgt, target, size_t(n) * kOut * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MLPC(hipStreamSynchronize(m->stream));
  m->ndata = long(n);
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_set_data");
}

int fvs_mlp_train(fvs_mlp *m, int steps, double *loss) try {
  if (!m) return fail(FVS_EINVAL, "null argument");
  if (!m->raw) return fail(FVS_ESTATE, "no training set (fvs_mlp_set_data)");
  if (steps < 0) return fail(FVS_EINVAL, "steps < 0");
  if (steps == 0) return 0;
  double *dl = nullptr;
  MLPC(hipMalloc(&dl, size_t(steps) * sizeof(double)));
  const int S = nsplit(m->M);
  const double inv_no = 1.0 / (double(m->M) * kOut);
  int rc = 0;
  if (hipEventRecord(m->ev0, m->stream) != hipSuccess) rc = fail(FVS_EHIP, "event");
  for (int s = 0; s < steps && !rc; ++s) {
    rc = train_pass(*m, m->M, {m->raw, m->tgt, m->M, m->ndata, m->opt.seed, m->t + 1});
    if (!rc) rc = launch_adam(*m, 2, S, (m->M + kHeadRows - 1) / kHeadRows, inv_no, dl + s, nullptr);
  }
  if (!rc) {
    hipError_t e = hipEventRecord(m->ev1, m->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(m->stream);
    if (e == hipSuccess) e = hipEventElapsedTime(&m->last_ms, m->ev0, m->ev1);
    if (e != hipSuccess) rc = fail(FVS_EHIP, std::string("training: ") + hipGetErrorString(e));
  }
  if (!rc && loss && hipMemcpy(loss, dl, size_t(steps) * sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
    rc = fail(FVS_EHIP, "copy of losses");
  (void)hipFree(dl);
  return rc;
} catch (...) {
  return host_exception("fvs_mlp_train");
}

static int grad_or_step(fvs_mlp *m, int n, const float *raw, const float *target, double *loss, float *grad,
                        bool update) {
  if (!m || !raw || !target) return fail(FVS_EINVAL, "null argument");
  if (n < 1 || n > m->M) return fail(FVS_EINVAL, "n must be 1..batch");
  const int M = round64(n);
  const int S = nsplit(M);
  if (int rc = stage_rows(*m, n, raw, target)) return rc;
  if (int rc = train_pass(*m, M, {m->iraw, m->itgt, n, 0, 0, 0})) return rc;
  if (int rc = launch_adam(*m, update ? 2 : 1, S, (M + kHeadRows - 1) / kHeadRows, 1.0 / (double(n) * kOut), m->lossh,
                           update ? nullptr : m->gtmp))
    return rc;
  if (grad) MLPC(hipMemcpyAsync(grad, m->gtmp, size_t(m->P) * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  double l = 0.0;
  MLPC(hipMemcpyAsync(&l, m->lossh, sizeof(double), hipMemcpyDeviceToHost, m->stream));
  MLPC(hipStreamSynchronize(m->stream));
  if (loss) *loss = l;
  return 0;
}

int fvs_mlp_grad(fvs_mlp *m, int n, const float *raw, const float *target, double *loss, float *grad) try {
  return grad_or_step(m, n, raw, target, loss, grad, false);
} catch (...) {
  return host_exception("fvs_mlp_grad");
}

int fvs_mlp_step(fvs_mlp *m, int n, const float *raw, const float *target, double *loss) try {
  return grad_or_step(m, n, raw, target, loss, nullptr, true);
} catch (...) {
  return host_exception("fvs_mlp_step");
}

int fvs_mlp_predict(fvs_mlp *m, long long n, const float *raw, float *out) try {
  if (!m || (n > 0 && (!raw || !out))) return fail(FVS_EINVAL, "null argument");
  if (n < 0) return fail(FVS_EINVAL, "n < 0");
  for (long long b = 0; b < n; b += m->M) {
    const int nb = int(std::min<long long>(m->M, n - b));
    const int M = round64(nb);
    if (int rc = stage_rows(*m, nb, raw + b * kRaw, nullptr)) return rc;
    if (int rc = predict_pass(*m, M, {m->iraw, nullptr, nb, 0, 0, 0})) return rc;
    MLPC(hipMemcpyAsync(out + b * kOut, m->Y, size_t(nb) * kOut * sizeof(float), hipMemcpyDeviceToHost, m->stream));
    MLPC(hipStreamSynchronize(m->stream));
  }
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_predict");
}

int fvs_mlp_kernel_times(fvs_mlp *m, int steps, double *ms6, double *flop6, int *launches6) try {
  if (!m || !ms6 || !flop6 || !launches6) return fail(FVS_EINVAL, "null argument");
  if (!m->raw) return fail(FVS_ESTATE, "no training set (fvs_mlp_set_data)");
  if (steps < 1) return fail(FVS_EINVAL, "steps must be positive");
  const int per_step = 2 * (MC_N - 1);
  const int need = per_step * steps;
  while (int(m->evpool.size()) < need) {
    hipEvent_t e;
    MLPC(hipEventCreate(&e));
    m->evpool.push_back(e);
  }
  m->evused = 0;
  m->evclass.clear();
  m->profiling = true;
  int rc = fvs_mlp_train(m, steps, nullptr);
  m->profiling = false;
  if (rc) return rc;
  double ms[MC_N] = {0}, cnt[MC_N] = {0};
  for (size_t k = 0; k < m->evclass.size(); ++k) {
    float t = 0.f;
    MLPC(hipEventElapsedTime(&t, m->evpool[2 * k], m->evpool[2 * k + 1]));
    ms[m->evclass[k]] += t;
    cnt[m->evclass[k]] += 1;
  }
  // matrix-core flops per launch (2 per multiply-add)
  const double M = m->M;
  double fl[MC_N] = {0};
  double fwd = 0;
  for (int l = 0; l < m->L; ++l) {
    fwd += 2.0 * M * (l == 0 ? kIn : kW) * kW;
  }
  fl[MC_FWD] = fwd;
  fl[MC_WGRAD] = fwd;
  fl[MC_BWD] = 2.0 * M * kW * kW * (m->L - 1);
  fl[MC_HEAD] = 2.0 * M * kW * kOut * 3.0;
  for (int k = 0; k < MC_N; ++k) {
    ms6[k] = cnt[k] ? ms[k] / cnt[k] : 0.0;
    flop6[k] = fl[k];
    launches6[k] = int(cnt[k] / steps);
  }
  return 0;
} catch (...) {
  return host_exception("fvs_mlp_kernel_times");
}

double fvs_mlp_last_elapsed_ms(const fvs_mlp *m) { return m ? double(m->last_ms) : 0.0; }

}  // extern "C"
