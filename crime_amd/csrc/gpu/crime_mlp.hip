// The C_l emulator's network (include/crime_mlp.h): one kernel takes a block of rows through every layer
// (BF16 MFMA, FP32 edge layers, activations in LDS), and in training back through them; a second one forms the
// deterministic split-K weight gradients and applies Adam.  A training step is those two, captured as a HIP
// graph (step counter, learning rate and minibatch RNG live on the device, so the graph replays unchanged).
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <condition_variable>
#include <exception>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "crime_mlp.h"
#include "gh_device.hpp"

using namespace crime;

namespace {

constexpr int NIN = CRIME_MLP_IN, WD = CRIME_MLP_WIDTH, NH = CRIME_MLP_HIDDEN;
constexpr int NMID = NH - 1;                          // square WD x WD layers
constexpr int64_t OFF_W0 = 0, OFF_MID = OFF_W0 + (int64_t)NIN * WD + WD;
constexpr int64_t MID_STRIDE = (int64_t)WD * WD + WD; // W_k then b_k
constexpr int64_t OFF_W5 = OFF_MID + NMID * MID_STRIDE;
constexpr int64_t NPARAM = OFF_W5 + WD + 1;
constexpr int KSPLIT = 256;                           // batch rows per split of a weight-gradient GEMM
constexpr int RROWS = 32;                             // batch rows per partial of the column reductions
constexpr uint32_t MLP_KEY1 = 0x4D4C5031u;            // second Philox key word of the minibatch draws

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

// per-handle device state read by the captured step
struct DevState {
  int step;        // Adam updates applied since set_params
  int step_b;      // k_mlp_rows' copy of step for k_mlp_update, which advances step itself
  int local;       // step index within the current train call (loss slot)
  int total;       // steps of the cosine schedule
  float lr0, b1, b2, eps;
  uint32_t seed;
  int64_t ndata;
  float lr, c1, c2;   // this step's learning rate and Adam bias corrections (k_mlp_rows, for k_mlp_update)
};

__device__ __forceinline__ uint16_t f2bf(float x)
{
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);   // round to nearest even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// four floats to BF16, round to nearest even: the bits of f2bf in one v_cvt_pk_bf16_f32 per pair
__device__ __forceinline__ uint2 pack4_bf16(float a, float b, float c, float d)
{
  typedef float fl4 __attribute__((ext_vector_type(4)));
  typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
  const fl4 v = {a, b, c, d};
  return __builtin_bit_cast(uint2, __builtin_convertvector(v, bf4));
}

// 1 / (1 + e^-z) as the correctly rounded quotient, without the operand scaling of a general division: the reciprocal
// of 1 <= d < 2^120 by a Newton step and two residual corrections in fused arithmetic (Markstein 1990, IBM J. Res. Dev.
// 34, 111; the quotient's bits are checked for every z by crime_mlp_silu_check)
__device__ __forceinline__ float sigm(float z)
{
  if (__builtin_expect(!(z > -80.0f), 0)) return 1.0f / (1.0f + expf(-z));
  const float d = 1.0f + expf(-z);
  const float r = __builtin_amdgcn_rcpf(d);
  const float r1 = fmaf(fmaf(-d, r, 1.0f), r, r);
  const float q = fmaf(fmaf(-d, r1, 1.0f), r1, r1);
  return fmaf(fmaf(-d, q, 1.0f), r1, q);
}

// bf16(z sigm(z)) of four values.  Most results do not depend on the last bits of sigm: with the hardware's
// exponential and reciprocal the product is within SILU_ULP units in the last place of z sigm(z) for z > SILU_MIN
// (its BF16 value is checked for every z by crime_mlp_silu_check), so unless it lies that close to a rounding boundary
// of BF16 its BF16 value is the same.  The others (one in 2600) take sigm.
constexpr unsigned SILU_ULP = 12;
constexpr float SILU_MIN = -9.0f;
__device__ __forceinline__ uint2 silu4_bf16(const float (&z)[4])
{
  float h[4];
  unsigned near = 0xffffu;
  float low = 0.0f;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const float e = __builtin_amdgcn_exp2f(z[v] * -1.44269504088896341f);
    h[v] = z[v] * __builtin_amdgcn_rcpf(1.0f + e);
    near = min(near, (__float_as_uint(h[v]) + (SILU_ULP - 0x8000u)) & 0xffffu);
    low = fminf(low, z[v]);
  }
  if (__builtin_expect(near <= 2 * SILU_ULP || !(low > SILU_MIN), 0)) {
#pragma unroll
    for (int v = 0; v < 4; v++) h[v] = z[v] * sigm(z[v]);
  }
  return pack4_bf16(h[0], h[1], h[2], h[3]);
}

// ---------------------------------------------------------------------------------------------
// The square layers run on v_mfma_f32_16x16x32_bf16 with the weights as the A operand and the
// activations as B (D = W^T h^T): lane l supplies W of feature l % 16 at the eight inputs 8 (l / 16) .. + 7,
// and h of row l % 16 at the same eight; D holds features 4 (l / 16) .. + 3 of row l % 16, four consecutive
// features of a row, which go back to the LDS tile as one 8-byte store.  The weights' BF16 copies lie in
// exactly that order, 16 bytes per lane and 1 KB per wave: frag(layer, tile of 16 outputs, step of 32 inputs).
// wf serves the forward product (outputs n, inputs k), wb the backward one (outputs k, inputs n).
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ size_t frag_index(int layer, int out, int in)
{
  const int t = out >> 4, s = in >> 5, l = (out & 15) + 16 * ((in & 31) >> 3);
  return ((((size_t)layer * 16 + t) * 8 + s) * 64 + l) * 8 + (in & 7);
}

constexpr int UPD_THREADS = 512;
constexpr int row_threads(int NT) { return 64 * (WD / 16) / NT; }   // a wave per NT tiles of 16 features
constexpr int HSTR = WD + 8;          // LDS row stride: 16 rows of one 16-byte column fall on distinct banks
constexpr int TR = RROWS;             // rows per workgroup of a training step: one partial of the column sums
constexpr int FWD_ROWS = 64;          // rows per workgroup of a large forward call
static_assert(TR == 32 && WD == 256, "k_mlp_rows' thread layout");

struct RowArgs {
  const float *X, *T, *Wt;       // inputs, targets, weights (the whole training set with gather)
  const float *p;
  const uint16_t *wf, *wb;
  float *Y;                      // forward only: outputs
  uint16_t *hp, *dzp;            // training: [4][octet of rows][feature][row % 8]
  float *part_in, *part_out, *part_b;
  DevState *st;
  float *loss;
  size_t stride;                 // elements per layer of hp, dzp
  int n, npart;                  // rows; partials allocated per layer in part_b
  int gather;
  float scale;                   // forward: not 0: write scale sinh(y) (the emulator's spectra) for y
};

__device__ __forceinline__ float spectrum(float y, float scale) { return (float)sinh((double)y) * scale; }

// One workgroup takes BM rows through the whole network without leaving the CU: the activations of the
// current layer stay in one LDS tile, the weights stream from L2 as fragments (prefetched across the
// epilogue), and a training step (TRAIN) carries on with the loss and the backward pass, its pre-activations
// held in registers from the forward half.
// A wave owns NT tiles of 16 features of every row.  What bounds it: up to 32 rows the 128 KB of weights per
// layer through the CU's vector cache and the latency of the layers in series; at 64 rows the SiLU epilogue
// (about 12 VALU instructions per element beside 512 MFMA flops), which the second workgroup of the CU overlaps.
// Measured: 65536 rows forward 82 us (418 TFLOP/s) against 321 us for one kernel per layer, which wrote and
// read every activation; 128-row workgroups (one per CU) 95 us.  256 rows 13 us (16-row workgroups) against
// 20 us (32 rows, NT = 2) and 50 us (one kernel per layer).  A training step's rows, 4096 of them: 40 us, and
// k_mlp_update 13 us, against 480 us for the 30 kernels of a step before.
template <int BM, int NT, bool TRAIN>
__global__ __launch_bounds__(row_threads(NT), 4) void k_mlp_rows(RowArgs g)
{
  constexpr int MT = BM / 16, NTHREADS = row_threads(NT);
  constexpr int NZ = TRAIN ? MT : 1;
  __shared__ __align__(16) uint16_t hs[BM * HSTR];
  __shared__ __align__(16) float xs[BM * NIN];
  __shared__ float ds[BM];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lg = lane >> 4;
  const int row0 = blockIdx.x * BM;
  const int f0 = 16 * NT * wv + 4 * lg;     // this lane's features: f0 + 16 nt + v
  uint4 w[NT][8];
  auto load_w = [&](const uint16_t *frags, int layer) {
#pragma unroll
    for (int nt = 0; nt < NT; nt++)
#pragma unroll
      for (int s = 0; s < 8; s++)
        w[nt][s] = *(const uint4 *)(frags + ((((size_t)layer * 16 + NT * wv + nt) * 8 + s) * 64 + lane) * 8);
  };
  load_w(g.wf, 0);
  float tgt = 0.f, wgt = 0.f;          // target and weight of row tid (tid < BM)
  if (tid < BM) {
    int64_t i = row0 + tid;
    const bool live = row0 + tid < g.n;
    if (TRAIN && g.gather) {
      u32x4 c = {{(uint32_t)g.st->step, (uint32_t)(row0 + tid), 0u, 0u}};
      u32x4 r = philox4x32_10(c, g.st->seed, MLP_KEY1);
      const uint64_t u = ((uint64_t)r.v[0] << 32) | r.v[1];
      i = (int64_t)(u % (uint64_t)g.st->ndata);
    }
    float4 x0 = make_float4(0, 0, 0, 0), x1 = x0;
    if (live) {
      x0 = *(const float4 *)(g.X + (size_t)i * NIN);
      x1 = *(const float4 *)(g.X + (size_t)i * NIN + 4);
      if (TRAIN) {
        tgt = g.T[i];
        wgt = g.Wt[i];
      }
    }
    *(float4 *)(xs + tid * NIN) = x0;
    *(float4 *)(xs + tid * NIN + 4) = x1;
  }
  if (TRAIN && blockIdx.x == 0 && tid == NTHREADS - 1) {
    const int st = g.st->step, total = g.st->total;
    const float frac = total > 0 ? fminf((float)st / (float)total, 1.0f) : 0.0f;
    g.st->step_b = st;
    g.st->lr = g.st->lr0 * 0.5f * (1.0f + cosf(3.14159265358979f * frac));
    g.st->c1 = 1.0f - powf(g.st->b1, (float)(st + 1));
    g.st->c2 = 1.0f - powf(g.st->b2, (float)(st + 1));
  }
  __syncthreads();

  float z[NZ][NT][TRAIN ? NH : 1][4];   // pre-activations of every layer (TRAIN)
  // input layer: z = b + sum_i x_i W0[i], FP32
#pragma unroll
  for (int nt = 0; nt < NT; nt++) {
    const int f = f0 + 16 * nt;
    float4 wc[NIN];
#pragma unroll
    for (int i = 0; i < NIN; i++) wc[i] = *(const float4 *)(g.p + OFF_W0 + (int64_t)i * WD + f);
    const float4 b = *(const float4 *)(g.p + OFF_W0 + (int64_t)NIN * WD + f);
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
      const float4 x0 = *(const float4 *)(xs + (16 * mt + lr) * NIN), x1 = *(const float4 *)(xs + (16 * mt + lr) * NIN + 4);
      const float x[NIN] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      float a[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int i = 0; i < NIN; i++) {
        a[0] = fmaf(x[i], wc[i].x, a[0]);
        a[1] = fmaf(x[i], wc[i].y, a[1]);
        a[2] = fmaf(x[i], wc[i].z, a[2]);
        a[3] = fmaf(x[i], wc[i].w, a[3]);
      }
      if constexpr (TRAIN)
        for (int v = 0; v < 4; v++) z[mt][nt][0][v] = a[v];
      *(uint2 *)(hs + (16 * mt + lr) * HSTR + f) = silu4_bf16(a);
    }
  }
  __syncthreads();

  // the LDS tile's rows 8 o .. 8 o + 7 of one feature as one 16-byte chunk
  auto octet = [&](int o, int f) {
    union { uint16_t e[8]; uint4 q; } u;
#pragma unroll
    for (int r = 0; r < 8; r++) u.e[r] = hs[(8 * o + r) * HSTR + f];
    return u.q;
  };
  auto mma = [&](f4 (&acc)[MT][NT]) {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
      for (int nt = 0; nt < NT; nt++) acc[mt][nt] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 8; s++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const bf16x8 h = __builtin_bit_cast(bf16x8, *(const uint4 *)(hs + (16 * mt + lr) * HSTR + 32 * s + 8 * lg));
        for (int nt = 0; nt < NT; nt++)
          acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[nt][s]), h, acc[mt][nt], 0, 0, 0);
      }
  };

#pragma unroll
  for (int k = 0; k < NMID; k++) {
    if constexpr (TRAIN) {   // the weight gradient's copy of this layer's input
      const int f = tid & 255;
#pragma unroll 1
      for (int o = tid >> 8; o < BM / 8; o += NTHREADS / 256)
        *(uint4 *)(g.hp + k * g.stride + ((size_t)(row0 / 8 + o) * WD + f) * 8) = octet(o, f);
    }
    f4 acc[MT][NT];
    mma(acc);
    if (k + 1 < NMID) load_w(g.wf, k + 1);
    else if (TRAIN) load_w(g.wb, NMID - 1);
    const float *bias = g.p + OFF_MID + k * MID_STRIDE + (int64_t)WD * WD;
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      const int f = f0 + 16 * nt;
      const float4 b = *(const float4 *)(bias + f);
      const float bb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        float zz[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          zz[v] = acc[mt][nt][v] + bb[v];
          if constexpr (TRAIN) z[mt][nt][k + 1][v] = zz[v];
        }
        *(uint2 *)(hs + (16 * mt + lr) * HSTR + f) = silu4_bf16(zz);
      }
    }
    __syncthreads();
  }

  // output layer, a wave per row: y = h5 . w5 + b5; training also d = 2 w (y - t) / n and the loss
  const float *w5 = g.p + OFF_W5;
  const float o0 = w5[lane], o1 = w5[lane + 64], o2 = w5[lane + 128], o3 = w5[lane + 192], b5 = w5[WD];
  for (int r = wv; r < BM; r += NTHREADS / 64) {
    const uint16_t *h = hs + r * HSTR + lane;
    float s = 0.f;
    s = fmaf(bf2f(h[0]), o0, s);
    s = fmaf(bf2f(h[64]), o1, s);
    s = fmaf(bf2f(h[128]), o2, s);
    s = fmaf(bf2f(h[192]), o3, s);
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if (lane == 0) ds[r] = s + b5;
  }
  __syncthreads();
  if constexpr (!TRAIN) {
    if (tid < BM && row0 + tid < g.n) g.Y[row0 + tid] = g.scale != 0.0f ? spectrum(ds[tid], g.scale) : ds[tid];
    return;
  }
  else {
    if (tid < BM) {
      const float e = ds[tid] - tgt;
      ds[tid] = 2.0f * wgt * e / (float)g.n;
      atomicAdd(g.loss + g.st->local, wgt * e * e / (float)g.n);
    }
    __syncthreads();
    // partials of dw5 = sum_r h5 d and db5 = sum_r d over the workgroup's rows
    if (tid < WD) {
      float a = 0.f, b = 0.f;
#pragma unroll 8
      for (int r = 0; r < BM; r++) {
        a = fmaf(bf2f(hs[r * HSTR + tid]), ds[r], a);
        b += ds[r];
      }
      g.part_out[(size_t)blockIdx.x * (WD + 1) + tid] = a;
      if (tid == 0) g.part_out[(size_t)blockIdx.x * (WD + 1) + WD] = b;
    }
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
      const int f = f0 + 16 * nt;
      const float wo[4] = {w5[f], w5[f + 1], w5[f + 2], w5[f + 3]};
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const float d = ds[16 * mt + lr];
        float q[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const float zz = z[mt][nt][NH - 1][v], sg = sigm(zz);
          q[v] = d * wo[v] * sg * (1.0f + zz * (1.0f - sg));
        }
        *(uint2 *)(hs + (16 * mt + lr) * HSTR + f) = pack4_bf16(q[0], q[1], q[2], q[3]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = NMID - 1; k >= 0; k--) {
      f4 acc[MT][NT];
      mma(acc);
      if (k > 0) load_w(g.wb, k - 1);
      // meanwhile the tile holds the gradient at square layer k's output: its column sums (the first four waves)
      // and the weight gradient's copy (the others)
      if (tid < WD) {
        float a = 0.f;
#pragma unroll 8
        for (int r = 0; r < BM; r++) a += bf2f(hs[r * HSTR + tid]);
        g.part_b[((size_t)k * g.npart + blockIdx.x) * WD + tid] = a;
      }
      else {
        const int f = tid & 255;
#pragma unroll 1
        for (int o = (tid >> 8) - 1; o < BM / 8; o += NTHREADS / 256 - 1)
          *(uint4 *)(g.dzp + k * g.stride + ((size_t)(row0 / 8 + o) * WD + f) * 8) = octet(o, f);
      }
      __syncthreads();
#pragma unroll
      for (int nt = 0; nt < NT; nt++) {
        const int f = f0 + 16 * nt;
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
          float q[4];
#pragma unroll
          for (int v = 0; v < 4; v++) {   // dz_prev = acc silu'(z_prev), silu' = s (1 + z (1 - s))
            const float zz = z[mt][nt][k][v], s = sigm(zz);
            q[v] = acc[mt][nt][v] * s * (1.0f + zz * (1.0f - s));
          }
          *(uint2 *)(hs + (16 * mt + lr) * HSTR + f) = pack4_bf16(q[0], q[1], q[2], q[3]);
        }
      }
      __syncthreads();
    }
    // partials of dW0 = x^T dz1 and db0 = sum_r dz1: part[block][i][c] (i < 8), part[block][8][c]
    if (tid < WD) {
      float a[NIN + 1] = {};
#pragma unroll 4
      for (int r = 0; r < BM; r++) {
        const float d = bf2f(hs[r * HSTR + tid]);
#pragma unroll
        for (int i = 0; i < NIN; i++) a[i] = fmaf(xs[r * NIN + i], d, a[i]);
        a[NIN] += d;
      }
      for (int i = 0; i <= NIN; i++) g.part_in[((size_t)blockIdx.x * (NIN + 1) + i) * WD + tid] = a[i];
    }
  }
}

// ---------------------------------------------------------------------------------------------
// gradients of every parameter and their Adam update (Kingma & Ba 2015), one launch.
// Workgroups 0 .. 255: a 32 x 32 tile of one square layer's dW = h^T dz.  The rows are summed in splits of
// KSPLIT (each split one chain of MFMAs from zero, as many splits at a time as there are waves), the splits in
// ascending order through LDS, so that the sum does not depend on the launch.  The operands are read as laid
// out by k_mlp_rows, 16 bytes per lane with no transposition.  The other workgroups: a thread per remaining
// parameter, over the row-chunk partials.
// ---------------------------------------------------------------------------------------------
struct UpdateArgs {
  float *p, *m, *v;
  float *grad;                   // not NULL: write the gradient there and leave the parameters alone
  uint16_t *wf, *wb;
  const uint16_t *hp, *dzp;
  const float *part_in, *part_out, *part_b;
  DevState *st;
  size_t stride;
  int n, npart, npart_alloc;     // rows; row-chunk partials; partials allocated per layer in part_b
};

constexpr int GT_ = 32;                                 // dW tile edge
constexpr int TILES = (WD / GT_) * (WD / GT_);          // per layer
constexpr int NSMALL = (NIN + 1) * WD + NMID * WD + WD + 1;
constexpr int UPD_BLOCKS = NMID * TILES + (NSMALL + UPD_THREADS - 1) / UPD_THREADS;

__device__ __forceinline__ float adam_update(const UpdateArgs &u, const DevState &a, int64_t i, float g)
{
  // fused products as written, the same on every build
#pragma clang fp contract(off)
  const float mi = fmaf(1.0f - a.b1, g, a.b1 * u.m[i]);
  const float vi = fmaf(a.b2, u.v[i], (1.0f - a.b2) * g * g);
  u.m[i] = mi;
  u.v[i] = vi;
  const float mh = mi / a.c1, vh = vi / a.c2;
  const float pi = u.p[i] - a.lr * mh / (sqrtf(vh) + a.eps);
  u.p[i] = pi;
  return pi;
}

__global__ __launch_bounds__(UPD_THREADS) void k_mlp_update(UpdateArgs u)
{
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, lr = lane & 15, lg = lane >> 4;
  const bool update = u.grad == nullptr;
  if (blockIdx.x < NMID * TILES) {
    constexpr int NW = UPD_THREADS / 64, PS = GT_ * (GT_ + 1);
    __shared__ float part[NW * PS];
    // blocks go to the eight XCDs in turn: two XCDs take one layer each, so that an XCD's L2 reads one layer's
    // operands (3 MB at 4096 rows) and not all four's
    static_assert(NMID == 4 && TILES % 2 == 0, "an XCD per half layer");
    const int xcd = blockIdx.x & 7, layer = xcd >> 1, tile = (xcd & 1) * (TILES / 2) + (blockIdx.x >> 3);
    const int i0 = (tile / (WD / GT_)) * GT_, j0 = (tile % (WD / GT_)) * GT_;
    const uint16_t *hp = u.hp + layer * u.stride, *dzp = u.dzp + layer * u.stride;
    const int ns = (u.n + KSPLIT - 1) / KSPLIT;
    constexpr int EL = GT_ * GT_ / UPD_THREADS;   // elements per thread
    float sum[EL] = {};
    for (int z0 = 0; z0 < ns; z0 += NW) {
      const int zs = z0 + wv;
      if (zs < ns) {
        const int kb = zs * KSPLIT, ke = u.n < kb + KSPLIT ? u.n : kb + KSPLIT;
        f4 acc[2][2];
        for (int i = 0; i < 2; i++)
          for (int j = 0; j < 2; j++) acc[i][j] = (f4){0.f, 0.f, 0.f, 0.f};
        auto step = [&](int r) {
          const size_t o = (size_t)(r / 8 + lg) * WD + lr;
          bf16x8 a[2], b[2];
          for (int i = 0; i < 2; i++) a[i] = __builtin_bit_cast(bf16x8, *(const uint4 *)(hp + (o + i0 + 16 * i) * 8));
          for (int j = 0; j < 2; j++) b[j] = __builtin_bit_cast(bf16x8, *(const uint4 *)(dzp + (o + j0 + 16 * j) * 8));
          for (int i = 0; i < 2; i++)
            for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        };
        if (ke - kb == KSPLIT) {   // a whole split: every load in flight before the first product
#pragma unroll
          for (int r = 0; r < KSPLIT; r += 32) step(kb + r);
        }
        else {
          for (int r = kb; r < ke; r += 32) step(r);
        }
        for (int i = 0; i < 2; i++)
          for (int j = 0; j < 2; j++)
            for (int v = 0; v < 4; v++)
              part[wv * PS + (16 * i + 4 * lg + v) * (GT_ + 1) + 16 * j + lr] = acc[i][j][v];
      }
      __syncthreads();
      const int nz = ns - z0 < NW ? ns - z0 : NW;
      for (int e = 0; e < EL; e++) {
        const int el = tid + e * UPD_THREADS, i = el / GT_, j = el % GT_;
        for (int q = 0; q < nz; q++) sum[e] += part[q * PS + i * (GT_ + 1) + j];
      }
      __syncthreads();
    }
    const DevState a = *u.st;
    for (int e = 0; e < EL; e++) {
      const int el = tid + e * UPD_THREADS, i = i0 + el / GT_, j = j0 + el % GT_;
      const int64_t idx = OFF_MID + layer * MID_STRIDE + (int64_t)i * WD + j;
      if (!update) {
        u.grad[idx] = sum[e];
        continue;
      }
      const uint16_t b = f2bf(adam_update(u, a, idx, sum[e]));
      u.wf[frag_index(layer, j, i)] = b;
      u.wb[frag_index(layer, i, j)] = b;
    }
    if (update && blockIdx.x == 0 && tid == 0) {
      u.st->step = u.st->step_b + 1;
      u.st->local += 1;
    }
    return;
  }
  const int q = (blockIdx.x - NMID * TILES) * UPD_THREADS + tid;
  if (q >= NSMALL) return;
  // parameter q of the input layer, the square layers' biases or the output layer: its index, partials and their stride
  constexpr int NI = (NIN + 1) * WD, NB = NMID * WD;
  int64_t idx;
  const float *part;
  int stride;
  if (q < NI) {
    idx = OFF_W0 + q;
    part = u.part_in + q;
    stride = NI;
  }
  else if (q < NI + NB) {
    const int k = (q - NI) / WD, c = (q - NI) % WD;
    idx = OFF_MID + k * MID_STRIDE + (int64_t)WD * WD + c;
    part = u.part_b + (size_t)k * u.npart_alloc * WD + c;
    stride = WD;
  }
  else {
    idx = OFF_W5 + (q - NI - NB);
    part = u.part_out + (q - NI - NB);
    stride = WD + 1;
  }
  float g = 0.f;
  int z = 0;
  for (; z + 16 <= u.npart; z += 16) {   // sixteen loads in flight, added in order
    float q[16];
#pragma unroll
    for (int e = 0; e < 16; e++) q[e] = part[(size_t)(z + e) * stride];
#pragma unroll
    for (int e = 0; e < 16; e++) g += q[e];
  }
  for (; z < u.npart; z++) g += part[(size_t)z * stride];
  if (!update) u.grad[idx] = g;
  else adam_update(u, *u.st, idx, g);
}

// the BF16 fragment copies of the square layers, from the FP32 parameters
__global__ __launch_bounds__(256) void k_pack_weights(const float *__restrict__ p, uint16_t *__restrict__ wf,
                                                      uint16_t *__restrict__ wb)
{
  const int i = blockIdx.x, j = threadIdx.x, k = blockIdx.y;
  const uint16_t b = f2bf(p[OFF_MID + k * MID_STRIDE + (int64_t)i * WD + j]);
  wf[frag_index(k, j, i)] = b;
  wb[frag_index(k, i, j)] = b;
}

}  // namespace

constexpr int PRED_SLOTS = 4, PRED_THREADS = 8;
constexpr int PRED_MIN = 4096, PRED_DIRECT = 24576, PRED_REUSE = 98304, PRED_ROWS = 65536;   // rows: see predict_impl

// pinned inputs and outputs of crime_mlp_predict, and the addresses the device has them at
struct HostRows {
  float *x = nullptr, *y = nullptr, *x_dev = nullptr, *y_dev = nullptr;
};

struct crime_mlp {
  int max_batch = 0, device = 0;
  hipStream_t stream = nullptr;
  float *p = nullptr, *m = nullptr, *v = nullptr, *grad = nullptr;
  uint16_t *wf = nullptr, *wb = nullptr;    // BF16 fragments of the square layers, forward and backward order
  float *X = nullptr, *T = nullptr, *Wt = nullptr, *Y = nullptr;
  uint16_t *hp = nullptr, *dzp = nullptr;   // [NMID][max_batch * WD] weight-gradient operands (k_mlp_rows)
  float *part_in = nullptr, *part_out = nullptr, *part_b = nullptr;
  DevState *st = nullptr;
  float *loss = nullptr;
  int loss_cap = 0;
  float *Xall = nullptr, *Tall = nullptr, *Wall = nullptr;
  int64_t ndata = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int graph_batch = 0;
  int use_graph = 1;                        // 0: every step enqueued directly (crime_mlp_set_graph)
  // crime_mlp_predict: pinned inputs and outputs of direct_rows rows, max_batch of them made with the handle
  int64_t direct_rows = 0;
  HostRows direct;
  // and of a long call's ring of chunks, ring_rows rows in all, whose inputs a stream of its own sends to ring_dx
  int64_t ring_rows = 0;
  HostRows ring;
  float *ring_dx = nullptr;
  hipEvent_t slot_in[PRED_SLOTS] = {}, slot_ev[PRED_SLOTS] = {};   // a slot's inputs are in ring_dx; its outputs in y
  hipStream_t copy = nullptr;
  std::string err;
};

static thread_local std::string g_mlp_err;

static int mlp_error(crime_mlp *h, int code, const char *fmt, ...)
{
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  if (h) h->err = buf;
  else g_mlp_err = buf;
  return code;
}

#define MLP_HIP(h, call)                                                                          \
  do {                                                                                                \
    hipError_t e_ = (call);                                                                           \
    if (e_ != hipSuccess) {                                                                           \
      (void)hipGetLastError(); /* reported here: a later launch check must not see it again */        \
      return mlp_error(h, e_ == hipErrorOutOfMemory ? CRIME_GH_ENOMEM : CRIME_GH_EHIP, "%s: %s", #call,     \
                       hipGetErrorString(e_));                                                        \
    }                                                                                                 \
  } while (0)

extern "C" int64_t crime_mlp_param_count(void) { return NPARAM; }
extern "C" const char *crime_mlp_last_error(const crime_mlp_t *h) { return h ? h->err.c_str() : g_mlp_err.c_str(); }

static void drop_graph(crime_mlp *h)
{
  if (h->exec) (void)hipGraphExecDestroy(h->exec);
  if (h->graph) (void)hipGraphDestroy(h->graph);
  h->exec = nullptr;
  h->graph = nullptr;
  h->graph_batch = 0;
}

static void drop_ring(crime_mlp *h)
{
  if (h->ring.x) (void)hipHostFree(h->ring.x);
  if (h->ring_dx) (void)hipFree(h->ring_dx);
  h->ring = HostRows{};
  h->ring_dx = nullptr;
  h->ring_rows = 0;
}

extern "C" void crime_mlp_destroy(crime_mlp_t *h)
{
  if (!h) return;
  (void)hipSetDevice(h->device);
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  if (h->copy) (void)hipStreamSynchronize(h->copy);
  drop_graph(h);
  drop_ring(h);
  if (h->direct.x) (void)hipHostFree(h->direct.x);
  for (int i = 0; i < PRED_SLOTS; i++) {
    if (h->slot_in[i]) (void)hipEventDestroy(h->slot_in[i]);
    if (h->slot_ev[i]) (void)hipEventDestroy(h->slot_ev[i]);
  }
  if (h->copy) (void)hipStreamDestroy(h->copy);
  void *bufs[] = {h->p, h->m, h->v, h->grad, h->wf, h->wb, h->X, h->T, h->Wt, h->Y, h->hp, h->dzp,
                  h->part_in, h->part_out, h->part_b, h->st, h->loss, h->Xall, h->Tall, h->Wall};
  for (void *b : bufs)
    if (b) (void)hipFree(b);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

static int nred_of(int n) { return (n + RROWS - 1) / RROWS; }

// pinned memory for `rows` rows, the outputs behind the inputs
static int alloc_rows(crime_mlp *h, int64_t rows, HostRows *r)
{
  MLP_HIP(h, hipHostMalloc((void **)&r->x, (size_t)rows * (NIN + 1) * sizeof(float), hipHostMallocDefault));
  MLP_HIP(h, hipHostGetDevicePointer((void **)&r->x_dev, r->x, 0));
  r->y = r->x + rows * NIN;
  r->y_dev = r->x_dev + rows * NIN;
  return 0;
}

static int ensure_direct(crime_mlp *h, int64_t rows)
{
  for (hipEvent_t &e : h->slot_ev)
    if (!e) MLP_HIP(h, hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (rows <= h->direct_rows) return 0;
  if (h->direct.x) (void)hipHostFree(h->direct.x);
  h->direct = HostRows{};
  h->direct_rows = 0;
  const int rc = alloc_rows(h, rows, &h->direct);
  if (!rc) h->direct_rows = rows;
  return rc;
}

static int ensure_ring(crime_mlp *h, int64_t rows)
{
  if (!h->copy) MLP_HIP(h, hipStreamCreateWithFlags(&h->copy, hipStreamNonBlocking));
  for (hipEvent_t &e : h->slot_in)
    if (!e) MLP_HIP(h, hipEventCreateWithFlags(&e, hipEventDisableTiming));
  for (hipEvent_t &e : h->slot_ev)
    if (!e) MLP_HIP(h, hipEventCreateWithFlags(&e, hipEventDisableTiming));
  if (rows <= h->ring_rows) return 0;
  drop_ring(h);
  const int rc = alloc_rows(h, rows, &h->ring);
  if (rc) return rc;
  MLP_HIP(h, hipMalloc((void **)&h->ring_dx, (size_t)rows * NIN * sizeof(float)));
  h->ring_rows = rows;
  return 0;
}

static int create_impl(crime_mlp *h, int max_batch, int device)
{
  if (max_batch < 64 || max_batch > 65536 || max_batch % 64)
    return mlp_error(h, CRIME_GH_EINVAL, "max_batch %d: a multiple of 64 in [64, 65536]", max_batch);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return mlp_error(h, CRIME_GH_ENODEV, "no HIP device");
  if (device < 0 || device >= ndev) return mlp_error(h, CRIME_GH_ENODEV, "device %d of %d", device, ndev);
  h->max_batch = max_batch;
  h->device = device;
  MLP_HIP(h, hipSetDevice(device));
  MLP_HIP(h, hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
  const size_t B = (size_t)max_batch;
  const int nr = nred_of(max_batch);
  MLP_HIP(h, hipMalloc((void **)&h->p, NPARAM * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->m, NPARAM * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->v, NPARAM * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->grad, NPARAM * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->wf, (size_t)NMID * WD * WD * sizeof(uint16_t)));
  MLP_HIP(h, hipMalloc((void **)&h->wb, (size_t)NMID * WD * WD * sizeof(uint16_t)));
  MLP_HIP(h, hipMalloc((void **)&h->X, B * NIN * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->T, B * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->Wt, B * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->Y, B * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->hp, NMID * B * WD * sizeof(uint16_t)));
  MLP_HIP(h, hipMalloc((void **)&h->dzp, NMID * B * WD * sizeof(uint16_t)));
  MLP_HIP(h, hipMalloc((void **)&h->part_in, (size_t)nr * (NIN + 1) * WD * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->part_out, (size_t)nr * (WD + 1) * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->part_b, (size_t)NMID * nr * WD * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->st, sizeof(DevState)));
  DevState s{};
  MLP_HIP(h, hipMemcpy(h->st, &s, sizeof(s), hipMemcpyHostToDevice));
  std::vector<float> zero(NPARAM, 0.0f);
  MLP_HIP(h, hipMemcpy(h->p, zero.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemcpy(h->m, zero.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemcpy(h->v, zero.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  return ensure_direct(h, std::min(PRED_DIRECT, max_batch));   // a first call finds them
}

extern "C" int crime_mlp_create(int max_batch, int device, crime_mlp_t **out)
{
  if (!out) return mlp_error(nullptr, CRIME_GH_EINVAL, "out is NULL");
  *out = nullptr;
  crime_mlp *h = new crime_mlp;
  int rc = create_impl(h, max_batch, device);
  if (rc) {
    g_mlp_err = h->err;
    crime_mlp_destroy(h);
    return rc;
  }
  *out = h;
  return 0;
}

extern "C" int crime_mlp_set_params(crime_mlp_t *h, const float *params)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (!params) return mlp_error(h, CRIME_GH_EINVAL, "params are NULL");
  MLP_HIP(h, hipSetDevice(h->device));
  MLP_HIP(h, hipMemcpy(h->p, params, NPARAM * sizeof(float), hipMemcpyHostToDevice));
  std::vector<float> zero(NPARAM, 0.0f);
  MLP_HIP(h, hipMemcpy(h->m, zero.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemcpy(h->v, zero.data(), NPARAM * sizeof(float), hipMemcpyHostToDevice));
  DevState s{};
  MLP_HIP(h, hipMemcpy(h->st, &s, sizeof(s), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_pack_weights, dim3(WD, NMID), dim3(WD), 0, h->stream, h->p, h->wf, h->wb);
  MLP_HIP(h, hipGetLastError());
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  return 0;
}

extern "C" int crime_mlp_get_params(crime_mlp_t *h, float *params)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (!params) return mlp_error(h, CRIME_GH_EINVAL, "params are NULL");
  MLP_HIP(h, hipSetDevice(h->device));
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  MLP_HIP(h, hipMemcpy(params, h->p, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}

static RowArgs row_args(crime_mlp *h, int n)
{
  RowArgs g{};
  g.X = h->X;
  g.T = h->T;
  g.Wt = h->Wt;
  g.p = h->p;
  g.wf = h->wf;
  g.wb = h->wb;
  g.Y = h->Y;
  g.hp = h->hp;
  g.dzp = h->dzp;
  g.part_in = h->part_in;
  g.part_out = h->part_out;
  g.part_b = h->part_b;
  g.st = h->st;
  g.loss = h->loss;
  g.stride = (size_t)h->max_batch * WD;
  g.n = n;
  g.npart = nred_of(h->max_batch);
  return g;
}

// forward for rows [0, n) of X (the handle's own input buffer unless given) on stream s (its own unless given).
// The fewest rows per workgroup that still give every one of the 256 CUs at most one workgroup, as the layers'
// latency counts there (256 rows: 13 us by 16, 20 us by 32); above that 64 rows, which read the weights less often.
static void enqueue_forward(crime_mlp *h, int n, hipStream_t s = nullptr, const float *X = nullptr, float *Y = nullptr,
                            float scale = 0.0f)
{
  if (!s) s = h->stream;
  RowArgs g = row_args(h, n);
  if (X) g.X = X;
  if (Y) g.Y = Y;
  g.scale = scale;
  auto launch = [&](auto bm, auto nt) {
    constexpr int BM = decltype(bm)::value, NT = decltype(nt)::value;
    hipLaunchKernelGGL((k_mlp_rows<BM, NT, false>), dim3((n + BM - 1) / BM), dim3(row_threads(NT)), 0, s, g);
  };
  using std::integral_constant;
  if (n <= 256 * 16) launch(integral_constant<int, 16>{}, integral_constant<int, 1>{});
  else if (n <= 256 * TR) launch(integral_constant<int, TR>{}, integral_constant<int, 1>{});
  else launch(integral_constant<int, FWD_ROWS>{}, integral_constant<int, 2>{});
}

// forward and backward for n rows (n % 64 == 0): of the training set drawn by Philox (gather), or of X, T, Wt
static void enqueue_rows(crime_mlp *h, int n, bool gather)
{
  RowArgs g = row_args(h, n);
  if (gather) {
    g.X = h->Xall;
    g.T = h->Tall;
    g.Wt = h->Wall;
    g.gather = 1;
  }
  hipLaunchKernelGGL((k_mlp_rows<TR, 1, true>), dim3(n / TR), dim3(row_threads(1)), 0, h->stream, g);
}

// the gradients of the last enqueue_rows: into grad, or the parameters' Adam update (grad NULL)
static void enqueue_update(crime_mlp *h, int n, float *grad)
{
  UpdateArgs u{};
  u.p = h->p;
  u.m = h->m;
  u.v = h->v;
  u.grad = grad;
  u.wf = h->wf;
  u.wb = h->wb;
  u.hp = h->hp;
  u.dzp = h->dzp;
  u.part_in = h->part_in;
  u.part_out = h->part_out;
  u.part_b = h->part_b;
  u.st = h->st;
  u.stride = (size_t)h->max_batch * WD;
  u.n = n;
  u.npart = nred_of(n);
  u.npart_alloc = nred_of(h->max_batch);
  hipLaunchKernelGGL(k_mlp_update, dim3(UPD_BLOCKS), dim3(UPD_THREADS), 0, h->stream, u);
}

static int ensure_loss(crime_mlp *h, int n)
{
  if (n <= h->loss_cap) return 0;
  drop_graph(h);  // the captured step holds the old buffer
  if (h->loss) MLP_HIP(h, hipFree(h->loss));
  h->loss = nullptr;
  h->loss_cap = 0;
  MLP_HIP(h, hipMalloc((void **)&h->loss, (size_t)n * sizeof(float)));
  h->loss_cap = n;
  return 0;
}

extern "C" int crime_mlp_forward(crime_mlp_t *h, int64_t n, const float *x, float *y)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (n < 1 || !x || !y) return mlp_error(h, CRIME_GH_EINVAL, "need n >= 1 and non-NULL x, y");
  MLP_HIP(h, hipSetDevice(h->device));
  for (int64_t i0 = 0; i0 < n; i0 += h->max_batch) {
    const int c = (int)(n - i0 < h->max_batch ? n - i0 : h->max_batch);
    MLP_HIP(h, hipMemcpyAsync(h->X, x + i0 * NIN, (size_t)c * NIN * sizeof(float), hipMemcpyHostToDevice, h->stream));
    enqueue_forward(h, c);
    MLP_HIP(h, hipGetLastError());
    MLP_HIP(h, hipMemcpyAsync(y + i0, h->Y, (size_t)c * sizeof(float), hipMemcpyDeviceToHost, h->stream));
  }
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  return 0;
}

// acc[i] (+)= w y[i]: the ensemble mean of crime_mlp_forward_mean
__global__ __launch_bounds__(256) void k_acc_rows(float *__restrict__ acc, const float *__restrict__ y, int n, float w,
                                                  int first)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) acc[i] = first ? w * y[i] : acc[i] + w * y[i];
}

extern "C" int crime_mlp_forward_mean(crime_mlp_t *const *hs, int nh, int64_t n, const float *x, float *y)
{
  if (!hs || nh < 1 || !hs[0]) return mlp_error(nullptr, CRIME_GH_EINVAL, "need nh >= 1 handles");
  crime_mlp *h0 = hs[0];
  if (n < 1 || !x || !y) return mlp_error(h0, CRIME_GH_EINVAL, "need n >= 1 and non-NULL x, y");
  int batch = h0->max_batch;
  for (int k = 0; k < nh; k++) {
    if (!hs[k]) return mlp_error(h0, CRIME_GH_EINVAL, "handle %d is NULL", k);
    if (hs[k]->device != h0->device) return mlp_error(h0, CRIME_GH_EINVAL, "handle %d is on another device", k);
    batch = std::min(batch, hs[k]->max_batch);
  }
  MLP_HIP(h0, hipSetDevice(h0->device));
  for (int k = 0; k < nh; k++) MLP_HIP(h0, hipStreamSynchronize(hs[k]->stream));  // no pending work on its buffers
  // every network reads the first handle's input buffer on the first handle's stream; the mean collects in
  // its target buffer (scratch outside a training step)
  hipStream_t s = h0->stream;
  const float w = 1.0f / (float)nh;
  for (int64_t i0 = 0; i0 < n; i0 += batch) {
    const int c = (int)(n - i0 < batch ? n - i0 : batch);
    MLP_HIP(h0, hipMemcpyAsync(h0->X, x + i0 * NIN, (size_t)c * NIN * sizeof(float), hipMemcpyHostToDevice, s));
    for (int k = 0; k < nh; k++) {
      enqueue_forward(hs[k], c, s, h0->X);
      hipLaunchKernelGGL(k_acc_rows, dim3((c + 255) / 256), dim3(256), 0, s, h0->T, hs[k]->Y, c, w, k == 0);
    }
    MLP_HIP(h0, hipGetLastError());
    MLP_HIP(h0, hipMemcpyAsync(y + i0, h0->T, (size_t)c * sizeof(float), hipMemcpyDeviceToHost, s));
  }
  MLP_HIP(h0, hipStreamSynchronize(s));
  return 0;
}

__global__ __launch_bounds__(256) void k_spectra(const float *__restrict__ y, int n, float scale, float *__restrict__ out)
{
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = spectrum(y[i], scale);
}

// rows [r0, r1) of the raw inputs as the network takes them: FP32, column 6 as (nu' - nu) / channel width
static void encode_rows(const double *x, int64_t r0, int64_t r1, float inv_dnu, float *out)
{
  for (int64_t r = r0; r < r1; r++, out += NIN) {
    for (int i = 0; i < NIN; i++) out[i] = (float)x[r * NIN + i];
    out[6] = (out[6] - out[5]) * inv_dnu;
  }
}

// Threads that encode the chunks of a call into the ring of slots, ENC_ROWS rows at a time in order; a chunk waits
// until its slot was given back.  Joined when it goes out of scope, however the call ends.
struct Encoders {
  static constexpr int ENC_ROWS = 4096;
  const double *x;
  int64_t n;
  int rows, slots;          // per chunk; ring
  float inv_dnu;
  float *hx;
  std::mutex mu;
  std::condition_variable cv;
  std::vector<int> left;    // blocks of each chunk not yet encoded
  int64_t next = 0;         // block to take
  int64_t open;             // chunks that may be written: [0, open)
  bool stop = false;
  std::vector<std::thread> workers;

  Encoders(const double *x_, int64_t n_, int rows_, int slots_, float inv_dnu_, float *hx_)
      : x(x_), n(n_), rows(rows_), slots(slots_), inv_dnu(inv_dnu_), hx(hx_), open(slots_)
  {
    for (int64_t c0 = 0; c0 < n; c0 += rows) left.push_back((int)((std::min(n - c0, (int64_t)rows) + ENC_ROWS - 1) / ENC_ROWS));
  }
  // encodes blocks; main: until chunk `until` is complete, else until none is left
  void work(int64_t until)
  {
    const int bpc = (rows + ENC_ROWS - 1) / ENC_ROWS;
    std::unique_lock<std::mutex> lk(mu);
    while (!stop) {
      if (until >= 0 && left[until] == 0) return;
      const int64_t c = next / bpc;
      if (c >= (int64_t)left.size() || c >= open) {
        if (until < 0 && c >= (int64_t)left.size()) return;
        cv.wait(lk);
        continue;
      }
      const int64_t b = next++ % bpc, r0 = c * rows + b * ENC_ROWS;
      const int64_t r1 = std::min(n, std::min(r0 + ENC_ROWS, (c + 1) * (int64_t)rows));
      if (r0 >= r1) continue;   // the last chunk has fewer blocks
      lk.unlock();
      encode_rows(x, r0, r1, inv_dnu, hx + ((size_t)(c % slots) * rows + (size_t)b * ENC_ROWS) * NIN);
      lk.lock();
      if (--left[c] == 0) cv.notify_all();
    }
  }
  void start(int count)
  {
    for (int i = 0; i < count; i++) {
      try {
        workers.emplace_back([this] { work(-1); });
      }
      catch (const std::exception &) {
        return;   // fewer threads: the caller encodes too
      }
    }
  }
  void give_back(int64_t chunk)
  {
    {
      std::lock_guard<std::mutex> lk(mu);
      open = chunk + 1 + slots;
    }
    cv.notify_all();
  }
  ~Encoders()
  {
    {
      std::lock_guard<std::mutex> lk(mu);
      stop = true;
    }
    cv.notify_all();
    for (std::thread &t : workers) t.join();
  }
};

// Up to PRED_REUSE rows of one network: its kernels read pinned inputs and write pinned outputs themselves, no copies
// between (256 rows: 26 us, against 42 with two copies).  The rows go in parts, so that one is encoded while the network
// runs on the one before: quarters of the call, PRED_MIN rows at least, as long as the pinned rows hold the call, then
// thirds of the pinned rows in turn (8192 rows, one workgroup for each CU; 6144 take as long).  8192 rows 47 us, 65536
// 196, 98304 287, against 66, 240 and 320 as chunks that are encoded, copied and computed; 131072 370 against 350.
// An ensemble takes up to PRED_DIRECT rows as one part, which its networks read from a device copy above PRED_MIN rows
// (three networks, 16384 rows: 128 us; in quarters 214).  The memory is the handle's from its creation unless its
// max_batch is smaller than the call (a new handle's first 5000 rows take 53 us, and 250 with memory pinned for
// them), and stays below 1 MB: from there on pinning it takes 0.4 ms more.
// Longer calls run in a ring of PRED_SLOTS chunks of PRED_ROWS rows: threads encode (one thread would take as long as
// all the rest), a second stream sends a chunk's inputs while the networks run on the one before, and outputs go
// straight to pinned memory and are handed out meanwhile.  A million rows: 1.35 ms, of which 1.3 are the kernels',
// against 7.7 with the encoding, copies and sinh of the whole call one after the other.
static int predict_impl(crime_mlp *const *hs, int nh, int64_t n, const double *x, float inv_dnu, float scale, float *y)
{
  crime_mlp *h = hs[0];
  // rows of one launch: an ensemble's networks leave their outputs in their handles' buffers
  int batch = PRED_ROWS;
  if (nh > 1)
    for (int k = 0; k < nh; k++) batch = std::min(batch, hs[k]->max_batch);
  MLP_HIP(h, hipSetDevice(h->device));
  for (int k = 1; k < nh; k++) MLP_HIP(h, hipStreamSynchronize(hs[k]->stream));  // no pending work on its buffers
  hipStream_t s = h->stream;
  // the networks on c rows of X, their spectra into Y
  auto forward = [&](int c, const float *X, float *Y) {
    if (nh == 1) {
      enqueue_forward(h, c, s, X, Y, scale);
      return;
    }
    for (int k = 0; k < nh; k++) {
      enqueue_forward(hs[k], c, s, X);
      hipLaunchKernelGGL(k_acc_rows, dim3((c + 255) / 256), dim3(256), 0, s, h->T, hs[k]->Y, c, 1.0f / (float)nh, k == 0);
    }
    hipLaunchKernelGGL(k_spectra, dim3((c + 255) / 256), dim3(256), 0, s, h->T, c, scale, Y);
  };
  if (n <= (nh == 1 ? PRED_REUSE : PRED_DIRECT)) {
    const int64_t held = std::min<int64_t>(n, PRED_DIRECT);   // rows in memory at a time
    const int rc = ensure_direct(h, (held + 63) / 64 * 64);
    if (rc) return rc;
    const int quarter = (int)((held + 4 * 64 - 1) / (4 * 64) * 64);
    const int part = nh > 1 ? batch : n > held ? PRED_DIRECT / 3 : std::max(PRED_MIN, quarter);
    const int64_t nparts = (n + part - 1) / part;
    const int64_t slots = n <= held ? nparts : std::min<int64_t>(PRED_SLOTS, held / part);
    auto count = [&](int64_t c) { return (int)std::min<int64_t>(part, n - c * part); };
    auto hand_out = [&](int64_t c) { memcpy(y + c * part, h->direct.y + c % slots * part, count(c) * sizeof(float)); };
    for (int64_t c = 0; c < nparts; c++) {
      const int64_t at = c % slots * part;
      if (c >= slots) {
        MLP_HIP(h, hipEventSynchronize(h->slot_ev[c % slots]));
        hand_out(c - slots);
      }
      const int m = count(c);
      encode_rows(x, c * part, c * part + m, inv_dnu, h->direct.x + at * NIN);
      const float *X = h->direct.x_dev + at * NIN;
      if (nh > 1 && m > PRED_MIN) {
        MLP_HIP(h, hipMemcpyAsync(h->X, h->direct.x + at * NIN, (size_t)m * NIN * sizeof(float), hipMemcpyHostToDevice, s));
        X = h->X;
      }
      forward(m, X, h->direct.y_dev + at);
      MLP_HIP(h, hipGetLastError());
      if (c + slots < nparts) MLP_HIP(h, hipEventRecord(h->slot_ev[c % slots], s));
    }
    MLP_HIP(h, hipStreamSynchronize(s));
    for (int64_t c = std::max<int64_t>(0, nparts - slots); c < nparts; c++) hand_out(c);
    return 0;
  }
  const int rows = batch;
  const int64_t nchunks = (n + rows - 1) / rows;
  const int slots = (int)std::min<int64_t>(PRED_SLOTS, nchunks);
  int rc = ensure_ring(h, (int64_t)slots * rows);
  if (rc) return rc;
  auto count = [&](int64_t c) { return (int)std::min<int64_t>(rows, n - c * rows); };
  auto hand_out = [&](int64_t c) -> int {
    MLP_HIP(h, hipEventSynchronize(h->slot_ev[c % slots]));
    memcpy(y + c * rows, h->ring.y + (size_t)(c % slots) * rows, (size_t)count(c) * sizeof(float));
    return 0;
  };
  Encoders enc(x, n, rows, slots, inv_dnu, h->ring.x);
  enc.start((int)std::min<int64_t>(PRED_THREADS, n / (2 * Encoders::ENC_ROWS)));
  int64_t out = 0;   // chunks handed out
  for (int64_t c = 0; c < nchunks && !rc; c++) {
    // a slot is given back ahead of its use, for the threads, if a later chunk has use for it
    if (c - out >= slots - 1 && out + slots < nchunks) {
      rc = hand_out(out);
      enc.give_back(out++);
      if (rc) break;
    }
    enc.work(c);
    const size_t at = (size_t)(c % slots) * rows;
    const int m = count(c);
    // the slot's device inputs were read by a chunk that is handed out
    MLP_HIP(h, hipMemcpyAsync(h->ring_dx + at * NIN, h->ring.x + at * NIN, (size_t)m * NIN * sizeof(float),
                              hipMemcpyHostToDevice, h->copy));
    MLP_HIP(h, hipEventRecord(h->slot_in[c % slots], h->copy));
    MLP_HIP(h, hipStreamWaitEvent(s, h->slot_in[c % slots], 0));
    forward(m, h->ring_dx + at * NIN, h->ring.y_dev + at);
    MLP_HIP(h, hipGetLastError());
    MLP_HIP(h, hipEventRecord(h->slot_ev[c % slots], s));
  }
  for (; out < nchunks && !rc; out++) rc = hand_out(out);
  return rc;
}

static void drain(crime_mlp *h)
{
  if (h->copy) (void)hipStreamSynchronize(h->copy);
  (void)hipStreamSynchronize(h->stream);
}

extern "C" int crime_mlp_predict(crime_mlp_t *const *hs, int nh, int64_t n, const double *x, float inv_dnu, float scale,
                                 float *y)
{
  if (!hs || nh < 1 || !hs[0]) return mlp_error(nullptr, CRIME_GH_EINVAL, "need nh >= 1 handles");
  crime_mlp *h = hs[0];
  if (n < 1 || !x || !y || !(scale > 0)) return mlp_error(h, CRIME_GH_EINVAL, "need n >= 1, non-NULL x, y and scale > 0");
  for (int k = 0; k < nh; k++) {
    if (!hs[k]) return mlp_error(h, CRIME_GH_EINVAL, "handle %d is NULL", k);
    if (hs[k]->device != h->device) return mlp_error(h, CRIME_GH_EINVAL, "handle %d is on another device", k);
  }
  try {
    const int rc = predict_impl(hs, nh, n, x, inv_dnu, scale, y);
    // nothing of a failed call may still read or write the slots
    if (rc) drain(h);
    return rc;
  }
  catch (const std::exception &e) {
    drain(h);
    return mlp_error(h, CRIME_GH_ENOMEM, "predict: %s", e.what());
  }
}

extern "C" int crime_mlp_loss_grad(crime_mlp_t *h, int n, const float *x, const float *t, const float *w,
                                   double *loss, float *grad)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (!x || !t || !loss || !grad) return mlp_error(h, CRIME_GH_EINVAL, "NULL argument");
  if (n < 64 || n > h->max_batch || n % 64)
    return mlp_error(h, CRIME_GH_EINVAL, "n %d: a multiple of 64 in [64, %d]", n, h->max_batch);
  MLP_HIP(h, hipSetDevice(h->device));
  int rc = ensure_loss(h, 1);
  if (rc) return rc;
  DevState s;
  MLP_HIP(h, hipMemcpy(&s, h->st, sizeof(s), hipMemcpyDeviceToHost));
  const int saved_local = s.local;
  s.local = 0;
  MLP_HIP(h, hipMemcpy(h->st, &s, sizeof(s), hipMemcpyHostToDevice));
  const float zero = 0.0f;
  MLP_HIP(h, hipMemcpy(h->loss, &zero, sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemcpy(h->X, x, (size_t)n * NIN * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemcpy(h->T, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  if (w) {
    MLP_HIP(h, hipMemcpy(h->Wt, w, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  } else {
    std::vector<float> ones((size_t)n, 1.0f);
    MLP_HIP(h, hipMemcpy(h->Wt, ones.data(), (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  }
  enqueue_rows(h, n, false);
  enqueue_update(h, n, h->grad);
  MLP_HIP(h, hipGetLastError());
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  float l = 0;
  MLP_HIP(h, hipMemcpy(&l, h->loss, sizeof(float), hipMemcpyDeviceToHost));
  MLP_HIP(h, hipMemcpy(grad, h->grad, NPARAM * sizeof(float), hipMemcpyDeviceToHost));
  s.local = saved_local;
  MLP_HIP(h, hipMemcpy(h->st, &s, sizeof(s), hipMemcpyHostToDevice));
  *loss = l;
  return 0;
}

extern "C" int crime_mlp_set_data(crime_mlp_t *h, int64_t n, const float *x, const float *t, const float *w)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (n < 1 || n > ((int64_t)1 << 40) || !x || !t) return mlp_error(h, CRIME_GH_EINVAL, "bad training set");
  MLP_HIP(h, hipSetDevice(h->device));
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  drop_graph(h);
  if (h->Xall) MLP_HIP(h, hipFree(h->Xall));
  if (h->Tall) MLP_HIP(h, hipFree(h->Tall));
  if (h->Wall) MLP_HIP(h, hipFree(h->Wall));
  h->Xall = h->Tall = h->Wall = nullptr;
  h->ndata = 0;
  MLP_HIP(h, hipMalloc((void **)&h->Xall, (size_t)n * NIN * sizeof(float)));
  MLP_HIP(h, hipMalloc((void **)&h->Tall, (size_t)n * sizeof(float)));
  MLP_HIP(h, hipMemcpy(h->Xall, x, (size_t)n * NIN * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemcpy(h->Tall, t, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMalloc((void **)&h->Wall, (size_t)n * sizeof(float)));
  if (w) {
    MLP_HIP(h, hipMemcpy(h->Wall, w, (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  } else {
    std::vector<float> ones((size_t)n, 1.0f);
    MLP_HIP(h, hipMemcpy(h->Wall, ones.data(), (size_t)n * sizeof(float), hipMemcpyHostToDevice));
  }
  h->ndata = n;
  return 0;
}

// counts[0]: floats whose BF16 SiLU (a group of four of it) is not that of z sigm(z); counts[1]: whose sigm is not
// the plain quotient; NaNs are equal to each other.  A workgroup takes 2^16 bit patterns.
__global__ __launch_bounds__(256) void k_silu_check(unsigned long long *__restrict__ counts)
{
  unsigned silu = 0, quot = 0;
  for (int i = 0; i < 256; i++) {
    const float z = __uint_as_float(blockIdx.x * 65536u + i * 256u + threadIdx.x);
    const float zz[4] = {z, z, z, z};
    const uint2 a = silu4_bf16(zz);
    const float s = sigm(z), q = 1.0f / (1.0f + expf(-z));
    const float x = bf2f((uint16_t)a.x), y = bf2f(f2bf(z * q));
    silu += !(x == y || (x != x && y != y)) || a.x != a.y || (a.x >> 16) != (a.x & 0xffffu);
    quot += !(__float_as_uint(s) == __float_as_uint(q) || (s != s && q != q));
  }
  if (silu) atomicAdd(counts, (unsigned long long)silu);
  if (quot) atomicAdd(counts + 1, (unsigned long long)quot);
}

extern "C" int crime_mlp_silu_check(crime_mlp_t *h, int64_t *counts)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (!counts) return mlp_error(h, CRIME_GH_EINVAL, "counts is NULL");
  MLP_HIP(h, hipSetDevice(h->device));
  unsigned long long zero[2] = {0, 0}, got[2], *d = (unsigned long long *)h->grad;   // scratch outside a loss_grad
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  MLP_HIP(h, hipMemcpy(d, zero, sizeof(zero), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(k_silu_check, dim3(65536), dim3(256), 0, h->stream, d);
  MLP_HIP(h, hipGetLastError());
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  MLP_HIP(h, hipMemcpy(got, d, sizeof(got), hipMemcpyDeviceToHost));
  counts[0] = (int64_t)got[0];
  counts[1] = (int64_t)got[1];
  return 0;
}

extern "C" int crime_mlp_set_graph(crime_mlp_t *h, int on)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  h->use_graph = on ? 1 : 0;
  return 0;
}

extern "C" int crime_mlp_train(crime_mlp_t *h, int steps, int batch, float lr0, int total_steps, float beta1,
                               float beta2, float eps, uint32_t seed, float *loss_out)
{
  if (!h) return mlp_error(nullptr, CRIME_GH_EINVAL, "handle is NULL");
  if (!h->ndata) return mlp_error(h, CRIME_GH_ESTATE, "train before set_data");
  if (steps < 1 || batch < 64 || batch > h->max_batch || batch % 64)
    return mlp_error(h, CRIME_GH_EINVAL, "steps %d, batch %d (a multiple of 64 <= %d)", steps, batch, h->max_batch);
  if (!(lr0 > 0) || total_steps < 1 || !(beta1 >= 0 && beta1 < 1) || !(beta2 >= 0 && beta2 < 1) || !(eps > 0))
    return mlp_error(h, CRIME_GH_EINVAL, "bad Adam hyper-parameters");
  MLP_HIP(h, hipSetDevice(h->device));
  int rc = ensure_loss(h, steps);
  if (rc) return rc;
  DevState s;
  MLP_HIP(h, hipMemcpy(&s, h->st, sizeof(s), hipMemcpyDeviceToHost));
  s.local = 0;
  s.total = total_steps;
  s.lr0 = lr0;
  s.b1 = beta1;
  s.b2 = beta2;
  s.eps = eps;
  s.seed = seed;
  s.ndata = h->ndata;
  MLP_HIP(h, hipMemcpy(h->st, &s, sizeof(s), hipMemcpyHostToDevice));
  MLP_HIP(h, hipMemset(h->loss, 0, (size_t)steps * sizeof(float)));
  if (!h->use_graph) {
    for (int i = 0; i < steps; i++) {
      enqueue_rows(h, batch, true);
      enqueue_update(h, batch, nullptr);
      MLP_HIP(h, hipGetLastError());
    }
    MLP_HIP(h, hipStreamSynchronize(h->stream));
    if (loss_out) MLP_HIP(h, hipMemcpy(loss_out, h->loss, (size_t)steps * sizeof(float), hipMemcpyDeviceToHost));
    return 0;
  }
  if (h->exec && h->graph_batch != batch) drop_graph(h);
  if (!h->exec) {
    MLP_HIP(h, hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
    enqueue_rows(h, batch, true);
    enqueue_update(h, batch, nullptr);
    hipError_t e = hipStreamEndCapture(h->stream, &h->graph);
    if (e != hipSuccess) {
      h->graph = nullptr;
      return mlp_error(h, CRIME_GH_EHIP, "step capture: %s", hipGetErrorString(e));
    }
    MLP_HIP(h, hipGraphInstantiate(&h->exec, h->graph, nullptr, nullptr, 0));
    h->graph_batch = batch;
  }
  for (int i = 0; i < steps; i++) MLP_HIP(h, hipGraphLaunch(h->exec, h->stream));
  MLP_HIP(h, hipStreamSynchronize(h->stream));
  if (loss_out) MLP_HIP(h, hipMemcpy(loss_out, h->loss, (size_t)steps * sizeof(float), hipMemcpyDeviceToHost));
  return 0;
}
