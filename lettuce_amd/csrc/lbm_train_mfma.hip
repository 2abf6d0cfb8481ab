// FP32 training kernels of the learned collision with the MLP on the FP32
// matrix instructions (v_mfma_f32_32x32x2_f32, FP32 products and sums): the
// forward step, and the adjoint fused with the parameter gradient.
//
// A wave owns 64 cells, one per lane, for the lattice arithmetic
// (lbm_train_cell.h).  The MLP runs on them as two blocks of 32 cells, one
// after the other, each layer as H^T = W X^T with the cells as columns: item r
// of lane l then holds unit unit(r, l / 32) of cell l % 32, which is the B
// operand of the next layer as it stands once that layer's K index is taken in
// the order of the items (step r contracts units unit(r, 0) and unit(r, 1)).
// So no layer moves data between lanes.  Layer 3 (3 rows) and its transposes,
// which would leave 29 of 32 rows idle, stay on the VALU, each half of the wave
// over its 16 units and the two halves added.
//
// The gradient of a layer's weights is a product over the cells, so its
// operands need the cells along K: the wave turns dz and a around through LDS
// (lane = unit, items = cells).  dW2 and [dW1, db1] accumulate in registers over
// all cells of the wave (persistent blocks), dW3 and the other biases in the
// lanes that hold them; a block writes one vector of partial sums, which
// grad_sum_kernel adds in block order.  The per-cell record of
// lbm_learned_train_backward (137 values, written and read back once per step)
// is not needed.
//
// Bound by issue: FP32 products on the matrix cores and the VALU's work (64
// SiLUs and their derivatives, the lattice) take about equal shares and hardly
// overlap at two waves per SIMD (VALU 42 %, MFMA 39 % of the adjoint's cycles).
// D2Q9, 2.1 M cells, before (one thread per cell on the VALU, the record, its
// reduction) and now: forward 168 / 105 us, adjoint and gradient 1000 / 289 us.
// The first layer's gradient on a 32-wide product, mostly padding, took 23 us
// more.
#include "lbm_train_mfma.h"

#include <algorithm>

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace lbm {

namespace {

constexpr int TM_WAVES = 4;
constexpr int TM_PITCH = 36;  // LDS rows of 32 floats: 16-byte aligned, conflict-free b128 reads
static_assert(TM_PITCH % 4 == 0 && HID % 4 == 0, "rows read as float4");

// unit held by item r of half h, in groups of four consecutive units
__device__ constexpr int unit(int r, int h) { return 8 * (r / 4) + 4 * h + r % 4; }

// both are read as float4: 16-byte aligned by declaration
struct alignas(16) WeightsLds {
  float w2[HID][TM_PITCH];   // W2 rows
  float w2t[HID][TM_PITCH];  // W2 columns
  float w1t[6][HID];         // W1 columns
  float w3[3][HID];
  float b1[HID], b2[HID], b3[4];
};
// a wave's turned operands; x rows 6 and 7 hold ones and zeros
struct alignas(16) TurnLds {
  float a1[HID][TM_PITCH], dz[HID][TM_PITCH], x[8][2 * TM_PITCH];
};

// The MLP runs in the log2 domain: an item holds t = -log2(e) z of its
// pre-activation z (the factor enters with the inputs and the biases), so
// 2^t = exp(-z) and t / (1 + 2^t) = -log2(e) silu(z) is the next layer's input
// in the same domain.  W2 and W3 take no factor; the output and the weight
// gradients, sums over such activations, take -ln(2).
constexpr float LOG2E = 1.44269504f, LN2 = 0.693147182f;

__device__ __forceinline__ void stage_weights(const float* P, WeightsLds& w) {
  for (int i = threadIdx.x; i < HID * HID; i += blockDim.x) {
    const float v = P[P_W2 + i];
    w.w2[i / HID][i % HID] = v;
    w.w2t[i % HID][i / HID] = v;
  }
  for (int i = threadIdx.x; i < HID * 6; i += blockDim.x) w.w1t[i % 6][i / 6] = P[P_W1 + i];
  for (int i = threadIdx.x; i < HID * 3; i += blockDim.x) w.w3[i / HID][i % HID] = P[P_W3 + i];
  for (int i = threadIdx.x; i < HID; i += blockDim.x) {
    w.b1[i] = -LOG2E * P[P_B1 + i];
    w.b2[i] = -LOG2E * P[P_B2 + i];
    if (i < 3) w.b3[i] = P[P_B3 + i];
  }
  __syncthreads();
}

// 16 floats in groups of four: p[8 q + 4 h + i] as item 4 q + i
__device__ __forceinline__ f32x16 items(const float* p, int h) {
  f32x16 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 t = *(const float4*)(p + 8 * q + 4 * h);
    v[4 * q] = t.x;
    v[4 * q + 1] = t.y;
    v[4 * q + 2] = t.z;
    v[4 * q + 3] = t.w;
  }
  return v;
}
// 16 consecutive floats
__device__ __forceinline__ f32x16 run16(const float* p) {
  f32x16 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float4 t = *(const float4*)(p + 4 * q);
    v[4 * q] = t.x;
    v[4 * q + 1] = t.y;
    v[4 * q + 2] = t.z;
    v[4 * q + 3] = t.w;
  }
  return v;
}

__device__ __forceinline__ void run8(const float* p, float (&v)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const float4 t = *(const float4*)(p + 4 * q);
    v[4 * q] = t.x;
    v[4 * q + 1] = t.y;
    v[4 * q + 2] = t.z;
    v[4 * q + 3] = t.w;
  }
}

// the upper half of a changes places with the lower half of b
__device__ __forceinline__ void swap_halves(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
// v of the cell in both halves, for the cells of block blk (lanes 32 blk ..)
__device__ __forceinline__ float of_block(float v, int blk) {
  float w = v;
  swap_halves(v, w);
  return blk ? w : v;
}
// the sum of v over the two halves, in both
__device__ __forceinline__ float add_halves(float v) {
  float w = v;
  swap_halves(v, w);
  return v + w;
}

// t <- t s, s = 1 / (1 + 2^t) by v_rcp_f32 and a Newton step (t is held below
// 126 there, where s < 2^-125, so that the step sees finite numbers);
// ds <- silu'(z) = s + z s (1 - s)
__device__ __forceinline__ void activate(f32x16& t, f32x16& ds) {
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const float d = 1.0f + __builtin_amdgcn_exp2f(__builtin_amdgcn_fmed3f(t[r], -126.f, 126.f));
    const float q = __builtin_amdgcn_rcpf(d);
    const float s = __builtin_fmaf(q, __builtin_fmaf(-d, q, 1.0f), q);
    t[r] *= s;
    const float a = -LN2 * t[r];
    ds[r] = __builtin_fmaf(-a, s, s + a);
  }
}

__device__ __forceinline__ f32x16 mfma16(const f32x16& a, const f32x16& b, f32x16 c) {
#pragma unroll
  for (int r = 0; r < 16; ++r) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[r], b[r], c, 0, 0, 0);
  return c;
}

// Phases of a block's MLP: memory operations and the schedule stay within one.
// Left alone, the compiler hoists the weights' LDS reads out of the loop over
// tiles and ahead of each other, which spills 259 registers.
__device__ __forceinline__ void phase() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// the MLP of the 32 cells of a block, up to the second layer's activations:
// xb the layer 1 operand, w1a its weights; a1, ds1, a2, ds2 in item layout
__device__ __forceinline__ void layers(const WeightsLds& w, const float (&w1a)[3],
                                       const float (&xb)[3], int h, int row, f32x16& a1, f32x16& ds1,
                                       f32x16& a2, f32x16& ds2) {
  a1 = items(w.b1, h);
#pragma unroll
  for (int j = 0; j < 3; ++j) a1 = __builtin_amdgcn_mfma_f32_32x32x2f32(w1a[j], xb[j], a1, 0, 0, 0);
  activate(a1, ds1);
  phase();
  a2 = mfma16(items(w.w2[row], h), a1, items(w.b2, h));
  phase();
  activate(a2, ds2);
  phase();
}

// raw rates 1/tau + W3 a2 + b3 of the block's cells, in both halves
__device__ __forceinline__ void rates(const WeightsLds& w, const f32x16& a2, float tau_inv, int h,
                                      float (&raw)[3]) {
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    phase();
    const f32x16 w3 = items(w.w3[k], h);
    float o = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) o = __builtin_fmaf(w3[r], a2[r], o);
    raw[k] = tau_inv + __builtin_fmaf(-LN2, add_halves(o), w.b3[k]);
  }
}

// layer 1 operands of the two blocks from the inputs of the lanes' own cells
__device__ __forceinline__ void block_inputs(const float (&x)[6], float (&xb)[2][3]) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    xb[0][j] = -LOG2E * x[2 * j];
    xb[1][j] = -LOG2E * x[2 * j + 1];
    swap_halves(xb[0][j], xb[1][j]);
  }
}

__device__ __forceinline__ void cell_tables32(const KParams& p, uint32_t c, int (&a0)[3],
                                              int (&a1)[3], int (&a2)[3]) {
  const uint32_t r = c / (uint32_t)p.n2;
  const int i2 = (int)(c - r * (uint32_t)p.n2), i0 = (int)(r / (uint32_t)p.n1);
  const int i1 = (int)(r - (uint32_t)i0 * (uint32_t)p.n1);
  axis_offsets(i0, p.n0, (int)p.s0, a0);  // fewer than 2^31 populations
  axis_offsets(i1, p.n1, p.s1, a1);
  axis_offsets(i2, p.n2, 1, a2);
}

// the pulled populations of a lane's cell; lanes past the last cell take the
// weights of a cell at rest, whose MLP inputs are finite
template <class S>
__device__ __forceinline__ void pull(const KParams& p, bool valid, const int (&a0)[3],
                                     const int (&a1)[3], const int (&a2)[3], float (&g)[S::Q]) {
  const float* fin = (const float*)p.fin;
#pragma unroll
  for (int q = 0; q < S::Q; ++q)
    g[q] = elem(fin + q * p.sq, (uint32_t)nb_offset<S>(q, -1, a0, a1, a2));
  if (!valid) {
#pragma unroll
    for (int q = 0; q < S::Q; ++q) g[q] = (float)S::w[q];
  }
}

}  // namespace

template <class S>
__global__ void __launch_bounds__(64 * TM_WAVES, 2)
    train_forward_mfma(const KParams p, const TrainArgs t, int tiles) {
  __shared__ WeightsLds w;
  stage_weights((const float*)t.params, w);
  const int lane = threadIdx.x & 63, h = lane >> 5, row = lane & 31;
  const float tau_inv = (float)p.tau_inv, s = (float)t.in_scale;
  const float lo = (float)t.rate_lo, hi = (float)t.rate_hi;
  float w1a[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) w1a[j] = w.w1t[2 * j + h][row];
  const uint32_t cells = (uint32_t)p.ncells;
  const int first = __builtin_amdgcn_readfirstlane(blockIdx.x * TM_WAVES + (threadIdx.x >> 6));
  for (int tile = first; tile < tiles; tile += gridDim.x * TM_WAVES) {
    const uint32_t c = (uint32_t)tile * 64u + lane;
    const bool valid = c < cells;
    int a0[3], a1[3], a2[3];
    cell_tables32(p, valid ? c : cells - 1, a0, a1, a2);
    float g[S::Q];
    pull<S>(p, valid, a0, a1, a2, g);
    CellFwd<S, float> F;
    features(g, s, F);
    float xb[2][3], r[3];
    block_inputs(F.x, xb);
#pragma unroll
    for (int blk = 0; blk < 2; ++blk) {
      f32x16 h1, d1, h2, d2;
      float raw[3];
      layers(w, w1a, xb[blk], h, row, h1, d1, h2, d2);
      rates(w, h2, tau_inv, h, raw);
#pragma unroll
      for (int k = 0; k < 3; ++k)
        if (blk == 0 || h == 1) r[k] = raw[k] < lo ? lo : (raw[k] > hi ? hi : raw[k]);
    }
    float out[S::Q];
    update(g, F, r, tau_inv, out);
    if (valid) {
      float* fout = (float*)p.fout;
      const uint32_t cell = (uint32_t)(a0[1] + a1[1] + a2[1]);
#pragma unroll
      for (int q = 0; q < S::Q; ++q) *elem_ptr(fout + q * p.sq, cell) = out[q];
    }
  }
}

// mu = (d step / d f)^T lam, and part[block] = the block's sum of the
// parameter gradient; lam as in train_backward_kernel
template <class S>
__global__ void __launch_bounds__(64 * TM_WAVES, 2)
    train_backward_mfma(const KParams p, const TrainArgs t, const float* __restrict__ lam_in,
                        int gathered, float* __restrict__ mu_out, float* __restrict__ part,
                        int tiles) {
  __shared__ WeightsLds w;
  __shared__ TurnLds turn[TM_WAVES];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = lane >> 5, row = lane & 31;
  TurnLds& T = turn[wave];
  for (int i = lane; i < 2 * TM_PITCH; i += 64) {
    T.x[6][i] = 1.0f;
    T.x[7][i] = 0.0f;
  }
  stage_weights((const float*)t.params, w);
  const float tau_inv = (float)p.tau_inv, s = (float)t.in_scale;
  const float lo = (float)t.rate_lo, hi = (float)t.rate_hi;
  float w1a[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) w1a[j] = w.w1t[2 * j + h][row];
  f32x16 g2 = {}, gb2 = {}, g3[3] = {};
  f32x4 g1[2] = {};
  float gb3[3] = {};
  const uint32_t cells = (uint32_t)p.ncells;
  const int first = __builtin_amdgcn_readfirstlane(blockIdx.x * TM_WAVES + wave);
  for (int tile = first; tile < tiles; tile += gridDim.x * TM_WAVES) {
    const uint32_t c = (uint32_t)tile * 64u + lane;
    const bool valid = c < cells;
    int a0[3], a1[3], a2[3];
    cell_tables32(p, valid ? c : cells - 1, a0, a1, a2);
    float g[S::Q], lam[S::Q];
    pull<S>(p, valid, a0, a1, a2, g);
    const uint32_t cell = (uint32_t)(a0[1] + a1[1] + a2[1]);
#pragma unroll
    for (int q = 0; q < S::Q; ++q)
      lam[q] = elem(lam_in + q * p.sq,
                    gathered ? (uint32_t)nb_offset<S>(q, +1, a0, a1, a2) : cell);
    CellFwd<S, float> F;
    CellAdj<S, float> A;
    float dr[3], r[3], gx[6];
    features(g, s, F);
    adjoint_rates(lam, F, A, dr);
    if (!valid) dr[0] = dr[1] = dr[2] = 0.f;  // no part in the gradient
    float xb[2][3];
    block_inputs(F.x, xb);
#pragma unroll
    for (int k = 0; k < 6; ++k) T.x[k][lane + (lane & 32 ? TM_PITCH - 32 : 0)] = F.x[k];
#pragma unroll 1
    for (int blk = 0; blk < 2; ++blk) {
      f32x16 h1, d1, h2, d2;
      float raw[3], go[3];
      const float xo[3] = {blk ? xb[1][0] : xb[0][0], blk ? xb[1][1] : xb[0][1],
                           blk ? xb[1][2] : xb[0][2]};
      layers(w, w1a, xo, h, row, h1, d1, h2, d2);
#pragma unroll
      for (int i = 0; i < 16; ++i) T.a1[unit(i, h)][row] = h1[i];
      phase();
      rates(w, h2, tau_inv, h, raw);
      f32x16 dz = {};
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const float q = of_block(dr[k], blk);
        go[k] = raw[k] >= lo && raw[k] <= hi ? q : 0.f;
        if (h == blk) r[k] = raw[k] < lo ? lo : (raw[k] > hi ? hi : raw[k]);
        gb3[k] += go[k];
        phase();
        const f32x16 w3 = items(w.w3[k], h);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          g3[k][i] = __builtin_fmaf(go[k], h2[i], g3[k][i]);
          dz[i] = __builtin_fmaf(w3[i], go[k], dz[i]);
        }
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        dz[i] *= d2[i];
        gb2[i] += dz[i];
        T.dz[unit(i, h)][row] = dz[i];
      }
      phase();
      f32x16 dz1 = {};
      dz1 = mfma16(items(w.w2t[row], h), dz, dz1);
      phase();
      // K runs over the block's cells: half h takes cells 16 h ..
      g2 = mfma16(run16(&T.dz[row][16 * h]), run16(&T.a1[row][16 * h]), g2);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        dz1[i] *= d1[i];
        T.dz[unit(i, h)][row] = dz1[i];
      }
      phase();
      // 7 columns: two products of 16 rows, each quarter of the wave 8 cells
      {
        const int quarter = lane >> 4, col = lane & 15;
        float xs[8];
        run8(&T.x[min(col, 7)][TM_PITCH * blk + 8 * quarter], xs);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          float dzs[8];
          run8(&T.dz[16 * half + col][8 * quarter], dzs);
#pragma unroll
          for (int i = 0; i < 8; ++i)
            g1[half] = __builtin_amdgcn_mfma_f32_16x16x4f32(dzs[i], xs[i], g1[half], 0, 0, 0);
        }
      }
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        phase();
        const f32x16 w1 = items(w.w1t[k], h);
        float v = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) v = __builtin_fmaf(w1[i], dz1[i], v);
        v = add_halves(v);
        if (h == blk) gx[k] = v;
      }
    }
    float mu[S::Q];
    adjoint(lam, F, A, r, gx, tau_inv, s, mu);
    if (valid) {
#pragma unroll
      for (int q = 0; q < S::Q; ++q) *elem_ptr(mu_out + q * p.sq, cell) = mu[q];
    }
  }

  // the lanes' sums over their cells, all waves at once, then the block's over
  // its waves, one after the other (with the lanes' sums in that loop, a launch
  // on 64 cells took 64 us, 28 so)
  auto over_cells = [](float v) {
    for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
  };
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    gb2[i] = over_cells(gb2[i]);
#pragma unroll
    for (int j = 0; j < 3; ++j) g3[j][i] = over_cells(g3[j][i]);
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) gb3[j] = over_cells(gb3[j]);
  __syncthreads();
  float* red = (float*)turn;
  for (int k = 0; k < TM_WAVES; ++k) {
    auto add = [&](int e, float v) { red[e] = k == 0 ? v : red[e] + v; };
    if (wave == k) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int u = unit(i, h);
        add(P_W2 + u * HID + row, -LN2 * g2[i]);
        if (row == 0) {
          add(P_B2 + u, gb2[i]);
#pragma unroll
          for (int j = 0; j < 3; ++j) add(P_W3 + j * HID + u, -LN2 * g3[j][i]);
        }
      }
      // item i of quarter k of a 16 x 16 product: row 4 k + i, column lane % 16
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int u = 16 * (i / 4) + 4 * (lane >> 4) + i % 4, col = lane & 15;
        if (col < 6) add(P_W1 + u * 6 + col, g1[i / 4][i % 4]);
        if (col == 6) add(P_B1 + u, g1[i / 4][i % 4]);
      }
#pragma unroll
      for (int j = 0; j < 3; ++j)
        if (lane == 0) add(P_B3 + j, gb3[j]);
    }
    __syncthreads();
  }
  for (int e = threadIdx.x; e < NPARAM; e += blockDim.x)
    part[(int64_t)blockIdx.x * NPARAM + e] = red[e];
}
static_assert(alignof(WeightsLds) == 16 && alignof(TurnLds) == 16, "float4 reads");
static_assert(sizeof(TurnLds) * TM_WAVES >= NPARAM * sizeof(float), "reduction area");

namespace {
int tiles_of(int64_t cells) { return (int)((cells + 63) / 64); }
}  // namespace

// two blocks per CU fit (LDS, registers); a wave sums at least one tile, and at
// most 32, 2048 cells in one FP32 sum whatever the size, as the partial sums of
// lbm_learned_grad_reduce
int train_mfma_blocks(int64_t cells) {
  const int64_t rounds = (cells + 64 * TM_WAVES - 1) / (64 * TM_WAVES);  // a tile per wave
  return (int)(rounds < 512 ? rounds : std::max<int64_t>(512, (rounds + 31) / 32));
}

void launch_train_forward_mfma(int32_t stencil, const KParams& p, const TrainArgs& t, hipStream_t s) {
  const int tiles = tiles_of(p.ncells);
  // four waves per SIMD fit
  const dim3 grid(std::min((tiles + TM_WAVES - 1) / TM_WAVES, 1024)), block(64 * TM_WAVES);
  if (stencil == LBM_D2Q9) hipLaunchKernelGGL(train_forward_mfma<D2Q9>, grid, block, 0, s, p, t, tiles);
  else hipLaunchKernelGGL(train_forward_mfma<D3Q27>, grid, block, 0, s, p, t, tiles);
}

void launch_train_backward_mfma(int32_t stencil, const KParams& p, const TrainArgs& t, const float* lam,
                                int gathered, float* mu, float* part, hipStream_t s) {
  const int tiles = tiles_of(p.ncells);
  const dim3 grid(train_mfma_blocks(p.ncells)), block(64 * TM_WAVES);
  if (stencil == LBM_D2Q9)
    hipLaunchKernelGGL(train_backward_mfma<D2Q9>, grid, block, 0, s, p, t, lam, gathered, mu, part, tiles);
  else
    hipLaunchKernelGGL(train_backward_mfma<D3Q27>, grid, block, 0, s, p, t, lam, gathered, mu, part, tiles);
}

}  // namespace lbm
