// Several fused steps per launch for 2D lattices (D2Q9), any extents,
// periodic or with a cell-class map: f_out = K^n(f_in), K the pull step of
// step_kernel, n up to kTile2dMaxSteps.
//
// Small 2D grids are bound by launches, not by work: a single step of 128^2
// to 250 x 187 cells takes 3 to 4.4 us on MI355X whatever it computes (so:
// 128^2 BGK FP32 1.5 us, 251 x 187 TRT FP64 2.0 us, a 250 x 125 channel 2.5 us
// per step, bound by each stage's chain of LDS reads, arithmetic and barrier: the
// VALU is busy 15 to 26 % of a launch).
// Here a block owns a tile of t1 x t2 cells and computes step s (s = 1 .. n) on
// the tile plus reach * (n - s) cells on each side, so it needs nothing from other
// blocks until the launch ends; the first step reads the input, the last one
// writes the output, and the populations between them stay in LDS (two
// buffers, one barrier per step), rounded to the storage format as a stored
// step rounds them.  The overlap is computed more than once, which costs
// nothing while the chip is mostly idle; the host weighs it (tile2d_choice).
//
// reach is 1 on periodic grids.  With a class map it is 2: an outlet cell
// gathers its neighbour x - dir, which itself pulls from one cell further.
//
// A run of n steps in lettuce's default order (collide, then stream) is n + 1
// stages: collide, n - 1 times stream and collide, stream.  The first stage of
// its first launch only collides (lead), the last one of its last launch only
// streams (trail).
//
// Rows of the grid wrap periodically, so the halo of a tile at the edge holds
// the cells of the opposite edge (the host keeps the halo within the extents:
// one wrap suffices).
#include "lbm_pull2d.h"
#include "lbm_tile2d.h"

namespace lbm {

// FP64 cells need more registers than 1024 threads leave
template <class ST>
constexpr int tile2d_max_threads() {
  return sizeof(typename ST::C) == 8 ? 512 : 1024;
}

// What a region cell of a masked grid does, worked out once per launch: bits
// 0-8 the populations bounced back from a solid source, 9-17 those not
// streamed, 18-21 the operator, 22-29 the class id.
constexpr uint32_t kTileRules = (1u << 18) - 1;
__device__ __forceinline__ uint32_t tile_op(uint32_t info) { return (info >> 18) & 15u; }
__device__ __forceinline__ uint32_t tile_class(uint32_t info) { return (info >> 22) & 255u; }

template <class S, class ST, int COLL, bool MASK>
__global__ void __launch_bounds__(tile2d_max_threads<ST>()) tile2d_kernel(const Tile2dParams P) {
  using C = typename ST::C;
  using T = typename ST::T;
  constexpr int Q = S::Q;
  extern __shared__ __align__(16) unsigned char tile2d_lds[];
  __shared__ lbm_cell_class ctl[MASK ? 256 : 1];
  const KParams& p = P.k;
  // the first step's region: the tile plus the halo m on each side; cells of
  // every later region are addressed in it
  const int m = P.reach * (P.steps - 1);
  const int W1 = P.t1 + 2 * m, W2 = P.t2 + 2 * m, cap = W1 * W2;
  uint32_t* info = (uint32_t*)tile2d_lds;                     // [cap], masked
  T* bufs = (T*)(tile2d_lds + (MASK ? 4 * ((cap + 1) & ~1) : 0));  // [2][Q][cap]
  if constexpr (MASK) {
    stage_classes(p, ctl);
    __syncthreads();
  }

  const int b1 = blockIdx.x / P.nt2, b2 = blockIdx.x - b1 * P.nt2;
  const int x0 = b1 * P.t1 - m, y0 = b2 * P.t2 - m;  // the region's first cell (unwrapped)
  const CollParams<C> cp = coll_params<C>(p);
  long long a0[3];
  axis_offsets(0, 1, 0LL, a0);  // the grid's single i0 plane
  KParams ps = p;               // the last step's store
  const bool lead = P.lead != 0;

  auto decode = [&](const T(&raw)[Q], C(&g)[Q]) {
#pragma unroll
    for (int q = 0; q < Q; ++q) g[q] = ST::dec(raw[q], shift_of<ST>(S::w[q], p));
  };
  // the pull from the input of grid cell (g1, g2) as stored, in two rounds of
  // loads with a class map (ids, then the populations they select); own: the
  // cell's own populations instead; returns its rules
  auto input_pull = [&](int g1, int g2, bool own, T(&raw)[Q]) {
    int a1[3], a2[3];
    axis_offsets(g1, p.n1, p.s1, a1);
    axis_offsets(g2, p.n2, 1, a2);
    const T* fin = (const T*)p.fin;
    uint32_t rules = 0;
    if constexpr (MASK) {
      PullIds<S> ids;
      const int cell = a1[1] + a2[1];
      load_pull_ids<S, MASK>(p, cell, a1, a2, ids);
      const lbm_cell_class& K = ctl[ids.c0];
      const bool near =
          (K.flags & (LBM_CLASS_NEAR_SOLID | LBM_CLASS_SOLID)) == LBM_CLASS_NEAR_SOLID;
      rules = (K.no_stream & 511u) << 9 | (uint32_t)K.op << 18 | ids.c0 << 22;
      if (near) {
#pragma unroll
        for (int q = 1; q < Q; ++q)
          rules |= (ctl[ids.src[q]].flags & LBM_CLASS_SOLID) ? 1u << q : 0u;
      }
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const bool bounce = (rules >> q) & 1u, keep = (rules >> (9 + q)) & 1u;
        const uint32_t at =
            (uint32_t)(own || bounce || keep ? cell : nb_in_plane<S>(q, -1, a1, a2));
        raw[q] = elem(fin, (uint32_t)(bounce && !own ? S::opp[q] : q) * (uint32_t)p.sq + at);
      }
    } else {
#pragma unroll
      for (int q = 0; q < Q; ++q)
        raw[q] = elem(fin + q * p.sq,
                      (uint32_t)(own ? a1[1] + a2[1] : nb_in_plane<S>(q, -1, a1, a2)));
    }
    return rules;
  };
  // the same of region cell r from the region buffer src of the step before
  auto region_pull = [&](const T* src, int r, uint32_t rules, T(&raw)[Q]) {
    if (!MASK || !__any((rules & kTileRules) != 0)) {
#pragma unroll
      for (int q = 0; q < Q; ++q) raw[q] = src[q * cap + r - go<S>(q, 1) * W2 - go<S>(q, 2)];
    } else {
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const bool bounce = (rules >> q) & 1u, keep = (rules >> (9 + q)) & 1u;
        raw[q] = src[(bounce ? S::opp[q] : q) * cap +
                     (bounce || keep ? r : r - go<S>(q, 1) * W2 - go<S>(q, 2))];
      }
    }
  };

  for (int s = 0; s < P.steps; ++s) {
    const int o = P.reach * s;
    const int w1 = W1 - 2 * o, w2 = W2 - 2 * o, n = w1 * w2;
    const float inv = 1.0f / (float)w2;
    const bool last = s + 1 == P.steps;
    const T* src = bufs + ((s + 1) & 1) * Q * cap;
    T* dst = bufs + (s & 1) * Q * cap;
    const uint32_t key = ST::stochastic ? sr_step_key(p.sr_seed, p.sr_step + (uint32_t)s) : 0u;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
      // i / w2 exactly: i + 1/2 is at least 1/2 away from a multiple of w2,
      // far more than the rounding of its product with 1 / w2 (i < 2^16)
      const int k1 = (int)(((float)i + 0.5f) * inv);
      const int r1 = o + k1, r2 = o + i - k1 * w2;
      const int r = r1 * W2 + r2;
      const int g1 = wrap(x0 + r1, p.n1), g2 = wrap(y0 + r2, p.n2);
      const int cell = g1 * p.s1 + g2;
      // tiles at the grid's end may reach past it: those cells are the first
      // ones of the opposite edge, which another tile stores
      const bool stored = x0 + r1 < p.n1 && y0 + r2 < p.n2;
      uint32_t rules = 0;
      T raw[Q];
      if (s == 0) {
        rules = input_pull(g1, g2, lead, raw);
        if (MASK) info[r] = rules;
      } else {
        if (MASK) rules = info[r];
        region_pull(src, r, rules, raw);
      }
      if (last && P.trail) {
        // streamed as stored: nothing is decoded or rounded again
        if (stored) {
          T* fout = (T*)p.fout;
#pragma unroll
          for (int q = 0; q < Q; ++q)
            __builtin_nontemporal_store(raw[q], elem_ptr(fout + q * p.sq, (uint32_t)cell));
        }
        continue;
      }
      C f[Q];
      decode(raw, f);
      const uint32_t op = MASK ? tile_op(rules) : (uint32_t)LBM_OP_COLLIDE;
      if (!MASK || op == LBM_OP_COLLIDE) {
        collide<S, C, COLL>(f, cp);
      } else {
        const lbm_cell_class& mine = ctl[tile_class(rules)];
        apply_boundary_op_nb<S, ST>(
            p, op, mine.flags, cell, f, [&]() -> const lbm_cell_class& { return mine; },
            [&](const lbm_cell_class& K, C(&g)[Q]) {
              T rn[Q];
              if (s == 0) {
                input_pull(wrap(g1 - K.dir[1], p.n1), wrap(g2 - K.dir[2], p.n2), lead, rn);
              } else {
                const int at = r - K.dir[1] * W2 - K.dir[2];
                region_pull(src, at, info[at], rn);
              }
              decode(rn, g);
            });
      }
      if (last) {
        if (stored) {
          ps.sr_step = p.sr_step + (uint32_t)s;
          const int a1[3] = {0, g1 * p.s1, 0}, a2[3] = {0, g2, 0};
          if (p.cached) store_cell<S, ST, MASK, false, false, false>(ps, cell, a0, a1, a2, 0, 0, f);
          else store_cell<S, ST, MASK, false>(ps, cell, a0, a1, a2, 0, 0, f);
        }
      } else {
        const uint32_t hs = ST::stochastic ? sr_cell(key, (uint32_t)cell) : 0u;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const C sh = shift_of<ST>(S::w[q], p);
          dst[q * cap + r] = ST::stochastic ? ST::enc_sr(f[q], sh, sr_bits(hs, q)) : ST::enc(f[q], sh);
        }
      }
    }
    if (!last) __syncthreads();
  }
}

namespace {

template <class ST, int COLL>
Tile2dFn pick_mask2d(bool mask) {
  return mask ? tile2d_kernel<D2Q9, ST, COLL, true> : tile2d_kernel<D2Q9, ST, COLL, false>;
}

template <class ST>
Tile2dFn pick_coll2d(int coll, bool mask) {
  switch (coll) {
    case LBM_COLL_NONE: return pick_mask2d<ST, LBM_COLL_NONE>(mask);
    case LBM_COLL_BGK: return pick_mask2d<ST, LBM_COLL_BGK>(mask);
    case LBM_COLL_TRT: return pick_mask2d<ST, LBM_COLL_TRT>(mask);
    case LBM_COLL_KBC: return pick_mask2d<ST, LBM_COLL_KBC>(mask);
    case LBM_COLL_BGK_GUO: return pick_mask2d<ST, LBM_COLL_BGK_GUO>(mask);
  }
  return nullptr;
}

}  // namespace

Tile2dFn pick_tile2d_kernel(int codec, int coll, bool mask) {
  switch (codec) {
    case LBM_F32: return pick_coll2d<StF32>(coll, mask);
    case LBM_F64: return pick_coll2d<StF64>(coll, mask);
    case LBM_F16_SHIFTED: return pick_coll2d<StF16>(coll, mask);
    case LBM_BF16_SHIFTED: return pick_coll2d<StBF16>(coll, mask);
    case kCodecBF16SR: return pick_coll2d<StBF16SR>(coll, mask);
  }
  return nullptr;
}

int64_t tile2d_lds_bytes(int t1, int t2, int steps, int reach, int storage_bytes, bool mask) {
  const int m = reach * (steps - 1);
  const int64_t cap = (int64_t)(t1 + 2 * m) * (t2 + 2 * m);
  return 2 * D2Q9::Q * cap * storage_bytes + (mask ? 4 * ((cap + 1) & ~(int64_t)1) : 0);
}

int64_t tile2d_static_lds_bytes() { return 256 * (int64_t)sizeof(lbm_cell_class); }

}  // namespace lbm
