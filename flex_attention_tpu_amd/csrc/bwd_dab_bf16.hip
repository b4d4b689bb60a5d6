// Gradient of an additive bias that several (batch, head) pairs share, bf16, head dim 128, gfx950:
//   dab[plane, i, j] = sum over the plane's pairs of P_ij (dP_ij - delta_i).
//
// Persistent work-groups of 8 waves walk 128 x 128 tiles, and in each the pairs that share it, whose sum they keep in registers:
// every element is written once, by one work-group, in the order of the pairs.  Wave w owns 64 q rows (w >> 2) x 32 keys (w & 3)
// of the tile as two MFMA blocks, lane = key: two waves a SIMD, of at most 256 registers.  Two products per pair (S, dP); Q and K
// of a pair share one half of the LDS, dO and V the other, and each half is refilled while the other one's product runs, across
// tiles too (one tile per work-group: 238 us, its first copies, bias loads and stores exposed; walking: 221 us).
//
// Why a pass of its own: the dk/dv pass has dP at hand, but one pair at a time, so it can only store a full-size float32 gradient
// per pair, which another pass sums.  On B=4, H=16, S=1500 with a bias shared by the batch that is 576 MB written and read
// again: 596 us of dk/dv with the stores (478 without) and 158 us for the sum, of a step of 1000 us; with this pass and the
// two-waves-a-SIMD dk/dv loop the step takes 750 us.
// BOUND: operands from the caches (1.2 GB over all tiles and pairs, 128 KB a step into LDS), each phase waiting for its
// copies: the products are 35 us of it.
#include "fa_common.hpp"
#include "launch.hpp"
#include "tile_io.hpp"

namespace fa {

namespace dab_cfg {
constexpr int T = 128;   // rows and keys of a tile (the dk/dv pass's block map)
constexpr int D = 128;
constexpr int LDS_BYTES = 8 * kTileElems * 2 + 4 * T * 4;   // Q, K | dO, V in 64-row tiles; lse and delta rows, two buffers
}  // namespace dab_cfg

__global__ __launch_bounds__(512, 1) void bwd_dab_bf16_kernel(BwdArgs a, int n_b, int n_h) {
  using namespace dab_cfg;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  bf16_t* sX = reinterpret_cast<bf16_t*>(smem_raw);   // Q rows 0-63, Q 64-127, K 0-63, K 64-127
  bf16_t* sY = sX + 4 * kTileElems;                   // dO, V the same
  float* sLse = reinterpret_cast<float*>(sY + 4 * kTileElems);
  float* sDl = sLse + 2 * T;

  const int nQ = a.map.nq, nK = a.map.nk;
  const int n_pairs = n_b * n_h;
  // A tile of the walk.  Planes are numbered batch-major over the dimensions that the bias has.  An XCD (work-groups j % 8) takes a
  // contiguous eighth of the tiles, which share operands, and its work-groups every n-th of them.
  struct Tile {
    int t, q0, k0, qb, kb, b0, h0, state;
  };
  const int n_tiles = a.B * a.Hq / n_pairs * nQ * nK;
  const int per = (n_tiles + 7) >> 3, end = min(n_tiles, ((int)(blockIdx.x & 7) + 1) * per);
  auto next_tile = [&](Tile& x, int t) {   // the first kept tile from t on, in steps of the XCD's work-groups
    for (; t < end; t += (int)(gridDim.x >> 3)) {
      const int plane = t / (nQ * nK), r = t - plane * nQ * nK;
      x.qb = r / nK;
      x.kb = r - x.qb * nK;
      x.state = __builtin_amdgcn_readfirstlane((int)a.map.state[r]);
      if (x.state == 0) continue;
      const int planes_h = a.Hq / n_h;
      x.b0 = n_b == 1 ? plane / planes_h : 0;
      x.h0 = n_h == 1 ? plane % planes_h : 0;
      x.q0 = tile_base(x.qb, T, a.Sq);
      x.k0 = tile_base(x.kb, T, a.Sk);
      break;
    }
    x.t = t;
    return t < end;
  };
  Tile cur, nxt;
  if (!next_tile(cur, (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3))) return;
  nxt = cur;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int hh = lane >> 5;
  const int group = a.Hq / a.Hkv;

  ScoreMod<kScoreBiasOnly> sm;
  // the tile's bias, shared by the pairs: element e of block c is row qw + 32 c + acc_row(e, hh), key kw + l32
  // (qw, kw: first row and key of the wave's part)
  f32x16 acc[2];
  float bias[2][16];
  auto load_bias = [&](const Tile& x) {
    sm.init(a.score, a.sm_scale, x.h0, x.b0);
    const unsigned lane_off = (unsigned)(4 * hh) * (unsigned)a.Sk + (unsigned)(x.k0 + 32 * (w & 3) + l32);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      sm.bias_rows(bias[c], x.q0 + 64 * (w >> 2) + 32 * c, lane_off);
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[c][e] = 0.f;
    }
  };

  TileLoader<8> loader;
  loader.init(w, lane);
  auto pair_of = [&](const Tile& x, int p, int& b, int& h) {
    const int pb = n_b == 1 ? 0 : p / n_h;
    b = x.b0 + pb;
    h = x.h0 + p - pb * n_h;
  };
  auto issue = [&](const void* rows, const void* keys, const Tile& x, int p, bf16_t* dst) {
    int b, h;
    pair_of(x, p, b, h);
    const bf16_t* r = static_cast<const bf16_t*>(rows) + ((size_t)(b * a.Hq + h) * a.Sq + (size_t)x.q0) * D;
    const bf16_t* k = static_cast<const bf16_t*>(keys) + ((size_t)(b * a.Hkv + h / group) * a.Sk + (size_t)x.k0) * D;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      loader.load(r + half * kTileElems, dst + half * kTileElems);
      loader.load(k + half * kTileElems, dst + (2 + half) * kTileElems);
    }
  };
  float l_st = 0.f, m_st = 0.f, dl_st = 0.f;
  auto load_rows = [&](const Tile& x, int p) {
    if (tid < T) {
      int b, h;
      pair_of(x, p, b, h);
      const size_t row = (size_t)(b * a.Hq + h) * a.Sq + (size_t)x.q0;
      l_st = (a.l + row)[tid];
      m_st = (a.m + row)[tid];
      dl_st = (a.delta + row)[tid];
    }
  };
  auto store_rows = [&](int buf) {
    if (tid < T) {   // (the loads' values are first touched here)
      sLse[buf * T + tid] = (l_st > 0.f) ? __builtin_fmaf(m_st, kLog2e, log2f(l_st)) : __builtin_huge_valf();
      sDl[buf * T + tid] = dl_st;
    }
  };
  unsigned r_off[8];
  const int r_sw = swz(l32);
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) r_off[ks] = (unsigned)(l32 * kTileD + (((2 * ks + hh) ^ r_sw) << 3)) * 2u;
  // the wave's 64 x 32 part of rows x keys^T, from one half of the LDS
  auto product = [&](const bf16_t* half, f32x16 (&c)[2]) {
    const char* rt = reinterpret_cast<const char*>(half + (w >> 2) * kTileElems);
    const char* kt = reinterpret_cast<const char*>(half + 2 * kTileElems) + (w & 3) * 32 * kTileD * 2;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int e = 0; e < 16; ++e) c[x][e] = 0.f;
    // (operands are read four products ahead: left to itself the compiler waits out the LDS latency in front of each)
    bf16x8 kf[2][2], rf[2][2][2];
    auto read = [&](int stage) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        kf[stage & 1][i] = *reinterpret_cast<const bf16x8*>(kt + r_off[2 * stage + i]);
#pragma unroll
        for (int x = 0; x < 2; ++x) rf[stage & 1][i][x] = *reinterpret_cast<const bf16x8*>(rt + r_off[2 * stage + i] + x * 32 * kTileD * 2);
      }
    };
    read(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int stage = 0; stage < 4; ++stage) {
      if (stage < 3) read(stage + 1);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int x = 0; x < 2; ++x) c[x] = mfma32(rf[stage & 1][i][x], kf[stage & 1][i], c[x]);
      if (stage < 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  issue(a.q, a.k, cur, 0, sX);
  load_rows(cur, 0);
  load_bias(cur);
  store_rows(0);
  wait_vmem_all();
  __syncthreads();
  // (tile, pair) steps; the operands of a step's first product are copied while the step before runs, across tiles too
  int p = 0;
  bool more = true;
  for (int step = 0; more; ++step) {
    const int buf = step & 1;
    f32x16 s[2], dp[2];
    issue(a.dout, a.v, cur, p, sY);
    product(sX, s);
    wait_vmem_all();
    __syncthreads();   // dO, V are there, Q, K are read
    const bool last = p + 1 == n_pairs;
    const int p_next = last ? 0 : p + 1;
    if (last) more = next_tile(nxt, cur.t + (int)(gridDim.x >> 3));
    if (more) {
      load_rows(nxt, p_next);
      issue(a.q, a.k, nxt, p_next, sX);
    }
    product(sY, dp);
    const int qw = cur.q0 + 64 * (w >> 2), kw = cur.k0 + 32 * (w & 3);   // the wave's part
    auto accumulate = [&](auto masked) {
      constexpr bool MASKED = decltype(masked)::value;
      MaskArgs mk = a.mask;
      int doc_j = 0;
      if (MASKED) {
        int b, h;
        pair_of(cur, p, b, h);
        mk = mask_of_batch(a.mask, b, a.Sq, a.Sk);
        if (mk.flags & FLEXATTN_MASK_DOC) doc_j = mk.doc_k[kw + l32];
      }
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int r0 = 32 * c + 8 * g + 4 * hh;   // the lane's q rows come in runs of 4
          const f32x4 lse4 = *reinterpret_cast<const f32x4*>(sLse + buf * T + 64 * (w >> 2) + r0);
          const f32x4 dl4 = *reinterpret_cast<const f32x4*>(sDl + buf * T + 64 * (w >> 2) + r0);
          int di[4] = {0, 0, 0, 0};
          if (MASKED && (mk.flags & FLEXATTN_MASK_DOC) != 0) {
            const auto d4 = *reinterpret_cast<const i32x4_a4*>(mk.doc_q + qw + r0);
            di[0] = d4[0]; di[1] = d4[1]; di[2] = d4[2]; di[3] = d4[3];
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int e = 4 * g + u;
            const float pe = fast_exp2(__builtin_fmaf(bias[c][e], kLog2e, sm.to_log2(s[c][e], 0, 0)) - lse4[u]);
            float gl = pe * (dp[c][e] - dl4[u]);
            if (MASKED) gl = keep_elem(mk, qw + r0 + u, kw + l32, di[u], doc_j) ? gl : 0.f;
            acc[c][e] += gl;
          }
        }
    };
    if (cur.state == 1) {
      accumulate(std::true_type{});
    } else {
      accumulate(std::false_type{});
    }
    if (more) store_rows(buf ^ 1);
    wait_vmem_all();
    if (last) {
      // (a last tile of a ragged length starts early: its first rows and keys belong to the tiles before.  The stores and the
      // next bias loads are left open: they have the next step's first product to complete in.)
      float* out = a.dab + ((size_t)(unsigned)sm.ab_row0 + (size_t)(qw + 4 * hh)) * (size_t)a.Sk + (size_t)(kw + l32);
      const int own_q = kw + l32 < cur.kb * T ? 64 : cur.qb * T - qw - 4 * hh;
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int r = 32 * c + acc_row(e, 0);
          if (r >= own_q) __builtin_nontemporal_store(acc[c][e], out + (size_t)r * a.Sk);
        }
      if (more) load_bias(nxt);
    }
    cur = nxt;
    p = p_next;
    __syncthreads();   // the next Q, K and row values are there, dO, V are read
  }
}

// Planes of the bias gradient, the pairs that share each, and the tiles that the kernel walks; -1: more than its int counters and their
// steps of a work-group hold.
static long long dab_tiles(const BwdArgs& a, int* n_b, int* n_h) {
  *n_b = a.score.ab_sb_rows == 0 ? a.B : 1;
  *n_h = a.score.ab_sh_rows == 0 ? a.Hq : 1;
  const long long planes = (long long)a.B * a.Hq / ((long long)*n_b * *n_h), per_plane = (long long)a.map.nq * a.map.nk;
  return (double)planes * (double)per_plane > (double)((1ll << 31) - 512) ? -1 : planes * per_plane;
}

// From 200 tiles on.  Kernel times of forward and backward, us, full-size gradient and its sum against this pass:
//                              2 pairs a tile   8               32              64
//    49 tiles (H=1, S=896)     112.6 / 108.6    119.5 / 131.0   148.5 / 210.6   267.8 / 368.2
//   128 tiles (H=2, S=1024)    129.6 / 122.6    143.4 / 147.9   351.3 / 322.8   723.9 / 647.6
//   196 tiles (H=1, S=1792)    204.7 / 189.2    219.7 / 216.4   555.8 / 443.1   1069  /  892
//   256 tiles (H=4, S=1024)    137.6 / 126.8    174.7 / 164.9   731.8 / 580.3   1441  / 1161
//   288 tiles (H=2, S=1536)    187.4 / 177.3    218.7 / 227.9   804.7 / 701.3   1509  / 1332
// Fewer tiles leave CUs idle for as long as a tile's pairs take, one after the other.  The number of pairs moves the line little: it
// lengthens that chain and the full-size gradient's bytes alike.  (288: a second round of the 256 work-groups with few tiles in it.)
bool bwd_dab_bf16_pays(const BwdArgs& a) {
  int n_b, n_h;
  return a.score.kind == FLEXATTN_SCORE_NONE && dab_tiles(a, &n_b, &n_h) >= 200 && n_b * n_h > 1;
}

int bwd_dab_bf16(const BwdArgs& a, hipStream_t stream) {
  using namespace dab_cfg;
  int n_b, n_h;
  const long long tiles = dab_tiles(a, &n_b, &n_h);
  if (tiles < 0) return set_error(FLEXATTN_ENOTSUP, "flexattn_bwd_dab: more than 2^31 - 512 tiles of the bias");
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(bwd_dab_bf16_kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
  if (attr != hipSuccess) return set_error(FLEXATTN_ELAUNCH, "hipFuncSetAttribute(dab): %s", hipGetErrorString(attr));
  const unsigned grid = tiles < 256 ? (unsigned)((tiles + 7) / 8 * 8) : 256u;   // one work-group per CU, the same number per XCD
  hipLaunchKernelGGL(bwd_dab_bf16_kernel, dim3(grid), dim3(512), LDS_BYTES, stream, a, n_b, n_h);
  return check_launch("flexattn_bwd_dab bf16");
}

}  // namespace fa
