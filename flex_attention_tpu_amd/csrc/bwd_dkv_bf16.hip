// Flex-attention dk/dv backward, bf16, head dim 128, gfx950.
//
// A work-group takes a KV tile of one (batch, kv head).  Q / dO rows stream through double-buffered LDS (LDS-direct loads,
// swizzled unpadded tiles) together with their lse and delta, for every query head of the KV group and every q tile the
// transposed block map lists.  Per tile:
//   S = Q K^T,  dP = dO V^T   (lane owns a kv column, accumulator rows are q),
//   P = exp2(S' - lse_q),  dS = P (dP - delta_q) f'(S),
//   dv^T += dO^T P,  dk^T += Q^T dS   (dO^T, Q^T via transposing LDS reads).
// Each dk/dv tile has exactly one writer, so the result is deterministic and needs no atomics.
//
// The plain score, the soft-cap and the global position bias (one query head per kv head) run generated, hand-scheduled instruction
// streams (gen_dkv_tile.py -> bwd_dkv_tile.inc) that software-pipeline MFMA, VALU and LDS work inside the wave with a fixed
// register allocation: 4 waves, 32 of the 128 kv rows each, K and V in registers as MFMA B operands.  Everything else runs kernels
// with a compiled loop: head dimension 128 with 8 waves and K and V in LDS, 256 with 4 waves on 64 kv rows (see there).
#include <cstdlib>
#include "fa_common.hpp"
#include "launch.hpp"
#include "tile_io.hpp"

#include <type_traits>

// v[68:199] and a[192:255] belong to the generated tile streams
#define FA_DKV_TILE_CLOBBERS "v68", "v69", "v70", "v71", "v72", "v73", "v74", "v75", "v76", "v77", "v78", "v79", "v80", "v81", "v82", \
  "v83", "v84", "v85", "v86", "v87", "v88", "v89", "v90", "v91", "v92", "v93", "v94", "v95", "v96", "v97", \
  "v98", "v99", "v100", "v101", "v102", "v103", "v104", "v105", "v106", "v107", "v108", "v109", "v110", \
  "v111", "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", \
  "v124", "v125", "v126", "v127", "v128", "v129", "v130", "v131", "v132", "v133", "v134", "v135", "v136", \
  "v137", "v138", "v139", "v140", "v141", "v142", "v143", "v144", "v145", "v146", "v147", "v148", "v149", \
  "v150", "v151", "v152", "v153", "v154", "v155", "v156", "v157", "v158", "v159", "v160", "v161", "v162", \
  "v163", "v164", "v165", "v166", "v167", "v168", "v169", "v170", "v171", "v172", "v173", "v174", "v175", \
  "v176", "v177", "v178", "v179", "v180", "v181", "v182", "v183", "v184", "v185", "v186", "v187", "v188", \
  "v189", "v190", "v191", "v192", "v193", "v194", "v195", "v196", "v197", "v198", "v199", "a192", "a193", \
  "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", \
  "a207", "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", \
  "a220", "a221", "a222", "a223", "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", \
  "a233", "a234", "a235", "a236", "a237", "a238", "a239", "a240", "a241", "a242", "a243", "a244", "a245", \
  "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"

// scalar registers of the generated run loop
#define FA_DKV_RUN_SGPRS "s60", "s61", "s62", "s63", "s64", "s65", "s66", "s67", "s68", "s69", "s70", "s71", "s72", "s73", "s74", "s75", "s76", "s77", "s78", "s79", "s80", "s81", "s82", "s83", "s84", "s85", "s86", "s87", "s88", "s89", "s90", "s91", "s92", "s93", "s94", "s95", "s96", "s97", "s98", "s99", "s100"

#include "bwd_dkv_tile.inc"

namespace fa {

namespace dkv_cfg {
constexpr int BNK = 128;  // kv rows per work-group
constexpr int BQ = 128;   // q rows per step (two 64-row LDS tiles)
constexpr size_t kDsBlockBytes = (size_t)BQ * BNK * 2;  // one exported dS block
constexpr int D = 128;
constexpr int MAX_LIST = 2048;       // longest q tile list the plain-score kernel caches in LDS (262144 tokens)
constexpr int PREFETCH_LIST = 1024;  // of which an item's prefetch carries this many in registers; the rest is read when the item starts
// (Q, dO) x 2 buffers x 2 tiles, lse x2, delta x2, run-loop tables, cached q tile list and its partial flags
constexpr int LDS_BYTES = 8 * kTileElems * 2 + 4 * BQ * 4 + 4 * 32 * 4 + MAX_LIST * 5 + kDocStageBytes + kMaxSortedItems * 4;
// compiled loop: K, V and (Q, dO) x 2 buffers of 64 rows, lse x2, delta x2 of 64 rows
constexpr int LOOP_LDS_BYTES = 8 * kTileElems * 2 + 4 * 64 * 4;
}  // namespace dkv_cfg


// The register-resident state of the generated tile streams.  Every asm statement that touches it
// names it with the same physical-register constraints, so the values stay where the streams
// expect them and the compiler keeps those registers free of anything else.
struct PinnedState {
  f32x16 dv[4], dk[4];  // a[0:63], a[64:127]
  bf16x8 k[8], v[8];    // a[128:159], a[160:191]
};
#define FA_DKV_PINNED(st)                                                                                   \
  "+{a[0:15]}"(st.dv[0]), "+{a[16:31]}"(st.dv[1]), "+{a[32:47]}"(st.dv[2]), "+{a[48:63]}"(st.dv[3]),        \
      "+{a[64:79]}"(st.dk[0]), "+{a[80:95]}"(st.dk[1]), "+{a[96:111]}"(st.dk[2]), "+{a[112:127]}"(st.dk[3]), \
      "+{a[128:131]}"(st.k[0]), "+{a[132:135]}"(st.k[1]), "+{a[136:139]}"(st.k[2]), "+{a[140:143]}"(st.k[3]), \
      "+{a[144:147]}"(st.k[4]), "+{a[148:151]}"(st.k[5]), "+{a[152:155]}"(st.k[6]), "+{a[156:159]}"(st.k[7]), \
      "+{a[160:163]}"(st.v[0]), "+{a[164:167]}"(st.v[1]), "+{a[168:171]}"(st.v[2]), "+{a[172:175]}"(st.v[3]), \
      "+{a[176:179]}"(st.v[4]), "+{a[180:183]}"(st.v[5]), "+{a[184:187]}"(st.v[6]), "+{a[188:191]}"(st.v[7])

// Score modifications: compiled C++ path.  One work-group = 8 waves = one 128-row kv tile; a loop iteration covers 64 q rows,
// half an entry of the kv tile's list.  Wave w takes kv rows 32 (w & 3) and q rows 32 (w >> 2) of the iteration: one 32 x 32
// block of S and dP, its element-wise work, and its share of dk and dv, which the two waves of a kv block add up through LDS
// at the end.  K and V lie in LDS (64 KB) beside the double-buffered Q and dO (64 KB).
// BOUND: the element-wise work (about 270 vector instructions per block, against 32 MFMAs of 32 cycles) and what of it the other
// wave's products do not cover.  Two waves a SIMD, of at most 256 registers each; four waves with K and V in registers and
// 128-row iterations had one wave a SIMD: symmetric ALiBi closure, B=8, H=4, S=2048, dk/dv with export 240 -> 180-198 us; bias,
// B=4, H=16, S=1500, 478 -> 350-378 us.  A higher priority for one of a SIMD's waves, or around the products, changed nothing.
// EXPORT: the kernel also writes the tile's bf16 dS (the B operands of the dk product: here with the score function's
// derivative and sm_scale in them) to a.ds, in the block layout of the generated streams' export (see there), for
// the dq pass from dS: a score function is then evaluated in one backward pass instead of two.
// AB: the call may have an additive bias (false: splits_bias() kinds without one).
// DAB (with EXPORT and a bias): the kernel stores the bias gradient as well.  (A variant of its own: with the stores behind
// a test the compiler associates the element-wise sums differently, and dk and dv would change a bit with the export.)
template <int SCORE, bool EXPORT, bool AB, bool DAB>
__global__ __launch_bounds__(512, 1) void bwd_dkv_bf16_d128_kernel(BwdArgs a) {
  using namespace dkv_cfg;
  constexpr bool kBias = SCORE == kScoreBiasOnly;             // a bias and no score function: launched as a kind of its own
  constexpr bool kNoBias = SCORE == FLEXATTN_SCORE_NONE || !AB;
  static_assert(!DAB || (EXPORT && !kNoBias), "the bias gradient comes with the export of a call with a bias");
  constexpr int HQ = 64;   // q rows per iteration
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  bf16_t* sK = reinterpret_cast<bf16_t*>(smem_raw);   // K rows 0-63, 64-127, V the same
  bf16_t* sQ = sK + 4 * kTileElems;                   // buffer b: Q at tile 2 b, dO at 2 b + 1
  float* sLse = reinterpret_cast<float*>(sQ + 4 * kTileElems);
  float* sDl = sLse + 2 * HQ;

  const int nKb = a.map.nk;
  const int nQ = a.map.nq;
  const int n_wg = a.B * a.Hkv * nKb;
  const int wg = xcd_remap(blockIdx.x, n_wg);
  int bhk, kb;  // (low kv tiles have the most q tiles under causal masks: they go first)
  block_item(wg, a.B, a.Hkv, nKb, kBias && a.score.ab_sb_rows == 0, bhk, kb);
  const int b = bhk / a.Hkv;
  const MaskArgs mk = mask_of_batch(a.mask, b, a.Sq, a.Sk);
  const int hk = bhk % a.Hkv;
  const int group = a.Hq / a.Hkv;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = w & 3, wq = w >> 2;   // the wave's kv block and its q block of an iteration
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  const int kv_local = wk * 32 + l32;
  const int k0 = tile_base(kb, BNK, a.Sk);
  const int k_idx = k0 + kv_local;
  const bool own_col = k_idx >= kb * BNK;   // (else a row of the kv tile before)
  const size_t kv_off = ((size_t)bhk * a.Sk + (size_t)k0) * D;
  int doc_j = 0;
  if (mk.flags & FLEXATTN_MASK_DOC) doc_j = mk.doc_k[k_idx];

  f32x16 dk_acc[4], dv_acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dk_acc[i][e] = 0.f;
      dv_acc[i][e] = 0.f;
    }

  const int n_tiles = a.map.cnt[kb];
  const int* tile_idx = a.map.idx + (size_t)kb * nQ;
  const bool ragged_q = nQ * BQ != a.Sq;   // (the last q tile then shares rows with the one before)
  const int n_iter = 2 * n_tiles * group;

  // (dS block of the list's first entry, for query head 0: read here, for a load in the loop would wait for the copies before it)
  const int ds_first = EXPORT ? __builtin_amdgcn_readfirstlane(a.ds_col[kb]) : 0;
  TileLoader<8> loader;
  loader.init(w, lane);
  // Iteration `it` covers rows 64 (it & 1) .. of list entry t of query head hk group + g, it = 2 (g n_tiles + t) + (it & 1).
  // `at` walks the entries one ahead of the iteration that computes; its q block index and state are fetched an entry ahead.
  int g_at = 0, t_at = 0;   // entry that is copied next
  int qb_at = 0, st_at = 0, qb_next = 0;
  if (n_iter > 0) {
    qb_at = __builtin_amdgcn_readfirstlane(tile_idx[0]);
    st_at = a.map.state[(size_t)qb_at * nKb + kb];
    qb_next = n_tiles > 1 ? tile_idx[1] : qb_at;
  }
  float l_st = 0.f, m_st = 0.f, dl_st = 0.f;
  size_t rbase = 0;   // first row of the rows that are copied next
  auto copy_of = [&](int n, int buf) {   // one of the wave's four pieces of them: Q, Q, dO, dO
    loader.load_block(static_cast<const bf16_t*>(n < 2 ? a.q : a.dout) + rbase * D, sQ + (2 * buf + (n >> 1)) * kTileElems, n & 1);
  };
  auto locate_rows = [&](int half) {
    rbase = ((size_t)(b * a.Hq + hk * group + g_at) * a.Sq + (size_t)(tile_base(qb_at, BQ, a.Sq) + half * HQ));
    if (tid < HQ) {
      unsigned at = 4u * (unsigned)tid;   // (opaque: three addresses per thread, kept through the loop, would spill)
      asm volatile("" : "+v"(at));
      l_st = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.l + rbase) + at);
      m_st = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.m + rbase) + at);
      dl_st = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.delta + rbase) + at);
    }
  };
  auto store_rows = [&](int buf) {
    if (tid < HQ) {   // (the loads' values are first touched here: touched where they are issued, every iteration waits for its copies there)
      sLse[buf * HQ + tid] = (l_st > 0.f) ? __builtin_fmaf(m_st, kLog2e, log2f(l_st)) : __builtin_huge_valf();
      sDl[buf * HQ + tid] = dl_st;
    }
  };
  auto advance = [&]() {   // `at` to the next entry
    if (++t_at == n_tiles) {
      t_at = 0;
      ++g_at;
    }
    qb_at = __builtin_amdgcn_readfirstlane(qb_next);
    st_at = a.map.state[(size_t)qb_at * nKb + kb];
    qb_next = tile_idx[t_at + 1 < n_tiles ? t_at + 1 : 0];
  };
  if (n_iter > 0) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      loader.load(static_cast<const bf16_t*>(a.k) + kv_off + half * kTileElems, sK + half * kTileElems);
      loader.load(static_cast<const bf16_t*>(a.v) + kv_off + half * kTileElems, sK + (2 + half) * kTileElems);
    }
    locate_rows(0);
#pragma unroll
    for (int n = 0; n < 4; ++n) copy_of(n, 0);
    store_rows(0);
  }
  wait_vmem_all();
  __syncthreads();

  // lane-constant byte offsets of the operand reads inside a tile (see tile_io.hpp)
  const int r_sw = swz(l32);
  const int t_row = 4 * hh + ((lane & 15) >> 2);
  const int t_chunk = 2 * ((lane & 31) >> 4) + ((lane & 3) >> 1);
  const int t_half = 4 * (lane & 1);
  unsigned r_off[8], t_off[4][2];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) r_off[ks] = (unsigned)(l32 * kTileD + (((2 * ks + hh) ^ r_sw) << 3)) * 2u;
#pragma unroll
  for (int db = 0; db < 4; ++db) {
    t_off[db][0] = (unsigned)(tile_off(t_row, 4 * db + t_chunk) + t_half) * 2u;
    t_off[db][1] = (unsigned)(tile_off(t_row + 8, 4 * db + t_chunk) + t_half) * 2u;
  }
  const char* kt = reinterpret_cast<const char*>(sK + (wk >> 1) * kTileElems) + (wk & 1) * 32 * kTileD * 2;
  const char* vt = kt + 2 * kTileElems * 2;

  constexpr int kOpenStores = EXPORT ? 2 : 0;
  float bias[16];
  ScoreMod<SCORE> sm;
  int qb = 0, st = 0, g = 0, t = 0;   // the entry that is computed
  for (int it = 0; it < n_iter; ++it) {
    const int buf = it & 1;
    if (buf == 0) {   // an entry's first half: the entry that was copied ahead
      if (it == 0 || g != g_at) sm.init(a.score, a.sm_scale, hk * group + g_at, b);
      qb = qb_at;
      st = st_at;
      g = g_at;
      t = t_at;
    }
    const bool partial = __builtin_amdgcn_readfirstlane(st) == 1 || (qb == nQ - 1 && ragged_q);
    const int q0 = tile_base(qb, BQ, a.Sq);
    const int cc = 2 * buf + wq;   // the wave's 32-row block of the q tile
    // (elements before this offset belong to the q tile before; a column of the kv tile before owns none)
    const int own = first_owned(qb, BQ, q0, 4 * hh, own_col);
    // An additive bias: a block's values are loaded behind the element-wise work of the block before and are there before
    // the next rows' copies are issued (vector-memory operations complete in order: behind the copies the first use would
    // wait for them too).
    const unsigned lane_off = (unsigned)(4 * hh) * (unsigned)a.Sk + (unsigned)k_idx;   // (of a bias or its gradient)
    if (kBias) {
      if (it == 0) sm.bias_rows(bias, q0 + 32 * cc, lane_off);
      wait_vmem<kOpenStores>();
    }
    const bool more = it + 1 < n_iter;
    if (more) {
      if (buf == 1) advance();
      locate_rows(buf ^ 1);
    }

    const char* qt = reinterpret_cast<const char*>(sQ + 2 * buf * kTileElems) + wq * 32 * kTileD * 2;
    const char* dot = qt + kTileElems * 2;
    f32x16 s_acc, dp_acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s_acc[e] = 0.f;
      dp_acc[e] = 0.f;
    }
    // (operands are read four products ahead: left to itself the compiler reads each pair in front of its product and waits
    // out the LDS latency 16 times)
    bf16x8 fa[2][4], fb[2][4];
    auto read_rows = [&](int stage) {   // stages 0, 1: Q and K, 2, 3: dO and V
      const char* ra = stage < 2 ? qt : dot;
      const char* rb = stage < 2 ? kt : vt;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        fa[stage & 1][i] = *reinterpret_cast<const bf16x8*>(ra + r_off[4 * (stage & 1) + i]);
        fb[stage & 1][i] = *reinterpret_cast<const bf16x8*>(rb + r_off[4 * (stage & 1) + i]);
      }
    };
    read_rows(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int stage = 0; stage < 4; ++stage) {
      if (stage < 3) read_rows(stage + 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (stage < 2) s_acc = mfma32(fa[stage & 1][i], fb[stage & 1][i], s_acc);
        else dp_acc = mfma32(fa[stage & 1][i], fb[stage & 1][i], dp_acc);
      }
      if (stage < 3) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // an MFMA,
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);   // two LDS reads
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (more) copy_of(stage, buf ^ 1);   // (under the products: in front of them, each copy holds the wave for some 50 cycles)
    }

    bf16x8 pb[2], dsb[2];
    // (DAB: the bias gradient, float32 [B, Hq, Sq, Sk], a row's 32 columns per store.  The block's 32 rows are a buffer of
    // their own: a store at an offset beyond it is dropped, which is how an element that another work-group owns is
    // left out; a branch around each of the 16 stores instead cuts the block into as many pieces for the scheduler.)
    __amdgpu_buffer_rsrc_t dab_block;
    if (DAB)
      dab_block = __builtin_amdgcn_make_buffer_rsrc(
          a.dab + ((size_t)(b * a.Hq + hk * group + g) * a.Sq + (size_t)(q0 + 32 * cc)) * a.Sk, 0, 32 * a.Sk * 4, 0x00020000);
    auto elementwise = [&](auto masked) {
      constexpr bool MASKED = decltype(masked)::value;
      const bool has_doc = MASKED && (mk.flags & FLEXATTN_MASK_DOC) != 0;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int r0 = 32 * cc + 8 * g4 + 4 * hh;  // the lane's q rows come in runs of 4
        const f32x4 lse4 = *reinterpret_cast<const f32x4*>(sLse + r0);
        const f32x4 dl4 = *reinterpret_cast<const f32x4*>(sDl + r0);
        int di[4] = {0, 0, 0, 0};
        if (MASKED && has_doc) {
          const auto d4 = *reinterpret_cast<const i32x4_a4*>(mk.doc_q + q0 + r0);
          di[0] = d4[0]; di[1] = d4[1]; di[2] = d4[2]; di[3] = d4[3];
        }
        float pv[4], dsv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = 4 * g4 + u;
          const int i = q0 + r0 + u;
          const float tv = sm.to_log2(s_acc[e], i, k_idx);
          float pe = fast_exp2((kBias ? __builtin_fmaf(bias[e], kLog2e, tv) : kNoBias ? tv : tv + sm.bias2(i, k_idx)) - lse4[u]);
          float gl = pe * (dp_acc[e] - dl4[u]);   // the gradient of the logit itself: what an additive bias receives
          float gd = gl * sm.dfactor(tv, s_acc[e], i, k_idx);
          unsigned dab_off = 4u * lane_off;
          if (MASKED) {
            const bool owned = 32 * cc + 8 * g4 + u >= own;
            const bool keep = keep_elem(mk, i, k_idx, di[u], doc_j) & owned;
            if (DAB) gl = keep ? gl : 0.f;
            pe = keep ? pe : 0.f;
            gd = keep ? gd : 0.f;
            // (rows and columns of the tiles before: the work-groups of those store them)
            dab_off = owned ? dab_off : ~0u;
          }
          if (DAB) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, gl), dab_block, (int)dab_off, (8 * g4 + u) * a.Sk * 4, 0);
          pv[u] = pe;
          dsv[u] = gd;
        }
        const bf16x2 p01 = pack_bf16(pv[0], pv[1]), p23 = pack_bf16(pv[2], pv[3]);
        const bf16x2 d01 = pack_bf16(dsv[0], dsv[1]), d23 = pack_bf16(dsv[2], dsv[3]);
        const int o = 4 * (g4 & 1);
        pb[g4 >> 1][o] = p01[0]; pb[g4 >> 1][o + 1] = p01[1]; pb[g4 >> 1][o + 2] = p23[0]; pb[g4 >> 1][o + 3] = p23[1];
        dsb[g4 >> 1][o] = d01[0]; dsb[g4 >> 1][o + 1] = d01[1]; dsb[g4 >> 1][o + 2] = d23[0]; dsb[g4 >> 1][o + 3] = d23[1];
      }
    };
    if (partial) {
      elementwise(std::true_type{});
    } else {
      elementwise(std::false_type{});
    }
    if (kBias && more) {
      ScoreMod<SCORE> of;   // (the next block's head, which an entry's second half shares)
      of.init(a.score, a.sm_scale, hk * group + g_at, b);
      of.bias_rows(bias, tile_base(qb_at, BQ, a.Sq) + 64 * (buf ^ 1) + 32 * wq, lane_off);
    }
    if constexpr (EXPORT) {
      // block of (query head, kept tile pair): head a.ds_pairs + a.ds_col[kv tile] + place of the q tile in the kv
      // tile's list; inside it kv block wk's 1 KB per (32-row q block cc, 16-row half u), lane L its 8 values
      char* blk = static_cast<char*>(a.ds) +
                  ((size_t)(b * a.Hq + hk * group + g) * (size_t)a.ds_pairs + (size_t)(ds_first + t)) * kDsBlockBytes +
                  8192 * wk + 16 * (2 * l32 + hh);
#pragma unroll
      for (int u = 0; u < 2; ++u) *reinterpret_cast<bf16x8*>(blk + 1024 * (2 * cc + u)) = dsb[u];
    }

    // transposed fragments of the block's rows, dv^T += dO^T P, dk^T += Q^T dS
    s16x4 tr[2][4][4];   // [16-row half][column block][dO low, dO high, Q low, Q high]
    auto read_tr = [&](int u) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          tr[u][db][i] = lds_read_tr16(reinterpret_cast<const bf16_t*>((i < 2 ? dot : qt) + t_off[db][i & 1] + 16 * u * kTileD * 2));
    };
    read_tr(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (u == 0) read_tr(1);
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        dv_acc[db] = mfma32(join_tr(tr[u][db][0], tr[u][db][1]), pb[u], dv_acc[db]);
        dk_acc[db] = mfma32(join_tr(tr[u][db][2], tr[u][db][3]), dsb[u], dk_acc[db]);
      }
      if (u == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }

    if (more) store_rows(buf ^ 1);
    // (the copies are there; what was issued behind them, the next bias values and the stores of dS, may stay open)
    wait_vmem<kOpenStores + (kBias ? 16 : 0)>();
    __syncthreads();
  }
  wait_vmem_all();

  // the two waves of a kv block add up: one finishes dk, the other dv
  {
    float* ex = reinterpret_cast<float*>(smem_raw) + (size_t)w * 64 * 64;   // 16 KB per wave
    auto put = [&](const f32x16 (&x)[4]) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4)
          *reinterpret_cast<f32x4*>(ex + ((4 * db + g4) * 64 + lane) * 4) =
              f32x4{x[db][4 * g4], x[db][4 * g4 + 1], x[db][4 * g4 + 2], x[db][4 * g4 + 3]};
    };
    if (wq == 0) put(dv_acc); else put(dk_acc);
    __syncthreads();
    const float* other = reinterpret_cast<const float*>(smem_raw) + (size_t)(w ^ 4) * 64 * 64;
    auto finish = [&](const f32x16 (&x)[4], bf16_t* out) {
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(other + ((4 * db + g4) * 64 + lane) * 4);
          const bf16x2 lo = pack_bf16(x[db][4 * g4] + y[0], x[db][4 * g4 + 1] + y[1]);
          const bf16x2 hi = pack_bf16(x[db][4 * g4 + 2] + y[2], x[db][4 * g4 + 3] + y[3]);
          const bf16x4 o = {lo[0], lo[1], hi[0], hi[1]};
          if (own_col) *reinterpret_cast<bf16x4*>(out + (size_t)kv_local * D + 32 * db + 8 * g4 + 4 * hh) = o;
        }
    };
    if (wq == 0) finish(dk_acc, static_cast<bf16_t*>(a.dk) + kv_off); else finish(dv_acc, static_cast<bf16_t*>(a.dv) + kv_off);
  }
}

// Head dimension 256: compiled C++ path.  One work-group = 4 waves = 64 kv rows, half a tile of the block map; a loop iteration
// covers 64 q rows, half an entry of the tile's list, as one LDS tile (tile_io.hpp) per 128-column panel at [buffer][panel].
// Wave w has kv rows 32 (w & 1) and, of the iteration, q rows 32 (w >> 1) for S and dP, over all 256 columns; P and dS go to the
// other wave of the kv rows through LDS, and each of the two adds the products of both q blocks to dk and dv in columns
// 128 (w >> 1): 128 accumulator registers and 128 of K and V, which leaves room to read operands ahead.
// BOUND: one wave a SIMD: an iteration is 64 MFMAs (2048 cycles) among some 700 instructions, copies into LDS of 64 KB and two
// barriers, 6280 cycles (with the export of dS).  The form before this one had 128 kv rows a work-group and all columns in each wave: 256
// accumulators beside K and V left 128 registers for everything else, operands were read in front of each product and the
// reloads of spilled registers, like the row values and the dS index read in the loop, waited for the copies in flight: dk/dv of
// B=4, H=16, S=4096, causal, 1776 -> 1520-1610 us, and twice the work-groups where few fill the chip.
// EXPORT: the pass also writes its bf16 dS, as bwd_dkv_bf16_d128_kernel does: at two panels the dq pass that recomputes S
// and dP costs three products of a 256-deep contraction, from dS one (B=4, H=16, S=4096, causal, forward and backward: 3.61
// -> 3.08 ms).
template <int SCORE, bool EXPORT, bool AB>
__global__ __launch_bounds__(256, 1) void bwd_dkv_bf16_wide_kernel(BwdArgs a) {
  using namespace dkv_cfg;
  constexpr bool kNoBias = SCORE == FLEXATTN_SCORE_NONE || !AB;   // (a bias without a score function: kScoreBiasOnly)
  constexpr int NP = 2, D = 128 * NP;
  constexpr int HQ = 64;                  // q rows per iteration
  constexpr int kPanel = kTileElems * 2;  // bytes
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  bf16_t* sQ = reinterpret_cast<bf16_t*>(smem_raw);
  bf16_t* sDO = sQ + 2 * NP * kTileElems;
  char* sX = reinterpret_cast<char*>(sDO + 2 * NP * kTileElems);   // P and dS of the four waves, 4 KB each
  float* sLse = reinterpret_cast<float*>(sX + 4 * 4096);
  float* sDl = sLse + 2 * HQ;

  const int nKb = a.map.nk;
  const int nQ = a.map.nq;
  const int n_wg = a.B * a.Hkv * nKb * 2;
  const int wg = xcd_remap(blockIdx.x, n_wg);
  const int bhk = wg / (2 * nKb);
  const int kb = (wg - bhk * 2 * nKb) >> 1, kx = wg & 1;   // tile of the block map and half of it
  const int b = bhk / a.Hkv;
  const MaskArgs mk = mask_of_batch(a.mask, b, a.Sq, a.Sk);
  const int hk = bhk % a.Hkv;
  const int group = a.Hq / a.Hkv;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w & 1, wc = w >> 1;   // the wave's kv rows; its q rows in S and dP, its columns in dk and dv
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  const int kv_local = 64 * kx + 32 * wr + l32;   // in the tile
  const int k0 = tile_base(kb, BNK, a.Sk);
  const int k_idx = k0 + kv_local;
  const bool own_col = k_idx >= kb * BNK;   // (else a row of the kv tile before)
  const size_t kv_off = ((size_t)bhk * a.Sk + (size_t)k0) * D;
  const bf16_t* Kg = static_cast<const bf16_t*>(a.k) + kv_off;
  const bf16_t* Vg = static_cast<const bf16_t*>(a.v) + kv_off;

  bf16x8 kreg[8 * NP], vreg[8 * NP];
#pragma unroll
  for (int ks = 0; ks < 8 * NP; ++ks) {
    kreg[ks] = *reinterpret_cast<const bf16x8*>(Kg + (size_t)kv_local * D + ks * 16 + hh * 8);
    vreg[ks] = *reinterpret_cast<const bf16x8*>(Vg + (size_t)kv_local * D + ks * 16 + hh * 8);
  }
  int doc_j = 0;
  if (mk.flags & FLEXATTN_MASK_DOC) doc_j = mk.doc_k[k_idx];

  f32x16 dk_acc[4], dv_acc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dk_acc[i][e] = 0.f;
      dv_acc[i][e] = 0.f;
    }

  const int n_tiles = a.map.cnt[kb];
  const int* tile_idx = a.map.idx + (size_t)kb * nQ;
  const bool ragged_q = nQ * BQ != a.Sq;   // (the last q tile then shares rows with the one before)
  const int n_iter = 2 * n_tiles * group;

  // (as in bwd_dkv_bf16_d128_kernel)
  const int ds_first = EXPORT ? __builtin_amdgcn_readfirstlane(a.ds_col[kb]) : 0;
  TileLoader<4, D> loader;
  loader.init(w, lane);
  // Iteration `it` covers rows 64 (it & 1) .. of a list entry of query head hk group + g.  The list is walked from its end:
  // under causal masks the lists of a head's kv tiles share their ends, and its work-groups then read the same rows at the same
  // time.  `at` names the entry that is copied next; its q block index and state are fetched an entry ahead.
  int g_at = 0, t_at = n_tiles - 1;
  int qb_at = 0, st_at = 0, qb_next = 0;
  if (n_iter > 0) {
    qb_at = __builtin_amdgcn_readfirstlane(tile_idx[t_at]);
    st_at = a.map.state[(size_t)qb_at * nKb + kb];
    qb_next = tile_idx[n_tiles > 1 ? t_at - 1 : t_at];
  }
  float l_st = 0.f, m_st = 0.f, dl_st = 0.f;
  size_t rbase = 0;   // first row of the rows that are copied next
  auto copy_of = [&](int n, int buf) {   // one of the wave's 16 KB-sized pieces of them: n = 8 panel + 4 (0: Q, 1: dO) + block
    const int pn = n >> 3;
    if (n & 4) loader.load_block(static_cast<const bf16_t*>(a.dout) + rbase * D + 128 * pn, sDO + (buf * NP + pn) * kTileElems, n & 3);
    else loader.load_block(static_cast<const bf16_t*>(a.q) + rbase * D + 128 * pn, sQ + (buf * NP + pn) * kTileElems, n & 3);
  };
  auto locate_rows = [&](int half) {
    rbase = ((size_t)(b * a.Hq + hk * group + g_at) * a.Sq + (size_t)(tile_base(qb_at, BQ, a.Sq) + half * HQ));
    if (tid < HQ) {
      unsigned at = 4u * (unsigned)tid;   // (opaque: three addresses per thread, kept through the loop, would spill)
      asm volatile("" : "+v"(at));
      l_st = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.l + rbase) + at);
      m_st = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.m + rbase) + at);
      dl_st = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.delta + rbase) + at);
    }
  };
  auto store_rows = [&](int buf) {
    if (tid < HQ) {   // (the loads' values are first touched here: touched where they are issued, every iteration waits for its copies there)
      sLse[buf * HQ + tid] = (l_st > 0.f) ? __builtin_fmaf(m_st, kLog2e, log2f(l_st)) : __builtin_huge_valf();
      sDl[buf * HQ + tid] = dl_st;
    }
  };
  auto advance = [&]() {   // `at` to the next entry
    if (--t_at < 0) {
      t_at = n_tiles - 1;
      ++g_at;
    }
    qb_at = __builtin_amdgcn_readfirstlane(qb_next);
    st_at = a.map.state[(size_t)qb_at * nKb + kb];
    qb_next = tile_idx[t_at > 0 ? t_at - 1 : n_tiles - 1];
  };
  if (n_iter > 0) {
    locate_rows(0);
#pragma unroll
    for (int n = 0; n < 8 * NP; ++n) copy_of(n, 0);
    store_rows(0);
  }
  wait_vmem_all();
  __syncthreads();

  // lane-constant byte offsets of the operand reads inside a tile (see tile_io.hpp)
  const int r_sw = swz(l32);
  const int t_row = 4 * hh + ((lane & 15) >> 2);
  const int t_chunk = 2 * ((lane & 31) >> 4) + ((lane & 3) >> 1);
  const int t_half = 4 * (lane & 1);
  unsigned r_off[8], t_off[4][2];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) r_off[ks] = (unsigned)(l32 * kTileD + (((2 * ks + hh) ^ r_sw) << 3)) * 2u;
#pragma unroll
  for (int db = 0; db < 4; ++db) {
    t_off[db][0] = (unsigned)(tile_off(t_row, 4 * db + t_chunk) + t_half) * 2u;
    t_off[db][1] = (unsigned)(tile_off(t_row + 8, 4 * db + t_chunk) + t_half) * 2u;
  }

  ScoreMod<SCORE> sm;
  int qb = 0, st = 0, g = 0, t = 0;   // the entry that is computed
  for (int it = 0; it < n_iter; ++it) {
    const int buf = it & 1;
    if (buf == 0) {   // an entry's first half: the entry that was copied ahead
      if (it == 0 || g != g_at) sm.init(a.score, a.sm_scale, hk * group + g_at, b);
      qb = qb_at;
      st = st_at;
      g = g_at;
      t = t_at;
    }
    const bool partial = __builtin_amdgcn_readfirstlane(st) == 1 || (qb == nQ - 1 && ragged_q);
    const int q0 = tile_base(qb, BQ, a.Sq);
    const int cc = 2 * buf + wc;   // the wave's 32-row block of the q tile
    // (elements before this offset belong to the q tile before; a column of the kv tile before owns none)
    const int own = first_owned(qb, BQ, q0, 4 * hh, own_col);
    const bool more = it + 1 < n_iter;
    if (more) {
      if (buf == 1) advance();
      locate_rows(buf ^ 1);
    }
    const char* qt = reinterpret_cast<const char*>(sQ + buf * NP * kTileElems);
    const char* dot = reinterpret_cast<const char*>(sDO + buf * NP * kTileElems);

    f32x16 s_acc, dp_acc;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      s_acc[e] = 0.f;
      dp_acc[e] = 0.f;
    }
    // (operands are read four products ahead: left to itself the compiler waits out the LDS latency in front of each)
    bf16x8 rf[2][4];
    auto read_rows = [&](int stage) {   // four k-steps each: those of Q, panel by panel, then those of dO
      const int at = stage % (2 * NP);
      const char* rows = (stage < 2 * NP ? qt : dot) + (at >> 1) * kPanel + wc * 32 * kTileD * 2;
#pragma unroll
      for (int i = 0; i < 4; ++i) rf[stage & 1][i] = *reinterpret_cast<const bf16x8*>(rows + r_off[4 * (at & 1) + i]);
    };
    read_rows(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int stage = 0; stage < 4 * NP; ++stage) {
      if (stage < 4 * NP - 1) read_rows(stage + 1);
      const int at = 4 * (stage % (2 * NP));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (stage < 2 * NP) s_acc = mfma32(rf[stage & 1][i], kreg[at + i], s_acc);
        else dp_acc = mfma32(rf[stage & 1][i], vreg[at + i], dp_acc);
      }
      if (stage < 4 * NP - 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // an MFMA,
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (more) {   // (under the products: in front of them, each copy holds the wave for some 50 cycles)
        copy_of(2 * stage, buf ^ 1);
        copy_of(2 * stage + 1, buf ^ 1);
      }
    }

    // dv^T += dO^T P, dk^T += Q^T dS in the wave's columns, over the q rows of both waves: groups of 16 rows, this wave's own
    // first; the next group's transposed fragments are read under this one's products
    s16x4 tr[2][4][4];   // [group & 1][column block][dO low, dO high, Q low, Q high]
    auto read_tr = [&](int ga) {
      const int off = (32 * (wc ^ (ga >> 1)) + 16 * (ga & 1)) * kTileD * 2 + wc * kPanel;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          tr[ga & 1][db][i] = lds_read_tr16(reinterpret_cast<const bf16_t*>((i < 2 ? dot : qt) + t_off[db][i & 1] + off));
    };
    read_tr(0);   // (in front of the element-wise work, which hides their latency)
    __builtin_amdgcn_sched_barrier(0);
    bf16x8 pb[2], dsb[2];
    auto elementwise = [&](auto masked) {
      constexpr bool MASKED = decltype(masked)::value;
      const bool has_doc = MASKED && (mk.flags & FLEXATTN_MASK_DOC) != 0;
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int r0 = 32 * cc + 8 * g4 + 4 * hh;  // the lane's q rows come in runs of 4 (64 buf + ..: the buffer's row values)
        const f32x4 lse4 = *reinterpret_cast<const f32x4*>(sLse + r0);
        const f32x4 dl4 = *reinterpret_cast<const f32x4*>(sDl + r0);
        int di[4] = {0, 0, 0, 0};
        if (MASKED && has_doc) {
          const auto d4 = *reinterpret_cast<const i32x4_a4*>(mk.doc_q + q0 + r0);
          di[0] = d4[0]; di[1] = d4[1]; di[2] = d4[2]; di[3] = d4[3];
        }
        float pv[4], dsv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int e = 4 * g4 + u;
          const int i = q0 + r0 + u;
          const float tv = sm.to_log2(s_acc[e], i, k_idx);
          float pe = fast_exp2(tv + (kNoBias ? 0.f : sm.bias2(i, k_idx)) - lse4[u]);
          float gd = pe * (dp_acc[e] - dl4[u]) * sm.dfactor(tv, s_acc[e], i, k_idx);
          if (MASKED) {
            const bool keep = keep_elem(mk, i, k_idx, di[u], doc_j) & (32 * cc + 8 * g4 + u >= own);
            pe = keep ? pe : 0.f;
            gd = keep ? gd : 0.f;
          }
          pv[u] = pe;
          dsv[u] = gd;
        }
        const bf16x2 p01 = pack_bf16(pv[0], pv[1]), p23 = pack_bf16(pv[2], pv[3]);
        const bf16x2 d01 = pack_bf16(dsv[0], dsv[1]), d23 = pack_bf16(dsv[2], dsv[3]);
        const int o = 4 * (g4 & 1);
        pb[g4 >> 1][o] = p01[0]; pb[g4 >> 1][o + 1] = p01[1]; pb[g4 >> 1][o + 2] = p23[0]; pb[g4 >> 1][o + 3] = p23[1];
        dsb[g4 >> 1][o] = d01[0]; dsb[g4 >> 1][o + 1] = d01[1]; dsb[g4 >> 1][o + 2] = d23[0]; dsb[g4 >> 1][o + 3] = d23[1];
      }
    };
    if (partial) {
      elementwise(std::true_type{});
    } else {
      elementwise(std::false_type{});
    }
    // P and dS to the other wave of these kv rows
    {
      char* mine = sX + w * 4096 + 16 * lane;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        *reinterpret_cast<bf16x8*>(mine + 1024 * u) = pb[u];
        *reinterpret_cast<bf16x8*>(mine + 2048 + 1024 * u) = dsb[u];
      }
    }
    if constexpr (EXPORT) {
      // (the block layout of bwd_dkv_bf16_d128_kernel's export)
      char* blk = static_cast<char*>(a.ds) +
                  ((size_t)(b * a.Hq + hk * group + g) * (size_t)a.ds_pairs + (size_t)(ds_first + t)) * kDsBlockBytes +
                  8192 * (2 * kx + wr) + 16 * (2 * l32 + hh);
#pragma unroll
      for (int u = 0; u < 2; ++u) *reinterpret_cast<bf16x8*>(blk + 1024 * (2 * cc + u)) = dsb[u];
    }

    auto products = [&](int ga, bf16x8 p, bf16x8 ds) {
#pragma unroll
      for (int db = 0; db < 4; ++db) {
        dv_acc[db] = mfma32(join_tr(tr[ga & 1][db][0], tr[ga & 1][db][1]), p, dv_acc[db]);
        dk_acc[db] = mfma32(join_tr(tr[ga & 1][db][2], tr[ga & 1][db][3]), ds, dk_acc[db]);
      }
    };
    auto interleave = [&]() {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_sched_barrier(0);
    read_tr(1);
    products(0, pb[0], dsb[0]);
    interleave();
    read_tr(2);
    products(1, pb[1], dsb[1]);
    interleave();
    // (the other wave's P and dS are there; copies and stores stay open over this barrier)
    __syncthreads();
    {
      const char* other = sX + (w ^ 2) * 4096 + 16 * lane;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        pb[u] = *reinterpret_cast<const bf16x8*>(other + 1024 * u);
        dsb[u] = *reinterpret_cast<const bf16x8*>(other + 2048 + 1024 * u);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    read_tr(3);
    products(2, pb[0], dsb[0]);
    interleave();
    products(3, pb[1], dsb[1]);

    if (more) store_rows(buf ^ 1);
    wait_vmem<EXPORT ? 2 : 0>();   // (the copies are there; the stores of dS behind them may stay open)
    __syncthreads();
  }

  if (!own_col) return;
  bf16_t* dKg = static_cast<bf16_t*>(a.dk) + kv_off + (size_t)kv_local * D + 128 * wc;
  bf16_t* dVg = static_cast<bf16_t*>(a.dv) + kv_off + (size_t)kv_local * D + 128 * wc;
#pragma unroll
  for (int db = 0; db < 4; ++db) {
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      bf16x2 lo = pack_bf16(dk_acc[db][4 * g4], dk_acc[db][4 * g4 + 1]);
      bf16x2 hi = pack_bf16(dk_acc[db][4 * g4 + 2], dk_acc[db][4 * g4 + 3]);
      const bf16x4 out = {lo[0], lo[1], hi[0], hi[1]};
      *reinterpret_cast<bf16x4*>(dKg + 32 * db + 8 * g4 + 4 * hh) = out;
      lo = pack_bf16(dv_acc[db][4 * g4], dv_acc[db][4 * g4 + 1]);
      hi = pack_bf16(dv_acc[db][4 * g4 + 2], dv_acc[db][4 * g4 + 3]);
      const bf16x4 out2 = {lo[0], lo[1], hi[0], hi[1]};
      *reinterpret_cast<bf16x4*>(dVg + 32 * db + 8 * g4 + 4 * hh) = out2;
    }
  }
}

template <int SCORE, bool EXPORT, bool AB = true>
static int launch_dkv_wide_on(const BwdArgs& a, hipStream_t stream) {
  if constexpr (AB && splits_bias(SCORE))
    if (a.score.ab == nullptr) return launch_dkv_wide_on<SCORE, EXPORT, false>(a, stream);
  if constexpr (SCORE == FLEXATTN_SCORE_NONE)
    if (a.score.ab != nullptr) return launch_dkv_wide_on<kScoreBiasOnly, EXPORT>(a, stream);
  using namespace dkv_cfg;
  constexpr int kLds = 8 * kTileElems * 2 + 4 * 4096 + 4 * 64 * 4;   // (Q, dO) x 2 buffers x 2 panels; P, dS; lse, delta x 2 buffers
  auto kern = bwd_dkv_bf16_wide_kernel<SCORE, EXPORT, AB>;
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  if (attr != hipSuccess) return set_error(FLEXATTN_ELAUNCH, "hipFuncSetAttribute(dkv): %s", hipGetErrorString(attr));
  const int n_wg = a.B * a.Hkv * a.map.nk * 2;
  hipLaunchKernelGGL(kern, dim3(n_wg), dim3(256), kLds, stream, a);
  return check_launch("flexattn_bwd_dkv bf16");
}
template <int SCORE>
static int launch_dkv_wide(const BwdArgs& a, hipStream_t stream) {
  return a.ds != nullptr ? launch_dkv_wide_on<SCORE, true>(a, stream) : launch_dkv_wide_on<SCORE, false>(a, stream);
}

#ifndef FLEXATTN_CUSTOM_ONLY
// ------------------------------------------------------------------------------------------------
// Plain score: the whole main loop runs inside generated asm statements (gen_dkv_tile.py).  One
// statement executes a run of consecutive full tiles, or one partial tile with the lane's keep bits;
// C++ only finds the runs, and builds the keep bits of partial tiles.  The kernel has no static
// shared memory, so the dynamic buffer starts at LDS address 0 (the run loop toggles buffers by
// address bits).
// ------------------------------------------------------------------------------------------------
// ALIBI: the score gets slopes[h] (j - i) added (one query head per kv head only).  With j0 the middle of
// the item's kv tile, exp2(t + a (j - i)) = exp2(t - a (i - j0)) 2^(a (j - j0)): the query's share joins
// -lse in the S chain's accumulator input, the key's share is a factor of whole dk / dv rows that the
// item epilogue applies, so the tile streams are those of the plain score.
// SOFTCAP: s' = cap tanh(s / cap).  The streams turn the chain's result times 2 log2(e) sm_scale / cap, u, into r = 1 / (2^u + 1) (tanh = 1 - 2 r), the exponent (cap' - lse) - 2 cap' r with
// cap' = cap log2(e) (LDS holds cap' - lse) and dS = P dP' r (1 - r); the factor 4 of 1 - tanh^2 = 4 r (1 - r)
// goes into dk with sm_scale.
// DOCS: the mask compares document ids; those of a partial q tile are staged through LDS (stage_doc_ids).
// (A template parameter: the staging code in the kernel costs the other masks registers.)
// EXPORT: the streams also write the step's bf16 dS (without sm_scale, as the dk product takes it) to a.ds, one
// 32 KB block per (query head, kept tile pair) at (head a.ds_pairs + a.ds_col[kv tile] + place of the q tile in the
// kv tile's list) 32 KB (the index of flexattn_build_ds_index: skipped pairs take no room); inside a block wave w
// (kv columns 32 w + L % 32) writes 1 KB per (32-row q block c, 16-row half u) at 8192 w + 1024 (2 c + u), lane L
// its 8 values (rows 8 (e / 4) + 4 (L / 32) + e % 4 of the half) at 16 (2 (L % 32) + L / 32).  bwd_dq_ds.hip reads it.
// HD: head dimension 128, or 64 (plain scores without export; see the forward).
template <int SCORE, bool DOCS, bool EXPORT = false, int HD = 128>
__global__ __launch_bounds__(256, 1) void bwd_dkv_bf16_d128_plain_kernel(BwdArgs a) {
  using namespace dkv_cfg;
  constexpr int D = HD;
  static_assert(HD == 128 || (SCORE == FLEXATTN_SCORE_NONE && !EXPORT), "streams of head dimension 64: plain scores");
  static_assert(!(EXPORT && SCORE == FLEXATTN_SCORE_ALIBI), "the position-bias streams keep the key's share out of dS");
  constexpr bool ALIBI = SCORE == FLEXATTN_SCORE_ALIBI;
  constexpr bool SOFTCAP = SCORE == FLEXATTN_SCORE_SOFTCAP;
  const float cap2 = SOFTCAP ? a.score.cap * kLog2e : 0.f;
  extern __shared__ __attribute__((aligned(1024))) char smem_raw[];
  bf16_t* sT = reinterpret_cast<bf16_t*>(smem_raw);
  float* sLse = reinterpret_cast<float*>(sT + 8 * kTileElems);
  float* sDl = sLse + 2 * BQ;

  const int nKb = a.map.nk;
  const int nQ = a.map.nq;
  const int n_wg = a.B * a.Hkv * nKb;
  const int group = a.Hq / a.Hkv;
  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int l32 = lane & 31;
  const int hh = lane >> 5;

  // One work-group per CU when the launcher found a balanced static schedule (persistent_ok):
  // it then runs n_wg / gridDim.x work items back to back, which saves the gap between the end of a
  // work-group and the start of the next one on the CU (only one fits at a time).
  const int n_items = n_wg / (int)gridDim.x;
  const int kv_local = w * 32 + l32;
  const int row = tid & (BQ - 1);
  // waves 0, 1 turn (l, m) into -lse for rows tid & 127; waves 2, 3 store -delta
  const bool lse_wave = w < 2;
  int* sIdx = reinterpret_cast<int*>(sDl + 2 * BQ) + 4 * 32;
  unsigned char* sPart = reinterpret_cast<unsigned char*>(sIdx + MAX_LIST);  // by q tile: 1 = partial with this kv tile
  TileLoader<4, HD> loader;
  loader.init(w, lane);

  // An item is kv tile kb of (batch, kv head) pair bhk.  Its addresses are cheap to derive from the
  // two numbers, so only those are carried from item to item.
  struct Geometry {
    int bhk, kb;
  };
  const PersistentPlan plan = persistent_plan((int)blockIdx.x, (int)gridDim.x, n_wg, nKb);
  // under document masks a persistent work-group takes its items from the longest-first schedule (sorted_items)
  const bool sorted = DOCS && gridDim.x != (unsigned)n_wg;
  int* sItems = reinterpret_cast<int*>(sPart + MAX_LIST) + 4 * 128;
  if (DOCS && sorted)
    sorted_items([&](int t) { return a.map.cnt[t]; }, nKb, n_wg / nKb, 1, (int)blockIdx.x, n_items, tid,
                 reinterpret_cast<int*>(smem_raw), sItems);
  auto geometry = [&](int item) {
    Geometry g;
    if (DOCS && sorted) {
      const int v = sItems[item];
      g.bhk = v >> 16;
      g.kb = v & 0xffff;
    } else {
      persistent_item(plan, item, (int)gridDim.x, n_wg, nKb, g.bhk, g.kb);
    }
    g.bhk = __builtin_amdgcn_readfirstlane(g.bhk);
    g.kb = __builtin_amdgcn_readfirstlane(g.kb);
    return g;
  };
  auto kv_base = [&](const Geometry& g) { return tile_base(g.kb, BNK, a.Sk); };
  auto kv_offset = [&](const Geometry& g) { return ((size_t)g.bhk * a.Sk + (size_t)kv_base(g)) * D; };
  const bool ragged_q = nQ * BQ != a.Sq;   // (the last q tile then shares rows with the one before: always masked)
  // (DOCS) document arrays given per batch entry: the rows of the entry of a (batch, kv head) pair
  auto doc_rows = [&](int bhk, int S) { return (DOCS && a.mask.doc_batched) ? (size_t)(bhk / a.Hkv) * (size_t)S : (size_t)0; };
  // (EXPORT) dS block of the item's kv tile against the first q tile of its list, for the group's first query
  // head: the blocks of a head are ordered kv tile by kv tile (a.ds_col[kb] pairs lie before kv tile kb), and
  // along each kv tile's q list
  auto ds_base = [&](const Geometry& g) {
    const int first = __builtin_amdgcn_readfirstlane(a.ds_col[g.kb]);
    return static_cast<char*>(a.ds) + (((size_t)g.bhk * group) * (size_t)a.ds_pairs + (size_t)first) * kDsBlockBytes;
  };
  // first row of the group's first query head: (b Hq + hk group) Sq with bhk = b Hkv + hk
  auto first_row = [&](const Geometry& g) { return (size_t)g.bhk * group * a.Sq; };

  // Everything an item needs from global memory before its first step is fetched while the previous
  // item runs: plain loads whose values are not touched until that item's last step is done.  (They
  // live in v[192:255] and the low registers, which the run loop leaves alone.)
  constexpr int kListRegs = PREFETCH_LIST / 256;
  struct ItemRegs {
    RowBlock k, v;                 // the wave's 32 K / V rows (full-row layout, see rows_load)
    int doc, n_tiles, qb0;         // list length and its first entry
    int qlo, qhi;                  // (DOCS) first and last q position that carries the column's document id, where known
    float na2;                     // -slopes[head] log2(e) (ALIBI)
    int idx[kListRegs];            // q list entries tid + 256 j
    unsigned char part[kListRegs]; // state of q tile tid + 256 j against this kv tile
  };
  // (opaque(): addresses derived from its result are computed where they are used instead of once
  // before the item loop, where they would have to be kept, spilled, through every run)
  auto opaque = [](int x) {
    asm volatile("" : "+v"(x));
    return x;
  };
  auto fetch = [&](const Geometry& g, ItemRegs& r) {
    const int tid_here = opaque(tid);
    const bf16_t* Kg = static_cast<const bf16_t*>(a.k) + kv_offset(g);
    const bf16_t* Vg = static_cast<const bf16_t*>(a.v) + kv_offset(g);
    rows_load<HD>(r.k, Kg + (size_t)(tid_here >> 6) * 32 * D, tid_here & 63);
    rows_load<HD>(r.v, Vg + (size_t)(tid_here >> 6) * 32 * D, tid_here & 63);
    const size_t dk_rows = doc_rows(g.bhk, a.Sk);
    r.doc = (a.mask.flags & FLEXATTN_MASK_DOC) ? a.mask.doc_k[dk_rows + kv_base(g) + kv_local] : 0;
    if constexpr (DOCS) {
      const bool have = a.mask.doc_k_range != nullptr;
      r.qlo = have ? a.mask.doc_k_range[2 * (dk_rows + kv_base(g) + kv_local)] : 0;
      r.qhi = have ? a.mask.doc_k_range[2 * (dk_rows + kv_base(g) + kv_local) + 1] : 0;
    }
    const int* tile_idx = a.map.idx + (size_t)g.kb * nQ;
    r.n_tiles = a.map.cnt[g.kb];
    r.qb0 = tile_idx[0];  // (nQ >= 1: always readable; used only if the list is not empty)
    r.na2 = ALIBI ? -a.score.slopes[g.bhk % a.Hkv] * kLog2e : 0.f;
#pragma unroll
    for (int j = 0; j < kListRegs; ++j) {
      const int t = tid_here + 256 * j;
      r.idx[j] = (t < nQ) ? tile_idx[t] : 0;  // (slots past the list length hold no valid entry and are never used)
      r.part[j] = (t < nQ) ? a.map.state[(size_t)t * a.map.nk + g.kb] : 0;
    }
  };
  // What is left of an item's fetched values once its K / V fragments sit in their registers.
  struct ItemHead {
    int doc, n_tiles, qb0, qlo, qhi;
    float na2;
    int idx[kListRegs];
    unsigned char part[kListRegs];
  };
  PinnedState st;
  // The streams multiply the fp32 products Q K^T by c2 (sm_scale * log2(e); softcap: 2 log2(e) sm_scale / cap)
  // on their way into the exponent; K itself goes in as it is.
  const float c2 = SOFTCAP ? 2.f * kLog2e * a.sm_scale / a.score.cap : a.sm_scale * kLog2e;
  auto scaled = [](unsigned two) { return two; };
  // (`stage`: the wave's 16 KB of a free LDS step buffer)
  auto consume = [&](const ItemRegs& r, ItemHead& c, char* stage) {
    u32x4 kw[8], vw[8];
    const int lane_here = opaque(lane);
    rows_to_fragments<HD>(r.k, stage, lane_here, kw);
    rows_to_fragments<HD>(r.v, stage + 8192, lane_here, vw);
#define FA_PUT(KS, KR, VR)                                                                                    \
  asm volatile(FA_DKV_PUT_KV_##KS                                                                             \
               : "={" KR "}"(st.k[KS]), "={" VR "}"(st.v[KS])                                                 \
               : "v"(scaled(kw[KS][0])), "v"(scaled(kw[KS][1])), "v"(scaled(kw[KS][2])), "v"(scaled(kw[KS][3])), \
                 "v"(vw[KS][0]), "v"(vw[KS][1]), "v"(vw[KS][2]), "v"(vw[KS][3]));
    FA_PUT(0, "a[128:131]", "a[160:163]") FA_PUT(1, "a[132:135]", "a[164:167]")
    FA_PUT(2, "a[136:139]", "a[168:171]") FA_PUT(3, "a[140:143]", "a[172:175]")
    FA_PUT(4, "a[144:147]", "a[176:179]") FA_PUT(5, "a[148:151]", "a[180:183]")
    FA_PUT(6, "a[152:155]", "a[184:187]") FA_PUT(7, "a[156:159]", "a[188:191]")
#undef FA_PUT
    c.doc = r.doc;
    if constexpr (DOCS) { c.qlo = r.qlo; c.qhi = r.qhi; }
    c.n_tiles = __builtin_amdgcn_readfirstlane(r.n_tiles);
    c.qb0 = __builtin_amdgcn_readfirstlane(r.qb0);
    c.na2 = ALIBI ? __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, r.na2))) : 0.f;
#pragma unroll
    for (int j = 0; j < kListRegs; ++j) {
      c.idx[j] = r.idx[j];
      c.part[j] = r.part[j];
    }
  };

  // Byte addresses of the lane's operand fragments and row values in LDS step buffer 0 (see
  // tile_io.hpp); the run loop flips them between the two buffers together with `buf`, across items too.
  const int r_sw = swz(l32);
  const int t_row = 4 * hh + ((lane & 15) >> 2);
  const int t_chunk = 2 * ((lane & 31) >> 4) + ((lane & 3) >> 1);
  const int t_half = 4 * (lane & 1);
  const unsigned base0 = (unsigned)(size_t)sT;
  unsigned ra[8], ta[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) ra[ks] = base0 + (unsigned)(l32 * kTileD + (((2 * ks + hh) ^ r_sw) << 3)) * 2u;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    ta[i] = base0 + (unsigned)(tile_off(t_row + 8 * (i & 1), 4 * (i >> 1) + t_chunk) + t_half) * 2u;
  unsigned la = (unsigned)(size_t)(sLse + 4 * hh);
  unsigned lw = (unsigned)(size_t)((lse_wave ? sLse : sDl) + BQ + row);  // this lane's row value of the NEXT buffer
  int buf = 0;
  bool resident = false;  // the item's first step was already copied into buffer `buf` by the previous item's last step

  ItemRegs pre;
  ItemHead cur;
  Geometry geo = geometry(0);
  fetch(geo, pre);
  consume(pre, cur, reinterpret_cast<char*>(sT + 4 * kTileElems) + w * 16384);

  for (int item = 0; item < n_items; ++item) {
  const int kb = geo.kb;
  const int k0 = kv_base(geo);
  const int k_idx = k0 + kv_local;
  const size_t kv_off = kv_offset(geo);
  const size_t rows0 = first_row(geo);
  const bf16_t* Qg = static_cast<const bf16_t*>(a.q) + rows0 * D;
  const bf16_t* dOg = static_cast<const bf16_t*>(a.dout) + rows0 * D;
  const float* rowa = (lse_wave ? a.l : a.delta) + rows0;
  const float* rowb = (lse_wave ? a.m : a.delta) + rows0;
  const int doc_j = cur.doc;
  // (DOCS) with sorted q ids the queries of the column's document are one interval: the keep bits of a partial tile
  // then have a closed form (keep_bits32_range) and no ids are read
  const bool ranged = DOCS && a.mask.doc_k_range != nullptr && keep_bits_have_range(a.mask);
  const int* tile_idx = a.map.idx + (size_t)kb * nQ;
  const int n_tiles = cur.n_tiles;
  const int n_iter = n_tiles * group;
  const float na2 = cur.na2;
  const int kc = k0 + BNK / 2;  // j0
  if (item > 0) __syncthreads();  // the previous item's list and row values are dead from here

  asm volatile(FA_DKV_ZERO_ACC
               : "={a[0:15]}"(st.dv[0]), "={a[16:31]}"(st.dv[1]), "={a[32:47]}"(st.dv[2]), "={a[48:63]}"(st.dv[3]),
                 "={a[64:79]}"(st.dk[0]), "={a[80:95]}"(st.dk[1]), "={a[96:111]}"(st.dk[2]), "={a[112:127]}"(st.dk[3]));

  // The kv tile's q list and which q tiles are partial against it, cached in LDS: finding runs of
  // full tiles then costs no global loads.
  const int tid_p = opaque(tid);  // (fresh per item: see opaque())
#pragma unroll
  for (int j = 0; j < kListRegs; ++j) {
    const int t = tid_p + 256 * j;
    if (t < nQ) {
      sIdx[t] = cur.idx[j];
      sPart[t] = (cur.part[j] == 1 || (ragged_q && t == nQ - 1)) ? 1 : 0;
    }
  }
  if (nQ > PREFETCH_LIST) {
    // columns longer than the prefetched part (more than 131072 tokens): the rest straight from global memory
    // (an item is then thousands of steps long: the wait does not show)
    for (int t = PREFETCH_LIST + tid_p; t < nQ; t += 256) {
      sIdx[t] = tile_idx[t];
      sPart[t] = (a.map.state[(size_t)t * a.map.nk + kb] == 1 || (ragged_q && t == nQ - 1)) ? 1 : 0;
    }
  }
  if (n_iter > 0 && !resident) {
    // first step into the current buffer: tiles (LDS-direct) and the lane's row value
    const size_t r0 = (size_t)tile_base(cur.qb0, BQ, a.Sq);
    bf16_t* dst = sT + (size_t)buf * 4 * kTileElems;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      loader.load(Qg + (r0 + half * kTileRows) * D, dst + half * kTileElems);
      loader.load(dOg + (r0 + half * kTileRows) * D, dst + (2 + half) * kTileElems);
    }
    const int row_p = tid_p & (BQ - 1);
    const float x = rowa[r0 + row_p], y = rowb[r0 + row_p];
    if (lse_wave) {  // (the streams want -lse: it is the accumulator input of the S chain)
      // (one fused multiply-add, as the streams' turn-around rounds the row values of every later step: an item's
      // results then do not depend on whether its first step was set up here or by the last step of the item before it)
      float neg_lse = (x > 0.f) ? -__builtin_fmaf(y, kLog2e, log2f(x)) : -__builtin_huge_valf();
      if (ALIBI) neg_lse = __builtin_fmaf((float)((int)r0 + row_p - kc), na2, neg_lse);
      if (SOFTCAP) neg_lse += cap2;
      sLse[buf * BQ + row_p] = neg_lse;
    } else {  // (and -delta, for the dP chain)
      sDl[buf * BQ + row_p] = -x;
    }
    wait_vmem_all();
  }
  resident = false;
  __syncthreads();
  // The next item's list lands while this item runs.  (The last item fetches itself again: every
  // path then redefines the fetched registers, so none of them has to live through the run loop.)
  const bool has_next = item + 1 < n_items;
  const Geometry geo_n = has_next ? geometry(item + 1) : geo;
  fetch(geo_n, pre);

  const unsigned tid4 = (unsigned)row * 4u;
  // (EXPORT) first dS block of this item and of the next one
  const size_t ds_item = EXPORT ? (size_t)ds_base(geo) : 0;
  const size_t ds_item_n = EXPORT ? (size_t)ds_base(geo_n) : 0;
  // Work-group constants of the run loop, one 32-dword table per wave behind the row values
  // (order: TABLE in gen_dkv_tile.py; the second half names the next item's first step, see below).
  // Written and read by the same wave: no barrier needed.
  unsigned* tbl = reinterpret_cast<unsigned*>(sDl + 2 * BQ) + w * 32;
  if (lane == 0) {
    tbl[0] = (unsigned)n_tiles;
    tbl[1] = (unsigned)(group - 1);
    tbl[2] = (unsigned)a.Sq;
    tbl[3] = base0 + (unsigned)w * 4096u;  // LDS address of the wave's first 1 KB block in buffer 0
    tbl[4] = __builtin_bit_cast(unsigned, SOFTCAP ? cap2 : na2);
    tbl[5] = lse_wave ? 1u : 0u;
    tbl[6] = (unsigned)(size_t)tile_idx;
    tbl[7] = (unsigned)((size_t)tile_idx >> 32);
    tbl[8] = (unsigned)(size_t)Qg;
    tbl[9] = (unsigned)((size_t)Qg >> 32);
    tbl[10] = (unsigned)(size_t)dOg;
    tbl[11] = (unsigned)((size_t)dOg >> 32);
    tbl[12] = (unsigned)(size_t)rowa;
    tbl[13] = (unsigned)((size_t)rowa >> 32);
    tbl[14] = (unsigned)(size_t)rowb;
    tbl[15] = (unsigned)((size_t)rowb >> 32);
    if (EXPORT) {
      const size_t ds0 = ds_item;
      tbl[28] = (unsigned)ds0;
      tbl[29] = (unsigned)(ds0 >> 32);
      tbl[30] = (unsigned)a.ds_pairs;   // blocks per query head
      tbl[31] = 0u;
    }
  }
  const unsigned tbl_addr = (unsigned)(size_t)tbl;

  // Step `it` is q tile tile_idx[it % n_tiles] of query head it / n_tiles of the group.  Carried:
  // the list positions of steps it + 1 and it + 2, the head of step it + 1, its q block index.
  int it = 0, g1 = 0, p1 = 1, p2 = 2;
  if (p1 >= n_tiles) { p1 -= n_tiles; g1 = 1; }
  if (p2 >= n_tiles) p2 -= n_tiles;
  if (p2 >= n_tiles) p2 -= n_tiles;
  int qb1 = (n_iter > 0) ? __builtin_amdgcn_readfirstlane(sIdx[p1]) : 0;

  while (it < n_iter) {
    // position of step `it` in the list, its q block and state
    int p0 = p1 - 1;
    if (p0 < 0) p0 += n_tiles;
    const int qb = __builtin_amdgcn_readfirstlane(sIdx[p0]);
    const bool partial = __builtin_amdgcn_readfirstlane((int)sPart[qb]) == 1;
    int it_end = it + 1;
    unsigned km[2] = {0u, 0u};
    if (partial) {
      // the lane's keep bits: element e of q block c sits at bit 16 (c & 1) + e of km[c >> 1]
      const int q0 = tile_base(qb, BQ, a.Sq);
      if constexpr (DOCS) {
        int* sDoc = reinterpret_cast<int*>(sPart + MAX_LIST) + w * 128;  // the wave's stage for document ids
        if (ranged) {
#pragma unroll
          for (int half = 0; half < 2; ++half)
            km[half] = keep_bits32_range<false>(a.mask, k_idx, q0 + 64 * half + 4 * hh, cur.qlo, cur.qhi);
        } else {
          stage_doc_ids(a.mask.doc_q + doc_rows(geo.bhk, a.Sq), q0, q0 + 64, lane, sDoc);
#pragma unroll
          for (int half = 0; half < 2; ++half)
            km[half] = keep_bits32_staged<false>(a.mask, k_idx, q0 + 64 * half + 4 * hh, doc_j, sDoc + 64 * half + 4 * hh);
        }
      } else {
#pragma unroll
        for (int half = 0; half < 2; ++half)
          km[half] = keep_bits32<false>(a.mask, k_idx, q0 + 64 * half + 4 * hh, doc_j, a.mask.doc_q);
      }
      // (rows and columns that the last tiles of ragged lengths share with the tiles before them: those own them.  opaque():
      // what only these tiles need is not kept through the runs)
      if (q0 != qb * BQ || k0 != kb * BNK) {
#pragma unroll
        for (int half = 0; half < 2; ++half)
          km[half] = opaque(kv_local) < kb * BNK - k0 ? 0u : km[half] & keep_bits_from(qb * BQ - q0 - 64 * half - 4 * (opaque(lane) >> 5));
      }
    } else {
      // the run of full tiles ends before the next partial one: lanes look 64 steps ahead at a time
      bool found = false;
      while (!found && it_end < n_iter) {
        const int j = it_end + lane;
        bool is_partial = false;
        if (j < n_iter) {
          const int pj = (p0 + (j - it)) % n_tiles;
          is_partial = sPart[sIdx[pj]] == 1;
        }
        const unsigned long long hits = __ballot(is_partial);
        if (hits != 0ull) {
          it_end += __builtin_ctzll(hits);
          found = true;
        } else {
          it_end = (it_end + 64 < n_iter) ? it_end + 64 : n_iter;
        }
      }
    }
    it_end = __builtin_amdgcn_readfirstlane(it_end);
    // The run that ends the item copies the next item's first step during its last step (bit 1 of
    // the flags; the table's second half says where it is).  The fetched values are first touched
    // here, an item's length after their loads were issued.
    int flags = partial ? 1 : 0;
    if (it_end == n_iter && has_next) {
      const int nt = __builtin_amdgcn_readfirstlane(pre.n_tiles);
      if (nt > 0) {
        flags |= 2;
        const int qb0_n = __builtin_amdgcn_readfirstlane(pre.qb0);
        const size_t rows_n = first_row(geo_n);
        const bf16_t* Qg_n = static_cast<const bf16_t*>(a.q) + rows_n * D;
        const bf16_t* dOg_n = static_cast<const bf16_t*>(a.dout) + rows_n * D;
        const float* rowa_n = (lse_wave ? a.l : a.delta) + rows_n;
        const float* rowb_n = (lse_wave ? a.m : a.delta) + rows_n;
        if (lane == 0) {
          tbl[16] = (unsigned)(size_t)Qg_n;
          tbl[17] = (unsigned)((size_t)Qg_n >> 32);
          tbl[18] = (unsigned)(size_t)dOg_n;
          tbl[19] = (unsigned)((size_t)dOg_n >> 32);
          tbl[20] = (unsigned)(size_t)rowa_n;
          tbl[21] = (unsigned)((size_t)rowa_n >> 32);
          tbl[22] = (unsigned)(size_t)rowb_n;
          tbl[23] = (unsigned)((size_t)rowb_n >> 32);
          tbl[24] = (unsigned)qb0_n;
          if (ALIBI) {
            tbl[26] = __builtin_bit_cast(unsigned, pre.na2);
            tbl[27] = (unsigned)(kv_base(geo_n) + BNK / 2);
          }
          if (EXPORT) {
            const size_t ds_n = ds_item_n;
            tbl[26] = (unsigned)ds_n;
            tbl[27] = (unsigned)(ds_n >> 32);
          }
        }
        resident = true;
      }
    }
    // no scalar operands (see gen_dkv_tile.py): the loop state travels in VGPRs
#define FA_DKV_CALL(RUN, CLOB_MORE, ...)                                                                                 \
  asm volatile(RUN                                                                                               \
               : FA_DKV_PINNED(st), [it] "+v"(it), [p1] "+v"(p1), [g1] "+v"(g1), [p2] "+v"(p2), [qb1] "+v"(qb1), \
                 [buf] "+v"(buf), [r0] "+v"(ra[0]), [r1] "+v"(ra[1]), [r2] "+v"(ra[2]), [r3] "+v"(ra[3]),       \
                 [r4] "+v"(ra[4]), [r5] "+v"(ra[5]), [r6] "+v"(ra[6]), [r7] "+v"(ra[7]), [t0] "+v"(ta[0]),       \
                 [t1] "+v"(ta[1]), [t2] "+v"(ta[2]), [t3] "+v"(ta[3]), [t4] "+v"(ta[4]), [t5] "+v"(ta[5]),       \
                 [t6] "+v"(ta[6]), [t7] "+v"(ta[7]), [la] "+v"(la), [lw] "+v"(lw)                                \
               : [it_end] "v"(it_end), [partial] "v"(flags), [tbl] "v"(tbl_addr), [g0] "v"(loader.goff[0]),      \
                 [g1v] "v"(loader.goff[1]), [g2] "v"(loader.goff[2]), [g3] "v"(loader.goff[3]), [m0] "v"(km[0]), \
                 [m1] "v"(km[1]), [tid4] "v"(tid4), [c2v] "v"(c2), ##__VA_ARGS__                                                \
               : "memory", "scc", "vcc", "m0", FA_DKV_RUN_SGPRS, "v67", FA_DKV_TILE_CLOBBERS CLOB_MORE)
#define FA_DKV_ALIBI_CLOBBERS , "s101"
#define FA_DKV_D64_CLOBBERS , "v200", "v201", "v202", "v203"
#define FA_DKV_DS_CLOBBERS , "s52", "s53", "s54", "s55", "s56", "s57", "s58", "s59"
    if constexpr (EXPORT) {
      // dS block of step `it` (head it / n_tiles of the group, place p0 in the q list) and the lane's place in
      // the wave's part
      const size_t ds_cur = ds_item + ((size_t)(it / n_tiles) * (size_t)a.ds_pairs + (size_t)p0) * kDsBlockBytes;
      const unsigned dslo = (unsigned)ds_cur, dshi = (unsigned)(ds_cur >> 32);
      const unsigned dsv = 8192u * (unsigned)w + 4096u + 16u * (unsigned)(2 * l32 + hh);
      if constexpr (SOFTCAP) {
        const float k2 = -2.f * cap2;
        FA_DKV_CALL(FA_DKV_RUN_SOFTCAP_DS, FA_DKV_ALIBI_CLOBBERS FA_DKV_DS_CLOBBERS, [k2] "v"(k2), [dslo] "v"(dslo),
                    [dshi] "v"(dshi), [dsv] "v"(dsv));
      } else {
        FA_DKV_CALL(FA_DKV_RUN_DS, FA_DKV_DS_CLOBBERS, [dslo] "v"(dslo), [dshi] "v"(dshi), [dsv] "v"(dsv));
      }
    } else if constexpr (ALIBI) {
      FA_DKV_CALL(FA_DKV_RUN_ALIBI, FA_DKV_ALIBI_CLOBBERS, [kc] "v"(kc));
    } else if constexpr (SOFTCAP) {
      const float k2 = -2.f * cap2;
      FA_DKV_CALL(FA_DKV_RUN_SOFTCAP, FA_DKV_ALIBI_CLOBBERS, [k2] "v"(k2));
    } else {
      if constexpr (HD == 64) { FA_DKV_CALL(FA_DKV_RUN_D64, FA_DKV_D64_CLOBBERS); } else { FA_DKV_CALL(FA_DKV_RUN, ); }
    }
#undef FA_DKV_CALL
#undef FA_DKV_DS_CLOBBERS
#undef FA_DKV_ALIBI_CLOBBERS
#undef FA_DKV_D64_CLOBBERS
    it = __builtin_amdgcn_readfirstlane(it);
    p1 = __builtin_amdgcn_readfirstlane(p1);
    buf = __builtin_amdgcn_readfirstlane(buf);
  }

  // ---- item epilogue ----
  // The next item's K / V fragments go into their registers before this item's stores are issued
  // (their loads are long done; behind the stores the wait would include the stores).
  // (buffer `buf` may hold the next item's first step: the other one is free)
  char* stage = reinterpret_cast<char*>(sT + (size_t)(buf ^ 1) * 4 * kTileElems) + w * 16384;
  consume(pre, cur, stage);

  // dk / dv: bf16 rows staged through the wave's 16 KB of the free LDS step buffer (16-byte chunks XOR-swizzled
  // by row), so that every store instruction writes four complete 256-byte rows.
  {
    const int lane_here = opaque(lane);
    const int row_here = lane_here & 31;
    const unsigned wr = (unsigned)row_here * 256u + 8u * (unsigned)(lane_here >> 5);
#define FA_GET(T, SRC, REG, MAT, DB, SCALE)                                                                        \
  if constexpr (32 * DB < HD) {                                                                                                                \
    float x[16];                                                                                                   \
    asm volatile(FA_DKV_GET_ACC_##T                                                                                \
                 : "=v"(x[0]), "=v"(x[1]), "=v"(x[2]), "=v"(x[3]), "=v"(x[4]), "=v"(x[5]), "=v"(x[6]), "=v"(x[7]), \
                   "=v"(x[8]), "=v"(x[9]), "=v"(x[10]), "=v"(x[11]), "=v"(x[12]), "=v"(x[13]), "=v"(x[14]),        \
                   "=v"(x[15])                                                                                     \
                 : "{" REG "}"(SRC));                                                                              \
    _Pragma("unroll") for (int g = 0; g < 4; ++g) {                                                                \
      const bf16x2 lo = pack_bf16(x[4 * g] * SCALE, x[4 * g + 1] * SCALE);                                         \
      const bf16x2 hi = pack_bf16(x[4 * g + 2] * SCALE, x[4 * g + 3] * SCALE);                                     \
      const bf16x4 out = {lo[0], lo[1], hi[0], hi[1]};                                                             \
      *reinterpret_cast<bf16x4*>(stage + MAT * 8192 + wr + (unsigned)(((4 * DB + g) ^ (row_here & 15)) << 4)) = out; \
    }                                                                                                              \
  }
    // the streams leave the constant sm_scale out of dS: dk takes it here; and both take the key's
    // share of a position bias
    const float ej = ALIBI ? exp2f(-na2 * (float)((lane_here & 31) + 32 * w - BNK / 2)) : 1.f;
    const float ek = (SOFTCAP ? 4.f : 1.f) * a.sm_scale * ej;
    FA_GET(0, st.dv[0], "a[0:15]", 1, 0, ej) FA_GET(1, st.dv[1], "a[16:31]", 1, 1, ej)
    FA_GET(2, st.dv[2], "a[32:47]", 1, 2, ej) FA_GET(3, st.dv[3], "a[48:63]", 1, 3, ej)
    FA_GET(4, st.dk[0], "a[64:79]", 0, 0, ek) FA_GET(5, st.dk[1], "a[80:95]", 0, 1, ek)
    FA_GET(6, st.dk[2], "a[96:111]", 0, 2, ek) FA_GET(7, st.dk[3], "a[112:127]", 0, 3, ek)
#undef FA_GET
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    bf16_t* dKg = static_cast<bf16_t*>(a.dk) + kv_off + (size_t)(w * 32) * D;
    bf16_t* dVg = static_cast<bf16_t*>(a.dv) + kv_off + (size_t)(w * 32) * D;
    const int r_first = kb * BNK - k0 - w * 32;   // (rows before it belong to the kv tile before)
    rows_store<HD, 2>(stage, {dKg, dVg}, lane_here, r_first);
  }
  geo = geo_n;
  }  // work items
}

#endif  // FLEXATTN_CUSTOM_ONLY

template <int SCORE, bool EXPORT, bool AB = true, bool DAB = false>
static int launch_dkv_on(const BwdArgs& a, hipStream_t stream) {
  if constexpr (AB && splits_bias(SCORE))
    if (a.score.ab == nullptr) return launch_dkv_on<SCORE, EXPORT, false>(a, stream);
  if constexpr (EXPORT && AB && !DAB && SCORE != FLEXATTN_SCORE_NONE)
    if (a.dab != nullptr) return launch_dkv_on<SCORE, true, true, true>(a, stream);   // (the caller has checked that there is a bias)
  using namespace dkv_cfg;
  auto kern = bwd_dkv_bf16_d128_kernel<SCORE, EXPORT, AB, DAB>;
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, LOOP_LDS_BYTES);
  if (attr != hipSuccess) return set_error(FLEXATTN_ELAUNCH, "hipFuncSetAttribute(dkv): %s", hipGetErrorString(attr));
  const int n_wg = a.B * a.Hkv * a.map.nk;
  hipLaunchKernelGGL(kern, dim3(n_wg), dim3(512), LOOP_LDS_BYTES, stream, a);
  return check_launch("flexattn_bwd_dkv bf16");
}
template <int SCORE>
static int launch_dkv(const BwdArgs& a, hipStream_t stream) {
  if constexpr (SCORE == FLEXATTN_SCORE_NONE)
    if (a.score.ab != nullptr) return launch_dkv<kScoreBiasOnly>(a, stream);
  return a.ds != nullptr ? launch_dkv_on<SCORE, true>(a, stream) : launch_dkv_on<SCORE, false>(a, stream);
}

#ifndef FLEXATTN_CUSTOM_ONLY
template <int SCORE, bool DOCS, bool EXPORT, int HD = 128>
static int launch_dkv_plain_on(const BwdArgs& a, hipStream_t stream) {
  using namespace dkv_cfg;
  auto kern = bwd_dkv_bf16_d128_plain_kernel<SCORE, DOCS, EXPORT, HD>;
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
  if (attr != hipSuccess) return set_error(FLEXATTN_ELAUNCH, "hipFuncSetAttribute(dkv): %s", hipGetErrorString(attr));
  const int n_wg = a.B * a.Hkv * a.map.nk;
  // (persistent_ok's schedule balances masks whose work per tile is linear in the tile index; document
  // masks take the longest-first schedule of sorted_items; what fits neither runs one item per work-group)
  const bool persistent = DOCS ? sorted_schedule_ok(n_wg, a.map.nk) : persistent_ok(n_wg, a.map.nk);
  const int grid = (persistent && n_wg > 256) ? 256 : n_wg;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), LDS_BYTES, stream, a);
  return check_launch("flexattn_bwd_dkv bf16");
}

template <int SCORE>
static int launch_dkv_plain(const BwdArgs& a, hipStream_t stream) {
  if constexpr (SCORE != FLEXATTN_SCORE_ALIBI) {
    if (a.ds != nullptr)
      return (a.mask.flags & FLEXATTN_MASK_DOC) ? launch_dkv_plain_on<SCORE, true, true>(a, stream)
                                                : launch_dkv_plain_on<SCORE, false, true>(a, stream);
  }
  return (a.mask.flags & FLEXATTN_MASK_DOC) ? launch_dkv_plain_on<SCORE, true, false>(a, stream)
                                            : launch_dkv_plain_on<SCORE, false, false>(a, stream);
}

#endif  // FLEXATTN_CUSTOM_ONLY

// Whether a request runs the generated-stream dk/dv kernel (else the one with a compiled main loop): the stream
// caches the q tile list in LDS, has no additive bias, serves the global position bias for one query head per kv
// head only, and a functor library of a compiled score function has no streams at all.
bool bwd_dkv_bf16_d128_on_stream(int kind, int flags, int nq, bool has_ab, int Hq, int Hkv) {
#ifdef FLEXATTN_CUSTOM_ONLY
  (void)kind; (void)flags; (void)nq; (void)has_ab; (void)Hq; (void)Hkv;
  return false;
#else
  const bool stream_ok = !(flags & FLEXATTN_FLAG_COMPILED_LOOP) && nq <= dkv_cfg::MAX_LIST && !has_ab;
  switch (kind) {
    case FLEXATTN_SCORE_NONE:
    case FLEXATTN_SCORE_SOFTCAP: return stream_ok;
    case FLEXATTN_SCORE_ALIBI: return stream_ok && Hq == Hkv;
  }
  return false;
#endif
}

int bwd_dkv_bf16_d128(const BwdArgs& a, hipStream_t stream) {
#ifdef FLEXATTN_CUSTOM_ONLY
  switch (a.score.kind) {
    case FLEXATTN_SCORE_NONE: return launch_dkv<FLEXATTN_SCORE_NONE>(a, stream);
    case FLEXATTN_SCORE_CUSTOM: return launch_dkv<FLEXATTN_SCORE_CUSTOM>(a, stream);
  }
  return set_error(FLEXATTN_ENOTSUP, "this functor library holds the plain and the compiled score function only (kind %d asked)", a.score.kind);
#else
  const bool on_stream = bwd_dkv_bf16_d128_on_stream(a.score.kind, a.flags, a.map.nq, a.score.ab != nullptr, a.Hq, a.Hkv);
  switch (a.score.kind) {
    case FLEXATTN_SCORE_NONE:
      return on_stream ? launch_dkv_plain<FLEXATTN_SCORE_NONE>(a, stream) : launch_dkv<FLEXATTN_SCORE_NONE>(a, stream);
    case FLEXATTN_SCORE_ALIBI:
      return on_stream ? launch_dkv_plain<FLEXATTN_SCORE_ALIBI>(a, stream) : launch_dkv<FLEXATTN_SCORE_ALIBI>(a, stream);
    case FLEXATTN_SCORE_SOFTCAP:
      return on_stream ? launch_dkv_plain<FLEXATTN_SCORE_SOFTCAP>(a, stream) : launch_dkv<FLEXATTN_SCORE_SOFTCAP>(a, stream);
    case FLEXATTN_SCORE_ALIBI_TILE: return launch_dkv<FLEXATTN_SCORE_ALIBI_TILE>(a, stream);
  }
  return set_error(FLEXATTN_EINVAL, "unknown score kind %d", a.score.kind);
#endif
}

// Head dim 64: the generated stream for plain scores (the rest: see fwd_bf16_d64).
int bwd_dkv_bf16_d64(const BwdArgs& a, hipStream_t stream) {
#ifndef FLEXATTN_CUSTOM_ONLY
  if (a.score.kind == FLEXATTN_SCORE_NONE && a.ds == nullptr &&
      bwd_dkv_bf16_d128_on_stream(a.score.kind, a.flags, a.map.nq, a.score.ab != nullptr, a.Hq, a.Hkv))
    return (a.mask.flags & FLEXATTN_MASK_DOC) ? launch_dkv_plain_on<FLEXATTN_SCORE_NONE, true, false, 64>(a, stream)
                                              : launch_dkv_plain_on<FLEXATTN_SCORE_NONE, false, false, 64>(a, stream);
#endif
  return set_error(FLEXATTN_ENOTSUP, "bf16 head dim 64: only plain scores without a bias (pad the operands to 128 columns)");
}

// Head dim 256: the kernel with a compiled main loop (two 128-column panels per row), every score kind.
int bwd_dkv_bf16_d256(const BwdArgs& a, hipStream_t stream) {
  switch (a.score.kind) {
    case FLEXATTN_SCORE_NONE: return launch_dkv_wide<FLEXATTN_SCORE_NONE>(a, stream);
#ifdef FLEXATTN_CUSTOM_ONLY
    case FLEXATTN_SCORE_CUSTOM: return launch_dkv_wide<FLEXATTN_SCORE_CUSTOM>(a, stream);
#else
    case FLEXATTN_SCORE_ALIBI: return launch_dkv_wide<FLEXATTN_SCORE_ALIBI>(a, stream);
    case FLEXATTN_SCORE_SOFTCAP: return launch_dkv_wide<FLEXATTN_SCORE_SOFTCAP>(a, stream);
    case FLEXATTN_SCORE_ALIBI_TILE: return launch_dkv_wide<FLEXATTN_SCORE_ALIBI_TILE>(a, stream);
#endif
  }
  return set_error(FLEXATTN_ENOTSUP, "score kind %d is not in this library", a.score.kind);
}

void bwd_dkv_bf16_d128_tile(int* bq, int* bk) {
  *bq = dkv_cfg::BQ;
  *bk = dkv_cfg::BNK;
}

}  // namespace fa
