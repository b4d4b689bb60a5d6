// Forward for few query rows against long keys (token generation), bf16, head dim 64 and 128, plain scores, no mask.
//
// Bound by reading K and V once.  The 128-row tiles of the other forward kernels spend that traffic badly here: one
// query row fills 1/128 of a tile, every query head of a kv head reads the keys again, and B Hq work-groups walk all
// keys each.  Here
//   - the query heads of a kv head are the rows of one tile (they lie one behind the other in memory: row r of kv head
//     h is row h group Sq + r of q, o, l and m), so K and V are read once;
//   - the keys are split over work-groups (decode_splits) and, inside one, over its four waves: tile t of the split
//     belongs to wave t % 4, which keeps its own softmax state; the four are merged through LDS at the end, the splits
//     by a second launch (decode_merge_kernel), both in fp32;
//   - a wave copies its tiles with LDS-direct loads into a ring of its own (two tiles of K and two of V): no barrier
//     in the loop, and 16-24 KB per wave stay in flight, 64-96 KB per CU.
// A tile is 32 LDS rows of 256 bytes: 32 keys at head dim 128, 64 at head dim 64 (key 2 r + p is half p of row r), so
// the copies and reads are the same for both.  Measured (us a call; before: the 128-row kernels): B=8, Hq=32, Hkv=8,
// D=128, 6001 keys, one query each (197 MB) 198 -> 40.8 (4.8 TB/s); the same at D=64 337 -> 24.8; B=1, 32768 keys 929 ->
// 31; B=16, Hq=Hkv=16, 8192 keys, five queries 322 -> 184 (5.8 TB/s); B=32, Hq=64, Hkv=8, 8192 keys, 16 queries (128 rows
// a kv head, the most that comes here) 1935 -> 310.
#include "fa_common.hpp"
#include "launch.hpp"
#include "tile_io.hpp"

namespace fa {

#ifndef FLEXATTN_CUSTOM_HEADER   // (the libraries of compiled closures hold no plain calls)

namespace dec_cfg {
constexpr int ROWS = 32;                    // LDS rows of a tile
constexpr int TILE_BYTES = ROWS * 256;      // 8 KB of K or V
constexpr int WAVE_BYTES = 4 * TILE_BYTES;  // K x2, V x2
constexpr int LDS_BYTES = 4 * WAVE_BYTES + 4 * 64 * 2 * 4;  // four waves' rings, (m, l) of up to 64 rows per wave
constexpr int MAX_ROWS = 128;               // query rows (group Sq) of a kv head
constexpr int MAX_SPLITS = 64;
}  // namespace dec_cfg

struct DecodeArgs {
  const bf16_t* q; const bf16_t* k; const bf16_t* v;
  bf16_t* o; float* l; float* m;
  float* work;    // [splits][heads rows][D] sums, then [splits][heads rows][2] (m, l); unused with one split
  int heads, rows, Sk, splits;   // heads: B Hkv; rows: query rows per kv head
  float sm_scale;
};

__device__ __forceinline__ void decode_copy(const char* g, unsigned dst, const unsigned (&goff)[4]) {
  // eight 1 KB blocks of four rows; rows 16 apart share their swizzle, so four lane offsets serve both halves
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const char* src = g + (i >> 2) * 4096;
    const unsigned to = dst + (unsigned)i * 1024u;
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(goff[i & 3]), "s"(src), "s"(to)
                 : "memory", "m0", "vcc");
  }
}

// NR: blocks of 32 query rows (1 or 2).
template <int D, int NR>
__global__ __launch_bounds__(256, 1) void decode_kernel(DecodeArgs a) {
  using namespace dec_cfg;
  constexpr int P = 128 / D;        // keys per LDS row
  constexpr int KEYS = ROWS * P;    // keys per tile
  constexpr int KS = D / 16;        // steps of a score's contraction
  constexpr int DB = D / 32;        // blocks of 32 output columns
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int l32 = lane & 31, hh = lane >> 5;
  // More than 64 query rows: a second work-group reads the same keys for the rest, eight ids on (ids go round-robin to
  // the XCDs: the same one, at about the same time).  (Four blocks of 32 rows in one wave spill 293 registers.)
  int hs = blockIdx.x, chunk = 0;
  if (a.rows > 64) {
    const int n_hs = a.heads * a.splits;
    if (n_hs % 8 == 0) {
      chunk = (hs >> 3) & 1;
      hs = ((hs >> 4) << 3) | (hs & 7);
    } else {
      chunk = hs & 1;
      hs >>= 1;
    }
  }
  const int head = hs / a.splits;
  const int split = hs % a.splits;
  const int rows = min(a.rows - 64 * chunk, 32 * NR);   // query rows of this work-group
  const int n_all = (a.Sk + KEYS - 1) / KEYS;
  const int t0 = (int)((long long)n_all * split / a.splits), t1 = (int)((long long)n_all * (split + 1) / a.splits);
  const int n = (t1 - t0 - w + 3) >> 2;   // tiles t0 + w, t0 + w + 4, ...; may be 0 or less

  const size_t row0 = (size_t)head * a.rows + 64 * chunk;
  const char* Kg = reinterpret_cast<const char*>(a.k + (size_t)head * a.Sk * D);
  const char* Vg = reinterpret_cast<const char*>(a.v + (size_t)head * a.Sk * D);

  // Q^T fragments: the lane's row, 8 consecutive columns per step (rows beyond the last repeat it)
  bf16x8 q[NR][KS];
#pragma unroll
  for (int nr = 0; nr < NR; ++nr) {
    const int r = min(32 * nr + l32, rows - 1);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
      q[nr][ks] = *reinterpret_cast<const bf16x8*>(a.q + (row0 + r) * D + ks * 16 + hh * 8);
  }
  wait_vmem_all();   // (the loop counts its own copies)

  unsigned goff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    goff[i] = (unsigned)(row * 256 + (((lane & 15) ^ swz(row)) << 4));
  }
  const unsigned ring = (unsigned)(size_t)(__attribute__((address_space(3))) char*)(smem) + (unsigned)w * WAVE_BYTES;
  const char* ring_p = smem + w * WAVE_BYTES;
  // (the last tile of a length that is no multiple of the tile starts early; its first keys are dropped below)
  auto first_key = [&](int it) { return tile_base(t0 + w + 4 * it, KEYS, a.Sk); };
  auto copy_k = [&](int it) { decode_copy(Kg + (size_t)first_key(it) * (2 * D), ring + (it & 1) * TILE_BYTES, goff); };
  auto copy_v = [&](int it) { decode_copy(Vg + (size_t)first_key(it) * (2 * D), ring + (2 + (it & 1)) * TILE_BYTES, goff); };

  const int k_sw = swz(l32);
  unsigned k_off[8], v_off[4][2];
#pragma unroll
  for (int c = 0; c < 8; ++c) k_off[c] = (unsigned)(l32 * 256 + (((2 * c + hh) ^ k_sw) << 4));
  {
    const int t_row = 4 * hh + ((lane & 15) >> 2);
    const int t_chunk = 2 * ((lane & 31) >> 4) + ((lane & 3) >> 1);
    const int t_half = 4 * (lane & 1);
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      v_off[db][0] = (unsigned)(tile_off(t_row, 4 * db + t_chunk) + t_half) * 2u;
      v_off[db][1] = (unsigned)(tile_off(t_row + 8, 4 * db + t_chunk) + t_half) * 2u;
    }
  }

  f32x16 acc[NR][DB];
  float m_run[NR], l_run[NR];
#pragma unroll
  for (int nr = 0; nr < NR; ++nr) {
    m_run[nr] = kNegInf;
    l_run[nr] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[nr][db][e] = 0.f;
  }
  const float c2 = a.sm_scale * kLog2e;

  if (n > 0) { copy_k(0); copy_v(0); }
  if (n > 1) { copy_k(1); copy_v(1); }
  for (int it = 0; it < n; ++it) {
    const int left = n - it;
    // copies behind this K tile: this V tile and, if there is one, the next tile's K and V (8 each)
    if (left > 1) wait_vmem<24>(); else wait_vmem<8>();
    const char* kt = ring_p + (it & 1) * TILE_BYTES;
    const char* vt = ring_p + (2 + (it & 1)) * TILE_BYTES;
    bf16x8 kf[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) kf[c] = *reinterpret_cast<const bf16x8*>(kt + k_off[c]);
    f32x16 s[NR][P];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr)
#pragma unroll
      for (int p = 0; p < P; ++p) {
#pragma unroll
        for (int e = 0; e < 16; ++e) s[nr][p][e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) s[nr][p] = mfma32(kf[KS * p + ks], q[nr][ks], s[nr][p]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (every read of this K buffer has returned)
    if (left > 2) copy_k(it + 2);

    const int k0 = first_key(it);
    const int own = (t0 + w + 4 * it) * KEYS - k0;   // (keys before it belong to the tile before)
    if (own > 0) {
#pragma unroll
      for (int nr = 0; nr < NR; ++nr)
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            s[nr][p][e] = P * (8 * (e >> 2) + (e & 3)) + p >= own - 4 * P * hh ? s[nr][p][e] : kNegInf;
    }
    bf16x8 pr[NR][P][2];
#pragma unroll
    for (int nr = 0; nr < NR; ++nr) {
      float mt = kNegInf;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 16; ++e) mt = fmaxf(mt, s[nr][p][e]);
      mt = half_max(mt);
      const float m_new = fmaxf(m_run[nr], mt);
      const float m_safe = (m_new == kNegInf) ? 0.f : m_new;
      if (__builtin_amdgcn_ballot_w64(m_new != m_run[nr]) != 0) {
        const float alpha = fast_exp2((m_run[nr] - m_safe) * c2);
        l_run[nr] *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[nr][db][e] *= alpha;
        m_run[nr] = m_new;
      }
      const float neg_m = -m_safe * c2;
      float lt = 0.f;
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
          const float p0 = fast_exp2(__builtin_fmaf(s[nr][p][e], c2, neg_m));
          const float p1 = fast_exp2(__builtin_fmaf(s[nr][p][e + 1], c2, neg_m));
          const bf16x2 pk = pack_bf16(p0, p1);
          lt += p0 + p1;
          pr[nr][p][e >> 3][e & 7] = pk[0];
          pr[nr][p][e >> 3][(e & 7) + 1] = pk[1];
        }
      l_run[nr] += lt;
    }
    // copies behind this V tile: the next tile's K and V and the K after it
    if (left > 2) wait_vmem<24>(); else if (left > 1) wait_vmem<16>(); else wait_vmem<0>();
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int db = 0; db < 4; ++db) {   // column blocks of the LDS row: head dim 64: dims 32 (db & 1) of key half db / 2
        const bf16x8 vf = join_tr(lds_read_tr16(reinterpret_cast<const bf16_t*>(vt + v_off[db][0] + tt * 16 * 256)),
                                  lds_read_tr16(reinterpret_cast<const bf16_t*>(vt + v_off[db][1] + tt * 16 * 256)));
#pragma unroll
        for (int nr = 0; nr < NR; ++nr) acc[nr][db % DB] = mfma32(vf, pr[nr][db / DB][tt], acc[nr][db % DB]);
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (left > 2) copy_v(it + 2);
  }

  // ---- merge the four waves, one block of 32 rows at a time ----
  float* sM = reinterpret_cast<float*>(smem + 4 * WAVE_BYTES);   // [wave][row]
  float* sL = sM + 4 * 64;
#pragma unroll
  for (int nr = 0; nr < NR; ++nr) {
    const float lt = half_sum(l_run[nr]);
    if (hh == 0) {
      sM[w * 64 + 32 * nr + l32] = m_run[nr];
      sL[w * 64 + 32 * nr + l32] = lt;
    }
  }
  constexpr int LD = D + 4;   // floats per staged row
  static_assert(4 * 32 * LD * 4 <= 4 * WAVE_BYTES, "the staged blocks fit the rings");
  float* sO = reinterpret_cast<float*>(smem);   // [wave][32 rows][LD]
  __syncthreads();   // (also: every wave is done with its ring)
  const size_t all_rows = (size_t)a.heads * a.rows;
#pragma unroll
  for (int nr = 0; nr < NR; ++nr) {
    float M = kNegInf;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) M = fmaxf(M, sM[ww * 64 + 32 * nr + l32]);
    const float m_safe = (M == kNegInf) ? 0.f : M;
    const float f = fast_exp2((m_run[nr] - m_safe) * c2);   // (a wave without keys: 0)
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        f32x4 x;
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = acc[nr][db][4 * g + u] * f;
        *reinterpret_cast<f32x4*>(sO + (w * 32 + l32) * LD + 32 * db + 8 * g + 4 * hh) = x;
      }
    __syncthreads();
    // thread -> (row, four columns); the waves' sums in a fixed order
    for (int at = (int)threadIdx.x; at < 32 * (D / 4); at += 256) {
      const int r = at / (D / 4), c = (at % (D / 4)) * 4;
      const int row = 32 * nr + r;
      if (row >= rows) break;   // (rows grow with `at`)
      float Mr = kNegInf, Lr = 0.f;
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) Mr = fmaxf(Mr, sM[ww * 64 + row]);
      const float Ms = (Mr == kNegInf) ? 0.f : Mr;
      f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ww = 0; ww < 4; ++ww) {
        Lr += sL[ww * 64 + row] * fast_exp2((sM[ww * 64 + row] - Ms) * c2);
        sum += *reinterpret_cast<const f32x4*>(sO + (ww * 32 + r) * LD + c);
      }
      const size_t gr = row0 + row;
      if (a.splits == 1) {
        const float inv = Lr > 0.f ? 1.0f / Lr : 0.f;
        const bf16x2 lo = pack_bf16(sum[0] * inv, sum[1] * inv), hi = pack_bf16(sum[2] * inv, sum[3] * inv);
        const bf16x4 out = {lo[0], lo[1], hi[0], hi[1]};
        *reinterpret_cast<bf16x4*>(a.o + gr * D + c) = out;
        if (c == 0 && a.l != nullptr) {
          a.l[gr] = Lr;
          a.m[gr] = Mr * a.sm_scale;
        }
      } else {
        *reinterpret_cast<f32x4*>(a.work + ((size_t)split * all_rows + gr) * D + c) = sum;
        if (c == 0) {
          float* ml = a.work + (size_t)a.splits * all_rows * D + ((size_t)split * all_rows + gr) * 2;
          ml[0] = Mr;
          ml[1] = Lr;
        }
      }
    }
    if (nr + 1 < NR) __syncthreads();
  }
}

// Merges the splits' sums: a work-group takes one row, its threads four columns of every (1024 / D)th split.  (A thread
// that walked all splits of its columns waited for one load after the other: 32 splits of 8 kv heads cost 20 us.)
template <int D>
__global__ __launch_bounds__(256) void decode_merge_kernel(DecodeArgs a) {
  constexpr int COLS = D / 4, GROUPS = 256 / COLS;
  static_assert(dec_cfg::MAX_SPLITS <= 64, "one lane per split");
  __shared__ f32x4 part[256];
  const size_t all_rows = (size_t)a.heads * a.rows;
  const size_t row = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int c = tid % COLS, g = tid / COLS;
  const float c2 = a.sm_scale * kLog2e;
  float mine = kNegInf, l = 0.f;   // lane s: maximum and sum of split s
  if (lane < a.splits) {
    const float* ml = a.work + (size_t)a.splits * all_rows * D + ((size_t)lane * all_rows + row) * 2;
    mine = ml[0];
    l = ml[1];
  }
  float M = mine;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) M = fmaxf(M, __shfl_xor(M, off));
  const float f = fast_exp2((mine - (M == kNegInf ? 0.f : M)) * c2);
  float L = l * f;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) L += __shfl_xor(L, off);
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < a.splits; s0 += GROUPS) {   // (the same trips for every lane of a wave: __shfl reads lane s)
    const int s = s0 + g;
    const float fs = __shfl(f, s & 63);
    if (s < a.splits) sum += *reinterpret_cast<const f32x4*>(a.work + ((size_t)s * all_rows + row) * D + 4 * c) * fs;
  }
  part[tid] = sum;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int o = 1; o < GROUPS; ++o) sum += part[o * COLS + c];
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  const bf16x2 lo = pack_bf16(sum[0] * inv, sum[1] * inv), hi = pack_bf16(sum[2] * inv, sum[3] * inv);
  const bf16x4 out = {lo[0], lo[1], hi[0], hi[1]};
  *reinterpret_cast<bf16x4*>(a.o + row * D + 4 * c) = out;
  if (c == 0 && a.l != nullptr) {
    a.l[row] = L;
    a.m[row] = M * a.sm_scale;
  }
}

// Key splits per kv head: the number of rounds of 256 work-groups (one per CU: the rings take 128 KB of LDS) times the
// tiles that a wave walks in one, plus what a work-group costs besides (start, first copies, merge: about as long as
// kOverhead tiles), made smallest; the fewest splits among equals.
static int chunks_of(int rows) { return rows > 64 ? 2 : 1; }
static int decode_splits(int heads, int tiles) {   // heads: times chunks_of(rows)
  constexpr int kOverhead = 4;
  long long best = -1;
  int splits = 1;
  for (int s = 1; s <= dec_cfg::MAX_SPLITS && (s == 1 || 4 * s <= tiles); ++s) {
    const long long rounds = ((long long)heads * s + 255) / 256;
    const long long cost = rounds * ((tiles + 4 * s - 1) / (4 * s) + kOverhead) + (s > 1 ? 2 : 0);
    if (best < 0 || cost < best) {
      best = cost;
      splits = s;
    }
  }
  return splits;
}

static int keys_per_tile(int D) { return dec_cfg::ROWS * (128 / D); }

bool fwd_decode_ok(int dtype, int B, int Hq, int Hkv, int Sq, int Sk, int D) {
  if (dtype != FLEXATTN_BF16 || (D != 64 && D != 128) || B <= 0 || Hq <= 0 || Hkv <= 0 || Sq <= 0 || Hq % Hkv != 0) return false;
  const long long rows = (long long)(Hq / Hkv) * Sq, heads = (long long)B * Hkv;
  return rows <= dec_cfg::MAX_ROWS && Sk >= keys_per_tile(D) && heads * 2 * dec_cfg::MAX_SPLITS < (1ll << 31);
}

int64_t fwd_decode_bytes(int B, int Hq, int Hkv, int Sq, int Sk, int D) {
  const int key_tiles = tiles_of(Sk, keys_per_tile(D));
  const int splits = decode_splits(B * Hkv * chunks_of(Hq / Hkv * Sq), key_tiles);
  return splits == 1 ? 0 : (int64_t)splits * B * Hq * Sq * (D + 2) * 4;
}

template <int D, int NR>
static int launch_decode(const DecodeArgs& d, hipStream_t stream) {
  auto kern = decode_kernel<D, NR>;
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                               dec_cfg::LDS_BYTES);
  if (attr != hipSuccess) return set_error(FLEXATTN_ELAUNCH, "hipFuncSetAttribute(decode): %s", hipGetErrorString(attr));
  hipLaunchKernelGGL(kern, dim3(d.heads * d.splits * chunks_of(d.rows)), dim3(256), dec_cfg::LDS_BYTES, stream, d);
  const int rc = check_launch("flexattn_fwd_decode");
  if (rc != FLEXATTN_OK || d.splits == 1) return rc;
  hipLaunchKernelGGL(decode_merge_kernel<D>, dim3(d.heads * d.rows), dim3(256), 0, stream, d);
  return check_launch("flexattn_fwd_decode (merge)");
}

template <int D>
static int launch_decode_rows(const DecodeArgs& d, hipStream_t stream) {
  if (d.rows <= 32) return launch_decode<D, 1>(d, stream);
  return launch_decode<D, 2>(d, stream);   // (more than 64 rows: two work-groups per split, see decode_kernel)
}

int fwd_decode(const FwdArgs& a, int D, void* work, hipStream_t stream) {
  DecodeArgs d;
  d.q = static_cast<const bf16_t*>(a.q); d.k = static_cast<const bf16_t*>(a.k); d.v = static_cast<const bf16_t*>(a.v);
  d.o = static_cast<bf16_t*>(a.o); d.l = a.l; d.m = a.m;
  d.work = static_cast<float*>(work);
  d.heads = a.B * a.Hkv;
  d.rows = a.Hq / a.Hkv * a.Sq;
  d.Sk = a.Sk;
  d.sm_scale = a.sm_scale;
  d.splits = decode_splits(d.heads * chunks_of(d.rows), tiles_of(a.Sk, keys_per_tile(D)));
  return D == 64 ? launch_decode_rows<64>(d, stream) : launch_decode_rows<128>(d, stream);
}

#else

bool fwd_decode_ok(int, int, int, int, int, int, int) { return false; }
int64_t fwd_decode_bytes(int, int, int, int, int, int) { return 0; }
int fwd_decode(const FwdArgs&, int, void*, hipStream_t) { return set_error(FLEXATTN_ENOTSUP, "not in this library"); }

#endif

}  // namespace fa
