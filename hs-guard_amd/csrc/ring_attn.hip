// Window-W GQA attention over a slot's ring and a row's own new keys (short ticks, 64-token window fills), or over
// the row's own keys alone (whole sequences), for gfx950 on MFMA.
//
// Contract: src/hs_guard/engine/ring_attention_kernel.py:7-26 (torch reference) with the v8 kernel's
// numerics and epilogue (src/hs_guard/engine/fused_kernels.py:288-356): keys in blocks of 32 (the W ring
// columns in order, then the tick's new keys), a running max per query row, probabilities rounded to bf16
// in the P.V product and summed in fp32, output / sum rounded to bf16, times bf16(sigmoid(gate)); the
// tick's keys/values are written into the ring in place after every read.
//
// Query rows r = l*G + g (token l, q group g) of one (row, kv head) form 16-row tiles, and a workgroup of 4 waves takes
// a group of 4 tiles. Both paths below run, per 32 keys, on v_mfma_f32_16x16x32_bf16,
//   S^T[key, m] = K . Q^T
//   O^T[d, m] += V^T . P^T   (A = V^T by LDS transpose reads of row-major V, B = P straight from the S^T accumulators:
//                             the k order of the product is the lane's own key order, so P never leaves registers)
// The S^T accumulator layout puts one query row per lane column, so maxima, sums and the O^T rescale are per-lane
// scalars. The in-place ring write is a second launch (ring_write_kernel) after all reads.
//
// attend_group (2 to 4 tiles): wave w takes tile w, and the keys pass through LDS 64 at a time for all waves, loaded
// into registers a fill ahead. The LDS reads of every wave's whole fill (256 KB per fill of a full group) bound it.
// attend_tile (one tile: a row of up to 16 / G tokens, or a longer row's last tile): one wave would do all the work, so
// the waves split the KEYS instead: of the tile's key blocks (the ring's in column order, then the new keys' from the
// first one it sees), wave w takes blocks w, w + 4, ..., at most SLOTS of them, its keys going straight from global
// memory into operand registers. Two phases, as in the decode kernel: every score and block maximum first; then, the
// reference's running max after block b being the prefix maximum m_b of the block maxima, each block's probabilities
// exp(s - m_b) in bf16 times its values, a wave chaining its blocks by exp(m_prev - m_b) and the waves' partial sums
// meeting in LDS with weights exp(m_last - m_final). No workgroup barrier inside the phases, and unconditional loads (a
// block the tile does not see reads the row's own first new keys): under branches they were waited for at once.
// Measured (W = 512, 16 q / 4 kv heads), with every tile on attend_group before and now:
// 72 padded rows of 2 to 64 steps 147 -> 92 us (49 us of it whole groups past their rows' lengths, which ran their
// keys), 64 rows of 4 steps 41.6 -> 28.0 us, one such row 34.9 -> 21.6 us. Splitting the keys of longer rows' tiles too
// reads K and V once per tile instead of once per group: 72 rows of 64 steps 264 us against 165. A sequence of 8,000
// tokens (no ring): 203 us, against 270 us over rings gathered from it (and 0.2 ms of gathers). Three rows of 900 tokens
// over rings (hsg_ring_prefill): 88 us, against 15 ticks of 25 us.
#include <math.h>

#include <type_traits>

#include "hsg_common.h"

namespace hsg {
namespace {

constexpr int D = 256;
constexpr int NW = 4;                  // waves per workgroup
constexpr int TQ = 16;                 // query rows of a tile
constexpr int KB = 32;                 // keys per softmax block (the reference's BN)
constexpr int W_MAX = 512;
constexpr int LB_MAX = 64;
constexpr int SLOTS = 5;               // attend_tile: key blocks of a wave: W / 32 ring blocks and 2 of new keys, or the 18 that the
                                       // window of a tile's up to 16 tokens can touch, over 4 waves
constexpr int KV_LOADS = 2 * D / KB;   // 16-byte K loads of a wave per block (and V loads)
constexpr int KF = 2 * KB;             // attend_group: keys per LDS fill

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) int i32x4;

struct RingParams {
  const uint16_t* q; int64_t q_sn, q_sl, q_sh, q_sg;
  uint16_t* ring_k; uint16_t* ring_v; int64_t ring_rows; int W;   // ring_k NULL: the row's own keys only
  const uint16_t* new_k; int64_t nk_sn, nk_sl, nk_sh;
  const uint16_t* new_v; int64_t nv_sn, nv_sl, nv_sh;
  const uint16_t* gate; int64_t g_sn, g_sl, g_sh, g_sg, g_off;
  const int64_t* ring_pos; const int64_t* slots; const int64_t* starts; const int64_t* lens;
  const int64_t* offsets;
  int lb, hkv, G;
  float scale;
  int write_ring;
  int min_len;
  int pairs;        // rows x kv heads
  int qgroups;      // workgroups (groups of NW tiles) per (row, kv head)
  int qg0;          // first group
  int sequences;    // rows of any length: each XCD takes a contiguous eighth of the workgroups
  uint16_t* out; int64_t o_sn, o_sl, o_sh, o_sg;
};

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 w) { return __builtin_bit_cast(bf16x8, w); }

constexpr int KP_NONE = -(1 << 30);    // an empty ring column
constexpr int KP_FAR = 1 << 29;        // clamp of a position relative to the row's start

// exp of the softmax argument on the hardware exp2 (v_exp_f32): exp(x) = 2^(x log2 e). The reference kernel
// takes tl.exp, Triton's fast exponential, here too (src/hs_guard/engine/fused_kernels.py:318-319,335-336).
__device__ __forceinline__ float exp_fast(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

// LDS transpose read (ds_read_b64_tr_b16): within each group of 16 lanes, lane 4q + e receives element e of
// the 4-element (8-byte) vectors addressed by lanes q, q + 4, q + 8, q + 12 of its group. With V row-major
// ([key][dim]), lane s of a group addressing key row r0 + (s >> 2), dims c0 + 4 (s & 3) .. +3 receives dim
// c0 + s of keys r0 .. r0 + 3: the A operand of O^T += V^T . P^T.
typedef __attribute__((ext_vector_type(4))) short s16x4_;
__device__ __forceinline__ u32x2 ld_tr4(const uint16_t* p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_*)(p)));
}

// Eight of them, of four dim tiles (LDS byte addresses a0 .. a3) and key rows 0 and 16, with one wait: the compiler
// issues its builtin one product ahead, an LDS round trip per product.
__device__ __forceinline__ void ld_tr_4x2(u32x2 (&v)[4][2], uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3) {
  static_assert(16 * D * 2 == 8192, "the offset below is 16 rows");
  asm volatile(
      "ds_read_b64_tr_b16 %0, %8\n\t"
      "ds_read_b64_tr_b16 %1, %8 offset:8192\n\t"
      "ds_read_b64_tr_b16 %2, %9\n\t"
      "ds_read_b64_tr_b16 %3, %9 offset:8192\n\t"
      "ds_read_b64_tr_b16 %4, %10\n\t"
      "ds_read_b64_tr_b16 %5, %10 offset:8192\n\t"
      "ds_read_b64_tr_b16 %6, %11\n\t"
      "ds_read_b64_tr_b16 %7, %11 offset:8192\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1]), "=&v"(v[2][0]), "=&v"(v[2][1]), "=&v"(v[3][0]),
        "=&v"(v[3][1])
      : "v"(a0), "v"(a1), "v"(a2), "v"(a3)
      : "memory");
}

// byte offset of an LDS pointer
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}

// Row pieces of 16 bytes in LDS: rows of 512 bytes whose 32-byte pairs of pieces are permuted, pair c of row r at
// c ^ (r & 15). A transpose read (16 rows x 32 bytes) and a row read of 16 rows (16 bytes at each of 4 offsets) then
// spread over all banks evenly. Element offset of piece `pc` of row r:
__device__ __forceinline__ int piece_at(int r, int pc) { return r * D + 8 * (2 * ((pc >> 1) ^ (r & 15)) + (pc & 1)); }

// The (row, kv head) of a workgroup: element pointers of its first token's query, new key, new value, gate and output
struct Row {
  const uint16_t* qrow;
  const uint16_t* krow;
  const uint16_t* vrow;
  const uint16_t* grow;   // NULL: no gate
  uint16_t* orow;
  const int64_t* ring_pos;
  int64_t slot, start, ring_base;
  int len, steps;         // valid tokens and output steps (padded rows: up to lb, the rest zeros)
  int RB;                 // ring blocks
};

struct SplitLds {
  uint16_t Vs[NW][KB * D];       // per wave: one block of V (piece_at), then the wave's O
  int kp_s[NW][W_MAX / NW];      // key position - start of the wave's ring columns; KP_NONE for an empty one
  float bm_s[TQ][NW * SLOTS];    // block maxima of each query row, -inf where nothing is seen
  float l_s[NW][TQ];             // per wave: weighted sum of each query row
};

struct GroupLds {
  uint16_t Ks[KF * D], Vs[KF * D];   // the fill's keys and values (piece_at)
  int kp[W_MAX];                     // key position - start of the ring columns; KP_NONE for an empty one
  uint32_t mask[NW];                 // per wave: bit f set if the ring's fill f has a key visible to the group
};

// ---------------------------------------------------------------------------------------------------------
// A group of up to NW tiles: wave w takes tile w, keys in fills of KF through LDS.
// ---------------------------------------------------------------------------------------------------------
__device__ __forceinline__ void attend_group(const RingParams& p, const Row& ro, int r_lo, GroupLds& lds, int lane, int wave) {
  const int tid = threadIdx.x;
  const int q4 = lane >> 4;                            // lane group: keys 4*q4 .., dims 8*q4 ..
  const int mcol = lane & 15;                          // the lane's query row within its tile
  const int W = p.W, G = p.G, RB = ro.RB, len = ro.len;
  const int M = G * ro.steps, Mv = G * len;
  const int r = r_lo + TQ * wave + mcol;
  const bool has_tile = r_lo + TQ * wave < Mv;
  const int rq = min(r, Mv - 1);                       // past the valid rows: the last one again, stored as zeros
  const int l_tok = rq / G;
  const int gq = rq - l_tok * G;
  bf16x8 qb[D / 32];
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks)
    qb[ks] = as_bf16x8(*reinterpret_cast<const u32x4*>(ro.qrow + l_tok * p.q_sl + gq * p.q_sg + 32 * ks + 8 * q4));
  // tokens of the group (all waves)
  const int l_lo = r_lo / G;
  const int l_hi = (min(r_lo + NW * TQ, Mv) - 1) / G;
  // Fills: the ring's, then those of the new keys the group sees (from new key j_lo). Every ring position goes to
  // LDS in one round trip, and the ring's fills that no query of the group sees are skipped.
  const int n_ring = (RB + 1) / 2;
  const int j_lo = max(0, l_lo - W + 1) / KF * KF;
  const int n_fills = n_ring + (l_hi - j_lo) / KF + 1;
  uint32_t my_mask = 0u;
  for (int c = tid; c < RB * KB; c += NW * 64) {
    const int64_t kpos = ro.ring_pos[c];
    const int64_t d = kpos - ro.start;
    int rel = (int)(d < -KP_FAR ? -KP_FAR : d > KP_FAR ? KP_FAR : d);
    if (kpos < 0) rel = KP_NONE;
    lds.kp[c] = rel;
    if (rel <= l_hi && rel > l_lo - W) my_mask |= 1u << (c / KF);
  }
  for (int o = 1; o < 64; o <<= 1) my_mask |= (uint32_t)__shfl_xor((int)my_mask, o, 64);
  if (lane == 0) lds.mask[wave] = my_mask;
  __syncthreads();
  const uint32_t ring_mask =
      __builtin_amdgcn_readfirstlane(lds.mask[0] | lds.mask[1] | lds.mask[2] | lds.mask[3]);
  auto next_fill = [&](int f) {   // first fill after f with a visible key (n_fills if none)
    ++f;
    if (f < n_ring) {
      const uint32_t rest = ring_mask >> f;
      f = rest ? f + __builtin_ctz(rest) : n_ring;
    }
    return f;
  };
  // Thread t holds piece t % 32 of keys t / 32 + 8 i (i < 8) of K and of V: every load instruction of a wave reads
  // two whole 512-byte key rows. Keys past the fill's valid ones repeat the last one and are zeroed when staged.
  u32x4 kr[8], vr[8];
  auto prefetch = [&](int f) __attribute__((always_inline)) {
    const bool ring = f < n_ring;
    const int c0 = ring ? f * KF : j_lo + (f - n_ring) * KF;
    const int last = ring ? min(KF, RB * KB - c0) - 1 : min(KF, len - c0) - 1;
    const uint16_t* kb = (ring ? p.ring_k + ro.ring_base + c0 * D : ro.krow + c0 * p.nk_sl);
    const uint16_t* vb = (ring ? p.ring_v + ro.ring_base + c0 * D : ro.vrow + c0 * p.nv_sl);
    const int64_t kst = ring ? D : p.nk_sl, vst = ring ? D : p.nv_sl;
    const int tl = lane_per_site(tid);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = min((tl >> 5) + 8 * i, last);
      // nontemporal, as the decode kernel's ring reads: a step's mixed tick ran 0.35 % faster (two A/B pairs
      // on MI355X), the rings no longer displacing what the neighbouring kernels reuse
      kr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(kb + key * kst + 8 * (tl & 31)));
      vr[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vb + key * vst + 8 * (tl & 31)));
    }
  };
  float m_run = -INFINITY, l_run = 0.f;   // l_run: this lane's keys only
  f32x4 O[D / 16];
#pragma unroll
  for (int t = 0; t < D / 16; ++t) O[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int rx = 4 * q4 + (mcol >> 2);    // the lane's key row of a transpose read (and + 16)
  int fcur = next_fill(-1);
  prefetch(fcur);
  for (; fcur < n_fills; fcur = next_fill(fcur)) {
    const bool ring = fcur < n_ring;
    const int c0 = ring ? fcur * KF : j_lo + (fcur - n_ring) * KF;
    const int nkeys = ring ? min(KF, RB * KB - c0) : min(KF, len - c0);
    __syncthreads();  // the previous fill's LDS reads are done
    {
      const int tl = lane_per_site(tid);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = (tl >> 5) + 8 * i;
        const bool live = key < nkeys;
        const int o = piece_at(key, tl & 31);
        *reinterpret_cast<u32x4*>(&lds.Ks[o]) = live ? kr[i] : (u32x4){0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(&lds.Vs[o]) = live ? vr[i] : (u32x4){0u, 0u, 0u, 0u};
      }
    }
    const int fnext = next_fill(fcur);
    if (fnext < n_fills) prefetch(fnext);
    __syncthreads();
    if (!has_tile) continue;
    // ---- S^T = K . Q^T for both softmax blocks of the fill first ----
    f32x4 S[2][2];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      S[sb][0] = S[sb][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
          S[sb][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              as_bf16x8(*reinterpret_cast<const u32x4*>(&lds.Ks[piece_at(sb * KB + 16 * kt + mcol, 4 * ks + q4)])), qb[ks],
              S[sb][kt], 0, 0, 0);
    }
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      if (sb * KB >= nkeys) break;
      // ---- mask, online softmax over the block (the lane's 8 keys: 4 q4 + i and 16 + 4 q4 + i) ----
      float s[8];
      float bmax = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        i32x4 rel;
        const int at = c0 + sb * KB + 16 * kt + 4 * q4;
        if (ring) {
          rel = *reinterpret_cast<const i32x4*>(&lds.kp[at]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) rel[i] = at + i;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {   // KP_NONE fails the second test, a new key past the row's end the first
          const bool ok = (rel[i] <= l_tok) & (rel[i] > l_tok - W);
          const float v = ok ? S[sb][kt][i] * p.scale : -INFINITY;
          s[4 * kt + i] = v;
          bmax = fmaxf(bmax, v);
        }
      }
      bmax = max_pair32(max_pair16(bmax));   // over q4 (lane xor 16, 32)
      const float m_new = fmaxf(m_run, bmax);
      const float m_safe = m_new == -INFINITY ? 0.f : m_new;
      const float alpha = exp_fast(m_run - m_safe);   // exp(-inf) = 0 before the first visible key
      l_run *= alpha;
      m_run = m_new;
      u32x4 pk;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p0 = exp_fast(s[2 * i] - m_safe);
        const float p1 = exp_fast(s[2 * i + 1] - m_safe);
        l_run += p0 + p1;
        pk[i] = pack_bf16x2(p0, p1);
      }
      const bf16x8 pb = as_bf16x8(pk);
      // ---- O^T += V^T . P^T over the block's 32 keys, in the lane's key order ----
#pragma unroll
      for (int t = 0; t < D / 16; ++t) {
        const uint16_t* vsrc = &lds.Vs[(sb * KB + rx) * D + 4 * (mcol & 3) + 16 * (t ^ rx)];
        const u32x2 lo = ld_tr4(vsrc);
        const u32x2 hi = ld_tr4(vsrc + 16 * D);
        O[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8((u32x4){lo[0], lo[1], hi[0], hi[1]}), pb, O[t] * alpha, 0,
                                                       0, 0);
      }
    }
  }
  // ---- normalise, gate, store this lane's row: dims 16 t + 4 q4 + i ----
  if (r < M) {
    l_run = add_xor32(add_xor16(l_run));
    const bool valid = r < Mv && l_run > 0.f;
    const int l_out = r / G;
    const int g_out = r - l_out * G;
    uint16_t* dst = ro.orow + l_out * p.o_sl + g_out * p.o_sg + 4 * q4;
    const uint16_t* gsrc = ro.grow ? ro.grow + l_out * p.g_sl + g_out * p.g_sg + 4 * q4 : nullptr;
    // every gate piece is loaded before the first store: out may alias gate as far as the compiler knows, so a
    // load after a store waits for it, and the 16 pieces were 16 serial memory round trips at the end of each
    // workgroup
    u32x2 gw[D / 16];
    if (gsrc) {
#pragma unroll
      for (int t = 0; t < D / 16; ++t) gw[t] = *reinterpret_cast<const u32x2*>(gsrc + 16 * t);
    }
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = valid ? rbf(quotient(O[t][i], l_run)) : 0.f;
      if (gsrc) {
        float gt[4];
        unpack2(gw[t][0], gt[0], gt[1]);
        unpack2(gw[t][1], gt[2], gt[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = y[i] * rbf(sigmoidf_(gt[i]));
      }
      store4_bf16(dst + 16 * t, y);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------
// One tile (16 query rows): the four waves split its keys.
// ---------------------------------------------------------------------------------------------------------
__device__ __forceinline__ void attend_tile(const RingParams& p, const Row& ro, int r_lo, SplitLds& lds, int lane, int wave) {
  auto& Vs = lds.Vs;
  auto& kp_s = lds.kp_s;
  auto& bm_s = lds.bm_s;
  auto& l_s = lds.l_s;
  const int tid = threadIdx.x;
  const int q4 = lane >> 4;                            // lane group: keys 4*q4 .., dims 8*q4 ..
  const int mcol = lane & 15;                          // the lane's query row within its tile
  const int W = p.W, G = p.G, RB = ro.RB, len = ro.len;
  const int M = G * ro.steps, Mv = G * len;
  uint16_t* const vlds = Vs[wave];
  // ---- this lane's query row and the tile's token range ----
  const int rq = min(r_lo + mcol, Mv - 1);   // past the valid rows: the last one again, never stored
  const int l_tok = rq / G;
  const int gq = rq - l_tok * G;
  const int l_lo = r_lo / G;
  const int l_hi = (min(r_lo + TQ, Mv) - 1) / G;
  bf16x8 qb[D / 32];
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks)
    qb[ks] = as_bf16x8(*reinterpret_cast<const u32x4*>(ro.qrow + l_tok * p.q_sl + gq * p.q_sg + 32 * ks + 8 * q4));

  // ---- positions of the wave's ring blocks w + 4 i; bit i: a key of block i is visible / all are to all ----
  uint32_t any = 0u, full = 0u;
  if (RB) {
    int64_t kpos[2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
      kpos[u] = ro.ring_pos[min(wave + NW * (2 * u + (lane >> 5)), RB - 1) * KB + (lane & 31)];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t d = kpos[u] - ro.start;
      int rel = (int)(d < -KP_FAR ? -KP_FAR : d > KP_FAR ? KP_FAR : d);
      if (kpos[u] < 0 || wave + NW * (2 * u + (lane >> 5)) >= RB) rel = KP_NONE;
      kp_s[wave][64 * u + lane] = rel;
      const uint64_t va = __ballot(rel <= l_hi && rel > l_lo - W);
      const uint64_t vf = __ballot(rel <= l_lo && rel > l_hi - W);
      any |= ((uint32_t)va ? 1u : 0u) << (2 * u) | ((uint32_t)(va >> 32) ? 1u : 0u) << (2 * u + 1);
      full |= ((uint32_t)vf == ~0u ? 1u : 0u) << (2 * u) | ((uint32_t)(vf >> 32) == ~0u ? 1u : 0u) << (2 * u + 1);
    }
    any = __builtin_amdgcn_readfirstlane(any);
    full = __builtin_amdgcn_readfirstlane(full);
  }
  // the new-key blocks the tile sees: cb0 .. cb1
  const int cb0 = max(0, l_lo - W + 1) / KB;
  const int cb1 = l_hi / KB;
  // the wave's blocks (ordinals wave + 4 i): bit i of seen / full as of any / full, over ring and new blocks
  uint32_t seen = any;
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
    const int c = cb0 + wave + NW * i - RB;
    if (wave + NW * i >= RB) {
      seen |= (c <= cb1 ? 1u : 0u) << i;
      full |= (c * KB + KB - 1 <= l_lo && c * KB > l_hi - W ? 1u : 0u) << i;
    }
  }
  // first row, row stride and last valid row of block i's keys or values; a block nobody sees reads the row's
  // first new keys
  auto rows_of = [&](int i, const uint16_t* ring, const uint16_t* fresh, int64_t stride, int64_t& st, int& last) {
    const int o = wave + NW * i;
    const bool live = (seen >> i & 1u) != 0;
    const bool from_ring = live && o < RB;
    const int j0 = live && !from_ring ? (cb0 + o - RB) * KB : 0;
    st = from_ring ? D : stride;
    last = from_ring ? KB - 1 : min(KB - 1, len - 1 - j0);
    return from_ring ? ring + ro.ring_base + o * (KB * D) : fresh + j0 * stride;
  };
  auto load_keys = [&](int i, u32x4 (&ka)[2][D / 32]) __attribute__((always_inline)) {
    int64_t st;
    int last;
    const uint16_t* base = rows_of(i, p.ring_k, ro.krow, p.nk_sl, st, last);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const uint16_t* src = base + min(16 * kt + mcol, last) * st + 8 * q4;
#pragma unroll
      for (int ks = 0; ks < D / 32; ++ks) ka[kt][ks] = *reinterpret_cast<const u32x4*>(src + 32 * ks);
    }
  };
  // V: load u covers rows 2 u, 2 u + 1 whole (a key past the last valid one repeats it; it is zeroed when staged)
  auto load_values = [&](int i, u32x4 (&va)[KV_LOADS]) __attribute__((always_inline)) {
    int64_t st;
    int last;
    const uint16_t* base = rows_of(i, p.ring_v, ro.vrow, p.nv_sl, st, last);
    const int lv = lane_per_site(lane);
#pragma unroll
    for (int u = 0; u < KV_LOADS; ++u)
      va[u] = *reinterpret_cast<const u32x4*>(base + min(2 * u + (lv >> 5), last) * st + 8 * (lv & 31));
  };
  for (int e = tid; e < TQ * NW * SLOTS; e += NW * 64) (&bm_s[0][0])[e] = -INFINITY;
  lds_barrier();   // kp_s and the empty block maxima are in LDS

  // ---- phase 1: scores of the blocks and their maxima; phase 2: probabilities and P.V ----
  float m_last = -INFINITY, m_fin = -INFINITY, l_run = 0.f;   // l_run: this lane's keys only
  f32x4 O[D / 16];
  auto attend = [&](auto first, auto step) __attribute__((always_inline)) {   // blocks FIRST, FIRST + STEP, ...
    constexpr int FIRST = decltype(first)::value, STEP = decltype(step)::value;
    float s[SLOTS][8];
    u32x4 va[KV_LOADS];
    {
      u32x4 ka[2][2][D / 32];
      load_keys(FIRST, ka[0]);
#pragma unroll
      for (int i = FIRST; i < SLOTS; i += STEP) {
        const int buf = (i - FIRST) / STEP & 1;
        if (i + STEP < SLOTS) load_keys(i + STEP, ka[buf ^ 1]);
        else load_values(FIRST, va);
        if (seen >> i & 1u) {
          f32x4 S[2];
#pragma unroll
          for (int kt = 0; kt < 2; ++kt) {
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < D / 32; ++ks)
              acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(ka[buf][kt][ks]), qb[ks], acc, 0, 0, 0);
            S[kt] = acc;
          }
          // scale and mask the lane's 8 keys 4 q4 + e and 16 + 4 q4 + e
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) s[i][4 * kt + e] = S[kt][e] * p.scale;
          if (!(full >> i & 1u)) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
              i32x4 rel;
              if (wave + NW * i < RB) {
                rel = *reinterpret_cast<const i32x4*>(&kp_s[wave][KB * min(i, W_MAX / NW / KB - 1) + 16 * kt + 4 * q4]);
              } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) rel[e] = (cb0 + wave + NW * i - RB) * KB + 16 * kt + 4 * q4 + e;
              }
#pragma unroll
              for (int e = 0; e < 4; ++e)   // KP_NONE fails the second
                s[i][4 * kt + e] = ((rel[e] <= l_tok) & (rel[e] > l_tok - W)) ? s[i][4 * kt + e] : -INFINITY;
            }
          }
          float bmax = -INFINITY;
#pragma unroll
          for (int e = 0; e < 8; ++e) bmax = fmaxf(bmax, s[i][e]);
          bmax = max_pair32(max_pair16(bmax));   // over q4 (lane xor 16, 32)
          if (q4 == 0) bm_s[mcol][wave + NW * i] = bmax;
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) s[i][e] = -INFINITY;
        }
      }
    }
    lds_barrier();   // every block maximum is in LDS
    // running max through each of the wave's blocks and over all of them
    float mb[SLOTS];
#pragma unroll
    for (int i = 0; i < SLOTS; ++i) {
      const f32x4 g = *reinterpret_cast<const f32x4*>(&bm_s[mcol][NW * i]);
      float own = m_fin;
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        own = fmaxf(own, w <= wave ? g[w] : -INFINITY);
        m_fin = fmaxf(m_fin, g[w]);
      }
      mb[i] = own;
    }
#pragma unroll
    for (int t = 0; t < D / 16; ++t) O[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = FIRST; i < SLOTS; i += STEP) {
      // V of block i from registers into LDS, the next block's loads behind it. Rows past the row's last key are zeros
      // there: their probability is zero, but 0 x an infinite value of that key would be NaN
      const int lv = lane_per_site(lane);
      const int last = wave + NW * i < RB ? KB - 1 : len - 1 - (cb0 + wave + NW * i - RB) * KB;
      if ((seen >> i & 1u) && last < KB - 1) {
#pragma unroll
        for (int u = 0; u < KV_LOADS; ++u)
          if (2 * u + (lv >> 5) > last) va[u] = (u32x4){0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int u = 0; u < KV_LOADS; ++u)
        *reinterpret_cast<u32x4*>(vlds + piece_at(2 * u + (lv >> 5), lv & 31)) = va[u];
      if (i + STEP < SLOTS) load_values(i + STEP, va);
      if (!(seen >> i & 1u)) continue;
      const float m = mb[i] == -INFINITY ? 0.f : mb[i];
      const float alpha = m_last == mb[i] ? 1.f : exp_fast(m_last - m);   // exp(-inf) = 0: nothing added so far
      m_last = mb[i];
      if (__ballot(alpha != 1.f)) {
        l_run *= alpha;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) O[t] *= alpha;
      }
      u32x4 pk;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = exp_fast(s[i][2 * e] - m);
        const float p1 = exp_fast(s[i][2 * e + 1] - m);
        l_run += p0 + p1;
        pk[e] = pack_bf16x2(p0, p1);
      }
      const bf16x8 pb = as_bf16x8(pk);
      // O^T += V^T . P^T over the block's 32 keys, in the lane's key order
      const int lt = lane_per_site(lane);
      const int rx = 4 * (lt >> 4) + ((lt & 15) >> 2);   // the lane's key row of a transpose read (and + 16)
      const uint32_t vbase = lds_offset(vlds) + 2 * (rx * D + 4 * (lt & 3));
#pragma unroll
      for (int t = 0; t < D / 16; t += 4) {
        u32x2 v[4][2];
        ld_tr_4x2(v, vbase + 32 * (t ^ rx), vbase + 32 * ((t + 1) ^ rx), vbase + 32 * ((t + 2) ^ rx),
                  vbase + 32 * ((t + 3) ^ rx));
#pragma unroll
        for (int u = 0; u < 4; ++u)
          O[t + u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              as_bf16x8((u32x4){v[u][0][0], v[u][0][1], v[u][1][0], v[u][1][1]}), pb, O[t + u], 0, 0, 0);
      }
    }
  };
  // A wave that sees none of its first SLOTS - 1 blocks (a row without history), or only its first and last (a history of up
  // to NW blocks), skips the others' loads: 72 rows of 4 steps over 100 keys 26.0 -> 19.1 us. The barrier
  // count is the same.
  using Slot = std::integral_constant<int, 1>;
  using Ends = std::integral_constant<int, SLOTS - 1>;
  if (seen & ((1u << (SLOTS - 1)) - 2)) attend(std::integral_constant<int, 0>{}, Slot{});
  else if (seen & 1u) attend(std::integral_constant<int, 0>{}, Ends{});
  else attend(Ends{}, Slot{});

  // ---- combine the waves: each leaves its weighted O (lane-linear 16-byte pieces) in its own Vs and takes dims
  // 64 w + 16 t + 4 q4 + i (t < 4) of every row ----
  const float wgt = m_last == -INFINITY ? 0.f : exp_fast(m_last - m_fin);
  const int lw = lane_per_site(lane);
  l_run = add_xor32(add_xor16(l_run)) * wgt;
  if (lw < TQ) l_s[wave][lw] = l_run;
  f32x4* const os = reinterpret_cast<f32x4*>(vlds) + lw;
#pragma unroll
  for (int t = 0; t < D / 16; ++t) os[t * 64] = O[t] * wgt;
  u32x2 gw[4];
  const int r = r_lo + (lw & 15);
  const int d0 = 64 * wave + 4 * (lw >> 4);
  const int l_out = min(r, M - 1) / G;
  const int g_out = min(r, M - 1) - l_out * G;
  if (ro.grow) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      gw[t] = *reinterpret_cast<const u32x2*>(ro.grow + l_out * p.g_sl + g_out * p.g_sg + d0 + 16 * t);
  }
  lds_barrier();
  float l_tot = 0.f;
  f32x4 o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    l_tot += l_s[w][lw & 15];
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] += reinterpret_cast<const f32x4*>(Vs[w])[(4 * wave + t) * 64 + lw];
  }
  if (r < M) {
    uint16_t* dst = ro.orow + l_out * p.o_sl + g_out * p.o_sg + d0;
    const bool valid = r < Mv && l_tot > 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = valid ? rbf(quotient(o[t][i], l_tot)) : 0.f;
      if (ro.grow) {
        float gt[4];
        unpack2(gw[t][0], gt[0], gt[1]);
        unpack2(gw[t][1], gt[2], gt[3]);
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = y[i] * rbf(sigmoidf_(gt[i]));
      }
      store4_bf16(dst + 16 * t, y);
    }
  }
}
__global__ __launch_bounds__(NW * 64, 2) void ring_attn_kernel(const RingParams p) {
  __shared__ union __align__(16) Lds {
    SplitLds split;
    GroupLds group;
    __device__ Lds() {}
  } lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Workgroups are dealt round-robin over the 8 XCDs. Ticks: query group slowest, so that consecutive workgroups take
  // consecutive (row, kv head) pairs (the live workgroups of a short-row tick spread over all XCDs, and a pair's
  // groups share one XCD's L2 when the pairs are a multiple of 8). Sequences: each XCD takes a
  // contiguous eighth of the groups, whose windows overlap.
  int pair, qg;
  if (!p.sequences) {
    qg = blockIdx.x / p.pairs;
    pair = blockIdx.x - qg * p.pairs;
  } else {
    const int i = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    pair = i / p.qgroups;
    qg = p.qg0 + i - pair * p.qgroups;
    if (pair >= p.pairs) return;
  }
  const int n = pair / p.hkv;
  const int h = pair - n * p.hkv;
  const bool padded = p.offsets == nullptr;
  Row ro;
  ro.slot = p.ring_k ? p.slots[n] : 0;
  ro.start = p.ring_k ? p.starts[n] : 0;
  int64_t len = p.lens[n];
  if (len < 0 || len > (padded ? LB_MAX : p.lb) || (p.ring_k && (ro.slot < 0 || ro.slot >= p.ring_rows))) len = 0;  // rejected
  if (padded && len > p.lb) len = p.lb;
  if (!padded && len < p.min_len) return;              // left to another kernel (single-step rows: decode)
  ro.len = (int)len;
  ro.steps = padded ? p.lb : ro.len;
  const int64_t base_tok = padded ? 0 : p.offsets[n];
  ro.qrow = p.q + (padded ? n * p.q_sn : base_tok * p.q_sl) + h * p.q_sh;
  ro.krow = p.new_k + (padded ? n * p.nk_sn : base_tok * p.nk_sl) + h * p.nk_sh;
  ro.vrow = p.new_v + (padded ? n * p.nv_sn : base_tok * p.nv_sl) + h * p.nv_sh;
  ro.grow = p.gate ? p.gate + (padded ? n * p.g_sn : base_tok * p.g_sl) + h * p.g_sh + p.g_off : nullptr;
  ro.orow = p.out + (padded ? n * p.o_sn : base_tok * p.o_sl) + h * p.o_sh;
  ro.RB = p.ring_k && len > 0 ? p.W / KB : 0;
  ro.ring_base = ((ro.slot * p.hkv + h) * (int64_t)(p.W + 1)) * D;
  ro.ring_pos = p.ring_pos + ro.slot * (int64_t)(p.W + 1);
  const int r_lo = qg * (NW * TQ);
  // a sequence's ring holds only positions before its start, which steps from W - 1 on do not see
  if (p.sequences && r_lo / p.G >= p.W - 1) ro.RB = 0;
  const int M = p.G * ro.steps, Mv = p.G * ro.len;      // query rows of this (row, kv head), and the valid ones
  // rows past the length of a padded row are zeros; attend_group and attend_tile store those of the tiles they take
  const int tiles = r_lo >= Mv ? 0 : min((Mv - r_lo + TQ - 1) / TQ, NW);
  const int z_lo = tiles > 1 ? M : r_lo + tiles * TQ;
  for (int e = threadIdx.x; e < (min(r_lo + NW * TQ, M) - z_lo) * (D / 4); e += NW * 64) {
    const int r = z_lo + e / (D / 4);
    const int l = r / p.G;
    *reinterpret_cast<u32x2*>(ro.orow + l * p.o_sl + (r - l * p.G) * p.o_sg + 4 * (e % (D / 4))) = (u32x2){0u, 0u};
  }
  // (a tile that may see ring blocks and many new-key blocks could need more than SLOTS of attend_tile's slots)
  if (tiles == 1 && (ro.RB == 0 || ro.len <= LB_MAX)) attend_tile(p, ro, r_lo, lds.split, lane, wave);
  else if (tiles > 0) attend_group(p, ro, r_lo, lds.group, lane, wave);
}

// In-place ring write of the tick's valid keys/values, launched after the attention kernel (whose query
// groups of one row run in different workgroups, so none of them may overwrite a column another still reads).
__global__ __launch_bounds__(256) void ring_write_kernel(const RingParams p) {
  const int n = blockIdx.x / p.hkv;
  const int h = blockIdx.x - n * p.hkv;
  // the row's reads are issued together (padded: lens stands in for the offset, unused) and checked without
  // short-circuit branches, each of which made the compiler wait for one read before issuing the next
  const bool padded = p.offsets == nullptr;
  const int64_t slot = p.slots[n];
  int64_t len = p.lens[n];
  const int64_t off = (padded ? p.lens : p.offsets)[n];
  const int64_t start = p.starts[n];
  const bool rejected = (slot < 0) | (slot >= p.ring_rows) | (len < 0) | (len > (padded ? LB_MAX : p.lb));
  if (rejected | (!padded & (len < p.min_len))) return;
  if (padded && len > p.lb) len = p.lb;
  const int64_t first = max(len - p.W, (int64_t)0);   // of a row longer than the window its last W steps stay
  const int64_t base_tok = padded ? 0 : off;
  const int64_t nk_row = (padded ? n * p.nk_sn : base_tok * p.nk_sl) + first * p.nk_sl;
  const int64_t nv_row = (padded ? n * p.nv_sn : base_tok * p.nv_sl) + first * p.nv_sl;
  const int64_t ring_base = ((slot * p.hkv + h) * (int64_t)(p.W + 1)) * D;
  const int c0 = (int)((start + first) % p.W);   // ring column of the first step written; at most W follow it
  // 8-byte pieces e = (token j, dims 4 i ..): a thread's pieces are loaded in batches of WB before any of them
  // is stored (the ring and the new rows could alias as far as the compiler knows, so a load after a store
  // would wait for it)
  constexpr int WB = 8;
  const int total = (int)(len - first) * (D / 4);
  for (int e0 = blockIdx.y * (256 * WB) + threadIdx.x; e0 < total; e0 += gridDim.y * (256 * WB)) {
    uint2 kw[WB], vw[WB];
#pragma unroll
    for (int u = 0; u < WB; ++u) {
      const int e = min(e0 + 256 * u, total - 1);
      const int j = e / (D / 4);
      const int d = (e - j * (D / 4)) * 4;
      kw[u] = *reinterpret_cast<const uint2*>(p.new_k + nk_row + j * p.nk_sl + h * p.nk_sh + d);
      vw[u] = *reinterpret_cast<const uint2*>(p.new_v + nv_row + j * p.nv_sl + h * p.nv_sh + d);
    }
#pragma unroll
    for (int u = 0; u < WB; ++u) {
      const int e = e0 + 256 * u;
      if (e < total) {
        const int j = e / (D / 4);
        const int d = (e - j * (D / 4)) * 4;
        const int col = c0 + j < p.W ? c0 + j : c0 + j - p.W;
        const int64_t dst = ring_base + (int64_t)col * D + d;
        *reinterpret_cast<uint2*>(p.ring_k + dst) = kw[u];
        *reinterpret_cast<uint2*>(p.ring_v + dst) = vw[u];
      }
    }
  }
}

}  // namespace
}  // namespace hsg

extern "C" int hsg_ring_attention(const void* q, int64_t q_sn, int64_t q_sl, int64_t q_sh, int64_t q_sg,
                                  void* ring_k, void* ring_v, int64_t ring_rows, int32_t window,
                                  const void* new_k, int64_t nk_sn, int64_t nk_sl, int64_t nk_sh,
                                  const void* new_v, int64_t nv_sn, int64_t nv_sl, int64_t nv_sh,
                                  const void* gate, int64_t g_sn, int64_t g_sl, int64_t g_sh, int64_t g_sg,
                                  int64_t g_off, const int64_t* ring_pos, const int64_t* slots,
                                  const int64_t* starts, const int64_t* lens, const int64_t* offsets,
                                  int32_t n_rows, int32_t lb, int32_t hkv, int32_t groups, int32_t head_dim,
                                  float scale, int32_t write_ring, int32_t min_len, void* out, int64_t o_sn,
                                  int64_t o_sl, int64_t o_sh, int64_t o_sg, void* stream) {
  using namespace hsg;
  if (n_rows < 0 || lb <= 0 || hkv <= 0 || groups <= 0 || ring_rows <= 0) return HSG_ERR_ARG;
  if (n_rows == 0) return HSG_OK;
  if (!q || !ring_k || !ring_v || !new_k || !new_v || !ring_pos || !slots || !starts || !lens || !out)
    return HSG_ERR_ARG;
  if (head_dim != D || window <= 0 || window > W_MAX || window % KB != 0 || lb > LB_MAX) return HSG_ERR_SHAPE;
  if (write_ring && lb > window) return HSG_ERR_SHAPE;  // two steps of one tick would share a ring column
  const int64_t s16[] = {q_sn, q_sl, q_sh, q_sg, nk_sn, nk_sl, nk_sh, nv_sn, nv_sl, nv_sh};
  for (int64_t s : s16)
    if (s % 8) return HSG_ERR_ALIGN;
  const int64_t s4[] = {g_sn, g_sl, g_sh, g_sg, g_off, o_sn, o_sl, o_sh, o_sg};
  for (int64_t s : s4)
    if (s % 4) return HSG_ERR_ALIGN;
  if (!aligned(q, 16) || !aligned(ring_k, 16) || !aligned(ring_v, 16) || !aligned(new_k, 16) ||
      !aligned(new_v, 16) || !aligned(out, 8) || (gate && !aligned(gate, 8)))
    return HSG_ERR_ALIGN;
  RingParams p{};
  p.q = static_cast<const uint16_t*>(q); p.q_sn = q_sn; p.q_sl = q_sl; p.q_sh = q_sh; p.q_sg = q_sg;
  p.ring_k = static_cast<uint16_t*>(ring_k); p.ring_v = static_cast<uint16_t*>(ring_v);
  p.ring_rows = ring_rows; p.W = window;
  p.new_k = static_cast<const uint16_t*>(new_k); p.nk_sn = nk_sn; p.nk_sl = nk_sl; p.nk_sh = nk_sh;
  p.new_v = static_cast<const uint16_t*>(new_v); p.nv_sn = nv_sn; p.nv_sl = nv_sl; p.nv_sh = nv_sh;
  p.gate = static_cast<const uint16_t*>(gate);
  p.g_sn = g_sn; p.g_sl = g_sl; p.g_sh = g_sh; p.g_sg = g_sg; p.g_off = g_off;
  p.ring_pos = ring_pos; p.slots = slots; p.starts = starts; p.lens = lens; p.offsets = offsets;
  p.lb = lb; p.hkv = hkv; p.G = groups; p.scale = scale; p.write_ring = write_ring; p.min_len = min_len;
  p.out = static_cast<uint16_t*>(out); p.o_sn = o_sn; p.o_sl = o_sl; p.o_sh = o_sh; p.o_sg = o_sg;
  p.pairs = n_rows * hkv;
  p.qgroups = (groups * lb + NW * TQ - 1) / (NW * TQ);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(ring_attn_kernel, dim3((unsigned)(p.pairs * p.qgroups)), dim3(NW * 64), 0, st, p);
  if (write_ring) hipLaunchKernelGGL(ring_write_kernel, dim3((unsigned)(n_rows * hkv)), dim3(256), 0, st, p);
  return launch_status();
}

extern "C" int hsg_window_attention(const void* q, int64_t q_sl, int64_t q_sh, int64_t q_sg, const void* k,
                                    int64_t k_sl, int64_t k_sh, const void* v, int64_t v_sl, int64_t v_sh,
                                    const void* gate, int64_t g_sl, int64_t g_sh, int64_t g_sg, int64_t g_off,
                                    const int64_t* lens, const int64_t* offsets, int32_t n_rows, int32_t max_len,
                                    int32_t first, int32_t count, int32_t window, int32_t hkv, int32_t groups,
                                    int32_t head_dim, float scale, void* out, int64_t o_sl, int64_t o_sh,
                                    int64_t o_sg, void* stream) {
  using namespace hsg;
  if (n_rows < 0 || max_len <= 0 || first < 0 || count <= 0 || hkv <= 0 || groups <= 0) return HSG_ERR_ARG;
  if (n_rows == 0) return HSG_OK;
  if (!q || !k || !v || !lens || !offsets || !out) return HSG_ERR_ARG;
  if (head_dim != D || window <= 0 || window > W_MAX) return HSG_ERR_SHAPE;
  constexpr int GR = NW * TQ;   // query rows of a workgroup
  const int64_t rows = (int64_t)groups * max_len;
  if (rows > (1 << 30) || (int64_t)first * groups % GR) return HSG_ERR_SHAPE;
  const int64_t strides[] = {q_sl, q_sh, q_sg, k_sl, k_sh, v_sl, v_sh};
  for (int64_t st : strides)
    if (st % 8) return HSG_ERR_ALIGN;
  const int64_t s4[] = {g_sl, g_sh, g_sg, g_off, o_sl, o_sh, o_sg};
  for (int64_t st : s4)
    if (st % 4) return HSG_ERR_ALIGN;
  if (!aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || !aligned(out, 8) || (gate && !aligned(gate, 8)))
    return HSG_ERR_ALIGN;
  if (first >= max_len) return HSG_OK;
  const int64_t last = (int64_t)first + count < max_len ? (int64_t)first + count : max_len;
  const int64_t qgroups = (last * groups + GR - 1) / GR - (int64_t)first * groups / GR;
  const int64_t blocks = ((int64_t)n_rows * hkv * qgroups + 7) / 8 * 8;
  if (blocks >= (1 << 24)) return HSG_ERR_SHAPE;   // a launch holds less than 2^32 threads
  RingParams p{};
  p.q = static_cast<const uint16_t*>(q); p.q_sl = q_sl; p.q_sh = q_sh; p.q_sg = q_sg;
  p.W = window;
  p.new_k = static_cast<const uint16_t*>(k); p.nk_sl = k_sl; p.nk_sh = k_sh;
  p.new_v = static_cast<const uint16_t*>(v); p.nv_sl = v_sl; p.nv_sh = v_sh;
  p.gate = static_cast<const uint16_t*>(gate); p.g_sl = g_sl; p.g_sh = g_sh; p.g_sg = g_sg; p.g_off = g_off;
  p.lens = lens; p.offsets = offsets;
  p.lb = max_len; p.hkv = hkv; p.G = groups; p.scale = scale; p.min_len = 0;
  p.pairs = n_rows * hkv;
  p.qgroups = (int)qgroups;
  p.qg0 = (int)((int64_t)first * groups / GR);
  p.sequences = 1;
  p.out = static_cast<uint16_t*>(out); p.o_sl = o_sl; p.o_sh = o_sh; p.o_sg = o_sg;
  hipLaunchKernelGGL(ring_attn_kernel, dim3((unsigned)blocks), dim3(NW * 64), 0, reinterpret_cast<hipStream_t>(stream), p);
  return launch_status();
}

extern "C" int hsg_ring_prefill(const void* q, int64_t q_sl, int64_t q_sh, int64_t q_sg, void* ring_k, void* ring_v,
                                int64_t ring_rows, int32_t window, const void* new_k, int64_t nk_sl, int64_t nk_sh,
                                const void* new_v, int64_t nv_sl, int64_t nv_sh, const void* gate, int64_t g_sl,
                                int64_t g_sh, int64_t g_sg, int64_t g_off, const int64_t* ring_pos,
                                const int64_t* slots, const int64_t* starts, const int64_t* lens,
                                const int64_t* offsets, int32_t n_rows, int32_t max_len, int32_t hkv, int32_t groups,
                                int32_t head_dim, float scale, void* out, int64_t o_sl, int64_t o_sh, int64_t o_sg,
                                void* stream) {
  using namespace hsg;
  if (n_rows < 0 || max_len <= 0 || hkv <= 0 || groups <= 0 || ring_rows <= 0) return HSG_ERR_ARG;
  if (n_rows == 0) return HSG_OK;
  if (!q || !ring_k || !ring_v || !new_k || !new_v || !ring_pos || !slots || !starts || !lens || !offsets || !out)
    return HSG_ERR_ARG;
  if (head_dim != D || window <= 0 || window > W_MAX || window % KB != 0) return HSG_ERR_SHAPE;
  if ((int64_t)groups * max_len > (1 << 30)) return HSG_ERR_SHAPE;
  const int64_t s16[] = {q_sl, q_sh, q_sg, nk_sl, nk_sh, nv_sl, nv_sh};
  for (int64_t st : s16)
    if (st % 8) return HSG_ERR_ALIGN;
  const int64_t s4[] = {g_sl, g_sh, g_sg, g_off, o_sl, o_sh, o_sg};
  for (int64_t st : s4)
    if (st % 4) return HSG_ERR_ALIGN;
  if (!aligned(q, 16) || !aligned(ring_k, 16) || !aligned(ring_v, 16) || !aligned(new_k, 16) ||
      !aligned(new_v, 16) || !aligned(out, 8) || (gate && !aligned(gate, 8)))
    return HSG_ERR_ALIGN;
  const int64_t qgroups = ((int64_t)groups * max_len + NW * TQ - 1) / (NW * TQ);
  const int64_t blocks = ((int64_t)n_rows * hkv * qgroups + 7) / 8 * 8;
  if (blocks >= (1 << 24)) return HSG_ERR_SHAPE;   // a launch holds less than 2^32 threads
  RingParams p{};
  p.q = static_cast<const uint16_t*>(q); p.q_sl = q_sl; p.q_sh = q_sh; p.q_sg = q_sg;
  p.ring_k = static_cast<uint16_t*>(ring_k); p.ring_v = static_cast<uint16_t*>(ring_v);
  p.ring_rows = ring_rows; p.W = window;
  p.new_k = static_cast<const uint16_t*>(new_k); p.nk_sl = nk_sl; p.nk_sh = nk_sh;
  p.new_v = static_cast<const uint16_t*>(new_v); p.nv_sl = nv_sl; p.nv_sh = nv_sh;
  p.gate = static_cast<const uint16_t*>(gate); p.g_sl = g_sl; p.g_sh = g_sh; p.g_sg = g_sg; p.g_off = g_off;
  p.ring_pos = ring_pos; p.slots = slots; p.starts = starts; p.lens = lens; p.offsets = offsets;
  p.lb = max_len; p.hkv = hkv; p.G = groups; p.scale = scale; p.write_ring = 1; p.min_len = 1;
  p.pairs = n_rows * hkv;
  p.qgroups = (int)qgroups;
  p.sequences = 1;
  p.out = static_cast<uint16_t*>(out); p.o_sl = o_sl; p.o_sh = o_sh; p.o_sg = o_sg;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(ring_attn_kernel, dim3((unsigned)blocks), dim3(NW * 64), 0, st, p);
  // 32 steps (one batch of the kernel) a workgroup: with one workgroup a pair, 12 pairs of 512 steps took 31 us
  const unsigned batches = (unsigned)((max_len < window ? max_len : window) + 31) / 32;
  hipLaunchKernelGGL(ring_write_kernel, dim3((unsigned)p.pairs, batches), dim3(256), 0, st, p);
  return launch_status();
}
