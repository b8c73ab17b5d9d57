// K3: write/encode of new tokens into compressed slots, two launches for all tokens of a layer.
// gfx950 / CDNA4.
//
// Few tokens per request (a decode step has one): 256-thread workgroups per token, so a batch of B
// tokens spreads its B x 450 KB of pinv and B x 132 KB of decoder reads over many CUs. Calls of more
// tokens take the same two launches in tiles of up to 16 tokens of one request
// (project_tiles_kernel, pack_tiles_kernel), which read its pinv and decoder once per tile:
//   K3a project  one workgroup per (token, 4 ranks): c[a] for its ranks over all H*d
//             dims, complete in the workgroup (wave sums, fixed order), left in the workspace
//                                                                  -- skipped when a fit gives (cq, cs)
//   K3b pack     one workgroup per (token, KV head): every head's workgroup quantises c alike,
//             then the rest for its head:
//   project   c[a] = sum_m M[m] * pinv[m][a], M = the token's raw key flattened m = h*d + j
//             (encode.py:322-324), fp32 in a fixed order          -- or take (cq, cs) from a fit
//   quantise  cs = max|c| * fp32(1/127) (1 if 0); cq = clamp(rint(c / cs), -128, 127)
//             (encode.py:328-332; the fp32 reciprocal multiply is torch-CUDA's scalar division,
//             select_triton.py:76-84; c/cs is a correctly rounded division)
//   residual  R[h][j] = K[h][j] - sum_a (cq[a]*cs) * decoder_f[a][h*d+j]   (encode.py:334-336)
//   rows      for every head: K residual row from R, V row from the value; each row picks exactly
//             k lanes by magnitude (ties -> lowest lane, select_triton.py:181-193), ruler =
//             rowmax * fp32(1/(2^(b-1)-1)) (1 * that if rowmax == 0), q = clamp(rint(x / ruler)),
//             bitmap MSB-first, codes MSB-first in lane order, fp16 ruler LE
//             (ttkv_packed_cache.py:203-231, select_triton.py:195-232)
//   store     coefficients, fp16 coefficient ruler, H K rows, H V rows, zero padding: the
//             bytes layout.pack_k_slots/pack_v_slots produce (layout.py:161-239), written at
//             slot_mapping[i] (encode.py:471-508).
// Selection, quantisation and packing are bit-exact functions of their float inputs (R and the
// value); the projection and reconstruction sums are fp32 with an implementation-defined order,
// as in the reference. Optional outputs expose c and R so tests can pin the bytes from there.
#include <math.h>

#include "ttkv_device.h"
#include "ttkv_host.h"

namespace ttkv {

constexpr int kWThreads = 256;

struct WriteArgs {
  Geom g;
  const void* key;
  int k_dtype;
  int64_t k_row_stride;
  const void* val;
  int v_dtype;
  int64_t v_row_stride;
  const int64_t* slot_mapping;
  int num_tokens;
  const int32_t* qsl;
  int num_reqs;
  const int32_t* bt;
  int64_t bt_row_stride;
  const int32_t* dec_map;
  int64_t num_blocks;
  const int8_t* dec_q;  // decoder pool (see dec_ranks)
  const float* dec_scale;
  const float* pinv_pool;
  int64_t n_dec_slots;
  int32_t* dec_used;  // [n_dec_slots] or null: set to 1 for every decoder slot a token uses
  const int8_t* cq_in;
  const float* cs_in;
  uint8_t* page;
  int64_t n_slots, slot_stride;
  float* c_out;
  float* r_out;
  int* err;
  int tok0;         // first token of this launch (tokens tok0 .. tok0 + num_tokens - 1)
  int tiles;        // at most so many tiles hold its tokens (tiled launches)
  float* ws_c;      // [num_tokens][r1] each token's projection c, from K3a for K3b
  int* ws_ds;       // [num_tokens] each token's decoder slot (or -1), from K3a for K3b
  float inv127, inv_rk, inv_rv;
};

// Decoder slot of the request whose first block is blk0, or -1.
__device__ __forceinline__ int decoder_of_block(const WriteArgs& a, int blk0) {
  const int ds = blk0 >= 0 && blk0 < a.num_blocks ? a.dec_map[blk0] : -1;
  return ds < 0 || ds >= a.n_dec_slots ? -1 : ds;
}

// Request of token i (qsl[r] <= i < qsl[r+1]; qsl is non-decreasing) and its decoder slot, or
// -1. Decode tokens come first in a step, one per request, so token i is usually request i: that
// guess, its first block id and the general count (r + 1 = the number of qsl[0..num_reqs) <= i,
// 64 per lane with one load each) are requested in one round trip; a confirmed guess leaves only
// the decoder map's round trip (two in all instead of three). Every lane of the wave must call
// it; all get the same answer.
__device__ int token_decoder(const WriteArgs& a, int i) {
  const int lane = threadIdx.x & 63;
  const bool guess = i < a.num_reqs;
  const int glo = guess ? a.qsl[i] : 0, ghi = guess ? a.qsl[i + 1] : 0;
  const int gblk = guess ? a.bt[(int64_t)i * a.bt_row_stride] : -1;
  int cnt = 0;
  for (int j0 = 0; j0 < a.num_reqs; j0 += 64) {
    const int j = j0 + lane;
    cnt += __builtin_popcountll(__ballot(j < a.num_reqs && a.qsl[j] <= i));
  }
  int blk0 = -1;
  if (guess && glo <= i && i < ghi) {
    blk0 = gblk;
  } else {
    const int r = cnt - 1;
    if (r >= 0 && i < a.qsl[r + 1]) blk0 = a.bt[(int64_t)r * a.bt_row_stride];
  }
  return decoder_of_block(a, blk0);
}

// Exact top-k select + quantise + pack of one 128-lane row held as lane l: x0 = dim l,
// x1 = dim l+64. Writes bitmap, codes and fp16 ruler at dst (any alignment). `sw` is this
// wave's LDS scratch of kStreamWords dwords. Every lane of the wave must call it.
//
// The k-th largest magnitude t is searched on the (monotone) magnitude bit pattern, between lo
// (at least k lanes are >= lo) and hi (fewer than k are >= hi). The first cut is the largest
// magnitude / 64 (six exponents), then the interval is halved, and the search ends as soon as a
// cut has exactly k lanes above it: about 10 steps of dependent ballots on rows of normal values
// where building t bit by bit takes 31. Rows with ties, or with a longer tail, take the steps
// they need (at most 32).
constexpr int kStreamWords = 17;  // 128 codes of 4 bits, and the word a 3-bit code may reach into

template <int BITS>
__device__ __forceinline__ void pack_row(float x0, float x1, int k, float inv_ruler, uint8_t* dst,
                                         uint32_t* sw) {
  constexpr int OFF = 1 << (BITS - 1);
  const int lane = threadIdx.x & 63;
  const uint32_t u0 = __builtin_bit_cast(uint32_t, fabsf(x0));
  const uint32_t u1 = __builtin_bit_cast(uint32_t, fabsf(x1));
  if (lane < kStreamWords) sw[lane] = 0;
  // Row max (always kept when k >= 1), as bits: non-negative floats order like their bits.
  const uint32_t mx = (uint32_t)wave_max_i((int)(u0 > u1 ? u0 : u1));
  uint32_t lo = 0, hi = mx + 1;
  int at_lo = kD;  // lanes >= lo
  uint32_t cut = mx > (6u << 23) ? mx - (6u << 23) : (lo + hi) >> 1;
  while (hi - lo > 1 && at_lo != k) {
    const int cnt = __builtin_popcountll(__ballot(u0 >= cut)) +
                    __builtin_popcountll(__ballot(u1 >= cut));
    if (cnt >= k) {
      lo = cut;
      at_lo = cnt;
    } else {
      hi = cut;
    }
    cut = lo + ((hi - lo) >> 1);
  }
  const uint64_t below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  uint64_t sel0 = __ballot(u0 >= lo), sel1 = __ballot(u1 >= lo);
  if (at_lo != k) {  // more than k lanes reach t = lo: those equal to it by lowest lane
    const uint64_t above0 = __ballot(u0 > lo), above1 = __ballot(u1 > lo);
    const int need = k - (__builtin_popcountll(above0) + __builtin_popcountll(above1));
    const uint64_t tie0 = sel0 & ~above0, tie1 = sel1 & ~above1;
    const int tr0 = __builtin_popcountll(tie0 & below);
    const int tr1 = __builtin_popcountll(tie0) + __builtin_popcountll(tie1 & below);
    sel0 = __ballot(u0 > lo || (u0 == lo && tr0 < need));
    sel1 = __ballot(u1 > lo || (u1 == lo && tr1 < need));
  }
  const bool s0 = (sel0 >> lane) & 1, s1 = (sel1 >> lane) & 1;
  const float rmax = __builtin_bit_cast(float, mx);
  const float sc = (rmax == 0.f ? 1.f : rmax) * inv_ruler;
  // Codes by rank (lane order), OR-ed into the big-endian stream words: code r at stream bits
  // [r * BITS, r * BITS + BITS).
  const int rank0 = __builtin_popcountll(sel0 & below);
  const int rank1 = __builtin_popcountll(sel0) + __builtin_popcountll(sel1 & below);
  auto put = [&](float x, int rank) {
    const float q = fminf(fmaxf(rintf(__fdiv_rn(x, sc)), (float)-OFF), (float)(OFF - 1));
    const uint32_t code = (uint32_t)((int)q + OFF);
    const int p = rank * BITS;
    const int sh = 32 - BITS - (p & 31);
    if (BITS == 4 || sh >= 0) {
      atomicOr(&sw[p >> 5], code << sh);
    } else {  // the code straddles two words
      atomicOr(&sw[p >> 5], code >> -sh);
      atomicOr(&sw[(p >> 5) + 1], code << (32 + sh));
    }
  };
  if (s0) put(x0, rank0);
  if (s1) put(x1, rank1);
  // (LDS accesses of one wave complete in order: the fences only keep the compiler from moving
  // them)
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int pb = (k * BITS + 7) / 8;
  // Bitmap: byte m holds dims 8m..8m+7, dim 8m at bit 7.
  if (lane < 16) {
    const uint64_t sel = lane < 8 ? sel0 : sel1;
    const uint32_t byte = (uint32_t)(sel >> (8 * (lane & 7))) & 0xffu;
    dst[lane] = (uint8_t)(__builtin_bitreverse32(byte) >> 24);
  }
  // Code stream: byte b = stream bits [8b, 8b+8), MSB first, zero beyond k codes.
  if (lane < pb) dst[16 + lane] = (uint8_t)(sw[lane >> 2] >> (24 - 8 * (lane & 3)));
  if (lane == 0) {
    const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)sc);
    dst[16 + pb] = (uint8_t)(hb & 0xff);
    dst[16 + pb + 1] = (uint8_t)(hb >> 8);
  }
  // the next row's clearing of `sw` stays behind this row's reads
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Scale of a 4-bit coefficient group whose largest magnitude is m: m / 7 (IEEE) rounded up to 8
// significant bits, then held within [2^-14, 9344], so that every q * scale (|q| <= 7) is an
// exact fp16 normal; 0 for an all-zero group.
__device__ inline float coef_group_scale(float m) {
  if (!(m > 0.f)) return 0.f;
  uint32_t u = __builtin_bit_cast(uint32_t, __fdiv_rn(m, 7.f));
  if (u & 0xffffu) u = (u & ~0xffffu) + 0x10000u;
  return fminf(fmaxf(__builtin_bit_cast(float, u), 0x1p-14f), 9344.f);
}

// Byte b of the 4-bit coefficient field: of word w = b / 4 it holds the nibbles of ranks lo (bits
// 0-3) and lo + 2 (bits 4-7), lo = 8w + 4j for byte j < 2 of the word, 8w + 4j - 7 for j >= 2.
// value(r) is q * scale exactly, so q = value / scale.
template <typename F>
__device__ __forceinline__ uint8_t nibble_byte(int b, int r1, F value, const float* gsc) {
  const int j = b & 3;
  const int lo = 8 * (b >> 2) + (j < 2 ? 4 * j : 4 * j - 7);
  uint32_t byte = 0;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int r = lo + 2 * e;
    if (r < r1) {
      const float sc = gsc[r >> 5];
      const int q = sc > 0.f ? (int)rintf(__fdiv_rn(value(r), sc)) : 0;
      byte |= ((uint32_t)q & 15u) << (4 * e);
    }
  }
  return (uint8_t)byte;
}

// K3a: the projection c = M_i . pinv of token i, one workgroup per (token, slice of kSliceRanks
// ranks). The pool holds each decoder's pseudo-inverse by rank (pinv_pool [slot][r1][H*d], row a
// = rank a's projection vector), so each wave reads whole rows: kWaveRanks ranks from a0 +
// kWaveRanks * w, each lane 16 of the H*d dims (four 16-byte loads per rank, 1 KB per wave
// instruction). Slices of 16 / 8 / 4 ranks measured 4.8 / 4.7 / 4.6 us per 8-token launch (more,
// smaller workgroups spread the pinv reads over more CUs). The wave sums each
// rank over its lanes with an xor butterfly, so every rank's sum is complete inside one workgroup
// and nothing is handed between workgroups; K3b quantises.
constexpr int kSliceRanks = 4;
constexpr int kWaveRanks = kSliceRanks / 4;  // ranks per wave

__host__ __device__ inline int project_slices(const Geom& g) {
  return (g.r1 + kSliceRanks - 1) / kSliceRanks;
}

// A tile: up to kTok tokens of one request, so that its pseudo-inverse and decoder are read once
// per tile and not once per token, and both contractions run on MFMA. (Tiles of 16 tokens whatever
// their requests need a pass per distinct decoder, about 7 us each one after another: 128 requests of 3
// tokens took 78 us, token by token 44.)
constexpr int kTok = 16;

// At most so many tiles hold n tokens of num_reqs requests (and those before and after them all).
__host__ inline int tile_bound(int n, int num_reqs) {
  return (int)((n + (int64_t)(kTok - 1) * std::min<int64_t>((int64_t)num_reqs + 2, n)) / kTok);
}

// The tile of block b of a launch's tile part, `per` blocks per tile. Blocks go round-robin over the
// 8 XCDs, so a tile's blocks are 8 apart: one XCD's L2 serves all of them the tile's keys, and
// merges the pieces of its slots' lines that they write.
__device__ __forceinline__ int tile_of(int b, int per) { return (b >> 3) / per * 8 + (b & 7); }
__host__ inline int tile_blocks(int tiles, int per) { return (tiles + 7) / 8 * 8 * per; }

// The tokens of one tile, tokens il0 .. il0 + nt - 1 of the launch (nt = 0: no such tile), and
// their request's first block id (-1: none).
struct TileTokens {
  int il0, nt, blk0;
};

// Tiles are numbered request by request; the tokens before the first request and after the last,
// which are refused unless they are padding, count as requests without a block. Lane j takes span j
// of 64 (one round trip), a scan of their tile counts finds the tile's. Every lane of the wave must
// call it; all get the same answer.
__device__ TileTokens find_tile(const WriteArgs& a, int tile) {
  const int lane = threadIdx.x & 63;
  const int s0 = a.tok0, s1 = a.tok0 + a.num_tokens;
  if (a.num_reqs == 1) {  // by scalar arithmetic (the scan costs 1 us of 47 with 2,048 tokens)
    const int q0 = min(max(a.qsl[0], s0), s1), q1 = min(max(a.qsl[1], q0), s1);
    const int head = (q0 - s0 + kTok - 1) / kTok, mid = (q1 - q0 + kTok - 1) / kTok;
    const bool in_head = tile < head, in_mid = !in_head && tile < head + mid;
    const int lo = in_head ? s0 : in_mid ? q0 : q1, hi = in_head ? q0 : in_mid ? q1 : s1;
    const int first = lo + (tile - (in_head ? 0 : in_mid ? head : head + mid)) * kTok;
    return {first - s0, min(kTok, max(hi - first, 0)), in_mid ? a.bt[0] : -1};
  }
  int before = 0;
  for (int j0 = 0; j0 < a.num_reqs + 2; j0 += 64) {  // span j: request j - 1
    const int j = j0 + lane, r = j - 1;
    int lo = j > 0 && r <= a.num_reqs ? a.qsl[r] : s0;
    int hi = j <= a.num_reqs ? a.qsl[j] : s1;
    const int blk = r >= 0 && r < a.num_reqs ? a.bt[(int64_t)r * a.bt_row_stride] : -1;
    lo = min(max(lo, s0), s1);
    hi = min(max(hi, lo), s1);
    const int own = r <= a.num_reqs ? (hi - lo + kTok - 1) / kTok : 0;
    int upto = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(upto, o);
      upto += lane >= o ? up : 0;
    }
    const uint64_t in = __ballot(before + upto - own <= tile && tile < before + upto);
    if (in) {
      const int l = __builtin_ctzll(in);
      auto at = [&](int v) { return __builtin_amdgcn_readlane(v, l); };
      const int first = at(lo) + (tile - (before + at(upto) - at(own))) * kTok;
      return {first - s0, min(kTok, at(hi) - first), at(blk)};
    }
    before += __builtin_amdgcn_readlane(upto, 63);
  }
  return {0, 0, -1};
}

__host__ __device__ inline int rank_groups(const Geom& g) { return (g.r1 + 15) / 16; }

// Four consecutive activations as loaded; KDT is their type, KVEC whether they take one wide load.
template <int KDT, bool KVEC>
struct RawAct4 {
  u32x4 w;
  __device__ __forceinline__ void load(const void* p, int64_t i) {
    if constexpr (KDT == TTKV_DTYPE_F32) {
      const uint32_t* q = (const uint32_t*)p + i;
      if constexpr (KVEC) {
        w = *gbl((const u32x4*)q);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = *gbl(q + j);
      }
    } else {
      const uint16_t* q = (const uint16_t*)p + i;
      if constexpr (KVEC) {
        const u32x2v x = *gbl((const u32x2v*)q);
        w[0] = x[0];
        w[1] = x[1];
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = *gbl(q + j);
      }
    }
  }
  __device__ __forceinline__ float value(int j) const {
    // (through a copy: a bit cast of a vector's element itself reads element 0)
    const uint32_t x = w[j];
    if constexpr (KDT == TTKV_DTYPE_F32) return __builtin_bit_cast(float, x);
    const uint32_t b = KVEC ? (w[j >> 1] >> (16 * (j & 1))) & 0xffffu : w[j];
    return KDT == TTKV_DTYPE_F16 ? f16_bits_to_float(b) : bf16_bits_to_float(b);
  }
};

// K3a for tiles: c[16 tokens][16 ranks] in one workgroup, fp32 MFMA 16x16x4 (A = the tokens' keys,
// B = the ranks' pinv rows). Wave w contracts its quarter of the H*d dims: per 16 dims each lane
// holds dims 4gq .. 4gq + 3 of its token and of its rank (one wide load each), and step j takes
// element j of both, so the contraction runs in an order of its own but over every dim once.
// Four accumulators take the steps j = 0..3 and are added pairwise, then the four waves' sums,
// so no chain of additions is longer than one wave's dims / 16. The keys are requested before the
// decoder is looked up.
// Bound: the round trips of the lookup and of the operands, 64 KB of pinv rows per workgroup from
// L2. 2,048 tokens: 18.8 us, where a workgroup per (token, 4 ranks) takes 103 us (450 KB of
// pinv per token).
template <int KDT, bool KVEC>
__global__ __launch_bounds__(kWThreads) void project_tiles_kernel(WriteArgs a) {
  __shared__ float part[4][kTok][kTok + 1];
  const Geom& g = a.g;
  const int rgs = rank_groups(g);
  const int tile = tile_of(blockIdx.x, rgs), rg = (int)(blockIdx.x >> 3) % rgs;
  if (tile >= a.tiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, gq = lane >> 4;
  const TileTokens tt = find_tile(a, tile);
  if (tt.nt == 0) return;
  const int il0 = tt.il0, nt = tt.nt;
  const int i0 = a.tok0 + il0;
  const int HD = g.H * kD;
  const int groups = HD >> 6;  // 16-dim groups per wave: 2 H
  const int64_t kb = (int64_t)(i0 + min(n, nt - 1)) * a.k_row_stride + 16 * wv * groups + 4 * gq;
  constexpr int kStep = 8;  // groups whose loads are in flight together
  RawAct4<KDT, KVEC> kx[kStep];
  auto load_keys = [&](int u0) {
#pragma unroll
    for (int u = 0; u < kStep; ++u) kx[u].load(a.key, kb + 16 * min(u0 + u, groups - 1));
  };
  load_keys(0);
  __builtin_amdgcn_sched_barrier(0);
  const int64_t slot = lane < nt ? a.slot_mapping[i0 + lane] : -1;
  const int ds = decoder_of_block(a, tt.blk0);
  if (rg == 0 && tid < nt) a.ws_ds[il0 + tid] = ds;
  const uint64_t ok = __ballot(slot >= 0 && slot < a.n_slots);
  if (ds < 0 || !ok) return;  // alike in every wave; K3b reports it
  const int rank = 16 * rg + n;
  const float* prow = a.pinv_pool + ((int64_t)ds * g.r1 + min(rank, g.r1 - 1)) * HD +
                      16 * wv * groups + 4 * gq;
  float4v acc[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f},
                    {0.f, 0.f, 0.f, 0.f}};
  for (int u0 = 0; u0 < groups; u0 += kStep) {
    float4v pv[kStep];
#pragma unroll
    for (int u = 0; u < kStep; ++u)
      pv[u] = *gbl((const float4v*)(prow + 16 * min(u0 + u, groups - 1)));
    if (u0) load_keys(u0);
    // (the scheduler would otherwise spread the loads between the MFMAs and wait for each)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kStep; ++u) {
      const bool in = u0 + u < groups;  // past the last group: zeros
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? kx[u].value(j) : 0.f,
                                                      in ? pv[u][j] : 0.f, acc[j], 0, 0, 0);
    }
  }
  const float4v s = (acc[0] + acc[1]) + (acc[2] + acc[3]);  // tokens 4gq .. 4gq + 3, rank n
#pragma unroll
  for (int i = 0; i < 4; ++i) part[wv][4 * gq + i][n] = s[i];
  __syncthreads();
  const int t = tid >> 4, r = tid & 15;
  if (((ok >> t) & 1) && 16 * rg + r < g.r1) {
    const float c = (part[0][t][r] + part[1][t][r]) + (part[2][t][r] + part[3][t][r]);
    a.ws_c[(int64_t)(il0 + t) * g.r1 + 16 * rg + r] = c;
    if (a.c_out) a.c_out[(int64_t)(i0 + t) * g.r1 + 16 * rg + r] = c;
  }
}

// K3a for single tokens: one workgroup per (token, kSliceRanks ranks).
__global__ __launch_bounds__(kWThreads) void write_project_kernel(WriteArgs a) {
  const int ns = project_slices(a.g);
  const int il = blockIdx.x / ns, sl = blockIdx.x % ns;
  const Geom& g = a.g;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int i = a.tok0 + il;  // il: the token's workspace row
  const int HD = g.H * kD;
  const int64_t slot = a.slot_mapping[i];
  // this lane's key dims 256j + 4 lane .. + 3, requested before the decoder lookup's round trips
  const int64_t kb = (int64_t)i * a.k_row_stride;
  const bool kvec = act_rows_aligned(a.key, a.k_dtype, a.k_row_stride);
  float kx[4][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d0 = 256 * j + 4 * lane;
    if (d0 < HD) {
      load_act_n<4>(a.key, a.k_dtype, kb + d0, kvec, kx[j]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) kx[j][e] = 0.f;
    }
  }
  const int ds = token_decoder(a, i);
  if (sl == 0 && tid == 0) a.ws_ds[il] = ds;
  if (ds < 0 || slot < 0 || slot >= a.n_slots) return;  // K3b reports it
  const int a0 = sl * kSliceRanks + kWaveRanks * wv;
  if (a0 >= g.r1) return;
  const float* prow = a.pinv_pool + (int64_t)ds * g.r1 * HD;
  float4v pv[kWaveRanks][4];
#pragma unroll
  for (int r = 0; r < kWaveRanks; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int d0 = 256 * j + 4 * lane;
      pv[r][j] = (a0 + r < g.r1 && d0 < HD)
                     ? *gbl((const float4v*)(prow + (int64_t)(a0 + r) * HD + d0))
                     : float4v{0.f, 0.f, 0.f, 0.f};
    }
  float acc[kWaveRanks];
#pragma unroll
  for (int r = 0; r < kWaveRanks; ++r) {
    acc[r] = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[r] = fmaf(kx[j][e], pv[r][j][e], acc[r]);
  }
  // butterfly: the same tree in every lane (operands only commuted), so every lane holds the sum
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int r = 0; r < kWaveRanks; ++r) acc[r] += __shfl_xor(acc[r], o);
  if (lane < kWaveRanks && a0 + lane < g.r1) {
    float c = acc[0];
#pragma unroll
    for (int r = 1; r < kWaveRanks; ++r) c = lane == r ? acc[r] : c;
    a.ws_c[(int64_t)il * g.r1 + a0 + lane] = c;
    if (a.c_out) a.c_out[(int64_t)i * g.r1 + a0 + lane] = c;
  }
}

// K3b for tiles: one 512-thread workgroup per (tile, head). Wave w quantises tokens 2w and 2w + 1
// (as the single token's workgroup does, lane l holding ranks l, l + 64, ..), the decoder's part
// of the keys is one fp32 MFMA contraction [128 dims x 16 tokens] (A = decoder values of dims 16w
// .. 16w + 15, B = c * cs), and each wave packs its tokens' K and V rows. The rows take most of
// the time (their selection is a chain of ballots), so the registers are held to what lets
// 6 waves share a SIMD.
// 2,048 tokens: 32 us (34 at 4 or 8 waves), where a workgroup per (token, head) takes 62 us.
constexpr int kPThreads = 512;
constexpr int kPWaves = kPThreads / 64;
constexpr int kPTok = kTok / kPWaves;  // tokens per wave
constexpr int kTileRanks = 256;
struct PackTileSmem {
  float coef[kTok][kTileRanks + 4];  // c * cs by rank (0 past r1)
  float rec[kTok][kD + 4];           // the decoder's part of each token's key
  float gsc[kPWaves][8];             // 4-bit mode: each wave's current token's group scales
  uint32_t stream[kPWaves][kStreamWords];
};

// Dims lane and 64 + lane of kPTok rows (elements rb[t] ..) as floats.
__device__ __forceinline__ void load_rows(const void* p, int dt, const int64_t rb[kPTok],
                                          float x[kPTok][2]) {
  const int lane = threadIdx.x & 63;
  if (dt == TTKV_DTYPE_F32) {
#pragma unroll
    for (int t = 0; t < kPTok; ++t)
#pragma unroll
      for (int e = 0; e < 2; ++e) x[t][e] = *gbl((const float*)p + rb[t] + 64 * e + lane);
    return;
  }
  uint32_t b[kPTok][2];
#pragma unroll
  for (int t = 0; t < kPTok; ++t)
#pragma unroll
    for (int e = 0; e < 2; ++e) b[t][e] = *gbl((const uint16_t*)p + rb[t] + 64 * e + lane);
#pragma unroll
  for (int t = 0; t < kPTok; ++t)
#pragma unroll
    for (int e = 0; e < 2; ++e)
      x[t][e] = dt == TTKV_DTYPE_F16 ? f16_bits_to_float(b[t][e]) : bf16_bits_to_float(b[t][e]);
}

template <int RB, int VB, int CM>
__global__ __launch_bounds__(kPThreads, 6) void pack_tiles_kernel(WriteArgs a) {
  __shared__ __align__(16) PackTileSmem S;
  const Geom& g = a.g;
  const int tile = tile_of(blockIdx.x, g.H), h = (int)(blockIdx.x >> 3) % g.H;
  if (tile >= a.tiles) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, gq = lane >> 4;
  const TileTokens tt = find_tile(a, tile);
  if (tt.nt == 0) return;
  const int il0 = tt.il0, nt = tt.nt;
  const int i0 = a.tok0 + il0;
  const int HD = g.H * kD;
  const int R = dec_ranks(g.r1);
  // the tile's slots (lane t: token t) and decoder, and this wave's tokens' rows
  const int64_t slot = lane < nt ? a.slot_mapping[i0 + lane] : -1;
  const int ds = a.cq_in ? decoder_of_block(a, tt.blk0) : a.ws_ds[il0];
  // (every load unconditional and behind no branch of its own, so that all are in flight together)
  const int nk = R >> 6;  // 64-rank groups in use
  float xk[kPTok][2], xv[kPTok][2], cw[kPTok][4] = {}, csin[kPTok];
  {
    int64_t kb[kPTok], vb[kPTok];
    int it[kPTok];
#pragma unroll
    for (int t = 0; t < kPTok; ++t) {
      it[t] = min(kPTok * wv + t, nt - 1);
      kb[t] = (int64_t)(i0 + it[t]) * a.k_row_stride + h * kD;
      vb[t] = (int64_t)(i0 + it[t]) * a.v_row_stride + h * kD;
    }
    load_rows(a.key, a.k_dtype, kb, xk);
    load_rows(a.val, a.v_dtype, vb, xv);
    if (a.cq_in) {
#pragma unroll
      for (int t = 0; t < kPTok; ++t) {
        csin[t] = a.cs_in[i0 + it[t]];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < nk) cw[t][k] = (float)*gbl(a.cq_in + (int64_t)(i0 + it[t]) * g.r1 + min(lane + 64 * k, g.r1 - 1));
      }
    } else {
#pragma unroll
      for (int t = 0; t < kPTok; ++t) {
        csin[t] = 1.f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < nk) cw[t][k] = *gbl(a.ws_c + (int64_t)(il0 + it[t]) * g.r1 + min(lane + 64 * k, g.r1 - 1));
      }
    }
#pragma unroll
    for (int t = 0; t < kPTok; ++t)
#pragma unroll
      for (int k = 0; k < 4; ++k) cw[t][k] = lane + 64 * k < g.r1 ? cw[t][k] : 0.f;
  }
  const bool live = slot >= 0;  // a negative slot id is vLLM's PAD_SLOT_ID: skipped silently
  if (h == 0 && wv == 0) {
    const bool bad_slot = __ballot(live && slot >= a.n_slots) != 0;
    const bool no_dec = __ballot(live && ds < 0) != 0;
    if (lane == 0 && (bad_slot || no_dec))
      atomicOr(a.err, (bad_slot ? TTKV_ERR_BAD_SLOT : 0) | (no_dec ? TTKV_ERR_NO_DECODER : 0));
    if (live && ds >= 0 && a.dec_used) a.dec_used[ds] = 1;
  }
  const uint64_t ok = __ballot(live && slot < a.n_slots && ds >= 0);
  if (!ok) return;  // alike in every wave
  // ---- quantise; each token's coefficients and padding are written by one of the heads
#pragma unroll
  for (int t = 0; t < kPTok; ++t) {
    const int tok = kPTok * wv + t;
    const int64_t sl = ((int64_t)__builtin_amdgcn_readlane((int)(slot >> 32), tok) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((int)slot, tok);
    uint8_t* base = a.page + sl * a.slot_stride;
    const bool store = tok % g.H == h && ((ok >> tok) & 1);  // the heads share the tokens
    float cs = csin[t], qv[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) qv[k] = cw[t][k];
    if (!a.cq_in) {
      if constexpr (CM == kCoefI8) {
        const float mx = wave_max(fmaxf(fmaxf(fabsf(qv[0]), fabsf(qv[1])),
                                        fmaxf(fabsf(qv[2]), fabsf(qv[3]))));
        cs = mx * a.inv127;
        if (cs == 0.f) cs = 1.f;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          if (k < nk) qv[k] = fminf(fmaxf(rintf(__fdiv_rn(qv[k], cs)), -128.f), 127.f);
      } else if constexpr (CM == kCoefF16) {
#pragma unroll
        for (int k = 0; k < 4; ++k) qv[k] = (float)(_Float16)qv[k];
      } else {  // group 2k + (lane >> 5) of ranks
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          if (k >= nk) break;
          float gm = fabsf(qv[k]);
#pragma unroll
          for (int o = 16; o > 0; o >>= 1) gm = fmaxf(gm, __shfl_xor(gm, o));
          const float sc = coef_group_scale(gm);
          if ((lane & 31) == 0) S.gsc[wv][2 * k + (lane >> 5)] = sc;
          qv[k] = sc > 0.f ? fminf(fmaxf(rintf(__fdiv_rn(qv[k], sc)), -7.f), 7.f) * sc : 0.f;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int r = lane + 64 * k;
      if (k >= nk) break;
      if (r >= g.r1) qv[k] = 0.f;
      if (r < R) S.coef[tok][r] = qv[k] * cs;
    }
    if (store) {  // wave-uniform
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int r = lane + 64 * k;
        if (r >= g.r1) continue;
        if constexpr (CM == kCoefI8) {
          base[r] = (uint8_t)(int8_t)(int)qv[k];
        } else if constexpr (CM == kCoefF16) {
          const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)qv[k]);
          base[2 * r] = (uint8_t)(hb & 0xff);
          base[2 * r + 1] = (uint8_t)(hb >> 8);
        }
      }
      if (CM == kCoefI8 && lane == 0) {
        const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)cs);
        base[g.coeff_bytes] = (uint8_t)(hb & 0xff);
        base[g.coeff_bytes + 1] = (uint8_t)(hb >> 8);
      }
      if constexpr (CM == kCoefI4G32) {
        // (this wave's LDS writes above are read back by the same wave, in order)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (lane < g.coef_groups) {
          const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)S.gsc[wv][lane]);
          base[g.coeff_bytes + 2 * lane] = (uint8_t)(hb & 0xff);
          base[g.coeff_bytes + 2 * lane + 1] = (uint8_t)(hb >> 8);
        }
        for (int b = lane; b < g.coeff_bytes; b += 64)
          base[b] = nibble_byte(b, g.r1, [&](int r) { return S.coef[tok][r]; }, S.gsc[wv]);
      }
      for (int b = g.k_field + g.H * g.k_row + lane; b < g.k_slot; b += 64) base[b] = 0;
      for (int b = g.k_slot + g.H * g.v_row + lane; b < g.blob; b += 64) base[b] = 0;
    }
    // the next token's group scales stay behind this one's reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  __syncthreads();
  // ---- the decoder's part of the keys: rec[token][dim], dims 16w .. 16w + 15 in this wave
  float4v rec;  // dims 16w + 4gq .. + 3 of token n
  {
    // per 64 ranks lane (n, gq) holds ranks 16gq .. 16gq + 15 of dim n (one 16-byte load) and of
    // token n; MFMA step (c, j) takes rank 16gq + 4c + j of every lane group
    float4v acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    const float* decs = a.dec_scale + (int64_t)ds * R + 16 * gq;
    const int8_t* decq = a.dec_q + ((int64_t)ds * HD + h * kD + 16 * wv + n) * R + 16 * gq;
    for (int s = 0; s < R; s += 64) {
      const u32x4 q16 = *gbl((const u32x4*)(decq + s));
      float4v rul[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) rul[c] = *gbl((const float4v*)(decs + s + 4 * c));
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int r = s + 16 * gq + 4 * c;
        const float4v cq = *(const float4v*)&S.coef[n][r];
#pragma unroll
        for (int j = 0; j < 4; ++j) rul[c][j] = r + j < g.r1 ? rul[c][j] : 0.f;
        float v[4];
        dec_values4(q16[c], rul[c], v);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[c & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], cq[j], acc[c & 1], 0, 0, 0);
      }
    }
    rec = acc[0] + acc[1];
  }
  *(float4v*)&S.rec[n][16 * wv + 4 * gq] = rec;
  __syncthreads();
  // ---- this wave's rows
#pragma unroll 1
  for (int t = 0; t < kPTok; ++t) {
    const int tok = kPTok * wv + t;
    if (!((ok >> tok) & 1)) continue;  // wave-uniform
    const int64_t sl = ((int64_t)__builtin_amdgcn_readlane((int)(slot >> 32), tok) << 32) |
                       (uint32_t)__builtin_amdgcn_readlane((int)slot, tok);
    uint8_t* base = a.page + sl * a.slot_stride;
    static_assert(kPTok == 2, "two tokens per wave");
    const float k0 = t ? xk[1][0] : xk[0][0], k1 = t ? xk[1][1] : xk[0][1];
    const float v0 = t ? xv[1][0] : xv[0][0], v1 = t ? xv[1][1] : xv[0][1];
    const float r0 = k0 - S.rec[tok][lane];
    const float r1v = k1 - S.rec[tok][64 + lane];
    if (a.r_out) {
      a.r_out[(int64_t)(i0 + tok) * HD + h * kD + lane] = r0;
      a.r_out[(int64_t)(i0 + tok) * HD + h * kD + 64 + lane] = r1v;
    }
    pack_row<RB>(r0, r1v, g.res_k, a.inv_rk, base + g.k_field + h * g.k_row, S.stream[wv]);
    pack_row<VB>(v0, v1, g.v_lanes, a.inv_rv, base + g.k_slot + h * g.v_row, S.stream[wv]);
  }
}

// K3b for single tokens, one workgroup per (token, head): residual of head h, then its K row and V
// row; head 0 also writes the coefficients.
template <int RB, int VB>
__global__ __launch_bounds__(kWThreads) void write_pack_kernel(WriteArgs a) {
  const int il = blockIdx.x / a.g.H, h = blockIdx.x % a.g.H;
  __shared__ __align__(16) float cqs[256];  // c * cs by rank (0 past r1)
  __shared__ __align__(16) float rul[256];  // decoder rank rulers (0 past r1)
  __shared__ float rp[kD];    // sum_a cqs[a] * dec[a][h*d + j]
  __shared__ uint32_t stream[2][kStreamWords];
  __shared__ float gsc[8];  // 4-bit mode: group scales
  const Geom& g = a.g;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int i = a.tok0 + il;  // il: the token's workspace rows
  const int HD = g.H * kD;
  const int64_t slot = a.slot_mapping[i];
  // Everything up to the decoder lookup depends only on the token index, so it is requested in
  // the same round trip as the slot id (before the PAD test below, which would otherwise wait
  // for the slot id first). The rows wave 0 (key) and wave 1 (value) pack:
  float xr0 = 0.f, xr1 = 0.f;
  if (wv == 0) {
    const int64_t kb = (int64_t)i * a.k_row_stride + h * kD;
    xr0 = load_act(a.key, a.k_dtype, kb + lane);
    xr1 = load_act(a.key, a.k_dtype, kb + 64 + lane);
  } else if (wv == 1) {
    const int64_t vb = (int64_t)i * a.v_row_stride + h * kD;
    xr0 = load_act(a.val, a.v_dtype, vb + lane);
    xr1 = load_act(a.val, a.v_dtype, vb + 64 + lane);
  }
  // the decoder slot from K3a's lookup when it ran; K3a's projection or the fit's coefficients
  const int ds_k3a = a.cq_in ? -1 : a.ws_ds[il];
  // K3a's projection: lane l loads ranks l, l + 64, l + 128, l + 192, so that every wave sees all
  // of them (the int8 ruler's max needs no barrier); thread t's own rank t is among them
  float cw[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int r = lane + 64 * k;
    cw[k] = (!a.cq_in && r < g.r1) ? a.ws_c[(int64_t)il * g.r1 + r] : 0.f;
  }
  const float cv = wv == 0 ? cw[0] : wv == 1 ? cw[1] : wv == 2 ? cw[2] : cw[3];
  float cs = a.cq_in ? a.cs_in[i] : 1.f;
  float qv = (a.cq_in && tid < g.r1) ? (float)a.cq_in[(int64_t)i * g.r1 + tid] : 0.f;
  // A negative slot id is vLLM's PAD_SLOT_ID (the padded tokens of a replayed graph): nothing
  // is written and nothing is refused, as vLLM's own cache writers skip them. Ids past the
  // cache are refused.
  if (slot < 0) return;
  const bool slot_ok = slot < a.n_slots;
  const int ds = a.cq_in ? token_decoder(a, i) : ds_k3a;
  if (h == 0 && tid == 0) {
    if (!slot_ok) atomicOr(a.err, TTKV_ERR_BAD_SLOT);
    if (ds < 0) atomicOr(a.err, TTKV_ERR_NO_DECODER);
    // the decoder registry's use flag (its eviction follows the last use, read by the host)
    if (ds >= 0 && a.dec_used) a.dec_used[ds] = 1;
  }
  if (ds < 0 || !slot_ok) return;
  // this head's decoder: wave w owns dims 32w .. 32w + 31; lane l reads column h*d + 32w + l/2,
  // ranks 64 (l & 1) .. + 63 of each 128-rank block (a lane pair reads one whole 128-byte column
  // line), requested before the coefficients are needed. The rank rulers are staged in LDS beside
  // the coefficients (thread t: rank t; r1 <= 256 threads, host-checked).
  const int R = dec_ranks(g.r1);
  const int cdim = 32 * wv + (lane >> 1);
  const int half = lane & 1;
  const int8_t* dcol = a.dec_q + ((int64_t)ds * HD + h * kD + cdim) * R + 64 * half;
  u32x4 dqv[4];
  auto load_ranks = [&](int b0) {
    if (b0 + 64 * half < R) {  // R = 64 (or 192): the second half has no ranks in the last block
#pragma unroll
      for (int c = 0; c < 4; ++c) dqv[c] = *gbl((const u32x4*)(dcol + b0 + 16 * c));
    }
  };
  load_ranks(0);
  if (!a.cq_in) {
    // Quantise the projection (every head's workgroup alike, so all agree): thread t holds rank t
    if (g.coef_mode == kCoefI8) {  // cs = max|c| * fp32(1/127), cq = clamp(rint(c / cs))
      float mx = fmaxf(fmaxf(fabsf(cw[0]), fabsf(cw[1])), fmaxf(fabsf(cw[2]), fabsf(cw[3])));
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
      cs = mx * a.inv127;
      if (cs == 0.f) cs = 1.f;
      if (tid < g.r1) qv = fminf(fmaxf(rintf(__fdiv_rn(cv, cs)), -128.f), 127.f);
    } else if (g.coef_mode == kCoefF16) {
      qv = (float)(_Float16)cv;  // round to nearest even
    } else {  // group k = ranks 32k .. 32k+31 = threads 32k .. 32k+31 (half a wave)
      float gm = fabsf(cv);
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) gm = fmaxf(gm, __shfl_xor(gm, o));
      const float sc = coef_group_scale(gm);
      if (tid < g.r1) qv = sc > 0.f ? fminf(fmaxf(rintf(__fdiv_rn(cv, sc)), -7.f), 7.f) * sc : 0.f;
      if ((tid & 31) == 0 && tid < g.r1) gsc[tid >> 5] = sc;
    }
  }
  if (tid < R) {
    rul[tid] = tid < g.r1 ? a.dec_scale[(int64_t)ds * R + tid] : 0.f;
    cqs[tid] = qv * cs;  // qv = 0 past r1
  }
  uint8_t* base = a.page + slot * a.slot_stride;
  if (h == 0) {
    if (g.coef_mode == kCoefI8) {
      if (tid < g.r1) base[tid] = (uint8_t)(int8_t)(int)qv;
      if (tid == 0) {
        const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)cs);
        base[g.coeff_bytes] = (uint8_t)(hb & 0xff);
        base[g.coeff_bytes + 1] = (uint8_t)(hb >> 8);
      }
    } else if (g.coef_mode == kCoefF16) {
      if (tid < g.r1) {  // qv is an fp16 value: the conversion is exact
        const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)qv);
        base[2 * tid] = (uint8_t)(hb & 0xff);
        base[2 * tid + 1] = (uint8_t)(hb >> 8);
      }
    }
    for (int b = g.k_field + g.H * g.k_row + tid; b < g.k_slot; b += kWThreads) base[b] = 0;
    for (int b = g.k_slot + g.H * g.v_row + tid; b < g.blob; b += kWThreads) base[b] = 0;
  }
  __syncthreads();
  if (g.coef_mode == kCoefI4G32 && h == 0 && tid < g.coef_groups) {  // the group scales (exact)
    const uint16_t hb = __builtin_bit_cast(uint16_t, (_Float16)gsc[tid]);
    base[g.coeff_bytes + 2 * tid] = (uint8_t)(hb & 0xff);
    base[g.coeff_bytes + 2 * tid + 1] = (uint8_t)(hb >> 8);
  }
  if (g.coef_mode == kCoefI4G32 && h == 0 && tid < g.coeff_bytes) {
    base[tid] = nibble_byte(tid, g.r1, [&](int r) { return cqs[r]; }, gsc);
  }
  // R[j] = K[h*d+j] - sum_a cqs[a] * dec[a][h*d+j], dec = float(q) * ruler exactly: each lane sums
  // its ranks in increasing order, then the two halves of the column are added
  float acc = 0.f;
  for (int b0 = 0; b0 < R; b0 += 128) {
    if (b0) load_ranks(b0);
    const int r0 = b0 + 64 * half;
    if (r0 < R) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int r = r0 + 16 * c + 4 * m;
          const float4v c4 = *(const float4v*)&cqs[r];
          float d[4];
          dec_values4(dqv[c][m], *(const float4v*)&rul[r], d);
#pragma unroll
          for (int k = 0; k < 4; ++k) acc = fmaf(c4[k], d[k], acc);
        }
    }
  }
  acc += __shfl_xor(acc, 1);
  if (half == 0) rp[cdim] = acc;
  __syncthreads();
  if (wv == 0) {
    const float r0 = xr0 - rp[lane];
    const float r1v = xr1 - rp[64 + lane];
    if (a.r_out) {
      a.r_out[(int64_t)i * HD + h * kD + lane] = r0;
      a.r_out[(int64_t)i * HD + h * kD + 64 + lane] = r1v;
    }
    pack_row<RB>(r0, r1v, g.res_k, a.inv_rk, base + g.k_field + h * g.k_row, stream[0]);
  } else if (wv == 1) {
    pack_row<VB>(xr0, xr1, g.v_lanes, a.inv_rv, base + g.k_slot + h * g.v_row, stream[1]);
  }
}

template <int RB, int VB>
static void launch_pack_tiles(const WriteArgs& b, int grid, hipStream_t st) {
  auto kfn = b.g.coef_mode == kCoefI8    ? pack_tiles_kernel<RB, VB, kCoefI8>
             : b.g.coef_mode == kCoefF16 ? pack_tiles_kernel<RB, VB, kCoefF16>
                                         : pack_tiles_kernel<RB, VB, kCoefI4G32>;
  hipLaunchKernelGGL(kfn, dim3(grid), dim3(kPThreads), 0, st, b);
}

template <int KDT>
static void launch_project_tiles(const WriteArgs& b, int grid, hipStream_t st) {
  const int64_t eb = KDT == TTKV_DTYPE_F32 ? 4 : 2;
  const bool vec = (uintptr_t)b.key % 16 == 0 && b.k_row_stride * eb % 16 == 0;
  auto kfn = vec ? project_tiles_kernel<KDT, true> : project_tiles_kernel<KDT, false>;
  hipLaunchKernelGGL(kfn, dim3(grid), dim3(kWThreads), 0, st, b);
}

// Fewest tokens of a launch that go in tiles: kMinTiled, and kTiledPerReq more for every further
// request (each can leave a tile partly filled, down to one token). Single tokens against tiles, graph
// replays, us: one request of 208 tokens 21.1 / 19.7, of 256 23.1 / 19.8, of 1,024 70.2 / 27.7; 2 x 97
// 21.2 / 21.1, 8 x 64 42.3 / 21.4, 64 x 4 30.0 / 26.6, 128 x 3 44.6 / 41.5, 256 x 3 83.2 / 76.7, 256 x 2
// 64.1 / 73.9; one token each of 31 requests and 200 of another 25.1 / 26.6, of 255 and 465 78.2 / 81.4.
constexpr int kMinTiled = 208, kTiledPerReq = 3;

static float inv_ruler_f32(int bits) { return (float)(1.0 / (double)((1 << (bits - 1)) - 1)); }

// Workspace: the shared 64 KiB counter region (unused here; kept so that one buffer can serve
// every entry point), then per token of a launch its projection (r1 floats) and decoder slot.
// Launches take at most kMaxCounters tokens each.
int64_t write_workspace_bytes(const Geom& g, int num_tokens) {
  const int64_t nt = std::min(std::max(num_tokens, 0), kMaxCounters);
  return kCounterBytes + nt * (g.r1 + 1) * 4;
}

int write_paged(const Geom& g, const void* key, int k_dtype, int64_t k_row_stride, const void* val,
                int v_dtype, int64_t v_row_stride, const int64_t* slot_mapping, int num_tokens,
                const int32_t* qsl, int num_reqs, const int32_t* bt, int64_t bt_row_stride,
                const int32_t* dec_map, int64_t num_blocks, const int8_t* dec_q,
                const float* dec_scale, const float* pinv_pool, int64_t n_dec_slots,
                int32_t* dec_used, const int8_t* cq_in, const float* cs_in, uint8_t* page,
                int64_t n_slots, int64_t slot_stride, float* c_out, float* r_out, void* ws,
                int64_t ws_bytes, int32_t* err, hipStream_t st) {
  if (g.d != kD) return host_fail(TTKV_E_UNSUPPORTED, "head dim must be 128");
  if (g.H > 8) return host_fail(TTKV_E_UNSUPPORTED, "H > 8 KV heads is not built");
  if (g.r1 > 256) return host_fail(TTKV_E_UNSUPPORTED, "r1 > 256 is not built");
  if (g.res_k < 1) return host_fail(TTKV_E_UNSUPPORTED, "res_k must be >= 1");
  if (!((g.res_bits == 3 && g.v_bits == 3) || (g.res_bits == 4 && g.v_bits == 4)))
    return host_fail(TTKV_E_UNSUPPORTED, "res_bits/v_bits must be 3/3 or 4/4");
  if (!key || !val || !slot_mapping || !qsl || !bt || !dec_map || !page || !err)
    return host_fail(TTKV_E_INVALID, "null pointer argument");
  if (!cq_in && !pinv_pool) return host_fail(TTKV_E_INVALID, "need pinv_pool or coeff_q_in");
  if (cq_in && !cs_in) return host_fail(TTKV_E_INVALID, "coeff_q_in needs coeff_scale_in");
  if (cq_in && g.coef_mode != kCoefI8)
    return host_fail(TTKV_E_INVALID, "coeff_q_in is int8: the fp16 and 4-bit coefficient modes "
                                     "quantise the projection themselves (pass pinv_pool)");
  if (slot_stride < g.blob) return host_fail(TTKV_E_INVALID, "slot stride smaller than the blob");
  if (k_dtype < 0 || k_dtype > 2 || v_dtype < 0 || v_dtype > 2)
    return host_fail(TTKV_E_INVALID, "dtype code");
  if (num_tokens < 0 || num_reqs < 0) return host_fail(TTKV_E_INVALID, "negative size");
  if (num_tokens == 0) return TTKV_OK;
  if (!cq_in) {
    const int64_t need = write_workspace_bytes(g, num_tokens);
    if (!ws || ws_bytes < need || (uintptr_t)ws % 256)
      return host_fail(TTKV_E_WORKSPACE, "write workspace needs " + std::to_string(need) +
                                             " bytes (256-aligned), got " +
                                             std::to_string(ws_bytes));
  }
  if (int rc = check_dec_pool(dec_q, dec_scale)) return rc;
  WriteArgs a{};
  a.g = g;
  a.key = key;
  a.k_dtype = k_dtype;
  a.k_row_stride = k_row_stride;
  a.val = val;
  a.v_dtype = v_dtype;
  a.v_row_stride = v_row_stride;
  a.slot_mapping = slot_mapping;
  a.num_tokens = num_tokens;
  a.qsl = qsl;
  a.num_reqs = num_reqs;
  a.bt = bt;
  a.bt_row_stride = bt_row_stride;
  a.dec_map = dec_map;
  a.num_blocks = num_blocks;
  a.dec_q = dec_q;
  a.dec_scale = dec_scale;
  a.pinv_pool = pinv_pool;
  a.n_dec_slots = n_dec_slots;
  a.dec_used = dec_used;
  a.cq_in = cq_in;
  a.cs_in = cs_in;
  a.page = page;
  a.n_slots = n_slots;
  a.slot_stride = slot_stride;
  a.c_out = c_out;
  a.r_out = r_out;
  a.err = err;
  a.inv127 = inv_ruler_f32(8);
  a.inv_rk = inv_ruler_f32(g.res_bits);
  a.inv_rv = inv_ruler_f32(g.v_bits);
  for (int t0 = 0; t0 < num_tokens; t0 += kMaxCounters) {
    WriteArgs b = a;
    b.tok0 = t0;
    b.num_tokens = std::min(kMaxCounters, num_tokens - t0);
    if (!cq_in) {
      b.ws_c = (float*)((char*)ws + kCounterBytes);
      b.ws_ds = (int*)(b.ws_c + (int64_t)b.num_tokens * g.r1);
    }
    b.tiles = tile_bound(b.num_tokens, num_reqs);
    const bool tiled = b.num_tokens >= kMinTiled + (int64_t)kTiledPerReq * std::max(num_reqs - 1, 0);
    const bool b3 = g.res_bits == 3;
    if (!tiled) {
      if (!cq_in)
        hipLaunchKernelGGL(write_project_kernel, dim3(b.num_tokens * project_slices(g)),
                           dim3(kWThreads), 0, st, b);
      auto kfn = b3 ? write_pack_kernel<3, 3> : write_pack_kernel<4, 4>;
      hipLaunchKernelGGL(kfn, dim3(b.num_tokens * g.H), dim3(kWThreads), 0, st, b);
      continue;
    }
    if (!cq_in) {
      const int grid = tile_blocks(b.tiles, rank_groups(g));
      if (k_dtype == TTKV_DTYPE_F32) launch_project_tiles<TTKV_DTYPE_F32>(b, grid, st);
      if (k_dtype == TTKV_DTYPE_F16) launch_project_tiles<TTKV_DTYPE_F16>(b, grid, st);
      if (k_dtype == TTKV_DTYPE_BF16) launch_project_tiles<TTKV_DTYPE_BF16>(b, grid, st);
    }
    const int grid = tile_blocks(b.tiles, g.H);
    if (b3) launch_pack_tiles<3, 3>(b, grid, st);
    if (!b3) launch_pack_tiles<4, 4>(b, grid, st);
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return host_fail(TTKV_E_LAUNCH, std::string("write launch: ") +
                                                          hipGetErrorString(e));
  return TTKV_OK;
}

}  // namespace ttkv
