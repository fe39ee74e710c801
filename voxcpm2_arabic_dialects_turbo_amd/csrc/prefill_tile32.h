// The bf16 prefill tile on 32x32x16 MFMA: one work item (query tile, sequence, kv head) of packed keys or of paged keys
// whose 64-key tiles lie inside one cache block (block_size a multiple of 64). Semantics as in prefill_attn.hip.
//
// An item is 32 RG query rows = (32 RG / G tokens) x (the G query heads of one kv head), as RG x KS waves: wave (rg, ks)
// owns rows [32 rg, 32 rg + 32) and keys [64 / KS * ks, ...) of every 64-key tile. With KS = 1 a wave sees every key;
// with KS = 2 two waves share a row block, each walking its half of every tile from one row max (the first tile's, over
// both halves), and merge (O, m, l) through LDS at the end: half the instructions, LDS reads and MFMAs per wave and key tile, which is
// what a short grid's time is made of (a chain of key tiles walked by one wave per SIMD, bound by instruction issue).
//
// Per tile and wave: S^T[keys x 32 rows] = K Q^T (Q^T in registers; lane = (row col = lane & 31, half h = lane >> 5)),
// softmax in fp32, O^T[128 d x 32 rows] += V^T P^T. A 32x32x16 MFMA does the work of two 16x16x32 with one operand read
// each, and a lane's 16 scores per 32-key block belong to one query row. P^T comes out of the score MFMA as the B operand
// of the P V MFMA: k-slot (h, e) of 16-key step s stands for key 16 s + 8 (e / 4) + 4 h + e % 4, and the transposed V
// reads (ds_read_b64_tr_b16: four keys of one column per lane) gather the same keys.
//
// K / V tiles go from global memory straight into LDS (buffer loads with the lds bit), double-buffered, the next tile's
// loads issued first thing in a tile (they are ten instructions: one descriptor each for K and V whose range ends at
// the sequence's last key, so keys past it read as zeros; one LDS base, the four pieces at immediate offsets). The
// 16-byte chunks of a 256-byte row are permuted against bank conflicts: chunk c of row R sits in slot c ^ (R & 15) of K
// (a fragment read's 16 rows hit 16 slots) and c ^ 4 (R & 3) of V (a transposed read's 4 rows x 4 chunks hit 16 slots).
#pragma once

#include <type_traits>

#include "vox_common.h"
#include "vox_kernels.h"

namespace vox {

namespace {

namespace pf32 {

constexpr int kD = 128;
constexpr int kBK = 64;         // keys per tile
constexpr int kTB = kBK * 256;  // bytes of one K or V tile in LDS
// word 3 of a raw buffer descriptor (32-bit data format; offsets in bytes, range-checked against num_records)
constexpr int kBufferWord3 = 0x00020000;

// Where an item's keys come from (one kernel instance each): packed rows; the paged cache; the paged cache with each
// sequence's new keys (positions nk - nq and later) from the step's rows (a riding KV store).
enum Source { kRows = 0, kCache = 1, kCacheNew = 2 };

typedef __attribute__((address_space(3))) void lds_void;

typedef u32x4 __attribute__((aligned(8))) u32x4_a8;  // output rows are 8-byte aligned

// The double-buffered K and V tiles: four distinct __shared__ arrays of the kernel, so the compiler can tell a tile's
// reads from the next tile's in-flight DMA writes.
struct Bufs {
  uint8_t* k0;
  uint8_t* k1;
  uint8_t* v0;
  uint8_t* v1;
  float* red;  // [2][4 waves][32] (two key halves)
};

// A sequence as an item sees it: its query rows [q0, q0 + nq), its first packed key row k0 (kRows), its keys nk, the
// position kn0 of its first new key; (paged) the block of its first tile and its block-table row, lane c holding column c.
struct Seq {
  int q0, nq, k0, nk, kn0, bid, bt_row;
};

template <int SRC, int RG, int KS>
__device__ __forceinline__ void item(const PrefillArgs& p, const int qt, const int b, const int g, const Bufs& bufs,
                                     const Seq& seq) {
  constexpr int ROWS = 32 * RG;      // query rows of the item
  constexpr int NW = RG * KS;        // waves
  constexpr int KT = 2 / KS;         // 32-key blocks per wave and tile
  constexpr int WR = kBK / NW;       // tile rows a wave loads
  constexpr int NP = WR / 4;         // its load instructions (4 rows each) for K, and for V
  static_assert(NW == 4 && (KS == 1 || KS == 2), "a wave takes 32-key blocks; the merge uses 8 KB a wave");

  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int rg = w % RG, ks = w / RG;
  const int lane = threadIdx.x & 63;
  const int col = lane & 31;
  const int h = lane >> 5;

  const int q0 = seq.q0, nq = seq.nq, k0 = seq.k0, nk = seq.nk, kn0 = seq.kn0, bid = seq.bid, bt_row = seq.bt_row;
  const int gsh = __builtin_ctz(p.group);  // the group divides 128: a power of two
  const int BQ = ROWS >> gsh;              // query tokens of the item

  // ---- this lane's query row
  const int rho = rg * 32 + col;
  const int tq = qt * BQ + (rho >> gsh);
  const int head = (g << gsh) + (rho & (p.group - 1));
  const bool row_ok = tq < nq && (p.row_limit <= 0 || (int64_t)q0 + tq < p.row_limit);
  const int qpos = nk - nq + tq;
  const int tq_last = min(nq, (qt + 1) * BQ) - 1;
  const int kv_end = p.causal ? min(nk, nk - nq + tq_last + 1) : nk;
  const int first_pos = nk - nq + qt * BQ;  // the position of the item's first query token

  // ---- tile loads: wave w fills rows [w WR, (w + 1) WR), piece i four of them; lane -> row 4 i + (lane >> 4), slot
  // lane & 15. A piece's LDS address is the wave's base plus an immediate i * 1024, which the hardware adds to the
  // memory offset too, so the lane offsets are less by it (never below zero: four rows are at least 1024 bytes).
  const int lr = lane >> 4;
  const uint32_t row_l = (uint32_t)(w * WR + lr);
  const uint32_t vsw = (uint32_t)(((lane & 15) ^ (lr << 2)) << 4);
  const uint32_t ksw = (uint32_t)(((lane & 15) ^ ((w * WR + lr) & 15)) << 4);  // ^ i << 6 for piece i
  const int rs = p.num_kv_heads * kD;  // elements between consecutive keys of the cache
  struct Place {  // a tile of the cache: its block, and its first key's place in the block
    int bid, in;
  };
  // One operand's part of a tile: the rows from `base` on, `stride` bytes apart; nrow: keys that exist from the tile's
  // first on (0: all zeros); sw: the lane's chunk of its row, ^ isw i for piece i.
  auto load_run = [&](uint8_t* d, const char* base, uint32_t stride, int nrow, uint32_t sw, auto isw) {
    const auto r = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), (short)0,
                                                     min(nrow, kBK) * (int)stride, kBufferWord3);
    lds_void* const l = (lds_void*)(d + w * (WR * 256));
    const uint32_t o = row_l * stride;
    constexpr uint32_t x = decltype(isw)::value;
#define VOX_DMA_PIECE(i)                                                                                            \
  if constexpr (NP > i)                                                                                             \
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, l, 16, o + (4 * i) * stride - 1024 * i + (sw ^ (i * x)), 0, 1024 * i, 0);
    VOX_DMA_PIECE(0)
    VOX_DMA_PIECE(1)
    VOX_DMA_PIECE(2)
    VOX_DMA_PIECE(3)
#undef VOX_DMA_PIECE
  };
  auto block_ok = [&](const Place& pl) { return pl.bid >= 0 && pl.bid < p.num_blocks; };
  // operand (K or V) of the tile at key kv0 into d
  auto load = [&](uint8_t* d, const uint16_t* src, int64_t src_stride, const uint16_t* cache, int kv0, const Place& pl,
                  uint32_t sw, auto isw) {
    if constexpr (SRC == kRows) {
      load_run(d, reinterpret_cast<const char*>(src + ((int64_t)k0 + kv0) * src_stride + g * kD),
               (uint32_t)src_stride * 2u, nk - kv0, sw, isw);
    } else {
      const bool ok = block_ok(pl);
      const uint16_t* base = cache + ((int64_t)(ok ? pl.bid : 0) * p.block_size + pl.in) * rs + g * kD;
      uint32_t stride = (uint32_t)rs * 2u;
      int nrow = ok ? nk - kv0 : 0;
      if constexpr (SRC == kCacheNew) {
        const uint16_t* const rows = src + ((int64_t)q0 + (kv0 - kn0)) * src_stride + g * kD;  // key kv0's, were it new
        if (__builtin_expect(kv0 < kn0 && kv0 + kBK > kn0 && kn0 < nk, 0)) {
          // cached and new keys: each lane's 16 bytes from the block or from the step's rows (keys past the last: the
          // last one again; they are masked). A tile of an unmapped block takes no weight: any row.
          constexpr uint32_t x = decltype(isw)::value;
          const int nold = ok ? kn0 - kv0 : 0, last = min(nk - kv0, kBK) - 1;
#pragma unroll
          for (int i = 0; i < NP; ++i) {
            const int row = min((int)row_l + 4 * i, last);
            const uint16_t* a = row < nold ? base + (int64_t)row * rs : rows + (int64_t)max(row, kn0 - kv0) * src_stride;
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)(a + ((sw ^ ((uint32_t)i * x)) >> 1)),
                (lds_void*)(d + w * (WR * 256) + i * 1024), 16, 0, 0);
          }
          return;
        }
        if (kv0 >= kn0) {
          base = rows;
          stride = (uint32_t)src_stride * 2u;
          nrow = nk - kv0;
        }
      }
      load_run(d, reinterpret_cast<const char*>(base), stride, nrow, sw, isw);
    }
  };
  auto load_k = [&](uint8_t* d, int kv0, const Place& pl) {
    load(d, p.k_src, p.k_row_stride, p.k_cache, kv0, pl, ksw, std::integral_constant<uint32_t, 64>{});
  };
  auto load_v = [&](uint8_t* d, int kv0, const Place& pl) {
    load(d, p.v_src, p.v_row_stride, p.v_cache, kv0, pl, vsw, std::integral_constant<uint32_t, 0>{});
  };
  // whether the tile at kv0 takes weight: one of an unmapped block (read as zeros) does not
  auto tile_ok = [&](int kv0, const Place& pl) {
    return SRC == kRows || (SRC == kCacheNew && kv0 >= kn0) || block_ok(pl);
  };
  int col_t = 0;
  auto next_place = [&](Place pl) -> Place {  // of the tile after it (calls in tile order)
    if constexpr (SRC != kRows) {
      pl.in += kBK;
      if (pl.in == p.block_size) {
        pl.in = 0;
        ++col_t;
        pl.bid = col_t < 64 ? __builtin_amdgcn_readlane(bt_row, col_t)
                            : p.block_tables[(int64_t)b * p.bt_stride + col_t];  // tables wider than 64 columns
      }
    }
    return pl;
  };

  // ---- per-tile steps
  const float c = p.scale_log2;
  const float rc = __builtin_amdgcn_rcpf(c);
  float m = -INFINITY, l = 0.f;
  f32x16 acc[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  // K fragment (key ks 64 / KS + kt 32 + col, chunk 2 s + h of its row) at byte kt 8192 + (krd ^ s << 5)
  const uint32_t frag = (uint32_t)(col * 256 + ((h ^ (col & 15)) << 4));
  const uint32_t krd = (uint32_t)(ks * KT * 8192) + frag;
  // transposed V read (dt, 16-key step s, half u): rows ks 64 / KS + 16 s + 8 u + 4 h + r (r = (lane & 15) >> 2), dims
  // dt 32 + 16 ((lane >> 4) & 1) + 4 (lane & 3), at byte s 4096 + u 2048 + (vrd ^ dt << 6)
  const int r4 = (lane >> 2) & 3;
  const uint32_t vrd = (uint32_t)((ks * KT * 32 + 4 * h + r4) * 256 + (r4 << 6) + (((lane >> 4) & 1) << 5) +
                                  ((lane & 3) << 3));
  u32x4 qop[8];
  auto scores = [&](const uint8_t* kd, f32x16 (&sc)[KT]) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) sc[kt][i] = 0.f;
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(kd + kt * 8192 + (krd ^ (uint32_t)(s << 5)));
        sc[kt] = mfma_32x32x16(a, qop[s], sc[kt]);
      }
  };
  // Key j is kept when j < nk and (causal) j <= qpos: one limit per lane, relative to the wave's first key. A tile of an
  // unmapped block (read as zeros) takes no weight.
  auto mask = [&](f32x16 (&sc)[KT], int kv0, bool ok) {
    if (kv0 + kBK > nk || (p.causal && kv0 + kBK - 1 > first_pos)) {
      const int last = (p.causal ? min(nk - 1, qpos) : nk - 1) - (kv0 + ks * KT * 32 + h * 4);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        // bit o: key kt 32 + o (+ 4 h) is kept (a bit extract and a bit select per score; compares and selects through
        // VCC, one after the other, took three times as long)
        const int lk = last - kt * 32;
        const uint32_t bits = lk >= 31 ? ~0u : lk < 0 ? 0u : (2u << lk) - 1u;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)bits, 8 * (i >> 2) + (i & 3), 1);
          sc[kt][i] = __uint_as_float((__float_as_uint(sc[kt][i]) & keep) | (0xff800000u & ~keep));
        }
      }
    }
    if (__builtin_expect(!ok, 0)) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sc[kt][i] = -INFINITY;
    }
  };
  // p = exp2(s c - m) of the wave's keys: the P V operand and the lane's partial row sum
  auto probs = [&](const f32x16 (&sc)[KT], u32x4 (&pb)[2 * KT]) -> float {
    const float mu = m == -INFINITY ? 0.f : m;
    float s4[4 * KT];
#pragma unroll
    for (int j = 0; j < 4 * KT; ++j) {
      float e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = fast_exp2(fmaf(sc[j >> 2][(j & 3) * 4 + i], c, -mu));
      s4[j] = (e[0] + e[1]) + (e[2] + e[3]);
      pb[j >> 1][(j & 1) * 2] = pack_bf16x2(e[0], e[1]);
      pb[j >> 1][(j & 1) * 2 + 1] = pack_bf16x2(e[2], e[3]);
    }
    float sum = (s4[0] + s4[1]) + (s4[2] + s4[3]);
    if constexpr (KT == 2) sum += (s4[4] + s4[5]) + (s4[6] + s4[7]);
    return sum;
  };
  auto row_max = [&](const f32x16 (&sc)[KT]) -> float {  // of the wave's keys, scaled (log2 units)
    float t = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) t = fmaxf(t, sc[kt][i]);
    return xhalf_max(t) * c;
  };
  // The row max is that of the first tile, and p stays <= 2^62: ahead of a tile with a score more than 62 (log2 units) past
  // it, or with a row's first key behind tiles without any, the row max moves (raise, a wave at a time). The scores are
  // looked at beside the last four P V MFMAs of the tile before, which have no softmax left to hide, and compared behind
  // its barrier. (Finding such a score by the row sum of its tile instead, with the accumulators already spoilt, and
  // walking the item a second time: 1 x 1000 tokens 30.9 us with one such key, 15.1 this way, 14.5 both with none;
  // 3 x 4096 314, 210 and 208, 210.)
  float lim = 0.f;  // the score (not scaled) from which on the row max moves
  auto raise = [&](const f32x16 (&sc)[KT]) {
    const float tm = row_max(sc);
    const bool up = tm > m + 8.f;
    const float alpha = up ? fast_exp2(m - tm) : 1.f;  // exp2(-inf) = 0 on a row's first update
    m = up ? tm : m;
    lim = (m + 62.f) * rc;
    l *= alpha;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) acc[dt] *= alpha;
  };
  // KS = 2: the first tile's row max over both of its halves, so that p and its rounding are those of an unsplit row (and
  // the int8 output's two forms quantize the same values). The barrier waits for LDS only, not for tiles in flight.
  [[maybe_unused]] auto shared_max = [&](float x) -> float {
    if (h == 0) bufs.red[w * 32 + col] = x;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    return fmaxf(x, bufs.red[(w ^ RG) * 32 + col]);
  };
  auto tile_barrier = [&]() {
    wait_vmem_all();  // this wave's part of the tiles in flight
    __syncthreads();  // ... every wave's, and the tiles read are free
  };

  // ---- the query rows, by DMA in the layout of a K tile (loaded straight into fragments, a wave's load would touch 32
  // rows for 32 bytes each), into buffers the first tiles leave free
  const int n = (kv_end + kBK - 1) / kBK;  // key tiles
  Place pl{bid, 0};                        // of the last K tile loaded
  bool ok = tile_ok(0, pl);                // whether the tile whose scores are held takes weight
  // The loop takes two tiles a round (fixed buffers: the compiler tells a tile's reads from the tiles in flight by the
  // arrays), with one tile before it where that leaves one: tile 0 then starts in the second buffers.
  const bool odd = n > 0 && (n - 1) % 2 != 0;
  uint8_t* const kfirst = odd ? bufs.k1 : bufs.k0;
  uint8_t* const ksecond = odd ? bufs.k0 : bufs.k1;
  uint8_t* const vfirst = odd ? bufs.v1 : bufs.v0;
  uint8_t* const vsecond = odd ? bufs.v0 : bufs.v1;
  f32x16 sa[KT], sb[KT];
  uint16_t* op = p.out + ((int64_t)q0 + tq) * p.out_row_stride + head * kD + h * 8;  // this lane's output row
  if (n > 0) {
    uint8_t* const qbuf = KS == 2 ? vsecond + rg * 8192 : (rg < 2 ? ksecond + rg * 8192 : vsecond + (rg - 2) * 8192);
    constexpr int NQ = 8 / KS;  // pieces (4 rows) this wave loads of its row block
    // (rows past the sequence or the limit read as zeros; their output is not stored)
    const int64_t tok0 = (int64_t)q0 + (int64_t)qt * BQ;
    int ntok = min(nq - qt * BQ, BQ);
    if (p.row_limit > 0) ntok = (int)max((int64_t)0, min((int64_t)ntok, p.row_limit - tok0));
    ntok = __builtin_amdgcn_readfirstlane(ntok);  // (clamped in a vector register)
    const uint16_t* const qb = p.q + tok0 * p.q_row_stride + (g << gsh) * kD;
    if (__builtin_expect(p.q_row_stride < (1 << 23), 1)) {
      const uint32_t sq = (uint32_t)p.q_row_stride * 2u;
      const auto rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(qb), (short)0, (uint32_t)ntok * sq,
                                                        kBufferWord3);
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int row = (ks * NQ + i) * 4 + lr;  // of the row block
        const int r = rg * 32 + row;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rq, (lds_void*)(qbuf + (ks * NQ + i) * 1024), 16,
            (uint32_t)(r >> gsh) * sq + (uint32_t)((r & (p.group - 1)) << 8) + (uint32_t)(((lane & 15) ^ (row & 15)) << 4), 0,
            0, 0);
      }
    } else {  // row strides past a descriptor's 32-bit offsets: per-lane addresses (the last valid row for those past it)
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        const int row = (ks * NQ + i) * 4 + lr;
        const int r = rg * 32 + row;
        const uint16_t* src = qb + (int64_t)max(min(r >> gsh, ntok - 1), 0) * p.q_row_stride +
                              (r & (p.group - 1)) * kD + (((lane & 15) ^ (row & 15)) << 3);
        if (ntok > 0)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                           (lds_void*)(qbuf + (ks * NQ + i) * 1024), 16, 0, 0);
      }
    }
    load_k(kfirst, 0, pl);
    load_v(vfirst, 0, pl);
    if (KS == 2 && n > 1) {
      pl = next_place(pl);
      load_k(ksecond, kBK, pl);
    }
    // the output address, computed while they arrive (not at the end of the item, where nothing else is left to run)
    asm volatile("" : "+v"(op));
    tile_barrier();
#pragma unroll
    for (int s = 0; s < 8; ++s) qop[s] = *reinterpret_cast<const u32x4*>(qbuf + (frag ^ (uint32_t)(s << 5)));
    if (KS == 1 && n > 1) {
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // every wave has its query rows
      pl = next_place(pl);
      load_k(ksecond, kBK, pl);
    }
    scores(kfirst, sa);
    mask(sa, 0, ok);
    m = row_max(sa);
    if constexpr (KS == 2) m = shared_max(m);
    if (n > 1) {  // (an item of one tile has no next one to wait for: 12 layers of 250 x 16 rows 150.7 -> 148.5 us)
      lim = (m + 62.f) * rc;
      if constexpr (KS == 1) tile_barrier();
    }
  }
  // One tile: the softmax of its scores (sc) beside the score MFMAs of the next tile (into sn) and its own first P V
  // MFMAs; the next V tile and the K tile after it are loaded meanwhile. In this order, pinned: an MFMA runs 32 cycles and
  // leaves the wave's issue slots free for about 1.3 elements' fma, exp, add and half a cvt, and for the LDS reads of
  // later MFMAs (a microbenchmark of one wave: 33 cycles per MFMA with that much softmax beside it, 32 without). With
  // two waves on a SIMD the issue slots are what is short: over 16 x 2048 tokens each wave issues in 41 % of its cycles
  // (the SIMD in 82 %), is ready behind the other in 36 % and waits in 23 %, 5 % for an LDS instruction's turn; the matrix
  // cores are busy 53 % of the time, at a clock of 1.7 GHz, with 5.2 VALU and 1.5 LDS instructions to an MFMA. Left to
  // itself the compiler runs the MFMAs together and the softmax together, and the two waves of a SIMD do not interleave
  // the two by themselves.
  auto step = [&](int t, const f32x16 (&sc)[KT], f32x16 (&sn)[KT], const uint8_t* kn, uint8_t* kfree, const uint8_t* vc,
                  uint8_t* vfree) {
    constexpr int NS = 8 * KT, NP2 = 8 * KT;        // score and P V MFMAs
    constexpr int SPAN = NS + (2 * KT - 1) * 4;     // MFMAs the softmax is spread over: the last P V step needs all of it
    constexpr int NE = 16 * KT;                     // elements per lane
    const float mu = m == -INFINITY ? 0.f : m;
    u32x4 pb[2 * KT];
    float e[4], sum = 0.f, top = -INFINITY;
    auto element = [&](int x) {  // element x (key block x / 16, register x % 16) of the tile's probabilities
      e[x & 3] = fast_exp2(fmaf(sc[x >> 4][x & 15], c, -mu));
      if (x & 1) pb[x >> 3][(x >> 1) & 3] = pack_bf16x2(e[(x & 3) - 1], e[x & 3]);
      if ((x & 3) == 3) {
        sum += (e[0] + e[1]) + (e[2] + e[3]);
        asm volatile("" : "+v"(sum));  // (here: sunk to the end of the tile, the adds would keep every e alive)
      }
    };
    constexpr int AH = KT == 1 ? 8 : 4;  // MFMAs whose operands are read ahead
    u32x4 kf[AH], vf[AH];
    auto read_k = [&](int i) {  // operand of score MFMA i (k-step i / KT, key block i % KT)
      kf[i % AH] = *reinterpret_cast<const u32x4*>(kn + (i % KT) * 8192 + (krd ^ (uint32_t)((i / KT) << 5)));
    };
    auto read_v = [&](int i) {  // operand of P V MFMA i (16-key step i / 4, dims block i % 4)
      const uint8_t* vp = vc + (i >> 2) * 4096 + (vrd ^ (uint32_t)((i & 3) << 6));
      const u32x2 lo = __builtin_bit_cast(u32x2, lds_read_tr16(reinterpret_cast<const uint16_t*>(vp)));
      const u32x2 hi = __builtin_bit_cast(u32x2, lds_read_tr16(reinterpret_cast<const uint16_t*>(vp + 2048)));
      vf[i % AH] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) sn[kt][i] = 0.f;
#pragma unroll
    for (int i = 0; i < AH; ++i) read_k(i);
    __builtin_amdgcn_sched_barrier(0);
    // the tile loads, while the first operands arrive
    load_v(vfree, (t + 1) * kBK, pl);
    ok = tile_ok((t + 1) * kBK, pl);
    if (t + 2 < n) {
      pl = next_place(pl);
      load_k(kfree, (t + 2) * kBK, pl);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NS + NP2; ++i) {
      if (i < NS)
        sn[i % KT] = mfma_32x32x16(kf[i % AH], qop[i / KT], sn[i % KT]);
      else
        acc[(i - NS) & 3] = mfma_32x32x16(vf[(i - NS) % AH], pb[(i - NS) >> 2], acc[(i - NS) & 3]);
      // later operands, two behind every second MFMA: half the waits (the tile is bound by issue; 1 x 1000 tokens 14.5 ->
      // 14.3 us, 3 x 4096 208.9 -> 208.3 against one behind each; four behind every fourth 14.6 and 211)
#pragma unroll
      for (int j = i - 1; (i & 1) && j <= i; ++j) {
        if (j + AH < NS)
          read_k(j + AH);
        else if (j + AH < NS + NP2)
          read_v(j + AH - NS);
      }
#pragma unroll
      for (int x = i * NE / SPAN; x < (i + 1) * NE / SPAN && x < NE; ++x) element(x);
      if (i >= NS + NP2 - 4) {  // this lane's largest score of the next tile (masked ones too)
        constexpr int N4 = NE / 4;
#pragma unroll
        for (int x = 0; x < N4; ++x) {
          const int y = (i - (NS + NP2 - 4)) * N4 + x;
          top = fmaxf(top, sn[y >> 4][y & 15]);
        }
        asm volatile("" : "+v"(top));  // (here)
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l += sum;
    mask(sn, (t + 1) * kBK, ok);
    tile_barrier();
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(top > lim) != 0, 0)) raise(sn);
  };
  if (n > 0) {
    int t = 0;
    if (odd) {
      step(0, sa, sb, bufs.k0, bufs.k1, bufs.v1, bufs.v0);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) sa[kt] = sb[kt];
      t = 1;
    }
    for (; t + 1 < n; t += 2) {
      step(t, sa, sb, bufs.k1, bufs.k0, bufs.v0, bufs.v1);
      step(t + 1, sb, sa, bufs.k0, bufs.k1, bufs.v1, bufs.v0);
    }
    // the last tile: its first V operands read while its softmax starts
    u32x4 pb[2 * KT], vf[8];
    auto read_v = [&](int i) {
      const uint8_t* vp = bufs.v0 + (i >> 2) * 4096 + (vrd ^ (uint32_t)((i & 3) << 6));
      const u32x2 lo = __builtin_bit_cast(u32x2, lds_read_tr16(reinterpret_cast<const uint16_t*>(vp)));
      const u32x2 hi = __builtin_bit_cast(u32x2, lds_read_tr16(reinterpret_cast<const uint16_t*>(vp + 2048)));
      vf[i & 7] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
#pragma unroll
    for (int i = 0; i < 8; ++i) read_v(i);
    l += probs(sa, pb);
#pragma unroll
    for (int i = 0; i < 8 * KT; ++i) {
      acc[i & 3] = mfma_32x32x16(vf[i & 7], pb[i >> 2], acc[i & 3]);
      if (i + 8 < 8 * KT) read_v(i + 8);
    }
  }
  // ---- epilogue: normalize, bf16
  const float L = xhalf_sum(l);
  // the 32-dim blocks [d0, d0 + nd) of O, normalized by inv
  auto store = [&](auto d0, auto nd, float inv) {
    constexpr int D0 = decltype(d0)::value, ND = decltype(nd)::value;
    u32x4 o[ND][2];
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int gp = 0; gp < 2; ++gp) {
        // lane half h holds dims 8 a + 4 h + [0, 4) of each 8-dim group a: the halves trade, so that half h stores the
        // 8 dims of group 2 gp + h
        uint32_t x[2], y[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          x[i] = pack_bf16x2(acc[D0 + dt][gp * 8 + 2 * i] * inv, acc[D0 + dt][gp * 8 + 2 * i + 1] * inv);
          y[i] = pack_bf16x2(acc[D0 + dt][gp * 8 + 4 + 2 * i] * inv, acc[D0 + dt][gp * 8 + 4 + 2 * i + 1] * inv);
        }
        const auto s0 = __builtin_amdgcn_permlane32_swap(x[0], y[0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(x[1], y[1], false, false);
        o[dt][gp] = u32x4{s0[0], s1[0], s0[1], s1[1]};
      }
    if (row_ok) {
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) *reinterpret_cast<u32x4_a8*>(op + (D0 + dt) * 32 + gp * 16) = o[dt][gp];
    }
  };
  using std::integral_constant;
  if constexpr (KS == 1) {
    store(integral_constant<int, 0>{}, integral_constant<int, 4>{}, L > 0.f ? 1.f / L : 0.f);
  } else {
    // the two waves of a row block hand each other half of their O: wave ks keeps dims [64 ks, 64 ks + 64)
    uint8_t* const mine = w < 2 ? bufs.k0 + w * 8192 : bufs.k1 + (w - 2) * 8192;
    const int pw = w ^ RG;  // the partner
    const uint8_t* const theirs = pw < 2 ? bufs.k0 + pw * 8192 : bufs.k1 + (pw - 2) * 8192;
    // (their p were taken against the same row max, and the parts add up, unless one of the waves has raised its own)
    __syncthreads();  // the last tile's reads are done
    auto merge = [&](auto half) {
      constexpr int OWN = 2 * decltype(half)::value, GIVE = 2 - OWN;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        *reinterpret_cast<f32x4*>(mine + j * 1024 + lane * 16) =
            f32x4{acc[GIVE + (j >> 2)][(j & 3) * 4], acc[GIVE + (j >> 2)][(j & 3) * 4 + 1],
                  acc[GIVE + (j >> 2)][(j & 3) * 4 + 2], acc[GIVE + (j >> 2)][(j & 3) * 4 + 3]};
      if (h == 0) {
        bufs.red[w * 32 + col] = L;
        bufs.red[128 + w * 32 + col] = m;
      }
      __syncthreads();
      float Lt = bufs.red[pw * 32 + col];
      const float mt = bufs.red[128 + pw * 32 + col];
      f32x4 y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = *reinterpret_cast<const f32x4*>(theirs + j * 1024 + lane * 16);
      float Ls = L;
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(m != mt) != 0, 0)) {
        const float M = fmaxf(m, mt);
        const float a = m == M ? 1.f : fast_exp2(m - M), at = mt == M ? 1.f : fast_exp2(mt - M);
        Ls *= a;
        Lt *= at;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          y[j] *= at;
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[OWN + (j >> 2)][(j & 3) * 4 + i] *= a;
        }
      }
      Ls += Lt;
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[OWN + (j >> 2)][(j & 3) * 4 + i] += y[j][i];
      store(integral_constant<int, OWN>{}, integral_constant<int, 2>{}, Ls > 0.f ? 1.f / Ls : 0.f);
    };
    if (ks == 0)
      merge(integral_constant<int, 0>{});
    else
      merge(integral_constant<int, 1>{});
  }
}

template <int SRC, int RG, int KS>
__device__ __forceinline__ void tile(const PrefillArgs& p, const int qt, const int b, const int g, const Bufs& bufs) {
  constexpr int ROWS = 32 * RG;
  const int lane = threadIdx.x & 63;

  // every argument in one batch of scalar loads (left to itself the compiler loads each where it is first used, a round
  // trip apiece on the way to the first tile loads: 2400 cycles from the bounds to the loads, 1000 this way)
  asm volatile("" ::"s"(p.q), "s"(p.q_row_stride), "s"(p.out), "s"(p.out_row_stride), "s"(p.cu_q), "s"(p.cu_k),
               "s"(p.group), "s"(p.causal), "s"(p.scale_log2), "s"(p.row_limit), "s"(p.skip_single));
  if constexpr (SRC != kCache)
    asm volatile("" ::"s"(p.k_src), "s"(p.v_src), "s"(p.k_row_stride), "s"(p.v_row_stride), "s"(p.num_kv_heads));
  if constexpr (SRC != kRows)
    asm volatile("" ::"s"(p.block_tables), "s"(p.bt_stride), "s"(p.max_blocks), "s"(p.block_size), "s"(p.num_blocks),
                 "s"(p.k_cache), "s"(p.v_cache), "s"(p.num_kv_heads));

  // ---- the sequence's bounds, and (paged) its block-table row beside them: lane c holds column c (c < 64), so the loop
  // takes each tile's block id with v_readlane; column 0 by a scalar load, for the first tile's DMA
  int q0 = b * p.uniform_q, q1 = q0 + p.uniform_q, k0 = b * p.uniform_k, k1 = k0 + p.uniform_k;
  if (p.cu_q) {
    q0 = p.cu_q[b];
    q1 = p.cu_q[b + 1];
    k0 = p.cu_k[b];
    k1 = p.cu_k[b + 1];
  }
  int bid = 0, bt_row = -1;
  if constexpr (SRC != kRows) {
    bid = p.block_tables[(int64_t)b * p.bt_stride];
    if (lane < p.max_blocks) bt_row = p.block_tables[(int64_t)b * p.bt_stride + lane];
  }
  const int nq = q1 - q0;
  const int kn0 = k1 - k0 - nq;  // position of the first new key
  const int nk = SRC == kRows ? k1 - k0 : min(k1 - k0, p.max_blocks * p.block_size);  // keys the table can address
  if (qt * (ROWS >> __builtin_ctz(p.group)) >= nq || (p.skip_single && nq == 1)) return;  // (one-query rows: the decode kernel's, in varlen mode)
  if (SRC != kCache && g >= p.num_kv_heads) return;         // a workgroup that only copies (a riding store)
  if constexpr (SRC == kCacheNew) {
    // A sequence without cached keys: a loop of its own that reads only the rows, with neither block ids nor a choice of
    // source a tile. A layer of a step of 1 x 237 tokens 8.7 -> 7.6 us, 1 x 1500 31.7 -> 23.7, 5 x 1000 44.1 -> 38.2,
    // 2 x 4000 171 -> 146.
    if (kn0 == 0) {
      item<kRows, RG, KS>(p, qt, b, g, bufs, Seq{q0, nq, q0, nk, 0, 0, -1});
      return;
    }
  }
  item<SRC, RG, KS>(p, qt, b, g, bufs, Seq{q0, nq, k0, nk, kn0, bid, bt_row});
}

}  // namespace pf32

}  // namespace

}  // namespace vox
