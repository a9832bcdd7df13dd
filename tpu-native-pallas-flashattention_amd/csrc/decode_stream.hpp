// Streaming single-query decode (gfx950): head_dim 64 and 128 for every dtype,
// 256 for bf16/f16.
//
// Replaces the decode launch of `flash_attention_decode`
// (flash_attention.py:555-589: the forward pallas_call with block_q = 1,
// kv_len = cache_len) and the `paged_flash_attention` pallas_call
// (paged.py:151-192, kernel :45-99). Other head dims, page sizes that are not
// a multiple of 4 (8 for 128-byte rows) and, off the 16-bit head_dim 128
// path, GQA groups of more than 16 heads use the generic kernel in decode.hip.
//
// The path is HBM-bound (about 4 FLOP per byte); the design keeps every CU's
// share of bytes in flight at all times with fully coalesced loads:
//  * Work list. A "sequence" is one (batch b, kv head, 16-head slice of the
//    GQA group); its keys [0, len_b) split into stages of SK keys (32; 16
//    for 512-byte rows). All sequences' stages, in order, form one global
//    list of S stages. The grid is persistent (as many one-wave workgroups as
//    fit on the chip) and wave w takes the contiguous range
//    [start(w), start(w + 1)) of that list, an equal share to within one
//    stage whatever the (paged) lengths are.
//  * All query heads of a group ride as the N columns of 16-column MFMAs, so
//    each K/V byte is read from HBM once (the reference grid runs per query
//    head and re-streams each KV head g times).
//  * K/V rows stream through a wave-private ring of NS LDS stages (8 KB of K
//    + 8 KB of V, half that for 128-byte rows, + the sequence's query rows).
//    The ring runs across sequence boundaries, so a wave never drains its
//    pipeline until its range ends. A stage is direct global->LDS loads
//    (buffer_load_dwordx4 ... lds) that each move whole rows, 1 KB contiguous
//    in HBM. They are issued from inline assembly, so the compiler does not
//    insert its conservative "wait for every LDS DMA" before each LDS read;
//    explicit vmcnt waits leave the NS - 2 younger stages in flight while a
//    stage is consumed. Whatever the row length, a CU holds about 64 KB in
//    flight: 4 resident waves of 16 KB stages, 8 of 8 KB ones. Measured
//    against the generic kernel, which runs these forms at one wave per key
//    chunk without a pipeline: bf16 head_dim 256, B=16 Hkv=8, 5003 keys
//    (656 MB): 200 us -> 101 us (3.3 -> 6.5 TB/s); float32 head_dim 64 paged,
//    page 16, B=16 Hkv=4, 64-2048 keys (35 MB): 66 us -> 14 us.
//  * Paged pool: each group of PG rows lies inside one page (page_size a
//    multiple of PG), so its page is a wave-uniform scalar load of the block
//    table and its buffer resource spans exactly that page's valid rows.
//  * Rows at or past the valid length lie outside the load's buffer range
//    and arrive as zeros (hardware bounds check): a NaN tail, -1 table
//    padding (never looked up: lookups stop below ceil(len / page_size)) and
//    unused pages cannot leak (flash_attention.py:95-100; paged.py:73-80, :93).
//  * A sequence whose stages all fall in one wave is finished by that wave
//    (o = acc / l, l == 0 -> 0; flash_attention.py:150-159, paged.py:95-99).
//    A sequence cut by wave boundaries leaves one partial (max, sum, acc)
//    per piece (slot piece_slot); pf_decode_stream_cut_kernel or
//    pf_decode_stream_combine_kernel merges them (launch_combine).
//
// LDS stage layout: row-major SK x RB-byte tiles with the 16-byte chunks of
// row r permuted by chunk ^ swz(r) (StreamGeo). Both read patterns are
// conflict-free:
//  * K as the A operand of S^T = K Q^T: the 16 lanes of a group read one
//    chunk index from 16 rows (row bits {0, 1, 3, 4} vary with 32-key stages,
//    {0, 1, 2, 3} with 16-key ones);
//  * 16-bit V^T through ds_read_b64_tr_b16: a 16-lane group reads 2 chunks of
//    4 consecutive rows (row bits {0, 1} vary). float32 V: a 16-lane group
//    reads one row, 16 bytes a lane; the four floats feed four MFMAs whose
//    output rows are the columns 4i + e.
#pragma once

#include "pf_common.hpp"
#include "pf_kernels.hpp"

#include <algorithm>
#include <mutex>

namespace pf {
namespace stream {

// Geometry of a stage for rows of D elements of T. FINE: 16-key stages for
// 256-byte rows too (DecodeParams::fine).
template <typename T, int D, bool FINE = false>
struct StreamGeo {
  static constexpr bool F32 = sizeof(T) == 4;
  static constexpr int RB = D * (int)sizeof(T);    // row bytes: 128, 256 or 512
  static constexpr int CPR = RB / 16;              // 16-byte chunks per row
  static constexpr int SK = RB == 512 || FINE ? 16 : 32;  // keys per stage
  static constexpr int KPL = SK / 4;               // keys per lane (of its head)
  static constexpr int NU = SK / 16;               // 16-key tiles per stage
  static constexpr int TILE = SK * RB;             // one stage of K (or V)
  static constexpr int NL = TILE / 1024;           // 64-lane loads per tile
  static constexpr int RPL = 1024 / RB;            // rows per load
  static constexpr int NACC = D / 16;              // O^T accumulators
  static_assert(RB == 128 || RB == 256 || RB == 512, "row sizes of the streaming kernel");
  // Query rows in LDS: at least one whole load (rows past the group are zeros).
  static constexpr int qrows(int qr) { return qr > RPL ? qr : RPL; }
  static constexpr int slot_bytes(int qr) { return 2 * TILE + qrows(qr) * RB; }
  // Chunk permutation of row r (XOR of the low bits of the chunk index). With
  // 128-byte rows two rows share a 256-byte bank window, so row bit 0 already
  // separates them and three bits are left.
  __host__ __device__ static constexpr int swz(int r) {
    if (RB == 128) return (((r >> 1) & 1) << 1) | ((r >> 3) & 1) | (((r >> 4) & 1) << 2);
    if (SK == 16) return ((r >> 2) & 1) | ((r & 3) << 1) | (((r >> 3) & 1) << 3);
    return ((r >> 3) & 1) | ((r & 3) << 1) | (((r >> 4) & 1) << 3);
  }
  static constexpr int QMASK = (CPR < 16 ? CPR : 16) - 1;  // query row permutation
};
// K/V stages are loaded non-temporal: each cache or pool byte is read once
// per call, and a read-once stream reaches a higher HBM rate that way
// (bench.py's read-form probe).
constexpr bool kKvNt = true;

typedef short i16x4 __attribute__((ext_vector_type(4)));

// Wait for the oldest issued stage; `younger` later stages (at least LPS
// loads each, loads complete in issue order) may stay in flight.
template <int NS, int LPS>
__device__ inline void wait_stage(int64_t younger) {
  if constexpr (NS >= 4) {
    if (younger >= 2) { wait_vm<2 * LPS>(); return; }
  }
  if constexpr (NS >= 3) {
    if (younger >= 1) { wait_vm<LPS>(); return; }
  }
  wait_vm<0>();
}

__device__ inline int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ inline int64_t uni64(int64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)x >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Scalar (wave-uniform) 32-bit load through the constant address space; the
// index is made provably uniform so the compiler emits s_load (the scalar
// counter), not a vector load whose wait would drain the LDS DMA queue.
__device__ inline int sload_i32(const int32_t* p, int64_t idx) {
  const __attribute__((address_space(4))) int32_t* cp = (const __attribute__((address_space(4))) int32_t*)p;
  return uni(cp[uni64(idx)]);
}

// 16x16 MFMAs with float32 accumulation; lane l holds A[l%16][k slots of
// l/16], B[k slots of l/16][l%16] and C[4(l/16) + r][l%16]. run: S^T over one
// 16-byte chunk of K and Q per lane (16-bit: one instruction over 32 columns;
// float32: four over 4 columns each).
template <typename T>
struct Mfma16;
template <>
struct Mfma16<bf16_t> {
  typedef bf16x8 Frag;
  __device__ static inline f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(Frag, a), __builtin_bit_cast(Frag, b), c, 0, 0,
                                                   0);
  }
  __device__ static inline f32x4 run16(u32x2 a, u32x2 b, f32x4 c) {
    typedef short v4i16 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(v4i16, a), __builtin_bit_cast(v4i16, b), c, 0,
                                                     0, 0);
  }
};
template <>
struct Mfma16<f16_t> {
  typedef f16x8 Frag;
  __device__ static inline f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(Frag, a), __builtin_bit_cast(Frag, b), c, 0, 0,
                                                  0);
  }
  __device__ static inline f32x4 run16(u32x2 a, u32x2 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(__builtin_bit_cast(f16x4, a), __builtin_bit_cast(f16x4, b), c, 0, 0,
                                                 0);
  }
};
template <>
struct Mfma16<float> {
  __device__ static inline f32x4 step(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static inline f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = step(x[e], y[e], c);
    return c;
  }
};

// Live keys of a decode step whose new token is at `pos` (0 for an invalid
// position: it attends nothing and writes nothing): linear cache pos + 1,
// ring min(pos + 1, cache_size) (model.py:475-476).
__device__ inline int step_len(const DecodeParams& p, int pos) {
  const bool valid = pos >= 0 && (p.ring != 0 || pos < p.cache_size) &&
                     (p.rope_cos == nullptr || pos < p.rope_len);
  if (!valid) return 0;
  return p.ring != 0 ? min(pos + 1, p.cache_size) : pos + 1;
}

// Valid keys of batch b: PG == 0 the one cache_len; PG == 1 (decode step)
// from b's position; paged: b's context length clamped to the table's reach.
// len_lane reads per lane (b may differ across lanes), seq_len with scalar
// loads (b wave-uniform).
template <int PG>
__device__ inline int len_lane(const DecodeParams& p, int b) {
  if constexpr (PG == 0) {
    return p.cache_len;
  } else if constexpr (PG == 1) {
    return step_len(p, p.positions[(int64_t)b * p.pos_stride]);
  } else {
    return min(max(p.context_lens[b], 0), p.pages_per_seq * p.page_size);
  }
}
template <int PG>
__device__ inline int seq_len(const DecodeParams& p, int b) {
  if constexpr (PG == 0) {
    return p.cache_len;
  } else if constexpr (PG == 1) {
    return step_len(p, sload_i32(p.positions, (int64_t)b * p.pos_stride));
  } else {
    return min(max(sload_i32(p.context_lens, b), 0), p.pages_per_seq * p.page_size);
  }
}

// a / b and a % b of a non-negative a: 32-bit division when a fits (it nearly
// always does; a 64-bit division is several hundred instructions).
__device__ inline int64_t div_pos(int64_t a, int b, int64_t* rem) {
  if (((uint64_t)a >> 32) == 0) {
    const uint32_t q = (uint32_t)a / (uint32_t)b;
    *rem = (uint32_t)a - q * (uint32_t)b;
    return q;
  }
  const int64_t q = a / b;
  *rem = a - q * b;
  return q;
}

// Balanced partition of the S-stage list over W waves: wave w takes
// [start(w), start(w + 1)).
struct Partition {
  int64_t q, rem;
  __device__ inline Partition(int64_t S, int W) { q = div_pos(S, W, &rem); }
  __device__ inline Partition(int64_t q_, int64_t rem_) : q(q_), rem(rem_) {}
  __device__ inline int64_t start(int w) const { return (int64_t)w * q + min((int64_t)w, rem); }
  __device__ inline int wave_of(int64_t s) const {
    int64_t r;
    const int64_t big = rem * (q + 1);
    if (s < big) return (int)div_pos(s, (int)(q + 1), &r);
    return (int)(rem + div_pos(s - big, (int)q, &r));
  }
};

// Workspace slot of the piece of sequence `seq` (= b * J + j) that wave w
// leaves; `late`: the sequence starts inside the wave's range. From one piece
// to the next along the stage list w or seq moves on, so w + seq names every
// piece once (W + B J slots). Many sequences: only the piece that opens a
// wave's range and the one that closes it can be partial (2 W slots).
__device__ inline int64_t piece_slot(const DecodeParams& p, int J, int w, int64_t seq, bool late) {
  return (int64_t)p.B * J <= p.n_waves ? w + seq : 2 * (int64_t)w + (late ? 1 : 0);
}

// Position in the stage list: batch b, sequence j = kv_head * n_hc + slice
// within the batch, stage st of nst = ceil(L / SK).
struct Cursor {
  int b, j, st, nst, L;
};

template <int PG, int SK>
__device__ inline void cursor_next(Cursor& c, const DecodeParams& p, int J) {
  if (++c.st < c.nst) return;
  c.st = 0;
  if (++c.j < J) return;
  c.j = 0;
  do {
    ++c.b;
    c.L = (c.b < p.B) ? seq_len<PG>(p, c.b) : 0;
  } while (c.b < p.B && c.L == 0);
  c.nst = (c.L + SK - 1) / SK;
}

__device__ inline int64_t readlane64(int64_t x, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)x >> 32), lane);
  return (int64_t)(((uint64_t)hi << 32) | lo);
}
// Inclusive scan over the 64 lanes.
__device__ inline int64_t scan64(int64_t x) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int64_t y = __shfl_up(x, o);
    if (lane >= o) x += y;
  }
  return x;
}

// The stage counts T_b = ceil(L_b / SK) * J of all batches, summed: lane l holds
// those of its `per` batches [l per, (l + 1) per), so one pass of independent
// loads, one scan and, past 64 batches, one look into one lane's share find
// any stage's batch. The lanes' loads lie in 64 cache lines, so a paged call
// takes 4 lengths with each. (64 batches after another, a scan each and once
// more for the total, took 30 us of every wave at 4096 batches.)
struct BatchScan {
  int per;       // batches per lane: 1, or a multiple of 4
  int L;         // per == 1: this lane's batch length (0 past B)
  int64_t t;     // stages of this lane's batches
  int64_t incl;  // stages up to and with them
  int64_t tot;   // S, the total
};
template <int PG, int SK>
__device__ inline BatchScan batch_scan(const DecodeParams& p, int J) {
  const int lane = threadIdx.x & 63;
  BatchScan r;
  r.per = 1;
  if (p.B <= 64) {
    r.L = lane < p.B ? len_lane<PG>(p, lane) : 0;
    r.t = (r.L + SK - 1) / SK;
  } else {
    typedef int i32x4u __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int NB = 16;  // lengths in flight
    r.per = (((p.B + 63) >> 6) + 3) & ~3;
    r.L = 0;
    r.t = 0;
    const int b0 = lane * r.per, b1 = min(b0 + r.per, p.B);
    int b = b0;
    for (; b + NB <= b1; b += NB) {
      int L[NB];
      if constexpr (PG > 1) {
#pragma unroll
        for (int u = 0; u < NB / 4; ++u) {
          const i32x4u x = *reinterpret_cast<const i32x4u*>(p.context_lens + b + 4 * u);
#pragma unroll
          for (int e = 0; e < 4; ++e) L[4 * u + e] = min(max(x[e], 0), p.pages_per_seq * p.page_size);
        }
      } else {
#pragma unroll
        for (int u = 0; u < NB; ++u) L[u] = len_lane<PG>(p, b + u);
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) r.t += (L[u] + SK - 1) / SK;
    }
    int L[NB];  // the share's rest
#pragma unroll
    for (int u = 0; u < NB; ++u) L[u] = b + u < b1 ? len_lane<PG>(p, b + u) : 0;
#pragma unroll
    for (int u = 0; u < NB; ++u) r.t += (L[u] + SK - 1) / SK;
  }
  r.t *= J;
  r.incl = scan64(r.t);
  r.tot = readlane64(r.incl, 63);
  return r;
}

// The cursor of stage s < S of the list.
template <int PG, int SK>
__device__ inline Cursor locate(const DecodeParams& p, int J, int64_t s, const BatchScan& sc) {
  const int lane = threadIdx.x & 63;
  const int ln = __builtin_ctzll(__ballot(sc.incl > s));
  int64_t before = readlane64(sc.incl - sc.t, ln);
  int b = ln, L = __builtin_amdgcn_readlane(sc.L, ln);
  if (sc.per > 1) {
    for (int i = 0; i < sc.per; i += 64) {
      const int bb = ln * sc.per + i + lane;
      const int Lb = i + lane < sc.per && bb < p.B ? len_lane<PG>(p, bb) : 0;
      const int64_t t = (int64_t)((Lb + SK - 1) / SK) * J, incl = scan64(t);
      const uint64_t hit = __ballot(before + incl > s);
      if (hit != 0) {
        const int in = __builtin_ctzll(hit);
        before += readlane64(incl - t, in);
        L = __builtin_amdgcn_readlane(Lb, in);
        b = ln * sc.per + i + in;
        break;
      }
      before += readlane64(incl, 63);
    }
  }
  const int nst = (L + SK - 1) / SK;
  int64_t st;
  const int j = (int)div_pos(uni64(s - before), nst, &st);
  return Cursor{uni(b), uni(j), uni((int)st), uni(nst), uni(L)};
}

// The stages of batches before b (wave-uniform).
template <int PG, int SK>
__device__ inline int64_t stages_before(const DecodeParams& p, int J, int b, const BatchScan& sc) {
  const int lane = threadIdx.x & 63;
  const int ln = sc.per == 1 ? b : (int)((uint32_t)b / (uint32_t)sc.per);
  int64_t before = readlane64(sc.incl - sc.t, ln);
  if (sc.per > 1) {
    int64_t t = 0;  // of this lane's share of lane ln's batches below b
    for (int bb = ln * sc.per + lane; bb < b; bb += 64) t += (len_lane<PG>(p, bb) + SK - 1) / SK;
    before += readlane64(scan64(t * J), 63);
  }
  return before;
}

// The same with one length for all batches: arithmetic.
template <int SK>
__device__ inline Cursor locate_uniform(const DecodeParams& p, int J, int64_t s) {
  const int nst = (p.cache_len + SK - 1) / SK;
  const int64_t per_b = (int64_t)nst * J;
  int64_t r, st;
  int b;
  if (p.B == 1) {
    b = 0;
    r = s;
  } else if ((per_b >> 31) == 0) {
    b = (int)div_pos(s, (int)per_b, &r);
  } else {
    b = (int)(s / per_b);
    r = s % per_b;
  }
  const int j = (int)div_pos(r, nst, &st);
  return Cursor{uni(b), uni(j), uni((int)st), uni(nst), uni(p.cache_len)};
}

// The stages of wave w of W: their count (returned) and, if any, the cursor
// of the first one; *part: the partition of all stages (PG == 0: the host
// divided).
template <int PG, int SK>
__device__ inline int64_t wave_plan(const DecodeParams& p, int J, int W, int w, Cursor* cc, Partition* part) {
  BatchScan sc;
  if constexpr (PG == 0) {
    *part = Partition(p.part_q, p.part_rem);
  } else {
    sc = batch_scan<PG, SK>(p, J);
    *part = Partition(sc.tot, W);
  }
  const int64_t s0 = part->start(w);
  const int64_t n = part->start(w + 1) - s0;
  if (n > 0) {
    if constexpr (PG == 0) *cc = locate_uniform<SK>(p, J, s0);
    else *cc = locate<PG, SK>(p, J, s0, sc);
  }
  return n;
}

// PG: 0 = contiguous cache, one length (cache_len) for every batch; 1 = the
// fused decode step (contiguous cache, per-batch positions in device memory,
// see below; 16-bit, D = 128); otherwise paged, PG = the rows of a group that
// lies inside one page (page_size % PG == 0; PG a multiple of the rows per
// load, at most SK): one table lookup and one pair of descriptors per group.
// QR: query rows staged per sequence (4 when the group has <= 4 heads, else 16).
//
// Decode step (PG == 1; model.py:340-347, :475-491): batch b's new token sits
// at pos = positions[b * pos_stride], its slot is pos (ring: pos % C) and the
// sequence is slots [0, step_len). At the start of each piece the wave reads
// pos, rotates its query fragments with table row pos (rotate-half, float32,
// rounded once to T: model.py:54-67) and prepares the new K row (rotated the
// same way) and V row in registers. The stage holding the slot is patched in
// LDS with those rows after its DMA lands -- the cache still holds the old
// slot contents, and no other stage holds that row -- and the wave that owns
// head slice 0 writes them to the cache slot. Every wave that reads the slot
// (one per head slice) patches its own copy, so no wave depends on another's
// global write within the launch.
//
// NWV = 1: the persistent grid of one-wave workgroups described above. NWV = 4
// (short sequences, few of them): a workgroup per sequence, its four waves
// taking a quarter of the stages each and merging through LDS at the end, so
// no piece leaves the workgroup and no second kernel runs.
template <typename T, int D, int PG, int NS, int QR, int NWV = 1, bool FINE = false>
__global__ __launch_bounds__(64 * NWV) void pf_decode_stream_kernel(DecodeParams p) {
  using MF = Mfma16<T>;
  using G = StreamGeo<T, D, FINE>;
  constexpr int SK = G::SK, RB = G::RB, KPL = G::KPL, NU = G::NU, NL = G::NL, RPL = G::RPL;
  constexpr int NSTEP = G::CPR / 4;  // K/Q chunk steps: lane group h reads chunk 4s + h
  constexpr int kSlotB = G::slot_bytes(QR);
  static_assert(PG != 1 || (D == 128 && !G::F32), "the decode step is written for 16-bit 128-column rows");
  static_assert(PG <= 1 || (PG % RPL == 0 && SK % PG == 0), "a page group is whole loads of one stage");
  __shared__ __attribute__((aligned(1024))) char smem_all[NWV * NS * kSlotB];

  const int lane = threadIdx.x & 63;
  const int wv = NWV > 1 ? uni((int)(threadIdx.x >> 6)) : 0;
  char* const smem = smem_all + wv * NS * kSlotB;  // this wave's ring
  const int i16 = lane & 15;
  const int h = lane >> 4;
  const int g = p.g;
  const int n_hc = (g + 15) >> 4;
  const int J = p.Hkv * n_hc;
  const int W = p.n_waves;
  const int w = blockIdx.x;

  Cursor cc;
  int64_t n;  // stages of this wave
  [[maybe_unused]] int per = 0;  // NWV > 1: stages per wave (the last ones may have fewer or none)
  if constexpr (NWV > 1) {
    const int b = w / J;
    cc = Cursor{b, w - b * J, 0, 0, seq_len<PG>(p, b)};
    cc.nst = (cc.L + SK - 1) / SK;
    per = (cc.nst + NWV - 1) / NWV;
    cc.st = wv * per;
    n = min(per, cc.nst - cc.st);
  } else {
    Partition part((int64_t)0, (int64_t)0);
    n = wave_plan<PG, SK>(p, J, W, w, &cc, &part);
    if (n <= 0) return;
  }

  const uint32_t lds0 = lds_u32(smem);
  const T* Kb = static_cast<const T*>(p.k);
  const T* Vb = static_cast<const T*>(p.v);
  const T* Qb = static_cast<const T*>(p.q);

  // Per-lane byte offset (within a stage's rows) of the chunk this lane
  // fetches for load i of a tile: 16-byte slot 64 i + lane.
  uint32_t loff[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int slot = 64 * i + lane, row = slot / G::CPR, c = slot % G::CPR;
    loff[i] = (uint32_t)(row * RB + 16 * (c ^ G::swz(row)));
  }

  // Issue the loads of the stage under cursor c into ring slot `slot`; with
  // `with_q`, first the query rows of c's head slice (rows past the group
  // arrive as zeros).
  auto issue = [&](const Cursor& c, int slot, bool with_q) {
    const uint32_t ldk = lds0 + (uint32_t)(slot * kSlotB);
    const uint32_t ldv = ldk + G::TILE;
    const int kvh = n_hc == 1 ? c.j : c.j / n_hc, hc = c.j - kvh * n_hc;
    if (with_q) {
      const int q0 = hc * 16;
      const int nq = min(QR, g - q0);
      const i32x4 dq = make_desc(Qb + ((int64_t)c.b * p.Hq + (int64_t)kvh * g + q0) * D, (uint32_t)(nq * RB));
#pragma unroll
      for (int i = 0; i < G::qrows(QR) / RPL; ++i) {
        const int qs = 64 * i + lane, row = qs / G::CPR, cq = qs % G::CPR;
        dma16(dq, (uint32_t)(row * RB + 16 * (cq ^ (row & G::QMASK))), ldv + G::TILE + 1024 * i);
      }
    }
    const int kv0 = c.st * SK;
    if constexpr (PG == 0 || PG == 1) {
      const int64_t seq = ((int64_t)c.b * p.Hkv + kvh) * (int64_t)p.cache_size * D;
      const i32x4 dk = make_desc(Kb + seq, (uint32_t)c.L * RB);
      const i32x4 dv = make_desc(Vb + seq, (uint32_t)c.L * RB);
      const uint32_t rb = (uint32_t)kv0 * RB;
#pragma unroll
      for (int i = 0; i < NL; ++i) dma16<kKvNt>(dk, rb + loff[i], ldk + 1024 * i);
#pragma unroll
      for (int i = 0; i < NL; ++i) dma16<kKvNt>(dv, rb + loff[i], ldv + 1024 * i);
    } else {
      const int ps = p.page_size;
      const int64_t trow = (int64_t)c.b * p.pages_per_seq;
      constexpr int kGroups = SK / PG;  // page-uniform groups per stage
      constexpr int kPer = NL / kGroups;
#pragma unroll
      for (int gi = 0; gi < kGroups; ++gi) {
        const int key0 = kv0 + gi * PG;
        // Groups at or past L load nothing (zero range) and look nothing up:
        // table entries at logical pages >= ceil(L / page_size) may be -1 or
        // lie past the table row.
        const bool live = key0 < c.L;
        const int lp = live ? key0 / ps : 0;
        int page = live ? sload_i32(p.block_tables, trow + lp) : 0;
        page = min(max(page, 0), p.num_pages - 1);
        const int prow0 = live ? lp * ps : key0;
        const int nvalid = live ? min(ps, c.L - prow0) : 0;
        const int64_t pbase = ((int64_t)page * p.Hkv + kvh) * (int64_t)ps * D;
        const i32x4 dk = make_desc(Kb + pbase, (uint32_t)(nvalid * RB));
        const i32x4 dv = make_desc(Vb + pbase, (uint32_t)(nvalid * RB));
        const uint32_t rb = (uint32_t)(kv0 - prow0) * RB;
#pragma unroll
        for (int j = 0; j < kPer; ++j) dma16<kKvNt>(dk, rb + loff[gi * kPer + j], ldk + 1024 * (gi * kPer + j));
#pragma unroll
        for (int j = 0; j < kPer; ++j) dma16<kKvNt>(dv, rb + loff[gi * kPer + j], ldv + 1024 * (gi * kPer + j));
      }
    }
  };

  // ---- decode step (PG == 1) --------------------------------------------
  // Per piece: the token's position, this lane's chunk of the new K row
  // (lanes 0-15, chunk i16, and its rotate-half partner i16 ^ 8) or V row
  // (lanes 16-31), and the table values the lane's rotations use (K: elements
  // 8 i16 .. +7; Q: 32 s + 8 h .. +7 for s = 0..3).
  struct StepData {
    int pos;
    u32x4 kv, kvp;
    f32x4 kc[2], ks[2];
    f32x4 qc[4][2], qs[4][2];
  };
  [[maybe_unused]] auto step_load = [&](const Cursor& c, StepData& d) {
    d.pos = sload_i32(p.positions, (int64_t)c.b * p.pos_stride);  // valid: the piece has keys
    const int kvh = n_hc == 1 ? c.j : c.j / n_hc;
    const int64_t src = ((int64_t)c.b * p.Hkv + kvh) * 128;
    if (lane < 32) {
      const T* nb = static_cast<const T*>(lane < 16 ? p.k_new : p.v_new) + src;
      d.kv = ldg16(nb + 8 * i16);
      d.kvp = ldg16(nb + 8 * (i16 ^ 8));
    }
    if (p.rope_cos != nullptr) {
      const float* cr = p.rope_cos + (int64_t)d.pos * 128;
      const float* sr = p.rope_sin + (int64_t)d.pos * 128;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        d.kc[u] = *reinterpret_cast<const f32x4*>(cr + 8 * i16 + 4 * u);
        d.ks[u] = *reinterpret_cast<const f32x4*>(sr + 8 * i16 + 4 * u);
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) {
          d.qc[s4][u] = *reinterpret_cast<const f32x4*>(cr + 32 * s4 + 8 * h + 4 * u);
          d.qs[s4][u] = *reinterpret_cast<const f32x4*>(sr + 32 * s4 + 8 * h + 4 * u);
        }
      }
    }
  };
  // Rotate-half RoPE of 8 consecutive elements d0 .. d0 + 7 of a 128-element
  // row whose partner elements (d +- 64) are in xp, with those elements'
  // table values: y = x cos - x' sin (first half), x cos + x' sin (second
  // half), float32, rounded once to T (model.py:54-67; fused_rope.py:43-50).
  auto rope8 = [&](const u32x4& x, const u32x4& xp, const f32x4* c, const f32x4* sn, bool first_half) -> u32x4 {
    float a[8], b2[8], y[8];
    chunk_to_f32<T>(x, a);
    chunk_to_f32<T>(xp, b2);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float ce = c[e >> 2][e & 3], se = sn[e >> 2][e & 3];
      y[e] = first_half ? a[e] * ce - b2[e] * se : a[e] * ce + b2[e] * se;
    }
    return f32_to_chunk<T>(y);
  };
  // New piece: the token's slot, the rotated query fragments (lane holds
  // Q[head i16][32 s + 8 h + e]; the partner of s is s ^ 2) and this lane's
  // new K (rotated) or V row chunk.
  [[maybe_unused]] auto step_apply = [&](const StepData& d, u32x4* q4, int& tslot, u32x4& row) {
    tslot = p.ring != 0 ? d.pos % p.cache_size : d.pos;
    row = d.kv;
    if (p.rope_cos != nullptr) {
      if (lane < 16) row = rope8(d.kv, d.kvp, d.kc, d.ks, i16 < 8);
      u32x4 qx[4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) qx[s4] = q4[s4];
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) q4[s4] = rope8(qx[s4], qx[s4 ^ 2], d.qc[s4], d.qs[s4], s4 < 2);
    }
  };
  // Stage holding the token's slot at row r: overwrite that row of the K and
  // V tiles (after the stage's DMA landed), and write it to the cache once
  // (head slice 0).
  [[maybe_unused]] auto step_patch = [&](const Cursor& c, char* tK, char* tV, int r, int tslot, const u32x4& row) {
    if (lane < 32) {
      char* t = lane < 16 ? tK : tV;
      sts16(t + r * RB + 16 * (i16 ^ G::swz(r)), row);
      const int kvh = n_hc == 1 ? c.j : c.j / n_hc, hc = c.j - kvh * n_hc;
      if (hc == 0) {
        T* out = static_cast<T*>(lane < 16 ? p.k_out : p.v_out);
        stg16(out + (((int64_t)c.b * p.Hkv + kvh) * p.cache_size + tslot) * 128 + 8 * i16, row);
      }
    }
    // this wave's LDS accesses run in order; keep the compiler from moving
    // the tile reads above the stores
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  [[maybe_unused]] StepData pend;  // NS == 2: the step data of the piece the next stage opens

  // Prologue: the first NS - 1 stages.
  Cursor pc = cc;
#pragma unroll
  for (int k = 0; k < NS - 1; ++k) {
    if (k < n) {
      issue(pc, k, k == 0 || pc.st == 0);
      if constexpr (PG == 1 && NS == 2) step_load(pc, pend);  // stage 0 opens a piece
      cursor_next<PG, SK>(pc, p, J);
    }
  }

  // Per-lane LDS read offsets.
  // K (A operand, tile u, step s): key row KPL(i16/4) + 4u + i16%4, chunk
  // 4s + h; steps past the 16 permuted chunks lie 256 bytes further on.
  constexpr int NKO = NSTEP < 4 ? NSTEP : 4;
  uint32_t koff[NU][NKO];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int row = KPL * (i16 >> 2) + 4 * u + (i16 & 3);
#pragma unroll
    for (int s = 0; s < NKO; ++s) koff[u][s] = (uint32_t)(row * RB + 16 * ((4 * s + h) ^ G::swz(row)));
  }
  // V. 16-bit (V^T as the A operand via transposing reads, d tile dt, key
  // group e): the lane addresses row KPL h + 4e + i16/4, columns 16dt +
  // 4(i16%4) .. +3. float32: row KPL h + t, chunk i16 (+ 16 blk).
  constexpr int NVO = G::F32 ? 1 : (G::NACC < 8 ? G::NACC : 8);
  constexpr int NVE = G::F32 ? KPL : NU;
  uint32_t voff[NVO][NVE];
#pragma unroll
  for (int e = 0; e < NVE; ++e) {
    if constexpr (G::F32) {
      const int row = KPL * h + e;
      voff[0][e] = (uint32_t)(row * RB + 16 * (i16 ^ G::swz(row)));
    } else {
      const int row = KPL * h + 4 * e + (i16 >> 2);
#pragma unroll
      for (int dt = 0; dt < NVO; ++dt) {
        const int chunk = 2 * dt + ((i16 >> 1) & 1);
        voff[dt][e] = (uint32_t)(row * RB + 16 * (chunk ^ G::swz(row)) + 8 * (i16 & 1));
      }
    }
  }

  u32x4 qf[NSTEP];
  // O^T accumulators: 16-bit tile dt, register r = column 16dt + 4h + r;
  // float32 tile 4 blk + e, register r = column 64 blk + 16h + 4r + e.
  f32x4 acc[G::NACC];
  float m_run = kNegInf, l_run = 0.f;
  int piece_st0 = 0;       // first stage (within the sequence) of the current piece
  bool first_piece = true;  // the current piece opens this wave's range
  // Decode step: the current piece's token slot and its new K (lanes 0-15,
  // 16-byte chunk i16) / V (lanes 16-31) row chunk.
  [[maybe_unused]] int tok_slot = -1;
  [[maybe_unused]] u32x4 new_row = (u32x4){0u, 0u, 0u, 0u};

  for (int64_t k = 0; k < n; ++k) {
    wait_stage<NS, 2 * NL>(min((int64_t)(NS - 2), n - 1 - k));
    const int slot = (int)(k % NS);
    char* const sK = smem + slot * kSlotB;
    char* const sV = sK + G::TILE;
    if (k == 0 || cc.st == 0) {
      // New piece: query fragments (B operand of S^T: lane holds chunk 4s + h
      // of head i16's row) and a fresh softmax state.
      const char* sQ = sV + G::TILE;
#pragma unroll
      for (int s = 0; s < NSTEP; ++s)
        qf[s] = (i16 < QR) ? lds16(sQ + i16 * RB + 16 * ((4 * s + h) ^ (i16 & G::QMASK))) : (u32x4){0u, 0u, 0u, 0u};
      if constexpr (PG == 1) {
        if constexpr (NS == 2) {
          step_apply(pend, qf, tok_slot, new_row);  // loaded with the stage's DMA
        } else {
          StepData d;
          step_load(cc, d);
          step_apply(d, qf, tok_slot, new_row);
        }
      }
#pragma unroll
      for (int dt = 0; dt < G::NACC; ++dt) acc[dt] = (f32x4)(0.f);
      m_run = kNegInf;
      l_run = 0.f;
      piece_st0 = cc.st;
    }
    if constexpr (PG == 1) {
      // the stage holding the new token's slot: its row comes from registers
      const int r = tok_slot - cc.st * SK;
      if (r >= 0 && r < SK) step_patch(cc, sK, sV, r, tok_slot, new_row);
    }
    if (k + NS - 1 < n) {
      issue(pc, (int)((k + NS - 1) % NS), pc.st == 0);
      if constexpr (PG == 1 && NS == 2) {
        // the next stage opens a piece: its step data arrive with its tiles
        if (pc.st == 0) step_load(pc, pend);
      }
      cursor_next<PG, SK>(pc, p, J);
    }

    const int kv0 = cc.st * SK;
    // S^T (SK keys x 16 heads): lane holds keys kv0 + KPL h + 4u + r, head i16.
    f32x4 s[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) s[u] = (f32x4)(0.f);
#pragma unroll
    for (int st = 0; st < NSTEP; ++st)
#pragma unroll
      for (int u = 0; u < NU; ++u)
        s[u] = MF::run(lds16(sK + koff[u][st % NKO] + 256 * (st / NKO)), qf[st], s[u]);

    float x[KPL];
    float mx = kNegInf;
#pragma unroll
    for (int t = 0; t < KPL; ++t) {
      const int key = kv0 + KPL * h + t;
      x[t] = key < cc.L ? s[t >> 2][t & 3] * p.scale_log2 : kNegInf;
      mx = fmaxf(mx, x[t]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == kNegInf) ? 0.f : m_new;
    const float alpha = exp2f(m_run - m_use);
    float rs = 0.f;
#pragma unroll
    for (int t = 0; t < KPL; ++t) {
      x[t] = exp2f(x[t] - m_use);
      rs += x[t];
    }
    l_run = l_run * alpha + rs;
    m_run = m_new;

    // O^T (D x 16 heads) += V^T . P^T
    if constexpr (G::F32) {
#pragma unroll
      for (int a = 0; a < G::NACC; ++a) acc[a] = acc[a] * alpha;
#pragma unroll
      for (int t = 0; t < KPL; ++t)
#pragma unroll
        for (int blk = 0; blk < D / 64; ++blk) {
          const f32x4 v = __builtin_bit_cast(f32x4, lds16(sV + voff[0][t] + 256 * blk));
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * blk + e] = MF::step(v[e], x[t], acc[4 * blk + e]);
        }
    } else {
      typedef T vk __attribute__((ext_vector_type(KPL)));
      vk pf;
#pragma unroll
      for (int t = 0; t < KPL; ++t) pf[t] = Elem<T>::from_f32(x[t]);
#pragma unroll
      for (int dt = 0; dt < G::NACC; ++dt) {
        i16x4 v[NU];
#pragma unroll
        for (int e = 0; e < NU; ++e)
          v[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(sV + voff[dt % NVO][e] + 256 * (dt / NVO)));
        if constexpr (SK == 32)
          acc[dt] = MF::run(__builtin_bit_cast(u32x4, __builtin_shufflevector(v[0], v[1], 0, 1, 2, 3, 4, 5, 6, 7)),
                            __builtin_bit_cast(u32x4, pf), acc[dt] * alpha);
        else
          acc[dt] = MF::run16(__builtin_bit_cast(u32x2, v[0]), __builtin_bit_cast(u32x2, pf), acc[dt] * alpha);
      }
    }

    if (cc.st == cc.nst - 1 || k == n - 1) {
      // ---- end of a piece ---------------------------------------------------
      float l_tot = l_run + __shfl_xor(l_run, 16);
      l_tot += __shfl_xor(l_tot, 32);
      // column d0 and value r of the lane's q-th group of 4 outputs (NACC groups)
      auto out4 = [&](int q, int& d0) -> f32x4 {
        if constexpr (G::F32) {
          const int blk = q >> 2, r = q & 3;
          d0 = 64 * blk + 16 * h + 4 * r;
          return (f32x4){acc[4 * blk][r], acc[4 * blk + 1][r], acc[4 * blk + 2][r], acc[4 * blk + 3][r]};
        } else {
          d0 = 16 * q + 4 * h;
          return acc[q];
        }
      };
      if constexpr (NWV > 1) {
        // this wave's ring is consumed: its piece goes there, for the merge
        float* po = reinterpret_cast<float*>(smem);
        if (i16 < QR) {
#pragma unroll
          for (int q = 0; q < G::NACC; ++q) {
            int d0;
            const f32x4 a = out4(q, d0);
            *reinterpret_cast<f32x4*>(po + i16 * D + d0) = a;
          }
          if (h == 0) *reinterpret_cast<f32x2*>(po + QR * D + 2 * i16) = (f32x2){m_run, l_tot};
        }
        break;
      }
      const int kvh = n_hc == 1 ? cc.j : cc.j / n_hc, hc = cc.j - kvh * n_hc;
      const int qh = hc * 16 + i16;
      if (piece_st0 == 0 && cc.st == cc.nst - 1) {
        // The whole sequence: finish it here.
        if (qh < g) {
          const float inv = (l_tot == 0.f) ? 0.f : 1.f / l_tot;
          T* out = static_cast<T*>(p.o) + ((int64_t)cc.b * p.Hq + (int64_t)kvh * g + qh) * D;
#pragma unroll
          for (int q = 0; q < G::NACC; ++q) {
            int d0;
            const f32x4 a = out4(q, d0);
            typedef T v4 __attribute__((ext_vector_type(4)));
            v4 y;
#pragma unroll
            for (int r = 0; r < 4; ++r) y[r] = Elem<T>::from_f32(a[r] * inv);
            *reinterpret_cast<v4*>(out + d0) = y;
          }
        }
      } else if (i16 < QR) {
        const int64_t pslot = piece_slot(p, J, w, (int64_t)cc.b * J + cc.j, !first_piece);
        float* po = p.part_o + (pslot * QR + i16) * D;
#pragma unroll
        for (int q = 0; q < G::NACC; ++q) {
          int d0;
          const f32x4 a = out4(q, d0);
          *reinterpret_cast<f32x4*>(po + d0) = a;
        }
        if (h == 0)
          *reinterpret_cast<f32x2*>(p.part_ml + (pslot * QR + i16) * 2) = (f32x2){m_run, l_tot};
      }
      first_piece = false;
    }
    cursor_next<PG, SK>(cc, p, J);
  }
  if constexpr (NWV > 1) {
    // o = sum_i acc_i 2^(m_i - M) / sum_i l_i 2^(m_i - M) over the waves' pieces
    // (none: o = 0), 4 columns of a head's row per thread.
    __syncthreads();
    const int kvh = n_hc == 1 ? cc.j : cc.j / n_hc, hc = cc.j - kvh * n_hc;
    const int nq = min(QR, g - hc * 16);
    T* const out = static_cast<T*>(p.o) + ((int64_t)cc.b * p.Hq + (int64_t)kvh * g + hc * 16) * D;
    for (int i = threadIdx.x; i < nq * (D / 4); i += 64 * NWV) {
      const int row = i / (D / 4), d0 = 4 * (i % (D / 4));
      f32x2 ml[NWV];
      float M = kNegInf;
#pragma unroll
      for (int v = 0; v < NWV; ++v) {
        ml[v] = (f32x2){kNegInf, 0.f};
        if (v * per < cc.nst)
          ml[v] = *reinterpret_cast<const f32x2*>(reinterpret_cast<float*>(smem_all + v * NS * kSlotB) + QR * D +
                                                  2 * row);
        M = fmaxf(M, ml[v][0]);
      }
      const float Mu = (M == kNegInf) ? 0.f : M;
      f32x4 o = (f32x4)(0.f);
      float l = 0.f;
#pragma unroll
      for (int v = 0; v < NWV; ++v) {
        if (v * per < cc.nst) {
          const float wt = exp2f(ml[v][0] - Mu);
          l += ml[v][1] * wt;
          o += *reinterpret_cast<const f32x4*>(reinterpret_cast<float*>(smem_all + v * NS * kSlotB) + row * D + d0) *
               wt;
        }
      }
      const float inv = (l == 0.f) ? 0.f : 1.f / l;
      typedef T v4 __attribute__((ext_vector_type(4)));
      v4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = Elem<T>::from_f32(o[e] * inv);
      *reinterpret_cast<v4*>(out + row * D + d0) = y;
    }
  }
}

// Merge the partial pieces of each (b, h) whose sequence was cut by wave
// boundaries: o = sum_i acc_i 2^(m_i - M) / sum_i l_i 2^(m_i - M); a batch
// with no valid key gives o = 0 (flash_attention.py:150-159; paged.py:95-99).
// Sequences that one wave covered were written by the main kernel.
//
// WPB waves share one (b, h)'s pieces, each taking a contiguous run of them
// and merging at the end through LDS. The pieces were just written by other
// XCDs, so every read of one is a trip past this XCD's L2: a wave reads up to
// 64 (max, sum) pairs with one load, a lane each, and the accumulators 8
// pieces at a time, instead of one dependent piece after another. One wave
// reading piece after piece took 30 us for 47 pieces of each of 32 heads (one
// sequence of 1500 keys, 8 kv heads); 8 waves a head take 5 us. At 8-9 pieces
// (B=16, 4096 keys): 7.5 -> 4.8 us.
template <typename T, int D, int PG, int QR, int WPB, bool FINE>
__global__ __launch_bounds__(64 * WPB) void pf_decode_stream_combine_kernel(DecodeParams p) {
  constexpr int SK = StreamGeo<T, D, FINE>::SK;
  constexpr int PER = D / 64;  // columns per lane
  constexpr int NB = 8;        // pieces in flight
  typedef float vp __attribute__((ext_vector_type(PER)));
  const int lane = threadIdx.x & 63;
  const int wv = uni((int)(threadIdx.x >> 6));
  const int bh = blockIdx.x;
  const int b = p.B == 1 ? 0 : bh / p.Hq, hq = bh - b * p.Hq;
  const int g = p.g;
  const int n_hc = (g + 15) >> 4;
  const int J = p.Hkv * n_hc;
  const int kvh = hq / g, qh = hq - kvh * g, hc = qh >> 4, qi = qh & 15;
  const int W = p.n_waves;

  // Global stage range [s0, s1) of this head's sequence.
  Partition part((int64_t)0, (int64_t)0);  // of all stages
  int64_t before = 0;     // stages of batches < b
  int L;
  if constexpr (PG == 0) {
    part = Partition(p.part_q, p.part_rem);
    L = p.cache_len;
    before = (int64_t)b * ((L + SK - 1) / SK) * J;
  } else {
    const BatchScan sc = batch_scan<PG, SK>(p, J);
    part = Partition(sc.tot, W);
    before = stages_before<PG, SK>(p, J, uni(b), sc);
    L = sc.per == 1 ? __builtin_amdgcn_readlane(sc.L, uni(b)) : seq_len<PG>(p, uni(b));
  }
  const int nst = (L + SK - 1) / SK;
  T* out = static_cast<T*>(p.o) + (int64_t)bh * D + PER * lane;
  if (nst == 0) {
    if (wv == 0) {
#pragma unroll
      for (int e = 0; e < PER; ++e) out[e] = Elem<T>::from_f32(0.f);
    }
    return;
  }
  const int64_t s0 = before + (int64_t)(kvh * n_hc + hc) * nst;
  const int wa = uni(part.wave_of(s0)), wb = uni(part.wave_of(s0 + nst - 1));
  if (wa == wb) return;  // finished by the main kernel (uniform over the workgroup)

  // Piece i is wave wa + i's; only the first can start inside a wave's range.
  const bool late = part.start(wa) < s0;
  const int64_t seq = (int64_t)b * J + kvh * n_hc + hc;
  const int np = wb - wa + 1;
  const int per = (np + WPB - 1) / WPB;
  const int i_end = min(np, (wv + 1) * per);
  float M = kNegInf, lsum = 0.f;  // lsum: per lane until the end
  vp o = (vp)(0.f);
  for (int i0 = wv * per; i0 < i_end; i0 += 64) {
    const int cnt = min(64, i_end - i0);
    f32x2 ml = {kNegInf, 0.f};
    if (lane < cnt) {
      const int i = i0 + lane;
      const int64_t slot = piece_slot(p, J, wa + i, seq, i == 0 && late);
      ml = *reinterpret_cast<const f32x2*>(p.part_ml + (slot * QR + qi) * 2);
    }
    float mc = ml[0];
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) mc = fmaxf(mc, __shfl_xor(mc, s));
    const float Mn = fmaxf(M, mc);
    const float Mu = (Mn == kNegInf) ? 0.f : Mn;
    const float back = exp2f(M - Mu);
    const float wt = lane < cnt ? exp2f(ml[0] - Mu) : 0.f;
    lsum = lsum * back + ml[1] * wt;
    o *= back;
    M = Mn;
    for (int j0 = 0; j0 < cnt; j0 += NB) {
      vp v[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        v[j] = (vp)(0.f);
        if (j0 + j < cnt) {
          const int i = i0 + j0 + j;
          const int64_t slot = piece_slot(p, J, wa + i, seq, i == 0 && late);
          v[j] = *reinterpret_cast<const vp*>(p.part_o + (slot * QR + qi) * D + PER * lane);
        }
      }
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (j0 + j < cnt) o += v[j] * __shfl(wt, j0 + j);
    }
  }
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) lsum += __shfl_xor(lsum, s);
  __shared__ float sm[WPB][2];
  __shared__ vp so[WPB][64];
  if (lane == 0) {
    sm[wv][0] = M;
    sm[wv][1] = lsum;
  }
  so[wv][lane] = o;
  __syncthreads();
  if (wv != 0) return;
  M = kNegInf;
#pragma unroll
  for (int i = 0; i < WPB; ++i) M = fmaxf(M, sm[i][0]);
  const float Mu = (M == kNegInf) ? 0.f : M;
  lsum = 0.f;
  o = (vp)(0.f);
#pragma unroll
  for (int i = 0; i < WPB; ++i) {
    if (i * per >= np) break;  // a wave without pieces holds nothing
    const float wt = exp2f(sm[i][0] - Mu);
    lsum += sm[i][1] * wt;
    o += so[i][lane] * wt;
  }
  const float inv = (lsum == 0.f) ? 0.f : 1.f / lsum;
#pragma unroll
  for (int e = 0; e < PER; ++e) out[e] = Elem<T>::from_f32(o[e] * inv);
}

// The same for sequences in few pieces: a workgroup per wave boundary, that is
// per place where a sequence can be cut at all. The first boundary inside a
// sequence takes it: one wave finds it in the work list for all four, and the
// workgroup's threads take 4 columns of a head each. The last workgroups write
// the zeros of batches without a valid key. Bound by the search's and the
// pieces' latency. A wave per (b, h), each with a search of its own, mostly to
// find that its sequence is whole, took 30 us at 19200 heads and, with the
// batch-by-batch search, 855 us at 65536 (bf16 head_dim 64, 300 x 64 and
// 4096 x 16 heads of up to 128 and 64 keys; now 8 and 10), more than the
// attention itself; at 2048 and 4096 heads of head_dim 128 5.0 -> 4.9 and
// 7.5 -> 5.9 us.
template <typename T, int D, int PG, int QR, bool FINE>
__global__ __launch_bounds__(256) void pf_decode_stream_cut_kernel(DecodeParams p) {
  constexpr int SK = StreamGeo<T, D, FINE>::SK;
  const int lane = threadIdx.x & 63;
  const int wv = uni((int)(threadIdx.x >> 6));
  const int g = p.g;
  const int n_hc = (g + 15) >> 4;
  const int J = p.Hkv * n_hc;
  const int W = p.n_waves;
  const int w = blockIdx.x + 1;
  if (PG != 0 && w >= W) {
    const int b = (w - W) * 4 + wv;
    if (b >= p.B || seq_len<PG>(p, b) > 0) return;
    typedef T v4 __attribute__((ext_vector_type(4)));
    v4* out = reinterpret_cast<v4*>(static_cast<T*>(p.o) + (int64_t)b * p.Hq * D);
    const int64_t n = (int64_t)p.Hq * (D / 4);
    for (int64_t i = lane; i < n; i += 64) out[i] = (v4)(Elem<T>::from_f32(0.f));
    return;
  }
  __shared__ int found[4];  // pieces, batch, sequence within it, late
  if (wv == 0) {
    Cursor c{0, 0, 0, 0, 0};
    Partition part((int64_t)0, (int64_t)0);
    int np = 0;
    bool late = false;
    if (wave_plan<PG, SK>(p, J, W, w, &c, &part) > 0 && c.st > 0) {
      const int64_t s0 = part.start(w) - c.st, before = part.start(w - 1);
      late = before < s0;
      if (before <= s0) np = part.wave_of(s0 + c.nst - 1) - w + 2;
    }
    if (lane == 0) {
      found[0] = np;
      found[1] = c.b;
      found[2] = c.j;
      found[3] = late;
    }
  }
  __syncthreads();
  const int np = uni(found[0]), b = uni(found[1]), j = uni(found[2]);
  const bool late = uni(found[3]) != 0;
  if (np == 0) return;
  const int kvh = j / n_hc, hc = j - kvh * n_hc;
  const int nq = min(16, g - 16 * hc);
  const int64_t seq = (int64_t)b * J + j;
  typedef T v4 __attribute__((ext_vector_type(4)));
  T* out = static_cast<T*>(p.o) + ((int64_t)b * p.Hq + (int64_t)kvh * g + hc * 16) * D;
  constexpr int NB = 8;  // pieces in flight
  for (int i = threadIdx.x; i < nq * (D / 4); i += 256) {
    const int qi = i / (D / 4), d0 = 4 * (i % (D / 4));
    float M = kNegInf, l = 0.f;
    f32x4 o = (f32x4)(0.f);
    for (int c0 = 0; c0 < np; c0 += NB) {
      float ls[NB];
      f32x2 ml[NB];
      f32x4 v[NB];
      float Mn = M;
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        ml[c] = (f32x2){kNegInf, 0.f};
        v[c] = (f32x4)(0.f);
        if (c0 + c < np) {
          const int64_t row = piece_slot(p, J, w - 1 + c0 + c, seq, c0 + c == 0 && late) * QR + qi;
          ml[c] = *reinterpret_cast<const f32x2*>(p.part_ml + row * 2);
          v[c] = *reinterpret_cast<const f32x4*>(p.part_o + row * D + d0);
        }
        Mn = fmaxf(Mn, ml[c][0]);
      }
      const float Mu = (Mn == kNegInf) ? 0.f : Mn;
      const float back = exp2f(M - Mu);
      o *= back;
#pragma unroll
      for (int c = 0; c < NB; ++c) {
        const float wt = exp2f(ml[c][0] - Mu);
        ls[c] = ml[c][1] * wt;
        o += v[c] * wt;
      }
      {
        // in the order of pf_decode_stream_combine_kernel's lanes, unfused: up
        // to NB pieces give its bits
#pragma clang fp contract(off)
        l = l * back + (((ls[0] + ls[1]) + (ls[2] + ls[3])) + ((ls[4] + ls[5]) + (ls[6] + ls[7])));
      }
      M = Mn;
    }
    const float inv = (l == 0.f) ? 0.f : 1.f / l;
    v4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = Elem<T>::from_f32(o[e] * inv);
    *reinterpret_cast<v4*>(out + qi * D + d0) = y;
  }
}

// The merge's form: the pieces of a sequence, about n_waves / sequences (and at
// most one per stage), decide. Few: a workgroup per wave boundary; more than 6,
// where the sequences are at most a sixth of the waves: 4 or 8 waves share the
// pieces of each (b, h).
template <typename T, int D, int PG, int QR, bool FINE>
hipError_t launch_combine(const DecodeParams& p, hipStream_t st) {
  const int64_t n_bh = (int64_t)p.B * p.Hq;
  const int64_t seqs = (int64_t)p.B * p.Hkv * ((p.Hq / p.Hkv + 15) / 16);
  const int64_t len = PG <= 1 ? p.cache_len : (int64_t)p.pages_per_seq * p.page_size;
  const int64_t pieces = std::min((int64_t)p.n_waves / seqs, len / StreamGeo<T, D, FINE>::SK) + 1;
  if (pieces > 32) {
    hipLaunchKernelGGL((pf_decode_stream_combine_kernel<T, D, PG, QR, 8, FINE>), dim3((unsigned)n_bh), dim3(512), 0, st, p);
  } else if (pieces > 6) {
    hipLaunchKernelGGL((pf_decode_stream_combine_kernel<T, D, PG, QR, 4, FINE>), dim3((unsigned)n_bh), dim3(256), 0, st, p);
  } else {
    const int64_t n = p.n_waves - 1 + (PG == 0 ? 0 : (p.B + 3) / 4);  // a wave per batch for the zeros
    if (n > 0)
      hipLaunchKernelGGL((pf_decode_stream_cut_kernel<T, D, PG, QR, FINE>), dim3((unsigned)n), dim3(256), 0, st, p);
  }
  return hipGetLastError();
}

// Short sequences (at most 12 stages: three a wave) and at most as many as are
// resident at once run a workgroup each (NWV = 4). One launch instead of two, and
// no trip of the pieces through memory: calls over 80-250 keys 8.0-9.8 us ->
// 5.1-6.6 us; from about 16 stages the longer chain costs what the second
// kernel did. A grid size set by hand (decode_waves) keeps the persistent grid.
constexpr int kShortWaves = 4, kShortStages = 12;
template <typename T, int D, int PG, int QR>
bool short_form(const DecodeParams& p) {
  using G = StreamGeo<T, D>;
  const int64_t seqs = (int64_t)p.B * p.Hkv * ((p.Hq / p.Hkv + 15) / 16);
  const int64_t len = PG <= 1 ? p.cache_len : (int64_t)p.pages_per_seq * p.page_size;
  constexpr int per_cu = 160 * 1024 / (kShortWaves * 2 * G::slot_bytes(QR));
  return per_cu > 0 && !p.fixed_grid && p.stages == 2 && seqs <= 256 * per_cu && len <= kShortStages * G::SK;
}

template <typename T, int D, int PG, int NS, int QR, bool FINE>
hipError_t launch_stream(const DecodeParams& p, hipStream_t st) {
  if constexpr (!FINE && NS == 2 && kShortWaves * 2 * StreamGeo<T, D>::slot_bytes(QR) <= 160 * 1024) {
    if (short_form<T, D, PG, QR>(p)) {
      const unsigned seqs = (unsigned)(p.B * p.Hkv * ((p.Hq / p.Hkv + 15) / 16));
      hipLaunchKernelGGL((pf_decode_stream_kernel<T, D, PG, 2, QR, kShortWaves>), dim3(seqs), dim3(64 * kShortWaves),
                         0, st, p);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((pf_decode_stream_kernel<T, D, PG, NS, QR, 1, FINE>), dim3((unsigned)p.n_waves), dim3(64), 0, st,
                     p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return launch_combine<T, D, PG, QR, FINE>(p, st);
}

// The ring depth is a tuning of the 16-bit head_dim 128 kernels; the others
// run two stages.
template <typename T, int D, int PG, int QR, bool FINE>
hipError_t launch_ns(const DecodeParams& p, hipStream_t st) {
  if constexpr (sizeof(T) == 2 && D == 128) {
    if (p.stages == 3) return launch_stream<T, D, PG, 3, QR, FINE>(p, st);
    if (p.stages == 4) return launch_stream<T, D, PG, 4, QR, FINE>(p, st);
  }
  return launch_stream<T, D, PG, 2, QR, FINE>(p, st);
}

template <typename T, int D, int PG, bool FINE = false>
hipError_t launch_qr(const DecodeParams& p, hipStream_t st) {
  return (p.Hq / p.Hkv <= 4) ? launch_ns<T, D, PG, 4, FINE>(p, st) : launch_ns<T, D, PG, 16, FINE>(p, st);
}

// Page groups: as many rows as one table lookup can serve (up to a stage).
// The smallest group is 4 rows, or one whole load of 128-byte rows.
template <typename T, int D>
hipError_t launch_pg(const DecodeParams& p, bool paged, hipStream_t st) {
  using G = StreamGeo<T, D>;
  if constexpr (sizeof(T) == 4 && D == 64) {
    if (p.fine) {
      if (!paged) return launch_qr<T, D, 0, true>(p, st);
      return p.page_size % 16 == 0 ? launch_qr<T, D, 16, true>(p, st) : launch_qr<T, D, 4, true>(p, st);
    }
  }
  if (!paged) {
    if constexpr (sizeof(T) == 2 && D == 128) {
      if (p.positions != nullptr) return launch_qr<T, D, 1>(p, st);
    }
    return p.positions != nullptr ? hipErrorInvalidValue : launch_qr<T, D, 0>(p, st);
  }
  if constexpr (G::SK == 32) {
    if (p.page_size % 32 == 0) return launch_qr<T, D, 32>(p, st);
  }
  if (p.page_size % 16 == 0) return launch_qr<T, D, 16>(p, st);
  return launch_qr<T, D, G::RPL == 8 ? 8 : 4>(p, st);
}

// Resident one-wave workgroups per CU (LDS-limited) of the kernel with `qr`
// query rows and an `ns`-stage ring, 0 if the query fails.
template <typename T, int D, int NS, int QR, bool FINE = false>
int blocks_per_cu() {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, pf_decode_stream_kernel<T, D, 0, NS, QR, 1, FINE>, 64, 0) !=
      hipSuccess)
    return 0;
  return n;
}

}  // namespace stream
}  // namespace pf
