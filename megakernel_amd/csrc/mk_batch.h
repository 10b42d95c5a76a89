// Batched greedy decode of up to 16 independent sequences.
//
// One decode step of all sequences is a fixed sequence of kernels, captured
// once into a HIP graph and replayed per step:
//   embed                 x[b] = E[tok[b]]
//   per layer:  qkv       rmsnorm(x) -> fused QKV GEMM           (16-row blocks)
//               attn      QK-norm + RoPE + KV append + split attention; the last
//                         split of each (sequence, kv head) merges the partials
//               o         O GEMM + residual                       (16-row blocks)
//               gu        rmsnorm(x) -> gate/up GEMM -> SiLU(g) * u
//               down      down GEMM + residual
//   lm                    final rmsnorm -> tied LM head GEMM -> per-sequence argmax
//   tok                   argmax keys -> tokens, positions + 1
// (reference phase order /root/reference/src/megakernel.cu:132-332, per sequence).
//
// With 16 sequences every weight block is used 16 times, so the GEMMs run on
// the matrix cores: v_mfma_f32_16x16x32_bf16 with the weight tile as the A
// operand (the tile layout of mk_config.h) and the 16 sequences' activations
// as the B operand (column n = sequence n).  Activations are fp32 and enter
// the products as two bf16 parts (hi = RNE(v), lo = RNE(v - hi); relative
// error <= 2^-17), two products per tile.  Kernel boundaries order every
// hand-off, so activations are ordinary cached loads and stores; only the
// attention merge hands partials between workgroups of one launch (write-through
// stores, an agent-scope counter, agent-scope loads).
#pragma once
#include <type_traits>

#include "mk_config.h"
#include "mk_device.h"
#include "mk_host.h"

namespace mk {
namespace batch {

constexpr int BMAX = 16;       // sequences per step (MFMA columns)
constexpr int GT = 512;        // threads of the GEMM kernels (8 waves)
constexpr int GW = GT / kWave;
#ifndef MK_BATCH_AT
#define MK_BATCH_AT 256
#endif
constexpr int AT = MK_BATCH_AT;  // threads of an attention item (4 waves)
static_assert(AT >= 4 * kWave, "the attention prologue takes q0, q1, k and v on waves 0-3");
constexpr int AW = AT / kWave;
#ifndef MK_BATCH_NBW
#define MK_BATCH_NBW 2
#endif
constexpr int NBW = MK_BATCH_NBW;  // 32-position blocks per wave and attention item
constexpr int CH = 32 * AW * NBW;  // positions per attention split
constexpr int PW = 2 * 64 + 4; // partial words per item for GQA 2, D 64: o[2][64], (m, l) x 2
// K splits of the GEMM kernels (whole 32-column tiles per split)
// (measured: splitting pays only for the K = F down projection, 64 blocks of
// 88 tiles; the others lose more to the reduction than they gain)
constexpr int KS_QKV = 1, KS_O = 1, KS_GU = 1, KS_DN = 4;

// Hand-off flags of one layer in the single-kernel step (bk_step), one word
// per producer: QKV blocks, merged (sequence, kv head) attention outputs, O
// blocks, gate / up blocks, down blocks.  A producer writes the step's epoch
// into its word after its outputs are acknowledged; a consumer waits until
// every word it needs holds the epoch.  One writer per word and no atomics:
// a single counter that every producer incremented serialised the
// increments at one memory channel (5-10 us per hand-off).
enum : int { FC_QKV = 0, FC_ATT, FC_O, FC_GU, FC_DN, FC_N };
constexpr int FLAG_MAX = 256;  // producers per phase (>= F/16, QKV/16, BMAX * NKV)
// Optional timestamps of bk_step per layer and workgroup: layer start, then
// inputs ready / done of QKV, attention, O, gate/up and down (a workgroup
// without a role in a phase leaves that phase's stamps 0).
enum : int { TR_START = 0, TR_QKV_IN, TR_QKV_DONE, TR_ATT_IN, TR_ATT_DONE, TR_O_IN, TR_O_DONE, TR_GU_IN,
             TR_GU_DONE, TR_DN_IN, TR_DN_DONE, TR_N };

struct BParams {
  const u32x4* wqkv;        // per layer [QKV/16][H/32] tiles
  const u32x4* wo;          // per layer [H/16][QD/32]
  const u32x4* wg;          // per layer gate [F/16][H/32]
  const u32x4* wu;          // per layer up
  const u32x4* wd;          // per layer down [H/16][F/32]
  const u32x4* lmhead;      // [V/16][H/32]
  const u32x4* lmhead8;     // optional FP8 (e4m3) copy [V/16][H/64][64] (bk_lm<S, true>)
  const float* lm_scale;    // [V] its power-of-two row scales
  long long u_qkv, u_o, u_gu, u_dn;  // 16-byte units per layer of each matrix
  const uint16_t* norms;    // [L][NORM_STRIDE] bf16
  const uint16_t* final_norm;
  uint16_t* kv;             // K caches [B][L][NKV][s_pad][D]
  uint16_t* kvt;            // V^T caches [B][L][NKV][s_pad/32][D][32]
  long long kv_seq;         // elements per sequence in each region
  float* kscale;            // FP8 cache (null: bf16): power-of-two scale per K row and per V
  float* vscale;            //   row, [B][L][NKV][s_pad]; codes at byte index = element index
  long long sc_seq;         // scales per sequence
  int s_pad;
  // activations, per slot (x_slot .. act_slot below: L + 1 slots of x / xg /
  // ssq, L of qkv / att / act; the per-phase kernels use slot 0)
  float* x;                 // [slot][2 consumers][H/16][BMAX][16] residual streams (x_at)
  uint16_t* xg;             // [slot][2 consumers][2 planes][H/32][64][8] x * gain as bf16 hi / lo parts (unit_at):
                            //   consumer 0 = attn_norm of the next QKV (or final_norm), 1 = ffn_norm
  float* ssq;               // [slot][2 consumers][H/16][BMAX] sums of squares of x per 16-row block
  float* qkv;               // [slot][BMAX][QKV] raw projections (a prefill: q normalised and rotated, k / v
                            //   only in the cache; qkv_head)
  uint16_t* att;            // [slot][2][QD/32][64][8] merged attention output, bf16 hi / lo parts
  uint16_t* act;            // [slot][2][F/32][64][8] SiLU(g) * u, bf16 hi / lo parts
  float* part;              // [BMAX][NKV][nsplit_max][PW] attention partials (a prefill: PC_WG of PC_PW floats)
  int* cnt;                 // [BMAX][NKV] finished splits of the current layer (a prefill: [NKV] per group)
  float* gpart;             // split-K partial block sums of the GEMM kernels
  int* gcnt;                // [256] finished K splits per 16-row block
  u64* keys;                // [BMAX] argmax keys of the step
  int* tok;                 // [BMAX] input tokens of the step
  int* pos;                 // [BMAX] position of the step's token
  int* out;                 // [max_steps][BMAX] produced tokens
  int* step;                // step counter (row of out)
  float* dbg_logits;        // optional [BMAX][V]
  const float* inv_freq;    // [D/2]
  float* rope;              // [BMAX][2][D/2] cos / sin of the step's position per sequence
  int* flags;               // bk_step: [L][FC_N][FLAG_MAX] hand-off flags (epoch of the last write)
  int* epoch;               // step epoch: bk_embed adds one per step, never reset
  u64* trace;               // bk_step (optional): [L][TR_N][G] device wall-clock stamps per workgroup
  int* err;                 // bk_step: MK_ERR_TIMEOUT when a hand-off wait gave up
  unsigned long long timeout_ticks;  // bk_step: wall-clock ticks a hand-off wait may take
  int B, L, V, nsplit_max, max_steps;
};

// Up to PG_MAX column groups that share one pass over the weights: a prefill
// pass of up to 1,024 prompt tokens is up to 64 groups of 16 columns, each
// with its own activation buffers, tokens and positions (the decode step is
// one group).
// Every kernel takes the group as blockIdx.y; the GEMM workgroups of one
// 16-row block differ in blockIdx.y only, so they run on one XCD (grid x a
// multiple of 8) at about the same time and share the block's weights
// through that XCD's L2.
constexpr int PG_MAX = 64;
template <int N>
struct PGroupN {  // groups in the kernel argument
  static constexpr int NG = N;
  BParams p[N];
  int n;  // groups in use, 1 .. N
};
using PGroup1 = PGroupN<1>;  // the decode step
// A prefill pass: group 0's parameters; group gi's activation buffers (x, xg,
// ssq, qkv, att, act, cnt, keys, rope) sit gi * gstride bytes after group 0's,
// its tokens and positions 16 gi entries after them.  part is one buffer for
// all groups; the GEMMs run the whole K and need no gpart / gcnt.
struct PGroup {
  static constexpr int NG = PG_MAX;
  BParams p;
  long long gstride;
  int n, ntok;  // groups and tokens of the pass
  int pos0;     // position of the pass's first token (group gi starts at pos0 + 16 gi)
};

template <class T>
__host__ __device__ __forceinline__ T* advance(T* q, long long bytes) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(q) + bytes);
}
// The parameters of column group gi of a pass (host and device), and of the
// workgroup's column group (blockIdx.y).
__host__ __device__ __forceinline__ BParams group_params(const PGroup& g, int gi) {
  const long long o = gi * g.gstride;
  BParams q = g.p;
  q.x = advance(q.x, o), q.xg = advance(q.xg, o), q.ssq = advance(q.ssq, o), q.qkv = advance(q.qkv, o);
  q.att = advance(q.att, o), q.act = advance(q.act, o), q.cnt = advance(q.cnt, o);
  q.keys = advance(q.keys, o), q.rope = advance(q.rope, o);
  q.tok += BMAX * gi, q.pos += BMAX * gi;
  q.B = g.ntok - BMAX * gi < BMAX ? g.ntok - BMAX * gi : BMAX;
  return q;
}
__device__ __forceinline__ const BParams& group_of(const PGroup1& g) { return g.p[0]; }
__device__ __forceinline__ BParams group_of(const PGroup& g) { return group_params(g, blockIdx.y); }

// ------------------------------------------------------------ helpers
// bf16 parts of an fp32 value: hi = RNE(v), lo = RNE(v - hi).
__device__ __forceinline__ void split2(float v, uint16_t& hi, uint16_t& lo) {
  hi = f32_to_bf16(v);
  lo = f32_to_bf16(v - bf16_to_f32(hi));
}

// u32x4 holding 8 bf16 with element e (0..7) replaced by v, in registers.
__device__ __forceinline__ u32x4 with_bf16(u32x4 x, int e, uint16_t v) {
  const unsigned keep = (e & 1) ? 0x0000ffffu : 0xffff0000u;
  const unsigned put = (e & 1) ? ((unsigned)v << 16) : (unsigned)v;
  u32x4 r = x;
#pragma unroll
  for (int c = 0; c < 4; ++c) r[c] = (c == (e >> 1)) ? ((x[c] & keep) | put) : x[c];
  return r;
}

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                 0, 0, 0);
}

// RMSNorm (reference rmsnorm.cuh:87-108) without a normalisation pass: the
// kernel that produces x also publishes x * gain as bf16 hi / lo parts (the B
// operand of the consuming product) and, per 16-row block and sequence, the
// sum of squares of its rows.  The consumer sums the H/16 partials in a fixed
// order, r_b = rsqrt(mean(x_b^2) + eps), and scales its outputs by r_b:
// W . (x * gain * r) = r * (W . (x * gain)).
// Activation slots.  The one-kernel step (bk_step) gives every layer its own
// copy of each activation buffer, so that within a launch every address is
// written once, before anything reads it: readers then use ordinary cached
// loads -- no cache can hold a stale copy, since every kernel starts with
// invalidated caches -- and only the writers' stores are write-through.  The
// per-phase kernels use slot 0 throughout (kernel boundaries order them).
// Slot s of x / xg / ssq holds, as consumer c = 0, the hidden state entering
// layer s with its attention-norm parts (s = L: the final-norm parts), and as
// c = 1 the state after layer s's O projection with its FFN-norm parts.
template <class S>
__device__ __forceinline__ float* x_slot(const BParams& p, int slot, int c) {
  return p.x + ((long long)(2 * slot + c) * BMAX) * S::H;
}
template <class S>
__device__ __forceinline__ uint16_t* xg_plane(const BParams& p, int slot, int c, int lohi) {
  return p.xg + ((long long)(4 * slot + 2 * c + lohi) * BMAX) * S::H;
}
template <class S>
__device__ __forceinline__ float* ssq_slot(const BParams& p, int slot, int c) {
  return p.ssq + (long long)(2 * slot + c) * (S::H / 16) * BMAX;
}
template <class S>
__device__ __forceinline__ float* qkv_slot(const BParams& p, int slot) {
  return p.qkv + (long long)slot * BMAX * S::QKV;
}
template <class S>
__device__ __forceinline__ uint16_t* att_slot(const BParams& p, int slot) {
  return p.att + (long long)slot * 2 * BMAX * S::QD;
}
template <class S>
__device__ __forceinline__ uint16_t* act_slot(const BParams& p, int slot) {
  return p.act + (long long)slot * 2 * BMAX * S::F;
}

// Layouts of the activations inside a slot (K columns, up to 16 sequences or
// tokens n).  The bf16 planes that feed a product (xg, att, act) are stored as
// its B operand: 1 KiB units of 32 k's, lane (k / 8 % 4) * 16 + n holding 8
// consecutive k's of column n, so a wave loads a unit with one contiguous
// 16-byte load per lane and an epilogue lane, which holds four rows of one
// column, stores 8 bytes.  (Row-major planes cost a load instruction 16 lines
// at a 2 KiB stride and an epilogue four 2-byte stores per plane.  With units a
// 1,024-token prefill went from 4.02 to 3.41 ms -- gate / up 39 -> 34, down 32
// -> 24, O 19 -> 12 us per layer -- and a batched step's QKV, O, gate / up and
// down from 5.0, 5.5, 6.6 and 7.2 to 4.6, 4.8, 5.1 and 6.3 us.)  The fp32 residual stream holds the
// 16 rows of a block per column, one 16-byte access per epilogue lane.
__device__ __forceinline__ int unit_at(int n, int k) { return ((k >> 5) * 64 + ((k >> 3) & 3) * 16 + n) * 8 + (k & 7); }
__device__ __forceinline__ void st4(uint16_t* a, const uint16_t (&v)[4]) {
  *reinterpret_cast<u32x2*>(a) = u32x2{v[0] | (unsigned)v[1] << 16, v[2] | (unsigned)v[3] << 16};
}
__device__ __forceinline__ int x_at(int n, int row) { return ((row >> 4) * BMAX + n) * 16 + (row & 15); }

// Epilogue of an x-producing 16-row block: thread t < 256 holds the new x of
// row rb * 16 + t / 16, sequence t % 16.  red: >= 256 floats of LDS.
// Stores of activations handed between workgroups: ordinary between kernels
// (SC1 false); inside the one-kernel step write-through at agent scope, and
// flagged on p.flags once acknowledged.
template <bool SC1, class T>
__device__ __forceinline__ void st_act(T* a, T v) {
  if constexpr (SC1) __hip_atomic_store(a, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *a = v;
}

template <class S, bool SC1 = false>
__device__ __forceinline__ void publish_x(const BParams& p, int slot, int c, const uint16_t* gain, int rb, float xn,
                                          float* red) {
  const int t = ltid(), row = rb * 16 + t / 16, b = t % 16;
  if (t < 256) {
    const bool on = b < p.B;
    if (on) {
      st_act<SC1>(x_slot<S>(p, slot, c) + x_at(b, row), xn);
      uint16_t h, o;
      split2(xn * bf16_to_f32(gain[row]), h, o);
      st_act<SC1>(xg_plane<S>(p, slot, c, 0) + unit_at(b, row), h);
      st_act<SC1>(xg_plane<S>(p, slot, c, 1) + unit_at(b, row), o);
    }
    red[t] = on ? xn * xn : 0.f;
  }
  __syncthreads();
  if (t < BMAX) {
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) ss += red[r * 16 + t];
    st_act<SC1>(ssq_slot<S>(p, slot, c) + (long long)rb * BMAX + t, ss);
  }
}

// r_b of slot / consumer c for b < BMAX into rr[0 .. BMAX) (read after a
// later barrier).  rr: RR_N floats of LDS; every thread of the workgroup
// calls this.  Sixteen threads per sequence each sum a run of the H/16 block
// sums (all their loads in flight together), then one thread per sequence
// adds the sixteen runs in order.
constexpr int RR_N = BMAX + 256;
template <class S>
__device__ __forceinline__ void rnorm(const BParams& p, int slot, int c, float* rr) {
  constexpr int NB = S::H / 16, PER = (NB + 15) / 16;
  const int t = ltid();
  if (t < 256) {
    const int b = t % 16, k = t / 16;
    const float* q = ssq_slot<S>(p, slot, c) + b;
    float v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = k * PER + i < NB ? q[(k * PER + i) * BMAX] : 0.f;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) sum += v[i];
    rr[BMAX + t] = sum;
  }
  __syncthreads();
  if (t < BMAX) {
    float ss = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) ss += rr[BMAX + k * 16 + t];
    rr[t] = rsqrtf(ss / (float)S::H + kRmsEps);
  }
}

// This wave's tiles of one 16-row block (tiles kt = w, w + GW, ... of KT),
// loaded into registers: the A operands of the block product.  Issued before
// the activations are staged, so the two latencies overlap.
template <int NT>
struct ATiles {  // NT tiles of a K range; wave w holds local tiles w, w + GW, ...
  static constexpr int TW = (NT + GW - 1) / GW;
  u32x4 t[TW];
};
template <int NT>
__device__ __forceinline__ void load_tiles(ATiles<NT>& a, const u32x4* __restrict__ blk, int kt0) {
  const unsigned l = lane_id();
  const int w = wave_id();
  const auto rs = make_rsrc(blk);
#pragma unroll
  for (int j = 0; j < ATiles<NT>::TW; ++j)
    a.t[j] = w + GW * j < NT ? buf_ld_nt(rs, l * 16u, (unsigned)(kt0 + w + GW * j) * 1024u) : u32x4{0u, 0u, 0u, 0u};
}

// The 16 activation columns of this wave's tiles: the B operands, from the
// planes' units (unit_at).  Loaded on their own, so
// a block can issue its other loads (norm sums, residual) before it waits.
template <int NT>
struct BCols {
  u32x4 h[ATiles<NT>::TW], l[ATiles<NT>::TW];
};
template <int NT>
__device__ __forceinline__ void load_cols(BCols<NT>& c, const uint16_t* hi, const uint16_t* lo, int kt0) {
  const int w = wave_id(), bo = 8 * (int)lane_id();
#pragma unroll
  for (int j = 0; j < ATiles<NT>::TW; ++j) {
    const int kt = kt0 + w + GW * j;
    if (w + GW * j < NT) {
      c.h[j] = *reinterpret_cast<const u32x4*>(hi + bo + 512 * kt);
      c.l[j] = *reinterpret_cast<const u32x4*>(lo + bo + 512 * kt);
    }
  }
}

// The tiles times the columns.  Lane (kg, n) returns rows 4 kg .. 4 kg + 3 of
// column n (this wave's share of the K sum).
template <int NT>
__device__ __forceinline__ f32x4 tiles_mma(const ATiles<NT>& a, const BCols<NT>& c) {
  const int w = wave_id();
  f32x4 a0 = f32x4{0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
  for (int j = 0; j < ATiles<NT>::TW; ++j) {
    if (w + GW * j < NT) {
      a0 = mfma(a.t[j], c.h[j], a0);
      a1 = mfma(a.t[j], c.l[j], a1);
    }
  }
  return a0 + a1;
}

// Two blocks' tiles (gate and up) times the same columns; each result equals
// tiles_mma of that block.
template <int NT>
__device__ __forceinline__ void tiles_mma2(const ATiles<NT>& a, const ATiles<NT>& b, const BCols<NT>& c, f32x4& ra,
                                           f32x4& rb) {
  const int w = wave_id();
  f32x4 a0 = f32x4{0.f, 0.f, 0.f, 0.f}, a1 = a0, b0 = a0, b1 = a0;
#pragma unroll
  for (int j = 0; j < ATiles<NT>::TW; ++j) {
    if (w + GW * j < NT) {
      a0 = mfma(a.t[j], c.h[j], a0);
      a1 = mfma(a.t[j], c.l[j], a1);
      b0 = mfma(b.t[j], c.h[j], b0);
      b1 = mfma(b.t[j], c.l[j], b1);
    }
  }
  ra = a0 + a1;
  rb = b0 + b1;
}

// K splits of a 16-row block run on KS workgroups; each publishes its block
// sums (thread t < 256: row t / 16, column t % 16; NV values per thread) with
// write-through stores, and the workgroup that completes the block (an
// agent-scope counter) adds the KS partials in split order -- the same sum in
// every run -- and runs the epilogue.  Returns true in that workgroup, with
// v[] replaced by the totals.  `last`: one int of LDS.
template <int NV>
__device__ __forceinline__ bool splitk_finish(const BParams& p, int rb, int ks, int KS, float (&v)[NV], int* last) {
  if (KS == 1) return true;  // one workgroup per block: its sums are the totals
  const int t = ltid();
  float* buf = p.gpart + ((long long)rb * KS) * 256 * NV;
  if (t < 256) {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      __hip_atomic_store(buf + ((long long)ks * NV + i) * 256 + t, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the partial is acknowledged before the count moves
  __syncthreads();
  if (t == 0) {
    const int done = __hip_atomic_fetch_add(p.gcnt + rb, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *last = done == KS - 1;
    if (*last) __hip_atomic_store(p.gcnt + rb, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-armed
  }
  __syncthreads();
  if (!*last) return false;
  if (t < 256) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      float sum = 0.f;
      for (int k = 0; k < KS; ++k)
        sum += __hip_atomic_load(buf + ((long long)k * NV + i) * 256 + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      v[i] = sum;
    }
  }
  return true;
}

// Cross-wave sum of a block's partial products: red[GW][16][17] in LDS.
// Returns, for thread t < 256, the total of row t / 16, column t % 16.
__device__ __forceinline__ float block_reduce(f32x4 acc, float* red) {
  const unsigned l = lane_id();
  const int w = wave_id();
  const int n = (int)(l & 15u), kg = (int)(l >> 4);
#pragma unroll
  for (int i = 0; i < 4; ++i) red[(w * 16 + 4 * kg + i) * 17 + n] = acc[i];
  __syncthreads();
  const int t = ltid();
  float s = 0.f;
  if (t < 256) {
#pragma unroll
    for (int ww = 0; ww < GW; ++ww) s += red[(ww * 16 + t / 16) * 17 + t % 16];
  }
  return s;
}

// ------------------------------------------------------------ kernels
// x[b] = E[tok[b]] (the tied embedding, gathered from the tile-layout LM head),
// published for layer 0's QKV.
template <class S, class G>
__global__ __launch_bounds__(256) void bk_embed(G pg) {
  __shared__ float xs[S::H];
  const BParams& p = group_of(pg);  // column group
  const int b = blockIdx.x;
  if (b >= BMAX) return;
  const int t = ltid();
  const bool on = b < p.B;
  const int t_ = on ? p.tok[b] : 0;
  const int tok = t_ < 0 ? 0 : (t_ >= p.V ? p.V - 1 : t_);  // tokens are validated on the host; never index outside
  for (int k = t; k < S::H; k += blockDim.x) {
    const int kt = k >> 5, q = (k >> 3) & 3, e = k & 7;
    const uint16_t* u = reinterpret_cast<const uint16_t*>(
        p.lmhead + ((long long)(tok >> 4) * S::KT_H + kt) * 64 + q * 16 + (tok & 15));
    const float xv = on ? bf16_to_f32(u[e]) : 0.f;
    xs[k] = xv;
    if (on) {
      x_slot<S>(p, 0, 0)[x_at(b, k)] = xv;
      uint16_t h, o;
      split2(xv * bf16_to_f32(p.norms[S::NORM_ATTN + k]), h, o);
      xg_plane<S>(p, 0, 0, 0)[unit_at(b, k)] = h;
      xg_plane<S>(p, 0, 0, 1)[unit_at(b, k)] = o;
    }
  }
  __syncthreads();
  for (int rb = t; rb < S::H / 16; rb += blockDim.x) {
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) ss += xs[rb * 16 + r] * xs[rb * 16 + r];
    ssq_slot<S>(p, 0, 0)[(long long)rb * BMAX + b] = ss;
  }
  if (t < S::D / 2) {  // RoPE angles of this step's position, shared by every layer
    float sn, cs;
    sincosf((float)(on ? p.pos[b] : 0) * p.inv_freq[t], &sn, &cs);
    p.rope[(b * 2 + 0) * (S::D / 2) + t] = cs;
    p.rope[(b * 2 + 1) * (S::D / 2) + t] = sn;
  }
  if (t == 0) p.keys[b] = 0ull;
  if (p.epoch && b == 0 && t == 0) *p.epoch += 1;  // this step's epoch for bk_step's hand-off flags
}

// Hand-off flag of producer `idx` of a phase of the one-kernel step: every
// thread's stores are acknowledged (write-through) before one thread writes
// the epoch.
__device__ __forceinline__ void fc_done(const BParams& p, int layer, int ph, int idx, int ep) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (ltid() == 0)
    __hip_atomic_store(p.flags + ((long long)layer * FC_N + ph) * FLAG_MAX + idx, ep, __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}

// Wait until the flags of producers 0 .. n - 1 of phase ph of `layer` hold
// epoch ep: wave 0 polls them (up to FLAG_MAX / 64 words per lane, all loads
// of a round in flight together), the workgroup follows; false when the
// wait gave up (p.err is set).
__device__ __forceinline__ bool fc_wait(const BParams& p, int layer, int ph, int n, int ep) {
  int ok = 1;
  if (wave_id() == 0) {
    const auto rs = make_rsrc(p.flags + ((long long)layer * FC_N + ph) * FLAG_MAX);
    const unsigned l = lane_id();
    Spin sp;
    while (true) {
      int v[FLAG_MAX / kWave];
#pragma unroll
      for (int k = 0; k < FLAG_MAX / kWave; ++k)
        v[k] = (int)l + kWave * k < n ? (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (l + kWave * k) * 4u, 0u, 16) : ep;
      bool ready = true;
#pragma unroll
      for (int k = 0; k < FLAG_MAX / kWave; ++k) ready &= v[k] == ep;
      if (__all(ready)) break;
      if (!sp.step(p.err, p.timeout_ticks)) {
        ok = 0;
        break;
      }
    }
  }
  return __syncthreads_and(ok) != 0;
}

// The GEMM phases as block functions.  FUSED (bk_step): the block's weight
// tiles are issued, then `ready()` waits for its inputs, which are read at
// agent scope, and the outputs are flagged on p.flags; otherwise (one kernel per
// phase) ready() is trivially true.  Each returns false only when ready()
// gave up.
struct NoWait {
  __device__ __forceinline__ bool operator()() const { return true; }
};

// rmsnorm(x) -> q|k|v rows of block rb for every sequence.
template <class S, bool FUSED, class Ready>
__device__ __forceinline__ bool qkv_block(const BParams& p, int layer, int ep, int rb, int ks, float* red, float* rr, int* last,
                                          const Ready& ready) {
  constexpr int NT = S::KT_H / KS_QKV;
  const int kt0 = ks * NT;
  ATiles<NT> a;
  load_tiles(a, p.wqkv + layer * p.u_qkv + (long long)rb * S::KT_H * 64, kt0);
  if (!ready()) return false;
  const int sl = FUSED ? layer : 0;
  BCols<NT> c;
  load_cols(c, xg_plane<S>(p, sl, 0, 0), xg_plane<S>(p, sl, 0, 1), kt0);
  rnorm<S>(p, sl, 0, rr);
  float v[1] = {block_reduce(tiles_mma(a, c), red)};
  if (!splitk_finish(p, rb, ks, KS_QKV, v, last)) return true;
  const int t = ltid(), row = rb * 16 + t / 16, b = t % 16;
  if (t < 256 && b < p.B) st_act<FUSED>(qkv_slot<S>(p, sl) + (long long)b * S::QKV + row, v[0] * rr[b]);
  if constexpr (FUSED) fc_done(p, layer, FC_QKV, rb, ep);
  return true;
}

// O projection + residual: x[b][row] += Wo[row] . att[b]; x published for the FFN norm.
template <class S, bool FUSED, class Ready>
__device__ __forceinline__ bool o_block(const BParams& p, int layer, int ep, int rb, int ks, float* red, int* last,
                                        const Ready& ready) {
  constexpr int NT = S::KT_Q / KS_O;
  const int kt0 = ks * NT;
  ATiles<NT> a;
  load_tiles(a, p.wo + layer * p.u_o + (long long)rb * S::KT_Q * 64, kt0);
  if (!ready()) return false;
  const int sl = FUSED ? layer : 0;
  const uint16_t* at = att_slot<S>(p, sl);
  BCols<NT> c;
  load_cols(c, at, at + BMAX * S::QD, kt0);
  const int t = ltid(), b = t % 16;
  const float xin = t < 256 && b < p.B ? x_slot<S>(p, sl, 0)[x_at(b, rb * 16 + t / 16)] : 0.f;
  float v[1] = {block_reduce(tiles_mma(a, c), red)};
  if (!splitk_finish(p, rb, ks, KS_O, v, last)) return true;
  const float xn = t < 256 && b < p.B ? xin + v[0] : 0.f;
  __syncthreads();  // red is reused
  publish_x<S, FUSED>(p, sl, 1, p.norms + (long long)layer * S::NORM_STRIDE + S::NORM_FFN, rb, xn, red);
  if constexpr (FUSED) fc_done(p, layer, FC_O, rb, ep);
  return true;
}

// rmsnorm(x) -> gate and up rows of block rb -> SiLU(g) * u parts.
template <class S, bool FUSED, class Ready>
__device__ __forceinline__ bool gu_block(const BParams& p, int layer, int ep, int rb, int ks, float* red, float* rr, int* last,
                                         const Ready& ready) {
  constexpr int NT = S::KT_H / KS_GU;
  const int kt0 = ks * NT;
  const long long off = (long long)rb * S::KT_H * 64;
  ATiles<NT> ag, au;
  load_tiles(ag, p.wg + layer * p.u_gu + off, kt0);
  load_tiles(au, p.wu + layer * p.u_gu + off, kt0);
  if (!ready()) return false;
  const int sl = FUSED ? layer : 0;
  BCols<NT> c;
  load_cols(c, xg_plane<S>(p, sl, 1, 0), xg_plane<S>(p, sl, 1, 1), kt0);
  rnorm<S>(p, sl, 1, rr);
  f32x4 pg, pu;
  tiles_mma2(ag, au, c, pg, pu);
  float v[2];
  v[0] = block_reduce(pg, red);
  __syncthreads();
  v[1] = block_reduce(pu, red);
  if (!splitk_finish(p, rb, ks, KS_GU, v, last)) return true;
  const int t = ltid(), row = rb * 16 + t / 16, b = t % 16;
  if (t < 256 && b < p.B) {
    const float g = v[0] * rr[b], u = v[1] * rr[b];
    uint16_t h, o;
    split2(g / (1.0f + __expf(-g)) * u, h, o);  // SiLU(g) * u (reference utils.cuh:59-61)
    st_act<FUSED>(act_slot<S>(p, sl) + unit_at(b, row), h);
    st_act<FUSED>(act_slot<S>(p, sl) + BMAX * S::F + unit_at(b, row), o);
  }
  if constexpr (FUSED) fc_done(p, layer, FC_GU, rb, ep);
  return true;
}

// Down projection + residual: x[b][row] += Wd[row] . act[b]; x published for
// the next layer's attention norm (the final norm after the last layer).
template <class S, bool FUSED, class Ready>
__device__ __forceinline__ bool down_block(const BParams& p, int layer, int ep, int rb, int ks, float* red, int* last,
                                           const Ready& ready) {
  static_assert(S::KT_F % KS_DN == 0, "whole tiles per K split");
  constexpr int NT = S::KT_F / KS_DN;
  const int kt0 = ks * NT;
  ATiles<NT> a;
  load_tiles(a, p.wd + layer * p.u_dn + (long long)rb * S::KT_F * 64, kt0);
  if (!ready()) return false;
  const int sl = FUSED ? layer : 0;
  const uint16_t* ac = act_slot<S>(p, sl);
  BCols<NT> c;
  load_cols(c, ac, ac + BMAX * S::F, kt0);
  const int t = ltid(), b = t % 16;
  // the residual, read by the workgroup that finishes the block (split 0 in
  // the one-kernel step, whichever split completes it otherwise)
  const float xin = (!FUSED || ks == 0) && t < 256 && b < p.B
                        ? x_slot<S>(p, sl, 1)[x_at(b, rb * 16 + t / 16)]
                        : 0.f;
  float v[1] = {block_reduce(tiles_mma(a, c), red)};
  if constexpr (FUSED) {
    // K splits 1.. publish their sums as (value, tag) words; split 0 polls
    // them and adds the splits in order, as splitk_finish does
    u64* buf = reinterpret_cast<u64*>(p.gpart) + (long long)rb * KS_DN * 256;
    const unsigned tag = (unsigned)ep * 64u + (unsigned)layer;
    if (ks != 0) {
      if (t < 256) __hip_atomic_store(buf + ks * 256 + t, ((u64)tag << 32) | f32_bits(v[0]), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
      return true;
    }
    int ok = 1;
    if (t < 256) {
      u64 wv[KS_DN - 1];
      Spin sp;
      while (true) {
        bool all = true;
#pragma unroll
        for (int k = 1; k < KS_DN; ++k) {
          wv[k - 1] = __hip_atomic_load(buf + k * 256 + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          all &= (unsigned)(wv[k - 1] >> 32) == tag;
        }
        if (all) break;
        if (!sp.step(p.err, p.timeout_ticks)) {
          ok = 0;
          break;
        }
      }
      float sum = 0.f;
      sum += v[0];
#pragma unroll
      for (int k = 1; k < KS_DN; ++k) sum += f32_from((unsigned)wv[k - 1]);
      v[0] = sum;
    }
    if (!__syncthreads_and(ok)) return false;
  } else if (!splitk_finish(p, rb, ks, KS_DN, v, last)) {
    return true;
  }
  const float xn = t < 256 && b < p.B ? xin + v[0] : 0.f;
  __syncthreads();  // red is reused
  const uint16_t* gain = layer + 1 < p.L ? p.norms + (long long)(layer + 1) * S::NORM_STRIDE + S::NORM_ATTN
                                         : p.final_norm;
  publish_x<S, FUSED>(p, FUSED ? layer + 1 : 0, 0, gain, rb, xn, red);
  if constexpr (FUSED) fc_done(p, layer, FC_DN, rb, ep);
  return true;
}

template <class S>
__global__ __launch_bounds__(GT) void bk_qkv(PGroup1 p, int layer) {
  __shared__ float red[GW * 16 * 17];
  __shared__ float rr[RR_N];
  __shared__ int last;
  qkv_block<S, false>(group_of(p), layer, 0, blockIdx.x / KS_QKV, blockIdx.x % KS_QKV, red, rr, &last, NoWait{});
}

template <class S>
__global__ __launch_bounds__(GT) void bk_o(PGroup1 p, int layer) {
  __shared__ float red[GW * 16 * 17];
  __shared__ int last;
  o_block<S, false>(group_of(p), layer, 0, blockIdx.x / KS_O, blockIdx.x % KS_O, red, &last, NoWait{});
}

template <class S>
__global__ __launch_bounds__(GT) void bk_gu(PGroup1 p, int layer) {
  __shared__ float red[GW * 16 * 17];
  __shared__ float rr[RR_N];
  __shared__ int last;
  gu_block<S, false>(group_of(p), layer, 0, blockIdx.x / KS_GU, blockIdx.x % KS_GU, red, rr, &last, NoWait{});
}

template <class S>
__global__ __launch_bounds__(GT) void bk_down(PGroup1 p, int layer) {
  __shared__ float red[GW * 16 * 17];
  __shared__ int last;
  down_block<S, false>(group_of(p), layer, 0, blockIdx.x / KS_DN, blockIdx.x % KS_DN, red, &last, NoWait{});
}

// ------------------------------------------------------------ prefill GEMMs
// A pass has 1 to 64 column groups.  A workgroup of W waves computes MR row
// blocks (gate / up: block pairs of 16 gate + 16 up rows) x NG groups over the
// whole K, split over its waves: wave w takes the 1 KiB units w, w + W, ... of
// every row block and column plane, straight into registers (weights as the A
// operand, the columns' bf16 hi / lo parts as two B operands of one
// accumulator), NBUF chunks of CW units in flight.  The waves' sums meet in
// LDS once, in wave order, and each wave runs the epilogue of its share of the
// tiles: QKV scales by the group's norm factor and finishes whole heads
// (qkv_head), gate / up applies SiLU, O and down add the residual and publish
// x (the next norm's parts and per-block sums of squares) as publish_x does;
// the epilogue's inputs are loaded before the product.
//
// What bounds it: a short pass the latency of one load round per kernel (23
// tokens: 5 - 7 us per GEMM, a kernel's fixed cost about 4), a long one the
// bytes that cross L2 per product.  No barrier and no LDS copy stands between
// a load and its product, and a wave's loads are all independent, so a
// workgroup keeps 64 - 256 KiB in flight.  The kernels before this staged both
// operands in LDS by chunks of K, with a barrier per chunk: every chunk waited
// for its loads (0.5 - 1.2 us each, 16 to 32 in a row).  us per layer inside
// whole passes (kernel trace), the LDS-tiled kernels on row-major planes -> now
// (QKV: before, its append kernel added; now, with the head epilogue):
//                    2 groups      13            32            64
//   QKV             14.4 -> 7.0   15.0 -> 8.1   15.6 -> 9.4   21.6 -> 14.7
//   O               11.6 -> 5.0   12.2 -> 5.2   12.7 -> 7.3   18.6 -> 10.5
//   gate / up       20.7 -> 7.0   26.6 -> 12.8  31.1 -> 18.0  38.2 -> 30.8
//   down            25.6 -> 7.1   24.8 -> 9.7   25.9 -> 13.3  31.5 -> 20.3
template <int MR_, int NG_, int CW_, int NBUF_, int W_>
struct PTile {
  static constexpr int MR = MR_, NG = NG_, CW = CW_, NBUF = NBUF_, W = W_;
};
enum PtOp : int { PT_QKV = 0, PT_O = 1, PT_DN = 2, PT_GU = 3 };
// One head (D = 64 rows, four row blocks) of the fused QKV product for the 16
// columns of a group, in one wave: lane (kg, n) holds rows 16 r + 4 kg + i of
// column n in v[r][i], so a head's sum of squares takes two cross-lane steps
// and a RoPE pair (d, d + 32) sits in one lane.  q: RMSNorm and RoPE (reference
// rmsnorm.cuh:57-84, attention.cuh:22-44), fp32 for the attention; k the same,
// then into the cache like v (reference kv_cache.cuh:58-78) -- before the
// attention kernel, so that a column sees the columns before it.  (A kernel of
// its own for k and v took 4.0 - 5.6 us per layer, and every attention
// workgroup normalised and rotated its queries again: 1,024 tokens 3,277 us,
// and 2,905 with both here.)
struct HeadIn {
  f32x4 cs[2], sn[2];  // RoPE cos / sin of dims 16 r + 4 kg + i, r = 0, 1
  u32x2 gain[4];       // QK-norm gains of the lane's rows
};
template <class S>
__device__ __forceinline__ void head_load(const BParams& p, int layer, int head, int n, int kg, HeadIn& in) {
  static_assert(S::D == 64, "heads of four row blocks");
  const uint16_t* g = p.norms + (long long)layer * S::NORM_STRIDE + (head < S::NQ ? S::NORM_Q : S::NORM_K);
#pragma unroll
  for (int r = 0; r < 4; ++r) in.gain[r] = *reinterpret_cast<const u32x2*>(g + 16 * r + 4 * kg);
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    in.cs[r] = *reinterpret_cast<const f32x4*>(p.rope + (n * 2 + 0) * (S::D / 2) + 16 * r + 4 * kg);
    in.sn[r] = *reinterpret_cast<const f32x4*>(p.rope + (n * 2 + 1) * (S::D / 2) + 16 * r + 4 * kg);
  }
}
template <class S>
__device__ __forceinline__ void qkv_head(const BParams& p, int layer, int head, int n, int kg, bool on, const HeadIn& in,
                                         f32x4 (&v)[4]) {
  constexpr int D = S::D;
  if (head < S::NQ + S::NKV) {
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) ss += v[r][i] * v[r][i];
    ss = sum_xor32(sum_xor16(ss));
    const float rn = rsqrtf(ss / (float)D + kRmsEps);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[r][i] = v[r][i] * rn * bf16_to_f32((uint16_t)(in.gain[r][i / 2] >> (16 * (i & 1))));
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a = v[r][i], b = v[r + 2][i];
        v[r][i] = a * in.cs[r][i] - b * in.sn[r][i];
        v[r + 2][i] = b * in.cs[r][i] + a * in.sn[r][i];
      }
  }
  if (head < S::NQ) {
    if (!on) return;
    float* q = qkv_slot<S>(p, 0) + (long long)n * S::QKV + head * D + 4 * kg;
#pragma unroll
    for (int r = 0; r < 4; ++r) *reinterpret_cast<f32x4*>(q + 16 * r) = v[r];
    return;
  }
  const bool isk = head < S::NQ + S::NKV;
  const int g = head - S::NQ - (isk ? 0 : S::NKV);
  const int pos = on ? p.pos[n] : 0;
  const long long base = ((long long)layer * S::NKV + g) * (long long)p.s_pad;
  const long long at = isk ? (base + pos) * D + 4 * kg : (base + pos / 32 * 32) * D + (long long)(4 * kg) * 32 + pos % 32;
  if (p.kscale) {  // FP8 row: codes and the power-of-two scale from the row's maximum
    float m = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) m = fmaxf(m, fabsf(v[r][i]));
    const int e = e4m3_row_exp(max_xor32(max_xor16(m)));
    if (!on) return;
    uint8_t* c = reinterpret_cast<uint8_t*>(isk ? p.kv : p.kvt) + at;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      uint8_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = (uint8_t)e4m3_encode(ldexpf(v[r][i], -e));
      if (isk) {
        *reinterpret_cast<uint32_t*>(c + 16 * r) = b[0] | (unsigned)b[1] << 8 | (unsigned)b[2] << 16 | (unsigned)b[3] << 24;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) c[(16 * r + i) * 32] = b[i];
      }
    }
    if (kg == 0) (isk ? p.kscale : p.vscale)[base + pos] = ldexpf(1.f, e);
  } else if (on) {
    uint16_t* c = (isk ? p.kv : p.kvt) + at;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      uint16_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = f32_to_bf16(v[r][i]);
      if (isk) {
        st4(c + 16 * r, b);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) c[(16 * r + i) * 32] = b[i];
      }
    }
  }
}

template <class S, int OP, class T>
__global__ __launch_bounds__(T::W * kWave) void bk_pgemm(PGroup pg, int layer) {
  constexpr int MR = T::MR, NGW = T::NG, W = T::W;
  constexpr bool GU = OP == PT_GU;
  constexpr int NB = GU ? 2 : 1;  // blocks per row tile
  constexpr int K = OP == PT_O ? S::QD : (OP == PT_DN ? S::F : S::H);
  constexpr int NT = K / 32, TW = NT / W, CW = T::CW < TW ? T::CW : TW;
  constexpr int NCH = (TW + CW - 1) / CW, NBUF = T::NBUF < NCH ? T::NBUF : NCH;
  static_assert(NT % W == 0, "whole units per wave");
  // epilogue units of a wave: one row tile, or for QKV one head, of a group
  constexpr int RU = OP == PT_QKV ? 4 : 1, MU = MR / RU;
  static_assert(MR % RU == 0, "whole heads");
  constexpr int TL = MU * NGW, TPW = (TL + W - 1) / W;
  __shared__ f32x4 red[W][MR * NGW][NB][kWave];
  const int rb0 = blockIdx.x * MR, g0 = blockIdx.y * NGW;
  const int ngr = pg.n - g0 < NGW ? pg.n - g0 : NGW;
  const int w = wave_id(), l = (int)lane_id();
  const int n = l & 15, kg = l >> 4;
  const BParams p0 = group_params(pg, g0);
  const long long gs = pg.gstride;
  const u32x4* wm[NB];
  if constexpr (GU) wm[0] = p0.wg + layer * p0.u_gu, wm[1] = p0.wu + layer * p0.u_gu;
  else wm[0] = OP == PT_QKV ? p0.wqkv + layer * p0.u_qkv : (OP == PT_O ? p0.wo + layer * p0.u_o : p0.wd + layer * p0.u_dn);
  const uint16_t* pl = OP == PT_QKV ? xg_plane<S>(p0, 0, 0, 0)
                                    : (GU ? xg_plane<S>(p0, 0, 1, 0) : (OP == PT_O ? att_slot<S>(p0, 0) : act_slot<S>(p0, 0)));
  // the epilogue's inputs first: the norm's block sums, or the residual rows
  constexpr bool NORM = OP == PT_QKV || GU;
  constexpr int NSB = S::H / 16, PER = NSB / 4;
  constexpr int CI = OP == PT_O ? 0 : 1, CO = 1 - CI;
  float sv[NORM ? TPW : 1][PER];
  f32x4 xr[TPW];
  u32x2 gw[TPW];
  HeadIn hin[OP == PT_QKV ? TPW : 1];
  const uint16_t* gain = OP == PT_O ? p0.norms + (long long)layer * S::NORM_STRIDE + S::NORM_FFN
                                    : (layer + 1 < p0.L ? p0.norms + (long long)(layer + 1) * S::NORM_STRIDE + S::NORM_ATTN
                                                        : p0.final_norm);
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int t = w + W * i, j = t / MU < ngr ? t / MU : 0;
    if constexpr (OP == PT_QKV) head_load<S>(group_params(pg, g0 + j), layer, rb0 / RU + t % MU, n, kg, hin[i]);
    if constexpr (NORM) {
      const float* q = advance(ssq_slot<S>(p0, 0, GU ? 1 : 0), j * gs) + n;
#pragma unroll
      for (int e = 0; e < PER; ++e) sv[i][e] = q[(kg * PER + e) * BMAX];
    } else {
      const int row = (rb0 + t % MU) * 16 + 4 * kg;
      xr[i] = *reinterpret_cast<const f32x4*>(advance(x_slot<S>(p0, 0, CI), j * gs) + x_at(n, row));
      gw[i] = *reinterpret_cast<const u32x2*>(gain + row);
    }
  }
  f32x4 acc[MR][NB][NGW];
#pragma unroll
  for (int r = 0; r < MR; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < NGW; ++j) acc[r][b][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 a[NBUF][CW][MR][NB], bh[NBUF][CW][NGW], bl[NBUF][CW][NGW];
  const auto issue = [&](int c, int q) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < CW; ++u) {
      if (c * CW + u >= TW) break;
      const int kt = w + W * (c * CW + u);
#pragma unroll
      for (int r = 0; r < MR; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b) a[q][u][r][b] = *(wm[b] + ((long long)(rb0 + r) * NT + kt) * 64 + l);
#pragma unroll
      for (int j = 0; j < NGW; ++j) {
        const uint16_t* s = pl + (j < ngr ? j : 0) * (gs / 2) + 512 * kt + 8 * l;
        bh[q][u][j] = *reinterpret_cast<const u32x4*>(s);
        bl[q][u][j] = *reinterpret_cast<const u32x4*>(s + BMAX * K);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int c = 0; c < NBUF; ++c) issue(c, c);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int q = c % NBUF;
#pragma unroll
    for (int u = 0; u < CW; ++u) {
      if (c * CW + u >= TW) break;
#pragma unroll
      for (int r = 0; r < MR; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int j = 0; j < NGW; ++j) acc[r][b][j] = mfma(a[q][u][r][b], bh[q][u][j], acc[r][b][j]);
#pragma unroll
      for (int r = 0; r < MR; ++r)
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int j = 0; j < NGW; ++j) acc[r][b][j] = mfma(a[q][u][r][b], bl[q][u][j], acc[r][b][j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (c + NBUF < NCH) issue(c + NBUF, q);
  }
#pragma unroll
  for (int r = 0; r < MR; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < NGW; ++j) red[w][j * MR + r][b][l] = acc[r][b][j];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int t = w + W * i, j = t / MU, rb = rb0 + t % MU * RU;
    if (t >= TL || j >= ngr) break;
    f32x4 v[RU][NB];
#pragma unroll
    for (int r = 0; r < RU; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int e = j * MR + t % MU * RU + r;
        v[r][b] = red[0][e][b][l];
#pragma unroll
        for (int k = 1; k < W; ++k) v[r][b] += red[k][e][b][l];
      }
    const BParams p = group_params(pg, g0 + j);
    const bool on = n < p.B;
    const int row = rb * 16 + 4 * kg;
    if constexpr (NORM) {
      float ss = 0.f;
#pragma unroll
      for (int e = 0; e < PER; ++e) ss += sv[i][e];
      ss = sum_xor32(sum_xor16(ss));
      const float rs = rsqrtf(ss / (float)S::H + kRmsEps);
      if constexpr (GU) {
        uint16_t h[4], o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = v[0][0][e] * rs, u = v[0][NB - 1][e] * rs;
          split2(g / (1.0f + __expf(-g)) * u, h[e], o[e]);  // SiLU(g) * u (reference utils.cuh:59-61)
        }
        if (on) {
          uint16_t* q = act_slot<S>(p, 0) + unit_at(n, row);
          st4(q, h);
          st4(q + BMAX * S::F, o);
        }
      } else {
        f32x4 hv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) hv[r] = v[r % RU][0] * rs;
        qkv_head<S>(p, layer, rb / 4, n, kg, on, hin[i], hv);
      }
    } else {
      f32x4 xn = xr[i] + v[0][0];
      uint16_t h[4], o[4];
      float sq = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (!on) xn[e] = 0.f;
        split2(xn[e] * bf16_to_f32((uint16_t)(gw[i][e / 2] >> (16 * (e & 1)))), h[e], o[e]);
        sq += xn[e] * xn[e];
      }
      if (on) {
        *reinterpret_cast<f32x4*>(x_slot<S>(p, 0, CO) + x_at(n, row)) = xn;
        st4(xg_plane<S>(p, 0, CO, 0) + unit_at(n, row), h);
        st4(xg_plane<S>(p, 0, CO, 1) + unit_at(n, row), o);
      }
      sq = sum_xor32(sum_xor16(sq));
      if (kg == 0) ssq_slot<S>(p, 0, CO)[(long long)rb * BMAX + n] = sq;
    }
  }
}

// Final rmsnorm -> tied LM head -> per-sequence argmax (reference
// sampling.cuh:32-117).  Each wave scores whole 16-row blocks; keys are
// ordered(logit) << 32 | (0xffffffff - index), combined with an atomic max, so
// the result is the largest logit and, among equal logits, the lowest index.
template <class S, bool F8 = false>
__global__ __launch_bounds__(GT) void bk_lm(BParams p, int slot) {
  // F8: the FP8 copy; a lane's 16 bytes (row l & 15, columns 64 u + 16 kg ..
  // + 15 of unit u) feed two MFMA k-steps, whose B operands take the same
  // columns of the hidden state; the row scale enters the conversion
  __shared__ __attribute__((aligned(16))) uint16_t hi[BMAX * S::H], lo[BMAX * S::H];  // B-operand units (unit_at)
  __shared__ u64 best_w[GW][BMAX];
  __shared__ float rr[RR_N];
  {  // the final-norm parts published by the last layer, copied to LDS
    const uint16_t *gh = xg_plane<S>(p, slot, 0, 0), *gl = xg_plane<S>(p, slot, 0, 1);
    for (int i = threadIdx.x; i < BMAX * S::H / 8; i += GT) {
      reinterpret_cast<u32x4*>(hi)[i] = reinterpret_cast<const u32x4*>(gh)[i];
      reinterpret_cast<u32x4*>(lo)[i] = reinterpret_cast<const u32x4*>(gl)[i];
    }
    rnorm<S>(p, slot, 0, rr);
  }
  __syncthreads();
  const unsigned l = lane_id();
  const int w = wave_id();
  const int n = (int)(l & 15u), kg = (int)(l >> 4);
  const int nb = p.V / 16;
  const int bo = 8 * (int)l;
  const float rn = rr[n];
  u64 best = 0ull;
  // the wave's blocks rb0, rb0 + stride, ... as a flat sequence of chunks of
  // U tiles; the next chunk's loads are issued before the current one's products
  constexpr int KT = F8 ? S::H / 64 : S::KT_H;  // 1 KiB units per 16-row block
  constexpr int U = KT < 8 ? KT : 8, CPB = KT / U;  // chunks per block
  static_assert(KT % U == 0, "whole chunks per block");
  const int rb0 = blockIdx.x * GW + w, stride = gridDim.x * GW;
  const int nblk = rb0 < nb ? (nb - 1 - rb0) / stride + 1 : 0;
  const int nch = nblk * CPB;
  u32x4 cur[U], nxt[U];
  auto load_chunk = [&](int c, u32x4* dst) {
    const int rb = rb0 + (c / CPB) * stride, k0 = (c % CPB) * U;
    const auto rs = make_rsrc((F8 ? p.lmhead8 : p.lmhead) + (long long)rb * KT * 64);
#pragma unroll
    for (int u = 0; u < U; ++u) dst[u] = buf_ld_nt(rs, l * 16u, (unsigned)(k0 + u) * 1024u);
  };
  if (nch > 0) load_chunk(0, cur);
  f32x4 a0 = f32x4{0.f, 0.f, 0.f, 0.f}, a1 = a0;
  for (int c = 0; c < nch; ++c) {
    if (c + 1 < nch) load_chunk(c + 1, nxt);
    const int k0 = (c % CPB) * U;
    if constexpr (F8) {
      const float sc = p.lm_scale[(long long)(rb0 + (c / CPB) * stride) * 16 + n];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kt = k0 + u;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const u32x4 wb = fp8x8_to_bf16x8_scaled(half ? u32x2{cur[u][2], cur[u][3]} : u32x2{cur[u][0], cur[u][1]}, sc);
          const int at = unit_at(n, 64 * kt + 16 * kg + 8 * half);
          a0 = mfma(wb, *reinterpret_cast<const u32x4*>(hi + at), a0);
          a1 = mfma(wb, *reinterpret_cast<const u32x4*>(lo + at), a1);
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int kt = k0 + u;
        a0 = mfma(cur[u], *reinterpret_cast<const u32x4*>(hi + bo + 512 * kt), a0);
        a1 = mfma(cur[u], *reinterpret_cast<const u32x4*>(lo + bo + 512 * kt), a1);
      }
    }
    if (c % CPB == CPB - 1) {  // the block is complete
      const int rb = rb0 + (c / CPB) * stride;
      const f32x4 acc = (a0 + a1) * rn;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const unsigned idx = (unsigned)(rb * 16 + 4 * kg + i);
        if (p.dbg_logits && n < p.B) p.dbg_logits[(long long)n * p.V + idx] = acc[i];
        const u64 key = ((u64)f32_order_key(acc[i]) << 32) | (u64)(0xffffffffu - idx);
        best = key > best ? key : best;
      }
      a0 = a1 = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < U; ++u) cur[u] = nxt[u];
  }
  // lanes n, n + 16, n + 32, n + 48 hold column n
#pragma unroll
  for (int m = 16; m <= 32; m <<= 1) {
    const u64 o = __shfl_xor(best, m);
    best = o > best ? o : best;
  }
  if (kg == 0) best_w[w][n] = best;
  __syncthreads();
  const int t = threadIdx.x;
  if (t < p.B) {
    u64 b = 0ull;
#pragma unroll
    for (int ww = 0; ww < GW; ++ww) b = best_w[ww][t] > b ? best_w[ww][t] : b;
    atomicMax(reinterpret_cast<unsigned long long*>(p.keys + t), (unsigned long long)b);
  }
}

// Tokens of the step from the argmax keys; positions advance.
__global__ void bk_tok(BParams p) {
  const int b = threadIdx.x;
  const int s = *p.step;
  if (b < p.B) {
    const int tok = (int)(0xffffffffu - (unsigned)(p.keys[b] & 0xffffffffull));
    p.tok[b] = tok;
    if (s < p.max_steps) p.out[(long long)s * BMAX + b] = tok;
    p.pos[b] += 1;
  }
  __syncthreads();
  if (b == 0) *p.step = s + 1;
}

// ------------------------------------------------------------ attention
// One item = (sequence b, kv head g, split s) of CH positions; wave w takes
// the 32-position block 4 s + w.  Both products of a block run on the matrix
// cores exactly as the batch-1 kernel does: scores^T = K . Qb with q split into
// three bf16 parts in rows 4 j + 0..2 (j = q head of the group), and
// out^T = V^T . Pb with the softmax weights split the same way.
template <class S>
struct AttnLds {
  static constexpr int D = S::D;
  float kcs[2];  // FP8: scales of position pos's K / V rows
  __attribute__((aligned(16))) uint16_t qb[16][D];       // q parts (A operand of the scores)
  __attribute__((aligned(16))) uint16_t pb[AW][16][32];  // weight parts (A operand of the output)
  __attribute__((aligned(16))) uint16_t kcur[D], vcur[D];  // K / V of position pos
  float rc[D / 2], rsn[D / 2];
  float mw[AW][2], lw[AW][2], ow[AW][2][D];
  float cm[AT / (2 * D)][2 * D], cl[AT / (2 * D)][2 * D], co[AT / (2 * D)][2 * D];  // split-group merge
  int last;
};

// K / V registers of one item: the wave's NBW 32-position blocks (4 s + w) +
// AW * q (blocks past the item repeat a valid block).  K8: the FP8 cache
// (codes converted to bf16 in registers, exact; the K row scale enters that
// conversion, the V row scale the softmax weight).
template <class S, bool K8>
struct AttnKV {
  using Reg = typename std::conditional<K8, u32x2, u32x4>::type;
  Reg kr[NBW][2][2], vr[NBW][S::D / 16];
  float sk[K8 ? NBW : 1][2], sv[K8 ? NBW : 1][2];  // FP8: scales of the lane's score positions
};
template <class S, bool K8>
__device__ __forceinline__ void attn_kv_load(const BParams& p, int layer, bool on, int b, int g, int s, int pos,
                                             AttnKV<S, K8>& r) {
  constexpr int D = S::D, NKV = S::NKV;
  const int n = on ? pos + 1 : 0;
  const int tid = ltid() % AT, w = tid / kWave, l = tid % kWave;
  const unsigned lu = (unsigned)l;
  const long long kbase = (long long)b * p.kv_seq + ((long long)layer * NKV + g) * (long long)p.s_pad * D;
  const long long sbase = (long long)b * p.sc_seq + ((long long)layer * NKV + g) * p.s_pad;
  if (!on) {  // no item: the registers hold nothing (no value carried from an earlier item)
#pragma unroll
    for (int q = 0; q < NBW; ++q) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) r.kr[q][h][kc] = __builtin_nondeterministic_value(r.kr[q][h][kc]);
        if constexpr (K8) {
          r.sk[q][h] = __builtin_nondeterministic_value(r.sk[q][h]);
          r.sv[q][h] = __builtin_nondeterministic_value(r.sv[q][h]);
        }
      }
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt) r.vr[q][dt] = __builtin_nondeterministic_value(r.vr[q][dt]);
    }
    return;
  }
#pragma unroll
  for (int q = 0; q < NBW; ++q) {
    int blk = s * AW * NBW + w + AW * q;
    blk = 32 * blk < n ? blk : s * AW * NBW;
    if constexpr (K8) {  // byte index = element index of the bf16 layout
      const auto rk = make_rsrc(reinterpret_cast<const uint8_t*>(p.kv) + kbase + (long long)blk * 32 * D);
      const auto rv = make_rsrc(reinterpret_cast<const uint8_t*>(p.kvt) + kbase + (long long)blk * 32 * D);
      const auto rks = make_rsrc(p.kscale + sbase + (long long)blk * 32);
      const auto rvs = make_rsrc(p.vscale + sbase + (long long)blk * 32);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
          r.kr[q][h][kc] =
              __builtin_amdgcn_raw_buffer_load_b64(rk, (16u * h + (lu & 15u)) * D + 32u * kc + 8u * (lu >> 4), 0u, 2);
        r.sk[q][h] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rks, (16u * h + (lu & 15u)) * 4u, 0u, 2));
        r.sv[q][h] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rvs, (16u * h + (lu & 15u)) * 4u, 0u, 2));
      }
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt)
        r.vr[q][dt] = __builtin_amdgcn_raw_buffer_load_b64(rv, (16u * dt + (lu & 15u)) * 32u + 8u * (lu >> 4), 0u, 2);
    } else {
      const auto rk = make_rsrc(p.kv + kbase + (long long)blk * 32 * D);
      const auto rv = make_rsrc(p.kvt + kbase + (long long)blk * 32 * D);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int kc = 0; kc < 2; ++kc)
          r.kr[q][h][kc] = __builtin_amdgcn_raw_buffer_load_b128(
              rk, ((16u * h + (lu & 15u)) * D + 32u * kc + 8u * (lu >> 4)) * 2u, 0u, 2);
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt)
        r.vr[q][dt] =
            __builtin_amdgcn_raw_buffer_load_b128(rv, ((16u * dt + (lu & 15u)) * 32u + 8u * (lu >> 4)) * 2u, 0u, 2);
    }
  }
}

// The item's code for AT threads (local thread threadIdx.x % AT).
// FUSED: inside bk_step, where the two AT-thread halves of a workgroup run
// two items and share every barrier: `on` false (a half without an item)
// passes the barriers only; the item reads its layer's qkv slot and writes
// its layer's att slot (write-through), flagged on p.flags.  Otherwise (bk_attn) one
// item per workgroup, always on.
// ready(): as for the GEMM blocks, between the K / V loads and the first read
// of q / k / v; the return is false only when it gave up.
template <class S, bool K8, bool FUSED, class Ready>
__device__ __forceinline__ bool attn_item(const BParams& p, int layer, int ep, AttnLds<S>& sm, bool on, int b, int g,
                                          int s, int nsplit, int pos, AttnKV<S, K8>& kv, const Ready& ready) {
  static_assert(S::GQA == 2 && S::D == 64, "batched attention is built for 2 q heads of 64 per kv head");
  constexpr int D = S::D, NKV = S::NKV;
  // K / V of the item's blocks are in kv (attn_kv_load, issued before)
  const int n = on ? pos + 1 : 0;
  const int tid = ltid() % AT, w = tid / kWave, l = tid % kWave;
  const int c16 = l & 15, rg = l >> 4;
  const long long kbase = (long long)b * p.kv_seq + ((long long)layer * NKV + g) * (long long)p.s_pad * D;
  const long long sbase = (long long)b * p.sc_seq + ((long long)layer * NKV + g) * p.s_pad;
  auto& kr = kv.kr;
  auto& vr = kv.vr;
  auto& sk = kv.sk;
  auto& sv = kv.sv;
  for (int i = tid; i < 16 * D; i += AT) (&sm.qb[0][0])[i] = 0;
  for (int i = tid; i < AW * 16 * 32; i += AT) (&sm.pb[0][0][0])[i] = 0;
  if (on && tid < D / 2) {
    sm.rc[tid] = p.rope[(b * 2 + 0) * (D / 2) + tid];
    sm.rsn[tid] = p.rope[(b * 2 + 1) * (D / 2) + tid];
  }
  if (!ready()) return false;
  __syncthreads();
  // 1. q heads (waves 0, 1), k (wave 2), v (wave 3) of position pos: QK-norm
  //    (reference rmsnorm.cuh:57-84) and RoPE rotate-half (attention.cuh:22-44)
  const int sl = FUSED ? layer : 0;
  const float* src = qkv_slot<S>(p, sl) + (long long)b * S::QKV +
                     (w < 2 ? (g * 2 + w) * D : (w == 2 ? S::QD + g * D : S::QD + S::KVD + g * D));
  const float v0 = on ? src[l] : 0.f;
  float v = v0;
  const bool own = on && pos >= s * CH && pos < (s + 1) * CH;
  if (on && w < 3) {
    const float ss = wave_sum(v * v);
    const uint16_t* gn = p.norms + (long long)layer * S::NORM_STRIDE + (w < 2 ? S::NORM_Q : S::NORM_K);
    v = v * rsqrtf(ss / (float)D + kRmsEps) * bf16_to_f32(gn[l]);
    const float partner = lane_xor32(v);
    const int d = l & 31;
    v = l < 32 ? v * sm.rc[d] - partner * sm.rsn[d] : v * sm.rc[d] + partner * sm.rsn[d];
    if (w < 2) {
      uint16_t h, m, o;
      split_bf16(v, h, m, o);
      sm.qb[4 * w + 0][l] = h;
      sm.qb[4 * w + 1][l] = m;
      sm.qb[4 * w + 2][l] = o;
    } else if constexpr (K8) {  // FP8 append: the row's power-of-two scale from the wave's max
      const int e = e4m3_row_exp(wave_max(fabsf(v)));
      const uint8_t code = (uint8_t)e4m3_encode(ldexpf(v, -e));
      reinterpret_cast<uint8_t*>(sm.kcur)[l] = code;
      if (l == 0) sm.kcs[0] = ldexpf(1.f, e);
      if (own) {
        reinterpret_cast<uint8_t*>(p.kv)[kbase + (long long)pos * D + l] = code;
        if (l == 0) p.kscale[sbase + pos] = ldexpf(1.f, e);
      }
    } else {
      const uint16_t kb = f32_to_bf16(v);
      sm.kcur[l] = kb;
      if (own) p.kv[kbase + (long long)pos * D + l] = kb;  // KV append (reference kv_cache.cuh:58-78)
    }
  } else if (on && w == 3) {
    if constexpr (K8) {
      const int e = e4m3_row_exp(wave_max(fabsf(v)));
      const uint8_t code = (uint8_t)e4m3_encode(ldexpf(v, -e));
      reinterpret_cast<uint8_t*>(sm.vcur)[l] = code;
      if (l == 0) sm.kcs[1] = ldexpf(1.f, e);
      if (own) {
        reinterpret_cast<uint8_t*>(p.kvt)[kbase + (long long)(pos / 32) * 32 * D + (long long)l * 32 + (pos % 32)] = code;
        if (l == 0) p.vscale[sbase + pos] = ldexpf(1.f, e);
      }
    } else {
      const uint16_t vb = f32_to_bf16(v);
      sm.vcur[l] = vb;
      if (own) p.kvt[kbase + (long long)(pos / 32) * 32 * D + (long long)l * 32 + (pos % 32)] = vb;
    }
  }
  __syncthreads();
  // 2. the wave's blocks: online softmax over them on the matrix cores
  const float scale = 1.0f / sqrtf((float)D);
  float m = -INFINITY, lsum = 0.f;
  f32x4 acc[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) acc[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int q = 0; q < NBW; ++q) {
    const int t0 = 32 * (s * AW * NBW + w + AW * q);
    if (t0 >= n) break;  // uniform over the wave (every block of an item that is off)
    // position pos takes K / V from LDS (this item appended them)
    if (pos >= t0 && pos < t0 + 32) {
      const int rp = pos - t0;
      if constexpr (K8) {
        if (c16 == (rp & 15)) {  // register arrays take compile-time indices only
          const uint8_t* kc8 = reinterpret_cast<const uint8_t*>(sm.kcur);
#pragma unroll
          for (int kc = 0; kc < 2; ++kc) {
            const u32x2 kv = *reinterpret_cast<const u32x2*>(&kc8[32 * kc + 8 * rg]);
            if (rp >> 4) kr[q][1][kc] = kv;
            else kr[q][0][kc] = kv;
          }
          if (rp >> 4) sk[q][1] = sm.kcs[0], sv[q][1] = sm.kcs[1];
          else sk[q][0] = sm.kcs[0], sv[q][0] = sm.kcs[1];
        }
        if (rg == (rp >> 3)) {
          const uint8_t* vc8 = reinterpret_cast<const uint8_t*>(sm.vcur);
#pragma unroll
          for (int dt = 0; dt < D / 16; ++dt) vr[q][dt] = set_u8(vr[q][dt], rp & 7, vc8[16 * dt + c16]);
        }
      } else {
        if (c16 == (rp & 15)) {  // register arrays take compile-time indices only
#pragma unroll
          for (int kc = 0; kc < 2; ++kc) {
            const u32x4 kv = *reinterpret_cast<const u32x4*>(&sm.kcur[32 * kc + 8 * rg]);
            if (rp >> 4) kr[q][1][kc] = kv;
            else kr[q][0][kc] = kv;
          }
        }
        if (rg == (rp >> 3)) {
#pragma unroll
          for (int dt = 0; dt < D / 16; ++dt) vr[q][dt] = with_bf16(vr[q][dt], rp & 7, sm.vcur[16 * dt + c16]);
        }
      }
    }
    float sc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 d4 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {  // q read from LDS per block: registers for a fifth workgroup per CU
        u32x4 kb;
        if constexpr (K8) kb = fp8x8_to_bf16x8_scaled(kr[q][h][kc], sk[q][h]);
        else kb = kr[q][h][kc];
        d4 = mfma(*reinterpret_cast<const u32x4*>(&sm.qb[c16][32 * kc + 8 * rg]), kb, d4);
      }
      const int t = t0 + 16 * h + c16;
      sc[h] = t < n ? ((d4[0] + d4[1]) + d4[2]) * scale : -INFINITY;
    }
    const float mn = fmaxf(m, group_max<16>(fmaxf(sc[0], sc[1])));  // finite: position t0 < n is valid
    const float alpha = __expf(m - mn);
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      sc[h] = __expf(sc[h] - m);
      ps += sc[h];
    }
    lsum = lsum * alpha + group_sum<16>(ps);
    if (rg < 2) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const Split3 a = split3(K8 ? sc[h] * sv[q][h] : sc[h]);
        sm.pb[w][4 * rg + 0][16 * h + c16] = (uint16_t)(a.hi >> 16);
        sm.pb[w][4 * rg + 1][16 * h + c16] = (uint16_t)(a.mid >> 16);
        sm.pb[w][4 * rg + 2][16 * h + c16] = (uint16_t)(a.lo >> 16);
      }
    }
    asm volatile("" ::: "memory");  // LDS operations of one wave complete in order
    const u32x4 pa = *reinterpret_cast<const u32x4*>(&sm.pb[w][c16][8 * rg]);
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[dt][i] *= alpha;
      if constexpr (K8) acc[dt] = mfma(pa, fp8x8_to_bf16x8_scaled(vr[q][dt], 1.0f), acc[dt]);
      else acc[dt] = mfma(pa, vr[q][dt], acc[dt]);
    }
  }
  // 3. combine the waves into the item's partial
  if (rg < 2) {
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) sm.ow[w][rg][16 * dt + c16] = (acc[dt][0] + acc[dt][1]) + acc[dt][2];
    if (c16 == 0) {
      sm.mw[w][rg] = m;
      sm.lw[w][rg] = lsum;
    }
  }
  __syncthreads();
  float* part = p.part + (((long long)b * NKV + g) * p.nsplit_max + s) * PW;
  if (on && tid < 2 * D) {
    const int h = tid / D, d = tid % D;
    float M = sm.mw[0][h];
#pragma unroll
    for (int i = 1; i < AW; ++i) M = fmaxf(M, sm.mw[i][h]);
    float o = 0.f, L = 0.f;
#pragma unroll
    for (int i = 0; i < AW; ++i) {
      const float f = __expf(sm.mw[i][h] - M);
      o = fmaf(f, sm.ow[i][h][d], o);
      L = fmaf(f, sm.lw[i][h], L);
    }
    __hip_atomic_store(part + tid, o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d == 0) {
      __hip_atomic_store(part + 2 * D + 2 * h, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(part + 2 * D + 2 * h + 1, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  // 4. the last split of (b, g) to finish merges: the partial stores above are
  //    acknowledged (write-through) before the counter moves
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    bool last = false;
    if (on) {
      int* c = p.cnt + b * NKV + g;
      const int done = __hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = done == nsplit - 1;
      if (last) __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // re-armed for the next layer
    }
    sm.last = last;
  }
  __syncthreads();
  const bool merge = sm.last;
  if (!FUSED && !merge) return true;  // one item per workgroup: nothing else shares its barriers
  // 5. the merge: thread (split group sg, output hd) reads output hd of every
  //    SG-th split, MG splits per load round (all loads of a round issued
  //    before any is used: one round trip, not one per split); the SG groups
  //    are then combined in LDS
  {
    constexpr int SG = AT / (2 * D), MG = 8;
    const int hd = tid % (2 * D), sg = tid / (2 * D), h = hd / D;
    const float* base = p.part + ((long long)b * NKV + g) * p.nsplit_max * PW;
    float M = -INFINITY, o = 0.f, L = 0.f;
    const int ns = merge ? nsplit : 0;
    for (int r0 = 0; r0 < ns; r0 += SG * MG) {
      float mv[MG], lv[MG], ov[MG];
#pragma unroll
      for (int u = 0; u < MG; ++u) {
        const int i = r0 + sg + SG * u;
        const float* pi = base + (long long)(i < ns ? i : 0) * PW;
        mv[u] = __hip_atomic_load(pi + 2 * D + 2 * h, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lv[u] = __hip_atomic_load(pi + 2 * D + 2 * h + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ov[u] = __hip_atomic_load(pi + hd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      float Mb = M;
#pragma unroll
      for (int u = 0; u < MG; ++u) Mb = r0 + sg + SG * u < ns ? fmaxf(Mb, mv[u]) : Mb;
      const float sc = M == -INFINITY ? 0.f : __expf(M - Mb);  // o, L are 0 while M is -inf
      o *= sc, L *= sc;
#pragma unroll
      for (int u = 0; u < MG; ++u) {
        const bool on_ = r0 + sg + SG * u < ns;  // select: skipped words hold anything
        const float f = __expf(mv[u] - Mb);
        o = on_ ? fmaf(f, ov[u], o) : o;
        L = on_ ? fmaf(f, lv[u], L) : L;
      }
      M = Mb;
    }
    sm.cm[sg][hd] = M, sm.cl[sg][hd] = L, sm.co[sg][hd] = o;
    __syncthreads();
    if (merge && tid < 2 * D) {
      float Mx = sm.cm[0][tid];  // group 0 holds split 0
#pragma unroll
      for (int k = 1; k < SG; ++k) Mx = fmaxf(Mx, sm.cm[k][tid]);
      float oo = 0.f, ll = 0.f;
#pragma unroll
      for (int k = 0; k < SG; ++k) {
        const float f = sm.cm[k][tid] == -INFINITY ? 0.f : __expf(sm.cm[k][tid] - Mx);
        oo = fmaf(f, sm.co[k][tid], oo);
        ll = fmaf(f, sm.cl[k][tid], ll);
      }
      uint16_t hi, lo;
      split2(oo / ll, hi, lo);
      const int k = unit_at(b, g * 2 * D + tid);
      st_act<FUSED>(att_slot<S>(p, sl) + k, hi);
      st_act<FUSED>(att_slot<S>(p, sl) + BMAX * S::QD + k, lo);
    }
  }
  if constexpr (FUSED) {  // the merged output is acknowledged before it is counted
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (merge && tid == 0)
      __hip_atomic_store(p.flags + ((long long)layer * FC_N + FC_ATT) * FLAG_MAX + b * NKV + g, ep, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
  }
  return true;
}

// Five 256-thread items per CU (<= 102 registers per lane): the 16-sequence
// step at KV 512-4096 has ~1,100 items; with four per CU the last ~10 % ran
// as a second, latency-bound residency wave.
constexpr int ATTN_WAVES_PER_EU = AT == 256 ? 5 : 2;
template <class S, bool K8>
__global__ __launch_bounds__(AT) __attribute__((amdgpu_waves_per_eu(ATTN_WAVES_PER_EU, ATTN_WAVES_PER_EU))) void bk_attn(
    PGroup1 pg, int layer) {
  __shared__ AttnLds<S> sm;
  const BParams& p = group_of(pg);  // column group
  // workgroup i runs on XCD i % 8: every split of one (sequence, kv head)
  // pair gets the same XCD, so the merging split reads its partials there; a
  // pair's splits are consecutive slots of its XCD (split-major numbering,
  // split 0 of every pair first, measured 3 % slower for the batched decode)
  static_assert((BMAX * S::NKV) % 8 == 0, "whole (sequence, kv head) pairs per XCD");
  const int xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
  const int bg = (slot / p.nsplit_max) * 8 + xcd, s = slot % p.nsplit_max;
  const int b = bg / S::NKV, g = bg % S::NKV;
  if (b >= p.B) return;
  const int pos = p.pos[b];
  const int nsplit = (pos + 1 + CH - 1) / CH;
  if (s >= nsplit) return;
  AttnKV<S, K8> kv;
  attn_kv_load<S, K8>(p, layer, true, b, g, s, pos, kv);
  attn_item<S, K8, false>(p, layer, 0, sm, true, b, g, s, nsplit, pos, kv, NoWait{});
}

// ------------------------------------------------------------ prefill attention
// One workgroup of AWc waves per (kv head g, column group): the group's
// <= 16 tokens x 2 q heads = 32 queries (query q: token q / 2, head 2 g + q % 2)
// as two 16-column tiles; wave w takes the 32-position K / V blocks w, w +
// AWc, ... of the causal prefix [0, the group's last position] with an
// online softmax per query, and the waves' states are combined at the end.
// Products (v_mfma_f32_16x16x32_bf16):
//   scores^T (16 positions x 16 queries) = K (A operand: the cache rows as
//     loaded) . Q^T (B operand: q in NPART bf16 parts, one product each);
//   out^T (16 dims x 16 queries) += V^T (A operand: the transposed cache, the
//     block's positions in the order the scores leave them in a lane) . P^T
//     (B operand: the softmax weights in NPART parts, built in registers).
// A lane holds 4 positions x 1 query of each 16-position score tile: the
// block max takes two cross-lane steps, the row sums stay per lane until the
// end, and the weights never pass through LDS.  NPART 3: q and the weights
// split exactly (hi + mid + lo by truncation); 2: hi + lo (RNE), relative
// error <= 2^-17.
// The score tiles take the positions of a block in the order 8 (r / 4) + 4 h +
// r % 4 (row r of tile h), so a lane's eight weights are eight consecutive
// positions and V^T is read 16 bytes at a time.
// What bounds it: the vector work beside the products (about 1,000 cycles of
// softmax and splitting per block step against 768 of matrix products) and,
// for a few groups, the load round trip of a wave's next block; two waves per
// SIMD.  us per layer inside whole passes (kernel trace), 64 groups at position
// 0 / 1,024 / 3,072: 20.4 / 36.5 / 66.5 with 8-byte V loads, non-temporal loads
// and one query tile after the other, 17.2 / 30.2 / 55.8 as it is; FP8 23.8 /
// 43.1 / 82.2 and 17.6 / 32.1 / 60.8; 13 groups at 1,500: 16.9 and 15.4.
// (Earlier measurements: three K / V register sets 23.2 against two 20.6; two
// parts 20.8 against three 21.6.)
#ifndef MK_PATTN_NPART
#define MK_PATTN_NPART 3
#endif
constexpr int PC_NQ = 2 * BMAX;  // queries of a workgroup (a column group x 2 q heads)
// Prefix splits (grid z): with few column groups a workgroup per (kv head,
// group) leaves most of the chip idle, so the prefix is cut into up to PC_NZ
// splits while there are at most PC_WG workgroups and the last group, whose
// prefix is the longest, keeps at least two blocks per wave (an earlier group's
// splits may be shorter); the split that finishes last merges (as in bk_attn).
constexpr int PC_WG = 256, PC_NZ = 16;
constexpr int PC_PW = PC_NQ * 64 + 2 * PC_NQ;  // floats of a split's partial: o[32][64], max[32], sum[32]
template <class S, bool K8>
struct PcKV {  // one block's K / V operands of a lane, as loaded (K8: FP8 codes, converted at use)
  using Reg = typename std::conditional<K8, u32x2, u32x4>::type;
  Reg k[2][2];  // [16-position half][32-dim chunk]
  Reg v[S::D / 16];  // [16-dim tile]: positions 8 gq .. 8 gq + 7
  f32x4 sk[2], sv[2];  // K8: row scales of the lane's score positions t0 + 8 gq + 4 h + i
};
// bf16 operand of a loaded register: FP8 codes converted exactly (scale 1)
__device__ __forceinline__ u32x4 pc_op(u32x4 r) { return r; }
__device__ __forceinline__ u32x4 pc_op(u32x2 r) { return fp8x8_to_bf16x8_scaled(r, 1.0f); }
template <class S, bool K8>
__device__ __forceinline__ void pc_load(const BParams& p, __amdgpu_buffer_rsrc_t rk, __amdgpu_buffer_rsrc_t rv,
                                        long long sbase, int t0, unsigned c16, unsigned gq, PcKV<S, K8>& r) {
  constexpr int D = S::D;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int kc = 0; kc < 2; ++kc) {
      const unsigned e = ((unsigned)t0 + 8u * (c16 >> 2) + 4u * h + (c16 & 3u)) * D + 32u * kc + 8u * gq;
      if constexpr (K8)
        r.k[h][kc] = __builtin_amdgcn_raw_buffer_load_b64(rk, e, 0u, 0);
      else
        r.k[h][kc] = __builtin_amdgcn_raw_buffer_load_b128(rk, e * 2u, 0u, 0);
    }
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) {
    const unsigned e = (unsigned)t0 * D + (16u * dt + c16) * 32u + 8u * gq;
    if constexpr (K8)
      r.v[dt] = __builtin_amdgcn_raw_buffer_load_b64(rv, e, 0u, 0);
    else
      r.v[dt] = __builtin_amdgcn_raw_buffer_load_b128(rv, e * 2u, 0u, 0);
  }
  if constexpr (K8) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      r.sk[h] = *reinterpret_cast<const f32x4*>(p.kscale + sbase + t0 + 8 * (int)gq + 4 * h);
      r.sv[h] = *reinterpret_cast<const f32x4*>(p.vscale + sbase + t0 + 8 * (int)gq + 4 * h);
    }
  }
}
// 8 fp32 values -> NPART bf16x8 parts (3: exact truncation split; 2: RNE hi + lo)
template <int NPART>
__device__ __forceinline__ void pc_parts(const float (&x)[8], u32x4 (&o)[NPART]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if constexpr (NPART == 3) {
      const Split3 a = split3(x[2 * e]), b = split3(x[2 * e + 1]);
      o[0][e] = pack_hi16(a.hi, b.hi);
      o[1][e] = pack_hi16(a.mid, b.mid);
      o[2][e] = pack_hi16(a.lo, b.lo);
    } else {
      uint32_t hi, lo;
      bf16_hilo2(x[2 * e], x[2 * e + 1], hi, lo);
      o[0][e] = hi;
      o[1][e] = lo;
    }
  }
}
template <class S, bool K8, int AWc, int NPART = MK_PATTN_NPART>
__global__ __launch_bounds__(AWc * kWave) __attribute__((amdgpu_waves_per_eu(2))) void bk_pattn(PGroup pg, int layer) {
  static_assert(S::GQA == 2 && S::D == 64, "2 q heads of 64 per kv head");
  static_assert(NPART == 2 || NPART == 3, "two or three bf16 parts");
  constexpr int D = S::D, NKV = S::NKV, NT = AWc * kWave, QT = PC_NQ / 16;
  // q is multiplied by log2(e) / sqrt(D) before it is split, so a score is
  // already the exponent of 2 of its softmax weight
  constexpr float kLog2Scale = 1.4426950408889634f / 8.0f;
  static_assert(D == 64, "1 / sqrt(D) = 1 / 8");
  __shared__ float ow[AWc][PC_NQ][D + 4];  // padded rows: the lanes of one store hit distinct banks
  __shared__ float mw[AWc][PC_NQ], lw[AWc][PC_NQ];
  // the longest prefixes (the last groups) first
  const int gi = pg.n - 1 - (int)blockIdx.y;
  const BParams p = group_params(pg, gi);
  const int g = blockIdx.x, tid = ltid(), w = wave_id(), l = (int)lane_id();
  const unsigned c16 = (unsigned)l & 15u, gq = (unsigned)l >> 4;
  const long long kbase = ((long long)layer * NKV + g) * (long long)p.s_pad * D;
  const long long sbase = ((long long)layer * NKV + g) * p.s_pad;
  const auto rk = K8 ? make_rsrc(reinterpret_cast<const uint8_t*>(p.kv) + kbase) : make_rsrc(p.kv + kbase);
  const auto rv = K8 ? make_rsrc(reinterpret_cast<const uint8_t*>(p.kvt) + kbase) : make_rsrc(p.kvt + kbase);
  const int p0 = pg.pos0 + BMAX * gi, pmax = p0 + p.B - 1, nall = pmax / 32 + 1;
  // this split's blocks [b0, nblk) of the prefix; the wave's first one is
  // loading during the prologue
  const int nz = gridDim.z, z = blockIdx.z, b0 = z * nall / nz, nblk = (z + 1) * nall / nz;
  PcKV<S, K8> cur, nxt;
  if (b0 + w < nblk) pc_load<S, K8>(p, rk, rv, sbase, 32 * (b0 + w), c16, gq, cur);
  __builtin_amdgcn_sched_barrier(0);
  // 1. the queries (normalised and rotated, qkv_head) as B operands, held for
  //    the whole loop: lane (gq, c16) takes dims 32 kc + 8 gq .. + 7 of query
  //    16 qt + c16 and splits them in registers
  u32x4 qb[QT][NPART][2];
  {
    f32x4 qv[QT][2][2];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      const int q = 16 * qt + (int)c16, col = q >> 1, j = q & 1;
      const float* src = qkv_slot<S>(p, 0) + (long long)(col < p.B ? col : 0) * S::QKV + (g * 2 + j) * D + 8 * gq;
#pragma unroll
      for (int kc = 0; kc < 2; ++kc)
#pragma unroll
        for (int e = 0; e < 2; ++e) qv[qt][kc][e] = *reinterpret_cast<const f32x4*>(src + 32 * kc + 4 * e);
    }
#pragma unroll
    for (int qt = 0; qt < QT; ++qt)
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        float x[8];
        u32x4 parts[NPART];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = qv[qt][kc][e / 4][e % 4] * kLog2Scale;  // log2 units, softmax scale included
        pc_parts<NPART>(x, parts);
#pragma unroll
        for (int pt = 0; pt < NPART; ++pt) qb[qt][pt][kc] = parts[pt];
      }
  }
  // 2. the wave's blocks
  float m[QT], ls[QT];
  int qpos[QT];
  f32x4 acc[QT][D / 16];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m[qt] = -INFINITY, ls[qt] = 0.f;
    const int col = (16 * qt + (int)c16) >> 1;
    qpos[qt] = col < p.B ? p0 + col : -1;  // -1: no token (every score masked)
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) acc[qt][dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // the first query's position when all 16 tokens exist, else -1: a block
  // that ends at or before it is visible to every query (no mask)
  const int qmin = p.B == BMAX ? p0 : -1;
  // the products and online-softmax step of both query tiles on a block (r:
  // its K / V operands), in one straight line so that one tile's vector work
  // runs beside the other's products; MASK: the causal mask and the guards of
  // a query that has no visible position yet
  const auto step = [&](auto mask_c, int t0, const PcKV<S, K8>& r) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask_c)::value;
    float sc[QT][2][4], mo[QT], mn[QT];
    f32x4 d4[QT][2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int kc = 0; kc < 2; ++kc) {
        const u32x4 ka = pc_op(r.k[h][kc]);
#pragma unroll
        for (int pt = 0; pt < NPART; ++pt)
#pragma unroll
          for (int qt = 0; qt < QT; ++qt)
            d4[qt][h] = mfma(ka, qb[qt][pt][kc], kc + pt == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : d4[qt][h]);
      }
    bool grew = false;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // K8: the K row scale (a power of two) multiplies the exact product
          const float x = K8 ? d4[qt][h][i] * r.sk[h][i] : d4[qt][h][i];
          sc[qt][h][i] = MASK && t0 + 8 * (int)gq + 4 * h + i > qpos[qt] ? -INFINITY : x;
        }
      float bm = fmaxf(fmaxf(fmaxf(sc[qt][0][0], sc[qt][0][1]), fmaxf(sc[qt][0][2], sc[qt][0][3])),
                       fmaxf(fmaxf(sc[qt][1][0], sc[qt][1][1]), fmaxf(sc[qt][1][2], sc[qt][1][3])));
      bm = max_xor32(max_xor16(bm));
      mo[qt] = m[qt], mn[qt] = fmaxf(m[qt], bm);
      m[qt] = mn[qt];
      grew |= mn[qt] != mo[qt];
    }
    // the running state is rescaled only when some query's maximum grew (the
    // factor is exactly 1 otherwise).  The branch is taken by the whole wave:
    // a query still without a visible position (mn = mo = -inf) keeps factor
    // 1, not exp2(-inf - -inf)
    if (__builtin_amdgcn_ballot_w64(grew)) {
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        const float alpha = MASK && mn[qt] == -INFINITY ? 1.f : exp2f(mo[qt] - mn[qt]);
        ls[qt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[qt][dt][i] *= alpha;
      }
    }
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      float pw[8], ps = 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // a query none of whose positions so far is visible keeps m = -inf
          // and weight 0 (no -inf - -inf)
          const float e = MASK && mn[qt] == -INFINITY ? 0.f : exp2f(sc[qt][h][i] - mn[qt]);
          ps += e;
          pw[4 * h + i] = K8 ? e * r.sv[h][i] : e;  // the V row scale enters the weight
        }
      ls[qt] += ps;
      u32x4 pb[NPART];
      pc_parts<NPART>(pw, pb);
#pragma unroll
      for (int pt = 0; pt < NPART; ++pt)
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) acc[qt][dt] = mfma(pc_op(r.v[dt]), pb[pt], acc[qt][dt]);
    }
  };
  const auto block = [&](int t0, const PcKV<S, K8>& r) __attribute__((always_inline)) {
    if (t0 + 31 <= qmin) step(std::false_type{}, t0, r);
    else step(std::true_type{}, t0, r);
  };
  // two register sets in turn (no copy between them: a copy would wait for
  // the next block's loads before the current block's products).  Every
  // iteration issues both sets' loads (past the prefix they repeat its last
  // block, unused), so that each product waits for exactly its own block's
  // loads: with a conditional issue the compiler's waits, merged over both
  // paths, also waited for the block after.
  // The scheduling barriers keep the loads where they are: the scheduler
  // otherwise sinks them to their first use.
  for (int kb = b0 + w; kb < nblk; kb += 2 * AWc) {
    pc_load<S, K8>(p, rk, rv, sbase, 32 * min(kb + AWc, nblk - 1), c16, gq, nxt);
    __builtin_amdgcn_sched_barrier(0);
    block(32 * kb, cur);
    if (kb + AWc >= nblk) break;
    pc_load<S, K8>(p, rk, rv, sbase, 32 * min(kb + 2 * AWc, nblk - 1), c16, gq, cur);
    __builtin_amdgcn_sched_barrier(0);
    block(32 * (kb + AWc), nxt);
  }
  // 3. combine the waves and write the output as bf16 hi / lo parts
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int q = 16 * qt + (int)c16;
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) ow[w][q][16 * dt + 4 * gq + i] = acc[qt][dt][i];
    const float lt = sum_xor32(sum_xor16(ls[qt]));
    if (gq == 0) {
      mw[w][q] = m[qt];
      lw[w][q] = lt;
    }
  }
  __syncthreads();
  // thread: OD dims of one query
  constexpr int OD = PC_NQ * D / NT;
  static_assert(OD == 4 || OD == 8, "whole 8-byte stores per thread");
  const int q = tid / (D / OD), d0 = tid % (D / OD) * OD, col = q >> 1, j = q & 1;
  float M = mw[0][q], o[OD], L = 0.f;
#pragma unroll
  for (int i = 1; i < AWc; ++i) M = fmaxf(M, mw[i][q]);
#pragma unroll
  for (int e = 0; e < OD; ++e) o[e] = 0.f;
#pragma unroll
  for (int i = 0; i < AWc; ++i) {
    const float f = mw[i][q] == -INFINITY ? 0.f : exp2f(mw[i][q] - M);
#pragma unroll
    for (int e = 0; e < OD; ++e) o[e] = fmaf(f, ow[i][q][d0 + e], o[e]);
    L = fmaf(f, lw[i][q], L);
  }
  if (nz > 1) {
    // the split's partial, written through and acknowledged before it is
    // counted; the last split of (group, kv head) adds them in split order
    __shared__ int last;
    float* part = pg.p.part + (long long)(gi * NKV + g) * nz * PC_PW;
    {
      float* mine = part + (long long)z * PC_PW;
#pragma unroll
      for (int e = 0; e < OD; ++e)
        __hip_atomic_store(mine + q * D + d0 + e, o[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d0 == 0) {
        __hip_atomic_store(mine + PC_NQ * D + q, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mine + PC_NQ * D + PC_NQ + q, L, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const int done = __hip_atomic_fetch_add(p.cnt + g, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = done == nz - 1;
      if (last) __hip_atomic_store(p.cnt + g, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next layer
    }
    __syncthreads();
    if (!last) return;
    float mv[PC_NZ], lv[PC_NZ], ov[PC_NZ][OD];  // every split's loads before the first use
#pragma unroll
    for (int k = 0; k < PC_NZ; ++k) {
      const float* pk = part + (long long)(k < nz ? k : 0) * PC_PW;
      if (k < nz) {
        mv[k] = __hip_atomic_load(pk + PC_NQ * D + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        lv[k] = __hip_atomic_load(pk + PC_NQ * D + PC_NQ + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int e = 0; e < OD; ++e)
          ov[k][e] = __hip_atomic_load(pk + q * D + d0 + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    M = -INFINITY, L = 0.f;
#pragma unroll
    for (int k = 0; k < PC_NZ; ++k) M = k < nz ? fmaxf(M, mv[k]) : M;
#pragma unroll
    for (int e = 0; e < OD; ++e) o[e] = 0.f;
#pragma unroll
    for (int k = 0; k < PC_NZ; ++k) {
      if (k < nz) {
        const float f = mv[k] == -INFINITY ? 0.f : exp2f(mv[k] - M);
#pragma unroll
        for (int e = 0; e < OD; ++e) o[e] = fmaf(f, ov[k][e], o[e]);
        L = fmaf(f, lv[k], L);
      }
    }
  }
  if (col >= p.B) return;
  uint16_t* a = att_slot<S>(p, 0) + unit_at(col, (g * 2 + j) * D + d0);
#pragma unroll
  for (int c = 0; c < OD; c += 4) {
    uint16_t hi[4], lo[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split2(o[c + e] / L, hi[e], lo[e]);
    st4(a + c, hi);
    st4(a + BMAX * S::QD + c, lo);
  }
}

// ------------------------------------------------------------ one-kernel step
// Workgroups of bk_step per CU (waves per SIMD = 2 x that): two, so twice the
// attention items run at once (<= 128 registers per lane).
#ifndef MK_STEP_WG_PER_CU
#define MK_STEP_WG_PER_CU 2
#endif
constexpr int STEP_WG_PER_CU = MK_STEP_WG_PER_CU;
constexpr int STEP_WAVES_PER_EU = 2 * STEP_WG_PER_CU;
// Every layer of a decode step in one persistent kernel: STEP_WG_PER_CU
// workgroups of GT threads per CU (all resident; the host checks the
// occupancy), each running
// its share of every phase of a layer in phase order and handing off through
// p.flags (one word per producer, the step's epoch once its outputs are out):
//   QKV block rb            on workgroup rb            waits: down of layer - 1 (H/16 blocks)
//   attention item pairs    pair j on workgroup (j + QKV/16) % G
//                                                      waits: every QKV block
//     (the two AT-thread halves of a workgroup run items 2j and 2j + 1)
//   O block rb              on workgroup (G - H/16 + rb) % G (G > H/16)
//                                                      waits: every (sequence, kv head) merged
//   gate/up block rb        on workgroup rb             waits: every O block
//   down piece (rb, ks)     on workgroup 4 rb + ks      waits: every gate/up block
//     (split 0 then waits for splits 1-3 of its block, whose sums carry a tag)
// Each block issues its weight loads before it waits, and every workgroup
// without a QKV block the K / V loads of its first attention pair at the
// layer start, so the loads overlap the hand-offs; every wait is for a phase that precedes it in the order
// above, and no phase waits for a later one, so the persistent grid cannot
// deadlock.  The arithmetic is that of the per-phase kernels (same block
// functions, same summation order): the logits are bit-identical.
template <class S, bool K8 = false>
__global__ __launch_bounds__(GT) __attribute__((amdgpu_waves_per_eu(STEP_WAVES_PER_EU, STEP_WAVES_PER_EU))) void bk_step(
    PGroup1 pg) {
  const BParams& p = pg.p[0];  // one group
  static_assert(GT == 2 * AT, "two attention items per workgroup");
  __shared__ float red[GW * 16 * 17];
  __shared__ float rr[RR_N];
  __shared__ int last;
  __shared__ AttnLds<S> att[2];
  __shared__ int icum[BMAX + 1], ins[BMAX], ipos[BMAX];
  const int G = gridDim.x, wg = blockIdx.x;
  if (threadIdx.x == 0) {  // attention items of the step: sequence b has NKV * nsplit_b, in (b, g, s) order
    int c = 0;
    for (int b = 0; b < BMAX; ++b) {
      const int pos = b < p.B ? p.pos[b] : 0;
      const int ns = b < p.B ? (pos + 1 + CH - 1) / CH : 0;
      icum[b] = c;
      ins[b] = ns;
      ipos[b] = pos;
      c += S::NKV * ns;
    }
    icum[BMAX] = c;
  }
  __syncthreads();
  const int n_items = icum[BMAX];
  const int ep = *p.epoch;  // this step's epoch (bk_embed advanced it)
  u64* const tr = p.trace;
  int layer = 0;
  auto stamp = [&](int ev) {
    if (tr && ltid() == 0) tr[((long long)layer * TR_N + ev) * G + wg] = wall_clock64();
  };
  // a wait followed by its "inputs ready" stamp
  auto waited = [&](bool ok, int ev) {
    stamp(ev);
    return ok;
  };
  // pair j on workgroup (j + QKV blocks) % G: the workgroups without a QKV
  // block take the first pairs; every workgroup issues the K / V loads of its
  // first pair at the layer start (they only read the cache)
  const int j0 = (wg - S::RB_QKV % G + G) % G;
  struct Item {
    bool on;
    int b, g, s, ns;
  };
  auto item_of = [&](int j) {
    const int i = 2 * j + ltid() / AT;
    Item it;
    it.on = i < n_items;
    int b = 0;
    while (b + 1 < BMAX && icum[b + 1] <= i) ++b;
    const int r = it.on ? i - icum[b] : 0;
    it.ns = ins[b] > 0 ? ins[b] : 1;
    it.b = b, it.g = r / it.ns, it.s = r % it.ns;
    return it;
  };
  for (; layer < p.L; ++layer) {
    stamp(TR_START);
    bool qkv_in = false;  // this layer's QKV flags already seen by this workgroup
    auto qkv_ready = [&] {
      if (qkv_in) return true;
      qkv_in = waited(fc_wait(p, layer, FC_QKV, S::RB_QKV, ep), TR_ATT_IN);
      return qkv_in;
    };
    int jn = j0;  // the next attention pair of this workgroup
    if (wg >= S::RB_QKV && 2 * j0 < n_items) {
      // no QKV block: the first pair's K / V loads are issued at the layer
      // start and overlap the QKV phase (a workgroup with a QKV block issues
      // them after it, in the loop below: both at once do not fit the registers)
      const Item it = item_of(j0);
      AttnKV<S, K8> kv;
      attn_kv_load<S, K8>(p, layer, it.on, it.b, it.g, it.s, ipos[it.b], kv);
      if (!attn_item<S, K8, true>(p, layer, ep, att[ltid() / AT], it.on, it.b, it.g, it.s, it.ns, ipos[it.b], kv,
                                  qkv_ready))
        return;
      stamp(TR_ATT_DONE);
      jn += G;
    } else {
      for (int rb = wg; rb < S::RB_QKV; rb += G) {
        if (!qkv_block<S, true>(p, layer, ep, rb, 0, red, rr, &last, [&] {
              return waited(layer == 0 || fc_wait(p, layer - 1, FC_DN, S::RB_H, ep), TR_QKV_IN);
            }))
          return;
        stamp(TR_QKV_DONE);
      }
    }
    for (int j = jn; 2 * j < n_items; j += G) {
      const Item it = item_of(j);
      AttnKV<S, K8> kv;
      attn_kv_load<S, K8>(p, layer, it.on, it.b, it.g, it.s, ipos[it.b], kv);
      if (!attn_item<S, K8, true>(p, layer, ep, att[ltid() / AT], it.on, it.b, it.g, it.s, it.ns, ipos[it.b], kv,
                                  qkv_ready))
        return;
      stamp(TR_ATT_DONE);
    }
    const int o_off = G > S::RB_H ? G - S::RB_H : 0;  // O on the last workgroups (fewest attention pairs)
    for (int rb = 0; rb < S::RB_H; ++rb)
      if ((rb + o_off) % G == wg) {
        if (!o_block<S, true>(p, layer, ep, rb, 0, red, &last,
                              [&] { return waited(fc_wait(p, layer, FC_ATT, p.B * S::NKV, ep), TR_O_IN); }))
          return;
        stamp(TR_O_DONE);
      }
    for (int rb = wg; rb < S::RB_F; rb += G) {
      if (!gu_block<S, true>(p, layer, ep, rb, 0, red, rr, &last,
                             [&] { return waited(fc_wait(p, layer, FC_O, S::RB_H, ep), TR_GU_IN); }))
        return;
      stamp(TR_GU_DONE);
    }
    // a workgroup with several down pieces runs its split-0 pieces (which
    // wait for the other splits of their block) after the others
    for (int pass = 0; pass < 2; ++pass)
      for (int k = wg; k < S::RB_H * KS_DN; k += G) {
        if ((k % KS_DN == 0) != (pass == 1)) continue;
        if (!down_block<S, true>(p, layer, ep, k / KS_DN, k % KS_DN, red, &last,
                                 [&] { return waited(fc_wait(p, layer, FC_GU, S::RB_F, ep), TR_DN_IN); }))
          return;
        stamp(TR_DN_DONE);
      }
  }
}

}  // namespace batch
}  // namespace mk
