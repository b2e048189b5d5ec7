// Single-query paged decode partial over one domain chunk.
//
// Replaces decode_local_partial / decode_local_compact_partial (ring.rs:625-639,
// :515-523): one query token per sequence, no causal mask (ring.rs:631-637), output
// normalised o and natural-log lse in fp32.  KV is read in place from the vLLM pool
// [2, num_blocks, bs, Hkv, D] (python/hcp_vllm_block_ring_plugin.py:8-14) through the
// sequence's block table -- no gather, no GQA expand copy.
//
// Work split (HBM-bound: every K/V byte is read exactly once):
//   * One launch covers every shard of every sequence (a decode partial has one shard, the
//     decode Q-ring one per domain).  A sequence's 16-token groups, shard after shard, are
//     dealt out in equal contiguous runs to `parts` x `subs` waves, whatever its own
//     length; grid = (parts, batch, ceil(Hkv / heads)), a workgroup holding `heads` kv
//     heads x `subs` runs of one part.  The subs of a part meet in LDS, the parts in the
//     LSE merge kernel.  plan_decode picks the three by modelled time: with a few sequences
//     a run is down to one group.
//   * Per 16 tokens a wave reads 16 K rows and 16 V rows of its head (4 KiB each for D=128,
//     bf16) straight from the pool; with many sequences a workgroup reads whole pool token
//     rows (heads = min(8, Hkv); 4 heads a workgroup: 0.7% slower on c4).
//   * Scores: S^T = K Q^T on MFMA 16x16x32 (A = 16 key rows loaded from the pool, 16
//     bytes per lane; B = the rep <= 16 query heads of the kv head -- the GQA group of
//     repeat_decode_kv_heads, ring.rs:496-512 -- zero-padded to 16 columns, held in
//     registers for the whole kernel).
//   * Online softmax per query head in the log2 domain; P goes through a small LDS
//     slot (broadcast reads) and PV runs on VALU with each lane owning 8 head-dim
//     values of 4 of the 16 keys for R query heads (R = 4, 8 or 16, the smallest that
//     holds rep; fp32 accumulators), reduced across lanes once at the end.
//   * Each part writes (o, lse) to the workspace; the LSE merge kernel combines the
//     parts of a sequence (heads = batch*Hq, q_len = 1).
#include <algorithm>

#include "kernels.hpp"
#include "../../include/hcp_ring.h"

namespace hcp {

struct DecodeArgs {
  const uint16_t* q;
  int64_t q_bs, q_hs;  // element strides: batch, head
  const uint16_t* pool;
  int64_t plane_elems;
  int64_t num_blocks;
  int32_t bs, hkv, hq, rep;
  DecodeSpan span[kMaxDomains];  // shards in merge order
  int32_t n_spans;
  int32_t heads, subs;  // kv heads and runs per workgroup
  int32_t gpb;          // 16-token groups per block (bs / 16)
  int32_t gpb_shift;    // its log2, or -1
  float scale_log2;
  float* ws_o;          // [parts][batch*hq][D]
  float* ws_lse;        // [parts][batch*hq]
  int32_t batch;
  int* err;
  int32_t dn;           // head dim of the pool rows, q and the partials (the D=128 kernel:
                        // any multiple of 8 up to 128, columns past it read as zeros)
};
static_assert(sizeof(DecodeArgs) <= 4096, "kernel arguments are limited to 4 KiB");

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ f32x4 mma16(u32x4 a, u32x4 b, f32x4 c);
template <>
__device__ __forceinline__ f32x4 mma16<kBF16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <>
__device__ __forceinline__ f32x4 mma16<kF16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

template <int DT>
__device__ __forceinline__ float lo_half(uint32_t w) {
  return DT == kBF16 ? __uint_as_float(w << 16) : f16_bits_to_f32(static_cast<uint16_t>(w & 0xffffu));
}
template <int DT>
__device__ __forceinline__ float hi_half(uint32_t w) {
  return DT == kBF16 ? __uint_as_float(w & 0xffff0000u) : f16_bits_to_f32(static_cast<uint16_t>(w >> 16));
}

constexpr float kNoMax = -1.0e30f;
constexpr int kDecWaves = 8;  // most waves per workgroup

// One wave per kv head and run.  Per 16-key group the wave needs the head's 16 K rows and 16 V
// rows (4 KiB each for D=128); the next group's loads are issued before a group is
// computed, and the block ids come from one table load per 64 groups.
template <int D, int DT, int R, bool PAD>
__global__ __launch_bounds__(512) void paged_decode_kernel(DecodeArgs a) {
  // PAD: head dim a.dn < D; the 16-byte columns past it are not loaded (zeros) nor stored
  const int dn = PAD ? a.dn : D;
  constexpr int KS = D / 32;        // k-steps of 32 for the QK^T product
  constexpr int DCH = D / 8;        // 8-wide d chunks per row (16 for D=128)
  constexpr int TPL = 16 * DCH / 64;  // keys per lane in PV (4 for D=128)

  __shared__ __attribute__((aligned(16))) float p_lds[kDecWaves][16][R];  // [wave][key][query col]
  // subs > 1: the waves' O, m and l (meet_bytes; a launch whose runs do not meet holds none of
  // it, and small workgroups stay as many to a CU as their registers allow)
  extern __shared__ __attribute__((aligned(16))) float meet_lds[];
  float (*const o_lds)[R][D] = reinterpret_cast<float (*)[R][D]>(meet_lds);
  float (*const m_lds)[R] = reinterpret_cast<float (*)[R]>(meet_lds + kDecWaves * R * D);
  float (*const l_lds)[R] = m_lds + kDecWaves;

  const int b = blockIdx.y;
  const int part = blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = wave / a.heads;
  const int kvh = blockIdx.z * a.heads + wave - sub * a.heads;
  const bool idle = kvh >= a.hkv;
  if (idle && a.subs == 1) return;  // no workgroup barrier below
  const int lane = threadIdx.x & 63;
  const int col = lane & 15;   // MFMA column = query head within the kv group
  const int grp = lane >> 4;   // MFMA k-group / key group
  // PV role: lane owns d chunk pv_dc (8 values) of keys pv_tg*TPL .. +TPL.
  const int pv_dc = lane % DCH;
  const int pv_tg = lane / DCH;

  // Tokens and 16-token groups of this sequence in shard s: table entries past its own
  // last group may be padding (ragged batches) and are neither read nor validated.
  auto span_end = [&](int s) __attribute__((always_inline)) -> int64_t {
    const DecodeSpan& sp = a.span[s];
    if (sp.seq_lens == nullptr) return sp.t1;
    return min(sp.t1, static_cast<int64_t>(__builtin_amdgcn_readfirstlane(sp.seq_lens[b])) - sp.len_off);
  };
  auto span_groups = [&](int s, int64_t t_end) __attribute__((always_inline)) {
    const int64_t t0 = a.span[s].t0;
    return t_end > t0 ? static_cast<int>((t_end + 15) / 16 - t0 / 16) : 0;
  };
  int total = 0;
  for (int s = 0; s < a.n_spans; ++s) total += span_groups(s, span_end(s));
  const int runs = gridDim.x * a.subs;
  const int run_len = (total + runs - 1) / runs;
  const int g0 = idle ? total : min((part * a.subs + sub) * run_len, total);
  const int g1 = min(g0 + run_len, total);

  // Q^T fragments: lane (col, grp) holds Q[head kvh*rep + col][grp*8 + 32*s .. +8].
  u32x4 qf[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    u32x4 v = {0, 0, 0, 0};
    if (!idle && col < a.rep && (!PAD || grp * 8 + 32 * s < dn))
      v = *reinterpret_cast<const u32x4*>(a.q + b * a.q_bs + (kvh * a.rep + col) * a.q_hs + grp * 8 + 32 * s);
    qf[s] = v;
  }

  // PV accumulators cover rep <= R query heads per kv head (checked by the launcher).
  float acc[R][8];
#pragma unroll
  for (int c = 0; c < R; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[c][e] = 0.f;
  float m_run = kNoMax, l_run = 0.f;

  const int64_t row_elems = static_cast<int64_t>(a.hkv) * dn;  // one slot, all heads

  struct Group {
    u32x4 k[KS];
    u32x4 v[TPL];
    int lo, hi;  // keys [lo, hi) of the group count
    bool ok;
  };
  // Cursor over the shards: groups [s_begin, s_end) of the sequence lie in shard s.
  int s = -1, s_begin = 0, s_end = 0;
  int64_t t_end = 0, t_beg = 0;
  int g_first = 0;                  // first group of the shard (t0 / 16)
  const int32_t* table = nullptr;
  int64_t table_len = 0;
  // Block ids of the run's groups, 64 at a time: lane i holds the table entry of group
  // ids_base + i, read back with readlane, so no group waits on a table load.  Keys of a
  // group lie in one table entry (bs is a multiple of 16).
  int ids = -1, ids_base = -64;
  auto load_group = [&](int g, Group& G) {
    if (g >= s_end) {
      do {
        ++s;
        s_begin = s_end;
        t_end = span_end(s);
        s_end += span_groups(s, t_end);
      } while (g >= s_end);
      const DecodeSpan& sp = a.span[s];
      t_beg = sp.t0;
      g_first = static_cast<int>(t_beg / 16);
      table = sp.tables + static_cast<int64_t>(b) * sp.table_stride;
      table_len = sp.table_len;
      ids_base = g - 64;
    }
    if (g - ids_base >= 64) {
      ids_base = g;
      const int gl = g_first + g - s_begin + lane;
      const int e = a.gpb_shift >= 0 ? gl >> a.gpb_shift : gl / a.gpb;
      ids = g + lane < min(g1, s_end) && e < table_len ? table[e] : -1;
    }
    const int32_t blk = __builtin_amdgcn_readlane(ids, g - ids_base);
    const int gl = g_first + g - s_begin;
    const int entry = a.gpb_shift >= 0 ? gl >> a.gpb_shift : gl / a.gpb;
    const int64_t tok0 = static_cast<int64_t>(gl) * 16;
    G.lo = __builtin_amdgcn_readfirstlane(static_cast<int>(t_beg > tok0 ? t_beg - tok0 : 0));
    G.hi = __builtin_amdgcn_readfirstlane(static_cast<int>(min(t_end - tok0, static_cast<int64_t>(16))));
    G.ok = blk >= 0 && blk < a.num_blocks;
    if (!G.ok) {
      if (lane == 0 && entry < table_len) atomicOr(a.err, 1);
#pragma unroll
      for (int s = 0; s < KS; ++s) G.k[s] = u32x4{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < TPL; ++j) G.v[j] = u32x4{0, 0, 0, 0};
      return;
    }
    const int slot0 = (gl - entry * a.gpb) * 16;
    const uint16_t* kslot = a.pool + (static_cast<int64_t>(blk) * a.bs + slot0) * row_elems + kvh * dn;
    const uint16_t* krow = kslot + col * row_elems + grp * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s)
      G.k[s] = !PAD || grp * 8 + 32 * s < dn ? __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(krow + 32 * s))
                                             : u32x4{0, 0, 0, 0};
    const uint16_t* vrow = kslot + a.plane_elems + pv_dc * 8;
    const bool v_in = !PAD || pv_dc * 8 < dn;
#pragma unroll
    for (int j = 0; j < TPL; ++j)
      G.v[j] = v_in ? __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(vrow + (pv_tg * TPL + j) * row_elems))
                    : u32x4{0, 0, 0, 0};
  };
  auto compute_group = [&](const Group& G) {
    if (!G.ok) return;
    // ---- S^T = K Q^T: lane (col = query, grp) holds keys grp*4 + i ----
    f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) s4 = mma16<DT>(G.k[s], qf[s], s4);
    float tmax = -INFINITY;
    float sv[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = grp * 4 + i;
      const bool ok = t >= G.lo && t < G.hi;
      sv[i] = ok ? s4[i] * a.scale_log2 : -INFINITY;
      tmax = fmaxf(tmax, sv[i]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float m_new = fmaxf(m_run, tmax);
    const float alpha = exp2f(m_run - m_new);
    m_run = m_new;
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float p = __builtin_amdgcn_exp2f(sv[i] - m_new);
      psum += p;
      if (col < R) p_lds[wave][grp * 4 + i][col] = p;
    }
    l_run = l_run * alpha + psum;  // per-lane partial over its keys (rescaled)
    // alpha of query column c lives in lane c.
    float al[R];
#pragma unroll
    for (int c = 0; c < R; ++c) al[c] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(alpha), c));
#pragma unroll
    for (int c = 0; c < R; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[c][e] *= al[c];
    __builtin_amdgcn_wave_barrier();
    // ---- O += P V (VALU): lane owns 8 head-dim values of keys pv_tg*TPL .. +TPL ----
#pragma unroll
    for (int j = 0; j < TPL; ++j) {
      const int key = pv_tg * TPL + j;
      const bool ok = key >= G.lo && key < G.hi;
      const u32x4 vv = ok ? G.v[j] : u32x4{0, 0, 0, 0};
      float vf[8];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        vf[2 * w] = lo_half<DT>(vv[w]);
        vf[2 * w + 1] = hi_half<DT>(vv[w]);
      }
#pragma unroll
      for (int c4 = 0; c4 < R; c4 += 4) {
        const float4 p4 = *reinterpret_cast<const float4*>(&p_lds[wave][key][c4]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          acc[c4][e] += p4.x * vf[e];
          acc[c4 + 1][e] += p4.y * vf[e];
          acc[c4 + 2][e] += p4.z * vf[e];
          acc[c4 + 3][e] += p4.w * vf[e];
        }
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  // Rolling double buffer: group g + 1 is loading while group g is computed.
  Group ga, gb;
  if (g0 < g1) load_group(g0, ga);
  for (int g = g0; g < g1; g += 2) {
    if (g + 1 < g1) load_group(g + 1, gb);
    compute_group(ga);
    if (g + 2 < g1) load_group(g + 2, ga);
    if (g + 1 < g1) compute_group(gb);
  }

  // ---- epilogue: reduce over key subgroups, normalise, write the part ----
  const int64_t ws_row_base = static_cast<int64_t>(part) * a.batch * a.hq + static_cast<int64_t>(b) * a.hq;
  float l = l_run;
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);  // lanes with the same col now hold the total over keys
#pragma unroll
  for (int c = 0; c < R; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float v = acc[c][e];
      // Lanes with equal pv_dc hold the same d for different key subgroups.
      for (int off = DCH; off < 64; off *= 2) v += __shfl_xor(v, off);
      acc[c][e] = v;
    }
  if (a.subs > 1) {
    // The runs of a part meet in LDS; wave `sub` of a kv head finishes its query heads
    // sub, sub + subs, ...
    if (pv_tg == 0) {
#pragma unroll
      for (int c = 0; c < R; ++c)
#pragma unroll
        for (int e = 0; e < 8; e += 4)
          *reinterpret_cast<float4*>(&o_lds[wave][c][pv_dc * 8 + e]) =
              make_float4(acc[c][e], acc[c][e + 1], acc[c][e + 2], acc[c][e + 3]);
    }
    if (lane < R) {
      m_lds[wave][lane] = m_run;
      l_lds[wave][lane] = l;
    }
    __syncthreads();
    if (idle) return;
    const int w0 = wave - sub * a.heads;
    for (int c = sub; c < a.rep; c += a.subs) {
      float m = kNoMax;
      for (int i = 0; i < a.subs; ++i) m = fmaxf(m, m_lds[w0 + i * a.heads][c]);
      float o[D / 64] = {}, den = 0.f;
      for (int i = 0; i < a.subs; ++i) {
        const int w = w0 + i * a.heads;
        const float f = exp2f(m_lds[w][c] - m);
        den += f * l_lds[w][c];
#pragma unroll
        for (int k = 0; k < D / 64; ++k) o[k] += f * o_lds[w][c][lane + 64 * k];
      }
      const float inv = den > 0.f ? 1.f / den : 0.f;
      const int64_t row = ws_row_base + kvh * a.rep + c;
#pragma unroll
      for (int k = 0; k < D / 64; ++k)
        if (!PAD || lane + 64 * k < dn) a.ws_o[row * dn + lane + 64 * k] = o[k] * inv;
      if (lane == 0) a.ws_lse[row] = den == 0.f ? -INFINITY : (m + __log2f(den)) * kLn2;  // NaN stays
    }
    return;
  }
  float lc[R];
#pragma unroll
  for (int c = 0; c < R; ++c) lc[c] = __shfl(l, c);
  if (pv_tg == 0 && (!PAD || pv_dc * 8 < dn)) {
#pragma unroll
    for (int c = 0; c < R; ++c) {
      if (c >= a.rep) break;
      const float inv = lc[c] > 0.f ? 1.f / lc[c] : 0.f;
      float* orow = a.ws_o + (ws_row_base + kvh * a.rep + c) * dn + pv_dc * 8;
      reinterpret_cast<float4*>(orow)[0] =
          make_float4(acc[c][0] * inv, acc[c][1] * inv, acc[c][2] * inv, acc[c][3] * inv);
      reinterpret_cast<float4*>(orow)[1] =
          make_float4(acc[c][4] * inv, acc[c][5] * inv, acc[c][6] * inv, acc[c][7] * inv);
    }
  }
  if (lane < a.rep && lane < R) {
    // lane c holds column c's total; a NaN one (a NaN key) stays, so the merge cannot take
    // the part for an empty one
    a.ws_lse[ws_row_base + kvh * a.rep + lane] = l == 0.f ? -INFINITY : (m_run + __log2f(l)) * kLn2;
  }
}

struct DecodePlan {
  int parts, heads, subs;
};

// Query heads per kv head the PV accumulators hold: the smallest of 4, 8, 16 >= rep.
int decode_width(int rep) { return rep <= 4 ? 4 : rep <= 8 ? 8 : 16; }
constexpr int kMaxParts = 64;  // partials of one LSE merge

size_t align_up256(size_t x) { return (x + 255) & ~static_cast<size_t>(255); }
// Workspace of `parts` partials of every (sequence, head): o, then lse.
size_t parts_bytes(int parts, int batch, int hq, int d) {
  const size_t rows = static_cast<size_t>(parts) * batch * hq;
  return align_up256(rows * d * sizeof(float)) + align_up256(rows * sizeof(float));
}

// LDS in which the runs of a workgroup meet.
size_t meet_bytes(int d, int r, int subs) {
  return subs > 1 ? static_cast<size_t>(kDecWaves) * r * ((d == 64 ? 64 : 128) + 2) * sizeof(float) : 0;
}

// 16-token groups of the longest sequence that the spans allow.
int64_t span_groups(int n, const DecodeSpan* spans) {
  int64_t groups = 0;
  for (int i = 0; i < n; ++i)
    if (spans[i].t1 > spans[i].t0) groups += (spans[i].t1 + 15) / 16 - spans[i].t0 / 16;
  require(groups <= INT32_MAX / 2, "paged_decode: too many tokens");  // the kernel counts them in 32 bits
  return std::max<int64_t>(groups, 1);
}

// Most parts of a plan: what one merge takes, no more than the groups, and within the static
// scratch of the entry point that uses it (at least one).  Never fewer for more groups.
int most_parts(int batch, int hq, int d, int64_t groups) {
  const int64_t fit = HCP_DECODE_STATIC_SCRATCH_BYTES / (sizeof(float) * (d + 1) * std::max<int64_t>(1, int64_t(batch) * hq));
  int parts = static_cast<int>(std::min<int64_t>({groups, kMaxParts, std::max<int64_t>(1, fit)}));
  while (parts > 1 && parts_bytes(parts, batch, hq, d) > HCP_DECODE_STATIC_SCRATCH_BYTES) --parts;
  return parts;
}

// ceil(a / b) of values that nearly always fit 32 bits, whose division takes a third of the time.
static int64_t quot(int64_t a, int64_t b) {
  if (((a + b) >> 32) == 0) return (static_cast<uint32_t>(a) + static_cast<uint32_t>(b) - 1) / static_cast<uint32_t>(b);
  return ceil_div(a, b);
}

// The plan with the least modelled time, in us, over 1, 2, 4 or 8 runs a workgroup, all kv
// heads of it (up to 8), half of them and so on, and parts that make short runs (up to 8
// groups) or that give every CU 1, 2, 3, ... workgroups:
//   * the fullest CU's share of the groups at a CU's rate (`group` per 16 tokens of a kv head
//     of 128 dims), or the groups of a run one after another (`chain` each) times the rounds
//     of resident workgroups, whichever is longer.  A CU takes in at most its own rate, so a
//     workgroup count that does not divide over the CUs costs its whole last round: 130
//     sequences of 700 tokens, 24/4 heads, took 64.7 us as 390 workgroups of 8 waves, 45 as
//     1560 of one.  Workgroups that read part of a token's row cost 2.5% more, and if their
//     runs lie apart as well (runs that meet) up to a third: 32 sequences of 8000 tokens,
//     32/8 heads, 190 us as 8 runs of one head a workgroup, 164 as 8 parts of whole rows.
//     Where the tokens are more than the Infinity Cache holds and only 8 waves are resident
//     a CU (R = 8 of 128 dims), single runs of part rows cost 10% more: 32 sequences of 3000
//     tokens, 64/8 heads, 84 us as 6 parts of two heads, 75 as 8 of whole rows;
//   * `meet` where runs meet in LDS, the more the wider the accumulators: one sequence of 40
//     tokens, 32/2 heads of 64 dims, 20.0 us with four runs that meet, 13.6 as three parts;
//   * the parts written and read again, the merge's chain over them and its batches of
//     loads in flight (32 parts of 128 dims, 64 of 64);
//   * the start of every workgroup.
// Per accumulator width R = 4, 8, 16 and head dim 128, 64.  Fitted on MI355X to 602 calls: 12
// head layouts (8/1 to 64/8 heads of 64, 96 and 128 dims), 1-400 sequences of 40-16384
// tokens, some 70 plans each: the model's choice among them is 1.6% above the fastest on
// average.  Against as many runs as fill the chip once, the heads halved while more than 16
// parts resulted, these calls take 8% less on average; 32/8, 16/2 and 14/2 heads, 1-64
// sequences: none more than 6% longer.
DecodePlan plan_decode(int batch, int hq, int hkv, int d, int n, const DecodeSpan* spans) {
  static const double group[3][2] = {{0.181, 0.157}, {0.229, 0.146}, {0.281, 0.322}};
  static const double chain[3][2] = {{1.09, 0.84}, {1.37, 0.78}, {1.97, 1.36}};
  static const double meet[3] = {1.1, 1.95, 6.9};
  static const int waves_per_cu[3][2] = {{12, 16}, {8, 12}, {8, 8}};  // resident, by registers
  constexpr double kPartRows = 0.025, kApart = 0.047, kPartRowsHbm = 1.1, kCacheBytes = 240e6;
  constexpr double kPartValue = 4.4e-6, kPart = 0.029, kPartBatch = 0.8, kStart = 0.05;
  const int64_t groups = span_groups(n, spans);
  const int r = decode_width(hq / hkv), w = r <= 4 ? 0 : r <= 8 ? 1 : 2, h = d == 64 ? 1 : 0;
  const int cus = device_cus(), most = most_parts(batch, hq, d, groups);
  const int whole = static_cast<int>(ceil_div(hkv, ceil_div(hkv, kDecWaves)));
  const double part = kPartValue * batch * hq * d + kPart;
  const bool uncached = w == 1 && h == 0 && 64.0 * groups * batch * hkv * d > kCacheBytes;  // 16 tokens of K and V a group
  DecodePlan best{1, whole, 1};
  double best_t = 0.0;
  for (int heads = whole;; heads = (heads + 1) / 2) {
    const int64_t rows = static_cast<int64_t>(batch) * ceil_div(hkv, heads);
    for (int subs = 1; heads * subs <= kDecWaves; subs *= 2) {
      const int waves = heads * subs, resident = std::max(1, waves_per_cu[w][h] / waves);
      const double apart = subs > 1 ? kApart * (static_cast<double>(whole) / heads - 1.0) : 0.0;
      const double unit = group[w][h] * d / 128 * waves * (1.0 + (heads < whole ? kPartRows : 0.0) + apart) *
                          (uncached && heads < whole && subs == 1 ? kPartRowsHbm : 1.0);
      const int64_t shares = std::min<int64_t>(ceil_div(groups, subs), most);  // most parts
      // Candidates that cannot win are left out: no plan of these heads and subs is better
      // than its groups spread evenly, none than the chain of its runs (host time of a plan
      // 0.1-0.7 us; 1.0-2.3 with every candidate worked out, in 64-bit divisions).
      const double fixed = subs > 1 ? meet[w] : 0.0;
      if (best_t > 0.0 && unit * rows * groups / (static_cast<double>(subs) * cus) + fixed + part >= best_t) continue;
      uint64_t seen = 0;
      auto consider = [&](int64_t want) {
        want = std::min(std::max<int64_t>(want, 1), shares);
        if (seen >> (want - 1) & 1) return;
        seen |= uint64_t(1) << (want - 1);
        const int64_t len = quot(groups, subs * want);  // groups of a run
        if (best_t > 0.0 && chain[w][h] * len + fixed >= best_t) return;
        const int64_t parts = quot(groups, subs * len), per_cu = quot(rows * parts, cus);
        const double run = static_cast<double>(len);
        const double t = std::max(unit * per_cu * run, chain[w][h] * run * quot(per_cu, resident)) +
                         fixed + part * parts + kPartBatch * ((parts - 1) / (h ? 64 : 32)) +
                         kStart * per_cu;
        if (best_t == 0.0 || t < best_t) {
          best = DecodePlan{static_cast<int>(parts), heads, subs};
          best_t = t;
        }
      };
      for (int64_t len : {1, 2, 3, 4, 6, 8}) consider(quot(groups, subs * len));
      if (rows >= cus)
        for (int64_t parts : {1, 2, 3, 4, 6, 8, 12}) consider(parts);
      else
        for (int k : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16}) {
          const int parts = k * cus / static_cast<int>(rows);
          consider(parts);
          if (parts >= shares) break;
        }
    }
    if (heads == 1) break;
  }
  return best;
}

// Covers these spans and any shorter ones: a workspace sized once for the longest context
// serves all of them.
size_t decode_workspace_bytes(int batch, int hq, int d, int n, const DecodeSpan* spans) {
  return parts_bytes(most_parts(batch, hq, d, span_groups(n, spans)), batch, hq, d);
}

template <int D, int DT, bool PAD = false>
static void launch_decode_kernel(int r, dim3 grid, int waves, const DecodeArgs& a, hipStream_t stream) {
  const size_t lds = meet_bytes(D, r, a.subs);
  switch (r) {
    case 4: paged_decode_kernel<D, DT, 4, PAD><<<grid, 64 * waves, lds, stream>>>(a); break;
    case 8: paged_decode_kernel<D, DT, 8, PAD><<<grid, 64 * waves, lds, stream>>>(a); break;
    default: paged_decode_kernel<D, DT, 16, PAD><<<grid, 64 * waves, lds, stream>>>(a); break;
  }
}

void launch_paged_decode(int dtype, int batch, int hq, int hkv, int d, const void* q, int64_t q_bs,
                         int64_t q_hs, const void* pool, int64_t num_blocks, int bs, int n,
                         const DecodeSpan* spans, float scale, int out_dtype, void* out, int64_t out_rs, float* lse,
                         void* ws, size_t ws_bytes, int* err, hipStream_t stream) {
  require(hq % hkv == 0 && hq / hkv <= 16, "paged_decode: num_q_heads/num_kv_heads must be <= 16");
  require(bs % 16 == 0, "paged_decode: block_size must be a multiple of 16");
  require(d > 0 && d <= 128 && d % 8 == 0, "paged_decode: head_dim must be a multiple of 8 up to 128");
  require(dtype == kBF16 || dtype == kF16, "paged_decode: dtype must be BF16 or F16");
  require(n >= 1 && n <= kMaxDomains, "paged_decode: 1 to 64 shards");
  for (int i = 0; i < n; ++i) require(spans[i].t0 >= 0 && spans[i].t0 < bs, "paged_decode: a span starts in its first block");
  const DecodePlan p = plan_decode(batch, hq, hkv, d, n, spans);
  const size_t need = parts_bytes(p.parts, batch, hq, d);
  require(ws != nullptr && ws_bytes >= need, "workspace too small: need " + std::to_string(need) + " bytes");
  const size_t rows = static_cast<size_t>(p.parts) * batch * hq;
  float* ws_o = static_cast<float*>(ws);
  float* ws_lse = reinterpret_cast<float*>(static_cast<char*>(ws) + align_up256(rows * d * sizeof(float)));

  DecodeArgs a;
  a.q = static_cast<const uint16_t*>(q);
  a.q_bs = q_bs;
  a.q_hs = q_hs;
  a.pool = static_cast<const uint16_t*>(pool);
  a.plane_elems = num_blocks * bs * hkv * static_cast<int64_t>(d);
  a.num_blocks = num_blocks;
  a.bs = bs;
  a.hkv = hkv;
  a.hq = hq;
  a.rep = hq / hkv;
  a.n_spans = n;
  for (int i = 0; i < n; ++i) a.span[i] = spans[i];
  a.heads = p.heads;
  a.subs = p.subs;
  a.gpb = bs / 16;
  a.gpb_shift = (a.gpb & (a.gpb - 1)) == 0 ? __builtin_ctz(a.gpb) : -1;
  a.scale_log2 = scale * kLog2e;
  a.ws_o = ws_o;
  a.ws_lse = ws_lse;
  a.batch = batch;
  a.err = err;
  a.dn = d;
  const int waves = p.heads * p.subs;
  const int r = decode_width(a.rep);
  const dim3 grid(static_cast<unsigned>(p.parts), static_cast<unsigned>(batch),
                  static_cast<unsigned>(ceil_div(hkv, p.heads)));
  // head dim 64: its own kernel; other multiples of 8 up to 128: the D=128 kernel with
  // the columns past d zero-padded
  if (dtype == kBF16) {
    if (d == 128) launch_decode_kernel<128, kBF16>(r, grid, waves, a, stream);
    else if (d == 64) launch_decode_kernel<64, kBF16>(r, grid, waves, a, stream);
    else launch_decode_kernel<128, kBF16, true>(r, grid, waves, a, stream);
  } else {
    if (d == 128) launch_decode_kernel<128, kF16>(r, grid, waves, a, stream);
    else if (d == 64) launch_decode_kernel<64, kF16>(r, grid, waves, a, stream);
    else launch_decode_kernel<128, kF16, true>(r, grid, waves, a, stream);
  }
  HCP_HIP(hipGetLastError());
  // Merge the parts of every (sequence, head): rows = batch*hq, one token each.
  const float* o_parts[kMaxParts];
  const float* l_parts[kMaxParts];
  for (int i = 0; i < p.parts; ++i) {
    o_parts[i] = ws_o + static_cast<size_t>(i) * batch * hq * d;
    l_parts[i] = ws_lse + static_cast<size_t>(i) * batch * hq;
  }
  launch_lse_merge(p.parts, o_parts, l_parts, batch * hq, 1, d, out_dtype, out, out_rs, out_rs, lse, 1, stream);
}

}  // namespace hcp
