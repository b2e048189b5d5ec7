// Fused QKV projection + RoPE + KV append: the producer of the ring operator's inputs.
//
// Replaces the head of HcpRingAttentionBackend::forward (ring.rs:1865-1936): three
// projections x W^T (+ bias), the head split, the rotary embedding of q and k
// (RotaryEmbedding::apply / rotate_pairs, rust/src/model/layers/rotary.rs:103-158) at
// each token's global position, and the KV-cache append (KvCache::update,
// cache.rs:191-251; the positioned slab append of self_driving.rs:180-228), as one
// matrix-core GEMM whose epilogue does everything after the accumulation:
//
//   * C^T = W X^T on v_mfma_f32_32x32x16 (A = weight rows, B = token rows, both
//     hidden-contiguous), so a lane owns one token and 16 features of each 32-feature
//     block.  A workgroup computes 256 features x 128, 256 or 384 tokens, 384 features
//     x 256 tokens or 128 x 128 (chosen per launch) with 8 waves of 64 features x half
//     the tokens, 192 x a quarter or 64 x a quarter: a wave's features come in pairs of
//     32-feature blocks at d and d + D/2 of one head, so each RoPE partner pair sits in
//     the same lane and register slot of the wave's two blocks -- the rotation needs no
//     data exchange.
//   * Weight and token tiles of 32 hidden values reach LDS through buffer_load ... lds
//     (four buffers, three stages in flight, eight and seven for 128 x 128 tiles; one
//     barrier per stage); chunk p of tile row r holds global chunk p ^ ((r >> 2) & 3),
//     which keeps the fragment reads free of bank conflicts.  The loop is software-pipelined:
//     a stage's DMA instructions are spread through the MFMAs of the stage three before it,
//     the second K half's fragments are read while the first half's MFMAs run, and the next
//     stage's barrier sits inside this stage's second half, so its first fragments arrive
//     while the matrix core still has this stage's MFMAs queued (measured on the Llama-3-8B layer:
//     +7.6% over one barrier and one DMA burst at each stage start).
//   * Epilogue, in fp32: + bias, rotate (x1 cos - x2 sin, x1 sin + x2 cos) with cos/sin
//     from the table row of the token's position, round once to the storage dtype and
//     store 8 consecutive head dims (16 bytes) per lane -- the two lanes holding halves
//     of an 8-dim group swap them with v_permlane32_swap, half the store instructions of
//     8-byte stores (+2.3% on the Llama-3-8B layer); 8-byte stores when a row start is
//     not 16-byte aligned: q into [Hq, L, D], k / v into [Hkv, L, D] views or appended to
//     the paged pool through the block table.
#include <cmath>

#include "kernels.hpp"
#include "lds_dma.hpp"

namespace hcp {


namespace {

constexpr int kQWaves = 8;
constexpr int kQThreads = kQWaves * 64;
constexpr int kQK = 32;                      // hidden values per stage
constexpr int kQRow = kQK * 2;               // bytes per tile row in LDS
constexpr int kQGroupM = 4;                  // token tiles per placement group

template <int DT>
struct QkvMfma;
template <>
struct QkvMfma<kBF16> {
  typedef bf16x8 frag;
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct QkvMfma<kF16> {
  typedef f16x8 frag;
  static __device__ __forceinline__ f32x16 mma(frag a, frag b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

__device__ __forceinline__ uint32_t qswz(int r) { return static_cast<uint32_t>((r >> 2) & 3); }

template <int DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  if constexpr (DT == kBF16) return f32x2_to_bf16x2_bits(a, b);
  else return static_cast<uint32_t>(f32_to_f16_bits(a)) | (static_cast<uint32_t>(f32_to_f16_bits(b)) << 16);
}

template <int DT>
__device__ __forceinline__ float ld16(const uint16_t* p) {
  return DT == kBF16 ? bf16_bits_to_f32(*p) : f16_bits_to_f32(*p);
}

// TF features x TN tokens per workgroup.  Each wave owns 2 x OB blocks of 32 x 32: with
// TF = 256 the features fbase and fbase + D/2 of one head (RoPE partners; group wf = w & 3)
// times the TN/2 tokens of half wt = w >> 2; with TF = 384 three such pairs 128 features
// apart (group wf = w & 1) times the 64 tokens of quarter wt = w >> 1; with TF = 128 one
// pair (group w & 1) times the 32 tokens of quarter w >> 1.  The side with more
// blocks is the outer one of the MFMA order, each of its fragments used for two MFMAs.
template <int DT, int D, int TF, int TN>
__global__ __launch_bounds__(kQThreads, 1) void qkv_rope_kernel(QkvArgs a) {
  using Ops = QkvMfma<DT>;
  using frag = typename Ops::frag;
  static_assert(TF == 256 || (TF == 384 && TN == 256) || (TF == 128 && TN == 128), "tile shapes");
  constexpr bool kFeatOuter = TF == 384;
  constexpr int WF = TF == 256 ? 4 : 2;         // feature groups of waves
  constexpr int WT = kQWaves / WF;              // token groups
  constexpr int OB = kFeatOuter ? 6 : TN / WT / 32;  // outer 32-blocks per wave (2 inner ones)
  constexpr int NP = kFeatOuter ? 3 : 1;        // RoPE pairs per wave
  constexpr int NT = kFeatOuter ? 2 : OB;       // 32-token blocks per wave
  constexpr int WJ = TF / 128;                  // weight-row DMA instructions per wave per stage
  constexpr int XJ = TN / 128;                  // token-row DMA instructions per wave per stage
  constexpr int kOperandW = TF * kQRow;
  constexpr int kOperandX = TN * kQRow;
  constexpr int kStage = kOperandW + kOperandX;
  constexpr int NB = TF == 128 ? 8 : 4;         // stage buffers, NB - 1 stages in flight
  constexpr int kPerStage = WJ + XJ;            // DMA instructions per wave per stage
  constexpr int kPair = D / 64;                 // pairs per head
  __shared__ __attribute__((aligned(1024))) uint8_t lds[NB * kStage];

  // ---- placement: groups of kQGroupM token tiles x every feature tile ----
  const int logical = xcd_remap(blockIdx.x, gridDim.x);
  const int per_group = kQGroupM * a.n_tiles_n;
  const int first_m = (logical / per_group) * kQGroupM;
  const int gsize = min(a.n_tiles_m - first_m, kQGroupM);
  const int in_group = logical % per_group;
  const int tok0 = (first_m + in_group % gsize) * TN;
  const int feat0 = (in_group / gsize) * TF;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int lcol = lane & 31, lhalf = lane >> 5;
  const int wf = wave % WF;  // feature group
  const int wt = wave / WF;  // token group
  const int fbase = D * (wf / kPair) + 32 * (wf % kPair);  // first feature of the group in the tile
  const int n_feat = a.nq + 2 * a.nkv;

  // ---- DMA roles: wave w copies weight rows (TF / 8) w .. (TF / 8) (w + 1) - 1, 16 an
  // instruction, and token rows (TN / 8) w .. (TN / 8) (w + 1) - 1 ----
  u32x4 srd_w[WJ];
#pragma unroll
  for (int j = 0; j < WJ; ++j) {
    const int frow = feat0 + (TF / 8) * wave + 16 * j;  // 16 rows never straddle q/k/v (boundaries are multiples of 128)
    int which = 0, local = frow;
    if (frow >= a.nq + a.nkv) {
      which = 2;
      local = frow - a.nq - a.nkv;
    } else if (frow >= a.nq) {
      which = 1;
      local = frow - a.nq;
    }
    const int64_t rows_left = frow >= n_feat ? 0 : (which == 0 ? a.nq : a.nkv) - local;
    srd_w[j] = make_srd(a.w[which] + static_cast<int64_t>(local) * a.hidden, rows_left * a.hidden * 2);
  }
  const int trow = tok0 + (TN / 8) * wave;
  const u32x4 srd_x = make_srd(a.x + static_cast<int64_t>(trow) * a.x_ss,
                               trow >= a.tokens ? 0 : (static_cast<int64_t>(a.tokens - trow) * a.x_ss * 2));
  // row lane >> 2 of an instruction's 16 weight rows; 16 instructions apart the swizzle key
  // (of the tile row) is the same
  const uint32_t w_voff = static_cast<uint32_t>((lane >> 2) * a.hidden * 2) + (((lane & 3) ^ qswz(lane >> 2)) << 4);
  uint32_t x_voff[XJ];
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const int r = 16 * j + (lane >> 2);        // row within the wave's token rows
    const int tr = (TN / 8) * wave + r;
    x_voff[j] = static_cast<uint32_t>(r * a.x_ss * 2) + (((lane & 3) ^ qswz(tr)) << 4);
  }
  const uint32_t lds0 = lds_offset(lds);
  // DMA instruction j (< kPerStage) of stage st into buffer buf: weight rows first.
  auto issue_one = [&](int st, int buf, int j) __attribute__((always_inline)) {
    const uint32_t kb = static_cast<uint32_t>(st) * kQRow;
    if (j < WJ) {
      dma16(srd_w[j], w_voff + kb, lds0 + buf * kStage + wave * ((TF / 8) * kQRow) + j * 1024);
    } else {
      dma16(srd_x, x_voff[j - WJ] + kb, lds0 + buf * kStage + kOperandW + wave * ((TN / 8) * kQRow) + (j - WJ) * 1024);
    }
  };
  auto issue = [&](int st, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < kPerStage; ++j) issue_one(st, buf, j);
  };

  // ---- fragment read offsets (bytes within a stage buffer) ----
  // Rows 32, 128 and D/2 apart share the swizzle key ((r >> 2) & 3 is unchanged by a
  // multiple of 16), so one offset per sub-step and operand serves every block.
  uint32_t w_rd[2], x_rd[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int c = 2 * s + lhalf;
    const int rw = fbase + lcol;
    w_rd[s] = rw * kQRow + ((c ^ qswz(rw)) << 4);
    const int rx = (TN / WT) * wt + lcol;
    x_rd[s] = kOperandW + rx * kQRow + ((c ^ qswz(rx)) << 4);
  }
  static_assert((D / 2) % 16 == 0, "swizzle key shared across the weight blocks");
  // fragment offsets: weight block k is half k % 2 of pair k / 2, token block k rows 32 k on
  auto w_at = [&](int s, int k) __attribute__((always_inline)) {
    return w_rd[s] + (128 * (k / 2) + (D / 2) * (k % 2)) * kQRow;
  };
  auto x_at = [&](int s, int k) __attribute__((always_inline)) { return x_rd[s] + 32 * k * kQRow; };
  auto in_at = [&](int s, int k) __attribute__((always_inline)) { return kFeatOuter ? x_at(s, k) : w_at(s, k); };
  auto out_at = [&](int s, int k) __attribute__((always_inline)) { return kFeatOuter ? w_at(s, k) : x_at(s, k); };
  auto mma = [](frag in, frag out, f32x16 c) __attribute__((always_inline)) {
    return kFeatOuter ? Ops::mma(out, in, c) : Ops::mma(in, out, c);
  };

  f32x16 acc[2][OB];  // [inner block][outer block]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int o = 0; o < OB; ++o)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][o][r] = 0.f;

  const int n_st = a.hidden / kQK;
#pragma unroll
  for (int st = 0; st < NB - 1; ++st)
    if (st < n_st) issue(st, st);

  // Stage st resident for every wave: this wave's DMA of it done (at most the stages
  // issued after it still in flight), this wave's reads of older stages done, then the
  // barrier.
  auto sync_stage = [&](int st) __attribute__((always_inline)) {
    const int after = min(NB - 2, max(0, n_st - 1 - st));
    if (after == NB - 2) wait_vmcnt<(NB - 2) * kPerStage>();
    else if (NB > 4 && after >= 4) wait_vmcnt<4 * kPerStage>();
    else if (NB > 4 && after >= 2) wait_vmcnt<2 * kPerStage>();
    else if (after == 1) wait_vmcnt<kPerStage>();
    else wait_vmcnt<0>();
    wait_lgkmcnt0();
    __syncthreads();
  };
  auto rd = [&](int bf, uint32_t off) __attribute__((always_inline)) {
    return __builtin_bit_cast(frag, *reinterpret_cast<const u32x4*>(lds + bf * kStage + off));
  };
  // MFMA (flat index over the stage) after which the next stage's barrier sits: after the
  // last DMA instruction and at least two outer blocks into the second K half.
  constexpr int kGap = OB == 1 ? 1 : 3;    // one DMA instruction after every third MFMA from the second
  constexpr int kOff = OB == 1 ? 0 : 1;    // (128 x 128 tiles: after each from the first)
  constexpr int kLast = kGap * (kPerStage - 1) + kOff;
  constexpr int kMidB = OB == 1 ? 3 : 2 * OB + 3;
  constexpr int kMidA = kLast > kMidB ? kLast : kMidB;
  constexpr int kMid = kMidA % 2 ? kMidA : kMidA + 1;
  constexpr int kMidO = (kMid - 2 * OB) / 2;  // last second-half outer block before it
  static_assert(kMid < 4 * OB, "barrier inside the stage");
  static_assert(kLast < 4 * OB, "every DMA instruction issued inside the stage");

  frag in0[2], out0[OB];  // first-half fragments of the current stage, read ahead
  if (n_st > 0) {
    sync_stage(0);
#pragma unroll
    for (int i = 0; i < 2; ++i) in0[i] = rd(0, in_at(0, i));
#pragma unroll
    for (int o = 0; o < OB; ++o) out0[o] = rd(0, out_at(0, o));
  }
  // compute(st, bufc): the MFMAs of stage st (buffer bufc).  The DMA of stage st + NB - 1
  // (into buffer bufc - 1, last read in stage st - 1, before this stage's barrier) is
  // spread through them, so the waves' address traffic does not queue at the stage start.
  auto compute = [&](int st, auto bufc) __attribute__((always_inline)) {
    constexpr int bf = decltype(bufc)::value;
    constexpr int nb = (bf + 1) % NB;
    const int pf = st + NB - 1 < n_st ? st + NB - 1 : -1;
    auto dma_after = [&](int m) __attribute__((always_inline)) {
      if (m % kGap == kOff % kGap && m / kGap < kPerStage && pf >= 0) {
        __builtin_amdgcn_sched_barrier(0);
        issue_one(pf, (bf + NB - 1) % NB, m / kGap);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    frag in1[2], out1[OB];
#pragma unroll
    for (int o = 0; o < OB; ++o) {
      if (o == OB - 1) {
#pragma unroll
        for (int i = 0; i < 2; ++i) in1[i] = rd(bf, in_at(1, i));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc[i][o] = mma(in0[i], out0[o], acc[i][o]);
        dma_after(2 * o + i);
      }
      out1[o] = rd(bf, out_at(1, o));
    }
#pragma unroll
    for (int o = 0; o < OB; ++o) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int m = 2 * OB + 2 * o + i;
        acc[i][o] = mma(in1[i], out1[o], acc[i][o]);
        dma_after(m);
        if (m == kMid) {  // after the last stage: an extra barrier and unused reads
          sync_stage(st + 1);
#pragma unroll
          for (int j = 0; j < 2; ++j) in0[j] = rd(nb, in_at(0, j));
#pragma unroll
          for (int t = 0; t <= kMidO; ++t) out0[t] = rd(nb, out_at(0, t));
        }
      }
      if (o > kMidO) out0[o] = rd(nb, out_at(0, o));
    }
  };
  for (int st = 0; st < n_st; st += NB) {
    compute(st, IntC<0>{});
    if (st + 1 < n_st) compute(st + 1, IntC<1>{});
    if (st + 2 < n_st) compute(st + 2, IntC<2>{});
    if (st + 3 < n_st) compute(st + 3, IntC<3>{});
    if constexpr (NB == 8) {
      if (st + 4 < n_st) compute(st + 4, IntC<4>{});
      if (st + 5 < n_st) compute(st + 5, IntC<5>{});
      if (st + 6 < n_st) compute(st + 6, IntC<6>{});
      if (st + 7 < n_st) compute(st + 7, IntC<7>{});
    }
  }

  // ---- epilogue ----
#pragma unroll
  for (int pr = 0; pr < NP; ++pr) {
    const int fw0 = feat0 + fbase + 128 * pr;  // first feature of the pair
    if (fw0 >= n_feat) return;
    int ow = 0, of = fw0;              // output tensor and its feature offset
    if (fw0 >= a.nq + a.nkv) {
      ow = 2;
      of = fw0 - a.nq - a.nkv;
    } else if (fw0 >= a.nq) {
      ow = 1;
      of = fw0 - a.nq;
    }
    const uint16_t* bias = a.bias[ow];
    const bool rot = a.rope && ow < 2;
    const int head = of / D;
    const int dh = of % D;             // head dim of block 0 (block 1 is dh + D/2)
    // 16-byte stores need every row start 16-byte aligned
    const bool st16 = (ow == 0 || a.pool == nullptr)
                          ? ((reinterpret_cast<uintptr_t>(a.out[ow]) | static_cast<uintptr_t>(a.out_hs[ow]) * 2 |
                              static_cast<uintptr_t>(a.out_ss[ow]) * 2) % 16) == 0
                          : reinterpret_cast<uintptr_t>(a.pool) % 16 == 0;
#pragma unroll
    for (int tb = 0; tb < NT; ++tb) {
      const int t = tok0 + (TN / WT) * wt + 32 * tb + lcol;
      if (t >= a.tokens) continue;
      float v[2][16];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int lf = (D / 2) * i + 8 * (r >> 2) + 4 * lhalf + (r & 3);
          v[i][r] = (kFeatOuter ? acc[tb][2 * pr + i][r] : acc[i][tb][r]) + (bias ? ld16<DT>(bias + of + lf) : 0.f);
        }
      if (rot) {
        const int64_t p = a.pos[t];
        if (p < 0 || p >= a.rope_rows) {
          if (lhalf == 0) atomicOr(a.err, 4);
        } else {
          const float* crow = a.rope_cos + p * (D / 2);
          const float* srow = a.rope_sin + p * (D / 2);
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int d0 = dh + 8 * g + 4 * lhalf;
            const float4 cs = *reinterpret_cast<const float4*>(crow + d0);
            const float4 sn = *reinterpret_cast<const float4*>(srow + d0);
            const float cc[4] = {cs.x, cs.y, cs.z, cs.w}, ss[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const float x1 = v[0][4 * g + i], x2 = v[1][4 * g + i];
              v[0][4 * g + i] = x1 * cc[i] - x2 * ss[i];
              v[1][4 * g + i] = x1 * ss[i] + x2 * cc[i];
            }
          }
        }
      }
      // store 4 consecutive head dims per (block, group)
      int32_t blk = 0;
      int64_t slot = 0;
      if (ow != 0 && a.pool != nullptr) {
        const int64_t sp = a.t0 + t - a.table_off;  // position of this token in the table
        const int64_t entry = sp / a.bs;
        blk = (sp >= 0 && entry < a.table_len) ? a.table[entry] : -1;
        if (blk < 0 || blk >= a.num_blocks) {
          if (lhalf == 0) atomicOr(a.err, 1);
          continue;
        }
        slot = sp - entry * a.bs;
      }
      uint16_t* row;
      if (ow == 0 || a.pool == nullptr) {
        row = a.out[ow] + head * a.out_hs[ow] + static_cast<int64_t>(t) * a.out_ss[ow];
      } else {
        row = a.pool + (ow == 2 ? a.plane_elems : 0) + ((static_cast<int64_t>(blk) * a.bs + slot) * a.hkv + head) * D;
      }
      u32x2 pk[2][4];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          pk[i][g][0] = pack2<DT>(v[i][4 * g], v[i][4 * g + 1]);
          pk[i][g][1] = pack2<DT>(v[i][4 * g + 2], v[i][4 * g + 3]);
        }
      if (st16) {
        // lanes 0-31 hold dims +0..3 of each 8-dim group, lanes 32-63 dims +4..7: after the
        // swap of groups (g, g + 1) lane lhalf = 0 holds all 8 dims of group g + 1 and
        // lhalf = 1 those of group g
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int g = 0; g < 4; g += 2) {
            u32x4 w;
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              const auto r = __builtin_amdgcn_permlane32_swap(pk[i][g + 1][k], pk[i][g][k], false, false);
              w[k] = r[0];
              w[2 + k] = r[1];
            }
            const int gs = g + 1 - lhalf;
            *reinterpret_cast<u32x4*>(row + dh + (D / 2) * i + 8 * gs) = w;
          }
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *reinterpret_cast<u32x2*>(row + dh + (D / 2) * i + 8 * g + 4 * lhalf) = pk[i][g];
      }
    }
  }
}

// Few tokens (a decode step, the tail of a prompt): the projection reads every weight for
// a handful of rows, so it is bound by the weights' bytes, and the tiled kernel's few
// workgroups (24 for a Llama-3-8B layer) leave most CUs idle.  Here a workgroup owns 32
// features -- 16 and their RoPE partners D/2 above -- times 16 TB tokens, and its 8 waves
// split the hidden dimension: each wave takes every eighth 64-value slice, streams its
// weight and token fragments straight from memory into registers (a weight is used by one
// wave only, so LDS would add nothing), and the eight partial tiles meet in LDS once, in a
// fixed order.  v_mfma_f32_16x16x32: A = 16 weight rows, B = 16 token rows; a lane owns
// one token and features 4 (lane / 16) .. + 3 of each 16.
// Measured on the Llama-3-8B layer (50 MB of weights): 1 token 12.4 us (was 46), 64 tokens
// 26 us (was 51).  At one token it is at the weights' 10 us; beyond, each workgroup also
// takes in every token row (8 KiB a token), and the CUs' intake, about 35 GB/s each,
// bounds it: whole 128-byte lines per load, a per-workgroup rotation of the slices and a
// deeper weight prefetch all measured the same or slower.
typedef float qf32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ qf32x4 mma16(bf16x8 a, bf16x8 b, qf32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ qf32x4 mma16(f16x8 a, f16x8 b, qf32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

template <int DT, int D, int TB>
__global__ __launch_bounds__(kQThreads, 1) void qkv_few_tokens_kernel(QkvArgs a) {
  using frag = typename QkvMfma<DT>::frag;
  constexpr int kPerHead = D / 32;           // feature tiles per head
  constexpr int SG = TB >= 8 ? 2 : 4;        // hidden steps (of 32) per load group
  constexpr uint32_t kOut = 0x80000000u;     // past every descriptor's records: reads zeros
  __shared__ __attribute__((aligned(16))) qf32x4 red[kQWaves][2][TB][64];

  const int logical = xcd_remap(blockIdx.x, gridDim.x);  // token tiles of a feature tile share its XCD's L2
  const int ft = logical / a.n_tiles_m;
  const int tok0 = (logical - ft * a.n_tiles_m) * 16 * TB;
  const int head = ft / kPerHead;            // over the q, k and v heads in turn
  const int d0 = (ft - head * kPerHead) * 16;
  const int nhq = a.nq / D, nhkv = a.nkv / D;
  const int which = head < nhq ? 0 : head < nhq + nhkv ? 1 : 2;
  const int lh = head - (which == 0 ? 0 : which == 1 ? nhq : nhq + nhkv);

  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int col = lane & 15, grp = lane >> 4;

  const uint16_t* wbase = a.w[which] + (static_cast<int64_t>(lh) * D + d0) * a.hidden;
  const auto wr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(wbase), 0, (D / 2 + 16) * a.hidden * 2, 0x00020000);
  const int rows = min(a.tokens - tok0, 16 * TB);
  const uint16_t* xbase = a.x + static_cast<int64_t>(tok0) * a.x_ss;
  const int x_rb = static_cast<int>(a.x_ss) * 2;
  const auto xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(xbase), 0, (rows - 1) * x_rb + a.hidden * 2, 0x00020000);
  const uint32_t w_off = static_cast<uint32_t>(col * a.hidden * 2 + grp * 16);
  const uint32_t x_off = static_cast<uint32_t>(col * x_rb + grp * 16);

  // Slice s of the hidden dimension is steps 2s and 2s + 1 (64 values, a 128-byte line of
  // each row); this wave's j-th step is step 2 (wave + 8 (j / 2)) + j % 2.
  const int n_st = a.hidden / kQK;
  const int n_sl = (n_st + 1) / 2;
  const int mine = wave < n_sl ? 2 * ((n_sl - wave + kQWaves - 1) / kQWaves) : 0;
  struct Group {
    u32x4 w[SG][2];
    u32x4 x[SG][TB];
  };
  auto load = [&](int j0, Group& g) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SG; ++j) {
      const int st = 2 * (wave + kQWaves * ((j0 + j) / 2)) + (j & 1);
      const uint32_t k = st < n_st ? static_cast<uint32_t>(st) * (kQK * 2) : kOut;
#pragma unroll
      for (int b = 0; b < 2; ++b)
        g.w[j][b] = __builtin_amdgcn_raw_buffer_load_b128(wr, w_off + k + static_cast<uint32_t>(b * (D / 2) * a.hidden * 2), 0, 0);
#pragma unroll
      for (int t = 0; t < TB; ++t)
        g.x[j][t] = __builtin_amdgcn_raw_buffer_load_b128(xr, x_off + k + static_cast<uint32_t>(16 * t * x_rb), 0, 0);
    }
  };
  qf32x4 acc[2][TB];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int t = 0; t < TB; ++t) acc[b][t] = qf32x4{0.f, 0.f, 0.f, 0.f};
  auto fold = [&](const Group& g) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < SG; ++j)
#pragma unroll
      for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int b = 0; b < 2; ++b)
          acc[b][t] = mma16(__builtin_bit_cast(frag, g.w[j][b]), __builtin_bit_cast(frag, g.x[j][t]), acc[b][t]);
  };
  Group ga, gb;
  load(0, ga);
  for (int j0 = 0; j0 < mine; j0 += 2 * SG) {
    load(j0 + SG, gb);
    fold(ga);
    load(j0 + 2 * SG, ga);
    fold(gb);
  }
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int t = 0; t < TB; ++t) red[wave][b][t][lane] = acc[b][t];
  __syncthreads();

  // ---- epilogue: wave t finishes token block t ----
  if (wave >= TB) return;
  const int t = tok0 + 16 * wave + col;
  if (t >= a.tokens) return;
  float v[2][4];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    qf32x4 sum = red[0][b][wave][lane];
#pragma unroll
    for (int w = 1; w < kQWaves; ++w) sum += red[w][b][wave][lane];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[b][i] = sum[i];
  }
  const int dh = d0 + 4 * grp;               // head dims dh .. + 3 and their partners + D/2
  if (const uint16_t* bias = a.bias[which]) {
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[b][i] += ld16<DT>(bias + lh * D + dh + b * (D / 2) + i);
  }
  if (a.rope && which < 2) {
    const int64_t p = a.pos[t];
    if (p < 0 || p >= a.rope_rows) {
      if (grp == 0) atomicOr(a.err, 4);
    } else {
      const float4 cs = *reinterpret_cast<const float4*>(a.rope_cos + p * (D / 2) + dh);
      const float4 sn = *reinterpret_cast<const float4*>(a.rope_sin + p * (D / 2) + dh);
      const float cc[4] = {cs.x, cs.y, cs.z, cs.w}, ss[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x1 = v[0][i], x2 = v[1][i];
        v[0][i] = x1 * cc[i] - x2 * ss[i];
        v[1][i] = x1 * ss[i] + x2 * cc[i];
      }
    }
  }
  uint16_t* row;
  if (which == 0 || a.pool == nullptr) {
    row = a.out[which] + lh * a.out_hs[which] + static_cast<int64_t>(t) * a.out_ss[which];
  } else {
    const int64_t sp = a.t0 + t - a.table_off;  // position of this token in the table
    const int64_t entry = sp / a.bs;
    const int32_t blk = (sp >= 0 && entry < a.table_len) ? a.table[entry] : -1;
    if (blk < 0 || blk >= a.num_blocks) {
      if (grp == 0) atomicOr(a.err, 1);
      return;
    }
    row = a.pool + (which == 2 ? a.plane_elems : 0) +
          ((static_cast<int64_t>(blk) * a.bs + (sp - entry * a.bs)) * a.hkv + lh) * D;
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    u32x2 w;
    w[0] = pack2<DT>(v[b][0], v[b][1]);
    w[1] = pack2<DT>(v[b][2], v[b][3]);
    *reinterpret_cast<u32x2*>(row + dh + b * (D / 2)) = w;
  }
}

constexpr int kRopeThreads = 256;
struct RopeArgs {
  float inv_freq[128];
  int32_t half;
  int64_t rows;
  float* cos;
  float* sin;
};

__global__ __launch_bounds__(kRopeThreads) void rope_table_kernel(RopeArgs a) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kRopeThreads + threadIdx.x;
  if (i >= a.rows * a.half) return;
  const int64_t m = i / a.half;
  const int j = static_cast<int>(i - m * a.half);
  // positions are exact in fp32 below 2^24; angle = m * inv_freq[j] in fp32
  const float ang = static_cast<float>(m) * a.inv_freq[j];
  a.cos[i] = cosf(ang);
  a.sin[i] = sinf(ang);
}

}  // namespace

void launch_rope_table(int d, int64_t rows, double base, float* cos, float* sin, hipStream_t stream) {
  require(d % 2 == 0 && d / 2 <= 128, "rope: head_dim must be even and <= 256");
  RopeArgs a{};
  a.half = d / 2;
  for (int j = 0; j < a.half; ++j)  // rotary.rs:72-78: 1 / base^(2j / dim) in f64, then f32
    a.inv_freq[j] = static_cast<float>(1.0 / std::pow(base, (2.0 * j) / d));
  a.rows = rows;
  a.cos = cos;
  a.sin = sin;
  const int64_t n = rows * a.half;
  if (n == 0) return;
  rope_table_kernel<<<static_cast<unsigned>(ceil_div(n, kRopeThreads)), kRopeThreads, 0, stream>>>(a);
  HCP_HIP(hipGetLastError());
}

// Tile (features x tokens) of 256 x 128, 256 x 256, 256 x 384, 384 x 256 or 128 x 128: the
// one with the least modelled time, i.e. rounds of workgroups over the device's compute
// units times the time one tile of that size takes relative to 256 x 256 (bigger tiles reuse
// each LDS fragment more), a partly filled last round counted as 0.5 + 0.5 x its fill (it
// runs at a higher clock with part of the chip idle).  Fitted to a sweep of the Llama-3-8B
// projection over 1024-24576 tokens on MI355X, the 128 x 128 tile to 150-8192 tokens of it
// and of Qwen2.5-3B's and Qwen2-0.5B's.  Llama-3-8B at 12288 tokens: 768 tiles of 256 x 384
// are 3 full rounds of 256 CUs; at 4096 tokens 256 of 384 x 256 are one, 177 us (384 of
// 256 x 256, one round and a half: 232); at 8192 tokens 354 against 376.  128 x 128 spreads a
// launch that fills less than a round over twice the CUs of 256 x 128: 256 tokens of
// Llama-3-8B 36 us against 55, 1024 of Qwen2.5-3B 25 against 37, 2048 of Qwen2-0.5B 17
// against 25; over more than a round it is the slower one (768 of Llama-3-8B: 74 against 72).
struct QkvTile {
  int tf, tn;
};
static QkvTile qkv_tile(int64_t n_feat, int64_t tokens) {
  const int cus = device_cus();
  const QkvTile tiles[5] = {{256, 256}, {256, 128}, {256, 384}, {384, 256}, {128, 128}};
  const double cost[5] = {1.0, 0.62, 1.41, 1.41, 0.42};
  int best = 0;
  double best_t = 0.0;
  for (int i = 0; i < 5; ++i) {
    const int64_t n = ceil_div(n_feat, tiles[i].tf) * ceil_div(tokens, tiles[i].tn);
    const int64_t full = n / cus;
    const double fill = static_cast<double>(n - full * cus) / cus;
    const double t = (static_cast<double>(full) + (fill > 0.0 ? 0.5 + 0.5 * fill : 0.0)) * cost[i];
    if (i == 0 || t < best_t - 1e-9) {
      best = i;
      best_t = t;
    }
  }
  return tiles[best];
}

template <int TB>
static void launch_few_tokens(int dtype, int d, const QkvArgs& a, unsigned grid, hipStream_t stream) {
  if (dtype == kBF16) {
    if (d == 128) qkv_few_tokens_kernel<kBF16, 128, TB><<<grid, kQThreads, 0, stream>>>(a);
    else qkv_few_tokens_kernel<kBF16, 64, TB><<<grid, kQThreads, 0, stream>>>(a);
  } else {
    if (d == 128) qkv_few_tokens_kernel<kF16, 128, TB><<<grid, kQThreads, 0, stream>>>(a);
    else qkv_few_tokens_kernel<kF16, 64, TB><<<grid, kQThreads, 0, stream>>>(a);
  }
}

// Token blocks (of 16) per workgroup of the few-tokens kernel, 0 where the tiled kernel is
// the faster one.  Its workgroups each take in every token row beside their weights, and past
// one round of the CUs that is paid again; the tiled kernel's time hardly depends on the
// tokens.  In us, few / tiled:
//   one round (up to 256 workgroups), up to 128 tokens: 32/8 heads of 128, hidden 4096: 1
//     token 13 / 32, 32 19 / 33, 64 27 / 34, 96 36 / 35, 128 41 / 36; 16/2, hidden 2048: 64
//     15 / 19, 128 22 / 20; 40/8, hidden 5120: 64 34 / 51, 128 50 / 56; and more tokens while
//     their tiles fit it too: 14/2 of 64, hidden 896: 160 12.7 / 12.3;
//   two rounds, up to 24: 64/8, hidden 8192 (320 workgroups): 1 41 / 58, 24 56 / 59, 33 70 /
//     59, 64 91 / 60, 128 148 / 65; 32/32, hidden 4096 (384): 24 31 / 33, 33 39 / 34, 128 79 / 37;
//   three, up to 16: 128/8, hidden 16384 (576): 1 130 / 153, 16 172 / 169, 64 313 / 190.
// Its per-lane offsets are 32-bit: the weight rows of a head and 128 token rows must span
// less than 2 GiB.
static int few_token_blocks(int64_t n_feat, int64_t tokens, int d, int64_t hidden, int64_t x_ss, int cus) {
  constexpr int64_t kSpan = int64_t(1) << 31;
  if (d * hidden * 2 >= kSpan || x_ss >= kSpan / 256) return 0;
  const int64_t rounds = ceil_div(n_feat / 32 * ceil_div(tokens, 128), cus);
  if (rounds > 1 && tokens > 48 / rounds) return 0;
  return tokens <= 16 ? 1 : tokens <= 32 ? 2 : tokens <= 64 ? 4 : 8;
}

void launch_qkv_rope(int dtype, int d, QkvArgs& a, hipStream_t stream) {
  const int n_feat = a.nq + 2 * a.nkv;
  if (a.tokens == 0) return;
  if (const int tb = few_token_blocks(n_feat, a.tokens, d, a.hidden, a.x_ss, device_cus())) {
    a.n_tiles_n = n_feat / 32;
    a.n_tiles_m = static_cast<int32_t>(ceil_div(a.tokens, 16 * tb));
    const unsigned grid = static_cast<unsigned>(a.n_tiles_n * a.n_tiles_m);
    if (tb == 1) launch_few_tokens<1>(dtype, d, a, grid, stream);
    else if (tb == 2) launch_few_tokens<2>(dtype, d, a, grid, stream);
    else if (tb == 4) launch_few_tokens<4>(dtype, d, a, grid, stream);
    else launch_few_tokens<8>(dtype, d, a, grid, stream);
    HCP_HIP(hipGetLastError());
    return;
  }
  const QkvTile tile = qkv_tile(n_feat, a.tokens);
  a.n_tiles_n = static_cast<int32_t>(ceil_div(n_feat, tile.tf));
  a.n_tiles_m = static_cast<int32_t>(ceil_div(a.tokens, tile.tn));
  const unsigned grid = static_cast<unsigned>(a.n_tiles_n * a.n_tiles_m);
  auto go = [&](auto tfc, auto tnc) {
    constexpr int TF = decltype(tfc)::value, TN = decltype(tnc)::value;
    if (dtype == kBF16) {
      if (d == 128) qkv_rope_kernel<kBF16, 128, TF, TN><<<grid, kQThreads, 0, stream>>>(a);
      else qkv_rope_kernel<kBF16, 64, TF, TN><<<grid, kQThreads, 0, stream>>>(a);
    } else {
      if (d == 128) qkv_rope_kernel<kF16, 128, TF, TN><<<grid, kQThreads, 0, stream>>>(a);
      else qkv_rope_kernel<kF16, 64, TF, TN><<<grid, kQThreads, 0, stream>>>(a);
    }
  };
  if (tile.tf == 384) go(IntC<384>{}, IntC<256>{});
  else if (tile.tf == 128) go(IntC<128>{}, IntC<128>{});
  else if (tile.tn == 128) go(IntC<256>{}, IntC<128>{});
  else if (tile.tn == 384) go(IntC<256>{}, IntC<384>{});
  else go(IntC<256>{}, IntC<256>{});
  HCP_HIP(hipGetLastError());
}

}  // namespace hcp
