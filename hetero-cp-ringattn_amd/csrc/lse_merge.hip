// LSE merge of ring-step partials (closed form of the re-entry merge in
// positioned_merge_compact_partial / decode_merge_packet, ring.rs:574-603, :647-663):
//   m = max_i lse_i,  w_i = e^(lse_i - m),
//   o = sum_i w_i o_i / sum_i w_i,  lse = m + ln sum_i w_i,  all -inf -> (0, -inf);
// a NaN LSE makes the row NaN.
//
// Layout: each partial is o [H, L, D] fp32 and lse [H, L] fp32 (as the block kernel
// writes them).  One row (h, t) = D fp32 is handled by D/4 lanes with 16-byte loads,
// so a wavefront covers 64*4/D rows per instruction, and each thread takes two
// consecutive rows (measured +2-4% over one on the c3 partials; four: +2-3%).  The partials are folded in one
// pass, in groups of up to 8 whose loads are all in flight together, with the running
// max, sum and accumulator rescaled when a group raises the max (the same closed form,
// grouped).  HBM-bound: algorithmic bytes per row = n*(4D + 4) read + (D*out_bytes + 4)
// written.
#include "kernels.hpp"
#include "lds_dma.hpp"

namespace hcp {

constexpr int kMaxMergeParts = 64;

struct MergeArgs {
  const float* o[kMaxMergeParts];
  const float* lse[kMaxMergeParts];
  int32_t n;
  int32_t heads;
  int64_t q_len;
  int32_t d;
  int32_t lanes_per_row;  // D/4 rounded up to a power of two
  void* out;
  int64_t out_hs, out_ss;  // elements
  float* lse_out;
  int64_t lse_out_hs;      // elements between heads of lse_out
};

// 16-byte streaming load: each partial is read once.
__device__ __forceinline__ float4 nt_load4(const float* p) {
  typedef float f4 __attribute__((ext_vector_type(4)));
  const f4 x = __builtin_nontemporal_load(reinterpret_cast<const f4*>(p));
  return make_float4(x[0], x[1], x[2], x[3]);
}

// LSE of a row from its largest partial LSE and the sum of the weights against it: -inf
// for a row of empty partials (sum 0), NaN where a partial's is.
__device__ __forceinline__ float merged_lse(float m, float den) {
  return den > 0.f ? m + __logf(den) : den == 0.f ? -INFINITY : den;
}

// Four consecutive values of a merged row in the output type.
template <int OUT_DT>
__device__ __forceinline__ void store_row4(void* out, int64_t at, float4 x) {
  if constexpr (OUT_DT == kF32) {
    store16_nt_sc1(static_cast<float*>(out) + at, __builtin_bit_cast(u32x4, x));
  } else {
    u32x2 w;
    if constexpr (OUT_DT == kBF16) {
      w[0] = static_cast<uint32_t>(f32_to_bf16_bits(x.x)) | (static_cast<uint32_t>(f32_to_bf16_bits(x.y)) << 16);
      w[1] = static_cast<uint32_t>(f32_to_bf16_bits(x.z)) | (static_cast<uint32_t>(f32_to_bf16_bits(x.w)) << 16);
    } else {
      w[0] = static_cast<uint32_t>(f32_to_f16_bits(x.x)) | (static_cast<uint32_t>(f32_to_f16_bits(x.y)) << 16);
      w[1] = static_cast<uint32_t>(f32_to_f16_bits(x.z)) | (static_cast<uint32_t>(f32_to_f16_bits(x.w)) << 16);
    }
    store8_nt_sc1(static_cast<uint16_t*>(out) + at, w);
  }
}

// Few rows, several partials (a decode step): one row per workgroup, whose 256 / lpr slots
// take every so-manieth partial with all their loads in flight, and meet in LDS.  The
// kernel below walks a row's partials in groups of 8, one memory latency each, on a handful
// of workgroups: that chain, not the bytes, bounds it (19 partials of 64 rows: 9.4 us).
// Decode steps with it and without: 4 sequences of 2085 tokens 18.9 / 23.7 us (32/8 heads),
// 4 of 16384 28.0 / 34.1 us (16/2 heads).
template <int OUT_DT>
__global__ __launch_bounds__(256) void lse_merge_few_rows_kernel(MergeArgs a) {
  constexpr int NP = 4;  // partials of a slot in flight together
  __shared__ float4 acc_l[256];
  __shared__ float m_l[256], den_l[256];
  const int lpr = a.lanes_per_row;
  const int slots = 256 / lpr;
  const int64_t row = blockIdx.x;
  const int slot = threadIdx.x / lpr;
  const int c = threadIdx.x % lpr * 4;
  const bool active = c < a.d;
  float m = -INFINITY, den = 0.f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int base = slot; base < a.n; base += NP * slots) {
    float l[NP];
    float4 v[NP];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const int i = base + u * slots;
      l[u] = i < a.n ? a.lse[i][row] : -INFINITY;
      v[u] = i < a.n && active ? nt_load4(a.o[i] + row * a.d + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float mn = m;
#pragma unroll
    for (int u = 0; u < NP; ++u) mn = fmaxf(mn, l[u]);
    // While every partial of the slot is empty the weights are taken against 0: an empty
    // one adds nothing, a NaN stays (the row's other slots may hold finite partials).
    const float ref = mn == -INFINITY ? 0.f : mn;
    const float sc = __expf(m - ref);
    den *= sc;
    acc.x *= sc; acc.y *= sc; acc.z *= sc; acc.w *= sc;
#pragma unroll
    for (int u = 0; u < NP; ++u) {
      const float w = __expf(l[u] - ref);
      den += w;
      acc.x += w * v[u].x; acc.y += w * v[u].y; acc.z += w * v[u].z; acc.w += w * v[u].w;
    }
    m = mn;
  }
  acc_l[threadIdx.x] = acc;
  m_l[threadIdx.x] = m;
  den_l[threadIdx.x] = den;
  __syncthreads();
  if (slot != 0) return;
  const int used = min(slots, a.n);  // slots past the last partial hold nothing
  float mt = -INFINITY;
  for (int s = 0; s < used; ++s) mt = fmaxf(mt, m_l[threadIdx.x + s * lpr]);
  float dt = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  if (mt != -INFINITY) {
    for (int s = 0; s < used; ++s) {
      const float w = __expf(m_l[threadIdx.x + s * lpr] - mt);
      const float4 x = acc_l[threadIdx.x + s * lpr];
      dt += w * den_l[threadIdx.x + s * lpr];
      o.x += w * x.x; o.y += w * x.y; o.z += w * x.z; o.w += w * x.w;
    }
  } else {  // no finite LSE: 0, or NaN with a NaN one
    for (int s = 0; s < used; ++s) dt += den_l[threadIdx.x + s * lpr];
  }
  const float inv = dt > 0.f ? 1.f / dt : dt;
  const int64_t h = row / a.q_len, t = row - h * a.q_len;
  if (active)
    store_row4<OUT_DT>(a.out, h * a.out_hs + t * a.out_ss + c, make_float4(o.x * inv, o.y * inv, o.z * inv, o.w * inv));
  if (a.lse_out != nullptr && threadIdx.x == 0) a.lse_out[h * a.lse_out_hs + t] = merged_lse(mt, dt);
}

template <int OUT_DT, int NP, int R>
__global__ __launch_bounds__(256) void lse_merge_kernel(MergeArgs a) {
  const int lpr = a.lanes_per_row;
  // R consecutive rows per thread (same 16-byte column of each): R * NP loads in flight.
  const int64_t row0 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / lpr * R;
  const int lane_in_row = threadIdx.x % lpr;
  const int64_t rows = static_cast<int64_t>(a.heads) * a.q_len;
  if (row0 >= rows) return;
  const int n = a.n;
  const int c = lane_in_row * 4;
  const bool active = c < a.d;

  // One pass over the partials in groups of NP: every load of a group (NP lse values
  // and NP 16-byte slices of o, for each of the R rows) is issued before any is used,
  // and the running (max, sum, acc) is rescaled when a group raises the max.
  float m[R], den[R];
  float4 acc[R];
#pragma unroll
  for (int k = 0; k < R; ++k) {
    m[k] = -INFINITY;
    den[k] = 0.f;
    acc[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  for (int base = 0; base < n; base += NP) {
    float l[R][NP];
    float4 v[R][NP];
#pragma unroll
    for (int k = 0; k < R; ++k)
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const bool in = base + u < n && row0 + k < rows;
        l[k][u] = in ? a.lse[base + u][row0 + k] : -INFINITY;
        v[k][u] = (in && active) ? nt_load4(a.o[base + u] + (row0 + k) * a.d + c)
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
    for (int k = 0; k < R; ++k) {
      float mg = l[k][0];
#pragma unroll
      for (int u = 1; u < NP; ++u) mg = fmaxf(mg, l[k][u]);
      const float mn = fmaxf(m[k], mg);
      if (mn == -INFINITY) {  // every partial so far is empty, or its LSE a NaN, which the sum keeps
#pragma unroll
        for (int u = 0; u < NP; ++u) den[k] += __expf(l[k][u]);
        continue;
      }
      const float sc = __expf(m[k] - mn);  // 0 while m = -inf
      den[k] *= sc;
      acc[k].x *= sc;
      acc[k].y *= sc;
      acc[k].z *= sc;
      acc[k].w *= sc;
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const float w = __expf(l[k][u] - mn);  // exp(-inf) = 0 for empty partials
        den[k] += w;
        acc[k].x += w * v[k][u].x;
        acc[k].y += w * v[k][u].y;
        acc[k].z += w * v[k][u].z;
        acc[k].w += w * v[k][u].w;
      }
      m[k] = mn;
    }
  }
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int64_t row = row0 + k;
    if (row >= rows) break;
    const int64_t h = row / a.q_len;
    const int64_t t = row - h * a.q_len;
    const float inv = den[k] > 0.f ? 1.f / den[k] : den[k];  // 0: empty; NaN stays
    if (active) {
      const int64_t base = h * a.out_hs + t * a.out_ss + c;
      store_row4<OUT_DT>(a.out, base, make_float4(acc[k].x * inv, acc[k].y * inv, acc[k].z * inv, acc[k].w * inv));
    }
    if (a.lse_out != nullptr && lane_in_row == 0) {
      a.lse_out[h * a.lse_out_hs + t] = merged_lse(m[k], den[k]);
    }
  }
}

void launch_lse_merge(int n, const float* const* o_parts, const float* const* lse_parts,
                      int heads, int64_t q_len, int d, int out_dtype, void* out, int64_t out_hs,
                      int64_t out_ss, float* lse_out, int64_t lse_out_hs, hipStream_t stream) {
  require(n >= 1 && n <= kMaxMergeParts, "lse_merge: num_parts must be in [1, 64]");
  require(d % 4 == 0 && d <= 256, "lse_merge: head_dim must be a multiple of 4, <= 256");
  if (q_len == 0 || heads == 0) return;
  MergeArgs a;
  for (int i = 0; i < n; ++i) {
    a.o[i] = o_parts[i];
    a.lse[i] = lse_parts[i];
  }
  a.n = n;
  a.heads = heads;
  a.q_len = q_len;
  a.d = d;
  int lpr = 1;
  while (lpr < d / 4) lpr *= 2;
  a.lanes_per_row = lpr;
  a.out = out;
  a.out_hs = out_hs;
  a.out_ss = out_ss;
  a.lse_out = lse_out;
  a.lse_out_hs = lse_out_hs;
#ifndef HCP_MERGE_R
#define HCP_MERGE_R 2
#endif
  constexpr int R = HCP_MERGE_R;
  const int64_t threads = ceil_div(static_cast<int64_t>(heads) * q_len, R) * lpr;
  const dim3 grid(static_cast<unsigned>(ceil_div(threads, 256)));
  const int64_t rows = static_cast<int64_t>(heads) * q_len;
  // One row per workgroup: up to four partials the kernel below has all loads of a row in
  // flight too, and with many rows it fills the chip as well and reads wider.  In us, below /
  // here, 128 dims: 4 partials of 64 rows 3.70 / 3.47; 8 of 64 4.50 / 3.48, of 1024 4.81 /
  // 4.05, of 1536 4.93 / 4.82, of 2048 4.85 / 5.28; 19 of 64 7.85 / 3.83, of 2048 8.70 / 7.40.
  if (n > 4 && rows <= 1024) {
    const dim3 g(static_cast<unsigned>(rows));
    switch (out_dtype) {
      case kBF16: lse_merge_few_rows_kernel<kBF16><<<g, 256, 0, stream>>>(a); break;
      case kF16: lse_merge_few_rows_kernel<kF16><<<g, 256, 0, stream>>>(a); break;
      case kF32: lse_merge_few_rows_kernel<kF32><<<g, 256, 0, stream>>>(a); break;
      default: throw Error(-6, "lse_merge: out_dtype must be BF16, F16 or F32");
    }
    HCP_HIP(hipGetLastError());
    return;
  }
  // Group size: all partials in one group up to 4, else groups of 8.
  auto go = [&](auto np) {
    constexpr int NP = decltype(np)::value;
    switch (out_dtype) {
      case kBF16: lse_merge_kernel<kBF16, NP, R><<<grid, 256, 0, stream>>>(a); break;
      case kF16: lse_merge_kernel<kF16, NP, R><<<grid, 256, 0, stream>>>(a); break;
      case kF32: lse_merge_kernel<kF32, NP, R><<<grid, 256, 0, stream>>>(a); break;
      default: throw Error(-6, "lse_merge: out_dtype must be BF16, F16 or F32");
    }
  };
  if (n == 1) go(IntC<1>{});
  else if (n == 2) go(IntC<2>{});
  else if (n <= 4) go(IntC<4>{});
  else go(IntC<8>{});
  HCP_HIP(hipGetLastError());
}

}  // namespace hcp
