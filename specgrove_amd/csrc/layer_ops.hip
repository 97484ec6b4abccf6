// Fused elementwise kernels of the target decoder layer stack (Qwen3 family)
// around the library projections, for the packed verification wave.
//
// The reference runs the Target's transformers decoder
// (engine.py:499-517 target_hidden_forward -> transformers' Qwen3 layers):
// per layer RMSNorm, q/k/v projections, per-head RMSNorm of q and k (QK-norm),
// rotary position embedding, attention, o projection, residual add, RMSNorm,
// gate/up projections, SiLU(gate) * up, down projection, residual add.  Here
// the projections are library GEMMs (hipBLASLt through torch.matmul) and every
// elementwise stage between them is one HBM pass:
//
//   sg_add_rmsnorm     residual add + RMSNorm (one read of each input, one
//                      write of each output);
//   sg_qk_norm_rope    QK-norm + RoPE of the merged q/k/v projection, writing
//                      q [R, Hq, D] for the attention and k/v [Hkv, R, D] as
//                      the wave's new cache rows;
//   sg_silu_mul        SiLU(gate) * up of the merged gate/up projection;
//   sg_gather_rows     the kept rows of several layers' hidden states side by
//                      side (the draft features, continuous_tree_block_decode.py
//                      :2144-2158).
//
// Arithmetic follows the transformers modules' rounding points: RMSNorm
// normalises in fp32, rounds to bf16, then multiplies by the bf16 weight and
// rounds again; RoPE uses bf16-rounded cos/sin of fp32 angles and rounds
// q*cos, rotate_half(q)*sin and their sum to bf16 in turn; SiLU rounds
// before the product with up.  Sums of squares run in fp32 in this kernel's
// own order, and 1/sqrt and sincos are the device's, so a normed or rotated
// value can still differ from transformers' by one bf16 ulp.
//
// All of them are bound by HBM (or the last-level cache, where the inputs are
// still there) once each load of a thread is issued before the first is used and
// the conversions to bf16 are gfx950's own.  One layer's four calls (hidden 4096,
// intermediate 12288, 32 q / 8 kv heads of 128) over 2,048 rows (336 MB), on new
// inputs in each call: 80.3 -> 75.4 us (the fused stages by themselves, repeated
// over one set of tensors: 79 -> 73.6 us; 1,024 rows 39.5 -> 38.6, 4,096 rows
// 140 -> 131).  Non-temporal stores: 3.5 us less over 2,048 rows, 25 us more in a
// 512-row decoder of four layers, where the next kernel reads the stored rows
// from the caches: not used.
#include <algorithm>
#include <cmath>

#include "sg_common.h"

namespace sg {
namespace {

constexpr int kNormThreads = 256;

__device__ __forceinline__ float block_sum(float v, float* scratch) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = 0.0f;
  const int waves = blockDim.x >> 6;
  for (int w = 0; w < waves; ++w) t += scratch[w];
  return t;
}

// The two bf16 halves of a word as floats, and both rounded to bf16 and back.
struct Pair {
  float lo, hi;
};
__device__ __forceinline__ Pair unpack(uint32_t v) {
  return {__uint_as_float(v << 16), __uint_as_float(v & 0xffff0000u)};
}
__device__ __forceinline__ Pair bf16r(float lo, float hi) { return unpack(pack_bf16x2(lo, hi)); }

// One row per workgroup; 8 bf16 (16 bytes) per thread and chunk, kChunks the
// fewest chunks that hold the row, so that every load of the row (the weight's
// too) is issued before the first is used.
// sum = x (+ residual); residual_out = bf16(sum) when requested;
// out = bf16(w * bf16(s * rsqrt(mean(s^2) + eps))), s = bf16(sum).
template <int kChunks, bool kResidual>
__global__ __launch_bounds__(kNormThreads) void add_rmsnorm_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ residual,
    const uint16_t* __restrict__ weight, uint16_t* __restrict__ out,
    uint16_t* __restrict__ residual_out, int hidden, int64_t x_stride, int64_t res_stride,
    int64_t out_stride, int64_t res_out_stride, float eps) {
  __shared__ float scratch[kNormThreads / 64];
  const int64_t row = blockIdx.x;
  const uint16_t* xr = x + row * x_stride;
  const uint16_t* rr = residual + row * res_stride;
  uint4 s[kChunks], b[kChunks], w[kChunks];
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int e = 8 * (threadIdx.x + c * kNormThreads);
    const bool live = e < hidden;
    s[c] = live ? *reinterpret_cast<const uint4*>(xr + e) : make_uint4(0u, 0u, 0u, 0u);
    if (kResidual)
      b[c] = live ? *reinterpret_cast<const uint4*>(rr + e) : make_uint4(0u, 0u, 0u, 0u);
  }
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int e = 8 * (threadIdx.x + c * kNormThreads);
    w[c] = e < hidden ? *reinterpret_cast<const uint4*>(weight + e) : make_uint4(0u, 0u, 0u, 0u);
  }
  float ss = 0.0f;
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    uint32_t v[4] = {s[c].x, s[c].y, s[c].z, s[c].w};
    if (kResidual) {
      const uint32_t bv[4] = {b[c].x, b[c].y, b[c].z, b[c].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const Pair p = unpack(v[k]), q = unpack(bv[k]);
        v[k] = pack_bf16x2(p.lo + q.lo, p.hi + q.hi);
      }
      s[c] = make_uint4(v[0], v[1], v[2], v[3]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const Pair p = unpack(v[k]);
      ss += p.lo * p.lo + p.hi * p.hi;
    }
  }
  if (residual_out != nullptr) {
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
      const int e = 8 * (threadIdx.x + c * kNormThreads);
      if (e < hidden)
        *reinterpret_cast<uint4*>(residual_out + row * res_out_stride + e) = s[c];
    }
  }
  const float total = block_sum(ss, scratch);
  const float r = 1.0f / sqrtf(total / static_cast<float>(hidden) + eps);
#pragma unroll
  for (int c = 0; c < kChunks; ++c) {
    const int e = 8 * (threadIdx.x + c * kNormThreads);
    if (e >= hidden) continue;
    const uint32_t v[4] = {s[c].x, s[c].y, s[c].z, s[c].w};
    const uint32_t wv[4] = {w[c].x, w[c].y, w[c].z, w[c].w};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const Pair p = unpack(v[k]), q = unpack(wv[k]);
      const Pair n = bf16r(p.lo * r, p.hi * r);
      o[k] = pack_bf16x2(q.lo * n.lo, q.hi * n.hi);
    }
    *reinterpret_cast<uint4*>(out + row * out_stride + e) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// One row per workgroup.  A head's D dims are D/8 lanes of 16 bytes (lane j
// holds dims 8j .. 8j+7), so a wave takes 64/(D/8) heads at a time with
// 16-byte loads and stores; the rotary partner of dim i < D/2 (dim i + D/2)
// sits in lane j ^ (D/16) of the same head.  Heads 0..Hq-1 are q (normed,
// rotated, written to q_out[row, h]), Hq..Hq+Hkv-1 are k (normed, rotated,
// written to k_out[h, row]), the rest v (copied to v_out[h, row]).  The
// row's bf16 cos / sin of the fp32 angles position * inv_freq[p] are made once
// per workgroup (one pair per thread) and read from LDS.
template <int D>
__global__ __launch_bounds__(kNormThreads) void qk_norm_rope_kernel(
    const uint16_t* __restrict__ qkv, int64_t qkv_stride, int hq, int hkv,
    const uint16_t* __restrict__ q_norm, const uint16_t* __restrict__ k_norm,
    const float* __restrict__ inv_freq, const int64_t* __restrict__ positions,
    uint16_t* __restrict__ q_out, int64_t q_row_stride, uint16_t* __restrict__ k_out,
    uint16_t* __restrict__ v_out, int64_t kv_head_stride, float eps) {
  constexpr int H2 = D / 2;
  constexpr int LPH = D / 8;        // lanes per head
  constexpr int HPW = kWave / LPH;  // heads per wave at a time
  constexpr int kBatch = 3;         // head groups of a wave loaded at a time
  __shared__ float s_cs[H2];
  __shared__ float s_sn[H2];
  const int64_t row = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int waves = blockDim.x >> 6;
  const int j = lane % LPH;             // 16-byte chunk of the head
  const int slot = lane / LPH;          // head of the wave's group
  const bool lower = j < LPH / 2;       // dims below D/2
  const int pair0 = 8 * (j % (LPH / 2));
  const int heads = hq + 2 * hkv;
  const uint16_t* src = qkv + row * qkv_stride + 8 * j;
  uint4 raw[kBatch];
  auto load = [&](int h0) {
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int h = h0 + b * waves * HPW + slot;
      raw[b] = h < heads ? *reinterpret_cast<const uint4*>(src + static_cast<int64_t>(h) * D)
                         : make_uint4(0u, 0u, 0u, 0u);
    }
  };
  // The row and the norm weights are on their way while the angles are made.
  load(wave * HPW);
  const uint4 wq = *reinterpret_cast<const uint4*>(q_norm + 8 * j);
  const uint4 wk = *reinterpret_cast<const uint4*>(k_norm + 8 * j);
  const float pos = static_cast<float>(positions[row]);
  for (int p = threadIdx.x; p < H2; p += blockDim.x) {
    float sv, cv;
    sincosf(pos * inv_freq[p], &sv, &cv);
    s_cs[p] = bf16_to_f32(f32_to_bf16(cv));
    s_sn[p] = bf16_to_f32(f32_to_bf16(sv));
  }
  __syncthreads();
  // The sign of rotate_half goes into the sine (bf16r(-v) = -bf16r(v)).
  float cs[8], sn[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    cs[k] = s_cs[pair0 + k];
    sn[k] = lower ? -s_sn[pair0 + k] : s_sn[pair0 + k];
  }
  for (int h0 = wave * HPW; h0 < heads;) {
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int h = h0 + b * waves * HPW + slot;
      const bool live = h < heads;
      const bool is_v = h >= hq + hkv;
      const uint32_t rv[4] = {raw[b].x, raw[b].y, raw[b].z, raw[b].w};
      Pair x[4];
      // RMS over the head's D dims: the lane's 8 squares, then the head's lanes.
      float ss = 0.0f;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        x[k] = unpack(rv[k]);
        ss += x[k].lo * x[k].lo;
        ss += x[k].hi * x[k].hi;
      }
#pragma unroll
      for (int d = LPH / 2; d >= 1; d >>= 1) ss += __shfl_xor(ss, d);
      const float r = 1.0f / sqrtf(ss / static_cast<float>(D) + eps);
      const uint4 wraw = h < hq ? wq : wk;
      const uint32_t wv[4] = {wraw.x, wraw.y, wraw.z, wraw.w};
      uint32_t nx[4], ny[4], o[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const Pair w = unpack(wv[k]);
        const Pair n = bf16r(x[k].lo * r, x[k].hi * r);
        nx[k] = pack_bf16x2(w.lo * n.lo, w.hi * n.hi);
      }
      // The rotary partner's normed values (exact: bf16 pairs).
#pragma unroll
      for (int k = 0; k < 4; ++k) ny[k] = __shfl_xor(nx[k], LPH / 2);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        // x*cos + rotate_half(x)*sin, rotate_half(x) = (-x2, x1), with the
        // rounding points of transformers' bf16 tensors: each product is
        // rounded to bf16, then their sum.
        const Pair a = unpack(nx[k]), p = unpack(ny[k]);
        const Pair ac = bf16r(a.lo * cs[2 * k], a.hi * cs[2 * k + 1]);
        const Pair bs = bf16r(p.lo * sn[2 * k], p.hi * sn[2 * k + 1]);
        o[k] = pack_bf16x2(ac.lo + bs.lo, ac.hi + bs.hi);
      }
      if (!live) continue;
      if (is_v) {
        *reinterpret_cast<uint4*>(v_out + static_cast<int64_t>(h - hq - hkv) * kv_head_stride +
                                  row * D + 8 * j) = raw[b];
      } else {
        uint16_t* dst = h < hq ? q_out + row * q_row_stride + static_cast<int64_t>(h) * D
                               : k_out + static_cast<int64_t>(h - hq) * kv_head_stride + row * D;
        *reinterpret_cast<uint4*>(dst + 8 * j) = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
    h0 += kBatch * waves * HPW;
    if (h0 < heads) load(h0);
  }
}

// out[r, i] = bf16(bf16(silu(gate[r, i])) * up[r, i]); gate = gu[r, :I],
// up = gu[r, I:2I].  A workgroup takes 256 chunks of 8 elements of one row (parts =
// workgroups per row), so that finding the row is one scalar division; two
// chunks a thread measured 4 % slower.  Plain loads: the non-temporal hint cost
// 15 % on what the caches hold (2,048 x 12,288: 25.8 -> 29.7 us alone) and gave
// nothing between the projections (up + SiLU + down 491 / 489 us at 2,048 rows,
// 876 / 876 at 4,096) or in a layer's four calls on new inputs (75.4 / 77.4 us).
constexpr int kSiluPart = 8 * 256;  // elements of a workgroup's part of a row
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gu,
                                                       int64_t gu_stride, int inter,
                                                       uint16_t* __restrict__ out,
                                                       int64_t out_stride, uint32_t parts,
                                                       int64_t items) {
  for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
    const int64_t row = item / parts;
    const uint32_t part = static_cast<uint32_t>(item - row * parts);
    const uint32_t e = part * kSiluPart + 8 * threadIdx.x;
    if (e >= static_cast<uint32_t>(inter)) continue;
    const uint16_t* gr = gu + row * gu_stride + e;
    const uint4 g = *reinterpret_cast<const uint4*>(gr);
    const uint4 u = *reinterpret_cast<const uint4*>(gr + inter);
    const uint32_t gv[4] = {g.x, g.y, g.z, g.w};
    const uint32_t uv[4] = {u.x, u.y, u.z, u.w};
    uint32_t o[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const Pair x = unpack(gv[q]), up = unpack(uv[q]);
      const Pair s = bf16r(x.lo / (1.0f + expf(-x.lo)), x.hi / (1.0f + expf(-x.hi)));
      o[q] = pack_bf16x2(s.lo * up.lo, s.hi * up.hi);
    }
    *reinterpret_cast<uint4*>(out + row * out_stride + e) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

// out[k, l*width .. (l+1)*width) = src_l[index[k], :width]; one workgroup per
// output row, 16-byte chunks.
__global__ __launch_bounds__(256) void gather_rows_kernel(const uint16_t* const* __restrict__ srcs,
                                                          int num_src, int64_t src_stride,
                                                          int width, int num_src_rows,
                                                          const int32_t* __restrict__ index,
                                                          uint16_t* __restrict__ out,
                                                          int64_t out_stride,
                                                          int32_t* __restrict__ status) {
  const int k = blockIdx.x;
  const int r = index[k];
  const bool ok = r >= 0 && r < num_src_rows;
  if (!ok && threadIdx.x == 0 && status != nullptr) atomicExch(status, SG_EINVAL);
  const int chunks = width / 8;
  for (int c = threadIdx.x; c < num_src * chunks; c += blockDim.x) {
    const int l = c / chunks;
    const int e = 8 * (c - l * chunks);
    const uint4 v = ok ? *reinterpret_cast<const uint4*>(srcs[l] + static_cast<int64_t>(r) *
                                                                       src_stride + e)
                       : make_uint4(0u, 0u, 0u, 0u);
    *reinterpret_cast<uint4*>(out + static_cast<int64_t>(k) * out_stride +
                              static_cast<int64_t>(l) * width + e) = v;
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace sg

extern "C" int sg_add_rmsnorm(const SgAddRmsNormArgs* args, sg_stream_t stream) {
  using namespace sg;
  clear_error();
  SG_REQUIRE(args != nullptr, "null args");
  const SgAddRmsNormArgs& a = *args;
  SG_REQUIRE(a.num_rows >= 0, "num_rows must be non-negative");
  SG_REQUIRE(a.hidden >= 8 && a.hidden % 8 == 0 && a.hidden <= 8 * 4 * kNormThreads,
             "hidden must be a multiple of 8 in [8, 8192]");
  if (a.num_rows == 0) return SG_OK;
  SG_REQUIRE(a.x_dev && a.weight_dev && a.out_dev, "null device pointer");
  SG_REQUIRE((a.x_stride | a.out_stride | (a.residual_dev ? a.residual_stride : 0) |
              (a.residual_out_dev ? a.residual_out_stride : 0)) % 8 == 0,
             "row strides must be multiples of 8 elements");
  SG_REQUIRE(aligned16(a.x_dev) && aligned16(a.weight_dev) && aligned16(a.out_dev) &&
                 (!a.residual_dev || aligned16(a.residual_dev)) &&
                 (!a.residual_out_dev || aligned16(a.residual_out_dev)),
             "tensors must be 16-byte aligned");
  auto go = [&](auto kernel) {
    kernel<<<dim3(a.num_rows), dim3(kNormThreads), 0, static_cast<hipStream_t>(stream)>>>(
        static_cast<const uint16_t*>(a.x_dev), static_cast<const uint16_t*>(a.residual_dev),
        static_cast<const uint16_t*>(a.weight_dev), static_cast<uint16_t*>(a.out_dev),
        static_cast<uint16_t*>(a.residual_out_dev), a.hidden, a.x_stride, a.residual_stride,
        a.out_stride, a.residual_out_stride, a.eps);
  };
  const bool res = a.residual_dev != nullptr;
  switch ((a.hidden + 8 * kNormThreads - 1) / (8 * kNormThreads)) {
    case 1: res ? go(add_rmsnorm_kernel<1, true>) : go(add_rmsnorm_kernel<1, false>); break;
    case 2: res ? go(add_rmsnorm_kernel<2, true>) : go(add_rmsnorm_kernel<2, false>); break;
    case 3: res ? go(add_rmsnorm_kernel<3, true>) : go(add_rmsnorm_kernel<3, false>); break;
    default: res ? go(add_rmsnorm_kernel<4, true>) : go(add_rmsnorm_kernel<4, false>); break;
  }
  SG_LAUNCH_CHECK();
  return SG_OK;
}

extern "C" int sg_qk_norm_rope(const SgQkNormRopeArgs* args, sg_stream_t stream) {
  using namespace sg;
  clear_error();
  SG_REQUIRE(args != nullptr, "null args");
  const SgQkNormRopeArgs& a = *args;
  SG_REQUIRE(a.num_rows >= 0, "num_rows must be non-negative");
  SG_REQUIRE(a.head_dim == 64 || a.head_dim == 128, "head_dim must be 64 or 128");
  SG_REQUIRE(a.num_q_heads >= 1 && a.num_kv_heads >= 1, "head counts must be positive");
  if (a.num_rows == 0) return SG_OK;
  SG_REQUIRE(a.qkv_dev && a.q_norm_dev && a.k_norm_dev && a.inv_freq_dev && a.positions_dev &&
                 a.q_out_dev && a.k_out_dev && a.v_out_dev,
             "null device pointer");
  SG_REQUIRE(a.qkv_row_stride >= static_cast<int64_t>(a.num_q_heads + 2 * a.num_kv_heads) *
                                     a.head_dim,
             "qkv row stride below the q/k/v width");
  SG_REQUIRE(a.q_row_stride >= static_cast<int64_t>(a.num_q_heads) * a.head_dim,
             "q row stride below Hq*D");
  SG_REQUIRE(a.kv_head_stride >= static_cast<int64_t>(a.num_rows) * a.head_dim,
             "k/v head stride below R*D");
  SG_REQUIRE((a.qkv_row_stride | a.q_row_stride | a.kv_head_stride) % 8 == 0,
             "row and head strides must be multiples of 8 elements");
  SG_REQUIRE(aligned16(a.qkv_dev) && aligned16(a.q_norm_dev) && aligned16(a.k_norm_dev) &&
                 aligned16(a.q_out_dev) && aligned16(a.k_out_dev) && aligned16(a.v_out_dev),
             "q/k/v, norm weights and outputs must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto go = [&](auto kernel) {
    kernel<<<dim3(a.num_rows), dim3(kNormThreads), 0, s>>>(
        static_cast<const uint16_t*>(a.qkv_dev), a.qkv_row_stride, a.num_q_heads,
        a.num_kv_heads, static_cast<const uint16_t*>(a.q_norm_dev),
        static_cast<const uint16_t*>(a.k_norm_dev), a.inv_freq_dev, a.positions_dev,
        static_cast<uint16_t*>(a.q_out_dev), a.q_row_stride, static_cast<uint16_t*>(a.k_out_dev),
        static_cast<uint16_t*>(a.v_out_dev), a.kv_head_stride, a.eps);
  };
  if (a.head_dim == 128) {
    go(qk_norm_rope_kernel<128>);
  } else {
    go(qk_norm_rope_kernel<64>);
  }
  SG_LAUNCH_CHECK();
  return SG_OK;
}

extern "C" int sg_silu_mul(const void* gate_up_dev, int64_t gate_up_row_stride,
                           int32_t num_rows, int32_t intermediate, void* out_dev,
                           int64_t out_row_stride, sg_stream_t stream) {
  using namespace sg;
  clear_error();
  SG_REQUIRE(num_rows >= 0 && intermediate >= 8 && intermediate % 8 == 0,
             "intermediate must be a positive multiple of 8");
  if (num_rows == 0) return SG_OK;
  SG_REQUIRE(gate_up_dev && out_dev, "null device pointer");
  SG_REQUIRE(gate_up_row_stride >= 2 * static_cast<int64_t>(intermediate) &&
                 out_row_stride >= intermediate && (gate_up_row_stride | out_row_stride) % 8 == 0,
             "row strides must cover the rows and be multiples of 8");
  SG_REQUIRE(aligned16(gate_up_dev) && aligned16(out_dev), "tensors must be 16-byte aligned");
  const uint32_t parts = (static_cast<uint32_t>(intermediate) + kSiluPart - 1) / kSiluPart;
  const int64_t items = static_cast<int64_t>(num_rows) * parts;
  silu_mul_kernel<<<dim3(static_cast<unsigned>(std::min<int64_t>(items, 1 << 20))), dim3(256), 0,
                    static_cast<hipStream_t>(stream)>>>(
      static_cast<const uint16_t*>(gate_up_dev), gate_up_row_stride, intermediate,
      static_cast<uint16_t*>(out_dev), out_row_stride, parts, items);
  SG_LAUNCH_CHECK();
  return SG_OK;
}

extern "C" int sg_gather_rows(const void* const* src_dev, int32_t num_src, int64_t src_row_stride,
                              int32_t width, int32_t num_src_rows, const int32_t* index_dev,
                              int32_t num_index, void* out_dev, int64_t out_row_stride,
                              int32_t* status_dev, sg_stream_t stream) {
  using namespace sg;
  clear_error();
  SG_REQUIRE(num_src >= 1 && width >= 8 && width % 8 == 0 && num_index >= 0 &&
                 num_src_rows >= 1,
             "need at least one source of a positive multiple of 8 columns");
  if (num_index == 0) return SG_OK;
  SG_REQUIRE(src_dev && index_dev && out_dev, "null device pointer");
  SG_REQUIRE(src_row_stride >= width && out_row_stride >= static_cast<int64_t>(num_src) * width &&
                 (src_row_stride | out_row_stride) % 8 == 0,
             "row strides must cover the rows and be multiples of 8");
  SG_REQUIRE(aligned16(out_dev), "out must be 16-byte aligned");
  gather_rows_kernel<<<dim3(num_index), dim3(256), 0, static_cast<hipStream_t>(stream)>>>(
      reinterpret_cast<const uint16_t* const*>(src_dev), num_src, src_row_stride, width,
      num_src_rows, index_dev, static_cast<uint16_t*>(out_dev), out_row_stride, status_dev);
  SG_LAUNCH_CHECK();
  return SG_OK;
}
