// Fused q/k offset-RMSNorm + partial RoPE + KV append for gfx950.
//
// Behaviour follows the reference kernel src/kernels/qk_norm_rope.cu:12-90 and, to the last bit,
// its CPU twin src/ref/ops.cpp:79-142:
//   y = x * r * w with r = 1 / sqrt(float(sum_sq / 256) + eps), sum_sq accumulated in double;
//   RoPE on dims [0, 64): (y_i, y_{i+32}) <- (y_i c - y_{i+32} s, y_{i+32} c + y_i s);
//   q -> fp16 (RNE); k (normed + rotated) and v (as projected) -> page row: int8 with one fp16
//   scale = fp16(amax / 127) per 64-dim group and codes clamp(rint(y / scale), -127, 127), or bf16.
//
// Work mapping (MI355X-first): one wave64 per (token, head row); rows are the nq q heads, then the
// nkv k heads, then the nkv v heads of a token. Lane l owns dims [4l, 4l + 4), so a 64-dim
// quantisation group is exactly 16 lanes (one DPP row) and RoPE partners (i, i + 32) sit 8 lanes
// apart. Contraction is off for the whole file and division / square root are correctly rounded, so
// every operation rounds exactly as the reference's IEEE single-precision code does. cos/sin come
// from a host-built table (same libm calls as the CPU reference), read per position.
//
// Mean of squares: the reference sums x_i^2 in double, left to right, and rounds the mean to float.
// x is bf16, so every x_i^2 is exact in double and two orders of summing them differ by less than
// 2^-43 relative; the kernels sum as a tree and replay the left-to-right sum only where that could
// change the rounded mean (mean_is_settled, about one row in 2^18).
//
// Larger launches (qk_norm_rope_append_rows_kernel): 16 lanes per row, four rows per wave, 16 dims per
// lane. A row's reductions are then four steps within a DPP row, shared by four rows, its division and
// square root too, and every access is 16 bytes per lane.
#include "append.hpp"

// No multiply-add fusion here either (append.hpp restores the default at its end).
#pragma clang fp contract(off)

namespace q38a {
namespace {

__global__ void __launch_bounds__(kWavesPerBlock * 64)
qk_norm_rope_append_kernel(AppendArgs p, BatchArgs batch, KvArgs kv, int jobs) {
  __shared__ double stage[kWavesPerBlock][kHeadDim];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int job = blockIdx.x * kWavesPerBlock + wave;
  if (job >= jobs) return;
  const int rows = p.nq + 2 * p.nkv;
  RowLoads L;
  L.m = job / rows;
  L.r = job % rows;
  // q head r at column r*256; k head h at (2nq + h)*256; v head h at (2nq + nkv + h)*256
  const int col = (L.r < p.nq ? L.r : p.nq + L.r) * kHeadDim;
  L.pos = batch.tok_pos[L.m];
  // (any alignment: the in-projection call takes every row stride and 2-byte aligned rows)
  __builtin_memcpy(&L.raw, p.proj + size_t(L.m) * p.ld_proj + col + 4 * lane, sizeof(L.raw));
  row_meta(p, batch, kv, lane, L);
  append_row(p, kv, stage[wave], lane, L);
}

// ---- four rows per wave ----------------------------------------------------------------------------

// Sum in double over each 16-lane DPP row, in a fixed order, the result in every lane of the row.
__device__ inline double row16_sum(double v) {
  auto lo = [](double x) { return uint32_t(__builtin_bit_cast(uint64_t, x)); };
  auto hi = [](double x) { return uint32_t(__builtin_bit_cast(uint64_t, x) >> 32); };
  auto add = [](double x, uint32_t l, uint32_t h) { return x + __builtin_bit_cast(double, (uint64_t(h) << 32) | l); };
  v = add(v, dpp_move<kDppXor1>(lo(v)), dpp_move<kDppXor1>(hi(v)));
  v = add(v, dpp_move<kDppXor2>(lo(v)), dpp_move<kDppXor2>(hi(v)));
  v = add(v, dpp_move<kDppHalfMirror>(lo(v)), dpp_move<kDppHalfMirror>(hi(v)));
  return add(v, dpp_move<kDppMirror>(lo(v)), dpp_move<kDppMirror>(hi(v)));
}

__device__ inline uint32_t pack16(uint16_t a, uint16_t b) { return uint32_t(a) | (uint32_t(b) << 16); }

// Two values as fp16 bits (f16_bits).
__device__ inline uint32_t f16_pair_bits(float a, float b) { return pack16(f16_bits(a), f16_bits(b)); }

// Wave w handles rows 4 w .. 4 w + 3 of one kind: the waves cover the tokens' q rows (token-major),
// then the k rows, then the v rows, so a wave's rows take the same path. Lane l: row l / 16, dims
// 16 (l % 16) .. + 15.
__global__ void __launch_bounds__(kWavesPerBlock * 64)
qk_norm_rope_append_rows_kernel(AppendArgs p, BatchArgs batch, KvArgs kv) {
  const int lane = threadIdx.x & 63, l16 = lane & 15;
  const int M = batch.num_tokens;
  const int qw = (M * p.nq + 3) / 4, kw = (M * p.nkv + 3) / 4;
  int w = __builtin_amdgcn_readfirstlane(blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6));
  if (w >= qw + 2 * kw) return;
  const bool is_q = w < qw, is_k = !is_q && w < qw + kw;
  w -= is_q ? 0 : is_k ? qw : qw + kw;
  const int heads = is_q ? p.nq : p.nkv;
  const int head0 = is_q ? 0 : is_k ? 2 * p.nq : 2 * p.nq + p.nkv;
  const bool valid = 4 * w + (lane >> 4) < M * heads;  // (lanes past the last row repeat it, unstored)
  const int row = valid ? 4 * w + (lane >> 4) : M * heads - 1;
  const int m = row / heads, head = row % heads;
  // the loads: proj and position, then the RoPE row and (k, v) the page
  const uint4* src = reinterpret_cast<const uint4*>(p.proj + size_t(m) * p.ld_proj + (head0 + head) * kHeadDim + 16 * l16);
  const int pos = batch.tok_pos[m];
  const uint4 raw0 = src[0], raw1 = src[1];
  const int slot = is_q ? 0 : batch.seq_slot[batch.tok_seq[m]];
  const bool pos_ok = pos >= 0 && pos < p.rope_rows;
  float x[16];
  {
    const uint32_t r[8] = {raw0.x, raw0.y, raw0.z, raw0.w, raw1.x, raw1.y, raw1.z, raw1.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[2 * i] = as_f32(r[i] << 16);
      x[2 * i + 1] = as_f32(r[i] & 0xffff0000u);
    }
  }
  const int page_idx = pos / kPageTokens;
  const bool store_ok = valid && !is_q && pos_ok && page_idx < kv.max_pages_per_seq;
  const int page = store_ok ? kv.block_table[size_t(slot) * kv.max_pages_per_seq + page_idx] : 0;

  if (is_q || is_k) {
    // lanes 0-1 of a row hold dims 0-31, lanes 2-3 dims 32-63
    const bool rot = l16 < 4 && pos_ok;
    float4 c[4], s[4];
    if (rot) {
      const float4* cs = reinterpret_cast<const float4*>(p.rope + size_t(pos) * kRotaryDim + 16 * (l16 & 1));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        c[i] = cs[i];
        s[i] = cs[8 + i];
      }
    }
    const float4* wp = reinterpret_cast<const float4*>((is_q ? p.q_norm : p.k_norm) + 16 * l16);
    const float4 wv[4] = {wp[0], wp[1], wp[2], wp[3]};
    double part = 0.0;
#pragma unroll
    for (int e = 0; e < 16; ++e) part += double(x[e]) * double(x[e]);
    double ss = row16_sum(part);
    if (__ballot(!mean_is_settled(ss))) {
      // the left-to-right sum: lane after lane of the row takes the running sum over its 16 dims
      double seq = 0.0;
      for (int l = 0; l < 16; ++l) {
        double t = seq;
#pragma unroll
        for (int e = 0; e < 16; ++e) t = __builtin_fma(double(x[e]), double(x[e]), t);  // (exact squares)
        seq = __shfl(t, (lane & 48) + l, 64);
      }
      ss = seq;
    }
    const float mean = float(ss / double(kHeadDim));
    const float rs = div_rn(1.0f, sqrt_rn(mean + p.eps));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float wl[4] = {wv[i].x, wv[i].y, wv[i].z, wv[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) x[4 * i + e] = (x[4 * i + e] * rs) * wl[e];
    }
    float partner[16];  // lane l16 ^ 2: the other half of each rotated pair
#pragma unroll
    for (int e = 0; e < 16; ++e) partner[e] = as_f32(dpp_move<kDppXor2>(as_u32(x[e])));
    if (rot) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float cl[4] = {c[i].x, c[i].y, c[i].z, c[i].w}, sl[4] = {s[i].x, s[i].y, s[i].z, s[i].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float a = x[4 * i + e] * cl[e], b = partner[4 * i + e] * sl[e];
          x[4 * i + e] = l16 < 2 ? a - b : a + b;
        }
      }
    }
  }

  if (is_q) {
    if (!valid) return;
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = pos_ok ? f16_pair_bits(x[2 * i], x[2 * i + 1]) : 0x7e007e00u;  // NaN flags a bad position
    uint4* dst = reinterpret_cast<uint4*>(p.q_out + (size_t(m) * p.nq + head) * kHeadDim + 16 * l16);
    dst[0] = uint4{h[0], h[1], h[2], h[3]};
    dst[1] = uint4{h[4], h[5], h[6], h[7]};
    return;
  }
  const int tok = pos % kPageTokens;
  uint8_t* base = kv.pool + size_t(p.attn_layer) * kv.layer_stride + size_t(page) * kv.page_bytes;
  if (kv.layout.dtype == Q38A_KV_BF16) {
    if (!store_ok) return;
    uint32_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = pack16(bf16_bits(x[2 * i]), bf16_bits(x[2 * i + 1]));
    uint4* dst = reinterpret_cast<uint4*>(base + (is_k ? kv.layout.k_row(head, tok) : kv.layout.v_row(head, tok)) + 32 * l16);
    dst[0] = uint4{h[0], h[1], h[2], h[3]};
    dst[1] = uint4{h[4], h[5], h[6], h[7]};
    return;
  }
  // int8: a 64-dim group is four lanes
  float amax = fabsf(x[0]);  // (as quantize_row_int8: a group of NaNs alone keeps NaN as its scale)
#pragma unroll
  for (int e = 1; e < 16; ++e) amax = fmaxf(amax, fabsf(x[e]));
  amax = fmaxf(amax, as_f32(dpp_move<kDppXor1>(as_u32(amax))));
  amax = fmaxf(amax, as_f32(dpp_move<kDppXor2>(as_u32(amax))));
  if (!store_ok) return;
  const uint16_t sbits = f16_bits(div_rn(amax, 127.0f));
  const float scale = f16_value(sbits);
  uint32_t packed[4] = {0, 0, 0, 0};
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    float q = 0.0f;
    if (scale > 0.0f) q = fminf(fmaxf(__builtin_rintf(div_rn(x[e], scale)), -127.0f), 127.0f);
    packed[e >> 2] |= (uint32_t(int32_t(q)) & 0xffu) << (8 * (e & 3));
  }
  if (!is_k && kv.layout.dtype == Q38A_KV_INT8_VT) {  // V codes transposed, scales group-major
#pragma unroll
    for (int e = 0; e < 16; ++e) base[kv.layout.vt_code(head, 16 * l16 + e, tok)] = uint8_t(packed[e >> 2] >> (8 * (e & 3)));
    if ((l16 & 3) == 0) *reinterpret_cast<uint16_t*>(base + kv.layout.vt_scale(head, l16 >> 2, tok)) = sbits;
    return;
  }
  *reinterpret_cast<uint4*>(base + (is_k ? kv.layout.k_row(head, tok) : kv.layout.v_row(head, tok)) + 16 * l16) =
      uint4{packed[0], packed[1], packed[2], packed[3]};
  if ((l16 & 3) == 0)
    reinterpret_cast<uint16_t*>(base + (is_k ? kv.layout.k_scales(head, tok) : kv.layout.v_scales(head, tok)))[l16 >> 2] = sbits;
}

}  // namespace

int launch_qk_norm_rope_append(const q38a_qk_norm_rope_params& p, const q38a_batch_desc& b,
                               const q38a_kv_cache_desc& kv, hipStream_t stream) {
  if (b.num_tokens == 0) return Q38A_OK;
  const int rows = p.num_q_heads + 2 * p.num_kv_heads;
  const long long jobs = (long long)b.num_tokens * rows;
  if (jobs > (1ll << 30)) return set_error(Q38A_ERR_INVALID, "qk_norm_rope_append: too many tokens (%d)", b.num_tokens);
  AppendArgs a{p.proj, p.ld_proj, p.q_norm, p.k_norm, p.eps, p.num_q_heads, p.num_kv_heads, p.q_out,
               p.attn_layer, p.rope_cos_sin, p.rope_rows};
  // Four rows per wave from 8,192 rows on (256 tokens of 24 + 4 + 4 heads: 5.5 us against 6.0; 512
  // tokens 7.0 against 8.9; 2,048 tokens 17.2 against 28.1, 67 MB, i.e. 3.9 TB/s), where the buffers
  // take its 16-byte accesses. Below, one row per wave keeps more of the GPU busy.
  auto aligned = [](const void* q, size_t to) { return reinterpret_cast<uintptr_t>(q) % to == 0; };
  const bool wide = jobs >= 8192 && p.ld_proj % 8 == 0 && aligned(p.proj, 16) && aligned(p.q_out, 16) &&
                    aligned(p.q_norm, 16) && aligned(p.k_norm, 16) && aligned(p.rope_cos_sin, 16) &&
                    aligned(kv.pool, 16) && kv.layer_stride % 16 == 0 && kv.page_bytes % 16 == 0;
  if (wide) {
    const int waves = (b.num_tokens * p.num_q_heads + 3) / 4 + 2 * ((b.num_tokens * p.num_kv_heads + 3) / 4);
    hipLaunchKernelGGL(qk_norm_rope_append_rows_kernel, dim3((waves + kWavesPerBlock - 1) / kWavesPerBlock),
                       dim3(kWavesPerBlock * 64), 0, stream, a, to_args(b), to_args(kv));
  } else {
    const int blocks = int((jobs + kWavesPerBlock - 1) / kWavesPerBlock);
    hipLaunchKernelGGL(qk_norm_rope_append_kernel, dim3(blocks), dim3(kWavesPerBlock * 64), 0, stream, a,
                       to_args(b), to_args(kv), int(jobs));
  }
  return check_hip(hipGetLastError(), "qk_norm_rope_append launch");
}

}  // namespace q38a
