// BQ-weight GEMM for gfx950 (q38a_qgemm), the attention in-projection with its q/k norm, RoPE and KV
// append (q38a_qgemm_qkv_append: the GEMM into proj, then the append launch) and the o-projection
// behind split decode (q38a_qgemm_merge_oproj).
//
// Semantics follow reference src/kernels/qgemm.cu:285-384 (epilogues) and :573-616 (launcher):
// C[M][N] = A[M][K] . W^T, W[n][k] = code * scale[n][k / 64], A bf16, fp32 accumulation; StoreBF16
// stores bf16(C * rs) with the folded-RMSNorm row scale rs, Residual adds C into the fp32 residual
// stream and refreshes its bf16 copy and its per-128-column sums of squares.
//
// MI355X design: v_mfma_f32_32x32x16_bf16 with the activations as the A operand and the weights as B.
// A lane of the B operand holds eight consecutive k of one column; the repacked weights (bq_repack.cpp)
// give it those codes as one 16-byte word per 64-k group (+ the high bits). A kernel per range of M:
//   * up to 8 rows on a wide weight or with the residual epilogue (qgemv_wide_kernel) and up to 64
//     (qgemm_small_kernel) a launch is a stream of weights: each wave dequantises its own columns'
//     words in registers. The codes enter the MFMA as the exact bf16 values 128 + u (u = the stored
//     unsigned code, two bit operations per pair); the offset and the per-(column, group) scale are
//     applied once per group in fp32:
//       C += scale[n][g] * (T_g - (128 + 2^(b-1)) * S_g),  T_g = sum_{k in g} a[m][k] (128 + u),
//     S_g = sum_{k in g} a[m][k] from MFMAs of A against a constant. T carries at most ~8 bits of
//     cancellation; the result keeps ~16 significant bits, far below the bf16 output's rounding.
//   * beyond, a workgroup dequantises its columns once into LDS for all its rows: up to about 1,000
//     rows (qgemm_tile_kernel) as the exact signed codes, the scale still in fp32 once per group; where
//     256 x 256 tiles fill the CUs (qgemm_big_kernel) as bf16(code x scale), the reference's rounding.
//   * where tiles leave CUs idle, K is split over several workgroups: each writes its fp32 partial tile
//     with write-through stores, counts its arrival on a per-tile counter, and the last to arrive sums
//     the slices in slice order (deterministic) and runs the epilogue, then resets the counter.
//   * the o-projection's A merged in the loader has a split-K kernel of its own (qgemv_kernel).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "decode.hpp"
#include "q38a_gemm.h"

namespace q38a {

int decode_grid(int* grid, int* target_items);
int launch_attention_merge(const q38a_attention_params& p, const q38a_batch_desc& b, hipStream_t stream);
int launch_qk_norm_rope_append(const q38a_qk_norm_rope_params& p, const q38a_batch_desc& b,
                               const q38a_kv_cache_desc& kv, hipStream_t stream);

namespace {

// A workgroup of the merging split-K kernel covers 32 rows x 256 columns: two sets (K parts) of 8 waves of
// one 32-column block, each set over half the slice's groups (twice the weight bytes in flight per
// CU), their sums added through LDS.
constexpr int kTileN = 256;
constexpr int kColWaves = kTileN / 32;
constexpr int kKParts = 2;
constexpr int kGemvThreads = 64 * kColWaves * kKParts;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

struct GemmArgs {
  const uint16_t* a;
  int m, n, k;
  const uint8_t* lo;
  const uint8_t* hi;
  const uint16_t* scales;
  int kind;
  void* out;
  int ldo, n_store;
  float* residual;
  uint16_t* xbf;
  float* partials_out;
  const float* partials_in;
  int norm_blocks;
  int wide_norm;  // partials_in's rows take 16-byte loads
  float inv_hidden, eps;
  int tiles_n, splits;
  int wide_out;  // the epilogue's buffers take 16-byte accesses (alignment of pointers and row strides)
  float* ws_partials;
  int* counters;
};

// The o-projection's A from decode split partials (q38a_qgemm_merge_oproj): A[row][256 h + d] is the
// gated merge of (decode row, q head h), as the decode launch's merge kernel computes it.
struct MergeIn {
  const float* scratch;
  const uint16_t* gate;
  int ld_gate, nq, nkv, max_splits, target_items;
};

// One lane's share of one (32-column block, group) of weights: 32 low nibbles, their high bits, and
// the column's scale.
struct BWords {
  u32x4 lo;
  u32x2 hi;
  uint32_t scale;  // bf16 bits in the low half (converted where used, so the load is not awaited early)
};

// A wave-uniform address kept in scalar registers (a buffer resource built from an address the
// compiler computed in vector registers would otherwise be legalised lane by lane).
template <class T>
__device__ inline T* uniform_ptr(T* p) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint64_t lo = uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v)));
  const uint64_t hi = uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(v >> 32)));
  return reinterpret_cast<T*>(lo | (hi << 32));
}

// Buffer resources over the three weight planes: the per-group offsets are wave-uniform (scalar
// offsets), the lane's part a fixed vector offset, so no per-load 64-bit address arithmetic.
struct BPlanes {
  __amdgpu_buffer_rsrc_t lo, hi, sc;
};

template <int BITS>
__device__ inline BPlanes make_bplanes(const GemmArgs& a) {
  const int units = (a.n / 32) * (a.k / 64);
  constexpr int hb = BITS == 4 ? 0 : BITS == 5 ? 4 : 8;
  BPlanes p;
  p.lo = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.lo), short(0), units * 1024, 0x00020000);
  p.hi = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(BITS == 4 ? a.lo : a.hi), short(0), units * 64 * hb,
                                           0x00020000);
  p.sc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.scales), short(0), units * 64, 0x00020000);
  return p;
}

// Cache policy of a buffer load: non-temporal (data read once).
constexpr int kNonTemporal = 2;

template <int BITS, int CPOL = 0>
__device__ inline void load_bwords(BWords& b, const BPlanes& p, int nb, int g, int G, int lane) {
  const int unit = nb * G + g;
  b.lo = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(p.lo, lane * 16, unit * 1024, CPOL));
  if constexpr (BITS == 5) b.hi = u32x2{__builtin_amdgcn_raw_buffer_load_b32(p.hi, lane * 4, unit * 256, CPOL), 0u};
  else if constexpr (BITS == 6)
    b.hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(p.hi, lane * 8, unit * 512, CPOL));
  else b.hi = u32x2{0u, 0u};
  b.scale = __builtin_amdgcn_raw_buffer_load_b16(p.sc, (lane & 31) * 2, unit * 64, CPOL);
}

// (x & m) | c: one v_and_or_b32. Plain code, not inline assembly: an MFMA reading a register that an
// inline-assembly instruction wrote gets no hazard wait states from the compiler (it does not count
// the assembly as a VALU write), and then reads stale values.
__device__ inline uint32_t and_or(uint32_t x, uint32_t m, uint32_t c) { return (x & m) | c; }

// Shift right by a signed constant (left when negative).
template <int R>
__device__ inline uint32_t shr(uint32_t x) {
  if constexpr (R > 0) return x >> R;
  else if constexpr (R < 0) return x << (-R);
  else return x;
}

// Pair P of step S of the B operand: two bf16 values 128 + u, exact: the low nibbles masked into
// the magic 0x4300 (one shift and one and-or; no shift at P = 0), the high bits masked in at bit 4.
template <int BITS, int S, int P>
__device__ inline uint32_t b_pair(const BWords& b, uint32_t magic) {
  constexpr int q = 4 * S + P;
  uint32_t w = and_or(shr<4 * P>(b.lo[S]), 0x000F000Fu, magic);
  if constexpr (BITS == 5) w = and_or(shr<q - 4>(b.hi.x), 0x00100010u, w);
  if constexpr (BITS == 6) w = and_or(shr<2 * (q & 7) - 4>(q < 8 ? b.hi.x : b.hi.y), 0x00300030u, w);
  return w;
}

template <int BITS, int S>
__device__ inline bf16x8_t b_operand(const BWords& b, uint32_t magic) {
  const u32x4 v{b_pair<BITS, S, 0>(b, magic), b_pair<BITS, S, 1>(b, magic), b_pair<BITS, S, 2>(b, magic),
                b_pair<BITS, S, 3>(b, magic)};
  return __builtin_bit_cast(bf16x8_t, v);
}

// Row scale of the folded RMSNorm (reference qgemm.cu:288-297): 64 partials of the row in flight
// per round (loads past the row's end re-read its last ones and are not added), summed in block
// order. Sixteen-byte loads where the rows take them: a lane reads its own row, so single floats
// cost a request per lane and partial, 40 instead of 10 a row for 5,120 hidden values.
__device__ inline float row_scale(const GemmArgs& a, int row) {
  if (!a.partials_in || row >= a.m) return 1.0f;
  const float* pr = a.partials_in + size_t(row) * a.norm_blocks;
  const int last = a.norm_blocks - 1;
  float s = 0.0f;
  if (a.wide_norm) {
    for (int b = 0; b < a.norm_blocks; b += 64) {
      float4 v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = reinterpret_cast<const float4*>(pr)[b + 4 * i < last ? b / 4 + i : last / 4];
#pragma unroll
      for (int i = 0; i < 16; ++i) s = b + 4 * i <= last ? (((s + v[i].x) + v[i].y) + v[i].z) + v[i].w : s;
    }
  } else {
    for (int b = 0; b < a.norm_blocks; b += 64) {
      float v[64];
#pragma unroll
      for (int i = 0; i < 64; ++i) v[i] = pr[b + i < last ? b + i : last];
#pragma unroll
      for (int i = 0; i < 64; ++i) s = b + i <= last ? s + v[i] : s;
    }
  }
  return 1.0f / __builtin_sqrtf(s * a.inv_hidden + a.eps);
}

struct alignas(16) GemmShared {
  union {
    float resid_ss[kColWaves][32];   // residual epilogue: per-wave sums of squares of its columns
    float kpart[kColWaves][16][64];  // the second K part's sums
  };
  float rs[32];                       // row scales of the folded RMSNorm (1 without partials_in)
  int last;
};

// The merging split-K kernel's end: split-K slices summed by the last workgroup to arrive, then the epilogue.
// C element e in this lane: row 8 (e / 4) + 4 (lane / 32) + e % 4, column 32 wave + lane % 32 of the
// tile. Every wave of the column tile calls it (K-part waves have ended); sh.rs holds the rows' scales.
// EQ: row quads of the MFMA output that can hold rows < M (the split-K traffic skips the others).
template <int EQ>
__device__ void tile_finish(const GemmArgs& a, GemmShared& sh, float16_t& C, int tn, int z, int wave, int lane) {
  constexpr int kRows = 32;
  const int kg = lane >> 5;
  auto row_of = [&](int e) { return 8 * (e >> 2) + 4 * kg + (e & 3); };
  const int col = tn * kTileN + 32 * wave + (lane & 31);

  // ---- split-K: the last of the tile's slices sums them in slice order -------------------------
  if (a.splits > 1) {
    float* part = a.ws_partials + size_t(tn) * a.splits * kRows * kTileN;
#pragma unroll
    for (int e = 0; e < 4 * EQ; ++e) {
      const int r = row_of(e);
      if (r < a.m)
        __hip_atomic_store(part + (size_t(z) * kRows + r) * kTileN + 32 * wave + (lane & 31), C[e], __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    // Hand-off without release/acquire fences: the partials are agent-scope atomic stores, which
    // gfx950 issues write-through past the XCD's L2 (sc1), s_waitcnt(0) waits until every one has
    // completed, the barrier orders all threads' completed stores before thread 0's arrival count,
    // and the last arrival reads the partials with agent-coherent (sc1) loads, which miss the
    // non-coherent L2. Agent-scope fences would add an L2 write-back (buffer_wbl2 sc1) and
    // invalidate (buffer_inv sc1) per workgroup: measured, they nearly doubled the small-M GEMM
    // (in-projection batch 8: 0.022 -> 0.041 ms; o-projection 0.017 -> 0.029 ms).
    __builtin_amdgcn_s_waitcnt(0);  // the write-through stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
      const int old = __hip_atomic_fetch_add(a.counters + tn, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.last = old == a.splits - 1;
      if (sh.last) __hip_atomic_store(a.counters + tn, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!sh.last) return;
    // the slices in slice order, this workgroup's own included (its stores have completed), read
    // with agent-coherent (sc1) buffer loads; kZB slices' loads are issued together (a batch past
    // the last slice re-reads the last one and discards it)
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        part, short(0), int(size_t(a.splits) * kRows * kTileN * sizeof(float)), 0x00020000);
    constexpr int kSc1 = 16;  // cache policy bit sc1
    constexpr int kZB = 16 / EQ;
#pragma unroll
    for (int e = 0; e < 16; ++e) C[e] = 0.0f;
    for (int zb = 0; zb < a.splits; zb += kZB) {
      float V[kZB][4 * EQ];
#pragma unroll
      for (int q = 0; q < kZB; ++q) {
        const int zz = zb + q < a.splits ? zb + q : a.splits - 1;
        const int zoff = zz * kRows * kTileN * int(sizeof(float));
#pragma unroll
        for (int e = 0; e < 4 * EQ; ++e) {
          const int off = (row_of(e) * kTileN + 32 * wave + (lane & 31)) * int(sizeof(float));
          V[q][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(prs, off, zoff, kSc1));
        }
      }
#pragma unroll
      for (int q = 0; q < kZB; ++q) {
        const bool use = zb + q < a.splits;
#pragma unroll
        for (int e = 0; e < 4 * EQ; ++e) C[e] = use ? C[e] + V[q][e] : C[e];
      }
    }
  }

  // ---- epilogues --------------------------------------------------------------------------------
  if (a.splits == 1) __syncthreads();  // sh.rs (the split-K path has passed barriers already)
  float rs[16];
#pragma unroll
  for (int e = 0; e < 16; ++e) rs[e] = sh.rs[row_of(e)];
  if (a.kind == Q38A_EPI_RESIDUAL) {
    // residual += C; xbf = bf16(residual); sums of squares per 128 columns (reference
    // qgemm.cu:356-380; the sum's order differs): the 32 lanes of each half wave, then the four
    // waves of each 128-column block in wave order
    float ss[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = row_of(e);
      ss[e] = 0.f;
      if (row < a.m) {
        float* res = a.residual + size_t(row) * a.n + col;
        const float x = *res + C[e];
        *res = x;
        a.xbf[size_t(row) * a.n + col] = bf16_bits(x);
        ss[e] = x * x;
      }
#pragma unroll
      for (int off = 16; off > 0; off >>= 1) ss[e] += __shfl_xor(ss[e], off, 64);
    }
    __syncthreads();
    if ((lane & 31) == 0) {
#pragma unroll
      for (int e = 0; e < 16; ++e) sh.resid_ss[wave][row_of(e)] = ss[e];
    }
    __syncthreads();
    if (threadIdx.x < 2 * kRows) {
      const int bw = threadIdx.x >> 5, r = threadIdx.x & 31;
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < 4; ++w) v += sh.resid_ss[4 * bw + w][r];
      if (r < a.m) a.partials_out[size_t(r) * a.norm_blocks + (tn * kTileN) / 128 + bw] = v;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int row = row_of(e);
      if (row >= a.m || col >= a.n_store) continue;
      const float y = C[e] * rs[e];
      if (a.kind == Q38A_EPI_STORE_F32) static_cast<float*>(a.out)[size_t(row) * a.ldo + col] = y;
      else static_cast<uint16_t*>(a.out)[size_t(row) * a.ldo + col] = bf16_bits(y);
    }
  }
}

// T = A . (128 + u) over a group's four 16-k steps of one column block, with A's steps in registers.
template <int BITS>
__device__ inline float16_t group_products(const u32x4 (&Ab)[4], const BWords& bw, uint32_t magic) {
  float16_t T = float16_t{};
  auto t_step = [&](auto step) {
    constexpr int s = decltype(step)::value;
    T = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, Ab[s]), b_operand<BITS, s>(bw, magic), T, 0,
                                                0, 0);
  };
  t_step(std::integral_constant<int, 0>{});
  t_step(std::integral_constant<int, 1>{});
  t_step(std::integral_constant<int, 2>{});
  t_step(std::integral_constant<int, 3>{});
  return T;
}

// ---- the epilogue of the tile kernels --------------------------------------------------------------
// A wave's output goes out in blocks of 32 rows x 64 columns, each laid out by rows in the wave's LDS
// block first, so that every store instruction covers whole 128- or 256-byte row runs.
typedef float OutBlock[32][64 + 4];

// Two MFMA outputs (columns 0-31 and 32-63) by rows: element e of a lane is row 8 (e / 4) + 4 (lane / 32)
// + e % 4, column lane % 32.
__device__ inline void block_to_rows(OutBlock& ot, const float16_t& left, const float16_t& right, int lane) {
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int r = 8 * (e >> 2) + 4 * (lane >> 5) + (e & 3);
    ot[r][lane & 31] = left[e];
    ot[r][32 + (lane & 31)] = right[e];
  }
}

// The block at (row0, col0): rs_of its rows' scales (store epilogues), ss its rows' sums of squares over
// the 64 columns (residual epilogue), both in LDS.
__device__ inline void store_block(const GemmArgs& a, const OutBlock& ot, int row0, int col0, const float* rs_of, float* ss,
                                   int lane) {
  if (a.kind == Q38A_EPI_RESIDUAL) {
    // four columns per lane, four rows per instruction
    const int c = 4 * (lane & 15), col = col0 + c;
    float ssum[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + (lane >> 4), row = row0 + r;
      const float4 y = *reinterpret_cast<const float4*>(&ot[r][c]);
      ssum[i] = 0.0f;
      if (row < a.m) {
        float* res = a.residual + size_t(row) * a.n + col;
        float x[4] = {y.x, y.y, y.z, y.w};
        if (a.wide_out) {
          const float4 p = *reinterpret_cast<const float4*>(res);
          x[0] += p.x;
          x[1] += p.y;
          x[2] += p.z;
          x[3] += p.w;
          *reinterpret_cast<float4*>(res) = float4{x[0], x[1], x[2], x[3]};
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            x[u] += res[u];
            res[u] = x[u];
          }
        }
        uint16_t* xb = a.xbf + size_t(row) * a.n + col;
        if (a.wide_out)
          *reinterpret_cast<uint2*>(xb) = uint2{uint32_t(bf16_bits(x[0])) | (uint32_t(bf16_bits(x[1])) << 16),
                                                uint32_t(bf16_bits(x[2])) | (uint32_t(bf16_bits(x[3])) << 16)};
        else
#pragma unroll
          for (int u = 0; u < 4; ++u) xb[u] = bf16_bits(x[u]);
        ssum[i] = x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3];
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) ssum[i] += __shfl_xor(ssum[i], o, 64);
      if ((lane & 15) == 0) ss[4 * i + (lane >> 4)] = ssum[i];
    }
  } else if (a.kind == Q38A_EPI_STORE_F32) {
    const int c = 4 * (lane & 15), col = col0 + c;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int r = 4 * i + (lane >> 4), row = row0 + r;
      if (row >= a.m) continue;
      const float rs = rs_of[r];
      const float4 y = *reinterpret_cast<const float4*>(&ot[r][c]);
      const float x[4] = {y.x * rs, y.y * rs, y.z * rs, y.w * rs};
      float* out = static_cast<float*>(a.out) + size_t(row) * a.ldo + col;
      if (a.wide_out && col + 4 <= a.n_store) *reinterpret_cast<float4*>(out) = float4{x[0], x[1], x[2], x[3]};
      else
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (col + u < a.n_store) out[u] = x[u];
    }
  } else {
    // eight columns per lane, eight rows per instruction
    const int c = 8 * (lane & 7), col = col0 + c;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 8 * i + (lane >> 3), row = row0 + r;
      if (row >= a.m) continue;
      const float rs = rs_of[r];
      const float4 y0 = *reinterpret_cast<const float4*>(&ot[r][c]), y1 = *reinterpret_cast<const float4*>(&ot[r][c + 4]);
      const uint16_t x[8] = {bf16_bits(y0.x * rs), bf16_bits(y0.y * rs), bf16_bits(y0.z * rs), bf16_bits(y0.w * rs),
                             bf16_bits(y1.x * rs), bf16_bits(y1.y * rs), bf16_bits(y1.z * rs), bf16_bits(y1.w * rs)};
      uint16_t* out = static_cast<uint16_t*>(a.out) + size_t(row) * a.ldo + col;
      if (a.wide_out && col + 8 <= a.n_store)
        *reinterpret_cast<u32x4*>(out) = u32x4{uint32_t(x[0]) | (uint32_t(x[1]) << 16), uint32_t(x[2]) | (uint32_t(x[3]) << 16),
                                               uint32_t(x[4]) | (uint32_t(x[5]) << 16), uint32_t(x[6]) | (uint32_t(x[7]) << 16)};
      else
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (col + u < a.n_store) out[u] = x[u];
    }
  }
}

// ---- 65 rows and more: 256 x 128 or 128 x 128 tiles, exact codes -------------------------------
// Eight waves of 64 x 64. The tile's columns are dequantised once per workgroup into LDS as the
// exact signed codes in bf16 (MFMA B operand layout: block, step, lane, 8 k) and shared by the
// waves of its rows; A rows come by the DMA path of buffer loads, 16-byte chunk c of a row in
// slot c ^ (row / 2 % 8): the 16 rows that one clock of an operand read takes then fall in 16 different
// quads of the 64 banks. Each 64-k group's products accumulate in their own registers (T, starting from
// zero) and C += scale * T in fp32 when the group is done: the codes are exact, so the only
// roundings are the fp32 sums'. One column block's T is folded while the other block's MFMAs run,
// and the last one's beside the next step's first MFMAs. KP: 64-k groups per step. With 256 rows a step
// is one group; with 128 rows two sets of four waves take one group each, and the sets' sums are added
// through LDS at the end (set 0 + set 1).
//
// Bound: the VALU beside the MFMA. Per 64 x 64 x 64 wave step 16 MFMAs (512 cycles) against 64 folds
// and 50 (5-bit codes, 256 rows) or 100 dequantisation instructions; two waves per SIMD hide about six
// vector instructions per MFMA (measured, register-only loops). In-projection at 512 rows, GEMM alone:
// 84 us, 0.9 us a step and ~10 us around them (897 TFLOP/s; hipBLASLt's plain bf16 product 90 us), against
// 216 us of the kernel before, which read both operands from global memory in every wave; 100 us with
// all waves in step, 93 with slot c ^ (row % 8).
constexpr int kTileWaves = 8;
constexpr int kTileThreads = 64 * kTileWaves;
constexpr int kTileCols = 128;  // two waves wide
constexpr int kTileMaxSplits = 8;
// rows per tile for WM waves of 64 rows; 64-k groups per step
__host__ __device__ constexpr int tile_rows(int wm) { return 64 * wm; }
__host__ __device__ constexpr int tile_kparts(int wm) { return kTileWaves / (2 * wm); }

template <int WM>
struct alignas(16) TileShared {
  union {
    struct {
      u32x4 a[3][256][8];  // [buffer][group of the step, row][slot]: 256 = rows x groups for every WM
      uint16_t b[2][tile_kparts(WM)][4][4][64][8];  // [buffer][group][block][step][lane][k]
    } s;
    struct {  // after the K loop
      union {
        float red[4][64][64];               // the second K part's sums: [wave][element][lane]
        OutBlock out[kTileWaves];           // 32 rows of a wave's tile
      };
      float rs[tile_rows(WM)];     // row scales of the folded RMSNorm
      float ss[2][tile_rows(WM)];  // residual epilogue: each wave column's sums of squares
      int last;
    } e;
  };
};

// 16 bytes per lane from the buffer to LDS at dst (wave-uniform) + 16 x lane, without registers.
__device__ inline void copy_to_lds(__amdgpu_buffer_rsrc_t r, u32x4* dst, int voffset, int soffset) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, voffset, soffset, 0, 0);
}

// s_waitcnt's immediate for "at most n vector memory loads in flight" (gfx9 encoding, the other counters
// not waited for). The loads retire in order, so it says that everything issued before the newest n has
// landed. n counts loads that the code after it reads: the compiler deletes the others, and a wait that
// counts a deleted load leaves the copy before it in flight.
constexpr int vm_in_flight(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }
// As well, that every LDS operation of the wave has completed.
constexpr int vm_in_flight_lds_done(int n) { return vm_in_flight(n) & ~0x0F00; }

// One thread's share of a step's weights: NS 16-k steps of one lane word (their low nibbles, 32
// bits a step) and the high bits of those steps.
template <int NS>
struct TileWords {
  uint32_t lo[NS];
  u32x2 hi;
};

// Steps [first, first + NS) of lane word l of block nb, group g (nb and g wave-uniform).
template <int BITS, int NS>
__device__ inline void load_tile_words(TileWords<NS>& w, const BPlanes& p, int nb, int g, int G, int l, int first) {
  const int unit = nb * G + g;
  if constexpr (NS == 4) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(p.lo, l * 16, unit * 1024, 0));
    w.lo[0] = v.x;
    w.lo[1] = v.y;
    w.lo[2] = v.z;
    w.lo[3] = v.w;
  } else {
    const u32x2 v =
        __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(p.lo, l * 16 + 4 * first, unit * 1024, 0));
    w.lo[0] = v.x;
    w.lo[1] = v.y;
  }
  if constexpr (BITS == 5) w.hi = u32x2{__builtin_amdgcn_raw_buffer_load_b32(p.hi, l * 4, unit * 256, 0), 0u};
  else if constexpr (BITS == 6 && NS == 4)
    w.hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(p.hi, l * 8, unit * 512, 0));
  else if constexpr (BITS == 6)  // steps 0-1 are in the first word, 2-3 in the second
    w.hi = u32x2{__builtin_amdgcn_raw_buffer_load_b32(p.hi, l * 8 + 2 * first, unit * 512, 0), 0u};
  else w.hi = u32x2{0u, 0u};
}

// (x & mask) | c in one instruction (the compiler splits it over a literal AND and an OR3). Only for
// values that vector instructions read: see and_or.
__device__ inline uint32_t and_or_valu(uint32_t x, uint32_t mask, uint32_t c) {
  uint32_t d;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(d) : "v"(x), "s"(mask), "v"(c));
  return d;
}

// Codes 2P and 2P + 1 of a lane word's step as a pair of signed codes in bf16, exact. lo: the step's
// nibbles, for P >= 2 already shifted right by 8; hi: the high bits. The fp16 values 2048 + 2 u (P
// even) or 2048 + 32 u (P odd: the nibble stays where it is), then one mixed-precision fma per code,
// which reads the fp16 half and takes the factor and the offset off, and one conversion of both.
template <int BITS, int S, int P>
__device__ inline uint32_t code_pair_bf16(uint32_t lo, uint32_t hi, uint32_t magic) {
  constexpr int q = 4 * S + P, up = P & 1 ? 4 : 0;  // the code's lowest bit in the fp16 mantissa
  uint32_t w = and_or_valu(lo, 0x000F000Fu << up, magic);
  if constexpr (BITS == 5) w = and_or_valu(shr<q - 4 - up>(hi), 0x00100010u << up, w);
  if constexpr (BITS == 6) w = and_or_valu(shr<2 * (q & 7) - 4 - up>(hi), 0x00300030u << up, w);
  constexpr float f = P & 1 ? 1.0f / 32 : 0.5f, off = -(2048.0f * f + float(1 << (BITS - 1)));
  const half2_t h = __builtin_bit_cast(half2_t, w);
  const float2_t x{__builtin_fmaf(float(h.x), f, off), __builtin_fmaf(float(h.y), f, off)};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2_t));
}

// Step S of the thread's words into LDS.
template <int BITS, int NS, int S>
__device__ inline void tile_dequant_step(uint16_t* dst, const TileWords<NS>& w, uint32_t hi, uint32_t magic) {
  const uint32_t lo = w.lo[S], lo8 = lo >> 8;
  const u32x4 v{code_pair_bf16<BITS, S, 0>(lo, hi, magic), code_pair_bf16<BITS, S, 1>(lo, hi, magic),
                code_pair_bf16<BITS, S, 2>(lo8, hi, magic), code_pair_bf16<BITS, S, 3>(lo8, hi, magic)};
  *reinterpret_cast<u32x4*>(dst) = v;
}

template <int BITS, int WM>
__global__ void __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) qgemm_tile_kernel(GemmArgs a) {
  constexpr int KP = tile_kparts(WM), BM = tile_rows(WM);
  constexpr int NS = KP == 1 ? 2 : 4;  // 16-k steps each thread dequantises per step
  __shared__ TileShared<WM> sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, kg = lane >> 5;
  const int kp = wave / (2 * WM), wi = wave % (2 * WM), wm = wi >> 1, wn = wi & 1;
  // tiles of one column block (the same weights) and its K slices on one XCD (blockIdx mod 8), when
  // the column blocks divide evenly
  const int tiles_m = (a.m + BM - 1) / BM, inner = tiles_m * a.splits;
  int tn, rest;
  if (a.tiles_n % 8 == 0) {
    const int idx = blockIdx.x >> 3;
    tn = (idx / inner) * 8 + (blockIdx.x & 7);
    rest = idx % inner;
  } else {
    tn = blockIdx.x / inner;
    rest = blockIdx.x % inner;
  }
  tn = __builtin_amdgcn_readfirstlane(tn);
  const int tm = __builtin_amdgcn_readfirstlane(rest / a.splits), z = __builtin_amdgcn_readfirstlane(rest % a.splits);
  const int m0 = tm * BM;
  const int G = a.k / 64;
  const int g0 = int((long long)z * G / a.splits), g1 = int((long long)(z + 1) * G / a.splits);
  const int steps = (g1 - g0 + KP - 1) / KP;
  const BPlanes bp = make_bplanes<BITS>(a);
  const int valid_rows = a.m - m0 < BM ? a.m - m0 : BM;
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(const_cast<uint16_t*>(a.a) + size_t(m0) * a.k), short(0), valid_rows * a.k * int(sizeof(uint16_t)),
      0x00020000);
  const uint32_t magic = 0x68006800u;  // fp16 2048 in both halves

  // the thread's lane word of the step's weights: group dkp of the step, block db, lane dl; with one
  // group per step, steps 2 dh and 2 dh + 1 of it
  const int dkp = KP == 1 ? 0 : wave >> 2, db = wave & 3, dh = KP == 1 ? wave >> 2 : 0, dl = lane;
  // Past the slice's last group every load repeats it (and meets A rows of zeros).
  auto gclamp = [&](int g) { return g < g1 - 1 ? g : g1 - 1; };
  // A rows of step t by DMA: wave w copies rows 32 w .. 32 w + 31 of the step's 256 (group, row)
  // pairs, 8 rows (1 KB) an instruction; a group past the slice's end loads zeros (outside the range)
  const int arow = (32 * wave) % BM + (lane >> 3), akp = (32 * wave) / BM;
  const int avoff = (arow * a.k + 8 * ((lane & 7) ^ (lane >> 4))) * 2;
  auto dma_a = [&](int t, int buf) {
    const int g = g0 + t * KP + akp;
    const int lost = g < g1 ? 0 : int(0x80000000u);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      copy_to_lds(ars, &sh.s.a[buf][32 * wave + 8 * i][0], ((i & 1 ? avoff ^ 64 : avoff) + 16 * i * a.k) | lost,
                  128 * gclamp(g));
  };
  auto load_words = [&](TileWords<NS>& w, int t) {
    load_tile_words<BITS, NS>(w, bp, 4 * tn + db, gclamp(g0 + t * KP + dkp), G, dl, NS == 2 ? 2 * dh : 0);
  };
  // bf16 bits of this lane's column scale in each of the wave's two column blocks
  auto load_scales = [&](uint32_t (&s)[2], int t) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
      s[j] = __builtin_amdgcn_raw_buffer_load_b16(bp.sc, (lane & 31) * 2,
                                                  ((4 * tn + 2 * wn + j) * G + gclamp(g0 + t * KP + kp)) * 64, 0);
  };
  auto high_bits = [&](const TileWords<NS>& w) {  // of the thread's own steps
    if constexpr (BITS == 5 && NS == 2) return w.hi.x >> (8 * dh);
    else return w.hi.x;
  };

  float16_t C[2][2], T[2][2];  // [column block][row block]
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      C[j][mb] = float16_t{};
      T[j][mb] = float16_t{};
    }
  // Words and scales go out three steps ahead (~3 us: each is read once, from HBM, by this workgroup's
  // XCD). Slot t % 4 holds the words dequantised in step t - 1 and the scales of step t.
  TileWords<NS> wq[4];
  uint32_t sc[4][2];
  float last_sc = 0.0f;
  auto dequant = [&](auto sc_, int buf, const TileWords<NS>& w) {
    constexpr int S = decltype(sc_)::value;
    // (6-bit words of four steps keep steps 2-3 in their second high word)
    const uint32_t hi = BITS == 6 && NS == 4 && S >= 2 ? w.hi.y : high_bits(w);
    tile_dequant_step<BITS, NS, S>(&sh.s.b[buf][dkp][db][2 * dh + S][dl][0], w, hi, magic);
  };
  using i0 = std::integral_constant<int, 0>;
  using i1 = std::integral_constant<int, 1>;
  using i2 = std::integral_constant<int, 2>;
  using i3 = std::integral_constant<int, 3>;
  const int ahead = wave >= 4 ? 1 : 0;
  auto dequant_all = [&](int buf, const TileWords<NS>& w) {
    dequant(i0{}, buf, w);
    dequant(i1{}, buf, w);
    if constexpr (NS == 4) {
      dequant(i2{}, buf, w);
      dequant(i3{}, buf, w);
    }
  };
  dma_a(0, 0);
  dma_a(1, 1);
  TileWords<NS> first[2];
  load_words(first[0], 0);
  load_words(first[1], 1);
  load_scales(sc[0], 0);
#pragma unroll
  for (int i = 1; i < 4; ++i) {
    load_words(wq[i], i + ahead);
    if (i < 3) load_scales(sc[i], i);
  }
  const float my_rs = int(threadIdx.x) < BM ? row_scale(a, m0 + threadIdx.x) : 0.0f;  // (with the first loads in flight)
  dequant_all(0, first[0]);
  if (ahead) dequant_all(1, first[1]);
  __builtin_amdgcn_s_waitcnt(0);  // the DMA copies of steps 0 and 1 have landed
  __syncthreads();

  auto fold = [&](int j, float s) {
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int e = 0; e < 16; ++e) C[j][mb][e] = __builtin_fmaf(s, T[j][mb][e], C[j][mb][e]);
  };
  // One step in two phases with a barrier after each: operand reads and loads, then the MFMAs with the
  // folds and the dequantisation in their shadow. Waves 4-7 run half a step behind waves 0-3, so of a
  // SIMD's two waves one is in each phase. Waves 0-3 dequantise step t + 1 beside the MFMAs of step t,
  // waves 4-7 step t + 2 (ahead = 1): either is then complete when waves 0-3 start to read it. The copies
  // of a step's A rows go out two steps ahead into the buffer read a step ago. Both overwrite what waves
  // 4-7 read in the phase before, so a wave's operand reads have returned when it passes the barrier
  // after them (in-projection, 512 rows: 390 us with the wait; with it only where tiles of 256 rows need
  // it, 391; o-projection, 519 rows: 253, 256). cur = t % 4 is a compile-time constant, so the register
  // rings are indexed statically.
  int abuf = 0;  // t mod 3: the A buffer of step t
  // (A plain barrier: __syncthreads would wait for every copy in flight. The empty assembly keeps the
  // compiler from moving memory accesses across it.)
  auto phase_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // TAIL: one of the up to three steps after the unrolled loop; no later step reads what they would load.
  constexpr int kCopies = 4, kLoads = (BITS == 4 ? 1 : 2) + 2;  // of a step: A copies; words and scales
  auto step = [&](int t, auto curc, auto tailc) {
    constexpr int cur = decltype(curc)::value;
    constexpr bool TAIL = decltype(tailc)::value;
    const TileWords<NS>& wnext = wq[(cur + 1) & 3];
    const int wbuf = (cur & 1) ^ 1 ^ ahead;
    bf16x8_t ao[4][2], bo[2][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const int r = 64 * wm + 32 * mb + (lane & 31);
        ao[s][mb] = __builtin_bit_cast(bf16x8_t, sh.s.a[abuf][kp * BM + r][(2 * s + kg) ^ ((r >> 1) & 7)]);
      }
      bo[0][s] = *reinterpret_cast<const bf16x8_t*>(&sh.s.b[cur & 1][kp][2 * wn][s][lane][0]);
    }
#pragma unroll
    for (int s = 0; s < 4; ++s)
      bo[1][s] = *reinterpret_cast<const bf16x8_t*>(&sh.s.b[cur & 1][kp][2 * wn + 1][s][lane][0]);
    __builtin_amdgcn_sched_barrier(0);
    dma_a(t + 2, abuf == 0 ? 2 : abuf - 1);
    // the wait at the phase's end counts the loads issued after the copies: keep that order
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!TAIL) {
      load_words(wq[cur], t + 4 + ahead);
      load_scales(sc[(cur + 3) & 3], t + 3);
      __builtin_amdgcn_sched_barrier(0);
    }
    // the copies of step t + 1 have landed: after them went out that step's loads, the copies of step
    // t + 2 and this step's loads; in the tail only the newest copies are sure to have. And the operand
    // reads have returned.
    __builtin_amdgcn_s_waitcnt(vm_in_flight_lds_done(TAIL ? kCopies : kLoads + kCopies + kLoads));
    phase_end();
    __builtin_amdgcn_s_setprio(1);
    fold(1, last_sc);  // the previous step's second column block
    dequant(i0{}, wbuf, wnext);
    if constexpr (NS == 4) dequant(i1{}, wbuf, wnext);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
          T[j][mb] =
              __builtin_amdgcn_mfma_f32_32x32x16_bf16(ao[s][mb], bo[j][s], s == 0 ? float16_t{} : T[j][mb], 0, 0, 0);
    fold(0, bf16_value(uint16_t(sc[cur][0])));
    if constexpr (NS == 4) {
      dequant(i2{}, wbuf, wnext);
      dequant(i3{}, wbuf, wnext);
    } else {
      dequant(i1{}, wbuf, wnext);
    }
    last_sc = bf16_value(uint16_t(sc[cur][1]));
    abuf = abuf == 2 ? 0 : abuf + 1;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
      __builtin_amdgcn_sched_group_barrier(0x002, NS == 4 ? 10 : 7, 0);  // then vector instructions
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's dequantised codes are in LDS
    phase_end();
  };
  if (wave >= 4) phase_end();
  int t = 0;
  for (; t + 3 < steps; t += 4) {
    step(t, i0{}, std::false_type{});
    step(t + 1, i1{}, std::false_type{});
    step(t + 2, i2{}, std::false_type{});
    step(t + 3, i3{}, std::false_type{});
  }
  if (t < steps) step(t, i0{}, std::true_type{});
  if (t + 1 < steps) step(t + 1, i1{}, std::true_type{});
  if (t + 2 < steps) step(t + 2, i2{}, std::true_type{});
  if (wave < 4) phase_end();
  fold(1, last_sc);
  // the copies past the last step have landed and every wave is past its last operand read: LDS is
  // free for the epilogue
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (int(threadIdx.x) < BM) sh.e.rs[threadIdx.x] = my_rs;

  // ---- the K parts' sums: part 0 + part 1, through LDS
  if constexpr (KP == 2) {
    if (kp == 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int e = 0; e < 16; ++e) sh.e.red[wi][(2 * j + mb) * 16 + e][lane] = C[j][mb][e];
    }
    __syncthreads();
    if (kp == 1) return;  // (barriers count only the waves still running)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e) C[j][mb][e] += sh.e.red[wi][(2 * j + mb) * 16 + e][lane];
  }
  __syncthreads();

  // ---- split-K: the tile's slices in slice order, summed by the last workgroup to arrive (the
  // hand-off of tile_finish: write-through stores, their completion, an arrival count, coherent loads)
  if (a.splits > 1) {
    constexpr int kSc1 = 16;                       // cache policy bit sc1
    constexpr int kWaveBytes = 64 * 64 * 4;        // a wave's sums: [quad][lane][4 floats]
    constexpr int kSliceBytes = 2 * WM * kWaveBytes;
    const int tile = tn * tiles_m + tm;
    float* part = uniform_ptr(a.ws_partials + size_t(tile) * a.splits * (kSliceBytes / 4));
    const __amdgpu_buffer_rsrc_t prs =
        __builtin_amdgcn_make_buffer_rsrc(part, short(0), a.splits * kSliceBytes, 0x00020000);
    const int off = wi * kWaveBytes + lane * 16;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x4 v{as_u32(C[j][mb][4 * q]), as_u32(C[j][mb][4 * q + 1]), as_u32(C[j][mb][4 * q + 2]),
                        as_u32(C[j][mb][4 * q + 3])};
          __builtin_amdgcn_raw_buffer_store_b128(v, prs, off + ((2 * j + mb) * 4 + q) * 1024, z * kSliceBytes, kSc1);
        }
    __builtin_amdgcn_s_waitcnt(0);  // the write-through stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
      const int old = __hip_atomic_fetch_add(a.counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.e.last = old == a.splits - 1;
      if (sh.e.last) __hip_atomic_store(a.counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!sh.e.last) return;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) C[j][mb] = float16_t{};
    // two slices' loads in flight (past the last slice: that one again, not added)
    u32x4 v[2][16];
    auto load_slice = [&](u32x4 (&d)[16], int zz) {
      const int zc = zz < a.splits ? zz : a.splits - 1;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        d[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(prs, off + i * 1024, zc * kSliceBytes, kSc1));
    };
    auto add_slice = [&](const u32x4 (&d)[16]) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float16_t& c = C[i >> 3][(i >> 2) & 1];
        c[4 * (i & 3)] += as_f32(d[i].x);
        c[4 * (i & 3) + 1] += as_f32(d[i].y);
        c[4 * (i & 3) + 2] += as_f32(d[i].z);
        c[4 * (i & 3) + 3] += as_f32(d[i].w);
      }
    };
    load_slice(v[0], 0);
    for (int zz = 0; zz < a.splits; zz += 2) {
      load_slice(v[1], zz + 1);
      add_slice(v[0]);
      load_slice(v[0], zz + 2);
      if (zz + 1 < a.splits) add_slice(v[1]);
    }
  }

  // ---- epilogue: 32 rows of the wave's 64 columns at a time through LDS
#pragma unroll
  for (int mb = 0; mb < 2; ++mb) {
    const int r0 = 64 * wm + 32 * mb;
    block_to_rows(sh.e.out[wave], C[0][mb], C[1][mb], lane);
    store_block(a, sh.e.out[wave], m0 + r0, tn * kTileCols + 64 * wn, sh.e.rs + r0, sh.e.ss[wn] + r0, lane);
  }
  if (a.kind == Q38A_EPI_RESIDUAL) {
    // the tile's 128 columns are one block of the sums of squares: its two waves' halves, in order
    __syncthreads();
    const int r = threadIdx.x;  // part 0's waves only: 2 WM x 64 threads >= BM
    if (r < BM && m0 + r < a.m) a.partials_out[size_t(m0 + r) * a.norm_blocks + tn] = sh.e.ss[0][r] + sh.e.ss[1][r];
  }
}

// ---- large M: 256 x 256 tiles, weights as bf16(code x scale) ------------------------------------
// As the tiles above, with eight waves of 64 rows x 128 columns and the weights staged in LDS as
// bf16(code x scale) (the reference's own weight rounding, qgemm.cu), so that the MFMA accumulates
// across groups directly. A group goes in two halves of 32 k, each a memory phase (12 operand reads,
// in the second half also the copies of A two groups ahead and the weights' loads) and a compute phase (16 MFMAs with half a
// lane word's dequantisation, ~3 vector instructions per MFMA), waves 4-7 one phase behind. The tile
// count fills the CUs, so no split-K.
//
// Bound: MFMA, at the clock the card holds under it. In-projection at 2,048 rows (448 tiles on 256 CUs: 2
// rounds for 1.75): 301 -> 265 us against the form with all waves in step and 2-byte stores (1,136 TFLOP/s;
// hipBLASLt's plain bf16 product 245-256 us on the same card; 285 and 327 us on cards with lower clocks).
constexpr int kBigRows = 256;
constexpr int kBigWaves = 8;
constexpr int kBigThreads = 64 * kBigWaves;

struct alignas(16) BigShared {
  union {
    struct {
      u32x4 a[3][kBigRows][8];       // three groups of the tile's A rows, [row][slot] as in TileShared
      uint16_t b[2][8][4][64][8];    // two groups of the tile's weights: [block][step][lane][k]
    } s;
    struct {  // after the K loop
      OutBlock out[kBigWaves];
      float rs[kBigRows];     // row scales of the folded RMSNorm
      float ss[4][kBigRows];  // residual epilogue: sums of squares of each 64 columns
    } e;
  };
};

// As code_pair_bf16, times the column's scale: bf16(code x scale), rounded once (the fma's result, 14
// significant bits, is exact). sc and off: the scale times the factor and the offset of even [0] and
// odd [1] pairs.
template <int BITS, int S, int P>
__device__ inline uint32_t scaled_pair_bf16(uint32_t lo, uint32_t hi, uint32_t magic, const float (&sc)[2],
                                           const float (&off)[2]) {
  constexpr int q = 4 * S + P, up = P & 1 ? 4 : 0;
  uint32_t w = and_or_valu(lo, 0x000F000Fu << up, magic);
  if constexpr (BITS == 5) w = and_or_valu(shr<q - 4 - up>(hi), 0x00100010u << up, w);
  if constexpr (BITS == 6) w = and_or_valu(shr<2 * (q & 7) - 4 - up>(hi), 0x00300030u << up, w);
  const half2_t h = __builtin_bit_cast(half2_t, w);
  const float2_t x{__builtin_fmaf(float(h.x), sc[P & 1], off[P & 1]), __builtin_fmaf(float(h.y), sc[P & 1], off[P & 1])};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, bf16x2_t));
}

template <int BITS>
__global__ void __launch_bounds__(kBigThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) qgemm_big_kernel(GemmArgs a) {
  __shared__ BigShared sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, kg = lane >> 5;
  const int wm = wave >> 1, wn = wave & 1;
  // (readfirstlane: wave-uniform values the buffer resources are built from stay in scalar registers)
  const int tn = __builtin_amdgcn_readfirstlane(blockIdx.x % a.tiles_n);
  const int m0 = __builtin_amdgcn_readfirstlane((blockIdx.x / a.tiles_n) * kBigRows);
  const int G = a.k / 64;
  const BPlanes bp = make_bplanes<BITS>(a);
  const uint32_t magic = 0x68006800u;  // fp16 2048 in both halves
  const int valid_rows = __builtin_amdgcn_readfirstlane(a.m - m0 < kBigRows ? a.m - m0 : kBigRows);
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(const_cast<uint16_t*>(a.a) + size_t(m0) * a.k), short(0), valid_rows * a.k * int(sizeof(uint16_t)),
      0x00020000);
  // Loads past the last group repeat it and are not used. A rows by DMA: wave w copies rows 32 w ..
  // 32 w + 31, 8 rows (1 KB) an instruction; rows past M load as zero through the buffer's range.
  auto gcl = [&](int g) { return g < G - 1 ? g : G - 1; };
  const int avoff = ((32 * wave + (lane >> 3)) * a.k + 8 * ((lane & 7) ^ (lane >> 4))) * 2;
  auto dma_a = [&](int g, int buf) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      copy_to_lds(ars, &sh.s.a[buf][32 * wave + 8 * i][0], (i & 1 ? avoff ^ 64 : avoff) + 16 * i * a.k, 128 * gcl(g));
  };
  // the thread's lane word of a group (block `wave` of the tile) and its column's scale, four groups
  // ahead: group g in slot g % 4 until its dequantisation beside group g - 1's MFMAs
  TileWords<4> wq[4];
  uint32_t sq[4];
  auto load_words = [&](int slot, int g) {
    load_tile_words<BITS, 4>(wq[slot], bp, 8 * tn + wave, gcl(g), G, lane, 0);
    sq[slot] = __builtin_amdgcn_raw_buffer_load_b16(bp.sc, (lane & 31) * 2, ((8 * tn + wave) * G + gcl(g)) * 64, 0);
  };
  auto dequant = [&](auto st, int buf, const TileWords<4>& w, const float (&sc)[2], const float (&off)[2]) {
    constexpr int S = decltype(st)::value;
    const uint32_t lo = w.lo[S], lo8 = lo >> 8, hi = BITS == 6 && S >= 2 ? w.hi.y : w.hi.x;
    const u32x4 v{scaled_pair_bf16<BITS, S, 0>(lo, hi, magic, sc, off), scaled_pair_bf16<BITS, S, 1>(lo, hi, magic, sc, off),
                  scaled_pair_bf16<BITS, S, 2>(lo8, hi, magic, sc, off), scaled_pair_bf16<BITS, S, 3>(lo8, hi, magic, sc, off)};
    *reinterpret_cast<u32x4*>(&sh.s.b[buf][wave][S][lane][0]) = v;
  };
  auto factors = [&](uint32_t bits, float (&sc)[2], float (&off)[2]) {
    const float s = bf16_value(uint16_t(bits));
    sc[0] = s * 0.5f;
    sc[1] = s * (1.0f / 32);
    off[0] = s * -(1024.0f + float(1 << (BITS - 1)));
    off[1] = s * -(64.0f + float(1 << (BITS - 1)));
  };

  float16_t C[2][4];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int j = 0; j < 4; ++j) C[mb][j] = float16_t{};

  using i0 = std::integral_constant<int, 0>;
  using i1 = std::integral_constant<int, 1>;
  using i2 = std::integral_constant<int, 2>;
  using i3 = std::integral_constant<int, 3>;
  dma_a(0, 0);
  dma_a(1, 1);
  load_words(0, 0);
  load_words(1, 1);
  load_words(2, 2);
  load_words(3, 3);
  const float my_rs = threadIdx.x < kBigRows ? row_scale(a, m0 + threadIdx.x) : 0.0f;  // (with the first loads in flight)
  {
    float sc[2], off[2];
    factors(sq[0], sc, off);
    dequant(i0{}, 0, wq[0], sc, off);
    dequant(i1{}, 0, wq[0], sc, off);
    dequant(i2{}, 0, wq[0], sc, off);
    dequant(i3{}, 0, wq[0], sc, off);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the DMA copies of groups 0 and 1 have landed
  __syncthreads();

  // One half of a group (steps 2 H and 2 H + 1): a memory and a compute phase with a barrier after each,
  // waves 4-7 one phase behind waves 0-3. A half's operands are complete when waves 0-3 read them (the
  // codes' same half of the group before was dequantised at least one phase earlier by either set of
  // waves), and the buffers are free when they are written: half H of group g + 1 goes where group
  // g - 1's half H was, the copies of group g + 2 (in the second half of group g) where group g - 1's rows
  // were; waves 4-7 read either two phases before at the latest, and used it in the one between. (In the
  // first half the copies would meet their last reads: 1,201 us with a wait for those, in-projection of
  // 2,048 rows over four layers, 1,194 so.) cur = g % 4 is a compile-time constant,
  // so the register ring is indexed statically.
  int abuf = 0;  // g mod 3
  auto phase_end = [&]() {  // (as in qgemm_tile_kernel)
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr int kCopies = 4, kLoads = (BITS == 4 ? 1 : 2) + 1;  // of a group: A copies; words and scale
  auto half = [&](int g, auto curc, auto hc, auto tailc) {  // TAIL: as in qgemm_tile_kernel
    constexpr int cur = decltype(curc)::value, H = decltype(hc)::value;
    constexpr bool TAIL = decltype(tailc)::value;
    bf16x8_t ao[2][2], bo[2][4];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const int r = 64 * wm + 32 * mb + (lane & 31);
        ao[s][mb] = __builtin_bit_cast(bf16x8_t, sh.s.a[abuf][r][(2 * (2 * H + s) + kg) ^ ((r >> 1) & 7)]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        bo[s][j] = *reinterpret_cast<const bf16x8_t*>(&sh.s.b[cur & 1][4 * wn + j][2 * H + s][lane][0]);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (H == 1) {
      dma_a(g + 2, abuf == 0 ? 2 : abuf - 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!TAIL) load_words(cur, g + 4);
      // the copies of group g + 1 have landed: after them went out one group's loads, the copies of
      // group g + 2 and another group's loads; in the tail only the newest copies are sure to have
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(vm_in_flight(TAIL ? kCopies : kLoads + kCopies + kLoads));
    }
    phase_end();
    __builtin_amdgcn_s_setprio(1);
    float sc[2], off[2];
    factors(sq[(cur + 1) & 3], sc, off);
    dequant(std::integral_constant<int, 2 * H>{}, (cur & 1) ^ 1, wq[(cur + 1) & 3], sc, off);
    dequant(std::integral_constant<int, 2 * H + 1>{}, (cur & 1) ^ 1, wq[(cur + 1) & 3], sc, off);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
          C[mb][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ao[s][mb], bo[s][j], C[mb][j], 0, 0, 0);
    if constexpr (H == 1) abuf = abuf == 2 ? 0 : abuf + 1;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA,
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);  // then vector instructions
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // this wave's dequantised codes are in LDS
    phase_end();
  };
  if (wave >= 4) phase_end();
  auto group = [&](int g, auto curc, auto tailc) {
    half(g, curc, i0{}, tailc);
    half(g, curc, i1{}, tailc);
  };
  int g = 0;
  for (; g + 3 < G; g += 4) {
    group(g, i0{}, std::false_type{});
    group(g + 1, i1{}, std::false_type{});
    group(g + 2, i2{}, std::false_type{});
    group(g + 3, i3{}, std::false_type{});
  }
  if (g < G) group(g, i0{}, std::true_type{});
  if (g + 1 < G) group(g + 1, i1{}, std::true_type{});
  if (g + 2 < G) group(g + 2, i2{}, std::true_type{});
  if (wave < 4) phase_end();
  // the copies past the last group have landed and every wave is past its last operand read
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x < kBigRows) sh.e.rs[threadIdx.x] = my_rs;
  __syncthreads();

  // ---- epilogue: blocks of 32 rows x 64 columns
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int jh = 0; jh < 2; ++jh) {
      const int r0 = 64 * wm + 32 * mb;
      block_to_rows(sh.e.out[wave], C[mb][2 * jh], C[mb][2 * jh + 1], lane);
      store_block(a, sh.e.out[wave], m0 + r0, tn * kTileN + 128 * wn + 64 * jh, sh.e.rs + r0, sh.e.ss[2 * wn + jh] + r0,
                  lane);
    }
  if (a.kind == Q38A_EPI_RESIDUAL) {
    __syncthreads();
    const int r = threadIdx.x & (kBigRows - 1), h = threadIdx.x / kBigRows;
    if (m0 + r < a.m)
      a.partials_out[size_t(m0 + r) * a.norm_blocks + 2 * tn + h] = sh.e.ss[2 * h][r] + sh.e.ss[2 * h + 1][r];
  }
}

// ---- the o-projection of up to 32 rows with the merge in its A staging: 32 x 256 tiles, sixteen waves
// A decode step's rows are few, so the launch is a stream of weights: per CU as many weight bytes
// in flight as registers allow. The workgroup's A slice (its rows x the slice's k) and the rows'
// group sums S_g are staged in LDS once; waves keep only weight words in their register pipeline
// (kGemvDepth groups deep). Two sets of eight waves (K parts) each cover half the slice's groups
// for all 256 columns and add their sums through LDS. EV: row quads of the MFMA output that can hold
// rows < M (1 for M <= 8: the epilogue arithmetic of the other 12 elements is skipped).
constexpr int kGemvDepth = 6;
constexpr int kSliceG = 20;                 // most 64-k groups in a workgroup's slice (LDS budget)
constexpr int kSliceStride = 64 * kSliceG + 8;  // bf16 per staged A row (+16 B against bank conflicts)

constexpr int kMaxNormBlocks = 64;  // folded-norm partials per row (hidden <= 8192)
constexpr int kStagePartials = (32 * kMaxNormBlocks + 1023) / 1024;  // partials per thread

struct alignas(16) GemvShared {
  uint16_t a[32][kSliceStride];  // the tile's A rows over the slice (rows >= M: stale)
  float s[kSliceG][32];          // S_g per row
  float p[32 * kMaxNormBlocks];  // the rows' folded-norm partials
};

// The staged A is the gated merge of decode split partials (MergeIn).
template <int BITS, int EV>
__global__ void __launch_bounds__(kGemvThreads) __attribute__((amdgpu_waves_per_eu(4)))
qgemv_kernel(GemmArgs a, BatchArgs batch, MergeIn mi) {
  __shared__ GemmShared sh;
  __shared__ GemvShared sv;
  const int hw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, wave = hw % kColWaves, kp = hw / kColWaves;
  const int kg = lane >> 5;
  const int z = blockIdx.x % a.splits, tn = blockIdx.x / a.splits;
  const int G = a.k / 64;
  const int gs0 = int((long long)z * G / a.splits), gs1 = int((long long)(z + 1) * G / a.splits);
  const int gm = gs0 + (gs1 - gs0) / kKParts;  // K part 0: [gs0, gm), part 1: [gm, gs1)
  const int g0 = kp == 0 ? gs0 : gm, g1 = kp == 0 ? gm : gs1;
  const int nb = tn * (kTileN / 32) + wave;  // this wave's 32-column block
  const int valid_rows = a.m;  // <= 32
  const BPlanes bp = make_bplanes<BITS>(a);

  // B pipeline first, then the staging loads, so one round trip covers them all; loads past the
  // part's end re-read its last group (unconditional loads keep the loop's waits exact)
  BWords B[kGemvDepth];
  const int glast = g1 - 1;
  auto gc = [&](int g) { return g < glast ? g : glast; };
#pragma unroll
  for (int d = 0; d + 1 < kGemvDepth; ++d) {
    load_bwords<BITS>(B[d], bp, nb, gc(g0 + d), G, lane);
    __builtin_amdgcn_sched_barrier(0);  // issue order per group, as in the loop (exact waits there)
  }
  // stage the A rows < M over the slice (16-byte chunks; LDS rows >= M keep whatever they hold: an
  // MFMA output row depends on its A row only, and rows >= M are never stored) and the partials
  // of the folded norm
  {
    {  // four dims of one (row, q head) per step; a row that is not a decode row (n != 1) is zero
      const DecodePlan pl = wave_decode_plan<true>(batch, mi.nkv, mi.max_splits, mi.target_items);
      const int qpr = 16 * (gs1 - gs0);  // quads per row
      for (int c = threadIdx.x; c < valid_rows * qpr; c += kGemvThreads) {
        const int r = c / qpr, kq = c % qpr, k = 64 * gs0 + 4 * kq;
        const int h = k / kHeadDim, d = k % kHeadDim, row = r;
        const int b = batch.tok_seq[row];
        const int L = decode_len(batch, b);
        uint16_t y[4] = {0, 0, 0, 0};
        if (L > 0)
          merge_quad(mi.scratch + (size_t(b) * mi.nq + h) * mi.max_splits * (kHeadDim + 2),
                     ceil_div_i(ceil_div_i(L, kPageTokens), pl.cp), kHeadDim + 2, d,
                     mi.gate + size_t(row) * mi.ld_gate + h * kHeadDim + d, y);
        *reinterpret_cast<uint2*>(&sv.a[r][4 * kq]) =
            uint2{uint32_t(y[0]) | (uint32_t(y[1]) << 16), uint32_t(y[2]) | (uint32_t(y[3]) << 16)};
      }
    }
    float pv[kStagePartials];
    const int np = valid_rows * a.norm_blocks;
#pragma unroll
    for (int i = 0; i < kStagePartials; ++i) {
      const int c = int(threadIdx.x) + i * kGemvThreads;
      if (a.partials_in && c < np) pv[i] = a.partials_in[c];
    }
#pragma unroll
    for (int i = 0; i < kStagePartials; ++i) {
      const int c = int(threadIdx.x) + i * kGemvThreads;
      if (a.partials_in && c < np) sv.p[c] = pv[i];
    }
    __syncthreads();
    // row scales (in block order, as row_scale) and group sums S_g (rows >= M: unused)
    if (threadIdx.x < 32) {
      float rs = 1.0f;
      if (a.partials_in && int(threadIdx.x) < valid_rows) {
        float acc = 0.0f;
        for (int b = 0; b < a.norm_blocks; ++b) acc += sv.p[threadIdx.x * a.norm_blocks + b];
        rs = 1.0f / __builtin_sqrtf(acc * a.inv_hidden + a.eps);
      }
      sh.rs[threadIdx.x] = rs;
    }
    const int ng = gs1 - gs0;
    for (int t = threadIdx.x; t < 32 * ng; t += kGemvThreads) {
      const int gl = t >> 5, r = t & 31;
      float acc = 0.0f;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const u32x4 w = *reinterpret_cast<const u32x4*>(&sv.a[r][64 * gl + 8 * c]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          acc += __builtin_bit_cast(float, w[i] << 16);
          acc += __builtin_bit_cast(float, w[i] & 0xFFFF0000u);
        }
      }
      sv.s[gl][r] = acc;
    }
    __syncthreads();
  }

  float16_t C = float16_t{};
  const float c0 = 128.0f + float(1 << (BITS - 1));
  const uint32_t magic = 0x43004300u;
  const int arow = lane & 31;
  for (int g = g0; g < g1; g += kGemvDepth) {
#pragma unroll
    for (int d = 0; d < kGemvDepth; ++d) {
      load_bwords<BITS>(B[(d + kGemvDepth - 1) % kGemvDepth], bp, nb, gc(g + d + kGemvDepth - 1), G, lane);
      __builtin_amdgcn_sched_barrier(0);
      const int gl = gc(g + d) - gs0;
      u32x4 Ab[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) Ab[s] = *reinterpret_cast<const u32x4*>(&sv.a[arow][64 * gl + 16 * s + 8 * kg]);
      const float16_t T = group_products<BITS>(Ab, B[d], magic);
      const float sc = g + d < g1 ? bf16_value(uint16_t(B[d].scale)) : 0.0f;
#pragma unroll
      for (int i = 0; i < EV; ++i) {
        const float4 sq = *reinterpret_cast<const float4*>(&sv.s[gl][8 * i + 4 * kg]);
        const float sr[4] = {sq.x, sq.y, sq.z, sq.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          C[4 * i + r] = __builtin_fmaf(sc, __builtin_fmaf(-c0, sr[r], T[4 * i + r]), C[4 * i + r]);
      }
    }
  }

  // part 1 hands its sums to part 0 and ends (barriers count only the waves still running)
  if (kp == 1) {
#pragma unroll
    for (int e = 0; e < 4 * EV; ++e) sh.kpart[wave][e][lane] = C[e];
  }
  __syncthreads();
  if (kp == 1) return;
#pragma unroll
  for (int e = 0; e < 4 * EV; ++e) C[e] += sh.kpart[wave][e][lane];
  __syncthreads();  // the union's other uses may overwrite kpart from here on
  tile_finish<EV>(a, sh, C, tn, z, wave, lane);
}

// ---- decode-size M (<= 8 rows) on a wide column grid: 64-column tiles over the whole K --------------
// One 8-wave workgroup per 64-column tile (the in-projection: 224 tiles for 256 CUs). The tile's K
// groups are cut into fixed chunks (two or three groups, both 32-column blocks); the waves take
// chunks from a counter in LDS as they finish, so a wave that the memory system serves late takes
// fewer (with a fixed share of K per wave, the workgroup waited ~4 us for its slowest wave after the
// mean wave was done). Each chunk's sums go to its own LDS slot and the slots are added in chunk
// order: the result does not depend on which wave took which chunk. A wave keeps its next group in
// flight across chunk boundaries (it claims the next chunk when it issues that chunk's first
// loads). A group's A rows come in one 16-byte load per lane (8 rows x 64 k, rows >= M load as
// zero) and pass through the wave's LDS buffer into the MFMA operand layout (loaded straight into
// that layout, 48 of a load's 64 lanes held rows >= 8, four loads per group). Weights are loaded
// non-temporal (read once). Only the 4 MFMA output elements per lane that can hold rows < 8 take
// the per-group epilogue arithmetic. StoreBF16 / StoreF32 only (the residual epilogue's 128-column
// sums of squares would span two tiles).
//
// Measured on the in-projection at M = 8 (HIP events, weights rotating through 8 copies): 17.1 us
// with a fixed share of K per wave and A loaded into the operand layout; 16.1 with the chunk
// claims; 15.0 with the compact A loads and non-temporal weights; 14.7 with 8 waves instead of 16.
// More groups in flight per wave (3 or 4), or 4 waves with 4 in flight, were slower (16-19 us), as
// was staging all of A in LDS once per workgroup (17.4 us).
constexpr int kWideWaves = 8;
constexpr int kWideRows = 8;
constexpr int kWideSlotFloats = 40 * 2 * 4 * 64;  // the chunks' sums in LDS (80 KB)
constexpr int kWideMaxSplits = 8;

// Chunks of a workgroup's Gs groups for tiles of nb 32-column blocks: at most as many as fill the
// LDS slots (40 of two blocks, 20 of four), at least one group each.
__host__ __device__ constexpr int wide_chunks(int nb, int gs) {
  return gs < kWideSlotFloats / (nb * 256) ? gs : kWideSlotFloats / (nb * 256);
}

struct alignas(16) WideShared {
  u32x4 a[kWideWaves][2][8][8];  // per wave and buffer: the group's A rows, [k chunk][row]
  float c[kWideSlotFloats];      // per chunk: [block][element (rows 4 kg + e)][lane]
  float rs[kWideRows];
  float ss[kWideWaves][2];       // residual epilogue: per wave, its two rows' sums of squares
  int next;                      // the next unclaimed chunk
  int last;                      // split-K: this workgroup arrived last
};

// NB: 32-column blocks per tile (2: StoreBF16 / StoreF32; 4: the residual epilogue, whose tile is
// one 128-column block of the sums of squares). gridDim.y: K splits; with more than one, every
// split writes its tile sums (write-through, as in the split-K kernel) and the last to arrive adds
// them in split order and runs the epilogue.
template <int BITS, int NB, bool RES>
__global__ void __launch_bounds__(64 * kWideWaves) qgemv_wide_kernel(GemmArgs a) {
  static_assert(!RES || NB == 4, "the residual epilogue needs 128-column tiles");
  constexpr int kOut = NB * 4 * 64 / (64 * kWideWaves);  // output values per thread
  __shared__ WideShared sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, kg = lane >> 5;
  const int tn = blockIdx.x, ks = blockIdx.y, KS = gridDim.y;
  const int G = a.k / 64;
  const int gb = ks * G / KS, Gs = (ks + 1) * G / KS - gb;
  const int NC = wide_chunks(NB, Gs);
  const int nb0 = tn * NB;
  // the counter's first value before any wave claims, and the row scales before any weight load (a
  // branch over outstanding loads would make the waits conservative)
  if (threadIdx.x == 0) sh.next = kWideWaves;
  __syncthreads();
  if (!RES && threadIdx.x < kWideRows) sh.rs[threadIdx.x] = row_scale(a, threadIdx.x);
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(const_cast<uint16_t*>(a.a)), short(0), a.m * a.k * int(sizeof(uint16_t)), 0x00020000);
  const BPlanes bp = make_bplanes<BITS>(a);
  // compact A loads: lane = 8 chunk + row (every lane useful; rows >= M load as zero)
  const int aoff = ((lane & 7) * a.k + 8 * (lane >> 3)) * int(sizeof(uint16_t));
  const float c0 = 128.0f + float(1 << (BITS - 1));
  const uint32_t magic = 0x43004300u;
  bf16x8_t ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = __bf16(1.0f);
  float C[NB][4];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) C[j][e] = 0.0f;
  auto chunk_begin = [&](int c) { return gb + c * Gs / NC; };
  // load cursor (wave-uniform): chunk lc (>= NC once the chunks are gone), group lg of it
  int lc = wave, lg = chunk_begin(wave), lend = chunk_begin(wave + 1);
  // two register buffers rotate over the groups
  constexpr int kDepth = 2;
  u32x4 A[kDepth];
  BWords B[kDepth][NB];
  int rc[kDepth], rg[kDepth];  // chunk and group in each buffer (wave-uniform)
  auto load_next = [&](int d) {
    if (lc < NC && lg == lend) {
      int c = 0;
      if (lane == 0) c = atomicAdd(&sh.next, 1);
      lc = __builtin_amdgcn_readfirstlane(c);
      if (lc < NC) { lg = chunk_begin(lc); lend = chunk_begin(lc + 1); }
    }
    const int g = lc < NC ? lg : gb;  // past the last chunk: a valid address, never used
    rc[d] = lc;
    rg[d] = lg;
    A[d] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ars, aoff, 128 * g, 0));
#pragma unroll
    for (int j = 0; j < NB; ++j) load_bwords<BITS, kNonTemporal>(B[d][j], bp, nb0 + j, g, G, lane);
    __builtin_amdgcn_sched_barrier(0);
    ++lg;
  };
  auto compute = [&](int d) {
    // through the wave's LDS buffer into the operand layout: row lane % 32 (rows >= 8 repeat rows
    // 0-7; their output rows are never read), k chunk 2 s + lane / 32
    sh.a[wave][d][lane >> 3][lane & 7] = A[d];
    u32x4 Ab[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) Ab[s] = sh.a[wave][d][2 * s + kg][lane & 7];
    // S (the rows' sums over the group) from two 16 x 16 x 32 MFMAs against ones: MFMA row r is
    // A row 4 (r / 8) + r % 4, so that output element e of lane l is row 4 (l / 32) + e, the row of
    // C element e (rows >= 8 of the 32 x 32 output are never read)
    float4_t S = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int h = 0; h < 2; ++h)
      S = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8_t, sh.a[wave][d][4 * h + (lane >> 4)][4 * ((lane >> 3) & 1) + (lane & 3)]), ones, S,
          0, 0, 0);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const float16_t T = group_products<BITS>(Ab, B[d][j], magic);
      const float sc = bf16_value(uint16_t(B[d][j].scale));
#pragma unroll
      for (int e = 0; e < 4; ++e) C[j][e] = __builtin_fmaf(sc, __builtin_fmaf(-c0, S[e], T[e]), C[j][e]);
    }
    if (rg[d] + 1 == chunk_begin(rc[d] + 1)) {  // the chunk's last group: its sums to its slot
      float* slot = sh.c + rc[d] * (NB * 256);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          slot[(4 * j + e) * 64 + lane] = C[j][e];
          C[j][e] = 0.0f;
        }
    }
  };
  load_next(0);
  for (;;) {
    load_next(1);
    if (rc[0] >= NC) break;
    compute(0);
    load_next(0);
    if (rc[1] >= NC) break;
    compute(1);
  }
  __syncthreads();
  // output value i of this thread: index x = t + 512 i = (block j, element e, lane l); the chunks'
  // sums in chunk order
  const int t = threadIdx.x;
  float v[kOut];
#pragma unroll
  for (int i = 0; i < kOut; ++i) {
    float x = 0.0f;
    for (int c = 0; c < NC; ++c) x += sh.c[c * (NB * 256) + t + 64 * kWideWaves * i];
    v[i] = x;
  }
  if (KS > 1) {
    // the tile's K splits: write-through partials, an arrival count, the last arrival sums them in
    // split order with agent-coherent loads (the hand-off of the split-K kernel, tile_finish)
    float* part = a.ws_partials + size_t(tn) * KS * (NB * 256);
#pragma unroll
    for (int i = 0; i < kOut; ++i)
      __hip_atomic_store(part + ks * (NB * 256) + t + 64 * kWideWaves * i, v[i], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // the write-through stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
      const int old = __hip_atomic_fetch_add(a.counters + tn, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.last = old == KS - 1;
      if (sh.last) __hip_atomic_store(a.counters + tn, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!sh.last) return;
    const __amdgpu_buffer_rsrc_t prs =
        __builtin_amdgcn_make_buffer_rsrc(part, short(0), KS * (NB * 256) * int(sizeof(float)), 0x00020000);
    constexpr int kSc1 = 16;  // cache policy bit sc1
    float V[kWideMaxSplits][kOut];
#pragma unroll
    for (int z = 0; z < kWideMaxSplits; ++z)
#pragma unroll
      for (int i = 0; i < kOut; ++i) {
        const int zz = z < KS ? z : KS - 1;  // past the last split: re-read it, not added
        V[z][i] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(prs, (t + 64 * kWideWaves * i) * 4, zz * NB * 1024, kSc1));
      }
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
      float x = 0.0f;
#pragma unroll
      for (int z = 0; z < kWideMaxSplits; ++z) x = z < KS ? x + V[z][i] : x;
      v[i] = x;
    }
  }
  if constexpr (RES) {
    // residual += C; xbf = bf16(residual); the tile's 128 columns' sums of squares per row: this
    // thread's values (blocks j and j + 2 of row 4 (l / 32) + e), then the 32 lanes of each half
    // wave, then the two waves of each row in wave order
    const int e = (t >> 6) & 3, l = t & 63, row = 4 * (l >> 5) + e;
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
      const int j = (t + 64 * kWideWaves * i) >> 8;
      const int col = tn * (32 * NB) + 32 * j + (l & 31);
      if (row < a.m) {
        float* res = a.residual + size_t(row) * a.n + col;
        const float x = *res + v[i];
        *res = x;
        a.xbf[size_t(row) * a.n + col] = bf16_bits(x);
        ss += x * x;
      }
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
    if ((lane & 31) == 0) sh.ss[wave][lane >> 5] = ss;
    __syncthreads();
    if (threadIdx.x < kWideRows) {
      // row r = 4 h + e: waves e and e + 4 (blocks 0-1 and 2-3 of element e), half h
      const int r = threadIdx.x, ee = r & 3, h = r >> 2;
      if (r < a.m) a.partials_out[size_t(r) * a.norm_blocks + tn] = sh.ss[ee][h] + sh.ss[ee + 4][h];
    }
  } else {
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
      const int x = t + 64 * kWideWaves * i, j = x >> 8, e = (x >> 6) & 3, l = x & 63;
      const int row = 4 * (l >> 5) + e, col = tn * (32 * NB) + 32 * j + (l & 31);
      if (row >= a.m || col >= a.n_store) continue;
      const float y = v[i] * sh.rs[row];
      if (a.kind == Q38A_EPI_STORE_F32) static_cast<float*>(a.out)[size_t(row) * a.ldo + col] = y;
      else static_cast<uint16_t*>(a.out)[size_t(row) * a.ldo + col] = bf16_bits(y);
    }
  }
}

// ---- 9 to 64 rows: the columns' weights straight into the MFMA operands ---------------------------
// Eight waves of (32 RB rows) x 64 columns over shares of K: CW column waves x 8 / CW K parts. A wave
// streams its weights from HBM into registers (every weight is dequantised once, by the wave whose
// columns it is, so they are not staged) and copies its A rows, which all workgroups share, from the
// L2 into an LDS buffer of its own, both one group ahead. (A rows loaded straight into the operand
// layout touched four times the cache lines: 24 instead of 20.7 us at 32 rows, 34 at 64.) Codes as bf16
// 128 + u; the group's products start from -(128 + 2^(b-1)) times the rows' sums (four more MFMAs of A
// against a constant, shared by the two column blocks), so T is A . codes and a group costs one fma per
// output. The K parts' sums meet in LDS in part order; with a K split over
// workgroups (CW = 2) the last to arrive adds the slices in slice order.
//
// Bound: the weight stream and, around it, one round trip of first loads and the sums' way through
// LDS. In-projection: 9 rows 24.3 -> 16.8 us with the append, 64 rows 36 -> 26.8; o-projection:
// 16 rows 21.9 -> 14.1, 64 rows 33 -> 22.3.
constexpr int kSmallWaves = 8;
constexpr int kSmallThreads = 64 * kSmallWaves;
constexpr int kSmallMaxRows = 64;
constexpr int kSmallMaxSplits = 8;

template <int RB>
struct alignas(16) SmallShared {
  union {
    u32x4 a[kSmallWaves][2][32 * RB][8];       // per wave: two groups' A rows, [row][slot] as in TileShared
    float part[kSmallWaves][RB * 2 * 16][64];  // the waves' sums: [row block, column block, element][lane]
    OutBlock out[2 * RB];                      // [column wave][row block]
  };
  float rs[32 * RB];     // row scales of the folded RMSNorm
  float ss[2][32 * RB];  // residual epilogue: each column wave's sums of squares
  int last;
};

// DMA: A by copies into LDS, which need rows of 16-byte alignment; otherwise through registers, with
// loads of any alignment.
template <int BITS, int RB, int CW, bool DMA>
__global__ void __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(2))) qgemm_small_kernel(GemmArgs a) {
  constexpr int KW = kSmallWaves / CW, kCols = 64 * CW;
  constexpr int kVals = CW * RB * 2 * 16 * 64 / kSmallThreads;  // outputs per thread
  __shared__ SmallShared<RB> sh;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, kg = lane >> 5;
  const int cw = wave % CW, kw = wave / CW;
  const int tn = blockIdx.x, z = blockIdx.y, Z = gridDim.y;
  const int G = a.k / 64;
  const int gb = z * G / Z, ge = (z + 1) * G / Z;
  const int g0 = gb + kw * (ge - gb) / KW, g1 = gb + (kw + 1) * (ge - gb) / KW;
  const int nb0 = tn * (kCols / 32) + 2 * cw;
  const BPlanes bp = make_bplanes<BITS>(a);
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      uniform_ptr(const_cast<uint16_t*>(a.a)), short(0), a.m * a.k * int(sizeof(uint16_t)), 0x00020000);
  // A rows of a group by DMA into the wave's own LDS buffer, 8 rows (1 KB) an instruction; rows past M
  // fall outside the buffer's range and load as zero
  const int avoff = ((lane >> 3) * a.k + 8 * ((lane & 7) ^ (lane >> 4))) * 2;
  const uint32_t magic = 0x43004300u;  // bf16 128 in both halves
  bf16x8_t neg;                        // -(128 + 2^(b-1)), exact in bf16
#pragma unroll
  for (int i = 0; i < 8; ++i) neg[i] = __bf16(-(128.0f + float(1 << (BITS - 1))));

  float16_t C[RB][2];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) C[rb][0] = C[rb][1] = float16_t{};
  BWords B[2][2];
  u32x4 R[2][DMA ? 1 : 4 * RB];  // without DMA: the groups' A rows on their way to LDS
  // unconditional loads (past the share's end they repeat its last group, cached and unused): a load
  // under a branch would make the loop's waits conservative
  auto load_group = [&](int d, int g) {
    const int gc = g < g1 - 1 ? g : (g1 > g0 ? g1 - 1 : gb);
    __builtin_amdgcn_sched_barrier(0);  // (the buffer's operand reads have returned: their MFMAs are issued)
#pragma unroll
    for (int i = 0; i < 4 * RB; ++i) {
      const int off = (i & 1 ? avoff ^ 64 : avoff) + 16 * i * a.k;
      if constexpr (DMA) {
        copy_to_lds(ars, &sh.a[wave][d][8 * i][0], off, 128 * gc);
      } else {
        // (rows past M load row 0: an output row depends on its own row only)
        const int at = 8 * i + (lane >> 3) < a.m ? off : avoff - (lane >> 3) * a.k * 2;
        __builtin_memcpy(&R[d][i], reinterpret_cast<const char*>(a.a) + at + 128 * gc, 16);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 2; ++j) load_bwords<BITS, kNonTemporal>(B[d][j], bp, nb0 + j, gc, G, lane);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto compute = [&](int d) {
    // this group's copies have landed: at most the next group's loads are in flight
    constexpr int kNext = 4 * RB + 2 * (BITS == 4 ? 2 : 3);
    if constexpr (DMA) {
      __builtin_amdgcn_s_waitcnt(vm_in_flight(kNext));
    } else {
#pragma unroll
      for (int i = 0; i < 4 * RB; ++i) sh.a[wave][d][8 * i + (lane >> 3)][lane & 7] = R[d][i];
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    u32x4 A[RB][4];
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int r = 32 * rb + (lane & 31);
        A[rb][s] = sh.a[wave][d][r][(2 * s + kg) ^ ((r >> 1) & 7)];
      }
    float16_t N[RB];  // the products' start
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        N[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, A[rb][s]), neg,
                                                        s == 0 ? float16_t{} : N[rb], 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float16_t T[RB];
      auto t_step = [&](auto st) {
        constexpr int s = decltype(st)::value;
        const bf16x8_t bo = b_operand<BITS, s>(B[d][j], magic);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
          T[rb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, A[rb][s]), bo,
                                                          s == 0 ? N[rb] : T[rb], 0, 0, 0);
      };
      t_step(std::integral_constant<int, 0>{});
      t_step(std::integral_constant<int, 1>{});
      t_step(std::integral_constant<int, 2>{});
      t_step(std::integral_constant<int, 3>{});
      const float sc = bf16_value(uint16_t(B[d][j].scale));
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int e = 0; e < 16; ++e) C[rb][j][e] = __builtin_fmaf(sc, T[rb][e], C[rb][j][e]);
    }
  };
  load_group(0, g0);
  if (int(threadIdx.x) < 32 * RB) sh.rs[threadIdx.x] = row_scale(a, threadIdx.x);  // (with the first loads in flight)
  int g = g0;
  for (; g + 1 < g1; g += 2) {
    load_group(1, g + 1);
    compute(0);
    load_group(0, g + 2);
    compute(1);
  }
  if (g < g1) {
    load_group(1, g + 1);  // (the wait in compute counts a following group's loads)
    compute(0);
  }
  __builtin_amdgcn_s_waitcnt(0);  // no copy in flight: LDS takes the sums
  __syncthreads();

  // ---- the K parts' sums in part order: value x = t + 512 i is (column wave, row block, column block,
  // element, lane)
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) sh.part[kw * CW + cw][(2 * rb + j) * 16 + e][lane] = C[rb][j][e];
  __syncthreads();
  float v[kVals];
#pragma unroll
  for (int i = 0; i < kVals; ++i) {
    const int x = int(threadIdx.x) + kSmallThreads * i, w = x / (RB * 2 * 16 * 64), r = x % (RB * 2 * 16 * 64);
    float y = 0.0f;
#pragma unroll
    for (int q = 0; q < KW; ++q) y += (&sh.part[q * CW + w][0][0])[r];
    v[i] = y;
  }
  if (Z > 1) {
    // the tile's slices (the hand-off of tile_finish)
    constexpr int kSc1 = 16, kSlice = kVals * kSmallThreads;  // floats
    float* part = uniform_ptr(a.ws_partials + size_t(tn) * Z * kSlice);
#pragma unroll
    for (int i = 0; i < kVals; ++i)
      __hip_atomic_store(part + z * kSlice + threadIdx.x + kSmallThreads * i, v[i], __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_s_waitcnt(0);  // the write-through stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
      const int old = __hip_atomic_fetch_add(a.counters + tn, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sh.last = old == Z - 1;
      if (sh.last) __hip_atomic_store(a.counters + tn, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!sh.last) return;
    const __amdgpu_buffer_rsrc_t prs =
        __builtin_amdgcn_make_buffer_rsrc(part, short(0), Z * kSlice * int(sizeof(float)), 0x00020000);
    float V[kSmallMaxSplits][kVals];
#pragma unroll
    for (int q = 0; q < kSmallMaxSplits; ++q)
#pragma unroll
      for (int i = 0; i < kVals; ++i) {
        const int zz = q < Z ? q : Z - 1;  // past the last slice: re-read it, not added
        V[q][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                prs, (int(threadIdx.x) + kSmallThreads * i) * 4, zz * kSlice * 4, kSc1));
      }
#pragma unroll
    for (int i = 0; i < kVals; ++i) {
      float y = 0.0f;
#pragma unroll
      for (int q = 0; q < kSmallMaxSplits; ++q) y = q < Z ? y + V[q][i] : y;
      v[i] = y;
    }
  }
  __syncthreads();  // the sums' slots have been read
#pragma unroll
  for (int i = 0; i < kVals; ++i) {
    const int x = int(threadIdx.x) + kSmallThreads * i, l = x & 63, e = (x >> 6) & 15, j = (x >> 10) & 1;
    const int rb = (x >> 11) % RB, w = x / (RB * 2048);
    sh.out[w * RB + rb][8 * (e >> 2) + 4 * (l >> 5) + (e & 3)][32 * j + (l & 31)] = v[i];
  }
  __syncthreads();
  if (wave < CW * RB) {
    const int w = wave / RB, rb = wave % RB;
    store_block(a, sh.out[wave], 32 * rb, tn * kCols + 64 * w, sh.rs + 32 * rb, sh.ss[w] + 32 * rb, lane);
  }
  if (CW == 2 && a.kind == Q38A_EPI_RESIDUAL) {
    __syncthreads();
    const int r = threadIdx.x;
    if (r < 32 * RB && r < a.m) a.partials_out[size_t(r) * a.norm_blocks + tn] = sh.ss[0][r] + sh.ss[1][r];
  }
}

// Column waves, tiles and K slices of the 9- to 64-row kernel. 64-column tiles over the whole K where they
// fill three quarters of the CUs and the epilogue allows it (the sums of squares of the residual one
// need 128 columns), otherwise 128-column tiles with K split to fill the CUs, at least a group per wave.
struct SmallPlan {
  int cw, tiles, splits;
  size_t partial_floats(int m) const {
    return splits > 1 ? size_t(tiles) * splits * (m > 32 ? 64 : 32) * 64 * cw : 0;
  }
};

SmallPlan plan_small(int m, int n, int k, int kind, int cus) {
  if (kind != Q38A_EPI_RESIDUAL && n / 64 >= (3 * cus) / 4) return SmallPlan{1, n / 64, 1};
  SmallPlan p{2, n / 128, 1};
  const int G = k / 64;
  int s = cus / p.tiles;
  if (s > kSmallMaxSplits) s = kSmallMaxSplits;
  if (s > G / 4) s = G / 4;
  p.splits = s < 1 ? 1 : s;
  return p;
}

// The wide-tile plan of a GEMM, or tiles = 0 when the shape does not take it: decode-size M, a
// store epilogue on a weight wide enough to fill the CUs with 64-column tiles (no split-K), or the
// residual epilogue on 128-column tiles with K split to fill the CUs.
struct WidePlan {
  int nb, tiles, splits;
};

WidePlan plan_wide(int m, int n, int k, int kind, int cus) {
  WidePlan p{0, 0, 1};
  const int G = k / 64;
  if (m > kWideRows) return p;
  if (kind != Q38A_EPI_RESIDUAL) {
    if (n / 64 >= (3 * cus) / 4 && wide_chunks(2, G) >= kWideWaves) p = WidePlan{2, n / 64, 1};
  } else if (n % 128 == 0) {
    const int tiles = n / 128;
    int s = cus / tiles;
    if (s > kWideMaxSplits) s = kWideMaxSplits;
    while (s > 1 && wide_chunks(4, G / s) < kWideWaves) --s;
    if (s >= 1 && tiles * s >= cus / 2 && wide_chunks(4, G / s) >= kWideWaves) p = WidePlan{4, tiles, s};
  }
  return p;
}

// Split-K plan of the merging kernel (m <= 32, one 1024-thread workgroup per CU): slices of at most
// kSliceG groups (the staged A), and at most as many as fill the CUs once without a second round;
// each of the two K parts keeps a group. tiles_n = 0: the shape does not take that kernel.
struct GemvPlan {
  int tiles_n, splits;
};

GemvPlan plan_gemv(int m, int n, int k, int cus) {
  GemvPlan p{0, 1};
  const int G = k / 64;
  if (m > 32 || G < 2) return p;
  p.tiles_n = n / kTileN;
  // fill the CUs, but keep about 12 groups per slice at least: a slice's fixed costs (staging, the
  // split-K tail) cost more than idle CUs below that (measured on the o-projection: 8 slices of 12
  // groups 17.6 us, 12 slices of 8 groups 19.0 us)
  const int s_min = (G + kSliceG - 1) / kSliceG, s_fill = cus / p.tiles_n, s_work = G / 12;
  int s = s_fill < s_work ? s_fill : s_work;
  if (s < s_min) s = s_min;
  if (s > G / kKParts) s = G / kKParts;
  if (s < s_min) s = s_min;  // (G / 2 >= ceil(G / 20) for every G >= 2)
  p.splits = s;
  return p;
}

// Tile height and K slices of the tile kernel (one workgroup per CU).
struct TilePlan {
  int wm, tiles_m, tiles_n, splits;
  size_t tiles() const { return size_t(tiles_m) * tiles_n; }
  size_t partial_floats() const { return splits > 1 ? tiles() * splits * tile_rows(wm) * kTileCols : 0; }
  size_t counters() const { return splits > 1 ? tiles() : 0; }
  bool fits(const q38a_gemm_workspace& ws) const {
    return splits == 1 || (ws.partials && ws.counters && ws.partial_floats >= partial_floats() &&
                           ws.num_counters > 0 && size_t(ws.num_counters) >= counters());
  }
};

// The height and slice count of the least estimated time, in us, from a sweep over both on the in-
// and the o-projection at 48 to 2,048 rows: rounds of one workgroup per CU, each of steps of 0.9 us
// (256 rows) or 1.12 us (128 rows, two groups), 12 us around them (first loads, epilogue) and, split,
// 5 + 3 s us for the hand-off. Within 6% of the best measured choice at every size of the sweep; on seven
// other weights (n 1,024 to 34,816, k 2,048 to 17,408, 96 to 1,000 rows) within 3% at 27 of 38 sizes, 20% at worst;
// e.g. in-projection: 128 rows 2 slices of 128-row tiles 38 us (1: 53, 4: 53), 384 rows 256-row
// tiles 83 us (128-row tiles 109); o-projection: 256 rows 3 slices of 128-row tiles 43 us (1: 72).
TilePlan plan_tile(int m, int n, int k, int cus, int max_splits) {
  const int G = k / 64;
  TilePlan best{};
  double best_cost = 1e30;
  for (int wm = 2; wm <= 4; wm += 2) {
    TilePlan p{wm, (m + tile_rows(wm) - 1) / tile_rows(wm), n / kTileCols, 1};
    for (int s = 1; s <= max_splits && s <= G; ++s) {
      p.splits = s;
      const size_t rounds = (p.tiles() * s + cus - 1) / cus;
      const int steps = ((G + s - 1) / s + tile_kparts(wm) - 1) / tile_kparts(wm);
      const double cost = rounds * (steps * (wm == 4 ? 0.9 : 1.12) + 12.0 + (s > 1 ? 5.0 + 3.0 * s : 0.0));
      if (cost < best_cost) {
        best = p;
        best_cost = cost;
      }
    }
  }
  return best;
}

// Without the planned split workspace, launches of fewer than two 64 x 256 tiles a CU are refused, whatever
// tiles they take; larger ones run unsplit (they fill the CUs anyway). What callers may leave out thus stays
// the same from one choice of kernels to the next.
bool tile_needs_workspace(int m, int n, int k, int cus) {
  return ((m + 63) / 64) * (n / kTileN) < 2 * cus && k / 64 >= 8;
}

// Whether the 256 x 256 tiles of the large-M kernel fill the CUs.
bool big_fits(int m, int n, int cus) { return m > 32 && ((m + kBigRows - 1) / kBigRows) * (n / kTileN) >= cus; }

}  // namespace

// Enough for every epilogue and every number of rows up to m, so that the workspace of a caller's
// largest launch serves the smaller ones too (a launch's own plan is not monotonic in m).
int gemm_workspace_size(int m, int n, int k, int cus, size_t out[2]) {
  out[0] = out[1] = 0;
  auto need = [&](size_t floats, size_t counters) {
    out[0] = std::max(out[0], floats);
    out[1] = std::max(out[1], counters);
  };
  if (m <= 0) return Q38A_OK;
  const GemvPlan p = plan_gemv(1, n, k, cus);  // the same for every m <= 32
  if (p.tiles_n > 0 && p.splits > 1) need(size_t(p.tiles_n) * p.splits * 32 * kTileN, size_t(p.tiles_n));
  const WidePlan wp = plan_wide(1, n, k, Q38A_EPI_RESIDUAL, cus);  // the same for every m <= kWideRows
  if (wp.tiles > 0 && wp.splits > 1) need(size_t(wp.tiles) * wp.splits * wp.nb * 256, size_t(wp.tiles));
  const int ms = m < kSmallMaxRows ? m : kSmallMaxRows;  // (its partials grow with m)
  for (const int kind : {Q38A_EPI_STORE_BF16, Q38A_EPI_RESIDUAL}) {
    const SmallPlan sp = plan_small(ms, n, k, kind, cus);
    if (sp.splits > 1) need(sp.partial_floats(ms), size_t(sp.tiles));
  }
  // the tile kernel's plan depends on m through its rows of 128-row tiles only
  for (int r = kSmallMaxRows + 1; r <= m && !big_fits(r, n, cus); r = (r + 127) / 128 * 128 + 1) {
    const TilePlan t = plan_tile(r, n, k, cus, kTileMaxSplits);
    need(t.partial_floats(), t.counters());
  }
  return Q38A_OK;
}

template <int BITS>
void launch_gemv(bool ev1, dim3 grid, hipStream_t stream, const GemmArgs& g, const BatchArgs& ba, const MergeIn& mi) {
  const dim3 block(kGemvThreads);
  if (ev1) hipLaunchKernelGGL((qgemv_kernel<BITS, 1>), grid, block, 0, stream, g, ba, mi);
  else hipLaunchKernelGGL((qgemv_kernel<BITS, 4>), grid, block, 0, stream, g, ba, mi);
}

template <int BITS>
void launch_small(int cw, dim3 grid, hipStream_t stream, const GemmArgs& g) {
  const dim3 block(kSmallThreads);
  if (g.m > 32) {
    if (cw == 1) hipLaunchKernelGGL((qgemm_small_kernel<BITS, 2, 1, true>), grid, block, 0, stream, g);
    else hipLaunchKernelGGL((qgemm_small_kernel<BITS, 2, 2, true>), grid, block, 0, stream, g);
  } else {
    if (cw == 1) hipLaunchKernelGGL((qgemm_small_kernel<BITS, 1, 1, true>), grid, block, 0, stream, g);
    else hipLaunchKernelGGL((qgemm_small_kernel<BITS, 1, 2, true>), grid, block, 0, stream, g);
  }
}

// A without 16-byte alignment: any number of rows, kSmallMaxRows a launch, on 128-column tiles.
template <int BITS>
void launch_unaligned(const SmallPlan& sp, hipStream_t stream, GemmArgs g) {
  const dim3 grid(unsigned(sp.tiles), unsigned(sp.splits)), block(kSmallThreads);
  const size_t rows = g.m;
  for (size_t done = 0; done < rows; done += kSmallMaxRows) {
    g.m = int(std::min(rows - done, size_t(kSmallMaxRows)));
    if (g.m > 32) hipLaunchKernelGGL((qgemm_small_kernel<BITS, 2, 2, false>), grid, block, 0, stream, g);
    else hipLaunchKernelGGL((qgemm_small_kernel<BITS, 1, 2, false>), grid, block, 0, stream, g);
    g.a += size_t(kSmallMaxRows) * g.k;
    if (g.kind == Q38A_EPI_RESIDUAL) {
      g.residual += size_t(kSmallMaxRows) * g.n;
      g.xbf += size_t(kSmallMaxRows) * g.n;
      g.partials_out += size_t(kSmallMaxRows) * g.norm_blocks;
    } else {
      g.out = static_cast<char*>(g.out) + size_t(kSmallMaxRows) * g.ldo * (g.kind == Q38A_EPI_STORE_F32 ? 4 : 2);
      if (g.partials_in) g.partials_in += size_t(kSmallMaxRows) * g.norm_blocks;
    }
  }
}

template <int BITS>
void launch_tile(int wm, dim3 grid, hipStream_t stream, const GemmArgs& g) {
  const dim3 block(kTileThreads);
  if (wm == 4) hipLaunchKernelGGL((qgemm_tile_kernel<BITS, 4>), grid, block, 0, stream, g);
  else hipLaunchKernelGGL((qgemm_tile_kernel<BITS, 2>), grid, block, 0, stream, g);
}

// ap: the in-projection append (the launch after the GEMM); mi: the o-projection's A
// merged from decode partials (only shapes of the small-M kernel: the caller checks
// gemm_merge_fits). b: the batch of either.
int launch_qgemm(const uint16_t* A, int m, const q38a_bq_weight& w, const q38a_gemm_epilogue& ep,
                 const q38a_gemm_workspace& ws, const q38a_qk_norm_rope_params* ap, const q38a_batch_desc* b,
                 const q38a_kv_cache_desc* kv, const MergeIn* mi, hipStream_t stream) {
  if (m <= 0) return Q38A_OK;
  int cus = 0;
  if (int rc = device_cu_count(&cus)) return rc;
  // (Up to 32 rows every call has to meet the limits of the split-K kernel, which only the merged A takes
  // now: what was refused stays refused.)
  const GemvPlan pl = plan_gemv(m, w.n, w.k, cus);
  const char* small_ws = "qgemm: workspace too small (q38a_qgemm_workspace_size)";
  if (pl.tiles_n > 0) {
    if (pl.splits > 1 && (!ws.partials || !ws.counters ||
                          ws.partial_floats < size_t(pl.tiles_n) * pl.splits * 32 * kTileN || ws.num_counters < pl.tiles_n))
      return set_error(Q38A_ERR_INVALID, small_ws);
    if (ep.partials_in && ep.kind != Q38A_EPI_RESIDUAL && ep.hidden / 128 > kMaxNormBlocks)
      return set_error(Q38A_ERR_INVALID, "qgemm: hidden %d above %d for the folded norm", ep.hidden,
                       128 * kMaxNormBlocks);
  } else if (mi) {
    return set_error(Q38A_ERR_INVALID, "qgemm: the merged A needs the small-M kernel");
  }
  GemmArgs g{};
  g.a = A;
  g.m = m;
  g.n = w.n;
  g.k = w.k;
  g.lo = w.lo;
  g.hi = w.hi;
  g.scales = w.scales;
  g.kind = ep.kind;
  g.out = ep.out;
  g.ldo = ep.ldo;
  g.n_store = ep.n_store > 0 ? ep.n_store : w.rows;
  g.residual = ep.residual;
  g.xbf = ep.xbf;
  g.partials_out = ep.partials_out;
  g.partials_in = ep.kind == Q38A_EPI_RESIDUAL ? nullptr : ep.partials_in;  // (the residual epilogue has no row scale)
  g.norm_blocks = ep.kind == Q38A_EPI_RESIDUAL ? w.n / 128 : ep.hidden / 128;
  g.inv_hidden = ep.hidden > 0 ? 1.0f / float(ep.hidden) : 0.0f;
  g.eps = ep.eps;
  g.ws_partials = ws.partials;
  g.counters = ws.counters;
  auto aligned = [](const void* p, size_t to) { return reinterpret_cast<uintptr_t>(p) % to == 0; };
  g.wide_out = ep.kind == Q38A_EPI_RESIDUAL ? aligned(ep.residual, 16) && aligned(ep.xbf, 8)
                                            : aligned(ep.out, 16) && ep.ldo % (ep.kind == Q38A_EPI_STORE_F32 ? 4 : 8) == 0;
  g.wide_norm = aligned(ep.partials_in, 16) && g.norm_blocks % 4 == 0;
  // the append as a launch of its own after the GEMM into proj: the same bits as the two calls
  auto then_append = [&]() -> int {
    if (int rc = check_hip(hipGetLastError(), "qgemm launch")) return rc;
    return ap ? launch_qk_norm_rope_append(*ap, *b, *kv, stream) : Q38A_OK;
  };
  // The tile, large-M and 9- to 64-row kernels copy A to LDS 16 bytes at a time, which is only sure to be right
  // for aligned rows; other A goes through registers, 64 rows a launch (in-projection, four layers: 16 rows
  // 111 us against 69, 64 rows 174 against 107, 512 rows 1,300 against 380).
  const bool copy_a = aligned(A, 16);
  // large M: 256 x 256 tiles with the weights dequantised once per workgroup, when those tiles fill
  // the CUs (below that the 128-column tiles, and their K slices, keep more of them busy)
  if (m > kSmallMaxRows && copy_a && big_fits(m, w.n, cus)) {
    g.tiles_n = w.n / kTileN;
    g.splits = 1;
    const dim3 bgrid(unsigned(((m + kBigRows - 1) / kBigRows) * g.tiles_n)), bblock{unsigned(kBigThreads)};
    switch (w.bits) {
      case 4: hipLaunchKernelGGL((qgemm_big_kernel<4>), bgrid, bblock, 0, stream, g); break;
      case 5: hipLaunchKernelGGL((qgemm_big_kernel<5>), bgrid, bblock, 0, stream, g); break;
      case 6: hipLaunchKernelGGL((qgemm_big_kernel<6>), bgrid, bblock, 0, stream, g); break;
      default: return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w.bits);
    }
    return then_append();
  }
  if (m > kSmallMaxRows && copy_a) {
    TilePlan tp = plan_tile(m, w.n, w.k, cus, kTileMaxSplits);
    if (!tp.fits(ws)) {
      if (tile_needs_workspace(m, w.n, w.k, cus)) return set_error(Q38A_ERR_INVALID, small_ws);
      tp = plan_tile(m, w.n, w.k, cus, 1);
    }
    g.tiles_n = tp.tiles_n;
    g.splits = tp.splits;
    const dim3 tgrid(unsigned(tp.tiles() * tp.splits));
    switch (w.bits) {
      case 4: launch_tile<4>(tp.wm, tgrid, stream, g); break;
      case 5: launch_tile<5>(tp.wm, tgrid, stream, g); break;
      case 6: launch_tile<6>(tp.wm, tgrid, stream, g); break;
      default: return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w.bits);
    }
    return then_append();
  }
  // decode-size M on a wide weight: the wide-tile kernel (store epilogues: 64-column tiles, no
  // split-K; residual: 128-column tiles, K split)
  const WidePlan wp = mi ? WidePlan{0, 0, 1} : plan_wide(m, w.n, w.k, ep.kind, cus);
  if (wp.tiles > 0 && (wp.splits == 1 || (ws.partials && ws.counters &&
                                          ws.partial_floats >= size_t(wp.tiles) * wp.splits * wp.nb * 256 &&
                                          ws.num_counters >= wp.tiles))) {
    const dim3 wgrid(unsigned(wp.tiles), unsigned(wp.splits)), wblock(64 * kWideWaves);
#define Q38A_WIDE(B)                                                                            \
  case B:                                                                                       \
    if (wp.nb == 4) hipLaunchKernelGGL((qgemv_wide_kernel<B, 4, true>), wgrid, wblock, 0, stream, g); \
    else hipLaunchKernelGGL((qgemv_wide_kernel<B, 2, false>), wgrid, wblock, 0, stream, g);       \
    break;
    switch (w.bits) {
      Q38A_WIDE(4)
      Q38A_WIDE(5)
      Q38A_WIDE(6)
      default: return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w.bits);
    }
#undef Q38A_WIDE
    return then_append();
  }
  // the other launches up to 64 rows: per layer 33 rows 23.2 us (in-projection with the append) and
  // 20.8 us (o-projection), 64 rows 26.8 and 22.3; the 64 x 256-column split-K tiles took 91.6, 65, 120
  // and 79 us
  if (!mi) {
    SmallPlan sp = plan_small(m, w.n, w.k, copy_a ? ep.kind : int(Q38A_EPI_RESIDUAL), cus);  // (128-column tiles)
    if (sp.splits > 1 && (!ws.partials || !ws.counters || ws.partial_floats < sp.partial_floats(m) || ws.num_counters < sp.tiles)) {
      if (pl.tiles_n == 0 && tile_needs_workspace(m, w.n, w.k, cus)) return set_error(Q38A_ERR_INVALID, small_ws);
      sp.splits = 1;
    }
    if (!copy_a) {
      switch (w.bits) {
        case 4: launch_unaligned<4>(sp, stream, g); break;
        case 5: launch_unaligned<5>(sp, stream, g); break;
        case 6: launch_unaligned<6>(sp, stream, g); break;
        default: return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w.bits);
      }
      return then_append();
    }
    const dim3 sgrid(unsigned(sp.tiles), unsigned(sp.splits));
    switch (w.bits) {
      case 4: launch_small<4>(sp.cw, sgrid, stream, g); break;
      case 5: launch_small<5>(sp.cw, sgrid, stream, g); break;
      case 6: launch_small<6>(sp.cw, sgrid, stream, g); break;
      default: return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w.bits);
    }
    return then_append();
  }
  // the merged A: the split-K kernel, whose staging merges
  const BatchArgs ba = to_args(*b);
  g.tiles_n = pl.tiles_n;
  g.splits = pl.splits;
  const dim3 grid(unsigned(pl.tiles_n * pl.splits));
  const bool ev1 = m <= 8;
  switch (w.bits) {
    case 4: launch_gemv<4>(ev1, grid, stream, g, ba, *mi); break;
    case 5: launch_gemv<5>(ev1, grid, stream, g, ba, *mi); break;
    case 6: launch_gemv<6>(ev1, grid, stream, g, ba, *mi); break;
    default: return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w.bits);
  }
  return check_hip(hipGetLastError(), "qgemm launch");
}

// Whether q38a_qgemm_merge_oproj runs the merge inside the GEMM for m rows (the small-M kernel).
bool gemm_merge_fits(int m, int n, int k, int cus) { return plan_gemv(m, n, k, cus).tiles_n > 0; }

}  // namespace q38a

using namespace q38a;

namespace {

int validate_gemm(const uint16_t* a, int m, const q38a_bq_weight* w, const q38a_gemm_epilogue* ep,
                  const q38a_gemm_workspace* ws) {
  if (!a || !w || !ep || !ws) return set_error(Q38A_ERR_INVALID, "qgemm: null argument");
  if (m < 0) return set_error(Q38A_ERR_INVALID, "qgemm: negative m");
  if (w->bits != 4 && w->bits != 5 && w->bits != 6)
    return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: %d-bit weights are not supported", w->bits);
  if (w->n <= 0 || w->k <= 0 || w->n % 256 || w->k % 64 || w->rows <= 0 || w->rows > w->n)
    return set_error(Q38A_ERR_INVALID, "qgemm: weight %d x %d (rows %d): n % 256 and k % 64 must be 0", w->n, w->k,
                     w->rows);
  if (!w->lo || !w->scales || (w->bits > 4 && !w->hi)) return set_error(Q38A_ERR_INVALID, "qgemm: null weight plane");
  if (ep->kind == Q38A_EPI_RESIDUAL) {
    if (!ep->residual || !ep->xbf || !ep->partials_out)
      return set_error(Q38A_ERR_INVALID, "qgemm: the residual epilogue needs residual, xbf and partials_out");
  } else if (ep->kind == Q38A_EPI_STORE_BF16 || ep->kind == Q38A_EPI_STORE_F32) {
    if (!ep->out || ep->ldo < (ep->n_store > 0 ? ep->n_store : w->rows))
      return set_error(Q38A_ERR_INVALID, "qgemm: out must be set and ldo must cover the stored columns");
  } else {
    return set_error(Q38A_ERR_UNSUPPORTED, "qgemm: epilogue kind %d is not supported", ep->kind);
  }
  if (ep->partials_in && (ep->hidden <= 0 || ep->hidden % 128))
    return set_error(Q38A_ERR_INVALID, "qgemm: folded-norm hidden size must be a positive multiple of 128");
  return Q38A_OK;
}

}  // namespace

extern "C" {

int q38a_qgemm_workspace_size(int m, int n, int k, size_t out[2]) {
  clear_error();
  if (!out || m < 0 || n <= 0 || k <= 0 || n % 256 || k % 64)
    return set_error(Q38A_ERR_INVALID, "qgemm_workspace_size: bad shape");
  int cus = 0;
  if (int rc = device_cu_count(&cus)) return rc;
  return gemm_workspace_size(m, n, k, cus, out);
}

int q38a_qgemm(const uint16_t* a, int m, const q38a_bq_weight* w, const q38a_gemm_epilogue* ep,
               const q38a_gemm_workspace* ws, void* stream) {
  clear_error();
  if (int rc = validate_gemm(a, m, w, ep, ws)) return rc;
  return launch_qgemm(a, m, *w, *ep, *ws, nullptr, nullptr, nullptr, nullptr, static_cast<hipStream_t>(stream));
}

int q38a_qgemm_qkv_append(const uint16_t* a, int m, const q38a_bq_weight* w, const q38a_gemm_epilogue* ep,
                          const q38a_gemm_workspace* ws, const q38a_qk_norm_rope_params* p,
                          const q38a_batch_desc* batch, const q38a_kv_cache_desc* kv, void* stream) {
  clear_error();
  if (int rc = validate_gemm(a, m, w, ep, ws)) return rc;
  if (!p || !batch || !kv) return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: null argument");
  if (ep->kind != Q38A_EPI_STORE_BF16)
    return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: the in-projection epilogue is STORE_BF16 into proj");
  if (int rc = validate_batch(batch, true)) return rc;
  if (int rc = validate_kv(kv)) return rc;
  if (batch->num_tokens != m) return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: m %d != batch tokens %d", m, batch->num_tokens);
  const int nq = p->num_q_heads, nkv = p->num_kv_heads;
  if (nq <= 0 || nkv <= 0 || nkv != kv->kv_heads || w->n != 2 * (nq + nkv) * kHeadDim || w->rows != w->n)
    return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: weight rows must be [q | gate | k | v] heads of 256");
  if (!p->q_out || !p->q_norm || !p->k_norm || !p->rope_cos_sin || p->rope_rows <= 0)
    return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: q_out, norms and the RoPE table must be set");
  if (ep->out != p->proj || ep->ldo != p->ld_proj)
    return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: the epilogue's out/ldo must be the append's proj/ld_proj");
  if (ep->n_store != 0 && ep->n_store != w->n)
    return set_error(Q38A_ERR_INVALID, "qgemm_qkv_append: n_store must cover the whole projection");
  return launch_qgemm(a, m, *w, *ep, *ws, p, batch, kv, nullptr, static_cast<hipStream_t>(stream));
}

namespace {

// in_loader: the merge in the small-M GEMM's A staging where the plan takes that kernel
int merge_oproj(const q38a_attention_params* attn, const q38a_batch_desc* batch, const q38a_bq_weight* w,
                const q38a_gemm_epilogue* ep, const q38a_gemm_workspace* ws, void* stream, bool in_loader) {
  clear_error();
  if (!attn || !batch) return set_error(Q38A_ERR_INVALID, "qgemm_merge_oproj: null argument");
  if (int rc = validate_gemm(attn->out, batch->num_tokens, w, ep, ws)) return rc;
  if (int rc = validate_batch(batch, true)) return rc;
  const int nq = attn->num_q_heads, nkv = attn->num_kv_heads;
  if (nq <= 0 || nkv <= 0 || nq % nkv || !attn->gate || !attn->split_scratch || attn->max_splits <= 0 ||
      attn->max_splits > kMaxMergeSplits || attn->ld_gate < nq * kHeadDim)
    return set_error(Q38A_ERR_INVALID, "qgemm_merge_oproj: attention heads, gate, split scratch or max_splits invalid");
  if (batch->num_tokens != batch->num_seqs)
    return set_error(Q38A_ERR_INVALID, "qgemm_merge_oproj: one token per sequence required (M %d, B %d)",
                     batch->num_tokens, batch->num_seqs);
  if (w->k != nq * kHeadDim)
    return set_error(Q38A_ERR_INVALID, "qgemm_merge_oproj: weight k %d != %d q heads x 256", w->k, nq);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  const int m = batch->num_tokens;
  int cus = 0, grid = 0, target = 0;
  if (int rc = device_cu_count(&cus)) return rc;
  if (int rc = decode_grid(&grid, &target)) return rc;
  if (!in_loader || !gemm_merge_fits(m, w->n, w->k, cus)) {
    // the merge kernel writes attn->out, which the GEMM reads
    if (int rc = launch_attention_merge(*attn, *batch, st)) return rc;
    return launch_qgemm(attn->out, m, *w, *ep, *ws, nullptr, batch, nullptr, nullptr, st);
  }
  const MergeIn mi{attn->split_scratch, attn->gate, attn->ld_gate, nq, nkv, attn->max_splits, target};
  return launch_qgemm(attn->out, m, *w, *ep, *ws, nullptr, batch, nullptr, &mi, st);
}

}  // namespace

int q38a_qgemm_merge_oproj(const q38a_attention_params* attn, const q38a_batch_desc* batch, const q38a_bq_weight* w,
                           const q38a_gemm_epilogue* ep, const q38a_gemm_workspace* ws, void* stream) {
  return merge_oproj(attn, batch, w, ep, ws, stream, false);
}

int q38a_qgemm_merge_oproj_in_loader(const q38a_attention_params* attn, const q38a_batch_desc* batch,
                                     const q38a_bq_weight* w, const q38a_gemm_epilogue* ep,
                                     const q38a_gemm_workspace* ws, void* stream) {
  return merge_oproj(attn, batch, w, ep, ws, stream, true);
}

}  // extern "C"
