// Mamba-2 SSD scan (mamba_ssm's mamba_chunk_scan_combined) on gfx950, in
// 64-step chunks with the chunk-local contractions on the matrix cores: in bf16
// pieces at float32 accuracy (ssd_pieces.h), or, in the chunk gradients of
// float32, fp16 and headdims and dstates other than 32, 64 and 64, 128, and in
// the per-sequence states, on v_mfma_f32_16x16x4_f32 with the storage type
// widened when a tile is staged.
//
// Per batch row b and head h (group g), with a_t = dt_t A and, inside a
// chunk, cs_t = a_0 + ... + a_t (so cs <= 0 and decays are exp of differences):
//   forward
//     F1  S_c  = sum_s exp(cs_L - cs_s) dt_s x_s B_s^T          (chunk-end state from 0)
//     F2  H_c  = exp(cs_L(c-1)) H_{c-1} + S_{c-1}               (state entering chunk c)
//     F3  Y    = (C B^T o M) (dt x) + diag(exp(cs)) C H_c^T + D x,  M[t][s] = exp(cs_t - cs_s) [s <= t]
//         out  = Y silu(z)
//   backward (dY the gradient of Y, dH_c^out that of the state leaving chunk c)
//     K1  the seed E_c = (diag(exp(cs)) C)^T dY of dL/dH_c from the chunk's own outputs
//     K2  dH^out_c = dH^in_{c+1} ; dH^in_c = exp(cs_L) dH^out_c + E_c (reverse over
//         chunks); dcs_L += <dH^out_c, exp(cs_L) H_c>
//     K3  per chunk: dG = dY (dt x)^T, dCB = dG o M, d(dt x) = (CB o M)^T dY
//         + B~ dH^out^T, dC = dCB B + diag(exp(cs)) dY H_c, dB = dCB^T C +
//         diag(w) (dt x) dH^out (B~ = diag(w) B, w_s = exp(cs_L - cs_s)), dcs
//         from all of them, da = suffix sums of dcs, then ddt, dx, dz and the
//         per-chunk partials of dA, dD, ddt_bias
//     a fixed-order reduce sums dB/dC over the head blocks of a group and the
//     partials.
// F1 and F2, and K1 and K2, run as one launch each (F12, K12) where enough
// workgroups walk the chunks in order (ssd_state_kernel).
// The chunk kernels (F3, K3) give a workgroup one chunk of `hb` heads of one
// group: B, C and C B^T are staged and formed once and each head reuses them;
// K3 keeps dB and dC of the block's heads in matrix-core accumulators.
// Chunks past the sequence end are padded with dt = 0 (no decay, no input).
#include "mcpu_common.h"
#include "scan_common.h"
#include "ssd_params.h"
#include "ssd_pieces.h"

namespace mcpu {

namespace {

constexpr int Q = kSsdQ;
constexpr int QP = Q + 4;          // padded row lengths of the LDS tiles (16-byte multiples)
constexpr int XP = kSsdMaxP + 4;
constexpr int NP = kSsdMaxN + 4;
constexpr int kThreads = 256;

__device__ __forceinline__ v4f mfma4(float a, float b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc[j] += A(16 x K) B(K x 16 columns 16 j ..) for column tiles j < NTC,
// operands float32 in LDS: A(i, k) = a[i ai + k ak] (a at the strip's first
// row), times `as` when SCALE (the lane's own row factor), B(k, c) = b[k bk +
// c bj]. K is a multiple of 16: four k-steps of operands are read before
// their products issue (and no more, to bound the registers). In each
// v_mfma_f32_16x16x4_f32 lane l supplies A(l % 16, k + l / 16) and B(k + l /
// 16, l % 16); lane l ends holding D(4 (l / 16) + e, l % 16) in acc[j][e].
template <int NTC, int NT, bool SCALE>
__device__ __forceinline__ void mma_n(v4f (&acc)[NT], const float* a, int ai, int ak, const float* b, int bk, int bj,
                                      int K, float as) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  const float* pa = a + r * ai + q * ak;
  const float* pb = b + q * bk + r * bj;
#pragma clang loop unroll(disable)
  for (int k0 = 0; k0 < K; k0 += 16) {
    float av[4], bv[4][NTC];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      av[u] = pa[(k0 + 4 * u) * ak];
      if (SCALE) av[u] *= as;
#pragma unroll
      for (int j = 0; j < NTC; ++j) bv[u][j] = pb[(k0 + 4 * u) * bk + 16 * j * bj];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int j = 0; j < NTC; ++j) acc[j] = mfma4(av[u], bv[u][j], acc[j]);
  }
}

// mma_n for a tile count nt (uniform, 1 <= nt <= NT) known only at run time:
// one branch picks the compile-time variant, so the products of a k-step
// issue back to back.
template <int NT, bool SCALE = false>
__device__ __forceinline__ void mma(v4f (&acc)[NT], int nt, const float* a, int ai, int ak, const float* b, int bk,
                                    int bj, int K, float as = 1.f) {
  static_assert(NT >= 1 && NT <= 8, "tile count");
  if (nt <= 0) return;
  switch (nt) {
    case 1: mma_n<1, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    case 2: if constexpr (NT >= 2) mma_n<2, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    case 3: if constexpr (NT >= 3) mma_n<3, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    case 4: if constexpr (NT >= 4) mma_n<4, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    case 5: if constexpr (NT >= 5) mma_n<5, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    case 6: if constexpr (NT >= 6) mma_n<6, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    case 7: if constexpr (NT >= 7) mma_n<7, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
    default: if constexpr (NT >= 8) mma_n<8, NT, SCALE>(acc, a, ai, ak, b, bk, bj, K, as); break;
  }
}

template <int NT>
__device__ __forceinline__ void zero(v4f (&acc)[NT]) {
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
}

// ---- four consecutive storage elements <-> float4 (16-byte aligned float32,
// 8-byte aligned 16-bit types) ----
// As loaded: float4 for float32, the raw 16-bit pairs otherwise. Prefetched
// tiles stay raw in registers and are widened where they are parked in LDS:
// widening next to the load would make the wave wait for the load there.
template <typename Tx> struct Raw4 { using type = uint2; };
template <> struct Raw4<float> { using type = float4; };
template <typename Tx> using raw4 = typename Raw4<Tx>::type;

template <typename Tx> __device__ __forceinline__ raw4<Tx> ld_raw(const Tx* p) {
  return *reinterpret_cast<const raw4<Tx>*>(p);
}
template <typename Tx> __device__ __forceinline__ raw4<Tx> raw_zero() { return make_uint2(0u, 0u); }
template <> __device__ __forceinline__ float4 raw_zero<float>() { return make_float4(0.f, 0.f, 0.f, 0.f); }
template <typename Tx> __device__ __forceinline__ float4 widen(raw4<Tx> u);
template <> __device__ __forceinline__ float4 widen<float>(float4 u) { return u; }
template <> __device__ __forceinline__ float4 widen<bf16>(uint2 u) {
  return make_float4(__builtin_bit_cast(float, u.x << 16), __builtin_bit_cast(float, u.x & 0xffff0000u),
                     __builtin_bit_cast(float, u.y << 16), __builtin_bit_cast(float, u.y & 0xffff0000u));
}
template <> __device__ __forceinline__ float4 widen<f16>(uint2 u) {
  auto h = [](uint32_t bits) { return static_cast<float>(__builtin_bit_cast(f16, static_cast<uint16_t>(bits))); };
  return make_float4(h(u.x & 0xffff), h(u.x >> 16), h(u.y & 0xffff), h(u.y >> 16));
}
template <typename Tx> __device__ __forceinline__ void st4(Tx* p, float4 v);
template <> __device__ __forceinline__ void st4<float>(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
template <> __device__ __forceinline__ void st4<bf16>(bf16* p, float4 v) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
}
template <> __device__ __forceinline__ void st4<f16>(f16* p, float4 v) {
  auto b = [](float f) { return static_cast<uint32_t>(__builtin_bit_cast(uint16_t, static_cast<f16>(f))); };
  *reinterpret_cast<uint2*>(p) = make_uint2(b(v.x) | (b(v.y) << 16), b(v.z) | (b(v.w) << 16));
}

__device__ __forceinline__ float4 scale4(float4 v, float s) { return make_float4(v.x * s, v.y * s, v.z * s, v.w * s); }

// The row of float4 number v of a tile with nv float4 per row: floor((v +
// 0.5) / nv) in float32 is exact for the tile sizes here (v < 2^11, nv <= 32:
// the quotient is at least 0.5 / nv away from an integer).
__device__ __forceinline__ int tile_row(int v, float inv_nv) {
  return static_cast<int>((static_cast<float>(v) + 0.5f) * inv_nv);
}

// The backward chunk kernel runs 8 waves: two per 16-row strip, splitting
// each product's column tiles.
constexpr int kThreads3 = 512;

// float4 per thread of the staged tiles: (64 x dstate) and (headdim x
// dstate) tiles, (64 x headdim) tiles and (headdim x 64-state half) tiles,
// for a workgroup of TPB threads.
template <int TPB = kThreads> constexpr int vec_n() { return Q * kSsdMaxN / 4 / TPB; }
template <int TPB = kThreads> constexpr int vec_x() { return Q * kSsdMaxP / 4 / TPB; }
constexpr int kVecN = vec_n();
constexpr int kVecX = vec_x();

// Registers x = rows r < nrows, columns c < ncols (multiple of 4) of
// src[r rs + c], four elements per entry, rows from nvalid on zero; thread
// tid holds entry number tid + k TPB of the row-major tile. The loads are
// issued here and waited for where the registers are used.
template <typename Tx, int V, int TPB = kThreads>
__device__ __forceinline__ void tile_load(raw4<Tx> (&x)[V], const Tx* src, int64_t rs, int nrows, int nvalid,
                                          int ncols) {
  const int nv = ncols >> 2, total = nrows * nv;
  const float inv = 1.0f / static_cast<float>(nv);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int v = threadIdx.x + k * TPB;
    x[k] = raw_zero<Tx>();
    if (v < total) {
      const int r = tile_row(v, inv);
      if (r < nvalid) x[k] = ld_raw<Tx>(src + r * rs + ((v - r * nv) << 2));
    }
  }
}

// LDS tile s (rows of ld floats) from registers filled by tile_load with the
// same nrows / ncols, widened to float32, times scale[r] when given.
template <typename Tx, int V, int TPB = kThreads>
__device__ __forceinline__ void tile_store(float* s, int ld, const raw4<Tx> (&x)[V], int nrows, int ncols,
                                           const float* scale = nullptr) {
  const int nv = ncols >> 2, total = nrows * nv;
  const float inv = 1.0f / static_cast<float>(nv);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int v = threadIdx.x + k * TPB;
    if (v < total) {
      const int r = tile_row(v, inv);
      const int c = (v - r * nv) << 2;
      const float4 f = widen<Tx>(x[k]);
      *reinterpret_cast<float4*>(s + r * ld + c) = scale ? scale4(f, scale[r]) : f;
    }
  }
}

// How TPB threads move a tile of NC columns (64 or 128), of which the first
// ncols exist, four elements at a time: NC / 4 threads to a row, so a thread
// keeps its column and steps down the rows. EXACT: ncols = NC.
template <int TPB, int NC, bool EXACT> struct TileMap {
  static constexpr int step = TPB / (NC / 4);
  int row, col;
  bool on;   // the thread's column exists
  __device__ __forceinline__ explicit TileMap(int ncols, int tid = threadIdx.x) {
    row = tid / (NC / 4);
    col = (tid % (NC / 4)) * 4;
    on = EXACT || col < ncols;
  }
};

// A lane's offset, kept apart from the uniform pointer it is added to: out of a
// loop the compiler would carry their 64-bit sum per lane, one for each tensor
// and entry, and spill.
__device__ __forceinline__ uint32_t lane_offset(uint32_t off) {
  asm volatile("" : "+v"(off));
  return off;
}

// Entry k of a thread: row m.row + k m.step of src, row stride rs elements, with
// nvalid rows. Every load is unconditional (what does not exist loads an
// element that does, and map_park zeroes it), so that a tile's loads issue
// together. Offsets from the uniform src are 32 bits: 64 rows of at most 65535
// heads.
template <typename Tx, int V, int TPB, int NC, bool EXACT>
__device__ __forceinline__ void map_load(raw4<Tx> (&x)[V], const TileMap<TPB, NC, EXACT>& m, const Tx* src,
                                         int64_t rs, int nvalid) {
  static_assert(V * TPB * 4 <= 64 * NC, "a thread's entries stay within 64 rows");
  const int col = m.on ? m.col : 0;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const int r = m.row + k * m.step < nvalid ? m.row + k * m.step : nvalid - 1;
    x[k] = ld_raw<Tx>(src + lane_offset(r * static_cast<uint32_t>(rs) + col));
  }
}

// Those entries as bf16 pieces (ssd_pieces.h) in LDS tile s; rows from nvalid
// on, and columns that do not exist, zero.
template <typename Tx, bool F32 = false, int V, int TPB, int NC, bool EXACT>
__device__ __forceinline__ void map_park(uint16_t* s, int ld, int plane, const TileMap<TPB, NC, EXACT>& m,
                                         const raw4<Tx> (&x)[V], int nvalid) {
  constexpr int NP = kPieces<Tx>;
  uint16_t* at = s + m.row * ld + m.col;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const raw4<Tx> v = m.on && m.row + k * m.step < nvalid ? x[k] : raw_zero<Tx>();
    uint16_t* to = at + k * m.step * ld;
    if constexpr (std::is_same_v<Tx, bf16>) {
      *reinterpret_cast<uint2*>(to) = v;
    } else {
      const float4 f = widen<Tx>(v);
      const float fv[4] = {f.x, f.y, f.z, f.w};
      uint2 o[NP];
      split4<NP, F32>(fv, o);
#pragma unroll
      for (int i = 0; i < NP; ++i) *reinterpret_cast<uint2*>(to + i * plane) = o[i];
    }
  }
}

// Four elements of a row of pieces, summed.
template <int NP> __device__ __forceinline__ float4 pieces4(const uint16_t* at, int plane) {
  float4 f = widen<bf16>(*reinterpret_cast<const uint2*>(at));
#pragma unroll
  for (int i = 1; i < NP; ++i) {
    const float4 g = widen<bf16>(*reinterpret_cast<const uint2*>(at + i * plane));
    f = make_float4(f.x + g.x, f.y + g.y, f.z + g.z, f.w + g.w);
  }
  return f;
}

// tile_load then tile_store.
template <typename Tx, int V, int TPB = kThreads>
__device__ __forceinline__ void stage(float* s, int ld, const Tx* src, int64_t rs, int nrows, int nvalid, int ncols,
                                      const float* scale = nullptr) {
  raw4<Tx> x[V];
  tile_load<Tx, V, TPB>(x, src, rs, nrows, nvalid, ncols);
  tile_store<Tx, V, TPB>(s, ld, x, nrows, ncols, scale);
}

// The dout tile of one head's chunk, and with HAS_Z its z and ysave (x layout from
// `off`), for a workgroup of TPB threads.
template <typename Tx, bool HAS_Z, int TPB = kThreads>
struct DyTiles {
  static constexpr int V = vec_x<TPB>();
  raw4<Tx> go[V], zz[V], yy[V];

  __device__ __forceinline__ void load(const SsdParams& p, int64_t off, int64_t rs, int nvalid, int ncols) {
    tile_load<Tx, V, TPB>(go, static_cast<const Tx*>(p.dout) + off, rs, Q, nvalid, ncols);
    if (HAS_Z) {
      tile_load<Tx, V, TPB>(zz, static_cast<const Tx*>(p.z) + off, rs, Q, nvalid, ncols);
      tile_load<Tx, V, TPB>(yy, static_cast<const Tx*>(p.ysave) + off, rs, Q, nvalid, ncols);
    }
  }

  // LDS tile of dY = dout silu(z) (dout without z); dz = dout y silu'(z) to rows
  // below nvalid.
  __device__ __forceinline__ void store(float* s, int ld, const SsdParams& p, int64_t off, int64_t rs, int nvalid,
                                        int ncols) const {
    const int nv = ncols >> 2, total = Q * nv;
    const float inv = 1.0f / static_cast<float>(nv);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const int v = threadIdx.x + k * TPB;
      if (v >= total) continue;
      const int r = tile_row(v, inv);
      const int c = (v - r * nv) << 2;
      float4 dz = make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 dy = dy_of(k, dz);
      if (HAS_Z && r < nvalid) st4<Tx>(static_cast<Tx*>(p.dz) + off + r * rs + c, dz);
      *reinterpret_cast<float4*>(s + r * ld + c) = dy;
    }
  }

  // dY of float4 number k, and with HAS_Z its dz.
  __device__ __forceinline__ float4 dy_of(int k, float4& dz) const {
    const float4 g4 = widen<Tx>(go[k]);
    if (!HAS_Z) return g4;
    const float4 z4 = widen<Tx>(zz[k]);
    const float gx[4] = {g4.x, g4.y, g4.z, g4.w}, zx[4] = {z4.x, z4.y, z4.z, z4.w};
    float d[4], sg[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      sg[u] = sigmoid(zx[u]);
      d[u] = gx[u] * zx[u] * sg[u];
    }
    const float4 y4 = widen<Tx>(yy[k]);
    const float yv[4] = {y4.x, y4.y, y4.z, y4.w};
    float dzv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) dzv[u] = gx[u] * yv[u] * sg[u] * (1.f + zx[u] * (1.f - sg[u]));
    dz = make_float4(dzv[0], dzv[1], dzv[2], dzv[3]);
    return make_float4(d[0], d[1], d[2], d[3]);
  }
};

// Inclusive prefix sum over the 64 lanes of a wave as a float pair hi + lo:
// each addition keeps its rounding error (Knuth's TwoSum) in lo, so a
// difference (hi_t - hi_s) + (lo_t - lo_s) is accurate relative to itself
// rather than to the size of the running sums.
// v comes as the pair v + vlo.
__device__ __forceinline__ void wave_prefix_sum2(float v, float& hi, float& lo, float vlo = 0.f) {
  const int lane = threadIdx.x & 63;
  hi = v;
  lo = vlo;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float oh = __shfl_up(hi, d, 64), ol = __shfl_up(lo, d, 64);
    if (lane >= d) {
      const float sum = hi + oh;
      const float bv = sum - hi;
      const float err = (hi - (sum - bv)) + (oh - bv);
      hi = sum;
      lo = (lo + ol) + err;
    }
  }
}

// exp(cs_t - cs_s) from the float pairs of the running sums.
__device__ __forceinline__ float seg_exp(const float* cs, const float* lo, int t, int s) {
  return fast_exp((cs[t] - cs[s]) + (lo[t] - lo[s]));
}

// Inclusive suffix sum over the 64 lanes of a wave (lane 63 first).
__device__ __forceinline__ float wave_suffix_sum(float v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float o = __shfl_down(v, d, 64);
    if (lane + d < 64) v += o;
  }
  return v;
}

// a + b as a float pair: the sum, its rounding error added to lo (TwoSum).
__device__ __forceinline__ float add2(float a, float b, float& lo) {
  const float sum = a + b, bv = sum - a;
  lo += (a - (sum - bv)) + (b - bv);
  return sum;
}

// The same of pairs v + lo (wave_prefix_sum2), rounded once: the terms nearly
// cancel over a chunk.
__device__ __forceinline__ float wave_suffix_sum2(float v, float vlo) {
  const int from = 63 - (threadIdx.x & 63);
  float hi, lo;
  wave_prefix_sum2(__shfl(v, from, 64), hi, lo, __shfl(vlo, from, 64));
  return __shfl(hi + lo, 63 - (threadIdx.x & 63), 64);
}

// Sum over the 64 lanes of a wave, in a fixed order, in every lane.
__device__ __forceinline__ float wave_total(float v) {
  v = row_allreduce16(v);
  v = swap_sum<32>(v, v);
  return swap_sum<16>(v, v);
}

// The effective step for dt + dt_bias = pre and, when grad, d(step)/d(raw
// dt): the softplus derivative, zero where the clamp to [dt_lo, dt_hi] is
// active. The clamp always applies, as in mamba_ssm (its default (0, inf)
// makes a negative raw step 0), and keeps a NaN step NaN, as torch.clamp does.
__device__ __forceinline__ float step_of(const SsdParams& p, float pre, float* grad) {
  float sg = 1.f;
  float st = pre;
  if (p.softplus) st = softplus_sigmoid(pre, sg);
  const bool inside = st >= p.dt_lo && st <= p.dt_hi;
  st = st < p.dt_lo ? p.dt_lo : (st > p.dt_hi ? p.dt_hi : st);
  if (!inside) sg = 0.f;
  if (grad) *grad = sg;
  return st;
}
// The same for (b, t, h); 0 past the sequence.
__device__ __forceinline__ float ssd_step(const SsdParams& p, int64_t b, int64_t t, int64_t h, float* grad) {
  if (t >= p.seqlen) {
    if (grad) *grad = 0.f;
    return 0.f;
  }
  return step_of(p, p.dt[(b * p.seqlen + t) * p.nheads + h] + (p.dt_bias ? p.dt_bias[h] : 0.f), grad);
}

// Chunk row (b, h, c) of the cs / step arrays.
__device__ __forceinline__ int64_t chunk_row(const SsdParams& p, int64_t b, int64_t h, int64_t c) {
  return ((b * p.nheads + h) * p.nchunks + c) * Q;
}

// Offset of the (b, c, h) state block in states / dstates.
__device__ __forceinline__ int64_t state_block(const SsdParams& p, int64_t b, int64_t c, int64_t h) {
  return ((b * p.nchunks + c) * p.nheads + h) * p.headdim * p.dstate;
}

// Steps of the chunk that exist.
__device__ __forceinline__ int chunk_steps(const SsdParams& p, int64_t t0) {
  return static_cast<int>(p.seqlen - t0 < Q ? p.seqlen - t0 : Q);
}

// Packed sequences. Kernels built with SEQ read p.seq_idx; without it every
// helper below folds to a constant (one sequence, id 0).
//
// Id of step t of batch row b: 0 before the first step (the initial state's
// id); steps past the sequence (a chunk's padding) take the last step's id.
template <bool SEQ>
__device__ __forceinline__ int32_t seq_of(const SsdParams& p, int64_t b, int64_t t) {
  if constexpr (!SEQ) return 0;
  if (t < 0) return 0;
  return p.seq_idx[b * p.seqlen + (t < p.seqlen ? t : p.seqlen - 1)];
}

// Ids do not decrease, so the steps of a chunk that share an id form a run.
// For the wave whose lane l stands for step t0 + l: the first step (in the
// chunk) of lane l's run.
template <bool SEQ>
__device__ __forceinline__ int run_first(const SsdParams& p, int64_t b, int64_t t0, int lane) {
  if constexpr (!SEQ) return 0;
  const bool starts = lane == 0 || seq_of<SEQ>(p, b, t0 + lane) != seq_of<SEQ>(p, b, t0 + lane - 1);
  const unsigned long long upto = __ballot(starts) & (~0ull >> (63 - lane));
  return 63 - __clzll(upto);
}

// Whether the state entering chunk c carries through it: the ids at the ends
// of chunks c - 1 and c agree (ids do not decrease, so none changes between).
template <bool SEQ>
__device__ __forceinline__ bool carries(const SsdParams& p, int64_t b, int64_t c) {
  if constexpr (!SEQ) return true;
  const int64_t end = (c + 1) * Q < p.seqlen ? (c + 1) * Q - 1 : p.seqlen - 1;
  return seq_of<SEQ>(p, b, end) == seq_of<SEQ>(p, b, c * Q - 1);
}

}  // namespace

// F2: walks the chunks in order, replacing each chunk-end state by the state
// entering the chunk, H_c = exp(cs_L(c-1)) H_{c-1} + S_{c-1} (H_0 = the
// initial state or 0), and writes the final state. One thread per state
// element; grid (nslices, nheads, batch). The next chunk's loads issue before
// this chunk's store.
template <bool SEQ>
__global__ void __launch_bounds__(kThreads) ssd_state_pass_kernel(const SsdParams p) {
  const int64_t PN = p.headdim * p.dstate, H = p.nheads;
  const int64_t e = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  const int64_t h = blockIdx.y, b = blockIdx.z;
  if (e >= PN) return;
  float run = p.init ? p.init[(b * H + h) * PN + e] : 0.f;
  float* st = p.states + state_block(p, b, 0, h) + e;
  const int64_t cstride = H * PN;
  const float* csl = p.cs + chunk_row(p, b, h, 0) + (Q - 1);
  float s = st[0], d = csl[0];
  for (int64_t c = 0; c < p.nchunks; ++c) {
    const float sc = s, dc = carries<SEQ>(p, b, c) ? fast_exp(d) : 0.f;
    if (c + 1 < p.nchunks) {
      s = st[(c + 1) * cstride];
      d = csl[(c + 1) * Q];
    }
    st[c * cstride] = run;
    run = fmaf(dc, run, sc);
  }
  if (p.final_states) p.final_states[(b * H + h) * PN + e] = run;
}

// The steps and running decays of every chunk, for the in-order kernels:
// one wave per (b, h, chunk), lane t owning step t. Grid (ceil(nchunks / 4),
// nheads, batch).
__global__ void __launch_bounds__(kThreads) ssd_chunk_decay_kernel(const SsdParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t c = static_cast<int64_t>(blockIdx.x) * (kThreads / 64) + (threadIdx.x >> 6);
  const int64_t h = blockIdx.y, b = blockIdx.z;
  if (c >= p.nchunks) return;
  const float st = ssd_step(p, b, c * Q + lane, h, nullptr);
  float cs, csl;
  wave_prefix_sum2(st * p.A[h], cs, csl);
  const int64_t row = chunk_row(p, b, h, c);
  p.cs[row + lane] = cs;
  p.cs_lo[row + lane] = csl;
  p.step[row + lane] = st;
}

// The thread's index for a kernel's second pass: what the compiler derives from it
// does not wait in registers through the first.
__device__ __forceinline__ int second_tid() {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  return tid;
}

constexpr int kLdS = 64 + 4;          // rows of the state kernel's 64-column tiles
constexpr int kPlaneS = Q * kLdS;

// Entries of map_load's mapping, times sc[k], in three pieces.
template <bool F32, int V, int TPB, int NC, bool EXACT>
__device__ __forceinline__ void park_scaled(uint16_t* s, const TileMap<TPB, NC, EXACT>& m, const float4 (&x)[V],
                                            const float (&sc)[V]) {
  uint16_t* at = s + m.row * kLdS + m.col;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const float fv[4] = {x[k].x * sc[k], x[k].y * sc[k], x[k].z * sc[k], x[k].w * sc[k]};
    uint2 o[3];
    split4<3, F32>(fv, o);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2*>(at + k * m.step * kLdS + i * kPlaneS) = o[i];
  }
}

template <typename Tx> struct StateLds {
  __align__(16) uint16_t A[3 * kPlaneS];             // the scaled x or dY (steps x headdim)
  __align__(16) uint16_t B[kPieces<Tx> * kPlaneS];   // B or C (steps x 64 states)
  float part[kThreads / 64];
};

// The states' products, in both directions and both forms. Per chunk c, for 64
// state columns of one head,
//   forward   U_c = sum_s exp(cs_L - cs_s) dt_s x_s B_s^T
//   backward  U_c = sum_t exp(cs_t) dY_t C_t^T
// as (rows p, columns n) in matrix-core accumulators, both operands in pieces
// and read transposed from the LDS tiles they are staged in.
//   WALK (F12, K12): the workgroup of (b, h, column block) walks the chunks in
//     the direction's order with the state X in the accumulators: it stores X
//     (the state entering the chunk, or the gradient of the one leaving it), then
//     X <- exp(cs_L) X + U_c, so that U never reaches memory. Grid (column
//     blocks, nheads, batch).
//   otherwise (F1, K1): the workgroup of (chunk, column block) stores U_c for
//     the passing kernel; forward, it also forms and saves the chunk's steps and
//     running decays. Grid (nchunks x column blocks, nheads, batch).
// EXACT: headdim 64, dstate 128; otherwise tiles are filled up with zeros. The
// next chunk's tiles load while the current products run.
// DCS (backward walk): also <X, exp(cs_L) H_c> over its columns to dcsL, for the
// float32 chunk gradients; the bf16 ones form it from tiles they read anyway.
// What bounds it is memory: x (or dout and z) once per column block, X out.
// Batch 4, seqlen 2048, 80 heads, bf16 with z: forward 138 us (3.7 TB/s), backward
// 171 us (3.9 TB/s), against 195 and 254 us on float32 tiles, the latter with
// H_c read for dcsL.
// F32: the pass on the float32 unit, for a workgroup whose pass in pieces ended with
// a value that is not finite (returned: 0 if there is none; none becomes finite again
// on the way).
template <typename Tx, bool HAS_Z, bool SEQ, bool BWD, bool WALK, bool EXACT, bool DCS, bool F32>
__device__ __forceinline__ float state_pass(const SsdParams& p, StateLds<Tx>& lds) {
  constexpr int TPB = kThreads, V = vec_x(), NX = kPieces<Tx>, NT = kSsdPassCols / 16;
  static_assert(!DCS || (BWD && WALK), "dcsL belongs to the backward walk");
  uint16_t* const s_A = lds.A;
  uint16_t* const s_B = lds.B;
  float (&s_part)[TPB / 64] = lds.part;
  const int tid = F32 ? second_tid() : threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int64_t L = p.seqlen, H = p.nheads, G = p.ngroups;
  const int64_t P = EXACT ? kSsdMaxP : p.headdim, N = EXACT ? kSsdMaxN : p.dstate;
  const uint32_t ncb = static_cast<uint32_t>((N + kSsdPassCols - 1) / kSsdPassCols);
  const int64_t blk = WALK ? blockIdx.x : blockIdx.x % ncb;
  const int64_t n0 = blk * kSsdPassCols;
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int64_t g = h / (H / G);
  const int ncol = static_cast<int>(N - n0 < kSsdPassCols ? N - n0 : kSsdPassCols);
  const bool act = EXACT || 16 * wave < P;
  const TileMap<TPB, kSsdMaxP, EXACT> ma(static_cast<int>(P), tid);
  const TileMap<TPB, kSsdPassCols, EXACT> mb(ncol, tid);
  // Accumulator element (j, e) of this lane: state row 16 wave + 4 q + e,
  // column n0 + 16 j + r, at offset eo + e N + 16 j of a (headdim x dstate) block.
  const uint32_t eo = static_cast<uint32_t>((16 * wave + 4 * q) * N + n0 + r);
  auto on = [&](int j) { return EXACT || (act && 16 * j < ncol); };
  v4f acc[NT];
  const Tx* const Ah = static_cast<const Tx*>(BWD ? p.dout : p.x) + b * L * H * P + h * P;
  const Tx* const Zh = static_cast<const Tx*>(p.z) + b * L * H * P + h * P;
  const Tx* const Bg = static_cast<const Tx*>(BWD ? p.C : p.B) + b * L * G * N + g * N + n0;
  raw4<Tx> ra[V], rz[V], rb[V];
  float ncs = 0.f, nlo = 0.f, nst = 0.f, nH[DCS ? NT : 1][4];
  auto fetch = [&](int64_t c) {
    const int64_t t0 = c * Q;
    const int nv = chunk_steps(p, t0);
    map_load<Tx>(ra, ma, Ah + t0 * H * P, H * P, nv);
    if constexpr (BWD && HAS_Z) map_load<Tx>(rz, ma, Zh + t0 * H * P, H * P, nv);
    map_load<Tx>(rb, mb, Bg + t0 * G * N, G * N, nv);
    const int64_t row = chunk_row(p, b, h, c);
    if constexpr (BWD || WALK) {
      const uint32_t at = lane_offset(lane);
      ncs = (p.cs + row)[at];
      nlo = (p.cs_lo + row)[at];
      if (!BWD) nst = (p.step + row)[at];
    } else {
      nst = ssd_step(p, b, t0 + lane, h, nullptr);
      wave_prefix_sum2(nst * p.A[h], ncs, nlo);
      if (blk == 0 && wave == 0) {
        p.cs[row + lane] = ncs;
        p.cs_lo[row + lane] = nlo;
        p.step[row + lane] = nst;
      }
    }
    if constexpr (DCS) {
      const float* hs = p.states + state_block(p, b, c, h);
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) nH[j][e] = on(j) ? hs[eo + e * N + 16 * j] : 0.f;
    }
  };
  float* const dcsl = DCS ? p.dcsL + (chunk_row(p, b, h, 0) / Q) * p.nslices + blk : nullptr;
  const int64_t only = WALK ? 0 : blockIdx.x / ncb;
  const int64_t count = WALK ? p.nchunks : 1;
  auto chunk_at = [&](int64_t i) { return WALK ? (BWD ? p.nchunks - 1 - i : i) : only; };
  int64_t pend = -1;        // chunk whose dcsL share awaits the cross-wave sum
  float pend_decay = 0.f;
  zero(acc);
  // The state the walk starts from. The second pass reads it back from where the first
  // put it, element by element in the same threads: the first has also written the
  // walk's end, which may lie over it.
  const float* init = F32 ? (BWD ? p.dstates : p.states) : BWD ? p.dfinal : p.init;
  if (WALK && init != nullptr) {
    const float* src = init + (F32 ? state_block(p, b, chunk_at(0), h) : (b * H + h) * P * N);
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (on(j)) acc[j][e] = src[eo + e * N + 16 * j];
  }
  fetch(chunk_at(0));
  for (int64_t i = 0; i < count; ++i) {
    const int64_t c = chunk_at(i), t0 = c * Q;
    const int nv = chunk_steps(p, t0);
    // Lane t: step t's factor. Packed sequences: forward only the chunk's last
    // run reaches its end, backward only the first reads the entering state.
    const float csL = __shfl(ncs, Q - 1, 64), loL = __shfl(nlo, Q - 1, 64);
    float f;
    if constexpr (BWD) {
      f = seq_of<SEQ>(p, b, t0 + lane) == seq_of<SEQ>(p, b, t0 - 1) ? fast_exp(ncs + nlo) : 0.f;
    } else {
      const bool reach = seq_of<SEQ>(p, b, t0 + lane) == seq_of<SEQ>(p, b, t0 + nv - 1);
      f = reach ? nst * fast_exp((csL - ncs) + (loL - nlo)) : 0.f;
    }
    const float decay = WALK && carries<SEQ>(p, b, c) ? fast_exp(csL + loL) : 0.f;
    float sc[V];
    float4 av[V];
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const int t = ma.row + k * ma.step;
      const bool in = ma.on && t < nv;
      sc[k] = __shfl(f, t, 64);
      av[k] = widen<Tx>(in ? ra[k] : raw_zero<Tx>());
      if constexpr (BWD && HAS_Z) {
        const float4 z = widen<Tx>(in ? rz[k] : raw_zero<Tx>());
        av[k] = make_float4(av[k].x * z.x * sigmoid(z.x), av[k].y * z.y * sigmoid(z.y),
                            av[k].z * z.z * sigmoid(z.z), av[k].w * z.w * sigmoid(z.w));
      }
    }
    float part = 0.f;
    if (WALK && act) {
      float* dst = (BWD ? p.dstates : p.states) + state_block(p, b, c, h);
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if (on(j))
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            dst[lane_offset(eo) + e * N + 16 * j] = acc[j][e];
            if constexpr (DCS) part = fmaf(acc[j][e], nH[j][e], part);
            acc[j][e] *= decay;
          }
    }
    if constexpr (DCS) part = wave_total(part);
    __syncthreads();  // the previous chunk's products are done with s_A and s_B; its parts are in
    if constexpr (DCS)
      if (pend >= 0 && tid == 0)
        dcsl[pend * p.nslices] = pend_decay * ((s_part[0] + s_part[1]) + (s_part[2] + s_part[3]));
    park_scaled<F32>(s_A, ma, av, sc);
    map_park<Tx, F32>(s_B, kLdS, kPlaneS, mb, rb, nv);
    if (i + 1 < count) fetch(chunk_at(i + 1));
    __syncthreads();
    if constexpr (DCS) {
      if (lane == 0) s_part[wave] = part;
      pend = c;
      pend_decay = decay;
    }
    if (act)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const Frag<3> a = frag_col<3>(s_A + 32 * k * kLdS + 16 * wave, kLdS, kPlaneS);
#pragma unroll
        for (int j = 0; j < NT; ++j)
          if (on(j)) acc[j] = mma32<F32>(a, frag_col<NX>(s_B + 32 * k * kLdS + 16 * j, kLdS, kPlaneS), acc[j]);
      }
  }
  if constexpr (DCS) {
    __syncthreads();
    if (pend >= 0 && tid == 0)
      dcsl[pend * p.nslices] = pend_decay * ((s_part[0] + s_part[1]) + (s_part[2] + s_part[3]));
  }
  float* end = WALK ? (BWD ? p.dinit : p.final_states) : (BWD ? p.dstates : p.states);
  if (end != nullptr && act) {
    end += WALK ? (b * H + h) * P * N : state_block(p, b, only, h);
#pragma unroll
    for (int j = 0; j < NT; ++j)
      if (on(j))
#pragma unroll
        for (int e = 0; e < 4; ++e) end[eo + e * N + 16 * j] = acc[j][e];
  }
  mma_wait(acc);
  float spoilt = 0.f;
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) spoilt = spoil(spoilt, acc[j][e]);
  return spoilt;
}

template <typename Tx, bool HAS_Z, bool SEQ, bool BWD, bool WALK, bool EXACT, bool DCS>
__global__ void __launch_bounds__(kThreads, 3) ssd_state_kernel(const SsdParams p) {
  __shared__ StateLds<Tx> lds;
  const float spoilt = state_pass<Tx, HAS_Z, SEQ, BWD, WALK, EXACT, DCS, false>(p, lds);
  if (__builtin_expect(__syncthreads_or(spoilt != 0.f), 0))
    state_pass<Tx, HAS_Z, SEQ, BWD, WALK, EXACT, DCS, true>(p, lds);
}

// F3: the chunk's outputs, Y = (C B^T o M) (dt x) + diag(exp(cs)) C H^T + D x,
// out = Y silu(z) (and Y itself into ysave when the backward needs it).
// Grid (nchunks, nhb, batch), 8 waves: wave w computes rows t of strip w % 4
// (16 rows), its half w / 4 taking steps s of [32 half, 32 half + 32) and states
// of [64 half, 64 half + 64); the halves' Y are added where it is stored. Every
// product runs on the bf16 matrix cores in pieces (ssd_pieces.h). A wave keeps
// its part of C and of (C B^T)^T (rows s, columns t) in registers for the
// block's heads, so G = C B^T o M dt is formed and split in the registers that
// G x reads it from, and only x and H go through LDS, as pieces, staged once per
// head. Tiles above the diagonal (s > t) are never formed.
// What bounds it is memory: x, z and H in, out and y out. At
// batch 4, seqlen 2048, 80 heads, bf16 with z it takes 137 us (4.9 TB/s) against
// 308 us on the float32 matrix cores; batch 4, seqlen 1000, 24 heads, float32:
// 32 against 48 us.
// MN: 64 or 128, at least dstate. EXACT: headdim is 64 and dstate MN (128 in
// every Mamba-2 model); otherwise tiles are filled up with zeros.
// In this order everything but the last pieces of H is within an LDS instruction's
// own 64 KB offset (with H first, float32 at 64 x 128 spills 6 registers).
template <typename Tx> struct ScanLds {
  __align__(16) uint16_t X[kPieces<Tx> * kPlaneP];   // x
  __align__(16) float cs[Q], csl[Q], dt[Q], D[kSsdMaxP];
  uint8_t first[Q];                                  // first step of each step's sequence run in the chunk
  __align__(16) uint16_t H[3 * kPlaneN];             // B (Q x N), then each head's entering state H (P x N), then Y
};

// The same outputs in float32, for a block whose products in pieces left one that is
// not finite. C B^T and C H^T, whose terms all belong to their element, run on the
// float32 matrix unit with operands straight from memory; G x adds the steps that an
// output has, and no others (0 times an infinite x is NaN), a lane's four rows per x.
// C B^T and G pass through LDS over H. Batch 4, seqlen 2048, 80 heads, bf16 with z, x
// all NaN: the forward takes 1.8 ms (11.4 one element at a time; 0.33 with finite x).
template <typename Tx, bool HAS_Z, bool SEQ>
__device__ __forceinline__ void chunk_scan_plain(const SsdParams& p, ScanLds<Tx>& lds) {
  constexpr int TPB = kThreads3;
  float* const s_CB = reinterpret_cast<float*>(lds.H);   // rows t of QP floats
  float* const s_G = s_CB + Q * QP;
  static_assert(2 * Q * QP * 4 <= sizeof(lds.H), "C B^T and G fit over H");
  const int tid = second_tid(), lane = tid & 63, wave = tid >> 6;
  const int ws = wave & 3, hf = wave >> 2;        // row strip, tiles 2 hf and 2 hf + 1 of 16 columns
  const int r = lane & 15, q = lane >> 4;
  const int64_t c = blockIdx.x, b = blockIdx.z;
  const int64_t L = p.seqlen, H = p.nheads, P = p.headdim, N = p.dstate, G = p.ngroups;
  const int64_t h0 = static_cast<int64_t>(blockIdx.y) * p.hb;
  const int64_t t0 = c * Q, bcoff = ((b * L + t0) * G + h0 / (H / G)) * N;
  const int nvalid = chunk_steps(p, t0);
  const bool enter = seq_of<SEQ>(p, b, t0) == seq_of<SEQ>(p, b, t0 - 1);
  // Rows and columns that do not exist repeat the last one and are not stored.
  const int64_t crow = bcoff + static_cast<int64_t>(min(16 * ws + r, nvalid - 1)) * G * N + q;
  int col[2], first[4];
  v4f acc[2];
#pragma unroll
  for (int e = 0; e < 4; ++e) first[e] = SEQ ? lds.first[16 * ws + 4 * q + e] : 0;
  int64_t brow[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int u = 32 * hf + 16 * j + r;
    col[j] = min(u, static_cast<int>(P) - 1);
    brow[j] = bcoff + static_cast<int64_t>(min(u, nvalid - 1)) * G * N + q;
    acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
  }
  int64_t n = 0;
  do {   // dstate is at least 16
    const float a = ld<Tx>(p.C, crow + n);
#pragma unroll
    for (int j = 0; j < 2; ++j)
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, ld<Tx>(p.B, brow[j] + n), acc[j], 0, 0, 0);
    n += 4;
  } while (n < N);
  mma_wait(acc);
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) s_CB[(16 * ws + 4 * q + e) * QP + 32 * hf + 16 * j + r] = acc[j][e];
  for (int64_t h = h0; h < h0 + p.hb; ++h) {
    const int64_t row = chunk_row(p, b, h, c), xoff = ((b * L + t0) * H + h) * P;
    const float* st = p.states + state_block(p, b, c, h) + q;
    __syncthreads();  // C B^T is there, and every thread is done with the previous head's G
    if (tid < Q) {
      lds.cs[tid] = p.cs[row + tid];
      lds.csl[tid] = p.cs_lo[row + tid];
      lds.dt[tid] = p.step[row + tid];
    }
    __syncthreads();
    for (int i = tid; i < Q * Q; i += TPB) {
      const int t = i / Q, u = i % Q;
      s_G[t * QP + u] = u <= t ? s_CB[t * QP + u] * seg_exp(lds.cs, lds.csl, t, u) * lds.dt[u] : 0.f;
    }
    __syncthreads();
    acc[0] = acc[1] = v4f{0.f, 0.f, 0.f, 0.f};
    n = 0;
    do {
      const float a = ld<Tx>(p.C, crow + n);
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, st[col[j] * N + n], acc[j], 0, 0, 0);
      n += 4;
    } while (n < N);
    mma_wait(acc);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int te = 16 * ws + 4 * q + e;
      const float ecs = fast_exp(lds.cs[te] + lds.csl[te]);
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[j][e] = enter && first[e] == 0 ? acc[j][e] * ecs : 0.f;
    }
    for (int s = 0; s < min(16 * ws + 16, nvalid); ++s) {
      float x[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) x[j] = ld<Tx>(p.x, xoff + s * H * P + col[j]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int te = 16 * ws + 4 * q + e;
        const float g = s_G[te * QP + s];
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j][e] = s <= te && s >= first[e] ? fmaf(g, x[j], acc[j][e]) : acc[j][e];
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int te = 16 * ws + 4 * q + e, pp = 32 * hf + 16 * j + r;
        if (te >= nvalid || pp >= P) continue;
        const int64_t at = xoff + te * H * P + pp;
        float y = acc[j][e];
        if (p.D) y = fmaf(p.D[h * P + pp], ld<Tx>(p.x, at), y);
        if (HAS_Z) {
          if (p.ysave) mcpu::st<Tx>(p.ysave, at, y);
          const float z = ld<Tx>(p.z, at);
          y *= z * sigmoid(z);
        }
        mcpu::st<Tx>(p.out, at, y);
      }
  }
}

template <typename Tx, bool HAS_Z, bool SEQ, int MN, bool EXACT>
__global__ void __launch_bounds__(kThreads3, 4) ssd_chunk_scan_kernel(const SsdParams p) {
  constexpr int TPB = kThreads3, NT = kSsdMaxP / 16;
  constexpr int NX = kPieces<Tx>, NK = MN / 64;   // k-steps of a half over the states
  constexpr int VX = vec_x<TPB>(), VN = Q * MN / 4 / TPB;
  __shared__ ScanLds<Tx> lds;
  uint16_t* const s_H = lds.H;
  uint16_t* const s_X = lds.X;
  float (&s_cs)[Q] = lds.cs;
  float (&s_csl)[Q] = lds.csl;
  float (&s_dt)[Q] = lds.dt;
  float (&s_D)[kSsdMaxP] = lds.D;
  uint8_t (&s_first)[Q] = lds.first;
  float* s_Y = reinterpret_cast<float*>(s_H);           // per half (Q x P), rows of XP floats
  static_assert(2 * Q * XP * 4 <= sizeof(lds.H), "Y fits over H");
  // x and z load once the products are done where three pieces of C leave no
  // registers for them before (spills: a reload waits for every load in flight).
  constexpr bool kLate = NX == 3;
  const int64_t c = blockIdx.x, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ws = wave & 3, hf = wave >> 2;        // row strip, half
  const int r = lane & 15, q = lane >> 4;
  const int64_t L = p.seqlen, H = p.nheads, G = p.ngroups;
  const int64_t P = EXACT ? kSsdMaxP : p.headdim, N = EXACT ? MN : p.dstate;
  const int64_t h0 = static_cast<int64_t>(blockIdx.y) * p.hb;
  const int64_t g = h0 / (H / G);
  const int64_t t0 = c * Q;
  const int nvalid = chunk_steps(p, t0);
  const int np = static_cast<int>(P / 16);
  const TileMap<TPB, kSsdMaxP, EXACT> mp(static_cast<int>(P));
  const TileMap<TPB, MN, EXACT> mn(static_cast<int>(N));
  // C, rows t = 16 ws + r: operand fragments over this half's states
  const int64_t bcoff = ((b * L + t0) * G + g) * N;
  auto c_frag = [&](int k) {
    const int t = 16 * ws + r, n = 32 * k + 8 * q;
    return frag_mem<Tx>(static_cast<const Tx*>(p.C) + bcoff + t * G * N + n, t < nvalid && n < N);
  };
  float spoilt = 0.f;
  Frag<NX> cf[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) cf[k] = c_frag(NK * hf + k);
  {
    raw4<Tx> rb[VN];
    map_load<Tx>(rb, mn, static_cast<const Tx*>(p.B) + bcoff, G * N, nvalid);
    map_park<Tx>(s_H, kLdN, kPlaneN, mn, rb, nvalid);
  }
  if (SEQ && wave == 0) s_first[lane] = static_cast<uint8_t>(run_first<SEQ>(p, b, t0, lane));
  // the entering state reaches the chunk's first run
  const bool enter = seq_of<SEQ>(p, b, t0) == seq_of<SEQ>(p, b, t0 - 1);
  // The next head's x tile, entering state and decays load into registers
  // while this head's products run.
  raw4<Tx> rx[VX], zc[VX];
  float4 rh[VN];
  float rcs = 0.f, rcsl = 0.f, rdt = 0.f, rD = 0.f;
  auto fetch = [&](int64_t h) {
    const int64_t row = chunk_row(p, b, h, c);
    if (tid < Q) {
      const uint32_t at = lane_offset(tid);
      rcs = (p.cs + row)[at];
      rcsl = (p.cs_lo + row)[at];
      rdt = (p.step + row)[at];
      if (p.D && tid < P) rD = (p.D + h * P)[at];
    }
    map_load<float>(rh, mn, p.states + state_block(p, b, c, h), N, static_cast<int>(P));
  };
  auto fetch_x = [&](int64_t h) {
    map_load<Tx>(rx, mp, static_cast<const Tx*>(p.x) + ((b * L + t0) * H + h) * P, H * P, nvalid);
  };
  fetch(h0);
  fetch_x(h0);
  __syncthreads();
  // runs of this lane's step t = 16 ws + r (M[t][s] needs first_t <= s <= t)
  // and of the rows t = 16 ws + 4 q + e it outputs
  const int first_t = SEQ ? s_first[16 * ws + r] : 0;
  bool from[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) from[e] = enter && (!SEQ || s_first[16 * ws + 4 * q + e] == 0);
  // (C B^T)^T: rows s of tiles 2 hf and 2 hf + 1, columns t of this strip
  v4f cb[2];
  zero(cb);
  for (int k = 0; k < 2 * NK; ++k) {
    const Frag<NX> ck = c_frag(k);
#pragma unroll
    for (int u = 0; u < 2; ++u)
      if (2 * hf + u <= ws)
        cb[u] = mma32(frag_row<NX>(s_H + 16 * (2 * hf + u) * kLdN + 32 * k, kLdN, kPlaneN), ck, cb[u]);
  }
  for (int i = 0; i < p.hb; ++i) {
    int64_t h = h0 + i;
    asm volatile("" : "+s"(h));
    const int64_t xoff = ((b * L + t0) * H + h) * P;
    __syncthreads();  // every wave is done with s_H (B, Y), s_X and s_cs
    if (tid < Q) {
      s_cs[tid] = rcs;
      s_csl[tid] = rcsl;
      s_dt[tid] = rdt;
      s_D[tid] = rD;
    }
    map_park<Tx>(s_X, kLdP, kPlaneP, mp, rx, nvalid);
    map_park<float>(s_H, kLdN, kPlaneN, mn, rh, static_cast<int>(P));
    __syncthreads();
    if (HAS_Z && !kLate) map_load<Tx>(zc, mp, static_cast<const Tx*>(p.z) + xoff, H * P, nvalid);
    if (i + 1 < p.hb) {
      fetch(h + 1);
      if (!kLate) fetch_x(h + 1);
    }
    v4f y[NT];
    zero(y);
    // C H^T over this half's states
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (EXACT || j < np)
          y[j] = mma32(cf[k], frag_row<3>(s_H + 16 * j * kLdN + 32 * (NK * hf + k), kLdN, kPlaneN), y[j]);
        if (NX == 3) __builtin_amdgcn_sched_barrier(0);  // one operand at a time: registers
      }
    float ecs[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int te = 16 * ws + 4 * q + e;
      ecs[e] = from[e] ? fast_exp(s_cs[te] + s_csl[te]) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) y[j][e] *= ecs[e];
    // G x over this half's steps s
    if (2 * hf <= ws) {
      const int t = 16 * ws + r;
      const float cst = s_cs[t], cslt = s_csl[t];
      v4f gt[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int s0 = 32 * hf + 16 * u + 4 * q;
        const float4 c4 = *reinterpret_cast<const float4*>(&s_cs[s0]);
        const float4 l4 = *reinterpret_cast<const float4*>(&s_csl[s0]);
        const float4 d4 = *reinterpret_cast<const float4*>(&s_dt[s0]);
        const float cv[4] = {c4.x, c4.y, c4.z, c4.w}, lv[4] = {l4.x, l4.y, l4.z, l4.w},
                    dv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int sx = s0 + e;
          const float m = cb[u][e] * fast_exp((cst - cv[e]) + (cslt - lv[e])) * dv[e];
          gt[u][e] = (sx <= t && sx >= first_t) ? m : 0.f;
        }
      }
      const Frag<3> ga = frag_acc<3>(gt[0], gt[1]);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (EXACT || j < np) y[j] = mma32(ga, frag_col<NX>(s_X + 32 * hf * kLdP + 16 * j, kLdP, kPlaneP), y[j]);
        if (NX == 3) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (kLate) {
      __builtin_amdgcn_sched_barrier(0);
      if (HAS_Z) map_load<Tx>(zc, mp, static_cast<const Tx*>(p.z) + xoff, H * P, nvalid);
      if (i + 1 < p.hb) fetch_x(h + 1);
    }
    __syncthreads();  // every wave is done reading s_H
    // Y (float32) over H, then out = (Y + D x) silu(z) four elements at a time.
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        if (EXACT || j < np) s_Y[(Q * hf + 16 * ws + 4 * q + e) * XP + 16 * j + r] = y[j][e];
    __syncthreads();
    {
#pragma unroll
      for (int k = 0; k < VX; ++k) {
        const int to = mp.row + k * mp.step, pp = mp.col;
        if (!mp.on || to >= nvalid) continue;
        const uint32_t at = lane_offset(to * static_cast<uint32_t>(H * P) + pp);
        const float4 ya = *reinterpret_cast<const float4*>(&s_Y[to * XP + pp]);
        const float4 yb = *reinterpret_cast<const float4*>(&s_Y[(Q + to) * XP + pp]);
        float o[4] = {ya.x + yb.x, ya.y + yb.y, ya.z + yb.z, ya.w + yb.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) spoilt = spoil(spoilt, o[u]);
        if (p.D) {
          const float4 d = *reinterpret_cast<const float4*>(&s_D[pp]), x4 = pieces4<NX>(s_X + to * kLdP + pp, kPlaneP);
          o[0] = fmaf(d.x, x4.x, o[0]);
          o[1] = fmaf(d.y, x4.y, o[1]);
          o[2] = fmaf(d.z, x4.z, o[2]);
          o[3] = fmaf(d.w, x4.w, o[3]);
        }
        if (HAS_Z) {
          if (p.ysave) st4<Tx>(static_cast<Tx*>(p.ysave) + xoff + at, make_float4(o[0], o[1], o[2], o[3]));
          const float4 z4 = widen<Tx>(zc[k]);
          const float zx[4] = {z4.x, z4.y, z4.z, z4.w};
#pragma unroll
          for (int u = 0; u < 4; ++u) o[u] *= zx[u] * sigmoid(zx[u]);
        }
        st4<Tx>(static_cast<Tx*>(p.out) + xoff + at, make_float4(o[0], o[1], o[2], o[3]));
      }
    }
  }
  if (__builtin_expect(__syncthreads_or(spoilt != 0.f), 0) && p.apart) chunk_scan_plain<Tx, HAS_Z, SEQ>(p, lds);
}

// K2: walks the chunks from the last: dH^out_c (gradient of the state leaving
// chunk c) replaces E_c in dstates, dH^in_c = exp(cs_L) dH^out_c + E_c
// carries on, and <dH^out_c, exp(cs_L) H_c> (this slice's share of dL/dcs_L)
// goes to dcsL. The gradient of the initial state is what is left after
// chunk 0. Grid (nslices, nheads, batch). The next chunk's loads issue before
// this chunk's store. DCS: false where the chunk-gradient kernel forms dcsL.
template <bool SEQ, bool DCS>
__global__ void __launch_bounds__(kThreads) ssd_bwd_pass_kernel(const SsdParams p) {
  __shared__ float s_part[kThreads / 64];
  const int64_t PN = p.headdim * p.dstate, H = p.nheads;
  const int64_t e = blockIdx.x * static_cast<int64_t>(kThreads) + threadIdx.x;
  const int64_t h = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool ok = e < PN;
  float run = (ok && p.dfinal) ? p.dfinal[(b * H + h) * PN + e] : 0.f;
  const int64_t base = state_block(p, b, 0, h) + (ok ? e : 0);
  const int64_t cstride = H * PN;
  const float* csl = p.cs + chunk_row(p, b, h, 0) + (Q - 1);
  float* dcsl = p.dcsL + (chunk_row(p, b, h, 0) / Q) * p.nslices + blockIdx.x;
  const int64_t last = p.nchunks - 1;
  float ec = ok ? p.dstates[base + last * cstride] : 0.f;
  float hin = DCS && ok ? p.states[base + last * cstride] : 0.f;
  float dl = csl[last * Q];
  for (int64_t c = last; c >= 0; --c) {
    const float ecc = ec, hc = hin, d = carries<SEQ>(p, b, c) ? fast_exp(dl) : 0.f;
    if (c > 0) {
      ec = ok ? p.dstates[base + (c - 1) * cstride] : 0.f;
      if (DCS) hin = ok ? p.states[base + (c - 1) * cstride] : 0.f;
      dl = csl[(c - 1) * Q];
    }
    if (ok) p.dstates[base + c * cstride] = run;
    if constexpr (DCS) {
      const float part = wave_total(run * d * hc);
      if (lane == 0) s_part[wave] = part;
      __syncthreads();
      if (threadIdx.x == 0) dcsl[c * p.nslices] = (s_part[0] + s_part[1]) + (s_part[2] + s_part[3]);
      __syncthreads();
    }
    run = fmaf(d, run, ecc);
  }
  if (ok && p.dinit) p.dinit[(b * H + h) * PN + e] = run;
}

// K3: every gradient of a chunk, for each head of the block. Grid (nchunks,
// nhb, batch), 8 waves: wave w owns rows [16 (w % 4), 16 (w % 4) + 16) of
// every Q-row product and half h = w / 4 of its column tiles (Q columns:
// tiles 2h, 2h + 1; headdim columns: the first or second half of the tiles;
// state columns: tiles 2h, 2h + 1 of each 64-state group). Two waves per SIMD
// hide each other's LDS and memory latency. Row sums over columns are
// combined across the two halves through LDS. dB and dC of the block's heads
// stay in accumulators and are written once, as the block's partial sums.
// In this order the tiles that rows are read from lie within an LDS instruction's own
// 64 KB offset of each other (with B and C first, 9 to 56 registers spill).
struct BwdF32Lds {
  __align__(16) float colp[16][Q];    // column sums of dG o G, per (row strip, lane quarter)
  float dD[16][kSsdMaxP];
  float half[2][4][Q];                // per column half: sum_s R, sum_n C.., sum_n B~.., sum_p ..
  float cs[Q], csl[Q], dt[Q], w[Q], ecs[Q], dcs[Q];
  float tot[8], wa[8], wb[8];
  __align__(4) uint8_t first[Q];      // first step of each step's sequence run in the chunk
  __align__(16) float X[Q][XP], dY[Q][XP];
  __align__(16) float U[Q][QP];       // G = C B^T o M, then dH^out (P x 64-state group)
  __align__(16) float V[Q][QP];       // dCB, then H (P x 64-state group), then dx
  __align__(16) float C[Q][NP], B[Q][NP];
};

// DCS: <dH^out, exp(cs_L) H_c> comes from the states' kernels as dcsL; otherwise it is
// formed here, from the tiles that are read anyway.
template <typename Tx, bool HAS_Z, bool SEQ, bool DCS>
__device__ __forceinline__ void bwd_chunk_f32(const SsdParams& p, BwdF32Lds& lds) {
  constexpr int TPB = kThreads3;
  constexpr int VX = vec_x<TPB>(), VN = vec_n<TPB>();
  float (&s_C)[Q][NP] = lds.C;
  float (&s_B)[Q][NP] = lds.B;
  float (&s_X)[Q][XP] = lds.X;
  float (&s_dY)[Q][XP] = lds.dY;
  float (&s_U)[Q][QP] = lds.U;
  float (&s_V)[Q][QP] = lds.V;
  float (&s_colp)[16][Q] = lds.colp;
  float (&s_dD)[16][kSsdMaxP] = lds.dD;
  float (&s_half)[2][4][Q] = lds.half;
  float (&s_cs)[Q] = lds.cs;
  float (&s_csl)[Q] = lds.csl;
  float (&s_dt)[Q] = lds.dt;
  float (&s_w)[Q] = lds.w;
  float (&s_ecs)[Q] = lds.ecs;
  float (&s_dcs)[Q] = lds.dcs;
  float (&s_tot)[8] = lds.tot;
  float (&s_wa)[8] = lds.wa;
  float (&s_wb)[8] = lds.wb;
  uint8_t (&s_first)[Q] = lds.first;
  const int64_t c = blockIdx.x, b = blockIdx.z;
  const int tid = DCS ? threadIdx.x : second_tid(), lane = tid & 63, wave = tid >> 6;
  const int ws = wave & 3, hf = wave >> 2;        // row strip, column half
  const int r = lane & 15, q = lane >> 4;
  const int64_t L = p.seqlen, H = p.nheads, P = p.headdim, N = p.dstate, G = p.ngroups;
  const int64_t h0 = static_cast<int64_t>(blockIdx.y) * p.hb;
  const int64_t g = h0 / (H / G);
  const int64_t t0 = c * Q;
  const int nvalid = chunk_steps(p, t0);
  const int np = static_cast<int>(P / 16), nn = static_cast<int>(N / 16);
  // headdim tiles of this wave: [p0, p0 + npw)
  const int pa = (np + 1) / 2;
  const int p0 = hf ? pa : 0, npw = hf ? np - pa : pa;
  // state tiles of this wave in the 64-state group starting at tile 4 grp
  auto ntw = [&](int grp) {
    const int nt = nn - 4 * grp < 4 ? nn - 4 * grp : 4;
    const int k = nt - 2 * hf;
    return k < 0 ? 0 : (k > 2 ? 2 : k);
  };
  {
    const int64_t off = ((b * L + t0) * G + g) * N;
    stage<Tx, VN, TPB>(&s_C[0][0], NP, static_cast<const Tx*>(p.C) + off, G * N, Q, nvalid, static_cast<int>(N));
    stage<Tx, VN, TPB>(&s_B[0][0], NP, static_cast<const Tx*>(p.B) + off, G * N, Q, nvalid, static_cast<int>(N));
  }
  // Packed sequences: step tid reaches the chunk's end state (w) and reads the
  // entering state (exp(cs)) only within one sequence.
  bool reach = true, from = true;
  if (wave == 0) {
    if (SEQ) s_first[lane] = static_cast<uint8_t>(run_first<SEQ>(p, b, t0, lane));
    const int32_t id = seq_of<SEQ>(p, b, t0 + lane);
    reach = id == seq_of<SEQ>(p, b, t0 + nvalid - 1);
    from = id == seq_of<SEQ>(p, b, t0 - 1);
  }
  __syncthreads();
  // runs of this thread's rows t = 16 ws + 4 q + e: M[t][s] needs first_t <= s <= t
  const uint32_t firsts = SEQ ? *reinterpret_cast<const uint32_t*>(&s_first[16 * ws + 4 * q]) : 0u;
  // C B^T, rows t of this strip, Q-column tiles 2 hf, 2 hf + 1
  v4f cb[2];
  zero(cb);
  mma(cb, 2, &s_C[16 * ws][0], NP, 1, &s_B[32 * hf][0], 1, NP, static_cast<int>(N));
  v4f dBa[2][2], dCa[2][2];   // [64-state group][tile of this wave]
#pragma unroll
  for (int grp = 0; grp < 2; ++grp) {
    zero(dBa[grp]);
    zero(dCa[grp]);
  }
  // The next head's x, dout, z and ysave tiles and decays load into
  // registers while this head's products run.
  raw4<Tx> rx[VX];
  DyTiles<Tx, HAS_Z, TPB> rdy;
  float rcs = 0.f, rcsl = 0.f, rdt = 0.f, rcsL = 0.f, rcslL = 0.f;
  auto fetch = [&](int64_t h) {
    const int64_t row = chunk_row(p, b, h, c);
    const int64_t xoff = ((b * L + t0) * H + h) * P;
    if (tid < Q) {
      rcs = p.cs[row + tid];
      rcsl = p.cs_lo[row + tid];
      rdt = p.step[row + tid];
      rcsL = p.cs[row + Q - 1];
      rcslL = p.cs_lo[row + Q - 1];
    }
    tile_load<Tx, VX, TPB>(rx, static_cast<const Tx*>(p.x) + xoff, H * P, Q, nvalid, static_cast<int>(P));
    rdy.load(p, xoff, H * P, nvalid, static_cast<int>(P));
  };
  fetch(h0);
  for (int i = 0; i < p.hb; ++i) {
    const int64_t h = h0 + i;
    const int64_t xoff = ((b * L + t0) * H + h) * P;
    const int64_t row = chunk_row(p, b, h, c);
    const int64_t sb = state_block(p, b, c, h);
    __syncthreads();  // every wave is done with the previous head's tiles
    if (tid < Q) {
      s_cs[tid] = rcs;
      s_csl[tid] = rcsl;
      s_dt[tid] = rdt;
      s_w[tid] = reach ? fast_exp((rcsL - rcs) + (rcslL - rcsl)) : 0.f;
      s_ecs[tid] = from ? fast_exp(rcs + rcsl) : 0.f;
    }
    tile_store<Tx, VX, TPB>(&s_X[0][0], XP, rx, Q, static_cast<int>(P));
    rdy.store(&s_dY[0][0], XP, p, xoff, H * P, nvalid, static_cast<int>(P));
    __syncthreads();
    if (i + 1 < p.hb) fetch(h + 1);
    // dGraw = dY x^T (rows t of this strip, this half's columns s); with M and
    // dt: G = CB o M, dCB = dt_s dGraw o M, R = dCB o CB (= dG o G). Row sums
    // of R per half and column sums per strip through LDS, in a fixed order.
    float rowsum[4] = {0.f, 0.f, 0.f, 0.f};
    {
      v4f dg[2];
      zero(dg);
      mma(dg, 2, &s_dY[16 * ws][0], XP, 1, &s_X[32 * hf][0], 1, XP, static_cast<int>(P));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float colsum = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 16 * ws + 4 * q + e, s = 32 * hf + 16 * j + r;
          const float m = (s <= t && s >= static_cast<int>((firsts >> (8 * e)) & 0xff)) ? seg_exp(s_cs, s_csl, t, s)
                                                                                     : 0.f;
          const float dcb = dg[j][e] * s_dt[s] * m;
          const float rv = dcb * cb[j][e];
          s_U[t][s] = cb[j][e] * m;
          s_V[t][s] = dcb;
          rowsum[e] += rv;
          colsum += rv;
        }
        s_colp[4 * ws + q][32 * hf + 16 * j + r] = colsum;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) rowsum[e] = row_allreduce16(rowsum[e]);
    if (r < 4) {
      float mine = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r == e) mine = rowsum[e];
      s_half[hf][0][16 * ws + 4 * q + r] = mine;
    }
    __syncthreads();
    // dcs_intra[t] = sum_s R[t][s] - sum_s R[s][t] (half 0's quarter lanes r < 4 own row t).
    if (hf == 0 && r < 4) {
      const int t = 16 * ws + 4 * q + r;
      float col = 0.f;
      for (int k = 0; k < 16; ++k) col += s_colp[k][t];
      s_dcs[t] = (s_half[0][0][t] + s_half[1][0][t]) - col;
    }
    // d(dt x)[s][p] = sum_t G[t][s] dY[t][p] (rows s of this strip, this half's headdim tiles).
    v4f dxa[2];
    zero(dxa);
    mma(dxa, npw, &s_U[0][16 * ws], 1, QP, &s_dY[0][16 * p0], XP, 1, Q);
    // dH^out and H of a 64-state group into registers, parked in s_U / s_V
    // once the products reading them are done: group 0's load under the dC /
    // dB products, group 1's under group 0's state products.
    float4 su[VX], sv[VX];
    auto load_states = [&](int grp) {
      const int n0 = 64 * grp;
      const int nw = static_cast<int>(N - n0 < 64 ? N - n0 : 64);
      tile_load<float, VX, TPB>(su, p.dstates + sb + n0, N, static_cast<int>(P), static_cast<int>(P), nw);
      tile_load<float, VX, TPB>(sv, p.states + sb + n0, N, static_cast<int>(P), static_cast<int>(P), nw);
    };
    load_states(0);
    // dC[t][n] += sum_s dCB[t][s] B[s][n] ; dB[s][n] += sum_t dCB[t][s] C[t][n] (this wave's state tiles).
#pragma unroll
    for (int grp = 0; grp < 2; ++grp) {
      const int nt = ntw(grp);
      const int col = 64 * grp + 32 * hf;
      mma(dCa[grp], nt, &s_V[16 * ws][0], QP, 1, &s_B[0][col], NP, 1, Q);
      mma(dBa[grp], nt, &s_V[0][16 * ws], 1, QP, &s_C[0][col], NP, 1, Q);
    }
    // State terms, over 64-state groups of dH^out and H.
    float a_row[4] = {0.f, 0.f, 0.f, 0.f};  // sum_n C[t][n] exp(cs_t) (dY H)[t][n]
    float b_row[4] = {0.f, 0.f, 0.f, 0.f};  // sum_n w_s B[s][n] ((dt x) dH)[s][n]
    const float dt_row = s_dt[16 * ws + r], w_row = s_w[16 * ws + r];
    float dh = 0.f;                         // this thread's part of <dH^out, H_c>
#pragma unroll
    for (int grp = 0; grp < kSsdMaxN / 64; ++grp) {
      const int n0 = 64 * grp;
      if (n0 >= N) break;
      const int nw = static_cast<int>(N - n0 < 64 ? N - n0 : 64);
      const int nt = ntw(grp);
      if (!DCS)
#pragma unroll
        for (int k = 0; k < VX; ++k)
          dh += fmaf(su[k].x, sv[k].x, su[k].y * sv[k].y) + fmaf(su[k].z, sv[k].z, su[k].w * sv[k].w);
      __syncthreads();  // every wave is done reading s_U / s_V
      tile_store<float, VX, TPB>(&s_U[0][0], QP, su, static_cast<int>(P), nw);
      tile_store<float, VX, TPB>(&s_V[0][0], QP, sv, static_cast<int>(P), nw);
      __syncthreads();
      if (n0 + 64 < N) load_states(grp + 1);
      v4f tv[2], yh[2];
      zero(tv);
      zero(yh);
      // tv[s][n] = sum_p dt_s x[s][p] dH[p][n] ; yh[t][n] = sum_p dY[t][p] H[p][n]
      mma<2, true>(tv, nt, &s_X[16 * ws][0], XP, 1, &s_U[0][32 * hf], QP, 1, static_cast<int>(P), dt_row);
      mma(yh, nt, &s_dY[16 * ws][0], XP, 1, &s_V[0][32 * hf], QP, 1, static_cast<int>(P));
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j >= nt) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int t = 16 * ws + 4 * q + e;
          const int n = n0 + 32 * hf + 16 * j + r;
          const float wt = s_w[t] * tv[j][e];
          const float ys = s_ecs[t] * yh[j][e];
          dBa[grp][j][e] += wt;
          dCa[grp][j][e] += ys;
          b_row[e] = fmaf(s_B[t][n], wt, b_row[e]);
          a_row[e] = fmaf(s_C[t][n], ys, a_row[e]);
        }
      }
      // d(dt x)[s][p] += sum_n w_s B[s][n] dH[p][n] (all states of the group, this half's headdim tiles)
      mma<2, true>(dxa, npw, &s_B[16 * ws][n0], NP, 1, &s_U[16 * p0][0], 1, QP, nw, w_row);
    }
    // sum_p d(dt x) x (for dstep) and dD partial sums over this half's headdim tiles.
    float c_row[4] = {0.f, 0.f, 0.f, 0.f};
    float dD_col[2] = {0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int s = 16 * ws + 4 * q + e;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j >= npw) continue;
        const int pp = 16 * (p0 + j) + r;
        const float xv = s_X[s][pp];
        c_row[e] = fmaf(dxa[j][e], xv, c_row[e]);
        dD_col[j] = fmaf(s_dY[s][pp], xv, dD_col[j]);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a_row[e] = row_allreduce16(a_row[e]);
      b_row[e] = row_allreduce16(b_row[e]);
      c_row[e] = row_allreduce16(c_row[e]);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (j < npw) s_dD[4 * ws + q][16 * (p0 + j) + r] = dD_col[j];
    // the chunk's sum of b_row is the cs_L term of the states' dependence on w
    float bsum = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) bsum += b_row[e];  // this quarter's 4 rows, alike in every lane of the row
    bsum = wave_total(r == 0 ? bsum : 0.f);
    if (!DCS) bsum = fmaf(s_ecs[Q - 1], wave_total(dh), bsum);
    if (lane == 0) s_tot[wave] = bsum;
    if (r < 4) {
      float av = 0.f, bv = 0.f, cv = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (r == e) {
          av = a_row[e];
          bv = b_row[e];
          cv = c_row[e];
        }
      const int t = 16 * ws + 4 * q + r;
      s_half[hf][1][t] = av;
      s_half[hf][2][t] = bv;
      s_half[hf][3][t] = cv;
    }
    __syncthreads();  // every wave is done reading s_U / s_V; halves' row sums are in
    // dx = dt d(dt x) + D dY into s_V, stored below four elements at a time
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int s = 16 * ws + 4 * q + e;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j >= npw) continue;
        const int pp = 16 * (p0 + j) + r;
        float dxv = dxa[j][e] * s_dt[s];
        if (p.D) dxv = fmaf(p.D[h * P + pp], s_dY[s][pp], dxv);
        s_V[s][pp] = dxv;
      }
    }
    if (wave == 0) {
      // dcs with the state terms, the cs_L terms, then da = suffix sums over the chunk
      float v = s_dcs[lane] + (s_half[0][1][lane] + s_half[1][1][lane]) -
                (s_half[0][2][lane] + s_half[1][2][lane]);
      if (lane == Q - 1) {
        float l = ((s_tot[0] + s_tot[1]) + (s_tot[2] + s_tot[3])) + ((s_tot[4] + s_tot[5]) + (s_tot[6] + s_tot[7]));
        if (DCS) {
          const float* dl = p.dcsL + (row / Q) * p.nslices;
          for (int64_t k = 0; k < p.nslices; ++k) l += dl[k];
        }
        v += l;
      }
      s_dcs[lane] = wave_suffix_sum(v);
    }
    __syncthreads();
    // dstep = sum_p d(dt x) x + da A, then through softplus / clamp / bias (half 0's quarter lanes).
    float ddt_raw = 0.f, dA_term = 0.f;
    if (hf == 0 && r < 4) {
      const int t = 16 * ws + 4 * q + r;
      if (t < nvalid) {
        float gfac;
        ssd_step(p, b, t0 + t, h, &gfac);
        const float da = s_dcs[t];
        const float c_all = s_half[0][3][t] + s_half[1][3][t];
        ddt_raw = fmaf(da, p.A[h], c_all) * gfac;
        dA_term = da * s_dt[t];
        p.ddt[(b * L + t0 + t) * H + h] = ddt_raw;
      }
    }
    {
      const int nv = np * 4;
      const float inv = 1.0f / static_cast<float>(nv);
#pragma unroll
      for (int k = 0; k < VX; ++k) {
        const int v = tid + k * TPB;
        if (v >= Q * nv) continue;
        const int s = tile_row(v, inv);
        if (s >= nvalid) continue;
        const int pp = (v - s * nv) << 2;
        st4<Tx>(static_cast<Tx*>(p.dx) + xoff + s * H * P + pp, *reinterpret_cast<const float4*>(&s_V[s][pp]));
      }
    }
    const float wa = wave_total(dA_term), wb = wave_total(ddt_raw);
    if (lane == 0) {
      s_wa[wave] = wa;
      s_wb[wave] = wb;
    }
    __syncthreads();
    const int64_t prt = (b * p.nchunks + c) * H + h;
    if (tid == 0) {
      p.dA_part[prt] = ((s_wa[0] + s_wa[1]) + (s_wa[2] + s_wa[3])) + ((s_wa[4] + s_wa[5]) + (s_wa[6] + s_wa[7]));
      p.dbias_part[prt] = ((s_wb[0] + s_wb[1]) + (s_wb[2] + s_wb[3])) + ((s_wb[4] + s_wb[5]) + (s_wb[6] + s_wb[7]));
    }
    if (tid < P) {
      float v = 0.f;
      for (int k = 0; k < 16; ++k) v += s_dD[k][tid];
      p.dD_part[prt * P + tid] = v;
    }
  }
  // the block's dB and dC partial sums (this wave's rows and state tiles)
  const int64_t hbk = blockIdx.y;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int t = 16 * ws + 4 * q + e;
    if (t >= nvalid) continue;
    const int64_t at = ((b * L + t0 + t) * p.nhb + hbk) * N;
#pragma unroll
    for (int grp = 0; grp < 2; ++grp) {
      const int nt = ntw(grp);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (j >= nt) continue;
        const int n = 64 * grp + 32 * hf + 16 * j + r;
        p.dC_part[at + n] = dCa[grp][j][e];
        p.dB_part[at + n] = dBa[grp][j][e];
      }
    }
  }
}

template <typename Tx, bool HAS_Z, bool SEQ>
__global__ void __launch_bounds__(kThreads3, 2) ssd_bwd_chunk_kernel(const SsdParams p) {
  __shared__ BwdF32Lds lds;
  bwd_chunk_f32<Tx, HAS_Z, SEQ, true>(p, lds);
}

// K3 for bf16 storage, headdim P 32 or 64 and dstate N 64 or 128: the same
// gradients with every product on the bf16 matrix cores in pieces
// (ssd_pieces.h): x, B and C are one piece as stored; dY, G, dCB, dH^out and H
// three. Waves 0-3 ("s") own 16 rows s each of d(dt x) and dB, waves 4-7 ("t")
// 16 rows t of dC:
//   - an s-wave forms C B^T and dG as (rows t, columns s), a t-wave as (rows s,
//     columns t), each over its own 16 columns, so what it makes of them (G, dCB)
//     is the operand of its next products where it stands, in registers, and
//     neither goes through LDS; tiles above the diagonal are never formed;
//   - products over rows of an LDS tile read it transposed (frag_col), so each
//     tile is stored once.
// dX = d(dt x), and its part W from the state, then pass through LDS once, where
// all threads take c = <x, dX>, b = dt <x, W> (the sum over states of B (dt x)
// dH^out) and dx, and one wave closes the chunk's decay gradients.
// What bounds it: the LDS holds one workgroup per CU, so its phases (park, chunk
// products, state groups, output) run one after the other with two waves per
// SIMD. The sizes are template arguments: with every loop bound known the
// prefetched tiles stay in registers (run-time bounds spill them, and a reload
// waits for every load in flight). Batch 4, seqlen 2048, 80 heads with z, forward
// and backward, these products against the float32 ones below: P 64, N 128 K3
// alone 485 against 971 us; the whole call at 64 x 64 724 against 1073,
// 32 x 128 715 against 1161, 32 x 64 541 against 833.
constexpr int kLdT = kSsdMaxN + 16;   // rows of B and C here, read mostly transposed: eight rows on 64 banks

// The small arrays first: with them last, beyond an LDS instruction's own 64 KB
// offset, P 64, N 128 spills 5 registers.
struct BwdChunkLds {
  __align__(16) float cs[Q], csl[Q], dt[Q], w[Q], ecs[Q];
  float row[Q], col[Q], a[Q], b[Q], c[Q], dh[8];
  float dD[8][kSsdMaxP];
  uint8_t first[Q], last[Q];                // ends of each step's sequence run in the chunk
  __align__(16) uint16_t X[kPlaneP], dY[3 * kPlaneP];
  __align__(16) uint16_t st[6 * kPlaneP];   // dH^out, then H, of a 64-state group; then dX and W
  __align__(16) uint16_t C[Q * kLdT], B[Q * kLdT];
};

// The waves of one kind, s (SW) or t: the head loop. The two kinds reach their
// barriers at different places in the code: the hardware counts arrivals, so both must
// pass the same number of them, in the same order, and nothing here may leave the loop
// early or skip one. Returns 0 if the sums that every factor of the block
// enters (C B^T, dB or dC, and the decay's gradient) are finite.
template <bool HAS_Z, bool SEQ, int P, int N, bool SW>
__device__ __forceinline__ float bwd_chunk_waves(const SsdParams& p, BwdChunkLds& lds) {
  constexpr int TPB = kThreads3, VX = Q * P / 4 / TPB;
  constexpr int PT = P / 16, PK = P / 32;                  // headdim tiles, and products' terms over it
  constexpr int NG = N / 64, VS = P * 64 / 4 / TPB;        // 64-state groups, and a thread's entries of one
  constexpr bool sw = SW;
  uint16_t (&s_X)[kPlaneP] = lds.X;
  uint16_t (&s_dY)[3 * kPlaneP] = lds.dY;
  float (&s_cs)[Q] = lds.cs;
  float (&s_csl)[Q] = lds.csl;
  float (&s_dt)[Q] = lds.dt;
  float (&s_w)[Q] = lds.w;
  float (&s_ecs)[Q] = lds.ecs;
  uint16_t* const s_dH = lds.st;
  uint16_t* const s_H = lds.st + 3 * kPlaneP;
  float* const s_dX = reinterpret_cast<float*>(lds.st);    // rows of XP floats
  float* const s_W = s_dX + Q * XP;
  static_assert(2 * Q * XP * 4 <= sizeof(lds.st), "dX and W fit over the states");
  const int64_t c = blockIdx.x, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int own = 16 * (wave & 3);                       // its strip's first row
  const int r = lane & 15, q = lane >> 4;
  const int64_t L = p.seqlen, H = p.nheads;
  const int64_t h0 = static_cast<int64_t>(blockIdx.y) * p.hb;
  const int64_t t0 = c * Q;
  const int nvalid = chunk_steps(p, t0);
  const TileMap<TPB, P, true> mp(P);
  const TileMap<TPB, 64, true> ms(64);
  // The strip's own matrix and the other: B and C for an s-wave, C and B for a t-wave.
  const uint16_t* const s_own = (sw ? lds.B : lds.C) + own * kLdT;
  const uint16_t* const s_oth = sw ? lds.C : lds.B;
  // C at this t-wave's dC elements, (rows t = own + 4 q + e, states 16 j + r), in pairs over j
  uint32_t cd[4][N / 32];
  // Wave 4 (a t-wave: those have registers to spare) keeps the chunk's per-step
  // values, lane t step t, and closes their gradients; wave 5 sums dD.
  const bool keeper = !SW && wave == 4;
  // Packed sequences: step `lane` reaches the chunk's end state (w) and reads the
  // entering state (exp(cs)) only within one sequence.
  bool reach = true, from = true;
  if (keeper) {
    if (SEQ) {
      const bool starts = lane == 0 || seq_of<SEQ>(p, b, t0 + lane) != seq_of<SEQ>(p, b, t0 + lane - 1);
      const unsigned long long begin = __ballot(starts);
      const unsigned long long later = lane == 63 ? 0ull : begin & (~0ull << (lane + 1));
      lds.first[lane] = static_cast<uint8_t>(run_first<SEQ>(p, b, t0, lane));
      lds.last[lane] = static_cast<uint8_t>(later ? __builtin_ctzll(later) - 1 : Q - 1);
    }
    const int32_t id = seq_of<SEQ>(p, b, t0 + lane);
    reach = id == seq_of<SEQ>(p, b, t0 + nvalid - 1);
    from = id == seq_of<SEQ>(p, b, t0 - 1);
  }
  // The next head's tiles and decays, and the next states, load into registers
  // while the current products run.
  raw4<bf16> rx[VX], rgo[VX], rz[VX], ry[VX];
  float4 su[VS], sv[VS];
  float rcs = 0.f, rcsl = 0.f, rdt = 0.f, rpre = 0.f;
  auto fetch = [&](int64_t h) {
    const int64_t row = chunk_row(p, b, h, c);
    const int64_t xoff = ((b * L + t0) * H + h) * P;
    if (keeper) {
      const uint32_t at = lane_offset(lane);
      rcs = (p.cs + row)[at];
      rcsl = (p.cs_lo + row)[at];
      rdt = (p.step + row)[at];
      rpre = (p.dt + (b * L + t0) * H + h)[lane_offset((lane < nvalid ? lane : 0) * static_cast<uint32_t>(H))];
    }
    map_load<bf16>(rx, mp, static_cast<const bf16*>(p.x) + xoff, H * P, nvalid);
    map_load<bf16>(rgo, mp, static_cast<const bf16*>(p.dout) + xoff, H * P, nvalid);
    if (HAS_Z) {
      map_load<bf16>(rz, mp, static_cast<const bf16*>(p.z) + xoff, H * P, nvalid);
      map_load<bf16>(ry, mp, static_cast<const bf16*>(p.ysave) + xoff, H * P, nvalid);
    }
  };
  auto fetch_states = [&](int64_t h, int grp) {
    const int64_t sb = state_block(p, b, c, h) + 64 * grp;
    map_load<float>(su, ms, p.dstates + sb, N, P);
    map_load<float>(sv, ms, p.states + sb, N, P);
  };
  auto park_states = [&](float& dh) {
    float v = 0.f;
#pragma unroll
    for (int k = 0; k < VS; ++k)
      v += fmaf(su[k].x, sv[k].x, su[k].y * sv[k].y) + fmaf(su[k].z, sv[k].z, su[k].w * sv[k].w);
    v = wave_total(v);
    dh += __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
    map_park<float>(s_dH, kLdP, kPlaneP, ms, su, P);
    map_park<float>(s_H, kLdP, kPlaneP, ms, sv, P);
  };
  fetch(h0);
  fetch_states(h0, 0);
  __syncthreads();
  // The run bound of this lane's own step: t <= last_s for an s-wave's column s
  // (with t >= s), s >= first_t for a t-wave's column t (with s <= t).
  const int step_own = own + r;
  const int bound = SEQ ? (sw ? lds.last[step_own] : lds.first[step_own]) : (sw ? Q - 1 : 0);
  // C B^T: rows = the other's steps (tile u), columns = own steps
  v4f cb[4];
  zero(cb);
#pragma unroll
  for (int k = 0; k < N / 32; ++k) {
    const Frag<1> o = frag_row<1>(s_own + 32 * k, kLdT, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) cb[u] = mma32(frag_row<1>(s_oth + 16 * u * kLdT + 32 * k, kLdT, 0), o, cb[u]);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (!sw)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int j = 0; j < N / 32; ++j) {
        const uint16_t* at = s_own + (4 * q + e) * kLdT + 32 * j + r;
        cd[e][j] = static_cast<uint32_t>(at[0]) | (static_cast<uint32_t>(at[16]) << 16);
      }
  float spoilt = 0.f;
  v4f acc[N / 16];   // dB (s-wave) or dC (t-wave): rows own + 4 q + e, states 16 j + r
  zero(acc);
  for (int i = 0; i < p.hb; ++i) {
    int64_t h = h0 + i;
    asm volatile("" : "+s"(h));
    const int64_t xoff = ((b * L + t0) * H + h) * P;
    __syncthreads();  // every wave is done with the previous head's tiles
    const float pre = rpre;   // the keeper: this head's raw steps
    float dh = 0.f;           // this wave's part of <dH^out, H_c>, uniform
    if (keeper) {
      const float csL = __shfl(rcs, Q - 1, 64), cslL = __shfl(rcsl, Q - 1, 64);
      s_cs[lane] = rcs;
      s_csl[lane] = rcsl;
      s_dt[lane] = rdt;
      s_w[lane] = reach ? fast_exp((csL - rcs) + (cslL - rcsl)) : 0.f;
      s_ecs[lane] = from ? fast_exp(rcs + rcsl) : 0.f;
    }
    map_park<bf16>(s_X, kLdP, kPlaneP, mp, rx, nvalid);
    {  // dY = dout silu(z), dz
#pragma unroll
      for (int k = 0; k < VX; ++k) {
        const int t = mp.row + k * mp.step;
        const bool in = t < nvalid;
        const float4 g4 = widen<bf16>(in ? rgo[k] : raw_zero<bf16>());
        float dy[4] = {g4.x, g4.y, g4.z, g4.w};
        if (HAS_Z) {
          const float4 z4 = widen<bf16>(rz[k]), y4 = widen<bf16>(ry[k]);
          const float zx[4] = {z4.x, z4.y, z4.z, z4.w}, yv[4] = {y4.x, y4.y, y4.z, y4.w};
          float dz[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float sg = sigmoid(zx[u]);
            dz[u] = dy[u] * yv[u] * sg * (1.f + zx[u] * (1.f - sg));
            dy[u] = in ? dy[u] * zx[u] * sg : 0.f;
          }
          if (in)
            st4<bf16>(static_cast<bf16*>(p.dz) + xoff + lane_offset(t * static_cast<uint32_t>(H * P) + mp.col),
                      make_float4(dz[0], dz[1], dz[2], dz[3]));
        }
        uint2 o[3];
        split4<3>(dy, o);
#pragma unroll
        for (int u = 0; u < 3; ++u) *reinterpret_cast<uint2*>(s_dY + u * kPlaneP + t * kLdP + mp.col) = o[u];
      }
    }
    park_states(dh);
    __syncthreads();
    if (NG > 1) fetch_states(h, 1);
    else if (i + 1 < p.hb) fetch_states(h + 1, 0);
    // This wave's own x (s) or dY (t) rows, terms over p in frag_col's order.
    Frag<1> xo[PK];
    Frag<3> yo[PK];
#pragma unroll
    for (int k = 0; k < PK; ++k) {
      if (sw) xo[k] = frag_row_as_col<1>(s_X + own * kLdP + 32 * k, kLdP, kPlaneP);
      else yo[k] = frag_row_as_col<3>(s_dY + own * kLdP + 32 * k, kLdP, kPlaneP);
    }
    v4f dxa[PT], dxs[PT];   // s-wave: d(dt x) from the chunk, and from the state before w
    zero(dxa);
    zero(dxs);
    // dG of each pair of tiles (32 of the other's steps), then G, dCB = dt_s dG
    // o M and R = dCB o C B^T, whose sum over the pair's rows is this lane's
    // column sum (s-wave) or row sum (t-wave) of R. Both leave out the diagonal,
    // whose decay is 1: it would only cancel between them, and round both.
    float rpart[4] = {0.f, 0.f, 0.f, 0.f};   // per tile: short chains of additions
    {
      const float cso = s_cs[step_own], cslo = s_csl[step_own], dto = s_dt[step_own];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        if (sw ? 32 * kt + 31 < own : 32 * kt > own) continue;   // above the diagonal
        v4f gv[2], dv[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int row0 = 32 * kt + 16 * u;
          v4f dg = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int k = 0; k < PK; ++k) {
            if (sw) dg = mma32(frag_row_as_col<3>(s_dY + row0 * kLdP + 32 * k, kLdP, kPlaneP), xo[k], dg);
            else dg = mma32(frag_row_as_col<1>(s_X + row0 * kLdP + 32 * k, kLdP, kPlaneP), yo[k], dg);
          }
          const int o0 = row0 + 4 * q;
          const float4 c4 = *reinterpret_cast<const float4*>(&s_cs[o0]);
          const float4 l4 = *reinterpret_cast<const float4*>(&s_csl[o0]);
          const float4 d4 = *reinterpret_cast<const float4*>(&s_dt[o0]);
          const float cv[4] = {c4.x, c4.y, c4.z, c4.w}, lv[4] = {l4.x, l4.y, l4.z, l4.w},
                      tv[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int o = o0 + e;
            const float dc = sw ? (cv[e] - cso) + (lv[e] - cslo) : (cso - cv[e]) + (cslo - lv[e]);
            const bool in = sw ? (o >= step_own && o <= bound) : (o <= step_own && o >= bound);
            const float m = in ? fast_exp(dc) : 0.f;
            gv[u][e] = cb[2 * kt + u][e] * m;
            dv[u][e] = dg[e] * (sw ? dto : tv[e]) * m;
            rpart[2 * kt + u] = fmaf(o == step_own ? 0.f : dv[u][e], cb[2 * kt + u][e], rpart[2 * kt + u]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        const Frag<3> df = frag_acc<3>(dv[0], dv[1]);
        if (sw) {  // d(dt x)[s][p] += sum_t G[t][s] dY[t][p]
          const Frag<3> gf = frag_acc<3>(gv[0], gv[1]);
#pragma unroll
          for (int j = 0; j < PT; ++j) {
            dxa[j] = mma32(gf, frag_col<3>(s_dY + 32 * kt * kLdP + 16 * j, kLdP, kPlaneP), dxa[j]);
            if (j & 1) __builtin_amdgcn_sched_barrier(0);  // two operands at a time: registers
          }
        }
        // dB[s][n] += sum_t dCB[t][s] C[t][n], or dC[t][n] += sum_s dCB[t][s] B[s][n]
#pragma unroll
        for (int j = 0; j < N / 16; ++j) {
          acc[j] = mma32(df, frag_col<1>(s_oth + 32 * kt * kLdT + 16 * j, kLdT, 0), acc[j]);
          if (j & 1) __builtin_amdgcn_sched_barrier(0);
        }
      }
      float rsum = (rpart[0] + rpart[1]) + (rpart[2] + rpart[3]);
      rsum = swap_sum<32>(rsum, rsum);
      rsum = swap_sum<16>(rsum, rsum);
      if (q == 0) (sw ? lds.col : lds.row)[step_own] = rsum;
    }
    if (i + 1 < p.hb) fetch(h + 1);   // here, not above: the chunk products need the registers
    // State terms, over 64-state groups of dH^out and H.
    const float4 f4 = *reinterpret_cast<const float4*>(sw ? &s_w[own + 4 * q] : &s_ecs[own + 4 * q]);
    const float4 t4 = *reinterpret_cast<const float4*>(&s_dt[own + 4 * q]);
    const float fr[4] = {f4.x, f4.y, f4.z, f4.w};   // w_s or exp(cs_t) of the rows own + 4 q + e
    const float dtr[4] = {t4.x, t4.y, t4.z, t4.w};
    float a_grp[N / 32][4] = {};                    // t-wave: sum_n C[t][n] exp(cs_t) (dY H)[t][n], 32 states each
#pragma unroll
    for (int grp = 0; grp < NG; ++grp) {
      if (grp == 1) {
        __syncthreads();  // every wave is done reading s_dH / s_H
        park_states(dh);
        __syncthreads();
        if (i + 1 < p.hb) fetch_states(h + 1, 0);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v4f tv = {0.f, 0.f, 0.f, 0.f};
        if (sw) {
          // (x dH)[s][n], and (B dH^T)[s][p] of headdim tile j
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            if (k < PK) tv = mma32(xo[k % PK], frag_col<3>(s_dH + 32 * k * kLdP + 16 * j, kLdP, kPlaneP), tv);
            if (j < PT)
              dxs[j % PT] = mma32(frag_row<1>(s_own + 64 * grp + 32 * k, kLdT, 0),
                                  frag_row<3>(s_dH + 16 * j * kLdP + 32 * k, kLdP, kPlaneP), dxs[j % PT]);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[4 * grp + j][e] = fmaf(fr[e] * dtr[e], tv[e], acc[4 * grp + j][e]);
        } else {
          // (dY H)[t][n]
#pragma unroll
          for (int k = 0; k < PK; ++k)
            tv = mma32(yo[k], frag_col<3>(s_H + 32 * k * kLdP + 16 * j, kLdP, kPlaneP), tv);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float ys = fr[e] * tv[e];
            acc[4 * grp + j][e] += ys;
            const uint32_t cw = cd[e][2 * grp + (j >> 1)];
            a_grp[2 * grp + (j >> 1)][e] =
                fmaf(__builtin_bit_cast(float, j & 1 ? cw & 0xffff0000u : cw << 16), ys, a_grp[2 * grp + (j >> 1)][e]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (lane == 0) lds.dh[wave] = dh;
    if (!sw) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = a_grp[0][e] + a_grp[1][e];
        if constexpr (NG > 1) a += a_grp[2][e] + a_grp[3][e];
        a = row_allreduce16(a);
        if (r == e) lds.a[own + 4 * q + e] = a;
      }
    }
    __syncthreads();  // every wave is done reading s_dH / s_H
    if (sw)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < PT; ++j) {
          const int at = (own + 4 * q + e) * XP + 16 * j + r;
          const float wv = fr[e] * dxs[j][e];
          s_W[at] = wv;
          s_dX[at] = dxa[j][e] + wv;
        }
    __syncthreads();
    // dx = dt dX + D dY; c = <x, dX>, b = dt <x, W> per row; dD over the rows
    {
      float dD[4] = {0.f, 0.f, 0.f, 0.f};
      float Dv[4] = {0.f, 0.f, 0.f, 0.f};
      if (p.D) ld4_elem<float>(p.D, h * P + mp.col, Dv);   // D may start at any element
#pragma unroll
      for (int k = 0; k < VX; ++k) {
        const int s = mp.row + k * mp.step;
        const float4 X4 = *reinterpret_cast<const float4*>(&s_dX[s * XP + mp.col]);
        const float4 W4 = *reinterpret_cast<const float4*>(&s_W[s * XP + mp.col]);
        const float4 x4 = pieces4<1>(s_X + s * kLdP + mp.col, kPlaneP);
        const float4 y4 = pieces4<3>(s_dY + s * kLdP + mp.col, kPlaneP);
        const float dt = s_dt[s];
        const float Xv[4] = {X4.x, X4.y, X4.z, X4.w}, Wv[4] = {W4.x, W4.y, W4.z, W4.w},
                    xv[4] = {x4.x, x4.y, x4.z, x4.w}, yv[4] = {y4.x, y4.y, y4.z, y4.w};
        float cr = fmaf(Xv[0], xv[0], Xv[1] * xv[1]) + fmaf(Xv[2], xv[2], Xv[3] * xv[3]);
        float br = fmaf(Wv[0], xv[0], Wv[1] * xv[1]) + fmaf(Wv[2], xv[2], Wv[3] * xv[3]);
        float o[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          dD[u] = fmaf(yv[u], xv[u], dD[u]);
          o[u] = fmaf(Dv[u], yv[u], Xv[u] * dt);
        }
        cr = lanes_allreduce<P / 4>(cr);
        br = lanes_allreduce<P / 4>(br);
        if (lane % (P / 4) == 0) {
          lds.c[s] = cr;
          lds.b[s] = br * dt;
        }
        if (s < nvalid)
          st4<bf16>(static_cast<bf16*>(p.dx) + xoff + lane_offset(s * static_cast<uint32_t>(H * P) + mp.col),
                    make_float4(o[0], o[1], o[2], o[3]));
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        dD[u] = swap_sum<32>(dD[u], dD[u]);
        dD[u] = swap_sum<16>(dD[u], dD[u]);
        if (P == 32) dD[u] += __shfl_xor(dD[u], 8, 64);
      }
      if (lane < P / 4) *reinterpret_cast<float4*>(&lds.dD[wave][4 * lane]) = make_float4(dD[0], dD[1], dD[2], dD[3]);
    }
    __syncthreads();
    const int64_t prt = (b * p.nchunks + c) * H + h;
    if (keeper) {
      // dcs = row sums - column sums of R + the state terms; the last step also
      // takes the cs_L terms (the states' dependence on w, and the entering
      // state's decay through the chunk, exp(cs_L) <dH^out, H_c>); da = suffix sums over the chunk; dstep = c + da A, then through
      // softplus / clamp / bias
      const float bv = lds.b[lane];
      float lo = 0.f;
      float v = add2(add2(lds.row[lane], -lds.col[lane], lo), add2(lds.a[lane], -bv, lo), lo);
      const float dhs = ((lds.dh[0] + lds.dh[1]) + (lds.dh[2] + lds.dh[3])) +
                        ((lds.dh[4] + lds.dh[5]) + (lds.dh[6] + lds.dh[7]));
      const float last = fmaf(s_ecs[Q - 1], dhs, wave_total(bv));
      if (lane == Q - 1) v = add2(v, last, lo);
      const float da = wave_suffix_sum2(v, lo);
      spoilt = spoil(spoilt, da);
      float ddt_raw = 0.f, dA_term = 0.f;
      if (lane < nvalid) {
        float gfac;
        step_of(p, pre + (p.dt_bias ? p.dt_bias[h] : 0.f), &gfac);
        ddt_raw = fmaf(da, p.A[h], lds.c[lane]) * gfac;
        dA_term = da * s_dt[lane];
        p.ddt[(b * L + t0 + lane) * H + h] = ddt_raw;
      }
      const float wa = wave_total(dA_term), wb = wave_total(ddt_raw);
      if (lane == 0) {
        p.dA_part[prt] = wa;
        p.dbias_part[prt] = wb;
      }
    } else if (!SW && wave == 5 && lane < P) {
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) v += lds.dD[k][lane];
      p.dD_part[prt * P + lane] = v;
    }
  }
  // the block's dB and dC partial sums
  float* const part = sw ? p.dB_part : p.dC_part;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int t = own + 4 * q + e;
    if (t >= nvalid) continue;
    const int64_t at = ((b * L + t0 + t) * p.nhb + blockIdx.y) * N;
#pragma unroll
    for (int j = 0; j < N / 16; ++j) part[at + 16 * j + r] = acc[j][e];
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int u = 0; u < 4; ++u) spoilt = spoil(spoilt, cb[u][e]);
#pragma unroll
    for (int j = 0; j < N / 16; ++j) spoilt = spoil(spoilt, acc[j][e]);
  }
  return spoilt;
}

template <bool HAS_Z, bool SEQ, int P, int N>
__global__ void __launch_bounds__(kThreads3, 2) ssd_bwd_chunk_bf16_kernel(const SsdParams p) {
  constexpr int TPB = kThreads3;
  __shared__ union {
    BwdChunkLds pieces;
    BwdF32Lds f32;
  } shared;
  BwdChunkLds& lds = shared.pieces;
  const int64_t c = blockIdx.x, b = blockIdx.z;
  const int64_t L = p.seqlen, G = p.ngroups;
  const int64_t g = static_cast<int64_t>(blockIdx.y) * p.hb / (p.nheads / G);
  const int64_t t0 = c * Q;
  const int nvalid = chunk_steps(p, t0);
  {
    const TileMap<TPB, N, true> mn(N);
    constexpr int VN = Q * N / 4 / TPB;
    const int64_t off = ((b * L + t0) * G + g) * N;
    raw4<bf16> rb[VN], rc[VN];
    map_load<bf16>(rb, mn, static_cast<const bf16*>(p.B) + off, G * N, nvalid);
    map_load<bf16>(rc, mn, static_cast<const bf16*>(p.C) + off, G * N, nvalid);
    map_park<bf16>(lds.B, kLdT, 0, mn, rb, nvalid);
    map_park<bf16>(lds.C, kLdT, 0, mn, rc, nvalid);
  }
  float spoilt;
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) < 4) spoilt = bwd_chunk_waves<HAS_Z, SEQ, P, N, true>(p, lds);
  else spoilt = bwd_chunk_waves<HAS_Z, SEQ, P, N, false>(p, lds);
  if (__builtin_expect(__syncthreads_or(spoilt != 0.f), 0) && p.apart)
    bwd_chunk_f32<bf16, HAS_Z, SEQ, false>(p, shared.f32);
}

// Per-sequence final states of packed sequences in batch row 0 (mamba_ssm's
// varlen states): entry i is the state after step e = cu[i + 1] - 1. From the
// chunk c holding e, h_e = exp(cs_e) H_c (when step e is in the entering
// state's sequence) + sum_s exp(cs_e - cs_s) dt_s x_s B_s^T over the steps
// s <= e of e's sequence in the chunk: one product on the matrix cores,
// started from the decayed entering state. Empty sequences, and offsets
// outside [0, seqlen], give zeros. Grid (nseqs, nheads); wave w computes state
// rows [16 w, 16 w + 16).
template <typename Tx, bool SEQ>
__global__ void __launch_bounds__(kThreads) ssd_varlen_state_kernel(const SsdParams p, const int32_t* cu,
                                                                     float* out) {
  __shared__ __align__(16) float s_B[Q][NP];
  __shared__ __align__(16) float s_x[Q][XP];
  __shared__ float s_sc[Q];
  const int64_t i = blockIdx.x, h = blockIdx.y, b = 0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int64_t L = p.seqlen, H = p.nheads, P = p.headdim, N = p.dstate, G = p.ngroups;
  const int64_t g = h / (H / G);
  const int nt = static_cast<int>(N / 16);
  const bool act = 16 * wave < P;
  const int64_t eo = (16 * wave + 4 * q) * N + r;   // accumulator (j, e) at eo + e N + 16 j of a block
  float* dst = out + (i * H + h) * P * N + eo;
  v4f acc[kSsdMaxN / 16];
  zero(acc);
  const int64_t start = cu[i], end = cu[i + 1];
  if (start < 0 || end > L || end <= start) {  // the same for the whole workgroup
    if (act)
#pragma unroll
      for (int j = 0; j < kSsdMaxN / 16; ++j)
        if (j < nt)
#pragma unroll
          for (int e = 0; e < 4; ++e) dst[e * N + 16 * j] = 0.f;
    return;
  }
  const int64_t last = end - 1, c = last / Q, t0 = c * Q;
  const int nv = static_cast<int>(last - t0 + 1);
  const int64_t row = chunk_row(p, b, h, c);
  const float cse = p.cs[row + nv - 1], loe = p.cs_lo[row + nv - 1];
  stage<Tx, kVecN>(&s_B[0][0], NP, static_cast<const Tx*>(p.B) + ((b * L + t0) * G + g) * N, G * N, Q, nv,
                   static_cast<int>(N));
  if (wave == 0) {
    const bool in = lane < nv && seq_of<SEQ>(p, b, t0 + lane) == seq_of<SEQ>(p, b, last);
    s_sc[lane] = in ? p.step[row + lane] * fast_exp((cse - p.cs[row + lane]) + (loe - p.cs_lo[row + lane])) : 0.f;
  }
  __syncthreads();
  stage<Tx, kVecX>(&s_x[0][0], XP, static_cast<const Tx*>(p.x) + ((b * L + t0) * H + h) * P, H * P, Q, nv,
                   static_cast<int>(P), s_sc);
  if (act && seq_of<SEQ>(p, b, last) == seq_of<SEQ>(p, b, t0 - 1)) {
    const float hd = fast_exp(cse + loe);
    const float* hs = p.states + state_block(p, b, c, h) + eo;
#pragma unroll
    for (int j = 0; j < kSsdMaxN / 16; ++j)
      if (j < nt)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[j][e] = hd * hs[e * N + 16 * j];
  }
  __syncthreads();
  if (act) {
    mma(acc, nt, &s_x[0][16 * wave], 1, XP, &s_B[0][0], NP, 1, Q);
#pragma unroll
    for (int j = 0; j < kSsdMaxN / 16; ++j)
      if (j < nt)
#pragma unroll
        for (int e = 0; e < 4; ++e) dst[e * N + 16 * j] = acc[j][e];
  }
}

namespace {

// Whether the chunk gradients run in bf16 pieces (and form their own dcsL).
template <typename Tx> bool bwd_in_pieces(const SsdParams& p) {
  return std::is_same_v<Tx, bf16> && (p.headdim == 64 || p.headdim == 32) && (p.dstate == 128 || p.dstate == 64);
}

bool exact_shape(const SsdParams& p) { return p.headdim == kSsdMaxP && p.dstate == kSsdMaxN; }

// The states' products of one direction: walking the chunks (in order), or per
// chunk, for every head (whatever the chunk kernels' head block).
template <typename Tx, bool SEQ, bool BWD>
hipError_t state_t(const SsdParams& p, hipStream_t st) {
  const int64_t ncb = (p.dstate + kSsdPassCols - 1) / kSsdPassCols;
  const dim3 grid(static_cast<unsigned>(p.in_order ? ncb : ncb * p.nchunks), static_cast<unsigned>(p.nheads),
                  static_cast<unsigned>(p.batch));
  auto go = [&](auto z, auto walk, auto exact, auto dcs) {
    hipLaunchKernelGGL((ssd_state_kernel<Tx, z.value, SEQ, BWD, walk.value, exact.value, dcs.value>), grid,
                       dim3(kThreads), 0, st, p);
  };
  auto shape = [&](auto z, auto walk, auto dcs) {
    constexpr bool never = std::is_same_v<Tx, bf16> && dcs.value;   // 64 x 128 runs in pieces
    if (!exact_shape(p)) go(z, walk, std::false_type{}, dcs);
    else if constexpr (!never) go(z, walk, std::true_type{}, dcs);
  };
  auto form = [&](auto z, auto walk) {
    if constexpr (BWD && walk.value) {
      if (!bwd_in_pieces<Tx>(p)) return shape(z, walk, std::true_type{});
      if constexpr (!std::is_same_v<Tx, bf16>) return;
    }
    shape(z, walk, std::false_type{});
  };
  auto gate = [&](auto z) {
    if (p.in_order) form(z, std::true_type{});
    else form(z, std::false_type{});
  };
  if (BWD && p.z) gate(std::integral_constant<bool, BWD>{});
  else gate(std::false_type{});
  return hipGetLastError();
}

template <typename Tx, bool SEQ>
hipError_t fwd_t(const SsdParams& p, hipStream_t st) {
  const dim3 chunks(static_cast<unsigned>(p.nchunks), static_cast<unsigned>(p.nhb), static_cast<unsigned>(p.batch));
  if (p.in_order) {
    const dim3 rows(static_cast<unsigned>((p.nchunks + kThreads / 64 - 1) / (kThreads / 64)),
                    static_cast<unsigned>(p.nheads), static_cast<unsigned>(p.batch));
    hipLaunchKernelGGL(ssd_chunk_decay_kernel, rows, dim3(kThreads), 0, st, p);
    if (hipError_t e = hipGetLastError()) return e;
  }
  if (hipError_t e = state_t<Tx, SEQ, false>(p, st)) return e;
  if (!p.in_order) {
    const dim3 slices(static_cast<unsigned>(p.nslices), static_cast<unsigned>(p.nheads),
                      static_cast<unsigned>(p.batch));
    hipLaunchKernelGGL(ssd_state_pass_kernel<SEQ>, slices, dim3(kThreads), 0, st, p);
    if (hipError_t e = hipGetLastError()) return e;
  }
  auto scan = [&](auto mn, auto exact) {
    if (p.z)
      hipLaunchKernelGGL((ssd_chunk_scan_kernel<Tx, true, SEQ, mn.value, exact.value>), chunks, dim3(kThreads3), 0, st, p);
    else
      hipLaunchKernelGGL((ssd_chunk_scan_kernel<Tx, false, SEQ, mn.value, exact.value>), chunks, dim3(kThreads3), 0, st, p);
  };
  if (exact_shape(p)) scan(std::integral_constant<int, 128>{}, std::true_type{});
  else if (p.dstate > 64) scan(std::integral_constant<int, 128>{}, std::false_type{});
  else scan(std::integral_constant<int, 64>{}, std::false_type{});
  return hipGetLastError();
}

template <typename Tx, bool SEQ>
hipError_t bwd_t(const SsdParams& p, hipStream_t st) {
  const dim3 chunks(static_cast<unsigned>(p.nchunks), static_cast<unsigned>(p.nhb), static_cast<unsigned>(p.batch));
  const bool pieces = bwd_in_pieces<Tx>(p);
  if (hipError_t e = state_t<Tx, SEQ, true>(p, st)) return e;
  if (!p.in_order) {
    const dim3 slices(static_cast<unsigned>(p.nslices), static_cast<unsigned>(p.nheads),
                      static_cast<unsigned>(p.batch));
    if (pieces) hipLaunchKernelGGL((ssd_bwd_pass_kernel<SEQ, false>), slices, dim3(kThreads), 0, st, p);
    else hipLaunchKernelGGL((ssd_bwd_pass_kernel<SEQ, true>), slices, dim3(kThreads), 0, st, p);
    if (hipError_t e = hipGetLastError()) return e;
  }
  if constexpr (std::is_same_v<Tx, bf16>) {
    if (pieces) {
      auto go = [&](auto hd, auto ds) {
        if (p.z)
          hipLaunchKernelGGL((ssd_bwd_chunk_bf16_kernel<true, SEQ, hd.value, ds.value>), chunks, dim3(kThreads3), 0, st, p);
        else
          hipLaunchKernelGGL((ssd_bwd_chunk_bf16_kernel<false, SEQ, hd.value, ds.value>), chunks, dim3(kThreads3), 0, st, p);
      };
      using n32 = std::integral_constant<int, 32>;
      using n64 = std::integral_constant<int, 64>;
      using n128 = std::integral_constant<int, 128>;
      if (p.headdim == 64) p.dstate == 128 ? go(n64{}, n128{}) : go(n64{}, n64{});
      else p.dstate == 128 ? go(n32{}, n128{}) : go(n32{}, n64{});
      return hipGetLastError();
    }
  }
  if (p.z) hipLaunchKernelGGL((ssd_bwd_chunk_kernel<Tx, true, SEQ>), chunks, dim3(kThreads3), 0, st, p);
  else hipLaunchKernelGGL((ssd_bwd_chunk_kernel<Tx, false, SEQ>), chunks, dim3(kThreads3), 0, st, p);
  return hipGetLastError();
}

}  // namespace

hipError_t ssd_fwd_launch(const SsdParams& p, int dtype, hipStream_t st) {
  const bool seq = p.seq_idx != nullptr;
  switch (dtype) {
    case MCPU_F32: return seq ? fwd_t<float, true>(p, st) : fwd_t<float, false>(p, st);
    case MCPU_BF16: return seq ? fwd_t<bf16, true>(p, st) : fwd_t<bf16, false>(p, st);
    default: return seq ? fwd_t<f16, true>(p, st) : fwd_t<f16, false>(p, st);
  }
}

hipError_t ssd_varlen_launch(const SsdParams& p, const int32_t* cu, int64_t nseqs, float* out, int dtype,
                             hipStream_t st) {
  const dim3 grid(static_cast<unsigned>(nseqs), static_cast<unsigned>(p.nheads));
  const bool seq = p.seq_idx != nullptr;
  switch (dtype) {
    case MCPU_F32:
      if (seq) hipLaunchKernelGGL((ssd_varlen_state_kernel<float, true>), grid, dim3(kThreads), 0, st, p, cu, out);
      else hipLaunchKernelGGL((ssd_varlen_state_kernel<float, false>), grid, dim3(kThreads), 0, st, p, cu, out);
      break;
    case MCPU_BF16:
      if (seq) hipLaunchKernelGGL((ssd_varlen_state_kernel<bf16, true>), grid, dim3(kThreads), 0, st, p, cu, out);
      else hipLaunchKernelGGL((ssd_varlen_state_kernel<bf16, false>), grid, dim3(kThreads), 0, st, p, cu, out);
      break;
    default:
      if (seq) hipLaunchKernelGGL((ssd_varlen_state_kernel<f16, true>), grid, dim3(kThreads), 0, st, p, cu, out);
      else hipLaunchKernelGGL((ssd_varlen_state_kernel<f16, false>), grid, dim3(kThreads), 0, st, p, cu, out);
  }
  return hipGetLastError();
}

hipError_t ssd_bwd_launch(const SsdParams& p, int dtype, hipStream_t st) {
  const bool seq = p.seq_idx != nullptr;
  switch (dtype) {
    case MCPU_F32: return seq ? bwd_t<float, true>(p, st) : bwd_t<float, false>(p, st);
    case MCPU_BF16: return seq ? bwd_t<bf16, true>(p, st) : bwd_t<bf16, false>(p, st);
    default: return seq ? bwd_t<f16, true>(p, st) : bwd_t<f16, false>(p, st);
  }
}

}  // namespace mcpu
