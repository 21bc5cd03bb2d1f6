// Selective state update (one decode step) on gfx950.
//
// Per row (batch, head, p) and state n (reference
// src/mamba_cpu/ops/selective_state_update.py:5-57):
//   dt    = softplus?(dt + dt_bias)
//   state = state * exp(dt * A) + dt * x * B[group]
//   out   = (<state, C[group]> + D * x) * silu(z)
// The state is read and written in place, and that is what bounds the call
// once the batch fills the GPU: 2 * 4 bytes per float32 state against a few
// instructions. Two kernels:
//   - dstate 16, 32, 64, 128 or 256 (every model's): LPR lanes per row, each
//     moving VPL vectors of four neighbouring states. The fewer lanes to a row,
//     the more rows to a wave for what is done once per row; 4 lanes up to 64
//     states (64 states 37 us, 8 lanes 39, 16 lanes 52; 32 states 17 against 23),
//     8 for 128 (70 us; 16 lanes 75; 4 lanes 74, of 222 registers), 16 for 256
//     (120 us, 117 of them without chains_sum's order; 8 lanes 135, for their
//     registers). Vectors need no more than their element's alignment, so any
//     base and strides run here.
//     (64, 80, 64, 128) float32 states with bf16 x, B and C: 70 us, 4.8 TB/s,
//     against 90 us with one state per lane and load and B and C cast to
//     float32 by two launches; (64, 5120, 16): 12.8 against 40.8 us.
//   - any other dstate: 16 lanes per row, lane j owning states j, j + 16, ...
// Both run row tiles of the (nheads, headdim) rows x batch, so the row decode is
// one 32-bit division. B and C are float32 or of x's type (Tb).
#include "mcpu_common.h"
#include "op_params.h"

namespace mcpu {

// The vector (of LPR in a row) that lane j moves: vector j, but with 8 lanes the upper
// quad's in the other order, for chains_sum.
template <int LPR> __device__ __forceinline__ int vector_of(int j) { return LPR == 8 && j >= 4 ? 11 - j : j; }

// <state, C> of a row whose lane j of LPR holds states 4 (vector_of(j) + LPR v) + i, in
// the last quad's lanes. The sum is that of one state per lane (VPL = 0 below, and the
// fused decode steps'), so that all give the same bits: 16 chains over the states m,
// m + 16, ..., then a tree over m. States 16 k .. 16 k + 16 are in quad k % (LPR / 4)
// of the row, so the chains pass from quad to quad where the row has more than one, by
// a mirror where it has two; what the other quads add meanwhile is not used.
template <int LPR, int VPL>
__device__ __forceinline__ float chains_sum(const float (&v)[4 * VPL], const float (&c)[4 * VPL]) {
  auto from_quad = [](float x) {
    if constexpr (LPR == 4) return x;
    else return dpp<LPR == 8 ? kRowHalfMirror : kRowRor4>(x);
  };
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < VPL * LPR / 4; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = 4 * (4 * k / LPR) + i;
      acc[i] = fmaf(v[at], c[at], k == 0 ? 0.f : from_quad(acc[i]));
    }
  float sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  sum += dpp<kQuadXor1>(sum);
  return sum + dpp<kQuadXor2>(sum);
}

// VPL > 0: dstate = 4 LPR VPL, lane j of a row owning states 4 (vector_of(j) + LPR v) + i.
// VPL = 0: any dstate up to 16 SPL, LPR = 16, lane j owning states j + 16 s.
template <typename Tx, typename Ts, typename Tb, int LPR, int VPL, int SPL>
__global__ void __launch_bounds__(256) state_update_kernel(const StateUpdateParams p) {
  constexpr int NS = VPL > 0 ? 4 * VPL : SPL;  // states of a lane
  const int j = threadIdx.x & (LPR - 1), jv = vector_of<LPR>(j);
  const uint32_t hp = blockIdx.x * (256u / LPR) + threadIdx.x / LPR;  // row within (nheads, headdim)
  // Whole rows share every branch, so the DPP reduction below never mixes
  // live and retired lanes of one row.
  if (hp >= static_cast<uint32_t>(p.nheads * p.headdim)) return;
  const uint32_t hd = static_cast<uint32_t>(p.headdim);
  const uint32_t h = hp / hd, pp = hp - h * hd;
  const int64_t g = h / static_cast<uint32_t>(p.nheads / p.ngroups);
  const int64_t N = p.dstate;
  for (int64_t b = blockIdx.y; b < p.batch; b += gridDim.y) {
    const int64_t rowid = b * p.nheads * p.headdim + hp;
    int64_t srow = b;
    if (p.state_idx != nullptr) {
      srow = p.state_idx[b];
      if (srow < 0 || srow >= p.state_batch) {
        if (j == 0) st<Tx>(p.out, rowid, 0.f);
        continue;
      }
    }
    const int64_t sbase = srow * p.sst[0] + h * p.sst[1] + pp * p.sst[2];
    const float* Arow = p.A + h * p.sA[0] + pp * p.sA[1];
    const int64_t Boff = b * p.sB[0] + g * p.sB[1], Coff = b * p.sC[0] + g * p.sC[1];
    // Every load of the lane's states first: a load after a store to the
    // state could not be moved above it, which would make each state a
    // memory round trip of its own.
    float sv[NS], av[NS], bv[NS], cv[NS];
    if constexpr (VPL > 0) {
#pragma unroll
      for (int v = 0; v < VPL; ++v) ld4_elem<Ts>(p.state, sbase + 4 * (jv + LPR * v), sv + 4 * v);
#pragma unroll
      for (int v = 0; v < VPL; ++v) {
        const int n = 4 * (jv + LPR * v);
        ld4_elem<Tb>(p.B, Boff + n, bv + 4 * v);
        ld4_elem<Tb>(p.C, Coff + n, cv + 4 * v);
        if (p.sA[2] == 1) {
          ld4_elem<float>(Arow, n, av + 4 * v);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) av[4 * v + i] = Arow[(n + i) * p.sA[2]];
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int n = j + 16 * s;
        const bool ok = n < N;
        sv[s] = ok ? ld<Ts>(p.state, sbase + n) : 0.f;
        av[s] = ok ? Arow[n * p.sA[2]] : 0.f;
        bv[s] = ok ? ld<Tb>(p.B, Boff + n) : 0.f;
        cv[s] = ok ? ld<Tb>(p.C, Coff + n) : 0.f;
      }
    }
    const float x = ld<Tx>(p.x, b * p.sx[0] + h * p.sx[1] + pp * p.sx[2]);
    float dt = ld<Tx>(p.dt, b * p.sdt[0] + h * p.sdt[1] + pp * p.sdt[2]);
    if (p.dt_bias != nullptr) dt += p.dt_bias[h * p.sbias[0] + pp * p.sbias[1]];
    if (p.softplus) dt = softplus(dt);
    const float dtx = dt * x;
    float acc = 0.f;
    if constexpr (VPL > 0) {
#pragma unroll
      for (int i = 0; i < NS; ++i) sv[i] = fmaf(sv[i], fast_exp(dt * av[i]), dtx * bv[i]);
#pragma unroll
      for (int v = 0; v < VPL; ++v) st4_elem<Ts>(p.state, sbase + 4 * (jv + LPR * v), sv + 4 * v);
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int n = j + 16 * s;
        if (n < N) {
          const float v = fmaf(sv[s], fast_exp(dt * av[s]), dtx * bv[s]);
          st<Ts>(p.state, sbase + n, v);
          acc = fmaf(v, cv[s], acc);
        }
      }
    }
    float y;
    if constexpr (VPL > 0) y = chains_sum<LPR, VPL>(sv, cv);
    else y = row_allreduce16(acc);
    if (j == (VPL > 0 ? LPR - 4 : 0)) {
      if (p.D != nullptr) y = fmaf(x, p.D[h * p.sD[0] + pp * p.sD[1]], y);
      if (p.z != nullptr) {
        const float zz = ld<Tx>(p.z, b * p.sz[0] + h * p.sz[1] + pp * p.sz[2]);
        y *= zz * sigmoid(zz);
      }
      st<Tx>(p.out, rowid, y);
    }
  }
}

template <typename Tx, typename Ts, typename Tb, int LPR, int VPL, int SPL>
static void launch_su_one(const StateUpdateParams& p, hipStream_t st) {
  const int64_t rows = p.nheads * p.headdim, per = 256 / LPR;
  const dim3 blocks(static_cast<unsigned>((rows + per - 1) / per),
                    static_cast<unsigned>(p.batch < 65535 ? p.batch : 65535));
  hipLaunchKernelGGL((state_update_kernel<Tx, Ts, Tb, LPR, VPL, SPL>), blocks, dim3(256), 0, st, p);
}

template <typename Tx, typename Ts, typename Tb>
static hipError_t launch_su_types(const StateUpdateParams& p, hipStream_t st) {
  const int64_t n = p.dstate;
  if (n == 16) launch_su_one<Tx, Ts, Tb, 4, 1, 0>(p, st);
  else if (n == 32) launch_su_one<Tx, Ts, Tb, 4, 2, 0>(p, st);
  else if (n == 64) launch_su_one<Tx, Ts, Tb, 4, 4, 0>(p, st);
  else if (n == 128) launch_su_one<Tx, Ts, Tb, 8, 4, 0>(p, st);
  else if (n == 256) launch_su_one<Tx, Ts, Tb, 16, 4, 0>(p, st);
  else if (n < 16) launch_su_one<Tx, Ts, Tb, 16, 0, 1>(p, st);
  else if (n < 32) launch_su_one<Tx, Ts, Tb, 16, 0, 2>(p, st);
  else if (n < 64) launch_su_one<Tx, Ts, Tb, 16, 0, 4>(p, st);
  else if (n < 128) launch_su_one<Tx, Ts, Tb, 16, 0, 8>(p, st);
  else launch_su_one<Tx, Ts, Tb, 16, 0, 16>(p, st);
  return hipGetLastError();
}

template <typename Tx, typename Ts>
static hipError_t launch_su(const StateUpdateParams& p, hipStream_t st) {
  if (p.bc_dtype == MCPU_F32) return launch_su_types<Tx, Ts, float>(p, st);
  return launch_su_types<Tx, Ts, Tx>(p, st);
}

template <typename Tx>
static hipError_t launch_su_state(const StateUpdateParams& p, int state_dtype, hipStream_t st) {
  switch (state_dtype) {
    case MCPU_F32: return launch_su<Tx, float>(p, st);
    case MCPU_BF16: return launch_su<Tx, bf16>(p, st);
    default: return launch_su<Tx, f16>(p, st);
  }
}

hipError_t state_update_launch(const StateUpdateParams& p, int dtype, int state_dtype, hipStream_t st) {
  if (p.batch * p.nheads * p.headdim == 0) return hipSuccess;
  switch (dtype) {
    case MCPU_F32: return launch_su_state<float>(p, state_dtype, st);
    case MCPU_BF16: return launch_su_state<bf16>(p, state_dtype, st);
    default: return launch_su_state<f16>(p, state_dtype, st);
  }
}

}  // namespace mcpu
