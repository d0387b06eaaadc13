// Converters and per-sample state of the noisy matrix-vector products, shared by the kernels that run them.
#pragma once
#include "kernels.h"

namespace rpu_amd {
namespace {

// lane i: the value of lane i ^ off, within rows of 16 lanes, where the values of lanes i and i ^ (2 off) (and above, in the
// row) are the same already: a butterfly that starts with the largest offset
template <int OFF> __device__ __forceinline__ float row_xor(float v) {
  static_assert(OFF == 8 || OFF == 4 || OFF == 2 || OFF == 1);
  constexpr int CTRL = OFF == 8 ? 0x128 : (OFF == 4 ? 0x124 : (OFF == 2 ? 0x4e : 0xb1)); // row_ror:8, row_ror:4, quad_perm
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// STOCH = false: for callers that have checked that the DAC draws no random numbers (no stochastic rounding, no input
// noise): the draws are then not even compiled in, which the fully unrolled callers pay for in registers
template <bool STOCH = true>
__device__ __forceinline__ float dac_value(float x, float scale, const IoDev &io, PhiloxKey key,
                                           uint32_t call, int round, int b, int k) {
  // value *= scale; discretize; clip; (+ noise); (asymmetry)      rpu_forward_backward_pass.cpp:583-602
  float v = x * scale;
  if (io.inp_res > 0.0f) {
    float q = v / io.inp_res;
    if (STOCH && io.inp_sto_round) {
      const Philox4 r = philox4x32_10((uint32_t)k, (uint32_t)b, call, RNG_INP_SR | ((uint32_t)round << 8), key.k0, key.k1);
      q = q + (u32_to_uniform(r.v[0]) - 0.5f);
    }
    v = rintf(q) * io.inp_res;
  }
  v = (v > io.inp_bound) ? io.inp_bound : v;
  v = (v < -io.inp_bound) ? -io.inp_bound : v;
  if (STOCH && io.inp_noise > 0.0f) {
    float n[4];
    philox_normal4((uint32_t)k, (uint32_t)b, call, RNG_INP_NOISE | ((uint32_t)round << 8), key, n);
    v += io.inp_noise * n[0];
  }
  if (io.inp_asym != 0.0f) {
    v = v < 0.0f ? v * (1.0f - io.inp_asym) : v;
  }
  return v;
}

// Stored elements of a sample: all K, or without the 1 of the bias column.  Loops that put several loads in flight read the
// elements below this number and set the 1 afterwards, in a branch that the whole wave takes or not: with a choice between
// load and constant at every element the loads are issued one by one (k_mvm_init, 256 samples of 1024 elements: 8.1 us
// instead of 6.9).
__device__ __forceinline__ int mvm_stored(const MvmArgs &a) { return a.K - a.in_one; }

// input scale of a round and the factor applied to its ADC output
__device__ __forceinline__ float round_scales(const MvmArgs &a, float nm, float red, float &fin) {
  const IoDev &io = a.io;
  const bool use_nm = io.noise_management != RPU_NM_NONE;
  const bool bm = io.bound_management != RPU_BM_NONE;
  float scale;
  if (a.transposed) {
    // backward: scale = 1 / nm ; result *= out_scale * nm
    if (use_nm && nm <= 0.0f) {
      scale = 0.0f;
      fin = 0.0f;
    } else {
      scale = use_nm ? 1.0f / nm : 1.0f;
      fin = use_nm ? io.out_scale * nm : io.out_scale;
    }
  } else if (use_nm && nm <= 0.0f && io.inp_noise <= 0.0f) {
    scale = 0.0f;
    fin = 0.0f;
  } else {
    scale = 1.0f;
    if (use_nm && nm > 0.0f) scale /= nm;
    if (bm) scale /= red;
    fin = io.out_scale / scale;
  }
  return scale;
}

// Noise-management value and reduction that sample b, now at (nm, red) with output factor fin, would use in
// the round after `round`; false when the reduction limit is reached or the sample is short-cut to zero
// (rpu_forward_backward_pass.cpp:944-983).
// np_known: the sample's AbsMaxNPSum scale where the caller has just computed it (the init kernel, whose other
// threads must not read back what its first thread is storing); null: read from the per-sample state.
__device__ __forceinline__ bool next_round_params(const MvmArgs &a, int round, int b, float fin, float &nm, float &red,
                                                  const float *np_known = nullptr) {
  const IoDev &io = a.io;
  if (fin == 0.0f) return false;
  const bool stop = ((int)red > io.max_bm_factor) || ((io.inp_res > 0.0f) && (red > io.max_bm_res / io.inp_res));
  if (stop) return false;
  red *= 2.0f;
  if (round == 0 && io.bound_management == RPU_BM_ITERATIVE_WORST_CASE && io.noise_management != RPU_NM_ABS_MAX_NP_SUM) {
    nm = np_known ? *np_known : a.st.nm_np[b];
    red = 1.0f;
  }
  return true;
}

} // namespace
} // namespace rpu_amd
