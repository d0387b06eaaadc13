// Noisy matrix-vector products of batches between the small ones (k_mvm_few) and those that fill large tiles, in one launch:
// noise management, DAC, contraction, ADC and every bound-management round, with the bits of the launches one by one.
//
// Such a call is a chain of latencies too: an init kernel, a round of 32 x 32 tiles on a quarter of the CUs or less (each wave
// 16 matrix steps of 64 cycles to 32 contraction indices, behind loads, LDS and a barrier), a launch for the rounds that are
// expected to be empty.  Here a workgroup takes 16 samples and 16 or 64 outputs: a step of 32 indices is 8 matrix instructions
// of 32 cycles, and four times as many workgroups are in flight.  It quantizes its samples' rows itself, keeps the quotients
// before the rounding in LDS (the rounds' inputs are halves of each other: they are rounded on the way into the registers,
// underneath the matrix instructions) and decides about further rounds as k_mvm_few does: the workgroups of a sample count
// themselves off, the last one copies out the round that stands (R = 3), or runs the rounds from R on alone.
//
// What bounds it: the chain from the inputs' loads over their maximum, the contraction, the barriers and the counters to the output.
// 512 x 512, 100 samples, three rounds: of the waves' cycles 58 % wait for such results, 19 % issue vector instructions, the matrix
// pipe is busy 11 %, LDS is waited for 0.3 % (one round: 63, 18, 5, 0.1).
// Launches one by one -> this one: 512 x 512, 100 samples 27.1 -> 15.8 us, 785 -> 256, 64 samples 39.3 -> 17.2.
//
// Sums are those of mvm_round_tile, bit for bit: four chains over the quarters of the padded contraction, wave w the w-th,
// added ((0 + 1) + 2) + 3; in a chain, steps of 32 indices in ascending order, in a step 0, 16, 1, 17, ..., 15, 31 (there the
// two half-waves hold 0 .. 15 and 16 .. 31).  The fp32 matrix instructions round after every product, in ascending order of
// their own contraction index: 32 x 32 x 2 and 16 x 16 x 4 are the same chain of fused multiply-adds.
#include "bf16_parts.h"
#include "mvm_device.h"

#include <algorithm>
#include <cmath>

namespace rpu_amd {

namespace {

constexpr int S = 16;           // samples of a workgroup
constexpr int KSTEP = 32;       // contraction indices of a step
constexpr int MOST_ROUNDS = MVM_WHOLE_ROUNDS; // worked out together
constexpr int THROUGH = 16;     // cache policy of a buffer access: past the XCD's L2, as an atomic access of the device's scope

typedef unsigned u32x4_bits __attribute__((ext_vector_type(4)));

struct WholeShared {
  int hits[MOST_ROUNDS * 2 * S]; // [R][2][S] saturation marks: upper, lower
  float fin[MOST_ROUNDS * S];    // [R][S] output factors
  float max[S], scale[S];
  int clip[4];
  int last;
};

__device__ __forceinline__ float two_to(int n) { return __builtin_bit_cast(float, (127 + n) << 23); }

template <bool WOC, int NB, int R> struct MvmWhole {
  static_assert((NB == 1 || NB == 2 || NB == 4) && (R == 1 || R == MOST_ROUNDS));
  typedef MvmWhole<WOC, 2, 1> Alone; // see alone()
  static constexpr int OB = 16 * NB;             // outputs of a workgroup; NB * i + n is row i of matrix product n
  static constexpr int AHEAD = NB == 1 ? 4 : 2;  // steps of weights in flight
  static constexpr int X_AHEAD = 8;              // inputs of a thread in flight, four at a time
  static constexpr int ROUND = 4 * NB * 256;     // partial sums of a round: [4 waves][NB][4][64 lanes]

  typedef f32x4 Weights[2 * NB]; // of a step: 8 NB values of a lane, see operands()

  const MvmArgs &a;
  float *const q; // LDS: [S][ld] inputs before rounding, in the order that a lane reads them
  float *part;    // LDS: partial sums [R][ROUND]
  WholeShared &sh;
  int lane, wave, steps, len, ld; // len: the row with what thread t / 16 pads it to, ld: with its distance to the next
  int s_begin, s_end; // steps of this wave
  __amdgpu_buffer_rsrc_t w_buffer;
  unsigned row_bytes;

  static __host__ __device__ int row(int K) { return (K + 63) / 64 * 64 + 4; }
  static __host__ __device__ size_t lds_bytes(int K) {
    // the partial sums take the place of the inputs, except where a workgroup goes on to further outputs
    const size_t inputs = sizeof(float) * S * row(K), sums = sizeof(float) * R * ROUND;
    const size_t alone = inputs + sizeof(float) * Alone::ROUND, own = inputs > sums ? inputs : sums;
    return own > alone ? own : alone;
  }

  __device__ __forceinline__ MvmWhole(const MvmArgs &a_, float *lds, WholeShared &sh_)
      : a(a_), q(lds), part(lds), sh(sh_), lane((int)threadIdx.x & 63), wave(uniform((int)threadIdx.x >> 6)), ld(row(a_.K)) {
    steps = (a.K + KSTEP - 1) / KSTEP;
    len = ld - 4;
    const int per_wave = (a.k_pad / KSTEP + 3) / 4; // as the waves of mvm_round_tile share the padded contraction
    s_begin = min(wave * per_wave, steps);
    s_end = min(s_begin + per_wave, steps);
    row_bytes = 4u * (unsigned)a.w_ld;
    w_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.w), 0,
                                                 (int)(((unsigned)(WOC ? a.K : a.O) - 1u) * row_bytes + 4u * (unsigned)(WOC ? a.O : a.K)), 0x00020000);
  }

  // Weights of a step.  Lane (r, h), r = lane % 16, takes part in the products with k = 16 (h % 2) + h / 2 + 2 j, j = 0 .. 7,
  // of the step, for the rows r of the NB matrix products.  What lies beyond the matrix reads as zero; what lies beyond a row
  // and within the matrix belongs to outputs that are not stored, or add() masks it.
  __device__ __forceinline__ void load(Weights &w, int step, int o_first) const {
    const int r = lane & 15, h = lane >> 4;
    if constexpr (WOC) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const unsigned from = (unsigned)(step * KSTEP + 16 * (h & 1) + (h >> 1) + 2 * j) * row_bytes + 4u * (unsigned)(o_first + NB * r);
        // value j of matrix product n: element (j NB + n) of the lane's values
        if constexpr (NB == 4) {
          w[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(w_buffer, from, 0, 0));
        } else if constexpr (NB == 2) {
          typedef float f32x2 __attribute__((ext_vector_type(2)));
          const f32x2 v = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(w_buffer, from, 0, 0));
          w[j / 2][2 * (j & 1)] = v[0];
          w[j / 2][2 * (j & 1) + 1] = v[1];
        } else {
          w[j / 4][j & 3] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(w_buffer, from, 0, 0));
        }
      }
    } else {
      // eight indices in a row, 16 (h % 2) + 8 (h / 2) ..: operands() trades them with lane ^ 32
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const unsigned from = (unsigned)(o_first + NB * r + n) * row_bytes + 4u * (unsigned)(step * KSTEP + 16 * (h & 1) + 8 * (h >> 1));
        w[2 * n] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(w_buffer, from, 0, 0));
        w[2 * n + 1] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(w_buffer, from + 16u, 0, 0));
      }
    }
  }
  __device__ __forceinline__ void operands(const Weights &w, float (&v)[NB][8]) const {
#pragma unroll
    for (int n = 0; n < NB; ++n) {
      if constexpr (WOC) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[n][j] = w[(j * NB + n) / 4][(j * NB + n) & 3];
      } else {
        // even indices of eight in the one register, odd ones in the other: the upper half-wave's even ones for the lower
        // half-wave's odd ones leave k = 2 j below and 2 j + 1 above
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 part4 = w[2 * n + i / 2];
          const float even = part4[2 * (i & 1)], odd = part4[2 * (i & 1) + 1];
          const auto swapped = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, even), __builtin_bit_cast(unsigned, odd), false, false);
          const unsigned first = swapped[0], second = swapped[1];
          v[n][i] = __builtin_bit_cast(float, first);
          v[n][4 + i] = __builtin_bit_cast(float, second);
        }
      }
    }
  }

  // Rows of the block's samples: thread t holds four elements at 4 (t % 16) of each 64, of row t / 16
  typedef f32x4 Inputs[X_AHEAD];
  __device__ __forceinline__ void load_inputs(Inputs &x, int b0, int k0) const {
    const int at = 4 * ((int)threadIdx.x & 15), b = min(b0 + ((int)threadIdx.x >> 4), a.m_batch - 1);
    const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(a.in), 0, (int)(4u * (unsigned)((long)(a.m_batch - 1) * a.in_sb + (long)(mvm_stored(a) - 1) * a.in_sk + 1)), 0x00020000);
    const unsigned step = 4u * (unsigned)a.in_sk, from = 4u * (unsigned)((long)b * a.in_sb) + step * (unsigned)(k0 + at);
    if (a.in_sk == 1) {
#pragma unroll
      for (int i = 0; i < X_AHEAD; ++i) {
        if (k0 + 64 * i < len) x[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(buffer, from + 256u * i, 0, 0));
      }
    } else {
#pragma unroll
      for (int i = 0; i < X_AHEAD; ++i) {
        if (k0 + 64 * i < len) {
#pragma unroll
          for (int c = 0; c < 4; ++c) x[i][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer, from + step * (unsigned)(64 * i + c), 0, 0));
        }
      }
    }
  }
  // Takes the values into the largest one, m, and leaves them in q
  __device__ __forceinline__ void keep_inputs(Inputs &x, int k0, float &m) const {
    const bool signed_max = a.io.noise_management == RPU_NM_MAX;
    const int stored = mvm_stored(a);
#pragma unroll
    for (int i = 0; i < X_AHEAD; ++i) {
      const int first = k0 + 64 * i;
      if (first >= len) break;
      if (first + 64 > stored) { // the row's end, perhaps with the bias column's 1 behind it, then zeros
        const int left = stored - first - 4 * ((int)threadIdx.x & 15);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          x[i][c] = c < left ? x[i][c] : (c < left + a.in_one ? 1.0f : 0.0f);
          m = c < left + a.in_one ? fmaxf(m, signed_max ? x[i][c] : fabsf(x[i][c])) : m;
        }
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) m = fmaxf(m, signed_max ? x[i][c] : fabsf(x[i][c]));
      }
      put(place(first), x[i]);
    }
  }
  // where this thread's four values of k0 .. k0 + 63 are in q: those of even index next to each other, those of odd index 16
  // behind them
  __device__ __forceinline__ float *place(int k0) const {
    const int at = 4 * ((int)threadIdx.x & 15);
    return q + ((int)threadIdx.x >> 4) * ld + k0 + (at & 32) + 8 * ((at >> 4) & 1) + ((at & 15) >> 1);
  }
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  __device__ __forceinline__ static void put(float *to, const f32x4 v) {
    *reinterpret_cast<f32x2 *>(to) = f32x2{v[0], v[2]};
    *reinterpret_cast<f32x2 *>(to + 16) = f32x2{v[1], v[3]};
  }
  // v / divisor, rounded as the division rounds it: with the divisor's reciprocal rounded to nearest, a product and one
  // correction are exact (Markstein 1990; compared with the division for 2400 divisors, with every mantissa), except where the
  // remainder leaves the range of numbers: smaller quotients round to zero, and larger ones are clipped (steps_are_exact).
  __device__ __forceinline__ static float quotient(float v, float divisor, float reciprocal) {
    const float first = v * reciprocal, second = __builtin_fmaf(__builtin_fmaf(-first, divisor, v), reciprocal, first);
    return fabsf(first) < 0x1p60f ? second : first;
  }
  // Leaves the block's inputs in q, the largest of each row in sh.max, its scale in sh.scale and in sh.clip, for each wave's
  // rows, a bit for each round in which one of them goes beyond the input range; x: as load_inputs(x, b0, 0); `red`: reduction
  // of the first round
  __device__ __forceinline__ void fill(Inputs &x, int b0, float nm_known, bool known, float red) const {
    const IoDev &io = a.io;
    const bool signed_max = io.noise_management == RPU_NM_MAX;
    float m = signed_max ? -INFINITY : 0.0f;
    for (int k0 = 0;;) {
      keep_inputs(x, k0, m);
      k0 += 64 * X_AHEAD;
      if (k0 >= len) break;
      load_inputs(x, b0, k0);
    }
    m = fmaxf(m, row_xor<8>(m));
    m = fmaxf(m, row_xor<4>(m));
    m = fmaxf(m, row_xor<2>(m));
    m = fmaxf(m, row_xor<1>(m));
    float fin;
    const float scale = round_scales(a, known ? nm_known : nm_of(m), red, fin);
    if (((int)threadIdx.x & 15) == 0) {
      sh.max[(int)threadIdx.x >> 4] = m;
      sh.scale[(int)threadIdx.x >> 4] = scale;
    }
    int clip = 0;
    float top = io.inp_res > 0.0f ? quotient(m * scale, io.inp_res, 1.0f / io.inp_res) : m * scale;
#pragma unroll
    for (int r = 0; r < R; ++r, top *= 0.5f) clip |= __ballot(signed_max || !((io.inp_res > 0.0f ? rintf(top) * io.inp_res : top) <= io.inp_bound)) ? 1 << r : 0;
    if (lane == 0) sh.clip[wave] = clip;
  }
  // (noise-management value of a sample with the largest input m)
  __device__ __forceinline__ float nm_of(float m) const {
    const IoDev &io = a.io;
    if (io.noise_management == RPU_NM_ABS_MAX || io.noise_management == RPU_NM_MAX) return io.nm_thres > 0.0f ? fminf(m, io.nm_thres) : m;
    if (io.noise_management == RPU_NM_CONSTANT) return io.nm_thres > 0.0f ? io.nm_thres : 1.0f;
    return 1.0f;
  }

  typedef f32x4 Sums[R][NB];
  // how the inputs of a lane's sample are converted
  struct Converter {
    int clip;
    float scale, resolution, reciprocal;
  };
  // the products of a step
  __device__ __forceinline__ void add(const Weights &w, int step, const Converter &by, Sums &sums) const {
    const IoDev &io = a.io;
    const float *const from = q + (lane & 15) * ld + step * KSTEP + 8 * (lane >> 4);
    const f32x4 x[2] = {*reinterpret_cast<const f32x4 *>(from), *reinterpret_cast<const f32x4 *>(from + 4)};
    float v[NB][8], in[R][8];
    operands(w, v);
#pragma unroll
    for (int j = 0; j < 8; ++j) in[0][j] = x[j / 4][j & 3] * by.scale;
    if (step * KSTEP + KSTEP > a.K) {
      // beyond the row: the next one's weights, and zeros times a scale that is infinite where the row's largest input is below
      // 2^-128
      const int left = a.K - step * KSTEP - 16 * ((lane >> 4) & 1) - (lane >> 5);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        in[0][j] = 2 * j < left ? in[0][j] : 0.0f;
        if constexpr (!WOC) {
#pragma unroll
          for (int n = 0; n < NB; ++n) v[n][j] = 2 * j < left ? v[n][j] : 0.0f;
        }
      }
    }
    if (by.resolution > 0.0f) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float y = quotient(in[0][j], by.resolution, by.reciprocal);
#pragma unroll
        for (int r = 0; r < R; ++r, y *= 0.5f) in[r][j] = rintf(y) * by.resolution;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int r = 1; r < R; ++r) in[r][j] = in[r - 1][j] * 0.5f;
      }
    }
    if (by.clip) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if (!((by.clip >> r) & 1)) break; // (a round's inputs are halves of those of the round before)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          float y = in[r][j];
          y = (y > io.inp_bound) ? io.inp_bound : y;
          in[r][j] = (y < -io.inp_bound) ? -io.inp_bound : y;
        }
      }
    }
    if (io.inp_asym != 0.0f) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int j = 0; j < 8; ++j) in[r][j] = in[r][j] < 0.0f ? in[r][j] * (1.0f - io.inp_asym) : in[r][j];
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int n = 0; n < NB; ++n) sums[r][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[n][j], in[r][j], sums[r][n], 0, 0, 0);
      }
    }
  }
  template <int N> __device__ __forceinline__ void start(Weights (&w)[N], int o_first) const {
#pragma unroll
    for (int u = 0; u < N; ++u) load(w[u], min(s_begin + u, steps - 1), o_first);
  }
  // w as start() leaves it; the partial sums go to `part` (after a barrier where that is where the inputs are)
  __device__ __forceinline__ void contract(Weights (&w)[AHEAD], int o_first, bool in_place) const {
    const Converter by = {uniform(sh.clip[0] | sh.clip[1] | sh.clip[2] | sh.clip[3]), sh.scale[lane & 15], a.io.inp_res, 1.0f / a.io.inp_res};
    Sums sums;
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int n = 0; n < NB; ++n) sums[r][n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    for (int step = s_begin; step < s_end; step += AHEAD) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        if (step + u >= s_end) break;
        add(w[u], step + u, by, sums);
        if (step + u + AHEAD < s_end) load(w[u], step + u + AHEAD, o_first);
      }
    }
    if (in_place) __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
      for (int n = 0; n < NB; ++n) {
#pragma unroll
        for (int i = 0; i < 4; ++i) part[r * ROUND + ((wave * NB + n) * 4 + i) * 64 + lane] = sums[r][n][i];
      }
    }
    __syncthreads();
  }

  // Adds up the partial sums of round `slot` and takes them through the ADC stage of `round`, marks to hits[slot], factors from
  // fin[slot]: COUNT outputs of sample lane % 16 to a thread, if it has its bit set in `live`.  COUNT = NB: those of row wave of
  // each four, NB (4 (lane / 16) + wave) .. of the block.  NB = 1, COUNT = 4: all four, one wave to a round (four outputs share
  // their draws).  rows: where the results are kept, null: the call's output; through: other workgroups read them, or have
  // written the same outputs
  template <int COUNT> __device__ __forceinline__ void finish(int b0, int o_first, int round, int slot, unsigned live, float *rows, bool through) const {
    static_assert(COUNT == NB || (NB == 1 && COUNT == 4));
    const IoDev &io = a.io;
    const int s = lane & 15, b = b0 + s, o0 = o_first + (COUNT == NB ? NB * (4 * (lane >> 4) + wave) : 4 * (lane >> 4));
    float y[COUNT];
#pragma unroll
    for (int n = 0; n < COUNT; ++n) {
      const float *const p = part + slot * ROUND + (COUNT == NB ? n * 4 + wave : n) * 64 + lane;
      y[n] = ((p[0] + p[NB * 256]) + p[2 * NB * 256]) + p[3 * NB * 256];
    }
    const float f = sh.fin[slot * S + s];
    if (o0 >= a.O || !((live >> s) & 1u)) return;
    float noise[COUNT];
    if (io.out_noise > 0.0f) {
      const Philox4 r = philox4x32_10((uint32_t)(o0 >> 2), (uint32_t)b, a.call, RNG_OUT_NOISE | ((uint32_t)round << 8), a.key.k0, a.key.k1);
      if constexpr (COUNT == 4) {
        box_muller(r.v[0], r.v[1], noise[0], noise[1]);
        box_muller(r.v[2], r.v[3], noise[2], noise[3]);
      } else {
        float n0, n1;
        box_muller((o0 & 2) ? r.v[2] : r.v[0], (o0 & 2) ? r.v[3] : r.v[1], n0, n1);
        noise[0] = COUNT == 1 && (o0 & 1) ? n1 : n0;
        if constexpr (COUNT == 2) noise[1] = n1;
      }
    }
    int up = 0, lo = 0;
    const float reciprocal = 1.0f / io.out_res;
    float *const out = rows ? rows + (long)b * a.O + o0 : a.out + (long)b * a.out_sb + (long)o0 * a.out_so;
    const long so = rows ? 1 : a.out_so;
#pragma unroll
    for (int n = 0; n < COUNT; ++n) {
      const int o = o0 + n;
      float v = y[n];
      if (io.out_asym > 0.0f) v = v < 0.0f ? v * (1.0f - io.out_asym) : v;
      if (io.out_noise > 0.0f) v += io.out_noise * noise[n];
      if (io.out_res > 0.0f) v = rintf(quotient(v, io.out_res, reciprocal)) * io.out_res;
      const bool over = v > io.out_bound, under = v < -io.out_bound;
      v = over ? io.out_bound : (under ? -io.out_bound : v);
      if (f == 0.0f) { // zero input: the reference short-cuts to a zero output
        v = 0.0f;
      } else {
        if (over && o < a.O) up = o + 1;
        if (under && o < a.O) lo = o + 1;
        v *= f;
      }
      if (o >= a.O - a.out_drop) continue;
      if (through) __hip_atomic_store(out + n * so, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else out[n * so] = v;
    }
    if (up) atomicMax(&sh.hits[2 * S * slot + s], up);
    if (lo) atomicMax(&sh.hits[2 * S * slot + S + s], lo);
  }

  // State of the samples, sample s in lane s of every wave: whether it is in the round that is being looked at, how many it
  // has run, its noise-management value
  struct Samples {
    bool live;
    int rounds;
    float nm;
  };
  // the samples that go on after `round`, whose marks are at hits[slot]; returns their number as bits
  __device__ __forceinline__ unsigned advance(int b0, int round, int slot, Samples &my) const {
    if (my.live) {
      const int up = sh.hits[2 * S * slot + lane], lo = sh.hits[2 * S * slot + S + lane];
      const bool failed = a.io.bm_test_negative_bound ? (up > 0 || lo > 0) : (up > lo);
      float nm = my.nm, red = two_to(round), fin;
      (void)round_scales(a, nm, red, fin);
      my.live = failed && round + 1 < a.max_rounds && next_round_params(a, round, b0 + lane, fin, nm, red);
      my.rounds += my.live ? 1 : 0;
    }
    return (unsigned)__ballot(my.live);
  }

  __device__ __forceinline__ void run(const int block_b, const int block_o) {
    const int t = (int)threadIdx.x, b0 = block_b * S, blocks_o = (a.O + OB - 1) / OB;
    // inputs first, then weights: the inputs are waited for first
    Inputs x;
    load_inputs(x, b0, 0);
    Weights w[AHEAD];
    start(w, block_o * OB);
    if (t < R * 2 * S) sh.hits[t] = 0;
    fill(x, b0, 0.0f, false, 1.0f);
    __syncthreads();
    Samples my;
    my.nm = nm_of(sh.max[lane % S]);
    my.live = lane < S && b0 + lane < a.m_batch;
    {
      float fin;
      (void)round_scales(a, my.nm, two_to(min(lane / S, R - 1)), fin);
      my.rounds = fin == 0.0f ? 0 : 1; // (lanes below S: of round 0)
      if (t < R * S) sh.fin[t] = fin;
    }
    unsigned live = (1u << min(S, a.m_batch - b0)) - 1u;
    contract(w, block_o * OB, true);
    const bool managed = a.max_rounds > 1, shared = managed && blocks_o > 1;
    float *const rows[3] = {nullptr, a.dual.buf[1], a.dual.buf[2]};
    if constexpr (NB == 1 && R == 3) {
      if (wave < R) finish<4>(b0, block_o * OB, wave, wave, live, wave == 0 ? rows[0] : (wave == 1 ? rows[1] : rows[2]), shared || wave > 0);
    } else {
#pragma unroll 1
      for (int r = 0; r < R; ++r) finish<NB>(b0, block_o * OB, r, r, live, r == 0 ? rows[0] : (r == 1 ? rows[1] : rows[2]), shared || r > 0);
    }
    if (managed) {
      // what this workgroup stored has arrived before it counts itself off, and so have its marks
      __syncthreads();
      if (shared) {
        int *const marks = a.few + a.m_batch; // [R][2][m_batch]: upper, lower; the counters before them
        const bool mine = t < R * 2 * S && b0 + t % S < a.m_batch;
        int *const mark = marks + (t / S) * a.m_batch + b0 + t % S;
        const int hit = mine ? sh.hits[t] : 0;
        if (hit) {
          const int old = atomicMax(mark, hit);
          asm volatile("" ::"v"(old));
        }
        __builtin_amdgcn_s_waitcnt(0);
        const int any = __syncthreads_or(hit != 0);
        // counter: workgroups in the lower half, those with marks in the upper
        if (t == 0) {
          const int before = atomicAdd(&a.few[block_b], any ? 0x10001 : 1);
          sh.last = (before & 0xffff) != blocks_o - 1 ? 0 : (before >= 0x10000 || any ? 2 : 1);
        }
        __syncthreads();
        const int last = uniform(sh.last);
        if (!last) return;
        // the last one reads the marks of all, and leaves them and the counter as it found them at first: zero
        if (t == 0) __hip_atomic_store(&a.few[block_b], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (last == 2) {
          if (t < R * 2 * S) sh.hits[t] = mine ? atomicExch(mark, 0) : 0;
          __syncthreads();
        }
      } else if (R > 1) {
        __builtin_amdgcn_s_waitcnt(0); // (what copy_out() reads)
        __syncthreads();
      }
      unsigned chosen[R]; // samples whose result is that of round r
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const unsigned before = live;
        live = advance(b0, r, r, my);
        chosen[r] = before & ~live;
      }
      if constexpr (R > 1) {
        if (chosen[1] | chosen[2]) copy_out(b0, chosen[1], chosen[2]);
      }
      if (live) { // the same for all threads
        __syncthreads();
        alone(block_b, live, my);
      }
    }
    if ((shared || block_o == 0) && wave == 0) {
      if (lane < S && b0 + lane < a.m_batch) a.st.rounds[b0 + lane] = my.rounds;
      const bool more = __ballot(lane < S && b0 + lane < a.m_batch && my.rounds > 1) != 0;
      const bool beyond = __ballot(lane < S && b0 + lane < a.m_batch && my.rounds > MOST_ROUNDS) != 0; // of the call's own, R may be 1
      // the host picks R by what it knows of the last calls: the last one it hears of, the last one with samples that went on
      if (managed && lane == 0) {
        if (more) __hip_atomic_store(a.few_seen, a.few_call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (beyond) __hip_atomic_store(a.few_seen + 2, a.few_call + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); // (0: none)
        if (block_b == 0) __hip_atomic_store(a.few_seen + 1, a.few_call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  // results of round 1 / 2 to the output, sixteen threads to a sample, 32 values of a thread in flight
  __device__ __forceinline__ void copy_out(int b0, unsigned first, unsigned second) const {
    const int t = (int)threadIdx.x, s = t >> 4;
    if (!(((first | second) >> s) & 1u)) return;
    const int stored = a.O - a.out_drop;
    const __amdgpu_buffer_rsrc_t first_rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.dual.buf[1]), 0, (int)(4u * (unsigned)a.m_batch * (unsigned)a.O), 0x00020000);
    const __amdgpu_buffer_rsrc_t second_rows = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.dual.buf[2]), 0, (int)(4u * (unsigned)a.m_batch * (unsigned)a.O), 0x00020000);
    const unsigned row_at = 4u * (unsigned)((long)(b0 + s) * a.O);
    for (int o0 = 4 * (t & 15); o0 < stored; o0 += 512) {
      f32x4 v[8];
      if ((first >> s) & 1u) {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(first_rows, row_at + 4u * (unsigned)(o0 + 64 * u), 0, THROUGH));
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(second_rows, row_at + 4u * (unsigned)(o0 + 64 * u), 0, THROUGH));
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int end = o0 + 64 * u + 4;
        if (a.out_so == 1 && end <= stored) {
          // up to the last output of the block's last sample (for one sample the distance to the next may be anything)
          const unsigned end_of_block = (unsigned)((long)(min(S, a.m_batch - b0) - 1) * a.out_sb + stored);
          const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(a.out + (long)b0 * a.out_sb, 0, (int)(4u * end_of_block), 0x00020000);
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_bits, v[u]), out, 4u * (unsigned)(s * a.out_sb + end - 4), 0, THROUGH);
          continue;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int o = o0 + 64 * u + c;
          if (o < stored) __hip_atomic_store(a.out + (long)(b0 + s) * a.out_sb + (long)o * a.out_so, v[u][c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
  }
  // The rounds from R on for the samples of `live`, by this workgroup, 32 outputs at a time
  __device__ __forceinline__ void alone(int block_b, unsigned live, Samples &my) {
    Alone all(a, q, sh);
    all.part = q + S * ld;
    for (int round = R; live; ++round) live = all.whole_round(block_b * S, round, live, my.live, my.rounds, my.nm);
  }
  __device__ __forceinline__ unsigned whole_round(int b0, int round, unsigned live, bool &on, int &rounds, float &nm) {
    const int t = (int)threadIdx.x;
    Inputs x;
    load_inputs(x, b0, 0);
    Weights w[AHEAD];
    start(w, 0);
    if (t < 2 * S) sh.hits[t] = 0;
    fill(x, b0, __shfl(nm, t >> 4), true, two_to(round));
    if (t < S) {
      float fin;
      (void)round_scales(a, nm, two_to(round), fin);
      sh.fin[t] = fin;
    }
    __syncthreads();
    for (int o_first = 0; o_first < a.O; o_first += OB) {
      contract(w, o_first, false);
      start(w, o_first + OB); // (beyond the outputs: not used)
      finish<NB>(b0, o_first, round, 0, live, nullptr, true);
      __syncthreads(); // the partial sums have been read
    }
    Samples my{on, rounds, nm};
    live = advance(b0, round, 0, my);
    on = my.live;
    rounds = my.rounds;
    __syncthreads();
    return live;
  }

  // workgroup number n -> block of samples, block of outputs.  From eight blocks of outputs on, those of an XCD (n % 8) are
  // next to each other: each L2 holds its own part of the weights.
  static __host__ __device__ int workgroups(int O, int m_batch) {
    const int bo = (O + OB - 1) / OB, bb = (m_batch + S - 1) / S;
    return bo < 8 ? bo * bb : 8 * ((bo + 7) / 8) * bb;
  }
  static __device__ __forceinline__ bool block_of(const MvmArgs &a, int n, int &block_b, int &block_o) {
    const int bo = (a.O + OB - 1) / OB;
    if (bo < 8) {
      block_o = n % bo;
      block_b = n / bo;
    } else {
      const int per = (bo + 7) / 8, m = n >> 3;
      block_o = (n & 7) * per + m % per;
      block_b = m / per;
    }
    return block_o < bo && block_b * S < a.m_batch;
  }
};

template <bool WOC, int NB, int R> __global__ __launch_bounds__(256, 2) void k_mvm_whole(MvmArgs a) {
  extern __shared__ __attribute__((aligned(16))) float whole_lds[];
  __shared__ WholeShared sh;
  typedef MvmWhole<WOC, NB, R> Whole;
  int block_b, block_o;
  if (Whole::block_of(a, (int)blockIdx.x, block_b, block_o)) Whole(a, whole_lds, sh).run(block_b, block_o);
}

// workgroups that the GPU holds at once: two to a CU by their registers, one where rows of more than 1088 inputs take half of
// its 160 KB of LDS
template <int NB, int R> int held(int K, int cus) {
  return std::min<int>(2, (int)(160 * 1024 / (MvmWhole<false, NB, R>::lds_bytes(K) + sizeof(WholeShared)))) * cus;
}

} // namespace

// Whether quotient() is the division for every value that a converter does not clip
static bool steps_are_exact(float resolution, float bound) {
  return !(resolution > 0.0f) || (resolution > 0x1p-60f && resolution < 0x1p60f && bound < 0x1p59f * resolution);
}

// The outputs of a workgroup: 16 where the GPU holds all of the call's workgroups at once, else 64, up to one set of those with
// bound management and two without.  us, the launches one by one / this one (forward: weights that saturate round 0 / that do
// not):
//   16 outputs: 512 x 512, 100 samples 27.1 / 15.8, 18.2 / 10.8; 256 28.5 / 21.3, 19.3 / 14.6; 785 -> 256, 64 39.3 / 17.2, 27.0 /
//   11.0; 513 -> 128, 512 45.2 / 18.0, 27.7 / 11.4; 1024 x 1024, 128 37.5 / 28.5, 22.2 / 18.1; 1500 x 1500 (one workgroup to a CU),
//   32 47.0 / 27.2, 28.0 / 15.3; backward 512 x 512, 400 15.0 / 9.3; 1024 x 1024, 128 17.6 / 11.8
//   64 outputs: 512 x 512, 512 31.4 / 28.7, 21.7 / 15.9, 1024 41.9 / 41.0, 26.9 / 20.1; 785 -> 256, 1024 52.6 / 35.6; 1024 x 1024, 300
//   60.9 / 50.9, 512 65.2 / 58.2; backward 1024 x 1024, 256 18.4 / 13.5, 1000 43.3 / 35.8; 512 x 512, 2000 32.7 / 23.2
//   beyond: forward 512 x 512, 1500 63 / 67, 38 / 33; 256 x 256, 4000 48 / 56, 33 / 26; 1024 x 1024, 768 88 / 97, 46 / 51.
// Rows along the inputs whose length is no multiple of 16 gain up to two sets of two workgroups to a CU: the other launches read
// them in unaligned pieces.  785 -> 256, 4000 155 / 97, 69 / 48; 300 -> 200, 3000 60 / 59, 42 / 28; 900 -> 700, 800 98 / 91, 52 / 44
// (1500 x 1500, one workgroup to a CU, 200 81 / 81, 37 / 43).
// Long aligned rows along the inputs, a single round: not with 64 outputs, whose 64 rows a wave reads 16 bytes at a time from 16
// of them (1024 x 1024 stored the other way round, backward, 256 16.6 / 16.6, 300 22.1 / 23.6, 1000 38 / 46).
// Large matrices whose 32 x 32 tiles are one to a CU stay with the others: these share the launch of rounds 0 and 1 there (k_mvm_dual)
// and read the weights once for 32 samples, where all samples end in round 1.  Without saturation / in round 1 / in round 2, the others
// and this one: 1024 x 1024, 256 samples 25.2 21.5 / 36.4 38.6 / 42.0 38.9, 160 23.1 19.8 / 34.1 35.0 / 38.7 35.4; 1024 -> 768, 320 25.1 25.8
// / 37.6 50.5 / 42.6 50.8; 544 -> 2048, 128 24.2 20.5 / 34.8 40.2 / 39.3 40.3; 1504 x 1504, 96 25.7 24.0 / 39.1 44.7 / 44.9 45.0 (so a call
// that does not saturate would gain up to 16 %).
int mvm_whole_outputs(const MvmArgs &a) {
  const IoDev &io = a.io;
  const int nm = io.noise_management, cus = a.cus > 0 ? a.cus : current_device_cus();
  if (io.perfect || a.in_index || a.pre_add || a.skip_if_zero || a.nm_phase || a.small_tiles_only || a.K > 2048 || a.K <= a.in_one) return 0;
  if (io.inp_sto_round || io.out_sto_round || io.inp_noise > 0.0f || !(io.inp_bound < 0x1p96f)) return 0;
  if (!steps_are_exact(io.inp_res, io.inp_bound) || !steps_are_exact(io.out_res, io.out_bound)) return 0;
  if (nm != RPU_NM_NONE && nm != RPU_NM_CONSTANT && nm != RPU_NM_ABS_MAX && nm != RPU_NM_MAX) return 0;
  if (io.bound_management != RPU_BM_NONE && (io.bound_management != RPU_BM_ITERATIVE || a.transposed)) return 0;
  // two rounds of short rows: the third one that is worked out with them costs more than their launches (16 -> 1024, 300 samples 22.9 /
  // 26.8; 64 -> 32, 4096 31.4 / 32.6)
  if (a.max_rounds == 2 && a.K <= 64) return 0;
  if (mvm_uses_large_tiles(a.m_batch, a.O)) return 0;
  // offsets of 32 bits
  if ((long)(a.w_oc ? a.K : a.O) * a.w_ld >= 1L << 28 || (long)a.m_batch * a.O >= 1L << 28) return 0;
  if ((long)a.m_batch * a.in_sb + (long)a.K * a.in_sk >= 1L << 28 || a.out_sb >= 1L << 24) return 0;
  const bool managed = a.max_rounds > 1, rounds = a.max_rounds > 2;
  if (managed && a.m_batch > mvm_whole_batch(a)) return 0;
  if (MvmWhole<false, 1, 1>::workgroups(a.O, a.m_batch) <= (rounds ? held<1, 3>(a.K, cus) : held<1, 1>(a.K, cus))) return 16;
  const bool ragged = !a.w_oc && (a.K & 15) != 0;
  const int tiles = mvm_round_workgroups(a);
  if (rounds && !ragged && a.K > 512 && (long)a.K * a.O > 1L << 19 && tiles <= cus && 2 * tiles > cus) return 0;
  if (!managed && !ragged && !a.w_oc && a.K > 512) return 0;
  const int set = rounds ? held<4, 3>(a.K, cus) : held<4, 1>(a.K, cus);
  const int sets = ragged ? set / cus : (managed ? 1 : 2);
  return MvmWhole<false, 4, 1>::workgroups(a.O, a.m_batch) <= sets * set ? 64 : 0;
}

// (the room for more samples than 4096 would be more than the rest of a small tile)
int mvm_whole_batch(const MvmArgs &a) {
  const int cus = a.cus > 0 ? a.cus : current_device_cus();
  return std::min(4096, S * (4 * cus / MvmWhole<false, 4, 1>::workgroups(a.O, S)));
}

void launch_mvm_whole(const MvmArgs &a, int outputs, int rounds, hipStream_t s) {
#define RPU_LAUNCH_WHOLE(WOC, NB, R) \
  hipLaunchKernelGGL((k_mvm_whole<WOC, NB, R>), dim3((unsigned)MvmWhole<WOC, NB, R>::workgroups(a.O, a.m_batch)), dim3(256), \
                     (MvmWhole<WOC, NB, R>::lds_bytes(a.K)), s, a)
#define RPU_PICK_WHOLE(NB, R) \
  do { \
    if (a.w_oc) RPU_LAUNCH_WHOLE(true, NB, R); \
    else RPU_LAUNCH_WHOLE(false, NB, R); \
  } while (0)
  if (outputs == 64) {
    if (rounds == 3) RPU_PICK_WHOLE(4, 3);
    else RPU_PICK_WHOLE(4, 1);
  } else {
    if (rounds == 3) RPU_PICK_WHOLE(1, 3);
    else RPU_PICK_WHOLE(1, 1);
  }
#undef RPU_PICK_WHOLE
#undef RPU_LAUNCH_WHOLE
}

} // namespace rpu_amd
