// Noisy matrix-vector products of small batches in one launch: noise management, DAC, contraction, ADC and every
// bound-management round.
//
// A batch of a few dozen samples is latency from end to end: an init kernel, a round of 32 x 32 tiles on a handful of CUs
// (each wave a chain of K / 4 matrix steps, mostly padding for one sample), and a launch for the rounds that are expected to
// be empty -- 4, 12 and 4 us for one sample on a 512 x 512 tile.  Here a workgroup takes S samples and OB outputs.  It
// reads and quantizes its samples' rows itself (every workgroup of a sample does: a few elements per thread), multiplies
// with plain fp32 multiply-adds, 64 weights of a thread in flight, and adds its threads' partial sums (chains of K / 16 terms)
// through LDS.  The workgroups of a sample count themselves off; the
// last one knows whether the sample saturated.  Where the tile's recent calls did, R = 3: the workgroups multiply the same
// weights with the inputs of rounds 0, 1 and 2 (V = R S rows) and keep all results, and the last one copies out what
// stands (as k_mvm_dual); a round beyond those it runs alone, block by block.  No list, no later launch.
// What bounds it: the chain from launch to loads, maximum, ADC and two atomics (about 1 us each), and how fast its code comes:
// it runs once through, and a jump over code that the call does not need waits for instructions.  So the random draws of the
// converters are compiled in only where
// the settings have them (STOCH), a thread works on one sample's row and not on all, loads have no branches (buffer
// loads: what lies beyond the matrix reads as zero) and what few calls need stands at the end.
// One sample on 512 x 512 8.8 -> 7.8 us a launch, 12 tiles of 512 x 512 with 8 samples 17.2 -> 10.1, 785 x 300 with 37 samples and
// three rounds 23.2 -> 16.8, backward 16.6 -> 7.0, 129 x 10 with 64 samples 9.3 -> 5.6.
// The streams of random numbers are those of the other kernels (element k, sample, round; four outputs to a draw).
#include "bf16_parts.h"
#include "mvm_device.h"

#include <algorithm>
#include <cmath>

namespace rpu_amd {

namespace {

// the largest value of a wave, the same in all lanes
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, row_xor<8>(v));
  v = fmaxf(v, row_xor<4>(v));
  v = fmaxf(v, row_xor<2>(v));
  v = fmaxf(v, row_xor<1>(v));
  const int i = __builtin_bit_cast(int, v);
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(i, i, 0x142, 0xa, 0xf, false))); // rows 1 and 3: of row 0, 2
  const int j = __builtin_bit_cast(int, v);
  v = fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(j, j, 0x143, 0xc, 0xf, false))); // rows 2 and 3: of row 1
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

constexpr int FEW_MOST_VALUES = 12; // R S at most
struct FewShared {
  int hits[2 * FEW_MOST_VALUES]; // [R][2][S] saturation marks: upper, lower
  float fin[FEW_MOST_VALUES];    // [R][S] output factors
  float max[4];                  // largest inputs, a wave each
  int last;
};

template <bool WOC, int S, int OB, int R, bool STOCH> struct MvmFew {
  typedef MvmFew<WOC, S, 64, 1, STOCH> Alone; // see alone()
  static constexpr int V = R * S;
  static_assert(V <= FEW_MOST_VALUES && (R == 1 || R == 3));
  // A load of a wave, and the order of every sum, are the same in all variants, so that any of them can run a call: part p of
  // an output's sixteen takes k = 4 p .. 4 p + 3 (mod 64) in ascending order, and the parts are added as a tree.
  //   weights along k: sixteen lanes next to each other read 64 weights of a row, a wave OB / 4 rows
  //   along the outputs: sixteen lanes read OB outputs of a row, each wave sixteen rows of 64
  static constexpr int PARTS = 16, K_LOAD = 64;
  static constexpr int WIDTH = WOC ? OB / 16 : 4;            // weights of a load
  static constexpr int LOADS = WOC ? 4 : OB / 16;            // loads of a thread for 64 contraction indices
  static constexpr int OUTPUTS = OB / 16;                    // sums of a thread, per row of inputs
  static constexpr int AHEAD = 256 / OB;                     // of 64 contraction indices, in flight: 64 weights of a thread
  static constexpr int PER_SUM = 256 / (S * OB);             // threads that add up an output
  static constexpr int PITCH = PARTS + 1;                    // of an output's partial sums in LDS
  static constexpr int THREADS = 256 / S;                    // threads of a sample's row
  static constexpr int STEP = 512, PER_THREAD = STEP / THREADS; // elements of a row, and of a thread, in flight together
  typedef float Load __attribute__((ext_vector_type(WIDTH)));
  typedef Load Chunk[LOADS]; // weights of 64 contraction indices

  const MvmArgs &a;
  const float *x_row; // the row of this thread's sample
  float *xs, *part;   // LDS: [R][S][k_len] quantized inputs, zero padded; [S][OB][PITCH]
  FewShared &sh;
  int k_len, whole;   // whole: blocks of 64 contraction indices without a branch at the row's end
  int lane, wave, s_mine, at; // this thread's sample of the block, and its first element of that row
  unsigned row_bytes, bytes;
  __amdgpu_buffer_rsrc_t w_buffer;
  unsigned w_at[WOC ? 1 : LOADS];

  static __host__ __device__ int padded(int K) { return (K + K_LOAD - 1) / K_LOAD * K_LOAD; }
  static __host__ __device__ size_t lds_bytes(int K) {
    const size_t own = sizeof(float) * ((size_t)V * padded(K) + S * OB * PITCH);
    if constexpr (OB == 64 && R == 1) return own;
    else return own > Alone::lds_bytes(K) ? own : Alone::lds_bytes(K);
  }

  __device__ __forceinline__ MvmFew(const MvmArgs &a_, float *lds, FewShared &shared_)
      : a(a_), xs(lds), part(lds + V * padded(a_.K)), sh(shared_), k_len(padded(a_.K)), lane((int)threadIdx.x & 63),
        wave(uniform((int)threadIdx.x >> 6)) {
    s_mine = wave * S / 4;
    at = (int)threadIdx.x % THREADS;
    whole = WOC ? k_len / K_LOAD : a.K / K_LOAD; // (along the outputs, rows beyond the last one are beyond the matrix)
    row_bytes = 4u * (unsigned)a.w_ld;
    bytes = ((unsigned)(WOC ? a.K : a.O) - 1u) * row_bytes + 4u * (unsigned)(WOC ? a.O : a.K);
    w_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.w), 0, (int)bytes, 0x00020000);
  }

  // from which output on the following loads are
  __device__ __forceinline__ void at_outputs(int o_first) {
    if constexpr (WOC) {
      w_at[0] = (unsigned)((wave * 4 + (lane >> 4)) * 4) * row_bytes + 4u * (unsigned)(o_first + WIDTH * (lane & 15));
    } else {
#pragma unroll
      for (int l = 0; l < LOADS; ++l) w_at[l] = (unsigned)(o_first + (wave * LOADS + l) * 4 + (lane >> 4)) * row_bytes + 16u * (unsigned)(lane & 15);
    }
  }
  // weights of block `k` of 64 contraction indices.  What lies beyond the matrix reads as zero, dword by dword; what lies beyond
  // a row and within the matrix belongs to outputs that are not stored, or to block `whole`, which rest() masks.
  __device__ __forceinline__ void load(Chunk &w, int k) const {
#pragma unroll
    for (int l = 0; l < LOADS; ++l) {
      const unsigned from = WOC ? w_at[0] + (unsigned)(k * K_LOAD + l) * row_bytes : w_at[WOC ? 0 : l] + 4u * K_LOAD * (unsigned)k;
      if constexpr (WIDTH == 4) w[l] = __builtin_bit_cast(Load, __builtin_amdgcn_raw_buffer_load_b128(w_buffer, from, 0, 0));
      else if constexpr (WIDTH == 2) w[l] = __builtin_bit_cast(Load, __builtin_amdgcn_raw_buffer_load_b64(w_buffer, from, 0, 0));
      else w[l][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(w_buffer, from, 0, 0));
    }
  }
  typedef float Sums[V][OUTPUTS];
  __device__ __forceinline__ void add(const Chunk &w, int k, Sums &sums) const {
    const int first = k * K_LOAD + (WOC ? (wave * 4 + (lane >> 4)) * 4 : 4 * (lane & 15));
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const f32x4 x = *reinterpret_cast<const f32x4 *>(xs + v * k_len + first);
#pragma unroll
      for (int l = 0; l < LOADS; ++l) {
#pragma unroll
        for (int q = 0; q < WIDTH; ++q) {
          if (WOC) sums[v][q] = __builtin_fmaf(w[l][q], x[l & 3], sums[v][q]);
          else sums[v][l] = __builtin_fmaf(w[l][q], x[q & 3], sums[v][l]);
        }
      }
    }
  }

  // The first AHEAD blocks, in two halves: the second one is asked for once the inputs have come.
  struct Weights {
    Chunk now[AHEAD], rest; // rest: block `whole`, part of which lies beyond the rows' ends (only with weights along k)
  };
  template <int HALF> __device__ __forceinline__ void start(Weights &w) const {
    if constexpr (HALF == 0) {
#pragma unroll
      for (int u = 0; u < AHEAD / 2; ++u) load(w.now[u], u);
      if (!WOC) load(w.rest, whole);
    } else if (whole > AHEAD / 2) {
#pragma unroll
      for (int u = AHEAD / 2; u < AHEAD; ++u) load(w.now[u], u);
    }
  }
  // this thread's sums; w as start() leaves it
  __device__ __forceinline__ void contract(Weights &w, Sums &sums) const {
#pragma unroll
    for (int v = 0; v < V; ++v) {
#pragma unroll
      for (int o = 0; o < OUTPUTS; ++o) sums[v][o] = 0.0f;
    }
    int k = 0;
    for (; k + AHEAD < whole; k += AHEAD) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        add(w.now[u], k + u, sums);
        load(w.now[u], k + u + AHEAD < whole ? k + u + AHEAD : whole); // (block `whole` is at hand and is not read here)
      }
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      if (k + u >= whole) break;
      add(w.now[u], k + u, sums);
    }
    if (!WOC && whole * K_LOAD < a.K) {
      const int left = a.K - whole * K_LOAD - 4 * (lane & 15);
#pragma unroll
      for (int l = 0; l < LOADS; ++l) {
#pragma unroll
        for (int q = 0; q < WIDTH; ++q) w.rest[l][q] = q < left ? w.rest[l][q] : 0.0f;
      }
      add(w.rest, whole, sums);
    }
  }
  // the sums of round r (of R) to LDS
  __device__ __forceinline__ void spread(const Sums &sums, int r) const {
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
      for (int o = 0; o < OUTPUTS; ++o) {
        const float v = sums[r * S + s][o];
        if (WOC) part[(s * OB + OUTPUTS * (lane & 15) + o) * PITCH + wave * 4 + (lane >> 4)] = v;
        else part[(s * OB + (wave * OUTPUTS + o) * 4 + (lane >> 4)) * PITCH + (lane & 15)] = v;
      }
    }
  }

  // adds up the partial sums and takes them through the ADC stage of `round` (mvm_adc_values, an output per thread), for the
  // samples of the block with their bit set in `live`, marks to hits[slot], factors from fin[slot].  rows: where the results are
  // kept, null: the call's output; through: other workgroups read them, or have written the same outputs
  __device__ __forceinline__ void finish(int b0, int o_first, int round, int slot, unsigned live, float *rows, bool through) {
    const int t = (int)threadIdx.x, sum = t / PER_SUM, s = sum / OB, o = o_first + sum % OB;
    constexpr int MINE = PARTS / PER_SUM;
    float p[MINE];
#pragma unroll
    for (int i = 0; i < MINE; ++i) p[i] = part[sum * PITCH + PER_SUM * i + t % PER_SUM];
    const float f = sh.fin[slot * S + s];
#pragma unroll
    for (int half = MINE / 2; half > 0; half >>= 1) {
#pragma unroll
      for (int i = 0; i < half; ++i) p[i] += p[i + half];
    }
    float y = p[0];
    if constexpr (PER_SUM > 8) y += row_xor<8>(y);
    if constexpr (PER_SUM > 4) y += row_xor<4>(y);
    if constexpr (PER_SUM > 2) y += row_xor<2>(y);
    if constexpr (PER_SUM > 1) y += row_xor<1>(y);
    if (t % PER_SUM != 0 || o >= a.O || !((live >> s) & 1u)) return;
    const IoDev &io = a.io;
    const int b = b0 + s;
    if (io.out_asym > 0.0f) y = y < 0.0f ? y * (1.0f - io.out_asym) : y;
    if (io.out_noise > 0.0f) {
      const Philox4 r = philox4x32_10((uint32_t)(o >> 2), (uint32_t)b, a.call, RNG_OUT_NOISE | ((uint32_t)round << 8), a.key.k0, a.key.k1);
      float n0, n1;
      box_muller((o & 2) ? r.v[2] : r.v[0], (o & 2) ? r.v[3] : r.v[1], n0, n1);
      y += io.out_noise * ((o & 1) ? n1 : n0);
    }
    if (io.out_res > 0.0f) {
      float q = y / io.out_res;
      if (STOCH && io.out_sto_round) {
        const Philox4 r = philox4x32_10((uint32_t)o, (uint32_t)b, a.call, RNG_OUT_SR | ((uint32_t)round << 8), a.key.k0, a.key.k1);
        q = q + (u32_to_uniform(r.v[0]) - 0.5f);
      }
      y = rintf(q) * io.out_res;
    }
    const bool over = y > io.out_bound, under = y < -io.out_bound;
    y = over ? io.out_bound : (under ? -io.out_bound : y);
    if (f == 0.0f) { // zero input: the reference short-cuts to a zero output
      y = 0.0f;
    } else {
      if (over) atomicMax(&sh.hits[2 * S * slot + s], o + 1);
      if (under) atomicMax(&sh.hits[2 * S * slot + S + s], o + 1);
      y *= f;
    }
    if (o >= a.O - a.out_drop) return;
    float *out = rows ? rows + (long)b * a.O + o : a.out + (long)b * a.out_sb + (long)o * a.out_so;
    if (through) __hip_atomic_store(out, y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // through the XCD's own L2
    else *out = y;
  }

  // element k of this thread's row (beyond the row: some element of it)
  __device__ __forceinline__ float stored_input(int k) const {
    const int stored = mvm_stored(a);
    const float v = x_row[(unsigned)min(k, stored - 1) * (unsigned)a.in_sk];
    return k < stored ? v : 1.0f;
  }

  // (nm_of: noise-management value of a sample with the largest input m)
  __device__ __forceinline__ float nm_of(float m) const {
    const IoDev &io = a.io;
    if (io.noise_management == RPU_NM_ABS_MAX || io.noise_management == RPU_NM_MAX) return io.nm_thres > 0.0f ? fminf(m, io.nm_thres) : m;
    if (io.noise_management == RPU_NM_CONSTANT) return io.nm_thres > 0.0f ? io.nm_thres : 1.0f;
    return 1.0f;
  }
  __device__ __forceinline__ static float reduction(int round) { return __builtin_bit_cast(float, (127 + round) << 23); } // 2^round

  // The DAC of round 0 to R - 1 for the element k of this thread's row: the rounds' scales are halves of each other, and so
  // are the quotients that are rounded (a value too small for that is zero in all of them, one too large at the bound: the few
  // calls with bounds beyond 2^96 work out one round at a time, Tile::few_args)
  __device__ __forceinline__ void quantize(float x, float scale, int b, int k) const {
    const IoDev &io = a.io;
    float q = x * scale;
    if (io.inp_res > 0.0f) q = q / io.inp_res;
#pragma unroll
    for (int r = 0; r < R; ++r, q *= 0.5f) {
      float v = q;
      if (io.inp_res > 0.0f) {
        if (STOCH && io.inp_sto_round) {
          const Philox4 u = philox4x32_10((uint32_t)k, (uint32_t)b, a.call, RNG_INP_SR | ((uint32_t)r << 8), a.key.k0, a.key.k1);
          v = v + (u32_to_uniform(u.v[0]) - 0.5f);
        }
        v = rintf(v) * io.inp_res;
      }
      v = (v > io.inp_bound) ? io.inp_bound : v;
      v = (v < -io.inp_bound) ? -io.inp_bound : v;
      if (STOCH && io.inp_noise > 0.0f) {
        float n[4];
        philox_normal4((uint32_t)k, (uint32_t)b, a.call, RNG_INP_NOISE | ((uint32_t)r << 8), a.key, n);
        v += io.inp_noise * n[0];
      }
      if (io.inp_asym != 0.0f) v = v < 0.0f ? v * (1.0f - io.inp_asym) : v;
      if (k < k_len) xs[(r * S + s_mine) * k_len + k] = k < a.K ? v : 0.0f;
    }
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
      const int s = lane;
      const int up = sh.hits[2 * S * slot + s], lo = sh.hits[2 * S * slot + S + s];
      const bool failed = a.io.bm_test_negative_bound ? (up > 0 || lo > 0) : (up > lo);
      float nm = my.nm, red = reduction(round), fin;
      (void)round_scales(a, nm, red, fin);
      my.live = failed && round + 1 < a.max_rounds && next_round_params(a, round, b0 + s, fin, nm, red);
      my.rounds += my.live ? 1 : 0;
    }
    return (unsigned)__ballot(my.live);
  }

  __device__ __forceinline__ void run(const int block_b, const int block_o) {
    const IoDev &io = a.io;
    const int t = (int)threadIdx.x, b0 = block_b * S, blocks_o = (a.O + OB - 1) / OB;
    const int b_mine = min(b0 + s_mine, a.m_batch - 1);
    x_row = a.in + (long)b_mine * a.in_sb;
    // inputs first, then the first half of the weights: the inputs are waited for first
    float x[PER_THREAD];
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) x[i] = stored_input(at + i * THREADS);
    Weights w;
    at_outputs(block_o * OB);
    start<0>(w);
    if (t < 2 * V) sh.hits[t] = 0;
    const bool signed_max = io.noise_management == RPU_NM_MAX;
    const float least = signed_max ? -INFINITY : 0.0f;
    float m = least;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) m = fmaxf(m, at + i * THREADS < a.K ? (signed_max ? x[i] : fabsf(x[i])) : least);
    for (int k0 = STEP; k0 < a.K; k0 += STEP) { // longer rows: the others wait in LDS, where their quantized values go
      float more[PER_THREAD];
#pragma unroll
      for (int i = 0; i < PER_THREAD; ++i) more[i] = stored_input(k0 + at + i * THREADS);
#pragma unroll
      for (int i = 0; i < PER_THREAD; ++i) {
        const int k = k0 + at + i * THREADS;
        m = fmaxf(m, k < a.K ? (signed_max ? more[i] : fabsf(more[i])) : least);
        if (k < k_len) xs[s_mine * k_len + k] = more[i];
      }
    }
    start<1>(w);
    m = wave_max(m);
    if (lane == 0) sh.max[wave] = m;
    if constexpr (S < 4) {
      __syncthreads();
      m = sh.max[s_mine * (4 / S)];
#pragma unroll
      for (int i = 1; i < 4 / S; ++i) m = fmaxf(m, sh.max[s_mine * (4 / S) + i]);
    }
    {
      float fin;
      const float scale = round_scales(a, nm_of(m), 1.0f, fin);
      for (int k0 = 0;;) {
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) {
          if (k0 + i * THREADS >= k_len) break; // the same for the workgroup
          quantize(x[i], scale, b_mine, k0 + at + i * THREADS);
        }
        k0 += STEP;
        if (k0 >= a.K) break;
#pragma unroll
        for (int i = 0; i < PER_THREAD; ++i) x[i] = k0 + at + i * THREADS < k_len ? xs[s_mine * k_len + k0 + at + i * THREADS] : 0.0f;
      }
    }
    __syncthreads();
    Samples my;
    {
      float top = sh.max[(lane % S) * (4 / S)];
#pragma unroll
      for (int i = 1; i < 4 / S; ++i) top = fmaxf(top, sh.max[(lane % S) * (4 / S) + i]);
      my.nm = nm_of(top);
      my.live = lane < S && b0 + lane < a.m_batch;
      float fin;
      (void)round_scales(a, my.nm, reduction(min(lane / S, R - 1)), fin);
      my.rounds = fin == 0.0f ? 0 : 1; // (lanes below S: of round 0)
      if (t < V) sh.fin[t] = fin;
    }
    unsigned live = (1u << min(S, a.m_batch - b0)) - 1u;
    Sums sums;
    contract(w, sums);
    const bool managed = a.max_rounds > 1, shared = managed && blocks_o > 1;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (r > 0) __syncthreads();
      spread(sums, r);
      __syncthreads();
      finish(b0, block_o * OB, r, r, live, r == 0 ? nullptr : (r == 1 ? a.dual.buf[1] : a.dual.buf[2]), shared || r > 0);
    }
    if (managed) {
      // what this workgroup stored has arrived before it counts itself off, and so have its marks
      if (shared || R > 1) __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
      if (shared) {
        int *const marks = a.few + a.m_batch; // [R][2][m_batch]: upper, lower; the counters before them
        const bool mine = t < 2 * V && b0 + t % S < a.m_batch;
        int *const mark = marks + (t / S) * a.m_batch + b0 + t % S;
        if (wave == 0) {
          const int hit = mine ? sh.hits[t] : 0;
          const bool any = __ballot(hit != 0) != 0;
          if (any) {
            if (hit) {
              const int old = atomicMax(mark, hit);
              asm volatile("" ::"v"(old));
            }
            __builtin_amdgcn_s_waitcnt(0);
          }
          // counter: workgroups in the lower half, those with marks in the upper
          if (lane == 0) {
            const int before = atomicAdd(&a.few[block_b], any ? 0x10001 : 1);
            sh.last = (before & 0xffff) != blocks_o - 1 ? 0 : (before >= 0x10000 || any ? 2 : 1);
          }
        }
        __syncthreads();
        const int last = uniform(sh.last);
        if (!last) return;
        // the last one reads the marks of all, and leaves them and the counter as it found them at first: zero
        if (t == 0) __hip_atomic_store(&a.few[block_b], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (last == 2) {
          if (t < 2 * V) sh.hits[t] = mine ? atomicExch(mark, 0) : 0;
          __syncthreads();
        }
      }
      unsigned chosen[R]; // samples whose result is that of round r
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const unsigned before = live;
        live = advance(b0, r, r, my);
        chosen[r] = before & ~live;
      }
      if constexpr (R > 1) {
#pragma unroll 1
        for (int r = 1; r < R; ++r) {
          const float *rows = r == 1 ? a.dual.buf[1] : a.dual.buf[2];
          const unsigned take = r == 1 ? chosen[1] : chosen[R - 1];
#pragma unroll 1
          for (int s = 0; s < S; ++s) {
            if (!((take >> s) & 1u)) continue;
            for (int o = t; o < a.O - a.out_drop; o += 256) {
              const float v = __hip_atomic_load(rows + (long)(b0 + s) * a.O + o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              __hip_atomic_store(a.out + (long)(b0 + s) * a.out_sb + (long)o * a.out_so, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
          }
        }
      }
      if (live) { // the same for all threads
        __syncthreads();
        alone(block_b, live, my);
      }
    }
    if ((shared || block_o == 0) && wave == 0) {
      if (lane < S && b0 + lane < a.m_batch) a.st.rounds[b0 + lane] = my.rounds;
      const bool more = __ballot(lane < S && b0 + lane < a.m_batch && my.rounds > 1) != 0;
      // the host picks R by what it knows of the last calls: the last one it hears of, the last one with samples that went on
      if (managed && lane == 0) {
        if (more) __hip_atomic_store(a.few_seen, a.few_call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        if (block_b == 0) __hip_atomic_store(a.few_seen + 1, a.few_call, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  // The rounds from R on for the samples of `live`, by this workgroup: block after block of 64 outputs, whatever the blocks of
  // the launch are (a block is one trip through the ADC stage: with blocks of 16 a round of a 512 x 512 tile took 35 us)
  __device__ __forceinline__ void alone(int block_b, unsigned live, Samples &my) {
    Alone all(a, xs, sh);
    const int b0 = block_b * S;
    all.x_row = x_row;
    for (int round = R; live; ++round) live = all.whole_round(b0, round, live, my.live, my.rounds, my.nm);
  }
  __device__ __forceinline__ unsigned whole_round(int b0, int round, unsigned live, bool &on, int &rounds, float &nm) {
    const int t = (int)threadIdx.x, b_mine = min(b0 + s_mine, a.m_batch - 1);
    const float red = reduction(round);
    Weights w;
    at_outputs(0);
    start<0>(w);
    start<1>(w);
    float fin;
    const float scale = round_scales(a, __shfl(nm, s_mine), red, fin);
    if (t < 2 * S) sh.hits[t] = 0;
    for (int k = at; k < k_len; k += THREADS) {
      xs[s_mine * k_len + k] = k < a.K ? dac_value<STOCH>(stored_input(k), scale, a.io, a.key, a.call, round, b_mine, k) : 0.0f;
    }
    if (at == 0) sh.fin[s_mine] = fin;
    for (int o_first = 0; o_first < a.O; o_first += OB) {
      __syncthreads(); // the inputs are there, the sums of the outputs before have been read
      Sums sums;
      contract(w, sums);
      spread(sums, 0);
      at_outputs(o_first + OB); // (beyond the outputs: zeros, not used)
      start<0>(w);
      start<1>(w);
      __syncthreads();
      finish(b0, o_first, round, 0, live, nullptr, true);
    }
    __syncthreads();
    Samples my{on, rounds, nm};
    live = advance(b0, round, 0, my);
    on = my.live;
    rounds = my.rounds;
    __syncthreads();
    return live;
  }

  // workgroup number n of a tile -> block of samples, block of outputs.  From eight blocks of outputs on, those of an XCD
  // (n % 8) are next to each other: each L2 holds its own part of the weights.
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

template <bool WOC, int S, int OB, int R, bool STOCH>
__global__ __launch_bounds__(256, 2) void k_mvm_few(MvmArgs a) {
  extern __shared__ __attribute__((aligned(16))) float few_lds[];
  __shared__ FewShared sh;
  typedef MvmFew<WOC, S, OB, R, STOCH> Few;
  int block_b, block_o;
  if (Few::block_of(a, (int)blockIdx.x, block_b, block_o)) Few(a, few_lds, sh).run(block_b, block_o);
}

// counters and marks of the tiles of a group, a workgroup for each tile
__global__ __launch_bounds__(256) void k_mvm_few_clear_group(MvmGroup g) {
  const MvmArgs &a = g.args[blockIdx.x];
  if (a.max_rounds < 2) return;
  for (int i = (int)threadIdx.x; i < 7 * a.m_batch; i += 256) a.few[i] = 0;
}

struct MvmFewGroup {
  MvmGroup group;
  MvmFewCalls calls;
};

// several tiles in one launch: start[t] .. start[t + 1] are the workgroups of tile t
template <bool WOC, int S, int OB, int R, bool STOCH>
__global__ __launch_bounds__(256, 2) void k_mvm_few_group(MvmFewGroup launch) {
  const MvmGroup &g = launch.group;
  extern __shared__ __attribute__((aligned(16))) float few_lds[];
  __shared__ FewShared sh;
  typedef MvmFew<WOC, S, OB, R, STOCH> Few;
  // the tile: as many of start[1 ..] as are not beyond this workgroup, 64 of them at a time
  int t = 0;
  for (int i = 0; i < g.n; i += 64) {
    const int at = i + ((int)threadIdx.x & 63);
    const unsigned long long before = __ballot(at + 1 < g.n && (int)blockIdx.x >= g.start[min(at + 1, g.n)]);
    t += __popcll(before);
    if (before != ~0ull) break;
  }
  t = uniform(t);
  MvmArgs a = g.args[t]; // scalar loads: t is the same for the whole workgroup
  if (launch.calls.count > 0) {
    a.in = launch.calls.in[t];
    a.out = launch.calls.out[t];
    a.call = launch.calls.call[t];
    a.few_call = launch.calls.few_call;
  }
  int block_b, block_o;
  if (Few::block_of(a, (int)blockIdx.x - g.start[t], block_b, block_o)) Few(a, few_lds, sh).run(block_b, block_o);
}

} // namespace

static int cus_of(const MvmArgs &a) { return a.cus > 0 ? a.cus : current_device_cus(); }

// whether the converters draw random numbers beyond the output noise
bool mvm_few_stoch(const MvmArgs &a) { return a.io.inp_sto_round || a.io.out_sto_round || a.io.inp_noise > 0.0f; }

// Blocks of the largest kind (four samples by 64 outputs) that a call launches for four of its samples
int mvm_few_blocks(int O) { return MvmFew<false, 4, 64, 1, false>::workgroups(O, 4); }

// The largest batch whose calls run as k_mvm_few.  A second set of blocks on a CU that holds two doubles the launch: the GPU
// has to hold all of them at once.  us, the other launches / one, at that line and beyond: 160 -> 100, backward, 600 samples
// 11.4 / 9.9, 800 11.7 / 15.5; 64 -> 32, 1000 17.0 / 7.8, 3000 16.7 / 17.5, backward 6000 11.5 / 21.7; 64 -> 2048, 64 17.4 /
// 16.6, 100 18.3 / 23.4; layers of tiles of at most 512 x 512, 768 -> 2304, 24 tokens 52 / 35, 32 28 / 32; 24 tiles of 300 x
// 300, 16 tokens 33 / 26, 24 33 / 39; 24 of 130 x 125, 64 tokens 28.5 / 32.7 (mvm_few_group_batch).
// (Measured on the kernel as it was with branches and all draws; this one is faster, the line is where it was: a call on this
// side of it adds in another order than one beyond.)
// Within it the multiply-adds: on either side of the line the launches cost the same.  The last samples here, the launches one
// by one / this one, and one sample more on k_mvm_whole:
//   forward, no saturation: 512 x 512, 50 (13 M) 18.1 / 9.6, 9.8; 1024 x 1024, 12 20.8 / 10.3, 11.9; 1500 x 1500, 5 28.1 / 12.9,
//   14.2; 785 x 300, 51 26.9 / 10.0, 11.2; 160 -> 100, 609 16.9 / 7.5, 9.0; 64 -> 32, 2048 15.3 / 5.7, 7.9
//   every sample in round 3 or later, which the last workgroup of a sample runs alone: 512 x 512, 50 70 / 54; 785 x 300, 51 108 /
//   45; 160 -> 100, 609 65 / 26; but 1024 x 1024, 12 64 / 87; 1500 x 1500, 5 82 / 205
//   backward: 512 x 512, 256 (67 M) 14.6 / 8.4, 9.3; 1024 x 1024, 64 17.6 / 11.0, 12.2; 1500 x 1500, 29 29.4 / 15.1, 12.3
int mvm_few_batch(const MvmArgs &a) {
  const IoDev &io = a.io;
  const int nm = io.noise_management;
  if (io.perfect || a.in_index || a.pre_add || a.skip_if_zero || a.nm_phase || a.small_tiles_only || a.K > 2048 || a.K <= a.in_one) return 0;
  // offsets of 32 bits
  if ((long)(a.w_oc ? a.K : a.O) * a.w_ld >= 1L << 28 || (long)a.K * a.in_sk >= 1L << 29) return 0;
  if (nm != RPU_NM_NONE && nm != RPU_NM_CONSTANT && nm != RPU_NM_ABS_MAX && nm != RPU_NM_MAX) return 0;
  if (io.bound_management != RPU_BM_NONE && (io.bound_management != RPU_BM_ITERATIVE || a.transposed)) return 0;
  const long per_cu = a.max_rounds > 1 ? 51200 : 262144; // multiply-adds
  // (a sample takes a load of 64 inputs by 16 outputs at least: a long batch on a tiny tile is not a small call)
  const long most = per_cu * cus_of(a) / ((long)((a.K + 63) & ~63) * ((a.O + 15) & ~15));
  return (int)std::min(most, 4L * (2 * cus_of(a) / mvm_few_blocks(a.O)));
}
// The same for a group of tiles whose calls have `blocks` blocks for four samples, all tiles taken together.
int mvm_few_group_batch(long blocks) { return (int)(4 * (2L * current_device_cus() / blocks)); }
// the variant of a launch of such calls: the smallest blocks of samples and outputs with at most two workgroups to a CU
int mvm_few_variant(const MvmArgs *const *calls, int n) {
  for (int v = 0; v < 3; ++v) {
    long workgroups = 0;
    for (int i = 0; i < n; ++i) workgroups += mvm_few_workgroups(*calls[i], v);
    if (workgroups <= 2L * current_device_cus()) return v;
  }
  return 3;
}

#define RPU_FEW_VARIANT(variant, CALL) \
  switch (variant) { \
  case 0: CALL(1, 16); break; \
  case 1: CALL(2, 32); break; \
  case 2: CALL(4, 32); break; \
  default: CALL(4, 64); break; \
  }

int mvm_few_workgroups(const MvmArgs &a, int variant) {
#define RPU_FEW_COUNT(S, OB) return MvmFew<false, S, OB, 1, false>::workgroups(a.O, a.m_batch)
  RPU_FEW_VARIANT(variant, RPU_FEW_COUNT)
#undef RPU_FEW_COUNT
}

#define RPU_LAUNCH_FEW_AS(KERNEL, ARGS, K, W_OC, ROUNDS, STOCH, S, OB) \
  if (W_OC) { \
    if (ROUNDS == 3) hipLaunchKernelGGL((KERNEL<true, S, OB, 3, STOCH>), grid, dim3(256), (MvmFew<true, S, OB, 3, STOCH>::lds_bytes(K)), s, ARGS); \
    else hipLaunchKernelGGL((KERNEL<true, S, OB, 1, STOCH>), grid, dim3(256), (MvmFew<true, S, OB, 1, STOCH>::lds_bytes(K)), s, ARGS); \
  } else { \
    if (ROUNDS == 3) hipLaunchKernelGGL((KERNEL<false, S, OB, 3, STOCH>), grid, dim3(256), (MvmFew<false, S, OB, 3, STOCH>::lds_bytes(K)), s, ARGS); \
    else hipLaunchKernelGGL((KERNEL<false, S, OB, 1, STOCH>), grid, dim3(256), (MvmFew<false, S, OB, 1, STOCH>::lds_bytes(K)), s, ARGS); \
  }

void launch_mvm_few(const MvmArgs &a, int variant, int rounds, hipStream_t s) {
  const dim3 grid((unsigned)mvm_few_workgroups(a, variant));
#define RPU_LAUNCH_FEW(S, OB) RPU_LAUNCH_FEW_AS(k_mvm_few, a, a.K, a.w_oc, rounds, false, S, OB)
#define RPU_LAUNCH_FEW_STOCH(S, OB) RPU_LAUNCH_FEW_AS(k_mvm_few, a, a.K, a.w_oc, rounds, true, S, OB)
  if (mvm_few_stoch(a)) {
    RPU_FEW_VARIANT(variant, RPU_LAUNCH_FEW_STOCH)
  } else {
    RPU_FEW_VARIANT(variant, RPU_LAUNCH_FEW)
  }
#undef RPU_LAUNCH_FEW_STOCH
#undef RPU_LAUNCH_FEW
}

void launch_mvm_few_clear_group(const MvmGroup &g, hipStream_t s) {
  hipLaunchKernelGGL(k_mvm_few_clear_group, dim3((unsigned)g.n), dim3(256), 0, s, g);
}

void launch_mvm_few_group(const MvmGroup &g, const MvmFewCalls &calls, int variant, int rounds, bool w_oc, bool stoch, int max_k,
                          int total_workgroups, hipStream_t s) {
  const MvmFewGroup launch{g, calls};
  const dim3 grid((unsigned)total_workgroups);
#define RPU_LAUNCH_FEW(S, OB) RPU_LAUNCH_FEW_AS(k_mvm_few_group, launch, max_k, w_oc, rounds, false, S, OB)
#define RPU_LAUNCH_FEW_STOCH(S, OB) RPU_LAUNCH_FEW_AS(k_mvm_few_group, launch, max_k, w_oc, rounds, true, S, OB)
  if (stoch) {
    RPU_FEW_VARIANT(variant, RPU_LAUNCH_FEW_STOCH)
  } else {
    RPU_FEW_VARIANT(variant, RPU_LAUNCH_FEW)
  }
#undef RPU_LAUNCH_FEW_STOCH
#undef RPU_LAUNCH_FEW
}
#undef RPU_LAUNCH_FEW_AS
#undef RPU_FEW_VARIANT

} // namespace rpu_amd
