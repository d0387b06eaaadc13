// Exact products (perfect IO, floating-point updates) of a size that fills the GPU: both operands split into bf16 parts once,
// by a launch of their own, then a contraction whose stages do nothing but move and multiply them.
//
//   k_product_parts  an operand's rows as three bf16 planes, in blocks of 128 rows x 32 terms laid out as the contraction
//                    stages them, whichever way the operand is stored (it takes the place of the copy into contiguous rows)
//   k_product        a workgroup makes 128 outputs x 128 (or 64) samples over a share of the terms
//   k_product_sum    adds the shares in their order, where there is more than one
//
// In the kernels that split what they stage (k_mvm_big, three parts) a wave issues 220 vector instructions for the 16 MFMAs of a
// stage and waits for a third of the rest: 27 % of the matrix pipe's time at 768 x 2304 outputs of 1024 terms.  Here a stage is
// 32 MFMAs and 18 reads of LDS to a wave, a byte staged meets more multiply-adds, and splitting the terms fills the CUs that
// few large tiles leave idle.  768 -> 2304, 1024 samples, row-major tile, backward call 76 -> 46 us (parts 9, product 32, sums 7);
// 1024 x 1024, 16384 samples, forward 311 -> 272: 1.1 PFLOP/s of bf16 products, a large library product reaches 1.2 on this card.
// There the matrix pipe is busy for 58 % of the cycles (at 1.9 GHz under that load), 49 % in the smaller call; what is left is the
// waits of a stage, for LDS (27 % of the cycles, no bank conflicts) and at its barrier.
#include "bf16_parts.h"
#include "kernels.h"

#include <algorithm>
#include <cmath>

namespace rpu_amd {
namespace {

constexpr int PT = PRODUCT_TILE;            // outputs of a workgroup tile, and rows of a block
constexpr int PK = 32;                      // terms of a stage
constexpr int PLANE = PT * PK;              // values of a plane of a block
constexpr int BLOCK = 3 * PLANE;            // ... of a block: the parts of PT rows x PK terms
constexpr int MOST_SHARES = 16;             // of the terms
constexpr float LIFT = 0x1p16f;             // the parts are those of this times the value (split_bf16)

// 64 rows x 64 terms of an operand: element (row, k) at src[row * s_r + k * s_k]; term one_k is 1 and not stored (-1: none)
__device__ __forceinline__ void product_parts_block(const float *src, long s_r, long s_k, int rows, int K, int one_k, int rb, int kb, __bf16 *parts,
                                                    int *flags, int stages, float safe, float (*tile)[65]) {
  const int t = (int)threadIdx.x, r0 = rb * 64, k0 = kb * 64;
  const int stored = one_k >= 0 ? one_k : K;
  const bool along_k = s_k == 1;
  // four neighbouring values of a thread, along the terms or else along the rows
  const int fast = (t & 15) * 4, slow = t >> 4;
  const long s_fast = along_k ? 1 : s_r, s_slow = along_k ? s_r : s_k;
  const int n_fast = along_k ? stored - k0 : rows - r0, n_slow = along_k ? rows - r0 : stored - k0;
  const float *from = src + (long)r0 * s_r + (long)k0 * s_k + (long)fast * s_fast;
  f32x4 v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = slow + 16 * i;
    v[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (at < n_slow) {
      const float *p = from + (long)at * s_slow;
      if (s_fast == 1 && fast + 3 < n_fast) {
        v[i] = *reinterpret_cast<const f32x4_unaligned *>(p);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (fast + e < n_fast) v[i][e] = p[(long)e * s_fast];
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = slow + 16 * i;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (along_k) tile[at][fast + e] = v[i][e];
      else tile[fast + e][at] = v[i][e];
    }
  }
  __syncthreads();
  const int row = t >> 2, chunk = t & 3;
  bool wide[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    float m = 0.0f;
    u32x4 part[3];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = 32 * p + 8 * chunk + 4 * half + e;
        x[e] = tile[row][k];
        if (k0 + k == one_k && r0 + row < rows) x[e] = 1.0f;
      }
      m = max_abs4(m, x);
      u32x2 hi, mid, lo;
      split_bf16<true>(x * LIFT, hi, mid, lo);
      part[0][2 * half] = hi.x; part[0][2 * half + 1] = hi.y;
      part[1][2 * half] = mid.x; part[1][2 * half + 1] = mid.y;
      part[2][2 * half] = lo.x; part[2][2 * half + 1] = lo.y;
    }
    wide[p] = !(m < safe);
    const int stage = 2 * kb + p;
    if (stage < stages) {
      __bf16 *dst = parts + ((long)(rb >> 1) * stages + stage) * BLOCK + big_x_offset((rb & 1) * 64 + row, chunk);
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4 *>(dst + q * PLANE) = part[q];
    }
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int any = __syncthreads_or(wide[p] ? 1 : 0);
    if (t == 0 && 2 * kb + p < stages) flags[(long)rb * stages + 2 * kb + p] = any;
  }
}

// Workgroups: blocks of 64 rows x 64 terms of the weights, then of the inputs; row blocks to full tiles of both.
__global__ __launch_bounds__(256) void k_product_parts(MvmArgs a, ProductArgs p) {
  __shared__ float tile[64][65];
  const int kbs = (p.stages + 1) / 2, w_blocks = 2 * p.tiles_o * kbs;
  int n = (int)blockIdx.x;
  if (n < w_blocks) {
    product_parts_block(a.w, a.w_oc ? 1 : a.w_ld, a.w_oc ? a.w_ld : 1, a.O, a.K, -1, n / kbs, n % kbs, p.w_parts, p.w_flags, p.stages, p.safe, tile);
  } else {
    n -= w_blocks;
    product_parts_block(a.in, a.in_sb, a.in_sk, a.m_batch, a.K, a.in_one ? a.K - 1 : -1, n / kbs, n % kbs, p.x_parts, p.x_flags, p.stages, p.safe, tile);
  }
}

// out = alpha * sum + beta * out for outputs o0 .. o0 + 3 of sample b
__device__ __forceinline__ void product_store(const MvmArgs &a, int b, int o0, f32x4 v) {
  const int o_end = a.O - a.out_drop;
  if (b >= a.m_batch || o0 >= o_end) return;
  float *out = a.out + (long)b * a.out_sb + (long)o0 * a.out_so;
  v *= a.alpha;
  if (a.out_so == 1 && o0 + 3 < o_end && ((uintptr_t)out & 15) == 0) {
    if (a.beta != 0.0f) v += a.beta * *reinterpret_cast<const f32x4 *>(out);
    *reinterpret_cast<f32x4 *>(out) = v;
    return;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (o0 + q < o_end) {
      float res = v[q];
      if (a.beta != 0.0f) res += a.beta * out[(long)q * a.out_so];
      out[(long)q * a.out_so] = res;
    }
  }
}

// A wave owns 64 outputs x 32 samples, a workgroup two waves of outputs and BT / 32 of samples.  A thread holds eight groups of
// four outputs: block of 32 outputs ob, group g, in the place where the MFMA leaves them.
constexpr int GROUPS = 8;
__device__ __forceinline__ void product_place(int t, int i, int &o, int &b) {
  const int lane = t & 63, wave = t >> 6, ob = i >> 2, g = i & 3;
  o = (wave & 1) * 64 + ob * 32 + g * 8 + (lane >> 5) * 4;
  b = (wave >> 1) * 32 + (lane & 31);
}

// Of the nine products of the parts, that of the two low ones (2^-36 of the whole) is left out.  Those of a low with a middle part
// (up to 2^-26 of the whole together) are small beside the rounding of a long dense sum, but not where few terms count: one
// term of 1024, largest error in units of the last place 0.51, without them 0.94.
// BT samples of a workgroup tile: 128 (eight waves, 96 KB of LDS for two stages in turn, one workgroup to a CU) or 64 (four waves,
// two workgroups to a CU).  Two waves to a SIMD either way: one reads fragments (18 for its 32 MFMAs) while the other multiplies.
// The next stage is on its way to registers while one is worked on.
template <int BT> __global__ __launch_bounds__(4 * BT, BT == 128 ? 1 : 2) void k_product(MvmArgs a, ProductArgs p) {
  constexpr int THREADS = 4 * BT, XPLANE = BT * PK;
  __shared__ __attribute__((aligned(16))) __bf16 lds_w[2][BLOCK], lds_x[2][3 * XPLANE];
  __shared__ int wide;
  // an XCD (workgroup n runs on XCD n % 8) walks tiles of one share of the terms that follow each other
  const int tiles = p.tiles_o * p.tiles_b, all = tiles * p.shares, per = (all + 7) >> 3;
  const int n = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || n >= all) return;
  const int share = n / tiles, tile = n - share * tiles, tile_b = tile / p.tiles_o, tile_o = tile - tile_b * p.tiles_o;
  const int s0 = share * p.stages_per_share, s1 = min(s0 + p.stages_per_share, p.stages);
  const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6, r = lane & 31, h = lane >> 5;
  const int block_b = BT == 128 ? tile_b : tile_b >> 1, half_b = BT == 128 ? 0 : tile_b & 1; // of the 128 rows of a block
  const u32x4 *w_src = reinterpret_cast<const u32x4 *>(p.w_parts + ((long)tile_o * p.stages + s0) * BLOCK) + t;
  const u32x4 *x_src = reinterpret_cast<const u32x4 *>(p.x_parts + ((long)block_b * p.stages + s0) * BLOCK + half_b * XPLANE) + t;
  constexpr int WL = BLOCK / 8 / THREADS, XL = 3 * XPLANE / 8 / THREADS; // 16-byte chunks of a thread per stage
  static_assert(XL == 3, "a plane of the inputs to a load");
  u32x4 gw[WL], gx[XL];
  auto gload = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < WL; ++i) gw[i] = w_src[THREADS * i];
#pragma unroll
    for (int i = 0; i < XL; ++i) gx[i] = x_src[PLANE / 8 * i];
    w_src += BLOCK / 8;
    x_src += BLOCK / 8;
  };
  auto store = [&](int buf) __attribute__((always_inline)) {
    u32x4 *w = reinterpret_cast<u32x4 *>(&lds_w[buf][0]) + t, *x = reinterpret_cast<u32x4 *>(&lds_x[buf][0]) + t;
#pragma unroll
    for (int i = 0; i < WL; ++i) w[THREADS * i] = gw[i];
#pragma unroll
    for (int i = 0; i < XL; ++i) x[XPLANE / 8 * i] = gx[i];
  };
  gload();
  { // whether a value of this share of the operands is out of the range of the parts
    int any = 0;
    for (int s = s0 + t; s < s1; s += THREADS) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        any |= p.w_flags[(long)(2 * tile_o + i) * p.stages + s];
        any |= p.x_flags[(long)(2 * block_b + (BT == 128 ? i : half_b)) * p.stages + s];
      }
    }
    if (t == 0) wide = 0;
    __syncthreads();
    if (any) wide = 1;
  }
  floatx16 acc[2], low[2];
#pragma unroll
  for (int ob = 0; ob < 2; ++ob) {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[ob][e] = low[ob][e] = 0.0f;
  }
  int w_off[2][2], x_off[2]; // [block][j]: values k = 16 h + 8 j .. + 7 of a stage
#pragma unroll
  for (int j = 0; j < 2; ++j) {
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) w_off[ob][j] = big_x_offset((wave & 1) * 64 + ob * 32 + r, h * 2 + j);
    x_off[j] = big_x_offset((wave >> 1) * 32 + r, h * 2 + j);
  }
  store(0);
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1;
    const bool next = s + 1 < s1;
    if (next) gload();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x8 w[2][3], x[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
#pragma unroll
        for (int ob = 0; ob < 2; ++ob) w[ob][q] = *reinterpret_cast<const bf16x8 *>(&lds_w[buf][w_off[ob][j] + q * PLANE]);
        x[q] = *reinterpret_cast<const bf16x8 *>(&lds_x[buf][x_off[j] + q * XPLANE]);
      }
      // part q of a weight with part m - q of an input, those that correct the product of the high parts to a sum of their own
#pragma unroll
      for (int m = 3; m >= 0; --m) {
#pragma unroll
        for (int q = 0; q <= min(m, 2); ++q) {
          if (m - q > 2) continue;
#pragma unroll
          for (int ob = 0; ob < 2; ++ob) {
            floatx16 &sum = m > 0 ? low[ob] : acc[ob];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ob][q], x[m - q], sum, 0, 0, 0);
          }
        }
      }
    }
    if (next) store(buf ^ 1);
    __syncthreads();
  }
  float unit = 1.0f / (LIFT * LIFT);
#pragma unroll
  for (int ob = 0; ob < 2; ++ob) acc[ob] += low[ob];
  if (wide) { // a value out of the range of the parts: this share of the tile again on the fp32 pipe, straight from memory
    unit = 1.0f;
    const long w_sr = a.w_oc ? 1 : a.w_ld, w_sk = a.w_oc ? a.w_ld : 1;
    const int stored = a.K - a.in_one;
    const float *w_row[2], *x_row = a.in + (long)min(tile_b * BT + (wave >> 1) * 32 + r, a.m_batch - 1) * a.in_sb;
#pragma unroll
    for (int ob = 0; ob < 2; ++ob) {
      w_row[ob] = a.w + (long)min(tile_o * PT + (wave & 1) * 64 + ob * 32 + r, a.O - 1) * w_sr;
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[ob][e] = 0.0f;
    }
#pragma unroll 1
    for (int k0 = s0 * PK; k0 < min(s1 * PK, a.K); k0 += 2) {
      const int k = k0 + h;
      const float x = k < stored ? x_row[k * a.in_sk] : (k < a.K ? 1.0f : 0.0f);
#pragma unroll
      for (int ob = 0; ob < 2; ++ob) acc[ob] = __builtin_amdgcn_mfma_f32_32x32x2f32(k < a.K ? w_row[ob][k * w_sk] : 0.0f, x, acc[ob], 0, 0, 0);
    }
  }
  f32x4 *partial = reinterpret_cast<f32x4 *>(p.partial) + (long)n * GROUPS * THREADS + t;
#pragma unroll
  for (int ob = 0; ob < 2; ++ob) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int i = ob * 4 + g;
      const f32x4 v = f32x4{acc[ob][4 * g], acc[ob][4 * g + 1], acc[ob][4 * g + 2], acc[ob][4 * g + 3]} * unit;
      if (p.shares > 1) {
        partial[i * THREADS] = v;
      } else {
        int o, b;
        product_place(t, i, o, b);
        product_store(a, tile_b * BT + b, tile_o * PT + o, v);
      }
    }
  }
}

// A workgroup adds an eighth of a tile: one group of every thread of k_product, or where outputs follow each other in memory the
// 16 groups, 256 bytes, of four samples of a wave (update of a [768][2304] matrix 14.1 -> 7.2 us).
template <int BT> __global__ __launch_bounds__(4 * BT) void k_product_sum(MvmArgs a, ProductArgs p) {
  constexpr int THREADS = 4 * BT;
  const int lane = (int)threadIdx.x & 63, tiles = p.tiles_o * p.tiles_b, tile = (int)blockIdx.x / GROUPS, part = (int)blockIdx.x % GROUPS;
  int t = (int)threadIdx.x, i = part;
  if (a.out_so == 1) {
    i = (lane & 15) >> 1;
    t = (t & ~63) + (lane & 1) * 32 + part * 4 + (lane >> 4);
  }
  const f32x4 *partial = reinterpret_cast<const f32x4 *>(p.partial) + ((long)tile * GROUPS + i) * THREADS + t;
  f32x4 v = partial[0];
#pragma unroll 4
  for (int s = 1; s < p.shares; ++s) v += partial[(long)s * tiles * GROUPS * THREADS];
  int o, b;
  product_place(t, i, o, b);
  const int tile_b = tile / p.tiles_o, tile_o = tile - tile_b * p.tiles_o;
  product_store(a, tile_b * BT + b, tile_o * PT + o, v);
}

} // namespace

// Whether a call of this size is worth the launch that splits its operands.  A tile makes room for the calls of fewer samples, too
// (product_room): large_tiles_aside, whether this or one of up to 63 samples less, which might not take the large tiles, could be.
static bool product_pays(const MvmArgs &a, int n_cus, bool large_tiles_aside) {
  const auto padded = [](double n, int to) { return std::ceil(n / to) * to; };
  // us, the launches of k_mvm_init and k_mvm_round or k_mvm_big / these.  From 3/4 G multiply-adds: 784 -> 256, 4096 samples (0.8
  // G) forward 43 / 35, update 53 / 34; 1024 x 1024, 1024 46 / 35, 16384 311 / 270, update 622 / 272; 768 -> 2304, 1024 58 / 52,
  // backward 76 / 46, update 58 / 45; 3072 x 3072, 512 145 / 114.  Below: 1024 x 1024, 512 23 / 28, 256 15 / 22; 512 x 512, 512 12
  // / 17; 3072 x 3072, 64 28 / 38, and few terms of a large product, which the split and the store are most of: 3072 x 3072 outputs
  // of 64 terms 39 / 50, of 128 64 / 59.
  const double work = (double)a.m_batch * a.O * a.K;
  // Less than that where the 32 x 32 kernel would walk a long chain of terms: 256 x 256 outputs of 4096 terms 35 / 27, 100 x 100 of
  // 16384 103 / 49, but 64 x 3072 of 2048 26 / 29
  const long tiles_32 = (long)((a.O + 31) / 32) * ((a.m_batch + 31) / 32);
  const double chain = (double)((tiles_32 + n_cus - 1) / n_cus) * a.K;
  const bool large = mvm_uses_large_tiles(a.m_batch, a.O);
  const bool long_chain = chain >= 4096.0 && work >= 0x1p27 && (large_tiles_aside || !large);
  // products per split value: few outputs or few samples leave a launch that splits and little else
  const double reuse = (double)a.m_batch * a.O / ((double)a.m_batch + a.O);
  if (!(work >= 0x1.8p29 && a.K >= 128 && reuse >= 96.0) && !(long_chain && reuse >= 32.0)) return false;
  // an update of operands that both lie along the terms, which the launches before have little to copy for: 1024 x 4096, 192 terms 29.5
  // / 32.9, 2048 x 2048, 192 31.0 / 32.6, 256 36.3 / 34.9
  const bool update = a.beta != 0.0f;
  if (update && a.in_sk == 1 && a.K < 256) return false;
  if (large && a.m_batch > 256) return true;
  // Few samples of a large matrix: the split of the weights is most of the call.  Time of either, us, fitted to 730 calls of 36 to 49152
  // samples, 100 to 32768 outputs, 128 to 50000 terms (60 take up to 13 % longer than the faster one): 8192 x 8192, 40 samples 104 / 211,
  // 4096 x 4096, 64 35 / 50, 128 54 / 64, 192 75 / 85, 224 93 / 88, 2048 x 2048, 256 31.9 / 33.2, 288 41.9 / 36.4, 1024 -> 16384, 128
  // 62 / 74.  Not by the way the weights are stored (the 32 x 32 kernel takes 0.0042 or 0.0054 a term): either way the same bits.
  const double samples = padded(a.m_batch, 64), outputs = padded(a.O, PT), terms = 1e-6 * a.K;
  double rows = 11.0 + 0.005 * chain + (a.O % 32 && tiles_32 > n_cus ? 11.0 : 0.0);
  if (large) { // two workgroups to a CU at a time
    const double large_rows = 20.5 + 0.022 * a.K * std::max(1.0, (a.O + 63) / 64 * (samples / 64) / (2 * n_cus));
    rows = large_tiles_aside ? std::max(rows, large_rows) : large_rows;
  }
  rows += 1.5 * a.m_batch * terms + (update ? 2e-6 * a.m_batch * a.O : 0.0);
  const double parts = 15.0 + 1.35 * (padded(a.m_batch, PT) + outputs) * terms + 10.5 * samples * outputs * a.K / 0x1p30;
  return rows > parts;
}
// the work of the call dealt out: tiles, shares of the terms
static void product_split(const MvmArgs &a, int n_cus, ProductArgs &p) {
  p = ProductArgs{};
  p.tiles_o = (a.O + PT - 1) / PT;
  p.stages = (a.K + PK - 1) / PK;
  p.safe = parts_safe(a.K);
  double best = 0.0;
  for (int bt = 64; bt <= 128; bt += 64) {
    const int tiles_b = (a.m_batch + bt - 1) / bt;
    const long tiles = (long)p.tiles_o * tiles_b;
    for (int shares = 1; shares <= MOST_SHARES && shares <= p.stages; ++shares) {
      const int per = (p.stages + shares - 1) / shares;
      if (shares > 1 && (shares - 1) * per >= p.stages) continue; // the last share would be empty
      // in stages of a CU that is full: the rounds of workgroups, a half-full one faster, each with a start and an end, and the
      // sums (512 x 512 outputs of 1024 terms 50 us with one share, 23 with eight; 1024 x 1024 of 1024 41 with two, 33 with four;
      // 2048 x 1024 of 1024 in one share 46 with 256 half workgroups, 56 with 128; 16384 x 1024 of 1024 251 with halves, 242)
      const long slots = (long)n_cus * (128 / bt), all = tiles * shares, last = all % slots;
      const double full = bt == 64 ? 1.04 : 1.0;
      double cost = (double)(all / slots) * (full * per + 3);
      if (last > 0) cost += (bt == 64 && last <= n_cus ? 0.8 : full) * per + 3;
      if (shares > 1) cost += 2 + 0.02 * (double)all * bt / 128;
      if (best == 0.0 || cost < best) {
        best = cost;
        p.sample_tile = bt; p.tiles_b = tiles_b; p.shares = shares; p.stages_per_share = per;
      }
    }
  }
}
constexpr size_t MOST_SCRATCH = (size_t)2 << 30; // rows padded to 128 are many times the operand of a long, narrow call

// Whether an exact call runs as k_product, and how
bool product_plan(const MvmArgs &a, ProductArgs &p) {
  if (!a.io.perfect || a.in_index || a.pre_add || a.skip_if_zero || a.nm_phase || a.small_tiles_only) return false;
  const int n_cus = a.cus > 0 ? a.cus : current_device_cus();
  if (!product_pays(a, n_cus, false)) return false;
  product_split(a, n_cus, p);
  return product_scratch(p, nullptr, nullptr) <= MOST_SCRATCH;
}
// Scratch of the largest such call with the sizes of `a` and no more samples (terms, where they are the samples): fewer samples can
// take more shares of the terms, and with them more room for the sums.
size_t product_room(MvmArgs a, bool terms_are_samples) {
  const int n_cus = a.cus > 0 ? a.cus : current_device_cus();
  int &samples = terms_are_samples ? a.K : a.m_batch;
  const int step = terms_are_samples ? PK : 64; // a stage, the smaller tile of samples
  a.beta = terms_are_samples ? 1.0f : 0.0f; // an update: those of delta weights pay for no smaller ones
  size_t room = 0;
  for (; samples > 0; samples = (samples - 1) / step * step) {
    ProductArgs p{};
    p.tiles_o = (a.O + PT - 1) / PT;
    p.tiles_b = (a.m_batch + PT - 1) / PT;
    p.stages = (a.K + PK - 1) / PK;
    p.sample_tile = PT;
    p.shares = MOST_SHARES;
    if (product_scratch(p, nullptr, nullptr) <= room) break; // nor can any smaller call need more
    p.shares = 1;
    // more shares save the last round of workgroups at most, and cost more than that for the sums of many tiles (product_split)
    const double tiles = (double)p.tiles_o * (p.tiles_b - 0.5);
    const bool one_share = 0.04 * tiles > p.stages + 1 + (double)p.tiles_o * (p.stages + 3 * MOST_SHARES) / (2 * n_cus);
    if (one_share && product_scratch(p, nullptr, nullptr) <= room) continue;
    MvmArgs fewer = a;
    if (terms_are_samples) fewer.K = std::max(a.K - (PK - 1), 1); // the fewest of this many stages
    if (!product_pays(a, n_cus, !terms_are_samples) && !(terms_are_samples && product_pays(fewer, n_cus, false))) continue;
    if (!one_share) product_split(a, n_cus, p);
    const size_t bytes = product_scratch(p, nullptr, nullptr);
    if (bytes <= MOST_SCRATCH) room = std::max(room, bytes);
  }
  return room;
}

static int sample_blocks(const ProductArgs &p) { return p.sample_tile == PT ? p.tiles_b : (p.tiles_b + 1) / 2; } // of 128 rows

size_t product_scratch(const ProductArgs &p, unsigned char *base, ProductArgs *out) {
  size_t off = 0;
  auto take = [&](size_t bytes) {
    unsigned char *at = base ? base + off : nullptr;
    off += (bytes + 255) & ~(size_t)255;
    return at;
  };
  const size_t block = (size_t)BLOCK * sizeof(__bf16);
  const size_t w_blocks = (size_t)p.tiles_o * p.stages, x_blocks = (size_t)sample_blocks(p) * p.stages;
  unsigned char *w = take(w_blocks * block), *x = take(x_blocks * block);
  unsigned char *wf = take(2 * w_blocks * sizeof(int)), *xf = take(2 * x_blocks * sizeof(int));
  unsigned char *sums = p.shares > 1 ? take((size_t)p.shares * p.tiles_o * p.tiles_b * PT * p.sample_tile * sizeof(float)) : nullptr;
  if (out) {
    out->w_parts = (__bf16 *)w; out->x_parts = (__bf16 *)x; out->w_flags = (int *)wf; out->x_flags = (int *)xf; out->partial = (float *)sums;
  }
  return off;
}

void launch_product_parts(const MvmArgs &a, const ProductArgs &p, hipStream_t s) {
  const int kbs = (p.stages + 1) / 2;
  hipLaunchKernelGGL(k_product_parts, dim3((unsigned)(2 * (p.tiles_o + sample_blocks(p)) * kbs)), dim3(256), 0, s, a, p);
}
void launch_product(const MvmArgs &a, const ProductArgs &p, hipStream_t s) {
  const int tiles = p.tiles_o * p.tiles_b;
  const dim3 grid((unsigned)(8 * ((tiles * p.shares + 7) / 8))), sums((unsigned)(GROUPS * tiles)), block((unsigned)(4 * p.sample_tile));
  if (p.sample_tile == 128) {
    hipLaunchKernelGGL(k_product<128>, grid, block, 0, s, a, p);
    if (p.shares > 1) hipLaunchKernelGGL(k_product_sum<128>, sums, block, 0, s, a, p);
  } else {
    hipLaunchKernelGGL(k_product<64>, grid, block, 0, s, a, p);
    if (p.shares > 1) hipLaunchKernelGGL(k_product_sum<64>, sums, block, 0, s, a, p);
  }
}

} // namespace rpu_amd
