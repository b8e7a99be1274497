// attention.hip -- causal attention of a prompt on gfx950's f32 matrix cores,
// with the bits of the CPU path
// (crates/rusticide-transformer/src/attention.rs:41-57,189-207,
//  crates/rusticide-simd/src/float.rs:23-62,
//  crates/rusticide-kernels/src/portable/norm.rs:17-30).
//
// The CPU path's order of float operations fits the f32 MFMA: one
// v_mfma_f32_16x16x4 adds its four products to the accumulator one fused
// multiply-add at a time, k ascending, each rounded to nearest with
// subnormals kept (tests/test_gpu_attention_edges.py compares it bit for bit
// with fmaf chains over normal, subnormal, overflowing, signed-zero, infinite
// and NaN operands).
//   * A score is eight interleaved chains of fused adds (dot's eight lanes),
//     added in order: chain l is an accumulator of its own, its k the
//     eight-wide chunks; the eight accumulators are then added in order.
//   * An output lane's value mix is one chain over the rows: k is the row.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "rh_device.h"
#include "rh_internal.h"
#include "rh_math.h"

namespace rh {

namespace {

constexpr uint32_t kStripQ = 16;       // (token, head) query rows a workgroup owns
constexpr uint32_t kStripWaves = 8;
constexpr uint32_t kStripThreads = 64u * kStripWaves;
constexpr size_t kLdsBytes = 160u * 1024u;  // a gfx950 workgroup's LDS
constexpr uint32_t kSumRounds = 6;     // checking rounds of the ordered sum

constexpr int kBufferRsrcWord3 = 0x00020000;  // gfx9 buffer resource: raw 32-bit dwords

typedef float v4f __attribute__((ext_vector_type(4)));

// A strip row holds one query row's scores, then its weights: four 16-byte
// slots per group of 16 cached rows, slot 4 group + kr holding rows 4i + kr,
// i = 0..3, of the group -- the four k of an MFMA step side by side across
// the lanes that read them, four steps a read. The slots of 16 are exchanged
// by their position so that lanes reading runs of a row, one run a lane,
// fall on distinct banks; the row's length (an odd number of slots) does the
// same for lanes reading one slot of 16 rows.
__device__ __forceinline__ uint32_t strip_slot(uint32_t f4) { return f4 ^ ((f4 >> 4) & 15u); }

__host__ __device__ constexpr uint32_t strip_stride(uint32_t groups) { return 16u * ((groups + 3u) & ~3u) + 4u; }

constexpr size_t strip_lds_bytes(uint32_t groups) {
  // strip | per-wave maxima [waves][16] | the exp table
  return 4u * (static_cast<size_t>(kStripQ) * strip_stride(groups) + kStripWaves * kStripQ) + 32u * 8u;
}

// x[i] / d, given inv = 1 / d in double, correctly rounded. The double
// quotient is within 2^-52 of x / d relatively; a quotient of two floats is
// never closer than 2^-49 to the midpoint of two normal floats, so rounding
// it gives the float nearest x / d. Subnormal midpoints have fewer bits and
// a quotient may be one: where the result is subnormal the division itself
// is taken (one branch for the four). A midpoint at the ends of that range,
// 2^-150 and 2^-126 - 2^-150, rounds out of it (to even), and the quotient
// that lands inside it by its error is among those divided.
template <typename V>
__device__ __forceinline__ void div_by(V& x, float d, double inv) {
  constexpr int kSubnormal = 0x90;  // v_cmp_class: subnormal of either sign
  float q[4];
  bool sub = false;
#pragma unroll
  for (uint32_t i = 0; i < 4u; i++) {
    q[i] = static_cast<float>(static_cast<double>(x[i]) * inv);
    sub |= __builtin_amdgcn_classf(q[i], kSubnormal);
  }
  if (sub) {
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) q[i] = __fdiv_rn(x[i], d);
  }
#pragma unroll
  for (uint32_t i = 0; i < 4u; i++) x[i] = q[i];
}

// Inclusive prefix sum over each half of the wave (approximate: guesses).
__device__ __forceinline__ double half_prefix_sum(double v) {
  v += dpp_fill0_f64<0x111>(v);
  v += dpp_fill0_f64<0x112>(v);
  v += dpp_fill0_f64<0x114>(v);
  v += dpp_fill0_f64<0x118>(v);
  v += dpp_fill0_f64<0x142, 0xA>(v);
  return v;
}

// Start guesses from increments, per half-wave: its first lane gets 0, lane
// k the increments of the lanes before it.
__device__ __forceinline__ float half_guess_starts(double d, uint32_t hl) {
  const float end = static_cast<float>(half_prefix_sum(d));
  const uint32_t prev = dpp_fill<kDppWaveShr1>(__float_as_uint(end), 0u);
  return __uint_as_float(hl == 0u ? 0u : prev);
}

__device__ __forceinline__ uint32_t half_prefix_maps_excl(uint32_t m, uint32_t hl) {
  m = map_after(m, dpp_fill<0x111>(m, kMapIdentity));
  m = map_after(m, dpp_fill<0x112>(m, kMapIdentity));
  m = map_after(m, dpp_fill<0x114>(m, kMapIdentity));
  m = map_after(m, dpp_fill<0x118>(m, kMapIdentity));
  m = map_after(m, dpp_fill<0x142, 0xA>(m, kMapIdentity));
  const uint32_t prev = dpp_fill<kDppWaveShr1>(m, kMapIdentity);
  return hl == 0u ? kMapIdentity : prev;
}

// The 16 values of group gi of a strip row, in row order.
__device__ __forceinline__ void load_group(const float* row, uint32_t gi, float (&x)[16]) {
#pragma unroll
  for (uint32_t kr = 0; kr < 4u; kr++) {
    const f32x4 t = reinterpret_cast<const f32x4*>(row)[strip_slot(4u * gi + kr)];
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) x[4u * i + kr] = t[i];
  }
}

// The sum in order from 0.0 of a strip row per half-wave (ordered_sum_wave's
// method, rh_device.h, with 32 lanes a sum): lane hl holds the run of `mine`
// groups from group hl * per on, `lanes` lanes hold values, and t is an
// approximate sum of the lane's run. Every lane of the wave calls it. `rounds`
// as ordered_sum_wave's, one a half-wave.
__device__ __forceinline__ float ordered_sum_half(const float* row, uint32_t per, uint32_t mine, uint32_t lanes,
                                                  uint32_t groups, float t, uint32_t* rounds = nullptr) {
  const uint32_t lane = __lane_id(), hl = lane & 31u, half = lane >> 5;
  const uint32_t g0 = hl * per;
  double d = t;
  {
    const float g = half_guess_starts(d, hl);
    float e = g;
    for (uint32_t c = 0; c < mine; c++) {
      float x[16];
      load_group(row, g0 + c, x);
#pragma unroll
      for (int i = 0; i < 16; i++) e += x[i];
    }
    d = static_cast<double>(e) - static_cast<double>(g);
  }
  for (uint32_t r = 1;; r++) {
    const float g = half_guess_starts(d, hl);
    const uint32_t gb = __float_as_uint(g);
    const float cand[3] = {g, __uint_as_float(gb - 1u), __uint_as_float(gb + 1u)};
    float s[3] = {cand[0], cand[1], cand[2]};
    for (uint32_t c = 0; c < mine; c++) {
      float x[16];
      load_group(row, g0 + c, x);
#pragma unroll
      for (int i = 0; i < 16; i++) {
        s[0] += x[i];
        s[1] += x[i];
        s[2] += x[i];
      }
    }
    uint32_t next = dpp_fill<kDppWaveShl1>(gb, 0u);
    asm volatile("" : "+v"(next));  // kept out of DPP combining, as in ordered_sum_wave4
    uint32_t map = 0x03000000u;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const uint32_t delta = __float_as_uint(s[i]) - next;
      const uint32_t neg = delta >> 31;
      const uint32_t mag = min(neg ? 0u - delta : delta, 2u);
      map |= min(2u * mag - neg, 3u) << (8 * i);
    }
    if (hl + 1u >= lanes) map = kMapIdentity;
    const uint32_t state = half_prefix_maps_excl(map, hl) & 0xFFu;
    const float mine_end = state == 1u ? s[1] : state == 2u ? s[2] : s[0];
    const uint64_t bad = __ballot(hl < lanes && state == 3u);
    const uint32_t bad_h = static_cast<uint32_t>(bad >> (32u * half));
    const uint32_t fb = bad_h ? static_cast<uint32_t>(__builtin_ctz(bad_h)) : lanes;  // >= 1
    if (bad == 0 || r == kSumRounds) {
      float end = __shfl(mine_end, static_cast<int>(32u * half + fb - 1u), 64);
      // unresolved runs of the last round are added one value at a time
      for (uint32_t c = fb * per; c < groups; c++) {
        float x[16];
        load_group(row, c, x);
#pragma unroll
        for (int i = 0; i < 16; i++) end += x[i];
      }
      if (rounds && hl == 0u) rounds[half] = bad_h ? r + 1u : r;
      return end;
    }
    const float start = state == 1u ? cand[1] : state == 2u ? cand[2] : cand[0];
    d = hl < fb ? static_cast<double>(mine_end) - static_cast<double>(start)
                : static_cast<double>(s[0]) - static_cast<double>(cand[0]);
  }
}

// The cached rows of one layer in the strips' operand order, a group of 16
// rows at a time: consecutive lanes of an operand hold consecutive rows (keys)
// or output lanes (values), which in row order lie apart, and a load whose
// lanes lie apart costs a cycle a lane (the strips read every row once for
// each 16 query rows: 256 tokens behind 1744 rows spent 15.6 us in the scores
// and 13.8 in the mix on such loads).
//   keys: [kv head][group][HD / 4 pieces of four values][operand row][4],
//         operand row j being row 4 (j % 4) + j / 4 of the group;
//   values: [kv head][group][HD / 16][k = row % 4][16 output lanes][row / 4].
// cap: groups a kv head has room for.
template <uint32_t HD>
__global__ __launch_bounds__(256) void pack_kv_kernel(const float* __restrict__ kcache,
                                                      const float* __restrict__ vcache, uint32_t kv, uint32_t rows,
                                                      uint32_t cap, float* __restrict__ kpack,
                                                      float* __restrict__ vpack) {
  const uint32_t g = blockIdx.x, kvh = blockIdx.y, off = kvh * HD;
  const size_t to = static_cast<size_t>(kvh * cap + g) * 16u * HD;
#pragma unroll
  for (uint32_t t = threadIdx.x; t < 4u * HD; t += 256u) {
    const uint32_t e4 = t % (HD / 4u), rr = t / (HD / 4u), j = (rr & 3u) * 4u + (rr >> 2);
    reinterpret_cast<f32x4*>(kpack + to)[16u * e4 + j] = *reinterpret_cast<const f32x4*>(
        kcache + static_cast<size_t>(min(16u * g + rr, rows - 1u)) * kv + off + 4u * e4);
    const uint32_t d = t % HD, kr = t / HD;
    f32x4 x;
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++)
      x[i] = vcache[static_cast<size_t>(min(16u * g + 4u * i + kr, rows - 1u)) * kv + off + d];
    reinterpret_cast<f32x4*>(vpack + to)[64u * (d >> 4) + 16u * kr + (d & 15u)] = x;
  }
}

// Workgroup b's tile of tokens and run of heads, for `tiles` tiles of hx runs.
// Workgroups go to the eight XCDs in turn: a tile's heads stay on one XCD while
// its 32 CUs hold them or every XCD has a tile; otherwise they go round (8
// tokens behind 2350 rows, 40 heads of 64 over 8 kv heads, one tile: 41 us a
// layer less; 32 heads over 32, 9 tokens: 4 less behind 2000 rows, 1 more at 9;
// 16 heads of 128, one tile: 1 more at 9, 0 at 700).
struct StripPlace {
  uint32_t tile, heads;
};
__host__ __device__ constexpr uint32_t strip_turn(uint32_t tiles, uint32_t hx) {
  return tiles < 8u && hx >= 32u ? tiles : 8u;
}
__host__ __device__ constexpr uint32_t strip_grid(uint32_t tiles, uint32_t hx) {
  const uint32_t turn = strip_turn(tiles, hx);
  return hx * ((tiles + turn - 1u) / turn * turn);
}
__host__ __device__ constexpr StripPlace strip_place(uint32_t b, uint32_t tiles, uint32_t hx) {
  const uint32_t turn = strip_turn(tiles, hx), k = b / turn;
  return {b % turn + turn * (k / hx), k % hx};
}

// A workgroup owns 16 query rows -- 16 >> hs_log tokens of (1 << hs_log)
// heads that share a kv head -- over all their cached rows, three phases
// apart by a barrier:
//   1. scores: each wave takes groups of 16 cached rows in turn, HD / 4
//      MFMAs a 16 x 16 tile, the keys straight from memory into the A operand;
//   2. softmax: each half-wave takes one query row: exp, the ordered sum,
//      the division, in LDS;
//   3. the value mix: wave w owns output lanes 16w .. of all 16 query rows,
//      one MFMA per four cached rows, values straight from memory. The groups
//      that reach past some query row's last cached row are added lane by
//      lane, so that no masked row enters a chain.
// The scores stay in LDS between the phases (64 bytes a cached row), which
// caps a launch at kStripMaxGroups groups.
// What bounds it: the two products' MFMAs, HD / 4 of 32 cycles each a 16 x 16
// tile on four SIMDs, 13 us of a strip over 2000 rows of 64; measured, the
// scores take 9.7 us of it, the mix, one chain a SIMD, 11.9, and the softmax
// between them, which one workgroup a CU cannot overlap, 13.
// 2000 tokens of 32 heads of 64 over 4 kv heads: 339-349 us a layer with the
// packing, against 2521 for attention_group_kernel (a workgroup a token and
// kv head); 700 tokens of 16 heads of 128: 50 us against 381 for
// attention_kernel.
// ONE: one workgroup has the CU (strips over half its LDS), so a wave has
// twice the registers, and keeps more of its loads in flight.
template <uint32_t HD, bool ONE>
__global__ __launch_bounds__(kStripThreads, !ONE && HD == 64u ? 4 : 2) void attention_strip_kernel(
    const float* __restrict__ q, const float* __restrict__ kpack, const float* __restrict__ vpack,
    const float* __restrict__ vcache, uint32_t cap, uint32_t width, uint32_t kv, uint32_t heads, uint32_t hs_log,
    uint32_t group, float scale, uint32_t start, uint32_t n, uint32_t tile0, uint32_t tiles, uint32_t stride,
    float* __restrict__ mixed) {
  constexpr uint32_t MQ = HD / 32u;   // MFMA steps of a score chain
  constexpr uint32_t DT = HD / 16u;   // output tiles of 16 lanes
  constexpr uint32_t KA = ONE ? 4u : 2u, kMixAhead = ONE ? 16u : 8u;  // groups of keys, of values requested ahead
  static_assert(DT <= kStripWaves, "a wave an output tile");
  extern __shared__ __align__(16) float sh[];
  float* const strip = sh;                              // [16][stride]
  float* const red = strip + kStripQ * stride;          // [waves][16]
  uint64_t* const table = reinterpret_cast<uint64_t*>(red + kStripWaves * kStripQ);
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(tid >> 6)));
  const uint32_t j = lane & 15u, kq = lane >> 4;        // the lane's query row (or operand row) and k
  const uint32_t tps = kStripQ >> hs_log;               // tokens a strip
  const StripPlace place = strip_place(blockIdx.x, tiles, heads >> hs_log);
  if (place.tile >= tiles) return;
  const uint32_t t0 = (tile0 + tiles - 1u - place.tile) * tps;  // the longest strips first
  const uint32_t h0 = place.heads << hs_log, off = (h0 / group) * HD;
  const uint32_t tj = t0 + (j >> hs_log), hj = h0 + (j & ((1u << hs_log) - 1u));
  const uint32_t tc = min(tj, n - 1u);                  // past the batch: its last token, not stored
  const uint32_t pos = start + tc;                      // the last cached row of query row j
  const uint32_t last = start + min(t0 + tps - 1u, n - 1u);
  const uint32_t groups = (last >> 4) + 1u, full = (start + t0 + 1u) >> 4;  // full: whole for every query row

  if (tid < 32u) table[tid] = exp_table_entry(tid);

  // ---- scores
  // chain l, step m: k = kq is chunk c = 4m + kq, element 8c + l
  const float* const qp = q + static_cast<size_t>(tc) * width + hj * HD + 8u * kq;
  f32x4 qf[MQ][2];
#pragma unroll
  for (uint32_t m = 0; m < MQ; m++)
#pragma unroll
    for (uint32_t u = 0; u < 2u; u++) qf[m][u] = *reinterpret_cast<const f32x4*>(qp + 32u * m + 4u * u);
  // the group's keys in operand order (pack_kv_kernel): D's registers i of
  // lane (j, kq) are rows 4i + kq, a slot of the strip
  const uint32_t pg = (h0 / group) * cap;  // the kv head's first packed group
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(kpack + static_cast<size_t>(pg) * 16u * HD), 0, static_cast<int>(groups * 64u * HD),
      kBufferRsrcWord3);
  auto load_k = [&](f32x4 (&f)[MQ][2], uint32_t gi) {
    const int base = static_cast<int>(min(gi, groups - 1u) * 64u * HD);
#pragma unroll
    for (uint32_t m = 0; m < MQ; m++)
#pragma unroll
      for (uint32_t u = 0; u < 2u; u++)
        f[m][u] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(krs, static_cast<int>(512u * kq + 16u * j),
                                                         base + static_cast<int>(256u * (8u * m + u)), 0));
  };
  const double inv_scale = 1.0 / static_cast<double>(scale);
  float mx = -INFINITY;
  auto score = [&](const f32x4 (&f)[MQ][2], uint32_t gi) {
    v4f acc[8];
#pragma unroll
    for (uint32_t m = 0; m < MQ; m++)
#pragma unroll
      for (uint32_t l = 0; l < 8u; l++)
        acc[l] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[m][l >> 2][l & 3u], qf[m][l >> 2][l & 3u],
                                                      m ? acc[l] : v4f{}, 0, 0, 0);
    f32x4 sc;
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) {
      float s = acc[0][i];
#pragma unroll
      for (uint32_t l = 1; l < 8u; l++) s += acc[l][i];
      sc[i] = s;
    }
    // attention.rs:189-207: over sqrt(head_dim); 8 is a power of two
    if constexpr (HD == 64u) sc *= 0.125f;
    else div_by(sc, scale, inv_scale);
    // past the query row's last cached row: -inf, which the maximum drops and
    // whose exp, 0, changes no sum
    if (gi >= full) {
#pragma unroll
      for (uint32_t i = 0; i < 4u; i++)
        if (16u * gi + 4u * i + kq > pos) sc[i] = -INFINITY;
    }
#pragma unroll
    for (uint32_t i = 0; i < 4u; i++) mx = fmaxf(mx, sc[i]);
    reinterpret_cast<f32x4*>(strip + j * stride)[strip_slot(4u * gi + kq)] = sc;
  };
  // KA register sets by turns, each requested again as soon as it is used (a
  // copy between sets would wait for its loads)
  f32x4 kf[KA][MQ][2];
#pragma unroll
  for (uint32_t a = 0; a < KA; a++) load_k(kf[a], wave + a * kStripWaves);
  uint32_t gw = wave;
  for (; gw + (KA - 1u) * kStripWaves < groups; gw += KA * kStripWaves) {
#pragma unroll
    for (uint32_t a = 0; a < KA; a++) {
      score(kf[a], gw + a * kStripWaves);
      load_k(kf[a], gw + (a + KA) * kStripWaves);
    }
  }
#pragma unroll
  for (uint32_t a = 0; a + 1u < KA; a++)
    if (gw + a * kStripWaves < groups) score(kf[a], gw + a * kStripWaves);
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (lane < kStripQ) red[wave * kStripQ + lane] = mx;
  __syncthreads();

  // ---- softmax (norm.rs:17-30): half-wave `half` of each wave takes query row jr
  {
    static_assert(kStripQ == 2u * kStripWaves, "a query row a half-wave");
    const uint32_t half = lane >> 5, hl = lane & 31u, jr = 2u * wave + half;
    const uint32_t rows = start + min(t0 + (jr >> hs_log), n - 1u) + 1u;
    float* const row = strip + jr * stride;
    float m = red[jr];
#pragma unroll
    for (uint32_t w = 1; w < kStripWaves; w++) m = fmaxf(m, red[w * kStripQ + jr]);
    const uint32_t per = (groups + 31u) >> 5;
    const uint32_t own = (rows + 15u) >> 4, lanes = (own + per - 1u) / per;
    const uint32_t mine = hl < lanes ? min(per, own - hl * per) : 0u;
    float t = 0.0f;
    for (uint32_t c = 0; c < mine; c++) {
      const uint32_t gi = hl * per + c;
#pragma unroll
      for (uint32_t kr = 0; kr < 4u; kr++) {
        f32x4* const at = reinterpret_cast<f32x4*>(row) + strip_slot(4u * gi + kr);
        f32x4 x = *at;
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
          // x - max is at most 0, or NaN
          const float d = x[i] - m, e = expf_ref_inner(d, [&](uint32_t k) { return table[k]; });
          x[i] = d < -0x1.9fe368p6f ? 0.0f : e;
        }
        *at = x;
        t += (x[0] + x[1]) + (x[2] + x[3]);
      }
    }
    const float sum = ordered_sum_half(row, per, mine, lanes, own, t);
    const double inv = 1.0 / static_cast<double>(sum);
    for (uint32_t c = 0; c < mine; c++) {
#pragma unroll
      for (uint32_t kr = 0; kr < 4u; kr++) {
        f32x4* const at = reinterpret_cast<f32x4*>(row) + strip_slot(4u * (hl * per + c) + kr);
        f32x4 x = *at;
        div_by(x, sum, inv);
        *at = x;
      }
    }
  }
  __syncthreads();

  // ---- value mix (float.rs:52-62): out starts at 0.0, each row fused in order
  if (wave >= DT) return;
  const f32x4* const wrow = reinterpret_cast<const f32x4*>(strip + j * stride);
  v4f acc{};
  if (full) {
    const __amdgpu_buffer_rsrc_t prs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(vpack + static_cast<size_t>(pg) * 16u * HD), 0, static_cast<int>(full * 64u * HD),
        kBufferRsrcWord3);
    f32x4 v[kMixAhead];
    auto load_v = [&](f32x4& x, uint32_t gi) {
      x = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                     prs, static_cast<int>(16u * lane),
                     static_cast<int>(min(gi, full - 1u) * 64u * HD + 1024u * wave), 0));
    };
    auto mix = [&](const f32x4& x, const f32x4& w) {
#pragma unroll
      for (uint32_t i = 0; i < 4u; i++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], w[i], acc, 0, 0, 0);
    };
    auto weights = [&](uint32_t gi) { return wrow[strip_slot(4u * min(gi, full - 1u) + kq)]; };
#pragma unroll
    for (uint32_t a = 0; a < kMixAhead; a++) load_v(v[a], a);
    f32x4 w[2] = {weights(0u), weights(1u)};
    uint32_t g0 = 0;
    // whole rounds of the register sets without a branch, so that the loads
    // in flight are counted exactly at each wait
    for (; g0 + kMixAhead <= full; g0 += kMixAhead) {
#pragma unroll
      for (uint32_t a = 0; a < kMixAhead; a++) {
        mix(v[a], w[a & 1u]);
        load_v(v[a], g0 + a + kMixAhead);
        w[a & 1u] = weights(g0 + a + 2u);
      }
    }
#pragma unroll
    for (uint32_t a = 0; a + 1u < kMixAhead; a++)
      if (g0 + a < full) {
        mix(v[a], w[a & 1u]);
        w[a & 1u] = weights(g0 + a + 2u);
      }
  }
  // acc[i] is query row j's output lane 16 wave + 4 kq + i
  const int kvb = static_cast<int>(4u * kv);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(vcache), 0, static_cast<int>(last + 1u) * kvb, kBufferRsrcWord3);
  for (uint32_t gi = full; gi < groups; gi++) {
    float w[16];
    load_group(reinterpret_cast<const float*>(wrow), gi, w);
#pragma unroll
    for (uint32_t half = 0; half < 16u; half += 8u) {
      f32x4 x[8];
#pragma unroll
      for (uint32_t r = 0; r < 8u; r++)
        x[r] = __builtin_bit_cast(
            f32x4, __builtin_amdgcn_raw_buffer_load_b128(vrs, static_cast<int>(4u * (off + 16u * wave + 4u * kq)),
                                                         static_cast<int>(min(16u * gi + half + r, last)) * kvb, 0));
#pragma unroll
      for (uint32_t r = 0; r < 8u; r++)
#pragma unroll
        for (uint32_t i = 0; i < 4u; i++) {
          const float s = __builtin_fmaf(x[r][i], w[half + r], acc[i]);
          acc[i] = 16u * gi + half + r <= pos ? s : acc[i];
        }
    }
  }
  if (tj < n)
    *reinterpret_cast<f32x4*>(mixed + static_cast<size_t>(tj) * width + hj * HD + 16u * wave + 4u * kq) =
        f32x4{acc[0], acc[1], acc[2], acc[3]};
}

// One token at position `start` behind more rows than attention_step_lds_kernel
// holds: two launches, so that neither the key nor the value rows pass through
// one CU a head. 32 heads of 64 behind 1800 rows: 23-25 us, against 53 for
// attention_step_kernel and 30 for one workgroup of 1024 threads a head; 16
// heads of 128 behind 712: 15.5 us, against 47 for qkv_post_kernel and
// attention_kernel.
//
// step_scores_kernel: a wave takes 16 cached rows of one kv head and forms the
// scores of up to 16 of its query heads, with the strips' MFMAs. It rotates q
// and the new key itself (portable/rope.rs:7-23) and appends the new rows to
// the caches; no wave reads those rows from them. scores: [head][pitch].
template <uint32_t HD>
__global__ __launch_bounds__(256) void step_scores_kernel(
    const float* __restrict__ qr, const float* __restrict__ kr, const float* __restrict__ vr,
    const float* __restrict__ rcos, const float* __restrict__ rsin, float* kcache, float* vcache, uint32_t kv,
    uint32_t group, float scale, uint32_t start, uint32_t pitch, float* __restrict__ scores) {
  constexpr uint32_t MQ = HD / 32u;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, j = lane & 15u, kq = lane >> 4;
  const uint32_t r0 = 64u * blockIdx.x + 16u * wave;
  if (r0 > start) return;
  const uint32_t kvh = blockIdx.y, jh = 16u * blockIdx.z + j, off = kvh * HD;
  const uint32_t h = kvh * group + min(jh, group - 1u);
  const uint32_t row = min(r0 + j, start);
  const bool fresh = row == start;
  const float* const kp = (fresh ? kr : kcache + static_cast<size_t>(row) * kv) + off + 8u * kq;
  const float* const qp = qr + static_cast<size_t>(h) * HD + 8u * kq;
  const size_t rot = static_cast<size_t>(start) * (HD / 2u) + 4u * kq;
  f32x4 qf[MQ][2], kf[MQ][2], c[MQ], sn[MQ];
#pragma unroll
  for (uint32_t m = 0; m < MQ; m++) {
    c[m] = *reinterpret_cast<const f32x4*>(rcos + rot + 16u * m);
    sn[m] = *reinterpret_cast<const f32x4*>(rsin + rot + 16u * m);
#pragma unroll
    for (uint32_t u = 0; u < 2u; u++) {
      qf[m][u] = *reinterpret_cast<const f32x4*>(qp + 32u * m + 4u * u);
      kf[m][u] = *reinterpret_cast<const f32x4*>(kp + 32u * m + 4u * u);
    }
  }
#pragma unroll
  for (uint32_t m = 0; m < MQ; m++)
#pragma unroll
    for (uint32_t u = 0; u < 2u; u++) {
      f32x4 y, z;
#pragma unroll
      for (uint32_t i = 0; i < 2u; i++) {
        const float co = c[m][2u * u + i], si = sn[m][2u * u + i];
        const float ql = qf[m][u][2u * i], qh = qf[m][u][2u * i + 1u];
        const float kl = kf[m][u][2u * i], kh = kf[m][u][2u * i + 1u];
        const float qhs = qh * si, qls = ql * si, khs = kh * si, kls = kl * si;
        y[2u * i] = __builtin_fmaf(ql, co, -qhs);
        y[2u * i + 1u] = __builtin_fmaf(qh, co, qls);
        z[2u * i] = __builtin_fmaf(kl, co, -khs);
        z[2u * i + 1u] = __builtin_fmaf(kh, co, kls);
      }
      qf[m][u] = y;
      if (fresh) kf[m][u] = z;
    }
  if (r0 + j == start && blockIdx.z == 0) {
    float* const kd = kcache + static_cast<size_t>(start) * kv + off + 8u * kq;
    float* const vd = vcache + static_cast<size_t>(start) * kv + off + 8u * kq;
#pragma unroll
    for (uint32_t m = 0; m < MQ; m++)
#pragma unroll
      for (uint32_t u = 0; u < 2u; u++) {
        *reinterpret_cast<f32x4*>(kd + 32u * m + 4u * u) = kf[m][u];
        *reinterpret_cast<f32x4*>(vd + 32u * m + 4u * u) =
            *reinterpret_cast<const f32x4*>(vr + off + 8u * kq + 32u * m + 4u * u);
      }
  }
  v4f acc[8];
#pragma unroll
  for (uint32_t m = 0; m < MQ; m++)
#pragma unroll
    for (uint32_t l = 0; l < 8u; l++)
      acc[l] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[m][l >> 2][l & 3u], qf[m][l >> 2][l & 3u], m ? acc[l] : v4f{},
                                                    0, 0, 0);
  f32x4 sc;
#pragma unroll
  for (uint32_t i = 0; i < 4u; i++) {
    float s = acc[0][i];
#pragma unroll
    for (uint32_t l = 1; l < 8u; l++) s += acc[l][i];
    sc[i] = s;
  }
  if constexpr (HD == 64u) sc *= 0.125f;
  else div_by(sc, scale, 1.0 / static_cast<double>(scale));
  // rows 4 kq + i of the wave's 16 for query head j (the pitch has room for
  // the rows past the last)
  if (jh < group) *reinterpret_cast<f32x4*>(scores + static_cast<size_t>(h) * pitch + r0 + 4u * kq) = sc;
}

// step_mix_kernel: a workgroup takes kStepD output lanes of one query head:
// the softmax over the head's scores (every such workgroup forms the same
// one), with its slice of the value rows on its way into LDS meanwhile; then
// the lanes' chains of fused adds over the rows, on one wave.
// What bounds it: that chain. A dependent fused add takes 4.2 cycles, a lane's
// LDS reads of four rows' values and weights about as long again each: 12
// cycles a row, 10.3 us of 15.3 behind 1800 rows, the ordered sum 1.1.
constexpr uint32_t kStepD = 8;
constexpr uint32_t kMixThreads = 512;
constexpr uint32_t kMixEarly = 2;  // pieces of value rows a thread loads before the softmax

// LDS: the value slice, four rows x kStepD lanes a block of 32 floats, the
// weights, a reduction.
constexpr size_t step_mix_lds_bytes(size_t rows) {
  return 4u * (((rows + 3u) / 4u) * 32u + wave_sum_floats(static_cast<uint32_t>(rows)) + 16u);
}

// Slot of output lane d in block r4: exchanged so that the stores of a wave
// (a lane's four rows of four lanes, transposed) fall on distinct banks.
__device__ __forceinline__ uint32_t mix_slot(uint32_t r4, uint32_t d) { return 8u * r4 + (d ^ ((r4 >> 1) & 3u)); }

template <uint32_t HD>
__global__ __launch_bounds__(kMixThreads) void step_mix_kernel(const float* __restrict__ scores,
                                                               const float* __restrict__ vcache, uint32_t kv,
                                                               uint32_t group, uint32_t rows, uint32_t pitch,
                                                               float* __restrict__ mixed) {
  constexpr uint32_t SL = HD / kStepD, NWV = kMixThreads / 64u;
  extern __shared__ __align__(16) float sh[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t r4s = (rows + 3u) / 4u;
  f32x4* const vt = reinterpret_cast<f32x4*>(sh);              // [r4s][8] (mix_slot)
  float* const ws = sh + r4s * 32u;                     // exps, then weights (wave_sum_index)
  float* const red = ws + wave_sum_floats(rows);         // [8] maxima, [8] the sum
  // workgroups go to the eight XCDs in turn: the slices of a head, which share
  // the lines of its values, on one of them
  const uint32_t H = gridDim.x / SL, b = blockIdx.x;
  const uint32_t h = H % 8u == 0 ? (b & 7u) + 8u * ((b >> 3) / SL) : b / SL;
  const uint32_t slice = H % 8u == 0 ? (b >> 3) % SL : b % SL, off = (h / group) * HD + kStepD * slice;
  const float* const sp = scores + static_cast<size_t>(h) * pitch;

  // four rows x four lanes of values a piece: piece f is block f / 2, lanes 4 (f % 2) ..
  const uint32_t pieces = 2u * r4s;
  auto load_piece = [&](f32x4 (&x)[4], uint32_t f) {
    const uint32_t r = 4u * (f >> 1), o = off + 4u * (f & 1u);
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++)
      x[k] = *reinterpret_cast<const f32x4*>(vcache + static_cast<size_t>(min(r + k, rows - 1u)) * kv + o);
  };
  auto store_piece = [&](const f32x4 (&x)[4], uint32_t f) {
    if (f >= pieces) return;
#pragma unroll
    for (uint32_t u = 0; u < 4u; u++)
      vt[mix_slot(f >> 1, 4u * (f & 1u) + u)] = f32x4{x[0][u], x[1][u], x[2][u], x[3][u]};
  };
  // a thread's first four scores, then its first values: loads return in order
  f32x4 s0 = *reinterpret_cast<const f32x4*>(sp + min(4u * tid, 4u * (r4s - 1u)));
  f32x4 early[kMixEarly][4];
#pragma unroll
  for (uint32_t k = 0; k < kMixEarly; k++) load_piece(early[k], tid + k * kMixThreads);

  // ---- softmax (norm.rs:17-30)
  float mx = -INFINITY;
  for (uint32_t i = 4u * tid; i < rows; i += 4u * kMixThreads) {
    const f32x4 x = i == 4u * tid ? s0 : *reinterpret_cast<const f32x4*>(sp + i);
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++)
      if (i + k < rows) mx = fmaxf(mx, x[k]);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = red[0];
#pragma unroll
  for (uint32_t k = 1; k < NWV; k++) mx = fmaxf(mx, red[k]);
  // the exps; the sum's identity up to the end of the last chunk of 32
  for (uint32_t i = 4u * tid; i < ((rows + 31u) & ~31u); i += 4u * kMixThreads) {
    f32x4 x = s0;
    if (i != 4u * tid) x = *reinterpret_cast<const f32x4*>(sp + min(i, 4u * (r4s - 1u)));
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) {
      const float e = expf_ref(x[k] - mx);
      x[k] = i + k < rows ? e : -0.0f;
    }
    *reinterpret_cast<f32x4*>(ws + wave_sum_index(i)) = x;
  }
#pragma unroll
  for (uint32_t k = 0; k < kMixEarly; k++) store_piece(early[k], tid + k * kMixThreads);
  __syncthreads();
  if (wave == 0) {
    const float sum = ordered_sum_wave(ws, rows, 0.0f);
    if (lane == 0) red[8] = sum;
  } else {
    for (uint32_t f = kMixEarly * kMixThreads + tid - 64u; f < pieces; f += kMixThreads - 64u) {
      f32x4 x[4];
      load_piece(x, f);
      store_piece(x, f);
    }
  }
  __syncthreads();
  {
    const float sum = red[8];
    const double inv = 1.0 / static_cast<double>(sum);
    for (uint32_t i = 4u * tid; i < rows; i += 4u * kMixThreads) {
      f32x4* const w = reinterpret_cast<f32x4*>(ws + wave_sum_index(i));
      f32x4 x = *w;
      div_by(x, sum, inv);
      *w = x;
    }
  }
  __syncthreads();
  if (wave != 0) return;

  // ---- value mix (float.rs:52-62): eight blocks of four rows in flight (LDS
  // reads are counted up to 15), each read again as soon as it is added, 32
  // rows on; a lane's reads sit at fixed offsets of four addresses (one for
  // each exchange of mix_slot)
  if (lane >= kStepD) return;
  float acc = 0.0f;
  uint32_t vo[4];
#pragma unroll
  for (uint32_t i = 0; i < 4u; i++) vo[i] = lane ^ i;
  const f32x4* const wt = reinterpret_cast<const f32x4*>(ws);
  f32x4 v[8], w[8];
  auto add = [&](uint32_t i) {
#pragma unroll
    for (uint32_t k = 0; k < 4u; k++) acc = __builtin_fmaf(v[i][k], w[i][k], acc);
  };
  const uint32_t chunks = rows >> 5;
  if (chunks) {
#pragma unroll
    for (uint32_t i = 0; i < 8u; i++) {
      v[i] = vt[vo[i >> 1] + 8u * i];
      w[i] = wt[i];
    }
    for (uint32_t c = 1; c < chunks; c++) {
#pragma unroll
      for (uint32_t i = 0; i < 4u; i++) vo[i] += 64u;
#pragma unroll
      for (uint32_t i = 0; i < 8u; i++) {
        add(i);
        v[i] = vt[vo[i >> 1] + 8u * i];
        w[i] = wt[9u * c + i];
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < 8u; i++) add(i);
  }
  for (uint32_t r = 32u * chunks; r < rows; r++)
    acc = __builtin_fmaf(reinterpret_cast<const float*>(vt + mix_slot(r >> 2, lane))[r & 3u], ws[wave_sum_index(r)],
                         acc);
  mixed[static_cast<size_t>(h) * HD + kStepD * slice + lane] = acc;
}

template <uint32_t HD>
hipError_t launch_step(const float* qr, const float* kr, const float* vr, const float* rcos, const float* rsin,
                       float* kcache, float* vcache, uint32_t heads, uint32_t kv, uint32_t group, float scale,
                       uint32_t start, float* scores, uint32_t pitch, float* mixed, hipStream_t s) {
  hipLaunchKernelGGL((step_scores_kernel<HD>), dim3(start / 64u + 1u, kv / HD, (group + 15u) / 16u), dim3(256), 0, s,
                     qr, kr, vr, rcos, rsin, kcache, vcache, kv, group, scale, start, pitch, scores);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((step_mix_kernel<HD>), dim3(heads * (HD / kStepD)), dim3(kMixThreads),
                     step_mix_lds_bytes(start + 1u), s, scores, vcache, kv, group, start + 1u, pitch, mixed);
  return hipGetLastError();
}

// q/k/v from the projections, token-major: q and k rotated
// (portable/rope.rs:7-23), k and v into the cache at positions start + t. One
// thread per rotation pair (q, k) or pair of value elements.
__global__ __launch_bounds__(256) void rope_append_kernel(const float* __restrict__ qr, const float* __restrict__ kr,
                                                          const float* __restrict__ vr, uint32_t width, uint32_t kv,
                                                          uint32_t head_dim, const float* __restrict__ rcos,
                                                          const float* __restrict__ rsin, uint32_t start,
                                                          float* __restrict__ q, float* __restrict__ kcache,
                                                          float* __restrict__ vcache) {
  const uint32_t t = blockIdx.y, i = blockIdx.x * 256u + threadIdx.x;
  const uint32_t pos = start + t, qp = width / 2u, kp = kv / 2u;
  if (i < qp + kp) {
    const bool is_q = i < qp;
    const uint32_t e = is_q ? i : i - qp, pairs = head_dim / 2u, p = e % pairs;
    const f32x2 x = reinterpret_cast<const f32x2*>(is_q ? qr + static_cast<size_t>(t) * width
                                                        : kr + static_cast<size_t>(t) * kv)[e];
    const float c = rcos[static_cast<size_t>(pos) * pairs + p], s = rsin[static_cast<size_t>(pos) * pairs + p];
    const float hs = x[1] * s, ls = x[0] * s;
    f32x2 y;
    y[0] = __builtin_fmaf(x[0], c, -hs);
    y[1] = __builtin_fmaf(x[1], c, ls);
    reinterpret_cast<f32x2*>(is_q ? q + static_cast<size_t>(t) * width : kcache + static_cast<size_t>(pos) * kv)[e] = y;
  } else if (i < qp + 2u * kp) {
    const uint32_t e = i - qp - kp;
    reinterpret_cast<f32x2*>(vcache + static_cast<size_t>(pos) * kv)[e] =
        reinterpret_cast<const f32x2*>(vr + static_cast<size_t>(t) * kv)[e];
  }
}

// The most groups of a strip of which `fit` share a CU's LDS.
constexpr uint32_t strip_max_groups(uint32_t fit) {
  uint32_t g = 0;
  while (strip_lds_bytes(g + 4u) * fit <= kLdsBytes) g += 4u;
  return g;
}
constexpr uint32_t kStripMaxGroups = strip_max_groups(1u), kStripHalfGroups = strip_max_groups(2u);

template <uint32_t HD>
hipError_t launch_strips(const float* q, const float* kcache, const float* vcache, float* pack, uint32_t cap,
                         uint32_t width, uint32_t kv, uint32_t heads, uint32_t group, float scale, uint32_t start,
                         uint32_t n, float* mixed, hipStream_t s) {
  float* const vpack = pack + static_cast<size_t>(cap) * 16u * kv;
  hipLaunchKernelGGL((pack_kv_kernel<HD>), dim3((start + n + 15u) / 16u, kv / HD), dim3(256), 0, s, kcache, vcache, kv,
                     start + n, cap, pack, vpack);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
  // heads a strip: the query heads of a kv head as far as 16 rows hold them
  // evenly (the tokens of a strip then span few rows past the shared groups)
  uint32_t hs_log = 0;
  while (hs_log < 4u && group % (2u << hs_log) == 0) hs_log++;
  const uint32_t tps = kStripQ >> hs_log, tiles = (n + tps - 1u) / tps;
  // tokens whose strips take less than half the LDS go in a launch of their
  // own, two workgroups a CU, where they have work for the whole chip
  const uint32_t half = 16u * kStripHalfGroups;  // rows of those strips
  uint32_t cut = half > start ? std::min(tiles, (half - start) / tps) : 0u;
  if (cut < tiles && cut * (heads >> hs_log) < 512u) cut = 0;
  for (uint32_t part = 0; part < 2u; part++) {
    const uint32_t t0 = part ? cut : 0u, t1 = part ? tiles : cut;
    if (t0 == t1) continue;
    const uint32_t groups = (start + std::min(t1 * tps, n) - 1u) / 16u + 1u;
    const auto fn = groups > kStripHalfGroups ? attention_strip_kernel<HD, true> : attention_strip_kernel<HD, false>;
    hipLaunchKernelGGL(fn, dim3(strip_grid(t1 - t0, heads >> hs_log)), dim3(kStripThreads),
                       strip_lds_bytes(groups), s, q, pack, vpack, vcache, cap, width, kv, heads, hs_log, group, scale,
                       start, n, t0, t1 - t0, strip_stride(groups), mixed);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// ---- test hooks' kernels, one wave each

// ordered_sum_half over values[0][0..n0) and values[1][0..n1), in strip rows
// of `stride` floats, +0.0 past their ends as the masked exps are.
__global__ __launch_bounds__(64) void ordered_sum_half_kernel(const float* values, uint32_t n0, uint32_t n1,
                                                              uint32_t groups, uint32_t stride, float* out,
                                                              uint32_t* rounds) {
  extern __shared__ __align__(16) float sh[];
  for (uint32_t j = 0; j < 2u; j++)
    for (uint32_t i = threadIdx.x; i < 16u * groups; i += 64u)
      sh[j * stride + 4u * strip_slot((i >> 4) * 4u + (i & 3u)) + ((i >> 2) & 3u)] =
          i < (j ? n1 : n0) ? values[j * 16u * groups + i] : 0.0f;
  __syncthreads();
  const uint32_t half = threadIdx.x >> 5, hl = threadIdx.x & 31u, rows = half ? n1 : n0;
  const float* const row = sh + half * stride;
  const uint32_t per = (groups + 31u) >> 5, own = (rows + 15u) >> 4, lanes = (own + per - 1u) / per;
  const uint32_t mine = hl < lanes ? min(per, own - hl * per) : 0u;
  float t = 0.0f;
  for (uint32_t c = 0; c < mine; c++) {
    float x[16];
    load_group(row, hl * per + c, x);
    for (int i = 0; i < 16; i++) t += x[i];
  }
  const float sum = ordered_sum_half(row, per, mine, lanes, own, t, rounds);
  if (hl == 0u) out[half] = sum;
}

// y[i] = x[i] / d by div_by, n a multiple of 4.
__global__ __launch_bounds__(64) void div_by_kernel(const float* x, uint32_t n, float d, float* y) {
  const double inv = 1.0 / static_cast<double>(d);
  for (uint32_t i = blockIdx.x * 64u + threadIdx.x; i < n / 4u; i += 64u * gridDim.x) {
    f32x4 v = reinterpret_cast<const f32x4*>(x)[i];
    div_by(v, d, inv);
    reinterpret_cast<f32x4*>(y)[i] = v;
  }
}

// d[16][16] = the MFMA chain over a[16][k] and b[k][16] from 0.0.
__global__ __launch_bounds__(64) void mfma_chain_kernel(const float* a, const float* b, uint32_t k, float* d) {
  const uint32_t j = threadIdx.x & 15u, kq = threadIdx.x >> 4;
  v4f acc{};
  for (uint32_t s = 0; s < k; s += 4u)
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j * k + s + kq], b[(s + kq) * 16u + j], acc, 0, 0, 0);
#pragma unroll
  for (uint32_t i = 0; i < 4u; i++) d[(4u * kq + i) * 16u + j] = acc[i];
}

constexpr size_t kMaxHookValues = size_t{1} << 24;

// in[0..n) to the device, `launch` on it and m floats of output, those back.
template <typename Launch>
rh_status run_hook(rh_ctx* ctx, const float* in, size_t n, float* out, size_t m, Launch launch) {
  if (hipSetDevice(ctx_device(ctx)) != hipSuccess) return RH_ERR_DEVICE;
  const hipStream_t s = static_cast<hipStream_t>(rh_stream(ctx));
  float *din = nullptr, *dout = nullptr;
  if (hipMalloc(reinterpret_cast<void**>(&din), n * 4u) != hipSuccess) return RH_ERR_OUT_OF_MEMORY;
  if (hipMalloc(reinterpret_cast<void**>(&dout), m * 4u) != hipSuccess) {
    (void)hipFree(din);
    return RH_ERR_OUT_OF_MEMORY;
  }
  hipError_t e = hipMemcpyAsync(din, in, n * 4u, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) {
    launch(din, dout, s);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipMemcpyAsync(out, dout, m * 4u, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  (void)hipFree(din);
  (void)hipFree(dout);
  return e == hipSuccess ? RH_OK : RH_ERR_DEVICE;
}

}  // namespace

// Rows (cached and new) from which a batch of n tokens takes strips: the
// lines where they and the kernels they replace measured the same. Strips cost
// a packing launch more, and where the O matrix's operand is `quantized` its
// launch; the others cost a workgroup per token and head (attention_kernel) or
// kv head (attention_group_kernel, `grouped`), free until they fill the chip.
// us a layer, strips less the other kernels, 32 heads of 64 unless stated:
//   grouped: eight heads a kv head -3 from 224 rows on (8 tokens); four, up to
//   8 tokens and quantized, +2 at 224 and -3 at 800, 12 tokens +2 at 260 and
//   -2 at 350, 48 tokens -3 at 224. 64 tokens, eight heads: 219 against 222 us
//   at 192 rows for two layers, which is why nothing here lies below 224.
//   token_major (k-quant GEMMs store q, k, v and the O rows token-major for
//   strips, row-major for attention_kernel): -1 to -6 from the first row on.
//   others, up to 256 (token, head) pairs, where the packing's share grows
//   with the kv width: 2 kv heads +1 at 700 rows, -1 at 1000; 16 kv heads +2 at
//   1000, -1 at 1400; 32 kv heads +3 at 1200, 0 at 1700. 384 pairs: +1 to +3 at
//   400, -4 at 1000; 768: +1 at 120, -2 at 260; 1536: -3 at 48.
//   16 heads of 128: 8 tokens +4 at 8 rows, +1 at 120, -3 at 224; 32 tokens +2
//   at 32, -9 at 180; 48 tokens -3 at 48.
size_t attention_strip_rows(size_t head_dim, size_t heads, size_t kv_heads, size_t n, bool grouped, bool quantized,
                            bool token_major) {
  const size_t pairs = n * heads;
  if (grouped) {
    if (heads / kv_heads == 8u || n >= 24u) return 224u;
    return quantized && n <= 8u ? 640u : 320u;
  }
  if (token_major) return 0u;
  if (head_dim == 128u) return pairs <= 256u ? 144u : pairs < 768u ? 64u : 0u;
  return pairs <= 256u ? 768u + kv_heads * head_dim / 2u : pairs <= 512u ? 512u : pairs < 1536u ? 160u : 0u;
}

bool attention_strip_ok(size_t head_dim, size_t heads, size_t kv_heads, size_t rows, size_t n, bool grouped,
                        bool quantized, bool token_major) {
  return attention_strip_shape(head_dim) && n >= 2u && rows <= 16u * kStripMaxGroups &&
         rows >= attention_strip_rows(head_dim, heads, kv_heads, n, grouped, quantized, token_major);
}

bool attention_strip_shape(size_t head_dim) { return head_dim == 64u || head_dim == 128u; }

// Groups a kv head has room for in the packed rows, and their floats.
static uint32_t strip_cap(size_t context) {
  return static_cast<uint32_t>(std::min<size_t>((context + 15u) / 16u, kStripMaxGroups));
}
size_t attention_pack_floats(size_t context, size_t kv) { return 2u * strip_cap(context) * size_t{16} * kv; }

hipError_t launch_attention_strip(const float* q, const float* kcache, const float* vcache, float* pack,
                                  size_t context, uint32_t width, uint32_t kv, uint32_t head_dim, float scale,
                                  uint32_t start, uint32_t n, float* mixed, hipStream_t s) {
  const uint32_t heads = width / head_dim, group = heads / (kv / head_dim), cap = strip_cap(context);
  if (head_dim == 64u)
    return launch_strips<64>(q, kcache, vcache, pack, cap, width, kv, heads, group, scale, start, n, mixed, s);
  return launch_strips<128>(q, kcache, vcache, pack, cap, width, kv, heads, group, scale, start, n, mixed, s);
}

// Heads of 64 up to 256 rows, a key row a thread of attention_step_kernel, stay
// there: generation, two launches less that one, +1.4 us a layer at 235 rows,
// -0.1 at 260, -1.0 at 320, -2.5 at 410 (8 to 32 heads). Heads of 128 gain at
// every length (-3.1 over the first 200 rows).
constexpr size_t kStepMinRows64 = 257;

// The most rows whose values and weights step_mix_kernel holds.
constexpr size_t step_max_rows() {
  size_t rows = 0;
  while (step_mix_lds_bytes(rows + 4u) <= kLdsBytes) rows += 4u;
  return rows;
}
constexpr size_t kStepMaxRows = step_max_rows();

bool attention_step_long_ok(size_t head_dim, size_t rows) {
  return ((head_dim == 64u && rows >= kStepMinRows64) || head_dim == 128u) && rows <= kStepMaxRows;
}

size_t attention_step_pitch(size_t context) { return (std::min(context, kStepMaxRows) + 63u) & ~size_t{63}; }

size_t attention_step_floats(size_t head_dim, size_t heads, size_t context) {
  return attention_step_long_ok(head_dim, std::min(context, kStepMaxRows)) ? heads * attention_step_pitch(context) : 0u;
}

hipError_t launch_attention_step_long(const float* qr, const float* kr, const float* vr, const float* rcos,
                                      const float* rsin, float* kcache, float* vcache, uint32_t heads, uint32_t kv,
                                      uint32_t head_dim, float scale, uint32_t start, float* scores, uint32_t pitch,
                                      float* mixed, hipStream_t s) {
  const uint32_t group = heads / (kv / head_dim);
  if (head_dim == 64u)
    return launch_step<64>(qr, kr, vr, rcos, rsin, kcache, vcache, heads, kv, group, scale, start, scores, pitch,
                           mixed, s);
  return launch_step<128>(qr, kr, vr, rcos, rsin, kcache, vcache, heads, kv, group, scale, start, scores, pitch, mixed,
                          s);
}

hipError_t launch_rope_append(const float* qr, const float* kr, const float* vr, uint32_t width, uint32_t kv,
                              uint32_t head_dim, const float* rcos, const float* rsin, uint32_t start, uint32_t n,
                              float* q, float* kcache, float* vcache, hipStream_t s) {
  const uint32_t work = width / 2u + kv;
  hipLaunchKernelGGL(rope_append_kernel, dim3((work + 255u) / 256u, n), dim3(256), 0, s, qr, kr, vr, width, kv,
                     head_dim, rcos, rsin, start, q, kcache, vcache);
  return hipGetLastError();
}

}  // namespace rh

extern "C" {

// Test hook: the softmax's ordered sums of a strip's two rows, values[0] and
// values[1] at a distance of whole groups of 16 (16 * groups floats each);
// rounds: as rh_ordered_sum_device, one a row.
rh_status rh_ordered_sum_half_device(rh_ctx* ctx, const float* values, size_t groups, size_t n0, size_t n1, float* sums,
                                     uint32_t* rounds) {
  if (!ctx || !values || !sums || !rounds || groups == 0 || groups > rh::kStripMaxGroups || n0 == 0 || n1 == 0 ||
      n0 > 16u * groups || n1 > 16u * groups)
    return RH_ERR_INVALID_ARGUMENT;
  float out[4] = {};
  const uint32_t g = static_cast<uint32_t>(groups), stride = rh::strip_stride(g);
  const rh_status st = rh::run_hook(ctx, values, 32u * groups, out, 4, [&](float* in, float* o, hipStream_t s) {
    hipLaunchKernelGGL(rh::ordered_sum_half_kernel, dim3(1), dim3(64), 8u * stride, s, in, static_cast<uint32_t>(n0),
                       static_cast<uint32_t>(n1), g, stride, o, reinterpret_cast<uint32_t*>(o + 2));
  });
  std::memcpy(sums, out, 8);
  std::memcpy(rounds, out + 2, 8);
  return st;
}

// Test hook: x[i] / d as the softmax divides its weights; n a multiple of 4.
rh_status rh_div_by_device(rh_ctx* ctx, const float* x, size_t n, float d, float* y) {
  if (!ctx || !x || !y || n == 0 || n % 4u || n > rh::kMaxHookValues) return RH_ERR_INVALID_ARGUMENT;
  return rh::run_hook(ctx, x, n, y, n, [&](float* in, float* o, hipStream_t s) {
    hipLaunchKernelGGL(rh::div_by_kernel, dim3(256), dim3(64), 0, s, in, static_cast<uint32_t>(n), d, o);
  });
}

// Test hook: the products of a[16][k] and b[k][16] (one after the other at ab)
// on the f32 matrix cores, as the attention kernels form their chains; k a
// multiple of 4.
rh_status rh_mfma_chain_device(rh_ctx* ctx, const float* ab, size_t k, float* d) {
  if (!ctx || !ab || !d || k == 0 || k % 4u || 32u * k > rh::kMaxHookValues) return RH_ERR_INVALID_ARGUMENT;
  return rh::run_hook(ctx, ab, 32u * k, d, 256, [&](float* in, float* o, hipStream_t s) {
    hipLaunchKernelGGL(rh::mfma_chain_kernel, dim3(1), dim3(64), 0, s, in, in + 16u * k, static_cast<uint32_t>(k), o);
  });
}

// Test hook: whether a batch of n tokens whose rows end at `rows` takes strips.
int rh_strip_route_host(size_t head_dim, size_t heads, size_t kv_heads, size_t rows, size_t n, int grouped,
                        int quantized, int token_major) {
  return rh::attention_strip_ok(head_dim, heads, kv_heads, rows, n, grouped, quantized, token_major);
}

// Test hook: whether a token at row `rows` takes the split step.
int rh_step_route_host(size_t head_dim, size_t rows) { return rh::attention_step_long_ok(head_dim, rows); }

// Test hook: floats of the split step's score scratch.
size_t rh_step_scratch_host(size_t head_dim, size_t heads, size_t context) {
  return rh::attention_step_floats(head_dim, heads, context);
}

// Test hook: workgroup b's tile and run of heads; returns the grid.
uint32_t rh_strip_place_host(uint32_t b, uint32_t tiles, uint32_t hx, uint32_t* tile, uint32_t* heads) {
  const rh::StripPlace at = rh::strip_place(b, tiles, hx);
  *tile = at.tile;
  *heads = at.heads;
  return rh::strip_grid(tiles, hx);
}

}  // extern "C"
