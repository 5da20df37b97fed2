// Backend::matmul with a bf16 weight (crates/yaxus-backend-cpu/src/lib.rs:234-248,
// 314-345) where matmul_bf16_rows (step_after.hpp, one 16 x 16 tile of the output per
// workgroup) reads its operands too often: passes of many rows, and few rows against
// many weight rows (logits). out[t][n] = x[t][:] . w[n][:], f32 activations and result.
// x goes in as three bf16 parts (its 24 significand bits cut in three by truncation), so
// every product is exact and only the f32 sums round; infinities are carried by the
// first part alone.
//
// Operand layouts of v_mfma_f32_16x16x32_bf16 as in step_after.hpp: A = 16 weight rows,
// B = 16 rows of one part of x, D: lane (c, g) holds out[t0 + c][n0 + 4g + i].
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "attn_decode.hpp"

namespace yx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// The bf16 parts of two f32 values, packed: h, m, l hold (value 1 << 16 | value 0). An
// infinite value has NaN in m and l unless kInf, which costs a compare and a select.
template <bool kInf>
__device__ __forceinline__ void split_bf16x3(float f0, float f1, uint32_t& h, uint32_t& m, uint32_t& l) {
  const float f[2] = {f0, f1};
  uint32_t hb[2], mb[2], lb[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    hb[i] = __float_as_uint(f[i]);
    float r = f[i] - __uint_as_float(hb[i] & 0xffff0000u);
    if (kInf && __builtin_isinf(f[i])) r = 0.0f;
    mb[i] = __float_as_uint(r);
    lb[i] = __float_as_uint(r - __uint_as_float(mb[i] & 0xffff0000u));
  }
  h = __builtin_amdgcn_perm(hb[1], hb[0], 0x07060302);  // the upper halves of both
  m = __builtin_amdgcn_perm(mb[1], mb[0], 0x07060302);
  l = __builtin_amdgcn_perm(lb[1], lb[0], 0x07060302);
}

// A lane's four outputs of a 16 x 16 tile: columns col .. col + 3 of one row.
__device__ __forceinline__ void store_out4(float* out, uint32_t row, uint32_t col, uint32_t n, bool wide,
                                           const f32x4& v) {
  float* o = out + static_cast<size_t>(row) * n + col;
  if (wide) {  // n a multiple of 4, out 16-byte aligned
    if (col < n) *reinterpret_cast<f32x4*>(o) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (col + i < n) o[i] = v[i];
  }
}

// ---- many rows -------------------------------------------------------------------
// A workgroup of 8 waves owns a TM x TN tile of the output (WM x WN waves) and walks k in
// stages of KU * 32: x (f32) and w go through registers into one of two LDS slots, x as
// its three parts, so a stage of x is cut up once per workgroup. What bounds it is the
// matrix pipe: three instructions per 16 x 16 x 32 (t 4096, k = n = 2048: 6.3M of them,
// 47 us at 2.1 GHz), and on gfx950 vector instructions beyond about one per matrix
// instruction add to that time, in the same wave or in the SIMD's other one. Hence:
//  - the waves form two groups half a stage apart (one wave of each per SIMD): while one
//    group's waves run their matrix instructions, the others read their operands from
//    LDS and write the next stage (matrix and data phases of all waves together: 98 us,
//    apart: 87 us);
//  - the parts of the next stage but one are computed between the matrix instructions,
//    one vector instruction after each (two: 91 us);
//  - loads are buffer loads from a scalar base (no address arithmetic; rows past t or n
//    lie beyond the resource and read zeros), two stages ahead;
//  - infinities are looked for by a running maximum (4 instructions per 8 values); a tile
//    that has one is done again with the parts that allow for them.
// LDS: per 32 k, chunks of 8 k in [row][4], chunk g of row r at g ^ (r / 2 % 4), so that
// 8 consecutive lanes of an operand read hit 128 different bytes (no bank conflicts
// counted).
// Accuracy: sums of at most an eighth of k (and at least two stages) are added to the
// result in f32, as matmul_bf16_rows adds its waves' eighths; one chain over k = 2048
// was 4.8e-7 off 64 bits (2-norm), this is 1.8e-7, as that kernel.
// With ks > 1 (grid y) the ks workgroups of a tile take consecutive stages and hand
// their tiles over as matmul_bf16_rows does.
// Measured (k = n = 2048): t 4096 702 -> 81 us (128 x 256 tiles, 425 TFLOP/s, 3x that in
// matrix instructions), t 2048 350 -> 54, t 512 90 -> 22, t 80 19.4 -> 12.0.
template <int TM_, int TN_, int WM_, int WN_, int KU_, int kWaves_>
struct MatmulTile {
  static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, KU = KU_, KT = 32 * KU_;
  static constexpr int kWavesPerSimd = kWaves_;  // for the register budget
};
static constexpr int kMatmulThreads = 512;
using MatmulTileA = MatmulTile<128, 256, 4, 2, 1, 2>;
using MatmulTileB = MatmulTile<128, 128, 4, 2, 1, 2>;
using MatmulTileC = MatmulTile<64, 128, 2, 4, 2, 2>;
using MatmulTileD = MatmulTile<64, 64, 2, 4, 2, 4>;

template <class T>
__global__ __launch_bounds__(kMatmulThreads, T::kWavesPerSimd) void matmul_bf16_tiles(
    const float* __restrict__ x, const uint16_t* __restrict__ w, float* __restrict__ out, uint32_t t,
    uint32_t k, uint32_t n, f32x4* __restrict__ part, uint32_t part_bytes,
    uint32_t* __restrict__ counters) {
  constexpr int TM = T::TM, TN = T::TN, KU = T::KU, KT = T::KT, TH = kMatmulThreads;
  static_assert(T::WM * T::WN * 64 == TH, "8 waves");
  constexpr int MT = TM / T::WM / 16, NT = TN / T::WN / 16;  // 16 x 16 tiles per wave
  // Chunks of 8 k per thread and stage.
  constexpr int XC = TM * KT / 8 / TH, WC = TN * KT / 8 / TH;
  static_assert(TM * KT / 8 == XC * TH && TN * KT / 8 == WC * TH, "whole rounds of chunks");
  constexpr int kOutside = 0x7ffffff0;  // beyond every resource: reads zeros
  __shared__ u16x8 xs[2][KU][3][TM * 4];
  __shared__ u16x8 ws[2][KU][TN * 4];
  __shared__ uint32_t last;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int c = lane & 15, g = lane >> 4, sw = g ^ ((c >> 1) & 3);
  const int wm = wave / T::WN, wn = wave % T::WN;
  // Tiles so that those running on one XCD (workgroups are dealt to the 8 XCDs in turn)
  // are consecutive, the operand with fewer tiles fastest: they share operands in its L2.
  const uint32_t ntn = (n + TN - 1) / TN, ntt = (t + TM - 1) / TM, tiles = ntn * ntt;
  const uint32_t xcd = blockIdx.x & 7;
  const uint32_t tile = xcd * (tiles >> 3) + min(xcd, tiles & 7) + (blockIdx.x >> 3);
  const uint32_t n0 = (ntn <= ntt ? tile % ntn : tile / ntt) * TN;
  const uint32_t t0 = (ntn <= ntt ? tile / ntn : tile % ntt) * TM;
  const uint32_t ks = gridDim.y, kp = blockIdx.y;
  const uint32_t stages = (k + KT - 1) / KT;
  const uint32_t s0 = static_cast<uint32_t>(static_cast<uint64_t>(stages) * kp / ks);
  const uint32_t s1 = static_cast<uint32_t>(static_cast<uint64_t>(stages) * (kp + 1) / ks);
  const uint32_t seg = max(2u, (stages >> 3) & ~1u);  // stages per partial sum (even: the slots alternate)

  int xd[XC], wd[WC], xo[XC], wo[WC];  // LDS chunk, global byte offset in the tile's rows
  uint32_t xk[XC], wk[WC];             // first k of the chunk within its stage
#pragma unroll
  for (int i = 0; i < XC; ++i) {
    const int id = i * TH + tid, row = id / (4 * KU), kc = id % (4 * KU);
    xk[i] = kc * 8;
    xo[i] = (row * static_cast<int>(k) + kc * 8) * 4;
    xd[i] = (kc / 4) * 3 * TM * 4 + row * 4 + ((kc & 3) ^ ((row >> 1) & 3));
  }
#pragma unroll
  for (int i = 0; i < WC; ++i) {
    const int id = i * TH + tid, row = id / (4 * KU), kc = id % (4 * KU);
    wk[i] = kc * 8;
    wo[i] = (row * static_cast<int>(k) + kc * 8) * 2;
    wd[i] = (kc / 4) * TN * 4 + row * 4 + ((kc & 3) ^ ((row >> 1) & 3));
  }
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(const_cast<float*>(x + static_cast<size_t>(t0) * k),
                                              min(t - t0, static_cast<uint32_t>(TM)) * k * 4);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(const_cast<uint16_t*>(w + static_cast<size_t>(n0) * k),
                                              min(n - n0, static_cast<uint32_t>(TN)) * k * 2);
  struct XRegs {
    f32x4 a[XC], b[XC];
  };
  struct WRegs {
    u16x8 v[WC];
  };
  struct XParts {
    u32x4 p[XC][3];
  };
  // Stage s (the last one again past the end, which nothing uses).
  const auto load_x = [&](XRegs& r, uint32_t s) {
    const uint32_t kb = min(s, s1 - 1) * KT;
    const bool tail = kb + KT > k;  // uniform
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const int o = tail && kb + xk[i] >= k ? kOutside : xo[i];
      r.a[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, kb * 4, 0));
      r.b[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, kb * 4 + 16, 0));
    }
  };
  const auto load_w = [&](WRegs& r, uint32_t s) {
    const uint32_t kb = min(s, s1 - 1) * KT;
    const bool tail = kb + KT > k;
#pragma unroll
    for (int i = 0; i < WC; ++i) {
      const int o = tail && kb + wk[i] >= k ? kOutside : wo[i];
      r.v[i] = __builtin_bit_cast(u16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, o, kb * 2, 0));
    }
  };
  float big = 0.0f;  // the largest |x| this thread has cut up
  const auto split = [&](XParts& o, const XRegs& r, auto inf) {
#pragma unroll
    for (int i = 0; i < XC; ++i) {
      const float v[8] = {r.a[i].x, r.a[i].y, r.a[i].z, r.a[i].w, r.b[i].x, r.b[i].y, r.b[i].z, r.b[i].w};
      // (The instruction itself: fmaxf and fabsf would canonicalise each operand first.)
      if (!decltype(inf)::value) {
#pragma unroll
        for (int e = 0; e < 8; e += 2)
          asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(big) : "v"(v[e]), "v"(v[e + 1]));
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t h, m, l;
        split_bf16x3<decltype(inf)::value>(v[2 * e], v[2 * e + 1], h, m, l);
        o.p[i][0][e] = h;
        o.p[i][1][e] = m;
        o.p[i][2][e] = l;
      }
    }
  };
  const auto write = [&](const XParts& xp, const WRegs& wr, int slot) {
    u16x8* xb = &xs[slot][0][0][0];
    u16x8* wb = &ws[slot][0][0];
#pragma unroll
    for (int i = 0; i < XC; ++i) {
#pragma unroll
      for (int q = 0; q < 3; ++q) xb[xd[i] + q * TM * 4] = __builtin_bit_cast(u16x8, xp.p[i][q]);
    }
#pragma unroll
    for (int i = 0; i < WC; ++i) wb[wd[i]] = wr.v[i];
  };
  bf16x8 wf[KU][NT], xf[KU][MT][3];
  const auto read_operands = [&](int slot) {
#pragma unroll
    for (int u = 0; u < KU; ++u) {
#pragma unroll
      for (int a = 0; a < NT; ++a)
        wf[u][a] = __builtin_bit_cast(bf16x8, ws[slot][u][(wn * NT * 16 + a * 16 + c) * 4 + sw]);
#pragma unroll
      for (int b = 0; b < MT; ++b)
#pragma unroll
        for (int q = 0; q < 3; ++q)
          xf[u][b][q] = __builtin_bit_cast(bf16x8, xs[slot][u][q][(wm * MT * 16 + b * 16 + c) * 4 + sw]);
    }
  };
  f32x4 acc[NT][MT], sum[NT][MT];
  const auto multiply = [&](auto first) {  // first: a new partial sum
#pragma unroll
    for (int u = 0; u < KU; ++u)
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
          for (int b = 0; b < MT; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wf[u][a], xf[u][b][q], decltype(first)::value && u == 0 && q == 0 ? f32x4{0, 0, 0, 0} : acc[a][b],
                0, 0, 0);
  };
  const auto barrier = []() {  // nothing moves from one phase to the other
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  // Every wave passes the same number of barriers: the late group one more before its
  // first stage, the other one more after its last. Stage s + 1 is in its slot once both
  // groups have passed the barrier that ends their data phase of stage s; that slot's
  // earlier content (stage s - 1) was last read in the data phases before those.
  const bool late = wave >= 4;
  XRegs xr[2];
  WRegs wr[2];
  XParts xp;
  const auto run = [&](auto inf) {
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < MT; ++b) sum[a][b] = f32x4{0, 0, 0, 0};
    load_x(xr[0], s0);
    load_w(wr[0], s0);
    load_x(xr[1], s0 + 1);
    load_w(wr[1], s0 + 1);
    split(xp, xr[0], inf);
    write(xp, wr[0], 0);
    load_x(xr[0], s0 + 2);
    load_w(wr[0], s0 + 2);
    split(xp, xr[1], inf);
    load_x(xr[1], s0 + 3);
    barrier();
    if (late) barrier();
    const auto stage = [&](uint32_t s, auto parity, auto first) {
      constexpr int P = decltype(parity)::value;
      write(xp, wr[P ^ 1], P ^ 1);
      load_w(wr[P ^ 1], s + 3);
      read_operands(P);
      barrier();
      __builtin_amdgcn_s_setprio(1);
      multiply(first);
      split(xp, xr[P], inf);
      load_x(xr[P], s + 4);
#pragma unroll
      for (int i = 0; i < KU * 3 * NT * MT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one matrix instruction,
        __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);  // one vector instruction
      }
      __builtin_amdgcn_s_setprio(0);
      barrier();
    };
    using Yes = std::true_type;
    using No = std::false_type;
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    for (uint32_t sb = s0; sb < s1; sb += seg) {
      const uint32_t ns = min(seg, s1 - sb);
      stage(sb, Even{}, Yes{});
      if (ns > 1) stage(sb + 1, Odd{}, No{});
      for (uint32_t i = 2; i < ns; i += 2) {
        stage(sb + i, Even{}, No{});
        if (i + 1 < ns) stage(sb + i + 1, Odd{}, No{});
      }
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) sum[a][b] = sum[a][b] + acc[a][b];
    }
    if (!late) barrier();
  };
  run(std::false_type{});
  if (__builtin_expect(__syncthreads_or(big == INFINITY), 0)) run(std::true_type{});

  if (ks > 1) {  // as matmul_bf16_rows: write-through partial tiles, an arrival count
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(part, part_bytes);
    constexpr uint32_t kTile = TM * TN / 4;  // in f32x4
    const uint32_t base = tile * ks * kTile + wave * MT * NT * 64 + lane;
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < MT; ++b)
        st4_coherent(rp, (base + kp * kTile + (a * MT + b) * 64) * 16, __builtin_bit_cast(float4, sum[a][b]));
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) {
      uint32_t* cnt = counters + static_cast<size_t>(tile) * kCounterStride;
      const uint32_t arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = arrived == ks - 1;
      if (last) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
      for (int b = 0; b < MT; ++b) sum[a][b] = f32x4{0, 0, 0, 0};
    for (uint32_t q = 0; q < ks; ++q)  // the parts in k order
#pragma unroll
      for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b)
          sum[a][b] = sum[a][b] + __builtin_bit_cast(f32x4, ld4_coherent(rp, (base + q * kTile + (a * MT + b) * 64) * 16));
  }
  const bool wide = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
  for (int b = 0; b < MT; ++b) {
    const uint32_t row = t0 + (wm * MT + b) * 16 + c;
    if (row >= t) continue;
#pragma unroll
    for (int a = 0; a < NT; ++a) store_out4(out, row, n0 + (wn * NT + a) * 16 + 4 * g, n, wide, sum[a][b]);
  }
}

// ---- few rows, many weight rows (logits) --------------------------------------------
// At most 16 rows of x against n weight rows of k = S * 256: bound by reading w. Each of a
// workgroup's 8 waves keeps the parts of its eighth of x (S steps of 32 k) in registers
// and streams that eighth of one 16-row tile of w after the other, the next tile's loads
// in flight while this one's are used; matmul_bf16_rows reads and cuts up x again for
// every tile (twice w's bytes from L2 and ~60 vector instructions per KiB of w). The waves'
// partial tiles meet in LDS, nb tiles at a time in one of two halves (so one barrier per
// nb tiles), and are added in wave order: the bits of matmul_bf16_rows without a split
// of k. Grid: at most one workgroup per CU; workgroup i takes batches i, i + grid, ...
// Measured (k 2048): 16 x 151936 222 -> 120 us (5.2 TB/s of w), 1 x 151936 128 -> 104,
// 16 x 16384 27 -> 15, 16 x 8192 14.9 -> 10.5; a third tile in flight or nontemporal
// loads are 2-30% slower.
static constexpr int kStreamWaves = 8;
static constexpr int kStreamMaxBatch = 8;  // one tile per wave to add up

template <int S>
__global__ __launch_bounds__(64 * kStreamWaves, 2) void matmul_bf16_stream(
    const float* __restrict__ x, const uint16_t* __restrict__ w, float* __restrict__ out, uint32_t t,
    uint32_t n, uint32_t nb) {
  constexpr uint32_t k = S * 32 * kStreamWaves;
  __shared__ f32x4 part[2][kStreamMaxBatch][kStreamWaves][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const uint32_t tiles = (n + 15) / 16, batches = (tiles + nb - 1) / nb;
  bf16x8 xf[S][3];
  {
    // Rows past t repeat the last one; their outputs are not stored.
    const float* xp = x + static_cast<size_t>(min(static_cast<uint32_t>(c), t - 1)) * k + wave * S * 32 + 8 * g;
#pragma unroll
    for (int u = 0; u < S; ++u) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(xp + u * 32);
      const f32x4 b = *reinterpret_cast<const f32x4*>(xp + u * 32 + 4);
      const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
      u32x4 p[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t h, m, l;
        split_bf16x3<true>(v[2 * e], v[2 * e + 1], h, m, l);
        p[0][e] = h;
        p[1][e] = m;
        p[2][e] = l;
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) xf[u][q] = __builtin_bit_cast(bf16x8, p[q]);
    }
  }
  const int voff = (c * static_cast<int>(k) + wave * S * 32 + 8 * g) * 2;
  const auto load = [&](u16x8 (&r)[S], uint32_t tile) {  // past the end: the last tile again, unused
    const uint32_t n0 = min(tile, tiles - 1) * 16;
    const __amdgpu_buffer_rsrc_t rw =
        make_rsrc(const_cast<uint16_t*>(w + static_cast<size_t>(n0) * k), min(n - n0, 16u) * k * 2);
#pragma unroll
    for (int u = 0; u < S; ++u)
      r[u] = __builtin_bit_cast(u16x8, __builtin_amdgcn_raw_buffer_load_b128(rw, voff + u * 64, 0, 0));
  };
  const bool wide = (n & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  u16x8 wv[2][S];
  uint32_t b = blockIdx.x, j = 0, half = 0;  // this tile: the j-th of batch b
  uint32_t lb = b, lj = 0;                   // the next one to load
  const auto next = [&]() {
    if (++lj == nb) {
      lj = 0;
      lb += gridDim.x;
    }
  };
  load(wv[0], lb * nb + lj);
  next();
  while (true) {
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      load(wv[d ^ 1], lb * nb + lj);
      next();
      f32x4 acc = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < S; ++u)
#pragma unroll
        for (int q = 0; q < 3; ++q)
          acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[d][u]), xf[u][q], acc, 0, 0, 0);
      part[half][j][wave][lane] = acc;
      if (++j < nb) continue;
      lds_barrier();  // the next tile's loads stay in flight
      const uint32_t tile = b * nb + wave;
      if (static_cast<uint32_t>(wave) < nb && tile < tiles) {
        f32x4 s = part[half][wave][0][lane];
#pragma unroll
        for (int q = 1; q < kStreamWaves; ++q) s = s + part[half][wave][q][lane];
        if (static_cast<uint32_t>(c) < t) store_out4(out, c, tile * 16 + 4 * g, n, wide, s);
      }
      half ^= 1;
      j = 0;
      b += gridDim.x;
      if (b >= batches) return;  // uniform: every wave of the workgroup
    }
  }
}

}  // namespace yx
