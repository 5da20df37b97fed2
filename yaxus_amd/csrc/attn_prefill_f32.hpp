// Paged prefill / chunked-prefill attention over the f32 arena (the reference's own K/V
// precision, crates/yaxus-backend-cpu/src/lib.rs:205-214): the same arithmetic as
// `LayerPass::attend` (crates/yaxus-backend-cpu/src/lib.rs:389-427) for passes with many
// rows per sequence, with f32 accumulation and every finite f32 K/V value the reference
// accepts served.
//
// Work items are built as for the f16 prefill kernel, with kPf32Rows = 128 logical rows
// (consecutive rows of one sequence, all query heads of one KV head) per workgroup of 8
// waves, 16 columns per wave. Such a tile runs on bf16 parts (prefill_f32_parts below); one
// whose values parts don't serve, and tiles of 64 rows, run on f32 products:
//
// prefill_f32_exact (v_mfma_f32_16x16x4_f32). Keys stream from HBM into an LDS ring of
// 32-key stages (two blocks of 16; global_load_lds_dwordx4, kLead stages in flight while
// one is computed), laid out in operand order so that every LDS read is one contiguous
// 1 KiB per wave. Per block of 16 keys and wave:
//   S^T[key][col] = K . Q^T     32 x v_mfma_f32_16x16x4_f32 (dims in steps of 4)
//   online softmax per column (permlane swaps across the 4 lane groups)
//   O^T += V^T P^T              32 x v_mfma_f32_16x16x4_f32 (keys in steps of 4)
// Operand layouts (lane l, c = l % 16, g = l / 16), those of the f32 decode kernel:
//   QK step 4t + e: lane holds K[key c][16t + 4g + e] and q[col c][16t + 4g + e];
//     S^T[key 4g + i][col c] is element i of the sum of the four step-parity
//     accumulators.
//   PV step (t, m): lane holds V[key 4g + t][64(m / 4) + 4c + m % 4] (A) and
//     P[key 4g + t][col c] (B); O lands as dims 64h + 16g + 4i + (0..3) of column c
//     in elements i of accumulators 4h .. 4h + 3.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "attn_prefill.hpp"
#include "matmul_bf16.hpp"

namespace yx {

// Two shapes: 8 waves (128 logical rows), one workgroup per CU; or 4 waves (64 rows) with a
// 2-stage ring (64 KiB), two workgroups per CU, f32 products only (taken on request).
template <int W>
struct Pf32Shape {
  static constexpr int kRows = W * 16;             // logical rows per work item (one tile per wave)
  static constexpr int kRing = W == 8 ? 4 : 2;     // LDS stages (32 KiB each)
  static constexpr int kLead = kRing - 1;          // stages in flight ahead of the one computed
  static constexpr int kRowsPerWave = 32 / W;      // stage rows (1 KiB each) each wave moves
};
static constexpr int kPf32Waves = 8;
static constexpr int kPf32Rows = Pf32Shape<8>::kRows;
static constexpr int kPf32SmallRows = Pf32Shape<4>::kRows;

// A split tile's hand-off once its partials are on their way: the last chunk to arrive
// merges the tile's chunks in chunk order.
template <int W>
__device__ __forceinline__ void finish_tile(const PrefillItem& it, uint32_t kh, uint32_t G, uint32_t hq,
                                            uint32_t hkv, float* __restrict__ out, __amdgpu_buffer_rsrc_t ro,
                                            __amdgpu_buffer_rsrc_t rml, uint32_t* __restrict__ counters, uint32_t part_rows) {
  __shared__ uint32_t last_chunk;
  const uint32_t nch = it.chunk_nch >> 16;
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t* cnt = counters + (static_cast<size_t>(it.counter) * hkv + kh) * kCounterStride;
    const uint32_t arrived = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_chunk = arrived == nch - 1;
    if (last_chunk) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last_chunk) return;
  merge_tile<64 * W, Pf32Shape<W>::kRows>(it.r0, it.nrows, it.part_base, nch, kh, G, hq, hkv, out, ro, rml, part_rows);
}

// The tile on f32 products.
template <int W>
__device__ __forceinline__ void prefill_f32_exact(
    const PrefillItem& it, float4 (*ring)[32 * 64], const uint32_t* pos,
    const uint32_t* __restrict__ pages, const float* __restrict__ kc, const float* __restrict__ vc,
    const float* q, float* __restrict__ out, uint32_t hq, uint32_t hkv, uint32_t bpp_shift,
    uint32_t window, float scale_log2, float* __restrict__ part_o, float2* __restrict__ part_ml,
    uint32_t* __restrict__ counters, uint32_t part_o_bytes, uint32_t part_ml_bytes, uint32_t part_rows) {
  // A ring of stages; each is 32 rows of 1 KiB: K of block b as rows 8b + t ([t][g][key c],
  // float4 = K[c][16t + 4g .. + 3]), then V of block b as rows 16 + 8b + 2t + h
  // ([t][h][g][c], float4 = V[4g + t][64h + 4c .. + 3]).
  using S = Pf32Shape<W>;
  constexpr int kRing = S::kRing, kLead = S::kLead, kRpw = S::kRowsPerWave;
  const uint32_t kh = blockIdx.x % hkv;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int c = lane & 15, g = lane >> 4;
  const uint32_t G = hq / hkv;
  const uint32_t nlog = it.nrows * G;

  const uint32_t bpp_mask = (1u << bpp_shift) - 1u;
  const size_t head_stride = static_cast<size_t>(16u << bpp_shift) * kD;
  const uint32_t* pt = pages + it.pt_off;
  const uint32_t nblk = it.blk1 - it.blk0;
  const uint32_t nst = (nblk + 1) / 2;  // stages of two blocks

  // Wave w moves stage rows kRpw * w .. kRpw * (w + 1) - 1, all of one block's K (rows
  // 0-15) or V (rows 16-31).
  const int row0 = wave * kRpw;
  const bool my_v = row0 >= 16;
  const uint32_t my_blk = static_cast<uint32_t>((row0 & 15) >> 3);
  uint32_t src_off[kRpw];  // bytes within the block, per row
#pragma unroll
  for (int r = 0; r < kRpw; ++r) {
    const int row = (row0 & 7) + r;  // row within the block's 8 rows
    if (!my_v)
      src_off[r] = static_cast<uint32_t>((c * kD + 16 * row + 4 * g) * 4);
    else
      src_off[r] = static_cast<uint32_t>(((4 * g + (row >> 1)) * kD + 64 * (row & 1) + 4 * c) * 4);
  }
  const uint32_t ring_base = static_cast<uint32_t>(
      reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) float4*)&ring[0][0]));
  // Page of the block the wave moves for stage st, read one stage ahead.
  auto page_of = [&](uint32_t st) __attribute__((always_inline)) {
    uint32_t b = it.blk0 + st * 2 + my_blk;
    b = b < it.blk1 ? b : it.blk1 - 1;  // past the end: re-read the last block (unused)
    return uint2{pt[b >> bpp_shift], b & bpp_mask};
  };
  uint2 next_page = page_of(0);
  auto issue = [&](uint32_t st) __attribute__((always_inline)) {
    const size_t elem = (static_cast<size_t>(next_page.x) * hkv + kh) * head_stride +
                        static_cast<size_t>(next_page.y) * 16 * kD;
    next_page = page_of(st + 1);
    const char* blk = reinterpret_cast<const char*>((my_v ? vc : kc) + elem);
    const uint32_t dst = ring_base + (st & (kRing - 1)) * (32 * 1024) + static_cast<uint32_t>(row0) * 1024u;
#pragma unroll
    for (int r = 0; r < kRpw; ++r) load_to_lds16(blk + src_off[r], dst + r * 1024);
  };

  // This lane's column: its row position, key window and q (dims 16t + 4g + 0..3) as
  // given; the summed products are scaled into log2 units once, per score.
  const uint32_t lr = wave * 16 + c;
  const bool has = lr < nlog;
  const uint32_t lrc = has ? lr : 0;
  const uint32_t rr = it.r0 + lrc / G, h = kh * G + lrc % G;
  const int p0 = static_cast<int>(pos[rr]);
  const int rpos = has ? p0 : -1;
  const int rlo = (window > 0 && p0 + 1 > static_cast<int>(window)) ? p0 + 1 - static_cast<int>(window) : 0;
  float4 qv[8];
  {
    const float* qp = q + (static_cast<size_t>(rr) * hq + h) * kD + 4 * g;
#pragma unroll
    for (int t = 0; t < 8; ++t) qv[t] = *reinterpret_cast<const float4*>(qp + 16 * t);
  }
  __asm__ volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < kLead; ++j) issue(j);
#pragma unroll
  for (int t = 0; t < 8; ++t)
    if (!has) qv[t] = float4{0, 0, 0, 0};

  // The wave's key range: blocks [wa, wb) hold a key some column of the wave sees.
  int mx = rpos, lo = has ? rlo : INT32_MAX, mn = rpos, hl = rlo;
#pragma unroll
  for (int s = 1; s < 16; s <<= 1) {
    mx = max(mx, __shfl_xor(mx, s));
    lo = min(lo, __shfl_xor(lo, s));
    mn = min(mn, __shfl_xor(mn, s));
    hl = max(hl, __shfl_xor(hl, s));
  }
  const int wmax = __builtin_amdgcn_readfirstlane(mx);
  const int wlo = __builtin_amdgcn_readfirstlane(lo);
  const int tmin = __builtin_amdgcn_readfirstlane(mn);  // -1 when the tile has an empty column
  const int tlo = __builtin_amdgcn_readfirstlane(hl);
  const int first_key = static_cast<int>(it.blk0 * 16);
  const int key_end = static_cast<int>(it.blk1 * 16);

  // The running maximum starts at the lowest finite value (f32 K and q may score down to it):
  // masked scores (-inf) give P = 0 and a column's first key rescales its zero state away.
  float m = kLowest, lsum = 0.0f;
  // How far the maximum may lag. Tiles that parts handed over may have V so large that only
  // weights of at most 1 keep its sums finite.
  constexpr float kLag = W == kPf32Waves ? 0.0f : kLazyRescale;
  floatx4 acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = floatx4{0, 0, 0, 0};

  auto block = [&](auto masked, const float4* kb, const float4* vb, int key0) __attribute__((always_inline)) {
    float4 kf[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) kf[t] = kb[t * 64 + lane];
    floatx4 sp[4] = {{0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      sp[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t].x, qv[t].x, sp[0], 0, 0, 0);
      sp[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t].y, qv[t].y, sp[1], 0, 0, 0);
      sp[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t].z, qv[t].z, sp[2], 0, 0, 0);
      sp[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t].w, qv[t].w, sp[3], 0, 0, 0);
    }
    float4 vf[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) vf[r] = vb[r * 64 + lane];
    float x[4], bmax = kLowest;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float s = ((sp[0][i] + sp[1][i]) + (sp[2][i] + sp[3][i])) * scale_log2;
      if constexpr (decltype(masked)::value) {
        const int kp = key0 + 4 * g + i;
        const bool ok = (kp >= rlo) & (kp <= rpos) & (kp < key_end);
        x[i] = ok ? s : -INFINITY;
      } else {
        x[i] = s;
      }
      bmax = fmaxf(bmax, x[i]);
    }
    const float mnew = fmaxf(m, max_xor32(max_xor16(bmax)));
    if (__builtin_amdgcn_ballot_w64(mnew > m + kLag)) {  // wave-uniform
      const float corr = __builtin_amdgcn_exp2f(m - mnew);
      lsum *= corr;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] *= corr;
      m = mnew;
    }
    float pr[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pr[i] = __builtin_amdgcn_exp2f(x[i] - m);
      lsum += pr[i];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int mm = 0; mm < 8; ++mm) {
        const float4 vv = vf[2 * t + mm / 4];
        const float a = (mm % 4 == 0) ? vv.x : (mm % 4 == 1) ? vv.y : (mm % 4 == 2) ? vv.z : vv.w;
        acc[mm] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, pr[t], acc[mm], 0, 0, 0);
      }
    }
  };

  for (uint32_t st = 0; st < nst; ++st) {
    // This wave's loads of stage st are done when at most the kLead - 1 later stages'
    // are in flight; the barrier makes every wave's rows visible, and every wave has
    // finished computing stage st - 1, whose slot stage st + kLead refills.
    __asm__ volatile("s_waitcnt vmcnt(%0)" ::"n"(kRpw * (kLead - 1)) : "memory");
    __builtin_amdgcn_s_barrier();
    __asm__ volatile("" ::: "memory");
    issue(st + kLead);
    const float4* sb = &ring[st & (kRing - 1)][0];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int key0 = first_key + static_cast<int>(st * 32 + b * 16);
      if (key0 > wmax || key0 + 15 < wlo || key0 >= key_end) continue;  // wave-uniform
      const bool whole = (key0 + 15 <= tmin) & (key0 >= tlo) & (key0 + 16 <= key_end);
      if (whole)
        block(std::false_type{}, sb + b * 8 * 64, sb + (16 + b * 8) * 64, key0);
      else
        block(std::true_type{}, sb + b * 8 * 64, sb + (16 + b * 8) * 64, key0);
    }
  }
  // No load into LDS may land after the workgroup ends.
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");

  const float l = sum_xor32(sum_xor16(lsum));
  const uint32_t nch = it.chunk_nch >> 16;
  if (nch <= 1) {
    if (!has) return;
    float* o = out + (static_cast<size_t>(rr) * hq + h) * kD;
    const float inv = 1.0f / l;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4*>(o + 64 * hh + 16 * g + 4 * i) =
            float4{acc[4 * hh][i] * inv, acc[4 * hh + 1][i] * inv, acc[4 * hh + 2][i] * inv,
                   acc[4 * hh + 3][i] * inv};
    return;
  }
  // A split tile: partials and the last chunk's merge, as in the binary16 kernel.
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(part_o, part_o_bytes);
  const __amdgpu_buffer_rsrc_t rml = make_rsrc(part_ml, part_ml_bytes);
  if (has) {
    const size_t slot = (static_cast<size_t>(it.part_base) + (it.chunk_nch & 0xffffu)) * hkv + kh;
    const size_t e = slot * part_rows + lr;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        st4_coherent(ro, static_cast<uint32_t>((e * kD + 64 * hh + 16 * g + 4 * i) * 4),
                     float4{acc[4 * hh][i], acc[4 * hh + 1][i], acc[4 * hh + 2][i], acc[4 * hh + 3][i]});
    if (g == 0) st2_coherent(rml, static_cast<uint32_t>(e * 8), float2{m, l});
  }
  finish_tile<W>(it, kh, G, hq, hkv, out, ro, rml, counters, part_rows);
}

// Two f32 values as three bf16 parts each, packed as split_bf16x3 does, but cut to nearest:
// |mid| is at most 2^-8 and |lo| 2^-16 of the value (2^-9 and 2^-18 of its power of two),
// either sign, where truncation gives up to 2^-7 and 2^-15, all of the value's sign. The same
// number of instructions. |f| below 0x1.ffp127 (from there on hi is infinite). `lost` gathers in its
// lower half the bits below bf16's range, 2^-133 (of values below 2^-110 only).
__device__ __forceinline__ void split_bf16x3_nearest(float f0, float f1, uint32_t& h, uint32_t& m, uint32_t& l,
                                                     uint32_t& lost) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  h = __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{f0, f1}, bf16x2));
  const float r0 = f0 - __uint_as_float(h << 16), r1 = f1 - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(uint32_t, __builtin_convertvector(floatx2{r0, r1}, bf16x2));
  const uint32_t s0 = __float_as_uint(r0 - __uint_as_float(m << 16));
  const uint32_t s1 = __float_as_uint(r1 - __uint_as_float(m & 0xffff0000u));
  l = __builtin_amdgcn_perm(s1, s0, 0x07060302);  // at most 8 bits are left: exact
  lost |= s0 | s1;
}

// The tile of 128 logical rows on bf16 products: K, V, q and P each as three bf16 parts
// (hi, mid, lo: the 24 significand bits cut to nearest, exactly), and of the nine products
// of two such numbers the six down to 2^-18 of the largest; what is left out (mid lo, lo mid,
// lo lo) is below 2^-26 of 2^(the exponents of k and q), either sign, half a rounding of the
// product to f32. (Parts cut by truncation lose up to 2^-21 of |k q|, always towards zero:
// on values just below a bf16 step, out of 1000 keys, 2.4e-5 off 64 bits where f32 products
// are 2.7e-6 and these 7e-7 off.) bf16 has f32's range, so every finite value is served, and
// f32 accumulation as before. Six v_mfma_f32_16x16x32_bf16 take 96 cycles where eight
// v_mfma_f32_16x16x4_f32 take 256.
// Returns false, with nothing written, where parts would not do: an infinity (0 * inf in a
// product of parts) or a NaN (a masked key's reaches the rows of its 32 keys here, of 16 in
// f32 products); K, q or the scale so large that parts below bf16's range matter to a
// score (at most 2^-133 * 2^70 * 2^7 dims * 2^20, 2^-36); a value of V with bits below that
// range, 2^-133 (one of 2^-110 keeps all 24; lost, an output made of such values alone would
// be as far off: 5.7e-4 at 2^-124); V of 2^100 and more (weights of up to 2^kLazyRescale times
// many such values might overflow where weights of at most 1 do not). The caller then runs the f32 products. (A weight's bits
// below 2^-133 are dropped: the exponential itself gives 0 below 2^-126.)
//
// Stages of 32 keys: each thread reads 8 dims of one key of K and of V (f32) into
// registers, one stage ahead, cuts them into parts and stores those to one of two LDS
// slots, as three planes each laid out like the binary16 kernel's stages: K [p][g][key] (16
// bytes: dims 32 p + 8 g ..), V [key][128] with 32-byte chunks XOR-swizzled by the key, read
// with the transposing LDS reads. One barrier per stage. The bounds are the matrix pipe (96
// instructions per wave and stage, 3072 cycles for a SIMD's two waves) and the LDS reads (48
// KiB per wave, 3072 cycles a CU); the conversions and the softmax, ~280 vector instructions
// a wave and stage, run beside them only in part: a stage takes 2.9 us, the matrix pipe is
// busy 42% of it. Two halves of the workgroup half a stage apart (three slots), V's planes
// in operand order (no transposing reads) and four dim groups' chains side by side each
// came out within 3% of this. Per layer with its write_rows, f32 products -> parts: 4 x 256
// rows after 100-4000 keys, 16/4 heads, 143 -> 95 us (45 -> 68 TFLOP/s); 512 after 3000, 24/4, 245
// -> 165; 16 x 256 after 8-2040 200 -> 133; 2 x 148, 24/4, 130 -> 88. Relative error
// against 64-bit results over these and windows, fresh passes and 20000 keys: 2.3e-7 to
// 3.7e-7, f32 products 2.5e-7 to 1.0e-6.
__device__ __forceinline__ bool prefill_f32_parts(
    const PrefillItem& it, char* lds, const uint32_t* pos,
    const uint32_t* __restrict__ pages, const float* __restrict__ kc, const float* __restrict__ vc,
    const float* q, float* __restrict__ out, uint32_t hq, uint32_t hkv, uint32_t bpp_shift,
    uint32_t window, float scale_log2, float* __restrict__ part_o, float2* __restrict__ part_ml,
    uint32_t* __restrict__ counters, uint32_t part_o_bytes, uint32_t part_ml_bytes, uint32_t part_rows) {
  constexpr int kSlot = 2 * 3 * 8192;  // bytes of a stage: K then V, three planes of two 4 KiB blocks
  constexpr int kV = 3 * 8192;
  const uint32_t kh = blockIdx.x % hkv;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const uint32_t G = hq / hkv;
  const uint32_t nlog = it.nrows * G;
  const uint32_t bpp_mask = (1u << bpp_shift) - 1u;
  const size_t head_stride = static_cast<size_t>(16u << bpp_shift) * kD;
  const uint32_t* pt = pages + it.pt_off;
  const uint32_t nst = (it.blk1 - it.blk0 + 1) / 2;

  // This thread's piece of a stage: K of block wave / 4, key c, dims 32 (wave % 4) + 8 g ..;
  // V of key 4 wave + g, dims 8 c .. (both in block wave / 4).
  const uint32_t my_blk = static_cast<uint32_t>(wave >> 2);
  const uint32_t k_src = static_cast<uint32_t>(c * kD + 32 * (wave & 3) + 8 * g);
  const uint32_t v_key = static_cast<uint32_t>(4 * (wave & 3) + g);
  const uint32_t v_src = v_key * kD + 8 * c;
  char* const k_dst = lds + my_blk * 4096 + (wave & 3) * 1024 + lane * 16;
  char* const v_dst = lds + kV + my_blk * 4096 + v_key * 256 + ((((c >> 1) ^ (v_key & 7)) << 1) + (c & 1)) * 16;
  auto page_of = [&](uint32_t st) __attribute__((always_inline)) {
    uint32_t b = it.blk0 + st * 2 + my_blk;
    b = b < it.blk1 ? b : it.blk1 - 1;  // past the end: the last block again (masked)
    return uint2{pt[b >> bpp_shift], b & bpp_mask};
  };
  if (fabsf(scale_log2) > 0x1p20f) return false;
  float4 kr[2], vr[2];
  auto load = [&](const uint2& page) __attribute__((always_inline)) {
    const size_t elem = (static_cast<size_t>(page.x) * hkv + kh) * head_stride + static_cast<size_t>(page.y) * 16 * kD;
    const float* ks = kc + elem + k_src;
    const float* vs = vc + elem + v_src;
    kr[0] = *reinterpret_cast<const float4*>(ks);
    kr[1] = *reinterpret_cast<const float4*>(ks + 4);
    vr[0] = *reinterpret_cast<const float4*>(vs);
    vr[1] = *reinterpret_cast<const float4*>(vs + 4);
  };
  float big = 0.0f, vbig = 0.0f;  // largest |K|, |q| and |V| met by this thread, or NaN
  uint32_t vlost = 0, unused = 0;
  auto split8 = [&](const float4& a, const float4& b, u32x4 (&p)[3], float& top, uint32_t& lost) __attribute__((always_inline)) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      __asm__("v_maximum3_f32 %0, %0, |%1|, |%2|" : "+v"(top) : "v"(v[2 * e]), "v"(v[2 * e + 1]));
      uint32_t h, m, l;
      split_bf16x3_nearest(v[2 * e], v[2 * e + 1], h, m, l, lost);
      p[0][e] = h;
      p[1][e] = m;
      p[2][e] = l;
    }
  };
  auto store = [&](uint32_t slot) __attribute__((always_inline)) {
    u32x4 p[3];
    split8(kr[0], kr[1], p, big, unused);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(k_dst + slot * kSlot + i * 8192) = p[i];
    split8(vr[0], vr[1], p, vbig, vlost);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(v_dst + slot * kSlot + i * 8192) = p[i];
  };

  // This lane's column, as in the f32 form.
  const uint32_t lr = wave * 16 + c;
  const bool has = lr < nlog;
  const uint32_t lrc = has ? lr : 0;
  const uint32_t rr = it.r0 + lrc / G, h = kh * G + lrc % G;
  const int p0 = static_cast<int>(pos[rr]);
  const int rpos = has ? p0 : -1;
  const int rlo = (window > 0 && p0 + 1 > static_cast<int>(window)) ? p0 + 1 - static_cast<int>(window) : 0;
  load(page_of(0));
  uint2 next_page = page_of(nst > 1 ? 1 : 0);
  bf16x8 qf[3][4];
  {
    const float* qp = q + (static_cast<size_t>(rr) * hq + h) * kD + 8 * g;
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      float4 a = *reinterpret_cast<const float4*>(qp + 32 * pp), b = *reinterpret_cast<const float4*>(qp + 32 * pp + 4);
      if (!has) a = b = float4{0, 0, 0, 0};
      u32x4 p[3];
      split8(a, b, p, big, unused);
#pragma unroll
      for (int i = 0; i < 3; ++i) qf[i][pp] = __builtin_bit_cast(bf16x8, p[i]);
    }
  }
  int mx = rpos, lo = has ? rlo : INT32_MAX, mn = rpos, hl = rlo;
#pragma unroll
  for (int s = 1; s < 16; s <<= 1) {
    mx = max(mx, __shfl_xor(mx, s));
    lo = min(lo, __shfl_xor(lo, s));
    mn = min(mn, __shfl_xor(mn, s));
    hl = max(hl, __shfl_xor(hl, s));
  }
  const int wmax = __builtin_amdgcn_readfirstlane(mx);
  const int wlo = __builtin_amdgcn_readfirstlane(lo);
  const int tmin = __builtin_amdgcn_readfirstlane(mn);  // -1 when the tile has an empty column
  const int tlo = __builtin_amdgcn_readfirstlane(hl);
  const int first_key = static_cast<int>(it.blk0 * 16);
  const int key_end = static_cast<int>(it.blk1 * 16);

  float m = kLowest, lsum = 0.0f;
  floatx4 acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = floatx4{0, 0, 0, 0};
  // Transposing-read offset of dim group j within a block of V (see the binary16 kernel).
  uint32_t vtr_off[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t k = 4u * g + (c >> 2);
    vtr_off[j] = k * 256u + 32u * (static_cast<uint32_t>(j) ^ (k & 7u)) + 8u * (c & 3);
  }
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));
  // The products kept, largest last: (part of K or V, part of q or P).
  constexpr int kPa[6] = {2, 1, 0, 1, 0, 0}, kPb[6] = {0, 1, 2, 0, 1, 0};

  auto compute = [&](auto masked, uint32_t slot, int key0) __attribute__((always_inline)) {
    const half8* kb = reinterpret_cast<const half8*>(lds + slot * kSlot);
    // The products of the hi parts and the others' small ones in sums of their own: a small
    // product added to a full score would round it once more (4.5e-7 off 64 bits with one
    // sum for 512 rows after 3000 keys, 2.8e-7 with two; f32 products 4.2e-7).
    floatx4 sc[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, sm[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
    for (int pp = 0; pp < 4; ++pp) {
      bf16x8 kf[2][3];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < 3; ++i)
          kf[b][i] = __builtin_bit_cast(bf16x8, kb[i * 512 + b * 256 + pp * 64 + lane]);
#pragma unroll
      for (int t = 0; t < 6; ++t)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          floatx4& to = t < 5 ? sm[b] : sc[b];
          to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[b][kPa[t]], qf[kPb[t]][pp], to, 0, 0, 0);
        }
    }
    float x[8], bmax = kLowest;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float s = (sc[e >> 2][e & 3] + sm[e >> 2][e & 3]) * scale_log2;
      if constexpr (decltype(masked)::value) {
        const int kp = key0 + (e >> 2) * 16 + 4 * g + (e & 3);
        const bool ok = (kp >= rlo) & (kp <= rpos) & (kp < key_end);
        x[e] = ok ? s : -INFINITY;
      } else {
        x[e] = s;
      }
      bmax = fmaxf(bmax, x[e]);
    }
    const float mnew = fmaxf(m, max_xor32(max_xor16(bmax)));
    if (__builtin_amdgcn_ballot_w64(mnew > m + kLazyRescale)) {  // wave-uniform
      const float corr = __builtin_amdgcn_exp2f(m - mnew);
      lsum *= corr;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] *= corr;
      m = mnew;
    }
    u32x4 pw[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = __builtin_amdgcn_exp2f(x[2 * e] - m), b = __builtin_amdgcn_exp2f(x[2 * e + 1] - m);
      lsum += a + b;
      uint32_t hh, mm, ll;
      split_bf16x3_nearest(a, b, hh, mm, ll, unused);
      pw[0][e] = hh;
      pw[1][e] = mm;
      pw[2][e] = ll;
    }
    bf16x8 pf[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) pf[i] = __builtin_bit_cast(bf16x8, pw[i]);
    const uint32_t vb = lds_base + slot * kSlot + kV;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      bf16x8 vf[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const lds_half4* src = reinterpret_cast<const lds_half4*>(
            reinterpret_cast<const __attribute__((address_space(3))) char*>(static_cast<uintptr_t>(vb + i * 8192u)) + vtr_off[j]);
        const half4 lo4 = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16(const_cast<lds_half4*>(src)));
        const half4 hi4 = __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16(const_cast<lds_half4*>(src + 512)));
        vf[i] = __builtin_bit_cast(bf16x8, half8{lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]});
      }
      floatx4 o = {0, 0, 0, 0};  // the pair's own sum: one rounding of the running one per pair
#pragma unroll
      for (int t = 0; t < 6; ++t) o = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[kPa[t]], pf[kPb[t]], o, 0, 0, 0);
      acc[j] = floatx4{acc[j][0] + o[0], acc[j][1] + o[1], acc[j][2] + o[2], acc[j][3] + o[3]};
    }
  };

  store(0);
  if (nst > 1) {
    load(next_page);
    next_page = page_of(nst > 2 ? 2 : 1);
  }
  lds_barrier();
  for (uint32_t st = 0; st < nst; ++st) {
    // Slot st + 1 was last read before the barrier that ended stage st - 1.
    if (st + 1 < nst) {
      store((st + 1) & 1);
      if (st + 2 < nst) {
        load(next_page);
        next_page = page_of(st + 3 < nst ? st + 3 : st + 2);
      }
    }
    const int key0 = first_key + static_cast<int>(st * 32);
    if (!(key0 > wmax || key0 + 31 < wlo)) {  // wave-uniform
      const bool whole = (key0 + 31 <= tmin) & (key0 >= tlo) & (key0 + 32 <= key_end);
      if (whole)
        compute(std::false_type{}, st & 1, key0);
      else
        compute(std::true_type{}, st & 1, key0);
    }
    lds_barrier();
  }
  // Values that parts don't serve: over to f32 products.
  if (__syncthreads_or(!(big < 0x1p70f) || !(vbig < 0x1p100f) || (vlost & 0xffffu) != 0)) {
    __syncthreads();
    return false;
  }

  const float l = sum_xor32(sum_xor16(lsum));
  if ((it.chunk_nch >> 16) <= 1) {
    if (!has) return true;
    float* o = out + (static_cast<size_t>(rr) * hq + h) * kD + 4 * g;
    const float inv = 1.0f / l;
#pragma unroll
    for (int j = 0; j < 8; ++j)  // acc[j][i] is dim 16 j + 4 g + i of the column
      *reinterpret_cast<float4*>(o + 16 * j) = float4{acc[j][0] * inv, acc[j][1] * inv, acc[j][2] * inv, acc[j][3] * inv};
    return true;
  }
  const __amdgpu_buffer_rsrc_t ro = make_rsrc(part_o, part_o_bytes);
  const __amdgpu_buffer_rsrc_t rml = make_rsrc(part_ml, part_ml_bytes);
  if (has) {
    const size_t slot = (static_cast<size_t>(it.part_base) + (it.chunk_nch & 0xffffu)) * hkv + kh;
    const size_t e = slot * part_rows + lr;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      st4_coherent(ro, static_cast<uint32_t>((e * kD + 16 * j + 4 * g) * 4),
                   float4{acc[j][0], acc[j][1], acc[j][2], acc[j][3]});
    if (g == 0) st2_coherent(rml, static_cast<uint32_t>(e * 8), float2{m, l});
  }
  finish_tile<kPf32Waves>(it, kh, G, hq, hkv, out, ro, rml, counters, part_rows);
  return true;
}

template <int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 2))) void paged_attn_prefill_f32(
    const PrefillItem* __restrict__ items, const uint32_t* pos,
    const uint32_t* __restrict__ pages, const float* __restrict__ kc, const float* __restrict__ vc,
    const float* q, float* __restrict__ out, uint32_t hq, uint32_t hkv, uint32_t bpp_shift,
    uint32_t window, float scale_log2, float* __restrict__ part_o, float2* __restrict__ part_ml,
    uint32_t* __restrict__ counters, uint32_t part_o_bytes, uint32_t part_ml_bytes, uint32_t part_rows) {
  __shared__ float4 ring[Pf32Shape<W>::kRing][32 * 64];
  const PrefillItem it = items[blockIdx.x / hkv];
  if constexpr (W == kPf32Waves) {
    static_assert(sizeof(ring) >= 2 * 2 * 3 * 8192, "two stages of parts");
    if (prefill_f32_parts(it, reinterpret_cast<char*>(&ring[0][0]), pos, pages, kc, vc, q, out, hq, hkv, bpp_shift,
                          window, scale_log2, part_o, part_ml, counters, part_o_bytes, part_ml_bytes, part_rows))
      return;
  }
  prefill_f32_exact<W>(it, ring, pos, pages, kc, vc, q, out, hq, hkv, bpp_shift, window, scale_log2, part_o, part_ml,
                       counters, part_o_bytes, part_ml_bytes, part_rows);
}

}  // namespace yx
