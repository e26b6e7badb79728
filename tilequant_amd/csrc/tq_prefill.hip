// tq_prefill.hip -- mixed INT8/16-bit tile GEMM for more than 64 tokens on
// token-blocked activation codes (tq_gemm_mixed_blocked).
//
// The whole-list kernel forms the sums of the row-major prefill kernels of
// tq_gemm.hip, bit for bit: one fp32 accumulator per output, the INT8 tiles of
// a row tile by column (exact INT32 tile product, then one FMA by
// sx[c] * sw[t]), then its 16-bit tiles by position (the reference's loop,
// gemm_rows_splitk_64x64.py:125-153).  The split kernel (few tokens, see
// split_waves) deals a row tile's tiles to 4 or 8 waves and adds their partial
// sums in wave order, as the decode kernels do.
#include <algorithm>
#include <vector>

#include "tq_common.h"

namespace tq {

typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

struct PrefillArgs {
  const int8_t* xq;        // token-blocked codes, nb 16-row blocks per column tile
  const float* sx;
  const int8_t* w8;
  const float* sw8;
  const int32_t* ids8;
  const int32_t* rp8;
  const uint16_t* xf;
  int64_t ldx;
  const uint16_t* w16;     // nullptr: no 16-bit tiles
  const int32_t* ids16;
  const int32_t* rp16;
  uint16_t* out;
  int64_t ldo;
  const uint16_t* bias;
  const int32_t* rows;     // row tile of each of n_slots slots (out of range: none), nullptr: identity
  int32_t* dump;           // DUMP instantiation: int32 [T8, dump_n, 64]
  int dump_r0, dump_n;
  int n, m, n_tr, n_tc, nb, n_slots, n_units;
  int out_bf16, layout, ovec;
};

// 32x32x16 MFMA on 16-bit operands (8 per lane: row / column lane % 32, k
// 8 (lane / 32) .. + 7).  Two of them over consecutive 16-deep slices give
// bitwise the 16x16x32 result (checked on MI355X, bf16 and fp16).
template <class XT>
__device__ inline v16f mfma32(v4i av, v4i bv, v16f c);
template <>
__device__ inline v16f mfma32<Bf16>(v4i av, v4i bv, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, av), __builtin_bit_cast(v8bf, bv), c, 0, 0, 0);
}
template <>
__device__ inline v16f mfma32<Fp16>(v4i av, v4i bv, v16f c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, av), __builtin_bit_cast(v8h, bv), c, 0, 0, 0);
}

// One INT8 tile's 32 FB features x 32 NT tokens: exact INT32 products (two chained
// 32x32x32 MFMAs per 32 x 32 block), then acc = fma((float)d, sc, acc) per
// element.  The MFMAs of block b + 1 are issued before the conversions of block
// b, so a wave alone on its SIMD does not sit out the MFMA latency, and each
// conversion goes out between two FMAs (on gfx950 a v_cvt of one wave and a
// v_fma of another issue together; measured 2.4 cycles per instruction for the
// alternating stream against 4.3 for either kind alone).  `ready(t)` waits for
// token block t's operands; `seen(f, t, d)` is the test dump.
template <int FB, int NT, class Ready, class Seen>
__device__ __attribute__((always_inline)) inline void tile_mac(v16f (&acc)[FB][NT], const v4i (&w)[FB][2],
                                                               v4i (&x)[NT][2], float sc, Ready&& ready, Seen&& seen) {
  v16i d[2];
#pragma unroll
  for (int b = 0; b <= FB * NT; ++b) {
    if (b < FB * NT) {
      const int f = b % FB, t = b / FB;
      if (f == 0) ready(t);
      const v16i z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
      d[b & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[f][0], x[t][0], z, 0, 0, 0);
      d[b & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[f][1], x[t][1], d[b & 1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (b > 0) {
      const int f = (b - 1) % FB, t = (b - 1) / FB;
      seen(f, t, d[(b - 1) & 1]);
      float c[16];
#pragma unroll
      for (int v = 0; v <= 16; ++v) {
        if (v < 16) {
          c[v] = (float)d[(b - 1) & 1][v];
          __builtin_amdgcn_sched_barrier(0);
        }
        if (v > 0) {
          acc[f][t][v - 1] = fmaf(c[v - 1], sc, acc[f][t][v - 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
}

// DUMP: token rows of d's 32 x 32 block (features f0 .., tokens row0 ..) into the test buffer.
__device__ inline void dump_block(const PrefillArgs& a, int p, int row0, int f0, int lane, const v16i& d) {
  const int rr = row0 + (lane & 31) - a.dump_r0;
  if ((unsigned)rr < (unsigned)a.dump_n)
#pragma unroll
    for (int v = 0; v < 16; ++v)
      a.dump[((int64_t)p * a.dump_n + rr) * 64 + f0 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)] = d[v];
}

// `rows` staged output rows of row tile r (128 bytes each, 16-byte chunk c of
// row R at slot c ^ (R % 8)) from token n0 on, by `threads` threads: CHUNKS
// chunks of each row from chunk ch0 on.
template <int CHUNKS = 8>
__device__ inline void store_rows(const PrefillArgs& a, const int8_t* staged, int r, int n0, int rows, int tid,
                                  int threads, int ch0 = 0) {
#pragma unroll 4
  for (int q = tid; q < rows * CHUNKS; q += threads) {
    const int rr = q / CHUNKS, ch = ch0 + q % CHUNKS, row = n0 + rr, col = r * 64 + ch * 8;
    const v4i val = *reinterpret_cast<const v4i*>(staged + rr * 128 + ((ch ^ (rr & 7)) * 16));
    if (row >= a.n || col >= a.m) continue;
    uint16_t* dst = a.out + (int64_t)row * a.ldo + col;
    if (a.ovec && col + 8 <= a.m) {
      *reinterpret_cast<v4i*>(dst) = val;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < a.m) dst[e] = (uint16_t)((uint32_t)val[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// Workgroup = 4 row tiles x 32 TB tokens; wave w owns the 64 features of slot
// 4 u + w and all of the tokens (2 x TB accumulator blocks of 32 x 32).  The
// weights are the MFMA's A operand and the tokens its B operand, so a lane
// holds four consecutive features of one token.
//
// INT8 phase, one step per column tile: the token slice (32 TB x 64 codes, one
// contiguous 1 KiB per 16 rows) is shared by the four waves through an 8-stage
// LDS ring; a wave's weight tile is its own and goes straight to registers,
// two steps ahead.  Two steps per barrier.  A wave whose row tile is 16-bit at
// a column skips the step's arithmetic.
//
// What bounds it: at thousands of tokens the VALU and matrix issue of the exact
// per-tile epilogue at the clock the power limit leaves (Gate/Up of
// Llama-3.2-3B at 8192 tokens 620 us; with all-zero operands, the same
// instructions, 470), below that each wave's serial walk of its list.  The
// 32x32 MFMAs hold the epilogue's registers in half as many instructions as
// 16x16 ones (register-only loop, two waves per SIMD: 53% of the INT8 peak
// against 41%), and token-blocked slices cross the LDS DMA path at twice the
// rate of row-major ones (probe of the loads alone: 25 against 12 TB/s).  Per
// Llama-3.2-3B layer (keep05, quantization included) against the row-major
// kernel: 2048 tokens 558 -> 424 us, 8192 tokens 1537 -> 1383 us; Qwen2.5-7B
// (clustered keep10, fp16) at 777 tokens 826 -> 488 us.
//
// NT <= TB: the 32-token blocks that a wave multiplies, fewer in a short last
// workgroup (the loads stay, so the waits count the same).
// 16-bit phase: see there.  Outputs are staged in the wave's quarter of the
// ring and leave as 128-byte rows.
constexpr int kPbCols = 304;     // column tiles (k <= 19456)
constexpr int kPbStages = 8;
constexpr int kPbAhead = 3;      // iterations (of two steps) a slice is fetched ahead

struct SlotTiles {           // one wave's row tile
  int r, lo8, hi8, lo16, hi16;
  bool active;
};

template <int TB>
struct BlockedLds {
  int8_t ring[kPbStages * TB * 2048];
  int pos[4][kPbCols];       // per wave: tile position by column, -1 none
  float sw[4][kPbCols];
  int cols16[kPbCols];       // SHARED16: the columns with a 16-bit tile
  int n_cols16;
};

template <class XT, int TB, int NT, bool SHARED16, bool DUMP>
__device__ __attribute__((always_inline)) inline void prefill_blocked_body(const PrefillArgs& a, BlockedLds<TB>& lds,
                                                                           const SlotTiles& tiles, int n0, bool any8,
                                                                           int lane, int wave) {
  constexpr int XB = TB * 2048;            // bytes of a stage
  constexpr int XL = TB / 2;               // stage blocks (1 KiB) fetched by each wave
  constexpr int kRegion = kPbStages * XB / 4;
  constexpr int kHalf = kRegion / 2;       // 16-bit phase: 16 TB tokens x 64 columns
  int8_t* ring = lds.ring;
  const int n_tc = a.n_tc;
  const int r = tiles.r, lo8 = tiles.lo8, hi8 = tiles.hi8, lo16 = tiles.lo16, hi16 = tiles.hi16;
  const int last8 = a.rp8[a.n_tr] - 1;     // any8: at least 0

  v16f acc[2][NT];
#pragma unroll
  for (int f = 0; f < 2; ++f)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[f][t][v] = 0.f;

  if (any8) {
    // ---- the wave's tile list by column -------------------------------------
    // (the column and block offsets are kept wave-uniform: scalar arithmetic)
    int xblk[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) xblk[i] = __builtin_amdgcn_readfirstlane(min(n0 / 16 + wave * XL + i, a.nb - 1)) * 1024;
    const int64_t xcol = (int64_t)a.nb * 1024;
    auto fetch_x = [&](int s) {            // the wave's share of column s's slice
      const int8_t* col = a.xq + (int64_t)__builtin_amdgcn_readfirstlane(min(s, n_tc - 1)) * xcol;
      int8_t* stage = ring + (s % kPbStages) * XB;
#pragma unroll
      for (int i = 0; i < XL; ++i) dma16(col + xblk[i] + lane * 16, stage + (wave * XL + i) * 1024);
    };
    int* pw = lds.pos[wave];
    float* sw = lds.sw[wave];
    for (int c = lane; c < n_tc; c += 64) pw[c] = -1;
    for (int p = lo8 + lane; p < hi8; p += 64) {
      const int c = col_of(a.ids8[p], r * n_tc, n_tc);
      pw[c] = p;
      sw[c] = a.sw8[p];
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int s = 0; s < 2 * kPbAhead; ++s) fetch_x(s);
    __builtin_amdgcn_sched_barrier(0);

    // weight operand (feature block f, K half h) of this lane inside a tile
    int woff[2];
#pragma unroll
    for (int f = 0; f < 2; ++f)
      woff[f] = a.layout == TQ_LAYOUT_MFMA
                    ? (2 * f + ((lane >> 4) & 1)) * 1024 + (lane >> 5) * 256 + (lane & 15) * 16
                    : (f * 32 + (lane & 31)) * 64 + (lane >> 5) * 16;
    const int wh = a.layout == TQ_LAYOUT_MFMA ? 512 : 32;
    v4i w[2][2][2];                        // [step parity][f][h]
    auto load_w = [&](v4i (&d)[2][2], int p) {
      const int8_t* t = a.w8 + (int64_t)min(max(p, 0), last8) * 4096;
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int h = 0; h < 2; ++h) d[f][h] = *reinterpret_cast<const v4i*>(t + woff[f] + h * wh);
    };
    const int p0 = pw[0], p1 = pw[min(1, n_tc - 1)];
    load_w(w[0], __builtin_amdgcn_readfirstlane(p0));
    __builtin_amdgcn_sched_barrier(0);
    load_w(w[1], __builtin_amdgcn_readfirstlane(p1));
    __builtin_amdgcn_sched_barrier(0);
    // The wave's share of slices 0 and 1 lands before the first barrier, past
    // which the other waves read it: only the later slices' fetches and both
    // steps' weights (2 x 4 loads) may stay in flight.
    if constexpr (DUMP) wait_vmcnt<0>();
    else wait_vmcnt<(2 * kPbAhead - 2) * XL + 8>();

    const uint32_t x_rd = lds_addr(ring) + ((lane >> 4) & 1) * 1024 + (lane >> 5) * 256 + (lane & 15) * 16;
    // window of 64 columns: lane i holds column c0 + i's scale and the
    // position of column c0 + i + 2's tile
    float wsc = 0.f;
    int wpn = 0;
    uint64_t mask = 0;
    auto step = [&](int s, v4i (&ws)[2][2]) {
      const int i = s & 63;
      // The weights were loaded two steps ago; since then one step's weights
      // (4 loads) and one iteration's slices (2 XL) were issued.  Waiting here,
      // outside the branch, keeps the count exact (inside it the compiler
      // waits for everything in flight).
      if constexpr (DUMP) wait_vmcnt<0>();
      else wait_vmcnt<2 * XL + 4>();
      if ((mask >> i) & 1) {
        const float sc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wsc), i));
        const uint32_t rd = x_rd + (s % kPbStages) * XB;
        v4i x[NT][2];
#pragma unroll
        for (int t = 0; t < NT; ++t)
          asm volatile(
              "ds_read_b128 %0, %2 offset:%3\n\t"
              "ds_read_b128 %1, %2 offset:%4"
              : "=&v"(x[t][0]), "=&v"(x[t][1])
              : "v"(rd), "n"(2048 * t), "n"(2048 * t + 512)
              : "memory");
        const int p = DUMP ? pw[s] : 0;
        tile_mac<2, NT>(
            acc, ws, x, sc,
            [&](int t) {
              // LDS reads return in order: token block t has landed when at
              // most 2 (NT - 1 - t) reads are outstanding
              if (t == NT - 1 || DUMP) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(x[t][0]), "+v"(x[t][1])::"memory");
              else if (t == NT - 2) asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(x[t][0]), "+v"(x[t][1])::"memory");
              else if (t == NT - 3) asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(x[t][0]), "+v"(x[t][1])::"memory");
              else asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(x[t][0]), "+v"(x[t][1])::"memory");
            },
            [&](int f, int t, const v16i& d) {
              if constexpr (DUMP) dump_block(a, p, n0 + 32 * t, 32 * f, lane, d);
            });
      }
      __builtin_amdgcn_sched_barrier(0);
      load_w(ws, __builtin_amdgcn_readlane(wpn, i));
      __builtin_amdgcn_sched_barrier(0);
    };
    const int iters = (n_tc + 1) / 2;
    for (int k = 0; k < iters; ++k) {
      const int s = 2 * k;
      // The wave's share of slices s and s + 1 has landed before the barrier
      // (vector memory operations complete in order): for k = 0 by the wait
      // above, for the prologue's other slices by the waits of the steps of
      // k = 0, and from k = kPbAhead on, fetched kPbAhead iterations ago, by
      // this one, as the two iterations since issued 2 (2 XL + 8) operations
      // after them.  Past the barrier every wave is done with the stages of
      // the previous iteration, which the fetch below reuses.
      if constexpr (DUMP) wait_vmcnt<0>();
      else wait_vmcnt<2 * (2 * XL + 8)>();
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      fetch_x(s + 2 * kPbAhead);
      fetch_x(s + 2 * kPbAhead + 1);
      __builtin_amdgcn_sched_barrier(0);
      if ((s & 63) == 0) {
        const int c = min(s + lane, n_tc - 1);
        const bool have = s + lane < n_tc && pw[c] >= 0;
        mask = __ballot(have);
        wsc = have ? a.sx[c] * sw[c] : 0.f;
        wpn = pw[min(s + lane + 2, n_tc - 1)];
      }
      step(s, w[0]);
      step(s + 1, w[1]);   // past the last column: no bit in the mask (the window's lanes stop at n_tc)
    }
    wait_vmcnt<0>();
  }
  __syncthreads();   // every wave is done with the ring

  int8_t* region = ring + wave * kRegion;
  if (a.w16 != nullptr) {
    // Activation rows: 128 bytes of a column tile, each DMA load 8 whole rows;
    // 16-byte chunk c of row R sits at slot c ^ (R % 8), so the operand reads
    // of 16 rows spread over the banks.
    const int xch = ((lane & 7) ^ (lane >> 3)) * 8;
    auto fetch_rows = [&](int c, int row0, int8_t* dst, auto loads) {
#pragma unroll
      for (int i = 0; i < decltype(loads)::value; ++i) {
        const int64_t row = min(n0 + row0 + 8 * i + (lane >> 3), a.n - 1);
        dma16(a.xf + row * a.ldx + c * 64 + xch, dst + i * 1024);
      }
    };
    int woff[2];
#pragma unroll
    for (int f = 0; f < 2; ++f)
      woff[f] = a.layout == TQ_LAYOUT_MFMA
                    ? (2 * f + ((lane >> 4) & 1)) * 1024 + (lane >> 5) * 128 + (lane & 15) * 8
                    : (f * 32 + (lane & 31)) * 64 + (lane >> 5) * 8;
    v4i w[2][2][4];                        // [parity][f][16-deep slice]
    auto load_w16 = [&](v4i (&d)[2][4], int q) {
      const uint16_t* t = a.w16 + (int64_t)q * 4096;
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
          d[f][kc] = *reinterpret_cast<const v4i*>(
              t + woff[f] + (a.layout == TQ_LAYOUT_MFMA ? (kc >> 1) * 512 + (kc & 1) * 256 : kc * 16));
    };
    uint32_t xrd[4];                       // chunk 2 kc + lane / 32 of row lane % 32, swizzled
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) xrd[kc] = (lane & 31) * 128 + (((2 * kc + (lane >> 5)) ^ (lane & 7)) * 16);
    auto block_mfma = [&](const v4i (&ws)[2][4], uint32_t base, auto t_tag) {   // token block t's 8 MFMAs
      constexpr int t = decltype(t_tag)::value;
      v4i x[4];
      asm volatile(
          "ds_read_b128 %0, %4\n\t"
          "ds_read_b128 %1, %5\n\t"
          "ds_read_b128 %2, %6\n\t"
          "ds_read_b128 %3, %7\n\t"
          "s_waitcnt lgkmcnt(0)"
          : "=&v"(x[0]), "=&v"(x[1]), "=&v"(x[2]), "=&v"(x[3])
          : "v"(base + xrd[0]), "v"(base + xrd[1]), "v"(base + xrd[2]), "v"(base + xrd[3])
          : "memory");
#pragma unroll
      for (int kc = 0; kc < 4; ++kc)
#pragma unroll
        for (int f = 0; f < 2; ++f) acc[f][t] = mfma32<XT>(ws[f][kc], x[kc], acc[f][t]);
    };
    if constexpr (SHARED16) {
      // A row tile mostly in 16 bits: the four waves walk the columns where
      // any of them has a 16-bit tile together, sharing each column's slice
      // (32 TB rows) through a 4-stage ring, two columns ahead.
      constexpr int SB = TB * 4096, XQ = TB;   // stage bytes; loads per wave and stage
      int* pw = lds.pos[wave];
      for (int c = lane; c < n_tc; c += 64) pw[c] = -1;
      for (int q = lo16 + lane; q < hi16; q += 64) pw[col_of(a.ids16[q], r * n_tc, n_tc)] = q;
      __syncthreads();
      if (wave == 0) {                     // the columns, in order
        int n = 0;
        for (int c0 = 0; c0 < n_tc; c0 += 64) {
          const int c = min(c0 + lane, n_tc - 1);
          const bool any = c0 + lane < n_tc && max(max(lds.pos[0][c], lds.pos[1][c]), max(lds.pos[2][c], lds.pos[3][c])) >= 0;
          const uint64_t b = __ballot(any);
          if (any) lds.cols16[n + __popcll(b & ((1ull << lane) - 1))] = c;
          n += __popcll(b);
        }
        if (lane == 0) lds.n_cols16 = n;
      }
      __syncthreads();
      const int nc = lds.n_cols16;
      auto entry = [&](int e) { return lds.cols16[min(e, nc - 1)]; };   // column of a list entry
      const int last16 = a.rp16[a.n_tr] - 1;
      auto fetch_stage = [&](int e, int c) {
        fetch_rows(c, wave * 8 * TB, ring + (e & 3) * SB + wave * XQ * 1024, std::integral_constant<int, XQ>{});
      };
      const int c1 = entry(1);
      const int c0 = entry(0);
      const int q0 = pw[c0], q1 = pw[c1];
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      fetch_stage(0, __builtin_amdgcn_readfirstlane(c0));
      load_w16(w[0], min(max(__builtin_amdgcn_readfirstlane(q0), 0), last16));
      __builtin_amdgcn_sched_barrier(0);
      fetch_stage(1, __builtin_amdgcn_readfirstlane(c1));
      load_w16(w[1], min(max(__builtin_amdgcn_readfirstlane(q1), 0), last16));
      __builtin_amdgcn_sched_barrier(0);
      int ecol = 0, eq = 0, eqn = 0;       // window: lane i: column and tile of entry w0 + i + 2, tile of entry w0 + i
      auto step16 = [&](int e, v4i (&ws)[2][4]) {
        const int i = e & 63;
        wait_vmcnt<XQ + 8>();              // the slice and the weights of entry e
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        fetch_stage(e + 2, __builtin_amdgcn_readlane(ecol, i));
        __builtin_amdgcn_sched_barrier(0);
        if (__builtin_amdgcn_readlane(eq, i) >= 0 && e < nc) {
          const uint32_t base = lds_addr(ring) + (e & 3) * SB;
          block_mfma(ws, base, std::integral_constant<int, 0>{});
          if constexpr (NT > 1) block_mfma(ws, base + 4096, std::integral_constant<int, 1>{});
          if constexpr (NT > 2) block_mfma(ws, base + 8192, std::integral_constant<int, 2>{});
          if constexpr (NT > 3) block_mfma(ws, base + 12288, std::integral_constant<int, 3>{});
        }
        __builtin_amdgcn_sched_barrier(0);
        load_w16(ws, min(max(__builtin_amdgcn_readlane(eqn, i), 0), last16));
        __builtin_amdgcn_sched_barrier(0);
      };
#pragma clang loop unroll(disable)
      for (int e = 0; e < nc; e += 2) {
        if ((e & 63) == 0) {
          const int cl = entry(e + lane);
          ecol = entry(e + lane + 2);
          eq = pw[cl];
          eqn = pw[ecol];
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(ecol), "+v"(eq), "+v"(eqn)::"memory");
        }
        step16(e, w[0]);
        step16(e + 1, w[1]);               // past the list: the last column again, not multiplied
      }
      wait_vmcnt<0>();
      __syncthreads();                     // every wave is done with the ring
    } else {
      // The waves are independent: each walks its own list, staging the
      // slice in its quarter of the ring in two token halves.
      const uint32_t rd = lds_addr(region);
      auto fetch_half = [&](int c, int half) {
        fetch_rows(c, half * 16 * TB, region + half * kHalf, std::integral_constant<int, 2 * TB>{});
      };
      auto half_mfma = [&](const v4i (&ws)[2][4], auto half_tag) {
        constexpr int H = decltype(half_tag)::value;
        constexpr int t = H * (TB / 2);
        if constexpr (t < NT) block_mfma(ws, rd + H * kHalf, std::integral_constant<int, t>{});
        if constexpr (TB == 4 && t + 1 < NT) block_mfma(ws, rd + H * kHalf + 4096, std::integral_constant<int, t + 1>{});
      };
      for (int q0 = lo16; q0 < hi16; q0 += 64) {
        const int cols = col_of(a.ids16[min(q0 + lane, hi16 - 1)], r * n_tc, n_tc);
        const int nq = min(64, hi16 - q0);
        fetch_half(__builtin_amdgcn_readlane(cols, 0), 0);
        load_w16(w[0], q0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_half(__builtin_amdgcn_readlane(cols, 0), 1);
        for (int i = 0; i < nq; ++i) {
          const int in = min(i + 1, nq - 1);
          const int cn = __builtin_amdgcn_readlane(cols, in);
          wait_vmcnt<2 * TB>();            // half 0 and the weights are here
          half_mfma(w[0], std::integral_constant<int, 0>{});
          __builtin_amdgcn_sched_barrier(0);
          fetch_half(cn, 0);
          __builtin_amdgcn_sched_barrier(0);
          wait_vmcnt<2 * TB>();            // half 1
          half_mfma(w[0], std::integral_constant<int, 1>{});
          __builtin_amdgcn_sched_barrier(0);
          load_w16(w[0], q0 + in);
          __builtin_amdgcn_sched_barrier(0);
          fetch_half(cn, 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        wait_vmcnt<0>();
      }
    }
  }
  if (!tiles.active) return;

  // ---- outputs: round, bias (double rounding), whole 128-byte rows ------------
  auto stage_out = [&](auto out_tag, auto bias_tag) {
    using OT = typename decltype(out_tag)::type;
    constexpr bool HB = decltype(bias_tag)::value;
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int feat = f * 32 + 8 * g + 4 * (lane >> 5);
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (HB)
#pragma unroll
          for (int e = 0; e < 4; ++e) bv[e] = OT::to_f32(a.bias[min(r * 64 + feat + e, a.m - 1)]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int row = t * 32 + (lane & 31);
          u32x2 y;
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            uint32_t y2 = OT::pack2(acc[f][t][4 * g + 2 * e], acc[f][t][4 * g + 2 * e + 1]);
            if constexpr (HB)   // the reference's double rounding: round(round(acc) + bias)
              y2 = OT::pack2(OT::to_f32((uint16_t)y2) + bv[2 * e], OT::to_f32((uint16_t)(y2 >> 16)) + bv[2 * e + 1]);
            y[e] = y2;
          }
          *reinterpret_cast<u32x2*>(region + row * 128 + (((f * 4 + g) ^ (row & 7)) * 16) + (lane >> 5) * 8) = y;
        }
      }
  };
  if (a.out_bf16) {
    if (a.bias) stage_out(TypeTag<Bf16>{}, std::true_type{});
    else stage_out(TypeTag<Bf16>{}, std::false_type{});
  } else {
    if (a.bias) stage_out(TypeTag<Fp16>{}, std::true_type{});
    else stage_out(TypeTag<Fp16>{}, std::false_type{});
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the wave reads back only its own rows
  store_rows(a, region, r, n0, 32 * NT, lane, 64);
}

template <class XT, int TB, bool DUMP = false>
__global__ void __launch_bounds__(256)
    __attribute__((amdgpu_waves_per_eu(DUMP ? 1 : (TB == 4 ? 2 : 3), DUMP ? 1 : (TB == 4 ? 2 : 3))))
gemm_prefill_blocked_kernel(PrefillArgs a) {
  __shared__ __align__(16) BlockedLds<TB> lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int unit = blockIdx.x % a.n_units, n0 = (blockIdx.x / a.n_units) * (32 * TB);
  // the four slots' tile ranges, one slot per lane (vector loads: one round
  // trip for the row tiles, one for their ranges)
  const int slot = unit * 4 + (lane & 3);
  int rv = slot;
  if (a.rows != nullptr) rv = a.rows[min(slot, a.n_slots - 1)];
  const bool okv = slot < a.n_slots && (unsigned)rv < (unsigned)a.n_tr;
  rv = okv ? rv : 0;
  const int32_t* rp16 = a.w16 != nullptr ? a.rp16 : a.rp8;   // every load unconditional: one round trip
  const int lo8v = a.rp8[rv], end8 = a.rp8[rv + 1], begin16 = rp16[rv], end16 = rp16[rv + 1];
  const int hi8v = okv ? end8 : lo8v;
  const bool has16 = okv && a.w16 != nullptr;
  const int lo16v = has16 ? begin16 : 0, hi16v = has16 ? end16 : 0;
  const bool any8 = __ballot(hi8v > lo8v) != 0;
  const bool heavy = __ballot(3 * (hi16v - lo16v) >= 2 * a.n_tc) != 0;
  auto of_wave = [&](int v) { return __builtin_amdgcn_readlane(v, wave); };
  const SlotTiles mine{of_wave(rv), of_wave(lo8v), of_wave(hi8v), of_wave(lo16v), of_wave(hi16v), of_wave(okv) != 0};
  // Row tiles mostly in 16 bits: the waves share the activation slices of the
  // 16-bit phase too (two programs, so that neither pays the other's registers).
  // A last workgroup of few tokens multiplies only the blocks it has (1, 2 or 4 of
  // them); it is dispatched last and fills the last wave of the grid.  Measured
  // on MI355X, cold weights, all blocks -> these: Qwen2.5-7B Gate/Up at 777
  // tokens (9 of 128 in the last) 220 -> 201 us, at 1030 279 -> 258;
  // Llama-3.2-3B Gate/Up at 1030 119 -> 97; Qwen2.5-7B O at 777 40 -> 38.
  const int left = a.n - n0;
  if (heavy) prefill_blocked_body<XT, TB, TB, true, DUMP>(a, lds, mine, n0, any8, lane, wave);
  else if (left > 16 * TB) prefill_blocked_body<XT, TB, TB, false, DUMP>(a, lds, mine, n0, any8, lane, wave);
  else if (TB == 4 && left > 32) prefill_blocked_body<XT, TB, TB / 2, false, DUMP>(a, lds, mine, n0, any8, lane, wave);
  else prefill_blocked_body<XT, TB, 1, false, DUMP>(a, lds, mine, n0, any8, lane, wave);
}

// ---- few tokens: the row tile's list split over the waves of a workgroup ------
//
// Workgroup = one row tile (FB = 2) or half of one (FB = 1) x 64 tokens: FB x 2
// accumulator blocks per wave.  Its W waves take the tile list round-robin (INT8 positions first, the 16-bit
// ones continuing the rotation, as the decode kernels do), each fetching its
// weight tiles and activation operands straight into registers, D tiles
// ahead, so no wave waits for another until the partial sums are added, in
// wave order, through LDS.  The first 16-bit tile's operands are fetched into the
// wave's LDS before the INT8 tiles are walked.  Bound by what a CU keeps in
// flight: cold weights arrive at about 48 GB/s per CU (Llama-3.2-3B Down, 1 MiB of
// operands per workgroup, takes 25 us on 48 CUs and on 144), so small grids are
// spread over more CUs by halving the row tiles.  Per Llama-3.2-3B layer at 128
// tokens (keep05, four projections, cold weights): 185 us with four row tiles per
// workgroup -> 68 us.
constexpr int kPdAhead = 2;        // tiles in flight per wave beyond the one multiplied (3 and 4: up to 20% slower)
constexpr int kPdRegion = 16384;   // LDS per wave: a 16-bit tile and its activation rows, or 64 x 64 fp32 partials

template <class XT, int FB, int D, bool DUMP = false>
__global__ void __launch_bounds__(512)
    __attribute__((amdgpu_waves_per_eu(DUMP ? 1 : 2, 2)))
gemm_prefill_split_kernel(PrefillArgs a) {
  extern __shared__ __align__(16) int8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int W = blockDim.x >> 6;
  const int n_tc = a.n_tc;
  // the token blocks of a row tile are dealt to one XCD back to back (workgroup
  // b runs on XCD b % 8), so its weights cross the fabric once
  const int ntb = (a.n + 63) / 64;
  constexpr int kParts = 2 / FB;           // workgroups sharing a row tile
  const int group = blockIdx.x >> 3, part = group % (kParts * ntb);
  const int r = (group / (kParts * ntb)) * 8 + (blockIdx.x & 7), n0 = (part / kParts) * 64, f0 = (part % kParts) * 32;
  if (r >= a.n_tr) return;
  const int lo8r = a.rp8[r], n8r = a.rp8[r + 1] - lo8r;
  const int cnt8 = n8r > wave ? (n8r - wave + W - 1) / W : 0;   // this wave's INT8 tiles
  const int32_t* rp16 = a.w16 != nullptr ? a.rp16 : a.rp8;
  const int lo16r = rp16[r], n16r = a.w16 != nullptr ? rp16[r + 1] - lo16r : 0;
  const int f16 = (wave - n8r % W + W) % W;
  const int cnt16 = n16r > f16 ? (n16r - f16 + W - 1) / W : 0;  // ... and 16-bit tiles
  const int first_q = lo16r + f16;
  int8_t* region = lds + wave * kPdRegion;
  const int rowpart = ((lane >> 4) & 1), kpart = lane >> 5, j = lane & 15;

  // 16-bit tile q of column tile c into the wave's region: 64 activation rows of
  // 128 bytes (16-byte chunk c of row R at slot c ^ (R % 8)), then the tile in
  // MFMA order (one KiB per 16 features x 32 columns).
  auto fetch16 = [&](int q, int c) {
    const int xch = ((lane & 7) ^ (lane >> 3)) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t row = min(n0 + 8 * i + (lane >> 3), a.n - 1);
      dma16(a.xf + row * a.ldx + c * 64 + xch, region + i * 1024);
    }
    const uint16_t* t = a.w16 + (int64_t)q * 4096 + f0 * 64;
    const int in_row = j * 64 + (lane >> 4) * 8;
#pragma unroll
    for (int i = 0; i < 4 * FB; ++i)       // i = 2 jb + h
      dma16(a.layout == TQ_LAYOUT_MFMA ? t + i * 512 + lane * 8 : t + (i >> 1) * 1024 + (i & 1) * 32 + in_row,
            region + 8192 + i * 1024);
  };
  auto cols16 = [&](int w0) {              // lane i: column of the wave's 16-bit tile w0 + i
    return col_of(a.ids16[first_q + min(w0 + lane, cnt16 - 1) * W], r * n_tc, n_tc);
  };
  // The first one's operands land while the INT8 tiles are multiplied.
  int wcol16 = 0;
  if (cnt16 > 0) {
    wcol16 = cols16(0);
    fetch16(first_q, __builtin_amdgcn_readlane(wcol16, 0));
  }

  v16f acc[FB][2];
#pragma unroll
  for (int f = 0; f < FB; ++f)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[f][t][v] = 0.f;

  if (cnt8 > 0) {
    int woff[FB];
#pragma unroll
    for (int f = 0; f < FB; ++f)
      woff[f] = f0 * 64 + (a.layout == TQ_LAYOUT_MFMA ? (2 * f + rowpart) * 1024 + kpart * 256 + j * 16
                                                      : (f * 32 + (lane & 31)) * 64 + kpart * 16);
    const int wh = a.layout == TQ_LAYOUT_MFMA ? 512 : 32;
    const int first_p = lo8r + wave;
    int xoff[2];                           // token block t's operand, K half 0 (blocks past the last re-read it)
#pragma unroll
    for (int t = 0; t < 2; ++t) xoff[t] = min(n0 / 16 + 2 * t + rowpart, a.nb - 1) * 1024 + kpart * 256 + j * 16;
    const int64_t xcol = (int64_t)a.nb * 1024;
    v4i w[D][FB][2], x[D][2][2];
    auto load_w = [&](v4i (&d)[FB][2], int i) {
      const int8_t* t = a.w8 + (int64_t)(first_p + min(i, cnt8 - 1) * W) * 4096;
#pragma unroll
      for (int f = 0; f < FB; ++f)
#pragma unroll
        for (int h = 0; h < 2; ++h) d[f][h] = *reinterpret_cast<const v4i*>(t + woff[f] + h * wh);
    };
    auto load_x = [&](v4i (&d)[2][2], int c) {
      const int8_t* b = a.xq + (int64_t)c * xcol;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) d[t][h] = *reinterpret_cast<const v4i*>(b + xoff[t] + h * 512);
    };
    // lane i of a window: the wave's tile w0 + i (the last one past the end)
    auto window = [&](int w0, int& c, float& sc) {
      const int p = first_p + min(w0 + lane, cnt8 - 1) * W;
      c = col_of(a.ids8[p], r * n_tc, n_tc);
      sc = a.sx[c] * a.sw8[p];
    };
    load_w(w[0], 0);                       // needs no column: in flight while the ids arrive
    __builtin_amdgcn_sched_barrier(0);
    int wc, wcn;
    float wsc, wscn;
    window(0, wc, wsc);
    window(64, wcn, wscn);
    __builtin_amdgcn_sched_barrier(0);
    // (the same order of loads as in the loop, so that its waits count exactly)
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (d > 0) load_w(w[d], d);
      __builtin_amdgcn_sched_barrier(0);
      load_x(x[d], __builtin_amdgcn_readlane(wc, d));
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma clang loop unroll(disable)
    for (int i0 = 0; i0 < cnt8; i0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        const int i = i0 + d, in = i + D;
        // tile i's operands: the loads of each of the D - 1 tiles after it
        // may stay in flight (waiting here, outside the branch, keeps the
        // compiler from waiting for everything)
        if constexpr (DUMP) wait_vmcnt<0>();
        else wait_vmcnt<(2 * FB + 4) * (D - 1)>();
        if (i < cnt8) {
          if (i > 0 && (i & 63) == 0) {
            wc = wcn;
            wsc = wscn;
            window(i + 64, wcn, wscn);
          }
          const float sc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wsc), i & 63));
          const int p = first_p + i * W;
          tile_mac<FB, 2>(
              acc, w[d], x[d], sc, [](int) {},
              [&](int f, int t, const v16i& m) {
                if constexpr (DUMP) dump_block(a, p, n0 + 32 * t, f0 + 32 * f, lane, m);
              });
        }
        __builtin_amdgcn_sched_barrier(0);
        const int cn = (in & 63) >= (i & 63) ? __builtin_amdgcn_readlane(wc, in & 63)
                                             : __builtin_amdgcn_readlane(wcn, in & 63);
        load_w(w[d], in);
        load_x(x[d], cn);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    wait_vmcnt<0>();
  }

  if (cnt16 > 0) {
    const uint32_t xrd0 = lds_addr(region) + (lane & 31) * 128;
    const uint32_t wrd = lds_addr(region) + 8192 + rowpart * 2048 + kpart * 256 + j * 16;
    for (int i = 0; i < cnt16; ++i) {
      wait_vmcnt<0>();
#pragma unroll
      for (int kc = 0; kc < 4; ++kc) {     // 16-deep slices, in order
        const uint32_t xrd = xrd0 + (((2 * kc + kpart) ^ (lane & 7)) * 16);
        const uint32_t wr = wrd + (kc >> 1) * 1024 + (kc & 1) * 512;
        v4i xv[2], wv[FB];
        asm volatile(
            "ds_read_b128 %0, %3\n\t"
            "ds_read_b128 %1, %3 offset:4096\n\t"
            "ds_read_b128 %2, %4\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(xv[0]), "=&v"(xv[1]), "=&v"(wv[0])
            : "v"(xrd), "v"(wr)
            : "memory");
        if constexpr (FB == 2)
          asm volatile("ds_read_b128 %0, %1 offset:4096\n\ts_waitcnt lgkmcnt(0)"
                       : "=&v"(wv[FB - 1])
                       : "v"(wr)
                       : "memory");
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int f = 0; f < FB; ++f) acc[f][t] = mfma32<XT>(wv[f], xv[t], acc[f][t]);
      }
      if (i + 1 < cnt16) {                 // every operand is in registers: refill
        if (((i + 1) & 63) == 0) wcol16 = cols16(i + 1);
        __builtin_amdgcn_sched_barrier(0);
        fetch16(first_q + (i + 1) * W, __builtin_amdgcn_readlane(wcol16, (i + 1) & 63));
      }
    }
  }

  // ---- outputs ------------------------------------------------------------------
  auto round4 = [&](const float* y, int feat) {   // four features of one token, rounded (+ bias, rounded again)
    u32x2 o;
    auto go = [&](auto out_tag) {
      using OT = typename decltype(out_tag)::type;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        uint32_t y2 = OT::pack2(y[2 * e], y[2 * e + 1]);
        if (a.bias != nullptr) {
          const int col = r * 64 + feat + 2 * e;
          const float b0 = OT::to_f32(a.bias[min(col, a.m - 1)]), b1 = OT::to_f32(a.bias[min(col + 1, a.m - 1)]);
          y2 = OT::pack2(OT::to_f32((uint16_t)y2) + b0, OT::to_f32((uint16_t)(y2 >> 16)) + b1);
        }
        o[e] = y2;
      }
    };
    if (a.out_bf16) go(TypeTag<Bf16>{});
    else go(TypeTag<Fp16>{});
    return o;
  };
  // Partial sums through LDS: chunk (f, t, g) of wave w is 64 lanes x 4
  // features, summed over the waves in wave order by wave (chunk % W); the
  // rounded outputs are staged and leave as 128-byte rows.
  int8_t* staged = lds + W * kPdRegion;
#pragma unroll
  for (int f = 0; f < FB; ++f)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *reinterpret_cast<v4f*>(region + (f * 8 + t * 4 + g) * 1024 + lane * 16) =
            v4f{acc[f][t][4 * g], acc[f][t][4 * g + 1], acc[f][t][4 * g + 2], acc[f][t][4 * g + 3]};
  __syncthreads();
  for (int q = wave; q < 8 * FB; q += W) {
    v4f s = *reinterpret_cast<const v4f*>(lds + q * 1024 + lane * 16);
    for (int u = 1; u < W; ++u) {
      const v4f p = *reinterpret_cast<const v4f*>(lds + u * kPdRegion + q * 1024 + lane * 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += p[e];
    }
    const int f = q >> 3, t = (q >> 2) & 1, g = q & 3, row = t * 32 + (lane & 31), feat = f0 + f * 32 + 8 * g + 4 * kpart;
    const float y[4] = {s[0], s[1], s[2], s[3]};
    *reinterpret_cast<u32x2*>(staged + row * 128 + (((f0 / 8 + f * 4 + g) ^ (row & 7)) * 16) + kpart * 8) = round4(y, feat);
  }
  __syncthreads();
  store_rows<4 * FB>(a, staged, r, n0, 64, threadIdx.x, blockDim.x, f0 / 8);
}

}  // namespace tq

using namespace tq;

// Schedule of n tokens.  Which sums are formed (W waves' partials, or one
// accumulator per output) depends on n and n_tc only, so stacked projections
// stay bitwise equal to their members.
//
// Split lists while whole-list workgroups leave most of the chip waiting for
// each wave's serial walk (0.56 us per tile).  Measured on MI355X, us per launch,
// whole list -> split over 4 waves, 128 / 192 / 384 / 512 tokens:
//   Llama-3.2-3B Q/K/V   35 -> 15   35 -> 15   35 -> 20   34 -> 27
//     O                  33 -> 10   32 -> 13   33 -> 16   33 -> 18
//     Gate/Up            38 -> 24   38 -> 33   48 -> 51   50 -> 63
//   Qwen2.5-7B Gate/Up   56 -> 54   90 -> 70   96 -> 125  142 -> 179
// Gate/Up alone stops gaining at 200-300 tokens; a layer's three together gain up
// to the limit, 192 / 320 / 384 tokens with uniform keep05 masks: Llama 103 -> 63,
// 113 -> 80, 114 -> 91; Qwen2.5-7B 149 -> 104, 171 -> 153, 177 -> 166; 14B 183 -> 126,
// 206 -> 178, 232 -> 204; with clustered keep10 masks at 384 7B loses (183 -> 191),
// 14B gains (236 -> 223).  The row-major kernels take 198-371 there.  Long lists
// (Down) longer, 192 / 1024 / 1500 tokens: Llama 80 -> 26, 77 -> 54, 103 -> 87;
// Qwen2.5-7B 174 -> 51, 173 -> 139, 229 -> 219; 14B 131 -> 41, 173 -> 131, 183 ->
// 221; at the limit of 1280 78, 194, 197 against 82, 236, 182.  Eight waves where the list is long and the grid small (192 tokens: 24,
// 46 and 39 against 26, 51 and 41 us; at 384 39, 84, 67 against 34, 76, 63).
constexpr int kSplitTokens = 384, kSplitLongTokens = 1280, kSplitLongTiles = 96, kSplitWideTokens = 256;
static int split_waves(int n, int n_tc) {
  if (n > (n_tc >= kSplitLongTiles ? kSplitLongTokens : kSplitTokens)) return 0;
  return n_tc >= kSplitLongTiles && n <= kSplitWideTokens ? 8 : 4;
}

// 64 or 128 tokens per workgroup otherwise (the same sums): the cheaper grid
// by the time of the most loaded CU.  A CU runs three 64-token workgroups or two
// 128-token ones together; measured on MI355X with 48-tile lists (us), 64
// tokens: 35 for one workgroup per CU, 51 for two, 68 for three; 128 tokens: 55
// and 83.  E.g. Llama-3.2-3B O at 2048 tokens 49 (64) vs 56 us, Gate/Up at 1024
// 102 vs 93, Q/K/V at 4096 120 vs 130, Gate/Up at 8192 701 vs 638.  From 64 units
// on, 128 tokens wherever a CU gets two of them: 64-token workgroups read the
// weights twice as often, and those of so many units do not stay in the L2s
// (Qwen2.5-7B Gate/Up at 777 / 2048 / 8192 tokens 268 / 669 / 2697 vs 229 / 476 /
// 1869 us).  Lists of other lengths scale both sides: over the four projections
// of Llama-3.2-3B, Qwen2.5-7B and 14B (48 to 296 tiles) at 400 to 4096 tokens the
// rule takes the faster side at 84 of 87 points and loses 1, 5 and 16% (Llama
// Gate/Up at 600 tokens, 81 vs 70 us) at the others.
static int blocked_tb(int n, int units) {
  constexpr int kCus = 256, kManyUnits = 64;
  const int64_t l2 = ((int64_t)units * ((n + 63) / 64) + kCus - 1) / kCus;
  const int64_t l4 = ((int64_t)units * ((n + 127) / 128) + kCus - 1) / kCus;
  if (units >= kManyUnits && l4 >= 2) return 4;
  const int64_t rest2[3] = {0, 35, 51};
  return (l4 / 2) * 83 + (l4 % 2) * 55 < (l2 / 3) * 68 + rest2[l2 % 3] ? 4 : 2;
}

// Half row tiles while the whole ones leave half of the CUs without work (the
// same sums).  Measured on MI355X with cold weights, whole -> half (us): Llama O
// (48 row tiles) at 128 tokens 12.7 -> 9.7, at 192 12.7 -> 11.6; Down (eight waves)
// at 128 24.9 -> 19.2, at 192 24.5 -> 28.9; Qwen2.5-7B Down (56) at 128 47.4 ->
// 36.9, at 192 46.5 -> 64.4; Q/K/V (80) at 128 14.9 -> 15.9.
constexpr int kSplitHalfGrid = 128;
static bool split_halves(int n, int n_tr) { return (int64_t)n_tr * ((n + 63) / 64) <= kSplitHalfGrid; }

template <class XT, int FB, bool DUMP>
static hipError_t launch_split(const PrefillArgs& a, int W, hipStream_t s) {
  constexpr auto kern = gemm_prefill_split_kernel<XT, FB, kPdAhead, DUMP>;
  const int64_t blocks = 8ll * ((a.n_tr + 7) / 8) * ((a.n + 63) / 64) * (2 / FB);
  if (blocks >= (1ll << 31)) return hipErrorInvalidValue;
  const size_t lds = (size_t)W * kPdRegion + 8192;
  const hipError_t e = allow_lds<kern>(lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(64 * W), lds, s, a);
  return hipGetLastError();
}

template <class XT, bool DUMP>
static hipError_t launch_blocked(PrefillArgs a, hipStream_t s) {
  if (const int W = split_waves(a.n, a.n_tc)) {
    return split_halves(a.n, a.n_tr) ? launch_split<XT, 1, DUMP>(a, W, s) : launch_split<XT, 2, DUMP>(a, W, s);
  }
  a.n_units = (a.n_slots + 3) / 4;
  const int tb = blocked_tb(a.n, a.n_units);
  const int64_t blocks = (int64_t)a.n_units * ((a.n + 32 * tb - 1) / (32 * tb));
  if (blocks >= (1ll << 31)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)blocks), block(256);
  if (tb == 4) hipLaunchKernelGGL((gemm_prefill_blocked_kernel<XT, 4, DUMP>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((gemm_prefill_blocked_kernel<XT, 2, DUMP>), grid, block, 0, s, a);
  return hipGetLastError();
}

extern "C" int tq_gemm_mixed_blocked(const int8_t* x_blocked, const float* sx, const int8_t* int8_tiles,
                                     const float* int8_scales, const int32_t* int8_tile_ids,
                                     const int32_t* int8_row_ptr, const void* x_fp, int64_t x_fp_stride_n, int x_dtype,
                                     const void* fp16_tiles, const int32_t* fp16_tile_ids, const int32_t* fp16_row_ptr,
                                     void* out, int64_t out_stride_n, int out_dtype, const void* bias, int n, int m,
                                     int k, int n_tr, int n_tc, int tile_layout, const int32_t* row_order, int n_slots,
                                     int32_t* products, int row0, int rows, void* stream) {
  if (n < 0 || m < 0 || n_tr < 0 || n_tc < 0 || k != n_tc * 64 || (int64_t)n_tr * 64 < m || n_tc > kPbCols)
    return TQ_ERR_ARG;
  if (x_dtype != TQ_DTYPE_BF16 && x_dtype != TQ_DTYPE_FP16) return TQ_ERR_DTYPE;
  if (out_dtype != TQ_DTYPE_BF16 && out_dtype != TQ_DTYPE_FP16) return TQ_ERR_DTYPE;
  if (tile_layout != TQ_LAYOUT_ROW_MAJOR && tile_layout != TQ_LAYOUT_MFMA) return TQ_ERR_DTYPE;
  if (n == 0 || m == 0) return TQ_OK;
  if (n_tc == 0 || int8_row_ptr == nullptr || out == nullptr || out_stride_n < m || x_blocked == nullptr || sx == nullptr)
    return TQ_ERR_ARG;
  const bool has16 = fp16_tiles != nullptr && fp16_tile_ids != nullptr && fp16_row_ptr != nullptr;
  if (has16 && (x_fp == nullptr || x_fp_stride_n < k)) return TQ_ERR_ARG;
  if (!aligned16(int8_tiles) || !aligned16(x_blocked) ||
      (has16 && (!aligned16(fp16_tiles) || !aligned16(x_fp) || (x_fp_stride_n % 8) != 0)))
    return TQ_ERR_ALIGN;
  if (row_order != nullptr && n_slots < 1) return TQ_ERR_ARG;
  if (products != nullptr && (x_dtype != TQ_DTYPE_BF16 || row0 < 0 || rows < 1 || rows > n - row0)) return TQ_ERR_ARG;
  PrefillArgs a{};
  a.xq = x_blocked; a.sx = sx; a.w8 = int8_tiles; a.sw8 = int8_scales; a.ids8 = int8_tile_ids; a.rp8 = int8_row_ptr;
  a.xf = has16 ? static_cast<const uint16_t*>(x_fp) : nullptr; a.ldx = x_fp_stride_n;
  a.w16 = has16 ? static_cast<const uint16_t*>(fp16_tiles) : nullptr;
  a.ids16 = fp16_tile_ids; a.rp16 = fp16_row_ptr;
  a.out = static_cast<uint16_t*>(out); a.ldo = out_stride_n; a.bias = static_cast<const uint16_t*>(bias);
  a.rows = row_order; a.n_slots = row_order != nullptr ? n_slots : n_tr; a.dump = products; a.dump_r0 = row0; a.dump_n = rows;
  a.n = n; a.m = m; a.n_tr = n_tr; a.n_tc = n_tc; a.nb = (n + 15) / 16;
  a.out_bf16 = out_dtype == TQ_DTYPE_BF16; a.layout = tile_layout;
  a.ovec = (out_stride_n % 8) == 0 && aligned16(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e;
  if (products != nullptr) e = launch_blocked<Bf16, true>(a, s);
  else if (x_dtype == TQ_DTYPE_BF16) e = launch_blocked<Bf16, false>(a, s);
  else e = launch_blocked<Fp16, false>(a, s);
  return (int)e;
}

extern "C" int tq_prompt_forward(const tq_prompt_desc* d) {
  if (d == nullptr) return TQ_ERR_ARG;
  if (d->quantize) {
    const int rc = tq_act_quant_blocked(d->x, d->x_stride, d->x_dtype, d->n, d->k, d->x_blocked, d->sx, d->workspace,
                                        d->workspace_elems, d->stream);
    if (rc != 0) return rc;
  }
  return tq_gemm_mixed_blocked(d->x_blocked, d->sx, d->int8_tiles, d->int8_scales, d->int8_tile_ids, d->int8_row_ptr,
                               d->x, d->x_stride, d->x_dtype, d->fp16_tiles, d->fp16_tile_ids, d->fp16_row_ptr, d->out,
                               d->out_stride, d->out_dtype, d->bias, d->n, d->m, d->k, d->n_tr, d->n_tc,
                               d->tile_layout, d->row_order, d->n_slots, nullptr, 0, 0, d->stream);
}

extern "C" int tq_gemm_row_order(const int32_t* fp16_row_ptr, int n_tr, int n_tc, int32_t* slots, int max_slots) {
  if (fp16_row_ptr == nullptr || slots == nullptr || n_tr < 1 || n_tc < 1 || max_slots < n_tr + 3) return TQ_ERR_ARG;
  std::vector<int32_t> order((size_t)n_tr);
  for (int r = 0; r < n_tr; ++r) order[r] = r;
  auto count = [&](int r) { return fp16_row_ptr[r + 1] - fp16_row_ptr[r]; };
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return count(a) > count(b); });
  int n = 0;
  size_t i = 0;
  for (; i < order.size() && 3 * (int64_t)count(order[i]) >= 2 * (int64_t)n_tc; ++i) slots[n++] = order[i];
  while (n % 4 != 0) slots[n++] = -1;
  for (; i < order.size(); ++i) slots[n++] = order[i];
  return n;
}
