// Attention core of the gpt-oss decoder layer: grouped-query attention with a
// learned per-head sink logit, causal and sliding-window masks.
//
// Semantics (transformers 5.15.0 models/gpt_oss/modeling_gpt_oss.py:235-264,
// eager_attention_forward, called from GptOssAttention.forward :295-336):
//   S[t, j]  = (q[t] . k[j]) * scaling  (+ mask: -inf where key j is hidden)
//   probs    = softmax over [S[t, 0..Tk-1], sink[h]]  (the sink column is
//              the head's logit, unscaled), then the sink column is dropped
//   out[t]   = sum_j probs[t, j] v[j]
// with key head h / (Hq / Hkv) serving query head h (repeat_kv, :203-212).
// Masks: none (every key visible: what the eager path does with
// attention_mask=None, the way the streaming runner calls the decoder,
// block_streamer/runners.py:327-335), causal (key j visible to query t at
// absolute position p = Tk - Tq + t when j <= p), or causal with a window w
// (also p - j < w: masking_utils' sliding-window overlay).
//
// The sink enters the online softmax as its starting state: running maximum
// = sink, running sum = exp(sink - sink) = 1, accumulator = 0.  Products run
// on bf16 MFMA (v_mfma_f32_32x32x16_bf16) with float32 accumulation; the
// probabilities are rounded to bf16 for the P.V product (as the eager path's
// cast to the value dtype).
//
// Rows: a workgroup of the forward and of the dq backward takes 128 rows of
// one (batch, key head); row R = t * G + i is query t of head G * hk + i
// (G = Hq / Hkv), so the G heads sharing a key head read each K/V tile once.
// Four waves, 32 rows each (lane c = row c of the wave), key tiles of 64.
// Short query grids (decoding: one row block per sequence and key head) split
// each row block's key tiles over several workgroups that write unnormalised
// partial sums; attn_split_combine_kernel merges them (bsa_attention_fwd_split).
//
// Orientation: S^T = K Q^T puts a query in each lane, so its row maximum and
// sum are one exchange between the two lane halves.  The K rows enter that
// MFMA permuted (pi below): lane half g then holds keys 8g .. 8g+7 and
// 16 + 8g .. 16 + 8g + 7 of each 32-key block, which is exactly the B
// operand of O^T += V^T P^T, so the probabilities never leave registers and
// the online-softmax rescale of query c stays in lane c.
//
// LDS: every tile is the natural row-major copy a DMA (global_load_lds)
// brings in: 64 rows x 128 bytes, 16-byte chunk c of row R at position
// c ^ sw(R), sw(R) = 4 * ((R >> 1) & 1) | ((R >> 2) & 3).  Two kinds of read
// use it: ds_read_b128 of 16 rows at one chunk (the operands K, V, Q, dO
// with rows permuted), whose 16 (R & 1, sw) pairs are distinct, and the
// transposing ds_read_b64_tr_b16 (V^T, K^T, Q^T, dO^T: in each 16-lane
// group, lane s addresses 4 elements of row k0 + s/4 at column m0 + 4(s%4)
// and lane i receives element i%4 of lanes i/4, 4 + i/4, 8 + i/4, 12 + i/4:
// column m0 + i at rows k0 .. k0+3), whose four rows land in four different
// 64-byte quarters of the 256-byte bank period.  Tiles stream through a ring
// of AT_NS stages, AT_NS - 1 ahead of the computation.
// ---------------------------------------------------------------------------
#include "bsa_common.h"

namespace bsa {

constexpr int AT_D = 64;                    // head dimension
constexpr int AT_BR = 128;                  // rows per workgroup (forward, dq)
constexpr int AT_BC = 64;                   // keys per tile
constexpr int AT_TILE = AT_BC * AT_D * 2;   // 8 KiB
constexpr int AT_NS = 2;                    // ring stages (forward, dq)

struct AttnArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const float* sinks;   // [Hq] or null (no sink)
  uint16_t* out;
  float* lse;           // [B][Hq][Tq] log2 of the softmax denominator in
                        // scaled-logit units (with the sink), or null
  int64_t sqb, sqt, sqh, skb, skt, skh, svb, svt, svh, sob, sot, soh;
  int B, Tq, Tk, Hq, Hkv, G;
  int causal, window;
  int rblocks;          // row blocks of 128
  float scale2;         // scaling * log2(e)
  // key-split forward (nsplit > 1): workgroup x = row block * nsplit + split
  // takes a contiguous share of the row block's key tiles and writes its rows'
  // unnormalised accumulators and (running max, sum) to part_o / part_ml at
  // row ((split * B + b) * Hkv + hk) * (Tq * G) + R; attn_split_combine_kernel
  // merges them
  int nsplit;
  float* part_o;        // [nsplit][B][Hkv][Tq * G][64]
  float* part_ml;       // [nsplit][B][Hkv][Tq * G][2]
};

typedef short s16x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int at_sw(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }

// Byte offset of 16-byte chunk `ch` of row `row` of a tile.
__device__ __forceinline__ uint32_t at_off(int row, int ch) {
  return (uint32_t)(row * 128 + ((ch ^ at_sw(row)) << 4));
}

// Transposing read: the address this lane supplies so that, for the rows
// k0 .. k0+3 (k0 = 16 s + 8 g + 4 h, g = lane / 32) and columns m0 + 0..15
// of its 16-lane group (m0 = 32 mb + 16 ((lane >> 4) & 1)), lane receives
// column m0 + lane % 16 at those four rows.
__device__ __forceinline__ uint32_t at_tr_off(int lane, int s, int h, int mb) {
  const int sl = lane & 15;
  const int row = 16 * s + 8 * (lane >> 5) + 4 * h + (sl >> 2);
  const int col = 32 * mb + 16 * ((lane >> 4) & 1) + 4 * (sl & 3);
  return (uint32_t)(row * 128 + ((((col >> 3) ^ at_sw(row)) << 4) | ((col & 7) << 1)));
}

__device__ __forceinline__ u32x4_t at_tr8(const uint8_t* tile, uint32_t o0, uint32_t o1) {
  typedef __attribute__((address_space(3))) s16x4_t lds_s16x4;
  const s16x4_t a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + o0));
  const s16x4_t b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + o1));
  const uint2 ua = __builtin_bit_cast(uint2, a), ub = __builtin_bit_cast(uint2, b);
  return u32x4_t{ua.x, ua.y, ub.x, ub.y};
}

// MFMA row r of S^T (or S) takes key (row) pi(r): with r = 8a + 4g + b
// (a 0..3, g 0..1, b 0..3), pi(r) = 16 (a >> 1) + 8g + 4 (a & 1) + b, so that
// output register v of lane half g is 8g + v (v < 8) or 16 + 8g + v - 8.
__device__ __forceinline__ int at_pi(int r) {
  const int a = r >> 3, g = (r >> 2) & 1, b = r & 3;
  return 16 * (a >> 1) + 8 * g + 4 * (a & 1) + b;
}

__device__ __forceinline__ f32x16_t at_mfma(const u32x4_t& a, const u32x4_t& b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                 c, 0, 0, 0);
}

// Two floats -> packed bf16 (v_cvt_pk_bf16_f32: round to nearest even).
__device__ __forceinline__ uint32_t at_pack2(float lo, float hi) {
  const bf16x2_t v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}

// max / sum of a value and its copy in lane ^ 32 (v_permlane32_swap: the
// pair holds both halves' values; combining them symmetrically gives every
// lane the same result, operands in the same order)
__device__ __forceinline__ float at_max32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float at_add32(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// s_waitcnt vmcnt(N) (expcnt and lgkmcnt not waited on)
template <int N>
__device__ __forceinline__ void at_wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Wait until at most min(ahead, MAXAHEAD) tiles of PER loads each are in flight.
template <int PER, int MAXAHEAD>
__device__ __forceinline__ void wait_vmcnt_tiles(int ahead) {
  if constexpr (MAXAHEAD <= 0) {
    at_wait_vmcnt<0>();
  } else {
    if (ahead >= MAXAHEAD) {
      at_wait_vmcnt<MAXAHEAD * PER>();
      return;
    }
    wait_vmcnt_tiles<PER, MAXAHEAD - 1>(ahead);
  }
}

// 16-byte DMA into LDS (per lane: source `src`; destination `lds` + 16 * lane,
// `lds` uniform).  Written in assembly because the compiler, seeing the
// builtin, waits for every DMA in flight (vmcnt(0)) before any transposing LDS
// read, i.e. for the next tile in the middle of the present one.  It counts no
// destination registers, so the kernels' own vmcnt waits and barriers are all
// that orders it; a vmcnt wait the compiler adds for loads of its own can
// only wait for more than it needs.  m0 is a reserved register that no clobber
// list can name: nothing else in these kernels may need it (an LDS DMA builtin
// beside them would, and the compiler could keep its m0 across this one).
__device__ __forceinline__ void at_dma16(const void* src, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory");
}
__device__ __forceinline__ void at_dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
               : "memory");
}
__device__ __forceinline__ void at_dma4(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base)
               : "memory");
}
__device__ __forceinline__ uint32_t at_lds(const void* p) { return (uint32_t)(uintptr_t)(lds_void*)p; }

// Row strides (bytes) up to which 64 rows stay within a 32-bit offset.
constexpr int64_t AT_NEAR = 1 << 24;

// Consecutive 64-row x 128-byte tiles by four waves: instruction m of wave w
// fills LDS bytes (256 m + 64 w + lane) * 16, i.e. row 32 m + 8 w + lane / 8,
// position lane & 7, from source chunk position ^ sw(row) (the same chunk for
// both m).  A tile wholly inside takes a uniform base, which moves on with the
// tiles, and the lane's 32-bit offset; rows past the last repeat it.
struct AtSrc {
  const uint8_t* base;  // row 0 (uniform)
  const uint8_t* next;  // row 0 of the next tile (uniform)
  int64_t stride;       // bytes per row (uniform)
  uint32_t off;         // this lane's row (m = 0) and chunk within a tile
};
__device__ __forceinline__ AtSrc at_src(const uint16_t* base, int64_t stride, int tile0, int wave, int lane) {
  const int row = 8 * wave + (lane >> 3);
  AtSrc s;
  s.base = reinterpret_cast<const uint8_t*>(base);
  s.stride = stride * 2;
  s.next = s.base + (int64_t)tile0 * (64 * s.stride);
  s.off = (uint32_t)row * (uint32_t)s.stride + ((lane & 7) ^ at_sw(row)) * 16;
  return s;
}
__device__ __forceinline__ void at_dma_tile(AtSrc& s, int row0, int rows, uint32_t lds, int wave, int lane) {
  if (row0 + 64 <= rows && s.stride <= AT_NEAR) {
    at_dma16(s.next, s.off, lds);
    at_dma16(s.next + 32 * s.stride, s.off, lds + 4096);
  } else {
    const int row = 8 * wave + (lane >> 3);
#pragma unroll
    for (int m = 0; m < 2; ++m)
      at_dma16(s.base + (int64_t)min(row0 + 32 * m + row, rows - 1) * s.stride + ((lane & 7) ^ at_sw(row)) * 16,
               lds + 4096 * m);
  }
  s.next += 64 * s.stride;
}

// The n lowest bits (n clamped to 0..32).
__device__ __forceinline__ uint32_t at_low(int n) {
  return (uint32_t)((1ull << min(max(n, 0), 32)) - 1ull);
}
// Visibility of 32 keys from j0 for the query that sees keys [lo, hi): bit i
// = key j0 + 8g + i (the keys a lane of half g holds are bits 0-7 and 16-23).
__device__ __forceinline__ uint32_t at_vis(int lo, int hi, int j0, int g) {
  return (at_low(hi - j0) & ~at_low(lo - j0)) >> (8 * g);
}
// All ones if register v's key is visible, else 0.
__device__ __forceinline__ uint32_t at_vis_mask(uint32_t vis, int v) {
  return (uint32_t)__builtin_amdgcn_sbfe((int)vis, v < 8 ? v : v + 8, 1);
}

// 32 x 64 accumulators in C layout (register 4 q + e of block db, lane (c, g):
// column c, d = 32 db + 8 q + 4 g + e) times f, as bf16 at row + d: the two
// lane halves exchange 8-byte halves so that every store is 16 bytes.
__device__ __forceinline__ void at_store_row(uint16_t* row, const f32x16_t (&acc)[2], float f, int g) {
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      uint32_t w[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 2; ++e)
          w[i][e] = at_pack2(acc[db][8 * q + 4 * i + 2 * e] * f, acc[db][8 * q + 4 * i + 2 * e + 1] * f);
      const auto x = __builtin_amdgcn_permlane32_swap(w[0][0], w[1][0], false, false);
      const auto y = __builtin_amdgcn_permlane32_swap(w[0][1], w[1][1], false, false);
      // half 0: d 16q .. 16q + 7, half 1: d 16q + 8 .. 16q + 15
      *reinterpret_cast<u32x4_t*>(row + 32 * db + 16 * q + 8 * g) = u32x4_t{x[0], y[0], x[1], y[1]};
    }
}

// Workgroup order of all three kernels: (batch, key head) pairs vary fastest,
// so the longest work of every pair starts first, and with a multiple of
// eight pairs all of a pair's workgroups run on one XCD, whose L2 holds the
// pair's keys and values (causal forward, 64/8 heads, against row blocks
// fastest: 8192 tokens 696 -> 611 us, 2048 tokens 72 -> 51 us).  A grid past
// the launch limit keeps (x, key head, batch) as its three dimensions.
struct AtBlock {
  int x, hk, b;
};
__device__ __forceinline__ AtBlock at_block(int B, int Hkv) {
  if (gridDim.y > 1 || gridDim.z > 1) return AtBlock{(int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
  const int pairs = B * Hkv;
  const int x = (int)blockIdx.x / pairs;
  const int pair = (int)blockIdx.x - x * pairs;
  const int b = pair / Hkv;
  return AtBlock{x, pair - b * Hkv, b};
}

// Row geometry of the forward and the dq backward.  Per lane: row R (query t,
// head h) and the keys [lo, hi) it sees; uniform: the workgroup's key tiles
// and the positions of the wave's first and last row.
struct AtRows {
  int R, t, h, rows, R0, lo, hi;
  int kt0, kt1;          // key tiles of the workgroup
  int ktf0, ktf1;        // of those, the tiles whose keys every row sees
  int wlo0, wlo1;        // first key seen by the wave's first / last row
  int whi0, whi1;        // one past the last key seen by them
  bool live_wave;
};

__device__ __forceinline__ AtRows at_rows(int Tq, int Tk, int G, int causal, int window, int rb, int hk, int wave,
                                          int c) {
  AtRows r;
  r.rows = Tq * G;
  r.R0 = rb * AT_BR;
  r.R = min(r.R0 + 32 * wave + c, r.rows - 1);  // rows past the end repeat the last (never stored)
  r.t = r.R / G;
  r.h = hk * G + (r.R - r.t * G);
  const int off = Tk - Tq;
  auto first = [&](int t) { return window > 0 ? max(0, off + t - window + 1) : 0; };
  auto end = [&](int t) { return causal ? min(Tk, off + t + 1) : Tk; };
  r.lo = first(r.t);
  r.hi = end(r.t);
  const int tw0 = min(r.R0 + 32 * wave, r.rows - 1) / G, tw1 = min(r.R0 + 32 * wave + 31, r.rows - 1) / G;
  r.wlo0 = first(tw0);
  r.wlo1 = first(tw1);
  r.whi0 = end(tw0);
  r.whi1 = end(tw1);
  r.kt0 = first(r.R0 / G) / AT_BC;
  r.kt1 = (end((min(r.R0 + AT_BR, r.rows) - 1) / G) + AT_BC - 1) / AT_BC;
  r.ktf0 = min(r.kt1, (first((min(r.R0 + AT_BR, r.rows) - 1) / G) + AT_BC - 1) / AT_BC);
  r.ktf1 = max(r.ktf0, end(r.R0 / G) / AT_BC);
  r.live_wave = r.R0 + 32 * wave < r.rows;
  return r;
}

// One key tile (its 32-key blocks KB0 .. KB1) of the forward for one wave.
// MASK: some of those keys are hidden from some of the wave's rows.
template <bool MASK, int KB0, int KB1>
__device__ __forceinline__ void at_fwd_tile(const uint8_t* K, const uint32_t (&koff)[4], const uint32_t (&voff)[2][2],
                                            const u32x4_t (&qf)[4], int j0, int lo, int hi, int g, float scale2,
                                            float& m, float& l, f32x16_t (&o)[2]) {
  constexpr int NK = KB1 - KB0 + 1;
  const uint8_t* V = K + AT_TILE;
  f32x16_t sc[NK];
#pragma unroll
  for (int kb = 0; kb < NK; ++kb) {
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[kb][v] = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      sc[kb] = at_mfma(*reinterpret_cast<const u32x4_t*>(K + koff[s] + 4096 * (KB0 + kb)), qf[s], sc[kb]);
  }
  // the maximum of the raw products (scale2 > 0), hidden keys at -inf
  float mt = -INFINITY;
#pragma unroll
  for (int kb = 0; kb < NK; ++kb) {
    if constexpr (MASK) {
      const uint32_t vis = at_vis(lo, hi, j0 + 32 * (KB0 + kb), g);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const uint32_t k = at_vis_mask(vis, v);
        sc[kb][v] = __uint_as_float((k & __float_as_uint(sc[kb][v])) | (~k & 0xFF800000u));
      }
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) mt = fmaxf(mt, sc[kb][v]);
  }
  // the accumulator is rescaled only when some row's maximum moved (every
  // other row has alpha = 1 exactly, or an accumulator still 0)
  const float mt2 = at_max32(mt) * scale2;
  const bool grow = mt2 > m;
  const float mn = grow ? mt2 : m;
  // a row that has seen nothing yet (no sink, every key so far hidden) keeps 0
  const float ms = mn == -INFINITY ? 0.f : mn;
  const float alpha = __builtin_amdgcn_exp2f(m - ms);
  float rs = 0.f;
  u32x4_t pf[2 * NK];  // P^T operands of the 16-key steps
#pragma unroll
  for (int kb = 0; kb < NK; ++kb)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[kb][8 * half + i], scale2, -ms));
        rs += p[i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) pf[2 * kb + half][i] = at_pack2(p[2 * i], p[2 * i + 1]);
    }
  rs = at_add32(rs);
  l = l * alpha + rs;
  m = mn;
  if (__builtin_amdgcn_ballot_w64(grow)) {
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[db][v] *= alpha;
  }
#pragma unroll
  for (int s = 0; s < 2 * NK; ++s)
#pragma unroll
    for (int db = 0; db < 2; ++db)
      o[db] = at_mfma(at_tr8(V + 2048 * (2 * KB0 + s), voff[db][0], voff[db][1]), pf[s], o[db]);
}

// Bound by VALU issue: a full tile is ~155 VALU instructions and 33
// exponentials for 16 MFMAs per wave, and neither occupancy (2, 3 and 4 waves
// per SIMD: 696, 692, 697 us at 8192 causal tokens, 64/8 heads) nor a software
// pipeline over tiles (735 against 735 us with the other costs as they were)
// moves it; fewer instructions do: no per-element branches, full tiles in a
// loop of their own, uniform DMA addresses (772 -> 692 us), then the order of
// the workgroups (611 us, 900 TFLOP/s; 128-key window 65 -> 54 us).
__global__ __launch_bounds__(256, 3) void attn_fwd_kernel(AttnArgs a) {
  extern __shared__ __align__(1024) uint8_t at_smem[];  // AT_NS stages of [K tile][V tile]
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31;
  const int g = lane >> 5;
  // the last row blocks have the most keys under a causal mask: start them first
  const int nsplit = a.nsplit > 1 ? a.nsplit : 1;
  const AtBlock blk = at_block(a.B, a.Hkv);
  const int sp = blk.x % nsplit;
  const int rb = a.rblocks - 1 - blk.x / nsplit;
  const int hk = blk.hk;
  const int b = blk.b;
  const AtRows rw = at_rows(a.Tq, a.Tk, a.G, a.causal, a.window, rb, hk, wave, c);
  // this workgroup's key tiles: all of the row block's, or split sp's share
  int kt_lo = rw.kt0, kt_hi = rw.kt1;
  if (nsplit > 1) {
    const int per = (rw.kt1 - rw.kt0 + nsplit - 1) / nsplit;
    kt_lo = min(rw.kt1, rw.kt0 + sp * per);
    kt_hi = min(rw.kt1, kt_lo + per);
  }

  AtSrc ks = at_src(a.k + b * a.skb + (int64_t)hk * a.skh, a.skt, kt_lo, wave, lane);
  AtSrc vs = at_src(a.v + b * a.svb + (int64_t)hk * a.svh, a.svt, kt_lo, wave, lane);
  const uint32_t lds0 = at_lds(at_smem) + 1024 * wave;
  auto issue = [&](int kt) {
    const uint32_t st = lds0 + (kt % AT_NS) * (2 * AT_TILE);
    at_dma_tile(ks, kt * AT_BC, a.Tk, st, wave, lane);
    at_dma_tile(vs, kt * AT_BC, a.Tk, st + AT_TILE, wave, lane);
  };
  constexpr int DPT = 4;  // DMA instructions per wave per tile

  // Q fragments (B operand of S^T): d 16s + 8g .. +7 of row c
  const uint16_t* qrow = a.q + b * a.sqb + (int64_t)rw.t * a.sqt + (int64_t)rw.h * a.sqh;
  u32x4_t qf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) qf[s] = *reinterpret_cast<const u32x4_t*>(qrow + 16 * s + 8 * g);
  constexpr float LOG2E = 1.4426950408889634f;
  // the sink is the starting state of split 0 only
  float m = a.sinks && sp == 0 ? a.sinks[rw.h] * LOG2E : -INFINITY;
  float l = a.sinks && sp == 0 ? 1.f : 0.f;
  for (int i = 0; i < AT_NS - 1; ++i)
    if (kt_lo + i < kt_hi) issue(kt_lo + i);

  // read offsets: K rows 32 kb + pi(c) at d chunk 2s + g (kb adds 4096);
  // V^T via transposing reads (d block db, 16-key step s adds 2048, halves h)
  uint32_t koff[4], voff[2][2];
#pragma unroll
  for (int s = 0; s < 4; ++s) koff[s] = at_off(at_pi(c), 2 * s + g);
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int h = 0; h < 2; ++h) voff[db][h] = at_tr_off(lane, 0, h, db);

  f32x16_t o[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[db][v] = 0.f;
  // the loads above land here, not inside the loop (where the wait would
  // drain the DMA ring on every tile)
#pragma unroll
  for (int s = 0; s < 4; ++s) asm volatile("" : "+v"(qf[s]));
  asm volatile("" : "+v"(m));

  // tile kt has landed once at most the tiles issued after it are in flight;
  // the barrier also certifies every wave's reads of tile kt - 1 are done,
  // whose stage takes tile kt + AT_NS - 1 (bare s_barrier: a __syncthreads()
  // fence would wait for that DMA too)
  auto turn = [&](int kt) {
    wait_vmcnt_tiles<DPT, AT_NS - 2>(kt_hi - 1 - kt);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + AT_NS - 1 < kt_hi) issue(kt + AT_NS - 1);
  };
  auto masked = [&](int kt0, int kt1) {
    for (int kt = kt0; kt < kt1; ++kt) {
      turn(kt);
      const uint8_t* K = at_smem + (kt % AT_NS) * (2 * AT_TILE);
      const int j0 = kt * AT_BC;
      // 32-key blocks that some of the wave's rows see (uniform)
      const bool live0 = rw.live_wave && j0 < rw.whi1 && j0 + 32 > rw.wlo0;
      const bool live1 = rw.live_wave && j0 + 32 < rw.whi1 && j0 + 64 > rw.wlo0;
      if (live0 && live1)
        at_fwd_tile<true, 0, 1>(K, koff, voff, qf, j0, rw.lo, rw.hi, g, a.scale2, m, l, o);
      else if (live0)
        at_fwd_tile<true, 0, 0>(K, koff, voff, qf, j0, rw.lo, rw.hi, g, a.scale2, m, l, o);
      else if (live1)
        at_fwd_tile<true, 1, 1>(K, koff, voff, qf, j0, rw.lo, rw.hi, g, a.scale2, m, l, o);
    }
  };
  // tiles every row sees, between the partly hidden ones at either end; each
  // run is a loop of its own so that no merge of the two forms costs register
  // copies on every tile
  const int f0 = min(max(rw.ktf0, kt_lo), kt_hi), f1 = min(max(rw.ktf1, f0), kt_hi);
  masked(kt_lo, f0);
  for (int kt = f0; kt < f1; ++kt) {
    turn(kt);
    if (rw.live_wave)
      at_fwd_tile<false, 0, 1>(at_smem + (kt % AT_NS) * (2 * AT_TILE), koff, voff, qf, 0, 0, 0, g, a.scale2, m, l, o);
  }
  masked(f1, kt_hi);

  if (rw.R0 + 32 * wave + c >= rw.rows) return;
  if (nsplit > 1) {
    const int64_t pidx = (((int64_t)sp * a.B + b) * a.Hkv + hk) * rw.rows + rw.R;
    float* po = a.part_o + pidx * AT_D;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const int d = 32 * db + 8 * q4 + 4 * g;
        *reinterpret_cast<f32x4_t*>(po + d) =
            f32x4_t{o[db][4 * q4], o[db][4 * q4 + 1], o[db][4 * q4 + 2], o[db][4 * q4 + 3]};
      }
    if (g == 0) *reinterpret_cast<float2*>(a.part_ml + pidx * 2) = make_float2(m, l);
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  at_store_row(a.out + b * a.sob + (int64_t)rw.t * a.sot + (int64_t)rw.h * a.soh, o, inv, g);
  // __builtin_amdgcn_logf is log2
  if (a.lse && g == 0) a.lse[((int64_t)b * a.Hq + rw.h) * a.Tq + rw.t] = m + __builtin_amdgcn_logf(l);
}

// Merge of the key splits, one wave per row (lane = d): with M = max_s m_s,
// w_s = 2^(m_s - M), out = sum_s w_s o_s / sum_s w_s l_s and lse = M +
// log2(sum_s w_s l_s), the splits added in split order (deterministic).
__global__ __launch_bounds__(256) void attn_split_combine_kernel(AttnArgs a, int B, int Hkv) {
  const int lane = threadIdx.x & 63;
  const int rows = a.Tq * a.G;
  const int64_t q = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (b, hk, R)
  if (q >= (int64_t)B * Hkv * rows) return;
  const int R = (int)(q % rows);
  const int64_t bh = q / rows;
  const int hk = (int)(bh % Hkv);
  const int b = (int)(bh / Hkv);
  const int ns = a.nsplit;  // <= 64
  const int64_t stride = (int64_t)B * Hkv * rows;  // rows per split
  float ms = -INFINITY, ls = 0.f;
  if (lane < ns) {
    const float2 v = *reinterpret_cast<const float2*>(a.part_ml + (lane * stride + q) * 2);
    ms = v.x;
    ls = v.y;
  }
  float mt = ms;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mt = fmaxf(mt, __shfl_xor(mt, off));
  const float w = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - mt);
  float lt = w * ls;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lt += __shfl_xor(lt, off);
  // eight splits' loads in flight at a time (added in split order); a split
  // with weight 0 holds zeros
  float acc = 0.f;
  const float* po = a.part_o + q * AT_D + lane;
  const int wi = __builtin_bit_cast(int, w);
  int sp = 0;
  for (; sp + 8 <= ns; sp += 8) {
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = po[(sp + j) * stride * AT_D];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += __builtin_bit_cast(float, __builtin_amdgcn_readlane(wi, sp + j)) * x[j];
  }
  for (; sp < ns; ++sp) acc += __builtin_bit_cast(float, __builtin_amdgcn_readlane(wi, sp)) * po[sp * stride * AT_D];
  const float inv = lt > 0.f ? 1.f / lt : 0.f;
  const int t = R / a.G;
  const int h = hk * a.G + (R - t * a.G);
  const __bf16 y = (__bf16)(acc * inv);
  a.out[b * a.sob + (int64_t)t * a.sot + (int64_t)h * a.soh + lane] = __builtin_bit_cast(uint16_t, y);
  if (a.lse && lane == 0) a.lse[((int64_t)b * a.Hq + h) * a.Tq + t] = mt + __builtin_amdgcn_logf(lt);
}

// ---------------------------------------------------------------------------
// Backward (the gradients autograd takes through eager_attention_forward,
// modeling_gpt_oss.py:235-264), from the forward's log2 denominators L:
//   p[t, j]  = 2^(S[t, j] * scaling * log2(e) - L[t])      (visible j, else 0)
//   D[t]     = dO[t] . O[t]       (= sum_j p dP: the sink has no value row)
//   dP[t, j] = dO[t] . v[j],   dS[t, j] = p (dP - D[t])
//   dq[t] = scaling * sum_j dS k[j],  dk[j] = scaling * sum_t dS q[t],
//   dv[j] = sum_t p[t, j] dO[t]
//   d sink[h] = -sum_t p_sink[t] D[t],  p_sink = 2^(sink log2(e) - L[t])
// Two kernels, no atomics: attn_bwd_dq (the forward's row blocks; it also
// writes each row's (L, D) in row order) and attn_bwd_dkv (key blocks, every
// row that sees them, the rows split over workgroups where the key blocks
// alone leave the chip idle; attn_bwd_reduce then adds the shares in order).
// ---------------------------------------------------------------------------
struct AttnBwdArgs {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  const uint16_t* o;    // forward output (strides so)
  const uint16_t* dout; // (strides sd)
  const float* lse;     // [B][Hq][Tq]
  float* stats;         // [B][Hkv][Tq * G][2]: (L, D) of row R, written by attn_bwd_dq
  uint16_t* dq;         // [B, Tq, Hq, 64] contiguous
  uint16_t* dk;         // [B, Tk, Hkv, 64] contiguous
  uint16_t* dv;
  int64_t sqb, sqt, sqh, skb, skt, skh, svb, svt, svh, sob, sot, soh, sdb, sdt, sdh;
  int B, Tq, Tk, Hq, Hkv, G;
  int causal, window;
  int rblocks;          // row blocks of 128
  float scale2, scaling;
  // dk/dv: workgroup x = key block * nsplit + split takes a contiguous share
  // of the rows that see the block; with nsplit > 1 it writes its unscaled
  // float32 sums to part at ((split * 2 + which) * B + b) * Hkv + hk, key, d
  // (which: 0 dk, 1 dv) and attn_bwd_reduce_kernel adds the splits in order
  int nsplit;
  float* part;
};

// 16 bf16 of a u32x4 pair -> float dot with another pair
__device__ __forceinline__ float at_dot8(const u32x4_t& x, const u32x4_t& y) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    s += __uint_as_float(x[i] << 16) * __uint_as_float(y[i] << 16) +
         __uint_as_float(x[i] & 0xFFFF0000u) * __uint_as_float(y[i] & 0xFFFF0000u);
  return s;
}

// dq: the forward's row blocks and K/V tile ring.  Per tile: S^T = K Q^T and
// dP^T = V dO^T (K and V rows permuted), dS^T in registers, dq^T += K^T dS^T
// (K^T by transposing reads of the K tile).
template <bool MASK, int KB0, int KB1>
__device__ __forceinline__ void at_dq_tile(const uint8_t* K, const uint32_t (&koff)[4], const uint32_t (&toff)[2][2],
                                           const u32x4_t (&qf)[4], const u32x4_t (&df)[4], int j0, int lo, int hi,
                                           int g, float scale2, float L, float D, f32x16_t (&dq)[2]) {
  const uint8_t* V = K + AT_TILE;
#pragma unroll
  for (int kb = KB0; kb <= KB1; ++kb) {
    f32x16_t sc, dp;
#pragma unroll
    for (int v = 0; v < 16; ++v) sc[v] = dp[v] = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      sc = at_mfma(*reinterpret_cast<const u32x4_t*>(K + koff[s] + 4096 * kb), qf[s], sc);
      dp = at_mfma(*reinterpret_cast<const u32x4_t*>(V + koff[s] + 4096 * kb), df[s], dp);
    }
    uint32_t vis = 0;
    if constexpr (MASK) vis = at_vis(lo, hi, j0 + 32 * kb, g);
    u32x4_t sf[2];  // dS^T operands of the two 16-key steps
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      float ds[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int v = 8 * half + i;
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[v], scale2, -L));
        if constexpr (MASK) p = __uint_as_float(__float_as_uint(p) & at_vis_mask(vis, v));
        ds[i] = p * (dp[v] - D);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) sf[half][i] = at_pack2(ds[2 * i], ds[2 * i + 1]);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int db = 0; db < 2; ++db)
        dq[db] = at_mfma(at_tr8(K + 2048 * (2 * kb + s), toff[db][0], toff[db][1]), sf[s], dq[db]);
  }
}

// 4096 causal tokens, 64/8 heads: 295 -> 204 us; 8192 with a 128-key window 100
// -> 67 us (the forward's changes).
__global__ __launch_bounds__(256, 3) void attn_bwd_dq_kernel(AttnBwdArgs a) {
  extern __shared__ __align__(1024) uint8_t at_smem[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31;
  const int g = lane >> 5;
  const AtBlock blk = at_block(a.B, a.Hkv);
  const int rb = a.rblocks - 1 - blk.x;
  const int hk = blk.hk;
  const int b = blk.b;
  const AtRows rw = at_rows(a.Tq, a.Tk, a.G, a.causal, a.window, rb, hk, wave, c);

  const uint16_t* qrow = a.q + b * a.sqb + (int64_t)rw.t * a.sqt + (int64_t)rw.h * a.sqh;
  const uint16_t* drow = a.dout + b * a.sdb + (int64_t)rw.t * a.sdt + (int64_t)rw.h * a.sdh;
  const uint16_t* orow = a.o + b * a.sob + (int64_t)rw.t * a.sot + (int64_t)rw.h * a.soh;
  u32x4_t qf[4], df[4], of[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    qf[s] = *reinterpret_cast<const u32x4_t*>(qrow + 16 * s + 8 * g);
    df[s] = *reinterpret_cast<const u32x4_t*>(drow + 16 * s + 8 * g);
    of[s] = *reinterpret_cast<const u32x4_t*>(orow + 16 * s + 8 * g);
  }
  float L = a.lse[((int64_t)b * a.Hq + rw.h) * a.Tq + rw.t];

  AtSrc ks = at_src(a.k + b * a.skb + (int64_t)hk * a.skh, a.skt, rw.kt0, wave, lane);
  AtSrc vs = at_src(a.v + b * a.svb + (int64_t)hk * a.svh, a.svt, rw.kt0, wave, lane);
  const uint32_t lds0 = at_lds(at_smem) + 1024 * wave;
  auto issue = [&](int kt) {
    const uint32_t st = lds0 + (kt % AT_NS) * (2 * AT_TILE);
    at_dma_tile(ks, kt * AT_BC, a.Tk, st, wave, lane);
    at_dma_tile(vs, kt * AT_BC, a.Tk, st + AT_TILE, wave, lane);
  };
  constexpr int DPT = 4;
  for (int i = 0; i < AT_NS - 1; ++i)
    if (rw.kt0 + i < rw.kt1) issue(rw.kt0 + i);

  float D = 0.f;
#pragma unroll
  for (int s = 0; s < 4; ++s) D += at_dot8(df[s], of[s]);
  D = at_add32(D);
  if (g == 0 && rw.R0 + 32 * wave + c < rw.rows) {
    const float2 st2 = {L, D};
    *reinterpret_cast<float2*>(a.stats + (((int64_t)b * a.Hkv + hk) * rw.rows + rw.R) * 2) = st2;
  }
  uint32_t koff[4], toff[2][2];
#pragma unroll
  for (int s = 0; s < 4; ++s) koff[s] = at_off(at_pi(c), 2 * s + g);
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int h = 0; h < 2; ++h) toff[db][h] = at_tr_off(lane, 0, h, db);

  f32x16_t dq[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) dq[db][v] = 0.f;
  // the loads above land here, not inside the loop (see the forward)
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    asm volatile("" : "+v"(qf[s]));
    asm volatile("" : "+v"(df[s]));
  }
  asm volatile("" : "+v"(L));

  auto turn = [&](int kt) {
    wait_vmcnt_tiles<DPT, AT_NS - 2>(rw.kt1 - 1 - kt);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (kt + AT_NS - 1 < rw.kt1) issue(kt + AT_NS - 1);
  };
  auto masked = [&](int kt0, int kt1) {
    for (int kt = kt0; kt < kt1; ++kt) {
      turn(kt);
      const uint8_t* K = at_smem + (kt % AT_NS) * (2 * AT_TILE);
      const int j0 = kt * AT_BC;
      const bool live0 = rw.live_wave && j0 < rw.whi1 && j0 + 32 > rw.wlo0;
      const bool live1 = rw.live_wave && j0 + 32 < rw.whi1 && j0 + 64 > rw.wlo0;
      if (live0) at_dq_tile<true, 0, 0>(K, koff, toff, qf, df, j0, rw.lo, rw.hi, g, a.scale2, L, D, dq);
      if (live1) at_dq_tile<true, 1, 1>(K, koff, toff, qf, df, j0, rw.lo, rw.hi, g, a.scale2, L, D, dq);
    }
  };
  // the forward's three runs of tiles
  masked(rw.kt0, rw.ktf0);
  for (int kt = rw.ktf0; kt < rw.ktf1; ++kt) {
    turn(kt);
    if (rw.live_wave)
      at_dq_tile<false, 0, 1>(at_smem + (kt % AT_NS) * (2 * AT_TILE), koff, toff, qf, df, 0, 0, 0, g, a.scale2, L, D, dq);
  }
  masked(rw.ktf1, rw.kt1);

  if (rw.R0 + 32 * wave + c >= rw.rows) return;
  at_store_row(a.dq + (((int64_t)b * a.Tq + rw.t) * a.Hq + rw.h) * AT_D, dq, a.scaling, g);
}

constexpr int AT_KB = 128;  // keys per dk/dv block (32 per wave)
constexpr int AT_RT = 32;   // rows per step of the dk/dv loop (a unit)
constexpr int AT_DKV_TILE = AT_RT * AT_D * 2;
constexpr int AT_DKV_STAGE = 2 * AT_DKV_TILE + 256;  // q tile, dO tile, (L, D) of the rows
constexpr int AT_DKV_NS = 4;                         // ring stages (3 and 6 measured within 2 %)
constexpr int AT_DKV_LDS = AT_DKV_NS * AT_DKV_STAGE;

// One unit of dk/dv for one wave: S = Q K^T and dP = dO V^T (register v: row 8g
// + v or 16 + 8g + v - 8 of the unit, key c), P and dS in registers, dv^T +=
// dO^T P and dk^T += q^T dS (A operands by transposing reads).
__device__ __forceinline__ void at_dkv_unit(const uint8_t* T, bool full, uint32_t vis, const uint32_t (&aoff)[4],
                                            const uint32_t (&toff)[2][2], const u32x4_t (&kf)[4],
                                            const u32x4_t (&vf)[4], int g, float scale2, f32x16_t (&dk)[2],
                                            f32x16_t (&dv)[2]) {
  const uint8_t* DO = T + AT_DKV_TILE;
  const float* ST = reinterpret_cast<const float*>(T + 2 * AT_DKV_TILE);
  f32x16_t sc, dp;
#pragma unroll
  for (int v = 0; v < 16; ++v) sc[v] = dp[v] = 0.f;
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    sc = at_mfma(*reinterpret_cast<const u32x4_t*>(T + aoff[s]), kf[s], sc);
    dp = at_mfma(*reinterpret_cast<const u32x4_t*>(DO + aoff[s]), vf[s], dp);
  }
  u32x4_t pf[2], sf[2];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    float p[8], ds[8];
#pragma unroll
    for (int i2 = 0; i2 < 4; ++i2) {
      const f32x4_t sd = *reinterpret_cast<const f32x4_t*>(ST + 2 * (16 * half + 8 * g + 2 * i2));  // (L, D) of two rows
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const int i = 2 * i2 + e;
        p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[8 * half + i], scale2, -sd[2 * e]));
        ds[i] = p[i] * (dp[8 * half + i] - sd[2 * e + 1]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      pf[half][i] = at_pack2(p[2 * i], p[2 * i + 1]);
      sf[half][i] = at_pack2(ds[2 * i], ds[2 * i + 1]);
    }
  }
  // Hidden P and dS to 0, as packed pairs: whatever the scaling's sign and
  // whatever (L, D) a row has, nothing of it reaches a key it does not see.
  if (!full) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t lo = at_vis_mask(vis, 8 * half + 2 * i), hi = at_vis_mask(vis, 8 * half + 2 * i + 1);
        const uint32_t k = (lo & 0xFFFFu) | (hi & 0xFFFF0000u);
        pf[half][i] &= k;
        sf[half][i] &= k;
      }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      dv[db] = at_mfma(at_tr8(DO + 2048 * s, toff[db][0], toff[db][1]), pf[s], dv[db]);
      dk[db] = at_mfma(at_tr8(T + 2048 * s, toff[db][0], toff[db][1]), sf[s], dk[db]);
    }
}

// dk, dv: key blocks of 128 keys of one (batch, key head); wave w keeps keys
// 32 w .. 32 w + 31 (their k and v rows as the B operands of S = Q K^T and dP =
// dO V^T, lane c = key c).  The workgroup walks its share of the rows that
// see one of its keys (R = t * G + i as in the forward) in units of 32,
// through a DMA ring: the q and dO tiles (rows permuted as A operands;
// q^T and dO^T by transposing reads for dv^T += dO^T P and dk^T += q^T dS) and
// the rows' (L, D).  Four waves with no common keys keep no sums to add at the
// end, and at 167 registers three workgroups share a CU, out of step with each
// other: one's MFMAs run under another's exponentials, where the eight waves
// of one workgroup met at the same barrier.  4096 causal tokens, 64/8 heads:
// 928 -> 325 us (of it the row splits 2x); 8192 with a 128-key window 228 ->
// 86 us.
__global__ __launch_bounds__(256, 3) void attn_bwd_dkv_kernel(AttnBwdArgs a) {
  extern __shared__ __align__(1024) uint8_t at_smem[];  // AT_DKV_NS stages
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c = lane & 31;
  const int g = lane >> 5;
  const AtBlock blk = at_block(a.B, a.Hkv);
  const int hk = blk.hk;
  const int b = blk.b;
  const int rows = a.Tq * a.G;
  const int off = a.Tk - a.Tq;  // position of query 0
  const uint16_t* qbase = a.q + b * a.sqb + (int64_t)hk * a.G * a.sqh;
  const uint16_t* dbase = a.dout + b * a.sdb + (int64_t)hk * a.G * a.sdh;
  const float* sbase = a.stats + ((int64_t)b * a.Hkv + hk) * rows * 2;

  // blocks in index order: under a causal mask the first have the most rows
  const int j0 = blk.x / a.nsplit * AT_KB;
  const int sp = blk.x % a.nsplit;
  // rows [first, end) that see key j
  auto row_first = [&](int j) { return a.causal ? max(0, j - off) * a.G : 0; };
  auto row_end = [&](int j) { return a.causal && a.window > 0 ? min(a.Tq, max(0, j + a.window - off)) * a.G : rows; };
  const int jlast = min(j0 + AT_KB, a.Tk) - 1;
  int r_begin = row_first(j0);
  const int r_end = max(r_begin, row_end(jlast));
  int nt = (r_end - r_begin + AT_RT - 1) / AT_RT;
  {
    const int per = (nt + a.nsplit - 1) / a.nsplit;
    const int t0 = min(nt, sp * per);
    nt = min(nt, t0 + per) - t0;
    r_begin += t0 * AT_RT;
  }

  const int jk = j0 + 32 * wave + c;
  const int jc = min(jk, a.Tk - 1);
  const uint16_t* krow = a.k + b * a.skb + (int64_t)jc * a.skt + (int64_t)hk * a.skh;
  const uint16_t* vrow = a.v + b * a.svb + (int64_t)jc * a.svt + (int64_t)hk * a.svh;
  u32x4_t kf[4], vf[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    kf[s] = *reinterpret_cast<const u32x4_t*>(krow + 16 * s + 8 * g);
    vf[s] = *reinterpret_cast<const u32x4_t*>(vrow + 16 * s + 8 * g);
  }
  // this lane's key is seen by rows [rlo, rhi), the wave's keys by all of
  // [wfull0, wfull1) and by none outside [wlive0, wlive1)
  const int rlo = row_first(jk), rhi = jk < a.Tk ? row_end(jk) : 0;
  const int jw0 = j0 + 32 * wave, jw1 = jw0 + 31;
  const int wfull0 = row_first(jw1), wfull1 = jw1 < a.Tk ? row_end(jw0) : 0;
  const int wlive0 = row_first(jw0), wlive1 = jw0 < a.Tk ? row_end(min(jw1, a.Tk - 1)) : 0;

  // A operands: rows pi(c) at d chunk 2s + g; transposing reads of d block db
  // (16-row step s adds 2048, halves h)
  uint32_t aoff[4], toff[2][2];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = at_off(at_pi(c), 2 * s + g);
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int h = 0; h < 2; ++h) toff[db][h] = at_tr_off(lane, 0, h, db);

  // Unit i: wave w fills rows 8w + lane / 8 of the q and dO tiles (source row
  // t = R / G, head R % G of the group); every wave writes the same 256 bytes
  // of (L, D).  Rows past the last repeat it.  r_begin is a multiple of G, so
  // when G divides the unit a row's head and its query within the unit do not
  // depend on the unit: a uniform base moves.
  const uint32_t lds0 = at_lds(at_smem);
  const int drow = 8 * wave + (lane >> 3);
  const int ch16 = ((lane & 7) ^ at_sw(drow)) * 16;
  const bool even = AT_RT % a.G == 0 && a.sqt <= AT_NEAR / 2 && a.sdt <= AT_NEAR / 2 && a.sqh <= AT_NEAR / 2 &&
                    a.sdh <= AT_NEAR / 2;
  const int tq = AT_RT / a.G;  // queries per unit when even
  const int64_t qstep = tq * a.sqt, dstep = tq * a.sdt;
  const uint16_t* qnext = qbase + (int64_t)(r_begin / a.G) * a.sqt;
  const uint16_t* dnext = dbase + (int64_t)(r_begin / a.G) * a.sdt;
  uint32_t qoff, doff;
  {
    const int tl = drow / a.G, hl = drow - tl * a.G;
    qoff = 2u * ((uint32_t)tl * (uint32_t)a.sqt + (uint32_t)hl * (uint32_t)a.sqh) + ch16;
    doff = 2u * ((uint32_t)tl * (uint32_t)a.sdt + (uint32_t)hl * (uint32_t)a.sdh) + ch16;
  }
  int irow = r_begin;            // first row of the next unit to fetch
  uint32_t ist = lds0;           // its stage
  auto issue = [&]() {
    if (even && irow + AT_RT <= rows) {
      at_dma16(qnext, qoff, ist + 1024 * wave);
      at_dma16(dnext, doff, ist + AT_DKV_TILE + 1024 * wave);
      at_dma4(sbase + 2 * (int64_t)irow, 4 * lane, ist + 2 * AT_DKV_TILE);
    } else {
      const int R = min(irow + drow, rows - 1);
      const int t = R / a.G;
      const int h = R - t * a.G;
      at_dma16(reinterpret_cast<const uint8_t*>(qbase + (int64_t)t * a.sqt + (int64_t)h * a.sqh) + ch16,
               ist + 1024 * wave);
      at_dma16(reinterpret_cast<const uint8_t*>(dbase + (int64_t)t * a.sdt + (int64_t)h * a.sdh) + ch16,
               ist + AT_DKV_TILE + 1024 * wave);
      at_dma4(sbase + 2 * (int64_t)min(irow, rows - 1),
              8 * min(lane >> 1, max(rows - 1 - irow, 0)) + 4 * (lane & 1), ist + 2 * AT_DKV_TILE);
    }
    irow += AT_RT;
    qnext += qstep;
    dnext += dstep;
    ist = ist + AT_DKV_STAGE == lds0 + AT_DKV_LDS ? lds0 : ist + AT_DKV_STAGE;
  };
  constexpr int DPT = 3;

  f32x16_t dk[2], dv[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int v = 0; v < 16; ++v) dk[db][v] = dv[db][v] = 0.f;

  for (int i = 0; i < AT_DKV_NS - 1; ++i)
    if (i < nt) issue();
  // the k and v loads land here, not inside the loop (see the forward)
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    asm volatile("" : "+v"(kf[s]));
    asm volatile("" : "+v"(vf[s]));
  }

  const uint8_t* T = at_smem;  // unit u's stage
  for (int u = 0; u < nt; ++u) {
    // unit u has landed; the barrier certifies every wave's reads of unit u -
    // 1 are done, whose stage takes unit u + AT_DKV_NS - 1
    wait_vmcnt_tiles<DPT, AT_DKV_NS - 2>(nt - 1 - u);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (u + AT_DKV_NS - 1 < nt) issue();
    const int r0 = r_begin + u * AT_RT;
    if (r0 + AT_RT > wlive0 && r0 < wlive1)
      at_dkv_unit(T, r0 >= wfull0 && r0 + AT_RT <= wfull1, at_vis(rlo, rhi, r0, g), aoff, toff, kf, vf, g, a.scale2,
                  dk, dv);
    T = T + AT_DKV_STAGE == at_smem + AT_DKV_LDS ? (const uint8_t*)at_smem : T + AT_DKV_STAGE;
  }

  if (jk < a.Tk) {
    if (a.nsplit > 1) {
#pragma unroll
      for (int which = 0; which < 2; ++which) {
        const f32x16_t* acc = which == 0 ? dk : dv;
        float* po = a.part + ((((int64_t)(sp * 2 + which) * a.B + b) * a.Hkv + hk) * a.Tk + jk) * AT_D;
#pragma unroll
        for (int db = 0; db < 2; ++db)
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4)
            *reinterpret_cast<f32x4_t*>(po + 32 * db + 8 * q4 + 4 * g) =
                f32x4_t{acc[db][4 * q4], acc[db][4 * q4 + 1], acc[db][4 * q4 + 2], acc[db][4 * q4 + 3]};
      }
      return;
    }
    const int64_t orow = (((int64_t)b * a.Tk + jk) * a.Hkv + hk) * AT_D;
    at_store_row(a.dk + orow, dk, a.scaling, g);
    at_store_row(a.dv + orow, dv, 1.f, g);
  }
}

// dk and dv from the row splits' sums, added in split order; one thread per
// four columns of one key of one head (blockIdx.z: dk, dv).
__global__ __launch_bounds__(256) void attn_bwd_reduce_kernel(AttnBwdArgs a, int B) {
  const int64_t n4 = (int64_t)B * a.Hkv * a.Tk * (AT_D / 4);
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const int which = blockIdx.z;
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(a.part) + which * n4 + i;
  f32x4_t s = *p;
  for (int k = 1; k < a.nsplit; ++k) s += p[2 * n4 * k];
  const float f = which == 0 ? a.scaling : 1.f;
  const int64_t row = i / (AT_D / 4);  // (b, hk, key)
  const int64_t bh = row / a.Tk;
  const int64_t key = row - bh * a.Tk;
  const int64_t b = bh / a.Hkv;
  uint16_t* out = (which == 0 ? a.dk : a.dv) + ((b * a.Tk + key) * a.Hkv + (bh - b * a.Hkv)) * AT_D + (i % (AT_D / 4)) * 4;
  uint2 w;
  w.x = at_pack2(s[0] * f, s[1] * f);
  w.y = at_pack2(s[2] * f, s[3] * f);
  *reinterpret_cast<uint2*>(out) = w;
}

constexpr int AT_FWD_LDS = AT_NS * 2 * AT_TILE;

static int at_allow_lds(const void* fn, int idx, int bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    set_error("no current HIP device");
    return BSA_EHIP;
  }
  static bool done[64][3];
  if (!done[dev][idx]) {
    if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
      set_error("attention: cannot allow %d bytes of LDS", bytes);
      return BSA_EHIP;
    }
    done[dev][idx] = true;
  }
  return BSA_OK;
}

static int at_check_common(const char* what, int64_t B, int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv,
                           int64_t head_dim, int causal, int64_t window) {
  BSA_REQUIRE(head_dim == AT_D, "%s: head_dim must be %d (got %lld)", what, AT_D, (long long)head_dim);
  BSA_REQUIRE(Hq % Hkv == 0 && Hq / Hkv <= 64, "%s: Hq (%lld) must be a multiple of Hkv (%lld), at most 64x", what,
              (long long)Hq, (long long)Hkv);
  BSA_REQUIRE(window >= 0 && (window == 0 || causal), "%s: a window needs the causal mask", what);
  BSA_REQUIRE(!causal || Tq <= Tk, "%s: causal with more queries (%lld) than keys (%lld)", what, (long long)Tq,
              (long long)Tk);
  BSA_REQUIRE(B < 65536 && Hkv < 65536 && Tq * (Hq / Hkv) < INT32_MAX / 2 && Tk < INT32_MAX / 2 && window < INT32_MAX,
              "%s: too large", what);
  return BSA_OK;
}

// A window that reaches past every key hides none: 0 (no window), which also
// keeps key + window within 32 bits.
static int at_window(int64_t window, int64_t Tk) { return window >= Tk ? 0 : (int)window; }

static int at_check_strides(const char* what, const int64_t* const* st, int n) {
  for (int j = 0; j < n; ++j)
    for (int i = 0; i < 3; ++i)
      BSA_REQUIRE(st[j][i] % 8 == 0 && st[j][i] >= 0,
                  "%s: strides (batch, sequence, head) must be non-negative multiples of 8 elements", what);
  return BSA_OK;
}

static inline bool at_al16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

// Key splits of the forward for a shape: enough workgroups for the chip
// (about AT_SPLIT_TARGET in all) when the (row block, key head, batch) grid
// alone is short of it and a row block sees at least AT_SPLIT_MIN_TILES key
// tiles; at least two tiles per split, at most 64 splits.  A function of the
// shape only, so results do not depend on the device.
#ifndef BSA_AT_SPLIT_TARGET
#define BSA_AT_SPLIT_TARGET 512
#endif
constexpr int64_t AT_SPLIT_TARGET = BSA_AT_SPLIT_TARGET;
constexpr int64_t AT_SPLIT_MIN_TILES = 8;
static int at_split_count(int64_t B, int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv, int causal, int64_t window) {
  if (B <= 0 || Tq <= 0 || Tk <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv) return 1;
  const int64_t G = Hq / Hkv;
  const int64_t base = (Tq * G + AT_BR - 1) / AT_BR * Hkv * B;
  if (base >= AT_SPLIT_TARGET) return 1;
  // key tiles of the row block that sees the most keys
  const int64_t keys = causal && window > 0 ? std::min<int64_t>(Tk, window + std::min<int64_t>(Tq, AT_BR)) : Tk;
  const int64_t tiles = (keys + AT_BC - 1) / AT_BC + (causal && window > 0 ? 1 : 0);
  if (tiles < AT_SPLIT_MIN_TILES) return 1;  // the merge launch costs more than a short range saves
  int64_t n = std::min<int64_t>((AT_SPLIT_TARGET + base - 1) / base, tiles / 2);
  n = std::min<int64_t>(n, 64);
  return n >= 2 ? (int)n : 1;
}

// Workspace layout of the key-split forward: part_o, then part_ml at a
// 256-byte boundary.
static int64_t at_split_bytes(int64_t nsplit, int64_t B, int64_t Tq, int64_t Hq) {
  if (nsplit <= 1) return 0;
  const int64_t rows = nsplit * B * Hq * Tq;  // = nsplit * B * Hkv * (Tq * G)
  const int64_t o = (rows * AT_D * 4 + 255) / 256 * 256;
  return o + (rows * 2 * 4 + 255) / 256 * 256;
}

// Shared checks and arguments of the two forward entry points.
static int at_fwd_args(AttnArgs& a, const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                       const void* v, const int64_t* v_strides, const float* sinks, int64_t B, int64_t Tq,
                       int64_t Tk, int64_t Hq, int64_t Hkv, int64_t head_dim, int causal, int64_t window,
                       float scaling, void* out, const int64_t* out_strides, float* lse) {
  BSA_REQUIRE(Tk > 0, "attention: queries without keys");
  BSA_REQUIRE(q && k && v && out && q_strides && k_strides && v_strides && out_strides, "attention: null pointer");
  int rc = at_check_common("attention", B, Tq, Tk, Hq, Hkv, head_dim, causal, window);
  if (rc) return rc;
  BSA_REQUIRE(at_al16(q) && at_al16(k) && at_al16(v) && at_al16(out), "attention: q, k, v and out must be 16-byte aligned");
  const int64_t* st[4] = {q_strides, k_strides, v_strides, out_strides};
  if ((rc = at_check_strides("attention", st, 4))) return rc;
  a = AttnArgs{};
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.sinks = sinks;
  a.out = static_cast<uint16_t*>(out);
  a.lse = lse;
  a.sqb = q_strides[0], a.sqt = q_strides[1], a.sqh = q_strides[2];
  a.skb = k_strides[0], a.skt = k_strides[1], a.skh = k_strides[2];
  a.svb = v_strides[0], a.svt = v_strides[1], a.svh = v_strides[2];
  a.sob = out_strides[0], a.sot = out_strides[1], a.soh = out_strides[2];
  a.B = (int)B;
  a.Tq = (int)Tq;
  a.Tk = (int)Tk;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.G = (int)(Hq / Hkv);
  a.causal = causal ? 1 : 0;
  a.window = at_window(window, Tk);
  a.scale2 = scaling * 1.4426950408889634f;
  a.nsplit = 1;
  return BSA_OK;
}

// The grid of n workgroups for each of B * Hkv pairs (at_block).
static dim3 at_grid(int64_t n, int64_t B, int64_t Hkv) {
  if (n * Hkv * B < (int64_t(1) << 23)) return dim3((unsigned)(n * Hkv * B));
  return dim3((unsigned)n, (unsigned)Hkv, (unsigned)B);
}

static int at_fwd_launch(AttnArgs& a, int64_t B, int64_t Hkv, hipStream_t st) {
  const int64_t rblocks = ((int64_t)a.Tq * a.G + AT_BR - 1) / AT_BR;
  a.rblocks = (int)rblocks;
  int rc = at_allow_lds(reinterpret_cast<const void*>(attn_fwd_kernel), 0, AT_FWD_LDS);
  if (rc) return rc;
  hipLaunchKernelGGL(attn_fwd_kernel, at_grid(rblocks * a.nsplit, B, Hkv), dim3(256),
                     AT_FWD_LDS, st, a);
  BSA_LAUNCH_CHECK("attention launch");
  if (a.nsplit > 1) {
    const int64_t nrow = B * Hkv * (int64_t)a.Tq * a.G;
    hipLaunchKernelGGL(attn_split_combine_kernel, dim3((unsigned)((nrow + 3) / 4)), dim3(256), 0, st, a, (int)B,
                       (int)Hkv);
    BSA_LAUNCH_CHECK("attention split combine launch");
  }
  return BSA_OK;
}

}  // namespace bsa

using namespace bsa;

extern "C" int bsa_attention_fwd(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                                 const void* v, const int64_t* v_strides, const float* sinks, int64_t B,
                                 int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv, int64_t head_dim, int causal,
                                 int64_t window, float scaling, void* out, const int64_t* out_strides, float* lse,
                                 void* stream) {
  clear_error();
  BSA_REQUIRE(B >= 0 && Tq >= 0 && Tk >= 0 && Hq > 0 && Hkv > 0, "attention: bad shape");
  if (B == 0 || Tq == 0) return BSA_OK;
  AttnArgs a;
  int rc = at_fwd_args(a, q, q_strides, k, k_strides, v, v_strides, sinks, B, Tq, Tk, Hq, Hkv, head_dim, causal,
                       window, scaling, out, out_strides, lse);
  if (rc) return rc;
  return at_fwd_launch(a, B, Hkv, static_cast<hipStream_t>(stream));
}

extern "C" int64_t bsa_attention_split_workspace_bytes(int64_t B, int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv,
                                                       int causal, int64_t window) {
  return at_split_bytes(at_split_count(B, Tq, Tk, Hq, Hkv, causal, window), B, Tq, Hq);
}

extern "C" int bsa_attention_fwd_split(const void* q, const int64_t* q_strides, const void* k,
                                       const int64_t* k_strides, const void* v, const int64_t* v_strides,
                                       const float* sinks, int64_t B, int64_t Tq, int64_t Tk, int64_t Hq,
                                       int64_t Hkv, int64_t head_dim, int causal, int64_t window, float scaling,
                                       void* out, const int64_t* out_strides, float* lse, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  clear_error();
  BSA_REQUIRE(B >= 0 && Tq >= 0 && Tk >= 0 && Hq > 0 && Hkv > 0, "attention: bad shape");
  if (B == 0 || Tq == 0) return BSA_OK;
  AttnArgs a;
  int rc = at_fwd_args(a, q, q_strides, k, k_strides, v, v_strides, sinks, B, Tq, Tk, Hq, Hkv, head_dim, causal,
                       window, scaling, out, out_strides, lse);
  if (rc) return rc;
  const int ns = at_split_count(B, Tq, Tk, Hq, Hkv, causal, window);
  if (ns > 1) {
    const int64_t need = at_split_bytes(ns, B, Tq, Hq);
    BSA_REQUIRE(workspace && reinterpret_cast<uintptr_t>(workspace) % 256 == 0 && workspace_bytes >= need,
                "attention: the key-split forward needs a 256-byte aligned workspace of %lld bytes (got %lld)",
                (long long)need, (long long)workspace_bytes);
    const int64_t rows = (int64_t)ns * B * Hq * Tq;
    a.nsplit = ns;
    a.part_o = static_cast<float*>(workspace);
    a.part_ml = reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + (rows * AT_D * 4 + 255) / 256 * 256);
  }
  return at_fwd_launch(a, B, Hkv, static_cast<hipStream_t>(stream));
}

// Row splits of dk/dv for a shape: enough workgroups for the 768 that the
// chip holds, a share keeping at least AT_BWD_SPLIT_MIN_UNITS units (its
// float32 sums, written and read once more, cost about as much as six).
// Under a causal mask without a window the blocks' lengths fall linearly and
// the longest share bounds the tail, so the grid aims higher, the more so
// where shares stay long.  Measured (64/8 heads, whole backward, 1 / 2 / 4 / 8 /
// 16 splits): causal 8192 - / 2000 / 1846 / 1858 / - us, causal 4096 - / 700 /
// 517 / 504 / 541 us, causal 2048 - / - / 203 / 163 / 184 us, 8192 with a
// 128-key window 160 / 179 / 194 us.  A function of the shape only, so results
// do not depend on the device.
constexpr int64_t AT_BWD_SPLIT_MIN_UNITS = 16;
static int at_bwd_split_count(int64_t B, int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv, int causal, int64_t window) {
  if (B <= 0 || Tq <= 0 || Tk <= 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv) return 1;
  const int64_t base = (Tk + AT_KB - 1) / AT_KB * Hkv * B;
  const int64_t queries = causal && window > 0 ? std::min<int64_t>(Tq, window + AT_KB) : Tq;
  const int64_t units = (queries * (Hq / Hkv) + AT_RT - 1) / AT_RT;  // of the longest block
  const int64_t target = !(causal && window == 0) ? 512 : (units >= 1024 ? 2048 : 1024);
  const int64_t n = std::min<int64_t>({(target + base - 1) / base, units / AT_BWD_SPLIT_MIN_UNITS, 32});
  return n >= 2 ? (int)n : 1;
}

static int64_t at_bwd_split_bytes(int64_t nsplit, int64_t B, int64_t Tk, int64_t Hkv) {
  return nsplit <= 1 ? 0 : nsplit * 2 * B * Hkv * Tk * AT_D * 4;
}

extern "C" int64_t bsa_attention_bwd_workspace_bytes(int64_t B, int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv,
                                                     int causal, int64_t window) {
  return at_bwd_split_bytes(at_bwd_split_count(B, Tq, Tk, Hq, Hkv, causal, window), B, Tk, Hkv);
}

static int at_bwd(const void* grad_out, const int64_t* grad_strides, const void* q, const int64_t* q_strides,
                  const void* k, const int64_t* k_strides, const void* v, const int64_t* v_strides, const void* out,
                  const int64_t* out_strides, const float* lse, int64_t B, int64_t Tq, int64_t Tk, int64_t Hq,
                  int64_t Hkv, int64_t head_dim, int causal, int64_t window, float scaling, void* grad_q,
                  void* grad_k, void* grad_v, float* row_stats, int nsplit, float* part, void* stream) {
  BSA_REQUIRE(B >= 0 && Tq >= 0 && Tk >= 0 && Hq > 0 && Hkv > 0, "attention bwd: bad shape");
  if (B == 0 || Tq == 0 || Tk == 0) return BSA_OK;
  BSA_REQUIRE(grad_out && q && k && v && out && lse && grad_q && grad_k && grad_v && row_stats && grad_strides &&
                  q_strides && k_strides && v_strides && out_strides,
              "attention bwd: null pointer");
  int rc = at_check_common("attention bwd", B, Tq, Tk, Hq, Hkv, head_dim, causal, window);
  if (rc) return rc;
  BSA_REQUIRE(at_al16(grad_out) && at_al16(q) && at_al16(k) && at_al16(v) && at_al16(out) && at_al16(grad_q) &&
                  at_al16(grad_k) && at_al16(grad_v) && at_al16(row_stats),
              "attention bwd: tensors must be 16-byte aligned");
  const int64_t* st[5] = {grad_strides, q_strides, k_strides, v_strides, out_strides};
  if ((rc = at_check_strides("attention bwd", st, 5))) return rc;
  AttnBwdArgs a{};
  a.q = static_cast<const uint16_t*>(q);
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint16_t*>(v);
  a.o = static_cast<const uint16_t*>(out);
  a.dout = static_cast<const uint16_t*>(grad_out);
  a.lse = lse;
  a.stats = row_stats;
  a.dq = static_cast<uint16_t*>(grad_q);
  a.dk = static_cast<uint16_t*>(grad_k);
  a.dv = static_cast<uint16_t*>(grad_v);
  a.sdb = grad_strides[0], a.sdt = grad_strides[1], a.sdh = grad_strides[2];
  a.sqb = q_strides[0], a.sqt = q_strides[1], a.sqh = q_strides[2];
  a.skb = k_strides[0], a.skt = k_strides[1], a.skh = k_strides[2];
  a.svb = v_strides[0], a.svt = v_strides[1], a.svh = v_strides[2];
  a.sob = out_strides[0], a.sot = out_strides[1], a.soh = out_strides[2];
  a.B = (int)B;
  a.Tq = (int)Tq;
  a.Tk = (int)Tk;
  a.Hq = (int)Hq;
  a.Hkv = (int)Hkv;
  a.G = (int)(Hq / Hkv);
  a.causal = causal ? 1 : 0;
  a.window = at_window(window, Tk);
  a.scale2 = scaling * 1.4426950408889634f;
  a.scaling = scaling;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t rblocks = (Tq * a.G + AT_BR - 1) / AT_BR;
  a.rblocks = (int)rblocks;
  if ((rc = at_allow_lds(reinterpret_cast<const void*>(attn_bwd_dq_kernel), 1, AT_FWD_LDS))) return rc;
  hipLaunchKernelGGL(attn_bwd_dq_kernel, at_grid(rblocks, B, Hkv), dim3(256), AT_FWD_LDS, s, a);
  BSA_LAUNCH_CHECK("attention bwd (dq) launch");
  a.nsplit = nsplit;
  a.part = part;
  const int64_t kgrid = (Tk + AT_KB - 1) / AT_KB * nsplit;
  if ((rc = at_allow_lds(reinterpret_cast<const void*>(attn_bwd_dkv_kernel), 2, AT_DKV_LDS))) return rc;
  hipLaunchKernelGGL(attn_bwd_dkv_kernel, at_grid(kgrid, B, Hkv), dim3(256),
                     AT_DKV_LDS, s, a);
  BSA_LAUNCH_CHECK("attention bwd (dk, dv) launch");
  if (nsplit > 1) {
    const int64_t n4 = B * Hkv * Tk * (AT_D / 4);
    hipLaunchKernelGGL(attn_bwd_reduce_kernel, dim3((unsigned)((n4 + 255) / 256), 1, 2), dim3(256), 0, s, a, (int)B);
    BSA_LAUNCH_CHECK("attention bwd (split sum) launch");
  }
  return BSA_OK;
}

extern "C" int bsa_attention_bwd(const void* grad_out, const int64_t* grad_strides, const void* q,
                                 const int64_t* q_strides, const void* k, const int64_t* k_strides, const void* v,
                                 const int64_t* v_strides, const void* out, const int64_t* out_strides,
                                 const float* lse, int64_t B, int64_t Tq, int64_t Tk, int64_t Hq, int64_t Hkv,
                                 int64_t head_dim, int causal, int64_t window, float scaling, void* grad_q,
                                 void* grad_k, void* grad_v, float* row_stats, void* stream) {
  clear_error();
  return at_bwd(grad_out, grad_strides, q, q_strides, k, k_strides, v, v_strides, out, out_strides, lse, B, Tq, Tk,
                Hq, Hkv, head_dim, causal, window, scaling, grad_q, grad_k, grad_v, row_stats, 1, nullptr, stream);
}

extern "C" int bsa_attention_bwd_split(const void* grad_out, const int64_t* grad_strides, const void* q,
                                       const int64_t* q_strides, const void* k, const int64_t* k_strides,
                                       const void* v, const int64_t* v_strides, const void* out,
                                       const int64_t* out_strides, const float* lse, int64_t B, int64_t Tq,
                                       int64_t Tk, int64_t Hq, int64_t Hkv, int64_t head_dim, int causal,
                                       int64_t window, float scaling, void* grad_q, void* grad_k, void* grad_v,
                                       float* row_stats, void* workspace, int64_t workspace_bytes, void* stream) {
  clear_error();
  const int ns = at_bwd_split_count(B, Tq, Tk, Hq, Hkv, causal, window);
  const int64_t need = at_bwd_split_bytes(ns, B, Tk, Hkv);
  BSA_REQUIRE(need == 0 || (workspace && at_al16(workspace) && workspace_bytes >= need),
              "attention bwd: the row-split backward needs a 16-byte aligned workspace of %lld bytes (got %lld)",
              (long long)need, (long long)workspace_bytes);
  return at_bwd(grad_out, grad_strides, q, q_strides, k, k_strides, v, v_strides, out, out_strides, lse, B, Tq, Tk,
                Hq, Hkv, head_dim, causal, window, scaling, grad_q, grad_k, grad_v, row_stats, ns,
                static_cast<float*>(workspace), stream);
}
