// Pieces shared by the pipelined GDN kernel (gdn.hip) and the prepared-tile kernels (gdn_scan.hip):
// arguments, lane helpers, operand layouts, the tile inverse and the snapshot store.
#pragma once

#include "common.h"

namespace dllm {

struct GdnStream {
  const void* q;
  const void* k;
  const void* v;
  const float* beta;
  const float* g;
  void* out;  // [B, T, Hv, Dv] contiguous
};

struct GdnArgs {
  GdnStream s[2];
  const float* init;  // [B, Hv, Dk, Dv] fp32 or null
  float* states;      // [B, T/chunk, Hv, Dk, Dv] fp32 or null
  long long q_sb, k_sb, v_sb, b_sb, g_sb;  // batch strides (elements)
  int q_st, q_sh, k_st, k_sh, v_st, v_sh, b_st, b_sh, g_st, g_sh;  // token / head strides
  int B, T, Hk, Hv, Dk, Dv;
  int sub;         // real rows per 32-row tile
  int snap_every;  // tiles per chunk
  float scale;     // applied to q after l2norm
  int l2norm;
  int vec_qk;  // q/k rows: 16-byte vector loads (aligned, Dk equal to the kernel width)
  int vec_v;   // v rows: 16-byte vector loads (aligned, Dv a multiple of the column window)
  int spin_limit;  // bounded waits give up (and report through dllm_status) after this many sleeps
  int wait_bias;   // 0; tests set a count the LDS wait never reaches, to exercise the give-up path
  // pipelined fork over a range of blocks: rows and snapshots per sequence of the full out and
  // states tensors (T and T / sub for a whole sequence), and the clean state the range starts
  // from (the snapshot of the block before it, in the states layout; null: zeros)
  int t_rows, snap_rows;
  const float* fork_init;
  // pipelined fork with the v channels' causal conv (width 4) + SiLU in the state waves: the v rows
  // read are the conv's inputs; weights [Hv * Dv, 4] (the v channels' rows; bf16, or fp32 in the
  // kernel's fp32-weight instantiation) and bias [Hv * Dv] of the same dtype, or null. t_first: the
  // sequence row of the launch's first row (the history before sequence row 0 is zero).
  const void* vconv_w;
  const void* vconv_b;
  int t_first;
  // the v channels' conv tails (the clean raw rows before each block, [B * nb, tails_cd, 3] from the
  // first v channel on), or null
  void* vtails;
  int tails_cd;
};

// Linear workgroup id such that consecutive ids run on the same XCD (dispatch is round-robin over
// the 8 XCDs): workgroups sharing a key head then share that XCD's L2.
__device__ __forceinline__ int xcd_linear_id(int bid, int n) {
  const int q = n >> 3, r = n & 7, x = bid & 7, i = bid >> 3;
  return (x < r) ? x * (q + 1) + i : r * (q + 1) + (x - r) * q + i;
}

// Returns x unchanged but opaque to the optimiser, so that uniform addresses derived from it are
// computed where they are used instead of being hoisted out of the tile loop (and spilled).
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+s"(x));
  return x;
}
// The same for a per-lane value: comparisons against it are evaluated where they are used instead
// of being hoisted out of the tile loop as lane masks held in (spilled) scalar registers.
__device__ __forceinline__ int opaque_v(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// DPP move; lanes whose source is outside the row read 0 (bound_ctrl).
template <int CTRL> __device__ __forceinline__ float dpp_mov(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true));
}

// Sum of squares of row l32 of a [32 x 128] bf16 operand held as four rho-ordered fragments (lane
// (l32, h) holds 64 of the row's values): paired bf16 dot products into four fp32 partial sums,
// then the other half of the row from lane l32 + 32 (or l32 - 32), so both lanes get the row total.
__device__ __forceinline__ float row_sumsq(const Frag<true> (&f)[4]) {
  float s[4];
#pragma unroll
  for (int kt = 0; kt < 4; ++kt) {
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bf16x2 lo = {f[kt].lo[2 * i], f[kt].lo[2 * i + 1]};
      const bf16x2 hi = {f[kt].hi[2 * i], f[kt].hi[2 * i + 1]};
      x = __builtin_amdgcn_fdot2_f32_bf16(lo, lo, x, false);
      x = __builtin_amdgcn_fdot2_f32_bf16(hi, hi, x, false);
    }
    s[kt] = x;
  }
  const float half = (s[0] + s[1]) + (s[2] + s[3]);
  // the other half from lane l ^ 32 (LDS crossbar permute); the sum is commutative, so the two
  // lanes of a row hold bit-identical totals
  const float other = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((__lane_id() ^ 32) << 2,
                                                                            __builtin_bit_cast(int, half)));
  return half + other;
}

// Pipelined-kernel operand convention. The state S is held with its rows (d) permuted inside each
// 32-row slice: accumulator row rho(v, h) holds d = 16 h + v. Fed back as a B operand, value v of
// lane (n, h) then carries d = 16 h + v, so every A operand contracted with it (W, Q) is read as 16
// CONSECUTIVE d of its row: two 16-byte LDS reads instead of four 8-byte ones. Products whose two
// operands both come from LDS rows (K K^T, K Q^T) use the same reads for both: the contraction pairs
// equal d whatever the order.
__device__ __forceinline__ void lds_frag_c(const bf16* base, int h, Frag<true>& f) {
  const bf16* p = base + 16 * h;
  f.lo = *(const bf16x8*)p;
  f.hi = *(const bf16x8*)(p + 8);
}
// Transposed read (as lds_frag_tr) whose result lane r = 8 m + 4 h' + e receives column
// 16 h' + 4 m + e of the 32-column slice: an A operand whose product rows come out in the permuted
// d order above. The transpose read hands each group of four result lanes the four consecutive
// columns one source lane addresses, so only the column-group addresses change.
__device__ __forceinline__ void lds_frag_tr_d(const bf16* base, int row_stride, int lane, Frag<true>& f) {
  typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
  const int s = lane & 15, j = s & 3;
  const bf16* p = base + (4 * (lane >> 5) + (s >> 2)) * row_stride + 16 * (j & 1) + 4 * (2 * ((lane >> 4) & 1) + (j >> 1));
  bf16x4 r[4];
#pragma unroll
  for (int m = 0; m < 4; ++m)
    r[m] = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(p + 8 * m * row_stride));
  f.lo = __builtin_shufflevector(r[0], r[1], 0, 1, 2, 3, 4, 5, 6, 7);
  f.hi = __builtin_shufflevector(r[2], r[3], 0, 1, 2, 3, 4, 5, 6, 7);
}

// Row stride (floats) of the [32][32] fp32 scratch of the tile inverse (gdn_inverse.inc).
constexpr int INV_ROW = 36;

// One fp32 element of a state snapshot: a non-temporal store (nothing in the launch reads the
// snapshot back) at device scope, so that the line is written through to memory instead of held
// dirty in the XCD's L2 until the launch ends. Issued as its own instruction, which also keeps the
// compiler from moving the stores among the update's products. Measured at the 27B-class layer:
// the fork 559.6 vs 594.3 us with the compiler's non-temporal store (571.2 us for the same nt
// store issued this way, 562.3 us with system scope), bit-identical; 253.1 vs 259.2 us at the
// 0.8B-class layer.
// OFF: an immediate byte offset from p.
template <int OFF> __device__ __forceinline__ void store_snapshot(float* p, float v) {
  asm volatile("global_store_dword %0, %1, off offset:%2 nt sc1" ::"v"(p), "v"(v), "i"(OFF) : "memory");
}
// The 16 values of one 32-row slice of a state wave's accumulator: rows 32 kt + 16 h + v of the
// snapshot (p0 = row 32 kt + 16 h), 512 bytes apart, as immediate offsets from two base addresses
// (v < 8 and v >= 8) instead of an address formed per store. With the v conv on the state waves
// (whose VALU is then the bound) this measured 604 vs 611 us at the 27B-class fork and 260 vs
// 270 us at the 0.8B-class, bit-identical (before it: 581 vs 561 us, slower).
__device__ __forceinline__ void store_snapshot_slice(float* p0, const f32x16& s) {
  float* const p1 = p0 + 8 * 128;
  store_snapshot<0>(p0, s[0]);
  store_snapshot<512>(p0, s[1]);
  store_snapshot<1024>(p0, s[2]);
  store_snapshot<1536>(p0, s[3]);
  store_snapshot<2048>(p0, s[4]);
  store_snapshot<2560>(p0, s[5]);
  store_snapshot<3072>(p0, s[6]);
  store_snapshot<3584>(p0, s[7]);
  store_snapshot<0>(p1, s[8]);
  store_snapshot<512>(p1, s[9]);
  store_snapshot<1024>(p1, s[10]);
  store_snapshot<1536>(p1, s[11]);
  store_snapshot<2048>(p1, s[12]);
  store_snapshot<2560>(p1, s[13]);
  store_snapshot<3072>(p1, s[14]);
  store_snapshot<3584>(p1, s[15]);
}

// Touch one 128-byte line per lane, so that the tile's operands wait in this XCD's L2 (no register
// result: the four bytes per lane land in a spare LDS area).
__device__ __forceinline__ void scan_touch(const void* src, const void* lds_base) {
  typedef const __attribute__((address_space(3))) void* lds_cptr;
  const unsigned m0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)(lds_cptr)lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(m0) : "memory", "m0");
}

// Launch arguments of one stream's whole sequence are filled by the entry points in gdn.hip; the
// prepared-tile path (gdn_scan.hip) takes the same arguments.
//
// Bytes of workspace the prepared-tile path needs, 0 where it is not taken; and the launches.
long long gdn_scan_workspace(int B, int T, int Hk, int Hv, int sub, int streams, bool states,
                             int* tiles_per_range);
int gdn_scan_launch(const GdnArgs& a, int streams, void* workspace, hipStream_t st);
// The same for the fp32 state fork (gdn_scan_f32.hip): D = Dk = Dv, 64 or 128.
long long gdn_fork32_workspace(int B, int L, int Hk, int Hv, int D, int block, bool states, int* tiles_per_range);
int gdn_fork32_launch(const GdnArgs& a, void* workspace, hipStream_t st);

}  // namespace dllm
