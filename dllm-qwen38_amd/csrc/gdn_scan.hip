// The gated delta rule (bf16 heads of 128 x 128) in two launches, for few (sequence, head) pairs.
//
// The pipelined kernel (gdn.hip) forms a tile's preparation (Gram products, the inverse T, P) one tile
// ahead, in the same workgroup as the recurrence. With few heads the chip is mostly idle and a tile
// lasts as long as that preparation, about 8k clocks, although only the state is sequential. Here
//   gdn_scan_prep_kernel  prepares every tile of every head at once and leaves the operands in a
//                         workspace, as the fragments the matrix instructions take;
//   gdn_scan_kernel       walks the tiles: one wave per stream and 32 value columns, every operand a
//                         coalesced register load issued a tile ahead, no row staging in LDS.
// Both do the pipelined kernel's arithmetic operation for operation (the same products in the same
// order, the same roundings), so the outputs and states are the same bits.
//
// Workspace per tile and sequence: per key head the K and Q fragments of each stream and the clean K^T
// fragments of the update (8 KB each), per value head and stream T1, T2 and P (2 KB each) and the
// row vectors. Sequences whose workspace would pass SCAN_WS_MAX are walked in ranges of tiles.
#include <algorithm>

#include "gdn_common.h"

namespace dllm {

struct ScanArgs {
  char* kq;                // [B][tiles][Hk][KQB]
  char* hd;                // [B][tiles][Hv][NS][HDB]
  const float* carry_in;   // state before the first tile [.., Hv, 128, 128], or null (zeros)
  long long carry_sb;      // its batch stride
  float* carry_out;        // state after the last tile [B, Hv, 128, 128], or null
  int ntiles;
};

constexpr int SCAN_FRAG = 8192;   // K, Q or K^T fragments of a tile: [4 slices][2 halves][64 lanes] x 16 bytes
constexpr int SCAN_TF = 2048;     // T1, T2 or P: [2 halves][64 lanes] x 16 bytes
constexpr int SCAN_HDB = 3 * SCAN_TF + 512;  // + EGQ, RNK, EGLK (32 floats each) and the tile's decay
constexpr int SCAN_V_EGQ = 3 * SCAN_TF, SCAN_V_RNK = SCAN_V_EGQ + 128, SCAN_V_EGLK = SCAN_V_EGQ + 256,
              SCAN_V_LAM = SCAN_V_EGQ + 384;
constexpr long long SCAN_WS_MAX = 96LL << 20, SCAN_TILE_MAX = 11LL << 18, SCAN_TILE_STATES = 2LL << 20;
// key-head block: clean K, Q, K^T, then noised K, Q
constexpr int scan_kqb(int ns) { return (ns == 2 ? 5 : 3) * SCAN_FRAG; }

__device__ __forceinline__ void scan_store_frag(char* base, int lane, const Frag<true>& f) {
  *(bf16x8*)(base + 16 * lane) = f.lo;
  *(bf16x8*)(base + 1024 + 16 * lane) = f.hi;
}
__device__ __forceinline__ void scan_load_frag(const char* base, int lane, Frag<true>& f) {
  f.lo = *(const bf16x8*)(base + 16 * lane);
  f.hi = *(const bf16x8*)(base + 1024 + 16 * lane);
}

struct PrepSmem {  // per wave, floats: A, T and Y of the inverse, row vectors (gamma, beta, factors)
  static constexpr int AF = 0, TF = AF + 32 * INV_ROW, YF = TF + 32 * INV_ROW, GAML = YF + 16 * 20, BET = GAML + 32,
                       BR = BET + 32, C1 = BR + 32, TOTAL = C1 + 32;
  static constexpr int QROW = 136;  // bf16 row stride of the K rows staged for the transposed fragments
  static_assert(32 * QROW * 2 <= (GAML - AF) * 4, "K rows fit the inverse's scratch");
};

// One workgroup per (sequence, tile, key head, stream); its waves (one per value head of the
// group, at most four) prepare the value heads in turn and share out the key head's fragment copies. Bound by latency: each value
// head is one wave's chain (Gram, mask, inverse), all tiles and heads at once.
template <int NS>
__global__ __launch_bounds__(256, 3) void gdn_scan_prep_kernel(GdnArgs a, ScanArgs w) {
  using SM = PrepSmem;
  using F = Frag<true>;
  constexpr int KT = 4;
  constexpr float LOG2E = 1.4426950408889634f;
  extern __shared__ __attribute__((aligned(16))) float scan_prep_smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int id = blockIdx.x;
  const int s = id % NS;
  id /= NS;
  const int hk = id % a.Hk;
  id /= a.Hk;
  const int c = id % w.ntiles, b = id / w.ntiles;
  const int rep = a.Hv / a.Hk;
  const GdnStream& st = a.s[s];
  float* const sm = scan_prep_smem + wave * SM::TOTAL;
  const int nw = blockDim.x >> 6;
  const int t0 = c * a.sub;

  // K and Q fragments of the tile (lane = row l32, 16 consecutive d of each 32-wide slice); rows past
  // the tile's real ones are zero
  F fk[KT], fq[KT];
  {
    const int row = t0 + min(l32, a.sub - 1);
    const bf16* kp = (const bf16*)st.k + b * a.k_sb + (long long)hk * a.k_sh + (long long)row * a.k_st + 16 * h;
    const bf16* qp = (const bf16*)st.q + b * a.q_sb + (long long)hk * a.q_sh + (long long)row * a.q_st + 16 * h;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      fk[kt].lo = *(const bf16x8*)(kp + 32 * kt);
      fk[kt].hi = *(const bf16x8*)(kp + 32 * kt + 8);
      fq[kt].lo = *(const bf16x8*)(qp + 32 * kt);
      fq[kt].hi = *(const bf16x8*)(qp + 32 * kt + 8);
    }
    if (l32 >= a.sub) {
      const bf16x8 z = {};
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) fk[kt].lo = fk[kt].hi = fq[kt].lo = fq[kt].hi = z;
    }
  }
  char* const kq = w.kq + ((long long)(b * w.ntiles + c) * a.Hk + hk) * scan_kqb(NS) + (s ? 3 * SCAN_FRAG : 0);
  if (0 == wave) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) scan_store_frag(kq + 2048 * kt, lane, fk[kt]);
  }
  if (1 % nw == wave) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) scan_store_frag(kq + SCAN_FRAG + 2048 * kt, lane, fq[kt]);
  }
  if (2 % nw == wave && s == 0) {
    bf16* const kr = (bf16*)sm;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      *(bf16x8*)(kr + l32 * SM::QROW + 32 * kt + 16 * h) = fk[kt].lo;
      *(bf16x8*)(kr + l32 * SM::QROW + 32 * kt + 16 * h + 8) = fk[kt].hi;
    }
    wave_lds_sync();
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      F f;
      lds_frag_tr_d(kr + 32 * kt, SM::QROW, lane, f);
      scan_store_frag(kq + 2 * SCAN_FRAG + 2048 * kt, lane, f);
    }
    wave_lds_sync();
  }

  for (int j = wave; j < rep; j += nw) {
    const int hv = hk * rep + j;
    char* const hd = w.hd + (((long long)(b * w.ntiles + c) * a.Hv + hv) * NS + s) * SCAN_HDB;
    const int row = t0 + min(l32, a.sub - 1);
    const float rg = st.g[b * a.g_sb + (long long)hv * a.g_sh + row * a.g_st];
    const float rb = st.beta[b * a.b_sb + (long long)hv * a.b_sh + row * a.b_st];
    // cumulative decay of the tile's rows (inclusive scan), as the pipelined kernel forms it
    float x = (h == 0 && l32 < a.sub) ? rg : 0.f;
    x += dpp_mov<0x111>(x);  // row_shr:1
    x += dpp_mov<0x112>(x);  // row_shr:2
    x += dpp_mov<0x114>(x);  // row_shr:4
    x += dpp_mov<0x118>(x);  // row_shr:8
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x142, 0xA, 0xF, false));
    const float gall = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 31));
    const float eg = __builtin_amdgcn_exp2f(x * LOG2E);            // lanes 0..31: e^gamma
    const float egl = __builtin_amdgcn_exp2f((gall - x) * LOG2E);  // e^(gamma_last - gamma)
    const float bet = l32 < a.sub ? rb : 0.f;
    // k and q row norms (both lanes of a row hold the row's)
    const float rj = a.l2norm ? rsqrtf(row_sumsq(fk) + 1e-6f) : 1.f;
    const float rqi = a.l2norm ? a.scale * rsqrtf(row_sumsq(fq) + 1e-6f) : a.scale;
    if (h == 0) {
      sm[SM::GAML + l32] = x * LOG2E;
      sm[SM::BET + l32] = bet;
      sm[SM::BR + l32] = bet * rj;
      sm[SM::C1 + l32] = bet * eg * rj;
      *(float*)(hd + SCAN_V_EGQ + 4 * l32) = eg * rqi;
      *(float*)(hd + SCAN_V_RNK + 4 * l32) = rj;
      *(float*)(hd + SCAN_V_EGLK + 4 * l32) = egl * rj;
      if (l32 == 31) *(float*)(hd + SCAN_V_LAM) = eg;
    }
    wave_lds_sync();
    f32x4 gam4[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) gam4[m] = *(const f32x4*)(sm + SM::GAML + 8 * m + 4 * h);
    const float gj = sm[SM::GAML + l32];
    {  // P^T = K Q^T (lane = query row, values = key rows), masked and scaled
      f32x16 acc = zero16();
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) mma32(acc, fk[kt], fq[kt]);
      f32x16 pv;
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float val = rqi * acc[4 * m + e] * __builtin_amdgcn_exp2f(gj - gam4[m][e]);
          pv[4 * m + e] = (8 * m + 4 * h + e <= l32) ? val : 0.f;
        }
      F fp;
      acc_to_frag(pv, fp);
      scan_store_frag(hd + 2 * SCAN_TF, lane, fp);
    }
    {  // A = mask(beta_i k^_i . k^_j e^(gamma_i - gamma_j)), j < i, and T = (I + A)^-1
      f32x16 acc = zero16();
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) mma32(acc, fk[kt], fk[kt]);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4 br4 = *(const f32x4*)(sm + SM::BR + 8 * m + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 8 * m + 4 * h + e;
          const float val = (br4[e] * rj) * acc[4 * m + e] * __builtin_amdgcn_exp2f(gam4[m][e] - gj);
          sm[SM::AF + i * INV_ROW + l32] = (l32 < i) ? val : 0.f;
        }
      }
      wave_lds_sync();
      {
        float* const AF = sm + SM::AF;
        float* const TF = sm + SM::TF;
        float* const YF = sm + SM::YF;
        const int lo = l32;
#include "gdn_inverse.inc"
      }
      f32x16 tv1, tv2;
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4 t4 = *(const f32x4*)(sm + SM::TF + l32 * INV_ROW + 8 * m + 4 * h);
        const f32x4 be4 = *(const f32x4*)(sm + SM::BET + 8 * m + 4 * h);
        const f32x4 c14 = *(const f32x4*)(sm + SM::C1 + 8 * m + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = 8 * m + 4 * h + e <= l32;
          tv1[4 * m + e] = in ? -(t4[e] * c14[e]) : 0.f;  // -T1 = -T diag(beta e^gamma / ||k||)
          tv2[4 * m + e] = in ? t4[e] * be4[e] : 0.f;     // T2 = T diag(beta)
        }
      }
      F f1, f2;
      acc_to_frag(tv1, f1);
      acc_to_frag(tv2, f2);
      scan_store_frag(hd, lane, f1);
      scan_store_frag(hd + SCAN_TF, lane, f2);
    }
    wave_lds_sync();  // the next head's vectors come after this one's reads
  }
}

struct ScanSmem {
  static constexpr int SB = 8192;       // state fragments of a tile: [4 slices][2 halves][64 lanes] x 16 bytes
  static constexpr int VB = 4096;       // V' of a tile and stream: [4][64 lanes] x 16 bytes
  static constexpr int OROW = 40;       // bf16 row stride of a staged [32 x 32] tile
  static constexpr int OB = 32 * OROW * 2;
  static constexpr int NSB = 3;         // state slots: the noised outputs read a state two phases after it
  // V' double-buffered per stream, the clean U double-buffered; per stream a staged V tile, per output wave a staged output tile,
  // per wave the tile's row vectors; 256 bytes that the touch loads land in
  static constexpr int O_S = 0, O_V = O_S + NSB * SB, O_U = O_V + 4 * VB, O_VT = O_U + 2 * VB, O_OT = O_VT + 2 * OB, O_X = O_OT + 2 * OB,
                       O_PF = O_X + 4 * 256, O_SN = O_PF + 256;
  static constexpr int SN = 16384;      // a state in fp32 on its way to its snapshot: [4 slices][4][64 lanes] x 16 bytes
  static constexpr int TOTAL = O_SN + 2 * SN;
};

// One workgroup per (sequence, value head, 32 value columns), its waves split by role so that the state's
// chain is all that wave 0 does:
//   wave 0     the clean state, in accumulators: per tile it publishes the state before the tile (as B
//              fragments) and V' = T2 V - T1 (K S) in LDS and updates the state;
//   wave 1     the clean outputs, from those, a tile behind;
//   wave 2, 3  (NS = 2) the noised V', a tile behind, and the noised outputs, two behind;
//   wave 2 NS  U = T2 V for wave 0, a tile ahead;
//   helpers    store the snapshots, handed over in LDS, a tile behind (in wave 0, whose later loads would
//              wait for the stores, they cost 25 of 81 us at B = 1, T = 1952, 48 heads), and the first one
//              touches the lines of the tile SCAN_AHEAD tiles on: a load from memory outlasts a tile.
// One barrier per tile. Every operand is a coalesced register load issued a tile ahead of its use.
constexpr int SCAN_AHEAD = 4, SCAN_HELPERS = 3;
template <int NS>
constexpr int scan_waves() { return 2 * NS + 1 + SCAN_HELPERS; }
template <int NS>
__global__ __launch_bounds__(64 * scan_waves<NS>()) void gdn_scan_kernel(GdnArgs a, ScanArgs w) {
  using SM = ScanSmem;
  using F = Frag<true>;
  constexpr int KT = 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[SM::TOTAL];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  const int s = wave == 2 * NS ? 0 : wave >> 1;  // the wave's stream
  const int lin = xcd_linear_id(blockIdx.x, gridDim.x);  // a head's column windows: one XCD
  const int cu = (lin & 3) * 32;
  const int hv = (lin >> 2) % a.Hv, b = (lin >> 2) / a.Hv;
  const int rep = a.Hv / a.Hk, hk = hv / rep;
  const int ntiles = w.ntiles;

  const long long kq_step = (long long)a.Hk * scan_kqb(NS), hd_step = (long long)a.Hv * NS * SCAN_HDB;
  const char* const kqb = w.kq + ((long long)b * w.ntiles * a.Hk + hk) * scan_kqb(NS);
  const char* const hdb = w.hd + ((long long)b * w.ntiles * a.Hv + hv) * NS * SCAN_HDB;
  // this wave's LDS writes have landed, then the barrier (global loads stay in flight); every wave runs
  // ntiles + NS of them
  auto tile_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  if (wave > 2 * NS) {
    constexpr int NHP = scan_waves<NS>() - 2 * NS - 1;
    const int hw = wave - 2 * NS - 1;
    // lanes 0..31: the clean v rows, 32..63: the noised ones (NS = 1: the same again)
    const bf16* const v0 = (const bf16*)a.s[0].v;
    const bf16* const v1 = (const bf16*)a.s[NS - 1].v;
    const bf16* const vl0 = (h ? v1 : v0) + b * a.v_sb + (long long)hv * a.v_sh + cu;
    // the workgroups of a key head's columns share its lines out among them, those of a head its own
    const int nk = 4 * rep, ik = 4 * (hv % rep) + (lin & 3);
    constexpr int LK = scan_kqb(NS) / 128, LH = NS * SCAN_HDB / 128;  // lines
    auto touch = [&](int c) {
      if (c >= ntiles || hw != 0) return;
      const char* const kl = kqb + c * kq_step;
      const char* const hl = hdb + c * hd_step;
      for (int i = ik * 64; i < LK; i += nk * 64) scan_touch(kl + 128 * min(i + lane, LK - 1), smem + SM::O_PF);
      if (lane < (LH + 3) / 4) scan_touch(hl + 128 * min(4 * lane + (lin & 3), LH - 1), smem + SM::O_PF);
      scan_touch(vl0 + (long long)(c * a.sub + min(l32, a.sub - 1)) * a.v_st, smem + SM::O_PF);
    };
#pragma unroll
    for (int c = 1; c < SCAN_AHEAD; ++c) touch(c);
    // snapshot rows: lane takes columns 4 (lane % 8) .. of row 8 i + lane / 8 of each 16-byte store; the state
    // lies in accumulator order, row r = 32 kt + 16 h' + 4 m + e, column n at [kt][m][32 h' + n][e]
    const float* const sn0 = (const float*)(smem + SM::O_SN) + 16 * (lane & 7) + ((lane >> 3) & 3) + 256 * (lane >> 5);
    float* const sp0 = a.states ? a.states + ((long long)b * a.snap_rows * a.Hv + hv) * (128LL * 128) + cu +
                                      (lane >> 3) * 128 + 4 * (lane & 7)
                                : nullptr;
    tile_barrier();
    for (int c = 0; c < ntiles + NS; ++c) {  // the last phases: no touch left, the barriers of the others
      touch(c + SCAN_AHEAD);
      if (c > 0 && c <= ntiles && sp0) {  // the state after tile c - 1
        const float* const sn = sn0 + ((c - 1) & 1) * (SM::SN / 4);
        float* const sp = sp0 + (long long)(c - 1) * a.Hv * (128LL * 128);
#pragma unroll
        for (int ii = 0; ii < (16 + NHP - 1) / NHP; ++ii) {  // rows 8 i .. 8 i + 7: slice i / 4, half (i / 2) % 2, m = 2 (i % 2) + lane / 32
          const int i = ii * NHP + hw;
          if (16 % NHP != 0 && i >= 16) break;
          const float* const q = sn + 1024 * (i >> 2) + 128 * ((i >> 1) & 1) + 512 * (i & 1);
          f32x4 x;
#pragma unroll
          for (int e = 0; e < 4; ++e) x[e] = q[4 * e];
          __builtin_nontemporal_store(x, (f32x4*)(sp + 8 * i * 128));
        }
      }
      if (c < ntiles + NS - 1) tile_barrier();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no touch in flight past the wave's end
    return;
  }

  const GdnStream& st = a.s[s];
  const char* const kq0 = kqb + (s ? 3 * SCAN_FRAG : 0);
  const char* const hd0 = hdb + s * SCAN_HDB;
  float* const xv = (float*)(smem + SM::O_X + wave * 256);  // 64 floats of row vectors (not the U wave's)
  float xr;
  auto load_frags = [&](int c, int off, F (&f)[KT]) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) scan_load_frag(kq0 + c * kq_step + off + 2048 * kt, lane, f[kt]);
  };
  auto load_x = [&](int c, int off) { xr = *(const float*)(hd0 + c * hd_step + off + 4 * lane); };
  // a row vector of the tile in accumulator layout: rows 8 m + 4 h + e
  auto row_vec = [&](int at, f32x4 (&x)[4]) {
#pragma unroll
    for (int m = 0; m < 4; ++m) x[m] = *(const f32x4*)(xv + at + 8 * m + 4 * h);
  };
  auto state_frag = [&](int c, int kt) { return (char*)smem + SM::O_S + (c % SM::NSB) * SM::SB + 2048 * kt; };
  unsigned char* const vb0 = smem + SM::O_V + 2 * s * SM::VB + 16 * lane;

  // the window's v rows of a tile: 16 bytes per lane of rows 16 i + lane / 4 (past the real rows: the last)
  const bf16* const vp0 = (const bf16*)st.v + b * a.v_sb + (long long)hv * a.v_sh + cu + 8 * (lane & 3);
  bf16* const vt = (bf16*)(smem + SM::O_VT + s * SM::OB);
  F t1, t2;
  bf16x8 vr[2];
  auto load_v = [&](int c) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
      vr[i] = *(const bf16x8*)(vp0 + (long long)(c * a.sub + min(16 * i + (lane >> 2), a.sub - 1)) * a.v_st);
  };
  auto load_t1 = [&](int c) { scan_load_frag(hd0 + c * hd_step, lane, t1); };
  auto load_t2 = [&](int c) { scan_load_frag(hd0 + c * hd_step + SCAN_TF, lane, t2); };
  auto u_product = [&](f32x16& vn) {  // U = T2 V (the V rows turned around in LDS)
    const bf16x8 z = {};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = 16 * i + (lane >> 2);
      *(bf16x8*)(vt + row * SM::OROW + 8 * (lane & 3)) = row < a.sub ? vr[i] : z;
    }
    wave_lds_sync();
    F fv;
    lds_frag_tr(vt, SM::OROW, lane, fv);
    mma32(vn, t2, fv);
  };
  auto publish = [&](unsigned char* to, const f32x16& x) {
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = x[4 * m + e];
      *(f32x4*)(to + 1024 * m) = y;
    }
  };
  unsigned char* const ub0 = smem + SM::O_U + 16 * lane;

  if (wave == 2 * NS) {  // ----------------------------------------------- U of the clean stream
    load_v(0);
    load_t2(0);
    for (int c = 0; c < ntiles + NS; ++c) {
      if (c < ntiles) {  // in phase c - 1, read in phase c
        const int cn = c + 1 < ntiles ? c + 1 : c;  // past the last tile: reloaded, unused
        f32x16 u = zero16();
        u_product(u);
        load_v(cn);
        load_t2(cn);
        publish(ub0 + (c & 1) * SM::VB, u);
      }
      tile_barrier();
    }
    return;
  }

  if (wave & 1) {  // ------------------------------------------------------- outputs of stream s
    const long long rs = (long long)a.Hv * a.Dv;  // token stride of the outputs
    bf16* const out0 = (bf16*)st.out + (long long)b * a.t_rows * rs + (long long)hv * a.Dv + cu;
    bf16* const ot = (bf16*)(smem + SM::O_OT + s * SM::OB);
    F qf[KT], p;
    auto load_p = [&](int c) { scan_load_frag(hd0 + c * hd_step + 2 * SCAN_TF, lane, p); };
    // the loads go out in the order of their uses here and in the loop, so that a wait for one leaves the
    // later ones in flight
    load_x(0, SCAN_V_EGQ);  // lanes 0..31 EGQ, 32..63 RNK
    load_frags(0, SCAN_FRAG, qf);
    load_p(0);
    tile_barrier();
    if (s == 1) tile_barrier();
    for (int c = 0; c < ntiles; ++c) {
      const int cn = c + 1 < ntiles ? c + 1 : c;  // past the last tile: reloaded, unused
      tile_barrier();  // tile c's state and V' are published
      xv[lane] = xr;
      load_x(cn, SCAN_V_EGQ);
      f32x16 qs = zero16(), vk;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        F sx;
        scan_load_frag(state_frag(c, kt), lane, sx);
        mma32(qs, qf[kt], sx);
      }
      load_frags(cn, SCAN_FRAG, qf);
      // O = diag(e^gamma scale/||q||) Q S + P (V' / ||k||)
      wave_lds_sync();
      f32x4 egq[4], rnk[4];
      row_vec(0, egq);
      row_vec(32, rnk);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4 x = *(const f32x4*)(vb0 + (c & 1) * SM::VB + 1024 * m);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vk[4 * m + e] = x[e] * rnk[m][e];
          qs[4 * m + e] *= egq[m][e];
        }
      }
      {
        F fv;
        acc_to_frag(vk, fv);
        mma32(qs, p, fv);
      }
      load_p(cn);
      // to rows of 64 bytes through LDS (this wave's own)
      bf16* const sp = ot + l32 + 4 * h * SM::OROW;
#pragma unroll
      for (int v = 0; v < 16; ++v) sp[(((v >> 2) << 3) + (v & 3)) * SM::OROW] = (bf16)qs[v];
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = 16 * i + (lane >> 2), ch = 8 * (lane & 3);
        const bf16x8 o8 = *(const bf16x8*)(ot + row * SM::OROW + ch);
        if (row < a.sub) *(bf16x8*)(out0 + (c * a.sub + row) * rs + ch) = o8;
      }
      wave_lds_sync();
    }
    if (NS == 2 && s == 0) tile_barrier();
    return;
  }

  // ------------------------------------------------------------------------- V' of stream s
  F kf[KT];
  if (NS == 2 && s == 1) {
    load_frags(0, 0, kf);
    load_v(0);
    load_t2(0);
    load_t1(0);
    tile_barrier();
    for (int c = 0; c < ntiles; ++c) {
      const int cn = c + 1 < ntiles ? c + 1 : c;
      tile_barrier();  // the state before tile c is published
      f32x16 ks = zero16(), vn = zero16();
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        F sx;
        scan_load_frag(state_frag(c, kt), lane, sx);
        mma32(ks, kf[kt], sx);
      }
      load_frags(cn, 0, kf);
      u_product(vn);
      load_v(cn);
      load_t2(cn);
      F fks;
      acc_to_frag(ks, fks);
      mma32(vn, t1, fks);  // V' = U - T1 (K S)
      load_t1(cn);
      publish(vb0 + (c & 1) * SM::VB, vn);
    }
    tile_barrier();
    return;
  }
  f32x16 S[KT];
  if (w.carry_in) {  // accumulator row rho(v, h) of slice kt is state row 32 kt + 16 h + v
    const float* ip = w.carry_in + b * w.carry_sb + (long long)hv * (128 * 128) + cu + 16 * h * 128 + l32;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) S[kt][v] = ip[(32 * kt + v) * 128];
  } else {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) S[kt] = zero16();
  }
  F ktf[KT];
  load_x(0, SCAN_V_EGLK);  // lanes 0..31 EGLK, lane 32 the tile's decay
  load_frags(0, 0, kf);
  load_t1(0);
  load_frags(0, 2 * SCAN_FRAG, ktf);
  tile_barrier();
  for (int c = 0; c < ntiles; ++c) {
    const int cn = c + 1 < ntiles ? c + 1 : c;
    f32x16 ks = zero16(), vn;
    xv[lane] = xr;
    const float lam = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, xr), 32));
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      F sx;
      acc_to_frag(S[kt], sx);
      mma32(ks, kf[kt], sx);
      scan_store_frag(state_frag(c, kt), lane, sx);
      // the decay of the state while the products run
#pragma unroll
      for (int v = 0; v < 16; ++v) S[kt][v] *= lam;
      __builtin_amdgcn_sched_barrier(0);
    }
    load_x(cn, SCAN_V_EGLK);
    load_frags(cn, 0, kf);
#pragma unroll
    for (int m = 0; m < 4; ++m) {  // U = T2 V
      const f32x4 x = *(const f32x4*)(ub0 + (c & 1) * SM::VB + 1024 * m);
#pragma unroll
      for (int e = 0; e < 4; ++e) vn[4 * m + e] = x[e];
    }
    f32x4 eglk[4];
    row_vec(0, eglk);
    {
      F fks;
      acc_to_frag(ks, fks);
      mma32(vn, t1, fks);  // V' = U - T1 (K S)
    }
    load_t1(cn);
    // S <- e^gamma_last S + K_raw^T (e^(gamma_last - gamma) / ||k|| V')
    {
      f32x16 vd;
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) vd[4 * m + e] = vn[4 * m + e] * eglk[m][e];
      F fd;
      acc_to_frag(vd, fd);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) mma32(S[kt], ktf[kt], fd);
    }
    publish(vb0 + (c & 1) * SM::VB, vn);
    load_frags(cn, 2 * SCAN_FRAG, ktf);
    if (a.states) {
      unsigned char* const sn = smem + SM::O_SN + (c & 1) * SM::SN + 16 * lane;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) publish(sn + 4096 * kt, S[kt]);
    }
    tile_barrier();
  }
  if constexpr (NS == 2) tile_barrier();
  if (w.carry_out) {
    float* op = w.carry_out + ((long long)b * a.Hv + hv) * (128LL * 128) + cu + 16 * h * 128 + l32;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int v = 0; v < 16; ++v) op[(32 * kt + v) * 128] = S[kt][v];
  }
}

static long long scan_tile_bytes(int B, int Hk, int Hv, int streams) {
  return (long long)B * ((long long)Hk * scan_kqb(streams) + (long long)Hv * streams * SCAN_HDB);
}

long long gdn_scan_workspace(int B, int T, int Hk, int Hv, int sub, int streams, bool states, int* tiles_per_range) {
  const int ntiles = T / sub;
  // Four workgroups per head, one per CU: past 64 heads a second round starts and the pipelined kernel, whose
  // workgroups hold a head (half a head up to 128), is the faster one (B = 8, 16 heads, L = 2048: 345
  // vs 553 us; B = 1, 48 heads: 226 vs 140). A few tiles are over before the second launch pays (eight
  // tiles of 48 heads on one stream 27.0 vs 24.8 us, ten 32.4 vs 24.8).
  // The operands of a tile step (all heads) past 2.75 MB, 2 MB where the states are written beside them, cost
  // more than the chain saves (L = 2048, 16 / 16 heads: B = 4, 3.5 MB, no states 272 vs 258 us; B = 3,
  // 2.6 MB, no states 218 vs 242, states 267 vs 250; 16 / 48 heads, B = 1, 1.3 MB, states 185 vs 229).
  const long long per = scan_tile_bytes(B, Hk, Hv, streams);
  if (ntiles < 10 || (long long)B * Hv > 64 || per > (states ? SCAN_TILE_STATES : SCAN_TILE_MAX)) return 0;
  const int most = (int)std::max(1LL, SCAN_WS_MAX / per);
  const int nr = (ntiles + most - 1) / most;
  const int tpr = (ntiles + nr - 1) / nr;
  if (tiles_per_range) *tiles_per_range = tpr;
  return per * tpr + (nr > 1 ? (long long)B * Hv * 128 * 128 * 4 : 0);
}

int gdn_scan_launch(const GdnArgs& a0, int streams, void* workspace, hipStream_t st) {
  int tpr = 0;
  gdn_scan_workspace(a0.B, a0.T, a0.Hk, a0.Hv, a0.sub, streams, a0.states != nullptr, &tpr);
  const int ntiles = a0.T / a0.sub;
  const long long snap = (long long)a0.Hv * 128 * 128;
  float* const carry = (float*)((char*)workspace + scan_tile_bytes(a0.B, a0.Hk, a0.Hv, streams) * tpr);
  for (int c0 = 0; c0 < ntiles; c0 += tpr) {
    const int n = std::min(tpr, ntiles - c0);
    const long long t = (long long)c0 * a0.sub;
    GdnArgs a = a0;
    for (int i = 0; i < streams; ++i) {
      GdnStream& s = a.s[i];
      s.q = (const bf16*)s.q + t * a.q_st;
      s.k = (const bf16*)s.k + t * a.k_st;
      s.v = (const bf16*)s.v + t * a.v_st;
      s.g += t * a.g_st;
      s.beta += t * a.b_st;
      s.out = (bf16*)s.out + t * a.Hv * a.Dv;
    }
    if (a.states) a.states += c0 * snap;
    a.T = n * a.sub;
    ScanArgs w = {};
    w.ntiles = n;
    w.kq = (char*)workspace;
    w.hd = w.kq + (long long)a.B * n * a.Hk * scan_kqb(streams);
    if (c0 == 0) {
      w.carry_in = a0.init;
      w.carry_sb = snap;
    } else if (a0.states) {
      w.carry_in = a0.states + (c0 - 1) * snap;
      w.carry_sb = a0.snap_rows * snap;
    } else {
      w.carry_in = carry;
      w.carry_sb = snap;
    }
    w.carry_out = !a0.states && c0 + n < ntiles ? carry : nullptr;
    const long long np = (long long)a.B * n * a.Hk * streams, ns = 4LL * a.B * a.Hv;
    if (np > 0x7fffffff) return fail(DLLM_EUNSUPPORTED, "gdn: grid too large");
    const int nw = std::min(4, a.Hv / a.Hk);
    const size_t plds = (size_t)nw * PrepSmem::TOTAL * sizeof(float);
    if (streams == 2) {
      gdn_scan_prep_kernel<2><<<dim3((unsigned)np), 64 * nw, plds, st>>>(a, w);
      gdn_scan_kernel<2><<<dim3((unsigned)ns), 64 * scan_waves<2>(), 0, st>>>(a, w);
    } else {
      gdn_scan_prep_kernel<1><<<dim3((unsigned)np), 64 * nw, plds, st>>>(a, w);
      gdn_scan_kernel<1><<<dim3((unsigned)ns), 64 * scan_waves<1>(), 0, st>>>(a, w);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(DLLM_ELAUNCH, "gdn scan launch: %s", hipGetErrorString(e));
  }
  return DLLM_OK;
}

}  // namespace dllm
