// The state fork in fp32 (heads of 64 x 64 and 128 x 128) in three launches.
//
// A tile's Gram products, its inverse T = (I + A)^-1, W = T1 K, U = T2 V and P depend on the tile's own
// rows, and its outputs on the state before it; only S <- e^gamma_last S + K~^T (U - W S) is sequential.
//   fork32_prep_kernel   every (tile, head, stream) at once: W, U, P and the row vectors, as the fragments
//                        the matrix instructions take, into a workspace;
//   fork32_state_kernel  the clean state alone, one workgroup per (sequence, head, 32 value columns), a wave
//                        per 32 state rows: a tile costs a wave two products of 32 x 32 x 32 (2 x 1024 clocks
//                        on the fp32 matrix cores), not the 16 of a wave that also forms U, both outputs
//                        and the update of all 128 rows;
//   fork32_out_kernel    the outputs of every (tile, head, stream), a wave per 32 columns, no LDS.
// Bound by the fp32 matrix cores (40k clocks per SIMD in all at eight tiles of 48 heads of 128) and the state
// chain (2.5k clocks a tile). The other path, the chunk kernel on the clean stream, then on every noised
// block from its copied initial state, walked a tile's whole work in one chain and formed T twice per head:
// conv and fork of one layer, 16 / 48 heads of 128, us there -> here: B = 1, L = 256 243 -> 87, and 70 with the conv's rows
// split (conv.hip), L = 32 99 -> 35, B = 2, L = 512 643 -> 252; four heads of 64, B = 1, L = 256 122 -> 38 (there one
// launch). At L = 256 the kernels take 18, 20 and 25 us, the matrix cores busy 25, 32 and 38% of them.
//
// Workspace per (sequence, tile): per key head the clean K^T, per (head, stream) W and U (4 KB per 32 state rows / value columns each; the
// state kernel leaves V' = U - W S of the clean stream in U's place), P (4 KB) and the row vectors; the
// states after each tile where the caller keeps none. Sequences past FORK32_WS_MAX are walked in ranges.
#include <algorithm>
#include <type_traits>

#include "gdn_common.h"

namespace dllm {

struct Fork32Args {
  char* hd;            // [B][ntiles][Hv][2] blocks of fork32_hdb bytes
  char* kt;            // [B][ntiles][Hk] clean K^T, 4 KB per 32 state rows
  const float* cin;    // state before the first tile [.., Hv, D, D], or null (zeros)
  long long cin_sb;    // its batch stride
  float* st;           // states after each tile [.., ntiles, Hv, D, D]
  long long st_sb;     // its batch stride
  float* cout;         // state after the last tile [B, Hv, D, D], or null
  int ntiles;
};

constexpr int FORK32_AHEAD = 5;  // tiles between a touch and the use
constexpr long long FORK32_WS_MAX = 128LL << 20;
// block of a (tile, head, stream): W, U, P, then EGQ, RNK, EGLK (32 floats each) and the tile's decay
constexpr int fork32_hdb(int kt) { return 2 * kt * 4096 + 4096 + 512; }
constexpr int F32V_EGQ = 0, F32V_RNK = 32, F32V_EGLK = 64, F32V_LAM = 96;

// 16 values per lane as four coalesced 1 KB rows of 16 bytes per lane
__device__ __forceinline__ void f32_store(char* base, int lane, const f32x16& x) {
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    f32x4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = x[4 * m + e];
    *(f32x4*)(base + 1024 * m + 16 * lane) = y;
  }
}
__device__ __forceinline__ void f32_store(char* base, int lane, const Frag<false>& f) {
  f32x16 x;
#pragma unroll
  for (int v = 0; v < 16; ++v) x[v] = f.v[v];
  f32_store(base, lane, x);
}
__device__ __forceinline__ void f32_load(const char* base, int lane, Frag<false>& f) {
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const f32x4 y = *(const f32x4*)(base + 1024 * m + 16 * lane);
#pragma unroll
    for (int e = 0; e < 4; ++e) f.v[4 * m + e] = y[e];
  }
}
// rows 8 m + 4 h + (0..3) of a row vector, in accumulator order
__device__ __forceinline__ void f32_rows(const float* v, int h, f32x4 (&x)[4]) {
#pragma unroll
  for (int m = 0; m < 4; ++m) x[m] = *(const f32x4*)(v + 8 * m + 4 * h);
}
// column l32 of 32 rows of stride rs (p uniform) in rho order; rows from `sub` on read as zero
__device__ __forceinline__ void f32_col(const float* p, int rs, int sub, int h, int l32, Frag<false>& f) {
  if (sub == 32) {  // one 32-bit lane offset for every row (at least 32 rows of a 32-bit extent)
    const unsigned lo = 4u * (unsigned)(4 * h * rs + l32);
#pragma unroll
    for (int v = 0; v < 16; ++v) f.v[v] = *(const float*)((const char*)(p + rho(v, 0) * rs) + lo);
    return;
  }
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int r = rho(v, h);
    const float x = p[min(r, sub - 1) * rs + l32];
    f.v[v] = r < sub ? x : 0.f;
  }
}

// One workgroup per (sequence, tile, key head, stream), a wave per 32 dims of the head. The Gram products are
// split over the waves by d (each reads its 32 columns of K and Q once) and summed in wave order through LDS.
// The value heads of the key head share them: up to KT at a time, each head's P and inverse on a wave of its own,
// then every wave its slice of every head's W and U.
template <int KT>
__global__ __launch_bounds__(64 * KT) void fork32_prep_kernel(GdnArgs a, Fork32Args w) {
  constexpr int HDB = fork32_hdb(KT);
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr int IS = 2 * 32 * INV_ROW + 16 * 20;  // A, T and Y of an inverse
  __shared__ __attribute__((aligned(16))) float part[2][KT][1024];
  __shared__ __attribute__((aligned(16))) float inv[KT][IS];
  __shared__ __attribute__((aligned(16))) float ss[2][KT][32];
  __shared__ __attribute__((aligned(16))) float vec[KT][4][32];  // gamma (log2 units), beta, beta / ||k||, beta e^gamma / ||k||
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  int id = xcd_linear_id(blockIdx.x, gridDim.x);  // a head's tiles: one XCD, in all three kernels
  const int c = id % w.ntiles;
  id /= w.ntiles;
  const int s = id & 1;
  id >>= 1;
  const int hk = id % a.Hk, b = id / a.Hk;
  const int rep = a.Hv / a.Hk;
  const GdnStream& st = a.s[s];
  const long long t0 = (long long)c * a.sub;

  Frag<false> fk, fq, ktr;
  const float* const kb = (const float*)st.k + b * a.k_sb + (long long)hk * a.k_sh + t0 * a.k_st + 32 * wave;
  const float* const qb = (const float*)st.q + b * a.q_sb + (long long)hk * a.q_sh + t0 * a.q_st + 32 * wave;
  const int row = min(l32, a.sub - 1);
  lds_frag(kb + (long long)row * a.k_st, h, fk);  // a row's rho-ordered slice, from memory
  lds_frag(qb + (long long)row * a.q_st, h, fq);
  f32_col(kb, a.k_st, a.sub, h, l32, ktr);
  if (l32 >= a.sub) {
#pragma unroll
    for (int v = 0; v < 16; ++v) fk.v[v] = fq.v[v] = 0.f;
  }
  {
    float xk = 0.f, xq = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      xk = __builtin_fmaf(fk.v[v], fk.v[v], xk);
      xq = __builtin_fmaf(fq.v[v], fq.v[v], xq);
    }
    xk += __shfl_xor(xk, 32);
    xq += __shfl_xor(xq, 32);
    if (h == 0) {
      ss[0][wave][l32] = xk;
      ss[1][wave][l32] = xq;
    }
  }
  {
    f32x16 kk = zero16(), kq = zero16();
    mma32(kk, fk, fk);
    mma32(kq, fk, fq);  // P^T: lane = query row, values = key rows
    f32_store((char*)part[0][wave], lane, kk);
    f32_store((char*)part[1][wave], lane, kq);
  }
  if (s == 0) f32_store(w.kt + (((long long)b * w.ntiles + c) * a.Hk + hk) * (KT * 4096) + 4096 * wave, lane, ktr);
  auto gram = [&](int which, Frag<false>& acc) {  // the waves' shares, summed in wave order
    f32_load((const char*)part[which][0], lane, acc);
#pragma unroll
    for (int i = 1; i < KT; ++i) {
      Frag<false> o;
      f32_load((const char*)part[which][i], lane, o);
#pragma unroll
      for (int v = 0; v < 16; ++v) acc.v[v] += o.v[v];
    }
  };
  for (int j0 = 0; j0 < rep; j0 += KT) {
    const int nj = min(KT, rep - j0);
    Frag<false> vtr[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) {
      const int hv = hk * rep + j0 + min(j, nj - 1);
      f32_col((const float*)st.v + b * a.v_sb + (long long)hv * a.v_sh + t0 * a.v_st + 32 * wave, a.v_st, a.sub, h, l32,
              vtr[j]);
    }
    const int hv = hk * rep + j0 + min(wave, nj - 1);
    const float rg = st.g[b * a.g_sb + (long long)hv * a.g_sh + (t0 + row) * a.g_st];
    const float rb = st.beta[b * a.b_sb + (long long)hv * a.b_sh + (t0 + row) * a.b_st];
    __syncthreads();  // the shares are in; the heads before are done with their T
    if (wave < nj) {
      char* const hd = w.hd + (((long long)(b * w.ntiles + c) * a.Hv + hv) * 2 + s) * HDB;
      // cumulative decay of the tile's rows (inclusive scan in lanes 0..31)
      float x = (h == 0 && l32 < a.sub) ? rg : 0.f;
      x += dpp_mov<0x111>(x);  // row_shr:1
      x += dpp_mov<0x112>(x);  // row_shr:2
      x += dpp_mov<0x114>(x);  // row_shr:4
      x += dpp_mov<0x118>(x);  // row_shr:8
      x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x142, 0xA, 0xF, false));
      const float gall = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 31));
      const float bet = l32 < a.sub ? rb : 0.f;
      const float eg = __builtin_amdgcn_exp2f(x * LOG2E);
      float sk = 0.f, sq = 0.f;
#pragma unroll
      for (int i = 0; i < KT; ++i) {
        sk += ss[0][i][l32];
        sq += ss[1][i][l32];
      }
      const float rj = a.l2norm ? rsqrtf(sk + 1e-6f) : 1.f;
      const float rqi = a.l2norm ? a.scale * rsqrtf(sq + 1e-6f) : a.scale;
      if (h == 0) {
        vec[wave][0][l32] = x * LOG2E;
        vec[wave][1][l32] = bet;
        vec[wave][2][l32] = bet * rj;
        vec[wave][3][l32] = bet * eg * rj;
        float* const vo = (float*)(hd + 2 * KT * 4096 + 4096);
        vo[F32V_EGQ + l32] = eg * rqi;
        vo[F32V_RNK + l32] = rj;
        vo[F32V_EGLK + l32] = __builtin_amdgcn_exp2f((gall - x) * LOG2E) * rj;
        if (l32 == 31) vo[F32V_LAM] = eg;
      }
      wave_lds_sync();
      f32x4 gam4[4], br4[4];
      f32_rows(vec[wave][0], h, gam4);
      f32_rows(vec[wave][2], h, br4);
      const float gj = vec[wave][0][l32];
      Frag<false> acc;
      gram(1, acc);
      f32x16 pv;
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float val = rqi * acc.v[4 * m + e] * __builtin_amdgcn_exp2f(gj - gam4[m][e]);
          pv[4 * m + e] = (8 * m + 4 * h + e <= l32) ? val : 0.f;
        }
      f32_store(hd + 2 * KT * 4096, lane, pv);
      gram(0, acc);
      float* const AF = inv[wave];
      float* const TF = AF + 32 * INV_ROW;
      float* const YF = TF + 32 * INV_ROW;
      const int lo = l32;
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 8 * m + 4 * h + e;
          const float val = (br4[m][e] * rj) * acc.v[4 * m + e] * __builtin_amdgcn_exp2f(gam4[m][e] - gj);
          AF[i * INV_ROW + l32] = (l32 < i) ? val : 0.f;
        }
      wave_lds_sync();
#include "gdn_inverse.inc"
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < KT; ++j) {
      if (j >= nj) break;
      const float* const TF = inv[j] + 32 * INV_ROW;
      Frag<false> t1, t2;  // T1 = T diag(beta e^gamma / ||k||), T2 = T diag(beta): lane = row
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4 t4 = *(const f32x4*)(TF + l32 * INV_ROW + 8 * m + 4 * h);
        const f32x4 be4 = *(const f32x4*)(vec[j][1] + 8 * m + 4 * h);
        const f32x4 c14 = *(const f32x4*)(vec[j][3] + 8 * m + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const bool in = 8 * m + 4 * h + e <= l32;
          t1.v[4 * m + e] = in ? t4[e] * c14[e] : 0.f;
          t2.v[4 * m + e] = in ? t4[e] * be4[e] : 0.f;
        }
      }
      char* const hd = w.hd + (((long long)(b * w.ntiles + c) * a.Hv + hk * rep + j0 + j) * 2 + s) * HDB;
      f32x16 wt = zero16(), u = zero16();
      mma32(wt, ktr, t1);  // W^T = K^T T1^T: lane = row of W, values = d, the A operand of W S
      mma32(u, t2, vtr[j]);
      f32_store(hd + 4096 * wave, lane, wt);
      f32_store(hd + 4096 * (KT + wave), lane, u);
    }
  }
}

// Waves 0 .. KT - 1 each hold 32 rows of the state's 32 columns and form their share of W S; the shares meet
// in LDS (one barrier per tile; loads stay in flight over it, two tiles ahead of their use), every wave sums them in wave order and updates
// its rows. Waves KT .. 2 KT - 1 store what the tile left in LDS, V' and, a tile behind, the state: the
// chain's waves have no store in flight that their loads would wait behind.
template <int KT>
__global__ __launch_bounds__(128 * KT) void fork32_state_kernel(GdnArgs a, Fork32Args w) {
  constexpr int HDB = fork32_hdb(KT), D = 32 * KT;
  __shared__ __attribute__((aligned(16))) float part[2][KT][1024];
  __shared__ __attribute__((aligned(16))) float snap[2][KT][1024];
  __shared__ __attribute__((aligned(16))) float touched[64];  // where touch loads land
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  const int lin = xcd_linear_id(blockIdx.x, gridDim.x);  // a head's column windows: one XCD
  const int win = lin % KT, cu = 32 * win;
  const int hv = (lin / KT) % a.Hv, b = lin / (KT * a.Hv);
  const int hk = hv / (a.Hv / a.Hk);
  const int ntiles = w.ntiles;
  const long long step = (long long)a.Hv * 2 * HDB;
  char* const hd0 = w.hd + ((long long)b * ntiles * a.Hv + hv) * 2 * HDB;
  const long long kstep = (long long)a.Hk * KT * 4096;
  const char* const kt0 = w.kt + ((long long)b * ntiles * a.Hk + hk) * KT * 4096;
  // this wave's LDS accesses are done, then the barrier; every wave runs ntiles + 1 of them
  auto tile_barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto share_sum = [&](int c, int m) {  // 16 bytes per lane of -V'
    f32x4 x = *(const f32x4*)(part[c & 1][0] + 256 * m + 4 * lane);
#pragma unroll
    for (int i = 1; i < KT; ++i) x += *(const f32x4*)(part[c & 1][i] + 256 * m + 4 * lane);
    return x;
  };

  if (wave >= KT) {
    const int k = wave - KT;
    float* const sp0 = w.st + b * w.st_sb + (long long)hv * D * D + (32 * k + 4 * h) * D + cu + l32;
    // the lines of a tile that this window brings in: W's slice, U's window and the row vectors from wave
    // KT, its share of K^T from wave KT + 1
    auto touch = [&](int c) {
      if (c >= ntiles) return;
      const char* const hd = hd0 + c * step;
      if (k == 0) {
        scan_touch(hd + 4096 * (h ? KT + win : win) + 128 * l32, touched);
        if (lane < 4) scan_touch(hd + 2 * KT * 4096 + 4096 + 128 * lane, touched);
      } else if (k == 1) {
        if (h == 0) scan_touch(kt0 + c * kstep + 4096 * win + 128 * l32, touched);
      }
    };
    for (int c = 2; c < FORK32_AHEAD; ++c) touch(c);
    for (int c = 0; c <= ntiles; ++c) {
      touch(c + FORK32_AHEAD);
      tile_barrier();
      if (c < ntiles) {
        for (int m = k; m < 4; m += KT)
          *(f32x4*)(hd0 + c * step + 4096 * (KT + win) + 1024 * m + 16 * lane) = -share_sum(c, m);
      }
      if (c > 0) {
        Frag<false> x;
        f32_load((const char*)snap[(c - 1) & 1][k], lane, x);
        float* const sp = sp0 + (long long)(c - 1) * a.Hv * D * D;
#pragma unroll
        for (int v = 0; v < 16; ++v) sp[rho(v, 0) * D] = x.v[v];
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no touch in flight past the wave's end
    return;
  }

  f32x16 S = zero16();
  if (w.cin) {
    const float* ip = w.cin + b * w.cin_sb + (long long)hv * D * D + 32 * wave * D + cu + l32;
#pragma unroll
    for (int v = 0; v < 16; ++v) S[v] = ip[rho(v, h) * D];
  }
  struct Tile {
    Frag<false> w, k, u;
    f32x4 eglk[4];
    float lam;
  };
  auto load_w = [&](int c, Tile& t) {
    const char* const hd = hd0 + c * step;
    f32_load(hd + 4096 * wave, lane, t.w);
    if (wave == 0) f32_load(hd + 4096 * (KT + win), lane, t.u);
  };
  auto load_k = [&](int c, Tile& t) {
    const float* const vo = (const float*)(hd0 + c * step + 2 * KT * 4096 + 4096);
    f32_rows(vo + F32V_EGLK, h, t.eglk);
    t.lam = vo[F32V_LAM];
    f32_load(kt0 + c * kstep + 4096 * wave, lane, t.k);
  };
  auto tile = [&](int c, Tile& t) {
    f32x16 acc = zero16();  // -V' = W S - U, wave 0's share starting from -U
    if (wave == 0) {
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] = -t.u.v[v];
    }
    Frag<false> fs;
    acc_to_frag(S, fs);
    mma32(acc, t.w, fs);
    f32_store((char*)part[c & 1][wave], lane, acc);
    const int cn = min(c + 2, ntiles - 1);  // past the last tile: reloaded, unused
    load_w(cn, t);
#pragma unroll
    for (int v = 0; v < 16; ++v) S[v] *= t.lam;
    tile_barrier();
    Frag<false> vd;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const f32x4 x = share_sum(c, m);
#pragma unroll
      for (int e = 0; e < 4; ++e) vd.v[4 * m + e] = -x[e] * t.eglk[m][e];
    }
    mma32(S, t.k, vd);
    load_k(cn, t);
    f32_store((char*)snap[c & 1][wave], lane, S);
  };
  Tile t0, t1;
  load_w(0, t0);
  load_k(0, t0);
  load_w(min(1, ntiles - 1), t1);
  load_k(min(1, ntiles - 1), t1);
  for (int c = 0; c < ntiles; c += 2) {
    tile(c, t0);
    if (c + 1 < ntiles) tile(c + 1, t1);
  }
  tile_barrier();
  if (w.cout) {
    float* op = w.cout + ((long long)b * a.Hv + hv) * D * D + 32 * wave * D + cu + l32;
#pragma unroll
    for (int v = 0; v < 16; ++v) op[rho(v, h) * D] = S[v];
  }
}

// Outputs O = diag(e^gamma scale / ||q||) Q S + P (V' / ||k||) of one (sequence, tile, head, stream) and 32
// columns per wave, S the clean state before the tile; the noised V' = U - W S, the clean one is stored. The waves
// of a SIMD hide each other's loads: a slice loaded during the products of the one before takes 134
// registers for 83 and measured 34 against 24 us (B = 1, L = 256, 48 heads of 128).
template <int KT>
__global__ __launch_bounds__(64 * KT) void fork32_out_kernel(GdnArgs a, Fork32Args w) {
  constexpr int HDB = fork32_hdb(KT), D = 32 * KT;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, h = lane >> 5, l32 = lane & 31;
  // an XCD takes consecutive (head, tile) pairs, the noised units first: they form V' as well, 1.8 times the
  // products of a clean unit, and every CU gets some of both
  const int pairs = a.B * a.Hv * w.ntiles, per = gridDim.x >> 4, slot = blockIdx.x >> 3;
  const int s = slot < per;
  int id = (blockIdx.x & 7) * per + (s ? slot : slot - per);
  if (id >= pairs) return;
  const int c = id % w.ntiles;
  id /= w.ntiles;
  const int hv = id % a.Hv, b = id / a.Hv;
  const int hk = hv / (a.Hv / a.Hk);
  const GdnStream& st = a.s[s];
  const int cu = 32 * wave;
  const long long t0 = (long long)c * a.sub;
  const char* const hd = w.hd + (((long long)(b * w.ntiles + c) * a.Hv + hv) * 2 + s) * HDB;
  const float* const sp = c > 0 ? w.st + b * w.st_sb + ((long long)(c - 1) * a.Hv + hv) * D * D
                                : (w.cin ? w.cin + b * w.cin_sb + (long long)hv * D * D : nullptr);
  const float* const vo = (const float*)(hd + 2 * KT * 4096 + 4096);
  float* const op = (float*)st.out + (((long long)b * a.t_rows + t0) * a.Hv + hv) * D + cu + l32;
  const int row = min(l32, a.sub - 1);
  const float* const qp = (const float*)st.q + b * a.q_sb + (long long)hk * a.q_sh + (t0 + row) * a.q_st;
  auto outputs = [&](auto noised) {
    f32x16 qs = zero16(), ws = zero16();
    Frag<false> u, p, vk;
    f32x4 egq[4], rnk[4];
    if (sp) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        Frag<false> fs, fq, fw;
#pragma unroll
        for (int v = 0; v < 16; ++v) fs.v[v] = sp[(32 * kt + rho(v, h)) * D + cu + l32];
        lds_frag(qp + 32 * kt, h, fq);  // rows past the tile's real ones are not stored
        mma32(qs, fq, fs);
        if constexpr (noised) {
          f32_load(hd + 4096 * kt, lane, fw);
          mma32(ws, fw, fs);
        }
      }
    }
    f32_load(hd + 4096 * (KT + wave), lane, u);
    f32_load(hd + 2 * KT * 4096, lane, p);
    f32_rows(vo + F32V_EGQ, h, egq);
    f32_rows(vo + F32V_RNK, h, rnk);
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int v = 4 * m + e;
        vk.v[v] = (noised ? u.v[v] - ws[v] : u.v[v]) * rnk[m][e];
        qs[v] *= egq[m][e];
      }
    mma32(qs, p, vk);
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = rho(v, h);
      if (r < a.sub) op[(long long)r * a.Hv * D] = qs[v];
    }
  };
  if (s) outputs(std::true_type{});
  else outputs(std::false_type{});
}

static long long fork32_operands(int B, int Hk, int Hv, int D) {  // bytes of a tile of every head
  return (long long)B * ((long long)Hv * 2 * fork32_hdb(D / 32) + (long long)Hk * D * 128);
}

// tiles per range and the workspace's bytes; 0 where one tile of all heads passes FORK32_WS_MAX
long long gdn_fork32_workspace(int B, int L, int Hk, int Hv, int D, int block, bool states, int* tiles_per_range) {
  const long long state = (long long)B * Hv * D * D * 4;
  const long long per = fork32_operands(B, Hk, Hv, D) + (states ? 0 : state);
  const int ntiles = L / block;
  if (per > FORK32_WS_MAX) return 0;
  const int most = (int)(FORK32_WS_MAX / per);
  const int nr = (ntiles + most - 1) / most, tpr = (ntiles + nr - 1) / nr;
  if (tiles_per_range) *tiles_per_range = tpr;
  return per * tpr + (nr > 1 && !states ? 2 * state : 0);
}

template <int KT>
static int fork32_range(const GdnArgs& a, const Fork32Args& w, hipStream_t st) {
  const long long preps = (long long)a.B * w.ntiles * a.Hk * 2, chains = (long long)a.B * a.Hv * KT;
  const long long outs = ((long long)a.B * w.ntiles * a.Hv + 7) / 8 * 16;
  if (outs > 0x7fffffff || chains > 0x7fffffff) return fail(DLLM_EUNSUPPORTED, "gdn: grid too large");
  fork32_prep_kernel<KT><<<dim3((unsigned)preps), 64 * KT, 0, st>>>(a, w);
  fork32_state_kernel<KT><<<dim3((unsigned)chains), 128 * KT, 0, st>>>(a, w);
  fork32_out_kernel<KT><<<dim3((unsigned)outs), 64 * KT, 0, st>>>(a, w);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(DLLM_ELAUNCH, "gdn fork32 launch: %s", hipGetErrorString(e));
  return DLLM_OK;
}

int gdn_fork32_launch(const GdnArgs& a0, void* workspace, hipStream_t st) {
  int tpr = 0;
  const int D = a0.Dk;
  gdn_fork32_workspace(a0.B, a0.T, a0.Hk, a0.Hv, D, a0.sub, a0.states != nullptr, &tpr);
  const int ntiles = a0.T / a0.sub;
  const long long snap = (long long)a0.Hv * D * D;
  // operands, then without kept states: the range's states and two carries, used in turn (a range's
  // outputs read the one that its state kernel started from)
  float* const wst = (float*)((char*)workspace + fork32_operands(a0.B, a0.Hk, a0.Hv, D) * tpr);
  float* const carry = wst + (long long)a0.B * tpr * snap;
  for (int c0 = 0, r = 0; c0 < ntiles; c0 += tpr, ++r) {
    const int n = std::min(tpr, ntiles - c0);
    const long long t = (long long)c0 * a0.sub;
    GdnArgs a = a0;
    for (int i = 0; i < 2; ++i) {
      GdnStream& s = a.s[i];
      s.q = (const float*)s.q + t * a.q_st;
      s.k = (const float*)s.k + t * a.k_st;
      s.v = (const float*)s.v + t * a.v_st;
      s.g += t * a.g_st;
      s.beta += t * a.b_st;
      s.out = (float*)s.out + t * a.Hv * a.Dv;
    }
    a.T = n * a.sub;
    Fork32Args w = {};
    w.hd = (char*)workspace;
    w.kt = w.hd + (long long)a.B * n * a.Hv * 2 * fork32_hdb(D / 32);
    w.ntiles = n;
    if (a0.states) {
      w.st = a0.states + c0 * snap;
      w.st_sb = a0.snap_rows * snap;
      w.cin = c0 > 0 ? a0.states + (c0 - 1) * snap : nullptr;
      w.cin_sb = w.st_sb;
    } else {
      w.st = wst;
      w.st_sb = n * snap;
      w.cin = c0 > 0 ? carry + (r & 1) * a0.B * snap : nullptr;
      w.cin_sb = snap;
      w.cout = c0 + n < ntiles ? carry + ((r + 1) & 1) * a0.B * snap : nullptr;
    }
    const int rc = D == 64 ? fork32_range<2>(a, w, st) : fork32_range<4>(a, w, st);
    if (rc != DLLM_OK) return rc;
  }
  return DLLM_OK;
}

}  // namespace dllm
