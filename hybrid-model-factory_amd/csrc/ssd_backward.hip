// Mamba2 SSD chunk scan backward (the gradients of mamba_chunk_scan_combined) for
// gfx950: bf16 MFMA products with fp32 accumulation, fp32 scalar chains.
//
// The forward (ssd_prefill.hip) per head h, chunk of L = 64 tokens, a_t = dt'_t A_h,
// A_t = sum_{s<=t} a_s from the chunk start (inclusive), chunk start state S0 and
// end state S1 (both P x N):
//   y'_t = sum_{s<=t} (C_t . B_s) e^{A_t - A_s} dt'_s x_s + e^{A_t} S0 C_t + D x_t
//   y_t  = y'_t silu(z_t)                        (y_t = y'_t without z)
//   S1   = e^{A_L} S0 + sum_s e^{A_L - A_s} dt'_s x_s B_s^T
// With g_t = dy_t silu(z_t) (dy_t without z), the gradient dS1 of the chunk's end
// state and, for s <= t,
//   M_ts = (C_t . B_s) e^{A_t - A_s},  Q_ts = g_t . x_s,  W_ts = dt'_s Q_ts e^{A_t - A_s}
// the backward is:
//   dS0   = e^{A_L} dS1 + sum_t e^{A_t} g_t C_t^T           (reverse scan over chunks)
//   dx_s  = sum_t M_ts dt'_s g_t + e^{A_L - A_s} dt'_s dS1 B_s + D g_s
//   dC_t  = sum_s W_ts B_s + e^{A_t} S0^T g_t
//   dB_s  = sum_t W_ts C_t + e^{A_L - A_s} dt'_s dS1^T x_s
//   ddt'_s = sum_t M_ts Q_ts + e^{A_L - A_s} x_s . (dS1 B_s)  +  A_h da_s
//   dA_t  (the cumulated log-decay): sum_s W_ts (C_t.B_s) - sum_u W_ut (C_u.B_t)
//           + g_t . (e^{A_t} S0 C_t) - dt'_t e^{A_L - A_t} x_t . (dS1 B_t)
//           + [t = L-1] <dS1, S1>
//   da_s  = sum_{t>=s} dA_t,   dA_h += sum_s dt'_s da_s
//   dz    = dy y' silu'(z),    dD_p += sum_t g_t[p] x_t[p]
//   d dt  = ddt' * [dt_min <= dt' <= dt_max] * (softplus ? sigmoid(dt + bias) : 1)
// with <dS1, S1> = e^{A_L} <dS1, S0> + sum_s dt'_s e^{A_L - A_s} x_s . (dS1 B_s), so
// S1 is never read.  These are the chain rule through the recurrence of
// oracle/ssd.py; mamba_ssm's backward (un-vendored) computes the same gradients
// with its own kernels (training/.../layers/mamba/mamba2.py:555-580 calls it).
//
// Launches over 64-token chunks (rows of a segment table, one chunk each):
//   ssd_bwd_states_kernel (block of rows, direction, head, 64 state rows): every chunk's
//                          start state S0 and end-state gradient dS1, and dS0 of the
//                          sequences' starts; before it, where rows are cut into several
//                          blocks, once more for the blocks' totals
//   ssd_bwd_group_kernel  (chunk, C group): everything else, for the group's heads
//                          in turn, the next head's inputs loading into registers
//                          during the current head's products; where B and C are
//                          grouped alike and there is no z gate
//   ssd_bwd_chunk_kernel  the same without those two conditions
// dC (and dB when B's groups are C's) sum over the workgroup's heads in registers;
// x shared by several heads (HX < H), or B shared wider than a C group, accumulate
// with fp32 atomics; everything else is stored.

#include <type_traits>

#include "common.hpp"
#include "mfma.hpp"
#include "ssd_backward_plan.hpp"

namespace hmx {
namespace ssdb {

constexpr int L = 64;
constexpr int NTHR = 256;

struct Params {
  const bf16* x; int64_t x_ts, x_hs;         // [T][HX][P]
  const bf16* B; int64_t b_ts, b_gs;         // [T][G][N]
  const bf16* C; int64_t c_ts, c_gs;         // [T][GC][N]
  const void* dt; int dt_dt; int64_t dt_ts, dt_hs;   // raw dt [T][H]
  const float* A;                            // [H]
  const float* D;                            // [H][P] or null
  const float* dt_bias;                      // [H] or null
  const bf16* z; int64_t z_ts, z_hs;         // [T][H][P] or null
  const bf16* dy; int64_t dy_ts, dy_hs;      // [T][H][P]
  const float* h0;                           // [nseq][H][P][N] or null (zero start)
  const float* dT;                           // [nseq][H][P][N] end-state gradients, or null
  const int* seg;                            // [nrows][8] segment rows (one chunk each)
  const int* seqs;                           // [nseq][2]: first row, rows
  int nrows, nseq;
  bf16* S0;                                  // ws [nrows][H][P][N]: chunk start states
  bf16* dS1;                                 // ws [nrows][H][P][N]: end-state gradients
  float* tot;                                // ws [2][blocks][H][P][N]: the states launch's
  float* tdec;                               // ws [2][blocks][H]: block totals and decays
  // outputs (contiguous)
  void* dx;    int x_shared;                 // [T][HX][P]
  void* dB;    int b_shared;                 // [T][G][N]
  void* dC;                                  // [T][GC][N]
  int gbf16;                                 // dx, dB, dC stored in bf16 (else fp32)
  bf16* dz;                                  // [T][H][P] or null
  float* ddt;                                // [T][H]
  float* dA;                                 // [H] (accumulated)
  float* dD;                                 // [H][P] (accumulated) or null
  float* dbias;                              // [H] (accumulated) or null
  float* dh0;                                // [nseq][H][P][N] or null
  int H, HX, G, GC, softplus;
  float dt_min, dt_max;
};

// segment row: sequence, first token, end token, chunk range, index in the
// sequence, first row of the sequence, rows of the sequence
struct Row { int n, bos, eos, c0, c1, idx, first, nseg; };
__device__ __forceinline__ Row load_row(const int* seg, int r) {
  const int* q = seg + r * 8;
  return Row{q[0], q[1], q[2], q[3], q[4], q[5], q[6], q[7]};
}

__device__ __forceinline__ float scan64(float x, int lane) {
  x = scan32(x);
  const float lo = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), 31));
  return lane >= 32 ? x + lo : x;
}

__device__ __forceinline__ float silu(float z) { return z * __builtin_amdgcn_rcpf(1.f + fast_exp(-z)); }

// a stored (not accumulated) gradient element, bf16 or fp32
__device__ __forceinline__ void st_grad(void* base, int64_t i, float v, int bf) {
  if (bf) static_cast<bf16*>(base)[i] = (bf16)v;
  else static_cast<float*>(base)[i] = v;
}

// Per-token scalars of a chunk, lane t of one wave: dt' (0 past the chunk's
// tokens), A_t, and the factor d dt'/d dt (clamp pass times the softplus slope).
struct Tok { float dtv, acs, fac; };
// dt prefetched for the next head: its raw bits (one load in either dtype
// branch), converted where the scalars are formed.  Converting at the load (as
// load_any does) would wait there for every load issued before it, the rest of
// the prefetch included.
__device__ __forceinline__ uint32_t ld_bits(const void* p, int64_t i, int dt) {
  if (dt == HMX_F32) return static_cast<const uint32_t*>(p)[i];
  return static_cast<const uint16_t*>(p)[i];
}
__device__ __forceinline__ float bits_f32(uint32_t b, int dt) {
  if (dt == HMX_F32) return __builtin_bit_cast(float, b);
  if (dt == HMX_BF16) return __builtin_bit_cast(float, b << 16);
  return (float)__builtin_bit_cast(f16, (uint16_t)b);
}
__device__ __forceinline__ Tok token_scalars_raw(const Params& p, int h, float dt_raw, int nval,
                                                 int lane) {
  float d = dt_raw + (p.dt_bias ? p.dt_bias[h] : 0.f);
  float sp = d, slope = 1.f;
  if (p.softplus) {
    sp = softplus20(d);
    slope = d > 20.f ? 1.f : 1.f / (1.f + fast_exp(-d));
  }
  float dtv = fminf(fmaxf(sp, p.dt_min), p.dt_max);
  // torch.clamp's gradient passes on [min, max]
  float fac = (sp >= p.dt_min && sp <= p.dt_max) ? slope : 0.f;
  if (lane >= nval) { dtv = 0.f; fac = 0.f; }
  const float acs = scan64(dtv * p.A[h], lane);
  return Tok{dtv, acs, fac};
}
constexpr int row_ld(int w) { return w == 64 ? w + 8 : w + 16; }

// ---------------------------------------------------------------------------
// states: every chunk's start state S0 and the gradient dS1 of its end state, one chain
// over the chunks in either direction (dir 0: S0(c+1) = e^{A_L} S0(c) + sum_s dt'_s
// e^{A_L - A_s} x_s B_s^T, forward; dir 1: dS1(c-1) = e^{A_L} dS1(c) + sum_t e^{A_t} g_t C_t^T,
// backward), held in fp32 MFMA accumulators; each chunk's state is stored in bf16 before
// the chunk is added.
//
// One workgroup per (block of Lr table rows, direction, head, 64 state rows), eight waves.
// A row that begins its sequence (ends it, backward) resets the chain to h0 (dT), so a
// block may hold several sequences.  Where a sequence crosses blocks, a launch before
// this one (TOT) has left each block's contribution and decay, and the chain starts from
// their sum over the sequence's blocks before it: two reads of x, dy, B and C in place of
// one, so blocks are cut only to fill the chip (see launch).
// What bounds it: memory, and the path to it.  Each chunk's terms as a launch of their
// own, then a scan over them, moved every state through memory twice more than this (a
// chunk's share written, read, its state written): 0.40 + 0.43 ms at 2 x 16384 tokens,
// H = 64, P = 64, N = 128, G = 8, where these chains take 0.49 (1.07 GB written, 0.67 GB
// read: 0.35 at the rate of a copy).  64 state rows per workgroup: with 32, two workgroups
// per CU load and stage every B and C row twice as often, 0.59 ms there.  (0.31 without
// the stores, 0.41 with cached inputs.)
// The loads of SD chunks are in flight; the LDS tiles alternate, one barrier per chunk;
// the scalar chain over a chunk's tokens runs in one wave of four, four chunks at a time.
// LDS: B's (C's) features in the order pos(n) = 32-block | bit 2 of n | bits 4,3 | bits 1,0,
// so that the two 16-row tiles of a 32-feature block leave 8 consecutive features of a
// state row in each lane (one 16-byte store) and the transposing reads stay contiguous.
// ---------------------------------------------------------------------------
constexpr int SP = 64;                    // state rows per workgroup
constexpr int STHR = 512;
constexpr int SD = 4;                     // chunks in flight

template <int N>
struct SLay {
  static constexpr int LDB = row_ld(N), LDX = SP + 16;      // rows 72 (36) and 40 dwords apart
  static constexpr int SZ_B = L * LDB, SET = SZ_B + L * LDX;   // elements
  static constexpr int SW = L + 4;                          // a chunk's weights and its decay
};

// One chunk's inputs in flight.
template <int N>
struct StateIn {
  bf16x8 m[L * N / 8 / STHR], x, z;
  int nval, fl, n, r;                     // tokens, row begins (1) / ends (2) a sequence, its n, row
};

template <int P, int N, bool TOT>
__global__ __launch_bounds__(STHR, 2) void ssd_bwd_states_kernel(Params p, int Lr, int nblk) {
  using Y = SLay<N>;
  constexpr int VB = L * N / 8 / STHR, TPR = N / 8;          // 16-byte pieces of a B row
  constexpr int NB = N / 32, PBW = N / 64;                   // 32-feature blocks; p tiles per wave
  __shared__ __align__(16) bf16 lds[2 * Y::SET];
  __shared__ __align__(16) float sW[8 * Y::SW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q4 = lane >> 4, l16 = lane & 15;
  const int H = p.H;
  const int tot = gridDim.x, id = blockIdx.x;
  int u = tot % 8 ? id : (id % 8) * (tot / 8) + id / 8;      // consecutive units on one XCD
  const int p0 = (u % (P / SP)) * SP;
  u /= P / SP;
  const int h = u % H;
  u /= H;
  const int dir = u & 1, b = u >> 1;
  int ra = b * Lr, rb = min(ra + Lr, p.nrows);
  if constexpr (TOT) {
    // needed by a block after (before) this one only if a sequence crosses into it; only
    // the crossing sequence's rows count
    if (dir == 0) {
      if (rb >= p.nrows) return;
      const Row nx = load_row(p.seg, rb);
      if (nx.idx == 0) return;
      ra = max(ra, nx.first);
    } else {
      if (ra == 0) return;
      const Row ro = load_row(p.seg, ra);
      if (ro.idx == 0) return;
      rb = min(rb, ro.first + ro.nseg);
    }
  }
  const int cnt = rb - ra;
  const int nb = wave % NB, pb0 = (wave / NB) * PBW;
  // this lane's part of the state: rows p0 + 16 (pb0 + i) + l16, features n_l .. n_l + 7
  const int n_l = 32 * nb + 8 * q4;
  const auto pn = [&](int i) { return (p0 + 16 * (pb0 + i) + l16) * N + n_l; };
  f32x4 X[PBW][2];
  const auto load_state = [&](const float* s) {     // [P][N] fp32, or null
#pragma unroll
    for (int i = 0; i < PBW; ++i)
#pragma unroll
      for (int a = 0; a < 2; ++a)
        X[i][a] = s ? *reinterpret_cast<const f32x4*>(s + pn(i) + 4 * a) : f32x4{0.f, 0.f, 0.f, 0.f};
  };
  const auto store_state = [&](float* s) {
#pragma unroll
    for (int i = 0; i < PBW; ++i)
#pragma unroll
      for (int a = 0; a < 2; ++a) *reinterpret_cast<f32x4*>(s + pn(i) + 4 * a) = X[i][a];
  };
  const float* init = dir ? p.dT : p.h0;
  const auto init_of = [&](int n) { return init ? init + ((int64_t)n * H + h) * P * N : nullptr; };
  const auto tot_at = [&](int j) { return p.tot + (((int64_t)dir * nblk + j) * H + h) * P * N; };
  const auto dec_at = [&](int j) -> float& { return p.tdec[((int64_t)dir * nblk + j) * H + h]; };
  load_state(nullptr);
  if (!TOT && b == 0 && dir == 1 && p.dh0) {
    // sequences without tokens: dh0 = dT
    for (int n0 = 0; n0 < p.nseq; n0 += 64) {
      uint64_t e = __ballot(n0 + lane < p.nseq && p.seqs[2 * min(n0 + lane, p.nseq - 1) + 1] == 0);
      for (; e; e &= e - 1) {
        const int n = n0 + __builtin_ctzll(e);
        load_state(init_of(n));
        store_state(p.dh0 + ((int64_t)n * H + h) * P * N);
      }
    }
    load_state(nullptr);
  }
  if (cnt <= 0) return;
  if (!TOT && nblk > 1) {
    // the sequence's blocks before this one
    const Row ro = load_row(p.seg, dir ? rb - 1 : ra);
    const int end = ro.first + ro.nseg - 1;
    const int j0 = dir ? end / Lr : ro.first / Lr;
    for (int j = j0; j != b; j += dir ? -1 : 1) {
      const float d = j == j0 ? 0.f : dec_at(j);
      const float* t = tot_at(j);
#pragma unroll
      for (int i = 0; i < PBW; ++i)
#pragma unroll
        for (int a = 0; a < 2; ++a)
          X[i][a] = X[i][a] * d + *reinterpret_cast<const f32x4*>(t + pn(i) + 4 * a);
    }
  }

  const bf16* mat = dir ? p.C + (int64_t)(h / (H / p.GC)) * p.c_gs : p.B + (int64_t)(h / (H / p.G)) * p.b_gs;
  const int64_t m_ts = dir ? p.c_ts : p.b_ts;
  const bf16* src = (dir ? p.dy + (int64_t)h * p.dy_hs : p.x + (int64_t)(h / (H / p.HX)) * p.x_hs) + p0;
  const int64_t s_ts = dir ? p.dy_ts : p.x_ts;
  const bool has_z = dir && p.z;
  const bf16* zs = has_z ? p.z + (int64_t)h * p.z_hs + p0 : nullptr;
  const bool f32dt = p.dt_dt == HMX_F32;
  const uint16_t* dts = static_cast<const uint16_t*>(p.dt);
  const float bias = p.dt_bias ? p.dt_bias[h] : 0.f, A_h = p.A[h];
  const int tx = tid / (SP / 8), cx = (tid % (SP / 8)) * 8;               // this thread's piece of x
  const int tm = tid / TPR, cm = (tid % TPR) * 8;            // and of B: rows tm + i STHR / TPR

  // The scalars of a chunk (its tokens' weights, its decay), a serial chain over the 64
  // lanes, are formed four chunks at a time, one per wave (waves w and w + 4 alike), two
  // groups of four ahead of the chunk (loads of dt) and one group ahead (the chain); sW
  // holds two groups.
  const auto row_of = [&](int m) { return dir ? rb - 1 - m : ra + m; };
  struct Span { int bos, eos; };
  struct Dt { uint16_t lo, hi; int nv; };  // dt of token `lane` as stored (an fp32's halves)
  const auto scal_row = [&](int grp) {     // of this wave's chunk of a group
    const int* r = p.seg + (int64_t)row_of(min(4 * grp + (wave & 3), cnt - 1)) * 8;
    return Span{r[1], r[2]};
  };
  const auto scal_fetch = [&](const Span& g) {
    const int nv = g.eos - g.bos;
    const int64_t t = nv > 0 ? g.bos + min(lane, nv - 1) : 0;      // (a row without tokens: any)
    const int64_t di = t * p.dt_ts + (int64_t)h * p.dt_hs;
    return Dt{dts[f32dt ? 2 * di : di], dts[f32dt ? 2 * di + 1 : di], nv};
  };
  const auto scal_form = [&](const Dt& g, int grp) {
    const uint32_t lo = g.lo, hi = g.hi;
    float dtv = (f32dt ? __builtin_bit_cast(float, lo | (hi << 16)) : bits_f32(lo, p.dt_dt)) + bias;
    if (p.softplus) dtv = softplus20(dtv);
    dtv = fminf(fmaxf(dtv, p.dt_min), p.dt_max);
    if (lane >= g.nv) dtv = 0.f;
    const float acs = scan64(dtv * A_h, lane);
    const float aend = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, acs), 63));
    float* o = sW + (4 * (grp & 1) + (wave & 3)) * Y::SW;
    o[lane] = dir ? fast_exp(acs) : dtv * fast_exp(aend - acs);
    if (lane == 0) o[L] = expf(aend);
  };

  // rows of the table, 64 chain positions at a time across the lanes
  int i_n = 0, i_bos = 0, i_nv = 0, i_fl = 0;
  const int64_t xo = tx * s_ts + cx, mo = tm * m_ts + cm, mi = (STHR / TPR) * m_ts, zo = tx * p.z_ts + cx;
  const auto fetch = [&](StateIn<N>& q, int m) {
    // past the last chunk: that one again (a load that may be skipped cannot be counted,
    // and the waits for the chunks in flight would be waits for all of them)
    const bool fresh = (m & 63) == 0 && m < cnt;
    m = min(m, cnt - 1);
    if (fresh) {
      const Row ro = load_row(p.seg, row_of(min(m + lane, cnt - 1)));
      i_n = ro.n;
      i_nv = ro.eos - ro.bos;
      i_bos = i_nv > 0 ? ro.bos : 0;
      i_fl = (ro.idx == 0 ? 1 : 0) | (ro.idx == ro.nseg - 1 ? 2 : 0);
    }
    const int64_t tok0 = __builtin_amdgcn_readlane(i_bos, m & 63);
    q.nval = __builtin_amdgcn_readlane(i_nv, m & 63);
    q.fl = __builtin_amdgcn_readlane(i_fl, m & 63);
    q.n = __builtin_amdgcn_readlane(i_n, m & 63);
    q.r = row_of(m);
    const bf16* sb = src + tok0 * s_ts;
    const bf16* mb = mat + tok0 * m_ts;
    int64_t ox = xo, oz = zo, om[VB];
#pragma unroll
    for (int i = 0; i < VB; ++i) om[i] = mo + i * mi;
    if (q.nval < L) {
      // rows past the chunk's tokens load its last one; their x is dropped where it is staged
      const int last = max(q.nval - 1, 0);
      ox = min(tx, last) * s_ts + cx;
      oz = min(tx, last) * p.z_ts + cx;
#pragma unroll
      for (int i = 0; i < VB; ++i) om[i] = min(tm + i * (STHR / TPR), last) * m_ts + cm;
    }
    q.x = *reinterpret_cast<const bf16x8*>(sb + ox);
#pragma unroll
    for (int i = 0; i < VB; ++i) q.m[i] = *reinterpret_cast<const bf16x8*>(mb + om[i]);
    if (has_z) q.z = *reinterpret_cast<const bf16x8*>(zs + tok0 * p.z_ts + oz);
  };

  float ldec = 1.f;                       // decay over the rows walked (TOT)
  const auto step = [&](StateIn<N>& q, int m) {
    bf16* sM = lds + (m & 1) * Y::SET;
    bf16* sX = sM + Y::SZ_B;
    const float* sw = sW + (m & 7) * Y::SW;
    const float wt = sw[tx], dec = sw[L];
    if (q.fl & (dir ? 2 : 1)) {
      load_state(init_of(q.n));
#pragma unroll
      for (int i = 0; i < PBW; ++i)
#pragma unroll
        for (int a = 0; a < 2; ++a) asm volatile("" : "+v"(X[i][a]));   // waited for here only
    }
    if constexpr (!TOT) {
      bf16* dst = (dir ? p.dS1 : p.S0) + ((int64_t)q.r * H + h) * P * N;
#pragma unroll
      for (int i = 0; i < PBW; ++i)
        *reinterpret_cast<bf16x8*>(dst + pn(i)) =
            bf16x8{(bf16)X[i][0][0], (bf16)X[i][0][1], (bf16)X[i][0][2], (bf16)X[i][0][3],
                   (bf16)X[i][1][0], (bf16)X[i][1][1], (bf16)X[i][1][2], (bf16)X[i][1][3]};
    } else {
      ldec *= dec;
    }
    {
      float v[8];
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (float)q.x[j];
      if (has_z) {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] *= silu((float)q.z[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (bf16)(tx < q.nval ? v[j] * wt : 0.f);
      *reinterpret_cast<bf16x8*>(sX + tx * Y::LDX + cx) = o;
#pragma unroll
      for (int i = 0; i < VB; ++i) {
        bf16* d = sM + (tm + i * (STHR / TPR)) * Y::LDB + (cm & ~31) + ((cm & 24) >> 1);
        const bf16x8 y = q.m[i];
        *reinterpret_cast<bf16x4*>(d) = bf16x4{y[0], y[1], y[2], y[3]};
        *reinterpret_cast<bf16x4*>(d + 16) = bf16x4{y[4], y[5], y[6], y[7]};
      }
    }
    const int fl = q.fl, n = q.n;
    fetch(q, m + SD);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < PBW; ++i)
#pragma unroll
      for (int a = 0; a < 2; ++a) X[i][a] *= dec;
#pragma unroll
    for (int k0 = 0; k0 < L; k0 += 32) {
      bf16x8 fa[2], fx[PBW];
#pragma unroll
      for (int a = 0; a < 2; ++a) fa[a] = frag_t_perm(sM, Y::LDB, k0, 32 * nb + 16 * a, lane);
#pragma unroll
      for (int i = 0; i < PBW; ++i) fx[i] = frag_t_perm(sX, Y::LDX, k0, 16 * (pb0 + i), lane);
#pragma unroll
      for (int i = 0; i < PBW; ++i)
#pragma unroll
        for (int a = 0; a < 2; ++a) X[i][a] = mfma16(fa[a], fx[i], X[i][a]);
    }
    if (!TOT && dir && (fl & 1) && p.dh0) store_state(p.dh0 + ((int64_t)n * H + h) * P * N);
  };
  static_assert(SD == 4, "one group of scalars per pass of the loop");
  const Span r0 = scal_row(0), r1 = scal_row(1);
  Span rn = scal_row(2);
  const Dt d0 = scal_fetch(r0);
  Dt dn = scal_fetch(r1);
  StateIn<N> q[SD];
#pragma unroll
  for (int j = 0; j < SD; ++j) {
    fetch(q[j], j);
    __builtin_amdgcn_sched_barrier(0);    // in this order: the loop's waits count on it
  }
  scal_form(d0, 0);
  lds_barrier();
  for (int m = 0;;) {
    scal_form(dn, m / 4 + 1);
    dn = scal_fetch(rn);
    rn = scal_row(m / 4 + 3);
    step(q[0], m);
    if (++m == cnt) break;
    step(q[1], m);
    if (++m == cnt) break;
    step(q[2], m);
    if (++m == cnt) break;
    step(q[3], m);
    if (++m == cnt) break;
  }
  if constexpr (TOT) {
    store_state(tot_at(b));
    if (p0 == 0 && tid == 0) dec_at(b) = ldec;
  }
}

// ---------------------------------------------------------------------------
// chunk kernel where B and C are grouped alike (G == GC) and there is no z gate:
// one workgroup of eight waves per (chunk, group), the group's heads in turn.
//
// Everything that depends on B and C alone is formed once per workgroup and held in
// registers: C B^T (its tiles of the wave), B as an MFMA operand, and B and C at the
// positions of the wave's gradient tiles.  Per head there remain five products,
//   Q = g x^T, g S0, x dS1, dS1 B^T and g^T (M dt'),
// where the general kernel below issues nine, because
//   - sum_h W_h B = (sum_h W_h) B and sum_h W_h^T C = (sum_h W_h)^T C: W is summed over
//     the heads in fp32 registers and its products are formed once per group;
//   - g_t . (S0 C_t) = C_t . (S0^T g_t) and x_s . (dS1 B_s) = B_s . (dS1^T x_s): the
//     decay gradient's state terms are dot products of rows that dC and dB need
//     anyway, so C S0^T is not formed and no x or g is read back;
//   - sum_t W_ts (C_t.B_s) = dt'_s sum_t M_ts Q_ts: one column sum serves both.
// Tiles: wave w holds token block w & 3 and half w >> 2 of the other dimension (key
// blocks of Q, p blocks of dx, n blocks of dC and dB).  Q and dx are formed transposed,
// so M goes to LDS and dx to memory as four consecutive elements per lane.
// LDS rows are 36 or 72 dwords in the interleaved feature order (mfma.hpp): row and
// transposing fragment reads are conflict-free.  At headdim 64 two sets of a head's
// tiles alternate: the next head is staged while this head's dx is formed (two
// barriers per head); at 128 one set fits, and the next head's loads are issued late,
// after the products whose tiles leave no registers for them.
// What bounds it: latency at two waves per SIMD, then memory (1.8 GB read and 0.45 GB
// written at 2 x 16384 tokens, H = 64, P = 64, N = 128, G = 8: 0.44 ms at the rate of a
// copy; S0 and dS1, 16 KB each per head and chunk, are 1.07 GB of it).  Measured there:
// 0.75 ms where ssd_bwd_chunk_kernel (four waves per CU, nine products, scalar LDS
// reads) takes 1.96.  In forward + backward, both with the chunk states still formed by
// two launches: 3.14 against 1.95 ms; at 8 x 4096 tokens, H = 32, P = N = 128 with 1, 4
// or 8 heads per group 3.13 against 2.27, 2.76 against 2.00, 2.70 against 1.97 ms; at
// 2 x 8192, H = 64, P = 64 with one head per group 2.17 against 1.47 ms.  (With the state
// chains 1.56 ms there and 1.82 at 8 x 4096 with one head per group.)
// ---------------------------------------------------------------------------
constexpr int GTHR = 512;

template <int P, int N>
struct GLay {
  static constexpr int LDP = row_ld(P), LDN = row_ld(N), LDM = row_ld(L);
  static constexpr int NSET = P == 64 ? 2 : 1;
  static constexpr int OFF_X = 0;                           // x    [L][LDP]
  static constexpr int OFF_G = OFF_X + L * LDP * 2;         // g    [L][LDP]
  static constexpr int OFF_S = OFF_G + L * LDP * 2;         // S0   [P][LDN]
  static constexpr int OFF_DS = OFF_S + P * LDN * 2;        // dS1  [P][LDN]
  static constexpr int OFF_SC = OFF_DS + P * LDN * 2;       // scalars of the head
  // dt', A, e^A, e^{A_L - A}, d dt'/d dt [L] each; D [P]; dD partials [8][P]; <dS1,S0> [8]
  static constexpr int F_D = 5 * L, F_DD = F_D + P, F_HD = F_DD + 8 * P;
  static constexpr int SET = OFF_SC + (F_HD + 8) * 4;
  static constexpr int OFF_M = NSET * SET;                  // M dt' (the heads' W at the end)
  // sums: rows of dt' M Q [2][L], columns of M Q [4][L], C.(S0 g) [2][L], B.(dS1 x) [2][L]
  static constexpr int OFF_R = OFF_M + L * LDM * 2;
  static constexpr int BYTES = OFF_R + 10 * L * 4;
  static_assert(BYTES <= 160 * 1024 && P >= L, "LDS budget");
};

// row and transposed fragments of interleaved bf16 rows (mfma.hpp)
__device__ __forceinline__ bf16x8 fr(const bf16* b, int ld, int r0, int k0, int lane) {
  return __builtin_bit_cast(bf16x8, frag_i(reinterpret_cast<const f16*>(b), ld, r0, k0, lane));
}
// transposed fragment (frag_t_i) of rows t0.., 16-column block c0 + c (c0 even, or c 0):
// a compile-time c stays an immediate offset
__device__ __forceinline__ bf16x8 fr_t(const bf16* b, int ld, int t0, int c0, int c, int lane) {
  const bf16* a = b + (4 * (lane >> 4) + ((lane & 15) >> 2)) * ld + icol4(c0, lane & 3) +
                  t0 * ld + icol4(c, 0);
  typedef __attribute__((address_space(3))) s16x4* lds4;
  const bf16x4 x = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(a)));
  const bf16x4 y = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(a + 16 * ld)));
  return bf16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
}
__device__ __forceinline__ void st8(bf16* row, int f0, const bf16x8& y) {
  store8_i(reinterpret_cast<f16*>(row), f0, __builtin_bit_cast(f16x8, y));
}

// Raw buffer resource over rows 0 .. nrows-1 (w elements of `es` bytes, ts elements
// apart): past its end nothing is read (zeros) or written.  The host keeps 64 rows of
// any stride inside 31-bit offsets.  Where ts < w (0: an operand constant over the
// tokens) the rows after nrows-1 overlap the ones before, so a load names them missing
// by row_off, not by their place.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const void* base, int nrows, int64_t ts,
                                                           int w, int es) {
  const uint32_t bytes = nrows > 0 ? (uint32_t)(((int64_t)(nrows - 1) * ts + w) * es) : 0u;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
constexpr uint32_t ROW_OFF = 1u << 31;    // past any resource
// byte offset of feature c of row t of a bf16 operand, past the resource's end for rows
// t >= nval (a select, not a branch: the loads stay countable)
__device__ __forceinline__ uint32_t row_off(int t, int64_t ts, int c, int nval) {
  return t < nval ? (uint32_t)((t * ts + c) * 2) : ROW_OFF;
}
__device__ __forceinline__ bf16x8 ld_row(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// One head's inputs for the chunk, in flight while the heads before it are computed.
template <int P, int N>
struct GroupIn {
  static constexpr int VX = L * P / 8 / GTHR, VS = P * N / 8 / GTHR;
  bf16x8 x[VX], dy[VX], s0[VS], ds[VS];
  uint32_t dt;   // of token `lane` (wave 0), as stored: converted where it is used
  float d;       // D of feature tid (tid < P)
};

template <int P, int N>
__global__ __launch_bounds__(GTHR, 2) void ssd_bwd_group_kernel(Params p) {
  using K = GLay<P, N>;
  using In = GroupIn<P, N>;
  constexpr int LDP = K::LDP, LDN = K::LDN, LDM = K::LDM;
  constexpr int VX = In::VX, VS = In::VS, VB = L * N / 8 / GTHR;
  constexpr int PW = P / 32, NW = N / 32;   // p and n blocks per wave
  constexpr int RX = GTHR / (P / 8), RS = GTHR / (N / 8);   // rows per staging pass
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q4 = lane >> 4, l16 = lane & 15;
  const int tb = wave & 3, half = wave >> 2;
  bf16* sM = reinterpret_cast<bf16*>(smem + K::OFF_M);
  float* sR = reinterpret_cast<float*>(smem + K::OFF_R);
  const auto set_bf = [&](int b, int off) { return reinterpret_cast<bf16*>(smem + b * K::SET + off); };
  const auto set_sc = [&](int b) { return reinterpret_cast<float*>(smem + b * K::SET + K::OFF_SC); };
  const auto at4 = [&](const float* f, int t) { return *reinterpret_cast<const f32x4*>(f + t); };

  const int H = p.H, GC = p.GC, HC = H / GC, HXS = H / p.HX;
  const int r = blockIdx.x / GC, gc = blockIdx.x % GC;
  const Row ro = load_row(p.seg, r);
  const int tok0 = ro.bos, nval = ro.eos - ro.bos;
  const int h_first = gc * HC;

  // B and C rows of the chunk into two sets of registers
  const auto fetch_bc = [&](int tid, bf16x8* bv, bf16x8* cv) {
    const auto rb = rows_rsrc(p.B + (int64_t)tok0 * p.b_ts + (int64_t)gc * p.b_gs, nval, p.b_ts, N, 2);
    const auto rc = rows_rsrc(p.C + (int64_t)tok0 * p.c_ts + (int64_t)gc * p.c_gs, nval, p.c_ts, N, 2);
#pragma unroll
    for (int i = 0; i < VB; ++i) {
      const int t = i * RS + tid / (N / 8), c = (tid % (N / 8)) * 8;
      bv[i] = ld_row(rb, row_off(t, p.b_ts, c, nval));
      cv[i] = ld_row(rc, row_off(t, p.c_ts, c, nval));
    }
  };
  const auto fetch = [&](int tid, int h, In& q) {
    const int lane = tid & 63;
    const auto rx = rows_rsrc(p.x + (int64_t)tok0 * p.x_ts + (int64_t)(h / HXS) * p.x_hs, nval, p.x_ts, P, 2);
    const auto ry = rows_rsrc(p.dy + (int64_t)tok0 * p.dy_ts + (int64_t)h * p.dy_hs, nval, p.dy_ts, P, 2);
#pragma unroll
    for (int i = 0; i < VX; ++i) {
      const int t = i * RX + tid / (P / 8), c = (tid % (P / 8)) * 8;
      q.x[i] = ld_row(rx, row_off(t, p.x_ts, c, nval));
      q.dy[i] = ld_row(ry, row_off(t, p.dy_ts, c, nval));
    }
    const bf16* s0 = p.S0 + ((int64_t)r * H + h) * P * N;
    const bf16* ds = p.dS1 + ((int64_t)r * H + h) * P * N;
#pragma unroll
    for (int i = 0; i < VS; ++i) {
      q.s0[i] = *reinterpret_cast<const bf16x8*>(s0 + (i * GTHR + tid) * 8);
      q.ds[i] = *reinterpret_cast<const bf16x8*>(ds + (i * GTHR + tid) * 8);
    }
    q.dt = (wave == 0 && lane < nval)
               ? ld_bits(p.dt, (int64_t)(tok0 + lane) * p.dt_ts + (int64_t)h * p.dt_hs, p.dt_dt) : 0u;
    q.d = (p.D && tid < P) ? p.D[(int64_t)h * P + tid] : 0.f;
  };
  In in;
  // in flight after head h's inputs: the next head, or after the last one B and C again
  // (in the registers of S0 and dS1) for the products at the end
  const auto fetch_next = [&](int tid, int h) {
    if (h < h_first + HC) fetch(tid, h, in);
    else fetch_bc(tid, in.s0, in.ds);
  };

  // ---- B and C through the S0 / dS1 tiles of set 0 into registers ------------------
  const auto stage_bc = [&](const bf16x8* bv, const bf16x8* cv, bf16* sb, bf16* sc) {
#pragma unroll
    for (int i = 0; i < VB; ++i) {
      const int t = i * RS + tid / (N / 8), c = (tid % (N / 8)) * 8;
      st8(sb + t * LDN, c, bv[i]);
      st8(sc + t * LDN, c, cv[i]);
    }
  };
  bf16x8 bfr[N / 32];        // B rows of token block tb (an operand of dS1 B^T)
  f32x4 cbt[2], wsum[2];     // (C B^T)^T and sum_h W_h^T, key block 2 half + j, query block tb
  bf16x4 creg[NW], breg[NW];  // C and B at rows 16 tb + 4 q4 + v, columns 16 (half NW + j) + l16
  f32x4 dC[NW], dB[NW];
  {
    bf16* sb = set_bf(0, K::OFF_S);
    bf16* sc = set_bf(0, K::OFF_DS);
    bf16x8 bv[VB], cv[VB];
    fetch_bc(tid, bv, cv);
    fetch(tid, h_first, in);
    stage_bc(bv, cv, sb, sc);
    // the tiles above the diagonal that M's products read (key block 1 of query block
    // 0, 3 of 2) stay zero
    if ((wave == 0 || wave == 2) && lane < 32) {
      const int t = 16 * wave + (lane >> 1), c = 16 * wave + 16 + 8 * (lane & 1);
      st8(sM + t * LDM, c, bf16x8{});
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < N / 32; ++k) bfr[k] = fr(sb, LDN, 16 * tb, 32 * k, lane);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      cbt[j] = wsum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < N / 32; ++k)
        cbt[j] = mfma16(fr(sb, LDN, 16 * (2 * half + j), 32 * k, lane), fr(sc, LDN, 16 * tb, 32 * k, lane), cbt[j]);
    }
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      dC[j] = dB[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int e = (16 * tb + 4 * q4 + v) * LDN + icol(16 * (half * NW + j) + l16);
        creg[j][v] = sc[e];
        breg[j][v] = sb[e];
      }
    }
    lds_barrier();   // set 0 is free again
  }

  // ---- one head's registers into set b: tiles, token scalars, D, the partial sums of
  // dD = sum_t g_t x_t and <dS1, S0> of each wave --------------------------------------
  const auto stage = [&](int tid, int b, int h) {
    const int lane = tid & 63, l16 = lane & 15;
    bf16 *sX = set_bf(b, K::OFF_X), *sG = set_bf(b, K::OFF_G);
    bf16 *sS = set_bf(b, K::OFF_S), *sDS = set_bf(b, K::OFF_DS);
    float* sf = set_sc(b);
    float dd[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < VX; ++i) {
      const int t = i * RX + tid / (P / 8), c = (tid % (P / 8)) * 8;
      st8(sX + t * LDP, c, in.x[i]);
      st8(sG + t * LDP, c, in.dy[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) dd[j] += (float)in.dy[i][j] * (float)in.x[i][j];
    }
    float hd = 0.f;
#pragma unroll
    for (int i = 0; i < VS; ++i) {
      const int e = (i * GTHR + tid) * 8;
      st8(sS + (e / N) * LDN, e % N, in.s0[i]);
      st8(sDS + (e / N) * LDN, e % N, in.ds[i]);
#pragma unroll
      for (int j = 0; j < 8; j += 2)
        hd = __builtin_amdgcn_fdot2_f32_bf16(bf16x2{in.s0[i][j], in.s0[i][j + 1]},
                                             bf16x2{in.ds[i][j], in.ds[i][j + 1]}, hd, false);
    }
    if (p.dD) {
      // over the wave's lanes of the same eight features: halving the values at each
      // exchange; lane l ends with feature 4 (l >> 5) + 2 (l >> 4 & 1) (+ (l >> 3 & 1))
#pragma unroll
      for (int j = 0; j < 4; ++j) dd[j] = pair_sum32(dd[j], dd[j + 4]);
#pragma unroll
      for (int j = 0; j < 2; ++j) dd[j] = pair_sum16(dd[j], dd[j + 2]);
      float* o = sf + K::F_DD + wave * P + 4 * (lane >> 5) + 2 * ((lane >> 4) & 1);
      if constexpr (P == 64) {
        const bool up = lane & 8;
        o[(lane & 7) * 8 + ((lane >> 3) & 1)] = (up ? dd[1] : dd[0]) + dppf<0x128>(up ? dd[0] : dd[1]);
      } else {
        o[l16 * 8] = dd[0];
        o[l16 * 8 + 1] = dd[1];
      }
    }
    hd = wave_sum_v(hd);
    if (lane == 0) sf[K::F_HD + wave] = hd;
    if (tid < P) sf[K::F_D + tid] = in.d;
    if (wave == 0) {
      const Tok tk = token_scalars_raw(p, h, bits_f32(in.dt, p.dt_dt), nval, lane);
      const float aend = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, tk.acs), 63));
      sf[lane] = tk.dtv;
      sf[L + lane] = tk.acs;
      sf[2 * L + lane] = fast_exp(tk.acs);
      sf[3 * L + lane] = fast_exp(aend - tk.acs);
      sf[4 * L + lane] = tk.fac;
    }
  };

  stage(tid, 0, h_first);
  if constexpr (K::NSET == 2) fetch_next(tid, h_first + 1);
  lds_barrier();

#pragma unroll 1
  for (int ih = 0; ih < HC; ++ih) {
    // opaque per head: the lane's LDS offsets are formed again instead of being hoisted
    // out of the loop into registers that the tiles need
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63, q4 = lane >> 4, l16 = lane & 15;
    const int h = h_first + ih, b = K::NSET == 2 ? (ih & 1) : 0;
    const bf16 *sX = set_bf(b, K::OFF_X), *sG = set_bf(b, K::OFF_G);
    const bf16 *sS = set_bf(b, K::OFF_S), *sDS = set_bf(b, K::OFF_DS);
    const float* sf = set_sc(b);
    if (p.dD && tid < P) {
      float s = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) s += sf[K::F_DD + w * P + tid];
      unsafeAtomicAdd(p.dD + (int64_t)h * P + tid, s);
    }
    // ---- Q^T (key rows, query columns), M dt' to LDS, W summed over the heads --------
    {
      float rowr = 0.f;   // sum over the wave's keys of dt'_s M_ts Q_ts, t = 16 tb + l16
      const float acs_t = sf[L + 16 * tb + l16];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int sb = 2 * half + j;
        if (sb > tb) continue;
        f32x4 qq = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < P / 32; ++k)
          qq = mfma16(fr(sX, LDP, 16 * sb, 32 * k, lane), fr(sG, LDP, 16 * tb, 32 * k, lane), qq);
        const f32x4 acs_s = at4(sf + L, 16 * sb + 4 * q4), dt_s = at4(sf, 16 * sb + 4 * q4);
        f32x4 u;
        bf16x4 md;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          float dec = fast_exp(acs_t - acs_s[v]);
          if (sb == tb && 4 * q4 + v > l16) dec = 0.f;
          const float e = dec * dt_s[v];
          u[v] = cbt[j][v] * qq[v] * dec;
          rowr += u[v] * dt_s[v];
          wsum[j][v] += qq[v] * e;
          md[v] = (bf16)(cbt[j][v] * e);
        }
        *reinterpret_cast<bf16x4*>(sM + (16 * tb + l16) * LDM + icol4(sb, q4)) = md;
        const float cs = row16_sum4(u, l16);
        if (l16 < 4) sR[(2 + tb) * L + 16 * sb + 4 * q4 + l16] = cs;
      }
      rowr = pair_sum16(rowr, rowr);
      rowr = pair_sum32(rowr, rowr);
      if (lane < 16) sR[half * L + 16 * tb + lane] = rowr;
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- dC += e^{A_t} g S0 and C_t . (S0^T g_t) ---------------------------------------
    {
      f32x4 acc[NW];
#pragma unroll
      for (int j = 0; j < NW; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < P / 32; ++k) {
        const bf16x8 a = fr(sG, LDP, 16 * tb, 32 * k, lane);
#pragma unroll
        for (int j = 0; j < NW; ++j)
          acc[j] = mfma16(a, fr_t(sS, LDN, 32 * k, half * NW, j, lane), acc[j]);
      }
      const f32x4 ea = at4(sf + 2 * L, 16 * tb + 4 * q4);
      f32x4 ds = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NW; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          ds[v] += (float)creg[j][v] * acc[j][v];
          dC[j][v] += ea[v] * acc[j][v];
        }
      const float s = row16_sum4(ds, l16);
      if (l16 < 4) sR[(6 + half) * L + 16 * tb + 4 * q4 + l16] = s;
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- dB += e dt' x dS1 and B_s . (dS1^T x_s) ---------------------------------------
    {
      f32x4 acc[NW];
#pragma unroll
      for (int j = 0; j < NW; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < P / 32; ++k) {
        const bf16x8 a = fr(sX, LDP, 16 * tb, 32 * k, lane);
#pragma unroll
        for (int j = 0; j < NW; ++j)
          acc[j] = mfma16(a, fr_t(sDS, LDN, 32 * k, half * NW, j, lane), acc[j]);
      }
      const f32x4 e = at4(sf + 3 * L, 16 * tb + 4 * q4), dt = at4(sf, 16 * tb + 4 * q4);
      f32x4 ds = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NW; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          ds[v] += (float)breg[j][v] * acc[j][v];
          dB[j][v] += e[v] * dt[v] * acc[j][v];
        }
      const float s = row16_sum4(ds, l16);
      if (l16 < 4) sR[(8 + half) * L + 16 * tb + 4 * q4 + l16] = s;
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- (dS1 B^T): p rows, key columns --------------------------------------------------
    f32x4 dh[PW];
#pragma unroll
    for (int i = 0; i < PW; ++i) {
      dh[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < N / 32; ++k)
        dh[i] = mfma16(fr(sDS, LDN, 16 * (half * PW + i), 32 * k, lane), bfr[k], dh[i]);
    }
    lds_barrier();   // M and the sums are whole

    if constexpr (K::NSET == 2) {
      if (ih + 1 < HC) {
        stage(tid, b ^ 1, h + 1);
        fetch_next(tid, h + 2);
      }
    } else {
      fetch_next(tid, h + 1);
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- dx^T = g^T (M dt') + e dt' (dS1 B^T) + D g ---------------------------------------
    {
      f32x4 acc[PW];
#pragma unroll
      for (int i = 0; i < PW; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        if (k == 0 && tb >= 2) continue;   // M's tiles above the diagonal
        const bf16x8 m = fr_t(sM, LDM, 32 * k, tb, 0, lane);
#pragma unroll
        for (int i = 0; i < PW; ++i)
          acc[i] = mfma16(fr_t(sG, LDP, 32 * k, half * PW, i, lane), m, acc[i]);
      }
      const int s = 16 * tb + l16, hx = h / HXS;
      const float f = sf[3 * L + s] * sf[s];
      const int es = p.gbf16 ? 2 : 4;
      const auto rx = rows_rsrc(static_cast<char*>(p.dx) + ((int64_t)tok0 * p.HX + hx) * P * es, nval,
                                (int64_t)p.HX * P, P, es);
#pragma unroll
      for (int i = 0; i < PW; ++i) {
        const int c = 16 * (half * PW + i) + 4 * q4;
        const bf16x4 g = *reinterpret_cast<const bf16x4*>(sG + s * LDP + icol4(half * PW, q4) + icol4(i, 0));
        const f32x4 dv = at4(sf + K::F_D, c);
        f32x4 d;
#pragma unroll
        for (int v = 0; v < 4; ++v) d[v] = acc[i][v] + f * dh[i][v] + dv[v] * (float)g[v];
        const uint32_t off = (uint32_t)((s * p.HX * P + c) * es);
        if (p.gbf16) {
          const bf16x4 o = {(bf16)d[0], (bf16)d[1], (bf16)d[2], (bf16)d[3]};
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, o), rx, off, 0, 0);
        } else if (!p.x_shared) {
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, d), rx, off, 0, 0);
        } else if (s < nval) {
          float* o = static_cast<float*>(p.dx) + ((int64_t)(tok0 + s) * p.HX + hx) * P + c;
#pragma unroll
          for (int v = 0; v < 4; ++v) unsafeAtomicAdd(o + v, d[v]);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ---- scalar chain on one wave: dA_t, da (reverse cumsum), d dt, dA_h, d dt_bias -------
    if (wave == (ih & 7)) {
      const int t = lane, tt = t >> 4;
      float cmq = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w)
        if (w >= tt) cmq += sR[(2 + w) * L + t];   // query blocks before the key's hold nothing
      const float dt_t = sf[t];
      const float dds = sf[3 * L + t] * (sR[8 * L + t] + sR[9 * L + t]);
      const float das = sf[2 * L + t] * (sR[6 * L + t] + sR[7 * L + t]);
      float dacs = sR[t] + sR[L + t] - dt_t * cmq + das - dt_t * dds;
      // <dS1, S1> = e^{A_L} <dS1, S0> + sum_s dt'_s e_s x_s . (dS1 B_s), on the last token
      const float tail = wave_sum_v(dt_t * dds);
      float hd = 0.f;
#pragma unroll
      for (int w = 0; w < 8; ++w) hd += sf[K::F_HD + w];
      if (t == L - 1) dacs += sf[2 * L + L - 1] * hd + tail;
      const float incl = scan64(dacs, lane);
      const float total = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, incl), 63));
      const float da = total - incl + dacs;   // sum_{u >= t} dA_u
      const float ddt = (cmq + dds + p.A[h] * da) * sf[4 * L + t];
      if (t < nval) p.ddt[(int64_t)(tok0 + t) * H + h] = ddt;
      const float sa = wave_sum_v(dt_t * da), sbias = wave_sum_v(ddt);
      if (lane == 0) {
        unsafeAtomicAdd(p.dA + h, sa);
        if (p.dbias) unsafeAtomicAdd(p.dbias + h, sbias);
      }
    }
    lds_barrier();   // this head's tiles, M and sums are free; the next head is staged
    if (K::NSET == 1 && ih + 1 < HC) {
      stage(tid, 0, h + 1);
      lds_barrier();
    }
  }

  // ---- dC += (sum_h W) B, dB += (sum_h W)^T C --------------------------------------------
  {
    bf16* sb = set_bf(0, K::OFF_S);
    bf16* sc = set_bf(0, K::OFF_DS);
    stage_bc(in.s0, in.ds, sb, sc);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int kb = 2 * half + j;
      if (kb > tb) continue;
      *reinterpret_cast<bf16x4*>(sM + (16 * tb + l16) * LDM + icol4(kb, q4)) =
          bf16x4{(bf16)wsum[j][0], (bf16)wsum[j][1], (bf16)wsum[j][2], (bf16)wsum[j][3]};
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k == 0 || tb >= 2) {
        const bf16x8 w = fr(sM, LDM, 16 * tb, 32 * k, lane);
#pragma unroll
        for (int j = 0; j < NW; ++j)
          dC[j] = mfma16(w, fr_t(sb, LDN, 32 * k, half * NW, j, lane), dC[j]);
      }
      if (k == 1 || tb < 2) {
        const bf16x8 w = fr_t(sM, LDM, 32 * k, tb, 0, lane);
#pragma unroll
        for (int j = 0; j < NW; ++j)
          dB[j] = mfma16(w, fr_t(sc, LDN, 32 * k, half * NW, j, lane), dB[j]);
      }
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int t = 16 * tb + 4 * q4 + v;
    if (t >= nval) continue;
    const int64_t row = ((int64_t)(tok0 + t) * GC + gc) * N + 16 * half * NW + l16;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      st_grad(p.dC, row + 16 * j, dC[j][v], p.gbf16);
      st_grad(p.dB, row + 16 * j, dB[j][v], p.gbf16);
    }
  }
}

// ---------------------------------------------------------------------------
// chunk kernel for a z gate, or B and C grouped differently
// ---------------------------------------------------------------------------
template <int P, int N>
struct Lay {
  static constexpr int LDX = P + 8, LDB = N + 8, LDM = L + 8;
  static constexpr int OFF_X = 0;                          // x        [L][LDX]
  static constexpr int OFF_G = OFF_X + L * LDX * 2;        // g        [L][LDX]
  // dy and z (for dz) fit only at P = 64; headdim 128 takes no z
  static constexpr int ZW = P == 64 ? L * LDX * 2 : 0;
  static constexpr int OFF_DY = OFF_G + L * LDX * 2;       // dy       [L][LDX] (z only)
  static constexpr int OFF_Z = OFF_DY + ZW;                // z        [L][LDX] (z only)
  static constexpr int OFF_B = OFF_Z + ZW;                 // B        [L][LDB]
  static constexpr int OFF_C = OFF_B + L * LDB * 2;        // C        [L][LDB]
  static constexpr int OFF_S = OFF_C + L * LDB * 2;        // S0       [P][LDB]
  static constexpr int OFF_DS = OFF_S + P * LDB * 2;       // dS1      [P][LDB]
  static constexpr int OFF_M = OFF_DS + P * LDB * 2;       // M dt'    [L][LDM]
  static constexpr int OFF_W = OFF_M + L * LDM * 2;        // W        [L][LDM]
  static constexpr int OFF_F = OFF_W + L * LDM * 2;        // fp32 scalars
  static constexpr int FDD = 16, FDV = 16 + P / L;         // dD and D: P floats each
  static constexpr int NF = 16 + 2 * (P / L);              // scalar arrays of L floats
  static constexpr int BYTES = OFF_F + NF * L * 4 + 64;
  static_assert(BYTES <= 160 * 1024, "LDS budget");
};
// scalar arrays
enum { F_DT, F_ACS, F_EA, F_E, F_FAC, F_ROWR, F_DAS, F_DDS,
       F_CMQ0, F_CR0 = F_CMQ0 + 4 };   // F_CR0 + 4 = 16 arrays, then dD and D (Lay)

// One head's inputs for the chunk, loaded into registers while the head before it
// is computed: x, dy, z rows (2 vectors per thread), S0 and dS1 (4 each), B rows
// (4, when B is not staged once per workgroup), the raw dt of token `lane` (wave 0)
// and D of feature `tid` (tid < 64).
template <int P, int N>
struct HeadIn {
  bf16x8 x[L * P / 8 / NTHR], dy[L * P / 8 / NTHR], z[L * P / 8 / NTHR];
  bf16x8 s0[P * N / 8 / NTHR], ds[P * N / 8 / NTHR], b[L * N / 8 / NTHR];
  uint32_t dt;   // as stored (converted where the scalars are formed)
  float d;
};

template <int P, int N>
__global__ __launch_bounds__(NTHR, 1) void ssd_bwd_chunk_kernel(Params p) {
  static_assert((P == 64 || P == 128) && (N == 64 || N == 128), "tile shape");
  // headdim 64 loads the next head's inputs during the current head's products;
  // at 128 they would not fit in registers beside the products' tiles
  constexpr bool AHEAD = P == 64;
  using K = Lay<P, N>;
  constexpr int LDX = K::LDX, LDB = K::LDB, LDM = K::LDM, NT = N / 16;
  extern __shared__ __align__(16) unsigned char smem[];
  bf16* sX = reinterpret_cast<bf16*>(smem + K::OFF_X);
  bf16* sG = reinterpret_cast<bf16*>(smem + K::OFF_G);
  bf16* sDY = reinterpret_cast<bf16*>(smem + K::OFF_DY);
  bf16* sZ = reinterpret_cast<bf16*>(smem + K::OFF_Z);
  bf16* sB = reinterpret_cast<bf16*>(smem + K::OFF_B);
  bf16* sC = reinterpret_cast<bf16*>(smem + K::OFF_C);
  bf16* sS = reinterpret_cast<bf16*>(smem + K::OFF_S);
  bf16* sDS = reinterpret_cast<bf16*>(smem + K::OFF_DS);
  bf16* sM = reinterpret_cast<bf16*>(smem + K::OFF_M);
  bf16* sW = reinterpret_cast<bf16*>(smem + K::OFF_W);
  float* sF = reinterpret_cast<float*>(smem + K::OFF_F);
  auto F = [&](int a, int t) -> float& { return sF[a * L + t]; };
  float* sHD = sF + K::NF * L;   // [0]: <dS1, S0>

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int q4 = lane >> 4, l16 = lane & 15;
  const int H = p.H, GC = p.GC, HC = H / GC, HB = H / p.G, HXS = H / p.HX;
  // one workgroup per (chunk, C group): the group's HC heads in turn
  const int r = blockIdx.x / GC, gc = blockIdx.x % GC;
  const Row ro = load_row(p.seg, r);
  const int tok0 = ro.bos, nval = ro.eos - ro.bos;
  const int h_first = gc * HC;
  // B staged once when the workgroup's heads are exactly one B group; dB then sums
  // over them in registers.  Otherwise B is per head (stored) or shared wider
  // (atomics).
  const bool b_once = p.G == GC;
  constexpr int VX = L * P / 8 / NTHR, VS = P * N / 8 / NTHR, VB = L * N / 8 / NTHR;

  if (tid == 0) sHD[0] = 0.f;
  if (tid < P) F(K::FDD, tid) = 0.f;
  // C (and B when shared by all the heads) once
#pragma unroll
  for (int i = 0; i < VB; ++i) {
    const int e = (i * NTHR + tid) * 8, t = e / N, c = e % N;
    bf16x8 cv = {}, bv = {};
    if (t < nval) {
      cv = *reinterpret_cast<const bf16x8*>(p.C + (int64_t)(tok0 + t) * p.c_ts + (int64_t)gc * p.c_gs + c);
      if (b_once)
        bv = *reinterpret_cast<const bf16x8*>(p.B + (int64_t)(tok0 + t) * p.b_ts +
                                              (int64_t)(h_first / HB) * p.b_gs + c);
    }
    *reinterpret_cast<bf16x8*>(sC + t * LDB + c) = cv;
    if (b_once) *reinterpret_cast<bf16x8*>(sB + t * LDB + c) = bv;
  }

  const auto fetch = [&](int h, HeadIn<P, N>& q) {
    const int hx = h / HXS, g = h / HB;
#pragma unroll
    for (int i = 0; i < VX; ++i) {
      const int e = (i * NTHR + tid) * 8, t = e / P, c = e % P;
      q.x[i] = q.dy[i] = q.z[i] = bf16x8{};
      if (t < nval) {
        q.x[i] = *reinterpret_cast<const bf16x8*>(p.x + (int64_t)(tok0 + t) * p.x_ts + (int64_t)hx * p.x_hs + c);
        q.dy[i] = *reinterpret_cast<const bf16x8*>(p.dy + (int64_t)(tok0 + t) * p.dy_ts + (int64_t)h * p.dy_hs + c);
        if (p.z) q.z[i] = *reinterpret_cast<const bf16x8*>(p.z + (int64_t)(tok0 + t) * p.z_ts + (int64_t)h * p.z_hs + c);
      }
    }
    const bf16* s0 = p.S0 + ((int64_t)r * H + h) * P * N;
    const bf16* ds = p.dS1 + ((int64_t)r * H + h) * P * N;
#pragma unroll
    for (int i = 0; i < VS; ++i) {
      const int e = (i * NTHR + tid) * 8;
      q.s0[i] = *reinterpret_cast<const bf16x8*>(s0 + e);
      q.ds[i] = *reinterpret_cast<const bf16x8*>(ds + e);
    }
    if (!b_once) {
#pragma unroll
      for (int i = 0; i < VB; ++i) {
        const int e = (i * NTHR + tid) * 8, t = e / N, c = e % N;
        q.b[i] = bf16x8{};
        if (t < nval)
          q.b[i] = *reinterpret_cast<const bf16x8*>(p.B + (int64_t)(tok0 + t) * p.b_ts + (int64_t)g * p.b_gs + c);
      }
    }
    q.dt = (wave == 0 && lane < nval)
               ? ld_bits(p.dt, (int64_t)(tok0 + lane) * p.dt_ts + (int64_t)h * p.dt_hs, p.dt_dt) : 0u;
    q.d = (p.D && tid < P) ? p.D[(int64_t)h * P + tid] : 0.f;
  };

  HeadIn<P, N> in;
  if constexpr (AHEAD) fetch(h_first, in);
  f32x4 dCacc[NT], dBacc[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j) { dCacc[j] = f32x4{0.f, 0.f, 0.f, 0.f}; dBacc[j] = dCacc[j]; }

  for (int ih = 0; ih < HC; ++ih) {
  const int h = h_first + ih, hx = h / HXS, g = h / HB;
  const float A_h = p.A[h];
  if constexpr (!AHEAD) fetch(h, in);

  // ---- staging from registers: x, g = dy silu(z), dy and z with the dD partials;
  // S0 and dS1 with <dS1, S0>; B when per head; the token scalars and D ----------
  {
    float dd[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < VX; ++i) {
      const int e = (i * NTHR + tid) * 8, t = e / P, c = e % P;
      bf16x8 gv;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float gj = (float)in.dy[i][j];
        if (p.z) gj *= silu((float)in.z[i][j]);
        gv[j] = (bf16)gj;
        dd[j] += gj * (float)in.x[i][j];
      }
      *reinterpret_cast<bf16x8*>(sX + t * LDX + c) = in.x[i];
      *reinterpret_cast<bf16x8*>(sG + t * LDX + c) = gv;
      if constexpr (P == 64) {
        if (p.z) {
          *reinterpret_cast<bf16x8*>(sDY + t * LDX + c) = in.dy[i];
          *reinterpret_cast<bf16x8*>(sZ + t * LDX + c) = in.z[i];
        }
      }
    }
    if (p.dD) {
      const int c = (tid * 8) % P;
#pragma unroll
      for (int j = 0; j < 8; ++j) atomicAdd(&F(K::FDD, c + j), dd[j]);
    }
    float hd = 0.f;
#pragma unroll
    for (int i = 0; i < VS; ++i) {
      const int e = (i * NTHR + tid) * 8, pr = e / N, c = e % N;
      *reinterpret_cast<bf16x8*>(sS + pr * LDB + c) = in.s0[i];
      *reinterpret_cast<bf16x8*>(sDS + pr * LDB + c) = in.ds[i];
#pragma unroll
      for (int j = 0; j < 8; ++j) hd += (float)in.s0[i][j] * (float)in.ds[i][j];
    }
    hd = wave_sum(hd);
    if (lane == 0) atomicAdd(sHD, hd);
    if (!b_once) {
#pragma unroll
      for (int i = 0; i < VB; ++i) {
        const int e = (i * NTHR + tid) * 8, t = e / N, c = e % N;
        *reinterpret_cast<bf16x8*>(sB + t * LDB + c) = in.b[i];
      }
    }
    if (tid < P) F(K::FDV, tid) = in.d;
    if (wave == 0) {
      const Tok tk = token_scalars_raw(p, h, bits_f32(in.dt, p.dt_dt), nval, lane);
      const float aend = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, tk.acs), 63));
      F(F_DT, lane) = tk.dtv;
      F(F_ACS, lane) = tk.acs;
      F(F_EA, lane) = fast_exp(tk.acs);
      F(F_E, lane) = fast_exp(aend - tk.acs);
      F(F_FAC, lane) = tk.fac;
    }
  }
  __syncthreads();
  // the next head's inputs load during this head's products (no other vector load
  // is issued until they are used)
  if constexpr (AHEAD) {
    if (ih + 1 < HC) fetch(h + 1, in);
  }
  if (p.dD && tid < P) {
    unsafeAtomicAdd(p.dD + (int64_t)h * P + tid, F(K::FDD, tid));
    F(K::FDD, tid) = 0.f;   // the next head's staging adds after the closing barrier
  }

  // ---- step A: CB and Q (rows t of wave's block, all s), M dt' and W to LDS ----
  {
    f32x4 cb[4], qq[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { cb[j] = f32x4{0.f, 0.f, 0.f, 0.f}; qq[j] = cb[j]; }
#pragma unroll
    for (int k0 = 0; k0 < N; k0 += 32) {
      const bf16x8 a = frag(sC, LDB, 16 * wave, k0, lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) cb[j] = mfma16(a, frag(sB, LDB, 16 * j, k0, lane), cb[j]);
    }
#pragma unroll
    for (int k0 = 0; k0 < P; k0 += 32) {
      const bf16x8 a = frag(sG, LDX, 16 * wave, k0, lane);
#pragma unroll
      for (int j = 0; j < 4; ++j) qq[j] = mfma16(a, frag(sX, LDX, 16 * j, k0, lane), qq[j]);
    }
    float rowr[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int s = 16 * j + l16;
      const float acs_s = F(F_ACS, s), dt_s = F(F_DT, s);
      float cmq = 0.f, cr = 0.f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int t = 16 * wave + 4 * q4 + v;
        const float dec = s <= t ? fast_exp(F(F_ACS, t) - acs_s) : 0.f;
        const float m = cb[j][v] * dec;
        const float w = dt_s * qq[j][v] * dec;
        const float rr = w * cb[j][v];
        cmq += m * qq[j][v];
        cr += rr;
        rowr[v] += rr;
        sM[t * LDM + s] = (bf16)(m * dt_s);
        sW[t * LDM + s] = (bf16)w;
      }
      // column sums over the wave's 16 rows: the four lane groups
      cmq += shfl_xor(cmq, 16);
      cmq += shfl_xor(cmq, 32);
      cr += shfl_xor(cr, 16);
      cr += shfl_xor(cr, 32);
      if (q4 == 0) {
        F(F_CMQ0 + wave, s) = cmq;
        F(F_CR0 + wave, s) = cr;
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float rs = row16_sum(rowr[v]);
      if (l16 == 0) F(F_ROWR, 16 * wave + 4 * q4 + v) = rs;
    }
  }
  __syncthreads();

  // ---- step B1: y' = M dt' x + e^{A_t} C S0^T + D x -> dz, and g . (e^A C S0^T) --
  {
    f32x4 yi[P / 16], ys[P / 16];
#pragma unroll
    for (int i = 0; i < P / 16; ++i) { yi[i] = f32x4{0.f, 0.f, 0.f, 0.f}; ys[i] = yi[i]; }
    if (P == 64 && p.z) {   // y' only feeds dz
#pragma unroll
      for (int k0 = 0; k0 < L; k0 += 32) {
        const bf16x8 a = frag(sM, LDM, 16 * wave, k0, lane);
#pragma unroll
        for (int i = 0; i < P / 16; ++i) yi[i] = mfma16(a, frag_t(sX, LDX, k0, 16 * i, lane), yi[i]);
      }
    }
#pragma unroll
    for (int k0 = 0; k0 < N; k0 += 32) {
      const bf16x8 a = frag(sC, LDB, 16 * wave, k0, lane);
#pragma unroll
      for (int i = 0; i < P / 16; ++i) ys[i] = mfma16(a, frag(sS, LDB, 16 * i, k0, lane), ys[i]);
    }
    float das[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int t = 16 * wave + 4 * q4 + v;
      const float ea = F(F_EA, t);
#pragma unroll
      for (int i = 0; i < P / 16; ++i) {
        const int pc = 16 * i + l16;
        const float y_s = ea * ys[i][v];
        das[v] += (float)sG[t * LDX + pc] * y_s;
        if (P == 64 && p.z && t < nval) {
          float yp = yi[i][v] + y_s;
          if (p.D) yp += F(K::FDV, pc) * (float)sX[t * LDX + pc];
          const float zf = (float)sZ[t * LDX + pc];
          const float sg = __builtin_amdgcn_rcpf(1.f + fast_exp(-zf));
          const float dsilu = sg * (1.f + zf * (1.f - sg));
          p.dz[(int64_t)(tok0 + t) * H * P + (int64_t)h * P + pc] =
              (bf16)((float)sDY[t * LDX + pc] * yp * dsilu);
        }
      }
      const float rs = row16_sum(das[v]);
      if (l16 == 0) F(F_DAS, t) = rs;
    }
  }

  // ---- step B2: dx = (M dt')^T g + e dt' (dS1 B)^T + D g, and x . (dS1 B) -------
  {
    f32x4 dxi[P / 16], dhb[P / 16];
#pragma unroll
    for (int i = 0; i < P / 16; ++i) { dxi[i] = f32x4{0.f, 0.f, 0.f, 0.f}; dhb[i] = dxi[i]; }
#pragma unroll
    for (int k0 = 0; k0 < L; k0 += 32) {
      const bf16x8 a = frag_t(sM, LDM, k0, 16 * wave, lane);
#pragma unroll
      for (int i = 0; i < P / 16; ++i) dxi[i] = mfma16(a, frag_t(sG, LDX, k0, 16 * i, lane), dxi[i]);
    }
#pragma unroll
    for (int k0 = 0; k0 < N; k0 += 32) {
      const bf16x8 a = frag(sB, LDB, 16 * wave, k0, lane);
#pragma unroll
      for (int i = 0; i < P / 16; ++i) dhb[i] = mfma16(a, frag(sDS, LDB, 16 * i, k0, lane), dhb[i]);
    }
    float dds[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int s = 16 * wave + 4 * q4 + v;
      const float e = F(F_E, s), dt_s = F(F_DT, s);
#pragma unroll
      for (int i = 0; i < P / 16; ++i) {
        const int pc = 16 * i + l16;
        dds[v] += (float)sX[s * LDX + pc] * dhb[i][v];
        if (s < nval) {
          float d = dxi[i][v] + e * dt_s * dhb[i][v];
          if (p.D) d += F(K::FDV, pc) * (float)sG[s * LDX + pc];
          const int64_t ix = (int64_t)(tok0 + s) * p.HX * P + (int64_t)hx * P + pc;
          if (p.x_shared) unsafeAtomicAdd(static_cast<float*>(p.dx) + ix, d);
          else st_grad(p.dx, ix, d, p.gbf16);
        }
      }
      const float rs = row16_sum(dds[v]);
      if (l16 == 0) F(F_DDS, s) = e * rs;
    }
  }

  // ---- step B3: dC += e^{A_t} g S0 + W B (summed over the workgroup's heads) -------
  {
    f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < P; k0 += 32) {
      const bf16x8 a = frag(sG, LDX, 16 * wave, k0, lane);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = mfma16(a, frag_t(sS, LDB, k0, 16 * j, lane), acc[j]);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float ea = F(F_EA, 16 * wave + 4 * q4 + v);
#pragma unroll
      for (int j = 0; j < NT; ++j) dCacc[j][v] += acc[j][v] * ea;
    }
#pragma unroll
    for (int k0 = 0; k0 < L; k0 += 32) {
      const bf16x8 a = frag(sW, LDM, 16 * wave, k0, lane);
#pragma unroll
      for (int j = 0; j < NT; ++j) dCacc[j] = mfma16(a, frag_t(sB, LDB, k0, 16 * j, lane), dCacc[j]);
    }
  }

  // ---- step B4: dB = e dt' x dS1 + W^T C (summed over the heads when B is staged
  // once; otherwise this head's, stored or added) ------------------------------------
  {
    f32x4 acc[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k0 = 0; k0 < P; k0 += 32) {
      const bf16x8 a = frag(sX, LDX, 16 * wave, k0, lane);
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = mfma16(a, frag_t(sDS, LDB, k0, 16 * j, lane), acc[j]);
    }
    if (!b_once) {
#pragma unroll
      for (int j = 0; j < NT; ++j) dBacc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int s_ = 16 * wave + 4 * q4 + v;
      const float f = F(F_E, s_) * F(F_DT, s_);
#pragma unroll
      for (int j = 0; j < NT; ++j) dBacc[j][v] += acc[j][v] * f;
    }
#pragma unroll
    for (int k0 = 0; k0 < L; k0 += 32) {
      const bf16x8 a = frag_t(sW, LDM, k0, 16 * wave, lane);
#pragma unroll
      for (int j = 0; j < NT; ++j) dBacc[j] = mfma16(a, frag_t(sC, LDB, k0, 16 * j, lane), dBacc[j]);
    }
    if (!b_once) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int s_ = 16 * wave + 4 * q4 + v;
        if (s_ >= nval) continue;
        const int64_t row = (int64_t)(tok0 + s_) * p.G * N + (int64_t)g * N;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          if (p.b_shared) unsafeAtomicAdd(static_cast<float*>(p.dB) + row + 16 * j + l16, dBacc[j][v]);
          else st_grad(p.dB, row + 16 * j + l16, dBacc[j][v], p.gbf16);
        }
      }
    }
  }
  __syncthreads();

  // ---- scalar chain: dA_t, da (reverse cumsum), d dt, dA_h, d dt_bias --------------
  if (wave == 0) {
    const int t = lane;
    const float dt_t = F(F_DT, t), dds = F(F_DDS, t);
    float dacs = F(F_ROWR, t) + F(F_DAS, t) - dt_t * dds;
    float cmq = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      dacs -= F(F_CR0 + w, t);
      cmq += F(F_CMQ0 + w, t);
    }
    // <dS1, S1> = e^{A_L} <dS1, S0> + sum_s dt'_s e_s x_s . (dS1 B_s), on the last token
    const float tail = wave_sum(dt_t * dds);
    const float aend = __builtin_bit_cast(float, __builtin_amdgcn_readlane(
        __builtin_bit_cast(int, F(F_ACS, t)), 63));
    if (t == L - 1) dacs += fast_exp(aend) * sHD[0] + tail;
    const float incl = scan64(dacs, lane);
    const float total = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, incl), 63));
    const float da = total - incl + dacs;   // sum_{u >= t} dA_u
    const float ddtv = cmq + dds + A_h * da;
    const float ddt_raw = ddtv * F(F_FAC, t);
    if (t < nval) p.ddt[(int64_t)(tok0 + t) * H + h] = ddt_raw;
    const float sa = wave_sum(dt_t * da);
    const float sb = wave_sum(ddt_raw);
    if (lane == 0) {
      unsafeAtomicAdd(p.dA + h, sa);
      if (p.dbias) unsafeAtomicAdd(p.dbias + h, sb);
      sHD[0] = 0.f;   // lane 63 read it above; the next head adds after the barrier
    }
  }
  __syncthreads();   // LDS free for the next head
  }   // heads

  // dC of the C group (and dB of the B group staged once), summed over the heads
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int t = 16 * wave + 4 * q4 + v;
    if (t >= nval) continue;
    const int64_t rc = (int64_t)(tok0 + t) * GC * N + (int64_t)gc * N;
    const int64_t rb = (int64_t)(tok0 + t) * p.G * N + (int64_t)gc * N;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      st_grad(p.dC, rc + 16 * j + l16, dCacc[j][v], p.gbf16);
      if (b_once) st_grad(p.dB, rb + 16 * j + l16, dBacc[j][v], p.gbf16);
    }
  }
}

template <int P, int N>
void launch(const Params& p, hipStream_t s) {
  constexpr int smem = Lay<P, N>::BYTES;
  (void)hipFuncSetAttribute((const void*)ssd_bwd_chunk_kernel<P, N>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  const int units = p.H * 2 * (P / SP);
  const auto [Lr, nblk] = state_blocks(p.nrows, units, cu_count());
  if (nblk > 1)
    hipLaunchKernelGGL((ssd_bwd_states_kernel<P, N, true>), dim3(units * nblk), dim3(STHR), 0, s, p, Lr, nblk);
  hipLaunchKernelGGL((ssd_bwd_states_kernel<P, N, false>), dim3(units * nblk), dim3(STHR), 0, s, p, Lr, nblk);
  if (p.nrows == 0) return;               // sequences without tokens only
  if (takes_group_kernel(p.G, p.GC, p.z != nullptr, p.x_ts, p.dy_ts, p.b_ts, p.c_ts, (int64_t)p.HX * P,
                         (uintptr_t)p.dx)) {
    constexpr int gsm = GLay<P, N>::BYTES;
    (void)hipFuncSetAttribute((const void*)ssd_bwd_group_kernel<P, N>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, gsm);
    hipLaunchKernelGGL((ssd_bwd_group_kernel<P, N>), dim3(p.nrows * p.GC), dim3(GTHR), gsm, s, p);
  } else {
    hipLaunchKernelGGL((ssd_bwd_chunk_kernel<P, N>), dim3(p.nrows * p.GC), dim3(NTHR), smem, s, p);
  }
}

}  // namespace ssdb
}  // namespace hmx

using namespace hmx;
using namespace hmx::ssdb;

extern "C" size_t hmx_ssd_chunk_bwd_workspace_bytes(int32_t nrows, int32_t H, int32_t P, int32_t N) {
  // S0, dS1 (bf16); the block totals (fp32, both directions, at most nrows / 8 blocks)
  // and their decays
  const size_t st = (size_t)nrows * H * P * N;
  return st * (2 + 2 + 1) + (size_t)nrows * H * 4 + 256;
}

extern "C" int hmx_ssd_chunk_bwd(
    const void* x, int64_t x_ts, int64_t x_hs, const void* B, int64_t b_ts, int64_t b_gs,
    const void* C, int64_t c_ts, int64_t c_gs, int32_t xbc_dtype, const void* dt, int32_t dt_dtype,
    int64_t dt_ts, int64_t dt_hs, const float* A, const float* D, const float* dt_bias,
    const void* z, int64_t z_ts, int64_t z_hs, const void* dy, int64_t dy_ts, int64_t dy_hs,
    const float* h0, const float* d_final, const int32_t* seg_table,
    int32_t nrows, const int32_t* seq_table, int32_t nseq, int32_t H, int32_t HX, int32_t G,
    int32_t GC, int32_t P, int32_t N, int32_t dt_softplus, float dt_min, float dt_max, void* dx,
    void* dB, void* dC, int32_t grad_dtype, void* dz, float* ddt, float* dA, float* dD, float* ddt_bias,
    float* dh0, void* workspace, size_t workspace_bytes, void* stream) {
  const char* fn = "hmx_ssd_chunk_bwd";
  HMX_REQUIRE(xbc_dtype == HMX_BF16, HMX_EUNSUPPORTED, "%s: x/B/C/z/dy must be bfloat16", fn);
  HMX_REQUIRE((P == 64 || P == 128) && (N == 64 || N == 128), HMX_EUNSUPPORTED,
              "%s: headdim and d_state in {64,128} (got %d, %d)", fn, P, N);
  HMX_REQUIRE(P == 64 || !z, HMX_EUNSUPPORTED, "%s: the z gate needs headdim 64", fn);
  HMX_REQUIRE(grad_dtype == HMX_F32 ||
                  (grad_dtype == HMX_BF16 && HX == H && (G == H || G == GC)),
              HMX_EUNSUPPORTED,
              "%s: dx / dB / dC in bf16 need unshared x and B (HX = H; G = H or G = GC)", fn);
  HMX_REQUIRE(H > 0 && HX > 0 && G > 0 && GC > 0 && H % HX == 0 && H % G == 0 && H % GC == 0,
              HMX_EINVAL, "%s: H=%d must be a multiple of HX=%d, G=%d and GC=%d", fn, H, HX, G, GC);
  HMX_REQUIRE(x && B && C && dt && A && dy && seg_table && seq_table && dx && dB && dC && ddt && dA &&
                  (!z || dz) && nrows >= 0 && nseq >= 0,
              HMX_EINVAL, "%s: null pointer", fn);
  HMX_REQUIRE(dt_dtype == HMX_F32 || dt_dtype == HMX_BF16 || dt_dtype == HMX_F16, HMX_EINVAL,
              "%s: dt dtype code %d", fn, dt_dtype);
  const int64_t strides[] = {x_ts, x_hs, b_ts, b_gs, c_ts, c_gs, dy_ts, dy_hs,
                             z ? z_ts : 8, z ? z_hs : 8};
  for (int64_t st : strides)
    HMX_REQUIRE(st % 8 == 0, HMX_EINVAL, "%s: token/head strides must be multiples of 8", fn);
  HMX_REQUIRE(((uintptr_t)x | (uintptr_t)B | (uintptr_t)C | (uintptr_t)dy | (uintptr_t)z |
               (uintptr_t)h0 | (uintptr_t)d_final | (uintptr_t)dh0) % 16 == 0,
              HMX_EINVAL, "%s: operands must be 16-byte aligned", fn);
  if (nrows == 0 && nseq == 0) return HMX_OK;
  const size_t need = hmx_ssd_chunk_bwd_workspace_bytes(nrows, H, P, N);
  HMX_REQUIRE(workspace && workspace_bytes >= need, HMX_EINVAL,
              "%s: workspace of %zu bytes needed, %zu given", fn, need, workspace_bytes);
  Params p;
  p.x = static_cast<const bf16*>(x); p.x_ts = x_ts; p.x_hs = x_hs;
  p.B = static_cast<const bf16*>(B); p.b_ts = b_ts; p.b_gs = b_gs;
  p.C = static_cast<const bf16*>(C); p.c_ts = c_ts; p.c_gs = c_gs;
  p.dt = dt; p.dt_dt = dt_dtype; p.dt_ts = dt_ts; p.dt_hs = dt_hs;
  p.A = A; p.D = D; p.dt_bias = dt_bias;
  p.z = static_cast<const bf16*>(z); p.z_ts = z_ts; p.z_hs = z_hs;
  p.dy = static_cast<const bf16*>(dy); p.dy_ts = dy_ts; p.dy_hs = dy_hs;
  p.h0 = h0; p.dT = d_final;
  p.seg = seg_table; p.seqs = seq_table; p.nrows = nrows; p.nseq = nseq;
  const size_t st = (size_t)nrows * H * P * N;
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  p.S0 = reinterpret_cast<bf16*>(ws);
  p.dS1 = reinterpret_cast<bf16*>(ws + st * 2);
  p.tot = reinterpret_cast<float*>(ws + st * 4);
  p.tdec = reinterpret_cast<float*>(ws + st * 5);
  p.dx = dx; p.x_shared = HX < H;
  p.dB = dB; p.b_shared = G < H;
  p.dC = dC; p.gbf16 = grad_dtype == HMX_BF16;
  p.dz = static_cast<bf16*>(dz); p.ddt = ddt; p.dA = dA; p.dD = dD; p.dbias = ddt_bias;
  p.dh0 = dh0;
  p.H = H; p.HX = HX; p.G = G; p.GC = GC; p.softplus = dt_softplus;
  p.dt_min = dt_min; p.dt_max = dt_max;
  hipStream_t s = (hipStream_t)stream;
  if (P == 64 && N == 128) launch<64, 128>(p, s);
  else if (P == 64) launch<64, 64>(p, s);
  else if (N == 128) launch<128, 128>(p, s);
  else launch<128, 64>(p, s);
  return check_launch(fn);
}
