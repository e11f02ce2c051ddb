// Router: f32 logits (sequential sum over d), top-k with lower-index tie-break (topk.h), softmax over the selection.
//
// Stands in for MaxText RoutedMoE's gate + top-k (third-party; configured by configs/stage1.yml:34-37 of the
// reference).  Logit order contract: logits[t,e] = (((x[t,0]w[0,e]) + x[t,1]w[1,e]) + ...) in f32, then
// + bias[e].  bf16 x bf16 products are exact in f32, so fused multiply-add and the CPU's separate multiply and
// add give the same bits: the result is reproducible bit for bit on the CPU whatever the thread mapping.
//
// Two paths.  The split path (the ABI's lsurge_router_topk, and shapes the fused kernel does not take): a logits
// kernel over (token block, expert block) tiles, then a selection kernel (one lane per token from 8192 tokens, else
// one wave per token).  The layer's fused path (E = 32, 64, 128 or 256, k <= 8): router_fused_kernel, one workgroup
// of 16 to 64 tokens x all experts computing the same logits on the f32 matrix cores, then top-k, softmax and the
// layout's per-64-token expert histograms in the same workgroup (described at the kernel).
#include "launchers.h"
#include "router_tiles.h"
#include "topk.h"

namespace {

using lsurge::TOPK_NO_ID;
using lsurge::TOPK_NO_KEY;
using lsurge::TopkList;
using lsurge::topk_before;
using lsurge::topk_key;
using lsurge::topk_logit;

// One round of a wave-per-token selection over the wave's keys (lane + 64 c is expert lane + 64 c of the token): the
// best candidate, the same in every lane, whose key is then removed.
template <int EC>
__device__ __forceinline__ void wave_take_best(uint32_t (&key)[EC], int lane, uint32_t* bk_out, int* bi_out) {
  uint32_t bk = TOPK_NO_KEY;
  int bi = TOPK_NO_ID;
#pragma unroll
  for (int c = 0; c < EC; ++c)
    if (key[c] > bk) {  // ascending experts: strictly larger keeps the lower index of a tie
      bk = key[c];
      bi = lane + 64 * c;
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const uint32_t ok = __shfl_xor(bk, o, 64);
    const int oi = __shfl_xor(bi, o, 64);
    if (topk_before(ok, oi, bk, bi)) {
      bk = ok;
      bi = oi;
    }
  }
#pragma unroll
  for (int c = 0; c < EC; ++c)
    if (lane + 64 * c == bi) key[c] = TOPK_NO_KEY;
  *bk_out = bk;
  *bi_out = bi;
}

constexpr int RT_TOK = 64;       // tokens per workgroup
constexpr int RT_DC = 32;        // d chunk staged in LDS
constexpr int RT_THREADS = 128;  // 16 token quads x 8 expert groups
constexpr int RT_EMAX = 256;

// LDS: x chunk transposed [RT_DC][RT_TOK] f32 (8 KB) + w chunk [RT_DC][EP] f32 (<= 32 KB).  After the d loop
// the w region holds the [RT_TOK][EP] logits (<= 64 KB, sized for that).
template <int EP>  // experts padded to a multiple of 32
__global__ __launch_bounds__(RT_THREADS) void router_topk_kernel(const bf16_t* __restrict__ x,
                                                                 const bf16_t* __restrict__ w,
                                                                 const float* __restrict__ bias, int T, int d,
                                                                 int E, int k, float* __restrict__ logits,
                                                                 int32_t* __restrict__ sel,
                                                                 float* __restrict__ weights) {
  constexpr int EPT = EP / 8;  // experts per thread (contiguous)
  __shared__ __attribute__((aligned(16))) float xs[RT_DC][RT_TOK];
  __shared__ __attribute__((aligned(16))) float ws[RT_TOK * EP > RT_DC * EP ? RT_TOK * EP : RT_DC * EP];
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * RT_TOK;
  const int eq = tid & 7;   // expert group: experts eq*EPT .. eq*EPT + EPT - 1
  const int tq = tid >> 3;  // token quad: tokens 4tq .. 4tq+3
  float acc[4][EPT];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int j = 0; j < EPT; ++j) acc[a][j] = 0.f;

  for (int d0 = 0; d0 < d; d0 += RT_DC) {
    const int dc = min(RT_DC, d - d0);
    // x[t0 .. t0+64, d0 .. d0+32): 8-element chunks (16 B), stored transposed as f32 (zeros past T / d)
    for (int c = tid; c < RT_TOK * RT_DC / 8; c += RT_THREADS) {
      const int tt = c / (RT_DC / 8), dd0 = (c % (RT_DC / 8)) * 8;
      const int t = t0 + tt;
      float v[8];
      if (t < T && dd0 + 8 <= dc && (d & 7) == 0) {
        const u32x4 u = *reinterpret_cast<const u32x4*>(x + (int64_t)t * d + d0 + dd0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          v[2 * i] = __uint_as_float(u[i] << 16);
          v[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
        }
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          v[i] = (t < T && dd0 + i < dc) ? bf16_to_f32(x[(int64_t)t * d + d0 + dd0 + i]) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) xs[dd0 + i][tt] = v[i];
    }
    // w[d0 .. d0+32, 0 .. E) as f32, experts padded with zeros
    for (int i = tid; i < RT_DC * EP; i += RT_THREADS) {
      const int dd = i / EP, e = i % EP;
      ws[i] = (dd < dc && e < E) ? bf16_to_f32(w[(int64_t)(d0 + dd) * E + e]) : 0.f;
    }
    __syncthreads();
    for (int dd = 0; dd < dc; ++dd) {
      const f32x4 xv = *reinterpret_cast<const f32x4*>(&xs[dd][4 * tq]);
#pragma unroll
      for (int c = 0; c < EPT / 4; ++c) {
        const f32x4 wv = *reinterpret_cast<const f32x4*>(&ws[dd * EP + eq * EPT + 4 * c]);
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[a][4 * c + i] = __builtin_fmaf(xv[a], wv[i], acc[a][4 * c + i]);
      }
    }
    __syncthreads();
  }
  // logits (+ bias) -> LDS [RT_TOK][EP] and global
  float* ls = ws;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int tt = 4 * tq + a;
    const int t = t0 + tt;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int e = eq * EPT + j;
      float v = acc[a][j];
      if (e < E && bias) v = v + bias[e];
      ls[tt * EP + e] = (e < E) ? v : -INFINITY;
      if (t < T && e < E && logits) logits[(int64_t)t * E + e] = v;
    }
  }
  __syncthreads();
  // top-k: one wave per token
  const int lane = tid & 63, wv = tid >> 6;
  for (int tt = wv; tt < RT_TOK; tt += RT_THREADS / 64) {
    const int t = t0 + tt;
    if (t >= T) break;
    constexpr int EC = (EP + 63) / 64;
    uint32_t key[EC];
#pragma unroll
    for (int c = 0; c < EC; ++c) {
      const int e = lane + 64 * c;
      key[c] = (e < E) ? topk_key(ls[tt * EP + e]) : TOPK_NO_KEY;
    }
    float top0 = 0.f, denom = 0.f;
    for (int j = 0; j < k; ++j) {
      uint32_t bk;
      int bi;
      wave_take_best(key, lane, &bk, &bi);
      const float bv = topk_logit(bk);
      if (j == 0) top0 = bv;
      const float z = __expf(bv - top0);
      denom += z;
      if (lane == 0) {
        sel[(int64_t)t * k + j] = bi;
        weights[(int64_t)t * k + j] = z;  // normalised below
      }
    }
    if (lane == 0) {
      const float inv = 1.f / denom;
      for (int j = 0; j < k; ++j) weights[(int64_t)t * k + j] *= inv;
    }
  }
}

// ---------------------------------------------------------------------------------------------- split path
// Logits kernel: workgroup = 64 tokens x 32 experts (256 threads, 4 tokens x 2 experts each), grid over token
// blocks x expert blocks, so there are enough waves to fill every SIMD; the d loop is the same sequential
// f32 sum as above.  The top-k then runs as its own kernel, one wave per token, over the logits in HBM.
//
// Lane layout: the 16 lanes of a row (lane / 16) share a token quad and hold 16 different expert pairs (lane % 16),
// so a row's x read is one LDS broadcast and its weight reads are 128 contiguous bytes.
constexpr int RL_TOK = 64, RL_EXP = 32, RL_DC = 64, RL_THREADS = 256;

// One d step of a thread's 4 tokens x 2 experts: x of the 4 tokens (one LDS read that the 16 lanes of the quad's row
// share) and the two weights; fmaf rounds once, so each logit stays the sequential f32 sum over d.
template <int WP>
__device__ __forceinline__ void logits_step(float (&acc)[4][2], const float* xrow, const float (*ws)[WP], int dd,
                                            int tq, int ep) {
  const f32x4 xv = *reinterpret_cast<const f32x4*>(xrow + 4 * tq);
  const float w0 = ws[dd][2 * ep], w1 = ws[dd][2 * ep + 1];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    acc[a][0] = __builtin_fmaf(xv[a], w0, acc[a][0]);
    acc[a][1] = __builtin_fmaf(xv[a], w1, acc[a][1]);
  }
}

__device__ __forceinline__ void unpack_bf16x8(const u32x4& u, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(u[i] << 16);
    v[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
  }
}

// LDS: two buffers of (x chunk transposed to [d][token] f32, w chunk [d][expert] f32).  When d and E are multiples
// of 8 the next chunk's global loads (raw bf16 in registers) are issued right after the barrier that publishes the
// current chunk, so their latency hides behind the current chunk's FMAs; other shapes load each chunk in place.
// Bank-conflict-free LDS traffic: a wave stages 64 consecutive tokens of one d row (lane = token) and w goes in as
// 16-byte stores of 4 consecutive experts (the x rows keep a padded pitch of RL_XP floats).
constexpr int RL_XP = RL_TOK + 4;
__global__ __launch_bounds__(RL_THREADS) void router_logits_kernel(const bf16_t* __restrict__ x,
                                                                   const bf16_t* __restrict__ w,
                                                                   const float* __restrict__ bias, int T, int d,
                                                                   int E, float* __restrict__ logits) {
  __shared__ __attribute__((aligned(16))) float xs[2][RL_DC][RL_XP];
  __shared__ __attribute__((aligned(16))) float ws[2][RL_DC][RL_EXP];
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * RL_TOK, e0 = blockIdx.y * RL_EXP;
  const int ep = tid & 15;   // experts e0 + 2 ep, e0 + 2 ep + 1 (position in the row of 16 lanes)
  const int tq = tid >> 4;   // tokens t0 + 4 tq .. + 3 (one row of 16 lanes)
  float acc[4][2] = {{0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}, {0.f, 0.f}};
  const bool vec = (d & 7) == 0 && (E & 7) == 0;
  // this thread's staging share: x token tid % 64 at d offsets 8 (tid / 64) and 8 (tid / 64 + 4) of the chunk; w d
  // row tid / 4, experts 8 (tid % 4) ..
  const int xtt = tid & 63, xc0 = tid >> 6;
  const int wdd = tid >> 2, wec = (tid & 3) * 8;

  auto compute = [&](int buf, int dc) {
    const float(*wsb)[RL_EXP] = ws[buf];
    if (dc == RL_DC) {
#pragma unroll 8
      for (int dd = 0; dd < RL_DC; ++dd) logits_step<RL_EXP>(acc, xs[buf][dd], wsb, dd, tq, ep);
    } else {
      for (int dd = 0; dd < dc; ++dd) logits_step<RL_EXP>(acc, xs[buf][dd], wsb, dd, tq, ep);
    }
  };

  if (vec) {
    u32x4 xr[2], wr;  // raw bf16 of the chunk being loaded (zeros outside the matrices)
    auto gload = [&](int d0) {
      const int dc = min(RL_DC, d - d0), t = t0 + xtt;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int dd0 = 8 * (xc0 + 4 * r);
        xr[r] = (t < T && dd0 < dc) ? *reinterpret_cast<const u32x4*>(x + (int64_t)t * d + d0 + dd0) : u32x4{0, 0, 0, 0};
      }
      wr = (wdd < dc && e0 + wec < E) ? *reinterpret_cast<const u32x4*>(w + (int64_t)(d0 + wdd) * E + e0 + wec)
                                      : u32x4{0, 0, 0, 0};
    };
    auto sstore = [&](int buf) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int dd0 = 8 * (xc0 + 4 * r);
        float v[8];
        unpack_bf16x8(xr[r], v);
#pragma unroll
        for (int i = 0; i < 8; ++i) xs[buf][dd0 + i][xtt] = v[i];
      }
      float v[8];
      unpack_bf16x8(wr, v);
      *reinterpret_cast<f32x4*>(&ws[buf][wdd][wec]) = f32x4{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<f32x4*>(&ws[buf][wdd][wec + 4]) = f32x4{v[4], v[5], v[6], v[7]};
    };
    gload(0);
    int buf = 0;
    for (int d0 = 0; d0 < d; d0 += RL_DC, buf ^= 1) {
      // buffer buf was last read two chunks ago, before the barrier of the previous chunk
      sstore(buf);
      __syncthreads();
      if (d0 + RL_DC < d) gload(d0 + RL_DC);
      compute(buf, min(RL_DC, d - d0));
    }
  } else {
    for (int d0 = 0; d0 < d; d0 += RL_DC) {
      const int dc = min(RL_DC, d - d0);
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int dd0 = 8 * (xc0 + 4 * r), t = t0 + xtt;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          xs[0][dd0 + i][xtt] = (t < T && dd0 + i < dc) ? bf16_to_f32(x[(int64_t)t * d + d0 + dd0 + i]) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        ws[0][wdd][wec + i] = (wdd < dc && e0 + wec + i < E) ? bf16_to_f32(w[(int64_t)(d0 + wdd) * E + e0 + wec + i]) : 0.f;
      __syncthreads();
      compute(0, dc);
      __syncthreads();
    }
  }
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const int t = t0 + 4 * tq + a;
    if (t >= T) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int e = e0 + 2 * ep + j;
      if (e < E) logits[(int64_t)t * E + e] = bias ? acc[a][j] + bias[e] : acc[a][j];
    }
  }
}

// ---------------------------------------------------------------------------------------------- workgroup-fused path
// Fused router of the layer (E = 32, 64, 128 or 256 experts, k <= 8): logits on the f32 matrix cores, then top-k,
// softmax and the expert histogram in the same workgroup.
//
// Logits.  v_mfma_f32_16x16x4_f32 adds its four products to the accumulator one after the other in ascending k, each
// with one f32 rounding: exactly the fmaf chain of router_logits_kernel, at twice the vector unit's rate (measured
// bit-equal on normal, wide-range, cancelling, subnormal and non-finite bf16 operands; the GPU tests compare the two
// kernels bit for bit).  One workgroup = TOK = 16 TT tokens x all E experts, one wave per 16 HT experts; a wave holds TT
// token tiles x HT expert tiles (HT = 2: expert 32 wave + 2 c + h is column c of tile h, so one dword of a row of W_r
// feeds both tiles).  Step s of a 32-deep block covers d = 4 s .. + 3, lane quarter q supplying d = 4 s + q:
//   x  goes through a double LDS buffer of DC-deep chunks, each block of a row stored by quarter ([q][8 steps] bf16),
//      so one 16-byte read gives a lane its operands of 8 steps; blocks are read one ahead of their use;
//   w  straight from L2 into registers, a ring of GD / 4 steps ahead of its use.
// Bound by the matrix pipe (32 HT cycles a step and token tile) once two waves share a SIMD, by load latency below that.
// TT = 1 gives the most workgroups, TT = 4 the fewest reads of W_r; the rule (router_tiles.h) takes the largest TT that
// still leaves 2048 waves (two per SIMD), so small batches spread over the CUs and a 1 MB W_r is read once per 64 tokens.
// At E = 256 the registers are held to 128, so that two 8-wave workgroups share a CU (656 -> 613 us at T = 65536, d =
// 2048); elsewhere the bound cost more than it gave.
// Replaced a vector-FMA kernel (4 tokens x 2-4 experts a thread, both operands as f32 through LDS, whose bandwidth
// bounded it).  Alone, before -> after: T = 4096, E = 64, d = 1024 45 -> 20 us; T = 16384, E = 64 55 -> 31 us; T =
// 16384, E = 128 97 -> 49 us; T = 65536, E = 256, d = 2048 1088 -> 613 us (matrix pipe alone: 455 us at the 150
// TFLOP/s that this instruction reaches).
//
// Then, in the same workgroup:
//  - the logits go to HBM and to an LDS tile [TOK][E + 1];
//  - top-k + softmax per token: L = E / (4 HT TT) lanes per token each keep a sorted list of the best 8 of their
//    EPL = 4 HT TT experts (scanned in ascending expert order), and k merge rounds take the best head of the L lists, in
//    the order of topk.h, as router_select_lane_kernel, whose softmax (in rank order) this repeats;
//  - the expert histogram of the workgroup's TOK k slots (LDS counters) -> hist[chunk of 64 tokens][E], the layout's
//    per-chunk counts.  A word of hist holds the counts of its chunk's four 16-token quarters in its bytes (a token
//    picks an expert at most once, so even 64 tokens fit one byte): a workgroup writes the TT bytes of its own
//    quarters (its count and zeros), and the layout adds the four bytes up.  No workgroup touches another's bytes, so
//    nothing has to be cleared first.
template <int E, int TT, int HT, int DC>
__global__ __launch_bounds__(4 * E / HT, E == 256 ? 4 : 1) void router_fused_kernel(
    const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, const float* __restrict__ bias, int T, int d, int k,
    float* __restrict__ logits, int32_t* __restrict__ sel, float* __restrict__ weights, uint8_t* __restrict__ hist) {
  constexpr int NT = 4 * E / HT, TOK = 16 * TT, L = NT / TOK, EPL = E / L;  // threads, tokens, lanes and experts a lane
  constexpr int GD = DC < 128 ? DC : 128;    // depth of the weight ring
  constexpr int XP = 2 * DC + 16;            // LDS row pitch in bytes (rows one 16-byte slot apart in the banks)
  static_assert(64 % L == 0 && L >= 1 && (HT == 1 || HT == 2), "fused router shape");
  constexpr int XS_B = 2 * TOK * XP, TILE_B = TOK * (E + 1) * 4;
  __shared__ __attribute__((aligned(16))) char sm[XS_B > TILE_B ? XS_B : TILE_B];
  __shared__ int32_t cnt[E];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int t0 = blockIdx.x * TOK;
  const int r = lane & 15, q = lane >> 4;
  for (int e = tid; e < E; e += NT) cnt[e] = 0;
  // staging: x pieces p = tid + NT i: token p / (DC / 8), d 8 (p % (DC / 8)) .. + 7 of the chunk (zeros past T), which
  // are two steps of every quarter
  constexpr int XQ = TOK * (DC / 8), XR = (XQ + NT - 1) / NT;
  u32x4 xr[XR];
  auto gx = [&](int d0) {
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      const int p = tid + NT * i, t = t0 + p / (DC / 8);
      xr[i] = p < XQ && t < T ? *reinterpret_cast<const u32x4*>(x + (int64_t)t * d + d0 + 8 * (p % (DC / 8)))
                              : u32x4{0, 0, 0, 0};
    }
  };
  auto sx = [&](int buf) {
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      const int p = tid + NT * i, c = p % (DC / 8);
      if (p < XQ) {
        char* o = sm + buf * TOK * XP + (p / (DC / 8)) * XP + 64 * (c >> 2) + 4 * (c & 3);
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // quarters 2 h and 2 h + 1: elements (q, q + 4) of the piece
          *reinterpret_cast<uint32_t*>(o + 32 * h) = __builtin_amdgcn_perm(xr[i][2 + h], xr[i][h], 0x05040100u);
          *reinterpret_cast<uint32_t*>(o + 32 * h + 16) = __builtin_amdgcn_perm(xr[i][2 + h], xr[i][h], 0x07060302u);
        }
      }
    }
  };
  const bf16_t* wl = w + (int64_t)q * E + HT * (16 * wv + r);  // this lane's experts of d row q
  auto gw = [&](int dd) {
    if constexpr (HT == 2) return *reinterpret_cast<const uint32_t*>(wl + (int64_t)dd * E);
    else return (uint32_t)wl[(int64_t)dd * E];
  };
  f32x4 acc[TT][HT];
#pragma unroll
  for (int a = 0; a < TT; ++a)
#pragma unroll
    for (int h = 0; h < HT; ++h) acc[a][h] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t wr[GD / 4];
  gx(0);
#pragma unroll
  for (int s = 0; s < GD / 4; ++s) wr[s] = gw(4 * s);
  u32x4 fa[2][TT];
  int buf = 0;
  for (int d0 = 0; d0 < d; d0 += DC, buf ^= 1) {  // d % DC == 0 (checked on the host)
    // buffer buf was last read two chunks ago, before the barrier of the previous chunk
    sx(buf);
    __syncthreads();
    gx(min(d0 + DC, d - DC));  // the next chunk (the last one again at the end, unused)
    const char* xa = sm + buf * TOK * XP + r * XP + 16 * q;  // this lane's row and quarter
    auto fread = [&](u32x4(&f)[TT], int blk) {
#pragma unroll
      for (int a = 0; a < TT; ++a) f[a] = *reinterpret_cast<const u32x4*>(xa + 16 * a * XP + 64 * blk);
    };
    fread(fa[0], 0);
    for (int g = 0; g < DC; g += GD) {
      const int dn = min(d0 + g + GD, d - GD);  // the ring's next depth (the last one again at the end, unused)
#pragma unroll
      for (int b = 0; b < GD / 32; ++b) {
        fread(fa[(b + 1) & 1], min(g / 32 + b + 1, DC / 32 - 1));
        float wc[8][HT];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
          wc[s][0] = __uint_as_float(wr[8 * b + s] << 16);
          if constexpr (HT == 2) wc[s][1] = __uint_as_float(wr[8 * b + s] & 0xffff0000u);
          wr[8 * b + s] = gw(dn + 32 * b + 4 * s);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
          for (int a = 0; a < TT; ++a) {
            const uint32_t u = fa[b & 1][a][s >> 1];
            const float xv = __uint_as_float(s & 1 ? u & 0xffff0000u : u << 16);
#pragma unroll
            for (int h = 0; h < HT; ++h) acc[a][h] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv, wc[s][h], acc[a][h], 0, 0, 0);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  __syncthreads();  // every wave is done with the staging buffers: they now hold the logits tile
  float* lt = reinterpret_cast<float*>(sm);
  const int e0 = HT * (16 * wv + r);
  float be[HT];
#pragma unroll
  for (int h = 0; h < HT; ++h) be[h] = bias ? bias[e0 + h] : 0.f;
#pragma unroll
  for (int a = 0; a < TT; ++a)
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // accumulator element i: token 4 q + i of the tile
      const int tt = 16 * a + 4 * q + i, t = t0 + tt;
      float v[HT];
#pragma unroll
      for (int h = 0; h < HT; ++h) lt[tt * (E + 1) + e0 + h] = v[h] = bias ? acc[a][h][i] + be[h] : acc[a][h][i];
      if (t < T) {
        float* lg = logits + (int64_t)t * E + e0;
        if constexpr (HT == 2) *reinterpret_cast<float2*>(lg) = float2{v[0], v[1]};
        else *lg = v[0];
      }
    }
  __syncthreads();
  // selection: token tid / L, lane part tid % L scans experts part, part + L, ... (ascending) into a sorted list of
  // its best KL = 8 (k <= 8, so a lane's share of the top k is always in it; the rest never matter), or all of them
  constexpr int KL = EPL < 8 ? EPL : 8;
  static_assert(L * KL >= 8, "the lists of a token hold its k <= 8 experts");
  const int tt = tid / L, part = tid % L, t = t0 + tt;
  TopkList<KL> list;
  list.clear();
#pragma unroll 1
  for (int c = 0; c < EPL; ++c) {
    const int e = part + L * c;
    list.insert(topk_key(lt[tt * (E + 1) + e]), e);
  }
  // k merge rounds over the L lanes of the token (an aligned group of L lanes of one wave).  The order is total, so the
  // lanes agree on the winner whatever the logits are, and exactly one of them advances: k distinct experts of [0, E)
  float top0 = 0.f, denom = 0.f, zj[8];
  int sj[8];
  int head = 0;
  for (int j = 0; j < k; ++j) {
    uint32_t bk;
    int hi;
    list.get(head, &bk, &hi);
    int bi = hi;
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
      const uint32_t ok = __shfl_xor(bk, o, 64);
      const int oi = __shfl_xor(bi, o, 64);
      if (topk_before(ok, oi, bk, bi)) {
        bk = ok;
        bi = oi;
      }
    }
    if (hi == bi) ++head;  // the lane that held the winner advances
    const float bv = topk_logit(bk);
    if (j == 0) top0 = bv;
    const float z = __expf(bv - top0);
    denom += z;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (q == j) {
        zj[q] = z;
        sj[q] = bi;
      }
  }
  if (part == 0 && t < T) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if (j < k) {
        sel[(int64_t)t * k + j] = sj[j];
        weights[(int64_t)t * k + j] = zj[j] / denom;
        atomicAdd(&cnt[sj[j]], 1);  // LDS counter: the count does not depend on the order
      }
    }
  }
  __syncthreads();
  // this workgroup's quarters of the 64-token chunk's words
  constexpr int PER = 4 / TT;
  uint8_t* hq = hist + (int64_t)(blockIdx.x / PER) * E * 4 + (blockIdx.x % PER) * TT;
  for (int e = tid; e < E; e += NT) {
    if constexpr (TT == 1) hq[4 * e] = (uint8_t)cnt[e];
    else if constexpr (TT == 2) *reinterpret_cast<uint16_t*>(hq + 4 * e) = (uint16_t)cnt[e];
    else *reinterpret_cast<uint32_t*>(hq + 4 * e) = (uint32_t)cnt[e];
  }
}

// one wave per token: top-k (the order of topk.h), softmax over the k
template <int EC>  // logits per lane: E <= 64 EC
__global__ __launch_bounds__(256) void router_select_kernel(const float* __restrict__ logits, int T, int E, int k,
                                                            int32_t* __restrict__ sel, float* __restrict__ weights) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  uint32_t key[EC];
#pragma unroll
  for (int c = 0; c < EC; ++c) {
    const int e = lane + 64 * c;
    key[c] = (e < E) ? topk_key(logits[(int64_t)t * E + e]) : TOPK_NO_KEY;
  }
  float top0 = 0.f, denom = 0.f, mine = 0.f;
  for (int j = 0; j < k; ++j) {
    uint32_t bk;
    int bi;
    wave_take_best(key, lane, &bk, &bi);
    const float bv = topk_logit(bk);
    if (j == 0) top0 = bv;
    const float z = __expf(bv - top0);
    denom += z;
    if (lane == j) mine = z;
    if (lane == 0) sel[(int64_t)t * k + j] = bi;
  }
  if (lane < k) weights[(int64_t)t * k + lane] = mine / denom;
}

// one lane per token: the k best logits (the order of topk.h) kept in a sorted register list while the token's logits
// are scanned in ascending expert order, then the softmax over them in rank order.  K >= k is the list's compile-time
// size.
template <int K>
__global__ __launch_bounds__(256) void router_select_lane_kernel(const float* __restrict__ logits, int T, int E, int k,
                                                                 int32_t* __restrict__ sel,
                                                                 float* __restrict__ weights) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= T) return;
  const float* l = logits + (int64_t)t * E;
  TopkList<K> best;
  best.clear();
  auto insert = [&](float v, int e) { best.insert(topk_key(v), e); };
  if ((E & 3) == 0) {
    for (int e = 0; e < E; e += 4) {
      const f32x4 q = *reinterpret_cast<const f32x4*>(l + e);
      insert(q[0], e);
      insert(q[1], e + 1);
      insert(q[2], e + 2);
      insert(q[3], e + 3);
    }
  } else {
    for (int e = 0; e < E; ++e) insert(l[e], e);
  }
  // softmax over the k best, denominator summed in rank order
  float denom = 0.f;
  const float top0 = topk_logit(best.key[0]);
#pragma unroll
  for (int j = 0; j < K; ++j)
    if (j < k) denom += __expf(topk_logit(best.key[j]) - top0);
#pragma unroll
  for (int j = 0; j < K; ++j) {
    if (j < k) {
      sel[(int64_t)t * k + j] = best.id[j];
      weights[(int64_t)t * k + j] = __expf(topk_logit(best.key[j]) - top0) / denom;
    }
  }
}

}  // namespace


extern "C" int lsurge_router_topk(const void* x, const void* w_r, const float* bias, int64_t t, int64_t d,
                                  int64_t e, int64_t k, float* logits, int32_t* sel, float* weights,
                                  lsurge_stream_t stream) {
  return lsurge::router_topk_impl(x, w_r, bias, t, d, e, k, logits, sel, weights, (hipStream_t)stream, nullptr);
}

bool lsurge::router_fused_ok(int64_t d, int64_t e, int64_t k) {
  return (e == 32 || e == 64 || e == 128 || e == 256) && k >= 1 && k <= 8 && d >= 64 && d % 64 == 0;
}

int lsurge::router_topk_impl(const void* x, const void* w_r, const float* bias, int64_t t, int64_t d, int64_t e,
                             int64_t k, float* logits, int32_t* sel, float* weights, hipStream_t stream,
                             hipEvent_t after_logits, int32_t* hist) {
  LSURGE_REQUIRE(x && w_r && sel && weights, "router_topk: null pointer");
  LSURGE_REQUIRE(t >= 0 && d > 0 && e >= 1 && e <= RT_EMAX && k >= 1 && k <= e, "router_topk: bad shape t=%lld d=%lld e=%lld k=%lld",
                 (long long)t, (long long)d, (long long)e, (long long)k);
  LSURGE_REQUIRE(t < (1ll << 31) && t * d < (1ll << 40), "router_topk: too large");
  if (t == 0) return LSURGE_OK;
  hipStream_t s = (hipStream_t)stream;
  if (hist) {  // workgroup-fused path: logits, top-k, softmax and the per-64-token histograms in one kernel
    LSURGE_REQUIRE(logits && router_fused_ok(d, e, k), "router_topk: shape d=%lld e=%lld k=%lld has no fused kernel",
                   (long long)d, (long long)e, (long long)k);
    const RouterTiles rt = router_tiles(t, d, e);
    const dim3 grid((unsigned)((t + 63) / 64 * (4 / rt.tt)));  // whole chunks: every byte of hist is written
#define RF_LAUNCH(E_, TT_, HT_, DC_)                                                                               \
  LSURGE_LAUNCH(KID_ROUTER, s,                                                                                     \
                hipLaunchKernelGGL((router_fused_kernel<E_, TT_, HT_, DC_>), grid, dim3(4 * E_ / HT_), 0, s,       \
                                   (const bf16_t*)x, (const bf16_t*)w_r, bias, (int)t, (int)d, (int)k, logits, sel, \
                                   weights, (uint8_t*)hist))
#define RF_DC(E_, TT_, HT_)                            \
  do {                                                 \
    if (rt.dc == 128) RF_LAUNCH(E_, TT_, HT_, 128);    \
    else RF_LAUNCH(E_, TT_, HT_, 64);                  \
  } while (0)
#define RF_CASE(E_)                       \
  do {                                    \
    if (rt.tt == 4) RF_DC(E_, 4, 2);      \
    else if (rt.tt == 2) RF_DC(E_, 2, 2); \
    else RF_DC(E_, 1, 2);                 \
  } while (0)
    if (rt.ht == 1 && e == 32) RF_DC(32, 1, 1);
    else if (rt.ht == 1) RF_DC(64, 1, 1);
    else if (e == 32) RF_CASE(32);
    else if (e == 64) RF_CASE(64);
    else if (e == 128) RF_CASE(128);
    else RF_CASE(256);
#undef RF_CASE
#undef RF_DC
#undef RF_LAUNCH
    if (after_logits && hipEventRecord(after_logits, s) != hipSuccess)
      return lsurge::set_error(LSURGE_ERR_LAUNCH, "router_topk: hipEventRecord failed");
    return LSURGE_OK;
  }
  if (logits && k <= 64) {  // split path: logits kernel over (token, expert) blocks, then one wave per token
    const dim3 lg((unsigned)((t + RL_TOK - 1) / RL_TOK), (unsigned)((e + RL_EXP - 1) / RL_EXP));
    LSURGE_LAUNCH(KID_ROUTER, s,
                  hipLaunchKernelGGL(router_logits_kernel, lg, dim3(RL_THREADS), 0, s, (const bf16_t*)x,
                                     (const bf16_t*)w_r, bias, (int)t, (int)d, (int)e, logits));
    if (after_logits && hipEventRecord(after_logits, s) != hipSuccess)
      return lsurge::set_error(LSURGE_ERR_LAUNCH, "router_topk: hipEventRecord failed");
    if (k <= 16 && t >= 8192) {  // lane per token (enough tokens to fill the GPU); else one wave per token
      const dim3 lg2((unsigned)((t + 255) / 256));
      if (k <= 8)
        LSURGE_LAUNCH(KID_ROUTER_SELECT, s,
                      hipLaunchKernelGGL(router_select_lane_kernel<8>, lg2, dim3(256), 0, s, logits, (int)t, (int)e,
                                         (int)k, sel, weights));
      else
        LSURGE_LAUNCH(KID_ROUTER_SELECT, s,
                      hipLaunchKernelGGL(router_select_lane_kernel<16>, lg2, dim3(256), 0, s, logits, (int)t, (int)e,
                                         (int)k, sel, weights));
      return LSURGE_OK;
    }
    const dim3 sg((unsigned)((t + 3) / 4));
#define RS_CASE(EC)                                                                                        \
  LSURGE_LAUNCH(KID_ROUTER_SELECT, s,                                                                      \
                hipLaunchKernelGGL(router_select_kernel<EC>, sg, dim3(256), 0, s, logits, (int)t, (int)e, (int)k, sel, \
                                   weights))
    if (e <= 64) RS_CASE(1);
    else if (e <= 128) RS_CASE(2);
    else RS_CASE(4);
#undef RS_CASE
    return LSURGE_OK;
  }
  if (after_logits && hipEventRecord(after_logits, s) != hipSuccess)  // one-kernel lane-per-token path
    return lsurge::set_error(LSURGE_ERR_LAUNCH, "router_topk: hipEventRecord failed");
  dim3 grid((unsigned)((t + RT_TOK - 1) / RT_TOK)), block(RT_THREADS);
  const bf16_t* xb = (const bf16_t*)x;
  const bf16_t* wb = (const bf16_t*)w_r;
#define RT_CASE(EP)                                                                                       \
  LSURGE_LAUNCH(KID_ROUTER, s,                                                                            \
                hipLaunchKernelGGL(router_topk_kernel<EP>, grid, block, 0, s, xb, wb, bias, (int)t, (int)d, \
                                   (int)e, (int)k, logits, sel, weights))
  if (e <= 32) RT_CASE(32);
  else if (e <= 64) RT_CASE(64);
  else if (e <= 128) RT_CASE(128);
  else RT_CASE(256);
#undef RT_CASE
  return LSURGE_OK;
}
