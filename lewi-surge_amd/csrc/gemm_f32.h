// Grouped GEMM on f32 operands with the bf16 matrix cores (the f32 operands of ragged_dot, modal/padded_gmm.py:67-68:
// the einsum runs in lhs.dtype).  An f32 value x is the sum of three bf16 terms x0 = bf16(x), x1 = bf16(x - x0),
// x2 = bf16(x - x0 - x1) (round to nearest even; each difference is exact in f32): 24 significant bits.  The product
// x y is the sum of the six term products of order <= 2 (x0 y0, x1 y0, x2 y0, x0 y1, x0 y2, x1 y1), each exact before
// the MFMA's f32 accumulation.  |x1| <= 2^-8 |x|, |x2| <= 2^-16 |x| and a split's remainder is at most 2^-24 |x|, so of
// what is left out x1 y2, x2 y1 and the two remainders' products are at most 2^-24 |x y| each (x2 y2 2^-32), together at
// most about 2^-22 |x y|.
//
// The split happens while the operands are staged: f32 values go from memory to registers, and from there as three
// bf16 planes into LDS, where the six products of a 16-deep step read each plane's fragments once (24 operand reads
// for 96 MFMAs a wave).  So the operands are read once, in f32, and nothing is written in between; the kernels are
// bound by the matrix cores (2 M K N times six products at the rate their power allows).  They replace a GEMM six times
// as deep over operands that a split kernel wrote out term by term (12 bytes a value).  M = 24576, K = 1024, N = 512, 64
// groups, forward / dlhs / drhs: 382 / 305 / 302 us with the splits -> 161 / 168 / 146 us (956 -> 459 us for the whole
// forward + backward), 1.25 PFLOP/s of bf16 products counting the rows that pad the 256-row tiles.
//
// Shape as the bf16 256 x 256 kernel (gemm256.h): one persistent workgroup of 4 waves per CU, a wave owning 128 x 128 of
// a 256 x 256 tile (256 accumulator registers).  A stage is 16 deep (2 x 3 planes of 8 KiB, double-buffered: 96 KiB) and
// holds six steps of 16 MFMAs, in the order (A term, B term) (0,0) (1,0) (2,0) (0,1) (0,2) (1,1).  Each step reads the
// fragments of the next ones and moves two of the stage's eight copies: split and LDS writes of the next stage's values,
// load of the stage after.  The last step starts with the stage barrier; its operands are the only ones not needed
// first, so it reads the next stage's (0,0) fragments.
#pragma once
#include "gemm256.h"

namespace lsgemm {
namespace f32x3 {

using g256::ctab;
using g256::ld16;
using g256::rsrc;
using g256::rsrc_t;
constexpr int BM = 256, BN = 256, BK = 16, NWG = g256::NWG;
constexpr int PLANE_BYTES = 256 * BK * 2;       // one bf16 term of one operand: 8 KiB
constexpr int OP_BYTES = 3 * PLANE_BYTES;
constexpr int STAGE_BYTES = 2 * OP_BYTES;       // A planes, then B planes
constexpr int RING_BYTES = 2 * STAGE_BYTES;
constexpr int STG_BYTES = 8192;                 // per-wave epilogue staging
constexpr int SMEM_BYTES = RING_BYTES + 4 * STG_BYTES;

// four f32 values -> their three bf16 terms at p, p + PLANE_BYTES and p + 2 PLANE_BYTES (8 bytes each)
__device__ __forceinline__ void put_terms(char* p, u32x4 v) {
  float r[4] = {__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    const u32x2 w = u32x2{pack_bf16x2(r[0], r[1]), pack_bf16x2(r[2], r[3])};
    *reinterpret_cast<u32x2*>(p + t * PLANE_BYTES) = w;
    if (t < 2) {
      r[0] -= __uint_as_float(w[0] << 16);
      r[1] -= __uint_as_float(w[0] & 0xffff0000u);
      r[2] -= __uint_as_float(w[1] << 16);
      r[3] -= __uint_as_float(w[1] & 0xffff0000u);
    }
  }
}

struct Frags {
  bf16x8 a[3][4], b[3][4];
};

// One stage from LDS half `cur`: six steps, see the top of the file.  fa(f, buf, t) / fb(f, buf, t): the four fragments
// of plane t; swrite(c, buf): copy c of the next stage to LDS; gload(c): the same copy of the stage after.
// NRA / NRB: LDS reads of a plane's four fragments.
template <int NRA, int NRB, class FA, class FB, class Swrite, class Gload, class Mma>
__device__ __forceinline__ void run_stage(Frags& f, int cur, FA&& fa, FB&& fb, Swrite&& swrite, Gload&& gload, Mma&& mma) {
  const int nxt = cur ^ 1;
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    if (s == 5) {
      // every wave's copies of the next stage are in LDS, and nobody reads the other half's previous stage any more
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      fa(f, nxt, 0);
      fb(f, nxt, 0);
    } else if (s < 2) {
      fa(f, cur, s + 1);
    } else if (s < 4) {
      fb(f, cur, s - 1);
    }
    if (s < 4) {
#pragma unroll
      for (int c = 2 * s; c < 2 * s + 2; ++c) {
        swrite(c, nxt);
        gload(c);
      }
    }
    constexpr int TA[6] = {0, 1, 2, 0, 0, 1}, TB[6] = {0, 0, 0, 1, 2, 1};
    mma(f, TA[s], TB[s]);
    const int nrd = s == 5 ? NRA + NRB : s < 2 ? NRA : s < 4 ? NRB : 0, nops = nrd + (s < 4 ? 8 : 0);
#pragma unroll
    for (int m = 0; m < 16; ++m) {
      __builtin_amdgcn_sched_group_barrier(g256::SG_MFMA, 1, 0);
      const int o0 = m * nops / 16, o1 = (m + 1) * nops / 16;
#pragma unroll
      for (int o = o0; o < o1; ++o) {
        if (o < nrd) __builtin_amdgcn_sched_group_barrier(g256::SG_DS_R, 1, 0);
        else if ((o - nrd) % 4 < 3) __builtin_amdgcn_sched_group_barrier(g256::SG_DS_W, 1, 0);
        else __builtin_amdgcn_sched_group_barrier(g256::SG_VMEM_R, 1, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// LDS of one plane.  K-major operand: rows of 16 k (32 bytes), the 16-byte half h of row r at slot h ^ ((r >> 3) & 1):
// 16 consecutive rows of one half cover all 64 banks once, and a wave's copy still writes 512 contiguous bytes.  N-major
// operand: two sub-tiles of 16 k rows x 128 columns in the layout of nm_off, read with the transpose read.
template <bool KMAJOR>
__device__ __forceinline__ void frags4(bf16x8 (&f)[4], const char* plane, int w, int lane) {  // wave half w: 128 rows / columns
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (KMAJOR)
      f[i] = as_bf16x8(*reinterpret_cast<const u32x4*>(plane + (w * 128 + 32 * i + (lane & 31)) * 32 +
                                                       16 * ((lane >> 5) ^ ((lane >> 3) & 1))));
    else
      f[i] = frag_n(reinterpret_cast<const bf16_t*>(plane) + w * (BK * 128), 0, 32 * i, lane);
  }
}
// byte offset in its plane of this thread's four values in copy i: K-major row 64 i + tid / 4, k 4 (tid % 4); N-major k
// row 4 i + tid / 64, columns 4 (tid % 64)
template <bool KMAJOR>
__device__ __forceinline__ uint32_t put_off(int i, int tid) {
  if (KMAJOR) return (uint32_t)((64 * i + (tid >> 2)) * 32 + 16 * (((tid >> 1) ^ (tid >> 5)) & 1) + 8 * (tid & 1));
  const int k = 4 * i + (tid >> 6), n = 4 * (tid & 63);
  return (uint32_t)((n >> 7) * (BK * 256) + 2 * nm_off(k, n & 127));
}

// 32 rows x 64 columns per pass of a wave's f32 accumulators to memory through its staging area: rows rbase + ., columns
// col0 .. of a buffer of row pitch pb bytes whose descriptor ends at the last row; columns >= N are dropped.  Branch-free
// as the epilogues of gemm256.h.
template <bool OUT16>
__device__ __forceinline__ void store_rows(const f32x16 (&acc)[4], char* stg, int lane, rsrc_t r, int rbase, uint32_t pb,
                                           int64_t col0, int64_t N) {
  const int fr = lane & 31, fh = lane >> 5;
#pragma unroll
  for (int jp = 0; jp < 2; ++jp) {
#pragma unroll
    for (int jj = 0; jj < 2; ++jj)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int ch = 8 * jj + 2 * q + fh;
        *reinterpret_cast<f32x4*>(stg + fr * 256 + ((ch ^ (fr & 15)) << 4)) =
            f32x4{acc[2 * jp + jj][4 * q], acc[2 * jp + jj][4 * q + 1], acc[2 * jp + jj][4 * q + 2], acc[2 * jp + jj][4 * q + 3]};
      }
#pragma unroll
    for (int it = 0; it < 8; ++it) {
      const int row = 4 * it + (lane >> 4), c = lane & 15;
      const u32x4 v = *reinterpret_cast<const u32x4*>(stg + row * 256 + ((c ^ (row & 15)) << 4));
      const int64_t col = col0 + 64 * jp + 4 * c;
      const uint32_t o = (uint32_t)(rbase + row) * pb;
      if (OUT16) {
        const uint2 h = pack_grad4(LSURGE_BF16, __builtin_bit_cast(f32x4, v));
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{h.x, h.y}, r, col < N ? o + (uint32_t)col * 2u : OOB, 0, 0);
      } else {
        __builtin_amdgcn_raw_buffer_store_b128(v, r, col < N ? o + (uint32_t)col * 4u : OOB, 0, 0);
      }
    }
  }
}

// C[tile rows, n tile] = A[tile rows, :] @ B[expert(tile)] over the 256-row tile table, f32 A and B (B_KN: [K, N] per
// expert; B_NK: [N, K]), f32 or bf16 C.  RowsArgs as g256::rows_kernel, with A and B pointing at f32 values.
template <int BMODE, bool OUT16>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void rows_kernel(RowsArgs a) {
  __shared__ __attribute__((aligned(1024))) char smem[SMEM_BYTES];
  constexpr bool BKM = BMODE == B_NK;
  const int ntr = min(ctab(a.num_tiles, 0), a.max_tiles), total = ntr * a.n_tiles;
  const int xcd = blockIdx.x % 8, nper = gridDim.x / 8;
  const int xbeg = (int)((int64_t)xcd * total / 8), xend = (int)((int64_t)(xcd + 1) * total / 8);
  int t_cur = xbeg + blockIdx.x / 8;
  if (t_cur >= xend) return;
  const float* A = reinterpret_cast<const float*>(a.A);
  const float* B = reinterpret_cast<const float*>(a.B);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int K = (int)a.K, N = (int)a.N;
  const int nk = ((K + 2 * BK - 1) / (2 * BK)) * 2;  // stages per tile, even (a trailing stage of zeros for odd counts)
  const uint32_t lda4 = (uint32_t)a.lda * 4u, ldb4 = (uint32_t)a.ldb * 4u;
  const int kc = 4 * (tid & 3);                                             // K-major: this thread's k within a stage
  const uint32_t ka = (uint32_t)(tid >> 2) * lda4 + 4u * kc, kb = (uint32_t)(tid >> 2) * ldb4 + 4u * kc;
  const uint32_t nb = (uint32_t)(tid >> 6) * ldb4 + 16u * (tid & 63);       // N-major B
  uint32_t wa[4], wb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    wa[i] = put_off<true>(i, tid);
    wb[i] = OP_BYTES + put_off<BKM>(i, tid);
  }
  // load cursor: stage lk of tile lt (past the last tile it re-reads that tile's first stages, which nothing consumes)
  int lt = t_cur, lk = 0;
  rsrc_t la, lb;
  bool ncol_ok = true;
  auto set_ld = [&]() {
    const int b = lt / a.n_tiles, nt = lt % a.n_tiles;
    const int64_t row0 = ctab(a.t_row0, b);
    const float* Bb = B + (int64_t)ctab(a.t_expert, b) * a.b_estride;
    const int64_t n0 = (int64_t)nt * BN;
    la = rsrc(A + row0 * a.lda, (int64_t)ctab(a.t_rows, b) * a.lda * 4);  // rows past the tile: zeros
    if (BKM) {
      lb = rsrc(Bb + n0 * a.ldb, min((int64_t)BN, (int64_t)N - n0) * a.ldb * 4);
    } else {
      lb = rsrc(Bb + n0, ((int64_t)K * a.ldb - n0) * 4);  // rows past K: zeros
      ncol_ok = n0 + 4 * (tid & 63) < N;
    }
  };
  set_ld();
  u32x4 R[8];
  auto gload = [&](int c) {
    const uint32_t k0 = (uint32_t)lk * BK;
    const bool kok = (int)k0 + kc < K;
    if (c < 4) R[c] = ld16(la, kok ? ka + (uint32_t)(64 * c) * lda4 + 4u * k0 : OOB);
    else if (BKM) R[c] = ld16(lb, kok ? kb + (uint32_t)(64 * (c - 4)) * ldb4 + 4u * k0 : OOB);
    else R[c] = ld16(lb, ncol_ok ? nb + (uint32_t)(4 * (c - 4) + k0) * ldb4 : OOB);
  };
  auto adv = [&]() {
    if (++lk == nk) {
      lk = 0;
      if (lt + nper < xend) {
        lt += nper;
        set_ld();
      }
    }
  };
  auto swrite = [&](int c, int buf) { put_terms(smem + buf * STAGE_BYTES + (c < 4 ? wa[c] : wb[c - 4]), R[c]); };
  auto fa = [&](Frags& f, int buf, int t) { frags4<true>(f.a[t], smem + buf * STAGE_BYTES + t * PLANE_BYTES, wm, lane); };
  auto fb = [&](Frags& f, int buf, int t) {
    frags4<BKM>(f.b[t], smem + buf * STAGE_BYTES + OP_BYTES + t * PLANE_BYTES, wn, lane);
  };
  f32x16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
  auto mma = [&](const Frags& f, int ta, int tb) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma32<LSURGE_BF16>(f.b[tb][j], f.a[ta][i], acc[i][j]);
  };
  // prologue: stage 0 in LDS half 0, stage 1 in registers
#pragma unroll
  for (int c = 0; c < 8; ++c) gload(c);
  adv();
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    swrite(c, 0);
    gload(c);
  }
  adv();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  Frags f;
  fa(f, 0, 0);
  fb(f, 0, 0);
  char* const stg = smem + RING_BYTES + wave * STG_BYTES;
  constexpr int NRB = BKM ? 4 : 8;
  while (true) {
    for (int kt = 0; kt < nk; kt += 2) {
      run_stage<4, NRB>(f, 0, fa, fb, swrite, gload, mma);
      adv();
      run_stage<4, NRB>(f, 1, fa, fb, swrite, gload, mma);
      adv();
    }
    int el = lane;  // opaque: the epilogue's offsets are formed here and not held across the K loop
    asm volatile("" : "+v"(el));
    const int b = t_cur / a.n_tiles, nt = t_cur % a.n_tiles, osz = OUT16 ? 2 : 4;
    const int64_t row0 = ctab(a.t_row0, b);
    const rsrc_t rC = rsrc((OUT16 ? reinterpret_cast<const char*>(a.C) : reinterpret_cast<const char*>(a.Cf)) + row0 * a.ldc * osz,
                           (int64_t)ctab(a.t_rows, b) * a.ldc * osz);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      store_rows<OUT16>(acc[i], stg, el, rC, wm * 128 + 32 * i, (uint32_t)a.ldc * osz, (int64_t)nt * BN + wn * 128, N);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
    }
    t_cur += nper;
    if (t_cur >= xend) break;
  }
  __builtin_amdgcn_s_waitcnt(0);  // the loads past the last tile land before the wave ends
}

// Weight gradient C_e[I, N] = A_e^T B_e of f32 A [rows, lda] and B [rows, ldb], reduced over the rows of a chunk of the
// chunk table (WgradArgs; partial slots as in gemm_wgrad_kernel), or, without one, of expert e = chunk (e_row0, e_rows).
// Both operands are N-major.  f32 C.
template <int UNUSED = 0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
void wgrad_kernel(WgradArgs a) {
  __shared__ __attribute__((aligned(1024))) char smem[SMEM_BYTES];
  const int nch = a.c_expert ? min(ctab(a.num_chunks, 0), a.max_chunks) : a.E;
  const int tpc = a.i_tiles * a.n_tiles;
  const int64_t total = (int64_t)nch * tpc;
  const int xcd = blockIdx.x % 8, nper = gridDim.x / 8;
  const int64_t xbeg = xcd * total / 8, xend = (xcd + 1) * total / 8;
  int64_t t_cur = xbeg + blockIdx.x / 8;
  if (t_cur >= xend) return;
  const float* A = reinterpret_cast<const float*>(a.A);
  const float* B = reinterpret_cast<const float*>(a.B);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int I = (int)a.I, N = (int)a.N;
  const uint32_t lda4 = (uint32_t)a.lda * 4u, ldb4 = (uint32_t)a.ldb * 4u;
  const int col = 4 * (tid & 63);
  auto row0_of = [&](int c) { return (int64_t)(a.c_expert ? ctab(a.c_row0, c) : ctab(a.e_row0, c)); };
  auto rows_of = [&](int c) { return a.c_expert ? ctab(a.c_rows, c) : ctab(a.e_rows, c); };
  auto stages_of = [](int rows) { return max(2, (rows + 2 * BK - 1) / (2 * BK) * 2); };  // even, at least one pair
  uint32_t wo[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) wo[i] = put_off<false>(i, tid);
  int64_t lt = t_cur;
  int lk = 0, l_nk = 2;
  rsrc_t la, lb;
  uint32_t ao, bo;  // byte offsets of this thread's columns in its first row (OOB: past I / N)
  auto set_ld = [&]() {
    const int c = (int)(lt / tpc), rem = (int)(lt % tpc), i0 = rem / a.n_tiles * BM, n0 = rem % a.n_tiles * BN;
    const int64_t row0 = row0_of(c);
    const int rows = rows_of(c);
    la = rsrc(A + row0 * a.lda, (int64_t)rows * a.lda * 4);  // rows past the chunk: zeros
    lb = rsrc(B + row0 * a.ldb, (int64_t)rows * a.ldb * 4);
    ao = i0 + col < I ? (uint32_t)(tid >> 6) * lda4 + 4u * (uint32_t)(i0 + col) : OOB;
    bo = n0 + col < N ? (uint32_t)(tid >> 6) * ldb4 + 4u * (uint32_t)(n0 + col) : OOB;
    l_nk = stages_of(rows);
  };
  set_ld();
  u32x4 R[8];
  auto gload = [&](int c) {
    const uint32_t r = (uint32_t)(4 * (c & 3) + lk * BK);
    if (c < 4) R[c] = ld16(la, ao & OOB ? OOB : ao + r * lda4);
    else R[c] = ld16(lb, bo & OOB ? OOB : bo + r * ldb4);
  };
  auto adv = [&]() {
    if (++lk == l_nk) {
      lk = 0;
      if (lt + nper < xend) {
        lt += nper;
        set_ld();
      }
    }
  };
  auto swrite = [&](int c, int buf) { put_terms(smem + buf * STAGE_BYTES + (c < 4 ? 0 : OP_BYTES) + wo[c & 3], R[c]); };
  auto fa = [&](Frags& f, int buf, int t) { frags4<false>(f.a[t], smem + buf * STAGE_BYTES + t * PLANE_BYTES, wm, lane); };
  auto fb = [&](Frags& f, int buf, int t) {
    frags4<false>(f.b[t], smem + buf * STAGE_BYTES + OP_BYTES + t * PLANE_BYTES, wn, lane);
  };
  f32x16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
  auto mma = [&](const Frags& f, int ta, int tb) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma32<LSURGE_BF16>(f.b[tb][j], f.a[ta][i], acc[i][j]);
  };
#pragma unroll
  for (int c = 0; c < 8; ++c) gload(c);
  adv();
#pragma unroll
  for (int c = 0; c < 8; ++c) {
    swrite(c, 0);
    gload(c);
  }
  adv();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  Frags f;
  fa(f, 0, 0);
  fb(f, 0, 0);
  char* const stg = smem + RING_BYTES + wave * STG_BYTES;
  while (true) {
    const int c = (int)(t_cur / tpc), rem = (int)(t_cur % tpc);
    const int nk = stages_of(rows_of(c));
    for (int kt = 0; kt < nk; kt += 2) {
      run_stage<8, 8>(f, 0, fa, fb, swrite, gload, mma);
      adv();
      run_stage<8, 8>(f, 1, fa, fb, swrite, gload, mma);
      adv();
    }
    int el = lane;
    asm volatile("" : "+v"(el));
    const int i0 = rem / a.n_tiles * BM, n0 = rem % a.n_tiles * BN;
    const int part = a.c_expert ? ctab(a.c_part, c) : -1, e = a.c_expert ? ctab(a.c_expert, c) : c;
    const int64_t pitch = part >= 0 ? N : a.ldc;
    const float* dst = part >= 0 ? a.part + (int64_t)part * I * N : a.C + (int64_t)e * a.c_estride;
    const rsrc_t rC = rsrc(dst + i0 * pitch, min((int64_t)BM, (int64_t)I - i0) * pitch * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      store_rows<false>(acc[i], stg, el, rC, wm * 128 + 32 * i, (uint32_t)pitch * 4u, (int64_t)n0 + wn * 128, N);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f32x16{};
    }
    t_cur += nper;
    if (t_cur >= xend) break;
  }
  __builtin_amdgcn_s_waitcnt(0);
}

}  // namespace f32x3
}  // namespace lsgemm
