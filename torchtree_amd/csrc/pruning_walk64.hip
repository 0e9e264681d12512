// Four-state FP64 passes with at most 4 categories as walks on the matrix cores: the post-order,
// and below it the pre-order.
//
// Reference: calculate_treelikelihood_discrete* (torchtree/evolution/tree_likelihood.py:40-278)
// at S = 4 in double precision.
//
// A wave walks the whole tree for 16 patterns (or four times 16) of one sample with all their
// categories, lane = pattern + 16 state. v_mfma_f64_4x4x4f64 multiplies four 4x4 blocks (A[i][k] in
// lane i + 4 b + 16 k, B[k][j] in lane j + 4 b + 16 k, D[i][j] in lane j + 4 b + 16 i), so with A =
// P in every block and B = four patterns each, a child's product of 16 patterns and one category is
// one instruction, operand and result have the same lanes, and nothing is shared between waves
// until the root sums of a 64-pattern tile's quarters.
//
// What bounds it: the chain of a node (product, maximum over states and categories, scaling) at
// small sizes, where one wave per 64 patterns with P through scalar loads left most of the chip
// idle; the partials' stores at large ones. The matrices of an entry are on their way for kDepth
// entries. Against that kernel, 4 categories with a gradient to follow: 211 taxa x 5003 patterns
// 374 -> 143 us, 64 x 100000 307 -> 244, 64 x 400000 867 -> 903 (eval only 852 -> 352); 64 x 997
// with one category about 55 -> 28.
#include "pruning.hpp"
#include "walk.hpp"

#include <math.h>

#include <type_traits>

namespace hx {

namespace {

using u2 = uint32_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ double buf_load(const __amdgpu_buffer_rsrc_t& r, unsigned off) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)off, 0, 0));
}

// [a0 a1 a2 a3], [b0 b1 b2 b3] (rows of 16 lanes) to [a0 b0 a2 b2], [a1 b1 a3 b3]
__device__ __forceinline__ void swap16(double& a, double& b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  const unsigned l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
  a = __builtin_bit_cast(double, (uint64_t)h0 << 32 | l0);
  b = __builtin_bit_cast(double, (uint64_t)h1 << 32 | l1);
}
// the same to [a0 a1 b0 b1], [a2 a3 b2 b3]
__device__ __forceinline__ void swap32(double& a, double& b) {
  const uint64_t x = __builtin_bit_cast(uint64_t, a), y = __builtin_bit_cast(uint64_t, b);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  const unsigned l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
  a = __builtin_bit_cast(double, (uint64_t)h0 << 32 | l0);
  b = __builtin_bit_cast(double, (uint64_t)h1 << 32 | l1);
}
// over the four states of a pattern (lanes 16 apart)
__device__ __forceinline__ double max_states(double v) {
  double w = v;
  swap16(v, w);
  w = v = fmax(v, w);
  swap32(v, w);
  return fmax(v, w);
}
__device__ __forceinline__ double sum_states(double v) {
  double w = v;
  swap16(v, w);
  w = v = v + w;
  swap32(v, w);
  return v + w;
}
__device__ __forceinline__ double sum_patterns(double v) {
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) v += __shfl_xor(v, o);
  return v;
}

}  // namespace

// LDS: the tip table, the quarters' root sums and exponent stacks.
static size_t post_walk64_lds(int C, int slots, int ncodes) {
  return (size_t)ncodes * 32 + 4 * (size_t)(5 + C) * 8 + 4 * (size_t)slots * 16 * 4 + 16;
}

// prog: walk.hpp, build_post4, without its drop bits (every partial is stored when a gradient may
// follow). A wave takes U quarters of the tile: 1 (block = 256) or 4 (block = 64, kDepth = 2), the
// same sums in the same order. grid = (ntiles, K).
template <int TIPS, int C, bool STORE, int U>
__global__ __launch_bounds__(256 / U) __attribute__((amdgpu_waves_per_eu(U == 1 || C < 3 ? 4 : 2))) void
k_post_walk64(PassArgs<double> a, const int* __restrict__ prog, int nprog, int slots) {
  constexpr int kDepth = U == 1 ? 4 : 2;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int q0 = U == 1 ? uni(threadIdx.x >> 6) : 0, lane = threadIdx.x & 63;  // first quarter
  const int pat = lane & 15, st = lane >> 4;
  const int tile = blockIdx.x, k = blockIdx.y;
  const int n0 = tile * 64 + q0 * 16, n = n0 + pat;
  // patterns of the wave; the others run as padding
  const int left = uni(max(0, min(16 * U, a.N - n0)));
  double* tbl = reinterpret_cast<double*>(smem_raw);                       // [ncodes][4]
  double* red = tbl + (TIPS == HX_TIPS_CODES ? a.ncodes * 4 : 0);          // [4][5 + C]
  int* est = reinterpret_cast<int*>(red + 4 * (5 + C)) + q0 * slots * 16;  // [slots][16 U]
  if constexpr (TIPS == HX_TIPS_CODES) {
    for (int q = threadIdx.x; q < a.ncodes * 4; q += 256 / U) tbl[q] = a.table[q];
    __syncthreads();
  }

  const double* mk = a.mats + (size_t)k * a.B * C * 16;
  const unsigned poff = 8u * (unsigned)((lane & 3) * 4 + st);  // P[i][k] of the lane
  // Category c of the lane's (pattern, state) in node slot s: base + s * sstride + c * cstride. Where the
  // pre-order walk below follows, the 64 values of 16 patterns are in lane order: neighbouring lanes at
  // neighbouring addresses, as a lane of a strided access is a lookup of its own in the vector L1.
  const size_t cstride = (size_t)a.np * 4, sstride = (size_t)a.K * C * cstride;
  double* base = a.partials + (size_t)k * C * cstride + (size_t)n0 * 4 + (a.lanes ? lane : pat * 4 + st);

  // program blocks: lane 4 j + q holds word q of entry 16 blk + j (past the end: zeros, an entry
  // of tip 0 whose operands exist)
  const auto pbuf = buf(prog, (size_t)nprog * kPost4Ints * 4);
  auto block = [&](int blk) {
    return (int)__builtin_amdgcn_raw_buffer_load_b32(pbuf, 4 * lane + 256 * blk, 0, 0);
  };
  int pcur = block(0), pnext = block(1);
  struct Entry {
    int c1, c2, v, m;
  };
  auto entry = [&](int i) __attribute__((always_inline)) {
    const int l = (i & 15) * kPost4Ints;
    return Entry{__builtin_amdgcn_readlane(pcur, l), __builtin_amdgcn_readlane(pcur, l + 1),
                 __builtin_amdgcn_readlane(pcur, l + 2), __builtin_amdgcn_readlane(pcur, l + 3)};
  };
  // Entries and their operands kDepth ahead, loaded on every path (an entry without a tip child
  // reads tip 0): the compiler waits at once for a load that only one path has. A result read back
  // from memory, which is rare, is loaded when it is needed.
  struct In {
    Entry e;
    double p1[C], p2[C], t1[U], t2[U];
    int code1[U], code2[U];
  };
  In in[kDepth];
  auto fetch = [&](int i, In& x) __attribute__((always_inline)) {
    x.e = entry(i);
    const auto r1 = buf(mk + (size_t)(unsigned)x.e.c1 * (C * 16), C * 128);
    const auto r2 = buf(mk + (size_t)(unsigned)x.e.c2 * (C * 16), C * 128);
    const int ty = x.e.m & 3, a1 = ty <= 1 ? x.e.c1 : 0, a2 = ty == 0 ? x.e.c2 : 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      x.p1[c] = buf_load(r1, poff + 128 * c);
      x.p2[c] = buf_load(r2, poff + 128 * c);
    }
    if constexpr (TIPS == HX_TIPS_CODES) {
      const auto s1 = buf(a.codes + (size_t)a1 * a.N + n0, left), s2 = buf(a.codes + (size_t)a2 * a.N + n0, left);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        x.code1[u] = __builtin_amdgcn_raw_buffer_load_b8(s1, pat + 16 * u, 0, 0);
        x.code2[u] = __builtin_amdgcn_raw_buffer_load_b8(s2, pat + 16 * u, 0, 0);
      }
    } else {
      const auto s1 = buf(a.dense + ((size_t)a1 * a.N + n0) * 4, left * 32);
      const auto s2 = buf(a.dense + ((size_t)a2 * a.N + n0) * 4, left * 32);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        x.t1[u] = buf_load(s1, 8u * (pat * 4 + st) + 512 * u);
        x.t2[u] = buf_load(s2, 8u * (pat * 4 + st) + 512 * u);
      }
    }
  };

  double y[U][C], h[U][C];  // the previous and the held result
  int E[U], Eh[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    E[u] = Eh[u] = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) y[u][c] = h[u][c] = 0.0;
  }
  auto step = [&](int i, In& x) __attribute__((always_inline)) {
    const Entry e = x.e;
    const int type = e.m & 3;
    if ((e.m >> 2) & 1) {  // the previous result waits (type 0)
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int c = 0; c < C; ++c) h[u][c] = y[u][c];
        Eh[u] = E[u];
      }
    }
    double l1[U][C];
    if (type == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double t = TIPS == HX_TIPS_CODES ? tbl[x.code2[u] * 4 + st] : x.t2[u];
#pragma unroll
        for (int c = 0; c < C; ++c) y[u][c] = t;
        E[u] = 0;
      }
    }
    if (type <= 1) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const double t = TIPS == HX_TIPS_CODES ? tbl[x.code1[u] * 4 + st] : x.t1[u];
#pragma unroll
        for (int c = 0; c < C; ++c) l1[u][c] = t;
      }
    } else if (type == 2) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int c = 0; c < C; ++c) l1[u][c] = h[u][c];
        E[u] += Eh[u];
      }
    } else {
      const double* src = base + (size_t)(e.c1 - a.T) * sstride;
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int c = 0; c < C; ++c) l1[u][c] = src[c * cstride + 64 * u];
        E[u] += est[((e.m >> 8) & 0xff) * 16 * U + 16 * u + pat];
      }
      // waited for here: after the branch every path would wait, and for all loads
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < C; ++c) asm volatile("" : "+v"(l1[u][c]));
    }
    double M[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      M[u] = 0.0;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const double y1 = __builtin_amdgcn_mfma_f64_4x4x4f64(x.p1[c], l1[u][c], 0.0, 0, 0, 0);
        const double y2 = __builtin_amdgcn_mfma_f64_4x4x4f64(x.p2[c], y[u][c], 0.0, 0, 0, 0);
        y[u][c] = y1 * y2;
        M[u] = fmax(M[u], y[u][c]);
      }
    }
    fetch(i + kDepth, x);
    const bool spill = (e.m >> 4) & 1;
    const bool keep = STORE ? i + 1 < nprog : spill;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const double m = max_states(M[u]);
      // brings the pattern's maximum into [0.5, 1); 0 for none or a non-finite one
      const int ex = m > 0.0 ? __builtin_amdgcn_frexp_exp(m) : 0;
#pragma unroll
      for (int c = 0; c < C; ++c) y[u][c] = __builtin_amdgcn_ldexp(y[u][c], -ex);
      E[u] += ex;
      if (spill && st == 0) est[((e.m >> 16) & 0xff) * 16 * U + 16 * u + pat] = E[u];
    }
    if (keep) {
      double* to = base + (size_t)(e.v - a.T) * sstride;
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int c = 0; c < C; ++c) to[c * cstride + 64 * u] = y[u][c];
    }
  };
#pragma unroll
  for (int d = 0; d < kDepth; ++d) fetch(d, in[d]);
  for (int i = 0; i < nprog;) {
    // (every time, and a whole turn before its use: see above)
    if (((i + kDepth) & 15) == 0) pcur = pnext;
    pnext = block(((i + kDepth) >> 4) + 1);
    __builtin_amdgcn_sched_barrier(0);
    step(i, in[0]);
    if (++i == nprog) break;
    step(i, in[1]);
    ++i;
    if constexpr (kDepth == 4) {
      if (i == nprog) break;
      step(i, in[2]);
      if (++i == nprog) break;
      step(i, in[kDepth - 1]);
      ++i;
    }
  }

  // root: site likelihood sum_c p_c pi.y_c (tree_likelihood.py:71-74, 215-220)
  const double pi = a.freqs[(size_t)k * a.freqs_ks + st];
  double pc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) pc[c] = a.props[(size_t)k * a.props_ks + c];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    double px[C], lik = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      px[c] = sum_states(pi * y[u][c]);
      lik += pc[c] * px[c];
    }
    double acc_l = 0.0, acc_f = 0.0, acc_p[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc_p[c] = 0.0;
    if (n + 16 * u < a.N) {
      const double w = a.weights[n + 16 * u], wi = w / lik;
      acc_l = w * (log(lik) + (double)E[u] * kLn2);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        acc_f += wi * (pc[c] * y[u][c]);
        acc_p[c] = wi * px[c];
      }
    }
    acc_l = sum_patterns(acc_l);
    acc_f = sum_patterns(acc_f);
#pragma unroll
    for (int c = 0; c < C; ++c) acc_p[c] = sum_patterns(acc_p[c]);
    if (pat == 0) {
      double* rq = red + (q0 + u) * (5 + C);
      rq[1 + st] = acc_f;
      if (st == 0) {
        rq[0] = acc_l;
#pragma unroll
        for (int c = 0; c < C; ++c) rq[5 + c] = acc_p[c];
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < 5 + C) {
    double s = 0.0;
    for (int w = 0; w < 4; ++w) s += red[w * (5 + C) + threadIdx.x];
    a.rootsums[((size_t)k * a.ntiles + tile) * (5 + C) + threadIdx.x] = s;
  }
}

// Pre-order, the gradient's pass (its terms: pruning_dna.hip, k_pre). A wave takes 16 patterns, a
// block the four quarters of a tile.
//
// The statistic sum_n Ut[n][i] L[n][j] contracts over patterns, so its operands have lane = state +
// 4 (pattern / 4) + 16 (pattern % 4) ("turned"). The product with its operands exchanged gives the
// turned result from the same registers, so each adjoint is carried in both layouts; partials, which
// come from memory in lane order, are turned by a lane permutation. A child's matrices are one
// contiguous load and become operands through LDS.
//
// A child's statistic of a tile is stored in the parent's own rows, which nothing reads any more:
// its partial was used at the entry before, its adjoint at this one. Waves meet once per entry, in
// LDS, one entry behind.
//
// What bounds it: the chain of an entry (LDS, product, likelihood, division, product, rescale) at 2
// waves per SIMD; the matrix cores are busy 11 % of it at 100,000 patterns. Kernel and sum, against a
// launch per level (k_pre) that read and wrote every adjoint: 64 taxa x 100000 patterns, 4
// categories 858 -> 503 us; 100 x 3000 at 8 samples, d/dtau 552 -> 218; 64 x 997, one category 70 ->
// 51; 211 x 5003 270 and 15 launches' gaps -> 292 (a tree of fewer levels goes by level:
// runs_pre_walk64, pruning.hip).
// Slower: partials and matrices in strided loads (820, 366 and 460 us of the three with 4
// categories), tips looked up an entry ahead without branches (+3 %); the same: one buffer for a
// node's categories.
static size_t pre_walk64_lds(int C, int ncodes) {
  return (size_t)ncodes * 32 + 2 * 4 * (size_t)C * 128 * 8 + 4 * (size_t)C * 32 * 8;
}

__device__ __forceinline__ double permute(int lane4, double v) {
  const uint64_t x = __builtin_bit_cast(uint64_t, v);
  const unsigned lo = __builtin_amdgcn_ds_bpermute(lane4, (int)(unsigned)x);
  const unsigned hi = __builtin_amdgcn_ds_bpermute(lane4, (int)(unsigned)(x >> 32));
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
  const uint64_t x = __builtin_bit_cast(uint64_t, v);
  const unsigned lo = __builtin_amdgcn_mov_dpp((int)(unsigned)x, CTRL, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_mov_dpp((int)(unsigned)(x >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
// over the four states of a pattern, turned (lanes 1 apart)
__device__ __forceinline__ double sum_quad(double v) {
  v += dpp<0xB1>(v);         // 1 0 3 2
  return v + dpp<0x4E>(v);   // 2 3 0 1
}
__device__ __forceinline__ double max_quad(double v) {
  v = fmax(v, dpp<0xB1>(v));
  return fmax(v, dpp<0x4E>(v));
}

// prog: walk.hpp, build_pre4; dropped cherries are stored here.
// grid = (ntiles, K).
template <int TIPS, int C>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_pre_walk64(
    PassArgs<double> a, const int* __restrict__ prog, int nprog) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int q0 = uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int pat = lane & 15, st = lane >> 4;
  const int tst = lane & 3, tpat = (lane & 12) + st;  // turned
  const int tile = blockIdx.x, k = blockIdx.y;
  const int n0 = tile * 64 + q0 * 16;
  const int left = uni(max(0, min(16, a.N - n0)));
  double* red = reinterpret_cast<double*>(smem_raw);  // [2][4 waves][child][C][64]
  double* pl = red + 2 * 4 * C * 128 + q0 * C * 32;   // [child][C][16], the wave's
  double* tbl = red + 2 * 4 * C * 128 + 4 * C * 32;   // [ncodes][4]
  if constexpr (TIPS == HX_TIPS_CODES) {
    for (int q = threadIdx.x; q < a.ncodes * 4; q += 256) tbl[q] = a.table[q];
    __syncthreads();
  }
  const double* mk = a.mats + (size_t)k * a.B * C * 16;
  const int pidx = tst * 4 + st, ptidx = st * 4 + tst;       // P[i][k] and P[k][i] of the lane
  const int turn = 4 * (tst * 16 + tpat), nat = 4 * (pat * 4 + st), nat_t = 4 * (tpat * 4 + tst);
  const size_t cstride = (size_t)a.np * 4, sstride = (size_t)a.K * C * cstride;
  double* base = a.partials + (size_t)k * C * cstride + (size_t)tile * 256;
  // A node's rows of this tile (a slot is 2048 ntiles K C bytes) and category c's of the wave's
  // patterns (any = false: an empty range). 64-bit products of the scalar unit cost more here than
  // the rest of an entry's addresses.
  const unsigned slot = (unsigned)(sstride >> 8);
  const size_t cbytes = cstride * 8;
  char* const base8 = reinterpret_cast<char*>(base);
  auto node = [&](int v) { return base8 + ((size_t)((unsigned)(v - a.T) * slot) << 11); };
  auto rows = [&](char* r, int c, bool any) { return buf(r + c * cbytes + q0 * 512, any ? 512 : 0); };
  const auto mbuf = buf(mk, (size_t)a.B * C * 128);

  // program blocks: lane 16 j + q holds word q of entry 4 blk + j (past the end: the last entry)
  auto block = [&](int blk) {
    return prog[min(4 * blk + (lane >> 4), nprog - 1) * kPre4Ints + (lane & 15)];
  };
  int pcur = block(0), pnext = block(1);
  // Entries and their operands kDepth ahead, loaded on every path (empty ranges read nothing); a
  // popped adjoint one ahead, since the entries between may push it.
  constexpr int kDepth = 4;
  struct In {
    int p, c1, c2, m;
    double mat[2];    // value lane of the child's [C][4][4]
    double l[2][C];   // partials
    double t[2];      // dense tips, value lane of [16][4]
    int code[2];
  };
  In in[kDepth];
  double up[C];
  auto fetch = [&](int i, In& x) __attribute__((always_inline)) {
    const int l = (i & 3) * kPre4Ints;
    x.p = __builtin_amdgcn_readlane(pcur, l);
    x.c1 = __builtin_amdgcn_readlane(pcur, l + 1);
    x.c2 = __builtin_amdgcn_readlane(pcur, l + 2);
    x.m = __builtin_amdgcn_readlane(pcur, l + 3);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int ch = h ? x.c2 : x.c1;
      const bool tip = ch < a.T;
      x.mat[h] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(mbuf, 8 * lane, ch * (C * 128), 0));
      const int t = tip ? ch : 0;
      if constexpr (TIPS == HX_TIPS_CODES)
        x.code[h] = __builtin_amdgcn_raw_buffer_load_b8(buf(a.codes + (size_t)t * a.N + n0, tip ? left : 0), pat, 0, 0);
      else
        x.t[h] = buf_load(buf(a.dense + ((size_t)t * a.N + n0) * 4, tip ? left * 32 : 0), 8 * lane);
      char* r = node(tip ? a.T : ch);
#pragma unroll
      for (int c = 0; c < C; ++c) x.l[h][c] = buf_load(rows(r, c, !tip), 8 * lane);
    }
  };

  const bool val = n0 + tpat < a.N;
  const double w = val ? a.weights[n0 + tpat] : 0.0;
  double pc[C], U[C], UT[C], held[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    pc[c] = a.props[(size_t)k * a.props_ks + c];
    U[c] = held[c] = a.freqs[(size_t)k * a.freqs_ks + st];
    UT[c] = a.freqs[(size_t)k * a.freqs_ks + tst];
  }
  auto mul = [](double x, double y) { return __builtin_amdgcn_mfma_f64_4x4x4f64(x, y, 0.0, 0, 0, 0); };

  // matrices of an entry, through the wave's LDS, to the operands of the products
  double pm[2][C];
  auto stage = [&](const In& x) __attribute__((always_inline)) {
    if (C == 4 || lane < 16 * C) {
      pl[lane] = x.mat[0];
      pl[C * 16 + lane] = x.mat[1];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < C; ++c) pm[h][c] = pl[(h * C + c) * 16 + pidx];
  };
  // The statistics of entry i: (child, category) values q0 and q0 + 4 of the four quarters, added in
  // order, then the four blocks of a product, to the rows of node p.
  constexpr int NF = (2 * C + 3) / 4;
  double fl[NF][4];
  auto gather = [&](int i) __attribute__((always_inline)) {
    lds_barrier();
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const int v = min(q0 + 4 * f, 2 * C - 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) fl[f][q] = red[(size_t)((i & 1) * 4 + q) * C * 128 + v * 64 + lane];
    }
  };
  auto flush = [&](int p) __attribute__((always_inline)) {
    char* to = node(p);
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const int v = q0 + 4 * f, h = v >= C, c = h ? v - C : v;
      double s = ((fl[f][0] + fl[f][1]) + fl[f][2]) + fl[f][3];
      s += dpp<0x124>(s);  // row rotations by 4 and 8 lanes
      s += dpp<0x128>(s);
      // (lanes of the other blocks: past the range)
      const unsigned at = (lane & 12) == 0 ? 8u * (4 * st + tst) : 1024u;
      if (v < 2 * C)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, s), buf(to + c * cbytes + h * 128, 128), (int)at, 0, 0);
    }
  };

  auto step = [&](int i, In& x, const In& nx, int& prev) __attribute__((always_inline)) {
    if ((x.m & 3) >= 2) {
      if ((x.m & 3) == 2) {
#pragma unroll
        for (int c = 0; c < C; ++c) U[c] = up[c];
      } else {
#pragma unroll
        for (int c = 0; c < C; ++c) U[c] = held[c];
      }
#pragma unroll
      for (int c = 0; c < C; ++c) UT[c] = permute(turn, U[c]);
    }
    char* ur = node(nx.p);
#pragma unroll
    for (int c = 0; c < C; ++c) up[c] = buf_load(rows(ur, c, (nx.m & 3) == 2), 8 * lane);
    double pt[2][C], L[2][C], LT[2][C];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < C; ++c) pt[h][c] = pl[(h * C + c) * 16 + ptidx];
    __builtin_amdgcn_wave_barrier();
    if (i > 0) gather(i - 1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if ((h ? x.c2 : x.c1) < a.T) {
        double t, tt;
        if constexpr (TIPS == HX_TIPS_CODES) {
          t = tbl[x.code[h] * 4 + st];
          tt = tbl[__builtin_amdgcn_ds_bpermute(4 * tpat, x.code[h]) * 4 + tst];
        } else {
          t = permute(nat, x.t[h]);
          tt = permute(nat_t, x.t[h]);
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
          L[h][c] = t;
          LT[h][c] = tt;
        }
      } else {
#pragma unroll
        for (int c = 0; c < C; ++c) {
          L[h][c] = x.l[h][c];
          LT[h][c] = permute(turn, x.l[h][c]);
        }
      }
    }
    double Ut[2][C], UtT[2][C], lik = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const double m1 = mul(pm[0][c], L[0][c]), m2 = mul(pm[1][c], L[1][c]);
      const double t1 = mul(L[0][c], pm[0][c]), t2 = mul(L[1][c], pm[1][c]);
      Ut[0][c] = U[c] * m2;
      Ut[1][c] = U[c] * m1;
      UtT[0][c] = UT[c] * t2;
      UtT[1][c] = UT[c] * t1;
      lik = fma(pc[c], UtT[0][c] * t1, lik);
    }
    stage(nx);
    lik = sum_quad(lik);
    const double coef = val ? w / lik : 0.0;
    if (i > 0) flush(prev);
    prev = x.p;
    double* out = red + (size_t)((i & 1) * 4 + q0) * C * 128 + lane;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < C; ++c)
        out[(h * C + c) * 64] = mul(coef * pc[c] * UtT[h][c], LT[h][c]);
    if ((x.m >> 6) & 3) {  // child 1's adjoint waits, in registers or over its partial
      double y[C], M = 0.0;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        y[c] = mul(pt[0][c], Ut[0][c]);
        M = fmax(M, y[c]);
      }
      M = max_states(M);
      const int ex = M > 0.0 ? __builtin_amdgcn_frexp_exp(M) : 0;
#pragma unroll
      for (int c = 0; c < C; ++c) y[c] = __builtin_amdgcn_ldexp(y[c], -ex);
      if (((x.m >> 6) & 3) == 2) {
#pragma unroll
        for (int c = 0; c < C; ++c) held[c] = y[c];
      } else {
        char* r = node(x.c1);
#pragma unroll
        for (int c = 0; c < C; ++c)
          __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, y[c]), rows(r, c, true), 8 * lane, 0, 0);
      }
    }
    if ((x.m >> 8) & 1) {  // child 2's goes on, each layout with its own scale
      double M = 0.0, MT = 0.0;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        U[c] = mul(pt[1][c], Ut[1][c]);
        UT[c] = mul(Ut[1][c], pt[1][c]);
        M = fmax(M, U[c]);
        MT = fmax(MT, UT[c]);
      }
      M = max_states(M);
      MT = max_quad(MT);
      const int ex = M > 0.0 ? __builtin_amdgcn_frexp_exp(M) : 0;
      const int et = MT > 0.0 ? __builtin_amdgcn_frexp_exp(MT) : 0;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        U[c] = __builtin_amdgcn_ldexp(U[c], -ex);
        UT[c] = __builtin_amdgcn_ldexp(UT[c], -et);
      }
    }
  };
  int prev = 0;
  auto run = [&](int i, In& x, const In& nx) __attribute__((always_inline)) {
    step(i, x, nx, prev);
    if (((i + kDepth) & 3) == 0) {
      pcur = pnext;
      pnext = block(((i + kDepth) >> 2) + 1);
    }
    fetch(i + kDepth, x);
  };
#pragma unroll
  for (int d = 0; d < kDepth; ++d) fetch(d, in[d]);
  stage(in[0]);
  for (int i = 0; i < nprog;) {
    run(i, in[0], in[1]);
    if (++i == nprog) break;
    run(i, in[1], in[2]);
    if (++i == nprog) break;
    run(i, in[2], in[3]);
    if (++i == nprog) break;
    run(i, in[3], in[0]);
    ++i;
  }
  gather(nprog - 1);
  flush(prev);
}

// The tiles' statistics, 32 C values of (category, child, entry) per node and sample, in parts of
// the tiles, each with eight loads in flight (43 us of the 503 above, 5 of 292). grid = (nprog, K), block = 32 C parts.
template <int C>
__global__ void k_reduce_walk64(PassArgs<double> a, const int* __restrict__ prog, double* __restrict__ out) {
  __shared__ double sm[1024];
  constexpr int NV = 32 * C, parts = 1024 / NV;
  const int* e = prog + (size_t)blockIdx.x * kPre4Ints;
  const int v = threadIdx.x % NV, part = threadIdx.x / NV, k = blockIdx.y, c = v >> 5, h = (v >> 4) & 1;
  const size_t cstride = (size_t)a.np * 4;
  const double* src = a.partials + (((size_t)(e[0] - a.T) * a.K + k) * C + c) * cstride + (v & 31);
  double s = 0.0;
  int t = part;
  for (; t + 7 * parts < a.ntiles; t += 8 * parts) {
    double x[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) x[q] = src[(size_t)(t + q * parts) * 256];
#pragma unroll
    for (int q = 0; q < 8; ++q) s += x[q];
  }
  for (; t < a.ntiles; t += parts) s += src[(size_t)t * 256];
  sm[threadIdx.x] = s;
  __syncthreads();
  if (part > 0) return;
  for (int q = 1; q < parts; ++q) s += sm[q * NV + v];
  const size_t kb = (size_t)k * a.B + e[1 + h];
  if (a.mats_dt == nullptr) {
    out[(kb * C + c) * 16 + (v & 15)] = s;
  } else {
    s *= a.mats_dt[(kb * C + c) * 16 + (v & 15)];
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) s += __shfl_xor(s, o);
    if ((v & 15) == 0) out[kb * C + c] = s;
  }
}

// -------------------------------------------------------------------- launcher
int launch_post_walk64(const PassArgs<double>& a, const int32_t* prog, int nprog, int slots, int tips,
                       bool store, hipStream_t st) {
  HX_REQUIRE(a.C >= 1 && a.C <= 4, HX_ERR_UNSUPPORTED, "post-order walk: categories");
  HX_REQUIRE(tips != HX_TIPS_CODES || a.T <= 65535, HX_ERR_UNSUPPORTED,
             "post-order walk: too many taxa");
  const size_t lds = post_walk64_lds(a.C, slots, tips == HX_TIPS_CODES ? a.ncodes : 0);
  const dim3 grid((unsigned)a.ntiles, (unsigned)a.K);
  // One wave per tile once there are three of them for every CU: it reads P once for 64 patterns,
  // but a wave per quarter is the shorter chain while there is room for four times the waves. 64
  // taxa x 4 (1) categories: 313 tiles 91 (72) us with one wave, 68 (47) with four; 782 tiles 136
  // (62) and 161 (67); 6250 tiles 903 (303) and 1066 (385). The sums are the same, so a sample's
  // result does not depend on the batch it is in.
  const bool wide = (size_t)a.ntiles * a.K >= 768;
#define HX_W64(TV, CV)                                                                     \
  do {                                                                                     \
    auto kern = wide ? (store ? k_post_walk64<TV, CV, true, 4> : k_post_walk64<TV, CV, false, 4>)  \
                     : (store ? k_post_walk64<TV, CV, true, 1> : k_post_walk64<TV, CV, false, 1>); \
    kern<<<grid, wide ? 64 : 256, lds, st>>>(a, prog, nprog, slots);                       \
  } while (0)
#define HX_W64_C(TV)            \
  switch (a.C) {                \
    case 1: HX_W64(TV, 1); break; \
    case 2: HX_W64(TV, 2); break; \
    case 3: HX_W64(TV, 3); break; \
    default: HX_W64(TV, 4);     \
  }
  if (tips == HX_TIPS_CODES) {
    HX_W64_C(HX_TIPS_CODES)
  } else {
    HX_W64_C(HX_TIPS_DENSE)
  }
#undef HX_W64_C
#undef HX_W64
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

int launch_pre_walk64(const PassArgs<double>& a, const int32_t* prog, int nprog, int tips, double* out,
                      hipStream_t st) {
  HX_REQUIRE(a.C >= 1 && a.C <= 4, HX_ERR_UNSUPPORTED, "pre-order walk: categories");
  const size_t lds = pre_walk64_lds(a.C, tips == HX_TIPS_CODES ? a.ncodes : 0);
  const dim3 grid((unsigned)a.ntiles, (unsigned)a.K), rgrid((unsigned)nprog, (unsigned)a.K);
#define HX_P64(CV)                                                                                     \
  do {                                                                                    \
    if (tips == HX_TIPS_CODES) k_pre_walk64<HX_TIPS_CODES, CV><<<grid, 256, lds, st>>>(a, prog, nprog); \
    else k_pre_walk64<HX_TIPS_DENSE, CV><<<grid, 256, lds, st>>>(a, prog, nprog);         \
    k_reduce_walk64<CV><<<rgrid, 1024 / (32 * CV) * (32 * CV), 0, st>>>(a, prog, out);    \
  } while (0)
  switch (a.C) {
    case 1: HX_P64(1); break;
    case 2: HX_P64(2); break;
    case 3: HX_P64(3); break;
    default: HX_P64(4);
  }
#undef HX_P64
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

}  // namespace hx
