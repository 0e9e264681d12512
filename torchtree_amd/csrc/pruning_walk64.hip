// Four-state FP64 post-order with at most 4 categories as a walk on the matrix cores.
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
  // category c of the lane's pattern in node slot s: base + s * sstride + c * cstride
  // (layout [slot][K][C][np][4])
  const size_t cstride = (size_t)a.np * 4, sstride = (size_t)a.K * C * cstride;
  double* base = a.partials + (size_t)k * C * cstride + (size_t)n * 4;
  // stores: lane (pattern, r) of group g holds the four states of the (quarter, category) 4 g + r
  constexpr int NG = (U * C + 3) / 4;
  size_t stoff[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) stoff[g] = (4 * g + st) % C * cstride + 64 * ((4 * g + st) / C);

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
      const double* src = base + (size_t)(e.c1 - a.T) * sstride + st;
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
      for (int g = 0; g < NG; ++g) {
        double z[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int f = 4 * g + r < U * C ? 4 * g + r : 0;
          z[r] = y[f / C][f % C];
        }
        swap16(z[0], z[1]);
        swap16(z[2], z[3]);
        swap32(z[0], z[2]);
        swap32(z[1], z[3]);
        if (4 * NG == U * C || 4 * g + st < U * C) {
          double2* dst = reinterpret_cast<double2*>(to + stoff[g]);
          dst[0] = make_double2(z[0], z[1]);
          dst[1] = make_double2(z[2], z[3]);
        }
      }
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

}  // namespace hx
