// Four-state (nucleotide) pruning kernels on the vector units: one fused post-order walk of the
// whole tree per pattern tile at more than 4 categories (FP32 and FP64; the other calls:
// pruning_walk.hip, pruning_walk64.hip), and the pre-order adjoint one tree level per launch for
// these and for FP64 calls of few patterns on large trees.
//
// Reference: calculate_treelikelihood_discrete* (torchtree/evolution/
// tree_likelihood.py:40-278) at S = 4, where each node update is two 4x4
// matrix-vector products per (sample, pattern, category): HBM-bound work.
//
// Partials use the category-major layout
//   partials [slot][K][C][np][4]  slot = node - T, np = 64 x tiles
// so a wave's accesses to one category are contiguous 16-byte vectors, and
// the padding lanes of the last tile have slots of their own.
//
// Post-order (k_post_walk): lane = pattern with all C categories in the lane,
// one wave per (tile, sample), walking the tree program; each internal
// partial is written once and read back only by the lane that wrote it, when
// a child waited on the stack. Pre-order: k_pre runs one tree level per
// launch with thread = (pattern, category).
#include "pruning.hpp"
#include "walk.hpp"

#include <math.h>

#include <type_traits>

namespace hx {

namespace {

template <typename R>
struct alignas(4 * sizeof(R)) V4 {
  R x[4];
};

template <typename R>
__device__ __forceinline__ V4<R> ld4(const R* p) {
  V4<R> v;
  if constexpr (sizeof(R) == 4) {
    const float4 q = *reinterpret_cast<const float4*>(p);
    v.x[0] = q.x, v.x[1] = q.y, v.x[2] = q.z, v.x[3] = q.w;
  } else {
    const double2 q0 = reinterpret_cast<const double2*>(p)[0];
    const double2 q1 = reinterpret_cast<const double2*>(p)[1];
    v.x[0] = q0.x, v.x[1] = q0.y, v.x[2] = q1.x, v.x[3] = q1.y;
  }
  return v;
}

template <typename R>
__device__ __forceinline__ void st4(R* p, const V4<R>& v) {
  if constexpr (sizeof(R) == 4) {
    *reinterpret_cast<float4*>(p) = make_float4(v.x[0], v.x[1], v.x[2], v.x[3]);
  } else {
    reinterpret_cast<double2*>(p)[0] = make_double2(v.x[0], v.x[1]);
    reinterpret_cast<double2*>(p)[1] = make_double2(v.x[2], v.x[3]);
  }
}

template <typename R>
__device__ __forceinline__ V4<R> zero4() {
  V4<R> v;
#pragma unroll
  for (int s = 0; s < 4; ++s) v.x[s] = R(0);
  return v;
}

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Read-only data read with wave-uniform addresses (the walk program, P
// matrices) goes through the constant address space so the compiler always
// uses scalar loads; those are counted apart from vector memory, so waiting
// for them never waits for the partials' stores.
template <typename T>
using cptr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ cptr<T> to_const(const T* p) {
  return (cptr<T>)p;
}

__device__ __forceinline__ float fmax_(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double fmax_(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ float frexp_(float m, int* e) { return frexpf(m, e); }
__device__ __forceinline__ double frexp_(double m, int* e) { return frexp(m, e); }
__device__ __forceinline__ float ldexp_(float x, int e) { return ldexpf(x, e); }
__device__ __forceinline__ double ldexp_(double x, int e) { return ldexp(x, e); }

// The 4x4 block at p (16 consecutive values, wave-uniform address).
template <typename R>
__device__ __forceinline__ void load_p16(cptr<R> p, R (&P)[16]) {
#pragma unroll
  for (int i = 0; i < 16; ++i) P[i] = p[i];
}

template <typename R>
__device__ __forceinline__ V4<R> mv(const R (&P)[16], const V4<R>& x) {
  V4<R> y;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    R acc = R(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = fma(P[4 * i + j], x.x[j], acc);
    y.x[i] = acc;
  }
  return y;
}

template <typename R>
__device__ __forceinline__ V4<R> mv_t(const R (&P)[16], const V4<R>& x) {
  V4<R> y;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    R acc = R(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = fma(P[4 * i + j], x.x[i], acc);
    y.x[j] = acc;
  }
  return y;
}

template <typename R>
__device__ __forceinline__ R max4(const V4<R>& v) {
  return fmax_(fmax_(v.x[0], v.x[1]), fmax_(v.x[2], v.x[3]));
}

// Exponent that brings the pattern maximum M into [0.5, 1); 0 for M = 0 or
// non-finite M (the partial then carries its value unscaled).
template <typename R>
__device__ __forceinline__ int scale_exp(R M) {
  int e = 0;
  if (M > R(0) && isfinite(M)) frexp_(M, &e);
  return e;
}

template <typename R>
__device__ __forceinline__ void scale4(V4<R>& v, int e) {
  if (e != 0) {
#pragma unroll
    for (int s = 0; s < 4; ++s) v.x[s] = ldexp_(v.x[s], -e);
  }
}

__device__ __forceinline__ size_t prow(int T, int K, int C, int N, int v, int k, int c) {
  return (((size_t)(v - T) * K + k) * C + c) * (size_t)N;
}

template <typename R, int TIPS>
__device__ __forceinline__ void stage_tbl(const PassArgs<R>& a, V4<R>* tbl, int nt) {
  if constexpr (TIPS == HX_TIPS_CODES) {
    for (int i = threadIdx.x; i < a.ncodes; i += nt) tbl[i] = ld4(a.table + 4 * i);
  }
}

// Outer-product accumulation g += w u (x) l.
template <typename R>
__device__ __forceinline__ void acc_outer(R (&g)[16], R w, const V4<R>& u, const V4<R>& l) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const R wu = w * u.x[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) g[4 * i + j] = fma(wu, l.x[j], g[4 * i + j]);
  }
}

}  // namespace

// ------------------------------------------------------------------ post-order
// A block of W waves walks the whole tree for one 64-pattern tile; wave w
// handles sample blockIdx.y * W + w and lane l pattern 64 tile + l with all C
// categories of it, so the rescaling maximum and the root likelihood never
// leave the lane and the waves never synchronise after staging. The tile's
// tip codes (T x 64 bytes) are staged in LDS once per block; P of each
// (branch, category) is wave-uniform (scalar loads, SGPR operands).
//
// prog: kWalkInts ints per internal node in walk order (walk.hpp). A child is
// a tip, the previous entry's result (registers), or an earlier result that
// waited on the stack: its partial is read back from the copy this lane
// wrote to HBM (in L2 in practice), issued one node ahead and before that
// node's stores so the wait for it does not wait for them, and its exponent
// comes from the lane's LDS stack. grid = (ntiles, ceil(K / W)), block = 64 W.
// CM: categories rounded up to a power of two (EXACT: C == CM).
__device__ __forceinline__ void store_row_f32(const __amdgpu_buffer_rsrc_t& r, unsigned off,
                                              const V4<float>& v) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const u4 w = {__float_as_uint(v.x[0]), __float_as_uint(v.x[1]), __float_as_uint(v.x[2]),
                __float_as_uint(v.x[3])};
  __builtin_amdgcn_raw_buffer_store_b128(w, r, (int)off, 0, 0);
}

template <typename R, int TIPS, int CM, bool EXACT>
__global__ __launch_bounds__(CM >= 8 ? 256 : 1024) void k_post_walk(PassArgs<R> a, const R* __restrict__ mats,
                                                    const int4* __restrict__ prog, int nprog,
                                                    int ne, int W) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int C = EXACT ? CM : a.C;
  const int wave = uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tile = blockIdx.x, k = blockIdx.y * W + wave;
  const int n = tile * 64 + lane;
  const bool val = n < a.N;
  uint8_t* lc = smem_raw;                                              // [T][64]
  const size_t lc_bytes = TIPS == HX_TIPS_CODES ? (size_t)a.T * 64 : 0;
  V4<R>* tbl = reinterpret_cast<V4<R>*>(smem_raw + lc_bytes);          // [ncodes]
  int* est = reinterpret_cast<int*>(tbl + (TIPS == HX_TIPS_CODES ? a.ncodes : 0)) +
             (size_t)wave * ne * 64;                                   // [W][ne][64]
  const int nt = blockDim.x;
  if constexpr (TIPS == HX_TIPS_CODES) {
    const size_t stride = (size_t)a.ntiles * 64;
    for (int i = threadIdx.x; i < a.T * 4; i += nt) {
      const int row = i >> 2, q = i & 3;
      *reinterpret_cast<uint4*>(lc + row * 64 + q * 16) =
          *reinterpret_cast<const uint4*>(a.codes_pad + row * stride + tile * 64 + q * 16);
    }
  }
  stage_tbl<R, TIPS>(a, tbl, nt);
  __syncthreads();
  if (k >= a.K) return;

  // element offsets: node slot s, category c of this lane's pattern at
  // base + s * sstride + c * cstride (layout [slot][K][C][np][4], np = 64 ntiles,
  // so the padding lanes of the last tile have slots of their own)
  const size_t cstride = (size_t)a.np * 4;
  const size_t sstride = (size_t)a.K * C * cstride;
  R* base = a.partials + (size_t)k * C * cstride + (size_t)n * 4;
  const cptr<R> mk = to_const(mats) + (size_t)k * a.B * C * 16;
  const cptr<int> cprog = to_const(reinterpret_cast<const int*>(prog));
  auto entry = [&](int i, int4& f0, int4& f1) {
    const cptr<int> q = cprog + (size_t)kWalkInts * i;
    f0.x = q[0], f0.y = q[1], f0.z = q[2], f0.w = q[3];
    f1.x = q[4], f1.y = q[5], f1.z = q[6], f1.w = q[7];
  };

  auto tip = [&](int ch) -> V4<R> {
    if constexpr (TIPS == HX_TIPS_CODES) return tbl[lc[ch * 64 + lane]];
    else return val ? ld4(a.dense + ((size_t)ch * a.N + n) * 4) : zero4<R>();
  };
  // Issued every node, for the stacked child of the next entry or, when it
  // has none, from this sample's P blocks (a few hot cache lines, value
  // unused): every iteration then issues the same vector memory operations,
  // so the wait for these loads counts only the older ones and not this
  // node's stores, and the placeholder loads never reach HBM.
  auto stacked_of = [&](const int4& f0, const int4& f1) {
    if ((f1.z & 0xff) == 2) return f0.y;
    if (((f1.z >> 8) & 0xff) == 2) return f0.z;
    return -1;
  };
  const R* hot = mats + (size_t)k * a.B * C * 16 + (lane & 3) * 4;
  auto readback = [&](int ch, V4<R>(&x)[CM]) {
    const bool real = ch >= 0;
    const R* p = base + (size_t)(real ? ch - a.T : 0) * sstride;
#pragma unroll
    for (int c = 0; c < CM; ++c)
      if (EXACT || c < C) x[c] = ld4(real ? p + (size_t)c * cstride : hot);
  };

  // The first entry of a walk has two tip children, so xs is first read
  // after a loop iteration has issued its read-back and stores.
  V4<R> y[CM], xs[CM];
  int E = 0;
  int4 e0, e1;
  entry(0, e0, e1);
  // entries 0 .. nprog-2 store their partial; the last entry is the root
  for (int i = 0; i < nprog; ++i) {
    const bool last = i + 1 == nprog;
    const int v = e0.x, l = e0.y, r = e0.z;
    const int sl = (e0.w & 0xff) - 1, sr = ((e0.w >> 8) & 0xff) - 1, so = e0.w >> 16;
    const int kl = e1.z & 0xff, kr = (e1.z >> 8) & 0xff;
    int4 f0 = e0, f1 = e1;
    if (i + 1 < nprog) entry(i + 1, f0, f1);
    V4<R> xl[CM], xr[CM];
    int El = 0, Er = 0;
    if (kl == 0) {
      const V4<R> t = tip(l);
#pragma unroll
      for (int c = 0; c < CM; ++c) xl[c] = t;
    } else if (kl == 1) {
#pragma unroll
      for (int c = 0; c < CM; ++c) xl[c] = y[c];
      El = E;
    } else {
#pragma unroll
      for (int c = 0; c < CM; ++c) xl[c] = xs[c];
      El = est[sl * 64 + lane];
    }
    if (kr == 0) {
      const V4<R> t = tip(r);
#pragma unroll
      for (int c = 0; c < CM; ++c) xr[c] = t;
    } else if (kr == 1) {
#pragma unroll
      for (int c = 0; c < CM; ++c) xr[c] = y[c];
      Er = E;
    } else {
#pragma unroll
      for (int c = 0; c < CM; ++c) xr[c] = xs[c];
      Er = est[sr * 64 + lane];
    }
    // P of (l, c) and (r, c); the loads of category c + 1 are issued before
    // category c is computed
    R M = R(0);
    R Pl[2][16], Pr[2][16];
    load_p16(mk + (size_t)l * C * 16, Pl[0]);
    load_p16(mk + (size_t)r * C * 16, Pr[0]);
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      if (EXACT || c < C) {
        if (c + 1 < CM && (EXACT || c + 1 < C)) {
          load_p16(mk + ((size_t)l * C + c + 1) * 16, Pl[(c + 1) & 1]);
          load_p16(mk + ((size_t)r * C + c + 1) * 16, Pr[(c + 1) & 1]);
        }
        const V4<R> yl = mv(Pl[c & 1], xl[c]);
        const V4<R> yr = mv(Pr[c & 1], xr[c]);
#pragma unroll
        for (int s = 0; s < 4; ++s) y[c].x[s] = yl.x[s] * yr.x[s];
        M = fmax_(M, max4(y[c]));
      } else {
        y[c] = zero4<R>();
      }
    }
    const int e = scale_exp(M);
#pragma unroll
    for (int c = 0; c < CM; ++c) scale4(y[c], e);
    E = El + Er + e;
    if (last) break;
    // the next entry's stacked child, before this node's stores
    readback(stacked_of(f0, f1), xs);
    if constexpr (sizeof(R) == 4) {
      // this node's C rows of this sample as one raw buffer: no address on the vector units (2 % of
      // the walk at 6 categories)
      const R* node = a.partials + (size_t)(v - a.T) * sstride + (size_t)k * C * cstride;
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<R*>(node), (short)0, (int)((size_t)C * cstride * sizeof(R)), 0x00020000);
#pragma unroll
      for (int c = 0; c < CM; ++c)
        if (EXACT || c < C) store_row_f32(rs, (unsigned)((c * cstride + (size_t)n * 4) * sizeof(R)), y[c]);
    } else {
      R* p = base + (size_t)(v - a.T) * sstride;
#pragma unroll
      for (int c = 0; c < CM; ++c)
        if (EXACT || c < C) st4(p + (size_t)c * cstride, y[c]);
    }
    est[so * 64 + lane] = E;
    e0 = f0;
    e1 = f1;
  }

  // root: site likelihood sum_c p_c pi.x_c (tree_likelihood.py:71-74, 215-220)
  R pi[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) pi[s] = a.freqs[(size_t)k * a.freqs_ks + s];
  R px[CM];
  R lik = R(0);
#pragma unroll
  for (int c = 0; c < CM; ++c) {
    px[c] = R(0);
    if (c < C) {
#pragma unroll
      for (int s = 0; s < 4; ++s) px[c] = fma(pi[s], y[c].x[s], px[c]);
      lik += a.props[(size_t)k * a.props_ks + c] * px[c];
    }
  }
  double acc[5 + CM];  // loglik, dfreqs[4], dprops[c]
#pragma unroll
  for (int q = 0; q < 5 + CM; ++q) acc[q] = 0.0;
  if (val) {
    const double w = a.weights[n];
    const double dl_ = (double)lik;
    const double wi = w / dl_;
    acc[0] = w * (log(dl_) + (double)E * kLn2);
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      if (c < C) {
        const R pc = a.props[(size_t)k * a.props_ks + c];
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[1 + s] += wi * (double)(pc * y[c].x[s]);
        acc[5 + c] = wi * (double)px[c];
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 5 + CM; ++q)
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) acc[q] += __shfl_xor(acc[q], o);
  double* out = a.rootsums + ((size_t)k * a.ntiles + tile) * (5 + C);
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 5 + CM; ++q)
      if (q < 5 + C) out[q] = acc[q];
  }
}

// ------------------------------------------------------------------- pre-order
// For parent p with children a, b and pre-order partial U_p (root: freqs):
//   Ut_a = U_p * (P_b L_b), Ut_b = U_p * (P_a L_a)
//   lik  = sum_c p_c Ut_a.(P_a L_a)                    (scaled site likelihood)
//   d loglik / d P_a[c][i][j] += w p_c Ut_a[i] L_a[j] / lik
//   U_a  = P_a^T Ut_a, rescaled (scale-free: every term is a ratio), written
//          over L_a in place
// Thread (pattern, category) with the CP = next_pow2(C) categories of a
// pattern in adjacent lanes: the likelihood sum and the rescaling maximum are
// shuffles within those lanes, so the tile loop has no barriers. The two P
// blocks are staged in LDS once per block; each branch statistic accumulates
// in registers over the block's chunk of 64-pattern tiles.
template <typename R>
struct PreTile {
  V4<R> U;
  V4<R> L[2];
  int code[2];
};

template <int CP, typename T>
__device__ __forceinline__ T qsum(T v) {
#pragma unroll
  for (int o = 1; o < CP; o <<= 1) v += __shfl_xor(v, o);
  return v;
}

template <int CP, typename T>
__device__ __forceinline__ T qmax(T v) {
#pragma unroll
  for (int o = 1; o < CP; o <<= 1) v = fmax_(v, __shfl_xor(v, o));
  return v;
}

// Entries of a 16-entry statistic transposed per pass so that the buffer
// [64][CP][NE + 1] stays within 36 KiB.
constexpr int pre_pass_entries(int cp, int rb) {
  int ne = 16;
  while (ne > 1 && (size_t)64 * cp * (ne + 1) * rb > 36 * 1024) ne >>= 1;
  return ne;
}

template <typename R, int TIPS, bool ROOT, int CP>
__global__ __launch_bounds__(64 * CP) void k_pre(PassArgs<R> a, const R* __restrict__ mats,
                                                 const R* __restrict__ mats_dt,
                                                 const int32_t* __restrict__ nodes) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int C = a.C, nt = 64 * CP;
  const int t = threadIdx.x, c = t % CP, pl = t / CP;
  const bool cval = c < C;
  const int cc = cval ? c : 0;
  const int chunk = blockIdx.x, k = blockIdx.y;
  const int p = nodes[blockIdx.z];
  int ch[2];
  bool in_c[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    ch[h] = a.kids[2 * p + h];
    in_c[h] = ch[h] >= a.T;
  }
  R* Ps = reinterpret_cast<R*>(smem_raw);                         // [2][C][16]
  V4<R>* tbl = reinterpret_cast<V4<R>*>(Ps + 2 * C * 16);         // [ncodes]
  // gb: [64 patterns][CP][NE + 1] statistic transpose for the chunk
  // reduction, NE of the 16 entries per pass
  constexpr int NE = pre_pass_entries(CP, sizeof(R));
  R* gb = reinterpret_cast<R*>(tbl + (TIPS == HX_TIPS_CODES ? a.ncodes : 0));
  for (int i = t; i < 2 * C * 16; i += nt) {
    const int h = i / (C * 16), rem = i - h * C * 16;
    Ps[i] = mats[((size_t)k * a.B + ch[h]) * C * 16 + rem];
  }
  stage_tbl<R, TIPS>(a, tbl, nt);

  const R pc = cval ? a.props[(size_t)k * a.props_ks + c] : R(0);
  V4<R> pi;
  if constexpr (ROOT) {
#pragma unroll
    for (int s = 0; s < 4; ++s) pi.x[s] = a.freqs[(size_t)k * a.freqs_ks + s];
  }
  R g[2][16];
#pragma unroll
  for (int i = 0; i < 16; ++i) g[0][i] = g[1][i] = R(0);

  auto fetch = [&](int tile, PreTile<R>& in) {
    const int n = tile * 64 + pl;
    in.U = zero4<R>();
    if constexpr (!ROOT) {
      if (cval) in.U = ld4(a.partials + (prow(a.T, a.K, C, a.np, p, k, cc) + n) * 4);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      in.L[h] = zero4<R>();
      in.code[h] = 0;
      if (in_c[h]) {
        if (cval) in.L[h] = ld4(a.partials + (prow(a.T, a.K, C, a.np, ch[h], k, cc) + n) * 4);
      } else if constexpr (TIPS == HX_TIPS_CODES) {
        if (n < a.N) in.code[h] = a.codes[(size_t)ch[h] * a.N + n];
      } else {
        if (n < a.N) in.L[h] = ld4(a.dense + ((size_t)ch[h] * a.N + n) * 4);
      }
    }
  };
  auto getP = [&](int h, R(&P)[16]) {
    const R* src = Ps + (h * C + cc) * 16;
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const V4<R> v = ld4(src + i);
      P[i] = v.x[0], P[i + 1] = v.x[1], P[i + 2] = v.x[2], P[i + 3] = v.x[3];
    }
  };

  // No software prefetch of the next tile: its registers cost a wave per
  // SIMD of occupancy, which hides the load latency better (measured).
  const int t0 = chunk * a.tiles_per_chunk;
  const int t1 = min(t0 + a.tiles_per_chunk, a.ntiles);
  __syncthreads();  // P blocks and code table staged
  for (int tile = t0; tile < t1; ++tile) {
    PreTile<R> cur;
    fetch(tile, cur);
    const int n = tile * 64 + pl;
    const bool val = n < a.N && cval;
    const R w = val ? (R)a.weights[n] : R(0);
    V4<R> U = cur.U;
    if constexpr (ROOT) U = cval ? pi : zero4<R>();
    V4<R> PL[2], Ut[2];
    R P[16];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (TIPS == HX_TIPS_CODES) {
        if (!in_c[h]) cur.L[h] = tbl[cur.code[h]];
      }
      getP(h, P);
      PL[h] = mv(P, cur.L[h]);
    }
    R d = R(0);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      Ut[0].x[s] = U.x[s] * PL[1].x[s];
      Ut[1].x[s] = U.x[s] * PL[0].x[s];
      d = fma(Ut[0].x[s], PL[0].x[s], d);
    }
    d = qsum<CP>(d * pc);
    const R coef = val ? w / d * pc : R(0);
    acc_outer(g[0], coef, Ut[0], cur.L[0]);
    acc_outer(g[1], coef, Ut[1], cur.L[1]);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (in_c[h]) {
        getP(h, P);
        V4<R> Uc = mv_t(P, Ut[h]);
        scale4(Uc, scale_exp(qmax<CP>(max4(Uc))));
        if (cval) st4(a.partials + (prow(a.T, a.K, C, a.np, ch[h], k, cc) + n) * 4, Uc);
      }
    }
  }

  // Chunk reduction of each branch statistic over the tile's 64 patterns:
  // transpose through LDS, thread (ci = (c, entry), part) sums 16 patterns,
  // then the 4 parts combine by shuffles (in double).
  auto flush = [&](const R(&gv)[16], int b) {
    const int part = t & 3, ci = t >> 2, c2 = ci >> 4, e = ci & 15;
    double sum = 0.0;
#pragma unroll
    for (int e0 = 0; e0 < 16; e0 += NE) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NE; ++i) gb[(pl * CP + c) * (NE + 1) + i] = gv[e0 + i];
      __syncthreads();
      if (e >= e0 && e < e0 + NE) {
#pragma unroll
        for (int j = 0; j < 16; ++j)
          sum += (double)gb[((part * 16 + j) * CP + c2) * (NE + 1) + (e - e0)];
      }
    }
    sum += __shfl_xor(sum, 1);
    sum += __shfl_xor(sum, 2);
    if (mats_dt != nullptr) {
      // lanes (c2, e, part) of one category c2 form one wave: contract over e
      double tv = (part == 0 && c2 < C)
                      ? sum * (double)mats_dt[(((size_t)k * a.B + b) * C + c2) * 16 + e] : 0.0;
#pragma unroll
      for (int o = 4; o < 64; o <<= 1) tv += __shfl_xor(tv, o);
      if ((t & 63) == 0 && c2 < C) a.gtau[(((size_t)b * a.K + k) * a.nchunks + chunk) * C + c2] = tv;
    } else if (part == 0 && c2 < C) {
      a.gpart[((((size_t)b * a.K + k) * a.nchunks + chunk) * C + c2) * 16 + e] = (R)sum;
    }
  };
#pragma unroll
  for (int h = 0; h < 2; ++h) flush(g[h], ch[h]);
}

// ------------------------------------------------------------------ launchers
static size_t tbl_bytes(int tips, int ncodes, size_t rb) {
  return tips == HX_TIPS_CODES ? (size_t)ncodes * 4 * rb : 0;
}

// Copies tip codes [T][N] into rows of ntiles * 64 bytes (zero padded) so the
// walk stages a tile's codes with aligned 16-byte loads.
// grid (ceil(npad / 1024), T): thread j4 writes bytes 4 j4 .. 4 j4 + 3 of row blockIdx.y as
// one 32-bit store (npad is a multiple of 64, so the stores are aligned)
__global__ void k_pad_codes(const uint8_t* __restrict__ codes, uint8_t* __restrict__ out, int T,
                            int N, int npad) {
  const int t = blockIdx.y;
  const int j = 4 * (blockIdx.x * blockDim.x + threadIdx.x);
  if (j >= npad) return;
  const uint8_t* src = codes + (size_t)t * N;
  uint32_t v = 0;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (j + q < N) v |= (uint32_t)src[j + q] << (8 * q);
  *reinterpret_cast<uint32_t*>(out + (size_t)t * npad + j) = v;
}

template <typename R>
int launch_post_dna(const PassArgs<R>& a, const int32_t* prog, int nprog, int need, int tips,
                    hipStream_t st) {
  // W samples share the staged codes; 8 keeps their P matrices (K B C 64 B
  // per sample) within L2; many categories need a smaller block (registers)
  const int wmax = a.C > 4 ? 4 : 8;
  int W = a.K < wmax ? a.K : wmax;
  while (W > 1 && dna_walk_lds(a.T, W, need, tips, a.ncodes, sizeof(R)) > kDnaWalkLdsMax) W >>= 1;
  const size_t lds = dna_walk_lds(a.T, W, need, tips, a.ncodes, sizeof(R));
  HX_REQUIRE(lds <= kDnaWalkLdsMax, HX_ERR_UNSUPPORTED,
             "post-order walk: tip codes of the tile exceed LDS (too many taxa)");
  HX_REQUIRE(sizeof(R) == 8 || (size_t)a.C * a.np * 4 * sizeof(R) < ((size_t)1 << 31),
             HX_ERR_UNSUPPORTED, "post-order walk: a node's rows of one sample exceed 2 GiB");
  if (tips == HX_TIPS_CODES) {
    const size_t npad = (size_t)a.ntiles * 64;
    HX_REQUIRE(a.T <= 65535, HX_ERR_UNSUPPORTED, "post-order walk: too many taxa");
    k_pad_codes<<<dim3((unsigned)((npad / 4 + 255) / 256), (unsigned)a.T), 256, 0, st>>>(
        a.codes, a.codes_pad, a.T, a.N, (int)npad);
  }
  dim3 grid(a.ntiles, (a.K + W - 1) / W);
  const int4* pg = reinterpret_cast<const int4*>(prog);
#define HX_WALK(CMV, EX)                                                                     \
  do {                                                                                       \
    auto kern = tips == HX_TIPS_CODES ? k_post_walk<R, HX_TIPS_CODES, CMV, EX>               \
                                      : k_post_walk<R, HX_TIPS_DENSE, CMV, EX>;              \
    if (lds > 64 * 1024)                                                                     \
      HX_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),                    \
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
    kern<<<grid, 64 * W, lds, st>>>(a, a.mats, pg, nprog, need, W);                          \
  } while (0)
  if constexpr (sizeof(R) == 4) {
    switch (a.C) {
      case 1: HX_WALK(1, true); break;
      case 2: HX_WALK(2, true); break;
      case 3: HX_WALK(4, false); break;
      case 4: HX_WALK(4, true); break;
      default:
        if (a.C <= 8) HX_WALK(8, false);
        else HX_WALK(16, false);
    }
  } else {
    HX_REQUIRE(a.C > 4, HX_ERR_INVALID_ARGUMENT, "post-order walk: categories");
    if (a.C <= 8) HX_WALK(8, false);
    else HX_WALK(16, false);
  }
#undef HX_WALK
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

template <typename R>
int launch_pre_dna(const PassArgs<R>& a, const int32_t* nodes, int width, int tips, bool root,
                   hipStream_t st) {
  const int cp = next_pow2(a.C);
  const size_t rb = sizeof(R);
  const int ne = pre_pass_entries(cp, (int)rb);
  const size_t lds = (size_t)2 * a.C * 16 * rb + tbl_bytes(tips, a.ncodes, rb) +
                     (size_t)64 * cp * (ne + 1) * rb;
  HX_REQUIRE(lds <= kDnaLdsBudget, HX_ERR_UNSUPPORTED, "pre-order LDS exceeds the 64 KiB budget");
  dim3 grid(a.nchunks, a.K, width);
  const int threads = 64 * cp;
#define HX_PRE(TV, RV, CPV) \
  k_pre<R, TV, RV, CPV><<<grid, threads, lds, st>>>(a, a.mats, a.mats_dt, nodes)
#define HX_PRE_T(CPV)                                                                        \
  if (tips == HX_TIPS_CODES) {                                                               \
    if (root) HX_PRE(HX_TIPS_CODES, true, CPV); else HX_PRE(HX_TIPS_CODES, false, CPV);      \
  } else {                                                                                   \
    if (root) HX_PRE(HX_TIPS_DENSE, true, CPV); else HX_PRE(HX_TIPS_DENSE, false, CPV);      \
  }
  switch (cp) {
    case 1: HX_PRE_T(1) break;
    case 2: HX_PRE_T(2) break;
    case 4: HX_PRE_T(4) break;
    case 8: HX_PRE_T(8) break;
    default: HX_PRE_T(16) break;
  }
#undef HX_PRE_T
#undef HX_PRE
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

template int launch_post_dna<float>(const PassArgs<float>&, const int32_t*, int, int, int,
                                    hipStream_t);
template int launch_post_dna<double>(const PassArgs<double>&, const int32_t*, int, int, int,
                                     hipStream_t);
template int launch_pre_dna<float>(const PassArgs<float>&, const int32_t*, int, int, bool,
                                   hipStream_t);
template int launch_pre_dna<double>(const PassArgs<double>&, const int32_t*, int, int, bool,
                                    hipStream_t);

}  // namespace hx
