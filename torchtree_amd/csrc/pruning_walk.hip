// Four-state FP32 pruning at up to 4 categories: the post-order and the pre-order pass, each one
// launch that walks the whole tree per 64-pattern tile with every 4 x 4 product on the matrix
// cores.
//
// Reference: calculate_treelikelihood_discrete* (torchtree/evolution/tree_likelihood.py:40-278)
// at S = 4, and its autograd backward.
//
// Lane = pattern, register = (category, state): that is both the B operand and the accumulator
// layout of v_mfma_f32_4x4x1_16b_f32 (B[b][col] in lane 4 b + col, D[b][row][col] in register row
// of lane 4 b + col), so y = P x takes four of them (one per state of x) and needs no data
// movement: block b works on patterns 4 b .. 4 b + 3, and its A operand, column j of P, is the
// same for every block. The instruction's block broadcast (CBSZ = 4, ABID) takes that column from
// one block of a register, and a register's 16 blocks hold the 16 columns of P for four
// categories: lane 16 c + 4 j + i carries P_c[i][j]. One 4-byte load per lane is therefore a whole
// [C][4][4] set of P, and the same load in memory order (lane 16 c + 4 i + j) is the set of P^T.
//
// What bounds the walks: at few waves (a served job of 413 taxa x 9,871 patterns, 8 samples: 1.2
// waves per SIMD) the instruction chain of one node, at many (512 taxa x 100,000 patterns, 32
// samples) the stores of the post-order and the LDS and issue slots of the pre-order. P used to
// sit in scalar registers, whose loads return out of order, so that each category of each node
// waited for a scalar-cache miss (about 0.5 us); as vector loads, counted in order, they run
// ahead. Measured against that, the whole call: 60 taxa x 431 patterns, 8 samples, d/dtau: 337 -> 187
// us; 413 x 9,871, 8 samples, d/dtau: 2.72 -> 1.55 ms; 512 x 20,011, 4 samples, log-likelihood alone:
// 1.13 -> 0.33 ms; 512 x 100,000, 32 samples, d/dP: 55.9 -> 47.4 ms (post-order 20.2 -> 14.8 ms,
// pre-order 33.9 -> 31.7 ms).
//
// Tried here and slower: categories across lanes instead of registers (16 to 64 patterns per wave,
// the statistic's transposes as products with the identity; d/dtau then in FP32 per pattern on both
// sides): 413 x 9,871 1.65-2.1 ms against 1.41, 512 x 100,000 58-77 ms against 48.6; a load around which the program branches (the register
// copies that join the two paths wait for it at once): the pre-order walks +8 %.
#include "pruning.hpp"
#include "walk.hpp"

#include <type_traits>
#include <utility>

namespace hx {

namespace {

using f4 = float __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

template <typename F, int... Is>
__device__ __forceinline__ void each_impl(F&& f, std::integer_sequence<int, Is...>) {
  (f(std::integral_constant<int, Is>{}), ...);
}
// f(0), f(1), ..., f(N - 1) with compile-time arguments
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  each_impl(f, std::make_integer_sequence<int, N>{});
}

// y_c = M_c x(c) for every category, M the P set p; x(c) is category c's vector. The four steps of
// a product depend on each other, so the categories take turns.
template <int CM, typename X>
__device__ __forceinline__ void mv4(float p, X&& x, f4 (&y)[CM]) {
#pragma unroll
  for (int c = 0; c < CM; ++c) y[c] = f4{0.f, 0.f, 0.f, 0.f};
  each<4>([&](auto j) {
    each<CM>([&](auto c) {
      constexpr int cc = decltype(c)::value, jj = decltype(j)::value;
      y[cc] = __builtin_amdgcn_mfma_f32_4x4x1f32(p, x(c)[jj], y[cc], 4, 4 * cc + jj, 0);
    });
  });
}

__device__ __forceinline__ float max4(const f4& v) {
  return fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
}

// Exponent that brings the pattern maximum M into [0.5, 1); 0 for M <= 0 or non-finite M.
__device__ __forceinline__ int scale_exp(float M) {
  const int e = __builtin_amdgcn_frexp_expf(M);  // 0 for zero, infinities and NaN
  return M > 0.f ? e : 0;
}

// One power of two over the C categories of a lane's pattern; returns its exponent.
template <int CM, bool EXACT>
__device__ __forceinline__ int rescale(f4 (&y)[CM], int C) {
  float M = 0.f;
#pragma unroll
  for (int c = 0; c < CM; ++c)
    if (EXACT || c < C) M = fmaxf(M, max4(y[c]));
  const int e = scale_exp(M);
#pragma unroll
  for (int c = 0; c < CM; ++c)
#pragma unroll
    for (int s = 0; s < 4; ++s) y[c][s] = ldexpf(y[c][s], -e);
  return e;
}

// Loads and stores go through raw buffers: a wave-uniform descriptor and offset in scalar
// registers plus one 32-bit lane offset, so no address is formed on the vector units.
using u4 = uint32_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float buf_load(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                          unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)lane_off, (int)off, 0));
}
// NT: streaming (non-temporal), for data that is read once
template <bool NT>
__device__ __forceinline__ f4 buf_load4(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                        unsigned off) {
  return __builtin_bit_cast(
      f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, (int)off, NT ? 2 : 0));
}
__device__ __forceinline__ void buf_store4(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                           unsigned off, const f4& v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), r, (int)lane_off, (int)off, 0);
}

template <int TIPS>
__device__ __forceinline__ void stage_table(const PassArgs<float>& a, f4* tbl) {
  if constexpr (TIPS == HX_TIPS_CODES) {
    for (int i = threadIdx.x; i < a.ncodes; i += blockDim.x)
      tbl[i] = *reinterpret_cast<const f4*>(a.table + 4 * i);
    __syncthreads();
  }
}

// Tip t's code (all codes lie within 4 GiB, checked at the launch) and dense partial at pattern n.
__device__ __forceinline__ int tip_code(const __amdgpu_buffer_rsrc_t& codes, unsigned t, unsigned N,
                                        unsigned n) {
  return __builtin_amdgcn_raw_buffer_load_b8(codes, (int)n, (int)(t * N), 0);
}
__device__ __forceinline__ f4 tip_row(const PassArgs<float>& a, int t, unsigned n) {
  return buf_load4<false>(buf(a.dense + (size_t)t * a.N * 4, (size_t)a.N * 16), n * 16, 0);
}

// Byte offset in a [C][4][4] set at which a lane reads its value of the P set (trans: of P^T).
// Lanes of categories past C repeat the last one, whose results are not used.
__device__ __forceinline__ unsigned p_offset(int lane, int C, bool trans) {
  const int c = min(lane >> 4, C - 1), q = (lane >> 2) & 3, r = lane & 3;
  return 4u * (unsigned)(trans ? 16 * c + 4 * q + r : 16 * c + 4 * r + q);
}

}  // namespace

// ------------------------------------------------------------------ post-order
// A wave walks the tree program (walk.hpp, build_post4) for one (tile, sample); waves share
// nothing but the tip table, so there is no barrier after staging. P sets and tip codes are
// loaded kAhead entries before their use, a spilled child one entry before, and the stores are
// issued for every entry (a dropped cherry's with an empty range, which the hardware discards),
// so the waits count loads exactly and never a recent store. The program itself comes in blocks of
// 16 entries, one word per lane, read by v_readlane: no scalar load is outstanding when the
// tip table is read from LDS (the two share a counter, and scalar loads return out of order).
// STORE: a gradient may follow, so every internal partial but the dropped cherries' and the root's
// is stored; otherwise (hx_loglik_value) only spilled results are.
// grid = (ntiles, ceil(K / W)), block = 64 W.
constexpr int kAhead = 3;

template <int TIPS>
struct PostIn {
  float p1, p2;
  int c1, c2;
  f4 t1, t2;  // dense tips
};

template <int TIPS, int CM, bool EXACT, bool STORE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_post_walk4(
    PassArgs<float> a, const float* __restrict__ mats, const int* __restrict__ prog, int nprog,
    int slots, int W) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int C = EXACT ? CM : a.C;
  const int wave = uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tile = blockIdx.x, k = blockIdx.y * W + wave;
  const int n = tile * 64 + lane;
  const bool val = n < a.N;
  f4* tbl = reinterpret_cast<f4*>(smem_raw);
  int* est = reinterpret_cast<int*>(tbl + (TIPS == HX_TIPS_CODES ? a.ncodes : 0)) +
             (size_t)wave * slots * 64;
  stage_table<TIPS>(a, tbl);
  if (k >= a.K) return;

  const size_t cstride = (size_t)a.np * 4;
  float* rows = a.partials + (size_t)k * C * cstride + (size_t)tile * 256;  // + slot, category
  const auto pbuf = buf(mats + (size_t)k * a.B * C * 16, (size_t)a.B * C * 64);
  const unsigned poff = p_offset(lane, C, false), loff = lane * 16u;
  const unsigned cbytes = (unsigned)(cstride * 4), nbytes = (C - 1) * cbytes + 1024;
  const unsigned nc = val ? n : a.N - 1;  // padding lanes read the last pattern's tips
  const auto cbuf = buf(a.codes, (size_t)a.T * a.N);
  const unsigned skb = (unsigned)((size_t)a.K * C * cstride >> 8);  // a slot's size in KiB
  auto node_buf = [&](int v, unsigned bytes) {
    return buf(reinterpret_cast<char*>(rows) + ((size_t)((unsigned)(v - a.T) * skb) << 10), bytes);
  };

  // program blocks: lane 4 j + q holds word q of entry 16 blk + j (past the end: the last entry)
  auto block = [&](int blk) {
    return prog[min(16 * blk + (lane >> 2), nprog - 1) * kPost4Ints + (lane & 3)];
  };
  int pcur = block(0), pnext = block(1);
  struct Entry {
    int c1, c2, v, m;
  };
  auto entry = [&](int i) {  // entry i of the current block
    const int l = (i & 15) * kPost4Ints;
    return Entry{__builtin_amdgcn_readlane(pcur, l), __builtin_amdgcn_readlane(pcur, l + 1),
                 __builtin_amdgcn_readlane(pcur, l + 2), __builtin_amdgcn_readlane(pcur, l + 3)};
  };
  auto fetch = [&](const Entry& e, PostIn<TIPS>& in) {
    in.p1 = buf_load(pbuf, poff, e.c1 * C * 64);
    in.p2 = buf_load(pbuf, poff, e.c2 * C * 64);
    const int t = e.m & 3;
    const int t1 = t <= 1 ? e.c1 : 0, t2 = t == 0 ? e.c2 : 0;
    if constexpr (TIPS == HX_TIPS_CODES) {
      in.c1 = tip_code(cbuf, t1, a.N, nc);
      in.c2 = tip_code(cbuf, t2, a.N, nc);
    } else {
      in.t1 = tip_row(a, t1, nc);
      in.t2 = tip_row(a, t2, nc);
    }
  };

  f4 y[CM], h[CM], xs[CM];
  int E = 0, Eh = 0;
#pragma unroll
  for (int c = 0; c < CM; ++c) y[c] = h[c] = xs[c] = f4{0.f, 0.f, 0.f, 0.f};
  // ring of kAhead + 1 entries (loads of entry i + kAhead are issued in entry i)
  constexpr int R = kAhead + 1;
  Entry ent[R];
  PostIn<TIPS> in[R];
  // (in order: the loop's waits are the weakest that hold for this entry too)
  each<R - 1>([&](auto j) {
    __builtin_amdgcn_sched_barrier(0);
    ent[j] = entry(j);
    fetch(ent[j], in[j]);
  });
  __builtin_amdgcn_sched_barrier(0);

  auto step = [&](int i, auto slot) __attribute__((always_inline)) {
    constexpr int s = decltype(slot)::value, nx = (s + 1) % R, ah = (s + kAhead) % R;
    const Entry e = ent[s];
    if (((i + kAhead) & 15) == 0) {
      pcur = pnext;
      pnext = block(((i + kAhead) >> 4) + 1);
    }
    ent[ah] = entry(i + kAhead);
    fetch(ent[ah], in[ah]);
    const PostIn<TIPS>& x = in[s];
    const int type = e.m & 3;
    if ((e.m >> 2) & 1) {
#pragma unroll
      for (int c = 0; c < CM; ++c) h[c] = y[c];
      Eh = E;
    }
    f4 y1[CM], y2[CM];
    if (type == 0) {
      f4 t;
      if constexpr (TIPS == HX_TIPS_CODES) t = tbl[x.c2]; else t = x.t2;
      mv4<CM>(x.p2, [&](auto) { return t; }, y2);
    } else {
      mv4<CM>(x.p2, [&](auto c) { return y[c]; }, y2);
    }
    if (type <= 1) {
      f4 t;
      if constexpr (TIPS == HX_TIPS_CODES) t = tbl[x.c1]; else t = x.t1;
      mv4<CM>(x.p1, [&](auto) { return t; }, y1);
      if (type == 0) E = 0;
    } else if (type == 2) {
      mv4<CM>(x.p1, [&](auto c) { return h[c]; }, y1);
      E += Eh;
    } else {
      mv4<CM>(x.p1, [&](auto c) { return xs[c]; }, y1);
      E += est[((e.m >> 8) & 0xff) * 64 + lane];
    }
#pragma unroll
    for (int c = 0; c < CM; ++c) y[c] = y1[c] * y2[c];
    E += rescale<CM, EXACT>(y, C);
    // the next entry's spilled child, before this node's stores
    if ((ent[nx].m & 3) == 3) {
      const auto r = node_buf(ent[nx].c1, nbytes);
#pragma unroll
      for (int c = 0; c < CM; ++c)
        if (EXACT || c < C) xs[c] = buf_load4<false>(r, loff, c * cbytes);
    }
    const bool spill = (e.m >> 4) & 1;
    if (spill) est[((e.m >> 16) & 0xff) * 64 + lane] = E;
    if (STORE || spill) {
      const bool empty = (((e.m >> 3) & 1) && a.drop) || i + 1 == nprog;  // (the root's: never read)
      const auto r = node_buf(e.v, empty ? 0 : nbytes);
#pragma unroll
      for (int c = 0; c < CM; ++c)
        if (EXACT || c < C) buf_store4(r, loff, c * cbytes, y[c]);
    }
  };
  static_assert(R == 4, "the ring's four steps");
  for (int i = 0; i < nprog; ++i) {
    step(i, std::integral_constant<int, 0>{});
    if (++i == nprog) break;
    step(i, std::integral_constant<int, 1>{});
    if (++i == nprog) break;
    step(i, std::integral_constant<int, 2>{});
    if (++i == nprog) break;
    step(i, std::integral_constant<int, 3>{});
  }

  // root: site likelihood sum_c p_c pi.x_c (tree_likelihood.py:71-74, 215-220)
  float pi[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) pi[s] = a.freqs[(size_t)k * a.freqs_ks + s];
  float px[CM];
  float lik = 0.f;
#pragma unroll
  for (int c = 0; c < CM; ++c) {
    px[c] = 0.f;
    if (c < C) {
#pragma unroll
      for (int s = 0; s < 4; ++s) px[c] = fmaf(pi[s], y[c][s], px[c]);
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
        const float pc = a.props[(size_t)k * a.props_ks + c];
#pragma unroll
        for (int s = 0; s < 4; ++s) acc[1 + s] += wi * (double)(pc * y[c][s]);
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
// A block's W waves walk the same program (walk.hpp, build_pre4) for W consecutive tiles of one
// sample, grid = (ceil(ntiles / W), K). Entry (p; 1, 2) with p's adjoint U (the frequencies at
// the root):
//   m_h  = P_h L_h,  Ut_1 = U * m_2,  Ut_2 = U * m_1        (per category)
//   lik  = sum_c p_c sum_s U m_1 m_2                         (scaled site likelihood)
//   G_h[c][i][j] = sum over patterns of (w p_c / lik) Ut_h[c][i] L_h[c][j], or
//   dtau_h[c]    = sum over i, j of G_h[c][i][j] dP_h/dtau[c][i][j]
//   U_h  = P_h^T Ut_h with one power-of-two rescale over all categories
// Every term is a ratio, so the scales of U and L cancel. A dropped cherry's partial is rebuilt
// from its two tips' codes; the continuing adjoint stays in registers, a pushed one too when
// nothing else is pushed before its pop, and otherwise in the child's own partials row, which has
// been read by then.
//
// All of an entry's loads are issued in the entry before it, ahead of that entry's store (the
// adjoint it pushes, which the next entry never pops); an empty range reads nothing.
//
// G: each wave writes (w / lik) Ut (rows 4c + i) and L (rows 4c + j) to LDS, pattern minor, and
// reads them back as the operands of 4 CM v_mfma_f32_4x4x1_16b_f32, whose blocks share the patterns
// of a category out: block (16 / CM) c + q sums its 4 x 4 outer products over 4 CM of them. Row
// rotations add four blocks; what is left of a category (4 / CM rows of 16 lanes) and the W waves'
// G meet in LDS one entry later (one barrier per entry, two buffers). With rows and products for
// four categories whatever their number (56 KB of LDS: 2 waves per SIMD) the calls of one category
// were behind a walk on the vector units, 64 taxa x 400,000 patterns, 4 samples, a caterpillar, d/dP:
// 1294 us against 1651 (1166 now); 256 x 100,000, 2 samples, 2 categories, d/dP: 1315 -> 1061.
//
// dtau: the 16 sums of a (child, category) meet dP/dtau in FP64 on their way out. Rows of dP/dtau sum
// to zero, so this contraction cancels. Done in FP32, per pattern and ahead of the sums, it needs no
// transposes, but its error against 64 bits was 1.04 to 1.1 times as large (the calls 60 taxa x 431
// patterns and 413 x 9871 at 8 samples took 135 and 1380 us so, 164 and 1504 as here); in FP64 per
// pattern they took 177 and 1854.
//
// Row stride (floats) of the LDS pattern transposes, and where a block's patterns lie: with four
// categories 16 running ones, with fewer fours 64 / CM apart. Either way the 16-byte reads of 16
// lanes (4 rows, 4 blocks) fall on different banks.
constexpr int xs_stride(int CM) { return CM == 4 ? 68 : 80; }

// v + (v from the lane `ROT` below in the same row of 16 lanes, cyclically): DPP row_ror
template <int ROT>
__device__ __forceinline__ float add_row_ror(float v) {
  static_assert(ROT > 0 && ROT < 16, "row rotation");
  return v + __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v),
                                                                 0x120 + ROT, 0xF, 0xF, true));
}
constexpr size_t pre4_lds_floats(int CM) {
  return (size_t)kPreWalkW * 3 * 4 * CM * xs_stride(CM) + 4 * kPreWalkW * 64;
}

template <int TIPS, int CM, bool EXACT, bool TAU>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CM == 4 ? 2 : 3))) void
k_pre_walk4(PassArgs<float> a, const float* __restrict__ mats, const float* __restrict__ mats_dt,
            const int* __restrict__ prog, int nprog) {
  constexpr int W = kPreWalkW;  // waves (tiles) per workgroup
  constexpr int RW = 4 * CM;    // rows of a transposed set
  constexpr int RC = 4 / CM;    // rows of 16 lanes per category
  constexpr int kXS = xs_stride(CM);
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int C = EXACT ? CM : a.C;
  const int wave = uni(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int chunk = blockIdx.x, k = blockIdx.y;
  const int tile = chunk * W + wave;
  // waves past the last tile repeat it with zero weight and store nothing
  const bool tval = tile < a.ntiles;
  const int tl = tval ? tile : a.ntiles - 1;
  const int n = tl * 64 + lane;
  const bool val = tval && n < a.N;
  float* sm = reinterpret_cast<float*>(smem_raw);
  float* xs = sm + (size_t)wave * 3 * RW * kXS;  // rows 4c + i: (w / lik) Ut[c][i] of one child
  float* ls = xs + RW * kXS;                     // [2] rows 4c + j: L[c][j] (a tip: rows j)
  float* red = sm + (size_t)W * 3 * RW * kXS;    // [2][2][W][64]
  f4* tbl = reinterpret_cast<f4*>(sm + pre4_lds_floats(CM));
  for (int i = lane; i < 3 * RW * kXS; i += 64) xs[i] = 0.f;  // rows of absent categories
  stage_table<TIPS>(a, tbl);

  const float w = val ? (float)a.weights[n] : 0.f;
  float pc[CM];
#pragma unroll
  for (int c = 0; c < CM; ++c) pc[c] = (EXACT || c < C) ? a.props[(size_t)k * a.props_ks + c] : 0.f;
  f4 pi;
#pragma unroll
  for (int s = 0; s < 4; ++s) pi[s] = a.freqs[(size_t)k * a.freqs_ks + s];

  const size_t cstride = (size_t)a.np * 4;
  float* rows = a.partials + (size_t)k * C * cstride + (size_t)tl * 256;  // + slot, category
  const size_t moff = (size_t)k * a.B * C * 16, mbytes = (size_t)a.B * C * 64;
  const auto pbuf = buf(mats + moff, mbytes), dbuf = buf(TAU ? mats_dt + moff : mats, mbytes);
  const unsigned pf = p_offset(lane, C, false), pt = p_offset(lane, C, true), loff = lane * 16u;
  const unsigned cbytes = (unsigned)(cstride * 4), nbytes = (C - 1) * cbytes + 1024;
  const unsigned nc = n < a.N ? n : a.N - 1;  // padding lanes read the last pattern's tips
  const auto cbuf = buf(a.codes, (size_t)a.T * a.N);
  const unsigned skb = (unsigned)((size_t)a.K * C * cstride >> 8);  // a slot's size in KiB
  auto node_buf = [&](int v, unsigned bytes) {
    return buf(reinterpret_cast<char*>(rows) + ((size_t)((unsigned)(v - a.T) * skb) << 10), bytes);
  };

  // program blocks: lane 16 j + q holds word q of entry 4 blk + j (past the end: the last entry)
  auto block = [&](int blk) {
    return prog[min(4 * blk + (lane >> 4), nprog - 1) * kPre4Ints + (lane & 15)];
  };
  int pcur = block(0), pnext = block(1);
  struct Entry {
    int p, c1, c2, m, g[4];
  };
  auto entry = [&](int i) {  // entry i of the current block
    const int l = (i & 3) * kPre4Ints;
    Entry e;
    e.p = __builtin_amdgcn_readlane(pcur, l);
    e.c1 = __builtin_amdgcn_readlane(pcur, l + 1);
    e.c2 = __builtin_amdgcn_readlane(pcur, l + 2);
    e.m = __builtin_amdgcn_readlane(pcur, l + 3);
#pragma unroll
    for (int q = 0; q < 4; ++q) e.g[q] = __builtin_amdgcn_readlane(pcur, l + 4 + q);
    return e;
  };
  // child h's partial: 0 a tip, 1 a dropped cherry, 2 stored
  const bool drops = TIPS == HX_TIPS_CODES && a.drop;
  auto kind = [&](int m, int h) {
    const int q = (m >> (2 + 2 * h)) & 3;
    return q == 1 && !drops ? 2 : q;
  };

  struct Small {
    float p[2], pt[2], g[2][2];         // P, P^T; P of a dropped cherry's tips
    int code[2][2];                     // a tip's code, or a dropped cherry's two
    f4 t[2];                            // dense tips
    float dp;                           // TAU: this thread's value of dP/dtau (flush_g)
  };
  Small in[2];
  f4 U[CM], held[CM], L0[CM], L1[CM], Up[CM];
#pragma unroll
  for (int c = 0; c < CM; ++c) U[c] = held[c] = pi;
  // The rows of a node, or nothing (an empty range reads no memory): the registers are written
  // on every path, since a branch around the loads would end in copies that wait for them.
  auto load_rows = [&](int node, bool any, f4(&x)[CM], auto nt) {
    const auto r = node_buf(node, any ? nbytes : 0);
    // a post-order partial is read once: streaming, so that pushed adjoints stay in L2
#pragma unroll
    for (int c = 0; c < CM; ++c)
      if (EXACT || c < C) x[c] = buf_load4<decltype(nt)::value>(r, loff, c * cbytes);
  };
  auto Lh = [&](auto h) -> f4(&)[CM] {
    if constexpr (decltype(h)::value == 0) return L0; else return L1;
  };
  // the statistic of thread t: value t mod CS of child t / CS's G
  const int CS = C * 16, sh = (int)threadIdx.x >= CS, se = threadIdx.x % CS;
  auto fetch_small = [&](const Entry& e, Small& x) {
    each<2>([&](auto hc) {
      constexpr int h = decltype(hc)::value;
      const int ch = h ? e.c2 : e.c1;
      x.p[h] = buf_load(pbuf, pf, ch * C * 64);
      const int kd = kind(e.m, h);
      if constexpr (TIPS == HX_TIPS_CODES) {
        x.code[h][0] = tip_code(cbuf, kd == 0 ? ch : e.g[2 * h], a.N, nc);
        x.code[h][1] = tip_code(cbuf, e.g[2 * h + 1], a.N, nc);
        x.g[h][0] = buf_load(pbuf, pf, e.g[2 * h] * C * 64);
        x.g[h][1] = buf_load(pbuf, pf, e.g[2 * h + 1] * C * 64);
      } else {
        x.t[h] = tip_row(a, kd == 0 ? ch : 0, nc);
      }
      x.pt[h] = buf_load(pbuf, pt, ch * C * 64);
    });
    if constexpr (TAU) x.dp = buf_load(dbuf, 4u * ((sh ? e.c2 : e.c1) * CS + se), 0);
  };
  auto fetch_rows = [&](const Entry& e) {
    load_rows(e.c1, kind(e.m, 0) == 2, L0, std::true_type{});
    load_rows(e.c2, kind(e.m, 1) == 2, L1, std::true_type{});
    load_rows(e.p, (e.m & 3) == 2, Up, std::false_type{});
  };

  // the statistics of entry i meet in LDS during entry i + 1
  const float spc = a.props[(size_t)k * a.props_ks + (se >> 4)];
  auto flush_g = [&](int b1, int b2, float dp, int par) {
    lds_barrier();
    if ((int)threadIdx.x < 2 * CS) {
      float s = 0.f;
#pragma unroll
      for (int q = 0; q < W; ++q)
#pragma unroll
        for (int r = 0; r < RC; ++r)
          s += red[((par * 2 + sh) * W + q) * 64 + (RC * (se >> 4) + r) * 16 + (se & 15)];
      const size_t at = ((size_t)(sh ? b2 : b1) * a.K + k) * a.nchunks + chunk;
      if constexpr (TAU) {
        double t = (double)(s * spc) * (double)dp;
#pragma unroll
        for (int o = 1; o < 16; o <<= 1) t += __shfl_xor(t, o);
        if ((se & 15) == 0) a.gtau[at * C + (se >> 4)] = t;
      } else {
        a.gpart[at * CS + se] = s * spc;
      }
    }
  };

  Entry cur = entry(0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_small(cur, in[0]);
  __builtin_amdgcn_sched_barrier(0);
  fetch_rows(cur);
  __builtin_amdgcn_sched_barrier(0);
  int fb1 = 0, fb2 = 0;
  float fdp = 0.f;
  auto step = [&](int i, auto slot) __attribute__((always_inline)) {
    constexpr int sl = decltype(slot)::value;
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    if (((i + 1) & 3) == 0) {
      pcur = pnext;
      pnext = block(((i + 1) >> 2) + 1);
    }
    const Entry nxt = entry(i + 1);
    fetch_small(nxt, in[1 - sl]);
    const Small& x = in[sl];
    const int m_ = cur.m, push = (m_ >> 6) & 3;
    if ((m_ & 3) == 2) {
#pragma unroll
      for (int c = 0; c < CM; ++c) U[c] = Up[c];
    } else if ((m_ & 3) == 3) {
#pragma unroll
      for (int c = 0; c < CM; ++c) U[c] = held[c];
    }
    // m_h = P_h L_h; L_h's rows go to LDS for the statistic
    f4 m[2][CM];
    each<2>([&](auto hc) {
      constexpr int h = decltype(hc)::value;
      f4(&L)[CM] = Lh(hc);
      const int kd = kind(m_, h);
      if (kd == 0) {
        f4 t;
        if constexpr (TIPS == HX_TIPS_CODES) t = tbl[x.code[h][0]];
        else t = x.t[h];
        mv4<CM>(x.p[h], [&](auto) { return t; }, m[h]);
#pragma unroll
        for (int s = 0; s < 4; ++s) ls[(RW * h + s) * kXS + lane] = t[s];
      } else {
        if constexpr (TIPS == HX_TIPS_CODES) {
          if (kd == 1) {
            // the cherry's partial before the post-order walk's power-of-two rescale: every
            // term below is a ratio in it. Of two such children one is rescaled, since the
            // product of two small ones could underflow.
            const f4 t0 = tbl[x.code[h][0]], t1 = tbl[x.code[h][1]];
            mv4<CM>(x.g[h][0], [&](auto) { return t0; }, L);
            mv4<CM>(x.g[h][1], [&](auto) { return t1; }, m[h]);
#pragma unroll
            for (int c = 0; c < CM; ++c) L[c] *= m[h][c];
            if (h == 0 && kind(m_, 1) == 1) rescale<CM, EXACT>(L, C);
          }
        }
        mv4<CM>(x.p[h], [&](auto c) { return L[c]; }, m[h]);
#pragma unroll
        for (int c = 0; c < CM; ++c)
          if (EXACT || c < C)
#pragma unroll
            for (int s = 0; s < 4; ++s) ls[(RW * h + 4 * c + s) * kXS + lane] = L[c][s];
      }
      __builtin_amdgcn_sched_barrier(0);  // one child's registers at a time
    });
    fetch_rows(nxt);  // the partials are used up: the next entry's
    // Ut, in m's place: m[0] becomes Ut_2, m[1] becomes Ut_1
    float lik = 0.f;
#pragma unroll
    for (int c = 0; c < CM; ++c) {
      if (EXACT || c < C) {
        float t = 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const float m1 = m[0][c][s], u1 = U[c][s] * m[1][c][s];
          m[0][c][s] = U[c][s] * m1;
          m[1][c][s] = u1;
          t = fmaf(u1, m1, t);
        }
        lik = fmaf(pc[c], t, lik);
      }
    }
    auto Ut = [&](auto hc) -> f4(&)[CM] { return m[1 - decltype(hc)::value]; };
    const float coef = (val && lik > 0.f) ? w * __builtin_amdgcn_rcpf(lik) : 0.f;
    // Block b = (16 / CM) c + q of the 4x4x1 product: lane 4b + i gives A[b][i] = (w / lik) Ut[c][i]
    // and lane 4b + j gives B[b][j] = L[c][j] of the block's pattern m in product m; register i of lane
    // 4b + j accumulates G[c][i][j] over those patterns. Child 2's Ut rows overwrite child 1's
    // after child 1's operand reads (LDS operations of a wave stay in order).
    const int g4 = lane >> 4, srow = 4 * (g4 / RC) + (lane & 3);
    const int scol = (CM == 4 ? 16 : 4) * ((lane >> 2) % (16 / CM));
    auto stat_rows = [&](auto hc) {
#pragma unroll
      for (int c = 0; c < CM; ++c)
        if (EXACT || c < C)
#pragma unroll
          for (int s = 0; s < 4; ++s) xs[(4 * c + s) * kXS + lane] = coef * Ut(hc)[c][s];
    };
    auto stat_mfma = [&](int h) {
      __builtin_amdgcn_wave_barrier();
      const int rl = RW * h + (kind(m_, h) == 0 ? (lane & 3) : srow);
      f4 g[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int u = 0; u < CM; ++u) {
        constexpr int US = CM == 4 ? 4 : 64 / CM;
        const f4 A = *reinterpret_cast<const f4*>(xs + srow * kXS + scol + US * u);
        const f4 Bv = *reinterpret_cast<const f4*>(ls + rl * kXS + scol + US * u);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          g[e & 1] = __builtin_amdgcn_mfma_f32_4x4x1f32(A[e], Bv[e], g[e & 1], 0, 0, 0);
      }
      __builtin_amdgcn_wave_barrier();
      return g[0] + g[1];
    };
    // The four blocks of a row of 16 lanes are added by row rotations; lane 16 r + j then holds row
    // r's share of G_h[r / RC][i][j] in register i and writes it to the wave's slot.
    auto stat_put = [&](int h, f4 g) {
#pragma unroll
      for (int r = 0; r < 4; ++r) g[r] = add_row_ror<8>(add_row_ror<4>(g[r]));
      if (((lane >> 2) & 3) == 0 && g4 < C * RC) {
        float* dst = red + (((i & 1) * 2 + h) * W + wave) * 64 + g4 * 16 + (lane & 3);
#pragma unroll
        for (int r = 0; r < 4; ++r) dst[4 * r] = g[r];
      }
    };
    stat_rows(H0{});
    // the barrier in here also keeps this entry's writes behind every read of entry i - 2
    if (i > 0) flush_g(fb1, fb2, fdp, (i - 1) & 1);
    fb1 = cur.c1;
    fb2 = cur.c2;
    if constexpr (TAU) fdp = x.dp;
    stat_put(0, stat_mfma(0));
    stat_rows(H1{});

    __builtin_amdgcn_sched_barrier(0);
    // adjoints of internal children
    if (push) {
      f4 Un[CM];
      mv4<CM>(x.pt[0], [&](auto c) { return Ut(H0{})[c]; }, Un);
      rescale<CM, EXACT>(Un, C);
      if (push == 2) {
#pragma unroll
        for (int c = 0; c < CM; ++c) held[c] = Un[c];
      } else if (tval) {
        const auto r = node_buf(cur.c1, nbytes);
#pragma unroll
        for (int c = 0; c < CM; ++c)
          if (EXACT || c < C) buf_store4(r, loff, c * cbytes, Un[c]);
      }
    }
    if ((m_ >> 8) & 1) {
      mv4<CM>(x.pt[1], [&](auto c) { return Ut(H1{})[c]; }, U);
      rescale<CM, EXACT>(U, C);
    }
    stat_put(1, stat_mfma(1));
    cur = nxt;
  };
  for (int i = 0; i < nprog; ++i) {
    step(i, std::integral_constant<int, 0>{});
    if (++i == nprog) break;
    step(i, std::integral_constant<int, 1>{});
  }
  flush_g(fb1, fb2, fdp, (nprog - 1) & 1);
}

// -------------------------------------------------------------------- launchers
static size_t table_bytes(int tips, int ncodes) {
  return tips == HX_TIPS_CODES ? (size_t)ncodes * 16 : 0;
}

template <int CM, bool EXACT>
static auto post_kernel(int tips, bool store) {
  if (tips == HX_TIPS_CODES)
    return store ? k_post_walk4<HX_TIPS_CODES, CM, EXACT, true>
                 : k_post_walk4<HX_TIPS_CODES, CM, EXACT, false>;
  return store ? k_post_walk4<HX_TIPS_DENSE, CM, EXACT, true>
               : k_post_walk4<HX_TIPS_DENSE, CM, EXACT, false>;
}

int launch_post_walk4(const PassArgs<float>& a, const int32_t* prog, int nprog, int slots, int tips,
                      bool store, hipStream_t st) {
  HX_REQUIRE(a.C >= 1 && a.C <= kPreWalkMaxC, HX_ERR_UNSUPPORTED, "post-order walk: categories");
  HX_REQUIRE((size_t)a.C * a.np * 16 < ((size_t)1 << 31), HX_ERR_UNSUPPORTED,
             "post-order walk: a node's rows of one sample exceed 2 GiB");
  // up to 4 samples share a tile's codes in the vector cache
  const int W = a.K < 4 ? a.K : 4;
  const size_t lds = table_bytes(tips, a.ncodes) + (size_t)W * slots * 256;
  HX_REQUIRE(lds <= 64 * 1024, HX_ERR_UNSUPPORTED, "post-order walk: LDS");
  const auto kern = a.C == 1   ? post_kernel<1, true>(tips, store)
                    : a.C == 2 ? post_kernel<2, true>(tips, store)
                    : a.C == 3 ? post_kernel<4, false>(tips, store)
                               : post_kernel<4, true>(tips, store);
  kern<<<dim3(a.ntiles, (a.K + W - 1) / W), 64 * W, lds, st>>>(a, a.mats, prog, nprog, slots, W);
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

template <int CM, bool EXACT>
static auto pre_kernel(int tips, bool tau) {
  if (tips == HX_TIPS_CODES)
    return tau ? k_pre_walk4<HX_TIPS_CODES, CM, EXACT, true>
               : k_pre_walk4<HX_TIPS_CODES, CM, EXACT, false>;
  return tau ? k_pre_walk4<HX_TIPS_DENSE, CM, EXACT, true>
             : k_pre_walk4<HX_TIPS_DENSE, CM, EXACT, false>;
}

int launch_pre_walk4(const PassArgs<float>& a, const int32_t* prog, int nprog, int tips,
                     hipStream_t st) {
  HX_REQUIRE(a.C >= 1 && a.C <= kPreWalkMaxC && a.nchunks == (a.ntiles + kPreWalkW - 1) / kPreWalkW,
             HX_ERR_UNSUPPORTED, "pre-order walk: chunking does not match the workgroup's tiles");
  const bool tau = a.mats_dt != nullptr;
  const size_t lds = pre4_lds_floats(a.C <= 2 ? a.C : 4) * 4 + table_bytes(tips, a.ncodes);
  HX_REQUIRE(lds <= 64 * 1024, HX_ERR_UNSUPPORTED, "pre-order walk: LDS");
  const auto kern = a.C == 1   ? pre_kernel<1, true>(tips, tau)
                    : a.C == 2 ? pre_kernel<2, true>(tips, tau)
                    : a.C == 3 ? pre_kernel<4, false>(tips, tau)
                               : pre_kernel<4, true>(tips, tau);
  kern<<<dim3(a.nchunks, a.K), 64 * kPreWalkW, lds, st>>>(a, a.mats, a.mats_dt, prog, nprog);
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

}  // namespace hx
