// Dense-state FP32 post-order (S != 4, at most 32 states and 4 categories) as one walk: a launch for
// the whole tree, for the calls that use_dwalk (layout.hpp) gives it: with few patterns on a large
// tree the level kernels are ahead. The partials and root sums are theirs to the bit.
//
// Reference: calculate_treelikelihood_discrete* (torchtree/evolution/tree_likelihood.py:40-278)
// at S != 4.
//
// A block walks the tree for one tile of 16 patterns of one sample, one wave per category with
// both children of a node: their products meet in registers, and only the rescaling maximum
// crosses waves, with one barrier per node. With lane = nn + 16 g and v_mfma_f32_16x16x4f32
// (A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k, D[i][j] in register i % 4 of lane
// j + 16 (i / 4)) the product is
//   Y[m][i] = sum_j L[m][j] P[i][j]   A = L, patterns x states; step q of lane group g is state g KV + q
// which leaves pattern 4 g + r, state 16 t + nn in register r of output tile t ("acc layout"); the
// next node's A operand is read back from the wave's own LDS tile.
//
// What bounds it: the chain of one node (matrix products 640 cycles at 20 states, then the maximum
// over lanes and waves, the barrier, the scaling and the LDS transpose), hidden behind the other
// blocks of the CU. A launch per tree level makes each level wait for its slowest block, reads every
// child back from memory and leaves the chip nearly empty at the narrow levels (about 30 us each).
// Measured against it, 20 states, 4 categories, FP32: 256 taxa x 20000 patterns 1815 -> 1005 us,
// 173 taxa x 3203 patterns at 8 samples 1495 -> 900 us; with split-BF16 products at the first size
// 1747 -> 1000 us (each operand is split when it is used). Past 32 states the operands of two children's matrices no longer fit a
// wave's registers (61 states: 64 x 2, fetched a node ahead).
#include "pruning.hpp"
#include "split.hpp"
#include "walk.hpp"

#include <math.h>

#include <type_traits>
#include <utility>

namespace hx {

namespace {

using f4 = float __attribute__((ext_vector_type(4)));
constexpr int kTile = 16;
constexpr unsigned kNowhere = 0x7fffff00u;  // lane offset past every buffer: loads 0, stores nothing

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float buf_load(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                          unsigned off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)lane_off, (int)off, 0));
}
__device__ __forceinline__ f4 buf_load4(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                        unsigned off) {
  return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane_off, (int)off, 0));
}
__device__ __forceinline__ void buf_store(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                          unsigned off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)lane_off, (int)off, 0);
}

// KV consecutive floats: one by one where a run may cross the buffer's end (each is then checked
// against it by itself), otherwise (FULL) 16 bytes at a time.
template <int KV, bool FULL>
__device__ __forceinline__ void load_run(const __amdgpu_buffer_rsrc_t& r, unsigned lane_off,
                                         unsigned off, float (&x)[KV]) {
  constexpr int V = FULL ? KV / 4 * 4 : 0;
#pragma unroll
  for (int q = 0; q < V; q += 4) {
    const f4 v = buf_load4(r, lane_off + 4 * q, off);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[q + e] = v[e];
  }
#pragma unroll
  for (int q = V; q < KV; ++q) x[q] = buf_load(r, lane_off + 4 * q, off);
}

// Reductions over the 16 lanes of a group by DPP row permutes. The maximum is taken on the bit
// patterns as signed integers (the inputs are maxima started at +0).
template <int CTRL>
__device__ __forceinline__ int dpp_i(int x) {
  return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
  return __builtin_bit_cast(float, dpp_i<CTRL>(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float max16(float v) {
  int x = __builtin_bit_cast(int, v);
  x = max(x, dpp_i<0xB1>(x));
  x = max(x, dpp_i<0x4E>(x));
  x = max(x, dpp_i<0x141>(x));
  x = max(x, dpp_i<0x140>(x));
  return __builtin_bit_cast(float, x);
}
__device__ __forceinline__ float sum16(float v) {
  v += dpp_f<0xB1>(v);
  v += dpp_f<0x4E>(v);
  v += dpp_f<0x141>(v);
  return v + dpp_f<0x140>(v);
}

// Exponent that brings the largest of a row's category maxima into [0.5, 1); 0 for none or
// non-finite ones.
__device__ __forceinline__ int row_exp(const f4& mv) {
  const float M = fmaxf(fmaxf(mv[0], mv[1]), fmaxf(mv[2], mv[3]));
  const int e = __builtin_amdgcn_frexp_expf(M);
  return M > 0.f ? e : 0;
}

// acc = A B over KV steps, on the FP32 matrix cores or as split products with the packs of the
// level kernels (FwdP)
template <int MT, int KV, bool SPLIT>
__device__ __forceinline__ void product(const float (&a)[KV], const float (&b)[MT][KV], f4 (&acc)[MT]) {
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f4{0.f, 0.f, 0.f, 0.f};
  if constexpr (SPLIT) {
    constexpr int KB = SplitShape<KV>::KB;
    static_assert(SplitShape<KV>::NB == 1, "one pack per lane");
    BfPack<KB> ap;
#pragma unroll
    for (int q = 0; q < KB; ++q) pack_set(ap, q, q < KV ? a[q < KV ? q : 0] : 0.f);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      BfPack<KB> bp;
#pragma unroll
      for (int q = 0; q < KB; ++q) pack_set(bp, q, q < KV ? b[t][q < KV ? q : 0] : 0.f);
      acc[t] = mma3(ap, bp, acc[t]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < KV; ++q)
#pragma unroll
      for (int t = 0; t < MT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], b[t][q], acc[t], 0, 0, 0);
  }
}

// The lane's offsets and the operand loads of one (tile, sample, category).
// FULL: S = 4 KV, every lane's run of states exists.
template <int MT, int KV, int TIPS, bool FULL>
struct Dense {
  static constexpr int LS = 16 * MT + 4;  // row stride of LDS tiles: rows 4 g + r on separate banks
  const PassArgs<float>& a;
  const int S, C, c, k, tile, lane, nn, g;
  const int CS, rows;       // floats per pattern; the tile's patterns
  const unsigned nrow;      // the lane's A row, clamped to the tile's last pattern
  unsigned pf[MT];          // lane offsets of its run of P rows
  unsigned lrow, acc_off[4], tile_bytes;
  float* tile0;       // the tile's rows of slot 0
  size_t slot_bytes;  // between slots
  bool last_ok, jok[KV];    // its state of the last output tile, its A states exist

  __device__ __forceinline__ Dense(const PassArgs<float>& a_, int S_, int c_, int k_, int tile_)
      : a(a_), S(S_), C(a_.C), c(c_), k(k_), tile(tile_), lane(threadIdx.x & 63),
        nn(threadIdx.x & 15), g((threadIdx.x & 63) >> 4), CS(a_.C * S_),
        rows(min(kTile, a_.N - tile_ * kTile)), nrow(min(nn, rows - 1)) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
      pf[t] = 16 * t + nn < S ? 4u * (unsigned)((16 * t + nn) * S + g * KV) : kNowhere;
    last_ok = 16 * (MT - 1) + nn < S;
    tile0 = a.partials + ((size_t)k * a.N + (size_t)tile * kTile) * CS;
    slot_bytes = (size_t)a.K * a.N * CS * 4;
    tile_bytes = (unsigned)(rows * CS * 4);
#pragma unroll
    for (int q = 0; q < KV; ++q) jok[q] = g * KV + q < S;
    lrow = 4u * (unsigned)(nrow * CS + c * S + g * KV);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      acc_off[r] = 4 * g + r < rows ? 4u * (unsigned)((4 * g + r) * CS + c * S + nn) : kNowhere;
  }
  // one category's matrix of a branch; a run past its end reads 0 and not the next matrix
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t mat(const float* m, int b) const {
    return buf(m + (((size_t)k * a.B + b) * C + c) * S * S, (size_t)S * S * 4);
  }
  __device__ __forceinline__ void load_p(const float* m, int b, float (&p)[MT][KV]) const {
    const auto r = mat(m, b);
#pragma unroll
    for (int t = 0; t < MT; ++t) load_run<KV, FULL>(r, pf[t], 0, p[t]);
  }
  // a node's rows of this tile, of all categories (any = false: an empty range)
  __device__ __forceinline__ float* slab(int v) const {
    return a.partials + (((size_t)(v - a.T) * a.K + k) * a.N + (size_t)tile * kTile) * CS;
  }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t node(int v, bool any) const {
    const unsigned i = any ? (unsigned)(v - a.T) : 0u;
    return buf(reinterpret_cast<char*>(tile0) + i * slot_bytes, any ? tile_bytes : 0u);
  }
  __device__ __forceinline__ int code(int t) const {
    return __builtin_amdgcn_raw_buffer_load_b8(buf(a.codes + (size_t)t * a.N + tile * kTile, rows),
                                               (int)nrow, 0, 0);
  }
  __device__ __forceinline__ void dense_row(int t, float (&x)[KV]) const {
    load_run<KV, FULL>(buf(a.dense + ((size_t)t * a.N + (size_t)tile * kTile) * S, (size_t)rows * S * 4),
                       4u * (unsigned)(nrow * S + g * KV), 0, x);
  }
  __device__ __forceinline__ void mask(float (&x)[KV]) const {
    if constexpr (FULL) return;
#pragma unroll
    for (int q = 0; q < KV; ++q) x[q] = jok[q] ? x[q] : 0.f;
  }
  __device__ __forceinline__ void store_acc(const __amdgpu_buffer_rsrc_t& r, const f4 (&x)[MT]) const {
#pragma unroll
    for (int t = 0; t < MT - 1; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q) buf_store(r, acc_off[q], 64 * t, x[t][q]);
    if (last_ok) {
#pragma unroll
      for (int q = 0; q < 4; ++q) buf_store(r, acc_off[q], 64 * (MT - 1), x[MT - 1][q]);
    }
  }
  // acc layout to the wave's LDS tile, and a row of it as an A operand
  __device__ __forceinline__ void put(float* lt, const f4 (&x)[MT]) const {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) lt[(4 * g + r) * LS + 16 * t + nn] = x[t][r];
  }
  __device__ __forceinline__ void get(const float* lt, float (&x)[KV]) const {
#pragma unroll
    for (int q = 0; q < KV; ++q) x[q] = lt[nn * LS + g * KV + q];
  }
};

}  // namespace

// LDS: per wave two tiles (the previous and a held result) and its exponent stack, per block the
// row maxima of two nodes and the tip table.
template <int MT>
static size_t post_dwalk_lds(int C, int S, int slots, int ncodes) {
  return (size_t)C * 2 * kTile * (16 * MT + 4) * 4 + 2 * kTile * 4 * 4 +
         ((size_t)ncodes * S + 64) * 4 + (size_t)C * slots * kTile * 4 + 16;
}

// ------------------------------------------------------------------ post-order
// prog: walk.hpp, build_post4, without its drop bits (every partial is stored when a gradient may
// follow). grid = ntiles * K, sample fastest, so that the blocks of one sample tend to share an
// XCD's L2, where its P matrices are read; block = 64 C. At 3 waves per SIMD nothing spills (107
// registers at 20 states); forced to 5 or 6 they do (256 taxa: +0 % and +55 % time).
template <int MT, int KV, int TIPS, bool FULL, bool STORE, bool SPLIT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void k_post_dwalk(
    PassArgs<float> a, const int* __restrict__ prog, int nprog, int slots, int S) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  using D = Dense<MT, KV, TIPS, FULL>;
  const int C = a.C, wave = uni(threadIdx.x >> 6);
  const int k = uni(blockIdx.x % a.K), tile = uni(blockIdx.x / a.K);
  const D d(a, S, wave, k, tile);
  const int lane = d.lane, nn = d.nn, g = d.g;
  float* tiles = reinterpret_cast<float*>(smem_raw) + (size_t)wave * 2 * kTile * D::LS;
  float* mx = reinterpret_cast<float*>(smem_raw) + (size_t)C * 2 * kTile * D::LS;  // [2][16][4]
  float* tbl = mx + 2 * kTile * 4;
  const int ntbl = TIPS == HX_TIPS_CODES ? a.ncodes * S : 0;
  int* est = reinterpret_cast<int*>(tbl + ntbl + 64) + (size_t)wave * slots * kTile;
  // categories C .. 3 of mx stay zero; states past a table row are masked, those past the table 0
  for (int q = threadIdx.x; q < 2 * kTile * 4; q += blockDim.x) mx[q] = 0.f;
  for (int q = threadIdx.x; q < ntbl + 64; q += blockDim.x) tbl[q] = q < ntbl ? a.table[q] : 0.f;
  __syncthreads();

  // program blocks: lane 4 j + q holds word q of entry 16 blk + j (past the end: the last entry)
  auto block = [&](int blk) {
    return prog[min(16 * blk + (lane >> 2), nprog - 1) * kPost4Ints + (lane & 3)];
  };
  int pcur = block(0), pnext = block(1);
  struct Entry {
    int c1, c2, v, m;
  };
  auto entry = [&](int i) {
    const int l = (i & 15) * kPost4Ints;
    return Entry{__builtin_amdgcn_readlane(pcur, l), __builtin_amdgcn_readlane(pcur, l + 1),
                 __builtin_amdgcn_readlane(pcur, l + 2), __builtin_amdgcn_readlane(pcur, l + 3)};
  };
  // the next entry's operands; loads are issued on every path (an empty range reads nothing)
  struct In {
    float p1[MT][KV], p2[MT][KV], x1[KV], x2[KV];  // x1: a spilled child or a dense tip
    int code1, code2;
  };
  In in[2];
  auto fetch = [&](const Entry& e, In& x) {
    const int ty = e.m & 3;
    d.load_p(a.mats, e.c1, x.p1);
    d.load_p(a.mats, e.c2, x.p2);
    const int t1 = ty <= 1 ? e.c1 : 0, t2 = ty == 0 ? e.c2 : 0;
    if constexpr (TIPS == HX_TIPS_CODES) {
      x.code1 = d.code(t1);
      x.code2 = d.code(t2);
      load_run<KV, FULL>(d.node(e.c1, ty == 3), d.lrow, 0, x.x1);
    } else {
      // the spilled rows or the tip's, by the descriptor
      const float* src = ty == 3 ? d.slab(e.c1) : a.dense + ((size_t)t1 * a.N + (size_t)tile * kTile) * S;
      const unsigned bytes = (unsigned)(d.rows * (ty == 3 ? d.CS : S) * 4);
      load_run<KV, FULL>(buf(src, bytes), ty == 3 ? d.lrow : 4u * (unsigned)(d.nrow * S + g * KV), 0,
                         x.x1);
      d.dense_row(t2, x.x2);
    }
  };

  f4 y[MT];
  int E[4] = {0, 0, 0, 0}, Eh[4] = {0, 0, 0, 0};
  int ci = 0;  // the tile that holds the previous result
  Entry cur = entry(0);
  fetch(cur, in[0]);
  auto step = [&](int i, auto slot) __attribute__((always_inline)) {
    constexpr int sl = decltype(slot)::value;
    if (((i + 1) & 15) == 0) pcur = pnext;
    pnext = block(((i + 1) >> 4) + 1);  // every time: a conditional load would be waited for at once
    const Entry nxt = entry(i + 1);
    fetch(nxt, in[1 - sl]);
    In& x = in[sl];
    const int type = cur.m & 3;
    if ((cur.m >> 2) & 1) {  // the previous result waits, later ones go to the other tile (type 0)
      ci ^= 1;
#pragma unroll
      for (int r = 0; r < 4; ++r) Eh[r] = E[r];
    }
    float* own = tiles + ci * kTile * D::LS;
    float a1[KV], a2[KV];
    if (type == 0) {
      if constexpr (TIPS == HX_TIPS_CODES) {
#pragma unroll
        for (int q = 0; q < KV; ++q) a2[q] = tbl[x.code2 * S + g * KV + q];
      } else {
#pragma unroll
        for (int q = 0; q < KV; ++q) a2[q] = x.x2[q];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) E[r] = 0;
    } else {
      d.get(own, a2);
    }
    if (type == 2) {
      d.get(tiles + (ci ^ 1) * kTile * D::LS, a1);
#pragma unroll
      for (int r = 0; r < 4; ++r) E[r] += Eh[r];
    } else if (TIPS == HX_TIPS_CODES && type <= 1) {
#pragma unroll
      for (int q = 0; q < KV; ++q) a1[q] = tbl[x.code1 * S + g * KV + q];
    } else {
#pragma unroll
      for (int q = 0; q < KV; ++q) a1[q] = x.x1[q];
    }
    if (type == 3) {
#pragma unroll
      for (int r = 0; r < 4; ++r) E[r] += est[((cur.m >> 8) & 0xff) * kTile + 4 * g + r];
    }
    d.mask(a1);
    d.mask(a2);
    f4 y2[MT];
    product<MT, KV, SPLIT>(a1, x.p1, y);
    product<MT, KV, SPLIT>(a2, x.p2, y2);
    float* m = mx + (i & 1) * kTile * 4;
#pragma unroll
    for (int t = 0; t < MT; ++t) y[t] *= y2[t];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = 0.f;
#pragma unroll
      for (int t = 0; t < MT; ++t) v = fmaxf(v, y[t][r]);
      v = max16(v);
      if (nn == 0) m[(4 * g + r) * 4 + wave] = v;
    }
    // one barrier: the next node writes the other half of mx, and every wave has read this half
    // before it passes the next node's barrier
    lds_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int e = row_exp(*reinterpret_cast<const f4*>(m + (4 * g + r) * 4));
#pragma unroll
      for (int t = 0; t < MT; ++t) y[t][r] = ldexpf(y[t][r], -e);
      E[r] += e;
    }
    d.put(own, y);
    const bool spill = (cur.m >> 4) & 1;
    if (spill && nn == 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) est[((cur.m >> 16) & 0xff) * kTile + 4 * g + r] = E[r];
    }
    if ((STORE && i + 1 < nprog) || spill) d.store_acc(d.node(cur.v, true), y);
    cur = nxt;
  };
  for (int i = 0; i < nprog; ++i) {
    step(i, std::integral_constant<int, 0>{});
    if (++i == nprog) break;
    step(i, std::integral_constant<int, 1>{});
  }

  // root: site likelihood sum_c p_c pi.y_c (tree_likelihood.py:71-74, 215-220)
  __syncthreads();
  const float pc = a.props[(size_t)k * a.props_ks + wave];
  float* pxs = mx;                                            // [16][4]
  double* red = reinterpret_cast<double*>(smem_raw);          // [C][16 MT] d/dfreqs shares (the tiles' room)
  float px[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    float v = 0.f;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int i = 16 * t + nn;
      v = fmaf(i < S ? a.freqs[(size_t)k * a.freqs_ks + i] : 0.f, y[t][r], v);
    }
    px[r] = sum16(v);
    if (nn == 0) pxs[(4 * g + r) * 4 + wave] = px[r];
  }
  __syncthreads();
  double acc_l = 0.0, acc_p = 0.0, acc_f[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc_f[t] = 0.0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = tile * kTile + 4 * g + r;
    if (4 * g + r >= d.rows) continue;
    double lik = 0.0;
    for (int cc = 0; cc < C; ++cc)
      lik += (double)(a.props[(size_t)k * a.props_ks + cc] * pxs[(4 * g + r) * 4 + cc]);
    const double w = a.weights[n], wi = w / lik;
    acc_l += w * (log(lik) + (double)E[r] * kLn2);
#pragma unroll
    for (int t = 0; t < MT; ++t) acc_f[t] += wi * (double)(pc * y[t][r]);
    acc_p += wi * (double)px[r];
  }
  // the lanes nn of a group g hold the same loglik and d/dprops terms
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) {
    acc_l += __shfl_xor(acc_l, o);
    acc_p += __shfl_xor(acc_p, o);
#pragma unroll
    for (int t = 0; t < MT; ++t) acc_f[t] += __shfl_xor(acc_f[t], o);
  }
  if (g == 0) {
#pragma unroll
    for (int t = 0; t < MT; ++t) red[wave * 16 * MT + 16 * t + nn] = acc_f[t];
  }
  __syncthreads();
  double* out = a.rootsums + ((size_t)k * a.ntiles + tile) * (1 + S + C);
  if (lane == 0) out[1 + S + wave] = acc_p;
  if (wave == 0) {
    if (lane == 0) out[0] = acc_l;
    if (lane < S) {
      double s = 0.0;
      for (int cc = 0; cc < C; ++cc) s += red[cc * 16 * MT + lane];
      out[1 + lane] = s;
    }
  }
}

// -------------------------------------------------------------------- launchers
int launch_post_dwalk(const PassArgs<float>& a, const int32_t* prog, int nprog, int slots, int tips,
                      int S, bool store, hipStream_t st) {
  HX_REQUIRE(S >= 2 && S <= 32 && a.C >= 1 && a.C <= 4, HX_ERR_UNSUPPORTED, "dense walk: shape");
  HX_REQUIRE((size_t)(a.N + 16) * a.C * S + 64 < ((size_t)1 << 31) &&
                 (size_t)a.ntiles * a.K < ((size_t)1 << 31),
             HX_ERR_UNSUPPORTED, "dense-state slab exceeds 31-bit offsets");
  // (the level kernels' limit: what they refuse stays refused)
  HX_REQUIRE((size_t)a.C * kTile * (S <= 16 ? 20 : 36) * 4 + 8 * kTile * 4 +
                     2 * (size_t)a.tiles_per_chunk * kTile + 64 <= 64 * 1024,
             HX_ERR_UNSUPPORTED, "dense-state post-order LDS exceeds 64 KiB");
  const int ncodes = tips == HX_TIPS_CODES ? a.ncodes : 0;
  const unsigned grid = (unsigned)a.ntiles * (unsigned)a.K;
#define HX_DW_K(MTV, KVV, FULLV, SPLITV)                                                     \
  (tips == HX_TIPS_CODES ? (store ? k_post_dwalk<MTV, KVV, HX_TIPS_CODES, FULLV, true, SPLITV>    \
                                  : k_post_dwalk<MTV, KVV, HX_TIPS_CODES, FULLV, false, SPLITV>)  \
                         : (store ? k_post_dwalk<MTV, KVV, HX_TIPS_DENSE, FULLV, true, SPLITV>    \
                                  : k_post_dwalk<MTV, KVV, HX_TIPS_DENSE, FULLV, false, SPLITV>))
#define HX_DW(MTV, KVV, FULLV)                                                               \
  do {                                                                                       \
    const size_t lds = post_dwalk_lds<MTV>(a.C, S, slots, ncodes);                           \
    auto kern = a.split ? HX_DW_K(MTV, KVV, FULLV, true) : HX_DW_K(MTV, KVV, FULLV, false);  \
    if (lds > 64 * 1024)                                                                     \
      HX_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),                    \
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)); \
    kern<<<grid, 64 * a.C, lds, st>>>(a, prog, nprog, slots, S);                             \
  } while (0)
  if (S <= 16) HX_DW(1, 4, false);
  else if (S == 20) HX_DW(2, 5, true);
  else if (S < 20) HX_DW(2, 5, false);
  else HX_DW(2, 8, false);
#undef HX_DW
#undef HX_DW_K
  HX_HIP_TRY(hipGetLastError());
  return HX_OK;
}

}  // namespace hx
