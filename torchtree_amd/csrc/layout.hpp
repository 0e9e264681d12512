// Host-side shape arithmetic of the library, free of HIP: the pattern tiling of a call, the
// kernel choices that change a workspace's layout, and the workspace layouts of hx_loglik*
// and of a resident job's evaluation. The HIP sources use it through common.hpp; the
// host-only test drivers build it with g++ under AddressSanitizer and UBSan.
#pragma once

#include <math.h>
#include <stddef.h>
#include <stdint.h>

#include "hiptree.h"

namespace hx {

constexpr int kBlock = 256;      // threads per block for the pruning kernels
constexpr int kWave = 64;        // CDNA wavefront
constexpr int kMaxCodes = 256;   // tip table rows held in LDS

inline int next_pow2(int x) {
  int p = 1;
  while (p < x) p <<= 1;
  return p;
}

inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// The precisions a call may ask for (HX_F32_BF16X3 stores FP32, as HX_F32 does).
inline bool dtype_ok(int dtype) {
  return dtype == HX_F32 || dtype == HX_F64 || dtype == HX_F32_BF16X3;
}

// Pattern tiling shared by every pass of one call: each block owns a chunk of
// consecutive pattern tiles for one (sample, node).
struct Tiling {
  int cp;               // lanes per pattern (C rounded up to a power of two)
  int ppb;              // patterns per tile (= kBlock / cp)
  int ntiles;
  int nchunks;
  int tiles_per_chunk;
};

// Dense states run on the matrix cores (pruning_mfma.hip) at up to 4 categories, in FP32
// (with or without split BF16 products) and FP64; otherwise on the wide kernels
// (pruning_wide.hip).
inline bool use_mfma(int C, int S, int dtype) {
  return (dtype == HX_F32 || dtype == HX_F64 || dtype == HX_F32_BF16X3) && S != 4 && C >= 1 &&
         C <= 4;
}

// LDS of one wide-kernel block, and its patterns per tile.
constexpr int kWideLdsBytes = 60 * 1024;
inline int wide_nt(int C, int S, int rb) {
  if (use_mfma(C, S, rb == 8 ? HX_F64 : HX_F32)) return 16;  // MFMA tiles of 16 patterns
  const int SP = S <= 32 ? 32 : 64;
  const int G = C * SP;
  int nt = kWideLdsBytes / (7 * G * rb);
  if (nt > 8) nt = 8;
  if (nt < 1) nt = 1;
  return nt;
}

// S == 4 uses tiles of 64 patterns (a wave per category, a lane per pattern);
// other S use tiles of wide_nt() patterns handled by (child, category, state)
// lanes.
// The chunking depends on N, S, C, the precision and the tile shape only, never on K: a sample's
// sums run in the same order whatever batch it is evaluated in, so its result is bitwise
// identical alone and in a batch. (K enters post_level_tiles and use_dwalk, which no result
// depends on.)
constexpr int kTargetChunks = 128;

// The four-state FP32 passes with at most kPreWalkMaxC categories are walks
// (pruning_walk.hip) at every size: choosing by size would make a sample's
// FP32 gradient depend on the batch it is evaluated in. The pre-order walk
// sums its branch statistics over the kPreWalkW tiles of a workgroup: one
// chunk per kPreWalkW tiles.
constexpr int kPreWalkW = 4;
constexpr int kPreWalkMaxC = 4;
inline bool use_pre_walk(int S, int C, int rb, int N, int K) {
  (void)N;
  (void)K;
  return S == 4 && rb == 4 && C <= kPreWalkMaxC;
}

inline Tiling make_tiling(int N, int C, int K, int S, int rb) {
  Tiling t;
  t.cp = next_pow2(C < 1 ? 1 : C);
  int min_tiles = 1;
  if (S == 4) {
    t.ppb = kWave;  // one wave per category, one lane per pattern
  } else {
    t.ppb = wide_nt(C, S, rb);
    // FP32 at 17..64 states: chunks of at least 8 tiles, since each chunk's d/dP partials
    // (C S^2 floats per branch) and its P set-up weigh as much as several tiles of partials
    // (128 taxa, 10k patterns, 61 states: at K = 32 the step 144 -> 128 ms, at K = 1 the
    // pre-order +2 %; the 200-request serving mix, whose smaller amino-acid slices get larger
    // chunks: +14 % served throughput)
    min_tiles = (S > 16 && rb == 4) ? 8 : 4;
  }
  t.ntiles = (N + t.ppb - 1) / t.ppb;
  if (use_pre_walk(S, C, rb, N, K)) {
    t.tiles_per_chunk = kPreWalkW;
    t.nchunks = (t.ntiles + kPreWalkW - 1) / kPreWalkW;
    return t;
  }
  int cap = t.ntiles / min_tiles;
  if (cap < 1) cap = 1;
  const int nch = cap < kTargetChunks ? cap : kTargetChunks;
  t.tiles_per_chunk = (t.ntiles + nch - 1) / nch;
  t.nchunks = (t.ntiles + t.tiles_per_chunk - 1) / t.tiles_per_chunk;
  return t;
}

// Tiles per block of a dense post-order level: nothing is summed over them, so it is chosen for the
// launch, and a result does not depend on it.
//
// At 33 states and more a block fills a CU. It costs its tiles and about `setup` more (P, which FP64
// loads in the lane order of its operand), and blocks beyond a round of the chip wait for the next:
// in the chunks of the gradient (8 tiles and more) the narrow levels near the root had 9 to 70 blocks
// a sample, and others a nearly empty last round (61 states, 128 taxa x 10000 patterns, split
// products: 1104 -> 968 us; FP32, 97 x 1217 at 8 samples: 1201 -> 984). `waves` is how many of the
// kernel a SIMD holds: 2, or 3 with FP32 products and coded tips, and with 1 or 2 categories more
// blocks of 2 C waves share a CU. (With 3 categories a third per SIMD gained nothing: blocks of 6
// waves.) At one category rounds are long and blocks leave them one by one, and past 10 tiles a longer
// chunk only coarsens the end: 33 to 61 states, 50 taxa x 20000 patterns at 8 samples, in percent
// behind the best of 2 to 48 tiles: FP32 9 to 11 (2 categories 6 to 11), FP64 6 to 7, split 5, with
// rounds of 1024 blocks and up to 64 tiles; 0 to 2 now.
//
// Below, blocks share a CU and hide each other's latency, and rounds of one block per CU leave it
// idle. There a level takes about (blocks / 256 + tail) (t + set-up), least at t ~ sqrt(tiles C) with
// a factor that grows with the set-up. Against every t of 1 to 16 on all levels, at 2, 8, 20 and 27
// states, 50 taxa x 100 patterns to 128 x 100000, 1 to 16 samples, this is 10 % behind the best of
// them at most and mostly ahead; rounds of one block per CU were 0 to 73 % behind. FP64, 2 states, 4
// categories, 50 taxa x 3000 patterns at 8 samples: 570 us in such rounds, 348 in the gradient's
// chunks, 333 now; 20 states, 128 x 20000: 1773 in such rounds, 1556 now.
//
// FP64 past 16 states holds 5 or 4 waves on a SIMD, so that a level of a few thousand blocks takes a few
// rounds of the chip, and a nearly empty last one shows: with up to four, t is the one with the least
// rounds (t + 1). 25 to 60 taxa, caterpillars, 4000 to 20000 patterns, 4 and 8 samples, 20 to 32 states, 2 to 4
// categories: 0.73 to 0.87 of the time without.
inline int post_level_tiles(int ntiles, int S, int C, int K, int width, bool f64, int waves = 2) {
  if (S <= 32) {
    const double q = S <= 16 ? 4096.0 : (S <= 20 ? 2048.0 : 1024.0);
    double t = sqrt((double)ntiles * K * width * C / q);
    if (f64 && S > 16 && C > 1) {
      const int simd = S <= 20 ? 5 : 4;  // waves of the kernel on a SIMD
      const double slots = 256.0 * (C == 2 ? simd : simd / 2);
      auto blocks = [&](double u) { return ceil(ntiles / u) * K * width; };
      auto cost = [&](double u) { return ceil(blocks(u) / slots) * (u + 1.0); };
      if (t < 1.0) t = 1.0;
      if (blocks(t) <= 4.0 * slots)
        for (int u = 1; u <= ntiles && u <= 64; ++u)
          if (cost(u) < cost(t)) t = u;
    }
    const int nch = (int)(ntiles / (t < 1.0 ? 1.0 : t) + 0.5), least = (ntiles + 63) / 64;
    return (ntiles + (nch > least ? nch : least) - 1) / (nch > least ? nch : least);  // even chunks
  }
  const double setup = f64 ? 4.0 : 1.0, slots = 256.0 * (C <= 2 ? 2 * waves / C : 1);
  int best = 1;
  double cost = 0.0;
  for (int t = 1; t <= ntiles && t <= (C == 1 ? 10 : 64); ++t) {
    const double blocks = (double)((ntiles + t - 1) / t) * K * width;
    const double c = ceil(blocks / slots) * (t + setup);
    if (t == 1 || c <= cost) best = t, cost = c;
  }
  return best;
}

// Whether the FP32 level kernels move rows with lanes along the states (NatRows) or load them as
// operands, a lane per pattern. Below 16 states, and up to 20 with few categories, rows are short:
// most lanes of a row load idle, and an operand load takes few lines. Operands against rows, the
// post- and the pre-order of 50 to 350 taxa x 60 to 20000 patterns: 2 and 8 states 0.80 to 1.02 and
// 0.84 to 1.05 (split products to 1.15, at 3000 patterns x 8 samples), 18 and 20 states with 1 to 3
// categories 0.80 to 1.21 and 0.87 to 1.05 (the larger ones at sizes that walk), with 4 0.99 to 1.29
// and 1.02 to 1.12; 16 states with several categories (50 to 200 taxa x 400 to 20000 patterns) 1.08 to
// 1.52 and, whole gradients, 1.00 to 1.49, but 13 to 15 states, whose rows straddle lines, 0.91 to 1.06
// and 0.90 to 1.13, the latter with dense tips and split products alone; 27 states 0.88 to 1.10 and 0.95
// to 1.11, 32 0.96 to 1.66 and 0.98 to 1.40.
//
// Split products of 17 and 19 states gain nothing by rows either (4 categories 1.03 to 1.19), and up to
// 20 states the post-order of a single tile takes operands: its P is used once, and comes faster so
// (1.04 to 1.33 with rows). With coded tips, whose rows come from the table's few lines either way, the
// post-order of 21 to 31 states does too at one tile (0.97 to 1.18 with rows) and with FP32 products at 3
// categories, whose blocks of 6 waves leave the rows' latency bare (1.00 to 1.16).
inline bool use_nat_rows(int S, int C, bool split, bool post, int ntiles, bool dense) {
  if (S > 20) return !(post && !dense && S < 32 && (ntiles == 1 || (C == 3 && !split)));
  if (post && ntiles == 1) return false;
  return S > 16 ? C >= 4 && !(split && S % 2) : S == 16 && C >= 2;
}

// Whether a dense FP32 or split-BF16 post-order runs as one walk of the tree (pruning_dwalk.hip) or
// by level (k_post_mfma_r). Both leave the same partials and root sums to the bit, so the choice may
// depend on the batch. Times in us, B blocks = tiles x samples, I internal nodes:
//   walk   8 + I (a + b C max(0, B - 256)): a node's chain a, whatever there is in flight up to a
//          block per CU, then the blocks' work. The states decide how P comes (pruning_dwalk.hip):
//          20 in 16-byte loads, the other sizes word by word, and rows of a multiple of 8 states
//          (past 20; of 16 with several categories) fall on the same banks. So do the rows of dense
//          tips, which come word by word at every size but 20 and weigh on the chain past 8 states.
//   levels (launch) x levels + I B C v.
// Measured at 2 to 32 states, 1 to 4 categories, coded and dense tips, 4 to 500 taxa (caterpillars to
// balanced trees), 1 to 100000 patterns and 1 to 32 samples, 7820 calls: the slower one costs more than
// 10 % in 91 of them and 20 % in 28, at most 51 % (4 taxa, where the root is a third of a call); with the walk everywhere 350 taxa x 60 patterns, 27
// states, 4 categories took 1068 us (levels 112), 128 x 400 at 20 states 163 (60); with coded tips'
// constants for dense ones 200 x 10000 at 16 samples, 18 states, 2 categories 5674 (3961).
constexpr int kDwalkMaxS = 32;
inline bool use_dwalk(int S, int C, int I, int levels, int ntiles, int K, bool dense = false,
                      bool split = false) {
  if (S > kDwalkMaxS) return false;
  const double blocks = (double)ntiles * K, past = blocks > 256 ? blocks - 256 : 0;
  const bool eights = S % 8 == 0;
  double a, b, launch, v;  // b and v in 1e-4 us
  if (S <= 16) {
    a = 0.73 + 0.08 * C, launch = 4.0 + 0.08 * C;
    b = S == 16 && C > 1 ? 10 : 5, v = 6.5;
    if (dense) {
      if (C > 2 && S >= 8) a += (S == 16 ? 0.3 : 0.1) * (C - 2);
      b = S == 16 ? 17.5 : (S == 8 ? 12.5 : (S > 8 ? 8.5 : 5.5));
      if (S >= 8) v = 8.8;
    }
  } else if (S == 20) {
    a = 0.84 + 0.1 * C, launch = 3.95 + 0.37 * C;
    b = 6, v = C < 4 ? 14 : 11.5;
  } else if (S < 20) {
    a = 0.8 + 0.27 * C, launch = 3.95 + 0.37 * C;
    b = dense ? 12 : 11, v = dense ? 11 : (C < 4 ? 13.5 : 12);
    if (split && !dense) b = 12.8, v = C == 2 || C == 3 ? 12 : 13;
  } else {
    a = 0.95 + 0.47 * C, launch = 4.7 + 0.22 * C;
    b = eights ? 1.24 * S : 17 + 0.7 * (S - 21), v = C == 3 ? 18 : 16;
    if (dense) {
      if (C > 2) a += (eights ? 0.75 : 0.3) * (C - 2);
      b += eights ? 14 : 6, v = C == 3 ? 17 : 14.5;
    }
  }
  return 8 + I * (a + 1e-4 * b * C * past) <= levels * launch + 1e-4 * I * blocks * C * v;
}

// Tiles per chunk of FP32 d/dtau at 33..64 states. A block's result is C doubles, so its chunk need not
// be as long as a d/dP one's (9 or 10 tiles here), and shorter ones fill the levels' last rounds
// better; but each sets P up, which weighs more the more blocks there are, and the sums may not depend
// on the batch, so it is chosen from the patterns and the waves of a block (2 C). Whole calls of 20 to 150
// taxa at 40 and 61 states against the d/dP chunks, one sample and 2 to 16: with 4 categories up to
// 1217 patterns 5 tiles took 0.61 to 0.92 and 0.64 to 1.02, at 1600 to 3000 6 tiles 0.76 to 0.98 and
// 0.80 to 1.04, at 4000 to 10000 8 tiles 0.92 to 1.00 and 0.94 to 1.01, where 5 lost up to 16 %; with
// one category 5 tiles at 3000 0.69 to 0.76 and 0.81 to 1.02, 6 at 8000 0.81 to 0.92 and 0.89 to 1.03.
// Past 16000 the d/dP chunks are 8 and more of themselves.
inline int tau_chunk_tiles(int ntiles, int C, int tiles_per_chunk) {
  const int x = ntiles * C;
  const int t = ntiles > 1000 ? tiles_per_chunk : (x <= 320 ? 5 : (x <= 800 ? 6 : (x <= 2560 ? 8 : tiles_per_chunk)));
  return t < tiles_per_chunk ? t : tiles_per_chunk;
}

// FP32 gradients at 33..64 states read P and P^T from zero-padded 64 x 64 copies.
inline bool use_ppad(int S, int dtype, int grad_mode) {
  return grad_mode != 0 && dtype != HX_F64 && S > 32 && S <= 64;
}

// Workspace of one hx_loglik* call: byte offsets of its regions.
struct WsLayout {
  size_t partials, tail, scales, rootsums, gpart, ppad, pcodes, total;  // tail: padding after the partials
};

// grad_mode: 0 loglik only, 1 d loglik / d mats, 2 d loglik / d tau.
// The layout depends on the tree only through its taxon count.
inline WsLayout ws_layout_t(int taxa, int S, int N, int C, int K, int dtype, int grad_mode) {
  const size_t rb = dtype == HX_F64 ? 8 : 4;
  const Tiling t = make_tiling(N, C, K, S, (int)rb);
  const size_t I = (size_t)taxa - 1, B = 2 * (size_t)taxa - 2;
  WsLayout w;
  size_t off = 0;
  w.partials = off;
  const size_t np = S == 4 ? (size_t)t.ntiles * 64 : (size_t)N;
  // dense states: the pre-order reads up to 16 C S + 64 elements past the
  // last (node, sample) slab (rows of the last tile past N, padded states)
  w.tail = off + I * K * np * C * S * rb;
  const size_t tail = S == 4 ? 0 : (16 * (size_t)C * S + 64) * rb;
  off = align_up(w.tail + tail, 256);
  w.scales = off;  // S = 4: 64-byte-aligned copy of the tip codes [T][ntiles * 64]
  if (S == 4) off = align_up(off + (size_t)taxa * t.ntiles * 64, 256);
  else off = align_up(off + I * K * (size_t)N * 4, 256);
  w.rootsums = off;
  off = align_up(off + (size_t)K * t.ntiles * (1 + S + C) * 8, 256);
  w.gpart = off;
  if (grad_mode == 1) off = align_up(off + B * K * (size_t)t.nchunks * C * S * S * rb, 256);
  if (grad_mode == 2) off = align_up(off + B * K * (size_t)t.nchunks * C * 8, 256);
  w.ppad = off;
  if (use_ppad(S, dtype, grad_mode)) off = align_up(off + B * K * (size_t)C * 2 * 64 * 64 * rb, 256);
  // four-state FP32: room for 16-bit tip codes and cherry code pairs, which the walks no longer
  // need (they read the caller's codes); kept so that workspace sizes, and the pattern slices
  // chosen by them, stay as they are
  w.pcodes = off;
  if (S == 4 && rb == 4)
    off = align_up(off + ((size_t)taxa + (size_t)taxa / 2) * t.ntiles * 64 * 2, 256);
  w.total = off;
  return w;
}

// hx_workspace_bytes for a tree of `taxa` taxa (the layout needs no plan).
inline size_t workspace_bytes_for(int taxa, int S, int N, int C, int K, int dtype, int grad_mode) {
  return ws_layout_t(taxa, S, N, C, K, dtype, grad_mode).total;
}

// Whether a call's walks leave cherries out of memory: 0 (the post-order walk stores no partial
// of a cherry, the pre-order walk rebuilds it from the two tips' codes) for four-state FP32 calls
// with tip codes that run as walks (use_pre_walk), -1 when every internal partial is stored.
inline int walk_drop_mode(int S, int C, int N, int K, int dtype, int tip_kind) {
  if (S != 4 || dtype == HX_F64 || tip_kind != HX_TIPS_CODES || !use_pre_walk(S, C, 4, N, K))
    return -1;
  return 0;
}

// Workspace of one resident-job evaluation (hx_job_eval): P (and dP/dtau), one pattern
// slice's pruning workspace, and the per-request sums.
struct JobWs {
  size_t mats, mats_dt, prune, prune_bytes, loglik_tmp, dtau_tmp, dtau_acc, total;
};

inline JobWs job_ws_shape(int taxa, int S, int slice, int C, int K, int dtype, int grad) {
  const size_t rb = dtype == HX_F64 ? 8 : 4;
  const size_t B = 2 * (size_t)taxa - 2;
  const size_t nm = (size_t)K * B * C * S * S;
  const size_t nt = (size_t)K * B * C;
  JobWs w{};
  size_t off = 0;
  w.mats = off;
  off = align_up(off + nm * rb, 256);
  if (grad) {
    w.mats_dt = off;
    off = align_up(off + nm * rb, 256);
  }
  w.prune = off;
  w.prune_bytes = workspace_bytes_for(taxa, S, slice, C, K, dtype, grad ? HX_GRAD_TAU : HX_GRAD_NONE);
  off = align_up(off + w.prune_bytes, 256);
  w.loglik_tmp = off;
  off = align_up(off + (size_t)K * 8, 256);
  if (grad) {
    w.dtau_tmp = off;
    off = align_up(off + nt * 8, 256);
    w.dtau_acc = off;
    off = align_up(off + nt * 8, 256);
  }
  w.total = off;
  return w;
}

}  // namespace hx
