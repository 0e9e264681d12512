// Declarations shared by the pruning translation units.
#pragma once

#include "common.hpp"

namespace hx {

template <typename R>
struct PassArgs {
  const int32_t* kids;  // [2T-1][2]
  int T, N, C, K, B;
  int ntiles, tiles_per_chunk, nchunks;
  int np;                 // pattern stride of the partials: N, or 64 ntiles for S = 4
  const R* mats;          // [K][B][C][S][S]
  const uint8_t* codes;   // [T][N]
  const R* table;         // [ncodes][S]
  int ncodes;
  const R* dense;         // [T][N][S]
  R* partials;            // [I][K][N][C][S]; S = 4: [I][K][C][np][4]
                          // (with `lanes`: [4][16] within 16 patterns)
  int32_t* scales;        // [I][K][N] (S != 4)
  uint8_t* codes_pad;     // S = 4: codes [T][ntiles * 64], rows 64-byte aligned (same memory)
  const R* freqs;
  int freqs_ks;           // stride between samples (0 or S)
  const R* props;
  int props_ks;           // stride between samples (0 or C)
  const double* weights;  // [N]
  double* rootsums;       // [K][nchunks][1+S+C]; S = 4: [K][ntiles][1+S+C]
  R* gpart;               // [B][K][nchunks][C][S][S]     (d loglik / d mats mode)
  const R* mats_dt;       // [K][B][C][S][S] dP/dtau; non-null selects d loglik / d tau mode
  double* gtau;           // [B][K][nchunks][C]            (d loglik / d tau mode)
  R* ppad;                // [K][B][C][2][64][64]: P and P^T zero-padded (FP32, 33..64 states);
                          // with `split`, each element holds its BF16 hi and lo halves
  int split;              // dense-state products as split BF16 on the matrix cores (FP32 only)
  // Four-state FP32 walks with tip codes: the post-order stores no cherry's partial and the
  // pre-order rebuilds it from the two tips' codes.
  int drop;
  int lanes;  // four-state FP64: partials in the lane order of the pre-order walk, which follows
  int root_parts;  // dense states: parts of the root's sums that a block takes (k_post_mfma)
};

constexpr double kLn2 = 0.69314718055994530942;

// Workgroup barrier that orders LDS only. __syncthreads() also waits for every
// outstanding global load and store of the wave (vmcnt(0)); the pruning
// kernels' barriers guard LDS tiles alone, since no wave reads global data
// that another wave of the same launch writes.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Dense-state (S != 4) launchers, defined in pruning_wide.hip.
template <typename R>
int launch_post_wide(const PassArgs<R>& a, const int32_t* nodes, int width, int tips, bool root,
                     int S, hipStream_t st);
template <typename R>
int launch_pre_wide(const PassArgs<R>& a, const int32_t* nodes, int width, int tips, bool root,
                    int S, hipStream_t st);

// Four-state kernels. Partials of S = 4 use the category-major layout [slot][K][C][np][4].
// FP32 at up to kPreWalkMaxC categories: both passes as walks on the matrix cores
// (pruning_walk.hip; use_pre_walk in layout.hpp). `store`: keep the partials for a gradient.
int launch_post_walk4(const PassArgs<float>& a, const int32_t* prog, int nprog, int slots, int tips,
                      bool store, hipStream_t st);
int launch_pre_walk4(const PassArgs<float>& a, const int32_t* prog, int nprog, int tips,
                     hipStream_t st);
// More than 4 categories (pruning_dna.hip): the post-order walk on the vector units
// and the pre-order adjoint one level per launch.
constexpr size_t kDnaLdsBudget = 64 * 1024;
constexpr size_t kDnaWalkLdsMax = 160 * 1024;  // gfx950 LDS per workgroup
// LDS of that post-order walk with W samples per block: it bounds the taxa of every four-state call
// with tip codes (about 2,500).
inline size_t dna_walk_lds(int T, int W, int need, int tips, int ncodes, size_t rb) {
  return (tips == HX_TIPS_CODES ? (size_t)T * 64 + (size_t)ncodes * 4 * rb : 0) +
         (size_t)W * need * 64 * 4;
}
template <typename R>
int launch_post_dna(const PassArgs<R>& a, const int32_t* prog, int nprog, int need, int tips,
                    hipStream_t st);
// FP64 with at most 4 categories: the post-order (pruning_walk64.hip).
int launch_post_walk64(const PassArgs<double>& a, const int32_t* prog, int nprog, int slots, int tips,
                       bool store, hipStream_t st);
// Its gradient: the pre-order and the sum of its statistics, d loglik / d mats or d tau in `out`.
int launch_pre_walk64(const PassArgs<double>& a, const int32_t* prog, int nprog, int tips, double* out,
                      hipStream_t st);
template <typename R>
int launch_pre_dna(const PassArgs<R>& a, const int32_t* nodes, int width, int tips, bool root,
                   hipStream_t st);

// Dense states as walks (pruning_dwalk.hip): FP32 and split-BF16 calls at up to kDwalkMaxS states
// and 4 categories (use_dwalk in layout.hpp). `store`: keep the partials for a gradient.
int launch_post_dwalk(const PassArgs<float>& a, const int32_t* prog, int nprog, int slots, int tips,
                      int S, bool store, hipStream_t st);

// Dense-state kernels on MFMA (pruning_mfma.hip, FP32 and FP64); used when
// use_mfma() (layout.hpp).
template <typename R>
int launch_mfma(bool post, const PassArgs<R>& a, const int32_t* nodes, int width, int tips,
                bool root, int S, hipStream_t st);

}  // namespace hx
