// Grouped GEMM of at most 32 rows in all and a long contraction for gfx950: one sequence being decoded, or a few.
//
// Such a GEMM reads the weights of the experts that have a row once and does next to nothing with them.  Tiles of the
// other kernels are too wide for it: 64 columns of all of K make 128 workgroups of FFN2 of one token, top-2 of 4096 /
// 14336, and with 768 / 3072 24 workgroups that walk 48 K steps one after the other.  Here a workgroup has 16 columns
// of one expert, its eight wavefronts an eighth of K each, and their sums meet in LDS: no plan, no partial tiles in
// memory, no reduction launch.
//
//   * nobody shares a weight, so the fragments come straight from memory: a lane takes 32 consecutive bytes of its
//     column's row and 64 lanes whole 128-byte lines of 16 rows, which two MFMAs then contract in an order of K of
//     their own (the tokens' fragments are loaded with the same addresses);
//   * two K tiles are in flight per wavefront while two are multiplied, 16 wavefronts per CU;
//   * the sum over K goes by eighths in a fixed order, so two calls give the same bits (not those of the other tiles).
//
// Bound by the weights where they are large, else by a chain of loads (offsets, row index, operands).  FFN2 of one token,
// top-2 of 8 experts, with the launches around it, in tiles of few.hip, in 256-row tiles and here: 4096 / 14336 59, 49
// and 37 us (6.3 TB/s); 2048 / 8192 37, 31 and 14; 1024 / 4096 21, 33 and 8; 768 / 3072 17, 46 and 8.
#include "ccf_common.h"
#include "gelu.h"
#include "plan.h"

#include <type_traits>

namespace ccf {
namespace {

constexpr int kThinWaves = 8;
constexpr int kThinK = 64;              // K elements of a step
constexpr int kThinMaxRows = 32;

__device__ __forceinline__ half8 thin_load(const half_t *p) { return *reinterpret_cast<const half8 *>(p); }

// RB blocks of 16 rows.
template <int kEpi, int RB>
__global__ void __launch_bounds__(kThinWaves * 64, 4)
thin_rows_kernel(FewArgs p, int n_col) {
  constexpr int kUnroll = 2;
  constexpr int LD = 16 + 4;
  __shared__ float s_part[kThinWaves][16 * RB][LD];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the workgroup's expert: the one of rank blockIdx.x / n_col among those with rows
  int rank = static_cast<int>(blockIdx.x) / n_col;
  const int n0 = (static_cast<int>(blockIdx.x) - rank * n_col) * 16;
  int e = -1, row0 = 0, rows = 0;
  for (int e0 = 0; e0 < p.E; e0 += 64) {
    int lo = 0, hi = 0;
    if (e0 + lane < p.E) {
      lo = p.offsets[e0 + lane];
      hi = p.offsets[e0 + lane + 1];
      lo = lo < p.max_rows ? lo : p.max_rows;
      hi = hi < p.max_rows ? hi : p.max_rows;
    }
    const unsigned long long live = __ballot(hi > lo);
    const int here = __popcll(live);
    if (rank < here) {
      const int before = __popcll(live & ((1ull << lane) - 1));
      const int who = __ffsll(__ballot(hi > lo && before == rank)) - 1;
      e = e0 + who;
      row0 = __builtin_amdgcn_readlane(lo, who);
      rows = __builtin_amdgcn_readlane(hi, who) - row0;
      break;
    }
    rank -= here;
  }
  if (e < 0) return;                                               // fewer experts have rows than the grid allows for
  rows = rows < 16 * RB ? rows : 16 * RB;

  // this lane's part of a K step: elements 16 (lane / 16) .. + 15 of row lane % 16 of every block (past the end: the
  // last row again, never stored)
  const int r16 = lane & 15, k_in = (lane >> 4) * 16;
  const int n = n0 + r16 < p.N ? n0 + r16 : p.N - 1;
  const half_t *w = p.B + (static_cast<size_t>(e) * p.N + n) * p.K + k_in, *x[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const int r = 16 * b + r16;
    int row = row0 + (r < rows ? r : rows - 1);
    if (p.a_rows) row = p.a_rows[row];
    x[b] = p.A + static_cast<size_t>(row) * p.K + k_in;
  }
  // K steps of this wavefront
  const int KT = p.K / kThinK, base = KT / kThinWaves, rem = KT % kThinWaves;
  const int first = wave * base + (wave < rem ? wave : rem), count = base + (wave < rem ? 1 : 0);
  float4v acc[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) acc[b] = float4v{0, 0, 0, 0};
  half8 wf[2][kUnroll][2], xf[2][kUnroll][RB][2];
  auto fetch = [&](int s, auto B_) {                               // K steps first + s ..; past the last one it again
    constexpr int buf = decltype(B_)::value;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int k = (first + (s + u < count ? s + u : count - 1)) * kThinK;
      wf[buf][u][0] = thin_load(w + k);
      wf[buf][u][1] = thin_load(w + k + 8);
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        xf[buf][u][b][0] = thin_load(x[b] + k);
        xf[buf][u][b][1] = thin_load(x[b] + k + 8);
      }
    }
  };
  auto multiply = [&](int s, auto B_) {
    constexpr int buf = decltype(B_)::value;
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      if (s + u >= count) break;                                   // uniform
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[buf][u][h], xf[buf][u][b][h], acc[b], 0, 0, 0);
    }
  };
  if (count > 0) {
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    fetch(0, even);
    for (int s = 0; s < count; s += 2 * kUnroll) {
      fetch(s + kUnroll, odd);
      __builtin_amdgcn_sched_barrier(0);
      multiply(s, even);
      __builtin_amdgcn_sched_barrier(0);
      fetch(s + 2 * kUnroll, even);
      __builtin_amdgcn_sched_barrier(0);
      multiply(s + kUnroll, odd);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // a lane holds one row and four consecutive columns of every block
#pragma unroll
  for (int b = 0; b < RB; ++b) *reinterpret_cast<float4v *>(&s_part[wave][16 * b + r16][4 * (lane >> 4)]) = acc[b];
  __syncthreads();
  const half_t *bias_e = p.bias ? p.bias + static_cast<size_t>(e) * p.N : nullptr;
  for (int o = threadIdx.x; o < rows * 16; o += kThinWaves * 64) {
    const int r = o / 16, col = n0 + o % 16;
    if (col >= p.N) continue;
    const int j = row0 + r;
    const size_t crow = p.c_rows ? static_cast<size_t>(p.c_rows[j]) : static_cast<size_t>(j);
    const float bias = bias_e ? static_cast<float>(bias_e[col]) : 0.0f;
    const float sc = p.row_scale ? static_cast<float>(p.row_scale[j]) : 1.0f;
    float v = s_part[0][r][o % 16];
#pragma unroll
    for (int i = 1; i < kThinWaves; ++i) v += s_part[i][r][o % 16];
    v += bias;
    v = kEpi == kFewPlain ? v * sc : gelu_erf(v);
    p.C[crow * p.N + col] = static_cast<half_t>(v);
  }
}

// Workgroups of 16 columns over all experts that may have rows.
long long thin_wgs(int max_rows, int E, int N) { return static_cast<long long>((N + 15) / 16) * (E < max_rows ? E : max_rows); }

// Two workgroups per CU at most: more of them are as many short ones, whose start costs more than their share of the
// weights (tiles of few.hip and here: FFN1 of one token, top-2 of 4096 / 14336, 1792 workgroups, 38 and 55 us; FFN2 of 8
// tokens of 32 experts of 1024 / 4096, 1024 workgroups, 22 and 25).  And eight wavefronts want two K tiles each (K of 768,
// 384 workgroups: 8.4 and 9.7).
//
// Within that, what takes the time here is the rounds of four K tiles that a wavefront has on their way, the rows of an
// expert that each of them fetches again, and a second workgroup on the CU, so both forms are priced in microseconds.
// Of 1295 GEMMs timed (K of 1024 to 4032, 1 to 32 experts, 64 to 512 workgroups, 1 to 32 rows) this takes the slower form
// by over 2 % in one (3.6 %), and by over 3 % where it stays with few.hip in six (4.6 % at most).  Tiles of few.hip and
// here: K of 1024, 256 workgroups, one expert: 16 rows 8.6 and 7.7, 32 rows 8.6 and 10.4; 512 workgroups, two experts: 2
// rows 8.7 and 9.0, 32 rows 8.7 and 14.3; K of 2048, 512 workgroups, 8 experts: 16 rows 13.4 and 9.9; one: 32 rows 13.0
// and 18.7.
//
// As many rows as experts and more of a K of 4096 and more are left to few.hip and to 256-row tiles that the plan cuts
// along K over the chip.  The times do not cross there (8 rows of 8 experts of 1024 / 4096: 27 us in those tiles, 21 in
// few.hip, 15 here; 2 of 2 of 4096 / 14336: 49, 59 and 37): the line keeps that form's calls as they were.
bool thin_rows_pays(int max_rows, int E, int N, int K) {
  const long long wgs = thin_wgs(max_rows, E, N);
  if (K < 2 * kThinWaves * kThinK || wgs > 512 || (max_rows >= E && K >= 64 * kThinK)) return false;
  const double rows = static_cast<double>(max_rows) / (E < max_rows ? E : max_rows);
  const int rounds = (K + 4 * kThinWaves * kThinK - 1) / (4 * kThinWaves * kThinK);
  const double here = 3.5 + (wgs <= 256 ? 1.0 : 2.5) * rounds * (2.1 + (max_rows > 16 ? 0.4 : 0.0) + 0.12 * rows);
  return here < 4.5 + 0.265 * K / kThinK;
}

}  // namespace

bool thin_rows_fits(int mode, int max_rows, int E, int N, int K, int epi, bool b_kn) {
  if ((mode != 1 && mode != 3) || b_kn || epi > kFewGelu || K % kThinK || E <= 0 || E > 1024 || max_rows <= 0 ||
      max_rows > kThinMaxRows || thin_wgs(max_rows, E, N) >= (1ll << 24))
    return false;
  return mode == 3 || thin_rows_pays(max_rows, E, N, K);
}

int thin_rows_gemm(const FewArgs &p, int epi, hipStream_t stream, const char *what) {
  const bool tall = p.max_rows > 16;
  void (*kernel)(FewArgs, int) = epi == kFewPlain ? (tall ? thin_rows_kernel<kFewPlain, 2> : thin_rows_kernel<kFewPlain, 1>)
                                                  : (tall ? thin_rows_kernel<kFewGelu, 2> : thin_rows_kernel<kFewGelu, 1>);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(thin_wgs(p.max_rows, p.E, p.N))), dim3(kThinWaves * 64), 0, stream, p,
                     (p.N + 15) / 16);
  return check_launch(what);
}

}  // namespace ccf
