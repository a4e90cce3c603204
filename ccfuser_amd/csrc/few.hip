// Grouped GEMM of few rows per expert for gfx950: decoding batches, short prompts, small layers.
//
// The 256-row tiles of ffn.hip leave most of the chip idle there: 32 rows per expert fill an eighth of a
// tile, and a layer of a few hundred rows makes a few dozen tiles for 256 CUs.  This kernel has tiles of 64
// or 128 rows by 64, 128 or 256 columns, picks among them on the device from the experts' row counts, and runs
// all of K in one workgroup: no plan launch in front, no partial tiles, no reduction behind.
//
//   * every workgroup derives its own tiles from the offsets (a scan over the experts and one binary search
//     per tile), so the launch stands alone;
//   * tiles of one column range lie side by side on an XCD, so an expert's second M tile reads the weights
//     from that XCD's L2;
//   * operands go to LDS with direct loads, 64 K elements per stage, as many stages as fit; the pipeline
//     runs on across a workgroup's tiles (the stages of the next tile are loaded under the last steps of
//     this one).  One workgroup of eight wavefronts per CU: two workgroups of four with half of the LDS each
//     measured the same at many tiles and up to a quarter slower at one tile per CU, whose weights then stream
//     through a pipeline of half the depth;
//   * accumulation runs over K in 32-wide steps in ascending order, as in the 256-row tiles: same bits.  By the rule, tiles
//     of large weights start inside K, at a place that the column gives, and go around: other bits than the 256-row tiles'
//     and than those of a call of more rows, the same for every tile shape and slot of an expert (starts_apart()).
//
// Bound by streaming the weights from HBM at 6.2 - 6.7 TB/s where they are large, by the latency of a few dependent
// steps where they are small.  FFN1 / FFN2 including their plan and reduction launches, 256-row tiles -> here:
// 8 experts of 4096 / 14336, 32 rows each: 202 -> 150 and 192 -> 140 us, 83 rows each: 199 -> 171 and 203 -> 163;
// 4 experts of 256 / 1024, 128 rows each: 21 -> 8 and 28 -> 10; FFN2 of 8 experts of 768 / 3072, 500 rows
// each: 62 -> 37; 16 experts of 1024 / 4096, 64 rows each: 31 -> 28 and 44 -> 26.
#include "ccf_common.h"
#include "gelu.h"
#include "gemm_tile.h"
#include "plan.h"

#include <cmath>

namespace ccf {
namespace {

constexpr int kFewThreads = 512;
constexpr int kFewLds = 163840;
constexpr int kFewMaxRounds = 64;      // most tiles of a workgroup: one per lane of the tile table
constexpr int kBK = 64;
// A K step of 64 and an epilogue (GELU, plain) by tile shape, in microseconds: fitted to 2520 timed launches of all
// shapes where the weights' bytes do not bound them, 4 to 9 % off each (before fragments were read ahead of their use, which
// took up to 16 % off a step: see few_rows_fits)
constexpr double kFewStepUs[6] = {0.274, 0.415, 0.705, 0.408, 0.600, 0.900};
constexpr double kFewEpiUs[2][6] = {{1.3, 2.2, 3.2, 2.7, 5.5, 8.7}, {0.8, 0.6, 0.5, 1.7, 3.3, 5.7}};

// Tile of 16 TM rows x 32 DB columns, 64 K elements per stage.  Eight wavefronts, 2 along the rows (wavefront half m
// holds the 16-row blocks m, m + 2, ...) x 4 along the columns (16 NB columns each): two wavefronts per SIMD, so one's
// LDS reads run under the other's MFMAs.
template <int TM_, int DB_>
struct FewCfg {
  static constexpr int TM = TM_, DB = DB_, TMW = TM / 2, NB = DB / 2, BN = 32 * DB;
  static constexpr int A_DMA = TM / 4, B_DMA = DB / 2, LOADS = A_DMA + B_DMA;             // 1 KB loads per wavefront and stage
  static constexpr int A_BYTES = 16 * TM * kBK * 2, STAGE = A_BYTES + BN * kBK * 2;
  static constexpr int FIT = kFewLds / STAGE, STAGES = FIT > 8 ? 8 : FIT;
  static_assert(TM % 4 == 0 && DB % 2 == 0 && STAGES >= 3 && (STAGES - 1) * LOADS < 63, "tile shape");
};

// One K half's fragments of a wavefront: row blocks 32 rows (4096 bytes) apart, column blocks 16 rows (2048 bytes) apart.
// For weights stored [K][N] (kKN) a column block's fragment is two transposing reads, K rows 0..3 and 4..7 of the lane's
// eight (8 BN bytes apart), at the lane's address XOR 32 J.  read() leaves the reads in flight; ready() waits until at most
// LATER reads that were issued behind them are, and ties the registers to the wait.
template <class C, bool kKN>
struct FewFrags {
  static constexpr int TMW = C::TMW, NB = C::NB, READS = TMW + (kKN ? 2 : 1) * NB;
  half8 a[TMW], b[NB];
  half4 lo[NB], hi[NB];
  __device__ __forceinline__ void read(uint32_t ra, uint32_t rb) {
    static_for<0, NB>([&](auto J) {
      constexpr int j = J.value;
      if constexpr (kKN) {
        lo[j] = lds_read_tr_b64<0>(rb ^ (32 * j));
        hi[j] = lds_read_tr_b64<8 * C::BN>(rb ^ (32 * j));
      } else {
        b[j] = lds_read_b128<2048 * j>(rb);
      }
    });
    static_for<0, TMW>([&](auto I) { a[I.value] = lds_read_b128<4096 * I.value>(ra); });
  }
  template <int LATER>
  __device__ __forceinline__ void ready() {
    static_assert(LATER < 15, "lgkmcnt has four bits");
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(LATER) : "memory");
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if constexpr (kKN) {
        asm volatile("" : "+v"(lo[j]), "+v"(hi[j]));
        b[j] = __builtin_shufflevector(lo[j], hi[j], 0, 1, 2, 3, 4, 5, 6, 7);
      } else {
        asm volatile("" : "+v"(b[j]));
      }
    }
#pragma unroll
    for (int i = 0; i < TMW; ++i) asm volatile("" : "+v"(a[i]));
  }
};

// A [K][N] weight tile in LDS: 64 K rows of BN columns, the 32-byte chunks of each span of 128 columns XOR-swizzled by
// the row (the layout of the 256-row tiles' main loop, gemm_tile.h).
__device__ __forceinline__ int few_kn_swz(int row) { return (row & 3) | (((row >> 3) & 1) << 2); }

// lds_dma16 with the non-temporal hint, for weights that one tile reads once: 6.2 TB/s from HBM instead of 5.5.  Weights
// that several M tiles share, or that a next call finds in the 256 MB Infinity Cache, do better without: the hint is for a
// tile that has its expert to itself where 320 MB pass before its weights are read again.  The kernel counts the experts
// that have rows; a layer's two products alternate, so each is half of that.  Microseconds without and with the hint:
//   a layer's two, again and again, 4 to 83 rows per expert: 8 experts with rows of 2304 / 8192 (302 MB each way) 124, 113;
//     of 4096 / 14336 334, 309; 16 of 2048 / 8192 245, 229; 4 of 2560 / 8192 (168 MB each) 78, 74, of 2304 / 8192 (151)
//     69, 69, of 2048 / 8192 (134) 62, 73; 2 of 4096 / 14336 (235) 141, 135, 1 of them (117) 85, 102
//   FFN1 alone: 8 of 2048 / 8192 (268 MB) 47, 66, of 2304 / 8192 (302) 51, 52, of 2560 / 8192 (336) 61, 57; 2 of 4096 /
//     14336 (235) 40, 54, 4 of them (470) 111, 105
// (Alone, 83 rows each of 8 of 2048 / 8192 do better with it, 68 and 59 for FFN2: the line goes by bytes, not rows.)
// A layer of 128 tokens, 8 experts of 4096 / 14336: 356 -> 333 us.
constexpr double kStreamBytes = 320e6;
__device__ __forceinline__ void lds_dma16_nt(const void *gptr, lds_char *lds_wave_base) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)gptr,
                                   (__attribute__((address_space(3))) void *)lds_wave_base, 16, 0, 2);
}

// Where the walk through K starts.  Rows of a [N][K] weight that are a multiple of 4 KB apart hold the same K at the same
// place of their pages, and workgroups that all start at the first K tile stay at about the same K: their loads fall on a
// few of the memory's channels at a time, on how few depends on where the weight happens to lie.  So where the weights
// come from HBM a tile's 256 columns go around from one of 16 places, 256 bytes apart.  The sum starts elsewhere (its error is
// the same), at a place that the column alone gives: not the tile's shape, nor the expert's slot, nor the other rows.
// Microseconds for a layer's two products in ascending order and so, two places of the weights each:
//   8 experts of 4096 / 14336, 32 rows each 313, 305 and 297, 296, 83 rows 347, 345 and 345, 344; two experts of it, one
//   row each 113 and 102; 64 rows of 16 of 2048 / 8192 250, 253 and 198, 199, 40 rows of 8 126 and 99; 40 rows of 16 of
//   1536 / 6144 127 and 119; 33 rows of 32 of 1024 / 4096 116, 112 and 105, 107; 64 rows of 8 of 3584 / 14336 314, 318 and 303.
// The places are sums of the shifted column number, the best of 90 such over 11 layers: the column number itself falls in
// with the channels' own pattern (those 16 of 2048 / 8192 206).  With 3 e added to it, places for every expert, 0 to 10 % faster
// again where N is 2048 and less, whose few column ranges have few places (64 rows of 32 of 2048 / 2048: 146 ascending, 107
// with 3 e, 117 here), the same at 4096 / 14336; but then an expert's results depend on its slot.
// Fewer rows than experts count as the others, so that a row's results are those of a larger call: the weights that they touch
// may stay in the cache, where it makes no difference (one row of 8 of 4096 / 14336 78.7 and 78.8, 8 of 32 of 1024 / 4096 39.4 and
// 39.2; four rows of the 8 202 and 147).
// Not for weights that stay in the Infinity Cache anyhow (134 MB: 64 rows each of 16 of 1024 / 4096 68.1 and 68.0, of 8 of 2048 /
// 4096 65.7 and 66.0; 151 MB: of 18 of 2048 / 2048 82 and 78), not for other row strides (5, 6, 7 and 10 KB, the first product of
// 8 experts of 2560 / 10240, 3072 / 12288, 3584 / 14336, 5120 / 13824: 100.8, 118.9, 154.2, 214 and 100.8, 118.8, 154.7, 215),
// and not for several M tiles an expert, where it wins and loses (200 rows of 8 of 2048 / 8192 183 and 174; 160 of 16 of 2048 /
// 6144, first product, 127 and 135).
constexpr double kRotateBytes = 160e6;
constexpr int kPlaces = 16, kPlaceStep = 2;        // K tiles of 128 bytes
bool can_start_apart(int K) {
  static_assert((kPlaces - 1) * kPlaceStep < 2048 / kBK, "a place inside the shortest K");
  return K % 2048 == 0;
}
bool starts_apart(int max_rows, int E, int N, int K) {
  return can_start_apart(K) && max_rows <= 128ll * E && 2.0 * E * N * K >= kRotateBytes;
}
__device__ __forceinline__ int first_k_tile(int n0) {
  const int c = n0 >> 8;
  return kPlaceStep * ((7 * c + 2 * (c >> 1) + 9 * (c >> 2) - (c >> 3) + 10 * (c >> 4)) & (kPlaces - 1));
}

// One lane's tile table entry.
struct FewTile {
  int e, row0, rows, n0;
  int alone;               // no other tile reads these weights
};

__device__ __forceinline__ FewTile tile_at(const FewTile &mine, int r) {
  return FewTile{__builtin_amdgcn_readlane(mine.e, r), __builtin_amdgcn_readlane(mine.row0, r),
                 __builtin_amdgcn_readlane(mine.rows, r), __builtin_amdgcn_readlane(mine.n0, r),
                 __builtin_amdgcn_readlane(mine.alone, r)};
}

// The workgroup's `nr` (>= 1) tiles, one after the other.  mine: lane r holds tile r.
template <class C, int kEpi, bool kKN, bool kStream>
__device__ __forceinline__ void few_run(const FewArgs &p, const FewTile &mine, int nr, lds_char *lds) {
  constexpr int TMW = C::TMW, NB = C::NB, S = C::STAGES;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 2, wn = wave & 3;
  const int KT = p.K / kBK;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));

  // this lane's fragment chunk of its first blocks, per K half: row lane % 16, K chunk lane / 16
  uint32_t a_off[2], b_off[2];
  {
    const int ra = wm * 16 + (lane & 15), rb = wn * (16 * NB) + (lane & 15);
#pragma unroll
    for (int sub = 0; sub < 2; ++sub) {
      const int c = sub * 4 + (lane >> 4);
      a_off[sub] = lds_base + (ra * 8 + (c ^ swz<8>(ra))) * 16;
      if constexpr (kKN) {
        // source lane i of its group of 16 points at K row 8 * group + i / 4, columns 4 (i % 4) ..
        const int i = lane & 15, row = sub * 32 + 8 * (lane >> 4) + (i >> 2), blk = wn * NB;
        b_off[sub] = lds_base + C::A_BYTES + row * (2 * C::BN) + (blk >> 3) * 256 + ((few_kn_swz(row) ^ (blk & 7)) << 5) + ((i & 3) << 3);
      } else {
        b_off[sub] = lds_base + C::A_BYTES + (rb * 8 + (c ^ swz<8>(rb))) * 16;
      }
    }
  }

  // The load side runs STAGES stages ahead: tile `it`, K tile `ik` of it.  Load j of a wavefront is 1 KB at
  // 1024 (8 j + wave) of the operand's part of the stage: eight 128-byte rows, or 1024 / (2 BN) K rows of a [K][N] tile.
  const half_t *a_src[C::A_DMA], *b_src[C::B_DMA];
  int it = 0, ik = 0, rot = 0;                                     // rot: the K tile that the walk starts with
  bool stream = false;                                             // the weights being loaded are read once
  const ptrdiff_t b_step = kKN ? static_cast<ptrdiff_t>(kBK) * p.N : kBK;
  auto sources = [&](const FewTile &t) {
    const half_t *Be = p.B + static_cast<size_t>(t.e) * p.N * p.K;
    stream = kStream && t.alone;
    if constexpr (!kKN)
      if (p.rotate) rot = first_k_tile(t.n0);
#pragma unroll
    for (int j = 0; j < C::A_DMA; ++j) {
      const int r = (j * 8 + wave) * 8 + (lane >> 3);
      int g = t.row0 + (r < t.rows ? r : t.rows - 1);              // padded tile rows re-read the last real row
      if (p.a_rows) g = p.a_rows[g];
      a_src[j] = p.A + static_cast<size_t>(g) * p.K + rot * kBK + ((lane & 7) ^ swz<8>(r)) * 8;
    }
#pragma unroll
    for (int j = 0; j < C::B_DMA; ++j) {
      if constexpr (kKN) {
        constexpr int UNITS = C::BN / 8;                           // 16-byte units of a K row
        const int r = (j * 8 + wave) * (64 / UNITS) + lane / UNITS, u = lane % UNITS, chunk = u >> 1;
        const int c = t.n0 + (chunk >> 3) * 128 + (((chunk & 7) ^ few_kn_swz(r)) << 4) + ((u & 1) << 3);
        b_src[j] = Be + static_cast<size_t>(r) * p.N + (c < p.N - 8 ? c : p.N - 8);
      } else {
        const int r = (j * 8 + wave) * 8 + (lane >> 3);
        const int n = (t.n0 + r) < p.N ? (t.n0 + r) : p.N - 1;
        b_src[j] = Be + static_cast<size_t>(n) * p.K + rot * kBK + ((lane & 7) ^ swz<8>(r)) * 8;
      }
    }
  };
  auto issue = [&](int stage) {
    lds_char *base = lds + stage * C::STAGE;
#pragma unroll
    for (int j = 0; j < C::A_DMA; ++j) lds_dma16(a_src[j], base + (j * 8 + wave) * 1024);
    if (kStream && stream) {
#pragma unroll
      for (int j = 0; j < C::B_DMA; ++j) lds_dma16_nt(b_src[j], base + C::A_BYTES + (j * 8 + wave) * 1024);
    } else {
#pragma unroll
      for (int j = 0; j < C::B_DMA; ++j) lds_dma16(b_src[j], base + C::A_BYTES + (j * 8 + wave) * 1024);
    }
    if (ik + 1 < KT) {
      ++ik;
      const ptrdiff_t back = !kKN && ik + rot == KT ? static_cast<ptrdiff_t>(p.K) : 0;       // from the last K tile to the first
#pragma unroll
      for (int j = 0; j < C::A_DMA; ++j) a_src[j] += kBK - back;
#pragma unroll
      for (int j = 0; j < C::B_DMA; ++j) b_src[j] += b_step - back;
    } else if (it + 1 < nr) {
      ++it;
      ik = 0;
      sources(tile_at(mine, it));
    }                                                              // past the end: the last K tile again, read by nobody
  };
  sources(tile_at(mine, 0));
#pragma unroll
  for (int s = 0; s < S; ++s) issue(s);

  // The fragments of a K half are read a half ahead of their use, so the barrier of a K step sits between its halves:
  // behind it the next stage is complete, and everyone has read all of this one, which takes the load of S steps ahead.
  FewFrags<C, kKN> f0, f1;
  wait_vmcnt<(S - 1) * C::LOADS>();
  block_barrier();
  f0.read(a_off[0], b_off[0]);
  int stage = 0;
  for (int r = 0; r < nr; ++r) {
    const FewTile t = tile_at(mine, r);
    const int live = (t.rows + 15) / 16;                           // 16-row blocks with real rows
    float4v acc[TMW][NB];
#pragma unroll
    for (int tm = 0; tm < TMW; ++tm)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) acc[tm][nb] = float4v{0, 0, 0, 0};
    auto multiply = [&](const FewFrags<C, kKN> &f) {
      static_for<0, TMW>([&](auto I) {
        constexpr int tm = I.value;
        if (2 * tm + wm < live) {                                  // uniform
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) acc[tm][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[nb], f.a[tm], acc[tm][nb], 0, 0, 0);
        }
      });
    };
    for (int kt = 0; kt < KT; ++kt) {
      const int next = stage == S - 1 ? 0 : stage + 1;
      const uint32_t so = stage * C::STAGE, sn = next * C::STAGE;
      f1.read(so + a_off[1], so + b_off[1]);
      f0.template ready<FewFrags<C, kKN>::READS>();
      multiply(f0);
      __builtin_amdgcn_sched_barrier(0);
      f1.template ready<0>();
      wait_vmcnt<(S - 2) * C::LOADS>();                            // the next stage has landed for this wavefront
      block_barrier();
      issue(stage);
      f0.read(sn + a_off[0], sn + b_off[0]);
      __builtin_amdgcn_sched_barrier(0);
      multiply(f1);
      __builtin_amdgcn_sched_barrier(0);
      stage = next;
    }
    f0.template ready<0>();                                        // the next tile's, or at the end nobody's
    // a lane holds one row and four consecutive columns of every block
    const half_t *bias_e = p.bias + static_cast<size_t>(t.e) * p.N;
    const int colb = t.n0 + wn * (16 * NB) + 4 * (lane >> 4);
#pragma unroll
    for (int tm = 0; tm < TMW; ++tm) {
      const int lr = (2 * tm + wm) * 16 + (lane & 15);
      if (2 * tm + wm >= live) break;                              // uniform
      const bool real = lr < t.rows;
      const int j = t.row0 + (real ? lr : t.rows - 1);
      const size_t crow = p.c_rows ? static_cast<size_t>(p.c_rows[j]) : static_cast<size_t>(j);
      const float sc = p.row_scale ? static_cast<float>(p.row_scale[j]) : 1.0f;
      half_t *dst = p.C + crow * p.N;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int col = colb + 16 * nb;
        if (!real || col >= p.N) continue;
        half4 bv = {0, 0, 0, 0};
        if (p.bias) bv = *reinterpret_cast<const half4 *>(bias_e + col);
        half4 o, pre;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          float x = acc[tm][nb][c] + static_cast<float>(bv[c]);
          if (kEpi == kFewPlain) {
            x *= sc;
          } else {
            pre[c] = static_cast<half_t>(x);
            x = gelu_erf(x);
          }
          o[c] = static_cast<half_t>(x);
        }
        *reinterpret_cast<half4 *>(dst + col) = o;
        if (kEpi == kFewGeluKeep) *reinterpret_cast<half4 *>(p.C2 + static_cast<size_t>(j) * p.N + col) = pre;
      }
    }
  }
  wait_vmcnt<0>();                                                 // no load into LDS outlives the workgroup
}

// Candidate tile shapes: index = 3 * (rows: 0 = 64, 1 = 128) + (columns: 0 = 64, 1 = 128, 2 = 256).
constexpr int kFewShapes = 6;

// kStream: the weights are large (a form of its own: the choice by tile in the loads of small ones cost 0.4 us of 36, two
// short launches of more code)
template <int kEpi, bool kKN, bool kStream>
__global__ void __launch_bounds__(kFewThreads)
few_rows_kernel(FewArgs p) {
  __shared__ __attribute__((aligned(1024))) char buf[kFewLds];
  int *s_off = reinterpret_cast<int *>(buf), *s_mt = s_off + 1056;  // tables of the tile search, before the pipeline starts
  static_assert(2 * 1056 * sizeof(int) <= kFewLds, "tables of 1024 experts");
  const int tid = threadIdx.x, lane = tid & 63;
  const int E = p.E;
  for (int e = tid; e <= E; e += kFewThreads) {
    const int v = p.offsets[e];
    s_off[e] = v < p.max_rows ? v : p.max_rows;                     // never past the caller's bound
  }
  __syncthreads();
  // M tiles of each height over all experts (every wavefront for itself)
  int m64 = 0, m128 = 0;
  for (int e = lane; e < E; e += 64) {
    int cnt = s_off[e + 1] - s_off[e];
    cnt = cnt > 0 ? cnt : 0;
    m64 += (cnt + 63) >> 6;
    m128 += (cnt + 127) >> 7;
  }
  [[maybe_unused]] int used = 0;                                    // experts with rows
  if constexpr (kStream)
    for (int e0 = 0; e0 < E; e0 += 64) used += __popcll(__ballot(e0 + lane < E && s_off[e0 + lane + 1] > s_off[e0 + lane]));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    m64 += __shfl_xor(m64, off, 64);
    m128 += __shfl_xor(m128, off, 64);
  }
  // price the shapes, one per lane: rounds of tiles times the rows of both operands that a K step loads.  Of 2520 timed
  // launches this takes a shape that is over 5 % slower than the best one in 120, on average 0.8 %; kFewStepUs did
  // so in 49, but was up to 14 % slower than this choice where most experts' rows end just past a tile.
  const int slots = gridDim.x >> 3;                                 // workgroups per XCD
  const int ci = lane < kFewShapes ? lane : 0;
  const int rsel = ci / 3, csel = ci - 3 * rsel;
  const int mt_l = rsel == 0 ? m64 : m128;
  const int per_x_l = (mt_l * ((p.N + (64 << csel) - 1) >> (6 + csel)) + 7) >> 3;
  const int rounds_l = (per_x_l + slots - 1) / slots;
  int key = INT_MAX;
  if (lane < kFewShapes && rounds_l <= kFewMaxRounds && (!kKN || csel > 0)) {      // no [K][N] layout of 64 columns
    key = (rounds_l * ((64 << rsel) + (64 << csel))) << 4 | lane;
  }
  if (lane == p.force && key != INT_MAX) key = lane;                // below every price
#pragma unroll
  for (int off = 4; off >= 1; off >>= 1) {
    const int other = __shfl_xor(key, off, 64);
    key = other < key ? other : key;
  }
  key = __builtin_amdgcn_readfirstlane(key);
  const int shape = key & 15;
  const int rs = shape / 3, cs = shape - 3 * rs;
  const int MT = __builtin_amdgcn_readfirstlane(rs == 0 ? m64 : m128);
  if (MT == 0) return;
  const int n_col = (p.N + (64 << cs) - 1) >> (6 + cs);
  const int T = MT * n_col, per_x = (T + 7) >> 3;
  // exclusive scan of the chosen M tiles
  if (tid < 64) {
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      int cnt = e0 + lane < E ? s_off[e0 + lane + 1] - s_off[e0 + lane] : 0;
      cnt = cnt > 0 ? cnt : 0;
      const int v = (cnt + (64 << rs) - 1) >> (6 + rs);
      int inc = v;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(inc, off, 64);
        if (lane >= off) inc += o;
      }
      if (e0 + lane < E) s_mt[e0 + lane] = carry + inc - v;
      carry += __shfl(inc, 63, 64);
    }
    if (lane == 0) s_mt[E] = carry;
  }
  __syncthreads();
  // workgroup j of XCD x has tiles x * per_x + j, + slots, ...; lane r finds tile r.  Tile order: expert, column
  // range, M tile.
  const int x = blockIdx.x & 7, first = blockIdx.x >> 3;
  int left = T - x * per_x;
  left = left < per_x ? left : per_x;                               // tiles of this XCD
  const int nr = first < left ? (left - first + slots - 1) / slots : 0;
  if (nr <= 0) return;
  FewTile mine;
  {
    const int i = first + (lane < nr ? lane : 0) * slots;
    const int t = x * per_x + i;
    int lo = 0, hi = E - 1;                                         // last expert whose tiles start at or before t
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_mt[mid] * n_col <= t) lo = mid;
      else hi = mid - 1;
    }
    const int mts = s_mt[lo + 1] - s_mt[lo], local = t - s_mt[lo] * n_col;
    const int ct = local / mts, m = local - ct * mts;
    const int cnt = s_off[lo + 1] - s_off[lo], r0 = m << (6 + rs), bm = 64 << rs;
    mine.e = lo;
    mine.row0 = s_off[lo] + r0;
    mine.rows = cnt - r0 < bm ? cnt - r0 : bm;
    mine.n0 = ct << (6 + cs);
    mine.alone = mts == 1;
  }
  __syncthreads();                                                  // the tables have been read
  lds_char *lds = (lds_char *)buf;
  auto go = [&](auto CI) {
    constexpr int i = CI.value;
    if constexpr (!kKN || i % 3 > 0)
      if (shape == i) {
        // two loops, not one that chooses: FFN2 of 64 rows of one of 16 experts of 2048 / 8192 takes 40 us, 46 with the
        // choice at every load (42 with the hint, 38 in the form of small weights)
        if (kStream && used >= p.stream_experts) few_run<FewCfg<4 << (i / 3), 2 << (i % 3)>, kEpi, kKN, kStream>(p, mine, nr, lds);
        else few_run<FewCfg<4 << (i / 3), 2 << (i % 3)>, kEpi, kKN, false>(p, mine, nr, lds);
      }
  };
  static_for<0, kFewShapes>(go);
}

// P(X > z) of a standard normal variable, within 2e-4: the rule below is on the host path of every GEMM, and an exp
// takes a third of an erfc's time.
double upper_tail(double z) { return 1 / (1 + std::exp(z * (1.5976 + 0.07056 * z * z))); }

}  // namespace

TileCount m_tiles(int max_rows, int E, int bm) {
  const int used = E < max_rows ? E : max_rows;
  if (used <= 0) return {0.0, 0.0};
  const double avg = static_cast<double>(max_rows) / used, sd = std::sqrt(avg * (1.0 - 1.0 / used));
  if (sd == 0) return {used * std::ceil(avg / bm), 0.0};
  // tiles of an expert: the sum over j of (rows > j bm)
  const double first = std::floor((avg - 5 * sd) / bm);
  const int j0 = first > 0 ? static_cast<int>(first) : 0;
  double m = j0, m2 = static_cast<double>(j0) * j0;
  for (int j = j0;; ++j) {
    const double p = upper_tail((static_cast<double>(j) * bm + 0.5 - avg) / sd);
    if (!(p >= 1e-4)) break;
    m += p;
    m2 += (2.0 * j + 1) * p;
  }
  return {used * m, used * (m2 > m * m ? m2 - m * m : 0.0)};
}

// Mean of ceil(M tiles * n_col / cus): the rounds that the workgroups of cus CUs take.
static double mean_rounds(const TileCount &t, int n_col, int cus) {
  const double sd = std::sqrt(t.var), per = static_cast<double>(cus) / n_col;     // M tiles of a round
  if (sd < 0.2) return std::ceil(t.mean / per - 1e-9);
  const double first = std::floor((t.mean - 4 * sd) / per);
  double rounds = first > 0 ? first : 0;
  for (double r = rounds;; r += 1) {
    const double p = upper_tail((std::floor(r * per) + 0.5 - t.mean) / sd);       // more M tiles than r rounds hold
    if (!(p >= 1e-3)) break;
    rounds += p;
  }
  return rounds;
}

SkinnyCount skinny_tiles(int max_rows, int E) {
  const int used = E < max_rows ? E : max_rows;
  if (used <= 0) return {0.0, 0.0};
  const double avg = static_cast<double>(max_rows) / used, sd = std::sqrt(avg * (1.0 - 1.0 / used));
  const auto at_most = [&](double x) { return sd > 0 ? 1 - upper_tail((x + 0.5 - avg) / sd) : (avg <= x ? 1.0 : 0.0); };
  const int j0 = avg > 5 * sd ? static_cast<int>((avg - 5 * sd) / 256) : 0, j1 = static_cast<int>((avg + 5 * sd) / 256);
  double full = 0, skinny = 0;
  for (int j = j0; j <= j1; ++j) {
    const double whole = at_most(256.0 * j), one = at_most(256.0 * j + 64), two = at_most(256.0 * j + 128);
    full += j * (two - at_most(256.0 * j - 1)) + (j + 1) * (at_most(256.0 * j + 256 - 1) - two);
    skinny += (one - whole) + 2 * (two - one);
  }
  return {used * full, used * skinny};
}

bool few_rows_fits(int mode, int max_rows, int E, int N, int K, int epi, bool b_kn, int cus) {
  if (!mode || epi > kFewGeluKeep || (b_kn && epi == kFewGeluKeep) || cus < 8 || K % kBK || E <= 0 || E > 1024 || max_rows <= 0)
    return false;
  // the tile table holds kFewMaxRounds tiles per workgroup of the largest shape
  const long long worst = (static_cast<long long>(max_rows) / 128 + E) * ((N + 255) / 256);
  if (worst >= static_cast<long long>(kFewMaxRounds - 1) * cus) return false;
  if (mode >= 2 || thin_rows_fits(mode, max_rows, E, N, K, epi, b_kn)) return true;
  // Where either is far ahead nothing is priced (0.3 to 0.8 us): three rounds of 256-row tiles waste too little for
  // smaller tiles to win, and a quarter of a round makes a single one of 128 x 128 tiles at most.
  const int n_tiles_n = (N + 255) / 256;
  if (static_cast<long long>(max_rows / 256) * n_tiles_n >= 3ll * cus) return false;
  if (K < 64 * kBK && 4 * (static_cast<long long>(max_rows) / 256 + E) * n_tiles_n <= cus) return true;
  // The 256-row tiles do 1.48 PFLOP/s inside a K step, the largest tile here 1.2: they win where they fill the chip
  // (FFN1 / FFN2, 256-row tiles and here: 8 experts of 3072 / 11008, 256 rows each: 184 and 230, 1024 rows of 768 / 3072:
  // 67 and 80 us), and lose where a few of them cannot (figures at the top; FFN2 of 16 experts of 2048 / 8192, 121 and
  // 200 rows each: 165 and 180 us there, 151 and 158 here).  Both forms are priced in microseconds for evenly popular
  // experts.  Their loads scatter, so a launch whose tiles fill a round, or two, just so may take one more: rounds are
  // an expectation over the tile counts.  Of 840 GEMMs timed in both forms (28 widths and numbers of experts, 32 to 700
  // rows each, means over three loads) the rule takes one that is over 4 % slower in 45, most of them by staying with the
  // 256-row tiles; rounding an expected count up did so in 57 and was up to 27 % slower than the 256-row tiles.  With
  // fragments read ahead and sums that start apart, both only here, the prices stayed: of 347 GEMMs (10 widths, 60 to 600
  // rows each, both weight layouts) 13 are over 4 % slower, 8 of them by staying with the 256-row tiles (20 % at most) and 5
  // [E, K, N] or short ones by leaving them (30 % at most: 61 rows of 4 of 3072 / 11008, FFN2, 73 cut along K and 95 here).
  // The weights, once, from HBM at 5.5 TB/s overlap with the steps, but not fully.
  const double used = E < max_rows ? E : max_rows, kt = K / kBK, weights = 2.0 * used * N * K / 5.5e6;
  const TileCount mt[2] = {m_tiles(max_rows, E, 64), m_tiles(max_rows, E, 128)};
  double key = 1e300, steps = 0;                                    // the shape that the kernel will choose
  for (int i = b_kn ? 1 : 0; i < kFewShapes; ++i) {
    if (b_kn && i % 3 == 0) continue;
    const int bm = 64 << (i / 3), bn = 64 << (i % 3);
    const double rounds = mean_rounds(mt[i / 3], (N + bn - 1) / bn, cus);
    if (rounds * (bm + bn) >= key) continue;
    key = rounds * (bm + bn);
    steps = rounds * (kt * kFewStepUs[i] + kFewEpiUs[epi == kFewPlain][i]);
  }
  const double mine = std::sqrt(steps * steps + weights * weights) + 5;
  // 256 x 256 tiles: 1.02 us a K step and the epilogue, fitted with the weights beside them (a step alone measures 1.2 to
  // 1.45 us); a last round of at most half the CUs is cut along K
  const TileCount big_mt = m_tiles(max_rows, E, 256);
  const double tile = kt * 1.02 + (epi == kFewPlain ? 5 : 15);
  if (kt >= 64) {
    const double rounds = big_mt.mean * n_tiles_n / cus, full = std::floor(rounds), part = rounds - full;
    double last = part > 0 ? tile : 0.0;
    if (part > 0 && part <= 0.5) {
      // the parts' steps, the reduction, and the partial tiles: fewer of them, and of their rows, with one or two rows
      // per expert (FFN2 of one token, top-2 of 8 experts of 4096 / 14336: 51 us cut, 60 here)
      const double rows = std::fmin(max_rows / used / 8, 1.0);
      const double cut = kt / std::fmin(std::floor(1 / part), 8.0) * 1.02 + 10 + 25 * rows + 42 * part;
      last = cut < tile ? cut : tile;
    }
    steps = full * tile + last;
  } else {
    steps = mean_rounds(big_mt, n_tiles_n, cus) * tile;
  }
  const double big = std::sqrt(steps * steps + weights * weights) + 5;
  return mine < 1.02 * big;
}

int few_rows_gemm(int mode, int places, FewArgs p, int epi, bool b_kn, bool in_layer, int cus, hipStream_t stream,
                  const char *what) {
  if (thin_rows_fits(mode, p.max_rows, p.E, p.N, p.K, epi, b_kn)) return thin_rows_gemm(p, epi, stream, what);
  p.force = mode >= 16 ? mode & 15 : -1;
  const double experts = std::ceil((in_layer ? kStreamBytes / 2 : kStreamBytes) / (2.0 * p.N * p.K));
  const bool large = experts <= (p.E < p.max_rows ? p.E : p.max_rows);
  p.stream_experts = large ? static_cast<int>(experts) : INT_MAX;
  p.rotate = places < 0 ? mode == 1 && starts_apart(p.max_rows, p.E, p.N, p.K) && !b_kn : places && can_start_apart(p.K) && !b_kn;
  const auto pick = [&](auto S_) -> void (*)(FewArgs) {
    constexpr bool S = decltype(S_)::value;
    if (b_kn) return epi == kFewPlain ? few_rows_kernel<kFewPlain, true, S> : few_rows_kernel<kFewGelu, true, S>;
    return epi == kFewPlain ? few_rows_kernel<kFewPlain, false, S>
                            : (epi == kFewGelu ? few_rows_kernel<kFewGelu, false, S> : few_rows_kernel<kFewGeluKeep, false, S>);
  };
  void (*kernel)(FewArgs) = large ? pick(std::true_type{}) : pick(std::false_type{});
  hipLaunchKernelGGL(kernel, dim3(cus), dim3(kFewThreads), 0, stream, p);
  return check_launch(what);
}

}  // namespace ccf
