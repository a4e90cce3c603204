// Top-k softmax gate for gfx950.
//
// logits[t, e] = sum_k x[t, k] * wg[e, k] + bg[e], then top-k and a softmax
// over the k selected logits (reference mix_moe/mix_moe/gates/naive_gate.py:31-38).
//
// The expert choice has to be reproducible bit for bit, so the fp32 sum is
// taken in one fixed order that a CPU can replay: K is cut into parts of 128
// consecutive elements (the last may be shorter); a part's sum starts at zero
// and takes its products one at a time in ascending K, acc = fma(x, w, acc);
// the part sums are added one after the other in ascending order, starting from
// the first; the bias is added last and the logit is rounded once to the input
// dtype.  The product of two fp16 values is exact in fp32, so for fp16 inputs
// the fused multiply-add is one rounding of acc + x*w however it is computed.
//
// That chain is what a K = 1 fp32 MFMA computes per output element
// (D = fma(A, B, C), round to nearest even: checked against fmaf chains on a
// CPU), so for fp16 inputs a wavefront runs it for a whole tile of tokens x
// experts at once: v_mfma_f32_32x32x1 (two 32 x 32 blocks) for more than 16
// experts, v_mfma_f32_16x16x1 (four 16 x 16 blocks) otherwise, one instruction
// per K element.  The blocks of an instruction are independent products, so a
// block is either another group of tokens or the same tokens on another part
// of K ("slot"): few tokens still fill the machine.  fp32 inputs keep multiply
// and add separate (two roundings): both on the vector unit, or with many tokens
// the multiplies as MFMAs onto zero.
#include "ccf_common.h"
#include "mfma_f32.h"
#include "plan.h"

#include <limits.h>
#include <type_traits>

namespace ccf {
int g_gate_waves = 8;    // most wavefronts of a gate workgroup (each takes other parts of K), 1..8
int g_gate_slots = 0;    // parts of K a wavefront works on at a time (1, 2, 4); 0 = by the token count
int g_gate_stream = -1;  // 1: every wavefront takes its tokens through all of K alone; 0: never; -1: with many tokens
namespace {

constexpr int kMaxTopK = 8;
constexpr int kPart = 128;          // K elements of a part
constexpr int kMaxWaves = 8;

template <typename T>
__device__ inline float round_to(float v) {
  return static_cast<float>(static_cast<T>(v));
}

__device__ inline bool better(float v, int id, float bv, int bid) {
  return v > bv || (v == bv && id < bid);
}

// The k best of a token so far (k <= KS), best first; ties keep the lower expert id.
template <int KS>
struct Best {
  float v[KS];
  int id[KS];
  __device__ inline void clear() {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      v[s] = -INFINITY;
      id[s] = INT_MAX;
    }
  }
  __device__ inline void offer(float nv, int nid, int k) {
    if constexpr (KS > 2) {                        // long lists: most offers end at the last kept entry
      float lv = v[0];
      int li = id[0];
#pragma unroll
      for (int s = 1; s < KS; ++s)
        if (s == k - 1) {
          lv = v[s];
          li = id[s];
        }
      if (!better(nv, nid, lv, li)) return;        // not among the k best
    }
    bool beats[KS];                                // short lists: no branch
#pragma unroll
    for (int s = 0; s < KS; ++s) beats[s] = better(nv, nid, v[s], id[s]);
#pragma unroll
    for (int s = KS - 1; s >= 0; --s) {
      if (s < k) {
        const int up = s > 0 ? s - 1 : 0;
        const bool ahead = s > 0 && beats[up];     // belongs further up: slot s takes its upper neighbour
        v[s] = ahead ? v[up] : (beats[s] ? nv : v[s]);
        id[s] = ahead ? id[up] : (beats[s] ? nid : id[s]);
      }
    }
  }
  // softmax over the k selected logits (slot 0 holds the maximum) and the writes
  template <typename T>
  __device__ inline void write(int t, int k, int64_t *__restrict__ idx_out, T *__restrict__ score_out) const {
    float ex[KS];
    float sum = 0.0f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      ex[s] = (s < k) ? expf(v[s] - v[0]) : 0.0f;
      sum += ex[s];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s < k) {
        idx_out[static_cast<size_t>(t) * k + s] = static_cast<int64_t>(id[s]);
        score_out[static_cast<size_t>(t) * k + s] = static_cast<T>(ex[s] / sum);
      }
    }
  }
};

// Leaves how many of the workgroup's token slots chose each expert, for the routing stage: the selection threads hold the
// ids, so the routing needs no pass of its own over idx to count them.  `row`: E ints of LDS that nothing else uses from
// here on; `mine`: this thread holds a token's list.  All threads of the workgroup call it, behind a barrier; with
// kFirstWave its first wavefront alone, which holds all lists, and the others make room for the next workgroup.  A list
// that NaN logits left short has entries that are no expert.
template <int KS, bool kFirstWave = false>
__device__ inline void leave_counts(const Best<KS> &best, bool mine, int k, int E, int *row, int32_t *__restrict__ wg_cnt) {
  const int step = kFirstWave ? 64 : static_cast<int>(blockDim.x);
  auto meet = [] {
    if constexpr (kFirstWave) {                      // a wavefront's LDS accesses happen in order
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    } else {
      __syncthreads();
    }
  };
  for (int e = threadIdx.x; e < E; e += step) row[e] = 0;
  meet();
  if (mine) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
      if (s < k && best.id[s] < E) atomicAdd(&row[best.id[s]], 1);
  }
  meet();
  for (int e = threadIdx.x; e < E; e += step) wg_cnt[static_cast<size_t>(blockIdx.x) * E + e] = row[e];
}

// Whether a gate of `wgs` workgroups of `wg_tokens` tokens leaves them: the table fits, and its rows tile the routing's
// chunks.  256 tokens of the stream form with eight experts each do not, nor does a top_k that is no power of two: the
// routing counts for itself then.
bool counts_fit(const int32_t *wg_cnt, long long wgs, int E, int wg_tokens, int k, long long max_cnt) {
  return wg_cnt && wgs * E <= max_cnt && kRouteChunk % (wg_tokens * k) == 0;
}

// fp16 gate.  An MFMA has 64 / N blocks; with S = 1 << LS slots, block b of a wavefront is
// token block b / S on slot b % S, so a wavefront covers TW = (64 / N / S) * N tokens and
// S parts of K at a time, and the wavefronts of a workgroup (all on the same TW tokens)
// cover waves * S parts per round.  Lane l of block b feeds row l % N of A with its
// token's x and column l % N of B with its expert's weights, zero where K, the tokens or
// the experts end (fma(0, 0, acc) = acc).
//
// A lane needs consecutive K of its own row, which is the opposite of a coalesced load, so
// the operands take the way through LDS: per stage of 32 K elements the wavefront fetches
// the 64 bytes of each of its 64 x rows and of its N*S weight rows with whole-line loads
// (four lanes per row), two stages ahead of their use, parks them in registers, and writes
// them into its own 10 KB of LDS one stage ahead; each lane then reads its row back in
// 16-byte pieces.  Only that wavefront touches the region, so the stage loop has no barrier.
//
// After a round the part sums wait in LDS (the same region) and are added in ascending part
// order onto the running sums; after the last round bias and rounding give the logits of one
// tile of N experts, of which one thread per token keeps the k best (k <= KS).
constexpr int kStageK = 32;                        // K elements of a stage
constexpr int kRowBytes = 80;                      // a row's 64 bytes of a stage + 16: bank spread
constexpr int kTileBytes = 64 * kRowBytes;         // one operand of a stage
constexpr int kRegionFloats = 2 * kTileBytes / 4;  // a wavefront's LDS: two operand tiles, later its part sums

template <int N, int LS, int KS>
__global__ void __launch_bounds__(kMaxWaves * 64)
gate_mfma_kernel(const half_t *__restrict__ x, const half_t *__restrict__ wg, const half_t *__restrict__ bg,
                 int tokens, int d, int E, int k, int64_t *__restrict__ idx_out,
                 half_t *__restrict__ score_out, half_t *__restrict__ logits_out, int32_t *__restrict__ wg_cnt) {
  using M = Mfma<N>;
  constexpr int kBlocks = 64 / N;
  constexpr int S = 1 << LS;
  static_assert(S <= kBlocks, "a slot is a block");
  constexpr int TW = (kBlocks / S) * N;            // tokens of a workgroup
  constexpr int kWLoads = N * S / 16;              // load instructions for the weight rows of a stage
  constexpr int kLd = N + 1;                       // row stride of the logit tile in LDS (bank spread)
  static_assert(64 * N * 4 <= kRegionFloats * 4, "part sums of a wavefront fit its region");
  extern __shared__ float s_mem[];
  const int waves = blockDim.x >> 6;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  float *region = s_mem + static_cast<size_t>(wave) * kRegionFloats;
  float *s_total = s_mem + static_cast<size_t>(waves) * kRegionFloats;   // [TW][kLd] running sums, then logits
  const int t0 = blockIdx.x * TW;
  const int nparts = (d + kPart - 1) / kPart;
  const int per_round = waves * S;
  const int rounds = (nparts + per_round - 1) / per_round;

  // as a reader: my block, row, slot
  const int blk = lane / N, r = lane % N;
  const int slot = blk & (S - 1);
  char *tile = reinterpret_cast<char *>(region);
  const char *my_x = tile + lane * kRowBytes;                              // x row of lane l is row l of the tile
  const char *my_w = tile + kTileBytes + (slot * N + r) * kRowBytes;       // weight rows: slot-major

  // as a loader: four lanes per row, 16 rows per instruction
  const int l_row = lane >> 2, l_piece = lane & 3;
  char *park_at = tile + l_row * kRowBytes + l_piece * 16;
  const half_t *x_src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int lr = 16 * i + l_row;
    int t = t0 + ((lr / N) >> LS) * N + lr % N;
    t = t < tokens ? t : tokens - 1;               // rows past the end repeat the last token
    x_src[i] = x + static_cast<size_t>(t) * d + (((lr / N) & (S - 1)) * kPart + l_piece * 8);
  }

  Best<KS> best;
  best.clear();

  for (int e0 = 0; e0 < E; e0 += N) {              // tiles of N experts
    const bool has_w = e0 + r < E;
    // the bias of the column this thread finishes (the same for all its elements: the
    // workgroup size is a multiple of N), asked for before the long part
    float my_bias = 0.0f;
    if (bg && e0 + static_cast<int>(threadIdx.x) % N < E) my_bias = static_cast<float>(bg[e0 + threadIdx.x % N]);
    const half_t *w_src[kWLoads];
#pragma unroll
    for (int i = 0; i < kWLoads; ++i) {
      const int wr = 16 * i + l_row;
      int e = e0 + wr % N;
      e = e < E ? e : E - 1;
      w_src[i] = wg + static_cast<size_t>(e) * d + ((wr / N) * kPart + l_piece * 8);
    }
    for (int rd = 0; rd < rounds; ++rd) {
      const int part0 = rd * per_round + wave * S;               // this wavefront's first part of the round
      if (part0 < nparts) {                        // uniform per wavefront
        int left = d - part0 * kPart;                            // the wavefront's first part is its longest
        left = left < kPart ? left : kPart;
        const int stages = (left + kStageK - 1) / kStageK;       // 1..4
        const int k0 = part0 * kPart;
        const int k_mine = k0 + slot * kPart;                    // where this lane's part starts (may be past d)
        typename M::Acc acc;
#pragma unroll
        for (int v = 0; v < M::kRegs; ++v) acc[v] = 0.0f;

        // Loads of stage s: every lane loads (from the start of the tensor where K has
        // ended) and unwanted pieces become zero when they are used, so there is no branch
        // around a load and the number of loads in flight is known where the waits go.
        int4v xa[4], wa[kWLoads], xb[4], wb[kWLoads];
        auto fetch = [&](int s, int4v (&xv)[4], int4v (&wv)[kWLoads]) {
          const int ks = k0 + s * kStageK;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int kx = ks + (((16 * i + l_row) / N) & (S - 1)) * kPart + l_piece * 8;
            xv[i] = *reinterpret_cast<const int4v *>(kx < d ? x_src[i] + ks : x);
          }
#pragma unroll
          for (int i = 0; i < kWLoads; ++i) {
            const int kw = ks + ((16 * i + l_row) / N) * kPart + l_piece * 8;
            wv[i] = *reinterpret_cast<const int4v *>(kw < d ? w_src[i] + ks : wg);
          }
        };
        auto park = [&](const int4v (&xv)[4], const int4v (&wv)[kWLoads]) {
#pragma unroll
          for (int i = 0; i < 4; ++i) *reinterpret_cast<int4v *>(park_at + 16 * i * kRowBytes) = xv[i];
#pragma unroll
          for (int i = 0; i < kWLoads; ++i)
            *reinterpret_cast<int4v *>(park_at + kTileBytes + 16 * i * kRowBytes) = wv[i];
        };
        auto take = [&](int c, half8 &vx, half8 &vw) {
          vx = *reinterpret_cast<const half8 *>(my_x + c * 16);
          vw = *reinterpret_cast<const half8 *>(my_w + c * 16);
        };
        auto run = [&](int s, int c, const half8 &vx, const half8 &vw) {
          const bool in = k_mine + s * kStageK + c * 8 < d;
          const half8 zero = {};
          const half8 xs = in ? vx : zero;
          const half8 ws = (in && has_w) ? vw : zero;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            acc = M::run(static_cast<float>(xs[j]), static_cast<float>(ws[j]), acc);
        };
        // One stage: its four pieces are read back two at a time; once the last read is on
        // its way (the LDS works in order) the next stage's operands overwrite the tiles
        // and the loads of the stage after that leave.  The scheduling barriers keep loads
        // and LDS traffic where they are written: left alone, the scheduler sinks each
        // load to just before its use.
        half8 ax, aw, bx, bw;
#define CCF_GATE_STAGE(s, PARK_NEXT)                                   \
  do {                                                                 \
    take(0, ax, aw);                                                   \
    take(1, bx, bw);                                                   \
    __builtin_amdgcn_sched_barrier(0);                                 \
    run(s, 0, ax, aw);                                                 \
    __builtin_amdgcn_sched_barrier(0);                                 \
    take(2, ax, aw);                                                   \
    __builtin_amdgcn_sched_barrier(0);                                 \
    run(s, 1, bx, bw);                                                 \
    __builtin_amdgcn_sched_barrier(0);                                 \
    take(3, bx, bw);                                                   \
    __builtin_amdgcn_sched_barrier(0);                                 \
    PARK_NEXT;                                                         \
    __builtin_amdgcn_sched_barrier(0);                                 \
    run(s, 2, ax, aw);                                                 \
    run(s, 3, bx, bw);                                                 \
    __builtin_amdgcn_sched_barrier(0);                                 \
  } while (0)
        fetch(0, xa, wa);
        fetch(1, xb, wb);
        __builtin_amdgcn_sched_barrier(0);
        park(xa, wa);                              // stage 0
        fetch(2, xa, wa);
        __builtin_amdgcn_sched_barrier(0);
        CCF_GATE_STAGE(0, park(xb, wb); fetch(3, xb, wb));
        if (stages > 1) {
          CCF_GATE_STAGE(1, park(xa, wa));
          if (stages > 2) {
            CCF_GATE_STAGE(2, park(xb, wb));
            if (stages > 3) CCF_GATE_STAGE(3, (void)0);
          }
        }
#undef CCF_GATE_STAGE
        // part sums into the same region, [slot][token][expert]
#pragma unroll
        for (int v = 0; v < M::kRegs; ++v) {
          const int ob = M::block(v);
          region[(static_cast<size_t>(ob & (S - 1)) * TW + (ob >> LS) * N + M::row(v, lane)) * N + r] = acc[v];
        }
      }
      __syncthreads();
      // running sums: the parts of this round in ascending order.  The part sums are read
      // eight at a time ahead of the additions, which stay one chain in part order.
      int np_round = nparts - rd * per_round;
      np_round = np_round < per_round ? np_round : per_round;
      for (int i = threadIdx.x; i < TW * N; i += blockDim.x) {
        const int tok = i / N, col = i % N;
        float t = rd == 0 ? 0.0f : s_total[tok * kLd + col];
        for (int q0 = 0; q0 < np_round; q0 += 8) {
          float ps[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            int q = q0 + u;
            q = q < np_round ? q : np_round - 1;
            ps[u] = s_mem[static_cast<size_t>(q >> LS) * kRegionFloats + (q & (S - 1)) * TW * N + i];
          }
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            const float sum = (rd == 0 && q0 + u == 0) ? ps[u] : t + ps[u];   // the first part starts the chain
            t = q0 + u < np_round ? sum : t;
          }
        }
        if (rd == rounds - 1) {
          const int e = e0 + col;
          if (e < E) {
            if (bg) t = t + my_bias;
            t = round_to<half_t>(t);
            if (logits_out && t0 + tok < tokens)
              logits_out[static_cast<size_t>(t0 + tok) * E + e] = static_cast<half_t>(t);
          }
        }
        s_total[tok * kLd + col] = t;
      }
      __syncthreads();
    }
    // one thread per token: the logits of this tile, ascending expert id
    if (threadIdx.x < TW && t0 + threadIdx.x < tokens) {
      const float *lg = s_total + threadIdx.x * kLd;
      const int ne = (E - e0) < N ? (E - e0) : N;
#pragma unroll
      for (int c0 = 0; c0 < N; c0 += 8) {          // eight logits read ahead of their offers
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = lg[c0 + u];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (c0 + u < ne) best.offer(v[u], e0 + c0 + u, k);
      }
    }
    // s_total is next written after the next tile's first barrier, which these threads reach later
  }
  if (threadIdx.x < TW && t0 + threadIdx.x < tokens)
    best.template write<half_t>(t0 + threadIdx.x, k, idx_out, score_out);
  // the wavefronts' regions are free since the last barrier
  if (wg_cnt) leave_counts<KS>(best, threadIdx.x < TW && t0 + threadIdx.x < tokens, k, E, reinterpret_cast<int *>(s_mem), wg_cnt);
}

// fp16 gate for many tokens: every wavefront works alone.  It takes TW tokens through all of
// K, S parts at a time ("round": 4 stages), in one unbroken stream of stages: the loads run
// five stages ahead of the MFMAs in four sets of registers, each set parked in the
// wavefront's LDS one stage ahead of its use, so after the first arrival the matrix pipe
// does not wait for memory again.  At the end of a round the part sums, which are registers
// of this lane, go onto the running sums in ascending part order; the logits of a tile of N
// experts pass through the wavefront's LDS once, for the selection (one lane per token) and
// the coalesced write.  No barrier before the expert counts of the workgroup.
constexpr int kStreamWaves = 4;

template <int N, int LS, int KS>
__global__ void __launch_bounds__(kStreamWaves * 64)
gate_stream_kernel(const half_t *__restrict__ x, const half_t *__restrict__ wg, const half_t *__restrict__ bg,
                   int tokens, int d, int E, int k, int64_t *__restrict__ idx_out,
                   half_t *__restrict__ score_out, half_t *__restrict__ logits_out, int32_t *__restrict__ wg_cnt) {
  using M = Mfma<N>;
  constexpr int kBlocks = 64 / N;
  constexpr int S = 1 << LS;
  static_assert(S <= kBlocks, "a slot is a block");
  constexpr int TB = kBlocks / S;                  // token blocks of a wavefront
  constexpr int TW = TB * N;                       // its tokens
  constexpr int RB = M::kRegs / kBlocks;           // accumulator registers of a block
  constexpr int kWLoads = N * S / 16;
  constexpr int kLd = N + 1;
  static_assert(TW * kLd <= kRegionFloats, "the logits of a tile fit the wavefront's region");
  extern __shared__ float s_mem[];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  float *region = s_mem + static_cast<size_t>(wave) * kRegionFloats;
  const int t0 = (blockIdx.x * kStreamWaves + wave) * TW;
  const int nparts = (d + kPart - 1) / kPart;
  const int rounds = (nparts + S - 1) / S;
  const bool ragged = d % (S * kPart) != 0;        // the last round has K elements to leave out

  const int blk = lane / N, r = lane % N;
  const int slot = blk & (S - 1);
  char *tile = reinterpret_cast<char *>(region);
  const char *my_x = tile + lane * kRowBytes;
  const char *my_w = tile + kTileBytes + (slot * N + r) * kRowBytes;
  const int l_row = lane >> 2, l_piece = lane & 3;
  char *park_at = tile + l_row * kRowBytes + l_piece * 16;

  Best<KS> best;
  best.clear();
  if (t0 < tokens) {                               // uniform per wavefront
    const half_t *x_src[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int lr = 16 * i + l_row;
      int t = t0 + ((lr / N) >> LS) * N + lr % N;
      t = t < tokens ? t : tokens - 1;
      x_src[i] = x + static_cast<size_t>(t) * d + (((lr / N) & (S - 1)) * kPart + l_piece * 8);
    }
    for (int e0 = 0; e0 < E; e0 += N) {
      // columns past the last expert repeat its weights; nothing reads their logits
      const bool has_w = e0 + r < E;
      float my_bias = 0.0f;
      if (bg && has_w) my_bias = static_cast<float>(bg[e0 + r]);
      const half_t *w_src[kWLoads];
#pragma unroll
      for (int i = 0; i < kWLoads; ++i) {
        const int wr = 16 * i + l_row;
        int e = e0 + wr % N;
        e = e < E ? e : E - 1;
        w_src[i] = wg + static_cast<size_t>(e) * d + ((wr / N) * kPart + l_piece * 8);
      }
      // stage g of the stream: round g / 4, K offset of the round's first part + (g % 4) * kStageK
      auto stage_k = [&](int g) { return (g >> 2) * (S * kPart) + (g & 3) * kStageK; };
      typedef int4v XSet[4];
      typedef int4v WSet[kWLoads];
      XSet xa, xb, xc, xd;
      WSet wa, wb, wc, wd;
      auto fetch = [&](int g, XSet &xv, WSet &wv) {   // past the end of K the loads read the start of x and wg
        const int ks = stage_k(g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kx = ks + (((16 * i + l_row) / N) & (S - 1)) * kPart + l_piece * 8;
          xv[i] = *reinterpret_cast<const int4v *>(kx < d ? x_src[i] + ks : x);
        }
#pragma unroll
        for (int i = 0; i < kWLoads; ++i) {
          const int kw = ks + ((16 * i + l_row) / N) * kPart + l_piece * 8;
          wv[i] = *reinterpret_cast<const int4v *>(kw < d ? w_src[i] + ks : wg);
        }
      };
      auto park = [&](const XSet &xv, const WSet &wv) {
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<int4v *>(park_at + 16 * i * kRowBytes) = xv[i];
#pragma unroll
        for (int i = 0; i < kWLoads; ++i)
          *reinterpret_cast<int4v *>(park_at + kTileBytes + 16 * i * kRowBytes) = wv[i];
      };
      auto take = [&](int c, half8 &vx, half8 &vw) {
        vx = *reinterpret_cast<const half8 *>(my_x + c * 16);
        vw = *reinterpret_cast<const half8 *>(my_w + c * 16);
      };
      typename M::Acc acc;
      // A piece is 8 K elements of a stage.  Its MFMAs run on fp32 copies made during the piece
      // before, in registers that no MFMA in flight reads: a conversion into a register that the
      // running MFMA still reads waits for that MFMA, and one wavefront per SIMD has nothing to
      // cover the wait with.
      auto convert = [&](auto rag, int g, int c, const half8 &vx, const half8 &vw, float (&fx)[8], float (&fw)[8]) {
        half8 xs = vx, ws = vw;
        if constexpr (decltype(rag)::value) {      // K ends inside a round: what lies past it counts as zero
          const bool in = stage_k(g) + slot * kPart + c * 8 < d;
          const half8 zero = {};
          xs = in ? vx : zero;
          ws = in ? vw : zero;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          fx[j] = static_cast<float>(xs[j]);
          fw[j] = static_cast<float>(ws[j]);
        }
      };
      auto mma = [&](const float (&fx)[8], const float (&fw)[8]) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = M::run(fx[j], fw[j], acc);
      };
      float total[TB * RB];
      half8 ax, aw, bx, bw;                        // pieces as read from LDS: even ones in a, odd ones in b
      float fax[8], faw[8], fbx[8], fbw[8];        // their fp32 copies
      // eight MFMAs with the next piece's conversions between them
#define CCF_GATE_PIECE(MMA_F, G, C, RAW, CONV_F)                       \
  do {                                                                 \
    __builtin_amdgcn_sched_barrier(0);                                 \
    mma(MMA_F##x, MMA_F##w);                                           \
    convert(rag, G, C, RAW##x, RAW##w, CONV_F##x, CONV_F##w);          \
    _Pragma("unroll") for (int q_ = 0; q_ < 8; ++q_) {                 \
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               \
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);               \
    }                                                                  \
    __builtin_amdgcn_sched_barrier(0);                                 \
  } while (0)
      // One stage, entered with piece 0 converted (fa) and piece 1 read (b).  Reads from LDS
      // run two pieces ahead, conversions one; the next stage is parked once this stage's last
      // read is on its way (the LDS works in order), and its first pieces are read behind that.
#define CCF_GATE_STAGE(g, PARK_NEXT)                                   \
  do {                                                                 \
    take(2, ax, aw);                                                   \
    CCF_GATE_PIECE(fa, g, 1, b, fb);                                   \
    take(3, bx, bw);                                                   \
    __builtin_amdgcn_sched_barrier(0);                                 \
    PARK_NEXT;                                                         \
    CCF_GATE_PIECE(fb, g, 2, a, fa);                                   \
    take(0, ax, aw);                                                   \
    CCF_GATE_PIECE(fa, g, 3, b, fb);                                   \
    take(1, bx, bw);                                                   \
    CCF_GATE_PIECE(fb, (g) + 1, 0, a, fa);                             \
  } while (0)
      auto all_rounds = [&](auto rag) {
      asm volatile("" ::: "memory");               // the tile is free: the previous expert tile's logits have been read
      fetch(0, xa, wa);
      fetch(1, xb, wb);
      fetch(2, xc, wc);
      fetch(3, xd, wd);
      __builtin_amdgcn_sched_barrier(0);
      park(xa, wa);                                // stage 0
      fetch(4, xa, wa);
      __builtin_amdgcn_sched_barrier(0);
      take(0, ax, aw);
      take(1, bx, bw);
      convert(rag, 0, 0, ax, aw, fax, faw);
      __builtin_amdgcn_sched_barrier(0);
      for (int rd = 0; rd < rounds; ++rd) {
        const int g = 4 * rd;
#pragma unroll
        for (int v = 0; v < M::kRegs; ++v) acc[v] = 0.0f;
        CCF_GATE_STAGE(g, park(xb, wb); fetch(g + 5, xb, wb));
        CCF_GATE_STAGE(g + 1, park(xc, wc); fetch(g + 6, xc, wc));
        CCF_GATE_STAGE(g + 2, park(xd, wd); fetch(g + 7, xd, wd));
        if (rd + 1 < rounds)
          CCF_GATE_STAGE(g + 3, park(xa, wa); fetch(g + 8, xa, wa));
        else
          CCF_GATE_STAGE(g + 3, (void)0);            // its reads ahead find the last stage again; nothing uses them
        // the round's part sums onto the running sums, ascending part order
#pragma unroll
        for (int tb = 0; tb < TB; ++tb)
#pragma unroll
          for (int sl = 0; sl < S; ++sl) {
            const int p = rd * S + sl;
            if (p < nparts) {
#pragma unroll
              for (int j = 0; j < RB; ++j) {
                const float ps = acc[(tb * S + sl) * RB + j];
                total[tb * RB + j] = p == 0 ? ps : total[tb * RB + j] + ps;
              }
            }
          }
      }
      };
      if (ragged) all_rounds(std::true_type{}); else all_rounds(std::false_type{});
#undef CCF_GATE_PIECE
#undef CCF_GATE_STAGE
      // logits of the tile: bias, one rounding, into the wavefront's LDS as [token][expert]
      asm volatile("" ::: "memory");
#pragma unroll
      for (int j = 0; j < TB * RB; ++j) {
        float t = total[j];
        if (has_w) {
          if (bg) t = t + my_bias;
          t = round_to<half_t>(t);
        }
        region[((j / RB) * N + M::row(j % RB, lane)) * kLd + r] = t;
      }
      asm volatile("" ::: "memory");
      __builtin_amdgcn_wave_barrier();
      if (logits_out) {
        for (int i = lane; i < TW * N; i += 64) {
          const int tok = i / N, col = i % N;
          if (e0 + col < E && t0 + tok < tokens)
            logits_out[static_cast<size_t>(t0 + tok) * E + e0 + col] = static_cast<half_t>(region[tok * kLd + col]);
        }
      }
      if (lane < TW && t0 + lane < tokens) {
        const float *lg = region + lane * kLd;
        const int ne = (E - e0) < N ? (E - e0) : N;
#pragma unroll
        for (int c0 = 0; c0 < N; c0 += 8) {
          float v[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) v[u] = lg[c0 + u];
#pragma unroll
          for (int u = 0; u < 8; ++u)
            if (c0 + u < ne) best.offer(v[u], e0 + c0 + u, k);
        }
      }
    }
    if (lane < TW && t0 + lane < tokens) best.template write<half_t>(t0 + lane, k, idx_out, score_out);
  }
  if (wg_cnt) {
    __syncthreads();
    leave_counts<KS>(best, lane < TW && t0 + lane < tokens, k, E, reinterpret_cast<int *>(s_mem), wg_cnt);
  }
}

// fp32 gate on the vector unit.  Each product is rounded before it is added, which an accumulating MFMA does not do, so
// the floor is two vector instructions per product: 4096 tokens x 64 experts x 2048 are 16.8 M wavefront instructions,
// 16 K per SIMD, ~20 us at the issue rate of a few wavefronts per SIMD.  What the kernel has to do is feed them:
//
// * A wavefront computes a tile of 8 TT tokens x 8 EE experts over one part of K (lane l: tokens l / 8 + 8 i,
//   experts l % 8 + 8 j), so four K elements of TT + EE rows read from LDS feed 8 TT EE instructions (8 reads for 128
//   and 10 for 128 at the largest tiles, 32 x 32 and 16 x 64; more tokens of more than 32 experts are
//   gate_f32_mfma_kernel's).  The wavefronts of a workgroup take different parts of the same tile.
// * Operands come in stages of 16 K elements: four lanes per row fetch its 64 bytes a stage ahead into registers,
//   which go into the other half of the wavefront's own LDS behind the stage's arithmetic: no barrier in the loop.
// * Rows are 80 bytes apart: the eight rows that a read touches start 20 banks apart, none in conflict.
// * Behind a round of parts their sums meet in LDS and are added in ascending order onto the running sums.
//
// TT shrinks with the tokens, so that 2049 and 4097 tokens still make 129 workgroups, EE with the experts.
// 4096 tokens x 2048, 64 experts, top-2: 42 us; 8192 x 2048, 32 experts: 39 us.
constexpr int kF32StageK = 16;                     // K elements of a stage
constexpr int kF32Row = kF32StageK + 4;            // row stride in LDS, floats

template <int TT, int EE>
struct GateF32Tile {
  static constexpr int WT = 8 * TT, WE = 8 * EE;   // tokens and experts of a tile
  static constexpr int ROWS = WT + WE;
  static constexpr int LOADS = (ROWS + 15) / 16;   // 16 rows per load instruction of a wavefront
  static constexpr int BUF = LOADS * 16 * kF32Row; // one stage, floats
  static constexpr int LD = WE + 1;                // row stride of the part sums and of the logits
  static constexpr int REGION = 2 * BUF > WT * LD ? 2 * BUF : WT * LD;   // a wavefront's LDS, floats
};

template <int KS>
__device__ inline void gate_f32_select(const float *row, int e0, int ne, int k, Best<KS> &best) {
  for (int e = 0; e < ne; ++e) best.offer(row[e], e0 + e, k);
}

template <int TT, int EE, int KS>
__global__ void __launch_bounds__(kMaxWaves * 64)
gate_f32_kernel(const float *__restrict__ x, const float *__restrict__ wg, const float *__restrict__ bg,
                int tokens, int d, int E, int k, int64_t *__restrict__ idx_out,
                float *__restrict__ score_out, float *__restrict__ logits_out, int32_t *__restrict__ wg_cnt) {
#pragma clang fp contract(off)
  using C = GateF32Tile<TT, EE>;
  extern __shared__ float s_mem[];
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  float *region = s_mem + static_cast<size_t>(wave) * C::REGION;
  float *s_logit = s_mem + static_cast<size_t>(waves) * C::REGION;       // [WT][LD] running sums, then logits
  const int t0 = blockIdx.x * C::WT;
  const int nparts = (d + kPart - 1) / kPart;
  const int l_row = lane >> 2, l_piece = lane & 3;                       // as a loader
  const int my_t = lane >> 3, my_e = lane & 7;                           // as a reader
  Best<KS> best;
  best.clear();
  for (int e0 = 0; e0 < E; e0 += C::WE) {
    // rows of this lane's loads: the tile's tokens, then its experts (past the end: a repeated row, never used)
    const float *src[C::LOADS];
#pragma unroll
    for (int i = 0; i < C::LOADS; ++i) {
      const int r = 16 * i + l_row;
      const int t = t0 + r < tokens ? t0 + r : tokens - 1;
      int e = e0 + r - C::WT;
      e = e < 0 ? 0 : (e < E ? e : E - 1);
      src[i] = (r < C::WT ? x + static_cast<size_t>(t) * d : wg + static_cast<size_t>(e) * d) + l_piece * 4;
    }
    for (int p0 = 0; p0 < nparts; p0 += waves) {
      const int part = p0 + wave;
      float acc[TT][EE];
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < EE; ++j) acc[i][j] = 0.0f;
      if (part < nparts) {                                               // uniform per wavefront
        const int k_lo = part * kPart;
        const int k_hi = k_lo + kPart < d ? k_lo + kPart : d;
        float4v reg[C::LOADS];
        // K past the part's end reads as zero, which adds nothing (a running sum is never -0)
        auto fetch = [&](int kk) {
          const bool in = kk + l_piece * 4 < k_hi;                       // d is a multiple of 8
#pragma unroll
          for (int i = 0; i < C::LOADS; ++i) {
            const float4v zero = {0.0f, 0.0f, 0.0f, 0.0f};
            reg[i] = in ? *reinterpret_cast<const float4v *>(src[i] + kk) : zero;
          }
        };
        auto park = [&](float *buf) {
#pragma unroll
          for (int i = 0; i < C::LOADS; ++i)
            *reinterpret_cast<float4v *>(buf + (16 * i + l_row) * kF32Row + l_piece * 4) = reg[i];
        };
        fetch(k_lo);
        park(region);
        int half = 0;
        for (int kk = k_lo; kk < k_hi; kk += kF32StageK) {
          const bool more = kk + kF32StageK < k_hi;
          if (more) fetch(kk + kF32StageK);
          const float *buf = region + half * C::BUF;
          // four K elements at a time, the next four read from LDS ahead of their use; the empty asm keeps
          // it at that: left alone, the compiler reads the whole stage up front and spills
          float4v xv[2][TT], wv[2][EE];
          auto take = [&](int c, float4v (&xr)[TT], float4v (&wr)[EE]) {
#pragma unroll
            for (int i = 0; i < TT; ++i) xr[i] = *reinterpret_cast<const float4v *>(buf + (my_t + 8 * i) * kF32Row + c);
#pragma unroll
            for (int j = 0; j < EE; ++j)
              wr[j] = *reinterpret_cast<const float4v *>(buf + (C::WT + my_e + 8 * j) * kF32Row + c);
          };
          take(0, xv[0], wv[0]);
#pragma unroll
          for (int c = 0; c < kF32StageK / 4; ++c) {
            asm volatile("" ::: "memory");
            if (c + 1 < kF32StageK / 4) take(4 * (c + 1), xv[(c + 1) & 1], wv[(c + 1) & 1]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
              for (int i = 0; i < TT; ++i)
#pragma unroll
                for (int j = 0; j < EE; ++j) {
                  const float prod = xv[c & 1][i][q] * wv[c & 1][j][q];
                  acc[i][j] = acc[i][j] + prod;
                }
#pragma unroll
            for (int i = 0; i < TT; ++i)
#pragma unroll
              for (int j = 0; j < EE; ++j) asm volatile("" : "+v"(acc[i][j]));
          }
          half ^= 1;
          if (more) park(region + half * C::BUF);
        }
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
          for (int j = 0; j < EE; ++j) region[(my_t + 8 * i) * C::LD + my_e + 8 * j] = acc[i][j];
      }
      __syncthreads();
      const int np = nparts - p0 < waves ? nparts - p0 : waves;
      const bool last = p0 + waves >= nparts;
      for (int o = threadIdx.x; o < C::WT * C::WE; o += blockDim.x) {
        const int t = o / C::WE, e = o % C::WE;
        const int at = t * C::LD + e;
        float s = p0 == 0 ? s_mem[at] : s_logit[at] + s_mem[at];
        for (int w = 1; w < np; ++w) s = s + s_mem[static_cast<size_t>(w) * C::REGION + at];
        if (last && e0 + e < E) {
          if (bg) s = s + bg[e0 + e];
          if (logits_out && t0 + t < tokens) logits_out[static_cast<size_t>(t0 + t) * E + e0 + e] = s;
        }
        s_logit[at] = s;
      }
      __syncthreads();
    }
    if (threadIdx.x < C::WT)
      gate_f32_select<KS>(s_logit + threadIdx.x * C::LD, e0, (E - e0) < C::WE ? (E - e0) : C::WE, k, best);
    // the next tile's logits are written behind the barrier that follows its first round's part sums
  }
  if (threadIdx.x < C::WT && t0 + threadIdx.x < tokens) best.template write<float>(t0 + threadIdx.x, k, idx_out, score_out);
  static_assert(C::REGION >= (EE >= 8 ? 1024 : 8 * EE), "a count per expert");
  // the first wavefront alone where a CU goes through several workgroups (as few as one of 8 tokens take 0.6 us longer with it)
  constexpr bool kMany = TT == 4;
  static_assert(C::WT <= 64, "lists in the first wavefront");
  if (wg_cnt && (!kMany || threadIdx.x < 64))
    leave_counts<KS, kMany>(best, threadIdx.x < C::WT && t0 + threadIdx.x < tokens, k, E, reinterpret_cast<int *>(s_mem), wg_cnt);
}

template <int TT, int EE>
int launch_gate_f32(const float *x, const float *wg, const float *bg, int tokens, int d, int E, int k, int64_t *idx_out,
                    float *score_out, float *logits_out, hipStream_t stream, int32_t *wg_cnt, long long max_cnt, int *tokens_per_wg) {
  using C = GateF32Tile<TT, EE>;
  const int nparts = (d + kPart - 1) / kPart;
  const int waves = nparts < kMaxWaves ? nparts : kMaxWaves;
  const size_t lds = sizeof(float) * (static_cast<size_t>(waves) * C::REGION + C::WT * C::LD);
  static_assert(sizeof(float) * (kMaxWaves * C::REGION + C::WT * C::LD) <= 160 * 1024, "LDS of a CU");
  auto kern = k <= 2 ? gate_f32_kernel<TT, EE, 2> : gate_f32_kernel<TT, EE, kMaxTopK>;
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(lds));
    if (e != hipSuccess) return fail(CCF_ERR_HIP, "gate: LDS attribute: %s", hipGetErrorString(e));
  }
  const int wgs = (tokens + C::WT - 1) / C::WT;
  if (!counts_fit(wg_cnt, wgs, E, C::WT, k, max_cnt)) wg_cnt = nullptr;
  if (wg_cnt && tokens_per_wg) *tokens_per_wg = C::WT;
  hipLaunchKernelGGL(kern, dim3(wgs), dim3(waves * 64), lds, stream, x, wg, bg, tokens, d, E, k,
                     idx_out, score_out, logits_out, wg_cnt);
  return check_launch("gate_f32_kernel");
}

template <int TT>
int launch_gate_f32_experts(const float *x, const float *wg, const float *bg, int tokens, int d, int E, int k,
                            int64_t *idx_out, float *score_out, float *logits_out, hipStream_t stream, int32_t *wg_cnt,
                            long long max_cnt, int *tokens_per_wg) {
  auto launch = E <= 8 ? launch_gate_f32<TT, 1> : (E <= 16 ? launch_gate_f32<TT, 2> : launch_gate_f32<TT, 4>);
  if constexpr (TT < 4) {                          // more tokens of more than 32 experts: gate_f32_on_mfma()
    if (E > 32) launch = launch_gate_f32<TT, 8>;
  }
  return launch(x, wg, bg, tokens, d, E, k, idx_out, score_out, logits_out, stream, wg_cnt, max_cnt, tokens_per_wg);
}

// The same order with the products on the matrix cores: fma(x, w, 0) of a K = 1 MFMA is the rounded product, subnormal
// ones included, for 2048 token-expert pairs in 64 cycles, and the vector unit has one addition per product left
// instead of two instructions.  (A product of -0 comes out as +0, which no running sum can tell: it starts at +0 and is
// never -0.)  They come one after the other, also with two wavefronts on a SIMD: a step takes 30 ns for the MFMA and 40
// for its 32 additions, against 80 for 64 vector instructions, and two LDS reads feed 32 of them instead of three.  (By the
// counters of the 8192 tokens below the matrix pipe is busy 26 % of the time and the vector unit 45 to 60.)
//
// * A wavefront computes 32 tokens x 64 experts (64 x 32, 64 x 16 for fewer experts) over one part of K, one product
//   tile ahead of the additions; the wavefronts of a workgroup take different parts of the same tile.
// * Operands come in stages of 16 K elements through the wavefront's own LDS, as above, into one buffer: a
//   wavefront's LDS accesses happen in order, so its writes of the next stage land behind its reads of this one.
//   The last stage of a part loads the first of the wavefront's next part.
// * LDS holds the part sums of two turns of the wavefronts (`turns`), so they meet at a barrier every second part: 8192
//   tokens x 2048, 64 experts 50.7 -> 48.8 us, x 4096 89.1 -> 86.3; 30000 x 3000, 48 experts 253 -> 243.
// * Eight threads select a token's experts (one per token: 4 us of 64 experts).
//
// On the vector unit and so, first form: 8192 tokens x 2048, 64 experts, top-2: 64 and 49 us; x 4096: 116 and 92; 32768 x
// 2048, 32 experts: 141 and 96.
template <int N, int WE>
struct GateF32Mfma {
  static constexpr int WT = 64 / N * N * N / WE;   // tokens of a tile
  static constexpr int ROWS = WT + WE;
  static constexpr int LOADS = (ROWS + 15) / 16;
  static constexpr int BUF = LOADS * 16 * kF32Row;
  static constexpr int LD = WE + 1;
  static constexpr int REGION = BUF > WT * LD ? BUF : WT * LD;           // a wavefront's LDS, floats
};

template <int N, int WE, int KS>
__global__ void __launch_bounds__(kMaxWaves * 64)
gate_f32_mfma_kernel(const float *__restrict__ x, const float *__restrict__ wg, const float *__restrict__ bg,
                     int tokens, int d, int E, int k, int64_t *__restrict__ idx_out,
                     float *__restrict__ score_out, float *__restrict__ logits_out, int32_t *__restrict__ wg_cnt, int turns) {
#pragma clang fp contract(off)
  using C = GateF32Mfma<N, WE>;
  using M = Mfma<N>;
  extern __shared__ float s_mem[];
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int held = waves * turns;                                        // parts whose sums LDS holds at a time
  float *s_logit = s_mem + static_cast<size_t>(held) * C::REGION;        // [WT][LD] running sums, then logits
  const int t0 = blockIdx.x * C::WT;
  const int nparts = (d + kPart - 1) / kPart;
  const int l_row = lane >> 2, l_piece = lane & 3;                       // as a loader
  // as a reader: the instruction's blocks are other tokens, or the same tokens and other experts
  const int my_t = WE == N ? lane : lane % N;
  const int my_e = C::WT + (WE == N ? lane % N : lane);
  // as a selector: 8 threads per token, every eighth expert each, where there are as many threads
  const int per = static_cast<int>(blockDim.x) >= 8 * C::WT ? 8 : 1;
  const int sel_t = threadIdx.x / per, sel_e = threadIdx.x % per;
  typename M::Acc zero;
#pragma unroll
  for (int v = 0; v < M::kRegs; ++v) zero[v] = 0.0f;
  Best<KS> best;
  best.clear();
  for (int e0 = 0; e0 < E; e0 += WE) {
    // this lane's rows of the tile's tokens, then of its experts (past the end: a repeated row, never used)
    const float *xb = x + static_cast<size_t>(t0) * d, *wb = wg + static_cast<size_t>(e0) * d;
    unsigned src[C::LOADS];
#pragma unroll
    for (int i = 0; i < C::LOADS; ++i) {
      const int r = 16 * i + l_row - (16 * i < C::WT ? 0 : C::WT);
      const int most = (16 * i < C::WT ? tokens - t0 : E - e0) - 1;
      src[i] = static_cast<unsigned>(r < most ? r : most) * d + l_piece * 4;
    }
    float4v reg[C::LOADS];
    // K past the part's end reads as zero, which adds nothing
    auto fetch = [&](int kk, int k_hi) {
      const bool in = kk + l_piece * 4 < k_hi;                           // d is a multiple of 8
#pragma unroll
      for (int i = 0; i < C::LOADS; ++i) {
        const float4v none = {0.0f, 0.0f, 0.0f, 0.0f};
        reg[i] = in ? *reinterpret_cast<const float4v *>((16 * i < C::WT ? xb : wb) + (src[i] + static_cast<unsigned>(kk))) : none;
      }
    };
    if (wave < nparts) fetch(wave * kPart, d);
    for (int p0 = 0; p0 < nparts; p0 += held) {
      for (int part = p0 + wave; part < nparts && part < p0 + held; part += waves) {   // uniform per wavefront
        float *region = s_mem + static_cast<size_t>(part - p0) * C::REGION;
        const int k_lo = part * kPart;
        const int k_hi = k_lo + kPart < d ? k_lo + kPart : d;
        float acc[M::kRegs];
#pragma unroll
        for (int v = 0; v < M::kRegs; ++v) acc[v] = 0.0f;
        for (int kk = k_lo; kk < k_hi; kk += kF32StageK) {
#pragma unroll
          for (int i = 0; i < C::LOADS; ++i)
            *reinterpret_cast<float4v *>(region + (16 * i + l_row) * kF32Row + l_piece * 4) = reg[i];
          // the next stage, at the part's end the first of this wavefront's next part
          const int next = kk + kF32StageK < k_hi ? kk + kF32StageK : k_lo + waves * kPart;
          if (next < d) fetch(next, d);
          asm volatile("" ::: "memory");                                 // the loads stay ahead of the arithmetic
          const float *xr = region + my_t * kF32Row, *wr = region + my_e * kF32Row;
          float4v xv[2], wv[2];
          xv[0] = *reinterpret_cast<const float4v *>(xr);
          wv[0] = *reinterpret_cast<const float4v *>(wr);
          typename M::Acc prod[2];
          prod[0] = M::run(xv[0][0], wv[0][0], zero);
#pragma unroll
          for (int q = 0; q < kF32StageK; ++q) {
            const int c = q >> 2, n = q + 1;
            if ((q & 3) == 0 && c + 1 < kF32StageK / 4) {
              xv[(c + 1) & 1] = *reinterpret_cast<const float4v *>(xr + 4 * (c + 1));
              wv[(c + 1) & 1] = *reinterpret_cast<const float4v *>(wr + 4 * (c + 1));
            }
            // the next products are issued ahead of these additions, and stay there (left alone, the compiler puts
            // them among the additions, which then wait)
            if (n < kF32StageK) prod[n & 1] = M::run(xv[(n >> 2) & 1][n & 3], wv[(n >> 2) & 1][n & 3], zero);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int v = 0; v < M::kRegs; ++v) {
              acc[v] = acc[v] + prod[q & 1][v];
              asm volatile("" : "+v"(acc[v]));
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int v = 0; v < M::kRegs; ++v) {
          const int b = M::block(v) * N, row = M::row(v, lane), col = lane % N;
          region[(WE == N ? b + row : row) * C::LD + (WE == N ? col : b + col)] = acc[v];
        }
      }
      __syncthreads();
      const int np = nparts - p0 < held ? nparts - p0 : held;
      const bool last = p0 + held >= nparts;
      for (int o = threadIdx.x; o < C::WT * WE; o += blockDim.x) {
        const int t = o / WE, e = o % WE;
        const int at = t * C::LD + e;
        float s = p0 == 0 ? 0.0f : s_logit[at];                          // (a part's sum is never -0)
        int w = 0;
        for (; w + kMaxWaves <= np; w += kMaxWaves) {                    // eight reads on their way
          float part[kMaxWaves];
#pragma unroll
          for (int u = 0; u < kMaxWaves; ++u) part[u] = s_mem[static_cast<size_t>(w + u) * C::REGION + at];
#pragma unroll
          for (int u = 0; u < kMaxWaves; ++u) s = s + part[u];
        }
        for (; w < np; ++w) s = s + s_mem[static_cast<size_t>(w) * C::REGION + at];
        if (last && e0 + e < E) {
          if (bg) s = s + bg[e0 + e];
          if (logits_out && t0 + t < tokens) logits_out[static_cast<size_t>(t0 + t) * E + e0 + e] = s;
        }
        s_logit[at] = s;
      }
      __syncthreads();
    }
    if (sel_t < C::WT) {
      const int ne = (E - e0) < WE ? (E - e0) : WE;
      for (int e = sel_e; e < ne; e += per) best.offer(s_logit[sel_t * C::LD + e], e0 + e, k);
    }
    // the next tile's logits are written behind the barrier that follows its first round's part sums
  }
  // lists of disjoint experts: (logit, expert) is a strict order, so it does not matter in which order they are offered
  for (int off = 1; off < per; off <<= 1) {
    float ov[KS];
    int oid[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      ov[s] = __shfl_xor(best.v[s], off, 64);
      oid[s] = __shfl_xor(best.id[s], off, 64);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
      if (s < k && oid[s] != INT_MAX) best.offer(ov[s], oid[s], k);
  }
  const bool mine = sel_t < C::WT && sel_e == 0 && t0 + sel_t < tokens;
  if (mine) best.template write<float>(t0 + sel_t, k, idx_out, score_out);
  static_assert(C::REGION >= (WE >= 64 ? 1024 : WE), "a count per expert");
  if (wg_cnt) leave_counts<KS>(best, mine, k, E, reinterpret_cast<int *>(s_mem), wg_cnt);
}

template <int N, int WE>
int launch_gate_f32_mfma(const float *x, const float *wg, const float *bg, int tokens, int d, int E, int k, int64_t *idx_out,
                         float *score_out, float *logits_out, hipStream_t stream, int32_t *wg_cnt, long long max_cnt, int *tokens_per_wg) {
  using C = GateF32Mfma<N, WE>;
  const int nparts = (d + kPart - 1) / kPart;
  const int waves = nparts < kMaxWaves ? nparts : kMaxWaves;
  const auto lds_of = [&](int turns) { return sizeof(float) * (static_cast<size_t>(waves) * turns * C::REGION + C::WT * C::LD); };
  // The 32-wide tiles' registers leave a CU one workgroup of eight wavefronts, which may as well have all of its LDS (not the
  // 16-wide ones': two of them run side by side)
  const int turns = N == 32 && nparts > waves && lds_of(2) <= 160 * 1024 ? 2 : 1;
  const size_t lds = lds_of(turns);
  static_assert(sizeof(float) * (kMaxWaves * C::REGION + C::WT * C::LD) <= 160 * 1024, "LDS of a CU");
  auto kern = k <= 2 ? gate_f32_mfma_kernel<N, WE, 2> : gate_f32_mfma_kernel<N, WE, kMaxTopK>;
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(lds));
    if (e != hipSuccess) return fail(CCF_ERR_HIP, "gate: LDS attribute: %s", hipGetErrorString(e));
  }
  const int wgs = (tokens + C::WT - 1) / C::WT;
  if (!counts_fit(wg_cnt, wgs, E, C::WT, k, max_cnt)) wg_cnt = nullptr;
  if (wg_cnt && tokens_per_wg) *tokens_per_wg = C::WT;
  hipLaunchKernelGGL(kern, dim3(wgs), dim3(waves * 64), lds, stream, x, wg, bg, tokens, d, E, k,
                     idx_out, score_out, logits_out, wg_cnt, turns);
  return check_launch("gate_f32_mfma_kernel");
}

// The same for few tokens where those tiles leave most of their lanes or wavefronts idle: one to three experts of a
// wide model (tiles have eight at least), or many experts of a narrow one (its one or two parts make as many wavefronts,
// which walk the experts' tiles one after the other).  One wavefront per token: a lane takes one (expert, part) pair at
// a time and walks the part in ascending K, then the lanes add each expert's part sums in order.
__global__ void __launch_bounds__(64)
gate_f32_walk_kernel(const float *__restrict__ x, const float *__restrict__ wg, const float *__restrict__ bg,
                     int d, int E, int k, int group, int64_t *__restrict__ idx_out,
                     float *__restrict__ score_out, float *__restrict__ logits_out) {
#pragma clang fp contract(off)
  extern __shared__ float s_mem[];
  const int lane = threadIdx.x, t = blockIdx.x;
  const int nparts = (d + kPart - 1) / kPart;
  float *s_logit = s_mem;                          // [E]
  float *s_part = s_mem + E;                       // [group][nparts]: `group` experts at a time
  const float *xrow = x + static_cast<size_t>(t) * d;
  for (int e0 = 0; e0 < E; e0 += group) {
    const int ne = (E - e0) < group ? (E - e0) : group;
    for (int q = lane; q < ne * nparts; q += kWave) {   // part fastest: neighbours read neighbouring K
      const int p = q % nparts;
      const float *wrow = wg + static_cast<size_t>(e0 + q / nparts) * d;
      const int k_end = (p + 1) * kPart < d ? (p + 1) * kPart : d;
      float acc = 0.0f;
      for (int kk = p * kPart; kk < k_end; kk += 4) {
        const float4v xv = *reinterpret_cast<const float4v *>(xrow + kk);
        const float4v wv = *reinterpret_cast<const float4v *>(wrow + kk);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float prod = xv[j] * wv[j];
          acc = acc + prod;
        }
      }
      s_part[q] = acc;
    }
    __syncthreads();
    for (int g = lane; g < ne; g += kWave) {
      float s = s_part[g * nparts];
      for (int p = 1; p < nparts; ++p) s = s + s_part[g * nparts + p];
      if (bg) s = s + bg[e0 + g];
      s_logit[e0 + g] = s;
      if (logits_out) logits_out[static_cast<size_t>(t) * E + e0 + g] = s;
    }
    __syncthreads();
  }
  if (lane == 0) {
    Best<kMaxTopK> best;
    best.clear();
    for (int e = 0; e < E; ++e) best.offer(s_logit[e], e, k);
    best.write<float>(t, k, idx_out, score_out);
  }
}

// Microseconds of the tiles and of a wavefront per token: 256 tokens of 4096, 1 expert: 12 and 8, 2: 12 and 9 (3: the
// tiles; of 8192: 22 and 20); 256 of 128, 33 experts: 15 and 12, 128: 37 and 28, 512: 140 and 94; of 256, 200: 60 and 55.
// More tokens fill the chip with either: 2048 of 128, 128 experts 37 and 53; 1024 of 256, 256: 69 and 86.
bool gate_f32_walks(int tokens, int d, int E) {
  if (E <= 3) return tokens * static_cast<long long>(E) <= 1024 && d > (E < 3 ? 2048 : 6144) && d <= 8192 * kPart;   // (LDS)
  return (E > 32 && d <= kPart && tokens <= (E > 64 ? 1024 : 512)) || (E > 128 && d <= 2 * kPart && tokens <= 512);
}

// Where the products run as MFMAs, in microseconds (vector unit, MFMA).  More than 32 experts: at 4097 tokens, where the
// vector unit's tiles grow to 32 tokens as well, 64 experts of 256: 32, 29; of 2048: 55, 43; of 7168: 157, 135 (4096
// tokens of 2048: 42, 46).  Up to 32 experts the tiles are twice as tall (8192 tokens of 2048, 32 experts: 39, 48; 8193:
// 61, 43) and want six parts of K (24576 of 512, 32 experts: 28, 28; 8193: 19, 24), and a second round of
// workgroups more of them (24576 tokens of 768, 32 experts: 46, 53; of 2048: 101, 86).  16 experts of a very wide model
// are bound by reading the tokens (16384 of 7168, 9 experts: 119, 126).
bool gate_f32_on_mfma(int tokens, int d, int E) {
  if (E > 32) return tokens > 4096;
  if (E <= 8 || tokens <= 8192 || d <= 5 * kPart) return false;
  return (tokens <= 16384 || d >= 12 * kPart) && (E > 16 || d <= 4096);
}

// fp16 gate of few tokens.  The MFMA tiles above have 16 tokens at least, and the 1024 instructions that 16 tokens of 4096
// and 16 experts take keep the one CU that has them busy for 4 us, the conversions of their operands for as long again.
// Here a thread walks one part of K of one expert for one token as a chain of 128 fused multiply-adds: the same chain, the
// same bits, and with 8 experts of 4096 four wavefronts, whose 256 chains run side by side.
//
// * A workgroup holds all expert rows and the rows of `group` tokens in LDS, fetched by direct loads that are all on their
//   way at once, and takes `wg_tokens` tokens, `group` at a time.  A part is 16 chunks of 16 bytes; chunk c of part i sits
//   at c ^ (i % 16), applied on the global side, so that lanes on neighbouring parts read other banks.
// * The part sums meet in LDS, a thread per token and expert adds them in part order, and one per token selects (top-3 and
//   more: as many rank them).
// * With `route` (one workgroup, at most 64 indices) the routing of the choice follows: a lane per index.
//
// Microseconds, MFMA tiles and here (the gate alone): see gate_f16_walk_group().
struct TinyRoute {
  int32_t *counts, *offsets;                       // counts null: no routing
  int64_t *pos;
  int32_t *src_row, *dst_row, *inv_pos;
  int64_t *idx_kept;
  int capacity;
};
constexpr int kTinyIndices = 64;
constexpr int kTinyBatches = 2;     // most turns of the one workgroup that gates and routes

// LDS of a workgroup, in bytes: expert rows, token rows, part sums, logits, biases, counts, routed indices
struct WalkLds {
  int x, part, logit, bias, row, idx, bytes;
};
__host__ __device__ inline WalkLds walk_lds(int E, int nparts, int group) {
  WalkLds l;
  l.x = (E * nparts * 256 + 1023) / 1024 * 1024;
  l.part = l.x + (group * nparts * 256 + 1023) / 1024 * 1024;
  l.logit = l.part + 4 * group * E * (nparts + 1);
  l.bias = l.logit + 4 * group * (E + 1);
  l.row = l.bias + 4 * E;
  l.idx = l.row + 4 * E;
  l.bytes = l.idx + 4 * 2 * kTinyIndices;
  return l;
}

template <int KS>
__global__ void __launch_bounds__(512)
gate_walk_kernel(const half_t *__restrict__ x, const half_t *__restrict__ wg, const half_t *__restrict__ bg,
                 int tokens, int d, int E, int k, int group, int wg_tokens, int64_t *__restrict__ idx_out,
                 half_t *__restrict__ score_out, half_t *__restrict__ logits_out, int32_t *__restrict__ wg_cnt,
                 TinyRoute route) {
  extern __shared__ __attribute__((aligned(1024))) char s_raw[];
  const int nparts = (d + kPart - 1) / kPart, chains = E * nparts;
  const WalkLds at = walk_lds(E, nparts, group);
  float *s_part = reinterpret_cast<float *>(s_raw + at.part), *s_logit = reinterpret_cast<float *>(s_raw + at.logit);
  float *s_bias = reinterpret_cast<float *>(s_raw + at.bias);
  int *s_row = reinterpret_cast<int *>(s_raw + at.row), *s_idx = reinterpret_cast<int *>(s_raw + at.idx);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const FastDiv by_parts(nparts), by_chains(chains), by_experts(E);

  // `rows` rows of base from row `first` on (past `last` that one again) into LDS at byte `to`
  auto fetch = [&](const half_t *base, int first, int rows, int last, int to) {
    const int parts = rows * nparts;
    for (int s0 = wave * 64; s0 < parts * 16; s0 += waves * 64) {
      const int s = s0 + lane, i = s >> 4, part = i < parts ? i : parts - 1;
      const int r = by_parts.div(part);
      const int row = first + r < last ? first + r : last;
      const int kk = (part - r * nparts) * kPart + (((s & 15) ^ (i & 15)) << 3);
      const half_t *src = base + static_cast<size_t>(row) * d + (kk < d ? kk : 0);       // past the end of K: never used
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                       (__attribute__((address_space(3))) void *)(s_raw + to + s0 * 16), 16, 0, 0);
    }
  };
  fetch(wg, 0, E, E - 1, 0);
  for (int e = tid; e < E; e += blockDim.x) {
    s_bias[e] = bg ? static_cast<float>(bg[e]) : 0.0f;
    s_row[e] = 0;
  }
  const int g = by_chains.div(tid), chain = tid - g * chains;
  const int e_of = by_parts.div(chain), p_of = chain - e_of * nparts;
  const bool full = d % kPart == 0;
  const int t_first = blockIdx.x * wg_tokens;
  for (int t0 = t_first; t0 < t_first + wg_tokens && t0 < tokens; t0 += group) {
    fetch(x, t0, group, tokens - 1, at.x);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (g < group) {
      const int xi = g * nparts + p_of;
      const char *wr = s_raw + chain * 256, *xr = s_raw + at.x + xi * 256;
      const int len = d - p_of * kPart;            // K elements left for this part
      float acc = 0.0f;
      auto walk = [&](auto FULL) {
#pragma unroll
        for (int c = 0; c < kPart / 8; ++c) {
          const half8 wv = *reinterpret_cast<const half8 *>(wr + ((c ^ (chain & 15)) << 4));
          const half8 xv = *reinterpret_cast<const half8 *>(xr + ((c ^ (xi & 15)) << 4));
          if (decltype(FULL)::value || c * 8 < len) {
#pragma unroll
            for (int j = 0; j < 8; ++j) acc = __builtin_fmaf(static_cast<float>(xv[j]), static_cast<float>(wv[j]), acc);
          }
        }
      };
      if (full) walk(std::true_type{});
      else walk(std::false_type{});
      s_part[(g * E + e_of) * (nparts + 1) + p_of] = acc;
    }
    __syncthreads();
    for (int i = tid; i < group * E; i += blockDim.x) {
      const int gi = by_experts.div(i), e = i - gi * E;
      const float *ps = s_part + i * (nparts + 1);
      float t = ps[0];
#pragma unroll 8
      for (int p = 1; p < nparts; ++p) t = t + ps[p];
      if (bg) t = t + s_bias[e];
      t = round_to<half_t>(t);
      if (logits_out && t0 + gi < tokens) logits_out[static_cast<size_t>(t0 + gi) * E + e] = static_cast<half_t>(t);
      s_logit[gi * (E + 1) + e] = t;
    }
    __syncthreads();
    // Long lists by rank: a thread per token and expert counts the experts in front of its own (NaN logits behind all,
    // as no expert: what a list that they left short holds) and puts it there, the part sums' place.  2048 tokens of
    // 1024, 16 experts, top-8: 20 us with one thread inserting into a list of eight, longer than the MFMA tiles' 17, and 10;
    // a token of 4096, 8 experts, top-3: 8.8, 14.5 and 7.5.
    float *s_v = s_part;
    int *s_id = reinterpret_cast<int *>(s_part + group * k);              // k <= E: no longer than the part sums
    if constexpr (KS > 2) {
      for (int i = tid; i < group * E; i += blockDim.x) {
        const int gi = by_experts.div(i), e = i - gi * E;
        const float *row = s_logit + gi * (E + 1);
        const float v = row[e];
        const bool none = v != v;
        int rank = 0;
#pragma unroll 8
        for (int o = 0; o < E; ++o) {
          const float ov = row[o];
          rank += none ? (ov == ov || o < e) : better(ov, o, v, e);
        }
        if (rank < k) {
          s_v[gi * k + rank] = none ? -INFINITY : v;
          s_id[gi * k + rank] = none ? INT_MAX : e;
        }
      }
      __syncthreads();
    }
    if (tid < group && t0 + tid < tokens) {
      Best<KS> best;
      best.clear();
      if constexpr (KS > 2) {
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (s < k) {
            best.v[s] = s_v[tid * k + s];
            best.id[s] = s_id[tid * k + s];
          }
      } else {
#pragma unroll 8
        for (int e = 0; e < E; ++e) best.offer(s_logit[tid * (E + 1) + e], e, k);
      }
      best.template write<half_t>(t0 + tid, k, idx_out, score_out);
#pragma unroll
      for (int s = 0; s < KS; ++s)
        if (s < k) {
          if (wg_cnt && best.id[s] < E) atomicAdd(&s_row[best.id[s]], 1);
          if (route.counts) s_idx[(t0 + tid) * k + s] = best.id[s];
        }
    }
    // the next tokens' rows land behind every thread's reads of these; their logits two barriers further on
  }
  if (wg_cnt) {
    __syncthreads();
    for (int e = tid; e < E; e += blockDim.x) wg_cnt[static_cast<size_t>(blockIdx.x) * E + e] = s_row[e];
  }
  if (!route.counts) return;
  // The routing, as pos_kernel does it: ranks in index order, the capacity, then the experts' starts.  A list that NaN
  // logits left short has entries that are no expert.
  int *s_kept = s_idx + kTinyIndices;
  const int n = tokens * k;
  __syncthreads();
  int e = INT_MAX, rank = 0;
  if (tid < n) {
    e = s_idx[tid];
    for (int q = 0; q < tid; ++q) rank += s_idx[q] == e;
    const bool kept = e < E && (route.capacity < 0 || rank < route.capacity);
    s_kept[tid] = kept ? e : INT_MAX;
  }
  __syncthreads();
  if (tid < n) {
    const bool kept = s_kept[tid] < E;
    int j = rank;
    for (int q = 0; q < n; ++q) j += s_kept[q] < e;
    if (kept) {
      route.pos[j] = tid;
      route.src_row[j] = tid / k;
      route.dst_row[j] = tid;
    }
    route.inv_pos[tid] = kept ? j : -1;
    route.idx_kept[tid] = kept ? e : -1;
  }
  for (int c = tid; c <= E; c += blockDim.x) {
    int start = 0, count = 0;
    for (int q = 0; q < n; ++q) {
      start += s_kept[q] < c;
      count += s_kept[q] == c;
    }
    route.offsets[c] = start;
    if (c < E) route.counts[c] = count;
  }
}

// (a knob away from its default asks for a form of the MFMA tiles)
bool gate_default_shape() { return g_gate_slots == 0 && g_gate_waves == kMaxWaves && g_gate_stream == -1; }

// Tokens that a workgroup of gate_walk_kernel takes at a time, 0: not a case for it.  The expert rows fit in LDS, and all
// workgroups are on the chip at once: a second round loads the expert rows again and loses to the MFMA tiles.  Microseconds
// (MFMA tiles, here): 8 experts of 4096, 1 token 11.4, 5.8, 333 tokens 12.0, 7.2, 512 (one round) 11.7, 7.4, 1024 12.4,
// 13.2; of 2048, 1536 (one round) 8.9, 7.0, 2048 9.0, 10.5; of 768, 8192 (one round) 11.8, 10.1, 16384 13.4, 15.9; 16
// experts of 1024, 2048 (one round) 8.7, 8.5, 4096 9.2, 14.8; 32 of 768, 768 (one round) 11.9, 8.1, 1536 12.0, 13.5; 4 of
// 256, 512 8.6, 4.0.
int gate_f16_walk_group(int tokens, int d, int E) {
  constexpr int kCus = 256, kLds = 160 * 1024, kMaxLds = 150 * 1024, kWgsPerCu = 8;
  const int nparts = (d + kPart - 1) / kPart;
  if (static_cast<long long>(E) * nparts > 512) return 0;
  const int chains = E * nparts;
  int group = 1;
  while (2 * group * chains <= 256 && group < tokens) group *= 2;
  const int lds = walk_lds(E, nparts, group).bytes;
  if (lds > kMaxLds) return 0;
  const int per_cu = kLds / lds < kWgsPerCu ? kLds / lds : kWgsPerCu;
  return (tokens + group - 1) / group <= kCus * per_cu ? group : 0;
}

int launch_gate_walk(const half_t *x, const half_t *wg, const half_t *bg, int tokens, int d, int E, int k, int group,
                     int64_t *idx_out, half_t *score_out, half_t *logits_out, hipStream_t stream, int32_t *wg_cnt,
                     long long max_cnt, int *tokens_per_wg, const TinyRoute &route) {
  const int nparts = (d + kPart - 1) / kPart, chains = E * nparts;
  const int threads = chains * group > 256 ? 512 : 256;
  const int wg_tokens = route.counts ? (tokens + group - 1) / group * group : group;
  const int wgs = (tokens + wg_tokens - 1) / wg_tokens;
  if (!counts_fit(wg_cnt, wgs, E, wg_tokens, k, max_cnt)) wg_cnt = nullptr;
  if (wg_cnt && tokens_per_wg) *tokens_per_wg = wg_tokens;
  const int lds = walk_lds(E, nparts, group).bytes;
  auto kern = k == 1 ? gate_walk_kernel<1> : (k == 2 ? gate_walk_kernel<2> : gate_walk_kernel<kMaxTopK>);
  if (lds > 65536) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return fail(CCF_ERR_HIP, "gate: LDS attribute: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(kern, dim3(wgs), dim3(threads), lds, stream, x, wg, bg, tokens, d, E, k, group, wg_tokens, idx_out, score_out,
                     logits_out, wg_cnt, route);
  return check_launch("gate_walk_kernel");
}

}  // namespace
}  // namespace ccf

namespace ccf {
// Gate and routing of a few tokens as one launch, by a workgroup that takes its tokens in two turns at most.  Microseconds
// as two launches (gate in MFMA tiles, then in walks; both with 5 of routing) and as one: 8 experts of 4096, 1 token 16.3,
// 10.8, 6.7, 2 (two turns) 16.5, 11.1, 9.9, 3 16.4, 11.1, 12.9; of 768, 8 (two turns) 12.4, 9.9, 8.7; 32 of 1024, 1 17.8,
// 11.6, 8.7.
bool gate_route_tiny_fits(int tokens, int d, int E, int k, int dtype, const void *x, const void *wg) {
  if (dtype != CCF_F16 || tokens <= 0 || d <= 0 || d % 8 || E <= 0 || E > 512 || k < 1 || k > kMaxTopK || k > E || !x || !wg ||
      !aligned16(x) || !aligned16(wg) || static_cast<long long>(tokens) * k > kTinyIndices || !gate_default_shape())
    return false;
  const int group = gate_f16_walk_group(tokens, d, E);
  return group > 0 && tokens <= kTinyBatches * group;
}

int gate_route_tiny(const void *x, const void *wg, const void *bg, int tokens, int d, int E, int k, int capacity, int64_t *idx,
                    void *score, int32_t *counts, int32_t *offsets, int64_t *pos, int32_t *src_row, int32_t *dst_row,
                    int32_t *inv_pos, int64_t *idx_kept, hipStream_t stream) {
  return launch_gate_walk(static_cast<const half_t *>(x), static_cast<const half_t *>(wg), static_cast<const half_t *>(bg), tokens, d,
                          E, k, gate_f16_walk_group(tokens, d, E), idx, static_cast<half_t *>(score), nullptr, stream, nullptr, 0,
                          nullptr, TinyRoute{counts, offsets, pos, src_row, dst_row, inv_pos, idx_kept, capacity});
}

// The gate; with wg_cnt (room for max_cnt ints) the tiled kernels also leave, per workgroup, how many of
// its token slots chose each expert ([workgroups][tot_expert], a workgroup covering *tokens_per_wg
// consecutive tokens), when that table is one that the routing can use (counts_fit); *tokens_per_wg = 0 says
// it was not written.
int gate_forward(const void *x, const void *wg, const void *bg, int tokens, int d_model, int tot_expert, int top_k,
                 int dtype, int64_t *idx_out, void *score_out, void *logits_out, ccf_stream_t stream,
                 int32_t *wg_cnt, long long max_cnt, int *tokens_per_wg) {
  if (tokens_per_wg) *tokens_per_wg = 0;
  CCF_REQUIRE(x && wg && idx_out && score_out, CCF_ERR_ARG, "gate: null pointer");
  CCF_REQUIRE(tokens >= 0 && d_model > 0 && tot_expert > 0, CCF_ERR_ARG, "gate: bad size");
  CCF_REQUIRE(d_model % 8 == 0, CCF_ERR_SHAPE, "gate: d_model=%d is not a multiple of 8", d_model);
  CCF_REQUIRE(top_k >= 1 && top_k <= kMaxTopK && top_k <= tot_expert, CCF_ERR_SHAPE,
              "gate: top_k=%d outside 1..min(%d, tot_expert=%d)", top_k, kMaxTopK, tot_expert);
  CCF_REQUIRE(tot_expert <= 1024, CCF_ERR_SHAPE, "gate: tot_expert=%d exceeds 1024", tot_expert);
  CCF_REQUIRE(dtype == CCF_F16 || dtype == CCF_F32, CCF_ERR_UNSUPPORTED, "gate: dtype %d", dtype);
  CCF_REQUIRE(aligned16(x) && aligned16(wg), CCF_ERR_ARG, "gate: x and wg must be 16-byte aligned");
  if (tokens == 0) return CCF_OK;
  const int nparts = (d_model + kPart - 1) / kPart;
  if (dtype == CCF_F32 && gate_f32_walks(tokens, d_model, tot_expert)) {
    // part sums of as many experts at a time as 32 KB hold
    int group = 8192 / nparts;
    group = group < 1 ? 1 : (group > tot_expert ? tot_expert : group);
    const size_t lds = sizeof(float) * (static_cast<size_t>(tot_expert) + static_cast<size_t>(group) * nparts);
    hipLaunchKernelGGL(gate_f32_walk_kernel, dim3(tokens), dim3(64), lds, as_stream(stream), static_cast<const float *>(x),
                       static_cast<const float *>(wg), static_cast<const float *>(bg), d_model, tot_expert, top_k, group,
                       idx_out, static_cast<float *>(score_out), static_cast<float *>(logits_out));
    return check_launch("gate_f32_walk_kernel");
  }
  if (dtype == CCF_F32 && gate_f32_on_mfma(tokens, d_model, tot_expert)) {
    auto launch = tot_expert <= 16 ? launch_gate_f32_mfma<16, 16>
                                   : (tot_expert <= 32 ? launch_gate_f32_mfma<32, 32> : launch_gate_f32_mfma<32, 64>);
    return launch(static_cast<const float *>(x), static_cast<const float *>(wg), static_cast<const float *>(bg), tokens,
                  d_model, tot_expert, top_k, idx_out, static_cast<float *>(score_out), static_cast<float *>(logits_out),
                  as_stream(stream), wg_cnt, max_cnt, tokens_per_wg);
  }
  if (dtype == CCF_F32) {
    auto launch = tokens > 4096 ? launch_gate_f32_experts<4>
                                : (tokens > 2048 ? launch_gate_f32_experts<2> : launch_gate_f32_experts<1>);
    return launch(static_cast<const float *>(x), static_cast<const float *>(wg), static_cast<const float *>(bg), tokens,
                  d_model, tot_expert, top_k, idx_out, static_cast<float *>(score_out), static_cast<float *>(logits_out),
                  as_stream(stream), wg_cnt, max_cnt, tokens_per_wg);
  }
  const int group = gate_default_shape() ? gate_f16_walk_group(tokens, d_model, tot_expert) : 0;
  if (group > 0)
    return launch_gate_walk(static_cast<const half_t *>(x), static_cast<const half_t *>(wg), static_cast<const half_t *>(bg), tokens,
                            d_model, tot_expert, top_k, group, idx_out, static_cast<half_t *>(score_out),
                            static_cast<half_t *>(logits_out), as_stream(stream), wg_cnt, max_cnt, tokens_per_wg, TinyRoute{});
  // Tile and slots.  With S slots a wavefront covers 64 / S tokens, so S grows while there
  // are fewer than four workgroups per CU and K has parts for the slots.
  const int n = tot_expert > 16 ? 32 : 16;
  const int blocks_per_mfma = 64 / n;
  int ls = 0;
  if (g_gate_slots) {
    while ((2 << ls) <= g_gate_slots && (2 << ls) <= blocks_per_mfma) ++ls;
  } else {
    while ((2 << ls) <= blocks_per_mfma && (2 << ls) <= nparts &&
           (tokens + (64 >> ls) - 1) / (64 >> ls) < 1024)
      ++ls;
  }
  const int slots = 1 << ls;
  const int tw = 64 >> ls;
  // With a wavefront or more per SIMD even when each works alone (two with the 16-wide tile, whose
  // MFMAs are shorter), the wavefronts stream through K on their own; with fewer, the wavefronts
  // of a workgroup share the parts of K.
  const int tiles = (tokens + tw - 1) / tw;
  const bool stream_form = g_gate_stream > 0 || (g_gate_stream < 0 && (tiles >= 2048 || (tiles >= 1024 && n == 32)));
  int waves = (nparts + slots - 1) / slots;
  int cap = g_gate_waves < kMaxWaves ? g_gate_waves : kMaxWaves;
  cap = cap < 1 ? 1 : cap;
  waves = waves < cap ? waves : cap;
  if (stream_form) waves = kStreamWaves;
  const int wg_tokens = stream_form ? kStreamWaves * tw : tw;
  const size_t lds = sizeof(float) * (static_cast<size_t>(waves) * kRegionFloats +
                                      (stream_form ? 0 : static_cast<size_t>(tw) * (n + 1)));
  CCF_REQUIRE(lds <= 160 * 1024, CCF_ERR_SHAPE, "gate: %zu bytes of LDS needed", lds);
  dim3 grid((tokens + wg_tokens - 1) / wg_tokens), block(waves * 64);
  if (counts_fit(wg_cnt, grid.x, tot_expert, wg_tokens, top_k, max_cnt)) {
    if (tokens_per_wg) *tokens_per_wg = wg_tokens;
  } else {
    wg_cnt = nullptr;
  }
#define CCF_GATE_LAUNCH(NN, LSV, KSV)                                                              \
  do {                                                                                             \
    auto kern = stream_form ? gate_stream_kernel<NN, LSV, KSV> : gate_mfma_kernel<NN, LSV, KSV>;   \
    if (lds > 65536) {                                                                             \
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),                     \
                                         hipFuncAttributeMaxDynamicSharedMemorySize,               \
                                         static_cast<int>(lds));                                   \
      if (e != hipSuccess) return fail(CCF_ERR_HIP, "gate: LDS attribute: %s", hipGetErrorString(e)); \
    }                                                                                              \
    hipLaunchKernelGGL(kern, grid, block, lds, as_stream(stream), static_cast<const half_t *>(x),  \
                       static_cast<const half_t *>(wg), static_cast<const half_t *>(bg), tokens,   \
                       d_model, tot_expert, top_k, idx_out, static_cast<half_t *>(score_out),      \
                       static_cast<half_t *>(logits_out), wg_cnt);                                 \
  } while (0)
#define CCF_GATE_K(NN, LSV)                                                  \
  do {                                                                       \
    if (top_k == 1) CCF_GATE_LAUNCH(NN, LSV, 1);                             \
    else if (top_k == 2) CCF_GATE_LAUNCH(NN, LSV, 2);                        \
    else CCF_GATE_LAUNCH(NN, LSV, kMaxTopK);                                 \
  } while (0)
  if (n == 32) {
    if (ls == 0) CCF_GATE_K(32, 0); else CCF_GATE_K(32, 1);
  } else {
    if (ls == 0) CCF_GATE_K(16, 0); else if (ls == 1) CCF_GATE_K(16, 1); else CCF_GATE_K(16, 2);
  }
#undef CCF_GATE_K
#undef CCF_GATE_LAUNCH
  return check_launch("gate_mfma_kernel");
}
}  // namespace ccf

namespace ccf {
namespace {

// ---- backward of the softmax over the selected logits and of the selection --------------
// A workgroup takes kGbTokens tokens: thread t computes the k values of its token,
//   g_j = s_j (grad_j - sum_i s_i grad_i)    (fp32),
// the workgroup zero-fills its rows of grad_logits and, behind a barrier, every thread stores its
// k values at their experts' columns.  The bias gradient is the column sum of the unrounded
// values: wavefront w sums experts w, w + 4, ... over the workgroup's tokens (lane l takes
// entries l, l + 64, ... in order, then a fixed tree over the lanes), so the result does not
// depend on scheduling; gate_bias_reduce_kernel adds the workgroups' sums in order.
constexpr int kGbTokens = 256;

__global__ void __launch_bounds__(kGbTokens)
gate_backward_kernel(const half_t *__restrict__ score, const half_t *__restrict__ grad_score,
                     const int64_t *__restrict__ idx, int tokens, int top_k, int E,
                     half_t *__restrict__ grad_logits, float *__restrict__ partial) {
  __shared__ float s_val[kGbTokens * kMaxTopK];
  __shared__ int s_idx[kGbTokens * kMaxTopK];
  const int t = threadIdx.x;
  const int tok0 = blockIdx.x * kGbTokens;
  const int tok = tok0 + t;
  float g[kMaxTopK];
  int ex[kMaxTopK];
  if (tok < tokens) {
    float s[kMaxTopK], dot = 0.0f;
    for (int j = 0; j < top_k; ++j) {
      s[j] = static_cast<float>(score[static_cast<size_t>(tok) * top_k + j]);
      g[j] = static_cast<float>(grad_score[static_cast<size_t>(tok) * top_k + j]);
      dot = fmaf(s[j], g[j], dot);
    }
    for (int j = 0; j < top_k; ++j) {
      g[j] = s[j] * (g[j] - dot);
      const int64_t e = idx[static_cast<size_t>(tok) * top_k + j];
      ex[j] = (e >= 0 && e < E) ? static_cast<int>(e) : -1;
    }
  } else {
    for (int j = 0; j < top_k; ++j) {
      g[j] = 0.0f;
      ex[j] = -1;
    }
  }
  for (int j = 0; j < top_k; ++j) {
    s_val[t * top_k + j] = g[j];
    s_idx[t * top_k + j] = ex[j];
  }
  // this workgroup's rows of grad_logits are one contiguous range
  const int n_tok = tokens - tok0 < kGbTokens ? tokens - tok0 : kGbTokens;
  half_t *rows = grad_logits + static_cast<size_t>(tok0) * E;
  const size_t n_el = static_cast<size_t>(n_tok) * E;
  for (size_t i = t; i < n_el; i += kGbTokens) rows[i] = static_cast<half_t>(0.0f);
  __syncthreads();                                  // the zeros are written (and s_val, s_idx)
  if (tok < tokens) {
    for (int j = 0; j < top_k; ++j)
      if (ex[j] >= 0) rows[static_cast<size_t>(t) * E + ex[j]] = static_cast<half_t>(g[j]);
  }
  if (!partial) return;
  const int lane = t & 63, wave = t >> 6;
  const int n_ent = kGbTokens * top_k;
  for (int e = wave; e < E; e += kGbTokens / 64) {
    float acc = 0.0f;
    for (int i = lane; i < n_ent; i += 64) acc += s_idx[i] == e ? s_val[i] : 0.0f;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) partial[static_cast<size_t>(blockIdx.x) * E + e] = acc;
  }
}

__global__ void __launch_bounds__(256)
gate_bias_reduce_kernel(const float *__restrict__ partial, int n_wg, int E, half_t *__restrict__ grad_bias) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= E) return;
  float acc = 0.0f;
  for (int w = 0; w < n_wg; ++w) acc += partial[static_cast<size_t>(w) * E + e];
  grad_bias[e] = static_cast<half_t>(acc);
}

// ---- the whole backward of the gate ------------------------------------------------------
// A token has k selected experts, so both products with the [T, E] gradient of the logits are sparse:
//   grad_x[t, :] = sum_j g[t, j] wg[e(t, j), :],   grad_wg[e, :] = sum over the (t, j) with e(t, j) = e of g[t, j] x[t, :],
// and the dense matrix is never made.  A workgroup takes a run of tokens and 512 columns, two per thread: it reads
// x once, writes grad_x, and adds the expert rows up in LDS, where a thread alone touches its two columns
// of every expert, so the order is the tokens' and two runs agree bit for bit.  gate_products_reduce_kernel adds the
// workgroups' partial rows in order and rounds once.  Bound by the chain of LDS additions of a run and by reading x and
// writing grad_x.  Against the softmax kernel, its reduction and two library products, GPU time: 1000 tokens of 256, 16
// experts 33 -> 16 us, 1999 of 768, 8: 22 -> 18, 4096 of 4096, 8: 42 -> 33, 32768 of 768, 8: 150 -> 65; and two launches
// instead of four, the products' 15 us of host time each (1999 tokens, host included: 58 -> 23).  More than 16 experts
// keep the products: the sums take so much LDS that a CU has one workgroup (8192 of 1024, 32: 47 against 57).  Since then eight
// tokens' loads are ahead of their use and the reduction has no remainder loop: 1000 of 256, 16 experts 16.6 -> 14.0 us, 1999
// of 768, 8: 18.7 -> 16.3, 4096 of 4096, 8: 33.1 -> 29.8, 32768 of 768, 8: 63.6 -> 56.4 (both launches, in a graph).  All 32 tokens'
// loads of a run at once: 50 us for the 1999 tokens.
//
// A wavefront holds the values of 64 tokens in its lanes and broadcasts them through scalar registers; the expert
// rows of wg sit in LDS, and the sums are plain reads and writes there (LDS float atomics run at ~190 cycles an
// instruction: 91 us instead of 18 for the 1999 tokens).
constexpr int kGpCols = 512;
constexpr int kGpMaxExpert = 16;                     // [E][512] floats and [E][512] halves of LDS: 48 KB

template <int KS>                                    // top_k <= KS
__global__ void __launch_bounds__(256)
gate_products_kernel(const half_t *__restrict__ score, const half_t *__restrict__ grad_score,
                     const int64_t *__restrict__ idx, const half_t *__restrict__ x, const half_t *__restrict__ wg,
                     int tokens, int top_k, int E, int d, int run, half_t *__restrict__ grad_x,
                     float *__restrict__ partial /* [n_run][E][d], or NULL */,
                     float *__restrict__ partial_b /* [n_run][E], or NULL */) {
  extern __shared__ float s_rows[];                  // [E][512] sums, then [E][512] halves of wg
  half_t *s_wg = reinterpret_cast<half_t *>(s_rows + E * kGpCols);
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int c = blockIdx.x * kGpCols + 2 * t;
  const bool in = c < d;                             // d is even
  const int cc = in ? c : 0;
  const int tok0 = blockIdx.y * run, tok1 = tok0 + run < tokens ? tok0 + run : tokens;
  // a thread reads and writes its own two columns only: no barrier
  for (int e0 = 0; e0 < E; e0 += 8) {
    half2v w[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) w[u] = *reinterpret_cast<const half2v *>(wg + static_cast<size_t>(e0 + u < E ? e0 + u : E - 1) * d + cc);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (e0 + u < E) {
        *reinterpret_cast<float2 *>(s_rows + (e0 + u) * kGpCols + 2 * t) = float2{0.0f, 0.0f};
        *reinterpret_cast<half2v *>(s_wg + (e0 + u) * kGpCols + 2 * t) = w[u];
      }
  }
  float bias = 0.0f;                                 // first wavefront of the first column range: expert = lane
  const bool want_b = partial_b && blockIdx.x == 0 && wave == 0;
  for (int base = tok0; base < tok1; base += 64) {
    const int n = tok1 - base < 64 ? tok1 - base : 64;
    float g[KS];
    int ex[KS];
    {
      const size_t at = static_cast<size_t>(base + (lane < n ? lane : n - 1)) * top_k;
      float dot = 0.0f, s[KS];
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        const bool on = j < top_k;
        s[j] = on ? static_cast<float>(score[at + (on ? j : 0)]) : 0.0f;
        g[j] = on ? static_cast<float>(grad_score[at + (on ? j : 0)]) : 0.0f;
        const int64_t e = on ? idx[at + (on ? j : 0)] : -1;
        ex[j] = e >= 0 && e < E ? static_cast<int>(e) : -1;
        if (on) dot = fmaf(s[j], g[j], dot);
      }
#pragma unroll
      for (int j = 0; j < KS; ++j) {
        g[j] = ex[j] >= 0 ? s[j] * (g[j] - dot) : 0.0f;
        ex[j] = ex[j] >= 0 ? ex[j] : 0;              // nobody's choice: adds zero
      }
    }
    constexpr int U = 8;                             // tokens whose loads leave together, ahead of the eight before them
    half2v xv[U], next[U];
    const auto load = [&](half2v (&to)[U], int q0) {
#pragma unroll
      for (int u = 0; u < U; ++u) to[u] = *reinterpret_cast<const half2v *>(x + static_cast<size_t>(base + (q0 + u < n ? q0 + u : n - 1)) * d + cc);
    };
    load(next, 0);
    for (int q0 = 0; q0 < n; q0 += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) xv[u] = next[u];
      load(next, q0 + U);                            // behind the last ones the last token again
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = q0 + u;
        if (q >= n) break;                           // uniform
        const float x0 = static_cast<float>(xv[u][0]), x1 = static_cast<float>(xv[u][1]);
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int j = 0; j < KS; ++j) {
          if (j >= top_k) break;
          const float gj = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, g[j]), q));
          const int e = __builtin_amdgcn_readlane(ex[j], q);
          const half2v w = *reinterpret_cast<const half2v *>(s_wg + e * kGpCols + 2 * t);
          a0 = fmaf(gj, static_cast<float>(w[0]), a0);
          a1 = fmaf(gj, static_cast<float>(w[1]), a1);
          float *row = s_rows + e * kGpCols + 2 * t;
          float2 sum = *reinterpret_cast<const float2 *>(row);
          sum.x = fmaf(gj, x0, sum.x);
          sum.y = fmaf(gj, x1, sum.y);
          *reinterpret_cast<float2 *>(row) = sum;
          if (want_b) bias += lane == e ? gj : 0.0f;
        }
        if (grad_x && in)
          *reinterpret_cast<half2v *>(grad_x + static_cast<size_t>(base + q) * d + c) = half2v{static_cast<half_t>(a0), static_cast<half_t>(a1)};
      }
    }
  }
  if (partial && in) {
    float *out = partial + static_cast<size_t>(blockIdx.y) * E * d + c;
    for (int e = 0; e < E; ++e)
      *reinterpret_cast<float2 *>(out + static_cast<size_t>(e) * d) = *reinterpret_cast<const float2 *>(s_rows + e * kGpCols + 2 * t);
  }
  if (want_b && lane < E) partial_b[static_cast<size_t>(blockIdx.y) * E + lane] = bias;
}

// Sum of n values `ld` apart, in order, N loads on their way together: past the end the first one is read again and left out
// (a remainder loop waits for each of its loads: 15 of 63).
template <int N, class T, class Add>
__device__ __forceinline__ void for_column(const T *col, size_t ld, int n, Add add) {
  for (int r = 0; r < n; r += N) {
    T v[N];
#pragma unroll
    for (int u = 0; u < N; ++u) v[u] = col[static_cast<size_t>(r + u < n ? r + u : 0) * ld];
#pragma unroll
    for (int u = 0; u < N; ++u)
      if (r + u < n) add(v[u]);
  }
}

// grad_wg (two columns per thread) and, in the workgroups behind them, grad_bias from the runs' partial sums, in order
__global__ void __launch_bounds__(256)
gate_products_reduce_kernel(const float *__restrict__ partial, const float *__restrict__ partial_b, int n_run, int E, int d,
                            half_t *__restrict__ grad_w, half_t *__restrict__ grad_bias, int w_wgs) {
  if (static_cast<int>(blockIdx.x) >= w_wgs) {
    const int e = threadIdx.x;
    if (e >= E) return;
    float acc = 0.0f;
    for_column<32>(partial_b + e, E, n_run, [&](float v) { acc += v; });
    grad_bias[e] = static_cast<half_t>(acc);
    return;
  }
  const size_t i = (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 2, n = static_cast<size_t>(E) * d;
  if (i >= n) return;
  float a0 = 0.0f, a1 = 0.0f;
  for_column<32>(reinterpret_cast<const float2 *>(partial + i), n / 2, n_run, [&](const float2 &v) {
    a0 += v.x;
    a1 += v.y;
  });
  *reinterpret_cast<half2v *>(grad_w + i) = half2v{static_cast<half_t>(a0), static_cast<half_t>(a1)};
}

// Tokens per run: about two workgroups per CU, and runs of 32 and more, which keeps the sums of the reduction short.
int products_run(int tokens, int d) {
  const int chunks = (d + kGpCols - 1) / kGpCols;
  const int most = 512 / chunks < 16 ? 16 : 512 / chunks;
  const int run = (tokens + most - 1) / most;
  return (run + 31) / 32 * 32;
}

}  // namespace
}  // namespace ccf

extern "C" size_t ccf_gate_backward_products_workspace_bytes(int tokens, int d_model, int tot_expert) {
  if (tokens <= 0 || d_model <= 0 || tot_expert <= 0 || tot_expert > ccf::kGpMaxExpert) return 0;
  const int run = ccf::products_run(tokens, d_model);
  return sizeof(float) * static_cast<size_t>((tokens + run - 1) / run) * tot_expert * (static_cast<size_t>(d_model) + 1);
}

extern "C" int ccf_gate_backward_products(const void *score, const void *grad_score, const int64_t *idx, const void *x,
                                          const void *wg, int tokens, int d_model, int tot_expert, int top_k, void *grad_x,
                                          void *grad_wg, void *grad_bias, void *workspace, size_t workspace_bytes,
                                          ccf_stream_t stream) {
  using namespace ccf;
  CCF_REQUIRE(score && grad_score && idx && x && wg && (grad_x || grad_wg || grad_bias), CCF_ERR_ARG,
              "gate_backward_products: null pointer");
  CCF_REQUIRE(tokens > 0 && d_model > 0 && d_model % 2 == 0 && tot_expert > 0 && tot_expert <= kGpMaxExpert, CCF_ERR_SHAPE,
              "gate_backward_products: %d tokens of %d and %d experts (tokens, an even width and 1..%d experts)", tokens,
              d_model, tot_expert, kGpMaxExpert);
  CCF_REQUIRE(top_k >= 1 && top_k <= kMaxTopK && top_k <= tot_expert, CCF_ERR_SHAPE,
              "gate_backward_products: top_k=%d outside 1..min(%d, tot_expert=%d)", top_k, kMaxTopK, tot_expert);
  const auto aligned4 = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; };
  CCF_REQUIRE(aligned4(x) && aligned4(wg) && aligned4(grad_x) && aligned4(grad_wg), CCF_ERR_ARG,
              "gate_backward_products: operands must be 4-byte aligned");
  const size_t need = ccf_gate_backward_products_workspace_bytes(tokens, d_model, tot_expert);
  CCF_REQUIRE(workspace && workspace_bytes >= need && (reinterpret_cast<uintptr_t>(workspace) & 7u) == 0, CCF_ERR_WORKSPACE,
              "gate_backward_products: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
  const int run = products_run(tokens, d_model), n_run = (tokens + run - 1) / run;
  float *partial = static_cast<float *>(workspace);
  float *partial_b = partial + static_cast<size_t>(n_run) * tot_expert * d_model;
  const size_t lds = (sizeof(float) + sizeof(half_t)) * kGpCols * tot_expert;
  const auto kernel = top_k <= 2 ? gate_products_kernel<2> : gate_products_kernel<kMaxTopK>;
  if (lds > 32768) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(lds));
    if (e != hipSuccess) return fail(CCF_ERR_HIP, "gate_backward_products: LDS attribute: %s", hipGetErrorString(e));
  }
  hipLaunchKernelGGL(kernel, dim3((d_model + kGpCols - 1) / kGpCols, n_run), dim3(256), lds, as_stream(stream),
                     static_cast<const half_t *>(score), static_cast<const half_t *>(grad_score), idx,
                     static_cast<const half_t *>(x), static_cast<const half_t *>(wg), tokens, top_k, tot_expert, d_model, run,
                     static_cast<half_t *>(grad_x), grad_wg ? partial : nullptr, grad_bias ? partial_b : nullptr);
  if (int rc = check_launch("gate_products_kernel")) return rc;
  if (!grad_wg && !grad_bias) return CCF_OK;
  const size_t pairs = static_cast<size_t>(tot_expert) * d_model / 2;
  const int w_wgs = grad_wg ? static_cast<int>((pairs + 255) / 256) : 0;
  hipLaunchKernelGGL(gate_products_reduce_kernel, dim3(w_wgs + (grad_bias ? 1 : 0)), dim3(256), 0, as_stream(stream), partial,
                     partial_b, n_run, tot_expert, d_model, static_cast<half_t *>(grad_wg), static_cast<half_t *>(grad_bias),
                     w_wgs);
  return check_launch("gate_products_reduce_kernel");
}

extern "C" size_t ccf_gate_backward_workspace_bytes(int tokens, int tot_expert) {
  if (tokens <= 0 || tot_expert <= 0) return 0;
  return sizeof(float) * static_cast<size_t>((tokens + ccf::kGbTokens - 1) / ccf::kGbTokens) * tot_expert;
}

extern "C" int ccf_gate_backward(const void *score, const void *grad_score, const int64_t *idx, int tokens,
                                 int top_k, int tot_expert, void *grad_logits, void *grad_bias, void *workspace,
                                 size_t workspace_bytes, ccf_stream_t stream) {
  using namespace ccf;
  CCF_REQUIRE(tokens >= 0 && tot_expert > 0 && tot_expert <= 1024, CCF_ERR_ARG, "gate_backward: bad size");
  CCF_REQUIRE(top_k >= 1 && top_k <= kMaxTopK && top_k <= tot_expert, CCF_ERR_SHAPE,
              "gate_backward: top_k=%d outside 1..min(%d, tot_expert=%d)", top_k, kMaxTopK, tot_expert);
  if (tokens == 0) {                                 // no rows to write; a sum over nothing
    if (!grad_bias) return CCF_OK;
    hipLaunchKernelGGL(gate_bias_reduce_kernel, dim3((tot_expert + 255) / 256), dim3(256), 0, as_stream(stream),
                       static_cast<const float *>(nullptr), 0, tot_expert, static_cast<half_t *>(grad_bias));
    return check_launch("gate_bias_reduce_kernel");
  }
  CCF_REQUIRE(score && grad_score && idx && grad_logits, CCF_ERR_ARG, "gate_backward: null pointer");
  const size_t need = ccf_gate_backward_workspace_bytes(tokens, tot_expert);
  CCF_REQUIRE(!grad_bias || (workspace && workspace_bytes >= need), CCF_ERR_WORKSPACE,
              "gate_backward: workspace of %zu bytes needed for the bias gradient, %zu given", need, workspace_bytes);
  const int n_wg = (tokens + kGbTokens - 1) / kGbTokens;
  hipLaunchKernelGGL(gate_backward_kernel, dim3(n_wg), dim3(kGbTokens), 0, as_stream(stream),
                     static_cast<const half_t *>(score), static_cast<const half_t *>(grad_score), idx, tokens, top_k,
                     tot_expert, static_cast<half_t *>(grad_logits), grad_bias ? static_cast<float *>(workspace) : nullptr);
  if (int rc = check_launch("gate_backward_kernel")) return rc;
  if (grad_bias) {
    hipLaunchKernelGGL(gate_bias_reduce_kernel, dim3((tot_expert + 255) / 256), dim3(256), 0, as_stream(stream),
                       static_cast<const float *>(workspace), n_wg, tot_expert, static_cast<half_t *>(grad_bias));
    return check_launch("gate_bias_reduce_kernel");
  }
  return CCF_OK;
}

extern "C" int ccf_gate_topk_softmax(const void *x, const void *wg, const void *bg, int tokens,
                                     int d_model, int tot_expert, int top_k, int dtype,
                                     int64_t *idx_out, void *score_out, void *logits_out,
                                     ccf_stream_t stream) {
  return ccf::gate_forward(x, wg, bg, tokens, d_model, tot_expert, top_k, dtype, idx_out, score_out, logits_out, stream,
                           nullptr, 0, nullptr);
}
