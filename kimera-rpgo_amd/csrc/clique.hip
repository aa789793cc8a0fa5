// Maximum clique on the bit-packed PCM adjacency.
//
// HEU_REF mode reproduces FMC::maxCliqueHeu (findCliqueHeu.cpp:32-117, called
// through findMaxCliqueHeu src/utils/GraphUtils.cpp:19-27) bit for bit:
//   * candidates c = 0..n-1 in order, skipped when best > deg(c)   (pruning 1)
//   * S = [c] ++ { u in N(c) : deg(u) >= best } ascending          (pruning 3)
//   * repeat: icc++, m = last of S, S = S /\ N(m) /\ {deg >= best} (pruning 5)
//   * the candidate beating best keeps the working buffer it leaves behind:
//     position p holds the value last written there, not the greedy picks.
// The sequential scan is split into speculative waves: every remaining
// candidate is evaluated in parallel against the current best (one wavefront
// per candidate, S as a bitset in registers), the first candidate that beats
// it is taken, and the scan resumes after it.  Each wave advances best, so
// the number of waves is the number of improvements.  The winner's buffer, the
// reference's stale one, then follows from its picks, every step at once
// (k_rp_*); small graphs, the allocation-free scan and the batch replay it step
// by step on one wavefront.
#include "rpgo_internal.h"

#include <algorithm>
#include <climits>
#include <mutex>
#include <vector>

namespace rpgo {

__global__ void k_degrees(int n, int W, const unsigned long long* __restrict__ adj,
                          int* __restrict__ deg) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n) return;
  // only bits u < n, u != v count (FMC's CSR skips the diagonal, graphIO.cpp:199)
  int s = 0;
  for (int w = 0; w < W; ++w) {
    unsigned long long b = adj[(size_t)v * W + w];
    if (w == W - 1 && (n & 63)) b &= (1ull << (n & 63)) - 1ull;
    if (w == (v >> 6)) b &= ~(1ull << (v & 63));
    s += __popcll(b);
  }
  deg[v] = s;
}

// first_reset (may be null): thread 0 also sets *first_reset to "no winner"
// (candidate n), which k_first_better lowers, so the scan needs no
// host-to-device copy
__global__ void k_dmask(int n, int W, int best, const int* __restrict__ deg,
                        unsigned long long* __restrict__ dmask, unsigned long long* __restrict__ first_reset) {
  const int w = blockIdx.x * blockDim.x + threadIdx.x;
  if (first_reset && w == 0) *first_reset = (unsigned long long)n << 32;
  if (w >= W) return;
  unsigned long long b = 0ull;
  for (int k = 0; k < 64; ++k) {
    const int u = w * 64 + k;
    if (u < n && deg[u] >= best) b |= 1ull << k;
  }
  dmask[w] = b;
}

// words per lane held in registers (n <= 64 * 64 * kMaxWPL)
constexpr int kMaxWPL = 8;
// row words from which the single-graph rounds walk the compacted subgraph
constexpr int kCompactMinW = 64;
// candidates of the single-graph scan's round after its first candidate
constexpr int kScanWindow = 256;
// search nodes the exact mode may visit before it reports failure
constexpr long long kExactNodeBudget = 400000000ll;

// Highest set bit over the wave's distributed bitset; -1 when empty.
// Word w = lane + 64 q, so the highest vertex lies in the highest q with a
// non-empty word, on the highest such lane: one ballot per q (scalar), then
// that lane's top bit by v_readlane, instead of a six-step shuffle reduction.
// Called by whole wavefronts (wave-uniform control flow).
__device__ __forceinline__ int wave_top_bit(const unsigned long long* S, int lane, int W) {
#pragma unroll
  for (int q = kMaxWPL - 1; q >= 0; --q) {
    if (64 * q >= W) continue;  // no words here (wave-uniform)
    const int w = lane + 64 * q;
    const unsigned long long lanes = __ballot(w < W && S[q] != 0ull);
    if (lanes) {
      const int L = 63 - __clzll(lanes);
      return __builtin_amdgcn_readlane(w * 64 + 63 - __clzll(S[q]), L);
    }
  }
  return -1;
}

__device__ __forceinline__ int wave_popcount(const unsigned long long* S) {
  int cnt = 0;
#pragma unroll
  for (int q = 0; q < kMaxWPL; ++q) cnt += __popcll(S[q]);
  return __ockl_wfred_add_i32(cnt);  // DPP wavefront sum
}

__device__ __forceinline__ unsigned long long readlane_u64(unsigned long long v, int l) {
  const unsigned int lo = __builtin_amdgcn_readlane((int)(unsigned int)v, l);
  const unsigned int hi = __builtin_amdgcn_readlane((int)(unsigned int)(v >> 32), l);
  return ((unsigned long long)hi << 32) | lo;
}

// Most rows of one block of the walk that are loaded together (half as many
// with four words a lane, all of them in flight).
constexpr int kWalkChunk = 16;

// Derived rows of an adjacency, for the walk: diag[v] = word v / 64 of row v
// (the 64 x 64 diagonal blocks, contiguous per block), g4 / g8 the ANDs of the
// rows 4 g .. 4 g + 3 and 8 g .. 8 g + 7 (rows of W words).  All null: none.
struct WalkAux {
  const unsigned long long* diag = nullptr;
  const unsigned long long* g4 = nullptr;
  const unsigned long long* g8 = nullptr;
};

// The rows to AND for a set of picks P of block wt: whole aligned groups of
// eight and of four picks take their group row, the rest their own.  Lane k
// returns the k-th row's address (the last one's past the end), *total their
// number; sl is 64 words of LDS.  Each lane places its own rows by a popcount:
// walking the masks a row at a time took the scalar unit longer than the loads.
__device__ __forceinline__ unsigned long long pick_rows(unsigned long long P, const unsigned long long* blk,
                                                        const WalkAux& x, int W, int wt, int lane,
                                                        unsigned long long* sl, int* total) {
  unsigned long long m8 = 0ull, m4 = 0ull, m1 = P;
  int n = 0;
  if (x.g4) {
    unsigned long long t = P & (P >> 1);
    t &= t >> 2;
    m8 = t & (t >> 4) & 0x0101010101010101ull;
    m4 = t & 0x1111111111111111ull & ~(m8 * 255ull);
    m1 = P & ~(m8 * 255ull) & ~(m4 * 15ull);
    if (lane < 8 && ((m8 >> (8 * lane)) & 1ull))
      sl[__popcll(m8 & ((1ull << (8 * lane)) - 1ull))] =
          reinterpret_cast<unsigned long long>(x.g8 + (size_t)(8 * wt + lane) * W);
    n = __popcll(m8);
    if (lane < 16 && ((m4 >> (4 * lane)) & 1ull))
      sl[n + __popcll(m4 & ((1ull << (4 * lane)) - 1ull))] =
          reinterpret_cast<unsigned long long>(x.g4 + (size_t)(16 * wt + lane) * W);
    n += __popcll(m4);
  }
  if ((m1 >> lane) & 1ull)
    sl[n + __popcll(m1 & ((1ull << lane) - 1ull))] = reinterpret_cast<unsigned long long>(blk + (size_t)lane * W);
  n += __popcll(m1);
  // LDS operations of a wavefront are performed in order; the fence keeps the
  // compiler from moving the read
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const unsigned long long v = sl[min(lane, n - 1)];
  __builtin_amdgcn_wave_barrier();
  *total = n;
  return v;
}

// S /\ rows at .. at + K - 1 of pick_rows' list.  A row past the last repeats
// it (a row ANDed twice changes nothing).  Lanes whose word of S is empty read
// word wt of the same rows, one shared line, and keep their zero.  Up to four
// words a lane, all K rows of all words are loaded together; wider bitsets go
// slot by slot, a slot empty on every lane skipped.
template <int K, int NQ>
__device__ __forceinline__ void and_rows(unsigned long long (&S)[NQ], unsigned long long rows, int at, int n_rows,
                                         int W, int wt, int lane) {
  const unsigned long long* rp[K];
#pragma unroll
  for (int k = 0; k < K; ++k)
    rp[k] = reinterpret_cast<const unsigned long long*>(readlane_u64(rows, min(at + k, n_rows - 1)));
  if (NQ <= 4) {
    unsigned long long r[NQ][K];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int w = lane + 64 * q;
      const int wa = (w < W && S[q] != 0ull) ? w : wt;
#pragma unroll
      for (int k = 0; k < K; ++k) r[q][k] = rp[k][wa];
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q)
#pragma unroll
      for (int k = 0; k < K; ++k) S[q] &= r[q][k];
  } else {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (64 * q >= W || !__ballot(lane + 64 * q < W && S[q] != 0ull)) continue;
      const int w = lane + 64 * q;
      const int wa = (w < W && S[q] != 0ull) ? w : wt;
      unsigned long long r[K];
#pragma unroll
      for (int k = 0; k < K; ++k) r[k] = rp[k][wa];
#pragma unroll
      for (int k = 0; k < K; ++k) S[q] &= r[k];
    }
  }
}

// Greedy size icc(c, best) of candidate c, one wavefront (S as a bitset in
// registers, word w = lane + 64 q; dmask holds the deg >= best filter, LDS or
// global).  The walk picks the highest vertex m of S and keeps S /\ N(m)
// until S is empty; it is taken a word of S at a time.  While S
// keeps a vertex of its highest non-empty word wt, every pick lies in wt: the
// vertices of S outside wt are all lower.  So the picks inside wt follow from
// the 64 x 64 diagonal block of the adjacency alone (one row word per vertex,
// loaded at once, the walk then runs on scalars by v_readlane), and the word
// leaves S when its last vertex is picked or removed.  The other words of S
// keep the common neighbours of those picks, whose rows are loaded
// kWalkChunk at a time with no load waiting on another.  A dense block then
// costs two or three load round trips per 64 vertices instead of one per pick.
// What bounds the rounds is the row words the walks load (thousands of walks
// at once) and, for the longest walk, its round trips.  In a near-complete
// block most picks fill whole groups of eight, so the group rows (WalkAux) cut
// both: about 15 rows a block instead of 61 where 96 % are picked.  Walks over
// 5,000 vertices took 0.48-0.9 ms a round with single rows and a scalar step
// per pick, 0.20-0.31 ms so; over 1,000 vertices 82 and 36 us.
// Only icc > best matters to the scan, so the walk stops early (INT_MIN) after a
// chunk of rows once it cannot get there (the word's picks are all counted,
// and every later pick removes at least itself from S, so at most |S| + 1
// increments remain); a candidate that beats best never stops early and
// returns its exact size, its picks as a bitset in picks_out (W words, may be
// null).
template <int NQ>
__device__ __forceinline__ int icc_walk_q(int W, int c, const unsigned long long* __restrict__ adj,
                                          const WalkAux& aux, const unsigned long long* dmask, int lane, int best,
                                          unsigned long long* sl, unsigned long long* __restrict__ picks_out) {
  unsigned long long S[NQ], T[NQ];
  int left = 0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int w = lane + 64 * q;
    S[q] = (w < W) ? (adj[(size_t)c * W + w] & dmask[w] &
                      ((w == (c >> 6)) ? ~(1ull << (c & 63)) : ~0ull))
                   : 0ull;
    T[q] = 0ull;
    left += __popcll(S[q]);
  }
  if (__ockl_wfred_add_i32(left) + 1 <= best) return INT_MIN;
  int picks = 0;
  // the diagonal words of block dwt, loaded while the block above it is walked
  int dwt = -1;
  unsigned long long dv = 0ull;
  for (;;) {
    // highest non-empty word wt of S and its vertices U (wave-uniform)
    int wt = -1;
    unsigned long long U = 0ull;
#pragma unroll
    for (int q = NQ - 1; q >= 0; --q) {
      if (wt >= 0 || 64 * q >= W) continue;  // no words here (wave-uniform)
      const unsigned long long lanes = __ballot(lane + 64 * q < W && S[q] != 0ull);
      if (lanes) {
        const int L = 63 - __clzll(lanes);
        wt = 64 * q + L;
        U = readlane_u64(S[q], L);
      }
    }
    if (wt < 0) break;  // S held only the seed c
    const unsigned long long* blk = adj + (size_t)64 * wt * W;  // rows 64 wt .. 64 wt + 63
    // lane k: the vertices of U below k that k's row lacks, for k in U (word wt
    // of row 64 wt + k; the other lanes read the top vertex's word and drop
    // it).  Picking k removes just these, so the picks are U less what the
    // picked vertices with a conflict remove, highest first: a few scalar steps
    // in a near-complete block, where a step per pick bound the rounds
    unsigned long long P = U;
    if (U & (U - 1)) {
      const bool in = (U >> lane) & 1ull;
      const int k = in ? lane : 63 - __clzll(U);
      unsigned long long v = dv;
      if (dwt != wt) v = aux.diag ? aux.diag[64 * wt + k] : blk[(size_t)k * W + wt];
      const unsigned long long x = in ? U & ~v & ((1ull << lane) - 1ull) : 0ull;
      unsigned long long C = __ballot(x != 0ull);
      while (C &= P) {
        const int h = 63 - __clzll(C);
        C ^= 1ull << h;
        P &= ~readlane_u64(x, h);
      }
    }
    picks += __popcll(P);
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      if (lane + 64 * q == wt) {
        S[q] = 0ull;
        T[q] = P;
      }
    if (aux.diag && wt > 0) {
      dwt = wt - 1;
      dv = aux.diag[64 * dwt + lane];
    }
    // S /\ N(p) over the picks p, a chunk of rows at a time; a short
    // remainder takes the next power of two, so few loads are wasted
    constexpr int KC = NQ == 4 ? kWalkChunk / 2 : kWalkChunk;
    int total;
    const unsigned long long rows = pick_rows(P, blk, aux, W, wt, lane, sl, &total);
    for (int at = 0; at < total;) {
      const int np = total - at;
      if (np > KC / 2) and_rows<KC, NQ>(S, rows, at, total, W, wt, lane);
      else if (np > KC / 4) and_rows<KC / 2, NQ>(S, rows, at, total, W, wt, lane);
      else if (np > 1) and_rows<KC / 4, NQ>(S, rows, at, total, W, wt, lane);
      else and_rows<1, NQ>(S, rows, at, total, W, wt, lane);
      at += KC;
      // every pick of word wt is already counted and S only shrinks
      left = 0;
#pragma unroll
      for (int q = 0; q < NQ; ++q) left += __popcll(S[q]);
      if (picks + __ockl_wfred_add_i32(left) + 1 <= best) return INT_MIN;
    }
  }
  if (picks_out && picks + 1 > best) {
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      if (lane + 64 * q < W) picks_out[lane + 64 * q] = T[q];
  }
  return picks + 1;
}

// one, two and four words a lane (up to 4,096, 8,192 and 16,384 vertices) load
// whole chunks at once; sl: 64 words of LDS per wavefront
__device__ __forceinline__ int icc_walk(int W, int c, const unsigned long long* __restrict__ adj, const WalkAux& aux,
                                        const unsigned long long* dmask, int lane, int best, unsigned long long* sl,
                                        unsigned long long* __restrict__ picks_out = nullptr) {
  if (W <= 64) return icc_walk_q<1>(W, c, adj, aux, dmask, lane, best, sl, picks_out);
  if (W <= 128) return icc_walk_q<2>(W, c, adj, aux, dmask, lane, best, sl, picks_out);
  if (W <= 256) return icc_walk_q<4>(W, c, adj, aux, dmask, lane, best, sl, picks_out);
  return icc_walk_q<kMaxWPL>(W, c, adj, aux, dmask, lane, best, sl, picks_out);
}

// The derived rows of n rows (*n_dev when given) of W = ceil(n/64) words: one
// thread per word of a group of eight.  Groups past the last whole one are
// never read (a pick set never covers them).
__global__ void __launch_bounds__(256) k_walk_aux(int n, const int* __restrict__ n_dev,
                                                  const unsigned long long* __restrict__ adj,
                                                  unsigned long long* __restrict__ diag,
                                                  unsigned long long* __restrict__ g4,
                                                  unsigned long long* __restrict__ g8) {
  if (n_dev) n = *n_dev;
  const int W = (n + 63) / 64, ng = (n + 7) / 8;
  const long long t = (long long)blockIdx.x * 256 + threadIdx.x;
  if (t >= (long long)ng * W) return;
  const int g = (int)(t / W), w = (int)(t - (long long)g * W);
  unsigned long long r[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int v = 8 * g + k;
    r[k] = v < n ? adj[(size_t)v * W + w] : 0ull;
    if (v < n && w == (v >> 6)) diag[v] = r[k];
  }
  const unsigned long long a = r[0] & r[1] & r[2] & r[3], b = r[4] & r[5] & r[6] & r[7];
  g4[(size_t)2 * g * W + w] = a;
  g4[(size_t)(2 * g + 1) * W + w] = b;
  g8[(size_t)g * W + w] = a & b;
}
constexpr size_t walk_aux_words(size_t n) {  // diag, then g4, then g8
  const size_t W = (n + 63) / 64, ng = (n + 7) / 8;
  return n + 3 * ng * W;
}
__host__ __device__ inline WalkAux walk_aux_at(unsigned long long* base, int n) {
  const size_t W = (size_t)(n + 63) / 64, ng = (size_t)(n + 7) / 8;
  return WalkAux{base, base + n, base + n + 2 * ng * W};
}

// Picks whose rows a replay stages in LDS at once: kReplayChunk x kMaxWPL x
// 64 words of 8 B (32 KB) per replaying wavefront.
constexpr int kReplayChunk = 8;
constexpr int kReplayLds = kReplayChunk * kMaxWPL * 64;

// Replay of the winning candidate c: the walk of icc_walk, one word of S at a
// time, that also writes the reference's buffer positions 0..s0-1 (position p
// keeps the value last written to it) and returns the greedy size.  One
// wavefront; rl is its LDS staging area (kReplayLds words).
// Step t (pick m_t, S_t -> S_{t+1}) leaves the list at s_{t+1} = 1 + |S_{t+1}|
// entries (the seed stays in front) and positions [s_{t+1}, s_t) keep S_t's
// entries: position p holds S_t's element of rank p - 1 in ascending order.
// The writes need |S_{t+1}| after every pick, so within word wt the picks'
// rows are staged in LDS kReplayChunk at a time (loads in flight together);
// the steps then run on registers and LDS: S_t is U_t (the rest of word wt,
// above every other vertex of S_t) and the lower words L_t.
__device__ __forceinline__ int replay_walk(int W, int c, const unsigned long long* __restrict__ adj,
                                           const unsigned long long* dmask, int* __restrict__ out, int lane,
                                           unsigned long long* rl, int* s0 = nullptr) {
  unsigned long long S[kMaxWPL];
#pragma unroll
  for (int q = 0; q < kMaxWPL; ++q) {
    const int w = lane + 64 * q;
    S[q] = (w < W) ? (adj[(size_t)c * W + w] & dmask[w] &
                      ((w == (c >> 6)) ? ~(1ull << (c & 63)) : ~0ull))
                   : 0ull;
  }
  if (lane == 0) out[0] = c;
  int s_t = 1 + wave_popcount(S);  // list size before the step
  if (s0) *s0 = s_t;                // positions 0 .. s_t - 1 are written
  int picks = 0;
  for (;;) {
    int wt = -1;
    unsigned long long U = 0ull;
#pragma unroll
    for (int q = kMaxWPL - 1; q >= 0; --q) {
      if (64 * q >= W) continue;
      const unsigned long long lanes = __ballot(lane + 64 * q < W && S[q] != 0ull);
      if (lanes) {
        const int L = 63 - __clzll(lanes);
        wt = 64 * q + L;
        U = readlane_u64(S[q], L);
        break;
      }
    }
    // S held only the seed: the last step leaves the list empty (s_t == 1,
    // nothing is written)
    if (wt < 0) return picks + 1;
#pragma unroll
    for (int q = 0; q < kMaxWPL; ++q)
      if (lane + 64 * q == wt) S[q] = 0ull;  // S is L_t from here
    const unsigned long long* blk = adj + (size_t)64 * wt * W;
    unsigned long long dw = 0ull;
    if (U & (U - 1)) {
      const bool in = (U >> lane) & 1ull;
      const unsigned long long v = blk[(size_t)(in ? lane : 63 - __clzll(U)) * W + wt];
      dw = in ? v : 0ull;
    }
    unsigned long long P = 0ull, Ug = U;
    while (Ug) {
      const int p = 63 - __clzll(Ug);
      P |= 1ull << p;
      Ug &= readlane_u64(dw, p) & ~(1ull << p);
    }
    while (P) {
      // the next kReplayChunk picks, highest first (a short chunk repeats
      // its first pick: ANDing a row twice changes nothing)
      int pk[kReplayChunk];
      int nk = 0;
#pragma unroll
      for (int k = 0; k < kReplayChunk; ++k) {
        pk[k] = P ? 63 - __clzll(P) : pk[0];
        if (P) {
          P &= ~(1ull << pk[k]);
          ++nk;
        }
      }
      // per word q: the chunk's row words loaded together, kept in LDS for
      // the writes (word lane + 64 q of pick k at rl[(k kMaxWPL + q) 64 +
      // lane]; each lane reads back only its own), and L after each pick with
      // its size; the kReplayChunk wave sums are then taken together
      unsigned long long L0[kMaxWPL];
      int cnt[kReplayChunk];
#pragma unroll
      for (int k = 0; k < kReplayChunk; ++k) cnt[k] = 0;
#pragma unroll
      for (int q = 0; q < kMaxWPL; ++q) {
        L0[q] = S[q];
        if (64 * q >= W) continue;
        const int w = lane + 64 * q;
        const int wa = (w < W && S[q] != 0ull) ? w : wt;  // dead lanes: one shared line
        unsigned long long r[kReplayChunk];
#pragma unroll
        for (int k = 0; k < kReplayChunk; ++k) r[k] = blk[(size_t)pk[k] * W + wa];
        unsigned long long a = S[q];
#pragma unroll
        for (int k = 0; k < kReplayChunk; ++k) {
          rl[(k * kMaxWPL + q) * 64 + lane] = r[k];
          a &= r[k];
          cnt[k] += __popcll(a);
        }
        S[q] = a;
      }
#pragma unroll
      for (int k = 0; k < kReplayChunk; ++k) cnt[k] = __ockl_wfred_add_i32(cnt[k]);
#pragma unroll
      for (int k = 0; k < kReplayChunk; ++k) {
        if (k >= nk) break;
        const int m = 63 - __clzll(U);  // the k-th staged pick
        const unsigned long long Un = U & readlane_u64(dw, m) & ~(1ull << m);
        const int s_next = 1 + __popcll(Un) + cnt[k];
        // positions [s_next, s_t): the top of S_t, first U_t (highest bit
        // first), then L_t, rebuilt from the staged rows when reached
        int p = s_t - 1;
        unsigned long long Ut = U;
        for (; p >= s_next && Ut; --p) {
          const int t = 63 - __clzll(Ut);
          if (lane == 0) out[p] = 64 * wt + t;
          Ut &= ~(1ull << t);
        }
        if (p >= s_next) {
          unsigned long long Lp[kMaxWPL];
#pragma unroll
          for (int q = 0; q < kMaxWPL; ++q) {
            Lp[q] = L0[q];
#pragma unroll
            for (int j = 0; j < k; ++j)
              if (64 * q < W) Lp[q] &= rl[(j * kMaxWPL + q) * 64 + lane];
          }
          for (; p >= s_next; --p) {
            const int t = wave_top_bit(Lp, lane, W);
            if (lane == 0) out[p] = t;
            const int w = t >> 6;
#pragma unroll
            for (int q = 0; q < kMaxWPL; ++q)
              if (lane + 64 * q == w) Lp[q] &= ~(1ull << (t & 63));
          }
        }
        U = Un;
        s_t = s_next;
        ++picks;
      }
    }
  }
}

// A walk against best stays inside the vertices with deg >= best (dmask): S
// starts within it and only shrinks, and the candidates that walk pass the
// same filter.  The rounds of the single-graph scan therefore walk the
// subgraph of those vertices, renumbered in the same order (so "highest"
// picks the same vertex), with rows of ceil(n'/64) words instead of W: the
// same sizes for fewer row bytes, which bound the rounds.
// One workgroup of 512: new indices by a scan of the dmask words' popcounts.
__global__ void __launch_bounds__(512) k_compact_index(int n, int W, const unsigned long long* __restrict__ dmask,
                                                       int* __restrict__ cidx, int* __restrict__ ccol,
                                                       unsigned long long* __restrict__ cdmask,
                                                       int* __restrict__ cn) {
  __shared__ int pre[512];
  const int t = threadIdx.x;
  const unsigned long long b = t < W ? dmask[t] : 0ull;
  pre[t] = __popcll(b);
  __syncthreads();
  for (int d = 1; d < 512; d <<= 1) {  // inclusive scan
    const int v = t >= d ? pre[t - d] : 0;
    __syncthreads();
    pre[t] += v;
    __syncthreads();
  }
  const int total = pre[511];
  int r = pre[t] - __popcll(b);
  if (t < W) {
    for (int k = 0; k < 64; ++k) {
      const int v = 64 * t + k;
      if (v >= n) break;
      if ((b >> k) & 1ull) {
        cidx[v] = r;
        ccol[r++] = v;
      } else {
        cidx[v] = -1;
      }
    }
  }
  if (t < W) {
    const int lo = 64 * t;
    cdmask[t] = total >= lo + 64 ? ~0ull : (total > lo ? (1ull << (total - lo)) - 1ull : 0ull);
  }
  if (t == 0) *cn = total;
}

// word w' of new row v': bits of old row ccol[v'] at old columns
// ccol[64 w' .. 64 w' + 63] (ascending, so the old words come in order)
__global__ void k_compact_adj(int n, int W, const unsigned long long* __restrict__ adj,
                              const int* __restrict__ ccol, const int* __restrict__ cn,
                              unsigned long long* __restrict__ cadj) {
  const int nc = *cn, Wc = (nc + 63) / 64;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (long long)nc * Wc) return;
  const int vr = (int)(t / Wc), wr = (int)(t % Wc);
  const unsigned long long* row = adj + (size_t)ccol[vr] * W;
  unsigned long long out = 0ull, cur = 0ull;
  int cw = -1;
  for (int k = 0; k < 64; ++k) {
    const int u2 = 64 * wr + k;
    if (u2 >= nc) break;
    const int u = ccol[u2];
    if ((u >> 6) != cw) {
      cw = u >> 6;
      cur = row[cw];
    }
    out |= ((cur >> (u & 63)) & 1ull) << k;
  }
  cadj[(size_t)vr * Wc + wr] = out;
}

// k_icc on the compacted graph; results by old index.
__global__ void __launch_bounds__(256) k_icc_compact(int n, int pos, int best, const int* __restrict__ deg,
                                                     const int* __restrict__ cidx, const int* __restrict__ cn,
                                                     const unsigned long long* __restrict__ cadj,
                                                     const unsigned long long* __restrict__ cdmask,
                                                     WalkAux aux, unsigned long long* __restrict__ picks,
                                                     int* __restrict__ icc_out) {
  const int c = pos + blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= n) return;
  const int lane = threadIdx.x & 63;
  if (best > deg[c]) {  // pruning 1
    if (lane == 0) icc_out[c] = INT_MIN;
    return;
  }
  __shared__ unsigned long long sl[4][64];
  const int Wc = (*cn + 63) / 64;
  const int icc = icc_walk(Wc, cidx[c], cadj, aux, cdmask, lane, best, sl[threadIdx.x >> 6],
                           picks + (size_t)cidx[c] * Wc);
  if (lane == 0) icc_out[c] = icc;
}

// ---------------------------------------------------------------------------
// The winner's buffer, all steps at once.  With the picks m_0, m_1, ... known
// from the walk, a vertex u of the first set S_0 leaves at step e(u), the first
// t with u not in N(m_t) (its own step if it is picked), so S_t is the set
// {u : e(u) >= t}, the list before step t has s_t = 1 + |S_t| entries, and
// step t leaves positions [s_{t+1}, s_t) holding the highest of S_t's vertices
// (replay_walk).  Exit steps come from one pass over the picks' rows, sizes
// from their histogram, and every step writes its positions by itself.  The
// sequential replay of a 4,816-vertex clique took 1.9 ms on one wavefront.
// The number of picks listed must be the greedy size less one, K, and S_0 must
// be empty after them; otherwise nothing is read from the list and the size
// reported is -1.
// ---------------------------------------------------------------------------
// Vertices from which this replaces replay_walk: five launches of about 5 us
// against 48 us for the step-by-step replay at 400 vertices, 7 us at 75
constexpr int kReplayParMin = 320;

// picks of candidate c as a list, highest first, in the graph's own numbering
// (ccol: old index of a compacted vertex, or null); 512 threads, one per word
__global__ void __launch_bounds__(512) k_winner_list(int c, int W, const int* __restrict__ cidx,
                                                     const int* __restrict__ ccol, const int* __restrict__ cn,
                                                     const unsigned long long* __restrict__ picks,
                                                     int* __restrict__ list, int* __restrict__ count) {
  __shared__ int suf[512];
  const int t = threadIdx.x;
  const int Wp = cn ? (*cn + 63) / 64 : W;
  const unsigned long long* row = picks + (size_t)(cidx ? cidx[c] : c) * Wp;
  unsigned long long b = t < Wp ? row[t] : 0ull;
  suf[t] = __popcll(b);
  __syncthreads();
  for (int d = 1; d < 512; d <<= 1) {  // inclusive suffix sums
    const int v = t + d < 512 ? suf[t + d] : 0;
    __syncthreads();
    suf[t] += v;
    __syncthreads();
  }
  int o = suf[t] - __popcll(b);
  while (b) {
    const int k = 63 - __clzll(b);
    b &= ~(1ull << k);
    const int v = 64 * t + k;
    list[o++] = ccol ? ccol[v] : v;
  }
  if (t == 0) *count = suf[0];
}

__device__ __forceinline__ unsigned long long replay_start_word(int c, int w, int W,
                                                                const unsigned long long* __restrict__ adj,
                                                                const unsigned long long* __restrict__ dmask) {
  return adj[(size_t)c * W + w] & dmask[w] & (w == (c >> 6) ? ~(1ull << (c & 63)) : ~0ull);
}

__global__ void k_rp_init(int n, int* __restrict__ exit_step, int* __restrict__ hist) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) exit_step[t] = INT_MAX;
  if (t <= n) hist[t] = 0;
}

// one wavefront per (word w, 64 picks): for every vertex of S_0's word w the
// first of these picks whose row lacks it
__global__ void __launch_bounds__(256) k_rp_exit(int W, int c, int K, const unsigned long long* __restrict__ adj,
                                                 const unsigned long long* __restrict__ dmask,
                                                 const int* __restrict__ list, const int* __restrict__ count,
                                                 int* __restrict__ exit_step) {
  const int w = blockIdx.x, j = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (64 * j >= K || *count != K) return;
  const unsigned long long s0 = replay_start_word(c, w, W, adj, dmask);
  if (!s0) return;
  const int t = 64 * j + lane;
  unsigned long long r = ~0ull;
  if (t < K) {
    const int m = list[t];
    r = adj[(size_t)m * W + w];
    if ((m >> 6) == w) r &= ~(1ull << (m & 63));
  }
  int first = 64;
#pragma unroll 8
  for (int b = 0; b < 64; ++b) {
    const unsigned long long z = __ballot(!((r >> b) & 1ull));
    if (lane == b && z) first = __builtin_ctzll(z);
  }
  if (((s0 >> lane) & 1ull) && first < 64) atomicMin(&exit_step[64 * w + lane], 64 * j + first);
}

// vertices per exit step; hist[K]: those still there after the last pick
__global__ void k_rp_hist(int n, int W, int c, int K, const unsigned long long* __restrict__ adj,
                          const unsigned long long* __restrict__ dmask, const int* __restrict__ exit_step,
                          int* __restrict__ hist) {
  const int u = blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n || !((replay_start_word(c, u >> 6, W, adj, dmask) >> (u & 63)) & 1ull)) return;
  atomicAdd(&hist[min(exit_step[u], K)], 1);
}

// sizes: sz[t] = s_t for t = 0 .. K, from s_K = 1 up; res[0] = greedy size,
// res[1] = s_0.  One workgroup.
__global__ void __launch_bounds__(1024) k_rp_sizes(int K, const int* __restrict__ hist, const int* __restrict__ count,
                                                   int* __restrict__ sz, int* __restrict__ res) {
  __shared__ int sum[16];
  __shared__ int base;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (tid == 0) {
    base = 1;
    sz[K] = 1;
  }
  __syncthreads();
  for (int hi = K; hi > 0; hi -= 1024) {  // steps hi-1 down to hi-1024
    const int t = hi - 1 - tid;
    int v = t >= 0 ? hist[t] : 0;
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(v, d);
      if (lane >= d) v += o;
    }
    if (lane == 63) sum[wid] = v;
    __syncthreads();
    int pre = base;
    for (int k = 0; k < wid; ++k) pre += sum[k];
    if (t >= 0) sz[t] = pre + v;
    __syncthreads();
    if (tid == 1023) base = pre + v;
    __syncthreads();
  }
  if (tid == 0) {
    res[0] = *count == K && hist[K] == 0 ? K + 1 : -1;
    res[1] = base;
  }
}

// one wavefront per step t: positions s_t - 1 down to s_{t+1} take S_t's
// highest vertices, from the pick m_t (the highest) down
__global__ void __launch_bounds__(256) k_rp_write(int n, int W, int c, int K,
                                                  const unsigned long long* __restrict__ adj,
                                                  const unsigned long long* __restrict__ dmask,
                                                  const int* __restrict__ list, const int* __restrict__ count,
                                                  const int* __restrict__ exit_step, const int* __restrict__ sz,
                                                  int* __restrict__ out) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x == 0) out[0] = c;
  if (t >= K || *count != K) return;
  int p = sz[t] - 1;
  const int lo = sz[t + 1];
  for (int w = list[t] >> 6; w >= 0 && p >= lo; --w) {
    const int u = 64 * w + lane;
    const unsigned long long s0 = replay_start_word(c, w, W, adj, dmask);
    const unsigned long long in = __ballot(((s0 >> lane) & 1ull) && u < n && exit_step[u] >= t);
    const int above = __popcll(in & ~((2ull << lane) - 1ull));  // S_t's vertices over u in this word
    if (((in >> lane) & 1ull) && p - above >= lo) out[p - above] = u;
    p -= __popcll(in);
  }
}

// One wavefront per candidate c >= pos: greedy size icc(c, best).
__global__ void __launch_bounds__(256) k_icc(int n, int W, int pos, int best,
                                             const unsigned long long* __restrict__ adj,
                                             const int* __restrict__ deg,
                                             const unsigned long long* __restrict__ dmask, WalkAux aux,
                                             unsigned long long* __restrict__ picks, int* __restrict__ icc_out) {
  const int c = pos + blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= n) return;
  const int lane = threadIdx.x & 63;
  if (best > deg[c]) {  // pruning 1
    if (lane == 0) icc_out[c] = INT_MIN;
    return;
  }
  __shared__ unsigned long long sl[4][64];
  const int icc = icc_walk(W, c, adj, aux, dmask, lane, best, sl[threadIdx.x >> 6],
                           picks ? picks + (size_t)c * W : nullptr);
  if (lane == 0) icc_out[c] = icc;
}

// the first candidate that beats best and its size, packed (candidate high)
__global__ void k_first_better(int end, int pos, int best, const int* __restrict__ icc,
                               unsigned long long* __restrict__ first) {
  const int c = pos + blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= end) return;
  const int k = icc[c];
  if (k > best) atomicMin(first, (unsigned long long)c << 32 | (unsigned int)k);
}

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2))) k_replay(int n, int W, int c, int best,
                                               const unsigned long long* __restrict__ adj,
                                               const unsigned long long* __restrict__ dmask,
                                               int* __restrict__ out, int* __restrict__ icc_out) {
  __shared__ unsigned long long rl[kReplayLds];
  const int icc = replay_walk(W, c, adj, dmask, out, threadIdx.x, rl);
  if (threadIdx.x == 0) *icc_out = icc;
  (void)best;
  (void)n;
}

// ---------------------------------------------------------------------------
// Batched heuristic: one workgroup of NW wavefronts per graph runs the whole
// sequential scan of FMC::maxCliqueHeu on the device.  Candidates are taken
// in rounds of NW consecutive ones (one per wavefront) against the current
// best; the first candidate of the first round that beats best is the one
// the sequential scan takes, and the scan resumes after it.  The winner is
// replayed by wavefront 0.  Graph g's adjacency starts at adj_off[g] with m[g]
// rows of ceil(m[g]/64) words; its degrees and clique go to lc_off[g].
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Chip-wide rounds of the batched scan.  One workgroup per graph leaves the
// largest graphs' scans on one CU each.  A round instead evaluates, for every
// graph still scanning, a window of kCbWindow candidates from its position
// with its current best, one wavefront each over the whole chip.  The first
// candidate of the window whose greedy size beats best is the scan's next
// winner: every candidate before it saw the same best in the sequential scan
// and did not beat it.  The position moves past the winner (or past the
// window), and candidates after a winner are evaluated again next round with
// the new best.
// ---------------------------------------------------------------------------
// 256 candidates per graph per round: on the 256-graph batch (up to ~6,000
// accepted loop closures per graph) the clique stage took 22.4 / 19.5 / 21.4 /
// 27.0 ms with windows of 128 / 256 / 512 / 1,024 on MI355X (wider windows
// re-evaluate more candidates after each winner, narrower ones need more rounds)
constexpr int kCbWindow = 256;   // candidates per graph per round
// vertices from which a graph of the batch gets group rows (3 ceil(n/8) rows,
// which fit the n rows of its adjacency region from 5 on)
constexpr int kCbGroupMin = 64;
constexpr int kCbExtraRounds = 8;  // rounds for winners, beyond one per window of the largest
                                   // graph; the per-graph scan finishes what is left

struct CbState {
  int best, pos, win, win_best;
};

__global__ void k_cb_init(int n_graphs, CbState* __restrict__ st) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g < n_graphs) st[g] = CbState{-1, 0, -1, -1};
}

// deg[v] of every vertex of every graph (vertex slots indexed like the loop
// closures; slots beyond a graph's accepted count are left alone)
__global__ void k_cb_degrees(long long n_slots, const int* __restrict__ slot_graph,
                             const long long* __restrict__ adj_off, const long long* __restrict__ lc_off,
                             const int* __restrict__ m_arr, const unsigned long long* __restrict__ adj_all,
                             int* __restrict__ deg_all, unsigned long long* __restrict__ diag_all) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_slots) return;
  const int g = slot_graph[t];
  const int v = (int)(t - lc_off[g]), n = m_arr[g];
  if (v >= n) return;
  const int W = (n + 63) / 64;
  const unsigned long long* A = adj_all + adj_off[g];
  int d = 0;
  for (int w = 0; w < W; ++w) {
    unsigned long long b = A[(size_t)v * W + w];
    if (w == W - 1 && (n & 63)) b &= (1ull << (n & 63)) - 1ull;
    if (w == (v >> 6)) b &= ~(1ull << (v & 63));
    d += __popcll(b);
  }
  deg_all[t] = d;
  diag_all[t] = A[(size_t)v * W + (v >> 6)];
}

// Group rows of every graph of at least kCbGroupMin vertices (WalkAux's g4 then
// g8, at the graph's adjacency offset): one wavefront per group of eight rows
__global__ void __launch_bounds__(256) k_cb_groups(long long n_slots, const int* __restrict__ slot_graph,
                                                   const long long* __restrict__ adj_off,
                                                   const long long* __restrict__ lc_off,
                                                   const int* __restrict__ m_arr,
                                                   const unsigned long long* __restrict__ adj_all,
                                                   unsigned long long* __restrict__ grp_all) {
  const long long t = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= n_slots) return;
  const int g = slot_graph[t];
  const int v = (int)(t - lc_off[g]), n = m_arr[g];
  if ((v & 7) || v >= n || n < kCbGroupMin) return;
  const int W = (n + 63) / 64, ng = (n + 7) / 8;
  const unsigned long long* A = adj_all + adj_off[g];
  unsigned long long* G = grp_all + adj_off[g];
  for (int w = threadIdx.x & 63; w < W; w += 64) {
    unsigned long long r[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = v + k < n ? A[(size_t)(v + k) * W + w] : 0ull;
    const unsigned long long a = r[0] & r[1] & r[2] & r[3], b = r[4] & r[5] & r[6] & r[7];
    G[(size_t)(v / 4) * W + w] = a;
    G[(size_t)(v / 4 + 1) * W + w] = b;
    G[(size_t)(2 * ng + v / 8) * W + w] = a & b;
  }
}

__device__ __forceinline__ WalkAux cb_aux(int n, long long adj_off, long long lc_off, const unsigned long long* diag,
                                          const unsigned long long* grp) {
  if (!diag) return WalkAux{};
  if (n < kCbGroupMin) return WalkAux{diag + lc_off, nullptr, nullptr};
  const int W = (n + 63) / 64, ng = (n + 7) / 8;
  return WalkAux{diag + lc_off, grp + adj_off, grp + adj_off + (size_t)2 * ng * W};
}

// degree filter deg >= best of every graph still scanning; word w of graph g
// at dm[lc_off[g] + w]
__global__ void k_cb_mask(long long n_slots, const int* __restrict__ slot_graph,
                          const long long* __restrict__ lc_off, const int* __restrict__ m_arr,
                          const int* __restrict__ deg_all, const CbState* __restrict__ st,
                          unsigned long long* __restrict__ dm) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_slots) return;
  const int g = slot_graph[t];
  const int w = (int)(t - lc_off[g]), n = m_arr[g];
  if (w >= (n + 63) / 64 || st[g].pos >= n) return;
  const int best = st[g].best;
  const int* deg = deg_all + lc_off[g];
  unsigned long long b = 0ull;
  for (int k = 0; k < 64; ++k) {
    const int u = w * 64 + k;
    if (u < n && deg[u] >= best) b |= 1ull << k;
  }
  dm[t] = b;
}

// one wavefront per (graph, window slot): greedy size of candidate pos + k.
// Workgroup b runs on XCD x = b % 8; the XCD's i-th workgroup takes window
// quarter i % (kCbWindow / 4) of the (i / (kCbWindow / 4))-th graph of XCD x's
// group in xorder, so each graph's walks share one L2.
__global__ void __launch_bounds__(256) k_cb_icc(int n_graphs, const long long* __restrict__ adj_off,
                                                const long long* __restrict__ lc_off,
                                                const int* __restrict__ m_arr,
                                                const unsigned long long* __restrict__ adj_all,
                                                const int* __restrict__ deg_all,
                                                const unsigned long long* __restrict__ dm,
                                                const CbState* __restrict__ st, const int* __restrict__ xorder,
                                                const unsigned long long* __restrict__ diag,
                                                const unsigned long long* __restrict__ grp,
                                                int* __restrict__ icc_out) {
  constexpr int kBlkPerGraph = kCbWindow / 4;
  const int x = blockIdx.x & 7;
  const int i = (int)(blockIdx.x >> 3);
  const int gi = xorder[n_graphs + x] + i / kBlkPerGraph;
  if (gi >= xorder[n_graphs + x + 1]) return;  // beyond this XCD's group
  const int g = xorder[gi];
  const int k = (i % kBlkPerGraph) * 4 + (threadIdx.x >> 6);
  const long long t = (long long)g * kCbWindow + k;
  const int n = m_arr[g], pos = st[g].pos, best = st[g].best;
  const int c = pos + k;
  if (pos >= n || c >= n) return;  // the select step reads only slots below n - pos
  const int lane = threadIdx.x & 63;
  __shared__ unsigned long long sl[4][64];
  int icc = INT_MIN;
  // best < 1: the window's first candidate wins (every greedy size is >= 1),
  // so the others need no walk
  if (!(best > deg_all[lc_off[g] + c]) && (best >= 1 || k == 0))  // pruning 1
    icc = icc_walk((n + 63) / 64, c, adj_all + adj_off[g], cb_aux(n, adj_off[g], lc_off[g], diag, grp), dm + lc_off[g],
                   lane, best, sl[threadIdx.x >> 6]);
  if (lane == 0) icc_out[t] = icc;
}

// one wavefront per graph: the window's first winner (by ballot over 64
// slots at a time), or the next window
__global__ void __launch_bounds__(256) k_cb_select(int n_graphs, const int* __restrict__ m_arr,
                                                   const int* __restrict__ icc, CbState* __restrict__ st) {
  const int g = blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (g >= n_graphs) return;
  CbState s = st[g];
  const int n = m_arr[g];
  if (s.pos >= n) return;
  const int span = min(kCbWindow, n - s.pos);
  const int* row = icc + (size_t)g * kCbWindow;
  int k = span;
  for (int base = 0; base < span; base += 64) {
    const int kk = base + lane;
    const unsigned long long b = __ballot(kk < span && row[kk] > s.best);
    if (b) {
      k = base + __builtin_ctzll(b);
      break;
    }
  }
  if (lane != 0) return;
  if (k < span) {
    s.win = s.pos + k;
    s.win_best = s.best;
    s.best = row[k];
    s.pos = s.pos + k + 1;
  } else {
    s.pos += span;
  }
  st[g] = s;
}

template <int NW>
__global__ void __launch_bounds__(64 * NW) k_clique_batch(int n_graphs, const long long* __restrict__ adj_off,
                                                          const long long* __restrict__ lc_off,
                                                          const int* __restrict__ m_arr,
                                                          const unsigned long long* __restrict__ adj_all,
                                                          int* __restrict__ deg_all, int* __restrict__ out_all,
                                                          int* __restrict__ k_out,
                                                          const CbState* __restrict__ start) {
  __shared__ unsigned long long dm[64 * kMaxWPL];
  __shared__ unsigned long long rl[kReplayLds];  // wavefront 0's replay
  __shared__ unsigned long long sl[NW][64];      // the walks' row lists
  __shared__ int s_icc[NW];
  __shared__ int s_win, s_win_icc;
  const int g = blockIdx.x;
  if (g >= n_graphs) return;
  const int n = m_arr[g];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (n <= 0) {
    if (tid == 0) k_out[g] = -1;  // maxCliqueHeu on an empty graph
    return;
  }
  const int W = (n + 63) / 64;
  if (W > 64 * kMaxWPL) {
    if (tid == 0) k_out[g] = INT_MIN;  // rejected on the host before launch
    return;
  }
  const unsigned long long* A = adj_all + adj_off[g];
  int* deg = deg_all + lc_off[g];
  int* out = out_all + lc_off[g];
  // after the chip-wide rounds the degrees are already there (k_cb_degrees)
  for (int v = start ? n : tid; v < n; v += 64 * NW) {
    int d = 0;
    for (int w = 0; w < W; ++w) {
      unsigned long long b = A[(size_t)v * W + w];
      if (w == W - 1 && (n & 63)) b &= (1ull << (n & 63)) - 1ull;
      if (w == (v >> 6)) b &= ~(1ull << (v & 63));
      d += __popcll(b);
    }
    deg[v] = d;
  }
  __syncthreads();
  // the scan so far (chip-wide rounds), or its start
  int best = -1, pos = 0, win = -1, win_best = -1;
  if (start) {
    best = start[g].best;
    pos = start[g].pos;
    win = start[g].win;
    win_best = start[g].win_best;
  }
  for (;;) {
    for (int w = tid; w < W; w += 64 * NW) {
      unsigned long long b = 0ull;
      for (int k = 0; k < 64; ++k) {
        const int u = w * 64 + k;
        if (u < n && deg[u] >= best) b |= 1ull << k;
      }
      dm[w] = b;
    }
    __syncthreads();
    bool found = false;
    for (int base = pos; base < n; base += NW) {
      const int c = base + wid;
      int icc = INT_MIN;
      // pruning 1; with best < 1 the first candidate wins (greedy sizes are >= 1)
      if (c < n && !(best > deg[c]) && (best >= 1 || wid == 0)) icc = icc_walk(W, c, A, WalkAux{}, dm, lane, best, sl[wid]);
      if (lane == 0) s_icc[wid] = icc;
      __syncthreads();
      if (tid == 0) {
        int first = -1, fi = 0;
        for (int k = 0; k < NW; ++k)
          if (s_icc[k] > best) {
            first = base + k;
            fi = s_icc[k];
            break;
          }
        s_win = first;
        s_win_icc = fi;
      }
      __syncthreads();
      const int first = s_win;
      if (first >= 0) {
        win = first;
        win_best = best;
        best = s_win_icc;
        pos = first + 1;
        found = true;
        break;
      }
    }
    __syncthreads();
    if (!found) break;
  }
  if (win >= 0) {
    for (int w = tid; w < W; w += 64 * NW) {
      unsigned long long b = 0ull;
      for (int k = 0; k < 64; ++k) {
        const int u = w * 64 + k;
        if (u < n && deg[u] >= win_best) b |= 1ull << k;
      }
      dm[w] = b;
    }
    __syncthreads();
    if (wid == 0) {
      const int icc = replay_walk(W, win, A, dm, out, lane, rl);
      if (lane == 0) k_out[g] = icc == best ? best : INT_MIN;
    }
  } else if (tid == 0) {
    k_out[g] = best;
  }
}

size_t clique_spread_state_bytes(int n_graphs) { return sizeof(CbState) * (size_t)(n_graphs > 0 ? n_graphs : 1); }
size_t clique_spread_icc_bytes(int n_graphs) {
  return sizeof(int) * (size_t)kCbWindow * (size_t)(n_graphs > 0 ? n_graphs : 1);
}

int clique_batch_launch(rpgo_ctx* ctx, int n_graphs, int waves, const long long* d_adj_off,
                        const long long* d_lc_off, const int* d_m, const unsigned long long* adj, int* deg,
                        int* out_idx, int* out_k, const CliqueSpread* spread) {
  hipStream_t st = ctx->stream;
  if (waves != 4 && waves != 8 && waves != 16) {
    set_error("clique_batch_launch: unsupported shape (%d wavefronts)", waves);
    return RPGO_ERR_ARG;
  }
  CbState* cs = nullptr;
  if (spread && spread->n_slots > 0) {
    cs = static_cast<CbState*>(spread->state);
    const long long ns = spread->n_slots;
    const unsigned sg = (unsigned)((ns + 255) / 256);
    k_cb_init<<<(n_graphs + 255) / 256, 256, 0, st>>>(n_graphs, cs);
    k_cb_degrees<<<sg, 256, 0, st>>>(ns, spread->slot_graph, d_adj_off, d_lc_off, d_m, adj, deg, spread->diag);
    k_cb_groups<<<(unsigned)((ns + 3) / 4), 256, 0, st>>>(ns, spread->slot_graph, d_adj_off, d_lc_off, d_m, adj,
                                                          spread->grp);
    const unsigned gi = (unsigned)(8ll * spread->xmax * (kCbWindow / 4));
    const int rounds = (int)((spread->max_slots + kCbWindow - 1) / kCbWindow) + kCbExtraRounds;
    for (int r = 0; r < rounds; ++r) {
      k_cb_mask<<<sg, 256, 0, st>>>(ns, spread->slot_graph, d_lc_off, d_m, deg, cs, spread->dm);
      k_cb_icc<<<gi, 256, 0, st>>>(n_graphs, d_adj_off, d_lc_off, d_m, adj, deg, spread->dm, cs, spread->xorder,
                                   spread->diag, spread->grp, spread->icc);
      k_cb_select<<<(n_graphs + 3) / 4, 256, 0, st>>>(n_graphs, d_m, spread->icc, cs);
    }
    RPGO_HIP_CHECK(hipGetLastError());
  }
#define RPGO_CB(NW) \
  k_clique_batch<NW><<<n_graphs, 64 * NW, 0, st>>>(n_graphs, d_adj_off, d_lc_off, d_m, adj, deg, out_idx, out_k, cs)
  if (waves == 4) RPGO_CB(4);
  else if (waves == 8) RPGO_CB(8);
  else RPGO_CB(16);
#undef RPGO_CB
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

int clique_walk_chunk() { return kWalkChunk; }

int clique_max_vertices() { return 64 * 64 * kMaxWPL; }

// Working memory of one heuristic scan over n vertices (W = ceil(n/64)):
// deg n ints, dmask W words, icc n ints, out n + 1 ints, best 4 ints.
struct ScanBufs {
  int* deg;
  unsigned long long* dmask;
  int* icc;
  int* out;
  int* best;
  // compacted graph of the rounds (all null: the rounds walk the full rows)
  int* cidx = nullptr;                  // n: new index of a vertex with deg >= best
  int* ccol = nullptr;                  // n: old index of new vertex v'
  unsigned long long* cdmask = nullptr;  // W: every new vertex
  unsigned long long* cadj = nullptr;    // n x W words (rows of ceil(n'/64) words)
  int* cn = nullptr;                     // n'
  // (with the compacted graph's) derived rows of the walked graph, picks of
  // the candidates, and the replay's list, exit steps, histogram and sizes
  unsigned long long* aux = nullptr;     // walk_aux_words(n)
  unsigned long long* picks = nullptr;   // n x W words
  int* replay = nullptr;                 // 4 n + 8 ints
};

// Greedy scan over candidates pos0 .. n-1 starting from the bound best0;
// mode EXACT continues with the exact search, mode HEU_REF replays the winner.
// bufs == nullptr: the context's grow-only buffers (allocated on demand).
static int clique_scan(rpgo_ctx* ctx, const uint64_t* d_adj_u64, int n, int mode, int pos0, int best0,
                       int32_t* idx_out, int32_t* k_out, const ScanBufs* bufs = nullptr);

int clique_run(rpgo_ctx* ctx, const uint64_t* d_adj_u64, int n, int mode, int32_t* idx_out,
               int32_t* k_out) {
  return clique_scan(ctx, d_adj_u64, n, mode, 0, -1, idx_out, k_out);
}

// ---------------------------------------------------------------------------
// Allocation-free heuristic scan (rpgo_max_clique_bits_noalloc).  Its working
// memory is this file-scope device array, one copy per GPU, held until the
// process ends.  Host code reaches it only through the address
// hipGetSymbolAddress returns on each device (the array's name is a host-side
// stand-in, not a device address); that lookup runs once per device, from
// rpgo_ctx_create, with the device current.
// ---------------------------------------------------------------------------
constexpr int kNoallocMaxVertices = RPGO_NOALLOC_MAX_VERTICES;
constexpr size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }
constexpr size_t kNaDeg = 0;
constexpr size_t kNaDmask = kNaDeg + align256(sizeof(int) * kNoallocMaxVertices);
constexpr size_t kNaIcc = kNaDmask + align256(sizeof(unsigned long long) * ((kNoallocMaxVertices + 63) / 64));
constexpr size_t kNaOut = kNaIcc + align256(sizeof(int) * kNoallocMaxVertices);
constexpr size_t kNaBest = kNaOut + align256(sizeof(int) * (kNoallocMaxVertices + 1));
constexpr size_t kNaBytes = kNaBest + 256;
static_assert(kNoallocMaxVertices <= 64 * 64 * kMaxWPL, "no-alloc maximum beyond the register bitset");

static __device__ __align__(256) unsigned char scratch[kNaBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

int clique_noalloc_init(int device) {
  if (device < 0 || device >= kMaxDevices) {
    set_error("clique_noalloc_init: device %d beyond the %d supported", device, kMaxDevices);
    return RPGO_ERR_ARG;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[device]) return RPGO_OK;
  void* ptr = nullptr;
  // the caller (rpgo_ctx_create) has made `device` current
  RPGO_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  g_scratch_ptr[device] = ptr;
  return RPGO_OK;
}

size_t clique_noalloc_bytes() { return kNaBytes; }

int clique_run_noalloc(rpgo_ctx* ctx, const uint64_t* d_adj_u64, int n, int32_t* idx_out, int32_t* k_out) {
  if (n > kNoallocMaxVertices) {
    set_error("rpgo_max_clique_bits_noalloc: %d vertices exceed the maximum %d", n, kNoallocMaxVertices);
    return RPGO_ERR_ARG;
  }
  void* base = nullptr;
  {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (ctx->device >= 0 && ctx->device < kMaxDevices) base = g_scratch_ptr[ctx->device];
  }
  if (!base) {
    set_error("rpgo_max_clique_bits_noalloc: scratch of device %d not set up", ctx->device);
    return RPGO_ERR_STATE;
  }
  unsigned char* b = static_cast<unsigned char*>(base);
  const ScanBufs bufs{reinterpret_cast<int*>(b + kNaDeg), reinterpret_cast<unsigned long long*>(b + kNaDmask),
                      reinterpret_cast<int*>(b + kNaIcc), reinterpret_cast<int*>(b + kNaOut),
                      reinterpret_cast<int*>(b + kNaBest)};
  return clique_scan(ctx, d_adj_u64, n, RPGO_CLIQUE_HEU_REF, 0, -1, idx_out, k_out, &bufs);
}

// FMC::maxCliqueHeuIncremental (findCliqueHeu.cpp:119-209) through
// findMaxCliqueHeuIncremental (GraphUtils.cpp:30-44): candidates are only the
// last num_new vertices, the bound starts at the previous clique size, and
// the size is reported only when it strictly grew (0 otherwise).
int clique_incremental(rpgo_ctx* ctx, const uint64_t* d_adj_u64, int n, int num_new, int prev_size,
                       int32_t* idx_out, int32_t* k_out) {
  if (num_new < 0 || num_new > n || prev_size < 0) {
    set_error("rpgo_max_clique_incremental: num_new %d / prev_size %d invalid for %d vertices", num_new,
              prev_size, n);
    return RPGO_ERR_ARG;
  }
  if (n <= 0 || num_new == 0) {
    *k_out = 0;
    return RPGO_OK;
  }
  int32_t k = 0;
  const int rc = clique_scan(ctx, d_adj_u64, n, RPGO_CLIQUE_HEU_REF, n - num_new, prev_size, idx_out, &k);
  if (rc) return rc;
  *k_out = k > prev_size ? k : 0;
  return RPGO_OK;
}

static int clique_scan(rpgo_ctx* ctx, const uint64_t* d_adj_u64, int n, int mode, int pos0, int best0,
                       int32_t* idx_out, int32_t* k_out, const ScanBufs* bufs) {
  CliqueState& s = ctx->clq;
  if (mode != RPGO_CLIQUE_HEU_REF && mode != RPGO_CLIQUE_EXACT) {
    set_error("rpgo_max_clique: unknown mode %d", mode);
    return RPGO_ERR_ARG;
  }
  if (n <= 0) {
    *k_out = mode == RPGO_CLIQUE_EXACT ? 0 : -1;  // FMC: maxClique finds nothing, maxCliqueHeu returns -1
    return RPGO_OK;
  }
  const int W = (n + 63) / 64;
  if (W > 64 * kMaxWPL) {
    set_error("rpgo_max_clique: %d vertices exceed the %d supported", n, 64 * 64 * kMaxWPL);
    return RPGO_ERR_ARG;
  }
  const unsigned long long* adj = reinterpret_cast<const unsigned long long*>(d_adj_u64);
  ScanBufs b;
  if (bufs) {
    b = *bufs;
  } else {
    int rc;
    if ((rc = s.deg.reserve(sizeof(int) * n))) return rc;
    if ((rc = s.dmask.reserve(sizeof(unsigned long long) * W))) return rc;
    if ((rc = s.icc.reserve(sizeof(int) * n))) return rc;
    if ((rc = s.out.reserve(sizeof(int) * (n + 1)))) return rc;
    if ((rc = s.best.reserve(sizeof(int) * 4))) return rc;
    if ((rc = s.cidx.reserve(sizeof(int) * n))) return rc;
    if ((rc = s.ccol.reserve(sizeof(int) * n))) return rc;
    if ((rc = s.cdmask.reserve(sizeof(unsigned long long) * W))) return rc;
    if ((rc = s.cadj.reserve(sizeof(unsigned long long) * (size_t)n * W))) return rc;
    if ((rc = s.cn.reserve(sizeof(int)))) return rc;
    if ((rc = s.caux.reserve(sizeof(unsigned long long) * walk_aux_words(n)))) return rc;
    if ((rc = s.picks.reserve(sizeof(unsigned long long) * (size_t)n * W))) return rc;
    if ((rc = s.replay.reserve(sizeof(int) * (4 * (size_t)n + 8)))) return rc;
    b = ScanBufs{s.deg.as<int>(), s.dmask.as<unsigned long long>(), s.icc.as<int>(), s.out.as<int>(),
                 s.best.as<int>(), s.cidx.as<int>(), s.ccol.as<int>(), s.cdmask.as<unsigned long long>(),
                 s.cadj.as<unsigned long long>(), s.cn.as<int>(), s.caux.as<unsigned long long>(),
                 s.picks.as<unsigned long long>(), s.replay.as<int>()};
  }
  hipStream_t st = ctx->stream;
  k_degrees<<<(n + 255) / 256, 256, 0, st>>>(n, W, adj, b.deg);
  RPGO_HIP_CHECK(hipGetLastError());
  int best = best0, pos = pos0, win = -1, win_best = -1;
  // d_best: the round's packed winner, then the replay's two results
  unsigned long long* d_first = reinterpret_cast<unsigned long long*>(b.best);
  int* d_res = b.best + 2;
  unsigned long long* h_first =
      reinterpret_cast<unsigned long long*>(static_cast<char*>(ctx->host_pinned) + kPinnedClique);
  const WalkAux aux = b.aux ? walk_aux_at(b.aux, n) : WalkAux{};
  unsigned long long *aux_diag = b.aux, *aux_g4 = nullptr, *aux_g8 = nullptr;
  if (b.aux) {
    aux_g4 = b.aux + (aux.g4 - b.aux);
    aux_g8 = b.aux + (aux.g8 - b.aux);
  }
  const unsigned aux_blocks = (unsigned)(((long long)((n + 7) / 8) * W + 255) / 256);
  const bool compact = b.cadj && W > kCompactMinW;
  const bool par = b.replay && n >= kReplayParMin;  // the replay from the winner's picks
  bool full_aux = false;
  int round = best0 < 1 ? 0 : 2;
  while (pos < n) {
    k_dmask<<<(W + 255) / 256, 256, 0, st>>>(n, W, best, b.deg, b.dmask, d_first);
    // best < 1: candidate pos wins (every greedy size is >= 1), so it alone is walked
    // The first candidate alone says little (an outlier's clique prunes nothing,
    // so every later candidate walks to its end) and a better one is near: the
    // round after it takes kScanWindow candidates (50k graph, 50 % outliers: 1.2
    // ms with all 9,999, 0.3 ms; 0.2 ms more when none of them wins)
    const int rem = best < 1 ? 1 : std::min(n - pos, round == 1 ? kScanWindow : n);
    ++round;
    const bool cmp = best >= 1 && compact;
    if (cmp) {
      // the round's subgraph of deg >= best, renumbered in order
      k_compact_index<<<1, 512, 0, st>>>(n, W, b.dmask, b.cidx, b.ccol, b.cdmask, b.cn);
      k_compact_adj<<<(unsigned)(((long long)n * W + 255) / 256), 256, 0, st>>>(n, W, adj, b.ccol, b.cn, b.cadj);
      k_walk_aux<<<aux_blocks, 256, 0, st>>>(n, b.cn, b.cadj, aux_diag, aux_g4, aux_g8);
      full_aux = false;
      k_icc_compact<<<(rem + 3) / 4, 256, 0, st>>>(pos + rem, pos, best, b.deg, b.cidx, b.cn, b.cadj, b.cdmask, aux, b.picks,
                                                   b.icc);
    } else {
      if (b.aux && !full_aux) k_walk_aux<<<aux_blocks, 256, 0, st>>>(n, nullptr, adj, aux_diag, aux_g4, aux_g8);
      full_aux = true;
      k_icc<<<(rem + 3) / 4, 256, 0, st>>>(pos + rem, W, pos, best, adj, b.deg, b.dmask, aux, b.picks, b.icc);
    }
    RPGO_HIP_CHECK(hipGetLastError());
    k_first_better<<<(rem + 255) / 256, 256, 0, st>>>(pos + rem, pos, best, b.icc, d_first);
    RPGO_HIP_CHECK(hipGetLastError());
    RPGO_HIP_CHECK(hipMemcpyAsync(h_first, d_first, sizeof(*h_first), hipMemcpyDeviceToHost, st));
    RPGO_HIP_CHECK(hipStreamSynchronize(st));
    const int first = (int)(*h_first >> 32);
    if (first >= n) {  // no winner in this window
      pos += rem;
      continue;
    }
    win = first;
    win_best = best;
    best = (int)(unsigned int)*h_first;
    pos = win + 1;
    if (par) {
      // the picks before the next round overwrites them
      k_winner_list<<<1, 512, 0, st>>>(win, W, cmp ? b.cidx : nullptr, cmp ? b.ccol : nullptr, cmp ? b.cn : nullptr,
                                       b.picks, b.replay, b.replay + n);
      RPGO_HIP_CHECK(hipGetLastError());
    }
  }
  if (mode == RPGO_CLIQUE_EXACT) {
    // the greedy size is a clique size that exists: the exact search's lower bound
    return clique_exact_run(ctx, adj, n, std::max(best, 1), idx_out, k_out, kExactNodeBudget);
  }
  if (win >= 0) {
    // dmask for the winner's threshold
    k_dmask<<<(W + 255) / 256, 256, 0, st>>>(n, W, win_best, b.deg, b.dmask, nullptr);
    if (par) {
      const int K = best - 1;  // picks
      int *list = b.replay, *count = list + n, *ex = count + 1, *hist = ex + n, *sz = hist + n + 1;
      k_rp_init<<<(n + 256) / 256, 256, 0, st>>>(n, ex, hist);
      if (K > 0) k_rp_exit<<<dim3(W, (K + 255) / 256), 256, 0, st>>>(W, win, K, adj, b.dmask, list, count, ex);
      k_rp_hist<<<(n + 255) / 256, 256, 0, st>>>(n, W, win, K, adj, b.dmask, ex, hist);
      k_rp_sizes<<<1, 1024, 0, st>>>(K, hist, count, sz, d_res);
      k_rp_write<<<std::max(1, (K + 3) / 4), 256, 0, st>>>(n, W, win, K, adj, b.dmask, list, count, ex, sz, b.out);
    } else {
      k_replay<<<1, 64, 0, st>>>(n, W, win, win_best, adj, b.dmask, b.out, d_res);
    }
    RPGO_HIP_CHECK(hipGetLastError());
    int* h_res = reinterpret_cast<int*>(h_first);
    RPGO_HIP_CHECK(hipMemcpyAsync(h_res, d_res, sizeof(int), hipMemcpyDeviceToHost, st));
    if (idx_out && best > 0)
      RPGO_HIP_CHECK(hipMemcpyAsync(idx_out, b.out, sizeof(int) * best, hipMemcpyDeviceToHost, st));
    RPGO_HIP_CHECK(hipStreamSynchronize(st));
    if (*h_res != best) {
      set_error("rpgo_max_clique: replay size %d differs from the scan's %d", *h_res, best);
      return RPGO_ERR_STATE;
    }
  }
  *k_out = best;
  return RPGO_OK;
}

}  // namespace rpgo
