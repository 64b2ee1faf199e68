// KV-cache token eviction and speculative-decoding verification for gfx950.
//
// ---- token eviction ----
// The reference (flash_attn_kernel.cu:4223-4344) bubble-sorts each batch
// row's attention scores ascending on one thread (swapping only when
// s[j] > s[j+1], i.e. a stable sort), evicts the `num_evict` lowest, and
// copies the kept K/V rows, in their original order, to the front of
// zero-filled outputs.  Here that is one launch, one workgroup per (batch,
// KV head, block of output rows): each derives its batch row's keep mask --
// token i is kept iff its stable ascending rank
//     #{j : s_j < s_i} + #{j < i : s_j == s_i}
// is >= num_evict, the position the stable sort gives it -- from a radix
// select of the num_evict-th smallest score, turns it into the destination ->
// source row map (a workgroup prefix count in LDS) and streams its output
// rows with 16-byte loads and stores: kept rows copied, the tail zero-filled.
// This is the HBM-bound part: kept rows are read once, every output row
// written once.
// Scores containing NaN are outside the contract (the reference's bubble sort
// then depends on where the NaN sits; the rank order does not).
#include "capi_internal.h"
#include "common.h"

namespace fa {
namespace evict {

constexpr int kMaxN = 1024;  // the reference's limit (shared arrays of 1024)
constexpr int kThreads = 256;
// Output rows per compaction workgroup: the largest of 128, 256 and 512
// that still gives every CU a workgroup (evict_rows_per_block).  Each
// workgroup runs the selection once for its rows, so fewer, longer
// workgroups spend less of the call selecting (config 8, B = 16, 8 heads,
// N = 1024: 128 rows 28.6 us, 256 rows 26.9, 512 rows 26.0, 1024 rows 32).
constexpr int kMinRowsPerBlock = 128;
constexpr int kMaxRowsPerBlock = 512;
constexpr long long kFillWorkgroups = 256;

// Block-wide exclusive prefix count of one flag per token (thread t owns
// tokens 4t .. 4t+3, in flag[0..3]); returns the count before thread t's first
// token and sets `total`.  `scratch` holds kThreads / 64 ints.
__device__ __forceinline__ int block_prefix(const int (&flag)[4], int* scratch, int& total) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cnt = flag[0] + flag[1] + flag[2] + flag[3];
  int incl = cnt;  // inclusive scan over the wave
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(incl, off, 64);
    if (lane >= off) incl += y;
  }
  __syncthreads();  // scratch may still be read by a previous call
  if (lane == 63) scratch[wave] = incl;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int w = 0; w < kThreads / 64; ++w) {
    before += (w < wave) ? scratch[w] : 0;
    total += scratch[w];
  }
  return before + incl - cnt;
}

// Order-preserving unsigned key of a (non-NaN) score: -0.0 and +0.0 compare
// equal as floats and so map to one key.
__device__ __forceinline__ uint32_t score_key(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x == 0.0f ? 0.0f : x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// One workgroup per (batch, KV head, block of output rows).  Every workgroup
// of batch row b derives row b's keep mask itself (1024 scores at most):
// a radix select (four 8-bit passes over LDS histograms) finds the key T of
// the num_evict-th smallest score and the count c of smaller ones; a token is
// evicted iff its key is below T, or equals T and fewer than num_evict - c
// equal keys precede it -- exactly the tokens whose stable ascending rank
// #{j : s_j < s_i} + #{j < i : s_j == s_i} is below num_evict, i.e. the first
// num_evict of the reference's stable sort.  A prefix count of the keep mask
// then gives the output -> source row map, and the workgroup streams its
// output rows: kept rows copied, the tail zero-filled.
template <bool VEC>
__global__ __launch_bounds__(kThreads) void evict_kernel(const half_t* __restrict__ k, const half_t* __restrict__ v,
                                                        const float* __restrict__ scores, int32_t* __restrict__ keep,
                                                        half_t* __restrict__ ko, half_t* __restrict__ vo, int H,
                                                        int N, int D, int num_evict, int rows_per_block) {
  static_assert(kThreads == 256 && 4 * kThreads == kMaxN, "one histogram bin and four tokens per thread");
  __shared__ int src_of[kMaxN];  // output row -> source row (kept rows only)
  __shared__ int hist[256];
  __shared__ int scratch[kThreads / 64];
  __shared__ int pick[2];
  const int bh = blockIdx.y;
  const int b = bh / H;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;

  // ---- keys of this thread's tokens 4t .. 4t+3 ----
  const float* sb = scores + static_cast<size_t>(b) * N;
  uint32_t key[4];
  bool valid[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int i = 4 * tid + q;
    valid[q] = i < N;
    key[q] = valid[q] ? score_key(sb[i]) : 0u;
  }
  const int E = num_evict;
  int keepf[4];
  if (E <= 0 || E >= N) {
#pragma unroll
    for (int q = 0; q < 4; ++q) keepf[q] = (valid[q] && E <= 0) ? 1 : 0;
  } else {
    // ---- radix select of the E-th smallest key (1-based) ----
    uint32_t prefix = 0u, himask = 0u;
    int need = E, below = 0;
#pragma unroll 1
    for (int shift = 24; shift >= 0; shift -= 8) {
      hist[tid] = 0;  // kThreads == 256 bins
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (valid[q] && (key[q] & himask) == prefix) atomicAdd(&hist[(key[q] >> shift) & 255u], 1);
      __syncthreads();
      if (wave == 0) {
        int c[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          c[j] = hist[4 * lane + j];
          sum += c[j];
        }
        int incl = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int y = __shfl_up(incl, off, 64);
          if (lane >= off) incl += y;
        }
        int run = incl - sum;  // keys in the bins before this lane's first bin
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // the bin where the running count first reaches `need` (one lane, one j)
          if (run < need && run + c[j] >= need) {
            pick[0] = 4 * lane + j;
            pick[1] = run;
          }
          run += c[j];
        }
      }
      __syncthreads();
      const int digit = pick[0];
      need -= pick[1];
      below += pick[1];
      prefix |= static_cast<uint32_t>(digit) << shift;
      himask |= 0xFFu << shift;
      __syncthreads();  // every thread has read pick before the next pass
    }
    // prefix = T; below = #{key < T}; the first E - below keys equal to T are evicted
    int eq[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) eq[q] = (valid[q] && key[q] == prefix) ? 1 : 0;
    int eq_total;
    int eq_before = block_prefix(eq, scratch, eq_total);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      keepf[q] = valid[q] && (key[q] > prefix || (eq[q] && eq_before >= E - below)) ? 1 : 0;
      eq_before += eq[q];
    }
  }
  // the mask output: written once per batch row
  if (bh % H == 0 && blockIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (valid[q]) keep[static_cast<size_t>(b) * N + 4 * tid + q] = keepf[q];
  }

  // ---- prefix count of kept tokens -> output row map ----
  int kept;
  int dst = block_prefix(keepf, scratch, kept);
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (keepf[q]) src_of[dst++] = 4 * tid + q;
  __syncthreads();

  // ---- output rows [r0, r0 + rows_per_block) of this (batch, head) ----
  const size_t base = static_cast<size_t>(bh) * N * D;
  const int r0 = blockIdx.x * rows_per_block;
  const int rows = min(rows_per_block, N - r0);
  if constexpr (VEC) {
    const int cpr = D / 8;  // 16-byte chunks per row
    const u32x4 zero = {0u, 0u, 0u, 0u};
    constexpr int U = 4;  // chunks in flight per thread: all loads, then all stores
    const int total = rows * cpr;
    for (int c0 = tid; c0 < total; c0 += U * kThreads) {
      u32x4 kx[U], vx[U];
      size_t dsto[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * kThreads;
        const int w = r0 + c / cpr;
        const int col = (c % cpr) * 8;
        dsto[u] = base + static_cast<size_t>(w) * D + col;
        kx[u] = zero;
        vx[u] = zero;
        if (c < total && w < kept) {
          const size_t srco = base + static_cast<size_t>(src_of[w]) * D + col;
          kx[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(k + srco));
          vx[u] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(v + srco));
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (c0 + u * kThreads < total) {
          *reinterpret_cast<u32x4*>(ko + dsto[u]) = kx[u];
          *reinterpret_cast<u32x4*>(vo + dsto[u]) = vx[u];
        }
      }
    }
  } else {
    for (int e = tid; e < rows * D; e += kThreads) {
      const int w = r0 + e / D;
      const int col = e % D;
      const size_t dsto = base + static_cast<size_t>(w) * D + col;
      if (w < kept) {
        const size_t srco = base + static_cast<size_t>(src_of[w]) * D + col;
        ko[dsto] = k[srco];
        vo[dsto] = v[srco];
      } else {
        ko[dsto] = static_cast<half_t>(0.0f);
        vo[dsto] = static_cast<half_t>(0.0f);
      }
    }
  }
}

}  // namespace evict

// ---- speculative verification ----
// The reference (flash_attn_kernel.cu:3853-4018) accepts draft token t at
// step i when r_i < min(1, p_t / (q_t + 1e-10)); at the first rejection it
// samples from max(target - draft, 0) / Z and draws a bonus token from the
// next target row, each by a running fp32 sum over the vocabulary compared
// against r (with its "tok == 0" update rule: a hit at index 0 is replaced by
// the next hit).  The sampled indices depend on the exact fp32 value of every
// partial sum, i.e. on the rounding of each of the V serial additions.
//
// Those serial sums are computed in parallel, bit for bit.  While the running
// sum s stays inside one binade it is n * g with g the ulp there and n an
// integer, and adding a term t >= 0 moves n by an integer that depends on t
// and, where t / g is a tie, on the parity of n alone.  A run of terms is
// therefore a map from the parity of n to an increment, a pair (d0, d1), found
// by adding the terms in fp32 to any sum of that binade with n even and to one
// with n odd; such pairs compose associatively, so lanes' pairs are scanned.
// Which binade a lane's terms meet is told by an estimate of the sums (a float
// prefix sum); a lane whose terms may cross into the next one is doubtful, and
// its terms are added one by one.  One wave puts the pieces together with the
// exact sum, and checks each piece against it: a wrong guess, a negative or
// non-finite term or a hit sends that 512-term chunk to a walk, which locates
// the lane concerned by the same scans and adds its terms in turn.  Only the
// row's first 128 terms, where the sum doubles every few, are all added in turn.
//
// Bound by the latency of these steps, not by bytes: of about 15 us a row of
// 32000 and scan, 4 us are the values' arrival, 2-3 us the first chunk, 3 us the
// records and 7 us the assembly (0.8 us for each of its half-dozen crossings).
// Two workgroups per row run concurrently: Z, then the residual sample; the
// bonus token.  One lane adding all the terms in turn from LDS, fed by a second
// wave, took 180 us for 16 rows of 32000 words and K = 4; scans that restarted
// at each binade 63 us; this takes 31-35 us (128000 words: 77-80 us).  The scans
// are compiled into the kernel: as calls, which reach LDS by generic addresses
// and keep registers in scratch, all-accepted batches (the bonus scan alone) took
// 19.2 us against 15.8.
namespace spec {

constexpr int kMaxK = 8;      // SPEC_MAX_K (flash_attn_kernel.cu:3851)
constexpr int kWaves = 16;
constexpr int kSpecThreads = kWaves * 64;
constexpr int kTerms = 8;               // consecutive terms per lane
constexpr int kChunk = 64 * kTerms;     // consecutive terms per wave
constexpr int kTiles = 4;               // chunks per wave and group
constexpr int kChunks = kTiles * kWaves;  // chunks per group: chunk c is wave c % 16's, one lane each when assembled
constexpr int kGroup = kChunks * kChunk;
static_assert(kChunks == 64, "one lane per chunk");
constexpr uint32_t kTop = 1u << 24;  // n at the end of a binade
constexpr uint32_t kCap = 1u << 25;  // increments saturate here (64 of them still fit 32 bits)

enum ChainMode { kZ = 0, kResidual = 1, kPrefix = 2, kBonus = 3 };

typedef float Terms __attribute__((ext_vector_type(kTerms)));
typedef Terms Terms4 __attribute__((aligned(4)));  // rows start at any 4-byte boundary

// Increment of n over a run of terms, for n even (d0) and odd (d1) before it.
struct Inc {
  uint32_t d0, d1;
};
__device__ __forceinline__ Inc then(Inc a, Inc b) {
  Inc c;
  c.d0 = min(a.d0 + ((a.d0 & 1u) ? b.d1 : b.d0), kCap);
  c.d1 = min(a.d1 + ((a.d1 & 1u) ? b.d0 : b.d1), kCap);
  return c;
}
__device__ __forceinline__ uint32_t advance(uint32_t n, Inc a) {
  const uint32_t d0 = a.d0, d1 = a.d1;
  return n + ((n & 1u) ? d1 : d0);
}

template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ void scan_step(Inc& x) {
  const Inc below = {dpp_from<CTRL, ROWS>(x.d0), dpp_from<CTRL, ROWS>(x.d1)};
  x = then(below, x);
}
// Inclusive scan over the wave.
__device__ __forceinline__ Inc scan_inc(Inc x) {
  if (__builtin_amdgcn_ballot_w64(x.d0 != x.d1) == 0) {
    // no tie in the wave: plain increments (64 * 2^25 at most)
    uint32_t d = wave_scan_add(x.d0);
    d = min(d, kCap);
    return Inc{d, d};
  }
  scan_step<kRowShr1>(x);
  scan_step<kRowShr2>(x);
  scan_step<kRowShr4>(x);
  scan_step<kRowShr8>(x);
  scan_step<kRowBcast15, 0xA>(x);
  scan_step<kRowBcast31, 0xC>(x);
  return x;
}

// The ulp grid of a sum s >= 0: s = n * 2^exp.
struct Grid {
  uint32_t n;
  int exp;
};
__device__ __forceinline__ Grid grid_of(float s) {
  const uint32_t u = __builtin_bit_cast(uint32_t, s);
  const uint32_t e = u >> 23;
  return Grid{(u & 0x7fffffu) | (e ? 0x800000u : 0u), static_cast<int>(e ? e : 1u) - 150};
}
__device__ __forceinline__ float sum_of(uint32_t n, int exp) {
  return __builtin_amdgcn_ldexpf(static_cast<float>(n), exp);
}
// sums the scans apply to: not negative, not infinite, not NaN
__device__ __forceinline__ bool on_grid(float s) { return s >= 0.0f && s < INFINITY; }

__device__ __forceinline__ float lane_value(float x, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), lane));
}

// Increments of n over a lane's terms, all >= 0, for a sum in the binade of
// `base` >= 0: the terms added to base with its last bit cleared, and set.  A
// sum that leaves the binade gives kCap.
__device__ __forceinline__ Inc lane_inc(const Terms& t, float base) {
  const uint32_t u = __builtin_bit_cast(uint32_t, base);
  float even = __builtin_bit_cast(float, u & ~1u), odd = __builtin_bit_cast(float, u | 1u);
#pragma unroll
  for (int e = 0; e < kTerms; ++e) {
    even += t[e];
    odd += t[e];
  }
  const uint32_t a = __builtin_bit_cast(uint32_t, even), b = __builtin_bit_cast(uint32_t, odd);
  // the last sum of base's binade is the first of the next; the lowest
  // exponent has two binades of one grid
  const uint32_t top = u < 0x00800000u ? 0x01000000u : (u & 0x7f800000u) + 0x00800000u;
  return Inc{a <= top ? a - (u & ~1u) : kCap, b <= top ? b - (u | 1u) : kCap};
}

// Where a chain stands: the running sum and what it has found.
struct Walk {
  float s;
  int tok;        // token found, valid with done
  int done;
};

// In kZ and kResidual a term that does not contribute (target <= draft, or
// past V) is -0.0, which leaves the sum unchanged and is never a hit; one that
// does has its sign bit clear.  Past V every mode has -0.0.
template <int MODE>
__device__ __forceinline__ bool contributes(float t, uint32_t v, uint32_t V) {
  if constexpr (MODE == kResidual) return !__builtin_signbit(t);
  return v < V;
}
template <int MODE>
__device__ __forceinline__ bool is_hit(float s, float r) {
  if constexpr (MODE == kZ) return false;
  if constexpr (MODE == kBonus) return s >= r;
  return r < s;
}

// One wave takes a chunk of terms (lane l: indices v0 .. v0 + kTerms), `w` to
// its end or to the token.  first: the row's first chunk, where the sum doubles
// every few terms: the terms of its first kSerialLanes lanes are added in turn
// from LDS (`first`).
constexpr int kSerialLanes = 16;
template <int MODE>
__device__ __forceinline__ void walk_chunk(const Terms& t, uint32_t v0, uint32_t V, float r, float* first, Walk& w) {
  const int lane = threadIdx.x & 63;
  bool bad = false, contrib = false;
#pragma unroll
  for (int e = 0; e < kTerms; ++e) {
    bad |= !(t[e] >= 0.0f && t[e] < INFINITY);
    contrib |= contributes<MODE>(t[e], v0 + e, V);
  }
  const uint64_t contribs = __builtin_amdgcn_ballot_w64(contrib);
  const bool any_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
  int from = 0;
  if (first != nullptr && !any_bad) {
    if (lane < kSerialLanes) *reinterpret_cast<Terms*>(first + lane * kTerms) = t;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    float x = w.s;
#pragma unroll
    for (int e = 0; e < kSerialLanes * kTerms; ++e) x += first[e];
    if (!((contribs & ((1ull << kSerialLanes) - 1)) && is_hit<MODE>(x, r))) {  // (or the hit is found below)
      w.s = lane_value(x, 0);
      from = kSerialLanes;
    }
  }
  while (from < 64) {
    int at = from;
    float s0 = w.s;
    if (on_grid(w.s)) {
      const Grid g = grid_of(w.s);
      Inc x = {0u, 0u};
      if (lane >= from && !bad) x = lane_inc(t, w.s);
      x = scan_inc(x);
      const uint32_t n = advance(g.n, x);
      const float s = sum_of(n, g.exp);
      const bool stop = lane >= from && (n > kTop || bad || (contrib && is_hit<MODE>(s, r)));
      const uint64_t stops = __builtin_amdgcn_ballot_w64(stop);
      if (stops == 0) {
        w.s = lane_value(s, 63);
        return;
      }
      at = __builtin_ctzll(stops);
      if (at > from) s0 = lane_value(s, at - 1);
    } else if (w.s != w.s) {
      return;  // NaN from here on: no comparison holds
    }
    // lane `at` adds its terms one by one (every lane does, its own are kept)
    float s = s0;
    int tok = -1;
#pragma unroll
    for (int e = 0; e < kTerms; ++e) {
      s += t[e];
      const uint32_t v = v0 + e;
      if (tok < 0 && v > 0 && contributes<MODE>(t[e], v, V) && is_hit<MODE>(s, r)) tok = static_cast<int>(v);
    }
    w.s = lane_value(s, at);
    tok = __builtin_amdgcn_readlane(tok, at);
    if (tok >= 0) {
      w.tok = tok;
      w.done = 1;
      return;
    }
    from = at + 1;
  }
}

// What a wave says about a chunk.  The lanes up to the first doubtful one move
// the sum on grid 2^exp by `head`; with at most kDoubtful doubtful lanes, `mid`
// holds their terms (-0.0 beyond) and `tail` is the increment of the lanes
// after them on grid 2^tail_exp.
constexpr int kDoubtful = 2;
enum Flags : int {
  kParts = 1,    // has doubtful lanes
  kWalkIt = 2,   // more of them, or a term that is negative or not finite
  kHasHead = 4,  // lanes before the doubtful ones
  kHasTail = 8,  // and after
  kContrib = 16  // a contributing term
};
struct Shared {
  float total[kChunks];  // estimated sum of each chunk's terms
  Inc head[kChunks], tail[kChunks];
  int exp[kChunks], tail_exp[kChunks], flags[kChunks];
  float mid[kChunks][kDoubtful * kTerms];
  __attribute__((aligned(16))) float first[kSerialLanes * kTerms];
  Walk w;
};

// row[v0 .. v0 + kTerms), 0 past V
__device__ __forceinline__ Terms load_terms(const float* row, uint32_t v0, uint32_t V) {
  Terms x;
  if (v0 + kTerms <= V) return *reinterpret_cast<const Terms4*>(row + v0);
#pragma unroll
  for (int e = 0; e < kTerms; ++e) x[e] = v0 + e < V ? row[v0 + e] : 0.0f;
  return x;
}

// The chain's terms from row values a (and b).
template <int MODE>
__device__ __forceinline__ Terms make_terms(const Terms& a, const Terms& b, float Z, uint32_t v0, uint32_t V) {
  Terms t;
#pragma unroll
  for (int e = 0; e < kTerms; ++e) {
    if constexpr (MODE == kZ || MODE == kResidual) {
      const float d = a[e] - b[e];
      t[e] = d > 0.0f && v0 + e < V ? (MODE == kZ ? d : d / Z) : -0.0f;
    } else {
      t[e] = v0 + e < V ? a[e] : -0.0f;
    }
  }
  return t;
}

// Serial scan of row a (minus row b for kZ / kResidual) over [0, V).
//  kZ:        *sum = the sum of the positive (a - b) in index order.
//  kResidual: cs += (a - b) / Z where a - b > 0; hit at such v when r < cs.
//  kPrefix:   cs += a; hit when r < cs.
//  kBonus:    cs += a; hit when cs >= r.
// Returns the reference's token: the first hit past index 0 (there, a hit at
// index 0 is replaced by the next one), 0 without one.  Every wave takes the
// same path through the barriers: what decides it is read from LDS after one.
// Indices are unsigned: the last group's ends pass 2^31 when V is within a
// group of it.
template <int MODE>
__device__ __forceinline__ int chain(const float* __restrict__ a, const float* __restrict__ b, uint32_t V, float Z,
                                     float r, float* sum, Shared& sh) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr bool kDiff = MODE == kZ || MODE == kResidual;
  auto terms_at = [&](uint32_t v0) {
    const Terms xa = load_terms(a, v0, V);
    const Terms xb = kDiff ? load_terms(b, v0, V) : Terms(0.0f);
    return make_terms<MODE>(xa, xb, Z, v0, V);
  };
  Walk w = {0.0f, 0, 0};
  for (uint32_t c0 = 0; c0 < V && !w.done && w.s == w.s; c0 += kGroup) {
    const uint32_t vw = c0 + (wave * 64 + lane) * kTerms;  // this lane's terms of its wave's first chunk
    Terms xa[kTiles], xb[kTiles], t[kTiles];
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      xa[j] = load_terms(a, vw + j * kWaves * kChunk, V);
      xb[j] = kDiff ? load_terms(b, vw + j * kWaves * kChunk, V) : Terms(0.0f);
    }
    float upto[kTiles];  // estimated sum of the chunk up to this lane's end
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      t[j] = make_terms<MODE>(xa[j], xb[j], Z, vw + j * kWaves * kChunk, V);
      float mine = 0.0f;
#pragma unroll
      for (int e = 0; e < kTerms; ++e) mine += t[j][e];
      upto[j] = wave_scan_add(mine);
      if (lane == 63) sh.total[j * kWaves + wave] = upto[j];
    }
    __syncthreads();
    const float chunk_end = w.s + wave_scan_add(sh.total[lane]);  // lane c: estimate at the end of chunk c
    if (c0 == 0 && wave == 0) {
      __builtin_amdgcn_s_setprio(3);  // everything waits for this walk
      walk_chunk<MODE>(t[0], vw, V, r, sh.first, w);
    }
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const int c = j * kWaves + wave;
      if (c0 == 0 && c == 0) continue;  // walked
      if (c0 + c * kChunk >= V) continue;
      const float start = (c > 0 ? lane_value(chunk_end, max(c - 1, 0)) : w.s);
      float mine = 0.0f, least = 0.0f;
      bool contrib = false;
#pragma unroll
      for (int e = 0; e < kTerms; ++e) {
        mine += t[j][e];
        least = fminf(least, t[j][e]);
        contrib |= contributes<MODE>(t[j][e], vw + j * kWaves * kChunk + e, V);
      }
      const bool bad = least < 0.0f || !(mine < INFINITY);  // (a NaN or infinite term shows in the sum)
      // The estimate of where the sum stands before and after the lane's terms
      // strays from the serial sum by far less than 2^-10; a wrong guess is
      // noticed when the pieces are put together and costs a walk.
      constexpr float kSlack = 1.0f / 1024.0f;
      const float lo = start + (upto[j] - mine);
      const int e0 = grid_of(lo * (1.0f - kSlack)).exp;
      const int e1 = grid_of((start + upto[j]) * (1.0f + kSlack)).exp;
      const uint64_t doubts = __builtin_amdgcn_ballot_w64(e0 != e1 || bad || !(lo >= 0.0f));
      const int x0 = doubts ? __builtin_ctzll(doubts) : 64;  // doubtful lanes [x0, x1)
      const int x1 = doubts ? 64 - __builtin_clzll(doubts) : 64;
      const int head_exp = __builtin_amdgcn_readlane(e0, 0);
      const int tail_exp = __builtin_amdgcn_readlane(e0, 63);
      const bool in_doubt = lane >= x0 && lane < x1;
      const Inc mine_inc = in_doubt ? Inc{0u, 0u} : lane_inc(t[j], lo);
      Inc head = {lane < x0 ? mine_inc.d0 : 0u, lane < x0 ? mine_inc.d1 : 0u};
      head = scan_inc(head);
      int flags = (x0 > 0 ? kHasHead : 0) | (__builtin_amdgcn_ballot_w64(contrib) ? kContrib : 0);
      // every lane of a run is on the run's grid
      bool off = __builtin_amdgcn_ballot_w64((lane < x0 && e0 != head_exp) || (lane >= x1 && e0 != tail_exp)) != 0;
      if (doubts) {
        flags |= kParts;
        off |= x1 - x0 > kDoubtful || __builtin_amdgcn_ballot_w64(bad) != 0;
        if (x1 < 64) {
          flags |= kHasTail;
          Inc tail = {lane >= x1 ? mine_inc.d0 : 0u, lane >= x1 ? mine_inc.d1 : 0u};
          tail = scan_inc(tail);
          if (lane == 63) sh.tail[c] = tail;
        }
        if (lane < kDoubtful * kTerms) sh.mid[c][lane] = -0.0f;
        if (in_doubt && lane < x0 + kDoubtful) {
#pragma unroll
          for (int e = 0; e < kTerms; ++e) sh.mid[c][(lane - x0) * kTerms + e] = t[j][e];
        }
      }
      if (off) flags |= kWalkIt;
      if (lane == 63) sh.head[c] = head;  // (lanes from x0 on add nothing)
      if (lane == 0) {
        sh.exp[c] = head_exp;
        sh.tail_exp[c] = tail_exp;
        sh.flags[c] = flags;
      }
    }
    __syncthreads();
    // ---- wave 0 puts the pieces together: lane c has chunk c's ----
    if (wave == 0) {
      const int chunks = static_cast<int>(min(static_cast<uint32_t>(kChunks), (V - c0 + kChunk - 1) / kChunk));
      int from = c0 == 0 ? 1 : 0;  // first chunk still to be added
      const Inc my_head = sh.head[lane];
      const int my_exp = sh.exp[lane], my_flags = sh.flags[lane];
      while (from < chunks && !w.done && w.s == w.s) {
        int at = from;
        bool walk = !on_grid(w.s);
        if (!walk) {
          const Grid g = grid_of(w.s);
          const bool mine = lane >= from && lane < chunks;
          const Inc y = scan_inc(Inc{mine ? my_head.d0 : 0u, mine ? my_head.d1 : 0u});
          const uint32_t n = advance(g.n, y);
          const float s = sum_of(n, g.exp);
          const bool stop = mine && ((my_flags & (kParts | kWalkIt)) || my_exp != g.exp || n > kTop ||
                                     ((my_flags & kContrib) && is_hit<MODE>(s, r)));
          const uint64_t stops = __builtin_amdgcn_ballot_w64(stop);
          at = stops ? __builtin_ctzll(stops) : chunks;
          if (at > from) w.s = lane_value(s, at - 1);
          if (at == chunks) break;
          const int fl = __builtin_amdgcn_readlane(my_flags, at);
          walk = (fl & (kParts | kWalkIt)) != kParts;
          if (!walk) {
            // head, doubtful terms one by one, tail
            const Inc head_at = sh.head[at], tail_at = sh.tail[at];
            float x = w.s;
            if (fl & kHasHead) {
              const Grid h = grid_of(x);
              const uint32_t m = advance(h.n, head_at);
              walk = sh.exp[at] != h.exp || m > kTop;
              x = sum_of(m, h.exp);
            }
#pragma unroll
            for (int e = 0; e < kDoubtful * kTerms; ++e) x += sh.mid[at][e];
            if (fl & kHasTail) {
              const Grid q = grid_of(x);
              const uint32_t m = advance(q.n, tail_at);
              walk |= !on_grid(x) || sh.tail_exp[at] != q.exp || m > kTop;
              x = sum_of(m, q.exp);
            }
            // sums only grow inside such a chunk: a hit anywhere shows at its end
            walk |= !on_grid(x) || ((fl & kContrib) && is_hit<MODE>(x, r));
            if (!walk) w.s = x;
          }
        }
        if (walk) {
          const uint32_t v0 = c0 + at * kChunk + lane * kTerms;
          walk_chunk<MODE>(terms_at(v0), v0, V, r, nullptr, w);
        }
        from = at + 1;
      }
      if (lane == 0) sh.w = w;
    }
    __syncthreads();
    w = sh.w;
    __builtin_amdgcn_s_setprio(0);
    // (sh.w and the records are written again only past the next group's first
    // barrier, or, by the next chain, past its own)
  }
  if (sum) *sum = w.s;
  return w.done ? w.tok : 0;
}

// Grid (B, 2): workgroup (b, 0) settles the acceptance steps of row b and,
// after a rejection, samples the residual (Z, then the residual scan);
// workgroup (b, 1) draws the bonus token.  Both run the acceptance steps
// themselves, lane i step i.
__global__ __launch_bounds__(kSpecThreads) void verify_kernel(
    const float* __restrict__ target, const float* __restrict__ draft, const int64_t* __restrict__ draft_tokens,
    const float* __restrict__ rand, int32_t* __restrict__ accepted, int64_t* __restrict__ out, int K, int V) {
  __shared__ Shared sh;
  const int b = blockIdx.x;
  const int role = blockIdx.y;
  const float* tb = target + static_cast<size_t>(b) * (K + 1) * V;
  const float* db = draft + static_cast<size_t>(b) * K * V;
  const int64_t* tok_b = draft_tokens + static_cast<size_t>(b) * K;
  const float* rb = rand + static_cast<size_t>(b) * K;
  int64_t* ob = out + static_cast<size_t>(b) * (K + 1);

  const int step = threadIdx.x & 63;
  int64_t tok = 0;
  bool rejects = false;
  if (step < K) {
    tok = tok_b[step];
    const float r = rb[step];
    const bool in_range = tok >= 0 && tok < V;
    const float p = in_range ? tb[static_cast<size_t>(step) * V + tok] : 0.0f;
    const float q = in_range ? db[static_cast<size_t>(step) * V + tok] : 0.0f;
    rejects = !(r < fminf(1.0f, p / (q + 1e-10f)));
  }
  const uint64_t rejections = __builtin_amdgcn_ballot_w64(rejects);
  const int rej = rejections ? __builtin_ctzll(rejections) : -1;
  const int acc = rej >= 0 ? rej : K;
  if (role == 0) {
    // every position is written: accepted tokens, then (after a rejection at
    // rej) the sample at rej, the bonus at rej + 1 (workgroup (b, 1)) and -1 beyond
    if (threadIdx.x < acc) ob[step] = tok;
    if (rej >= 0 && static_cast<int>(threadIdx.x) >= rej + 2 && static_cast<int>(threadIdx.x) <= K) ob[threadIdx.x] = -1;
    if (threadIdx.x == 0) accepted[b] = acc;
    if (rej >= 0) {
      const float* ti = tb + static_cast<size_t>(rej) * V;
      const float* di = db + static_cast<size_t>(rej) * V;
      float Z;
      chain<kZ>(ti, di, V, 0.0f, 0.0f, &Z, sh);
      const int s = Z > 0.0f ? chain<kResidual>(ti, di, V, Z, rb[rej], nullptr, sh)
                             : chain<kPrefix>(ti, nullptr, V, 0.0f, rb[rej], nullptr, sh);
      if (threadIdx.x == 0) ob[rej] = s;
    }
  } else {
    const int row = rej >= 0 ? rej + 1 : K;
    const float r = rb[rej >= 0 ? min(rej, K - 1) : K - 1];
    const int bonus = chain<kBonus>(tb + static_cast<size_t>(row) * V, nullptr, V, 0.0f, r, nullptr, sh);
    if (threadIdx.x == 0) ob[row] = bonus;
  }
}

}  // namespace spec
}  // namespace fa

using namespace fa;
using namespace fa::evict;

extern "C" int fa_token_eviction(const void* k, const void* v, const float* attn_scores, void* k_out, void* v_out,
                                 int32_t* keep_mask, int B, int H_KV, int N, int D, int num_evict, void* stream) {
  const char* fn = "fa_token_eviction";
  if (B < 0 || H_KV <= 0 || N < 0 || D <= 0)
    return set_error(FA_ERR_INVALID_ARG, "%s: bad sizes (B=%d H_KV=%d N=%d D=%d)", fn, B, H_KV, N, D);
  if (N > kMaxN) return set_error(FA_ERR_UNSUPPORTED, "%s: N=%d exceeds %d", fn, N, kMaxN);
  if (static_cast<long long>(B) * H_KV > 65535) return set_error(FA_ERR_UNSUPPORTED, "%s: B*H_KV exceeds 65535", fn);
  if (B == 0 || N == 0) return FA_OK;
  if (!k || !v || !attn_scores || !k_out || !v_out || !keep_mask)
    return set_error(FA_ERR_INVALID_ARG, "%s: null pointer", fn);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool vec = D % 8 == 0 && aligned16(k) && aligned16(v) && aligned16(k_out) && aligned16(v_out);
  int rpb = kMaxRowsPerBlock;
  while (rpb > kMinRowsPerBlock && static_cast<long long>(B) * H_KV * ceil_div(N, rpb) < kFillWorkgroups) rpb /= 2;
  const dim3 grid(ceil_div(N, rpb), B * H_KV);
  const half_t* kh = static_cast<const half_t*>(k);
  const half_t* vh = static_cast<const half_t*>(v);
  if (vec)
    hipLaunchKernelGGL(evict_kernel<true>, grid, dim3(kThreads), 0, st, kh, vh, attn_scores, keep_mask,
                       static_cast<half_t*>(k_out), static_cast<half_t*>(v_out), H_KV, N, D, num_evict, rpb);
  else
    hipLaunchKernelGGL(evict_kernel<false>, grid, dim3(kThreads), 0, st, kh, vh, attn_scores, keep_mask,
                       static_cast<half_t*>(k_out), static_cast<half_t*>(v_out), H_KV, N, D, num_evict, rpb);
  return check_launch(fn);
}

extern "C" int fa_speculative_verify(const float* target_probs, const float* draft_probs, const int64_t* draft_tokens,
                                     const float* random_vals, int32_t* accepted_count, int64_t* output_tokens, int B,
                                     int K, int vocab_size, void* stream) {
  const char* fn = "fa_speculative_verify";
  if (B < 0 || vocab_size <= 0)
    return set_error(FA_ERR_INVALID_ARG, "%s: bad sizes (B=%d vocab=%d)", fn, B, vocab_size);
  if (K < 1 || K > spec::kMaxK) return set_error(FA_ERR_INVALID_ARG, "%s: K=%d outside [1, %d]", fn, K, spec::kMaxK);
  if (B == 0) return FA_OK;
  if (!target_probs || !draft_probs || !draft_tokens || !random_vals || !accepted_count || !output_tokens)
    return set_error(FA_ERR_INVALID_ARG, "%s: null pointer", fn);
  hipLaunchKernelGGL(spec::verify_kernel, dim3(B, 2), dim3(spec::kSpecThreads), 0, static_cast<hipStream_t>(stream), target_probs,
                     draft_probs, draft_tokens, random_vals, accepted_count, output_tokens, K, vocab_size);
  return check_launch(fn);
}
