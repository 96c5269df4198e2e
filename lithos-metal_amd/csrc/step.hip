// The serial ops of a GPU-resident decode loop (ops/embed.py `embed`, ops/sample.py `argmax`, the advance of
// runtime/src/metal_core.mm:256-386 with the StepState fields of core/step_state.py:28-73): small kernels that run
// once per step so a captured step replays unchanged; everything that varies lives in mi_step_state.
#include "mi_common.h"

#include <time.h>

#include <algorithm>
#include <chrono>
#include <deque>
#include <mutex>
#include <vector>

static_assert(sizeof(mi_step_state) == 272, "mi_step_state: the 272-byte layout");

namespace {

constexpr int EMBED_THREADS = 256;
constexpr int ARGMAX_THREADS = 256;

// one block per (token, 2048-column span): 8 BF16 per thread, 16-byte loads
__global__ __launch_bounds__(EMBED_THREADS) void embed_rows(mi_embed_desc d) {
  const int i = blockIdx.y;
  const int col = (blockIdx.x * EMBED_THREADS + threadIdx.x) * 8;
  if (col >= d.hidden) return;
  const int tok = d.tokens[i];
  const long long row = (tok >= 0 && tok < d.vocab) ? tok : 0;
  // T16 BF16 slab: tile = 16 rows × (hidden / 32) chunks of 512 elements; inside a chunk, column group q (8 columns)
  // of row r sits at q·128 + r·8
  const long long at = d.t16 ? ((row >> 4) * (d.hidden >> 5) + (col >> 5)) * 512 + ((col >> 3) & 3) * 128 + (row & 15) * 8
                             : row * d.hidden + col;
  const uint4 v = *reinterpret_cast<const uint4*>(d.table + at);
  *reinterpret_cast<uint4*>(d.out + (long long)i * d.ldo + col) = v;
}

__device__ __forceinline__ bool better(float v, int i, float bv, int bi) {
  return v > bv || (v == bv && i < bi);          // NaN compares false: never replaces a number
}

// The order "larger value, then lower index" over the numbers is total, so combining partial results in any order
// gives the same answer: the spans of a row run in parallel and the last one to finish folds them.
// Logits per workgroup: 16 a thread. (8 a thread, twice the workgroups, publishing twice the partials: rows of 248320 x 1 /
// 4 / 16 5.7 / 9.7 / 26.8 us, 16 a thread 5.4 / 7.4 / 16.1. Only a draw for one or two rows is faster with 8, its noise is
// work for every logit: 248320 28.0 → 27.2 us, see sample_layout)
constexpr int ARGMAX_SPAN = ARGMAX_THREADS * 16;
constexpr int ARGMAX_MAX_SPANS = 256;
constexpr size_t ARGMAX_COUNTERS = 256;            // bytes: 16 per-row arrival counters, padded

__device__ __forceinline__ void st_dev8(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_dev8(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void block_best(float& bv, int& bi, float* sv, int* si) {
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o);
    const int oi = __shfl_xor(bi, o);
    if (better(ov, oi, bv, bi)) { bv = ov; bi = oi; }
  }
  const int w = threadIdx.x / 64;
  if ((threadIdx.x & 63) == 0) { sv[w] = bv; si[w] = bi; }
  __syncthreads();
  bv = sv[0];
  bi = si[0];
  for (int k = 1; k < ARGMAX_THREADS / 64; ++k)
    if (better(sv[k], si[k], bv, bi)) { bv = sv[k]; bi = si[k]; }
}

// ---- stochastic sampling (kernels/common/sample.metal, nn/sampling_ref.py) -------------------------------------
// The draw is argmax over the kept logits (v >= tau) of v / temperature + g_i, g_i = −log(−log(u_i)), u_i from a
// splitmix64 hash of (seed, step, token row, index): the reference's counter-based noise, so a draw is reproducible
// bit for bit and checkable against the host restatement.
struct SampleCtx {
  const float* tau;                // per row: the logit threshold (sample_threshold); null: keep every logit
  float inv_t;
  uint32_t seed_lo, seed_hi, step;
  const mi_step_state* st;         // when set: seed = (rng_hi, rng_lo) and step come from the step state
};

__device__ __forceinline__ float uniform01(uint32_t seed_lo, uint32_t seed_hi, uint32_t step, uint32_t t, uint32_t i) {
  uint64_t x = ((uint64_t)seed_hi << 32) | seed_lo;
  x += (uint64_t)step * 0x9E3779B97F4A7C15ull + (uint64_t)t * 0xC2B2AE3D27D4EB4Full + (uint64_t)i * 0x165667B19E3779F9ull;
  x ^= x >> 30;                    // the splitmix64 finalizer
  x *= 0xBF58476D1CE4E5B9ull;
  x ^= x >> 27;
  x *= 0x94D049BB133111EBull;
  x ^= x >> 31;
  return ((float)((x >> 41) & 0x7FFFFFull) + 0.5f) * (1.0f / 8388608.0f);   // 23 bits: u in (0, 1), never 1
}

// BF16 bits → a 16-bit key that orders like the value (sign flipped: negative values reversed)
__device__ __forceinline__ uint32_t key16(uint32_t bits) { return bits & 0x8000u ? (~bits) & 0xFFFFu : bits | 0x8000u; }
__device__ __forceinline__ float key_val(uint32_t key) {
  const uint32_t bits = key & 0x8000u ? key & 0x7FFFu : (~key) & 0xFFFFu;
  return __uint_as_float(bits << 16);
}

constexpr uint32_t HIST_KEYS = 65536;
constexpr int SELECT_THREADS = 1024;
constexpr int SELECT_WAVES = SELECT_THREADS / 64;
constexpr uint32_t WAVE_KEYS = HIST_KEYS / SELECT_WAVES;   // keys per wave, descending from 65535 − 4096·w
constexpr int KEY_BLOCK = 64;                              // keys a thread counts and merges (1024 blocks)
constexpr int PART_U64 = KEY_BLOCK * 2 / 8;                // a block's 16-bit counts, in 8-byte words
constexpr int SELECT_MIN_WGS = 4;
constexpr int SELECT_SPAN_MAX = 65528;                     // logits per workgroup: a 16-bit count cannot overflow

template <typename T>
__device__ __forceinline__ T wave_total(T v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// A row's counts as sample_threshold's last workgroup holds them: 16 bits a key in LDS, and the few carries past them
// (each at least 32768 logits of a row of at most 2^20)
constexpr int MAX_CARRY = 32;
constexpr int CARRY_SPAN = 32760;                          // logits one workgroup counts between two sweeps of carries
struct KeyCounts {
  const uint16_t* h;
  const uint32_t* carry_key;
  const uint32_t* carry;
  int n_carry;
  __device__ __forceinline__ uint32_t operator()(uint32_t k) const {
    uint32_t c = h[k];
    for (int i = 0; i < n_carry; ++i) c += carry_key[i] == k ? carry[i] : 0u;
    return c;
  }
};

// The chunks of 64 keys of a wave (lane 0 the highest key of a chunk) that hold a count, from the top, four at a time:
// f(q[4], cnt[4], n) for the next n chunks (past n: chunk 63, its count taken as 0); f returns whether to stop
template <typename F>
__device__ __forceinline__ void for_chunks(const KeyCounts& kc, unsigned long long occ, uint32_t hi, int lane, F f) {
  while (occ) {
    int q[4], n = 0;
    uint32_t c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      q[j] = occ ? __builtin_ctzll(occ) : 63;
      n += occ ? 1 : 0;
      occ &= occ - 1;                               // 0 stays 0
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) c[j] = kc(hi - 64 * q[j] - lane);
#pragma unroll
    for (int j = 1; j < 4; ++j) c[j] = j < n ? c[j] : 0u;
    if (f(q, c)) return;
  }
}

// the key where a descending cumulative sum starting at `run` first reaches `target`, walking this wave's keys; -inf
// when it has none, the lowest when the sums' order leaves the target a rounding short. A chunk's total (a balanced
// tree over the lanes, as lane 63 of its inclusive prefix) moves the sum on; only a chunk that may hold the target (a
// margin of 2^-16 covers the prefix's other order of the same sum) has its prefix formed, through the lane exchanges
template <bool MASS>
__device__ __forceinline__ float walk_to(const KeyCounts& kc, unsigned long long occ, uint32_t hi, float vmax, float inv_t,
                                         float run, float target, int lane) {
  float res = -INFINITY;
  for_chunks(kc, occ, hi, lane, [&](const int (&q)[4], const uint32_t (&c)[4]) {
    float x[4], tot[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t k = hi - 64 * q[j] - lane;
      x[j] = MASS ? (c[j] ? (float)c[j] * expf((key_val(k) - vmax) * inv_t) : 0.0f) : (float)c[j];
      tot[j] = wave_sum(x[j]);
    }
    for (int j = 0; j < 4; ++j) {
      const float xj = j == 0 ? x[0] : j == 1 ? x[1] : j == 2 ? x[2] : x[3];
      const float tj = j == 0 ? tot[0] : j == 1 ? tot[1] : j == 2 ? tot[2] : tot[3];
      const uint32_t cj = j == 0 ? c[0] : j == 1 ? c[1] : j == 2 ? c[2] : c[3];
      const uint32_t top = hi - 64 * (j == 0 ? q[0] : j == 1 ? q[1] : j == 2 ? q[2] : q[3]);
      const unsigned long long nz = __ballot(cj != 0u);
      if ((run + tj) * (1.0f + 1.0f / 65536.0f) >= target) {
        float s = xj;
        for (int off = 1; off < 64; off <<= 1) {    // inclusive prefix over the lanes
          const float u = __shfl_up(s, off);
          s = lane >= off ? s + u : s;
        }
        const unsigned long long hit = __ballot(cj != 0u && run + s >= target);
        if (hit) {
          res = key_val(top - (uint32_t)__builtin_ctzll(hit));
          return true;
        }
      }
      if (nz) res = key_val(top - (63u - (uint32_t)__builtin_clzll(nz)));   // the lowest key with a count so far
      run += tj;
    }
    return false;
  });
  return res;
}

// grid (workgroups, rows): the threshold tau of each row (sample.metal `sample_select`), the most restrictive of
// top-k (the k-th largest logit, ties kept), top-p (the key at which the descending cumulative softmax mass of
// logits / temperature first reaches p of the total — of the top-k set's mass with flag 8) and min-p (max +
// temperature · log(min_p)), from the counts of the row's logit keys.
//
// What bounds it is latency: half a megabyte of logits, but 65536 counters. Counting with device-scope atomics on a
// table in memory took 88 us for a row of 248320 logits (hot keys serialize at the coherence point) and walking that
// table from one workgroup 49 us. Here a workgroup counts its span in LDS, 16 bits a key (128 KB, so a span stays under
// 65536 logits; at least four workgroups a row, so that counting is short), publishes the blocks of 64 keys that hold
// anything with a 1024-bit map of them (device-scope stores), and the row's last workgroup to arrive adds the published
// blocks to its own and finds tau, looking only at the chunks of keys that hold a count: 20 us for that row (counting
// 6, publishing and arriving 5, merging 3, the sums and the walk 6), and 49 us with the draw for 16 rows. Six or eight
// workgroups a row count faster and merge slower (27 us with the draw either way at 248320 logits, 21 → 23 us at 32000).
// Every loop over the keys is rolled: with the counts in registers the kernel was 93 KB of straight-line code, and
// fetching it cost more than its work.
//
// The sums keep one fixed order: wave w owns the keys 65535 − 4096·w − [0, 4096), lane l the keys ≡ 63 − l mod 64,
// added from the top down; lanes, then waves; the wave whose share crosses the target walks its keys in order.
__global__ __launch_bounds__(SELECT_THREADS) void sample_threshold(const uint16_t* logits, int ld, int vocab, int span,
                                                                   uint32_t* counters, unsigned long long* maps,
                                                                   unsigned long long* part, float* tau, int top_k,
                                                                   float temperature, float top_p, float min_p,
                                                                   uint32_t flags) {
  extern __shared__ __attribute__((aligned(16))) uint32_t h16[];   // [32768]: the counts of keys 2i, 2i + 1
  __shared__ uint32_t wmax[SELECT_WAVES];
  __shared__ uint32_t wcnt[SELECT_WAVES];
  __shared__ float wmass[SELECT_WAVES], wmass_k[SELECT_WAVES];
  __shared__ float res[2];
  __shared__ int last;
  __shared__ uint32_t carry_key[MAX_CARRY], carry[MAX_CARRY], n_carry;
  const int tid = threadIdx.x, lane = tid & 63, row = blockIdx.y, nb = gridDim.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lo = blockIdx.x * span, n = min(span, vocab - lo);     // n >= 1
  const uint16_t* p = logits + (long long)row * ld + lo;

  // ---- count this span ------------------------------------------------------------------------------------------
#pragma unroll
  for (int i = 0; i < (int)HIST_KEYS / 2 / 4 / SELECT_THREADS; ++i)
    reinterpret_cast<uint4*>(h16)[i * SELECT_THREADS + tid] = uint4{0u, 0u, 0u, 0u};
  if (tid == 0) n_carry = 0;
  __syncthreads();
  auto count = [&](uint32_t bits) {
    const uint32_t k = key16(bits);
    atomicAdd(&h16[k >> 1], (k & 1u) ? 0x10000u : 1u);
  };
  auto count_span = [&](const uint16_t* p, int n) {
    const int nv = (reinterpret_cast<uintptr_t>(p) & 15) == 0 ? n / 8 : 0;   // whole 16-byte vectors of an aligned row
    constexpr int UN = 4;                                                    // vectors in flight per thread
    for (int v0 = tid; v0 < nv; v0 += UN * SELECT_THREADS) {
      uint4 q[UN];
#pragma unroll
      for (int i = 0; i < UN; ++i) q[i] = reinterpret_cast<const uint4*>(p)[min(v0 + i * SELECT_THREADS, nv - 1)];
#pragma unroll
      for (int i = 0; i < UN; ++i) {
        if (v0 + i * SELECT_THREADS >= nv) break;
        const uint32_t qw[4] = {q[i].x, q[i].y, q[i].z, q[i].w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          count(qw[e] & 0xFFFFu);
          count(qw[e] >> 16);
        }
      }
    }
    for (int c = 8 * nv + tid; c < n; c += 8 * SELECT_THREADS) {             // the rest, or an unaligned row
      uint16_t b[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = p[min(c + i * SELECT_THREADS, n - 1)];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (c + i * SELECT_THREADS < n) count(b[i]);
    }
    __syncthreads();
  };
  // a row in one workgroup (no room for more in the workspace): the counts from 32768 on go to the carries between spans
  const int sub = n > SELECT_SPAN_MAX ? CARRY_SPAN : n;
#pragma unroll 1
  for (int at = 0;;) {
    count_span(p + at, min(sub, n - at));
    at += sub;
    if (at >= n) break;
    for (int i = 0; i < KEY_BLOCK / 2; ++i) {
      const int word = tid * (KEY_BLOCK / 2) + ((i + tid) & (KEY_BLOCK / 2 - 1));
      const uint32_t c = h16[word];
      if (!(c & 0x80008000u)) continue;
      h16[word] = c & 0x7FFF7FFFu;
      for (int e = 0; e < 2; ++e)
        if ((c >> (16 * e + 15)) & 1u) {
          const uint32_t slot = atomicAdd(&n_carry, 1u);
          if (slot < MAX_CARRY) { carry_key[slot] = 2 * word + e; carry[slot] = 32768u; }
        }
    }
    __syncthreads();
  }

  if (nb > 1) {
    // ---- publish: thread b the block of keys 64·b .. + 63, its 16 words in an order rotated by the thread (no bank
    // conflicts; the thread of the same number adds them in the same order), word i of every block side by side
    unsigned long long* mine = reinterpret_cast<unsigned long long*>(h16) + tid * PART_U64;
    const long long at = (long long)row * nb + blockIdx.x;
    unsigned long long any = 0, v[PART_U64];
#pragma unroll
    for (int i = 0; i < PART_U64; ++i) any |= v[i] = mine[(i + tid) & (PART_U64 - 1)];
    if (any) {
      unsigned long long* dst = part + at * PART_U64 * SELECT_THREADS + tid;
#pragma unroll
      for (int i = 0; i < PART_U64; ++i) st_dev8(dst + i * SELECT_THREADS, v[i]);
    }
    const unsigned long long map = __ballot(any != 0);
    if (lane == 0) st_dev8(maps + at * SELECT_WAVES + w, map);
    // every wave's stores acknowledged at the coherence point before the row's count moves
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const uint32_t prev = __hip_atomic_fetch_add(counters + row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = prev == (uint32_t)(nb - 1);
      if (last) __hip_atomic_store(counters + row, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!last) return;

    // ---- the row's last workgroup: add the other workgroups' blocks, three workgroups at a time. Wave w adds word w of
    // the blocks; it goes through the groups of 64 blocks that any of the three holds, four groups' loads in flight. A
    // block its map leaves out was not written: read, and not added
    constexpr int MG = 3, BG = 4;
    static_assert(SELECT_WAVES == PART_U64, "wave w adds word w of every block");
    auto wg_of = [&](int i) { return (long long)row * nb + (blockIdx.x + 1 + i) % nb; };   // the others, i < nb − 1
    for (int g0 = 0; g0 < nb - 1; g0 += MG) {
      unsigned long long m[MG], held = 0;              // lane l: the maps' words of blocks 64·(l % 16) .. + 63
#pragma unroll
      for (int g = 0; g < MG; ++g) m[g] = ld_dev8(maps + wg_of(min(g0 + g, nb - 2)) * SELECT_WAVES + (lane & 15));
#pragma unroll
      for (int g = 0; g < MG; ++g) {
        if (g0 + g >= nb - 1) m[g] = 0;                // past the last: re-read, not added
        held |= m[g];
      }
      uint32_t todo = (uint32_t)__ballot(held != 0) & 0xFFFFu;
      while (todo) {
        unsigned long long buf[BG][MG];
        int bg[BG], nbg = 0;
#pragma unroll
        for (int j = 0; j < BG; ++j) {                 // past the last group: the group before again, not added
          if (todo) { bg[j] = __builtin_ctz(todo); ++nbg; } else { bg[j] = bg[max(j - 1, 0)]; }
          todo &= todo - 1;
#pragma unroll
          for (int g = 0; g < MG; ++g)
            buf[j][g] = ld_dev8(part + (wg_of(min(g0 + g, nb - 2)) * PART_U64 + w) * SELECT_THREADS + 64 * bg[j] + lane);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < BG; ++j) {
          if (j >= nbg) break;
          unsigned long long x[MG];
#pragma unroll
          for (int g = 0; g < MG; ++g) {
            const unsigned long long on = (unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)m[g], bg[j]) |
                                          ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(m[g] >> 32), bg[j]) << 32);
            x[g] = (on >> lane) & 1ull ? buf[j][g] : 0ull;
          }
          const int b = 64 * bg[j] + lane, word = b * PART_U64 + ((w + b) & (PART_U64 - 1));
          unsigned long long* at64 = reinterpret_cast<unsigned long long*>(h16) + word;
          const unsigned long long own = *at64;
          uint32_t c[4] = {(uint32_t)own & 0xFFFFu, (uint32_t)own >> 16, (uint32_t)(own >> 32) & 0xFFFFu, (uint32_t)(own >> 48)};
#pragma unroll
          for (int g = 0; g < MG; ++g) {
            c[0] += (uint32_t)x[g] & 0xFFFFu;
            c[1] += (uint32_t)x[g] >> 16;
            c[2] += (uint32_t)(x[g] >> 32) & 0xFFFFu;
            c[3] += (uint32_t)(x[g] >> 48);
          }
          *at64 = (unsigned long long)((c[0] & 0xFFFFu) | (c[1] << 16)) |
                  ((unsigned long long)((c[2] & 0xFFFFu) | (c[3] << 16)) << 32);
          if ((c[0] | c[1] | c[2] | c[3]) >> 16) {     // a key past 65535
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (c[e] >> 16) {
                const uint32_t slot = atomicAdd(&n_carry, 1u);
                if (slot < MAX_CARRY) { carry_key[slot] = 4 * word + e; carry[slot] = c[e] & 0xFFFF0000u; }
              }
          }
        }
      }
    }
    __syncthreads();
  }

  // ---- tau: thread (w, l) takes the keys hi − 64·q − l, hi = 65535 − 4096·w; occ: the chunks q that hold a count -----
  const KeyCounts kc{reinterpret_cast<const uint16_t*>(h16), carry_key, carry, (int)min(n_carry, (uint32_t)MAX_CARRY)};
  const uint32_t hi = HIST_KEYS - 1 - (uint32_t)w * WAVE_KEYS;
  unsigned long long occ = 0;
  for (int q0 = 0; q0 < 64; q0 += 16) {
    uint32_t c[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) c[j] = kc.h[hi - 64 * (q0 + j) - lane];
#pragma unroll
    for (int j = 0; j < 16; ++j) occ |= __ballot(c[j] != 0u) ? 1ull << (q0 + j) : 0ull;
  }
  if (kc.n_carry)                                   // a count of 65536, …: its low bits may be 0
    for (int i = 0; i < kc.n_carry; ++i)
      if (carry_key[i] <= hi && carry_key[i] > hi - WAVE_KEYS) occ |= 1ull << ((hi - carry_key[i]) >> 6);
  uint32_t km = 0;                                  // the wave's highest key with a count
  if (occ) {
    const uint32_t top = hi - 64 * (uint32_t)__builtin_ctzll(occ);
    km = top - (uint32_t)__builtin_ctzll(__ballot(kc(top - lane) != 0u));
  }
  if (lane == 0) wmax[w] = km;
  if (tid == 0) { res[0] = -INFINITY; res[1] = -INFINITY; }
  __syncthreads();
  uint32_t gmax = 0;
#pragma unroll
  for (int i = 0; i < SELECT_WAVES; ++i) gmax = max(gmax, wmax[i]);
  const float vmax = key_val(gmax), inv_t = 1.0f / temperature;
  float tau_k = -INFINITY, tau_p = -INFINITY, tau_m = -INFINITY;
  if (flags & 1u) {                                 // top-k: counts are exact
    uint32_t c = 0;
    for_chunks(kc, occ, hi, lane, [&](const int (&)[4], const uint32_t (&x)[4]) {
      c += x[0] + x[1] + x[2] + x[3];
      return false;
    });
    c = wave_total(c);
    if (lane == 0) wcnt[w] = c;
    __syncthreads();
    uint32_t before = 0;
    for (int i = 0; i < w; ++i) before += wcnt[i];
    if (before < (uint32_t)top_k && before + wcnt[w] >= (uint32_t)top_k) {
      const float kk = walk_to<false>(kc, occ, hi, vmax, inv_t, (float)before, (float)top_k, lane);
      if (lane == 0) res[0] = kk;
    }
    __syncthreads();
    tau_k = res[0];                                 // k beyond the vocabulary: every logit kept (−inf)
  }
  if (flags & 2u) {
    float m = 0.0f, mk = 0.0f;
    for_chunks(kc, occ, hi, lane, [&](const int (&q)[4], const uint32_t (&c)[4]) {
      float kv[4], x[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kv[j] = key_val(hi - 64 * q[j] - lane);
        x[j] = (float)c[j] * expf((kv[j] - vmax) * inv_t);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        m = c[j] ? m + x[j] : m;
        mk = c[j] && kv[j] >= tau_k ? mk + x[j] : mk;
      }
      return false;
    });
    m = wave_total(m);
    mk = wave_total(mk);
    if (lane == 0) { wmass[w] = m; wmass_k[w] = mk; }
    __syncthreads();
    float total = 0.0f, before = 0.0f;
    for (int i = 0; i < SELECT_WAVES; ++i) total += (flags & 9u) == 9u ? wmass_k[i] : wmass[i];
    for (int i = 0; i < w; ++i) before += wmass[i];
    const float target = top_p * total;
    if (before < target && before + wmass[w] >= target) {
      const float kp = walk_to<true>(kc, occ, hi, vmax, inv_t, before, target, lane);
      if (lane == 0) res[1] = kp;
    }
    __syncthreads();
    tau_p = res[1];
  }
  if (flags & 4u) tau_m = vmax + temperature * logf(min_p);
  if (tid == 0) tau[row] = fmaxf(fmaxf(tau_k, tau_p), tau_m);
}

// grid (spans, rows): each workgroup scans `span` logits of one row with 16-byte loads, publishes its best,
// and the last workgroup of the row to arrive folds the row's partials and resets the row's counter. SAMPLE: the
// value of a BF16 logit v >= tau is v / temperature + its Gumbel noise, any other logit is left out.
template <bool SAMPLE>
__global__ __launch_bounds__(ARGMAX_THREADS) void argmax_spans(mi_argmax_desc d, int span, uint32_t* counters,
                                                               unsigned long long* part, SampleCtx sc) {
  __shared__ float sv[ARGMAX_THREADS / 64];
  __shared__ int si[ARGMAX_THREADS / 64];
  __shared__ int last;
  const int row = blockIdx.y, nb = gridDim.x, tid = threadIdx.x;
  const int lo = blockIdx.x * span, hi = min(lo + span, d.vocab);
  float bv = -INFINITY;
  int bi = 0x7FFFFFFF;
  float th = 0.0f;
  uint32_t seed_lo = 0, seed_hi = 0, step = 0;
  if constexpr (SAMPLE) {
    th = sc.tau ? sc.tau[row] : -INFINITY;          // null: every logit kept
    seed_lo = sc.st ? (uint32_t)sc.st->rng_lo : sc.seed_lo;
    seed_hi = sc.st ? (uint32_t)sc.st->rng_hi : sc.seed_hi;
    step = sc.st ? sc.st->step : sc.step;
  }
  if (!SAMPLE && d.f32) {
    const float* p = static_cast<const float*>(d.logits) + (long long)row * d.ld;
    const bool vec = ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)lo * 4) & 15) == 0;
    for (int c = lo + tid * 4; c < hi; c += ARGMAX_THREADS * 4) {
      float v[4];
      if (vec && c + 4 <= hi) {
        const float4 q = *reinterpret_cast<const float4*>(p + c);
        v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
      } else {
        for (int e = 0; e < 4; ++e) v[e] = c + e < hi ? p[c + e] : NAN;
      }
      for (int e = 0; e < 4; ++e)
        if (better(v[e], c + e, bv, bi)) { bv = v[e]; bi = c + e; }
    }
  } else {
    const uint16_t* p = static_cast<const uint16_t*>(d.logits) + (long long)row * d.ld;
    const bool vec = ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)lo * 2) & 15) == 0;
    for (int c = lo + tid * 8; c < hi; c += ARGMAX_THREADS * 8) {
      uint32_t w[4];
      if (vec && c + 8 <= hi) {
        const uint4 q = *reinterpret_cast<const uint4*>(p + c);
        w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
      } else {
        for (int e = 0; e < 4; ++e) {
          const uint32_t a = c + 2 * e < hi ? p[c + 2 * e] : 0x7FC0u;          // past the end: NaN
          const uint32_t b = c + 2 * e + 1 < hi ? p[c + 2 * e + 1] : 0x7FC0u;
          w[e] = a | (b << 16);
        }
      }
      for (int e = 0; e < 4; ++e) {
        float v0 = __uint_as_float(w[e] << 16), v1 = __uint_as_float(w[e] & 0xFFFF0000u);
        if constexpr (SAMPLE) {
          v0 = v0 >= th ? v0 * sc.inv_t - logf(-logf(uniform01(seed_lo, seed_hi, step, row, c + 2 * e))) : NAN;
          v1 = v1 >= th ? v1 * sc.inv_t - logf(-logf(uniform01(seed_lo, seed_hi, step, row, c + 2 * e + 1))) : NAN;
        }
        if (better(v0, c + 2 * e, bv, bi)) { bv = v0; bi = c + 2 * e; }
        if (better(v1, c + 2 * e + 1, bv, bi)) { bv = v1; bi = c + 2 * e + 1; }
      }
    }
  }
  block_best(bv, bi, sv, si);
  // published without a fence (an agent-scope release writes back the whole L2): the partial's device-scope store is
  // acknowledged before the row's count moves, and the last workgroup reads the partials with device-scope loads
  if (tid == 0) {
    st_dev8(part + row * nb + blockIdx.x,
            (unsigned long long)__float_as_uint(bv) | ((unsigned long long)(uint32_t)bi << 32));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(&counters[row], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)(nb - 1);
  }
  __syncthreads();
  if (!last) return;
  bv = -INFINITY;
  bi = 0x7FFFFFFF;
  for (int k = tid; k < nb; k += ARGMAX_THREADS) {
    const unsigned long long q = ld_dev8(part + row * nb + k);
    const float qv = __uint_as_float((uint32_t)q);
    const int qi = (int)(uint32_t)(q >> 32);
    if (better(qv, qi, bv, bi)) { bv = qv; bi = qi; }
  }
  __syncthreads();                                  // sv / si are reused
  block_best(bv, bi, sv, si);
  if (tid == 0) {
    d.ids[row] = bi == 0x7FFFFFFF ? -1 : bi;        // no number in the row
    __hip_atomic_store(&counters[row], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

__device__ __forceinline__ void publish_ctl(uint32_t* ctl, const mi_step_state* st) {
  if (ctl) {                                        // posted writes to pinned host memory: the pump polls these
    __atomic_store_n(&ctl[2], st->error, __ATOMIC_RELAXED);
    __atomic_store_n(&ctl[1], st->done, __ATOMIC_RELEASE);
  }
}

// one thread: the ring, the position and the stop conditions
__global__ __launch_bounds__(64) void advance_step(mi_advance_desc d) {
  if (threadIdx.x != 0) return;
  mi_step_state* st = d.state;
  if (st->done) return;
  const uint32_t t = min(max(st->t_this_step, 1u), (uint32_t)MI_STEP_T_MAX);   // a state the host left inconsistent
  if (st->prefill_left > 0) {                       // a prompt chunk: no token leaves the step
    st->position += t;
    st->step += 1;
    if (d.ctx_cap && st->position >= d.ctx_cap) { st->error = 2; st->done = 1; }
    publish_ctl(d.host_ctl, st);
    return;
  }
  const int32_t tok = d.tokens[t - 1];
  const uint32_t head = st->ring_head;
  if (head - st->ring_tail >= d.ring_cap) {         // the host has not drained: overflow
    st->error = 1;
    st->done = 1;
    publish_ctl(d.host_ctl, st);
    return;
  }
  d.ring[head % d.ring_cap] = ((uint64_t)(head + 1) << 32) | (uint32_t)tok;
  st->ring_head = head + 1;
  if (st->stop_at && head + 1 >= st->stop_at) st->done = 1;
  st->pending_tokens[0] = tok;
  st->position += t;
  st->step += 1;
  st->t_this_step = 1;
  for (int i = 0; i < d.n_eos; ++i)
    if (tok == d.eos[i]) st->done = 1;
  if (d.ctx_cap && st->position >= d.ctx_cap) { st->error = 2; st->done = 1; }
  publish_ctl(d.host_ctl, st);
}

int argmax_spans_of(int vocab) { return (vocab + ARGMAX_SPAN - 1) / ARGMAX_SPAN; }

// the 8-byte partials of a workspace that starts on 4 bytes lie 4 before where they would (the counters end long before)
char* down8(void* ws) { return reinterpret_cast<char*>(reinterpret_cast<uintptr_t>(ws) & ~(uintptr_t)7); }

// sample_threshold's workgroups per row and the logits each counts (a multiple of 8: rows stay 16-byte aligned)
int select_span_of(int vocab, int* wgs) {
  const int n = std::max(SELECT_MIN_WGS, (vocab + SELECT_SPAN_MAX - 1) / SELECT_SPAN_MAX);
  const int span = ((vocab + n - 1) / n + 7) / 8 * 8;
  *wgs = (vocab + span - 1) / span;
  return span;
}

__global__ __launch_bounds__(64) void verify_select_step(mi_verify_select_desc d) {
  if (threadIdx.x != 0) return;
  mi_step_state* st = d.state;
  if (st->done) return;
  if (d.lm) st->drafter_ctx_len = st->position + (st->prefill_left > 0 ? 0u : d.gamma);
  else st->drafter_ctx_len += st->n_inject;
  st->n_inject = 0;
  if (st->prefill_left > 0) return;                 // the host feeds the next prompt chunk
  for (uint32_t k = 0; k < d.gamma; ++k) {
    st->draft_tokens[k] = d.drafts[k];
    st->confidence[k] = d.conf[k];
    if (d.log_cap) d.conf_log[(st->step % d.log_cap) * 16 + k] = d.conf[k];
  }
  uint32_t lmax = min(d.gamma, d.t_max - 1);
  if (d.ctx_cap) {                                  // the verify rows position … position + L must fit the caches
    if (st->position >= d.ctx_cap) { st->error = 2; st->done = 1; return; }
    lmax = min(lmax, d.ctx_cap - st->position - 1);
  }
  uint32_t L = 0;
  if (d.mode == 2) {
    L = min((uint32_t)fmaxf(d.threshold, 0.f), lmax);
  } else if (d.mode == 1) {
    float survive = 1.f, expected = 1.f, best = 1.f / d.cost[0];
    for (uint32_t l = 1; l <= lmax; ++l) {
      survive *= d.conf[l - 1];
      expected += survive;
      const float score = expected / d.cost[l];
      if (score > best) { best = score; L = l; }
    }
  } else if (d.threshold <= 0.f) {
    L = lmax;
  } else {
    while (L < lmax && d.conf[L] >= d.threshold) ++L;
  }
  st->gamma = d.gamma;
  st->verify_len = L;
  st->pending_tokens[0] = st->anchor;
  for (uint32_t k = 0; k < L; ++k) st->pending_tokens[k + 1] = d.drafts[k];
  st->t_this_step = 1 + L;
}

__device__ __forceinline__ bool is_eos(const int32_t* eos, int n, int32_t tok) {
  bool hit = false;
  for (int i = 0; i < n; ++i) hit |= tok == eos[i];
  return hit;
}

__global__ __launch_bounds__(64) void accept_scan_step(mi_accept_scan_desc d) {
  if (threadIdx.x != 0) return;
  mi_step_state* st = d.state;
  if (st->done) return;
  // the step's rows and verify length as the state holds them, kept inside the token rows whatever the host left
  // there (t in 1..16, L <= t - 1), so no row index falls outside the step
  const uint32_t t = min(max(st->t_this_step, 1u), (uint32_t)MI_STEP_T_MAX);
  if (st->prefill_left > 0) {                       // a prompt chunk: nothing to verify; its rows are injected next
    if (d.log_cap) d.log[st->step % d.log_cap] = (t << 16) | 0xFFFFu;
    st->position += t;
    st->step += 1;
    st->n_inject = t;
    st->checkpoint_index = t;
    st->n_chain = 0;
    if (d.ctx_cap && st->position >= d.ctx_cap) { st->error = 2; st->done = 1; }
    publish_ctl(d.host_ctl, st);
    return;
  }
  const uint32_t L = min(st->verify_len, t - 1);
  const uint32_t base = t - 1 - L;                  // the anchor's row
  uint32_t acc = 0;
  while (acc < L && d.tokens[base + acc] == st->pending_tokens[base + acc + 1]) ++acc;
  const int32_t bonus = d.tokens[base + acc];
  uint32_t head = st->ring_head;
  if (head + acc + 1 - st->ring_tail > d.ring_cap) {  // not enough ring room: the host fell behind
    st->error = 1;
    st->done = 1;
    publish_ctl(d.host_ctl, st);
    return;
  }
  uint32_t committed = 0;
  int32_t last = bonus;
  bool stop = false;
  for (uint32_t k = 0; k <= acc; ++k) {
    const int32_t tok = k < acc ? st->pending_tokens[base + k + 1] : bonus;
    d.ring[head % d.ring_cap] = ((uint64_t)(head + 1) << 32) | (uint32_t)tok;
    ++head;
    ++committed;
    last = tok;
    if (is_eos(d.eos, d.n_eos, tok)) { stop = true; break; }   // nothing after the first EOS is committed
  }
  if (d.log_cap) d.log[st->step % d.log_cap] = (committed << 16) | (L << 8) | acc;
  st->ring_head = head;
  if (st->stop_at && head >= st->stop_at) stop = true;
  st->accepted = acc;
  st->anchor = last;
  st->position += base + committed;
  st->step += 1;
  st->verify_len = 0;
  st->t_this_step = 1;
  st->n_inject = base + committed;
  st->checkpoint_index = base + committed;
  st->n_chain = 1;
  if (d.lm) st->n_inject = st->position > st->drafter_ctx_len ? st->position - st->drafter_ctx_len : 0;
  if (stop) st->done = 1;
  if (d.ctx_cap && st->position >= d.ctx_cap) { st->error = 2; st->done = 1; }
  publish_ctl(d.host_ctl, st);
}

double now_ms() {
  return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

double thread_cpu_ms() {
  timespec ts;
  clock_gettime(CLOCK_THREAD_CPUTIME_ID, &ts);
  return ts.tv_sec * 1e3 + ts.tv_nsec / 1e6;
}

// take slots while the next expected sequence number is present (slots of batches still running may be written in
// any order, so the GPU's head is never trusted), then publish the tail
bool drain_ring(mi_runner_desc* d) {
  const volatile uint64_t* slots = d->ring;
  uint32_t tail = __atomic_load_n(&d->host_ctl[0], __ATOMIC_RELAXED);
  bool full = false;
  for (;;) {
    const uint64_t v = slots[tail % d->ring_capacity];
    if ((uint32_t)(v >> 32) != tail + 1) break;
    if (d->n_tokens >= d->tokens_capacity) { full = true; break; }
    d->tokens[d->n_tokens++] = (int32_t)(uint32_t)v;
    ++tail;
  }
  __atomic_store_n(&d->host_ctl[0], tail, __ATOMIC_RELEASE);
  return full;
}

}  // namespace

extern "C" {

int mi_runner_run(mi_runner_desc* d, mi_runner_stats* st) {
  MI_REQUIRE(d && st && d->graph_exec && (d->state || d->state_ring_tail) && d->ring && d->host_ctl &&
             (d->tokens || !d->tokens_capacity), "mi_runner_run: null pointer");
  MI_REQUIRE(!d->state_done == !d->state_error, "mi_runner_run: state_done and state_error go together");
  MI_REQUIRE(d->ring_capacity > 0 && d->launches_per_batch > 0 && d->in_flight > 0,
             "mi_runner_run: ring_capacity, launches_per_batch and in_flight must be >= 1");
  MI_REQUIRE(d->n_tokens <= d->tokens_capacity, "mi_runner_run: n_tokens exceeds tokens_capacity");
  *st = mi_runner_stats{};
  hipStream_t s = static_cast<hipStream_t>(d->stream);
  auto exec = static_cast<hipGraphExec_t>(d->graph_exec);
  struct Batch { hipEvent_t a, b; };
  std::vector<Batch> pool(d->in_flight);
  for (auto& b : pool) {
    MI_TRY_HIP(hipEventCreate(&b.a), "hipEventCreate");
    MI_TRY_HIP(hipEventCreate(&b.b), "hipEventCreate");
  }
  auto release = [&]() { for (auto& b : pool) { (void)hipEventDestroy(b.a); (void)hipEventDestroy(b.b); } };
  const double t0 = now_ms(), c0 = thread_cpu_ms();
  const uint64_t first = d->n_tokens;
  std::deque<size_t> pending;
  size_t next = 0;
  bool full = false;
  hipError_t err = hipSuccess;
  auto observe = [&]() {
    Batch& b = pool[pending.front()];
    pending.pop_front();
    const double w = now_ms();
    // poll with short sleeps: the pump thread stays idle while the GPU works (hipEventSynchronize spins)
    hipError_t e;
    while ((e = hipEventQuery(b.b)) == hipErrorNotReady) {
      const timespec nap{0, 20000};
      nanosleep(&nap, nullptr);
    }
    st->wait_ms += now_ms() - w;
    if (e != hipSuccess && err == hipSuccess) err = e;
    float ms = 0.f;
    if (e == hipSuccess && hipEventElapsedTime(&ms, b.a, b.b) == hipSuccess) st->gpu_ms += ms;
    st->batches++;
    full = drain_ring(d) || full;
    st->done = __atomic_load_n(d->state_done ? d->state_done : &d->host_ctl[1], __ATOMIC_ACQUIRE);
    st->error = __atomic_load_n(d->state_error ? d->state_error : &d->host_ctl[2], __ATOMIC_RELAXED);
  };
  while (st->launches < d->max_launches && !st->done && !full && err == hipSuccess &&
         (d->max_tokens == 0 || d->n_tokens - first < d->max_tokens)) {
    const double l = now_ms();
    const uint32_t n = (uint32_t)std::min<uint64_t>(d->launches_per_batch, d->max_launches - st->launches);
    Batch& b = pool[next];
    // the tail the GPU checks for overflow: the host's value when the copy runs (it only grows)
    if (d->state_ring_tail)       // a host-resident state: a newer tail than the copy would give is as correct
      __atomic_store_n(d->state_ring_tail, __atomic_load_n(&d->host_ctl[0], __ATOMIC_RELAXED), __ATOMIC_RELEASE);
    else
      err = hipMemcpyAsync(&d->state->ring_tail, &d->host_ctl[0], sizeof(uint32_t), hipMemcpyHostToDevice, s);
    if (err == hipSuccess) err = hipEventRecord(b.a, s);
    for (uint32_t i = 0; i < n && err == hipSuccess; ++i) err = hipGraphLaunch(exec, s);
    if (err == hipSuccess) err = hipEventRecord(b.b, s);
    st->launch_ms += now_ms() - l;
    if (err != hipSuccess) break;
    pending.push_back(next);
    next = (next + 1) % pool.size();
    st->launches += n;
    while (pending.size() >= d->in_flight) observe();
  }
  while (!pending.empty()) observe();
  st->wall_ms = now_ms() - t0;
  st->host_busy_ms = thread_cpu_ms() - c0;
  st->tokens = d->n_tokens - first;
  release();
  MI_TRY_HIP(err, "mi_runner_run");
  return MI_OK;
}

int mi_embed(const mi_embed_desc* d, void* stream) {
  MI_REQUIRE(d && d->tokens && d->table && d->out, "mi_embed: null pointer");
  MI_REQUIRE(d->t >= 1 && d->t <= 16 && d->vocab > 0 && d->hidden > 0 && d->hidden % 8 == 0 && d->ldo >= d->hidden &&
             d->ldo % 8 == 0, "mi_embed: bad shape");
  MI_REQUIRE(((uintptr_t)d->table & 15) == 0 && ((uintptr_t)d->out & 15) == 0, "mi_embed: table / out alignment");
  MI_REQUIRE(!d->t16 || d->hidden % 32 == 0, "mi_embed: a T16 table needs hidden %% 32 == 0");
  const dim3 grid((d->hidden / 8 + EMBED_THREADS - 1) / EMBED_THREADS, d->t);
  hipLaunchKernelGGL(embed_rows, grid, dim3(EMBED_THREADS), 0, static_cast<hipStream_t>(stream), *d);
  MI_TRY_HIP(hipGetLastError(), "embed launch");
  return MI_OK;
}

size_t mi_argmax_workspace_bytes(const mi_argmax_desc* d) {
  if (!d || d->t < 1 || d->vocab < 1) return 0;
  return ARGMAX_COUNTERS + (size_t)d->t * argmax_spans_of(d->vocab) * sizeof(unsigned long long);
}

int mi_argmax(const mi_argmax_desc* d, void* stream) {
  MI_REQUIRE(d && d->logits && d->ids, "mi_argmax: null pointer");
  MI_REQUIRE(d->t >= 1 && d->t <= 16 && d->vocab > 0 && d->ld >= d->vocab, "mi_argmax: bad shape");
  const int nb = argmax_spans_of(d->vocab);
  MI_REQUIRE(nb <= ARGMAX_MAX_SPANS, "mi_argmax: vocab %d exceeds %d", d->vocab, ARGMAX_MAX_SPANS * ARGMAX_SPAN);
  const size_t need = mi_argmax_workspace_bytes(d);
  void* ws = d->workspace;
  if (ws) {
    MI_REQUIRE(d->workspace_bytes >= need, "mi_argmax: workspace %zu B < %zu B", d->workspace_bytes, need);
  } else if (int rc = mi_library_scratch(MI_SCRATCH_ARGMAX, need, static_cast<hipStream_t>(stream), &ws)) {
    return rc;
  }
  auto* counters = static_cast<uint32_t*>(ws);
  auto* part = reinterpret_cast<unsigned long long*>(down8(ws) + ARGMAX_COUNTERS);
  hipLaunchKernelGGL(argmax_spans<false>, dim3(nb, d->t), dim3(ARGMAX_THREADS), 0, static_cast<hipStream_t>(stream),
                     *d, ARGMAX_SPAN, counters, part, SampleCtx{});
  MI_TRY_HIP(hipGetLastError(), "argmax launch");
  return MI_OK;
}

// workspace: argmax counters (16, then sample_threshold's 16) | partials | tau[16] | per (row, workgroup of
// sample_threshold): the maps of its key blocks [16] u64 | the blocks' 16-bit counts [1024][64]
struct SampleLayout {
  int span, wgs;                // the draw's logits per workgroup, sample_threshold's workgroups per row and their span
  int count_span;
  size_t off_tau, off_map, off_part, bytes;
};
SampleLayout sample_layout(int t, int vocab) {
  SampleLayout l{};
  l.span = t <= 2 ? ARGMAX_SPAN / 2 : ARGMAX_SPAN;
  l.count_span = select_span_of(vocab, &l.wgs);
  l.off_tau = (ARGMAX_COUNTERS + (size_t)t * ((vocab + l.span - 1) / l.span) * sizeof(unsigned long long) + 255) / 256 * 256;
  l.off_map = l.off_tau + 256;
  l.off_part = l.off_map + (size_t)t * l.wgs * SELECT_WAVES * sizeof(unsigned long long);
  l.bytes = l.off_part + (size_t)t * l.wgs * SELECT_THREADS * PART_U64 * sizeof(unsigned long long);
  return l;
}
// The least that a call takes, what it asks callers for: 256 KB a row, where the workgroups' counts need 128 KB each and
// at least four. With less than sample_layout's bytes one workgroup counts a row (nothing to publish): 248320 logits
// 27 → 50 us with the draw, 32000 as fast
SampleLayout sample_least(int t, int vocab) {
  SampleLayout l{};
  l.span = ARGMAX_SPAN;
  l.wgs = 1;
  l.count_span = vocab;
  l.off_tau = (ARGMAX_COUNTERS + (size_t)t * argmax_spans_of(vocab) * sizeof(unsigned long long) + 255) / 256 * 256;
  l.off_map = l.off_part = l.off_tau + 256;
  l.bytes = l.off_part + (size_t)t * HIST_KEYS * sizeof(uint32_t);
  return l;
}

size_t mi_sample_workspace_bytes(const mi_sample_desc* d) {
  if (!d || d->t < 1 || d->vocab < 1) return 0;
  return sample_least(d->t, d->vocab).bytes;
}

int mi_sample(const mi_sample_desc* d, void* stream) {
  MI_REQUIRE(d && d->logits && d->ids, "mi_sample: null pointer");
  MI_REQUIRE(d->t >= 1 && d->t <= 16 && d->vocab > 0 && d->ld >= d->vocab, "mi_sample: bad shape");
  MI_REQUIRE(d->temperature > 0.0f && d->top_k >= 0 && d->top_p >= 0.0f && d->min_p >= 0.0f,
             "mi_sample: temperature > 0, top_k / top_p / min_p >= 0 (temperature 0 is mi_argmax)");
  MI_REQUIRE(argmax_spans_of(d->vocab) <= ARGMAX_MAX_SPANS, "mi_sample: vocab %d exceeds %d", d->vocab,
             ARGMAX_MAX_SPANS * ARGMAX_SPAN);
  SampleLayout l = sample_layout(d->t, d->vocab);
  const SampleLayout least = sample_least(d->t, d->vocab);
  void* ws = d->workspace;
  if (ws) {
    MI_REQUIRE(d->workspace_bytes >= least.bytes, "mi_sample: workspace %zu B < %zu B", d->workspace_bytes, least.bytes);
    if (d->workspace_bytes < l.bytes) l = least;
  } else if (mi_library_scratch(MI_SCRATCH_ARGMAX, l.bytes, static_cast<hipStream_t>(stream), &ws)) {
    l = least;                                      // it cannot grow (a capture): what it holds may be enough
    if (int rc = mi_library_scratch(MI_SCRATCH_ARGMAX, l.bytes, static_cast<hipStream_t>(stream), &ws)) return rc;
  }
  char* wb = down8(ws);
  auto* counters = static_cast<uint32_t*>(ws);
  auto* part = reinterpret_cast<unsigned long long*>(wb + ARGMAX_COUNTERS);
  auto* tau = reinterpret_cast<float*>(wb + l.off_tau);
  uint32_t flags = 0;
  if (d->top_k > 0) flags |= 1u;
  if (d->top_p > 0.0f && d->top_p < 1.0f) flags |= 2u;
  if (d->min_p > 0.0f) flags |= 4u;
  if (d->topp_in_topk) flags |= 8u;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (flags & 7u) {
    const size_t lds = HIST_KEYS / 2 * sizeof(uint32_t);
    static std::once_flag once;                     // more than 64 KB of dynamic LDS must be allowed once
    std::call_once(once, [&] {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(sample_threshold),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      (void)hipGetLastError();
    });
    hipLaunchKernelGGL(sample_threshold, dim3(l.wgs, d->t), dim3(SELECT_THREADS), lds, s, d->logits, d->ld, d->vocab, l.count_span,
                       counters + 16, reinterpret_cast<unsigned long long*>(wb + l.off_map),
                       reinterpret_cast<unsigned long long*>(wb + l.off_part), tau, d->top_k, d->temperature, d->top_p,
                       d->min_p, flags);
  } else {
    tau = nullptr;                                  // nothing to cut: keep every logit
  }
  mi_argmax_desc am{};
  am.t = d->t; am.vocab = d->vocab; am.logits = d->logits; am.ld = d->ld; am.f32 = 0; am.ids = d->ids;
  SampleCtx sc{tau, 1.0f / d->temperature, (uint32_t)d->seed, (uint32_t)(d->seed >> 32), d->step, d->state};
  hipLaunchKernelGGL(argmax_spans<true>, dim3((d->vocab + l.span - 1) / l.span, d->t), dim3(ARGMAX_THREADS), 0, s, am, l.span, counters,
                     part, sc);
  MI_TRY_HIP(hipGetLastError(), "sample launch");
  return MI_OK;
}

int mi_advance(const mi_advance_desc* d, void* stream) {
  MI_REQUIRE(d && d->state && d->tokens && d->ring, "mi_advance: null pointer");
  MI_REQUIRE(d->ring_cap >= 1 && d->n_eos >= 0 && d->n_eos <= 8, "mi_advance: ring_cap >= 1, n_eos in 0..8");
  hipLaunchKernelGGL(advance_step, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), *d);
  MI_TRY_HIP(hipGetLastError(), "advance launch");
  return MI_OK;
}

int mi_verify_select(const mi_verify_select_desc* d, void* stream) {
  MI_REQUIRE(d && d->state && (d->gamma == 0 || (d->drafts && d->conf)), "mi_verify_select: null pointer");
  MI_REQUIRE(d->gamma <= MI_STEP_GAMMA_MAX && d->t_max >= 1 && d->t_max <= MI_STEP_T_MAX && d->mode <= 2,
             "mi_verify_select: gamma <= %d, t_max in 1..%d, mode 0..2", MI_STEP_GAMMA_MAX, MI_STEP_T_MAX);
  MI_REQUIRE(!d->log_cap || d->conf_log, "mi_verify_select: log_cap without conf_log");
  if (d->mode == 1)
    for (uint32_t l = 0; l <= d->gamma && l < 16; ++l)
      MI_REQUIRE(d->cost[l] > 0.f, "mi_verify_select: cost[%u] must be positive", l);
  hipLaunchKernelGGL(verify_select_step, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), *d);
  MI_TRY_HIP(hipGetLastError(), "verify_select launch");
  return MI_OK;
}

int mi_accept_scan(const mi_accept_scan_desc* d, void* stream) {
  MI_REQUIRE(d && d->state && d->tokens && d->ring, "mi_accept_scan: null pointer");
  MI_REQUIRE(d->ring_cap >= 1 && d->n_eos >= 0 && d->n_eos <= 8, "mi_accept_scan: ring_cap >= 1, n_eos in 0..8");
  MI_REQUIRE(!d->log_cap || d->log, "mi_accept_scan: log_cap without log");
  hipLaunchKernelGGL(accept_scan_step, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), *d);
  MI_TRY_HIP(hipGetLastError(), "accept_scan launch");
  return MI_OK;
}

void* mi_host_alloc(size_t bytes) {
  void* p = nullptr;
  if (hipHostMalloc(&p, bytes, hipHostMallocCoherent) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  return p;
}

int mi_host_free(void* p) {
  if (p) MI_TRY_HIP(hipHostFree(p), "hipHostFree");
  return MI_OK;
}

}  // extern "C"
