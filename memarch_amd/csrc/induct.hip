// induct.hip — keys-and-locks pointer candidates for MI355X (gfx950): memarch's `FullLM2._induct_raw`
// (full2.py:1499-1535; numpy twin memarch_jax/memarch_jax/induct.py:17-43) and the pointer candidate c1 of the
// mixture producer (full2.py:1559-1563).
//
// For every position t of a text and every lock k (0: the token x[t]; 1: the pair (x[t-1], x[t]); 2: the triple
// (x[t-2], x[t-1], x[t]); missing predecessors are a sentinel that equals no token), last_k[t] is the latest
// j < t whose key equals t's. The candidate is x[last_k[t] + 1] (causal: last + 1 <= t). A position t < k has no
// complete key: it has no last and is no other position's last, so only positions t >= k are entered below.
//
// No sort. A hash table gives every key a slot, and "the previous position with the same slot" follows in two steps:
//   1. insert: each position finds or claims the slot of its key (open addressing; the entry is the claiming position,
//      whose tokens are compared, so a slot stands for exactly one key whatever the hash does; the table has more
//      slots than positions, so a probe always ends). One wave takes one chunk of 64 consecutive positions: matching
//      the slots across its lanes (one ballot per slot bit) gives each lane the previous lane with its key and marks
//      the first and the last lane of every key in the chunk;
//   2. link: one wave walks a text's chunks in order over a table of the latest position per slot: a key's first lane
//      reads it (the previous position, in an earlier chunk), its last lane writes it. A wave's LDS accesses execute
//      in order, so the walk does not wait for a chunk's reads before the next chunk's: every lane reads and writes,
//      the ones with nothing to do at a spare entry of their own, since a branch around an access would wait for it.
// The time is the walk (0.06 us per chunk, 0.03 with the infos of PACK texts, 0.11 in longer ones) and the latencies of
// the steps around it. The work is linear in T up to 32768 tokens, where one walk per lock covers a text; above, every
// part of k_ind_link walks the whole text and the parts grow with T (about 760 per lock at 2^24), so its work grows
// with T^2, spread over the GPU: one text of 2^20 1.60 ms, of 2^22 16.6 ms, of 2^24 191 ms (the sorts this replaced
// took 143, 687 and 3296).
//   k_induct       T <= 8192: one workgroup per text, tables in LDS (32-bit entries; infos and links of 16 bits), all
//                  locks at once up to 2048 tokens, one after the other above.
//   k_ind_*        longer texts, T up to 2^24, on a caller-sized workspace: the insert of all locks and texts over the
//                  whole GPU on tables in global memory, then the walks with the latest positions in LDS (k_ind_walk
//                  up to 32768 positions; k_ind_link above: a text with more slots than a workgroup's LDS holds takes
//                  several workgroups that each keep to their own slots), then the outputs.
// Measured (3 locks): 32 texts x 1024 tokens 12.3 us, 59.6 with the bitonic sorts this replaced; 4 x 8192 84 us against
// 435; 4 x 16384 39 us (insert 21, walks 8; k_ind_link walks them in 34) against 1082.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstddef>

#include "../../include/mce_induct.h"

namespace {

// Positions per text of k_induct: what one workgroup's LDS holds. A batch of texts pays for the line there, few long
// texts do not: 3 locks, us, k_induct against the workspace path at the same lengths (built for the comparison):
//   texts x 2049    1: 24 / 21   16: 25 / 25   64: 26 / 40     300: 50 / 123
//   texts x 4096    1: 44 / 23   16: 45 / 33   64: 46 / 68     300: 90 / 238
//   texts x 8192    1: 83 / 24   16: 85 / 46   64: 87 / 113    128: 90 / 205
constexpr int IND_TMAX = 8192;
constexpr int IND_SMALL = 2048;  // up to here all locks' tables fit at once, with the tokens
constexpr int IND_THREADS_MAX = 1024;
constexpr int LINK_AHEAD = 8;    // chunks of a walk whose infos and reads are in flight together
constexpr uint32_t NONE16 = 0xFFFFu;      // empty 16-bit entry / no previous position
constexpr uint32_t NONE32 = 0xFFFFFFFFu;  // empty 32-bit entry

// Hash of the (k+1)-gram that ends at t (t >= k): multiply-and-fold rounds with odd 64-bit constants (the fractions of
// the golden ratio, sqrt 2 and sqrt 3).
__device__ __forceinline__ uint64_t key_hash(const int64_t* __restrict__ x, int t, int k) {
  uint64_t h = (uint64_t)x[t] * 0x9E3779B97F4A7C15ull;
  h ^= h >> 32;
  if (k > 0) {
    h = (h + (uint64_t)x[t - 1]) * 0x6A09E667F3BCC909ull;
    h ^= h >> 29;
  }
  if (k > 1) {
    h = (h + (uint64_t)x[t - 2]) * 0xBB67AE8584CAA73Bull;
    h ^= h >> 32;
  }
  h *= 0x9E3779B97F4A7C15ull;
  return h ^ (h >> 32);
}
__device__ __forceinline__ bool same_key(const int64_t* __restrict__ x, int a, int b, int k) {
  // no short circuit: all of a key's loads go out together
  int64_t d = x[a] ^ x[b];
  if (k > 0) d |= x[a - 1] ^ x[b - 1];
  if (k > 1) d |= x[a - 2] ^ x[b - 2];
  return d == 0;
}
// The lanes of `valid` whose v (below 2^bits) equals this lane's.
__device__ __forceinline__ uint64_t match_lanes(uint32_t v, int bits, uint64_t valid) {
  uint32_t lo = (uint32_t)valid, hi = (uint32_t)(valid >> 32);
#pragma unroll 4
  for (int b = 0; b < bits; ++b) {
    const uint32_t one = (uint32_t)((int32_t)(v << (31 - b)) >> 31);  // the bit in every position
    const uint64_t bal = __builtin_amdgcn_ballot_w64(one != 0);
    lo &= ~((uint32_t)bal ^ one);
    hi &= ~((uint32_t)(bal >> 32) ^ one);
  }
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ int high_bit(uint64_t m) { return 63 - __builtin_clzll(m); }
// Orders this wave's LDS accesses before the call ahead of those after it, where a walk's lanes hand positions to each
// other: the hardware executes a wave's LDS accesses in order, and this keeps the compiler to it (no instruction).
__device__ __forceinline__ void wave_lds_order() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local"); }

// Outputs of positions i0, i0 + step, ... of a text (xt: its tokens; row0: its first position's flat index) from
// last_at(k, t), the previous position with t's k-gram or -1. cand, on and src go out flat over (t, k), so that the
// lanes of a wave write consecutive elements.
template <typename LastAt>
__device__ void emit(const int64_t* xt, int64_t row0, int T, int locks, int longest, LastAt last_at,
                     const int64_t* __restrict__ bucket, int64_t nbucket, int64_t c1_none, int64_t* __restrict__ cand,
                     uint8_t* __restrict__ on, int64_t* __restrict__ src, int64_t* __restrict__ bk,
                     int64_t* __restrict__ c1, int i0, int step) {
  if (cand != nullptr || on != nullptr || src != nullptr) {
    for (int i = i0; i < T * locks; i += step) {
      const int t = i / locks, k = i - t * locks;
      const int l = last_at(k, t);
      bool o = l >= 0;
      if (longest)
        for (int j = k + 1; j < locks; ++j) o = o && last_at(j, t) < 0;
      const int64_t oi = row0 * locks + i;
      if (cand != nullptr) cand[oi] = l >= 0 ? xt[l + 1] : 0;
      if (on != nullptr) on[oi] = o ? 1 : 0;
      if (src != nullptr) src[oi] = l >= 0 ? (int64_t)l + 1 : 0;
    }
  }
  if (c1 == nullptr && bk == nullptr) return;
  for (int t = i0; t < T; t += step) {
    if (c1 != nullptr) {
      int64_t sum = 0;
      bool any = false, longer = false;
      for (int k = locks - 1; k >= 0; --k) {
        const int l = last_at(k, t);
        if (l < 0 || (longest && longer)) continue;
        sum += xt[l + 1];
        any = longer = true;
      }
      c1[row0 + t] = any ? sum : c1_none;
    }
    if (bk != nullptr) {
      int64_t b = 0;
      if (bucket != nullptr) {
        int64_t xi = xt[t];
        xi = xi < nbucket - 1 ? xi : nbucket - 1;
        b = bucket[xi < 0 ? 0 : xi];
      }
      bk[row0 + t] = b;
    }
  }
}

// ---------------------------------------------------------------------------------------------------------
// One workgroup per text. The slot of t's key (hash h) in a table of mask + 1 slots, found or claimed: an entry is the
// claiming position with 16 bits of its key's hash above, so that nearly every entry of another key is passed without
// a look at its tokens; an odd step over a power of two of slots visits every one.
__device__ __forceinline__ uint32_t lds_slot(uint32_t* tab, uint32_t mask, uint64_t h, const int64_t* x, int t, int k) {
  const uint32_t tag = (uint32_t)(h >> 16) & 0xFFFFu, mine = (tag << 16) | (uint32_t)t;
  const uint32_t step = (uint32_t)(h >> 40) | 1u;
  uint32_t s = (uint32_t)(h >> 32) & mask;
  while (true) {
    const uint32_t e = atomicCAS(tab + s, NONE32, mine);
    if (e == NONE32 || (e >> 16 == tag && same_key(x, (int)(e & 0xFFFFu), t, k))) return s;
    s = (s + step) & mask;
  }
}

// TM: the most positions; LP: locks per round; XL: the tokens are kept in LDS too. Info of a position: its slot (below
// 2 TM <= 2^14), bit 14 set for the first and bit 15 for the last lane of its key in the chunk.
template <int TM, int LP, bool XL>
__global__ __launch_bounds__(IND_THREADS_MAX) void k_induct(const int64_t* __restrict__ x, int T, int Tp, int locks,
                                                            int longest, const int64_t* __restrict__ bucket,
                                                            int64_t nbucket, int64_t c1_none,
                                                            int64_t* __restrict__ cand, uint8_t* __restrict__ on,
                                                            int64_t* __restrict__ src, int64_t* __restrict__ bk,
                                                            int64_t* __restrict__ c1) {
  __shared__ uint32_t tab[LP][2 * TM + 64];  // (and a walk's 64 spare entries)
  __shared__ uint16_t info[LP][TM];
  __shared__ uint16_t last[3][TM + 64];
  __shared__ int64_t xs[XL ? TM : 1];
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, nw = nt >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t* xg = x + (int64_t)blockIdx.x * T;
  const int64_t* xt = XL ? xs : xg;
  const int nch = (T + 63) >> 6;
  const uint32_t mask = 2 * (uint32_t)Tp - 1;
  const int bits = 32 - __builtin_clz(mask);
  if constexpr (XL)
    for (int i = tid; i < T; i += nt) xs[i] = xg[i];

  for (int k0 = 0; k0 < locks; k0 += LP) {
    const int lp = min(LP, locks - k0);
    for (int q = 0; q < lp; ++q)
      for (int i = tid; i < 2 * Tp; i += nt) tab[q][i] = NONE32;
    __syncthreads();
    for (int it = wave; it < lp * nch; it += nw) {
      const int q = it / nch, t = (it - q * nch) * 64 + lane, k = k0 + q;
      const bool ok = t < T && t >= k;
      uint32_t s = 0;
      if (ok) s = lds_slot(tab[q], mask, key_hash(xt, t, k), xt, t, k);
      const uint64_t m = match_lanes(s, bits, __builtin_amdgcn_ballot_w64(ok));
      const uint64_t below = m & ((uint64_t(1) << lane) - 1);
      const bool first = ok && below == 0, final = ok && (m >> lane) == 1;
      info[q][t] = (uint16_t)(s | (first ? 1u << 14 : 0u) | (final ? 1u << 15 : 0u));
      last[k][t] = (uint16_t)(below != 0 && ok ? (uint32_t)(t - lane + high_bit(below)) : NONE16);
    }
    __syncthreads();
    // the tables again, now as the latest position per slot
    for (int q = 0; q < lp; ++q)
      for (int i = tid; i < 2 * Tp; i += nt) tab[q][i] = NONE32;
    __syncthreads();
    if (wave < lp) {
      uint32_t* latest = tab[wave];
      for (int c0 = 0; c0 < nch; c0 += LINK_AHEAD) {
        uint32_t f[LINK_AHEAD], r[LINK_AHEAD];
#pragma unroll
        for (int u = 0; u < LINK_AHEAD; ++u) f[u] = info[wave][min(c0 + u, nch - 1) * 64 + lane];
#pragma unroll
        for (int u = 0; u < LINK_AHEAD; ++u) {
          const uint32_t s = f[u] & 0x3FFFu;
          r[u] = latest[f[u] & (1u << 14) ? s : 2 * TM + lane];
          wave_lds_order();
          latest[f[u] & (1u << 15) ? s : 2 * TM + lane] = (uint32_t)((c0 + u) * 64 + lane);
          wave_lds_order();
        }
#pragma unroll
        for (int u = 0; u < LINK_AHEAD; ++u)
          last[k0 + wave][c0 + u < nch && (f[u] & (1u << 14)) ? (c0 + u) * 64 + lane : TM + lane] = (uint16_t)r[u];
      }
    }
    __syncthreads();
  }
  emit(xt, (int64_t)blockIdx.x * T, T, locks, longest,
       [&](int k, int t) { return last[k][t] == NONE16 ? -1 : (int)last[k][t]; }, bucket, nbucket, c1_none, cand, on,
       src, bk, c1, tid, nt);
}

// ---------------------------------------------------------------------------------------------------------
// Long texts.
constexpr int64_t IND_LONG_MAX = int64_t(1) << 24;  // positions per text of the long path
constexpr int LINK_BYTES = 144 * 1024;              // LDS of a walk's latest positions
constexpr int LINK_THREADS = 256, LONG_AHEAD = 32;
// Info of a position: its slot plus one (at most 2^25 - 1), bit 25 set for the last lane of its key in the chunk, the
// lane of the previous position with its key in the chunk (its own lane: none) in bits 26-31; 0 for t < k.
constexpr uint32_t SLOT_MASK = (1u << 25) - 1;
// Texts of at most PACK_T positions, whose slots fit in 16 bits, have the two table indexes of the walk instead (the
// walk is bound by its instructions, and these need none to be worked out): in the low half the entry to read, the slot
// for the first lane of its key in the chunk, else slots + the lane of the previous position with its key in the chunk
// (its own lane: none), a spare entry; in the high half the entry to write, the slot for the last lane, else the lane's
// spare entry. The links then hold what the walk read, and k_ind_emit takes the rest from the infos.
constexpr int64_t PACK_T = 32768;
constexpr size_t PACK_SLOTS = 65536 - 64;

// Workspace of one text: the locks' tables, `slots` 32-bit entries each, from the start of the text's part (later
// the links last[locks][T] i32: the tables are then no longer needed), and the infos [locks][T] u32 at `info`.
struct LongLayout {
  size_t info, bytes;
  uint32_t slots;
};
inline size_t align256(size_t x) { return (x + 255) & ~size_t(255); }
inline int64_t pow2_at_least(int64_t T) {
  int64_t p = 1;
  while (p < T) p <<= 1;
  return p;
}
// The size is 12 bytes per position of T rounded up to a power of two, plus 4 * locks + 8 per position; the tables
// take all of it but the infos, at most 2 slots per padded position: never fewer than 1.66 slots per position.
LongLayout long_layout(int64_t T, int locks) {
  const size_t tp = (size_t)pow2_at_least(T);
  LongLayout l{};
  const size_t tables = align256(8 * tp) + align256(4 * tp) + align256(8 * (size_t)T);
  l.info = tables;
  l.bytes = tables + align256(4 * (size_t)locks * (size_t)T);
  const size_t slots = std::min(2 * tp, tables / (4 * (size_t)locks));
  l.slots = (uint32_t)std::min(slots, T <= PACK_T ? PACK_SLOTS : (size_t)SLOT_MASK - 1);
  return l;
}

// Empty tables: block (.., text).
__global__ __launch_bounds__(256) void k_ind_clear(char* __restrict__ ws, size_t per_text, uint32_t entries) {
  uint32_t* tab = reinterpret_cast<uint32_t*>(ws + (size_t)blockIdx.y * per_text);
  for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < entries; i += gridDim.x * 256) tab[i] = NONE32;
}

// Slot of t's key (hash h) in a table in global memory, found or claimed. An entry, once set, never changes: the
// claiming position in bits 0-23 (< 2^24) and 7 bits of its key's hash above, so that nearly every entry of another
// key is passed without a look at its tokens. The first probes go to independent places (the tables are up to 60%
// full, where linear probing alone forms long runs, and a wave waits for its slowest lane), the later ones are linear,
// so that they visit every slot.
__device__ __forceinline__ uint32_t place(uint32_t h, uint32_t slots) {
  return (uint32_t)(((uint64_t)h * slots) >> 32);
}
__device__ __forceinline__ uint32_t global_slot(uint32_t* tab, uint32_t slots, uint64_t h,
                                                const int64_t* __restrict__ x, int t, int k) {
  const uint32_t tag = (uint32_t)(h >> 40) & 0x7Fu, mine = (tag << 24) | (uint32_t)t;
  uint32_t g = (uint32_t)h, s = place(g, slots);
  for (int probe = 0;; ++probe) {
    const uint32_t e = atomicCAS(tab + s, NONE32, mine);
    if (e == NONE32 || (e >> 24 == tag && same_key(x, (int)(e & 0xFFFFFFu), t, k))) return s;
    if (probe < 6) {
      g = g * 0x9E3779B1u + (uint32_t)(h >> 32);
      s = place(g, slots);
    } else if (++s == slots) {
      s = 0;
    }
  }
}

// The infos (PACK: of texts of at most PACK_T positions): a wave per (chunk, lock), 4 chunks per block; block (chunk
// group * locks + lock, text). Lanes that start at the same slot let the lowest of them go first and take its slot
// where their key is the same, so that a frequent key costs one access of its entry per chunk.
template <bool PACK>
__global__ __launch_bounds__(256) void k_ind_insert(const int64_t* __restrict__ x, int T, int locks, int bits,
                                                    char* __restrict__ ws, size_t per_text, size_t off_info,
                                                    uint32_t slots) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int k = (int)blockIdx.x % locks, t = ((int)blockIdx.x / locks * 4 + wave) * 64 + lane;
  const int64_t* xt = x + (int64_t)blockIdx.y * T;
  char* base = ws + (size_t)blockIdx.y * per_text;
  uint32_t* tab = reinterpret_cast<uint32_t*>(base) + (size_t)k * slots;
  uint32_t* info = reinterpret_cast<uint32_t*>(base + off_info) + (size_t)k * T;
  const bool ok = t < T && t >= k;
  const uint64_t valid = __builtin_amdgcn_ballot_w64(ok);
  const uint64_t h = ok ? key_hash(xt, t, k) : 0;
  uint32_t s = place((uint32_t)h, slots);
  uint64_t m = match_lanes(s, bits, valid);
  const int lead = ok ? __builtin_ctzll(m) : lane;
  if (ok && lead == lane) s = global_slot(tab, slots, h, xt, t, k);
  const uint32_t ls = __shfl(s, lead);
  // another key that starts at the leader's slot (rare) makes the wave match its lanes again
  const bool same = lead == lane || (ok && same_key(xt, t - lane + lead, t, k));
  if (ok && lead != lane) s = same ? ls : global_slot(tab, slots, h, xt, t, k);
  if (__builtin_amdgcn_ballot_w64(ok && !same) != 0) m = match_lanes(s, bits, valid);
  const uint64_t below = m & ((uint64_t(1) << lane) - 1);
  const int prev = below != 0 ? high_bit(below) : lane;
  if (t >= T) return;
  const bool final = ok && (m >> lane) == 1;
  if constexpr (PACK)
    info[t] = (ok && below == 0 ? s : slots + (ok ? prev : lane)) | ((final ? s : slots + lane) << 16);
  else
    info[t] = ok ? (s + 1) | (final ? 1u << 25 : 0u) | ((uint32_t)prev << 26) : 0u;
}

// A 32-bit word at byte offset `off` of a buffer of `bytes` bytes: out-of-range offsets load 0 and store nothing, so a
// walk needs no branch around its accesses. (The whole offset goes into the per-lane operand: the scalar one is not
// part of the bounds check.)
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc make_rsrc(void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)bytes, 0x00020000);
}

// The walk of a PACK text: block (lock, text); its first wave goes through the chunks, LONG_AHEAD at a time, the infos
// of the next ones in flight.
__global__ __launch_bounds__(LINK_THREADS) void k_ind_walk(int T, char* __restrict__ ws, size_t per_text,
                                                           size_t off_info, uint32_t slots) {
  __shared__ __attribute__((aligned(16))) uint16_t latest[PACK_SLOTS + 64];
  const size_t k = blockIdx.x;
  char* base = ws + (size_t)blockIdx.y * per_text;
  const Rsrc info = make_rsrc(base + off_info + 4 * k * T, 4 * (uint32_t)T);
  const Rsrc link = make_rsrc(base + 4 * k * T, 4 * (uint32_t)T);
  for (uint32_t i = threadIdx.x; i < (slots + 7) / 8; i += LINK_THREADS)
    reinterpret_cast<uint4*>(latest)[i] = uint4{NONE32, NONE32, NONE32, NONE32};
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x, nch = (T + 63) >> 6;
  const uint32_t idle = (slots + lane) * 0x10001u;  // past the text: nothing to read or write
  uint32_t nx[LONG_AHEAD];
#pragma unroll
  for (int u = 0; u < LONG_AHEAD; ++u) nx[u] = __builtin_amdgcn_raw_buffer_load_b32(info, lane * 4 + u * 256, 0, 0);
  for (int c0 = 0; c0 < nch; c0 += LONG_AHEAD) {
    uint32_t f[LONG_AHEAD], l[LONG_AHEAD];
#pragma unroll
    for (int u = 0; u < LONG_AHEAD; ++u) {
      f[u] = nx[u];
      nx[u] = __builtin_amdgcn_raw_buffer_load_b32(info, lane * 4 + (c0 + LONG_AHEAD + u) * 256, 0, 0);
    }
    if ((c0 + LONG_AHEAD) * 64 > T) {  // the last batch
#pragma unroll
      for (int u = 0; u < LONG_AHEAD; ++u)
        if ((c0 + u) * 64 + lane >= T) f[u] = idle;
    }
#pragma unroll
    for (int u = 0; u < LONG_AHEAD; ++u) {
      l[u] = latest[f[u] & 0xFFFFu];
      wave_lds_order();
      latest[f[u] >> 16] = (uint16_t)((c0 + u) * 64 + lane);
      wave_lds_order();
    }
#pragma unroll
    for (int u = 0; u < LONG_AHEAD; ++u)
      __builtin_amdgcn_raw_buffer_store_b32(l[u], link, lane * 4 + (c0 + u) * 256, 0, 0);
  }
}

// The walks of longer texts: block (part * locks + lock, text) links the positions whose slots are in
// [part * CAP, (part + 1) * CAP). P: the type of a position (16 bits while every position and the empty mark fit). The
// first wave walks; the infos of the next LONG_AHEAD chunks are loaded before a batch of chunks is walked, so that the
// walk (about 0.06 us per chunk) covers their latency.
template <typename P>
__global__ __launch_bounds__(LINK_THREADS) void k_ind_link(int T, int locks, char* __restrict__ ws, size_t per_text,
                                                           size_t off_info) {
  constexpr uint32_t CAP = LINK_BYTES / sizeof(P);
  constexpr int LA = LONG_AHEAD;
  __shared__ __attribute__((aligned(16))) P latest[CAP + 64];  // and the spare entries
  const int k = (int)blockIdx.x % locks;
  const uint32_t lo = ((uint32_t)blockIdx.x / (uint32_t)locks) * CAP;
  char* base = ws + (size_t)blockIdx.y * per_text;
  const Rsrc info = make_rsrc(base + off_info + 4 * (size_t)k * T, 4 * (uint32_t)T);
  const Rsrc link = make_rsrc(base + 4 * (size_t)k * T, 4 * (uint32_t)T);
  for (uint32_t i = threadIdx.x; i < LINK_BYTES / 16; i += LINK_THREADS)
    reinterpret_cast<uint4*>(latest)[i] = uint4{NONE32, NONE32, NONE32, NONE32};
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const int lane = threadIdx.x, nch = (T + 63) >> 6;
  uint32_t nx[LA];
#pragma unroll
  for (int u = 0; u < LA; ++u) nx[u] = __builtin_amdgcn_raw_buffer_load_b32(info, (u * 64 + lane) * 4, 0, 0);
  for (int c0 = 0; c0 < nch; c0 += LA) {
    uint32_t f[LA], l[LA];
#pragma unroll
    for (int u = 0; u < LA; ++u) {
      f[u] = nx[u];
      nx[u] = __builtin_amdgcn_raw_buffer_load_b32(info, ((c0 + LA + u) * 64 + lane) * 4, 0, 0);
    }
#pragma unroll
    for (int u = 0; u < LA; ++u) {
      const uint32_t s = (f[u] & SLOT_MASK) - 1 - lo;
      const bool mine = f[u] != 0 && s < CAP;
      l[u] = latest[mine && (int)(f[u] >> 26) == lane ? s : CAP + lane];
      wave_lds_order();
      latest[mine && (f[u] & (1u << 25)) ? s : CAP + lane] = (P)((c0 + u) * 64 + lane);
      wave_lds_order();
    }
#pragma unroll
    for (int u = 0; u < LA; ++u) {
      const int t0 = (c0 + u) * 64, t = t0 + lane, prev = (int)(f[u] >> 26);
      const bool none = f[u] == 0;
      const int r = none ? -1 : prev != lane ? t0 + prev : l[u] == (P)NONE32 ? -1 : (int)l[u];
      // a position without a key (t < k) belongs to the first part
      const bool mine = none ? lo == 0 : (f[u] & SLOT_MASK) - 1 - lo < CAP;
      __builtin_amdgcn_raw_buffer_store_b32((uint32_t)r, link, mine ? t * 4 : -4, 0, 0);
    }
  }
}

template <bool PACK>
__global__ __launch_bounds__(256) void k_ind_emit(const int64_t* __restrict__ x, int T, int locks, int longest,
                                                  const int64_t* __restrict__ bucket, int64_t nbucket, int64_t c1_none,
                                                  const char* __restrict__ ws, size_t per_text,
                                                  int64_t* __restrict__ cand, uint8_t* __restrict__ on,
                                                  int64_t* __restrict__ src, int64_t* __restrict__ bk,
                                                  int64_t* __restrict__ c1, int64_t text0, size_t off_info,
                                                  uint32_t slots) {
  const int32_t* last = reinterpret_cast<const int32_t*>(ws + (size_t)blockIdx.y * per_text);
  const uint32_t* info = reinterpret_cast<const uint32_t*>(ws + (size_t)blockIdx.y * per_text + off_info);
  const int64_t row0 = (text0 + blockIdx.y) * T;
  emit(x + (int64_t)blockIdx.y * T, row0, T, locks, longest,
       [&](int k, int t) {
         const int l = last[(size_t)k * T + t];
         if constexpr (PACK) {
           const uint32_t f = info[(size_t)k * T + t] & 0xFFFFu;
           if (f < slots) return l == (int)NONE16 ? -1 : l;
           return (int)(f - slots) == (t & 63) ? -1 : (t & ~63) + (int)(f - slots);
         }
         return l;
       },
       bucket, nbucket, c1_none, cand, on, src, bk, c1,
       (int)blockIdx.x * 256 + (int)threadIdx.x, (int)gridDim.x * 256);
}

thread_local int g_induct_hip_error = 0;  // the calling thread's last failed launch

int launched() {
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess) return MCE_INDUCT_OK;
  g_induct_hip_error = (int)e;
  return MCE_INDUCT_ELAUNCH;
}

}  // namespace

extern "C" {

int mce_induct(const int64_t* x, int64_t B, int64_t T, int locks, int longest, const int64_t* bucket,
               int64_t nbucket, int64_t c1_none, int64_t* cand, uint8_t* on, int64_t* src, int64_t* bk, int64_t* c1,
               void* stream) {
  if (B < 0 || T < 0 || T > IND_TMAX || locks < 1 || locks > 3) return MCE_INDUCT_EINVAL;
  if (bucket != nullptr && nbucket <= 0) return MCE_INDUCT_EINVAL;
  if (B == 0 || T == 0) return MCE_INDUCT_OK;
  if (x == nullptr || B > INT32_MAX) return MCE_INDUCT_EINVAL;
  int Tp = 1;
  while (Tp < T) Tp <<= 1;
  // a wave per chunk and lock, as far as a workgroup goes
  const int nt = (int)std::min<int64_t>(IND_THREADS_MAX, (T + 63) / 64 * 64 * locks);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (T <= IND_SMALL)
    hipLaunchKernelGGL((k_induct<IND_SMALL, 3, true>), dim3((unsigned)B), dim3(nt), 0, st, x, (int)T, Tp, locks,
                       longest ? 1 : 0, bucket, nbucket, c1_none, cand, on, src, bk, c1);
  else
    hipLaunchKernelGGL((k_induct<IND_TMAX, 1, false>), dim3((unsigned)B), dim3(nt), 0, st, x, (int)T, Tp, locks,
                       longest ? 1 : 0, bucket, nbucket, c1_none, cand, on, src, bk, c1);
  return launched();
}

int mce_induct_max_len(void) { return IND_TMAX; }

size_t mce_induct_ws_bytes(int64_t B, int64_t T, int locks) {
  if (B <= 0 || T <= IND_TMAX || T > IND_LONG_MAX || locks < 1 || locks > 3) return 0;
  const size_t per = long_layout(T, locks).bytes;
  if ((uint64_t)B > SIZE_MAX / per) return 0;
  return (size_t)B * per;
}

int mce_induct_ws(const int64_t* x, int64_t B, int64_t T, int locks, int longest, const int64_t* bucket,
                  int64_t nbucket, int64_t c1_none, int64_t* cand, uint8_t* on, int64_t* src, int64_t* bk, int64_t* c1,
                  void* ws, size_t ws_bytes, void* stream) {
  if (B < 0 || T < 0 || T > IND_LONG_MAX || locks < 1 || locks > 3) return MCE_INDUCT_EINVAL;
  if (T <= IND_TMAX)
    return mce_induct(x, B, T, locks, longest, bucket, nbucket, c1_none, cand, on, src, bk, c1, stream);
  if (bucket != nullptr && nbucket <= 0) return MCE_INDUCT_EINVAL;
  if (B == 0) return MCE_INDUCT_OK;
  if (x == nullptr || B > INT32_MAX) return MCE_INDUCT_EINVAL;
  const size_t need = mce_induct_ws_bytes(B, T, locks);
  if (need == 0 || ws == nullptr || ws_bytes < need || (reinterpret_cast<uintptr_t>(ws) & 255))
    return MCE_INDUCT_EINVAL;
  const LongLayout l = long_layout(T, locks);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  int bits = 1;
  while ((uint32_t(1) << bits) < l.slots) ++bits;
  const bool small = T < (int64_t)NONE16;  // 16-bit positions
  const uint32_t cap = LINK_BYTES / (small ? 2 : 4), parts = (l.slots + cap - 1) / cap;
  const uint32_t entries = l.slots * (uint32_t)locks;
  const unsigned groups = (unsigned)((T + 255) / 256);
  const int64_t batch = 32768;  // texts per launch (the grid's second dimension)
  int rc;
  for (int64_t b0 = 0; b0 < B; b0 += batch) {
    const unsigned nb = (unsigned)std::min(batch, B - b0);
    char* w = static_cast<char*>(ws) + (size_t)b0 * l.bytes;
    hipLaunchKernelGGL(k_ind_clear, dim3(std::min(1024u, (entries + 1023) / 1024), nb), dim3(256), 0, st, w, l.bytes,
                       entries);
    if ((rc = launched())) return rc;
    const dim3 igrid(groups * (unsigned)locks, nb), egrid(std::min(4096u, groups), nb);
    const int64_t* xb = x + b0 * T;
    const int tt = (int)T, lo = longest ? 1 : 0;
    if (T <= PACK_T) {
      hipLaunchKernelGGL((k_ind_insert<true>), igrid, dim3(256), 0, st, xb, tt, locks, bits, w, l.bytes, l.info,
                         l.slots);
      if ((rc = launched())) return rc;
      hipLaunchKernelGGL(k_ind_walk, dim3((unsigned)locks, nb), dim3(LINK_THREADS), 0, st, tt, w, l.bytes, l.info,
                         l.slots);
      if ((rc = launched())) return rc;
      hipLaunchKernelGGL((k_ind_emit<true>), egrid, dim3(256), 0, st, xb, tt, locks, lo, bucket, nbucket, c1_none, w,
                         l.bytes, cand, on, src, bk, c1, b0, l.info, l.slots);
      if ((rc = launched())) return rc;
      continue;
    }
    hipLaunchKernelGGL((k_ind_insert<false>), igrid, dim3(256), 0, st, xb, tt, locks, bits, w, l.bytes, l.info,
                       l.slots);
    if ((rc = launched())) return rc;
    if (small)
      hipLaunchKernelGGL((k_ind_link<uint16_t>), dim3(parts * (unsigned)locks, nb), dim3(LINK_THREADS), 0, st, tt,
                         locks, w, l.bytes, l.info);
    else
      hipLaunchKernelGGL((k_ind_link<uint32_t>), dim3(parts * (unsigned)locks, nb), dim3(LINK_THREADS), 0, st, tt,
                         locks, w, l.bytes, l.info);
    if ((rc = launched())) return rc;
    hipLaunchKernelGGL((k_ind_emit<false>), egrid, dim3(256), 0, st, xb, tt, locks, lo, bucket, nbucket, c1_none, w,
                       l.bytes, cand, on, src, bk, c1, b0, l.info, l.slots);
    if ((rc = launched())) return rc;
  }
  return MCE_INDUCT_OK;
}

}  // extern "C"
