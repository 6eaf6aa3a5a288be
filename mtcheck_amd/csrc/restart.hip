// restart.hip -- rebuild checkpoint k from the diff chain ref_id..k.
//
// Semantics: src/tree_approach.cpp:712-1128.  A chunk takes its bytes from the
// newest diff of the chain that covers its leaf, either from that diff's own
// first-occurrence data or, for a shifted-duplicate entry (node, prev) with source
// checkpoint s, from the first-occurrence region of diff s that contains prev.
// Instead of the reference's per-diff pass over every chunk, the chain is resolved
// once into a per-chunk (diff, data slot) cover array, then one scatter copy runs.
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>

#include "internal.hpp"

namespace mtc {

constexpr uint32_t kRThreads = 256;
constexpr uint64_t kNoKey = ~0ull;
// Cover entries: the covering diff's chain position + 1 above the byte address of the
// chunk's bytes; zero: not covered.  Diffs are covered in any order, the newest wins
// by atomic max.  Chains of more than kCoverPos diffs take several passes.
constexpr uint32_t kAddrBits = 47;
constexpr uint64_t kAddrMask = (1ull << kAddrBits) - 1;
constexpr uint32_t kCoverPos = (1u << (64 - kAddrBits)) - 1;

static uint32_t rgrid(uint64_t items, uint32_t cap = 1u << 20) {
  uint64_t g = (items + kRThreads - 1) / kRThreads;
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(g, cap));
}

__device__ __forceinline__ uint32_t ld32(const uint8_t* p) {
  return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// Hash set (diff position, root node) -> region index, for prev lookups.
__device__ __forceinline__ uint64_t rs_home(uint64_t key, uint64_t mask) {
  key ^= key >> 33;
  key *= 0xff51afd7ed558ccdULL;
  key ^= key >> 33;
  return key & mask;
}

__device__ __forceinline__ uint32_t rs_find(const uint64_t* keys, const uint32_t* vals, uint64_t mask, uint64_t key) {
  uint64_t s = rs_home(key, mask);
  for (uint64_t probes = 0; probes <= mask; probes++) {
    const uint64_t k = keys[s];
    if (k == key) return vals[s];
    if (k == kNoKey) return ~0u;
    s = (s + 1) & mask;
  }
  return ~0u;
}

// The tables of a chain of L diffs, by chain position p (one array of 64-bit words;
// prefix arrays have L + 1 entries).
enum : uint32_t { M_FIRST, M_DATA, M_CHUNKS, M_SHIFT, M_TABLE, M_PS, M_CUM, M_REGION, M_CBASE, M_SBASE, M_ARRAYS };
__host__ __device__ constexpr uint64_t meta_words(uint64_t L) { return M_ARRAYS * L + 3; }

struct Chain {
  uint32_t L;
  uint32_t n, C;
  uint32_t ref;
  uint32_t idb;      // added to every stored id (0 for tree diffs, whose ids are node ids; n - 1
                     // for basic diffs, whose ids are chunk indices: leaf n - 1 + c holds chunk c)
  Geo g;
  const uint64_t* meta;
  uint32_t* region;  // per root of every diff, then one end marker: sizes, then their running totals
  uint32_t* cum;     // per diff: inclusive running count of its shifted entries by checkpoint id
  uint64_t* keys;    // the (position, root) set
  uint32_t* vals;
  uint64_t mask;
  uint64_t* cover;
  uint32_t* err;
  volatile uint32_t* err_host;  // pinned copy (may be null): an error's bits, one word each

  __device__ const uint64_t* first() const { return meta; }                        // address of the F roots
  __device__ const uint64_t* data() const { return meta + (uint64_t)M_DATA * L; }  // address of the data section
  __device__ const uint64_t* chunks() const { return meta + (uint64_t)M_CHUNKS * L; }  // whole chunks it can hold
  __device__ const uint64_t* shift() const { return meta + (uint64_t)M_SHIFT * L; }    // address of the S pairs
  __device__ const uint64_t* table() const { return meta + (uint64_t)M_TABLE * L; }    // address of the P table
  __device__ const uint64_t* ps() const { return meta + (uint64_t)M_PS * L; }          // P << 32 | S
  __device__ const uint64_t* cum_off() const { return meta + (uint64_t)M_CUM * L; }
  __device__ const uint64_t* region_base() const { return meta + (uint64_t)M_REGION * L; }     // L + 1
  __device__ const uint64_t* chunk_base() const { return meta + (uint64_t)M_CBASE * L + 1; }   // L + 1: running chunks()
  __device__ const uint64_t* shift_base() const { return meta + (uint64_t)M_SBASE * L + 2; }   // L + 1: running S

  __device__ void fail(uint32_t bit) const {
    atomicOr(err, bit);
    if (err_host) err_host[bit == ERR_TABLE_FULL ? 1 : 0] = bit;
  }
  __device__ uint32_t roots(uint32_t p) const { return (uint32_t)(region_base()[p + 1] - region_base()[p] - 1); }
};

// The position whose share of a prefix array (L + 1 entries) holds i.
__device__ __forceinline__ uint32_t owner(const uint64_t* base, uint32_t lo, uint32_t hi, uint64_t i) {
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (base[mid] <= i) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Everything a restart reads before it is written starts here: the chain's tables
// (from `src`, host-visible memory), the set, the cover array and the counts.
__global__ __launch_bounds__(kRThreads) void k_r_init(const uint64_t* src, uint64_t* meta, uint64_t meta_n, uint64_t* keys,
                                                      uint64_t keys_n, uint64_t* cover, uint64_t cover_n, uint32_t* cum,
                                                      uint64_t cum_n, uint32_t* err) {
  const uint64_t t = (uint64_t)blockIdx.x * kRThreads + threadIdx.x, s = (uint64_t)gridDim.x * kRThreads;
  if (t == 0) *err = 0;
  if (src)
    for (uint64_t i = t; i < meta_n; i += s) meta[i] = src[i];
  for (uint64_t i = t; i < keys_n; i += s) keys[i] = kNoKey;
  for (uint64_t i = t; i < cum_n; i += s) cum[i] = 0;
  ulonglong2* c2 = reinterpret_cast<ulonglong2*>(cover);
  for (uint64_t i = t; i < cover_n / 2; i += s) c2[i] = ulonglong2{0, 0};
  if (t == 0 && (cover_n & 1)) cover[cover_n - 1] = 0;
}

// One block: the inclusive running count, by checkpoint id ref..ref+p, of the shifted
// entries of diff p (its prior-checkpoint table, src/tree_approach.cpp:872-883),
// checked against the diff's S.
__device__ void cum_block(const Chain& c, uint32_t p) {
  __shared__ uint32_t ws[kRThreads / 64];
  const uint32_t P = (uint32_t)(c.ps()[p] >> 32), S = (uint32_t)c.ps()[p];
  const uint8_t* tab = reinterpret_cast<const uint8_t*>(c.table()[p]);
  uint32_t* cnt = c.cum + c.cum_off()[p];
  for (uint32_t i = threadIdx.x; i < P; i += kRThreads) {
    const uint32_t id = ld32(tab + 8ull * i), m = ld32(tab + 8ull * i + 4);
    if (id < c.ref || id - c.ref > p) c.fail(ERR_CORRUPT);
    else atomicAdd(&cnt[id - c.ref], m);
  }
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t carry = 0;
  for (uint64_t b = 0; b <= p; b += kRThreads) {
    const uint64_t i = b + threadIdx.x;
    uint32_t x = i <= p ? __hip_atomic_load(&cnt[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(x, o);
      if (lane >= (uint32_t)o) x += y;
    }
    if (lane == 63) ws[w] = x;
    __syncthreads();
    uint32_t pre = carry;
    for (uint32_t k = 0; k < kRThreads / 64; k++) {
      if (k < w) pre += ws[k];
      carry += ws[k];
    }
    if (i <= p) cnt[i] = pre + x;
    __syncthreads();
  }
  if (threadIdx.x == 0 && carry != S) c.fail(ERR_CORRUPT);
}

// Every diff's first-occurrence roots in one launch: the region size of each, and its
// entry in the (diff position, root node) set that resolves shifted entries' sources.
// The last L blocks build the running counts of shifted entries.
__global__ __launch_bounds__(kRThreads) void k_r_roots(Chain c, uint32_t nblk) {
  if (blockIdx.x >= nblk) {
    cum_block(c, blockIdx.x - nblk);
    return;
  }
  const uint64_t* base = c.region_base();
  const uint64_t words = base[c.L];
  for (uint64_t i = (uint64_t)blockIdx.x * kRThreads + threadIdx.x; i < words; i += (uint64_t)nblk * kRThreads) {
    const uint32_t p = owner(base, 0, c.L, i);
    if (i + 1 == base[p + 1]) {  // the diff's end marker
      c.region[i] = 0;
      continue;
    }
    const uint32_t r = (uint32_t)(i - base[p]);
    const uint64_t node = (uint64_t)ld32(reinterpret_cast<const uint8_t*>(c.first()[p]) + 4ull * r) + c.idb;
    if (node >= 2ull * c.g.n - 1) {
      c.fail(ERR_CORRUPT);
      c.region[i] = 0;
      continue;
    }
    c.region[i] = leaf_count(c.g, (uint32_t)node);
    const uint64_t key = ((uint64_t)p << 32) | node;
    uint64_t s = rs_home(key, c.mask);
    bool placed = false;
    for (uint64_t probes = 0; probes <= c.mask; probes++) {
      const uint64_t old = atomicCAS((unsigned long long*)&c.keys[s], (unsigned long long)kNoKey, (unsigned long long)key);
      if (old == kNoKey) {
        c.vals[s] = r;
        placed = true;
        break;
      }
      if (old == key) {  // the same root twice in one diff
        c.fail(ERR_CORRUPT);
        placed = true;
        break;
      }
      s = (s + 1) & c.mask;
    }
    if (!placed) c.fail(ERR_TABLE_FULL);
  }
}

// One diff's regions: slots of its data section -> chunks, the last region found being
// kept for the next slot (a baseline often has one region for the whole buffer).
struct Regions {
  const uint32_t* reg;
  const uint8_t* roots;
  uint32_t F, g0, total;
  uint32_t from = 1, to = 0;  // slots of the region found last
  uint32_t run0 = 0, run1 = 0, cnt0 = 0;  // its chunks: cnt0 from run0 on, then from run1 on

  __device__ Regions(const Chain& c, uint32_t p)
      : reg(c.region + c.region_base()[p]), roots(reinterpret_cast<const uint8_t*>(c.first()[p])), F(c.roots(p)),
        g0(reg[0]), total(reg[F] - g0) {
    if (total > c.chunks()[p]) {  // the data section is shorter than its regions
      c.fail(ERR_CORRUPT);
      total = 0;
    }
  }
  __device__ uint32_t chunk(const Chain& c, uint32_t j) {  // j < total
    if (j < from || j >= to) {
      uint32_t lo = 0, hi = F;
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (reg[mid] - g0 <= j) lo = mid;
        else hi = mid;
      }
      from = reg[lo] - g0;
      to = reg[lo + 1] - g0;
      uint32_t st[2], ct[2];
      const int r = leaf_runs(c.g, ld32(roots + 4ull * lo) + c.idb, st, ct);
      run0 = st[0];
      run1 = r == 2 ? st[1] : 0u;
      cnt0 = ct[0];
    }
    const uint32_t k = j - from;
    return k < cnt0 ? run0 + k : run1 + (k - cnt0);
  }
};

// Diffs are covered in one of two ways.  Most share a launch, in which the newest entry of
// a chunk stands by atomic max: that needs no order.  Plain stores run at three times an
// atomic's rate, but need a launch of their own, after the earlier diffs' and before the
// later ones'.  So are covered the first-occurrence chunks of the pass's oldest diff, which
// holds nearly the whole buffer when it is the baseline, and any diff's if it stores
// kCoverPlain chunks; its shifted entries too if there are as many.  1 GiB in 48-byte chunks
// (22 million), all but the oldest diff by atomics / so: a chain of three whole rewrites 750
// / 510 us, of half constant buffers (a shifted entry a chunk) 1040 / 880; 256 MiB in
// 64-byte chunks (2^22) rewritten 212 / 177, in 96-byte chunks no difference.  (Where one of
// many shifted entries spans half the buffer, which one wavefront walks, less runs beside
// it: 21.1 / 21.6 ms.)
constexpr uint64_t kCoverPlain = 1u << 22;

// First-occurrence chunks of diff p of the pass that starts at lo, by plain stores.
__global__ __launch_bounds__(kRThreads) void k_r_cover_base(Chain c, uint32_t lo, uint32_t p) {
  if (*c.err) return;
  Regions d(c, p);
  const uint64_t top = (uint64_t)(p - lo + 1) << kAddrBits, data = c.data()[p];
  for (uint64_t j = (uint64_t)blockIdx.x * kRThreads + threadIdx.x; j < d.total; j += (uint64_t)gridDim.x * kRThreads)
    c.cover[d.chunk(c, (uint32_t)j)] = top | (data + j * c.C);
}

// First-occurrence chunks of diffs flo .. hi - 1 (nblk blocks) and shifted entries of diffs
// slo .. hi - 1 (the other blocks) of the pass that starts at lo.  Each leaf of a shifted
// entry's `node` takes the data slot of the matching leaf of `prev` inside the source diff's
// region (src/tree_approach.cpp:887-925, 1058-1118); a wavefront shares the leaves of its
// larger entries.  PLAIN: one diff's shifted entries, by plain stores.
constexpr uint32_t kShiftOwn = 4;  // most leaves a lane covers by itself
template <bool PLAIN>
__global__ __launch_bounds__(kRThreads) void k_r_cover_rest(Chain c, uint32_t lo, uint32_t flo, uint32_t slo, uint32_t hi,
                                                            uint32_t nblk) {
  if (*c.err) return;
  if (!PLAIN && blockIdx.x < nblk) {
    const uint64_t* base = c.chunk_base();
    const uint64_t end = base[hi];
    for (uint64_t j = base[flo] + (uint64_t)blockIdx.x * kRThreads + threadIdx.x; j < end; j += (uint64_t)nblk * kRThreads) {
      const uint32_t p = owner(base, flo, hi, j);
      const uint64_t slot = j - base[p];
      Regions d(c, p);
      if (slot >= d.total) continue;
      atomicMax((unsigned long long*)&c.cover[d.chunk(c, (uint32_t)slot)],
                (unsigned long long)(((uint64_t)(p - lo + 1) << kAddrBits) | (c.data()[p] + slot * c.C)));
    }
    return;
  }
  const uint64_t* base = c.shift_base();
  const uint64_t end = base[hi];
  const uint64_t nodes = 2ull * c.g.n - 1;
  const uint32_t lane = lane_id();
  const uint64_t stride = (uint64_t)(gridDim.x - nblk) * kRThreads;
  for (uint64_t w0 = base[slo] + (uint64_t)(blockIdx.x - nblk) * kRThreads + (threadIdx.x & ~63u); w0 < end; w0 += stride) {
    const uint64_t i = w0 + lane;
    uint32_t node = 0, prev = 0, root = 0, rbase = 0, spos = 0, cnt = 0, p = 0;
    bool ok = i < end;
    if (ok) {
      p = owner(base, slo, hi, i);
      const uint32_t e = (uint32_t)(i - base[p]);
      const uint8_t* sh = reinterpret_cast<const uint8_t*>(c.shift()[p]) + 8ull * e;
      node = ld32(sh);
      prev = ld32(sh + 4);
      ok = node < nodes && prev < nodes;
      if (ok) {
        const uint32_t* cum = c.cum + c.cum_off()[p];
        uint32_t l = 0, h = p + 1;  // smallest checkpoint whose running count exceeds e
        while (l < h) {
          const uint32_t mid = (l + h) >> 1;
          if (e < cum[mid]) h = mid;
          else l = mid + 1;
        }
        spos = l;  // chain position of the source checkpoint
        ok = l <= p;
      }
      uint32_t region = ~0u;
      if (ok) {
        for (uint32_t anc = prev;; anc = (anc - 1) >> 1) {
          region = rs_find(c.keys, c.vals, c.mask, ((uint64_t)spos << 32) | anc);
          if (region != ~0u || anc == 0) break;
        }
        ok = region != ~0u;
      }
      if (ok) {
        root = ld32(reinterpret_cast<const uint8_t*>(c.first()[spos]) + 4ull * region) + c.idb;
        const uint32_t* reg = c.region + c.region_base()[spos];
        rbase = reg[region] - reg[0];
        cnt = leaf_count(c.g, node);
        ok = cnt == leaf_count(c.g, prev);
      }
      if (!ok) {
        c.fail(ERR_CORRUPT);
        cnt = 0;
      }
    }
    auto cover_leaves = [&](uint32_t nd, uint32_t pv, uint32_t rt, uint32_t rb, uint32_t sp, uint32_t pos, uint32_t from,
                            uint32_t step, uint32_t count) {
      uint32_t rs[2], rc[2], ns[2], nc[2], ps[2], pc[2];
      const int rr = leaf_runs(c.g, rt, rs, rc);
      const int nr = leaf_runs(c.g, nd, ns, nc);
      const int pr = leaf_runs(c.g, pv, ps, pc);
      const uint64_t top = (uint64_t)(pos - lo + 1) << kAddrBits, data = c.data()[sp], cap = c.chunks()[sp];
      for (uint32_t j = from; j < count; j += step) {
        const uint64_t slot = (uint64_t)rb + run_rank(rr, rs, rc, run_at(pr, ps, pc, j));
        if (slot >= cap) {
          c.fail(ERR_CORRUPT);
          break;
        }
        uint64_t* at = &c.cover[run_at(nr, ns, nc, j)];
        const uint64_t v = top | (data + slot * c.C);
        if (PLAIN) *at = v;
        else atomicMax((unsigned long long*)at, (unsigned long long)v);
      }
    };
    if (cnt && cnt <= kShiftOwn) cover_leaves(node, prev, root, rbase, spos, p, 0, 1, cnt);
    uint64_t big = __ballot(cnt > kShiftOwn);
    while (big) {
      const int l = __ffsll((long long)big) - 1;
      big &= big - 1;
      cover_leaves(__shfl(node, l), __shfl(prev, l), __shfl(root, l), __shfl(rbase, l), __shfl(spos, l), __shfl(p, l), lane,
                   64, __shfl(cnt, l));
    }
  }
}

// Between two passes over a long chain: the cover keeps its addresses below every
// position of the next pass.
__global__ void k_r_cover_age(uint64_t* cover, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * kRThreads + threadIdx.x; i < n; i += (uint64_t)gridDim.x * kRThreads)
    if (cover[i]) cover[i] &= kAddrMask;
}

// One scatter copy: out[chunk] = the bytes its cover names.  No loop: a block copies
// 16 KiB with four 16-byte loads a thread before its stores (a wait for a load also
// waits for the stores before it).  The card's copy rate bounds it: 8 GiB in 3.04 ms
// (5.65 TB/s read and written), 3.53 ms as 8192 looping blocks.  C a power of
// two of at least 16, 16-byte aligned out, 4-byte aligned data sections.
constexpr uint32_t kCopyUnits = 4;
__global__ __launch_bounds__(kRThreads) void k_r_copy(Chain c, uint64_t datalen, uint32_t ulog, uint8_t* out) {
  if (*c.err) return;
  const uint64_t blk = wide_block(), units = datalen / 16, u0 = blk * (kCopyUnits * kRThreads) + threadIdx.x;
  uint64_t e[kCopyUnits];
#pragma unroll
  for (uint32_t i = 0; i < kCopyUnits; i++) {
    const uint64_t u = u0 + i * kRThreads;
    e[i] = u < units ? c.cover[u >> ulog] : 1;
    if (!e[i]) c.fail(ERR_CORRUPT);
  }
  uint4 v[kCopyUnits];
#pragma unroll
  for (uint32_t i = 0; i < kCopyUnits; i++) {
    const uint64_t u = u0 + i * kRThreads;
    if (u < units && e[i])
      v[i] = ld_stream16_a4(reinterpret_cast<const uint8_t*>(e[i] & kAddrMask) + 16 * (u & ((1u << ulog) - 1)));
  }
#pragma unroll
  for (uint32_t i = 0; i < kCopyUnits; i++) {
    const uint64_t u = u0 + i * kRThreads;
    if (u < units && e[i]) st_stream16(out + 16 * u, v[i]);
  }
  if (blk == 0 && threadIdx.x < (datalen & 15)) {  // the short last chunk's last bytes
    const uint64_t o = 16 * units + threadIdx.x, ce = c.cover[o / c.C];
    if (ce) out[o] = reinterpret_cast<const uint8_t*>(ce & kAddrMask)[o % c.C];
    else c.fail(ERR_CORRUPT);
  }
}

// The same for any chunk size and alignment, in whole words of the output (mis: where it
// starts in one): W bytes a thread.  W = 16, chunks of at least 16 bytes: words that lie in
// one chunk, or in two that are neighbours in the diff too, are cut out of the aligned words
// that hold them, others gathered byte by byte.  W = 4, smaller chunks: a word a thread, so
// that neighbours store side by side (64 MiB in 4-byte chunks, three versions, 1098 us; with
// 16 bytes a thread, stored one by one, 1600, as 256-chunk tiles of bytes 1190).
template <uint32_t W>
__global__ __launch_bounds__(kRThreads) void k_r_copy_any(Chain c, uint64_t datalen, uint8_t* out) {
  if (*c.err) return;
  const uint32_t mis = (uint32_t)(uintptr_t)out & 3;
  const uint64_t t = wide_block() * kRThreads + threadIdx.x;
  auto chunk_of = [&](uint64_t o) { return o >> 32 ? o / c.C : (uint64_t)((uint32_t)o / c.C); };
  auto word = [&](uint64_t j) {
    const uint64_t o = 4 * j > mis ? 4 * j - mis : 0u, end = min<uint64_t>(4 * j + 4 - mis, datalen);
    if (o >= end) return;
    uint64_t k = chunk_of(o);
    uint32_t w = (uint32_t)(o - k * c.C), x = 0;
    bool ok = true;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
      if (o + i >= end) continue;
      const uint64_t e = c.cover[k];
      if (e) x |= (uint32_t) reinterpret_cast<const uint8_t*>(e & kAddrMask)[w] << (8 * i);
      else ok = false;
      if (++w == c.C) {
        w = 0;
        k++;
      }
    }
    if (!ok) c.fail(ERR_CORRUPT);
    else if (end - o == 4) *reinterpret_cast<uint32_t*>(out + o) = x;
    else
      for (uint32_t i = 0; o + i < end; i++) out[o + i] = (uint8_t)(x >> (8 * i));
  };
  if (W == 4) {
    word(t);
    return;
  }
  if (16 * t >= datalen + mis) return;
  if (t || !mis) {
    const uint64_t o = 16 * t - mis, k = chunk_of(o);
    const uint32_t w = (uint32_t)(o - k * c.C);
    const uint64_t e = c.cover[k];
    if (o + 16 <= datalen && e && ((uint64_t)w + 16 <= c.C || (c.cover[k + 1] & kAddrMask) == (e & kAddrMask) + c.C)) {
      const uint64_t src = (e & kAddrMask) + w;
      const uint32_t sh = (uint32_t)src & 3;
      const uint32_t* q = reinterpret_cast<const uint32_t*>(src - sh);
      const uint4 v = ld_stream16_a4(q);
      const uint32_t x = sh ? q[4] : 0u;
      st_stream16_a4(out + o, uint4{__builtin_amdgcn_alignbyte(v.y, v.x, sh), __builtin_amdgcn_alignbyte(v.z, v.y, sh),
                                    __builtin_amdgcn_alignbyte(v.w, v.z, sh), __builtin_amdgcn_alignbyte(x, v.w, sh)});
      return;
    }
  }
#pragma unroll 1
  for (uint32_t i = 0; i < 4; i++) word(4 * t + i);
}

// The headers of the chain that ends in diff k (a device chain's), read where they lie:
// hdr[0] is k's, hdr[1 + i] that of its i-th diff (ref_id + i).  ptrs and sizes (from
// diff `first` on; entries below the chain are not looked at) and hdr are pinned host
// memory: one launch and one synchronisation for the whole chain.  A missing or short
// diff leaves its header as it is.
__global__ __launch_bounds__(kRThreads) void k_r_headers(const uint64_t* ptrs, const uint64_t* sizes, uint32_t first,
                                                         uint32_t k, uint32_t* hdr) {
  const uint32_t ref = ld32(reinterpret_cast<const uint8_t*>(ptrs[k - first]));
  const uint32_t L = ref >= first && ref <= k ? k - ref + 1 : 0u;
  for (uint64_t i = (uint64_t)blockIdx.x * kRThreads + threadIdx.x; i < 8ull * (L + 1ull); i += (uint64_t)gridDim.x * kRThreads) {
    const uint64_t h = i / 8, w = i % 8;
    const uint64_t idx = (h == 0 ? k : ref + (h - 1)) - first;
    if (ptrs[idx] && sizes[idx] >= sizeof(mtc_header)) hdr[i] = ld32(reinterpret_cast<const uint8_t*>(ptrs[idx]) + 4 * w);
  }
}

struct RestartScratch {
  hipEvent_t ev[3] = {nullptr, nullptr, nullptr};  // start, chain uploaded, done
  Workspace ws;
  DevBuf<uint32_t> err, region, set_vals, cum;
  DevBuf<uint64_t> set_keys, cover, meta;
  uint8_t* stage = nullptr;  // pinned: diff addresses and sizes, headers, per-position tables, error words
  uint64_t stage_cap = 0;
  bool busy = false;  // a restart that did not reach its end may still use the scratch
};

// Pinned staging that grows by at least half (no restart is using it).
static void pinned_reserve(uint8_t*& p, uint64_t& cap, uint64_t want) {
  if (want <= cap) return;
  const uint64_t c = std::max<uint64_t>({want, cap + cap / 2, 4096});
  if (p) (void)hipHostFree(p);
  p = nullptr;
  cap = 0;
  MTC_HIP(hipHostMalloc((void**)&p, c));
  cap = c;
}

static std::mutex& scratch_mutex() {
  static std::mutex m;
  return m;
}

// Scratch of one device, kept until the process ends.
static RestartScratch& scratch_for(int dev) {
  static std::map<int, RestartScratch*> all;
  RestartScratch*& r = all[dev];
  if (!r) r = new RestartScratch();
  return *r;
}

// The calling thread's last restart: upload of a host chain, and the whole restart
// (restart_timers of src/tree_approach.cpp:1792-1793).
static thread_local float g_restart_ms[2] = {0, 0};

void last_restart_times(float* upload_ms, float* total_ms) {
  if (upload_ms) *upload_ms = g_restart_ms[0];
  if (total_ms) *total_ms = g_restart_ms[1];
}

static void throw_err(uint32_t e) {
  if (e & ERR_TABLE_FULL) throw Status{MTC_ERR_OUT_OF_MEMORY, "restart root set overflow"};
  if (e) throw Status{MTC_ERR_CORRUPT_DIFF, "diff chain is inconsistent (err bits " + std::to_string(e) + ")"};
}

static void check_err(uint32_t* err_d, hipStream_t st) {
  uint32_t e = 0;
  MTC_HIP(hipMemcpyAsync(&e, err_d, sizeof(uint32_t), hipMemcpyDeviceToHost, st));
  MTC_HIP(hipStreamSynchronize(st));
  throw_err(e);
}

// The header of the requested checkpoint.
static void check_last(const mtc_header& hk, uint32_t k, uint64_t out_len) {
  if (hk.chkpt_id != k || hk.ref_id > k || hk.chunk_size == 0 || hk.datalen == 0)
    throw Status{MTC_ERR_CORRUPT_DIFF, "bad header of the requested diff"};
  if (out_len < hk.datalen) throw Status{MTC_ERR_BUFFER_TOO_SMALL, "output shorter than datalen"};
  if ((hk.datalen + hk.chunk_size - 1) / hk.chunk_size > (1ull << 31)) throw Status{MTC_ERR_CORRUPT_DIFF, "too many chunks"};
}

// Totals of a chain, known from its headers and sizes.
struct ChainSums {
  uint64_t F = 0, S = 0, chunks = 0, cum = 0;
  bool words = true;  // every data section is 4-byte aligned
};

// Fills the tables of a chain (meta_words(L) words) from its headers, device
// addresses and sizes; every diff is checked against the last one's header.
static ChainSums fill_meta(uint64_t* m, const mtc_header* hs, const uint64_t* addr, const uint64_t* sizes, uint32_t L,
                           const mtc_header& hk, bool basic) {
  ChainSums t;
  uint64_t* region = m + (uint64_t)M_REGION * L;
  uint64_t* cbase = m + (uint64_t)M_CBASE * L + 1;
  uint64_t* sbase = m + (uint64_t)M_SBASE * L + 2;
  for (uint32_t p = 0; p < L; p++) {
    const uint32_t idx = hk.ref_id + p;
    const mtc_header& h = hs[p];
    if (h.chkpt_id != idx || h.ref_id != hk.ref_id || h.datalen != hk.datalen || h.chunk_size != hk.chunk_size)
      throw Status{MTC_ERR_CORRUPT_DIFF, "diff " + std::to_string(idx) + " does not belong to the chain"};
    if (basic && (h.num_prior_chkpts || h.num_shift_dupl))
      throw Status{MTC_ERR_CORRUPT_DIFF, "diff " + std::to_string(idx) + " is not a basic diff"};
    const uint64_t off_table = 32 + 4ull * h.num_first_ocur, off_shift = off_table + 8ull * h.num_prior_chkpts;
    const uint64_t off_data = off_shift + 8ull * h.num_shift_dupl;
    if (off_data > sizes[p]) throw Status{MTC_ERR_CORRUPT_DIFF, "diff shorter than its metadata"};
    const uint64_t chunks = (sizes[p] - off_data) / hk.chunk_size;
    if (h.num_first_ocur && !chunks) throw Status{MTC_ERR_CORRUPT_DIFF, "data section shorter than its regions"};
    if ((addr[p] + sizes[p]) >> kAddrBits) throw Status{MTC_ERR_INVALID_ARG, "diff address above 2^47"};
    m[(uint64_t)M_FIRST * L + p] = addr[p] + 32;
    m[(uint64_t)M_DATA * L + p] = addr[p] + off_data;
    m[(uint64_t)M_CHUNKS * L + p] = chunks;
    m[(uint64_t)M_SHIFT * L + p] = addr[p] + off_shift;
    m[(uint64_t)M_TABLE * L + p] = addr[p] + off_table;
    m[(uint64_t)M_PS * L + p] = ((uint64_t)h.num_prior_chkpts << 32) | h.num_shift_dupl;
    m[(uint64_t)M_CUM * L + p] = t.cum;
    region[p] = t.F + p;
    cbase[p] = t.chunks;
    sbase[p] = t.S;
    t.F += h.num_first_ocur;
    t.S += h.num_shift_dupl;
    t.chunks += chunks;
    t.cum += p + 1;
    t.words = t.words && (addr[p] + off_data) % 4 == 0;
  }
  region[L] = t.F + L;
  cbase[L] = t.chunks;
  sbase[L] = t.S;
  return t;
}

static uint64_t set_slots(uint64_t roots) {
  uint64_t cap = 16;
  while (cap < 2 * roots) cap <<= 1;
  return cap;
}

// The restart's launches, the chain's tables being in c.meta's source: the set and
// counts, the region offsets (scan), the cover and the copy.  They come in a fixed
// number whatever the chain's length: with one set of them per diff, ten diffs took 45
// launches, each waiting for its own chain of lookups (64 MiB of 128-byte chunks,
// restart and 4 KiB digests: 683 us, 194 us so).  Every later kernel stops at an error of an earlier one.
template <class Scan>
static void launch_restart(const Chain& c, const uint64_t* meta_src, const uint64_t* m, const ChainSums& t, uint64_t datalen,
                           uint8_t* out, hipStream_t st, Scan scan) {
  const uint32_t L = c.L, n = c.n;
  k_r_init<<<rgrid(std::max<uint64_t>({n / 2, t.cum, c.mask + 1, meta_words(L)})), kRThreads, 0, st>>>(
      meta_src, const_cast<uint64_t*>(c.meta), meta_words(L), c.keys, c.mask + 1, c.cover, n, c.cum, t.cum, c.err);
  const uint32_t rblk = rgrid(t.F + L);
  k_r_roots<<<rblk + L, kRThreads, 0, st>>>(c, rblk);
  MTC_HIP(hipGetLastError());
  scan();
  const uint64_t* cbase = m + (uint64_t)M_CBASE * L + 1;
  const uint64_t* sbase = m + (uint64_t)M_SBASE * L + 2;
  for (uint64_t lo = 0; lo < L; lo += kCoverPos) {
    const uint32_t hi = (uint32_t)std::min<uint64_t>(L, lo + kCoverPos);
    if (lo) k_r_cover_age<<<rgrid(n), kRThreads, 0, st>>>(c.cover, n);
    auto blocks = [](uint64_t items) { return items ? rgrid(items) : 0u; };
    uint32_t flo = (uint32_t)lo, slo = flo;  // the first diffs whose chunks, and whose shifted entries, are not covered yet
    auto together = [&](uint32_t end) {      // all before end
      const uint32_t fblk = blocks(cbase[end] - cbase[flo]), sblk = blocks(sbase[end] - sbase[slo]);
      if (fblk + sblk) k_r_cover_rest<false><<<fblk + sblk, kRThreads, 0, st>>>(c, (uint32_t)lo, flo, slo, end, fblk);
      flo = slo = end;
    };
    for (uint32_t p = flo; p < hi; p++) {
      const uint64_t first = cbase[p + 1] - cbase[p], shifted = sbase[p + 1] - sbase[p];
      const bool f = p == lo || first >= kCoverPlain, s = shifted >= kCoverPlain;
      if (!f && !s) continue;
      together(p);
      if (f) k_r_cover_base<<<rgrid(first, 4096), kRThreads, 0, st>>>(c, (uint32_t)lo, flo++);
      if (s) k_r_cover_rest<true><<<rgrid(shifted), kRThreads, 0, st>>>(c, (uint32_t)lo, p, slo++, p + 1, 0);
    }
    together(hi);
    MTC_HIP(hipGetLastError());
  }
  const uint32_t C = c.C;
  if (C >= 16 && (C & (C - 1)) == 0 && (uintptr_t)out % 16 == 0 && t.words)
    k_r_copy<<<wide_grid((datalen / 16 + kCopyUnits * kRThreads - 1) / (kCopyUnits * kRThreads)), kRThreads, 0, st>>>(
        c, datalen, (uint32_t)__builtin_ctz(C) - 4, out);
  else if (const uint64_t end = datalen + ((uintptr_t)out & 3); C < 16)
    k_r_copy_any<4><<<wide_grid((end + 4 * kRThreads - 1) / (4 * kRThreads)), kRThreads, 0, st>>>(c, datalen, out);
  else
    k_r_copy_any<16><<<wide_grid((end + 16 * kRThreads - 1) / (16 * kRThreads)), kRThreads, 0, st>>>(c, datalen, out);
  MTC_HIP(hipGetLastError());
}

// Device chains of which this many diffs come before the restarted one or fewer have
// their headers read in one launch (the addresses of all of them are staged).
constexpr uint32_t kHeadersAtOnce = 4096;

void restart_impl(const void* const* diffs, const uint64_t* sizes, uint32_t count, uint32_t k, bool on_device,
                  uint8_t* out, uint64_t out_len, hipStream_t st, bool basic) {
  if (!diffs || !sizes || k >= count || !diffs[k]) throw Status{MTC_ERR_INVALID_ARG, "bad diff chain arguments"};
  // Scratch buffers are kept per device between restarts (grow-only); one restart
  // at a time uses them.
  int dev = 0;
  MTC_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> guard(scratch_mutex());
  RestartScratch& rs = scratch_for(dev);
  g_restart_ms[0] = g_restart_ms[1] = 0;
  if (rs.busy) MTC_HIP(hipDeviceSynchronize());
  rs.busy = false;
  if (!rs.ev[0])
    for (auto& e : rs.ev) MTC_HIP(hipEventCreate(&e));
  MTC_HIP(hipEventRecord(rs.ev[0], st));
  auto present = [&](uint64_t idx) {
    if (!diffs[idx] || sizes[idx] < sizeof(mtc_header)) throw Status{MTC_ERR_CORRUPT_DIFF, "missing or short diff"};
  };
  present(k);
  mtc_header hk{};
  std::vector<mtc_header> hs;
  if (!on_device) {
    std::memcpy(&hk, diffs[k], sizeof(hk));
  } else if (k < kHeadersAtOnce) {
    pinned_reserve(rs.stage, rs.stage_cap, 16ull * (k + 1) + sizeof(mtc_header) * (k + 2ull));
    uint64_t* ptrs = reinterpret_cast<uint64_t*>(rs.stage);
    for (uint32_t i = 0; i <= k; i++) ptrs[i] = reinterpret_cast<uint64_t>(diffs[i]);
    std::memcpy(ptrs + (k + 1), sizes, 8ull * (k + 1));
    mtc_header* hdr = reinterpret_cast<mtc_header*>(ptrs + 2ull * (k + 1));
    rs.busy = true;
    k_r_headers<<<rgrid(8ull * (k + 2), 64), kRThreads, 0, st>>>(ptrs, ptrs + (k + 1), 0, k, reinterpret_cast<uint32_t*>(hdr));
    MTC_HIP(hipGetLastError());
    MTC_HIP(hipStreamSynchronize(st));
    rs.busy = false;
    hk = hdr[0];
    if (hk.ref_id <= k) hs.assign(hdr + 1, hdr + 1 + (k - hk.ref_id + 1));
  } else {
    MTC_HIP(hipMemcpyAsync(&hk, diffs[k], sizeof(hk), hipMemcpyDeviceToHost, st));
    MTC_HIP(hipStreamSynchronize(st));
  }
  check_last(hk, k, out_len);
  const uint64_t C = hk.chunk_size;
  const uint32_t n = (uint32_t)((hk.datalen + C - 1) / C), ref = hk.ref_id, L = k - ref + 1;
  for (uint32_t p = 0; p < L; p++) present(ref + (uint64_t)p);
  if (hs.empty()) {
    hs.resize(L);
    if (!on_device) {
      for (uint32_t p = 0; p < L; p++) std::memcpy(&hs[p], diffs[ref + (uint64_t)p], sizeof(mtc_header));
    } else {
      pinned_reserve(rs.stage, rs.stage_cap, 16ull * L + sizeof(mtc_header) * (L + 1ull));
      uint64_t* ptrs = reinterpret_cast<uint64_t*>(rs.stage);
      for (uint32_t p = 0; p < L; p++) ptrs[p] = reinterpret_cast<uint64_t>(diffs[ref + (uint64_t)p]);
      std::memcpy(ptrs + L, sizes + ref, 8ull * L);
      mtc_header* hdr = reinterpret_cast<mtc_header*>(ptrs + 2ull * L);
      rs.busy = true;
      k_r_headers<<<rgrid(8ull * (L + 1ull), 1024), kRThreads, 0, st>>>(ptrs, ptrs + L, ref, k, reinterpret_cast<uint32_t*>(hdr));
      MTC_HIP(hipGetLastError());
      MTC_HIP(hipStreamSynchronize(st));
      rs.busy = false;
      hs.assign(hdr + 1, hdr + 1 + L);
    }
  }
  // Chain layout, with host diffs uploaded once: an exact-size upload, freed when the
  // restart returns (a chain can be as large as the buffer, so it is not kept).
  std::vector<uint64_t> addr(L);
  DevBuf<uint8_t> upload;
  if (on_device) {
    for (uint32_t p = 0; p < L; p++) addr[p] = reinterpret_cast<uint64_t>(diffs[ref + (uint64_t)p]);
  } else {
    uint64_t total = 0;
    for (uint32_t p = 0; p < L; p++) {
      addr[p] = total;
      total += (sizes[ref + (uint64_t)p] + 255) & ~255ull;
    }
    upload.ensure(total);
    for (uint32_t p = 0; p < L; p++) addr[p] += reinterpret_cast<uint64_t>(upload.p);
  }
  const uint64_t words = meta_words(L);
  pinned_reserve(rs.stage, rs.stage_cap, 8 * words + 8);
  uint64_t* m = reinterpret_cast<uint64_t*>(rs.stage);
  volatile uint32_t* err_h = reinterpret_cast<volatile uint32_t*>(m + words);
  const ChainSums t = fill_meta(m, hs.data(), addr.data(), sizes + ref, L, hk, basic);
  err_h[0] = err_h[1] = 0;
  if (!on_device) {
    for (uint32_t p = 0; p < L; p++)
      MTC_HIP(hipMemcpyAsync(reinterpret_cast<void*>(addr[p]), diffs[ref + (uint64_t)p], sizes[ref + (uint64_t)p],
                             hipMemcpyHostToDevice, st));
    MTC_HIP(hipEventRecord(rs.ev[1], st));
  }
  const uint64_t cap = set_slots(t.F);
  rs.err.ensure(1);
  rs.region.reserve(t.F + L);
  rs.set_keys.ensure(cap);
  rs.set_vals.ensure(cap);
  rs.cover.ensure(n);
  rs.cum.reserve(t.cum);
  rs.meta.reserve(words);
  Chain c{L, n, (uint32_t)C, ref, basic ? n - 1 : 0u, make_geo(n), rs.meta.p, rs.region.p, rs.cum.p, rs.set_keys.p,
          rs.set_vals.p, cap - 1, rs.cover.p, rs.err.p, err_h};
  rs.busy = true;
  launch_restart(c, m, m, t, hk.datalen, out, st,
                 [&] { exclusive_scan_u32(c.region, c.region, t.F + L, nullptr, rs.ws, st); });
  MTC_HIP(hipEventRecord(rs.ev[2], st));
  MTC_HIP(hipStreamSynchronize(st));
  rs.busy = false;
  throw_err(err_h[0] | err_h[1]);
  if (!on_device) MTC_HIP(hipEventElapsedTime(&g_restart_ms[0], rs.ev[0], rs.ev[1]));  // else nothing was uploaded
  MTC_HIP(hipEventElapsedTime(&g_restart_ms[1], rs.ev[0], rs.ev[2]));
}

// ---------------------------------------------------------------------------
// Restart without allocation (mtc_restart_noalloc).  Every scratch buffer of the
// restart above -- the cover array, the (position, root) set, region offsets, the
// per-position tables and scan partials -- is carved from one static device array
// per GPU, and the host side uses no pinned staging: headers come back through one
// gather kernel and one small copy, and the running counts of shifted entries by
// source checkpoint are built on the device.  Chains are device-resident tree
// diffs of at most kNoAllocMaxChain checkpoints.
// ---------------------------------------------------------------------------
constexpr uint64_t kNoAllocScratch = 64ull << 20;  // bytes of `scratch` on each GPU
constexpr uint32_t kNoAllocMaxChain = 256;         // diffs from ref_id to the restarted checkpoint
constexpr int kNoAllocMaxDevices = 64;

static __device__ __align__(256) uint8_t scratch[kNoAllocScratch];

// Per GPU: the device address of `scratch` (taken once, with that GPU current) and
// the lock that keeps restarts on one GPU from sharing the array at the same time.
struct NoAllocDevice {
  std::mutex mu;
  uint8_t* ptr = nullptr;
};
static NoAllocDevice g_noalloc[kNoAllocMaxDevices];

// The 32-byte headers of the chain's diffs, gathered next to each other.
__global__ void k_r_gather_headers(const uint64_t* ptrs, uint32_t L, uint32_t* out) {
  const uint32_t i = blockIdx.x * kRThreads + threadIdx.x;
  if (i >= 8 * L) return;
  out[i] = ld32(reinterpret_cast<const uint8_t*>(ptrs[i / 8]) + 4 * (i % 8));
}

// Bump carving of the scratch array (256-byte aligned pieces).
struct Carve {
  uint64_t off = 0;
  uint64_t take(uint64_t bytes) {
    const uint64_t o = off;
    off = (off + bytes + 255) & ~255ull;
    return o;
  }
};

void restart_noalloc_impl(const void* const* diffs, const uint64_t* sizes, uint32_t count, uint32_t k, uint8_t* out,
                          uint64_t out_len, hipStream_t st) {
  if (!diffs || !sizes || k >= count || !diffs[k]) throw Status{MTC_ERR_INVALID_ARG, "bad diff chain arguments"};
  int dev = 0;
  MTC_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kNoAllocMaxDevices) throw Status{MTC_ERR_INVALID_ARG, "device ordinal above 63"};
  NoAllocDevice& nd = g_noalloc[dev];
  std::lock_guard<std::mutex> guard(nd.mu);
  if (!nd.ptr) {  // once per GPU, with it current: the device copy of `scratch`
    void* p = nullptr;
    MTC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw Status{MTC_ERR_HIP, "no device address for the restart scratch"};
    nd.ptr = static_cast<uint8_t*>(p);
  }
  uint8_t* const base = nd.ptr;
  g_restart_ms[0] = g_restart_ms[1] = 0;
  if (sizes[k] < sizeof(mtc_header)) throw Status{MTC_ERR_CORRUPT_DIFF, "missing or short diff"};
  mtc_header hk;
  MTC_HIP(hipMemcpyAsync(&hk, diffs[k], sizeof(hk), hipMemcpyDeviceToHost, st));
  MTC_HIP(hipStreamSynchronize(st));
  check_last(hk, k, out_len);
  const uint64_t C = hk.chunk_size;
  const uint32_t n = (uint32_t)((hk.datalen + C - 1) / C), ref = hk.ref_id, L = k - ref + 1;
  if (L > kNoAllocMaxChain)
    throw Status{MTC_ERR_INVALID_ARG, "the no-allocation restart takes chains of at most 256 diffs"};

  // Headers of the chain: one gather kernel, one copy.  The tables come to lie where
  // the addresses and headers were.
  Carve cv;
  uint32_t* err_p = reinterpret_cast<uint32_t*>(base + cv.take(4));
  uint8_t* const lead = base + cv.take(std::max<uint64_t>(8ull * L + 32ull * L, 8 * meta_words(L)));
  uint64_t* ptrs_d = reinterpret_cast<uint64_t*>(lead);
  uint32_t* hdr_d = reinterpret_cast<uint32_t*>(lead + 8ull * L);
  uint64_t ptrs_h[kNoAllocMaxChain];
  for (uint32_t p = 0; p < L; p++) {
    const uint32_t idx = ref + p;
    if (!diffs[idx] || sizes[idx] < sizeof(mtc_header)) throw Status{MTC_ERR_CORRUPT_DIFF, "missing or short diff"};
    ptrs_h[p] = reinterpret_cast<uint64_t>(diffs[idx]);
  }
  MTC_HIP(hipMemcpyAsync(ptrs_d, ptrs_h, 8ull * L, hipMemcpyHostToDevice, st));
  k_r_gather_headers<<<rgrid(8ull * L), kRThreads, 0, st>>>(ptrs_d, L, hdr_d);
  MTC_HIP(hipGetLastError());
  mtc_header hs[kNoAllocMaxChain];
  MTC_HIP(hipMemcpyAsync(hs, hdr_d, 32ull * L, hipMemcpyDeviceToHost, st));
  MTC_HIP(hipStreamSynchronize(st));

  // Chain layout (the same checks as the allocating restart).
  uint64_t meta_h[meta_words(kNoAllocMaxChain)];
  const ChainSums t = fill_meta(meta_h, hs, ptrs_h, sizes + ref, L, hk, false);
  uint32_t maxF = 0;
  for (uint32_t p = 0; p < L; p++) {
    if (hs[p].num_prior_chkpts > p + 1) throw Status{MTC_ERR_CORRUPT_DIFF, "prior-checkpoint table longer than the chain"};
    maxF = std::max(maxF, hs[p].num_first_ocur);
  }
  const uint64_t cap = set_slots(t.F);
  uint64_t* cover_p = reinterpret_cast<uint64_t*>(base + cv.take(8ull * n));
  uint64_t* keys_p = reinterpret_cast<uint64_t*>(base + cv.take(8 * cap));
  uint32_t* vals_p = reinterpret_cast<uint32_t*>(base + cv.take(4 * cap));
  const uint64_t off_region = cv.take(4 * (t.F + L));
  const uint64_t off_cum = cv.take(4 * t.cum);
  uint64_t off_sums[3];
  for (int d = 0; d < 3; d++) off_sums[d] = cv.take(4 * scan_sums_words(maxF, d));
  if (cv.off > kNoAllocScratch)
    throw Status{MTC_ERR_INVALID_ARG, "this restart needs " + std::to_string(cv.off) +
                                          " bytes of scratch; the no-allocation restart has 64 MiB per GPU"};
  uint32_t* region_p = reinterpret_cast<uint32_t*>(base + off_region);
  uint64_t* meta_p = reinterpret_cast<uint64_t*>(lead);
  uint32_t* const sums[3] = {reinterpret_cast<uint32_t*>(base + off_sums[0]),
                             reinterpret_cast<uint32_t*>(base + off_sums[1]),
                             reinterpret_cast<uint32_t*>(base + off_sums[2])};
  MTC_HIP(hipMemcpyAsync(meta_p, meta_h, 8 * meta_words(L), hipMemcpyHostToDevice, st));
  Chain c{L, n, (uint32_t)C, ref, 0u, make_geo(n), meta_p, region_p, reinterpret_cast<uint32_t*>(base + off_cum), keys_p,
          vals_p, cap - 1, cover_p, err_p, nullptr};
  // Region offsets diff by diff: the scan's scratch is sized for the largest one.
  launch_restart(c, nullptr, meta_h, t, hk.datalen, out, st, [&] {
    const uint64_t* region = meta_h + (uint64_t)M_REGION * L;
    for (uint32_t p = 0; p < L; p++) {
      uint32_t* ro = region_p + region[p];
      exclusive_scan_u32_fixed(ro, ro, hs[p].num_first_ocur, ro + hs[p].num_first_ocur, sums, st);
    }
  });
  check_err(err_p, st);
}

}  // namespace mtc
