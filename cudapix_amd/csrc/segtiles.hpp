// segtiles.hpp -- the tiles of the persistent segment kernel (segsieve.hip)
// and of the streaming kernel (stream.hip): hard-leaf phi sieve of one
// LDS-resident bitmap segment per tile, with the P2 prime count of the same
// segment as an epilogue; easy-leaf and P2-lookup tiles.
//
// Layout: bit 8q + i of a segment is the integer lo + 30q + r_i, r_i the i-th
// of the eight residues coprime to 30 (lo a multiple of 30), so a segment of
// SB = 32*K*T bits covers 3.75 SB integers -- 1.875 times what the odd numbers
// alone would give the same LDS, and every cost per (segment, stage) is spread
// over that many more integers.  The bits sit in units of 1024 (32 words and
// one padding word); thread t owns K/32 units, wave w the units of its 64
// threads.
//
// A tile is one segment of a group of up to CPX_GROUP queries (similar x,
// same wheel): the sieve state after stage b does not depend on x, so the
// tile sieves the segment once and evaluates every member's leaves against
// it.
//
// Hard leaves (replaces S2glob::S2ctl + S2hardHost, src/sieve/S2_hard_device.cu:264-355,
// src/sieve/S2_hard_host.cu:115-191; DR split p <= x^(1/4), src/Deleglise-Rivat/S3.cu:8):
//   The segment starts as the wheel of the first cs primes.  Stages b (p = p_b,
//   cs < b <= B, while p^2 <= x/lo for some member) run in chunks: the block
//   first lists the chunk's items, the (stage, member) pairs with leaf
//   candidates in the segment (x/p, the candidate range), each wave finds its
//   part of every item's range, then walks the chunk's stages on its own, with
//   no block barrier:
//     L  leaves of p whose n = x/(p m) falls in the wave's bits, all members'
//        in one list: m with mu(m) != 0 and lpf(m) > p from the leaf table of
//        the m coprime to 30030 (p^2 <= y) or m prime (p^2 > y); the wave
//        publishes its in-wave prefix counts and counts phi_wave(n) = prefix of
//        the unit + popcounts of its words below n; sum mu * phi_wave per
//        member, sum mu per wave and item;
//     X  cross off the multiples of p in the wave's bits, recording the
//        removals.
//   At the end of a chunk the block adds the survivors of the earlier waves
//   to every leaf's count (from the per-stage, per-wave removals and sums of
//   mu), and writes T_b (survivors before stage b) and sum_b(mu); the carry
//   kernel adds sum_b prefix_b(seg) * sum_b(mu) over the segments (the
//   decomposition the reference does with scanVectorized/addMultiply,
//   src/sieve/S2_hard_device.cu:357-375).
//
// P2: the segments holding x/p for a member's P2 primes p in (y, sqrt x]
// get, on replica 0 of their tile (on all of them where the primes are many), the rest of a prime sieve (primes above
// the last stage up to sqrt(hi)) and each such member's P2 counts; see
// p2_epilogue.
#pragma once
#include "cpx_device.hpp"

#ifndef P2_WAVE_P
#define P2_WAVE_P 1024     // P2 sieve: primes below this are crossed by a whole wave
#endif
#define P2_U 4             // P2 primes of a lane in flight (1, 2 and 4 are even)
static_assert(CPX_GROUP == 32, "member slots: 1, 8 or 32");

// Stages of a chunk at most, by member slots (one item per thread is tested).
template <int GS>
struct ChunkStages {
  static constexpr uint32_t SST = GS == 1 ? 64 : (GS <= 8 ? 32 : 16);
};

// A group member's share of the current segment (zero when its hard range
// ends before the segment).
struct GroupMember {
  uint64_t stage_off;   // its stage table
  uint64_t toff;        // hard_T index of its stage 0 in this segment's row
  uint64_t moff;        // hard_M index of its stage 0 for this replica
  uint32_t y;
  uint32_t nst;         // its active stages in the segment
  uint32_t on;          // the segment is in its hard range (1), and in its P2 range (2)
  uint32_t pad;
};

template <int T, int K>
struct SegShared {
  static constexpr uint32_t NW = T / CPX_WAVE, NU = T * (K / 32);
  // items of a chunk: as many as the LDS left by two blocks per CU holds
  static constexpr uint32_t NI = NW >= 8 ? 96 : 128;
  // survivors of each unit's four quarters, a byte each (a quarter's 256 bits
  // lose at least the multiples of 7 and 11), kept in the stages that count
  // their removals one by one and published at a stage with leaves
  uint32_t cnt[NU];
  // published at a stage with leaves: the unit's in-wave exclusive prefix
  uint32_t ipre[NU];
  long long acc[NW][CPX_GROUP];  // sum of mu * phi by wave and member
  GroupMember gm[CPX_GROUP];
  uint32_t wtot[NW];             // wave totals (P2)
  int32_t wsum[NW];              // per-wave sums
  unsigned long long red_u[NW];
  // the chunk: its items, in stage order
  uint64_t xp[NI];               // floor(x / p), low 64 bits
  uint16_t xph[NI];              // ... and bits 64-79 (nonzero only for x above 2^68)
  uint16_t kg[NI];               // stage * 32 + member
  uint32_t cbase[NI];            // first candidate: index of the leaf table or of a prime
  uint32_t ccnt[NI];             // candidates | HARD_SPARSE
  int32_t wm[NI][NW];            // sum of mu of each wave's leaves
  uint16_t dw[64][NW];           // survivors each wave removes at each stage
  uint32_t gmask[32];            // members with an item at the stage (member slots > 1)
  uint8_t ist[68];               // first item of each stage
  uint32_t c0[NW];               // each wave's survivors at the chunk start
  uint32_t wcount[NW];
  uint32_t clen;
  uint32_t tile;
};

// A block's LDS, one object at a fixed address, so that the bitmap's and the
// tables' addresses are instruction offsets: units of 32 words and one of padding.
template <int T, int K>
struct SegLds {
  SegShared<T, K> sh;
  __attribute__((aligned(16))) uint32_t bits[SegShared<T, K>::NU * 33];
  // waves per SIMD that a CU's LDS holds: the register budget (4 for 512 threads x 32 words)
  static constexpr int waves()
  {
    return 163840 / (int)sizeof(SegLds) * (T / CPX_WAVE) / 4 > 0 ? 163840 / (int)sizeof(SegLds) * (T / CPX_WAVE) / 4 : 1;
  }
};

#define HARD_NC_MASK 0x7fffffffu
#define HARD_SPARSE 0x80000000u    // p^2 > y: candidates are primes
// Stages with p below this cross without returns and recount the wave's
// bits afterwards (a popcount per word of the thread); above, each removal
// is taken off its quarter's count.  Steps of a wave per stage: 1024/p.
#ifndef HARD_RECOUNT_P
#define HARD_RECOUNT_P 128
#endif

// threadIdx.x, opaque: what one part of a tile derives from it is not kept in
// registers through the others (20 -> 6 spilled registers in the 512-thread
// kernel; two 512-query batches 30.8 -> 29.7 ms).
__device__ __forceinline__ uint32_t own_thread()
{
  uint32_t t = threadIdx.x;
  asm("" : "+v"(t));
  return t;
}

// Word of bit j of a bitmap in padded units.  (One shift-add forms the byte
// offset; the compiler's own form takes two shifts, two masks and an add.)
__device__ __forceinline__ uint32_t *unit_word(uint32_t *bits, uint32_t j)
{
  const uint32_t w = j >> 5, u = j >> 10;
  uint32_t o;
  asm("v_add_lshl_u32 %0, %1, %2, 2" : "=v"(o) : "v"(w), "v"(u));
  return (uint32_t *)((char *)bits + o);
}

// Survivors of the four quarters of a unit, a byte each.
__device__ __forceinline__ uint32_t unit_counts(const uint32_t *w)
{
  uint32_t q[4] = {0, 0, 0, 0};
#pragma unroll
  for (uint32_t j = 0; j < 32; j++) q[j >> 3] += cpx_popc32(w[j]);
  return q[0] | q[1] << 8 | q[2] << 16 | q[3] << 24;
}
__device__ __forceinline__ uint32_t unit_total(uint32_t c) { return __builtin_amdgcn_sad_u8(c, 0u, 0u); }

// Publish the wave's prefix counts from its threads' unit counts.
template <int UPT>
__device__ __forceinline__ uint32_t publish_units(const uint32_t (&c)[UPT], uint32_t *ipre)
{
  uint32_t s = 0;
#pragma unroll
  for (int u = 0; u < UPT; u++) s = __builtin_amdgcn_sad_u8(c[u], 0u, s);
  const uint32_t incl = wave_incl_scan(s);
  uint32_t ex = incl - s;
#pragma unroll
  for (int u = 0; u < UPT; u++) {
    ipre[threadIdx.x * UPT + u] = ex;
    ex = __builtin_amdgcn_sad_u8(c[u], 0u, ex);
  }
  return (uint32_t)__builtin_amdgcn_readlane((int)incl, CPX_WAVE - 1);
}

// Survivors at or below bit g of the units from `bits`, of which ipre and cnt
// hold the published prefixes and quarter counts.  The quarter's eight words,
// the published words and the bit's own word are loaded before any is used, so
// the count costs one LDS round trip; words at or above the bit's are masked out.
__device__ __forceinline__ uint32_t unit_count_to(const uint32_t *bits, const uint32_t *ipre, const uint32_t *cnt,
                                                  uint32_t g)
{
  const uint32_t u = g >> 10, nf = (g >> 5) & 7u;
  const uint32_t *w = bits + ((g >> 5) & ~7u) + u;
  uint32_t wd[8];
#pragma unroll
  for (uint32_t r = 0; r < 8; r++) wd[r] = w[r];
  const uint32_t part = w[nf], pre = ipre[u], q = cnt[u];
  const uint32_t full = (1u << nf) - 1u;
  uint32_t c = __builtin_amdgcn_sad_u8(q & ((1u << ((g >> 5) & 24u)) - 1u), 0u, pre);
#pragma unroll
  for (uint32_t r = 0; r < 8; r++) c += cpx_popc32(wd[r] & (uint32_t)__builtin_amdgcn_sbfe((int)full, r, 1u));
  return c + cpx_popc32(part & ((2u << (g & 31u)) - 1u));
}

// Number of table entries m <= M: primes (sparse) or leaf-table m's.
__device__ __forceinline__ uint32_t leaf_rank(const BatchDev &bd, bool sparse, uint32_t M)
{
  return sparse ? (uint32_t)pi_lookup(bd.pitab, M) : cop30030_upto(M);
}

// floor((xph 2^64 + xp) / d), or ~0 where it is 2^50 or more (above every m <= y).
__device__ __forceinline__ uint64_t leaf_bound(uint64_t xp, uint32_t xph, uint64_t d, double inv)
{
  if (d == 0 || !cpx_quot_below_2_50(xp, xph, d)) return ~0ull;
  return xph ? cpx_div_recip_w(xp, xph, d, inv) : cpx_div_recip(xp, d, inv);
}

// Items of the stages [s0, s0 + se) (the stage primes are primes[cs + s0 + k],
// shared by the members), one (stage, member) per thread: x/p and the
// candidates of the leaves m in (x/(p hi), x/(p lo)], m > y/p.  Only those with
// candidates become items; a chunk ends before the stage whose items no longer
// fit.  Returns the chunk's stages; *ni = its items.  Block barriers inside.
template <int T, int K, int GS>
__device__ __forceinline__ uint32_t hard_items(const BatchDev &bd, SegShared<T, K> &sh, uint32_t s0,
                                               uint32_t se, uint64_t lo, uint64_t hi, double inv_lo,
                                               double inv_hi, uint32_t *ni)
{
  constexpr uint32_t NW = T / CPX_WAVE, NI = SegShared<T, K>::NI;
  const uint32_t t = own_thread();
  const uint32_t lane = t % CPX_WAVE, wv = t / CPX_WAVE;
  const uint32_t k = t / GS, g = t % GS;
  uint32_t nc = 0, cb = 0, xph = 0;
  uint64_t xp = 0;
  bool sparse = false;
  if (k < se) {
    const GroupMember &m = sh.gm[g];
    if (s0 + k < m.nst) {
      const StageDev sd = bd.stages[m.stage_off + s0 + k];
      const uint64_t p = sd.p, y = m.y;
      xp = sd.xp;
      xph = sd.xph;
      sparse = p * p > y;
      uint64_t mhi = min(y, leaf_bound(xp, xph, lo, inv_lo));
      uint64_t mlo = leaf_bound(xp, xph, hi, inv_hi);
      if (sparse) mhi = min(mhi, sd.xp3);                // q above x/p^3: pi-table lookups
      mlo = max(mlo, (uint64_t)sd.ylo);
      if (sparse) mlo = max(mlo, p);
      if (mlo < mhi) {
        cb = leaf_rank(bd, sparse, (uint32_t)mlo);
        nc = leaf_rank(bd, sparse, (uint32_t)mhi) - cb;
      }
    }
  }
  const uint64_t bal = __ballot(nc != 0);
  if (lane == 0) sh.wcount[wv] = (uint32_t)__popcll(bal);
  if (t == 0) sh.clen = se;
  __syncthreads();
  uint32_t rank = 0, total = 0;
#pragma unroll
  for (uint32_t w = 0; w < NW; w++) {
    rank += w < wv ? sh.wcount[w] : 0u;
    total += sh.wcount[w];
  }
  rank += __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
  if (g == 0 && k < se) {
    const uint32_t gm = (uint32_t)(bal >> lane) & (GS == 32 ? ~0u : (1u << GS) - 1u);
    sh.ist[k] = (uint8_t)min(rank, 255u);
    if (GS > 1) sh.gmask[k] = gm;
    if (rank + cpx_popc32(gm) > NI) atomicMin(&sh.clen, k);
  }
  if (nc && rank < NI) {
    sh.xp[rank] = xp;
    sh.xph[rank] = (uint16_t)xph;
    sh.kg[rank] = (uint16_t)(k * 32 + g);
    sh.cbase[rank] = cb;
    sh.ccnt[rank] = nc | (sparse ? HARD_SPARSE : 0u);
  }
  __syncthreads();
  const uint32_t n = (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.clen);
  *ni = n < se ? (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.ist[n]) : total;
  return n;
}

// Lane l's value of v for a per-lane l; every lane must be active.
__device__ __forceinline__ uint32_t lane_get(uint32_t v, uint32_t l)
{
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(l * 4), (int)v);
}
__device__ __forceinline__ uint32_t lane_read(uint32_t v, uint32_t l)      // wave-uniform l
{
  return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)l);
}

// Add one window of list entries [fb, fb + 64) (lane l holds entry fb + l:
// val = mu * phi_wave, sg = mu, zero past the list) to the sums of item
// lanes: a lane gains the sums over its entries [my_lo, my_hi).  One wave
// scan of val * 256 + sg, read at each item's ends: with at least 7 and 11
// sieved out |val| <= 0.78 * 2^17 for K <= 64, so a window's sum is below 2^31
// and its low byte is the sum of sg.
template <int K>
__device__ __forceinline__ void hard_lane_accumulate(int32_t val, int32_t sg, uint32_t fb, uint32_t my_lo,
                                                     uint32_t my_hi, int64_t &acc, int32_t &wmv)
{
  // list offsets are below 2^31: an item has at most 0.192 y candidates (m
  // coprime to 30030), and groups of more than one member have y < 2^28, so
  // 32 of them at most 1.65e9
  const int32_t lo = min(max((int32_t)my_lo - (int32_t)fb, 0), CPX_WAVE);
  const int32_t hi = min(max((int32_t)my_hi - (int32_t)fb, 0), CPX_WAVE);
  auto range = [&](uint32_t S) {
    const uint32_t shi = lane_get(S, (uint32_t)(hi > 0 ? hi - 1 : 0));
    const uint32_t slo = lane_get(S, (uint32_t)(lo > 0 ? lo - 1 : 0));
    return (int32_t)((hi > 0 ? shi : 0u) - (lo > 0 ? slo : 0u));
  };
  if (K <= 64) {
    const int32_t d = range(wave_incl_scan((uint32_t)(val * 256 + sg)));
    const int32_t sgs = (int32_t)((uint32_t)d << 24) >> 24;
    acc += (d - sgs) >> 8;
    wmv += sgs;
  } else {
    acc += range(wave_incl_scan((uint32_t)val));
    wmv += range(wave_incl_scan((uint32_t)sg));
  }
}

// End of a chunk of stages [s0, s0 + n) (all threads call and keep
// `running`): writes, for every member g and its active stages b, T_b =
// survivors of the segment before stage b (replica 0) and this replica's sum
// of mu, and adds to every member's sum the part of its leaves' phi that the
// in-wave count left out -- the survivors of the earlier waves at the stage:
//   sum over items i (stage k) of wm[i][w] * (A_w - sum_{j<k} sum_{w'<w} dw[j][w'])
// with A_w the earlier waves' survivors at the chunk start.  kk: the stages
// of the items lane and lane + 64.
template <int T, int K, int GS>
__device__ __forceinline__ void hard_flush(const BatchDev &bd, SegShared<T, K> &sh, uint32_t s0,
                                           uint32_t n, uint32_t ni, const uint32_t (&kk)[2],
                                           uint32_t &running, bool write_T, int64_t &acc)
{
  constexpr uint32_t NW = T / CPX_WAVE, SST = ChunkStages<GS>::SST;
  const uint32_t lane = lane_id(), wv = wave_id();
  __syncthreads();
  uint32_t Gk = 0, D = 0;
  if (lane < n) {
#pragma unroll
    for (uint32_t w = 0; w < NW; w++) {
      const uint32_t d = sh.dw[lane][w];
      D += d;
      Gk += w < wv ? d : 0u;
    }
  }
  if (NW > 1) {
    uint32_t A = 0;
#pragma unroll
    for (uint32_t w = 0; w < NW; w++) A += w < wv ? sh.c0[w] : 0u;
    const uint32_t R = wave_incl_scan(Gk) - Gk;
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) {
      if (h * CPX_WAVE >= ni) break;
      const uint32_t i = h * CPX_WAVE + lane, Rk = lane_get(R, kk[h]);
      if (i < ni) {
        const int64_t v = (int64_t)sh.wm[i][wv] * ((int64_t)A - (int64_t)Rk);
        if (GS == 1) acc += v;
        else if (v) atomicAdd((unsigned long long *)&sh.acc[wv][sh.kg[i] & 31u], (unsigned long long)v);
      }
    }
  }
  // T_b and the sums of mu: a wave writes SST stages of 64/SST members at a time
  const uint32_t incl = wave_incl_scan(D);
  const uint32_t Tk = running - (incl - D);
  running -= lane_read(incl, CPX_WAVE - 1);
  const uint32_t k = lane % SST, Tw = lane_get(Tk, k);
  for (uint32_t g = wv * (CPX_WAVE / SST) + lane / SST; g < GS; g += NW * (CPX_WAVE / SST)) {
    const GroupMember &m = sh.gm[g];
    if (k >= n || s0 + k >= m.nst) continue;
    uint32_t i = sh.ist[k];
    bool has;
    if (GS == 1) {
      has = i < (k + 1 < n ? (uint32_t)sh.ist[k + 1] : ni);
    } else {
      const uint32_t gm = sh.gmask[k];
      has = (gm >> g) & 1u;
      i += cpx_popc32(gm & ((1u << g) - 1u));
    }
    int32_t ms = 0;
    if (has) {
#pragma unroll
      for (uint32_t w = 0; w < NW; w++) ms += sh.wm[i][w];
    }
    if (write_T) st_out(&bd.hard_T[m.toff + s0 + k], Tw);
    st_out(&bd.hard_M[m.moff + s0 + k], ms);
  }
  __syncthreads();
}

// P2 leaves of a segment (replaces the windowed upper_bound count of
// src/P2.cu:76-133), run by a hard tile after its stages: the
// bitmap already holds [lo, hi) sieved by the wheel and by the stage primes
// below primes[kfirst]; the primes from index kfirst with p^2 < hi are
// crossed here, which leaves exactly the primes above the largest
// p2_e of the members.  Then, for each member whose P2 range holds the
// segment and each of its P2 primes p in (max(y, x/hi), min(sqrt x, x/lo)]
// (pi-table bits, block-strided), the count of primes in (p2_e, x/p] held in
// this segment; per member and segment: primes in (p2_e, hi), number of p,
// sum of the counts.  The carry is applied in the combine kernel.
//
// Replica 0 does this alone, or where the P2 primes are many (CPX_P2_SHARE) all
// replicas do, each the sieve and its share of the primes.  The first segments
// of a small x hold most of them: at 1e12 segment 0 counts 37 K, 74 us of one
// block bound by VALU issue (about 100 instructions a count) while the others
// are done.  Shared, pi(1e12) takes 325 us instead of 400, 1e13 with fresh tables
// 735 instead of 820 (100 of it the table's); with the threshold at 2 to 8
// entries a thread the same, at 32 or more nothing is shared at 1e12.
template <int T, int K>
__device__ __forceinline__ void p2_epilogue(const BatchDev &bd, const GroupDev &grp, uint64_t seg,
                                            uint32_t rep, uint32_t nrep, uint64_t lo, uint32_t kfirst,
                                            uint32_t *lds, SegShared<T, K> &sh)
{
  constexpr uint32_t NW = T / CPX_WAVE, UPT = K / 32, WU = CPX_WAVE * UPT;
  constexpr uint32_t SB = 32u * K * T;
  const uint32_t t = own_thread();
  const uint32_t lane = t % CPX_WAVE, wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(t / CPX_WAVE));
  const uint64_t hi = lo + SB / 8 * 30, base = lo / 30;
  const uint32_t *__restrict__ sp = bd.primes;
  const uint32_t np_all = (uint32_t)bd.nprimes;

  // (the same f64 estimate in every replica)
  bool share = false;
  if (nrep > 1) {
    double ents = 0;
    if (lane < grp.n && (sh.gm[lane].on & 2u)) {
      const QueryDev &q = bd.queries[grp.q[lane]];
      const double xf = (double)q.x_hi * 0x1p64 + (double)q.x_lo, sq = (double)q.sqrtx;
      const double pm = lo ? fmin(sq, xf / (double)lo) : sq;
      ents = fmax(0.0, pm - fmax((double)q.y, xf / (double)hi)) * (1.0 / 64);
    }
    share = wave_sum((unsigned long long)ents) > (unsigned long long)CPX_P2_SHARE * T;
  }
  if (rep && !share) {
    if (t < grp.n && (sh.gm[t].on & 2u)) {
      const QueryDev &q = bd.queries[grp.q[t]];
      const uint64_t mr = q.mrow_base + bd.rowinfo[q.hard_row0 + seg].mrow + rep;
      st_out(&bd.p2_np[mr], 0u);
      st_out(&bd.p2_loc[mr], (uint64_t)0);
    }
    return;
  }
  // member g's P2 primes of the segment, (pmin, pmax], in lane g of every wave
  uint64_t pmin = 0, pmax = 0;
  if (lane < grp.n && (sh.gm[lane].on & 2u)) {
    const QueryDev &q = bd.queries[grp.q[lane]];
    const u128 x = ((u128)q.x_hi << 64) | q.x_lo;
    pmax = lo ? min(q.sqrtx, cpx_div128_to64(x, lo)) : q.sqrtx;
    pmin = max(q.y, cpx_div128_to64(x, hi));
    pmin = min(pmin, pmax);
  }
  const uint32_t e0 = share ? rep * T + t : t, estep = share ? nrep * T : T;

  __syncthreads();
  // primes below P2_WAVE_P have many multiples: one prime per wave, eight
  // classes of multiples times eight in step, so no lane walks a long chain
  // alone.  (The wave's next 64 primes and their constants sit in its lanes;
  // fetched one by one they cost pi(1e9) 6 us of 160.)
  {
    const CrossLane cl(lane);
    uint32_t n = CPX_WAVE;
    for (uint32_t k0 = kfirst + wv; n == CPX_WAVE && k0 < np_all; k0 += NW * CPX_WAVE) {
      const uint32_t k = k0 + NW * lane, pk = sp[min(k, np_all - 1)];
      n = (uint32_t)__popcll(__ballot(k < np_all && pk < P2_WAVE_P && (uint64_t)pk * pk < hi));
      const uint32_t d8k = 8 * (uint32_t)(base - cpx_div_leaf(base, (double)base, pk) * pk);
      const uint32_t ack = pk / 30u << 6 | cop30_class8(pk);
      for (uint32_t i = 0; i < n; i++) {
        const uint32_t p = lane_read(pk, i), ac = lane_read(ack, i);
        const uint32_t p8 = 8 * p, p64 = 64 * p;
        uint32_t j = cl.first(ac >> 6, ac & 63u, p8, lane_read(d8k, i)) + (lane >> 3) * p8;
        if (base == 0 && lane == 0) j += p64;             // p itself
        for (; j < SB; j += p64) atomicAnd(unit_word(lds, j), ~(1u << (j & 31u)));
      }
    }
  }
  // the rest: one prime per lane, class after class
  for (uint32_t k = kfirst + t; k < np_all; k += T) {
    const uint32_t p = sp[k];
    if ((uint64_t)p * p >= hi) break;
    if (p < P2_WAVE_P) continue;
    const uint32_t p8 = 8 * p, a = p / 30u;
    const uint32_t d8 = 8 * (uint32_t)(base - cpx_div_leaf(base, (double)base, p) * p);
    // (the table is symmetric: the lane constants of p's own class are its bytes by class of multiple)
    const uint64_t eb = cop30_products.e[cop30_class8(p) >> 3];
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
      uint32_t j = a * (8 * cop30_residue(i)) + ((uint32_t)(eb >> (8 * i)) & 255u) - d8;
      j = min(j, j + p8);
      if (i == 0 && base == 0) j += p8;                 // p itself
      for (; j < SB; j += p8) atomicAnd(unit_word(lds, j), ~(1u << (j & 31u)));   // SB + 8p < 2^32
    }
  }
  __syncthreads();
  {
    uint32_t c[UPT];
#pragma unroll
    for (uint32_t u = 0; u < UPT; u++) c[u] = sh.cnt[t * UPT + u] = unit_counts(lds + (t * UPT + u) * 33);
    const uint32_t ws = publish_units<(int)UPT>(c, sh.ipre);
    if (lane == 0) sh.wtot[wv] = ws;
  }
  __syncthreads();
  uint32_t wp[NW], tot = 0;
#pragma unroll
  for (uint32_t w = 0; w < NW; w++) { wp[w] = tot; tot += sh.wtot[w]; }
  // survivors at or below n (lo <= n < hi)
  auto count_to = [&](uint64_t n) {
    const uint32_t bits = cop30_upto((uint32_t)(n - lo)), b = max(bits, 1u) - 1, wave = (b >> 10) / WU;
    uint32_t pre = 0;
#pragma unroll
    for (uint32_t w = 0; w < NW; w++) pre = wave == w ? wp[w] : pre;
    return bits ? pre + unit_count_to(lds, sh.ipre, sh.cnt, b) : 0u;
  };
  for (uint32_t g = 0; g < grp.n; g++) {
    if (!(sh.gm[g].on & 2u)) continue;
    const QueryDev &q = bd.queries[grp.q[g]];
    const u128 x = ((u128)q.x_hi << 64) | q.x_lo;
    // x / p < z < 2^50 for every P2 prime: the reciprocal divide when p < 2^32
    const bool fastdiv = q.sqrtx < (1ull << 32);
    const double xf = (double)x;
    // survivors at or below p2_e (1, the stage primes and what is below
    // sqrt x are not counted): only the first segment of the range has any
    const uint32_t ce = q.p2_e >= lo ? count_to(min(q.p2_e, hi - 1)) : 0u;

    unsigned long long loc = 0;
    uint32_t np = 0;
    const uint64_t p_lo = lane_read((uint32_t)pmin, g) | (uint64_t)lane_read((uint32_t)(pmin >> 32), g) << 32;
    const uint64_t p_hi = lane_read((uint32_t)pmax, g) | (uint64_t)lane_read((uint32_t)(pmax >> 32), g) << 32;
    if (p_hi > p_lo) {
      const uint64_t e_lo = (p_lo + 1) >> 6, e_hi = p_hi >> 6;
      for (uint64_t e = e_lo + e0; e <= e_hi; e += estep) {
        const PiEntry pe = bd.pitab[e];
        uint32_t b = pe.bits;
        const uint64_t base64 = 64 * e;
        // keep odd integers base64 + 2i + 1 in (p_lo, p_hi]
        if (p_hi < base64 + 63) b &= cpx_lowmask32((uint32_t)((p_hi - base64 + 1) >> 1));
        if (p_lo > base64) {
          const uint64_t kk = (p_lo - base64 + 1) >> 1;     // bits for integers <= p_lo
          b = kk >= 32 ? 0u : (b & ~cpx_lowmask32((uint32_t)kk));
        }
        np += cpx_popc32(b);
        while (b && fastdiv) {                              // lo <= x / p < hi
          bool on[P2_U];
          uint64_t v[P2_U];
#pragma unroll
          for (uint32_t u = 0; u < P2_U; u++) {
            on[u] = b != 0;
            const uint32_t i = on[u] ? __builtin_ctz(b) : 0u;
            b &= b - 1;
            v[u] = on[u] ? cpx_div_leaf(q.x_lo, xf, (uint32_t)(base64 + 2 * i + 1)) : lo;
          }
#pragma unroll
          for (uint32_t u = 0; u < P2_U; u++) {
            const uint32_t ct = count_to(v[u]);
            loc += on[u] ? ct - ce : 0u;
          }
        }
        for (; b; b &= b - 1) loc += count_to(cpx_div128_to64(x, base64 + 2 * __builtin_ctz(b) + 1)) - ce;
      }
    }
    loc = wave_sum(loc);
    const uint32_t npw = wave_sum(np);
    if (lane == 0) { sh.red_u[wv] = loc; sh.wsum[wv] = (int32_t)npw; }
    __syncthreads();
    if (t == 0) {
      unsigned long long L = 0;
      uint32_t N = 0;
      for (uint32_t w = 0; w < NW; w++) { L += sh.red_u[w]; N += (uint32_t)sh.wsum[w]; }
      const uint64_t mr = q.mrow_base + bd.rowinfo[q.hard_row0 + seg].mrow + rep;
      if (rep == 0) st_out(&bd.p2_cnt[q.p2_row0 + (seg - q.p2_seg0)], (uint32_t)(tot - ce));
      st_out(&bd.p2_np[mr], (uint32_t)N);
      st_out(&bd.p2_loc[mr], (uint64_t)L);
    }
    __syncthreads();
  }
}

// The stage chunks of one tile with GS member slots: leaves, cross-off and
// chunk flushes; adds the members' sums of mu * phi to sh.acc.
//
// Cross-off: the multiples of p coprime to 30 in the wave's bits are eight
// arithmetic progressions of stride 8p bits; the wave takes eight of each at a
// time (lane & 7 the class, lane >> 3 the step), so a stage of a prime above
// 1024 (K = 32) is one LDS and-with-return per lane.  (With every thread
// crossing its own bits instead, one multiple or none each, a stage cost the
// wave about 50 instructions to find the lanes' first multiples.)
//
// Bound by VALU issue: at x = 1e17 the SIMDs have a VALU instruction in flight
// 78 % of the time (6.1e9 of them in 13.4 ms, 4 cycles each), so what counts is
// instructions per (wave, stage).  Against odd-only bits, own-bits crossing,
// candidates from every odd m and groups of 8, the layout above took two
// 512-query batches to 1e15 from 64.2 to 35.5 ms, 1e16 from 7.7 to 5.4 ms, 1e18
// from 153 to 97 ms.  First multiples of eight stages at a time, four stages'
// operations in flight, removals taken off byte counters and one LDS object at a
// fixed address took a stage of a prime above 1024 from 35 to 20 VALU
// instructions: 1e16 4.36 -> 4.05 ms, 1e18 79.2 -> 68.4 ms, 1e12 431 -> 402 us.
template <int T, int K, int GS>
__device__ __forceinline__ void hard_chunks(const BatchDev &bd, SegShared<T, K> &sh, uint32_t *lds,
                                            uint32_t cs, uint32_t nst, uint32_t rep, uint32_t cstep,
                                            uint64_t lo, uint64_t hi)
{
  constexpr uint32_t NW = T / CPX_WAVE, UPT = K / 32, WU = CPX_WAVE * UPT, WB = WU * 1024;
  constexpr uint32_t SST = ChunkStages<GS>::SST < T / GS ? ChunkStages<GS>::SST : T / GS;
  const uint32_t t = own_thread();
  const uint32_t lane = t % CPX_WAVE;
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_id());
  const uint64_t lo_w = lo + (uint64_t)wv * (WB / 8 * 30), hi_w = lo_w + WB / 8 * 30;
  const double inv_lo_w = lo_w ? 1.0 / (double)lo_w : 0.0, inv_hi_w = 1.0 / (double)hi_w;
  const double inv_lo = lo ? 1.0 / (double)lo : 0.0, inv_hi = 1.0 / (double)hi;
  const uint64_t base_w = lo_w / 30;
  const uint32_t wbit = wv * WB;                        // the wave's bits start here
  const CrossLane cl(lane);

  // survivors: the thread's units, the wave, the segment
  uint32_t cr[UPT];
  uint32_t wcur = 0, running = 0;
#pragma unroll
  for (uint32_t u = 0; u < UPT; u++) {
    cr[u] = unit_counts(lds + (t * UPT + u) * 33);
    wcur += unit_total(cr[u]);
  }
  wcur = wave_sum(wcur);
  if (lane == 0) sh.wsum[wv] = (int32_t)wcur;
  __syncthreads();
#pragma unroll
  for (uint32_t w = 0; w < NW; w++) running += (uint32_t)sh.wsum[w];
  bool counted = false;                                 // counts live in sh.cnt, not in cr

  int64_t acc = 0;                                      // GS = 1: sum of mu * phi, per lane
  for (uint32_t s0 = 0; s0 < nst;) {
    const uint32_t se = min(SST, nst - s0);
    // stage constants, stage k in lane k: p, 8 (base mod p), p / 30 and the class of p
    // (p < 2^21: the pi table's reach bounds x^(1/4))
    const uint32_t pk = bd.primes[cs + s0 + min(lane, se - 1)];
    uint32_t ni;
    const uint32_t n = hard_items<T, K, GS>(bd, sh, s0, se, lo, hi, inv_lo, inv_hi, &ni);
    const uint32_t d8k = 8 * (uint32_t)(base_w - cpx_div_leaf(base_w, (double)base_w, pk) * pk);
    const uint32_t ack = pk / 30u << 6 | cop30_class8(pk);
    const uint32_t istk = sh.ist[lane];
    if (lane == 0) sh.c0[wv] = wcur;
    // the wave's candidates [ia, ia + in) of the items lane and lane + 64
    uint32_t ia[2], in[2], kk[2];
    uint64_t im[2];
#pragma unroll
    for (uint32_t h = 0; h < 2; h++) {
      ia[h] = in[h] = kk[h] = 0;
      im[h] = 0;
      if (h * CPX_WAVE >= ni) continue;
      const uint32_t i = h * CPX_WAVE + lane;
      if (i < ni) {
        const uint32_t kg = sh.kg[i], cc = sh.ccnt[i], nc = cc & HARD_NC_MASK, cb = sh.cbase[i];
        const uint64_t xp = sh.xp[i], y = sh.gm[GS == 1 ? 0 : kg & 31u].y;
        const uint32_t xph = sh.xph[i];
        kk[h] = kg >> 5;
        const bool sparse = cc & HARD_SPARSE;
        // n in [lo_w, hi_w) <=> floor(x/p / hi_w) < m <= floor(x/p / lo_w)
        const uint32_t ra = leaf_rank(bd, sparse, (uint32_t)min(y, leaf_bound(xp, xph, hi_w, inv_hi_w)));
        const uint32_t rb = leaf_rank(bd, sparse, (uint32_t)min(y, leaf_bound(xp, xph, lo_w, inv_lo_w)));
        const uint32_t a = min(ra > cb ? ra - cb : 0u, nc), b = min(rb > cb ? rb - cb : 0u, nc);
        ia[h] = cb + a;
        in[h] = b > a ? b - a : 0u;
        sh.wm[i][wv] = 0;
      }
      im[h] = __ballot(in[h] != 0);
    }

    // the next stage with candidates of the wave: stage nk, items [is, ie),
    // ntot candidates in one list; item is + l takes list offsets [my_lo, my_hi)
    // of lane l and starts at candidate ml
    uint32_t nk = n, is = 0, ie = 0, ntot = 0, my_lo = 0, my_hi = 0, ml = 0;
    // this lane's next list entry: its item and candidate, loaded ahead
    uint32_t fi = 0;
    int2 pf = {0, 0};
    // (every lane calls; f may lie past the list)
    auto entry = [&](uint32_t f, uint32_t &it) {
      if (GS == 1) {
        it = is;
        return ml + f;
      }
      uint32_t l = 0;                                   // items that end at or before f
#pragma unroll
      for (uint32_t st = GS / 2; st; st >>= 1) l += f >= lane_get(my_hi, l + st - 1) ? st : 0u;
      it = is + l;
      return lane_get(ml, l) + f - lane_get(my_lo, l);
    };
    auto fetch = [&](uint32_t it, uint32_t c) {
      int2 v = {0, 0};
      if (sh.ccnt[it] & HARD_SPARSE) v.x = (int)bd.primes[c];
      else v = bd.mleaf[c];
      return v;
    };
    auto prepare = [&]() {
      if (!(im[0] | im[1])) {
        nk = n;
        return;
      }
      uint32_t i;
      if (im[0]) {
        i = (uint32_t)__builtin_ctzll(im[0]);
        nk = lane_read(kk[0], i);
      } else {
        i = (uint32_t)__builtin_ctzll(im[1]);
        nk = lane_read(kk[1], i);
        i += CPX_WAVE;
      }
      is = lane_read(istk, nk);
      ie = nk + 1 < n ? lane_read(istk, nk + 1 < CPX_WAVE ? nk + 1 : 0u) : ni;
      if (GS == 1) {
        ntot = lane_read(in[0], is);
        ml = lane_read(ia[0], is);
        im[0] &= im[0] - 1;
      } else {
        const uint32_t src = is + lane;
        const uint32_t n0 = lane_get(in[0], src & 63u), m0 = lane_get(ia[0], src & 63u);
        uint32_t nl = n0;
        ml = m0;
        if (ie > CPX_WAVE) {
          const uint32_t n1 = lane_get(in[1], src & 63u), m1 = lane_get(ia[1], src & 63u);
          if (src >= CPX_WAVE) { nl = n1; ml = m1; }
        }
        if (src >= ie) nl = 0;
        my_hi = wave_incl_scan(nl);
        my_lo = my_hi - nl;
        ntot = lane_read(my_hi, CPX_WAVE - 1);
        // the stage's items are done
        im[0] = ie >= CPX_WAVE ? 0ull : im[0] >> ie << ie;
        if (ie > CPX_WAVE) im[1] = ie >= 2 * CPX_WAVE ? 0ull : im[1] >> (ie - CPX_WAVE) << (ie - CPX_WAVE);
      }
      const uint32_t f = rep * CPX_WAVE + lane;
      uint32_t c = entry(f, fi);
      if (f < ntot) pf = fetch(fi, c);
    };
    prepare();

    uint32_t dwk = 0;                                   // the wave's removals of stage k, in lane k
    auto removed = [&](uint32_t k, uint32_t wd) {
      wcur -= wd;
      dwk = lane == k ? wd : dwk;
    };
    // first multiples as bits of the segment, class by class: of the eight
    // stages from 8 fg (fj) and from 8 fg + 8 (fn), stage (lane >> 3), class lane & 7
    uint32_t fg = 0, fj, fn;
    auto firsts = [&](uint32_t g) {
      const uint32_t st = 8 * g + (lane >> 3), ac = lane_get(ack, st);
      return cl.first(ac >> 6, ac & 63u, 8 * lane_get(pk, st), lane_get(d8k, st)) + wbit;
    };
    fj = firsts(0);
    fn = firsts(1);
    // this lane's first multiple of the primes of stages k, k + 1, .. (at most eight)
    auto first_of = [&](uint32_t k, uint32_t count, uint32_t *j) {
      while (k >> 3 > fg) {
        fg++;
        fj = fn;
        fn = firsts(fg + 1);
      }
#pragma unroll
      for (uint32_t u = 0; u < count; u++)
        j[u] = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(4 * (lane & 7u) + 32 * ((k + u) & 7u)),
                                                      (int)((k + u) >> 3 > fg ? fn : fj));
#pragma unroll
      for (uint32_t u = 0; u < count; u++) j[u] += __umul24(lane >> 3, 8 * lane_read(pk, k + u));
    };
    // one multiple j: whether its bit (m) was still set, taken off its quarter's count
    auto hit = [&](uint32_t j, uint32_t m, uint32_t old) {
      const bool h = (old & m) != 0;
      const uint64_t all = __builtin_amdgcn_ballot_w64(h);
      if (h) atomicSub(&sh.cnt[j >> 10], 1u << ((j >> 5) & 24u));
      return all;
    };
    for (uint32_t k = 0; k < n;) {
      const uint32_t p = lane_read(pk, k);
      if (!counted && p >= HARD_RECOUNT_P) {            // from here on removals are counted one by one
#pragma unroll
        for (uint32_t u = 0; u < UPT; u++) sh.cnt[t * UPT + u] = cr[u];
        counted = true;
      }
      if (k == nk) {
        // ---- leaves of p whose n falls in this wave's bits (state: crossed
        //      by p_1 .. p_{b-1}), all members' in one list; the wave
        //      publishes its own prefix, no other wave is involved
        int64_t as = 0;                                 // this item lane's sums (GS > 1)
        int32_t ws = 0;                                 // sum of mu: the item lane's, or the wave's (GS = 1)
        if (ntot > rep * CPX_WAVE) {
#pragma unroll
          for (uint32_t u = 0; u < UPT; u++) {
            if (counted) cr[u] = sh.cnt[t * UPT + u];
            else sh.cnt[t * UPT + u] = cr[u];
          }
          (void)publish_units<(int)UPT>(cr, sh.ipre);
          for (uint32_t fb = rep * CPX_WAVE; fb < ntot; fb += cstep) {   // every lane runs every window
            const uint32_t f = fb + lane;
            if (fb != rep * CPX_WAVE) {
              const uint32_t c = entry(f, fi);
              if (f < ntot) pf = fetch(fi, c);
            }
            int32_t val = 0, sg = 0;
            if (f < ntot) {
              if (sh.ccnt[fi] & HARD_SPARSE) {
                sg = -1;                                        // a prime
              } else {                                          // mu(m) = 0 or lpf(m) <= p: no leaf
                const uint32_t av = (uint32_t)(pf.y < 0 ? -pf.y : pf.y);
                sg = av <= p ? 0 : (pf.y > 0 ? 1 : -1);
              }
              if (sg) {
                const uint64_t xp = sh.xp[fi];
                const double xpf = (double)xp + (double)sh.xph[fi] * 0x1p64;
                const uint64_t nn = cpx_div_leaf(xp, xpf, (uint32_t)pf.x);   // lo_w <= nn < hi_w
                const uint32_t bits = cop30_upto((uint32_t)nn - (uint32_t)lo_w);   // 0 .. WB
                const uint32_t ct = unit_count_to(lds, sh.ipre, sh.cnt, max(bits, 1u) - 1 + wbit);
                const int32_t cn = bits ? (int32_t)ct : 0;
                val = sg > 0 ? cn : -cn;
              }
            }
            if (GS == 1) {
              acc += val;
              ws += (int32_t)__popcll(__ballot(sg > 0)) - (int32_t)__popcll(__ballot(sg < 0));
            } else {
              hard_lane_accumulate<K>(val, sg, fb, my_lo, my_hi, as, ws);
            }
          }
          if (GS == 1) {
            if (lane == 0) sh.wm[is][wv] = ws;
          } else if (is + lane < ie) {
            const uint32_t i = is + lane;
            sh.wm[i][wv] = ws;
            if (as) atomicAdd((unsigned long long *)&sh.acc[wv][sh.kg[i] & 31u], (unsigned long long)as);
          }
        }
        prepare();
      }
      // ---- cross off the multiples of p in the wave's bits, and of the
      //      stages after it that have no leaves here: with at most one multiple
      //      per lane four stages go together, the LDS taking the wave's
      //      operations in order, so that their round trips overlap
      const uint32_t kend = min(nk, n);                 // (> k)
      const uint32_t jend = wbit + WB;
      if (64 * p >= WB) {
        for (; k + 3 < kend; k += 4) {
          uint32_t j[4], m[4], old[4];
          first_of(k, 4, j);
#pragma unroll
          for (uint32_t u = 0; u < 4; u++) {
            m[u] = 1u << (j[u] & 31u);
            old[u] = 0;
            if (j[u] < jend) old[u] = atomicAnd(unit_word(lds, j[u]), ~m[u]);
          }
          // the four stages' removals (below 2^16) to lanes k .. k + 3
          uint64_t wd4 = 0;
#pragma unroll
          for (uint32_t u = 0; u < 4; u++) {
            const uint32_t wd = (uint32_t)__popcll(hit(j[u], m[u], old[u]));
            wcur -= wd;
            wd4 |= (uint64_t)wd << (16 * u);
          }
          const uint32_t to = lane - k;
          dwk = to < 4 ? (uint32_t)(wd4 >> (16 * to)) & 0xffffu : dwk;
        }
        for (; k < kend; k++) {
          uint32_t j, old = 0;
          first_of(k, 1, &j);
          const uint32_t m = 1u << (j & 31u);
          if (j < jend) old = atomicAnd(unit_word(lds, j), ~m);
          removed(k, (uint32_t)__popcll(hit(j, m, old)));
        }
        continue;
      }
      const uint32_t p64 = 64 * p;                      // (64 p bits: whole words, so a lane keeps its bit)
      uint32_t j, wd;
      first_of(k, 1, &j);
      const uint32_t m = 1u << (j & 31u);
      if (p < HARD_RECOUNT_P) {
        const uint32_t p2 = 2 * p, we = jend >> 5;
        uint32_t w = j >> 5;
        for (; w + 3 * p2 < we; w += 4 * p2) {
          const uint32_t w1 = w + p2, w2 = w1 + p2, w3 = w2 + p2;
          atomicAnd(&lds[w + (w >> 5)], ~m);
          atomicAnd(&lds[w1 + (w1 >> 5)], ~m);
          atomicAnd(&lds[w2 + (w2 >> 5)], ~m);
          atomicAnd(&lds[w3 + (w3 >> 5)], ~m);
        }
        for (; w < we; w += p2) atomicAnd(&lds[w + (w >> 5)], ~m);
        uint32_t s = 0;
#pragma unroll
        for (uint32_t u = 0; u < UPT; u++) {
          cr[u] = unit_counts(lds + (t * UPT + u) * 33);
          s += unit_total(cr[u]);
        }
        wd = wcur - wave_sum(s);
      } else {
        // (every lane takes every step: the ballots count the removals)
        wd = 0;
        const uint32_t steps = (WB + p64 - 1) / p64;    // (first multiples are below 64 p)
        for (uint32_t i = 0; i < steps; i += 2, j += 2 * p64) {
          const uint32_t j1 = j + p64;
          uint32_t o0 = 0, o1 = 0;
          if (j < jend) o0 = atomicAnd(unit_word(lds, j), ~m);
          if (j1 < jend) o1 = atomicAnd(unit_word(lds, j1), ~m);
          wd += (uint32_t)__popcll(hit(j, m, o0));
          wd += (uint32_t)__popcll(hit(j1, m, o1));
        }
      }
      removed(k, wd);
      k++;
    }
    if (lane < n) sh.dw[lane][wv] = (uint16_t)dwk;
    hard_flush<T, K, GS>(bd, sh, s0, n, ni, kk, running, rep == 0, acc);
    s0 += n;
  }
  if (GS == 1) {
    const long long a = wave_sum((long long)acc);
    if (lane == 0) sh.acc[wv][0] = a;
  }
}

// One tile: segment `seg` of a group, replica `rep` of `nrep`.  The wheel
// and the stage primes sieve the segment once; every member's leaves are
// evaluated against that one bitmap.
template <int T, int K>
__device__ __forceinline__ void hard_segment(const BatchDev &bd, const TileDev &tile, uint32_t *lds,
                                             SegShared<T, K> &sh)
{
  constexpr uint32_t NW = T / CPX_WAVE, G = CPX_GROUP, SB = 32u * K * T;
  const uint32_t t = own_thread();
  const uint64_t seg = tile.seg;
  const uint64_t lo = seg * (SB / 8 * 30), hi = lo + SB / 8 * 30;
  const GroupDev &grp = bd.groups[tile.group];
  const uint32_t rep = tile.rep;
  const uint32_t cs = bd.queries[grp.q[0]].cs;          // members share the wheel
  const WheelInfo wi = bd.winfo[cs];
  // members' rows of this segment: counters of the active stages only (the
  // plan sized each row for ri.act stages)
  for (uint32_t g = t; g < G; g += T) {
    GroupMember m{};
    if (g < grp.n) {
      const QueryDev &q = bd.queries[grp.q[g]];
      if (seg < q.hard_nseg) {
        const HardRowInfo ri = bd.rowinfo[q.hard_row0 + seg];
        m.y = (uint32_t)q.y;
        m.stage_off = q.stage_off;
        m.toff = q.tm_off + ri.toff - bd.pass_toff;
        m.moff = q.m_off + ri.moff - bd.pass_moff + (uint64_t)rep * ri.act;
        m.nst = min(q.nstage, ri.act);
        m.on = 1u | (seg >= q.p2_seg0 && seg < q.p2_seg0 + q.p2_nseg ? 2u : 0u);
      }
    }
    sh.gm[g] = m;
  }
  for (uint32_t i = t; i < NW * G; i += T) (&sh.acc[0][0])[i] = 0;
  const uint32_t cstep = CPX_WAVE * (uint32_t)tile.nrep;   // candidate stride of a lane

  {
    // segment word w is pattern word (seg * words + w) mod period; the index
    // steps by T mod period instead of a division per word, so the loads of
    // the unrolled loop go out together
    const uint32_t *__restrict__ pat = reinterpret_cast<const uint32_t *>(bd.wheel + wi.pat_off);
    const uint32_t P = wi.pat_period, step = (uint32_t)T % P;
    uint32_t idx = (uint32_t)((seg * (uint64_t)(SB / 32) + t) % P);
#pragma unroll 8
    for (uint32_t w = t; w < SB / 32; w += T) {
      lds[w + (w >> 5)] = pat[idx];
      idx += step;
      if (idx >= P) idx -= P;
    }
  }
  __syncthreads();
  uint32_t nst = 0, p2any = 0;                          // stages of the segment: the members' most
  for (uint32_t g = 0; g < grp.n; g++) { nst = max(nst, sh.gm[g].nst); p2any |= sh.gm[g].on & 2u; }
  nst = (uint32_t)__builtin_amdgcn_readfirstlane((int)nst);
  if (grp.n == 1) hard_chunks<T, K, 1>(bd, sh, lds, cs, nst, rep, cstep, lo, hi);
  else if (grp.n <= 8) hard_chunks<T, K, 8>(bd, sh, lds, cs, nst, rep, cstep, lo, hi);
  else hard_chunks<T, K, 32>(bd, sh, lds, cs, nst, rep, cstep, lo, hi);
  __syncthreads();
  for (uint32_t g = t; g < grp.n; g += T) {
    if (!(sh.gm[g].on & 1u)) continue;
    const QueryDev &q = bd.queries[grp.q[g]];
    const uint64_t row = q.hard_row0 + seg;
    long long tt = 0;
    for (uint32_t w = 0; w < NW; w++) tt += sh.acc[w][g];
    st_out(&bd.hard_acc[q.mrow_base + bd.rowinfo[row].mrow + rep], (int64_t)tt);
  }
  if (p2any) p2_epilogue<T, K>(bd, grp, seg, rep, tile.nrep, lo, cs + nst, lds, sh);
}

// Easy leaves (replaces S2_a / V_a / V_b, src/Deleglise-Rivat/S2.cu:72-99,
// src/V.cu:22-124) of one descriptor, as a tile of the persistent kernel:
//   V = sum_{x^(1/4) < p <= cbrt x} sum_{p < q <= min(y, x/p^2)} [pi(x/pq) - pi(p) + 2]
// over the descriptor's primes p = primes[j], j in [begin, end) (all these
// leaves have x/pq < p^2).  The block sets up T primes at a time in parallel
// (x/p, the q range, the (2 - pi(p)) terms), then strides its threads over
// each prime's q's with U = 4 independent prime -> quotient -> pi-table
// chains per thread.  Uses the first 5T words of the segment LDS.
//
// Where the q's pass s = floor(sqrt(x/p)), those above it need no lookups of
// their own: with Q the upper end of the q's, counting the pairs of primes
// (q, r), s < q <= Q, r <= x/(pq), by r instead of by q gives
//   sum_{s < q <= Q} pi(x/pq) = sum_{r <= s} [pi(min(Q, x/pr)) - pi(s)]
//     = pi(R) (pi(Q) - pi(s)) + sum_{R < r <= s} [pi(x/pr) - pi(s)],  R = min(s, x/(pQ)),
// and every r in (R, s] is also a q of the range (R is at least its lower
// end: p <= x/(pQ) as Q <= x/p^2, and x/p^3 <= x/(pQ) where Q = y < p^2), so
// those lookups count twice.  The tiles are bound by the rate of divergent
// gathers, and at x = 1e18 this leaves about a third of them.  Solves with it, before
// and after: 1e16 5.40 -> 4.92 ms, 1e18 97.2 -> 79.1 ms, 2e19 799 -> 657 ms;
// where y <= sqrt(x/p) for most p (512 queries to 1e15) nothing changes.
template <int T, int K>
__device__ __forceinline__ void easy_tile(const BatchDev &bd, uint32_t di, uint32_t *lds, SegShared<T, K> &sh)
{
  constexpr uint32_t U = 4;
  constexpr uint32_t SBT = T < 256 ? T : 256, SUB = T / SBT, BIG = 8 * U * T;
  uint64_t *sxp = reinterpret_cast<uint64_t *>(lds);    // x / p of the chunk's primes
  uint32_t *sk1 = lds + 2 * T;                          // pi(min(y, x / p^2)): q indices end here
  uint32_t *sk0 = lds + 3 * T;                          // max(j + 1, pi(x / p^3)): and start here
  uint32_t *skr = lds + 4 * T;                          // and from here on count twice
  const uint32_t t = own_thread();
  const BlockDesc d = bd.easy_desc[di];
  const QueryDev &q = bd.queries[d.query];
  const u128 x = ((u128)q.x_hi << 64) | q.x_lo;
  // a descriptor of hard leaves (its part in the hard group) adds mu * phi
  const bool hard = d.part >= q.n_ord_parts + q.n_triv_parts + q.n_easy_parts;
  i128 sum = 0;
  for (uint64_t j0 = d.begin; j0 < d.end; j0 += T) {
    const uint32_t nj = (uint32_t)min((uint64_t)T, d.end - j0);
    if (t < nj) {
      const uint64_t j = j0 + t;
      const uint64_t p = bd.primes[j];
      const uint64_t xp = cpx_div128_to64(x, p);
      // every bound first, then their table entries in one round trip
      const uint64_t v = (xp >> 50) < p ? cpx_div_smallq(xp, p) : xp / p;
      const uint64_t qmax = min(q.y, v);
      // q > x/p^3 (x/(pq) < p^2): no bound above x^(1/4), where x/p^3 < p
      uint64_t t3 = p;
      if (hard) t3 = max(p, min(q.y, (v >> 50) < p ? cpx_div_smallq(v, p) : v / p));
      const uint64_t s = min(isqrt64_dev(xp), qmax);
      const uint64_t R = min(s, cpx_div_smallq(xp, qmax));     // x/(p y) <= z < 2^50, or about p
      const uint64_t k1 = pi_lookup(bd.pitab, qmax), ks = pi_lookup(bd.pitab, s);
      const uint64_t kR = pi_lookup(bd.pitab, R), k3 = pi_lookup(bd.pitab, t3);
      const uint64_t k0 = max(j + 1, k3);
      uint64_t kend = k1, kr = k1;
      if (k1 > k0) {
        sum += (i128)(k1 - k0) * (1 - (i128)j);                // (2 - pi(p)) per q, pi(p) = j + 1
        if (s < qmax && ks > k0) {
          kend = ks;
          kr = kR;
          sum += (i128)(kr * (k1 - ks)) - (i128)(ks * (ks - kr));
        }
      }
      sxp[t] = xp;
      sk1[t] = (uint32_t)kend;
      sk0[t] = (uint32_t)k0;
      skr[t] = (uint32_t)kr;
    }
    __syncthreads();
    // primes with at least BIG q's take the whole block one at a time (U * T
    // slots per step); the others go to sub-blocks of SBT threads, every SUB-th
    // prime to one sub-block (U * SBT slots per step: fewer idle lanes in a
    // prime's last step)
    for (uint32_t pass = 0; pass < 2; pass++) {
      const uint32_t nthr = pass ? SBT : T, stride = U * nthr, tl = pass ? t % SBT : t;
      for (uint32_t jj = pass ? t / SBT : 0; jj < nj; jj += pass ? SUB : 1) {
        const uint64_t kend = sk1[jj], kbeg = sk0[jj], xp = sxp[jj];
        if (kend <= kbeg || ((kend - kbeg >= BIG) != (pass == 0))) continue;
        // a chain past k1 repeats index k and is masked; x/(p q) < x/p^2 <
        // 2^50, so the reciprocal divide with the tabulated 1/q is exact
        const double xpf = (double)xp;
        const uint64_t kr = min(kend, (uint64_t)skr[jj]);
        uint64_t s = 0;
        // the q's that count twice, then those that count once
        for (uint32_t once = 0; once < 2; once++) {
          const uint64_t k0 = once ? kbeg : kr, k1 = once ? kr : kend;
          s += s;
          for (uint64_t k = k0 + tl; k < k1; k += stride) {
            uint32_t qv[U];
            double rv[U];
            bool ok[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
              ok[u] = k + u * nthr < k1;
              const uint64_t kk = ok[u] ? k + u * nthr : k;
              qv[u] = bd.primes[kk];
              rv[u] = bd.prinv[kk];
            }
            PiEntry pe[U];
            uint32_t ix[U];
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
              const uint64_t v = cpx_div_leaf_r(xp, xpf, qv[u], rv[u]);
              ix[u] = (uint32_t)(((v & 63) + 1) >> 1) | (v >= 2 ? 0x80u : 0u);
              pe[u] = bd.pitab[v >> 6];
            }
#pragma unroll
            for (uint32_t u = 0; u < U; u++) {
              const uint32_t c = (ix[u] >> 7) + pe[u].count + cpx_popc32(pe[u].bits & cpx_lowmask32(ix[u] & 63));
              s += ok[u] ? c : 0u;
            }
          }
        }
        sum += (i128)s;
      }
    }
    __syncthreads();
  }
  // block sum: wave sums, then wave 0 adds them
  sum = wave_sum_i128(sum);
  i128 *red = reinterpret_cast<i128 *>(lds);
  if (lane_id() == 0) red[wave_id()] = sum;
  __syncthreads();
  if (t == 0) {
    i128 tot = 0;
    for (uint32_t w = 0; w < T / CPX_WAVE; w++) tot += red[w];
    st_out(&bd.parts[q.part_off + d.part], hard ? -tot : tot);
  }
  (void)sh;
}

// P2 by lookups (replaces the windowed upper_bound count of src/P2.cu:76-133)
// for one descriptor, as a tile of the persistent kernel: the sum of
// pi(x/p) over P2 primes p = primes[k], k in [begin, end) (y < p <= sqrt x,
// x < 2^64), x/p by the reciprocal divide with the tabulated 1/p (x/p <=
// x/(y+1) < 2^50), pi from the resident table, which reaches x/(y+1); four
// independent chains per thread.  k_combine subtracts sum (pi(p) - 1) in
// closed form.  Uses the first T/16 words of the segment LDS.
template <int T, int K>
__device__ __forceinline__ void p2tab_tile(const BatchDev &bd, uint32_t di, uint32_t *lds)
{
  constexpr uint32_t U = 4;
  const uint32_t t = own_thread();
  const BlockDesc d = bd.p2_desc[di];
  const QueryDev &q = bd.queries[d.query];
  const uint64_t x = q.x_lo;
  const double xf = (double)x;
  uint64_t s = 0;
  for (uint64_t k = d.begin + t; k < d.end; k += U * T) {
    uint64_t v[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint64_t kk = k + u * T < d.end ? k + u * T : k;
      v[u] = cpx_div_leaf_r(x, xf, bd.primes[kk], bd.prinv[kk]);
    }
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      const uint64_t c = pi_lookup(bd.pitab, v[u]);
      s += k + u * T < d.end ? c : 0u;
    }
  }
  const uint64_t ws = wave_sum(s);
  uint64_t *red = reinterpret_cast<uint64_t *>(lds);
  if (lane_id() == 0) red[wave_id()] = ws;
  __syncthreads();
  if (t == 0) {
    i128 tot = 0;
    for (uint32_t w = 0; w < T / CPX_WAVE; w++) tot += (i128)red[w];
    st_out(&bd.parts[q.part_off + d.part], (i128)tot);
  }
}

