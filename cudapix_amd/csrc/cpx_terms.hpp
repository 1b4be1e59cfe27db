// cpx_terms.hpp -- block-level bodies of the cheap terms, the hard-leaf
// carry and the per-query combine, shared by their grid-stride kernels
// (terms.hip) and by the streaming kernel, which runs them as tiles.  Every
// function is written for a block of NT threads (a multiple of 64) and takes
// its LDS scratch from the caller.
#pragma once
#include "cpx_device.hpp"

// ----------------------------------------------------------- ordinary
// S0 = sum over odd n <= y with lpf(n) > p_c of mu(n) * phi(x/n, c),
// phi(u, c) = floor(u / W_c) * totient(W_c) + phi(u mod W_c, c)
// (src/ordinary.cu:101-115 and :118-135 for 128-bit x).  Items: odd index i,
// n = 2i + 1.  Returns this thread's share of descriptor d.
template <uint32_t NT>
__device__ __forceinline__ i128 ordinary_part(const BatchDev &bd, const BlockDesc &d, uint32_t t)
{
  const QueryDev &q = bd.queries[d.query];
  const u128 x = ((u128)q.x_hi << 64) | q.x_lo;
  const WheelInfo wi = bd.winfo[q.c];
  const PiEntry *wh = bd.wheel + wi.off;
  i128 sum = 0;
  for (uint64_t i = d.begin + t; i < d.end; i += NT) {
    int32_t v = bd.mlpf[i];
    uint32_t av = (uint32_t)(v < 0 ? -v : v);
    if (av <= wi.pc) continue;
    uint64_t n = 2 * i + 1;
    uint64_t rr;
    u128 m = cpx_div128_64(x, n, &rr);
    uint64_t r;
    u128 k = cpx_div128_64(m, wi.W, &r);
    uint32_t kk = (uint32_t)((r + 1) >> 1);
    PiEntry e = wh[kk >> 5];
    uint64_t ph = e.count + cpx_popc32(e.bits & cpx_lowmask32(kk & 31u));
    i128 phi = (i128)(k * wi.totient) + (i128)ph;
    sum += v > 0 ? phi : -phi;
  }
  return sum;
}

// ------------------------------------------- hard leaves of wheel stages
// The segment sieve starts from the wheel of the first q.cs primes; the hard
// leaves of the stages c < b <= cs, p = p_b, need no sieve: with b - 1 <= 7
// primes below p, phi(x/(p m), b - 1) is the wheel's closed form, as in the
// ordinary leaves.  This thread's share of
//   sum over odd m of d, m > y/p, lpf(m) > p of mu(m) phi(x/(p m), b - 1).
// Bound by the integer divides (a 128/64 one per m, two per leaf).
template <uint32_t NT>
__device__ __forceinline__ i128 direct_part(const BatchDev &bd, const BlockDesc &d, uint32_t t)
{
  const QueryDev &q = bd.queries[d.query];
  const u128 x = ((u128)q.x_hi << 64) | q.x_lo;
  const uint32_t p0 = bd.primes[q.c];
  i128 sum = 0;
  for (uint64_t i = d.begin + t; i < d.end; i += NT) {
    const int32_t v = bd.mlpf[i];
    const uint32_t av = (uint32_t)(v < 0 ? -v : v);
    if (av <= p0) continue;
    const uint64_t m = 2 * i + 1;
    uint64_t r;
    const u128 u = cpx_div128_64(x, m, &r);
    i128 s = 0;
    for (uint32_t b = q.c; b < q.cs; b++) {
      const uint32_t p = bd.primes[b];
      if (av <= p) break;
      if (m * p <= q.y) continue;
      const WheelInfo wi = bd.winfo[b];
      const u128 k = cpx_div128_64(cpx_div128_64(u, p, &r), wi.W, &r);
      const uint32_t kk = (uint32_t)((r + 1) >> 1);
      const PiEntry e = bd.wheel[wi.off + (kk >> 5)];
      s += (i128)(k * wi.totient) + (i128)(e.count + cpx_popc32(e.bits & cpx_lowmask32(kk & 31u)));
    }
    sum += v > 0 ? s : -s;
  }
  return sum;
}

// ------------------------------------------------------------ trivial U
// U = sum over primes sqrt(z) < p <= cbrt(x) of [pi(y) - pi(x / p^2)]
// (src/trivial.cu:31-62).  Items: prime index i (p = primes[i]).
template <uint32_t NT>
__device__ __forceinline__ i128 trivial_part(const BatchDev &bd, const BlockDesc &d, uint32_t t)
{
  const QueryDev &q = bd.queries[d.query];
  const u128 x = ((u128)q.x_hi << 64) | q.x_lo;
  i128 sum = 0;
  for (uint64_t i = d.begin + t; i < d.end; i += NT) {
    uint64_t p = bd.primes[i];
    uint64_t qq = cpx_div128_to64(x, p * p);    // < y
    sum += (i128)q.a - (i128)pi_lookup(bd.pitab, qq);
  }
  return sum;
}

// -------------------------------------------------------- hard carry
// Hard-leaf carry of stages [s0, s0 + ns) (ns <= CPX_FIN_STAGES) of one
// query: for each of them
//   carry_s = sum over segments r (in order, while s is active in r) of
//             msum_s(r) * (T_s(0) + ... + T_s(r-1))
// with msum_s(r) the replicas' sum(mu) of the leaves of p_s in segment r and
// T_s(r) its survivors before stage s.  Activity is a prefix of the segments;
// the descriptor says how many rows stage s0 is active in (begin = s0 | rows << 32).
// The block's threads are FIN_STAGES columns by NT / FIN_STAGES runs of
// consecutive rows: a thread walks its run for one stage, adding up T, msum and
// msum times the T's before it in the run; the runs' totals of T then give each
// run's base.  Bound by the latency of a run's chain of row records and entries:
// four rows are in flight and the next four records are fetched ahead.  With
// one row per thread and a scan over the block for every 128 rows the carry
// took 830 us of a 512-query batch to 1e15, 230 us at 1e16 and 2.8 ms at 1e18.
template <uint32_t NT>
struct FinShared {
  i128 red[NT / CPX_WAVE];
  unsigned long long run[NT];      // survivors of a run, by stage
};

// Writes the descriptor's carry to bd.parts; every thread of the block calls it.
// In a run in passes it takes the pass's rows only, starts each stage's
// prefix from hard_base (the survivors of the earlier passes' segments),
// writes the advanced totals back, and adds to the partial sum after the
// first pass: the stages' carries over the passes then sum to the one-launch carry.
template <uint32_t NT>
__device__ __forceinline__ void hard_fin_desc(const BatchDev &bd, const BlockDesc &d, FinShared<NT> &fs)
{
  constexpr uint32_t FS = CPX_FIN_STAGES, RUNS = NT / FS, U = 4;
  const uint32_t t = threadIdx.x, j = t % FS, run = t / FS;
  const QueryDev &q = bd.queries[d.query];
  const uint32_t s = (uint32_t)d.begin + j;
  const bool on = s < d.end;
  const uint64_t r_lo = bd.pass_r0, r_hi = min(d.begin >> 32, bd.pass_r1);
  const uint64_t per = r_hi > r_lo ? (r_hi - r_lo + RUNS - 1) / RUNS : 0;
  const uint64_t ra = r_lo + run * per, rb = min(ra + per, r_hi);
  const HardRowInfo *__restrict__ info = bd.rowinfo + q.hard_row0;
  const uint32_t *__restrict__ T = bd.hard_T + (q.tm_off - bd.pass_toff) + s;
  const int32_t *__restrict__ M = bd.hard_M + (q.m_off - bd.pass_moff) + s;
  unsigned long long pre = 0;
  long long ms = 0;
  i128 carry = 0;
  HardRowInfo ri[U];
  auto fetch = [&](uint64_t r) {
#pragma unroll
    for (uint32_t u = 0; u < U; u++)
      if (r + u < rb) ri[u] = info[r + u];
      else ri[u].act = 0;
  };
  if (on) fetch(ra);
  for (uint64_t r = ra; on && r < rb && s < ri[0].act; r += U) {
    HardRowInfo c[U];
    uint32_t tv[U];
    long long m[U];
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      c[u] = ri[u];
      tv[u] = 0;
      m[u] = 0;
      if (s < c[u].act) {
        tv[u] = T[c[u].toff];
        m[u] = M[c[u].moff];
      }
    }
    fetch(r + U);
#pragma unroll
    for (uint32_t u = 0; u < U; u++) {
      if (s < c[u].act)
        for (uint32_t k = 1; k < c[u].nrep; k++) m[u] += M[c[u].moff + (uint64_t)k * c[u].act];
      carry += (i128)pre * m[u];
      pre += tv[u];
      ms += m[u];
    }
  }
  fs.run[t] = pre;
  // (read before the barrier: the last run's threads advance it after theirs)
  unsigned long long base = bd.hard_base && on ? bd.hard_base[s] : 0ull;
  __syncthreads();
  for (uint32_t k = 0; k < run; k++) base += fs.run[k * FS + j];
  carry += (i128)base * ms;
  if (bd.hard_base && on && run == RUNS - 1) bd.hard_base[s] = base + pre;
  __syncthreads();
  i128 tt = block_sum_i128(carry, fs.red);
  if (t == 0) {
    i128 *out = &bd.parts[q.part_off + d.part];
    st_out(out, bd.pass_add ? *out + tt : tt);
  }
}

// ------------------------------------------------------------- combine
// One query: P2 carry scan over P2 segments, hard local sums, then
//   pi = S0 + (S1 + U) + V + S3 + pi(y) - 1 - P2
// (src/Deleglise-Rivat/deleglise-rivat.cpp:77).  With table_pi the query's
// pi(sqrt x) and pi(p2_e) are read from the pi table here instead of from
// the record (the streaming path has no setup kernel).
template <uint32_t NT>
struct CombShared {
  i128 red[5][NT / CPX_WAVE];
  i128 sum[5];
  uint64_t wtot[NT / CPX_WAVE];
};

static __device__ __forceinline__ void put_i128(uint64_t out[2], i128 v)
{
  out[0] = (uint64_t)v;
  out[1] = (uint64_t)((u128)v >> 64);
}

// A result record, written word by word with system-scope coherence: the
// streaming kernel's results live in pinned host memory that the host reads
// while the kernel still runs.
static __device__ __forceinline__ void st_result(ResultDev *dst, const ResultDev &r)
{
  const uint64_t *src = reinterpret_cast<const uint64_t *>(&r);
  uint64_t *d = reinterpret_cast<uint64_t *>(dst);
  for (uint32_t k = 0; k < sizeof(ResultDev) / 8; k++)
    __hip_atomic_store(d + k, src[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <uint32_t NT>
__device__ __forceinline__ void combine_query(const BatchDev &bd, uint32_t qi, CombShared<NT> &cs,
                                              bool table_pi)
{
  const uint32_t t = threadIdx.x;
  const QueryDev &q = bd.queries[qi];
  const uint64_t pi_e = table_pi ? pi_lookup(bd.pitab, q.p2_e) : q.pi_e;
  const uint64_t pi_sqrtx = table_pi ? pi_lookup(bd.pitab, q.sqrtx) : q.pi_sqrtx;
  // P2: sum over segments of loc + np * (pi(p2_e) + primes in earlier segments),
  // a run of consecutive segments a thread, then the runs' totals.  (A latency
  // chain: four rows in flight.  At 1e18, one row a thread and a scan for every
  // 256 rows, each a chain of its own, took 430 us.)
  i128 p2 = 0;
  {
    constexpr uint32_t U = 4;
    const uint64_t per = (q.p2_nseg + NT - 1) / NT, ra = per * t, rb = min(ra + per, q.p2_nseg);
    const HardRowInfo *__restrict__ info = bd.rowinfo + q.hard_row0 + q.p2_seg0;
    const uint32_t *__restrict__ cnt = bd.p2_cnt + q.p2_row0, *__restrict__ nps = bd.p2_np + q.mrow_base;
    const uint64_t *__restrict__ locs = bd.p2_loc + q.mrow_base;
    uint64_t pre = 0, nsum = 0;
    for (uint64_t r = ra; r < rb; r += U) {
      uint32_t mr[U], nr[U];
      uint64_t c[U], np[U], loc[U];
#pragma unroll
      for (uint32_t u = 0; u < U; u++) {
        const bool in = r + u < rb;
        mr[u] = in ? info[r + u].mrow : 0u;
        nr[u] = in ? info[r + u].nrep : 0u;
        c[u] = in ? cnt[r + u] : 0u;
      }
#pragma unroll
      for (uint32_t u = 0; u < U; u++) {
        np[u] = nr[u] ? nps[mr[u]] : 0u;
        loc[u] = nr[u] ? locs[mr[u]] : 0ull;
      }
#pragma unroll
      for (uint32_t u = 0; u < U; u++) {
        for (uint32_t k = 1; k < nr[u]; k++) { np[u] += nps[mr[u] + k]; loc[u] += locs[mr[u] + k]; }
        p2 += (i128)loc[u] + (i128)np[u] * pre;
        pre += c[u];
        nsum += np[u];
      }
    }
    const uint64_t incl = wave_incl_scan(pre);
    if (lane_id() == CPX_WAVE - 1) cs.wtot[wave_id()] = incl;
    __syncthreads();
    uint64_t base = pi_e + incl - pre;
    for (uint32_t w = 0; w < wave_id(); w++) base += cs.wtot[w];
    p2 += (i128)nsum * base;
  }
  // hard: local sums
  i128 hacc = 0;
#pragma unroll 4
  for (uint64_t r = t; r < q.hard_nmrow; r += NT) hacc += bd.hard_acc[q.mrow_base + r];
  if (t == 0 && q.small) {
    ResultDev res;
    i128 pi = (i128)pi_lookup(bd.pitab, q.x_lo);
    put_i128(res.pi, pi);
    put_i128(res.ordinary, 0);
    put_i128(res.trivial, 0);
    put_i128(res.easy, 0);
    put_i128(res.hard, 0);
    put_i128(res.p2, 0);
    res.pi_y = q.a;
    res.status = 1;
    st_result(&bd.results[qi], res);
  }
  // the term partial sums, by term (ordinary | trivial U | easy | hard carry
  // | P2 lookups)
  i128 ps0 = 0, psu = 0, psv = 0, psh = hacc, psp = p2;
  if (!q.small) {
    const i128 *pp = bd.parts + q.part_off;
    const uint32_t n0 = q.n_ord_parts, n1 = n0 + q.n_triv_parts, n2 = n1 + q.n_easy_parts,
                   n3 = n2 + q.n_hard_parts, n4 = n3 + q.n_p2_parts;
#pragma unroll 2
    for (uint32_t i = t; i < n4; i += NT) {
      const i128 v = pp[i];
      if (i < n0) ps0 += v;
      else if (i < n1) psu += v;
      else if (i < n2) psv += v;
      else if (i < n3) psh += v;
      else psp += v;
    }
  }
  // the block's five sums behind one pair of barriers
  const i128 part[5] = {ps0, psu, psv, psh, psp};
#pragma unroll
  for (uint32_t j = 0; j < 5; j++) {
    const i128 s = wave_sum_i128(part[j]);
    if (lane_id() == 0) cs.red[j][wave_id()] = s;
  }
  __syncthreads();
  if (t < 5) {
    i128 s = 0;
    for (uint32_t w = 0; w < NT / CPX_WAVE; w++) s += cs.red[t][w];
    cs.sum[t] = s;
  }
  __syncthreads();
  if (t == 0 && !q.small) {
    const i128 s0 = cs.sum[0], u = cs.sum[1], v = cs.sum[2];
    // S1 = C(pi(y) - pi(cbrt x), 2)
    i128 kk = (i128)q.a - (i128)q.pi_cbrt;
    i128 s1 = kk > 0 ? kk * (kk - 1) / 2 : 0;
    i128 triv = s1 + u;
    i128 hard = -cs.sum[3];
    // P2 = sum pi(x/p) - sum_{p} (pi(p) - 1), pi(p) = a+1 .. A
    i128 A = (i128)pi_sqrtx, a = (i128)q.a;
    i128 P2 = 0;
    if (A > a) P2 = cs.sum[4] - (A * (A - 1) / 2 - a * (a - 1) / 2);
    i128 pi = s0 + triv + v + hard + a - 1 - P2;
    ResultDev res;
    put_i128(res.pi, pi);
    put_i128(res.ordinary, s0);
    put_i128(res.trivial, triv);
    put_i128(res.easy, v);
    put_i128(res.hard, hard);
    put_i128(res.p2, P2);
    res.pi_y = q.a;
    res.status = 1;
    st_result(&bd.results[qi], res);
  }
  __syncthreads();
}
