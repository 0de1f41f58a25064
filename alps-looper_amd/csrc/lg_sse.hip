// "loop; sse" (sse.C:174-400): the same loop clusters on the stochastic
// series expansion.  A chain's operator string (series order) is walked step
// by step: before each kept operator, and again after each insertion, a gap
// tries an insertion when (n + 1) u < beta W_tot (W_tot sums every location's
// graphs: lattice bonds, the single-ion term's in-site bonds, the transverse
// field's site operators; the location and graph from words 2 and 3, kept if
// compatible); a diagonal operator is removed when beta W_tot u < n (the next
// one follows with no gap between) or else regraphed by choose_diagonal
// (graph_impl.h:297-312); an off-diagonal one by choose_offdiagonal and
// flips its spins.  Step k of the walk takes the words
// Philox(sweep, 6, 0, k).  The new string then becomes bond-major operators
// at times p / n, on which the path-integral cluster stage runs unchanged
// (lengths in units of the string), and the flipped types return to the
// string.
#include <hip/hip_runtime.h>

#include "lg_common.h"
#include "lg_device.h"
#include "lg_kernels.h"

namespace lg {

namespace {
constexpr int SSE_THREADS = 64;
constexpr int SSE_NONE = 0xffff;   // no site
constexpr int SSE_MOST = 1 << 30;  // above every operator count

// ones of m from bit k on (at most 64 - k)
__device__ __forceinline__ int run_length(unsigned long long m, int k) {
  return (int)min((unsigned)__ffsll((long long)(~m >> k)) - 1u, (unsigned)(64 - k));
}
__device__ __forceinline__ int lane_of(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ int with_lane(int v, int l, int x) { return lane_id() == l ? x : v; }
}  // namespace

// The walk, one wave per chain.  A step's decision depends on the operator
// count and the spins that the steps before it leave, so the steps are
// serial; but the lanes hold what each of the next 64 steps would need -- the
// largest count n at which its insertion is tried, the smallest at which its
// removal succeeds, its location -- and each of the next 64 old operators,
// and the walk moves by whole runs: of insertions (up to the first step whose
// insertion fails, counting those before it into n), of removals (up to the
// first operator that stays or is off-diagonal).  A run is one compare per
// lane and a count of trailing ones, in scalar registers.  Which locations
// are compatible is a 64-bit mask that an off-diagonal operator updates by
// comparing its two sites with every lane's.  A lone wave is bound by the
// instructions it issues (about 6 clocks each), so the loop only notes where
// each lane's operator goes in the new string and which step's word decides
// its graph; the operators, the spins and the string follow for all lanes at
// once when the next 64 steps or operators come in.  One step at a time with
// words, sites and spins from LDS took 280 ns a step (16.7 ms for the coldest
// of 512 chains of 32^2, about 60000 steps); runs with every emitted
// operator stored in the loop 8.9 ms.
__global__ void __launch_bounds__(SSE_THREADS) k_sse_walk(DevBatch B) {
  if (blockIdx.x == 0 && threadIdx.x == 0) scan_advance_epoch(B);  // for k_scan, which follows
  if (__builtin_amdgcn_readfirstlane((int)overflowed(B))) return;  // (another chain may set it meanwhile: one answer a wave)
  const int c = blockIdx.x;
  const ChainDev& P = B.chains[c];
  __shared__ uint32_t spw[SSE_MAX_SITES / 32];            // spins, a bit each
  __shared__ int cnt[SSE_MAX_BONDS], off[SSE_MAX_BONDS];  // operators and off-diagonal ones stored per bond
  __shared__ uint32_t ends[SSE_MAX_BONDS];                // source | target << 16; a site operator's target SSE_NONE
  __shared__ int ring[2 * SSE_THREADS];                   // the last emitted operators, stored 64 at a time
  const int lane = threadIdx.x;
  const int Nb = P.Nb, nb_lat = P.nb_lat, nb_real = P.nb_real;
  for (int s0 = 0; s0 < P.N; s0 += 64) {
    const unsigned long long m = __ballot(s0 + lane < P.N && B.spins_old[P.old_site_base + min(s0 + lane, P.N - 1)]);
    if (lane == 0) spw[s0 >> 5] = (uint32_t)m;
    if (lane == 1) spw[(s0 >> 5) + 1] = (uint32_t)(m >> 32);
  }
  for (int b = lane; b < Nb; b += SSE_THREADS) {
    int s0, s1;
    op_sites(P, b, s0, s1);
    cnt[b] = off[b] = 0;
    ends[b] = (uint32_t)s0 | ((uint32_t)(b >= nb_real ? SSE_NONE : s1) << 16);
  }
  __syncthreads();
  auto spin_of = [&](int s) -> int { return (int)((spw[s >> 5] >> (s & 31)) & 1u); };
  const uint32_t sweep = B.sweep[c];
  const int n_old = __builtin_amdgcn_readfirstlane(B.bo_old[P.old_bond_base + Nb] - B.bo_old[P.old_bond_base]);
  const int* const so = B.sse_old + P.sse_base;
  int* const sn = B.sse_new + P.sse_base;
  int* const rank_at = B.sse_perm + P.sse_base;  // an emitted operator's number on its bond,
  int* const koff_at = B.l0 + P.sse_base;        // and the off-diagonal ones before it (scratch until the linking)
  const double bw = P.beta * P.sse_wtot;
  const int cap = P.sse_cap, nsite = P.N;
  const uint32_t key0 = P.key0, key1 = P.key1;
  // (values, not the descriptor: a choice between two of its fields would be
  // one between addresses, with the descriptor in scratch memory)
  const uint64_t toff = P.toff, dtoff = P.dtoff, pd0 = P.pdiag[0], pd1 = P.pdiag[1], dpd0 = P.dpdiag[0], dpd1 = P.dpdiag[1];
  const uint64_t cls0 = P.sse_cls[0], cls1 = P.sse_cls[1], tl0 = P.sse_tl[0], tl1 = P.sse_tl[1], tl2 = P.sse_tl[2];
  const uint64_t td0 = P.sse_td[0], td1 = P.sse_td[1], td2 = P.sse_td[2];
  int bits = 0;  // bits of a bond index
  while ((1 << bits) < Nb) ++bits;

  // the lanes' steps: step xbase + lane, the next one k
  int xbase = -SSE_THREADS, k = SSE_THREADS;
  int ins_at = 0, rem_at = 0;                // (see below)
  int z = 0;                                 // word 2
  int ne = 0, s0 = SSE_NONE, s1 = SSE_NONE;  // the insertion's operator and sites
  int pos_ins = -1;                          // its place in the new string, once inserted
  unsigned long long compat = 0;             // its location is compatible with the spins
  // the lanes' old operators: number obase + lane, the next one i of iend
  int obase = -SSE_THREADS, i = 0, iend = 0;
  int el = 0, q0 = SSE_NONE, q1 = SSE_NONE;
  int pos_op = -1, z_op = 0;                 // its place, once kept, and the word that decides its graph
  unsigned long long diag = 0;               // diagonal ones
  unsigned long long anti = 0;               // kept diagonal ones on an antiparallel pair
  int next_el = lane < n_old ? so[lane] : 0;
  int nop = n_old, out = 0, stored = 0;

  bool gap = true;

  while (true) {
    // ---- the next 64 steps, or the next 64 old operators (reached from the
    // walk below when either runs out) ----
    // the lanes' emitted operators go into the ring, the spins become up to date
    if (pos_ins >= 0) ring[pos_ins & (2 * SSE_THREADS - 1)] = ne;
    pos_ins = -1;
    if (pos_op >= 0) {
      const int b = el >> 3;
      const bool site = b >= nb_real, insite = b >= nb_lat && !site;
      const uint64_t zk = (uint32_t)z_op;
      int g;
      if (el & 1) {
        g = zk < (insite ? dtoff : toff) ? 0 : 1;
        atomicXor(&spw[q0 >> 5], 1u << (q0 & 31));
        if (!site) atomicXor(&spw[q1 >> 5], 1u << (q1 & 31));  // a site operator flips its one spin
      } else {
        const int cc = ((anti >> lane) & 1) ? 0 : 1;
        const uint64_t pd = insite ? (cc ? dpd1 : dpd0) : (cc ? pd1 : pd0);
        g = (zk < pd ? 0 : 2) ^ cc;
      }
      ring[pos_op & (2 * SSE_THREADS - 1)] = (b << 3) | (site ? 0 : g << 1) | (el & 1);
    }
    pos_op = -1;
    anti = 0;
    const bool end = out > cap || (!gap && i == iend && obase + SSE_THREADS >= n_old);
    // full 64s of the string (at the end the rest too): the operators, and
    // each one's number on its bond (the lanes of equal bonds found by
    // ballots over the bits of the bond index)
    while (stored + SSE_THREADS <= out || (end && stored < out)) {
      const bool have = stored + lane < min(out, cap);
      const int e = have ? ring[(stored + lane) & (2 * SSE_THREADS - 1)] : 0;
      const int b = e >> 3;
      unsigned long long same = __ballot(have);
      const unsigned long long odd = __ballot(have && (e & 1));
      for (int q = 0; q < bits; ++q) {
        const bool bit = (b >> q) & 1;
        const unsigned long long v = __ballot(bit);
        same &= bit ? v : ~v;
      }
      if (have) {
        const unsigned long long below = same & ((1ull << lane) - 1);
        const int r = cnt[b] + __popcll(below), ko = off[b] + __popcll(below & odd);
        sn[stored + lane] = e;
        rank_at[stored + lane] = r;
        koff_at[stored + lane] = ko;
        if ((same >> lane) == 1) {  // the last lane of its bond
          cnt[b] = r + 1;
          off[b] = ko + (e & 1);
        }
      }
      stored += SSE_THREADS;
    }
    if (end) break;
    if (k == SSE_THREADS) {
      xbase += SSE_THREADS;
      k = 0;
      const U4 x = philox(sweep, STAGE_SSE, 0u, (uint32_t)(xbase + lane), key0, key1);
      const double u = uniform53(x);
      // insertion tried iff (n + 1) u < bw: n + 1 up to the largest m with m u < bw
      const double est = bw / u;
      int m = est < (double)SSE_MOST ? (int)est : SSE_MOST;
      while (m < SSE_MOST && (double)(m + 1) * u < bw) ++m;
      while (m > 0 && !((double)m * u < bw)) --m;
      ins_at = m - 1 - lane;  // tried iff n - (steps before it) <= this, every one of those an insertion
      // removal iff bw u < n
      const double d = bw * u;
      rem_at = (d < (double)SSE_MOST ? (int)d + 1 : SSE_MOST) + lane;  // removed iff n + (steps before it) >= this, every one a removal
      z = (int)x.z;
      int b, g = 0;
      const uint64_t z64 = x.z;
      if (z64 < cls0) {
        b = (int)(((uint64_t)x.w * (uint64_t)nb_lat) >> 32);
        g = (int)(z64 >= tl0) + (int)(z64 >= tl1) + (int)(z64 >= tl2);
      } else if (z64 < cls1) {
        b = nb_lat + (int)(((uint64_t)x.w * (uint64_t)(nb_real - nb_lat)) >> 32);
        g = (int)(z64 >= td0) + (int)(z64 >= td1) + (int)(z64 >= td2);
      } else {  // a site operator: the site graph, compatible with either spin
        b = nb_real + (int)(((uint64_t)x.w * (uint64_t)nsite) >> 32);
      }
      ne = (b << 3) | (g << 1);
      s0 = s1 = SSE_NONE;
      bool ok = true;
      if (b < nb_real) {
        const uint32_t e2 = ends[b];
        s0 = (int)(e2 & 0xffffu);
        s1 = (int)(e2 >> 16);
        ok = ((g & 1) ^ spin_of(s0) ^ spin_of(s1)) != 0;
      }
      compat = __ballot(ok);
    }
    if (!gap && i == iend) {
      obase += SSE_THREADS;
      i = 0;
      iend = min(64, n_old - obase);
      el = next_el;
      next_el = obase + SSE_THREADS + lane < n_old ? so[obase + SSE_THREADS + lane] : 0;
      q0 = q1 = SSE_NONE;
      if (lane < iend) {
        const uint32_t e2 = ends[el >> 3];
        q0 = (int)(e2 & 0xffffu);
        q1 = (int)(e2 >> 16);
      }
      diag = __ballot(lane < iend && (el & 1) == 0);
    }

    // ---- the walk ----
    while (true) {
      if (gap) {
        // insertions up to the first step that fails
        const int r = run_length(__ballot(ins_at >= nop - k) & compat, k);
        if ((unsigned)(lane - k) < (unsigned)r) pos_ins = out - k + lane;
        out += r;
        nop += r;
        k += r;
        if (k == SSE_THREADS) break;
        ++k;
        gap = false;
        if (k == SSE_THREADS || i == iend) break;
      }
      // removals up to the next operator that stays (past the string's end no
      // bit of diag is set)
      const int rr = min(run_length(diag, i), run_length(__ballot(rem_at <= nop + k), k));
      nop -= rr;
      k += rr;
      i += rr;
      if (k == SSE_THREADS || i == iend) break;
      z_op = with_lane(z_op, i, lane_of(z, k));
      pos_op = with_lane(pos_op, i, out);
      const int t0 = lane_of(q0, i), t1 = lane_of(q1, i);
      if ((diag >> i) & 1) {
        // regraphed by its pair's spins: those of the last 64, and the
        // off-diagonal operators kept since
        if (t1 != SSE_NONE) {
          const unsigned long long since = __ballot(pos_op >= 0 && (el & 1));
          const unsigned long long hit = __ballot(q0 == t0) ^ __ballot(q1 == t0) ^ __ballot(q0 == t1) ^ __ballot(q1 == t1);
          if ((spin_of(t0) ^ spin_of(t1) ^ __popcll(since & hit)) & 1) anti |= 1ull << i;
        }
      } else {  // its spins flip (a site operator's target SSE_NONE meets the lanes without sites twice)
        compat ^= __ballot(s0 == t0) ^ __ballot(s1 == t0) ^ __ballot(s0 == t1) ^ __ballot(s1 == t1);
      }
      ++out;
      ++k;
      ++i;
      gap = true;
      if (k == SSE_THREADS) break;
    }
  }
  if (out > cap && lane == 0) atomicOr(B.flags, FLAG_OP_OVERFLOW);
  __syncthreads();
  for (int b = lane; b < Nb; b += SSE_THREADS) {
    B.counts[P.bond_base + b] = cnt[b];
    // each bond's diagonal operators, as the path-integral diagonal update
    // leaves them (k_end_sweep counts the off-diagonal ones for the sign)
    B.acc_count[P.bond_base + b] = cnt[b] - off[b];
  }
}

// the new string into bond-major order (series order within a bond), times
// p / n; perm[p] = the operator index of string position p.  SSE_SPLIT
// workgroups share a chain (one wave ranking 64 elements at a time took
// 2.7 ms on 512 chains of 32^2; the walk now leaves the ranks).
constexpr int SSE_SPLIT = 4;

__global__ void __launch_bounds__(256) k_sse_scatter(DevBatch B) {
  if (overflowed(B)) return;
  const int c = blockIdx.x / SSE_SPLIT, part = blockIdx.x % SSE_SPLIT;
  const ChainDev& P = B.chains[c];
  const int n = B.bo_new[P.bond_base + P.Nb] - B.bo_new[P.bond_base];
  const int* sn = B.sse_new + P.sse_base;
  int* perm = B.sse_perm + P.sse_base;  // holds the number on the bond
  const int* koff = B.l0 + P.sse_base;
  const int bond_base = P.bond_base;
  const double dn = (double)n;
  for (int p = part * 256 + (int)threadIdx.x; p < n; p += SSE_SPLIT * 256) {
    const int el = sn[p], gb = bond_base + (el >> 3);
    const int pos = B.bo_new[gb] + perm[p];
    B.ot_new[pos] = (double)p / dn;
    B.oi_new[pos] = (gb << 3) | (el & 7);
    B.kc_new[pos] = koff[p];
    perm[p] = pos;
  }
}

// the flipped operator types back into the string
__global__ void __launch_bounds__(256) k_sse_gather(DevBatch B) {
  if (overflowed(B)) return;
  const int c = blockIdx.x / SSE_SPLIT, part = blockIdx.x % SSE_SPLIT;
  const ChainDev& P = B.chains[c];
  // (k_end_sweep has moved the chain's old bases to the configuration just built)
  const int o0 = B.bo_new[P.bond_base], n = B.bo_new[P.bond_base + P.Nb] - o0;
  int* sn = B.sse_new + P.sse_base;
  const int* perm = B.sse_perm + P.sse_base;
  for (int p = part * 256 + (int)threadIdx.x; p < n; p += SSE_SPLIT * 256) sn[p] = (sn[p] & ~1) | (B.oi_new[perm[p]] & 1);
}

void launch_sse_walk(const DevBatch& B, hipStream_t st) {
  hipLaunchKernelGGL(k_sse_walk, dim3(B.nchains), dim3(SSE_THREADS), 0, st, B);
}
void launch_sse_scatter(const DevBatch& B, hipStream_t st) {
  hipLaunchKernelGGL(k_sse_scatter, dim3(B.nchains * SSE_SPLIT), dim3(256), 0, st, B);
}
void launch_sse_gather(const DevBatch& B, hipStream_t st) {
  hipLaunchKernelGGL(k_sse_gather, dim3(B.nchains * SSE_SPLIT), dim3(256), 0, st, B);
}

}  // namespace lg
