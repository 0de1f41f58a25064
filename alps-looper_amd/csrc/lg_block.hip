// One workgroup per chain: whole sweeps of a chain inside one workgroup, many
// sweeps per launch (gfx950).
//
// The kernels of lg_kernels.hip cut a sweep into eight or nine launches over
// flat arrays.  A chain of a few hundred to a few tens of thousands of
// operators does not fill them: each launch then costs its own start and a
// chain of dependent loads (7-14 us a kernel, whatever the size), and in a
// batch of many chains every per-operator step walks through global memory.
// Here a chain's workgroup keeps the sweep's random-access state in LDS --
// operator and segment offsets, event times cut to 31 bits for the searches
// (equal cuts are decided by the full time), off-diagonal bitmaps with
// prefix counts, the union-find parents as 16-bit words, the clusters'
// accumulators -- and streams the rest (times, types, segment arrays) in
// order.  The steps are those of lg_kernels.hip and so are the results: the
// same Philox counters, integer times, event order and cut rules.
//
// A chain's new configuration goes to a region of its own (ChainDev::blk_op,
// blk_node), so that no chain waits for the operator counts of others; its
// last offsets are blk_nops / blk_nnodes.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "lg_common.h"
#include "lg_device.h"
#include "lg_kernels.h"

namespace lg {

namespace {

extern __shared__ __align__(16) unsigned char blk_lds[];

// event time cut to 31 bits, in the upper bits of a word (bit 0 is free);
// ascending with the time, times from 1 on share the last value
__device__ __forceinline__ uint32_t cut_time(double t) {
  return (t >= 1.0 ? 0x7fffffffu : (uint32_t)(t * 2147483648.0)) << 1;
}

// bond lists of a site: the lattice's, the in-site bonds', its own operators'
__host__ __device__ __forceinline__ int chain_lists(const ChainDev& P) {
  return site_lists(P) + (P.npair > 0 ? P.nv - 1 : 0) + (P.Nb > P.nb_real ? 1 : 0);
}

// a value that is the same in every lane, in a scalar register
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }

// ---- block-wide helpers (every thread of the workgroup calls them) ---------
// inclusive prefix over the wave's lanes by data-parallel-primitive moves
// (rows of 16, then the rows' last lanes on to the rows above): six dependent
// VALU steps instead of six LDS permutes
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_add(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, true);
}
__device__ __forceinline__ int row_scan(int v) {  // within each row of 16 lanes
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  return dpp_add<0x118, 0xf>(v);
}
__device__ __forceinline__ int wave_scan(int v) {
  v = row_scan(v);
  v = dpp_add<0x142, 0xa>(v);
  return dpp_add<0x143, 0xc>(v);
}

// exclusive prefix of v over the workgroup's threads, and the total; wsum: 16
// words, not those of the call before (one barrier between two uses is enough)
__device__ __forceinline__ int blk_scan(int v, int* wsum, int* total) {
  const int lane = lane_id(), w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const int x = wave_scan(v);
  if (lane == 63) wsum[w] = x;
  __syncthreads();
  const int t = row_scan(lane < nw ? wsum[lane] : 0);
  *total = __shfl(t, nw - 1, 64);
  const int off = __shfl(t, w > 0 ? w - 1 : 0, 64);
  return (w > 0 ? off : 0) + x - v;
}

// a[0..n) in LDS to its exclusive prefix sums, a[n] the total; the caller's
// writes of a are behind a barrier, and the result is behind one
__device__ __forceinline__ int blk_prefix(int* a, int n, int* wsum) {
  const int items = (n + (int)blockDim.x - 1) / (int)blockDim.x;
  const int lo = min((int)threadIdx.x * items, n), hi = min(lo + items, n);
  int sum = 0;
  for (int i = lo; i < hi; ++i) sum += a[i];
  int tot;
  int off = blk_scan(sum, wsum, &tot);
  for (int i = lo; i < hi; ++i) {
    const int v = a[i];
    a[i] = off;
    off += v;
  }
  if (threadIdx.x == 0) a[n] = tot;
  __syncthreads();
  return tot;
}

// st(x, ld(x)) for x in [0, n) over the workgroup, U loads of a thread in
// flight (16 waves a CU cannot hide a load's latency one item at a time)
template <int U, class LD, class ST>
__device__ __forceinline__ void blk_each(int n, LD ld, ST st) {
  const int T = blockDim.x;
  for (int x0 = threadIdx.x; x0 < n; x0 += U * T) {
    decltype(ld(0)) v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = ld(min(x0 + u * T, n - 1));
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (x0 + u * T < n) st(x0 + u * T, v[u]);
  }
}

// a set of bits [0, n) in LDS with the counts before each 64-bit word
struct Bits {
  unsigned long long* w;  // [n / 64 + 1]
  int* pre;               // [n / 64 + 2]
  __device__ __forceinline__ int rank(int x) const {
    const int q = x >> 6;
    return pre[q] + __popcll(w[q] & ((1ull << (x & 63)) - 1));
  }
  __device__ __forceinline__ bool has(int x) const { return (w[x >> 6] >> (x & 63)) & 1; }
};
__host__ __device__ __forceinline__ int bits_words(int n) { return n / 64 + 1; }
__host__ __device__ __forceinline__ int bits_bytes(int n) { return bits_words(n) * 8 + ((bits_words(n) + 2) & ~1) * 4; }
__device__ __forceinline__ Bits bits_at(unsigned char* p, int n) {
  return Bits{(unsigned long long*)p, (int*)(p + (size_t)bits_words(n) * 8)};
}
// counts before each word, from the words (behind a barrier)
__device__ __forceinline__ int bits_count(const Bits& s, int n, int* wsum) {
  const int nw = bits_words(n);
  if (nw <= (int)blockDim.x) {  // a word per thread
    const int q = threadIdx.x;
    const int v = q < nw ? __popcll(s.w[q]) : 0;
    int tot;
    const int off = blk_scan(v, wsum, &tot);
    if (q < nw) s.pre[q] = off;
    if (q == 0) s.pre[nw] = tot;
    __syncthreads();
    return tot;
  }
  for (int q = threadIdx.x; q < nw; q += blockDim.x) s.pre[q] = __popcll(s.w[q]);
  __syncthreads();
  return blk_prefix(s.pre, nw, wsum);
}
// word x >> 6 of the set from each lane's bit (a wave holds 64 consecutive x)
__device__ __forceinline__ void bits_put(const Bits& s, int x, bool v) {
  const unsigned long long m = __ballot(v);
  if (lane_id() == 0) s.w[x >> 6] = m;
}

// ---- event times of the searches: cut in LDS (32 or 16 bits), or full -----
// below(i): the event's cut time is below the searched one's; same(i): the
// cuts are equal, and the full times decide
struct Cut32 {  // 31 bits of the time | spin
  const uint32_t* h;
  const double* full;
  uint32_t hx;
  __device__ __forceinline__ void at(double x) { hx = cut_time(x); }
  __device__ __forceinline__ bool below(int i) const { return h[i] < hx; }
  __device__ __forceinline__ bool same(int i) const { return (h[i] ^ hx) < 2u; }
  __device__ __forceinline__ int spin(int i) const { return (int)(h[i] & 1u); }
  __device__ __forceinline__ double time(int i) const { return full[i]; }
};
struct Cut16 {  // 15 bits of the time | spin (about one search in a thousand reads full times)
  const uint16_t* h;
  const double* full;
  uint32_t hx;
  __device__ __forceinline__ void at(double x) { hx = (cut_time(x) >> 17) << 1; }
  __device__ __forceinline__ bool below(int i) const { return h[i] < hx; }
  __device__ __forceinline__ bool same(int i) const { return (h[i] ^ hx) < 2u; }
  __device__ __forceinline__ int spin(int i) const { return h[i] & 1; }
  __device__ __forceinline__ double time(int i) const { return full[i]; }
};
struct FullTimes {
  const double* full;
  const uint8_t* seg;
  double x;
  __device__ __forceinline__ void at(double t) { x = t; }
  __device__ __forceinline__ bool below(int i) const { return full[i] < x; }
  __device__ __forceinline__ bool same(int i) const { return full[i] == x; }
  __device__ __forceinline__ int spin(int i) const { return seg[i]; }
  __device__ __forceinline__ double time(int i) const { return full[i]; }
};

// first of the events [r, end) not below x (or, ties, above x), from the
// first one whose cut is not below x's
template <class TS>
__device__ __forceinline__ int settle(const TS& t, int r, int end, bool ties, double x) {
  while (r < end && t.same(r)) {
    const double v = t.time(r);
    if (ties ? !(v <= x) : !(v < x)) break;
    ++r;
  }
  return r;
}

// ---- union-find: parents as 16-bit words in LDS, or as ints in memory -----
// (the hooking rule of lg_kernels.hip: the larger root goes under the smaller)
struct Parents16 {
  uint16_t* p;
  __device__ __forceinline__ int get(int x) const {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __device__ __forceinline__ void set(int x, int v) const {
    __hip_atomic_store(p + x, (uint16_t)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // hook root a under b; returns a's parent before (a on success)
  __device__ __forceinline__ int hook(int a, int b) const {
    unsigned int* w = (unsigned int*)p + (a >> 1);
    const int sh = (a & 1) * 16;
    unsigned int old = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    while (true) {
      const int cur = (int)((old >> sh) & 0xffffu);
      if (cur != a) return cur;
      const unsigned int seen = atomicCAS(w, old, (old & ~(0xffffu << sh)) | ((unsigned int)b << sh));
      if (seen == old) return a;
      old = seen;
    }
  }
};
struct ParentsMem {
  int* p;
  __device__ __forceinline__ int get(int x) const {
    return __hip_atomic_load(p + x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ void set(int x, int v) const {
    __hip_atomic_store(p + x, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __device__ __forceinline__ int hook(int a, int b) const { return atomicCAS(p + a, a, b); }
};
template <class U>
__device__ __forceinline__ int blk_find(const U& u, int x) {
  int p;
  while ((p = u.get(x)) != x) x = p;
  return x;
}
template <class U>
__device__ __forceinline__ void blk_unite(const U& u, int a, int b) {
  a = blk_find(u, a);
  b = blk_find(u, b);
  while (a != b) {
    if (a < b) { const int t = a; a = b; b = t; }
    const int old = u.hook(a, b);
    if (old == a) return;
    a = blk_find(u, old);
    b = blk_find(u, b);
  }
}

// A segment's flags here (bits 0-1: its class, as ClusterAcc counts it; bits
// 2-3: the winding of the event above it, for the event's source site)
enum : uint8_t { SEG_GAUGE = 1, SEG_DOWN = 2, SEG_X = 4, SEG_Y = 8, SEG_FIRST = 16, SEG_EMPTY = 32, SEG_NOWRAP = 64 };

// ---------------------------------------------------------------------------
// a chain's working state, the same in every thread of its workgroup
// ---------------------------------------------------------------------------
struct Chain {
  int *bo, *so;           // LDS: operator offsets per bond, segment offsets per site (previous configuration)
  int *bn, *sn;           // LDS: those being built
  uint32_t* ends;         // LDS: source | target << 16 of every bond
  uint32_t* into;         // LDS: the lattice bonds of which a site is the target (square: y | x << 16; plain chains)
  uint16_t* lists;        // LDS: a site's nl bonds, site-major (GEN)
  int nl;
  uint8_t* spin;          // LDS: tau = 0 spins
  uint8_t* sbase;         // LDS: tau = 0 spin ^ the off-diagonal parities before the site's lists | gauge << 1
  unsigned char* rest;    // LDS from here on: by step
  int rest_bytes;
  int n, m;               // operators and segments of the previous configuration
};

// Diagonal update (diag_count_bond of lg_kernels.hip) in two loops.  The first
// draws the bonds' Poisson candidates into the chain's list (time; bond |
// graph << 14 | number on the bond << 16).  Groups of G lanes take bonds from
// a counter, so that a lane is busy whatever its bonds' numbers (one bond per
// lane in turn would wait for the largest of 64 bonds).  The second tests the
// candidates against the previous world lines, one per lane: drawing and
// testing in one loop held twice the registers and ran the searches with the
// lanes of finished bonds idle.
template <int G, bool GEN>
__device__ __forceinline__ void blk_draw(const DevBatch& B, const ChainDev& P, uint32_t sweep, double scale_lat,
                                         double scale_in, double scale_site, double* list, uint32_t* list_bond,
                                         int cap, int* next, int* ncand) {
  const int lane = lane_id(), gl = lane & (G - 1), gbase = lane & ~(G - 1);
  const uint64_t below = (1ull << lane) - 1;
  const int Nb = P.Nb, kmax = ((P.cand_cap + 31) / 32) * 32;
  bool fresh = true;
  int b = 0, cls = 0;
  uint64_t Tb = 0;
  int kb = 0;
  double scale = scale_lat;
  while (true) {
    if (fresh) {
      int q = 0;
      if (gl == 0) q = atomicAdd(next, 1);
      if (G > 1) q = __shfl(q, gbase, 64);
      b = q;
      if (b >= Nb) break;
      if (GEN) {
        cls = b >= P.nb_real ? 2 : (b >= P.nb_lat ? 1 : 0);
        scale = cls == 2 ? scale_site : (cls == 1 ? scale_in : scale_lat);
        if (!(cls == 2 ? P.site_w > 0 : (cls == 1 ? P.dwsum > 0 : P.has_weight != 0))) continue;
      }
      Tb = 0;
      kb = 0;
      fresh = false;
    }
    const U4 x = philox(sweep, STAGE_DIAG, (uint32_t)b, (uint32_t)(kb + gl), P.key0, P.key1);
    uint64_t incl = exp_gap(x, scale);
    if (G > 1) {
#pragma unroll
      for (int d = 1; d < G; d <<= 1) {
        const uint32_t lo = __shfl_up((unsigned int)(incl & 0xffffffffu), d, G);
        const uint32_t hi = __shfl_up((unsigned int)(incl >> 32), d, G);
        if (gl >= d) incl += ((uint64_t)hi << 32) | lo;
      }
    }
    const uint64_t T = Tb + incl;
    if (T < TGRID) {
      int g;
      const uint64_t z = x.z;
      if (!GEN || cls == 0) g = (int)(z >= P.thr[0]) + (int)(z >= P.thr[1]) + (int)(z >= P.thr[2]);
      else if (cls == 1) g = (int)(z >= P.dthr[0]) + (int)(z >= P.dthr[1]) + (int)(z >= P.dthr[2]);
      else g = 0;
      const uint64_t m = __ballot(true);
      const int lead = __ffsll((long long)m) - 1;
      int base = 0;
      if (lane == lead) base = atomicAdd(ncand, __popcll(m));
      const int at = __shfl(base, lead, 64) + __popcll(m & below), k = kb + gl;
      if (at < cap && k < kmax) {
        list[at] = (double)T * TGRID_INV;
        list_bond[at] = (uint32_t)b | ((uint32_t)g << 14) | ((uint32_t)k << 16);
      } else {
        atomicOr(B.flags + 1, FLAG_CAND_OVERFLOW);
      }
    }
    if (G > 1) {
      const uint32_t lo = __shfl((unsigned int)(incl & 0xffffffffu), G - 1, G);
      const uint32_t hi = __shfl((unsigned int)(incl >> 32), G - 1, G);
      Tb += ((uint64_t)hi << 32) | lo;
    } else {
      Tb = T;
    }
    kb += G;
    fresh = Tb >= TGRID || kb > kmax;  // (draws beyond the slots: flagged above; the loop is bounded)
  }
}

// accepted candidates: bit (number on the bond) of the bond's words in acc
template <bool GEN, class TS>
__device__ __forceinline__ void blk_test(const ChainDev& P, const Chain& S, const TS times, int ncand,
                                         const double* list, const uint32_t* list_bond, uint32_t* acc, int wpb) {
  struct Cand { uint32_t v; double tau; };
  blk_each<2>(ncand, [&](int e) { return Cand{list_bond[e], list[e]}; }, [&](int, const Cand& cd) {
    const uint32_t v = cd.v;
    const double tau = cd.tau;
    const int b = (int)(v & 0x3fffu), g = (int)(v >> 14) & 3, k = (int)(v >> 16);
    const uint32_t en = S.ends[b];
    const int s0 = (int)(en & 0xffffu), s1 = (int)(en >> 16);
    const int n0 = S.so[s0], x0 = S.so[s0 + 1], n1 = S.so[s1], x1 = S.so[s1 + 1];
    TS t = times;
    t.at(tau);
    int l0 = n0, c0 = x0 - n0, l1 = n1, c1 = x1 - n1;
    while ((c0 | c1) > 0) {  // first event not below tau on both sites, a step of each at a time
      const int h0 = c0 >> 1, h1 = c1 >> 1;
      const bool u0 = c0 > 0 && t.below(l0 + h0), u1 = c1 > 0 && t.below(l1 + h1);
      if (u0) { l0 += h0 + 1; c0 -= h0 + 1; } else { c0 = h0; }
      if (u1) { l1 += h1 + 1; c1 -= h1 + 1; } else { c1 = h1; }
    }
    l0 = settle(t, l0, x0, false, tau);
    l1 = settle(t, l1, x1, false, tau);
    // an event of exactly this time on either site rejects the candidate
    const bool tie = (l0 < x0 && t.same(l0) && t.time(l0) == tau) || (l1 < x1 && t.same(l1) && t.time(l1) == tau);
    const int p = t.spin(l0 < x0 ? l0 : n0) ^ t.spin(l1 < x1 ? l1 : n1) ^ g;
    if (!tie && ((GEN && b >= P.nb_real) || (p & 1))) atomicOr(&acc[b * wpb + (k >> 5)], 1u << (k & 31));
  });
}

// rank of each accepted candidate among its bond's previous operators (times
// ordered), and with it its place in the new operator list
template <class TS>
__device__ __forceinline__ void blk_place(const ChainDev& P, const Chain& S, const TS times, const Bits& off,
                                          const Bits& occ, int ncand, const double* list, const uint32_t* list_bond,
                                          const uint32_t* acc, int wpb, double* ot_new, int* oi_new) {
  struct Cand { uint32_t v; double tau; };
  blk_each<2>(ncand, [&](int e) { return Cand{list_bond[e], list[e]}; }, [&](int, const Cand& cd) {
    const uint32_t v = cd.v;
    const int b = (int)(v & 0x3fffu), k = (int)(v >> 16);
    const uint32_t* w = acc + b * wpb;
    const uint32_t word = w[k >> 5];
    if (!((word >> (k & 31)) & 1u)) return;
    int j = __popc(word & ((1u << (k & 31)) - 1));
    for (int i = 0; i < (k >> 5); ++i) j += __popc(w[i]);
    const double tau = cd.tau;
    TS t = times;
    t.at(tau);
    const int lo = S.bo[b], end = S.bo[b + 1];
    int r = lo, len = end - lo;
    while (len > 0) {
      const int h = len >> 1;
      if (t.below(r + h)) { r += h + 1; len -= h + 1; } else { len = h; }
    }
    r = settle(t, r, end, false, tau);
    const int pos = S.bn[b] + j + off.rank(r) - off.rank(lo);
    ot_new[pos] = tau;
    oi_new[pos] = ((P.bond_base + b) << 3) | ((int)((v >> 14) & 3u) << 1);
    atomicOr(&occ.w[pos >> 6], 1ull << (pos & 63));
  });
}

// World-line linking, one thread per operator (k_link_ops of lg_kernels.hip):
// par(x) = parity of the off-diagonal operators before x; bit 0 of S.sbase[s]
// the tau = 0 spin ^ the parities at the starts of the site's lists, so that
// the spin below an event is that ^ the parities at its positions in the
// lists; bit 1 set where the gauge is -1.
template <bool GEN, class TS, class PAR>
__device__ __forceinline__ void blk_link(const ChainDev& P, const Chain& S, const TS times, PAR par, int n,
                                         const double* ot, const int* oi, double* evt, uint8_t* evflags, int* l0,
                                         int* l1) {
  const bool chain = P.kind == 0;
  const int bond_base = P.bond_base;
  struct Op { int info; double tau; };
  blk_each<2>(n, [&](int k) { return Op{oi[k], ot[k]}; }, [&](int k, const Op& op) {
    const int info = op.info;
    const int b = (info >> 3) - bond_base;
    const double tau = op.tau;
    TS t = times;
    t.at(tau);
    const uint32_t e = S.ends[b];
    const bool site = GEN && b >= P.nb_real;
    const bool lattice = !GEN || b < P.nb_lat;
    const int dflag = GEN ? (!lattice ? 0 : (bond_dir(P, b) ? SEG_Y : SEG_X)) : ((chain || (b & 1)) ? SEG_X : SEG_Y);
    const int own = k - S.bn[b], kpar = par(k);
    int leg[2];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      if (GEN && side && site) { leg[1] = leg[0]; break; }
      const int s = side ? (int)(e >> 16) : (int)(e & 0xffffu);
      const int base = S.sbase[s];
      int rank = own, sp = base ^ kpar;
      if (!GEN) {
        // the site's other lists (three on the square lattice, one on the
        // chain) searched together, a step of each at a time
        int o0, o1 = b, o2 = b;
        const uint32_t in = S.into[s];  // the bonds of which the site is the target
        if (chain) {
          o0 = side ? s : (int)in;
        } else {
          const int y = (int)(in & 0xffffu), x = (int)(in >> 16);
          o0 = side ? 2 * s : (b ^ 1);
          o1 = side ? 2 * s + 1 : y;
          o2 = side ? ((b & 1) ? y : x) : x;
        }
        const int a0 = S.bn[o0], a1 = S.bn[o1], a2 = S.bn[o2];
        const int e0 = S.bn[o0 + 1], e1 = S.bn[o1 + 1], e2 = S.bn[o2 + 1];
        // (the chain's second and third list stand for its own: empty)
        int r0 = a0, r1 = a1, r2 = a2, c0 = o0 != b ? e0 - a0 : 0, c1 = chain ? 0 : e1 - a1, c2 = chain ? 0 : e2 - a2;
        while ((c0 | c1 | c2) > 0) {
          const int h0 = c0 >> 1, h1 = c1 >> 1, h2 = c2 >> 1;
          const bool u0 = c0 > 0 && t.below(r0 + h0), u1 = c1 > 0 && t.below(r1 + h1), u2 = c2 > 0 && t.below(r2 + h2);
          if (u0) { r0 += h0 + 1; c0 -= h0 + 1; } else { c0 = h0; }
          if (u1) { r1 += h1 + 1; c1 -= h1 + 1; } else { c1 = h1; }
          if (u2) { r2 += h2 + 1; c2 -= h2 + 1; } else { c2 = h2; }
        }
        if (o0 != b) { r0 = settle(t, r0, e0, o0 < b, tau); rank += r0 - a0; sp ^= par(r0); }
        if (!chain) {
          r1 = settle(t, r1, e1, o1 < b, tau);
          r2 = settle(t, r2, e2, o2 < b, tau);
          rank += r1 - a1 + r2 - a2;
          sp ^= par(r1) ^ par(r2);
        }
      } else {
        auto other = [&](int bp) {
          if (bp == b) return;
          const int lo = S.bn[bp], end = S.bn[bp + 1];
          int r = lo, len = end - lo;
          while (len > 0) {
            const int h = len >> 1;
            if (t.below(r + h)) { r += h + 1; len -= h + 1; } else { len = h; }
          }
          r = settle(t, r, end, bp < b, tau);
          rank += r - lo;
          sp ^= par(r);
        };
        for (int i = 0; i < S.nl; ++i) other(S.lists[s * S.nl + i]);
      }
      const int node = S.sn[s] + rank;
      const bool split = GEN && P.nv > 1;
      const int gflag = (base >> 1) & SEG_GAUGE;
      evt[node] = tau;
      evflags[node] = (uint8_t)(gflag | ((sp & 1) << 1) | (side ? 0 : dflag) | (rank == 0 ? SEG_FIRST : 0) |
                                (split && rank == 0 ? SEG_NOWRAP : 0));
      if (split && node + 2 == S.sn[s + 1]) {  // the last event: the site's top segment, up to tau = 1
        evt[node + 1] = 1.0;
        evflags[node + 1] = (uint8_t)(gflag | (((sp ^ info) & 1) << 1));
      }
      leg[side] = node;
    }
    l0[k] = leg[0];
    l1[k] = leg[1];
  });
}

// segment above the event below which `node` lies, on site s
__device__ __forceinline__ int blk_up(const Chain& S, int node, int s) {
  return node + 1 == S.sn[s + 1] ? S.sn[s] : node + 1;
}

// unions of every operator by its graph (graph_impl.h:277-295)
template <bool GEN, class U>
__device__ __forceinline__ void blk_unions(const ChainDev& P, const Chain& S, const U u, int n, const int* oi,
                                           const int* l0, const int* l1) {
  struct Op { int info, a0, a1; };
  blk_each<4>(n, [&](int k) { return Op{oi[k], l0[k], l1[k]}; }, [&](int, const Op& op) {
    const int info = op.info;
    const int b = (info >> 3) - P.bond_base;
    if (GEN && b >= P.nb_real) return;  // a site operator cuts the world line
    const int g = (info >> 1) & 3;
    const uint32_t e = S.ends[b];
    const int a0 = op.a0, a1 = op.a1;
    const int b0 = blk_up(S, a0, (int)(e & 0xffffu)), b1 = blk_up(S, a1, (int)(e >> 16));
    if (g & 2) {            // frozen: all four legs
      blk_unite(u, a0, a1);
      blk_unite(u, b0, b1);
      blk_unite(u, a0, b0);
    } else if (g == 0) {    // horizontal cut
      blk_unite(u, a0, a1);
      blk_unite(u, b0, b1);
    } else {                // cross
      blk_unite(u, a0, b1);
      blk_unite(u, a1, b0);
    }
  });
}

// unions, the tau boundary of virtual sites, then every segment's root in
// place of its parent; roots: the set of the root segments, whose rank in it
// numbers the clusters; root_of: their segments.  Returns their number.
template <bool GEN, class U>
__device__ __forceinline__ int blk_clusters(const ChainDev& P, const Chain& S, const U u, uint32_t sweep, int n, int m,
                                             const int* oi, const int* l0, const int* l1, const uint8_t* evflags,
                                             const Bits& roots, int* root_of, int* wsum) {
  for (int x = threadIdx.x; x < m; x += blockDim.x) u.set(x, x);
  __syncthreads();
  blk_unions<GEN>(P, S, u, n, oi, l0, l1);
  if (GEN && P.nv > 1) {
    const int nr = P.N / P.nv;
    for (int r = threadIdx.x; r < nr; r += blockDim.x) {
      int bot[MAX_NV], top[MAX_NV];
      uint32_t bs = 0, es = 0;
#pragma unroll
      for (int a = 0; a < MAX_NV; ++a) {
        bot[a] = top[a] = 0;
        if (a < P.nv) {
          bot[a] = S.sn[r * P.nv + a];
          top[a] = S.sn[r * P.nv + a + 1] - 1;
          bs |= (uint32_t)((evflags[bot[a]] >> 1) & 1) << a;
          es |= (uint32_t)((evflags[top[a]] >> 1) & 1) << a;
        }
      }
      join_boundary(P, sweep, r, bot, top, bs, es, [&](int a, int b) { blk_unite(u, a, b); });
    }
  }
  __syncthreads();
  const int end = bits_words(m) * 64;
  for (int x = threadIdx.x; x < end; x += blockDim.x) {
    bool root = false;
    if (x < m) {
      const int r = blk_find(u, x);
      root = r == x;
      u.set(x, r);  // (an ancestor: walks through x still end at r)
    }
    bits_put(roots, x, root);
  }
  __syncthreads();
  const int nc = bits_count(roots, m, wsum);
  for (int x = threadIdx.x; x < m; x += blockDim.x)
    if (roots.has(x)) root_of[roots.rank(x)] = x;
  return nc;
}

// the collector's accumulators of a cluster: 4 class lengths, the tau = 0
// segments of the 4 classes (16 bits each), the packed winding
constexpr int ACC_BYTES = 48;
struct Acc {
  double* L;              // [W][4]
  unsigned long long* n;  // [W]
  unsigned long long* w;  // [W]
  int W;
  // a segment of cluster a: its length, and the winding d0, d1 (-1 .. 1)
  __device__ __forceinline__ void add(int a, double len, int cls, int d0, int d1) const {
    unsafeAtomicAdd(&L[4 * a + cls], len);
    if (d0 | d1) atomicAdd(&w[a], (unsigned long long)pack_winding(d0, d1));
  }
};
// winding of a segment with flags fl above one with flags flo (stiffness.h:94-105)
__device__ __forceinline__ void seg_winding(int fl, int flo, int& d0, int& d1) {
  const int x = ((fl >> 2) & 1) - ((flo >> 2) & 1), y = ((fl >> 3) & 1) - ((flo >> 3) & 1);
  d0 = (fl & SEG_DOWN) ? -x : x;
  d1 = (fl & SEG_DOWN) ? -y : y;
}

}  // namespace

// Bound by the instructions of one CU (80000 vector instructions a sweep at
// 2400 operators, which the CU's four SIMDs issue in 33 of 61 us; the rest is
// barriers, LDS and loads), so the steps hold little per operator; 256, 512 or
// 1024 threads by the operators, as few as keep a step's loads in flight, so
// that small chains share a CU.  A sweep of 450 operators: 65 us in eight
// launches, 27 here; 512 chains of up to 24000 operators: 1.30 and 0.59 ms,
// the largest chain's time (link 116 us, unions 98, estimator 115, draws 64,
// tests 46, places 75 of it).
// GEN: virtual sites (S > 1/2), in-site bonds (single-ion term) or site
// operators (transverse field); the plain instance carries none of it.
// (1024 threads: 128 VGPRs; one workgroup per CU at the full LDS)
template <bool GEN>
__global__ void __launch_bounds__(1024) k_chain_sweeps(DevBatch B, BlockArgs A) {
  // (the same answer for every wave of the workgroup: this kernel raises its
  // own flags in the second word, which k_chain_stop passes on after it)
  if (overflowed(B)) return;
  __shared__ int s_next, s_ncand, s_wsum[2][16];
  __shared__ double s_red[16][NCOL];
  int* const ws0 = s_wsum[0];
  int* const ws1 = s_wsum[1];
  const int tid = threadIdx.x, T = blockDim.x;
  const int c = uni(A.order[blockIdx.x]);
  // (the descriptor through the constant address space: scalar loads where a
  // field is used, instead of a hundred registers held for the whole kernel;
  // nothing writes it before the end)
  const ChainDev& P = *(const ChainDev*)(const __attribute__((address_space(4))) ChainDev*)(uintptr_t)(B.chains + c);
  const int N = P.N, Nb = P.Nb;
  double beta = P.beta, scale_lat = P.scale, scale_in = P.dscale, scale_site = P.site_scale;
  uint32_t sweep = (uint32_t)uni((int)B.sweep[c]);

  // ---- LDS: the chain's tables, then space used step by step ----
  Chain S;
  unsigned char* at = blk_lds;
  auto take = [&](int bytes) { unsigned char* p = at; at += (bytes + 7) & ~7; return p; };
  S.bo = (int*)take((Nb + 1) * 4);
  S.bn = (int*)take((Nb + 1) * 4);
  S.so = (int*)take((N + 1) * 4);
  S.sn = (int*)take((N + 1) * 4);
  S.ends = (uint32_t*)take(Nb * 4);
  S.nl = GEN ? chain_lists(P) : 0;
  S.into = (uint32_t*)take(GEN ? 0 : N * 4);
  S.lists = (uint16_t*)take(GEN ? N * S.nl * 2 : 0);
  S.spin = (uint8_t*)take(N);
  S.sbase = (uint8_t*)take(N);
  S.rest = at;
  S.rest_bytes = A.lds - (int)(at - blk_lds);
  for (int b = tid; b < Nb; b += T) {
    int s0, s1;
    op_sites(P, b, s0, s1);
    S.ends[b] = (uint32_t)s0 | ((uint32_t)s1 << 16);
  }
  if (GEN) {
    const int z = site_lists(P), nd = P.npair > 0 ? P.nv - 1 : 0;
    for (int q = tid; q < N * S.nl; q += T) {
      const int s = q / S.nl, i = q - s * S.nl;
      S.lists[q] = (uint16_t)(i < z ? site_bond(P, s, i) : (i < z + nd ? dpair_bond(P, s, i - z) : P.nb_real + s));
    }
  }
  if (!GEN)
    for (int s = tid; s < N; s += T)
      S.into[s] = P.kind == 0 ? (uint32_t)real_site_bond(P, s, 1)
                              : (uint32_t)real_site_bond(P, s, 2) | ((uint32_t)real_site_bond(P, s, 3) << 16);
  const int ob = P.old_bond_base, os = P.old_site_base;
  const int op0 = uni(B.bo_old[ob]), nd0 = uni(B.soff_old[os]);
  S.n = uni(A.packed ? B.bo_old[ob + Nb] - op0 : A.nops[c]);
  S.m = uni(A.packed ? B.soff_old[os + N] - nd0 : A.nnodes[c]);
  if (S.n > P.blk_opcap || S.m > P.blk_nodecap) {  // (the tables below are sized for the region)
    if (tid == 0) atomicOr(B.flags + 1, S.n > P.blk_opcap ? FLAG_OP_OVERFLOW : FLAG_NODE_OVERFLOW);
    return;
  }
  for (int b = tid; b < Nb; b += T) S.bo[b] = B.bo_old[ob + b] - op0;
  for (int s = tid; s < N; s += T) { S.so[s] = B.soff_old[os + s] - nd0; S.spin[s] = B.spins_old[os + s]; }
  if (tid == 0) { S.bo[Nb] = S.n; S.so[N] = S.m; }
  // the two configurations' arrays at this chain's place: the previous one's
  // for the first sweep, the chain's region afterwards
  const double* ot_old = B.ot_old + op0;
  const int* oi_old = B.oi_old + op0;
  const double* evt_old = B.evt_old + nd0;
  const uint8_t* seg_old = B.segspin_old + nd0;
  int old_bond_base = ob;
  // scratch of the chain's region
  double* const list = B.cand_t + P.cand_base;
  uint32_t* const list_bond = (uint32_t*)B.kc_new + P.blk_op;
  const int list_cap = min(P.blk_opcap, Nb * P.cand_cap);
  int* const kept_at = B.kpre + P.blk_op;
  int* const l0 = B.l0 + P.blk_op;
  int* const l1 = B.l1 + P.blk_op;
  uint8_t* const evflags = B.evflags + P.blk_node;
  int* const parents = B.parent + P.blk_node;
  int* const root_of = A.root_of + P.blk_node;
  double* const seg_len = A.seg_len + P.blk_node;
  uint32_t* const seg_info = A.seg_info + P.blk_node;
  const int wpb = (P.cand_cap + 31) / 32;
  __syncthreads();
  {  // off-diagonal operators of the configuration
    const Bits off = bits_at(S.rest, S.n);
    const int end = bits_words(S.n) * 64;
    for (int k = tid; k < end; k += T) bits_put(off, k, k < S.n && (oi_old[k] & 1));
    __syncthreads();
    bits_count(off, S.n, ws0);
  }

  for (int it = 0; it < A.nsweeps; ++it) {
    double* const ot_new = ((it & 1) ? const_cast<double*>(B.ot_old) : B.ot_new) + P.blk_op;
    int* const oi_new = ((it & 1) ? const_cast<int*>(B.oi_old) : B.oi_new) + P.blk_op;
    double* const evt_new = ((it & 1) ? const_cast<double*>(B.evt_old) : B.evt_new) + P.blk_node;
    uint8_t* const seg_new = ((it & 1) ? const_cast<uint8_t*>(B.segspin_old) : B.segspin_new) + P.blk_node;
    const Bits off = bits_at(S.rest, S.n);
    uint32_t* const acc = (uint32_t*)(S.rest + bits_bytes(S.n));
    const int acc_bytes = (Nb * wpb * 4 + 7) & ~7;
    unsigned char* const sp1 = (unsigned char*)acc + acc_bytes;
    const int sp1_bytes = S.rest_bytes - bits_bytes(S.n) - acc_bytes;

    // ---- diagonal update: the bonds' candidates ----
    const int cut1 = sp1_bytes >= 4 * S.m ? 32 : (sp1_bytes >= 2 * S.m ? 16 : 0);
    if (cut1 == 32) {
      blk_each<4>(S.m, [&](int x) { return cut_time(evt_old[x]) | seg_old[x]; }, [&](int x, uint32_t v) { ((uint32_t*)sp1)[x] = v; });
    } else if (cut1 == 16) {
      blk_each<4>(S.m, [&](int x) { return ((cut_time(evt_old[x]) >> 17) << 1) | seg_old[x]; }, [&](int x, uint32_t v) { ((uint16_t*)sp1)[x] = (uint16_t)v; });
    }
    for (int k = tid; k < S.n; k += T)
      if (off.has(k)) kept_at[off.rank(k)] = k;
    for (int i = tid; i < Nb * wpb; i += T) acc[i] = 0;
    if (tid == 0) { s_next = 0; s_ncand = 0; }
    __syncthreads();
    if (GEN || P.has_weight) {
      // one lane per bond when there are bonds for the lanes; small lattices
      // share a bond's draws over 4 or 16 lanes
      if (Nb * 4 > 2 * T) blk_draw<1, GEN>(B, P, sweep, scale_lat, scale_in, scale_site, list, list_bond, list_cap, &s_next, &s_ncand);
      else if (Nb * 16 > 2 * T) blk_draw<4, GEN>(B, P, sweep, scale_lat, scale_in, scale_site, list, list_bond, list_cap, &s_next, &s_ncand);
      else blk_draw<16, GEN>(B, P, sweep, scale_lat, scale_in, scale_site, list, list_bond, list_cap, &s_next, &s_ncand);
    }
    __syncthreads();
    const int ncand = min(uni(s_ncand), list_cap);
    // ---- candidates against the previous world lines ----
    if (cut1 == 32) blk_test<GEN>(P, S, Cut32{(const uint32_t*)sp1, evt_old, 0}, ncand, list, list_bond, acc, wpb);
    else if (cut1 == 16) blk_test<GEN>(P, S, Cut16{(const uint16_t*)sp1, evt_old, 0}, ncand, list, list_bond, acc, wpb);
    else blk_test<GEN>(P, S, FullTimes{evt_old, seg_old, 0}, ncand, list, list_bond, acc, wpb);
    __syncthreads();
    // ---- offsets of the new operators and segments ----
    for (int b = tid; b < Nb; b += T) {
      int q = off.rank(S.bo[b + 1]) - off.rank(S.bo[b]);
      for (int i = 0; i < wpb; ++i) q += __popc(acc[b * wpb + i]);
      S.bn[b] = q;
    }
    __syncthreads();
    const int n = uni(blk_prefix(S.bn, Nb, ws1));
    for (int s = tid; s < N; s += T) {
      int q = 0;
      auto add = [&](int b) { q += S.bn[b + 1] - S.bn[b]; };
      if (!GEN) {
        const uint32_t in = S.into[s];
        if (P.kind == 0) { add(s); add((int)in); }
        else { add(2 * s); add(2 * s + 1); add((int)(in & 0xffffu)); add((int)(in >> 16)); }
      } else {
        for (int i = 0; i < S.nl; ++i) add(S.lists[s * S.nl + i]);
      }
      S.sn[s] = q == 0 ? 1 : (GEN && P.nv > 1 ? q + 1 : q);
      S.sbase[s] = (uint8_t)((q == 0 ? 1 : 0) | (gauge(P, s) < 0 ? 2 : 0));  // (bit 0: event-free, until the linking's parity goes there)
    }
    __syncthreads();
    const int m = uni(blk_prefix(S.sn, N, ws0));
    if (n > P.blk_opcap || m > P.blk_nodecap) {
      // the operators or segments do not fit (uniform over the workgroup).
      // The offsets of the launch's earlier sweeps are not written out and
      // the host takes the next arrays for the configuration: none is whole
      // from here on, and the host gives none out (Batch::config_lost)
      if (tid == 0) atomicOr(B.flags + 1, n > P.blk_opcap ? FLAG_OP_OVERFLOW : FLAG_NODE_OVERFLOW);
      return;
    }
    for (int s = tid; s < N; s += T) {
      const int node = S.sn[s];
      if (S.sbase[s] & 1) {  // event-free site: one segment spanning [0,1)
        evt_new[node] = EMPTY_TIME;
        evflags[node] = (uint8_t)(SEG_EMPTY | SEG_FIRST | ((S.sbase[s] >> 1) & SEG_GAUGE) | (S.spin[s] << 1));
      }
    }
    // ---- the new operator list ----
    const Bits occ = bits_at(sp1, n);  // places of the accepted candidates, then the kept operators' places
    unsigned char* const sp2 = sp1 + bits_bytes(n);
    const int sp2_bytes = sp1_bytes - bits_bytes(n);
    const int nw = bits_words(n);
    for (int q = tid; q < nw; q += T) occ.w[q] = 0;
    const bool cut2 = sp2_bytes >= 4 * S.n;
    if (cut2)
      blk_each<4>(S.n, [&](int k) { return cut_time(ot_old[k]); }, [&](int k, uint32_t v) { ((uint32_t*)sp2)[k] = v; });
    __syncthreads();
    if (cut2) blk_place(P, S, Cut32{(const uint32_t*)sp2, ot_old, 0}, off, occ, ncand, list, list_bond, acc, wpb, ot_new, oi_new);
    else blk_place(P, S, FullTimes{ot_old, nullptr, 0}, off, occ, ncand, list, list_bond, acc, wpb, ot_new, oi_new);
    __syncthreads();
    // the places left are the kept operators', in their order: both lists are
    // sorted by (bond, time)
    for (int q = tid; q < nw; q += T) {
      const int rem = n - q * 64;
      occ.w[q] = ~occ.w[q] & (rem >= 64 ? ~0ull : (rem <= 0 ? 0ull : (1ull << rem) - 1));
    }
    __syncthreads();
    const int nkept = uni(bits_count(occ, n, ws1));
    // ---- kept operators ----
    const Bits& kept = occ;  // also: the new configuration's off-diagonal operators before the flip
    struct Kept { int i, info; double tau; };
    blk_each<4>(n,
                [&](int x) {
                  const int i = min(kept.rank(x), nkept - 1), k = nkept > 0 ? kept_at[i] : 0;
                  return Kept{i, oi_old[k], ot_old[k]};
                },
                [&](int x, const Kept& o) {
                  if (!kept.has(x)) return;
                  const int b = (o.info >> 3) - old_bond_base;
                  const int kr = o.i - off.rank(S.bo[b]);
                  const U4 w = philox(sweep, STAGE_REGRAPH, (uint32_t)b, (uint32_t)kr, P.key0, P.key1);
                  const uint64_t toff = (GEN && b >= P.nb_lat) ? (b >= P.nb_real ? (1ull << 32) : P.dtoff) : P.toff;
                  ot_new[x] = o.tau;
                  oi_new[x] = ((P.bond_base + b) << 3) | (((uint64_t)w.x < toff ? 0 : 1) << 1) | 1;
                });
    // sign problem: the off-diagonal operators of negative weight before the
    // flip (path_integral.C:551-576)
    int neg = 0;
    if (P.sgn_lattice) neg += kept.rank(S.bn[P.nb_lat]) - kept.rank(0);
    if (P.sgn_site) neg += nkept - kept.rank(S.bn[P.nb_real]);
    __syncthreads();
    // parities of the off-diagonal operators before each place, over the
    // previous configuration's set and the candidates' bits (which hold at
    // least a bit for each operator); the rest of the space follows
    unsigned long long* const pword = (unsigned long long*)S.rest;
    const uint32_t* const pbits = (const uint32_t*)pword;   // 2 * nw words
    for (int q = tid; q < nw; q += T) {
      unsigned long long v = kept.w[q] << 1;  // bit x: parity of the bits below x
      v ^= v << 1; v ^= v << 2; v ^= v << 4; v ^= v << 8; v ^= v << 16; v ^= v << 32;
      if (kept.pre[q] & 1) v = ~v;
      pword[q] = v;
    }
    __syncthreads();
    // ---- linking ----
    unsigned char* const sp3 = S.rest + (size_t)nw * 8;
    const int sp3_bytes = S.rest_bytes - nw * 8;
    auto par = [&](int x) -> int { return (int)((pbits[x >> 5] >> (x & 31)) & 1u); };
    const int cut3 = sp3_bytes >= 4 * n ? 32 : (sp3_bytes >= 2 * n ? 16 : 0);
    if (cut3 == 32) {
      blk_each<4>(n, [&](int k) { return cut_time(ot_new[k]); }, [&](int k, uint32_t v) { ((uint32_t*)sp3)[k] = v; });
    } else if (cut3 == 16) {
      blk_each<4>(n, [&](int k) { return (cut_time(ot_new[k]) >> 17) << 1; }, [&](int k, uint32_t v) { ((uint16_t*)sp3)[k] = (uint16_t)v; });
    }
    for (int s = tid; s < N; s += T) {
      int v = S.spin[s];
      auto add = [&](int b) { v ^= par(S.bn[b]); };
      if (!GEN) {
        const uint32_t in = S.into[s];
        if (P.kind == 0) { add(s); add((int)in); }
        else { add(2 * s); add(2 * s + 1); add((int)(in & 0xffffu)); add((int)(in >> 16)); }
      } else {
        for (int i = 0; i < S.nl; ++i) add(S.lists[s * S.nl + i]);
      }
      S.sbase[s] = (uint8_t)((v & 1) | (S.sbase[s] & 2));
    }
    __syncthreads();
    if (cut3 == 32) blk_link<GEN>(P, S, Cut32{(const uint32_t*)sp3, ot_new, 0}, par, n, ot_new, oi_new, evt_new, evflags, l0, l1);
    else if (cut3 == 16) blk_link<GEN>(P, S, Cut16{(const uint16_t*)sp3, ot_new, 0}, par, n, ot_new, oi_new, evt_new, evflags, l0, l1);
    else blk_link<GEN>(P, S, FullTimes{ot_new, nullptr, 0}, par, n, ot_new, oi_new, evt_new, evflags, l0, l1);
    __syncthreads();
    // ---- clusters ----
    // the space of the earlier steps is free from here on: the segments' flip
    // bits, the clusters' flip bits, the root set, then parents (16-bit where
    // they fit) and accumulators
    const int mw = bits_words(m);
    unsigned long long* const nflip = (unsigned long long*)S.rest;
    unsigned long long* const cflip = nflip + mw;
    const Bits roots = bits_at(S.rest + 16 * mw, m);
    unsigned char* const sp4 = S.rest + 16 * mw + bits_bytes(m);
    const int sp4_bytes = S.rest_bytes - 16 * mw - bits_bytes(m), pb = (2 * m + 7) & ~7;
    uint16_t* const p16 = (uint16_t*)sp4;
    const bool lds_p = m < 65536 && sp4_bytes >= pb;
    const int nc = uni(lds_p ? blk_clusters<GEN>(P, S, Parents16{p16}, sweep, n, m, oi_new, l0, l1, evflags, roots, root_of, ws0)
                             : blk_clusters<GEN>(P, S, ParentsMem{parents}, sweep, n, m, oi_new, l0, l1, evflags, roots, root_of, ws0));
    __syncthreads();
    // ---- flip bits (one bit of the root's Philox counter per cluster) ----
    const bool field = P.h != 0.0;
    if (!field) {
      const int end = (nc + 63) & ~63;
      for (int i = tid; i < end; i += T) {
        bool f = false;
        if (i < nc) f = philox(sweep, STAGE_FLIP, (uint32_t)root_of[i], 0u, P.key0, P.key1).x & 1u;
        const unsigned long long mk = __ballot(f);
        if (lane_id() == 0) cflip[i >> 6] = mk;
      }
    }
    // ---- estimators ----
    // accumulators behind the parents when every cluster has its own there;
    // else the segments' terms go to memory first, and the clusters take the
    // whole space a window at a time
    const bool direct = lds_p && sp4_bytes - pb >= ((nc + 63) & ~63) * ACC_BYTES;
    Acc ac;
    ac.W = direct ? (nc + 63) & ~63 : min((nc + 63) & ~63, (sp4_bytes / ACC_BYTES) & ~63);
    unsigned char* const wbase = direct ? sp4 + pb : sp4;
    ac.L = (double*)wbase;
    ac.n = (unsigned long long*)(wbase + (size_t)32 * ac.W);
    ac.w = ac.n + ac.W;
    if (direct)
      for (int i = tid; i < 6 * ac.W; i += T) ((unsigned long long*)wbase)[i] = 0;
    __syncthreads();
    auto root_at = [&](int x) -> int { return lds_p ? (int)p16[x] : ParentsMem{parents}.get(x); };
    // a segment's terms: into its cluster's accumulator, or to memory
    auto account = [&](int x, int id, double len, int fl, int flo) {
      int d0, d1;
      seg_winding(fl, flo, d0, d1);
      if (direct) {
        ac.add(id, len, fl & 3, d0, d1);
      } else {
        seg_len[x] = len;
        seg_info[x] = (uint32_t)id | ((uint32_t)(fl & 3) << 24) | ((uint32_t)(fl & SEG_FIRST) << 22) |
                      ((uint32_t)(d0 + 1) << 27) | ((uint32_t)(d1 + 1) << 29);
      }
    };
    {
      // U segments per thread at a time, every load of them before its use
      constexpr int U = 2;
      const int end = mw * 64;
      for (int x0 = tid; x0 < end; x0 += U * T) {
        int root[U], fl[U], flo[U];
        double thi[U], tlo[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int x = min(x0 + u * T, m - 1), lower = max(x - 1, 0);
          fl[u] = evflags[x];
          thi[u] = evt_new[x];
          tlo[u] = evt_new[lower];
          flo[u] = evflags[lower];
          root[u] = root_at(x);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int x = x0 + u * T;
          if ((x & ~63) >= end) break;  // (wave-uniform)
          bool f = false;
          if (x < m) {
            const int id = roots.rank(root[u]);
            if (!field) {
              f = (((const uint32_t*)cflip)[id >> 5] >> (id & 31)) & 1;
              seg_new[x] = (uint8_t)(((fl[u] >> 1) & 1) ^ (int)f);
            }
            if (!(fl[u] & SEG_FIRST)) account(x, id, thi[u] - tlo[u], fl[u], flo[u]);
          }
          const unsigned long long mk = __ballot(f);
          if (lane_id() == 0) nflip[x >> 6] = mk;
        }
      }
      // the sites' first segments: the segment below is the site's last (the
      // line wraps through tau = 1), a virtual site's begins at tau = 0; the
      // tau = 0 boundary counts with them
      for (int s = tid; s < N; s += T) {
        const int x = S.sn[s], last = S.sn[s + 1] - 1;
        const int fx = evflags[x], fy = evflags[last];
        const double tx = evt_new[x], ty = evt_new[last];
        const int id = roots.rank(root_at(x));
        const bool empty = (fx & SEG_EMPTY) != 0, nowrap = GEN && (fx & SEG_NOWRAP);
        const double len = empty ? 1.0 : (nowrap ? tx : (tx + 1.0) - ty);
        account(x, id, len, fx, empty ? fx : (nowrap ? 0 : fy));
        if (direct) atomicAdd(&ac.n[id], 1ull << (16 * (fx & 3)));
      }
    }
    __syncthreads();
    // the clusters' terms: by four waves when they are few, whose sums over
    // the lanes would cost the other waves more than the terms themselves
    const int TT = nc <= 1024 ? min(T, 256) : T;
    double v[NCOL];
#pragma unroll
    for (int q = 0; q < NCOL; ++q) v[q] = 0;
    for (int w0 = 0; w0 < nc; w0 += ac.W) {
      if (!direct) {
        for (int i = tid; i < 6 * ac.W; i += T) ((unsigned long long*)wbase)[i] = 0;
        __syncthreads();
        struct Seg { uint32_t info; double len; };
        blk_each<4>(m, [&](int x) { return Seg{seg_info[x], seg_len[x]}; },
                    [&](int, const Seg& g) {
                      const int a = (int)(g.info & 0xffffffu) - w0;
                      if ((unsigned)a < (unsigned)ac.W) {
                        const int cls = (int)(g.info >> 24) & 3;
                        ac.add(a, g.len, cls, (int)((g.info >> 27) & 3) - 1, (int)((g.info >> 29) & 3) - 1);
                        if ((g.info >> 26) & 1) atomicAdd(&ac.n[a], 1ull << (16 * cls));
                      }
                    });
        __syncthreads();
      }
      const int wend = min(ac.W, nc - w0), wround = (wend + 63) & ~63;
      for (int i = tid; i < wround; i += TT) {
        if (tid >= TT) break;
        bool f = false;
        if (i < wend) {
          ClusterAcc a;
#pragma unroll
          for (int q = 0; q < 4; ++q) a.L[q] = ac.L[4 * i + q];
          const unsigned long long cn = ac.n[i];
#pragma unroll
          for (int q = 0; q < 4; ++q) a.n[q] = (int)((cn >> (16 * q)) & 0xffffu);
          a.w = (long long)ac.w[i];
          if (field) {
            // k_field_flip of lg_kernels.hip
            const double umag = 0.5 * ((a.L[0] + a.L[1]) - (a.L[2] + a.L[3]));
            const double xw = beta * (-P.h * umag);
            const double u = uniform53(philox(sweep, STAGE_FLIP, (uint32_t)root_of[w0 + i], 0u, P.key0, P.key1));
            f = (2.0 * u - 1.0) < det_tanh(xw);
          } else {
            f = (cflip[(w0 + i) >> 6] >> ((w0 + i) & 63)) & 1;
          }
          double t[NCOL];
          cluster_terms(a, P.h, f, t);
#pragma unroll
          for (int q = 0; q < NCOL; ++q) v[q] += t[q];
        }
        if (field) {
          const unsigned long long mk = __ballot(f);
          if (lane_id() == 0) cflip[(w0 + i) >> 6] = mk;
        }
      }
      if (!direct) __syncthreads();
    }
    // the threads' sums (waves past the clusters hold zeros and skip it)
    const int tw = (min(nc, TT) + 63) / 64;
    if ((tid >> 6) < tw) {
#pragma unroll
      for (int q = 0; q < NCOL; ++q) v[q] = wave_total(v[q]);
      if (lane_id() == 63)
        for (int q = 0; q < NCOL; ++q) s_red[tid >> 6][q] = v[q];
    }
    // ---- flips ----
    if (field) {
      __syncthreads();
      const int end = mw * 64;
      for (int x = tid; x < end; x += T) {
        bool f = false;
        if (x < m) {
          const int id = direct ? roots.rank((int)p16[x]) : (int)(seg_info[x] & 0xffffffu);
          f = (cflip[id >> 6] >> (id & 63)) & 1;
          seg_new[x] = (uint8_t)(((evflags[x] >> 1) & 1) ^ (int)f);
        }
        const unsigned long long mk = __ballot(f);
        if (lane_id() == 0) nflip[x >> 6] = mk;
      }
    }
    __syncthreads();
    auto flip_of = [&](int x) -> int { return (int)((nflip[x >> 6] >> (x & 63)) & 1); };
    for (int s = tid; s < N; s += T) S.spin[s] ^= (uint8_t)flip_of(S.sn[s]);
    // the new off-diagonal set goes behind the segments' flip bits first
    unsigned long long* const noff = cflip;
    {
      constexpr int U = 4;
      for (int k0 = tid; k0 < nw * 64; k0 += U * T) {
        int info[U], a0[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = max(0, min(k0 + u * T, n - 1));
          info[u] = oi_new[k];
          a0[u] = l0[k];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int k = k0 + u * T;
          if ((k & ~63) >= nw * 64) break;  // (wave-uniform)
          bool o = false;
          if (k < n) {
            const int b0 = blk_up(S, a0[u], (int)(S.ends[(info[u] >> 3) - P.bond_base] & 0xffffu));
            const int f = flip_of(a0[u]) ^ flip_of(b0);
            if (f) oi_new[k] = info[u] ^ 1;
            o = (info[u] ^ f) & 1;
          }
          const unsigned long long mk = __ballot(o);
          if (lane_id() == 0) noff[k >> 6] = mk;
        }
      }
    }
    // ---- record ----
    double* const out = B.rec_ring + ((size_t)(A.slot0 + it) * B.nchains + c) * R_COUNT;
    if (tid < NCOL) {
      double t = 0;
      for (int w = 0; w < tw; ++w) t += s_red[w][tid];
      out[term_slot(tid)] = t;
      if (term_slot(tid) == R_EFIELD) out[R_ENERGY] = P.offset_total - (double)n / beta + t;
    }
    if (tid == NCOL) {
      out[R_NOP] = (double)n;
      out[R_BETA] = beta;
      out[R_SWEEP] = (double)sweep;
      out[R_SIGN] = (neg & 1) ? -1.0 : 1.0;
    }
    ++sweep;
    if (P.sched_n > 0) {  // annealing: the next sweep's inverse temperature
      beta = 1.0 / schedule_temperature(B.sched + 2 * P.sched_off, P.sched_n, (int)sweep);
      scale_lat = candidate_scale(beta, P.wsum);
      scale_site = candidate_scale(beta, P.site_w);
      scale_in = candidate_scale(beta, P.dwsum);
    }
    __syncthreads();
    // ---- the new configuration is the next sweep's previous one ----
    {
      // (the words move down over the flip bits; a thread's words at a time,
      // read by every thread before any is written)
      const Bits next = bits_at(S.rest, n);
      for (int q0 = 0; q0 < nw; q0 += T) {
        const unsigned long long v = q0 + tid < nw ? noff[q0 + tid] : 0;
        __syncthreads();
        if (q0 + tid < nw) next.w[q0 + tid] = v;
      }
      __syncthreads();
      bits_count(next, n, ws1);
    }
    int* t;
    t = S.bo; S.bo = S.bn; S.bn = t;
    t = S.so; S.so = S.sn; S.sn = t;
    S.n = n;
    S.m = m;
    old_bond_base = P.bond_base;
    ot_old = ot_new; oi_old = oi_new; evt_old = evt_new; seg_old = seg_new;
  }

  // ---- offsets, spins and counters of the last configuration ----
  const bool odd = A.nsweeps & 1;
  int* const bo_out = odd ? B.bo_new : const_cast<int*>(B.bo_old);
  int* const so_out = odd ? B.soff_new : const_cast<int*>(B.soff_old);
  uint8_t* const sp_out = odd ? B.spins_new : const_cast<uint8_t*>(B.spins_old);
  for (int b = tid; b < Nb; b += T) bo_out[P.bond_base + b] = P.blk_op + S.bo[b];
  for (int s = tid; s < N; s += T) {
    so_out[P.site_base + s] = P.blk_node + S.so[s];
    sp_out[P.site_base + s] = S.spin[s];
  }
  if (tid == 0) {
    if (B.nchains == 1) {  // one chain: the packed form too
      bo_out[Nb] = S.n;
      so_out[N] = S.m;
    }
    A.nops[c] = S.n;
    A.nnodes[c] = S.m;
    B.sweep[c] = sweep;
    ChainDev* Wc = B.chains + c;
    Wc->old_site_base = P.site_base;
    Wc->old_bond_base = P.bond_base;
    if (P.sched_n > 0) {
      Wc->beta = beta;
      Wc->scale = scale_lat;
      Wc->site_scale = scale_site;
      Wc->dscale = scale_in;
    }
  }
}

// What a launch of k_chain_sweeps raised stops the launches after it.
__global__ void k_chain_stop(DevBatch B) {
  if (B.flags[1]) B.flags[0] |= B.flags[1];
}

// Packed form of a batch whose chains stand in regions of their own: chain c's
// operators to op_base[c], its segments to node_base[c], into the other
// configuration's arrays; the batch's last chain closes the offsets.
__global__ void __launch_bounds__(256) k_pack(DevBatch B, const int* nops, const int* nnodes, const int* op_base,
                                              const int* node_base) {
  const int c = blockIdx.x;
  const ChainDev& P = B.chains[c];
  const int n = nops[c], m = nnodes[c], ob = op_base[c], nb = node_base[c];
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    B.ot_new[ob + k] = B.ot_old[P.blk_op + k];
    B.oi_new[ob + k] = B.oi_old[P.blk_op + k];
  }
  for (int x = threadIdx.x; x < m; x += blockDim.x) {
    B.evt_new[nb + x] = B.evt_old[P.blk_node + x];
    B.segspin_new[nb + x] = B.segspin_old[P.blk_node + x];
  }
  for (int b = threadIdx.x; b < P.Nb; b += blockDim.x)
    B.bo_new[P.bond_base + b] = B.bo_old[P.bond_base + b] - P.blk_op + ob;
  for (int s = threadIdx.x; s < P.N; s += blockDim.x) {
    B.soff_new[P.site_base + s] = B.soff_old[P.site_base + s] - P.blk_node + nb;
    B.spins_new[P.site_base + s] = B.spins_old[P.site_base + s];
  }
  if (c == B.nchains - 1 && threadIdx.x == 0) {
    B.bo_new[B.nbonds] = ob + n;
    B.soff_new[B.nsites] = nb + m;
  }
}

// LDS of the tables a workgroup keeps for a chain throughout, and of the
// accepted candidates' bits
static int blk_tables(const ChainDev& d) {
  auto r = [](int x) { return (x + 7) & ~7; };
  return 2 * r((d.Nb + 1) * 4) + 2 * r((d.N + 1) * 4) + r(d.Nb * 4) + r(d.N * 4) + r(d.N * 2 * chain_lists(d)) + 2 * r(d.N);
}
static int blk_accept(const ChainDev& d) { return (d.Nb * ((d.cand_cap + 31) / 32) * 4 + 7) & ~7; }

int block_lds_least(const ChainDev& d) {
  const int lists = 2 * bits_bytes(d.blk_opcap) + blk_accept(d) + bits_words(d.blk_opcap) * 8;
  const int clusters = std::max(16 * bits_words(d.blk_nodecap) + bits_bytes(d.blk_nodecap) + 64 * ACC_BYTES,
                                8 * bits_words(d.blk_nodecap) + 8 * bits_words(d.blk_opcap));
  return blk_tables(d) + std::max(lists, clusters);
}

int block_lds_for(const ChainDev& d, int n) {
  const int m = 2 * n + d.N;
  const int diag = bits_bytes(n) + blk_accept(d) + 4 * m;
  const int link = 2 * bits_bytes(n) + blk_accept(d) + bits_words(n) * 8 + 4 * n;
  const int clusters = 16 * bits_words(m) + bits_bytes(m) + 2 * m + 8 + (n * 6 / 10 + d.N / 2 + 64) * ACC_BYTES;
  return blk_tables(d) + std::max(diag, std::max(link, clusters));
}

int block_prepare() {
  for (const void* k : {(const void*)k_chain_sweeps<false>, (const void*)k_chain_sweeps<true>})
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, BLOCK_LDS_MAX) != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
  return 1;
}

void launch_pack(const DevBatch& B, const int* nops, const int* nnodes, const int* op_base, const int* node_base,
                 hipStream_t st) {
  hipLaunchKernelGGL(k_pack, dim3(B.nchains), dim3(256), 0, st, B, nops, nnodes, op_base, node_base);
}

void launch_chain_stop(const DevBatch& B, hipStream_t st) { hipLaunchKernelGGL(k_chain_stop, dim3(1), dim3(1), 0, st, B); }

void launch_chain_sweeps(const DevBatch& B, const BlockArgs& A, bool general, int threads, hipStream_t st) {
  if (general) hipLaunchKernelGGL(k_chain_sweeps<true>, dim3(A.grid), dim3(threads), A.lds, st, B, A);
  else hipLaunchKernelGGL(k_chain_sweeps<false>, dim3(A.grid), dim3(threads), A.lds, st, B, A);
}

}  // namespace lg
