// Device helpers shared by the sweep kernels (lg_kernels.hip) and the
// one-workgroup-per-chain sweep (lg_block.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "lg_common.h"
#include "lg_kernels.h"

namespace lg {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__device__ __forceinline__ bool overflowed(const DevBatch& B) {
  return __hip_atomic_load(B.flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

// one thread, in the kernel before a scan: clear the ticket, next epoch
// (never 0, the value of freshly cleared status words)
__device__ __forceinline__ void scan_advance_epoch(const DevBatch& B) {
  B.scan_ctl[0] = 0;
  uint32_t e = ((uint32_t)B.scan_ctl[1] + 1u) & 0x3fffffffu;
  B.scan_ctl[1] = (int)(e == 0 ? 1u : e);
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Sum of v over the wave, in its last lane, by DPP adds: the same sum by
// shuffles is a dozen LDS operations, which for the collector's 19 terms took
// a seventh of its time (chain L=1024, beta=1000: 30 -> 26 us).  k_estimate,
// which has two and no register left, is faster with wave_sum_d (121 us
// against 129 at square 128^2, beta=128).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
  return v + __longlong_as_double((long long)(((unsigned long long)(uint32_t)hi << 32) | (uint32_t)lo));
}
__device__ __forceinline__ double wave_total(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);
  return dpp_add<0x143, 0xc>(v);
}

// one of eight values by a run-time index, chosen from registers
template <typename T>
__device__ __forceinline__ T pick8(int i, T a0, T a1, T a2, T a3, T a4, T a5, T a6, T a7) {
  return i < 4 ? (i == 0 ? a0 : i == 1 ? a1 : i == 2 ? a2 : a3) : (i == 4 ? a4 : i == 5 ? a5 : i == 6 ? a6 : a7);
}

// tau boundary of the virtual sites (S > 1/2; path_integral.C:589-615, the
// S > 1/2 branch of the symmetrization): per real site, the tau = 0 ends
// (lowest segments) of its nv virtual sites are joined to their tau = 1 ends
// (top segments) by a permutation that maps equal spins onto each other,
// uniform among those that do (looper::partitioned_random_shuffle,
// looper/permutation.h:88-112).  For each spin value u = 0, 1 in turn, the
// bottoms of spin u in virtual-site order are matched to the tops of spin u
// in virtual-site order permuted by Fisher-Yates: for i = n_u - 1 down to 1,
// j = i - (x mod (i + 1)) with x the next word of the stream (word k is word
// k mod 4 of Philox(sweep, STAGE_BOUNDARY, real site, k / 4)), swap
// positions i and j.  (The spins at tau = 1 are those at tau = 0 in some
// order: every update keeps each real site's magnetization periodic.)  For
// nv = 2 with equal spins this is the exchange iff bit 0 of the first word
// is set.  nv <= 8, so a permutation lives in one
// register as eight 4-bit fields.  bot / top: the real site's lowest and top
// segments, bs / es: their spins, bit a for virtual site a.
template <class Unite>
__device__ __forceinline__ void join_boundary(const ChainDev& P, uint32_t sweep, int r, const int* bot, const int* top,
                                              uint32_t bs, uint32_t es, Unite unite) {
  constexpr int NV = MAX_NV;
  const int nv = P.nv;
  const uint32_t all = (1u << nv) - 1;
  // words 0..3, and 4..7 when the two shuffles can take more than four
  // (n_0 - 1 + n_1 - 1 <= nv - 1 words in all)
  const U4 x0 = philox(sweep, STAGE_BOUNDARY, (uint32_t)r, 0u, P.key0, P.key1);
  U4 x1 = {0u, 0u, 0u, 0u};
  if (nv > 5) x1 = philox(sweep, STAGE_BOUNDARY, (uint32_t)r, 1u, P.key0, P.key1);
  int k = 0;
  uint32_t perm[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int n = __popc(u ? (bs & all) : (~bs & all));
    uint32_t p = 0x76543210u;
#pragma unroll
    for (int i = NV - 1; i >= 1; --i) {
      if (i < n) {
        const uint32_t w = pick8(k, x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w);
        const int j = i - (int)(w % (uint32_t)(i + 1));
        ++k;
        const uint32_t vi = (p >> (4 * i)) & 15u, vj = (p >> (4 * j)) & 15u;
        p &= ~((15u << (4 * i)) | (15u << (4 * j)));
        p |= (vi << (4 * j)) | (vj << (4 * i));
      }
    }
    perm[u] = p;
  }
#pragma unroll
  for (int a = 0; a < NV; ++a) {
    if (a >= nv) continue;
    const uint32_t u = (bs >> a) & 1u;
    const uint32_t cls_b = u ? bs : ~bs, cls_e = u ? es : ~es;
    const int rank = __popc(cls_b & all & ((1u << a) - 1));
    const int t = (int)(((u ? perm[1] : perm[0]) >> (4 * rank)) & 15u);
    // the top of spin u with rank t among the tops of spin u
    int target = 0, cnt = 0;
#pragma unroll
    for (int q = 0; q < NV; ++q) {
      if (q < nv && ((cls_e >> q) & 1u)) {
        if (cnt == t) target = q;
        ++cnt;
      }
    }
    unite(bot[a], pick8(target, top[0], top[1], top[2], top[3], top[4], top[5], top[6], top[7]));
  }
}

constexpr int NCOL = NUM_COLLECTOR_TERMS;

// Collector terms of one cluster.  h, flip: the chain's field and the
// cluster's flip; the field weight of the cluster is w = -h umag
// (cluster.h:50-63) and its Zeeman energy after the flip flip ? -w : w
// (path_integral.C:852-858).
__device__ __forceinline__ void cluster_terms(const ClusterAcc& a, double h, int flip, double* v) {
  const double L0 = a.L[0], L1 = a.L[1], L2 = a.L[2], L3 = a.L[3];
  const int n0 = a.n[0], n1 = a.n[1], n2 = a.n[2], n3 = a.n[3];
  int w0, w1;
  unpack_winding(a.w, w0, w1);
  // per-cluster improved estimates (susceptibility.h:96-147 with sigma = 1-2c)
  const double usize0 = 0.5 * (n0 + n1 + n2 + n3), umag0 = 0.5 * (n0 + n1 - n2 - n3);
  const double ssize0 = 0.5 * (n0 - n1 + n2 - n3), smag0 = 0.5 * (n0 - n1 - n2 + n3);
  const double usize = 0.5 * ((L0 + L1) + (L2 + L3)), umag = 0.5 * ((L0 + L1) - (L2 + L3));
  const double ssize = 0.5 * ((L0 - L1) + (L2 - L3)), smag = 0.5 * ((L0 - L1) - (L2 - L3));
  v[0] = 1.0;  // clusters
  v[1] = umag0;
  v[2] = usize0 * usize0;
  v[3] = umag0 * umag0;
  v[4] = v[2] * v[2];
  v[5] = v[3] * v[3];
  v[6] = usize * usize;
  v[7] = umag * umag;
  v[8] = smag0;
  v[9] = ssize0 * ssize0;
  v[10] = smag0 * smag0;
  v[11] = v[9] * v[9];
  v[12] = v[10] * v[10];
  v[13] = ssize * ssize;
  v[14] = smag * smag;
  v[15] = 0.25 * ((double)w0 * w0 + (double)w1 * w1);
  v[16] = umag;   // normal estimator: tau-integrated magnetization
  v[17] = smag;
  const double wf = -h * umag;
  v[18] = flip ? -wf : wf;
}

// record slot of collector term q (R_NC, R_UMAG0 .. R_W2, R_UMAGA, R_SMAGA, R_EFIELD)
__device__ __forceinline__ int term_slot(int q) {
  return q == 0 ? R_NC : (q <= 15 ? R_UMAG0 + (q - 1) : R_UMAGA + (q - 16));
}

}  // namespace lg
