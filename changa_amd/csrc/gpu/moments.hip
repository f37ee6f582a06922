// GPU multipole build: bucket P2M and level-synchronous M2M, in FP64.
//
// CPU semantics followed: GenericTreeNode::makeBucket (GenericTreeNode.h:
// 219-257) with MultipoleMoments::operator+=(particle) (MultipoleMoments.h:
// 276-352) for buckets, LocalTreeBuilder::doneChildren (Compute.cpp:
// 2534-2580) with operator+=(MultipoleMoments) (MultipoleMoments.h:207-272)
// for internal nodes, and calculateRadiusFarthestParticle /
// FarthestCorner (MultipoleMoments.h:460-505) for the expansion radius. The
// arithmetic kernels of the reference are momMakeFmomr, momShiftFmomr,
// momScaledAddFmomr and momRescaleFmomr (moments.c:202-268, 772-846,
// 1002-1058).
//
// Formulation. Moments are kept as "complete" symmetric components
// C(a,b,c) (a x's, b y's, c z's; orders 0 and 2..4, 35 slots with order 1
// unused). A bucket accumulates the raw moments sum_i m_i dx^a dy^b dz^c
// about its centre of mass and projects them once onto the symmetric
// trace-free (STF) subspace; the incremental per-particle shifting of the CPU
// build is the same sum. An internal node shifts each child's STF moments by
// the binomial rule for raw moments, R(a,b,c) = sum C(a,a1) C(b,b1) C(c,c1)
// Q(a1,b1,c1) d^(a-a1, b-b1, c-c1) (the dipole about a centre of mass is
// zero), adds the two children and projects onto the STF subspace again
// (trace parts of lower orders vanish under the projection). The shift runs
// axis by axis (moment_shift_axis), 105 FMAs per child. Stored moments
// are divided by radius^order (radius-scaled reduced moments).
#include "stf.h"

namespace cgpu {

// reduced (FMOMR order) <-> complete
__device__ __forceinline__ void complete_from_reduced(const double* q, double* C) {
  C[0] = q[0];
  C[1] = C[2] = C[3] = 0.0;
  C[cidx(2, 0, 0)] = q[1]; C[cidx(0, 2, 0)] = q[2]; C[cidx(1, 1, 0)] = q[3];
  C[cidx(1, 0, 1)] = q[4]; C[cidx(0, 1, 1)] = q[5];
  C[cidx(3, 0, 0)] = q[6]; C[cidx(1, 2, 0)] = q[7]; C[cidx(2, 1, 0)] = q[8];
  C[cidx(0, 3, 0)] = q[9]; C[cidx(2, 0, 1)] = q[10]; C[cidx(0, 2, 1)] = q[11];
  C[cidx(1, 1, 1)] = q[12];
  C[cidx(4, 0, 0)] = q[13]; C[cidx(1, 3, 0)] = q[14]; C[cidx(3, 1, 0)] = q[15];
  C[cidx(0, 4, 0)] = q[16]; C[cidx(3, 0, 1)] = q[17]; C[cidx(0, 3, 1)] = q[18];
  C[cidx(2, 2, 0)] = q[19]; C[cidx(2, 1, 1)] = q[20]; C[cidx(1, 2, 1)] = q[21];
  // z-heavy components from tracelessness, in increasing c
#pragma unroll
  for (int n = 2; n <= 4; ++n)
#pragma unroll
    for (int c = 2; c <= n; ++c)
#pragma unroll
      for (int a = 0; a <= n - c; ++a) {
        const int b = n - c - a;
        C[cidx(a, b, c)] = -(C[cidx(a + 2, b, c - 2)] + C[cidx(a, b + 2, c - 2)]);
      }
}

__device__ __forceinline__ void reduced_from_complete(const double* C, double* q) {
  q[0] = C[0];
  q[1] = C[cidx(2, 0, 0)]; q[2] = C[cidx(0, 2, 0)]; q[3] = C[cidx(1, 1, 0)];
  q[4] = C[cidx(1, 0, 1)]; q[5] = C[cidx(0, 1, 1)];
  q[6] = C[cidx(3, 0, 0)]; q[7] = C[cidx(1, 2, 0)]; q[8] = C[cidx(2, 1, 0)];
  q[9] = C[cidx(0, 3, 0)]; q[10] = C[cidx(2, 0, 1)]; q[11] = C[cidx(0, 2, 1)];
  q[12] = C[cidx(1, 1, 1)];
  q[13] = C[cidx(4, 0, 0)]; q[14] = C[cidx(1, 3, 0)]; q[15] = C[cidx(3, 1, 0)];
  q[16] = C[cidx(0, 4, 0)]; q[17] = C[cidx(3, 0, 1)]; q[18] = C[cidx(0, 3, 1)];
  q[19] = C[cidx(2, 2, 0)]; q[20] = C[cidx(2, 1, 1)]; q[21] = C[cidx(1, 2, 1)];
}

// Raw moments about a centre displaced by -d along one axis, in place:
// M'(a) = sum_{a1 <= a} binom(a, a1) d^(a - a1) M(a1) on every line of fixed
// exponents of the other two axes. This is the transpose of the Taylor
// shift's repeated synthetic division: n (n + 1) / 2 FMAs on a line of
// degree n, 35 per axis (the direct binomial sum over all three axes takes
// ~1,500 operations). Order-1 slots take part: they are zero about the
// child's centre of mass but not after the first axis.
template <int AXIS>
__device__ __forceinline__ void moment_shift_axis(double* P, double d) {
#pragma unroll
  for (int u = 0; u <= 4; ++u)
#pragma unroll
    for (int v = 0; v <= 4 - u; ++v) {
      const int n = 4 - u - v;  // degree along AXIS on this line
#pragma unroll
      for (int k = n - 1; k >= 0; --k)
#pragma unroll
        for (int e = k; e < n; ++e) {
          const int lo = AXIS == 0 ? cidx(e, u, v) : AXIS == 1 ? cidx(u, e, v) : cidx(u, v, e);
          const int hi = AXIS == 0 ? cidx(e + 1, u, v)
                                   : AXIS == 1 ? cidx(u, e + 1, v) : cidx(u, v, e + 1);
          P[hi] = fma(d, P[lo], P[hi]);
        }
    }
}

// write node outputs: node64 record, wire moments, cm64
__device__ __forceinline__ void emit(int nd, const double* g, const double* C, double u,
                                     CudaMultipoleMoments* out, double* node64, double* cm64) {
  double q[22];
  reduced_from_complete(C, q);
  const double iu = 1.0 / u;
  const double s2 = iu * iu, s3 = s2 * iu, s4 = s3 * iu;
#pragma unroll
  for (int k = 1; k < 22; ++k) q[k] *= (k < 6 ? s2 : k < 13 ? s3 : s4);
  double* rec = node64 + (size_t)nd * 34;
#pragma unroll
  for (int k = 0; k < 12; ++k) rec[k] = g[k];
  rec[3] = u;
#pragma unroll
  for (int k = 0; k < 22; ++k) rec[12 + k] = q[k];
  if (cm64) {
    cm64[3 * (size_t)nd] = g[0];
    cm64[3 * (size_t)nd + 1] = g[1];
    cm64[3 * (size_t)nd + 2] = g[2];
  }
  CudaMultipoleMoments m;
  m.radius = (float)u;
  m.soft = (float)g[4];
  m.totalMass = (float)g[5];
  m.cm.x = (float)g[0];
  m.cm.y = (float)g[1];
  m.cm.z = (float)g[2];
  m.xx = (float)q[1]; m.xy = (float)q[3]; m.xz = (float)q[4]; m.yy = (float)q[2]; m.yz = (float)q[5];
  m.xxx = (float)q[6]; m.xyy = (float)q[7]; m.xxy = (float)q[8]; m.yyy = (float)q[9];
  m.xxz = (float)q[10]; m.yyz = (float)q[11]; m.xyz = (float)q[12];
  m.xxxx = (float)q[13]; m.xyyy = (float)q[14]; m.xxxy = (float)q[15]; m.yyyy = (float)q[16];
  m.xxxz = (float)q[17]; m.yyyz = (float)q[18]; m.xxyy = (float)q[19]; m.xxyz = (float)q[20];
  m.xyyz = (float)q[21];
  out[nd] = m;
}

// Sum of v over the 4 lanes of a bucket's group (lanes 4g..4g+3), by an xor
// butterfly: every lane of the group gets the same bits ((v0 + v1) + (v2 + v3)
// up to commutation).
__device__ __forceinline__ double group4_sum(double v) {
  v += __shfl_xor(v, 1);
  return v + __shfl_xor(v, 2);
}
__device__ __forceinline__ double group4_min(double v) {
  v = fmin(v, __shfl_xor(v, 1));
  return fmin(v, __shfl_xor(v, 2));
}
__device__ __forceinline__ double group4_max(double v) {
  v = fmax(v, __shfl_xor(v, 1));
  return fmax(v, __shfl_xor(v, 2));
}

constexpr int kMomBlock = 256;
constexpr int kMomNodes = 128;  // nodes per block
constexpr int kMomHeld = 4;     // particles a lane keeps in registers between the passes

// node outputs of a leaf without particles: mass 0, centre 0 / 0, its box inside out
__device__ __forceinline__ void emit_empty(int nd, double u, CudaMultipoleMoments* out,
                                           double* node64, double* cm64) {
  constexpr double nan = __builtin_nan(""), inf = HUGE_VAL;
  const double g[12] = {nan, nan, nan, u, nan, 0.0, inf, inf, inf, -inf, -inf, -inf};
  const double C[35] = {};
  emit(nd, g, C, u, out, node64, cm64);
}

// Buckets (leaf nodes). A block takes kMomNodes consecutive nodes, compacts
// its leaves into LDS, and gives each leaf a group of 4 lanes: lane j of the
// group takes particles first + j, first + j + 4, ..., so each group reads its
// bucket's particles as contiguous 4-particle runs and every cache line it
// touches is used up within about one step (one lane per bucket, walking its
// own particles, kept ~10^5 partly read lines live at once and fetched each
// line several times over). Pass 1: mass, mass-weighted position and
// softening, bounding box; pass 2: the raw moments about the centre of mass
// and the farthest particle, summed over the group. The first kMomHeld
// particles of a lane (a whole bucket of 16) are loaded together and kept
// between the passes; a larger bucket's others are read again. One lane per
// bucket then projects and writes the records. About half the nodes are
// leaves, so 128 nodes keep the block's 64 groups busy once (256 nodes: two
// rounds in turn, 6 us longer on a tree that does not fill the device). With
// three wavefronts per SIMD (7 spills) instead of the 182 registers' two the
// build of the 2^22 halos takes 323 us, 329; of the 256^3 box 1,167, 1,187.
__global__ __launch_bounds__(kMomBlock) __attribute__((amdgpu_waves_per_eu(3))) void bucket_moments_kernel(
    int nNodes, const int* first, const int* count, const int* child, const double* boxRadius,
    const double* pos, const double* mass, const double* soft, CudaMultipoleMoments* out,
    double* node64, double* cm64) {
  __shared__ int leaves[kMomNodes];
  __shared__ int wave_base[kMomBlock / kWave + 1];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const int nd0 = blockIdx.x * kMomNodes + tid;
  const bool node = tid < kMomNodes && nd0 < nNodes;
  const int c0 = node ? child[2 * (size_t)nd0] : 0, n0 = node ? count[nd0] : 0;
  const bool leaf = c0 < 0 && n0 > 0;
  // a leaf without particles has nothing to load (handled here: as a branch
  // around the loads below it cost 25 to 56 more spills, and 6% of a small step)
  if (c0 < 0 && n0 <= 0) emit_empty(nd0, boxRadius[nd0], out, node64, cm64);
  const unsigned long long bal = __ballot(leaf);
  if (lane == 0) wave_base[wv + 1] = __popcll(bal);
  __syncthreads();
  if (tid == 0) {
    wave_base[0] = 0;
    for (int w = 1; w <= kMomBlock / kWave; ++w) wave_base[w] += wave_base[w - 1];
  }
  __syncthreads();
  if (leaf) leaves[wave_base[wv] + __popcll(bal & ((1ull << lane) - 1ull))] = nd0;
  __syncthreads();
  const int nleaf = wave_base[kMomBlock / kWave];
  const int sub = tid & 3;
  // a group's 4 lanes run the same trip counts, so its shuffles always pair
  // active lanes
  for (int j = tid >> 2; j < nleaf; j += kMomBlock / 4) {
    const int nd = leaves[j];
    const int f = first[nd], cnt = count[nd];
    double M = 0, sx = 0, sy = 0, sz = 0, ss = 0;
    double lo0 = HUGE_VAL, lo1 = HUGE_VAL, lo2 = HUGE_VAL;
    double hi0 = -HUGE_VAL, hi1 = -HUGE_VAL, hi2 = -HUGE_VAL;
    double hm[kMomHeld], hx[kMomHeld], hy[kMomHeld], hz[kMomHeld], hs[kMomHeld];
#pragma unroll
    for (int t = 0; t < kMomHeld; ++t) {
      const int i = min(f + sub + 4 * t, f + cnt - 1);
      hm[t] = mass[i];
      hx[t] = pos[3 * (size_t)i];
      hy[t] = pos[3 * (size_t)i + 1];
      hz[t] = pos[3 * (size_t)i + 2];
      hs[t] = soft[i];
    }
    auto first_pass = [&](double m, double x, double y, double z, double h) {
      M += m;
      sx += m * x;
      sy += m * y;
      sz += m * z;
      ss += m * h;
      lo0 = fmin(lo0, x); lo1 = fmin(lo1, y); lo2 = fmin(lo2, z);
      hi0 = fmax(hi0, x); hi1 = fmax(hi1, y); hi2 = fmax(hi2, z);
    };
#pragma unroll
    for (int t = 0; t < kMomHeld; ++t)
      if (sub + 4 * t < cnt) first_pass(hm[t], hx[t], hy[t], hz[t], hs[t]);
    for (int i = f + sub + 4 * kMomHeld; i < f + cnt; i += 4)
      first_pass(mass[i], pos[3 * (size_t)i], pos[3 * (size_t)i + 1], pos[3 * (size_t)i + 2],
                 soft[i]);
    double g[12];
    M = group4_sum(M);
    g[0] = group4_sum(sx) / M;
    g[1] = group4_sum(sy) / M;
    g[2] = group4_sum(sz) / M;
    g[4] = group4_sum(ss) / M;
    g[5] = M;
    g[6] = group4_min(lo0); g[7] = group4_min(lo1); g[8] = group4_min(lo2);
    g[9] = group4_max(hi0); g[10] = group4_max(hi1); g[11] = group4_max(hi2);
    double T[35];
#pragma unroll
    for (int k = 0; k < 35; ++k) T[k] = 0.0;
    double r2max = 0.0;
    auto second_pass = [&](double m, double x, double y, double z) {
      const double dx = x - g[0], dy = y - g[1], dz = z - g[2];
      r2max = fmax(r2max, dx * dx + dy * dy + dz * dz);
      double px[5], py[5], pz[5];
      px[0] = m;
      py[0] = pz[0] = 1.0;
#pragma unroll
      for (int k = 1; k < 5; ++k) {
        px[k] = px[k - 1] * dx;
        py[k] = py[k - 1] * dy;
        pz[k] = pz[k - 1] * dz;
      }
#pragma unroll
      for (int n = 2; n <= 4; ++n)
#pragma unroll
        for (int a = 0; a <= n; ++a)
#pragma unroll
          for (int b = 0; b <= n - a; ++b) {
            const int c = n - a - b;
            T[cidx(a, b, c)] += px[a] * py[b] * pz[c];
          }
    };
#pragma unroll
    for (int t = 0; t < kMomHeld; ++t)
      if (sub + 4 * t < cnt) second_pass(hm[t], hx[t], hy[t], hz[t]);
    for (int i = f + sub + 4 * kMomHeld; i < f + cnt; i += 4)
      second_pass(mass[i], pos[3 * (size_t)i], pos[3 * (size_t)i + 1], pos[3 * (size_t)i + 2]);
    T[0] = M;
#pragma unroll
    for (int n = 2; n <= 4; ++n)
#pragma unroll
      for (int a = 0; a <= n; ++a)
#pragma unroll
        for (int b = 0; b <= n - a; ++b) {
          const int k = cidx(a, b, n - a - b);
          T[k] = group4_sum(T[k]);
        }
    r2max = group4_max(r2max);
    if (sub == 0) {
      stf_project(T);
      const double u = (cnt > 1 && r2max > 0.0) ? sqrt(r2max) : boxRadius[nd];
      g[3] = u;
      emit(nd, g, T, u, out, node64, cm64);
    }
  }
}

// Two lanes per internal node of depth range [lo, hi), one per child: each
// shifts its child's moments to the node's centre of mass, a lane exchange
// adds them, and the even lane projects and writes. One lane per node
// shifting both children in turn measured 1-3% slower for the whole build.
__global__ __launch_bounds__(128) void internal_moments_kernel(int lo, int hi, const int* child,
                                                               CudaMultipoleMoments* out,
                                                               double* node64, double* cm64) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x, sub = t & 1;
  const int nd = lo + (t >> 1);
  if (nd >= hi) return;
  const int c = child[2 * (size_t)nd + sub];
  if (c < 0) return;  // a leaf: both lanes
  const double* r = node64 + (size_t)c * 34;
  double v[34];
#pragma unroll
  for (int k = 0; k < 34; ++k) v[k] = r[k];
  // this child's value and its sibling's, first child first
  auto both = [&](double a, double& x0, double& x1) {
    const double o = __shfl_xor(a, 1);
    x0 = sub ? o : a;
    x1 = sub ? a : o;
  };
  double g[12], M0, M1;
  both(v[5], M0, M1);
  const double M = M0 + M1;
  g[5] = M;
  double a0, a1;
  both(v[4], a0, a1);
  g[4] = (M0 * a0 + M1 * a1) / M;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    both(v[k], a0, a1);
    g[k] = (M0 * a0 + M1 * a1) / M;
    g[6 + k] = fmin(v[6 + k], __shfl_xor(v[6 + k], 1));
    g[9 + k] = fmax(v[9 + k], __shfl_xor(v[9 + k], 1));
  }
  double d2 = 0.0;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    double e1 = g[k] - g[6 + k], e2 = g[9 + k] - g[k];
    double e = e1 > e2 ? e1 : e2;
    d2 += e * e;
  }
  const double u = sqrt(d2);
  g[3] = u;
  double q[22], C[35];
  const double uc = v[3], s2 = uc * uc, s3 = s2 * uc, s4 = s3 * uc;
#pragma unroll
  for (int k = 0; k < 22; ++k) q[k] = v[12 + k] * (k == 0 ? 1.0 : k < 6 ? s2 : k < 13 ? s3 : s4);
  complete_from_reduced(q, C);
  moment_shift_axis<0>(C, v[0] - g[0]);
  moment_shift_axis<1>(C, v[1] - g[1]);
  moment_shift_axis<2>(C, v[2] - g[2]);
#pragma unroll
  for (int k = 0; k < 35; ++k) C[k] += __shfl_xor(C[k], 1);
  if (sub) return;
  stf_project(C);
  emit(nd, g, C, u, out, node64, cm64);
}
// Several depths in one launch, for depths of few nodes, whose own launches
// wait on one another: one wavefront per node of the depths [d0, d0 + n),
// each taking its moments straight from its descendants at depth d0 + n (or
// leaves above it), one per lane, at most 2^n <= 64 of them: lane j follows
// bit s of j at its s-th step down, and a leaf met early belongs to the lane
// whose remaining bits are zero. The shift and the projection are the
// per-depth kernel's; shifting a descendant at once instead of through the
// nodes between differs in FP64 rounding only.
//
// A per-depth launch of few nodes takes 3.4 us whatever their number (the
// chain of one node: index, record, two shifts, projection, stores); a
// launch of up to six depths about 7. kGroupNodes, the nodes of a run of
// depths up to which it goes into one launch: a wavefront per node does up
// to 32 times the shifts, which must stay below the launches saved. Build
// time with 0 (a launch per depth) / 1,024 / 4,096 / 16,384 nodes: 2^16
// Plummer 160 / 112 / 89 / 84 us, 128^3 box 267 / 236 / 227 / 250, 2^22
// halos 412 / 371 / 360 / 383; 2^12 Plummer 108 / 54 / 54 / 55.
constexpr int kGroupLevels = 6;
constexpr int kGroupNodes = 4096;
struct GroupLevels {
  int n;                      // depths of this launch
  int off[kGroupLevels + 1];  // node range of depth d0 + i: [off[i], off[i + 1])
};

__global__ __launch_bounds__(kWave) void group_moments_kernel(GroupLevels lv, const int* child,
                                                              CudaMultipoleMoments* out,
                                                              double* node64, double* cm64) {
  __shared__ double red[35][kWave + 1];
  const int lane = threadIdx.x;
  const int nd = lv.off[0] + blockIdx.x;
  int c0 = child[2 * (size_t)nd], c1 = child[2 * (size_t)nd + 1];
  if (c0 < 0) return;  // a leaf: its moments are there
  int i = 0;
  while (i + 1 < lv.n && nd >= lv.off[i + 1]) ++i;
  const int steps = lv.n - i;
  bool mine = lane < (1 << steps);
  int src = (lane & 1) ? c1 : c0;
  for (int s = 1; s < steps; ++s) {
    if (mine) {
      c0 = child[2 * (size_t)src];
      c1 = child[2 * (size_t)src + 1];
      if (c0 >= 0) {
        src = ((lane >> s) & 1) ? c1 : c0;
      } else {
        mine = (lane >> s) == 0;
        break;
      }
    }
  }
  const double* r = node64 + (size_t)src * 34;
  double v[34] = {};
  if (mine) {
#pragma unroll
    for (int k = 0; k < 34; ++k) v[k] = r[k];
  }
  // mass, centre of mass, softening, bounding box over the lanes
  double sum[5] = {v[5], v[5] * v[0], v[5] * v[1], v[5] * v[2], v[5] * v[4]};
  double lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lo[k] = mine ? v[6 + k] : HUGE_VAL;
    hi[k] = mine ? v[9 + k] : -HUGE_VAL;
  }
  for (int m = 1; m < (1 << steps); m <<= 1) {
#pragma unroll
    for (int k = 0; k < 5; ++k) sum[k] += __shfl_xor(sum[k], m, kWave);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = fmin(lo[k], __shfl_xor(lo[k], m, kWave));
      hi[k] = fmax(hi[k], __shfl_xor(hi[k], m, kWave));
    }
  }
  double g[12];
  const double M = sum[0];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    g[k] = sum[1 + k] / M;
    g[6 + k] = lo[k];
    g[9 + k] = hi[k];
  }
  g[4] = sum[4] / M;
  g[5] = M;
  double C[35];
  {
    double q[22];
    const double s2 = v[3] * v[3], s3 = s2 * v[3], s4 = s3 * v[3];
#pragma unroll
    for (int k = 0; k < 22; ++k)
      q[k] = v[12 + k] * (k == 0 ? 1.0 : k < 6 ? s2 : k < 13 ? s3 : s4);
    complete_from_reduced(q, C);
    moment_shift_axis<0>(C, v[0] - g[0]);
    moment_shift_axis<1>(C, v[1] - g[1]);
    moment_shift_axis<2>(C, v[2] - g[2]);
  }
  if (lane < (1 << steps)) {
#pragma unroll
    for (int k = 0; k < 35; ++k) red[k][lane] = mine ? C[k] : 0.0;
  }
  __syncthreads();
  if (lane < 35) {
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    const int n = 1 << steps;
    for (int j = 0; j < n; j += 4)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j + u < n) t[u] += red[lane][j + u];
    red[lane][0] = (t[0] + t[1]) + (t[2] + t[3]);
  }
  __syncthreads();
  if (lane == 0) {
    double d2 = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const double e1 = g[k] - g[6 + k], e2 = g[9 + k] - g[k];
      const double e = e1 > e2 ? e1 : e2;
      d2 += e * e;
    }
    const double u = sqrt(d2);
    g[3] = u;
#pragma unroll
    for (int k = 0; k < 35; ++k) C[k] = red[k][0];
    stf_project(C);
    emit(nd, g, C, u, out, node64, cm64);
  }
}

}  // namespace cgpu

using namespace cgpu;

extern "C" int changaBuildMoments(int nNodes, int nDepths, const int* levelOffsets,
                                  const int* first, const int* count, const int* child,
                                  const double* boxRadius, const double* pos, const double* mass,
                                  const double* soft, CudaMultipoleMoments* moments,
                                  double* node64, double* cm64, void* stream) {
  if (nNodes <= 0) return 0;
  if (!levelOffsets || !first || !count || !child || !boxRadius || !pos || !mass || !soft ||
      !moments || !node64)
    return fail("changaBuildMoments: missing argument", hipErrorInvalidValue, __FILE__, __LINE__);
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(bucket_moments_kernel, dim3((nNodes + kMomNodes - 1) / kMomNodes),
                     dim3(kMomBlock), 0, s, nNodes,
                     first, count, child, boxRadius, pos, mass, soft, moments, node64, cm64);
  CGPU_CHECK(hipGetLastError());
  // The deepest depth holds leaves only. Above it, runs of depths with at
  // most kGroupNodes nodes together go into one launch.
  for (int d = nDepths - 2; d >= 0;) {
    GroupLevels lv = {};
    int d0 = d + 1;
    while (d0 > 0 && d + 1 - (d0 - 1) <= kGroupLevels &&
           levelOffsets[d + 1] - levelOffsets[d0 - 1] <= kGroupNodes)
      --d0;
    if (d0 < d) {
      lv.n = d + 1 - d0;
      for (int i = 0; i <= lv.n; ++i) lv.off[i] = levelOffsets[d0 + i];
      const int nodes = lv.off[lv.n] - lv.off[0];
      if (nodes > 0) {
        hipLaunchKernelGGL(group_moments_kernel, dim3(nodes), dim3(kWave), 0, s, lv, child,
                           moments, node64, cm64);
        CGPU_CHECK(hipGetLastError());
      }
      d = d0 - 1;
      continue;
    }
    const int lo = levelOffsets[d], hi = levelOffsets[d + 1];
    --d;
    if (hi <= lo) continue;
    hipLaunchKernelGGL(internal_moments_kernel, dim3((hi - lo + 63) / 64), dim3(128), 0, s, lo,
                       hi, child, moments, node64, cm64);
    CGPU_CHECK(hipGetLastError());
  }
  return 0;
}
