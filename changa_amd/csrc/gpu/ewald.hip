// Ewald correction kernel: real-space replica sum plus k-space h-loop of the
// root multipole, per active particle.
//
// CPU semantics followed: TreePiece::BucketEwald (Ewald.cpp:72-281). The
// GPU work split of the reference is EwaldKernel (HostCUDA.cu:1958-2192).
//
//  - d = x - cm_root. Real space: lattice vectors n in [-nEwReps, nEwReps]^3
//    (nEwReps = max(ceil(fEwCut), nReps)); a term is skipped when
//    |d + nL|^2 > (fEwCut L)^2 unless n is in the "hole" |n_i| <= nReps, whose
//    terms use -erf (the tree already summed those replicas) instead of erfc.
//  - Radial kernels g_0..g_5 by the recursion g_(n+1) = (2n+1) g_n / r^2 +
//    (2 alpha^2)^n ka e^(-alpha^2 r^2) / r^2, or by the two-term series about
//    r = 0 when r^2 < 1.2e-3 L^2 (the CPU switch, Ewald.cpp:119).
//  - Multipole contraction with the root's STF moments at unit scale:
//    phi -= sum_n (1/n!) g_n Q_n . r^n,
//    a   += sum_n (1/n!) [n g_n Q_n . r^(n-1) - g_(n+1) (Q_n . r^n) r].
//  - k space: phi += hC cos(k.d) + hS sin(k.d), a += k (hC sin - hS cos).
//
// Precision: the central replica (n = 0, the only term that can reach small
// r, where the -erf kernels cancel catastrophically in FP32) is evaluated in
// FP64 with the CPU's series switch; every other term in FP32. All per-particle
// sums run in FP64 and are added into the FP32 result array at the end.
//
// Work split: one lane per active particle in tree order, so a wavefront
// holds spatially close particles. Each wavefront bounds its particles' d,
// keeps only the lattice vectors any of them can need (compacted into LDS),
// then every lane applies the exact per-particle test. The h-loop table is
// staged in LDS (dynamic size; no 80-entry limit).
//
// Bound by FP32 VALU issue: about 80 replica terms of 165 instructions and 73
// k-space pairs of 26 per particle. 2^21 particles take 0.68 ms (0.92 with
// library error functions, 185 instructions a term, all 146 k-space entries,
// divisions in the candidate search and four wavefronts per SIMD).
#include "ewald_body.h"

namespace cgpu {

// The root's moments for the FP32 replica terms: Q_n / n! with the trace
// combinations formed, one value for the whole wavefront (scalar registers:
// 25 vector registers fewer, so five wavefronts per SIMD instead of four).
struct EwaldMom32 {
  float m, xx, yy, xy, xz, yz, zz;
  float xxx, xyy, xxy, yyy, xxz, yyz, xyz, q3a, q3b;
  float xxxx, xyyy, xxxy, yyyy, xxxz, yyyz, xxyy, xxyz, xyyz, q4a, q4b, q4c;
};

__device__ __forceinline__ float uniform(double v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int((float)v)));
}

__device__ __forceinline__ EwaldMom32 ewald_mom32(const Mom22<double>& Q) {
  const double h = 0.5, s = 1.0 / 6.0, f = 1.0 / 24.0;
  EwaldMom32 o;
  o.m = uniform(Q.m);
  o.xx = uniform(h * Q.xx); o.yy = uniform(h * Q.yy); o.xy = uniform(h * Q.xy);
  o.xz = uniform(h * Q.xz); o.yz = uniform(h * Q.yz); o.zz = uniform(-h * (Q.xx + Q.yy));
  o.xxx = uniform(s * Q.xxx); o.xyy = uniform(s * Q.xyy); o.xxy = uniform(s * Q.xxy);
  o.yyy = uniform(s * Q.yyy); o.xxz = uniform(s * Q.xxz); o.yyz = uniform(s * Q.yyz);
  o.xyz = uniform(s * Q.xyz);
  o.q3a = uniform(-s * (Q.xxx + Q.xyy)); o.q3b = uniform(-s * (Q.xxy + Q.yyy));
  o.xxxx = uniform(f * Q.xxxx); o.xyyy = uniform(f * Q.xyyy); o.xxxy = uniform(f * Q.xxxy);
  o.yyyy = uniform(f * Q.yyyy); o.xxxz = uniform(f * Q.xxxz); o.yyyz = uniform(f * Q.yyyz);
  o.xxyy = uniform(f * Q.xxyy); o.xxyz = uniform(f * Q.xxyz); o.xyyz = uniform(f * Q.xyyz);
  o.q4a = uniform(-f * (Q.xxxx + Q.xxyy)); o.q4b = uniform(-f * (Q.yyyy + Q.xxyy));
  o.q4c = uniform(-f * (Q.xxxy + Q.xyyy));
  return o;
}

// One replica term (ewald_term's sums) with V_n = Q_n . r^(n-1) / n! and
// p_n = V_n . r:  pot = -(g0 m + g2 p2 + g3 p3 + g4 p4),
//   a = 2 g2 V2 + 3 g3 V3 + 4 g4 V4 - (g1 m + g3 p2 + g4 p3 + g5 p4) r.
__device__ __forceinline__ void ewald_term32(const EwaldMom32& Q, float x, float y, float z,
                                             const float* g, float& pot, float& ax, float& ay,
                                             float& az) {
  const float x2 = x * x, y2 = y * y, z2 = z * z;
  const float fxx = x2 - z2, fyy = y2 - z2;
  const float x_2 = x + x, y_2 = y + y;
  const float fxy = x_2 * y, fxz = x_2 * z, fyz = y_2 * z;
  const float fxxx = x * __builtin_fmaf(-3.0f, z2, x2), fyyy = y * __builtin_fmaf(-3.0f, z2, y2);
  const float fxyy = (3.0f * x) * fyy, fxxy = (3.0f * y) * fxx;
  const float fxxz = z * __builtin_fmaf(3.0f, x2, -z2), fyyz = z * __builtin_fmaf(3.0f, y2, -z2);
  const float fxyz = (3.0f * z) * fxy;
  const float v2x = Q.xx * x + Q.xy * y + Q.xz * z;
  const float v2y = Q.xy * x + Q.yy * y + Q.yz * z;
  const float v2z = Q.xz * x + Q.yz * y + Q.zz * z;
  const float v3x = Q.xxx * fxx + Q.xyy * fyy + Q.xxy * fxy + Q.xxz * fxz + Q.xyz * fyz;
  const float v3y = Q.xyy * fxy + Q.xxy * fxx + Q.yyy * fyy + Q.yyz * fyz + Q.xyz * fxz;
  const float v3z = Q.xxz * fxx + Q.yyz * fyy + Q.xyz * fxy + Q.q3a * fxz + Q.q3b * fyz;
  const float v4x = Q.xxxx * fxxx + Q.xxyy * fxyy + Q.xxxy * fxxy + Q.xyyy * fyyy +
                    Q.xxxz * fxxz + Q.xyyz * fyyz + Q.xxyz * fxyz;
  const float v4y = Q.yyyy * fyyy + Q.xxyy * fxxy + Q.xxxy * fxxx + Q.xyyy * fxyy +
                    Q.xyyz * fxyz + Q.xxyz * fxxz + Q.yyyz * fyyz;
  const float v4z = Q.xxxz * fxxx + Q.xyyz * fxyy + Q.xxyz * fxxy + Q.yyyz * fyyy + Q.q4a * fxxz +
                    Q.q4b * fyyz + Q.q4c * fxyz;
  const float p2 = v2x * x + v2y * y + v2z * z;
  const float p3 = v3x * x + v3y * y + v3z * z;
  const float p4 = v4x * x + v4y * y + v4z * z;
  pot = -(g[0] * Q.m + g[2] * p2 + g[3] * p3 + g[4] * p4);
  const float ta = g[1] * Q.m + g[3] * p2 + g[4] * p3 + g[5] * p4;
  const float c2 = 2.0f * g[2], c3 = 3.0f * g[3], c4 = 4.0f * g[4];
  ax = c2 * v2x + c3 * v3x + c4 * v4x - ta * x;
  ay = c2 * v2y + c3 * v3y + c4 * v4y - ta * y;
  az = c2 * v2z + c3 * v3z + c4 * v4z - ta * z;
}

// radial32 with the error functions of x = alpha r >= 1 (all but a few
// particles near a replica's copy of the root centre) from the exponential
// the recursion needs anyway: erfc(x) = e^(-x^2) P(t), t = 1 / (1 + x / 2),
// -erf = erfc - 1. P: degree-7 least-maximum fit of erfc(x) e^(x^2) on
// 0.98 <= x <= 6.3 (own fit, relative error 1e-8; 2.2e-7 up to 7, 5.2e-6 up
// to 9.2, 1e-4 up to 15, where it does not matter: erfc is below 1e-17 past
// 6.3, far under the sums' FP64 rounding of terms of order one). With
// e^(-x^2) from the unrounded x^2 the relative error of erfc is at most
// 3.4e-7 for x <= 6.2, where erfcf of the rounded x gives 6.5e-6, at a third
// of its instructions.
__device__ __forceinline__ void radial32_fast(float r2, float hole, float alpha, float alpha2,
                                              float ka, float inner2, float* g) {
  const float dir = rsqrtf(r2), ir2 = dir * dir;
  const float x = alpha * (r2 * dir);
  if (r2 < inner2 || x < 1.0f) {
    radial32(r2, hole != 0.0f, alpha, alpha2, ka, inner2, g);
    return;
  }
  const float ex = expf(-alpha2 * r2);
  const float t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.5f, x, 1.0f));
  float pt = 1.008342766e-01f;
  pt = __builtin_fmaf(pt, t, -4.093811133e-01f);
  pt = __builtin_fmaf(pt, t, 4.758980659e-01f);
  pt = __builtin_fmaf(pt, t, -3.587170541e-02f);
  pt = __builtin_fmaf(pt, t, 3.166909518e-01f);
  pt = __builtin_fmaf(pt, t, 2.681522595e-01f);
  pt = __builtin_fmaf(pt, t, 2.836491832e-01f);
  pt = __builtin_fmaf(pt, t, -7.436778299e-05f);
  g[0] = __builtin_fmaf(ex, pt, -hole) * dir;
  const float e = ka * ex * ir2;
  float s = 1.0f;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    g[k + 1] = (2 * k + 1) * g[k] * ir2 + s * e;
    s *= 2 * alpha2;
  }
}

// LDS beside the k-space table, whose size is the caller's: 32 bytes an entry,
// in all at most the CU's 160 KB (4,348 entries). The runtime does not refuse
// a launch that asks for more, the queue aborts; launch_ewald checks.
struct EwLds {
  // lattice offsets (n L, hole flag): all of them, then those that some
  // particle of the wavefront needs, in place
  float4 cand[kEwBlock / kWave][kEwMaxCand];
  // the k-space table as weights on the cube |h_i| <= kEwCube (zero off the table)
  float2 cube[kEwCubeN];
  int n_outside, n_uneven;
};
constexpr size_t kEwLdsMax = 160 * 1024;

__global__ __launch_bounds__(kEwBlock) __attribute__((amdgpu_waves_per_eu(5))) void ewald_kernel(const CompactPartData* parts,
                                                         VariablePartData* vars,
                                                         const int* markers, int first, int n,
                                                         const EwtData* ewt, const double* pos64,
                                                         const double* root, EwaldParams p) {
  // h-loop table: per entry (k, hC) and (h as integers, hS); dynamic size
  extern __shared__ float4 sh[];
  __shared__ EwLds lds;
  auto& cand = lds.cand;
  auto& cube = lds.cube;
  int &n_outside = lds.n_outside, &n_uneven = lds.n_uneven;

  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  const float kscale = (float)(p.L / (2.0 * M_PI));  // k -> integer h
  for (int i = tid; i < kEwCubeN; i += kEwBlock) cube[i] = make_float2(0.0f, 0.0f);
  if (tid == 0) n_outside = n_uneven = 0;
  __syncthreads();
  for (int i = tid; i < p.nH; i += kEwBlock) {
    EwtData e = ewt[i];
    const float hx = rintf(e.hx * kscale), hy = rintf(e.hy * kscale), hz = rintf(e.hz * kscale);
    sh[2 * i] = make_float4(e.hx, e.hy, e.hz, e.hCfac);
    sh[2 * i + 1] = make_float4(hx, hy, hz, e.hSfac);
    if (fabsf(hx) <= kEwCube && fabsf(hy) <= kEwCube && fabsf(hz) <= kEwCube) {
      const int ci = ((int)hx + kEwCube) * kEwCubeW * kEwCubeW + ((int)hy + kEwCube) * kEwCubeW +
                     (int)hz + kEwCube;
      cube[ci] = make_float2(e.hCfac, e.hSfac);
    } else {
      atomicAdd(&n_outside, 1);
    }
  }

  // hC is even in h and hS odd (Ewald.cpp:359-381), so h and -h give the same
  // term: with a table that holds both, the cube's upper half is doubled and
  // the lower one cleared (and its planes skipped); any other table is kept
  __syncthreads();
  if (tid < kEwCubeN / 2) {
    const float2 u = cube[tid], v = cube[kEwCubeN - 1 - tid];
    if (u.x != v.x || u.y != -v.y) atomicAdd(&n_uneven, 1);
  }
  __syncthreads();
  const bool even = n_uneven == 0;
  if (even && tid < kEwCubeN / 2) {
    const float2 v = cube[kEwCubeN - 1 - tid];
    cube[kEwCubeN - 1 - tid] = make_float2(2.0f * v.x, 2.0f * v.y);
    cube[tid] = make_float2(0.0f, 0.0f);
  }

  // root centre of mass, k = 0 term and moments: from the device root record
  // (changaEwaldRoot) when there is one, else from the parameters
  const double cmx = root ? root[0] : p.cmx, cmy = root ? root[1] : p.cmy,
               cmz = root ? root[2] : p.cmz;
  const double mk1 = root ? root[3] * M_PI / (p.alpha2 * p.L * p.L * p.L) : p.mk1;
  const int gi = blockIdx.x * kEwBlock + tid;
  const bool live = gi < n;
  const int id = live ? (markers ? markers[gi] : first + gi) : (markers ? markers[n - 1] : first + n - 1);
  double dx, dy, dz;
  if (pos64) {
    dx = pos64[3 * (size_t)id] - cmx;
    dy = pos64[3 * (size_t)id + 1] - cmy;
    dz = pos64[3 * (size_t)id + 2] - cmz;
  } else {
    CompactPartData q = parts[id];
    dx = (double)q.position.x - cmx;
    dy = (double)q.position.y - cmy;
    dz = (double)q.position.z - cmz;
  }
  // wavefront bounding box of d (dead lanes hold a live lane's particle)
  float lo[3] = {(float)dx, (float)dy, (float)dz}, hi[3] = {lo[0], lo[1], lo[2]};
#pragma unroll
  for (int m = 1; m < kWave; m <<= 1)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      lo[k] = fminf(lo[k], __shfl_xor(lo[k], m, kWave));
      hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], m, kWave));
    }
  // the lattice vectors, found once for the block
  const int W = 2 * p.nEwReps + 1, NC = W * W * W;
  const float Lf = (float)p.L, cut2f = (float)p.cut2;
  for (int c = tid; c < NC; c += kEwBlock) {
    const int ix = c / (W * W) - p.nEwReps, iy = (c / W) % W - p.nEwReps, iz = c % W - p.nEwReps;
    const bool hole = abs(ix) <= p.nReps && abs(iy) <= p.nReps && abs(iz) <= p.nReps;
#pragma unroll
    for (int w = 0; w < kEwBlock / kWave; ++w)
      cand[w][c] = make_float4(ix * Lf, iy * Lf, iz * Lf, hole ? 1.0f : 0.0f);
  }
  __syncthreads();
  // those that some particle of the wavefront needs, compacted: a step writes
  // at most as many entries as were read up to its end, after its reads
  int nc = 0;
  for (int c0 = 0; c0 < NC; c0 += kWave) {
    const int c = c0 + lane;
    const float4 v = cand[wv][min(c, NC - 1)];
    const float n[3] = {v.x, v.y, v.z};
    const bool hole = v.w != 0.0f, centre = v.x == 0.0f && v.y == 0.0f && v.z == 0.0f;
    float d2 = 0.f;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const float l = lo[k] + n[k], h = hi[k] + n[k];
      const float e = l > 0.f ? l : (h < 0.f ? -h : 0.f);
      d2 += e * e;
    }
    // slack for FP32 rounding of the bound; the per-particle test is exact
    const bool need = c < NC && !centre && (hole || d2 <= cut2f * 1.0001f + 1e-6f * Lf * Lf);
    const unsigned long long mask = __ballot(need);
    if (need) cand[wv][nc + __popcll(mask & ((1ull << lane) - 1ull))] = v;
    nc += __popcll(mask);
  }
  __syncthreads();

  Mom22<double> Qd;
  {
    double* qd = &Qd.m;
#pragma unroll
    for (int k = 0; k < 22; ++k) qd[k] = root ? root[4 + k] : p.q[k];
  }
  const EwaldMom32 Qf = ewald_mom32(Qd);
  double pot = mk1, ax = 0, ay = 0, az = 0;
  // central replica in FP64
  {
    double g[6];
    radial64(dx * dx + dy * dy + dz * dz, p.nReps >= 0, p, g);
    ewald_term<double>(Qd, dx, dy, dz, g, pot, ax, ay, az);
  }
  const float fx = (float)dx, fy = (float)dy, fz = (float)dz;
  const float alpha = (float)p.alpha, alpha2 = (float)p.alpha2, ka = (float)p.ka,
              inner2 = (float)p.inner2, cut2 = (float)p.cut2;
  for (int k = 0; k < nc; ++k) {
    const float4 cv = cand[wv][k];
    float x = fx + cv.x, y = fy + cv.y, z = fz + cv.z;
    float r2 = x * x + y * y + z * z;
    if (r2 > cut2 && cv.w == 0.0f) continue;
    float g[6];
    radial32_fast(r2, cv.w, alpha, alpha2, ka, inner2, g);
    float tp, tx, ty, tz;
    ewald_term32(Qf, x, y, z, g, tp, tx, ty, tz);
    pot += tp;
    ax += tx;
    ay += ty;
    az += tz;
  }
  // k space. On the cube |h_i| <= kEwCube: e^(2 pi i h.u) (u = d / L) as the
  // product of per-axis powers of e^(2 pi i u_x) etc., which are formed once
  // per particle; the plane hx is advanced by one complex multiplication.
  // Compensated FP32 sums within a plane (the residual c is subtracted when
  // the plane's sum is carried into FP64), FP64 across planes.
  const float iL = (float)(1.0 / p.L);
  const float ux = fx * iL, uy = fy * iL, uz = fz * iL;
  {
    float2 ey[kEwCubeW], ez[kEwCubeW];
    float2 e1x;
    sincospif(2.0f * ux, &e1x.y, &e1x.x);
    axis_powers(uy, ey);
    axis_powers(uz, ez);
    const int hx0 = even ? 0 : -kEwCube;
    float2 ex = even ? make_float2(1.0f, 0.0f) : cpow_neg(e1x);  // e^(2 pi i hx0 u_x)
    const float kf = (float)(2.0 * M_PI / p.L);
    for (int hx = hx0; hx <= kEwCube; ++hx) {
      KahanF sp, st, sy, sz;
      const float2* cw = cube + (hx + kEwCube) * kEwCubeW * kEwCubeW;
#pragma unroll
      for (int hy = -kEwCube; hy <= kEwCube; ++hy) {
        const float2 exy = cmul(ex, ey[hy + kEwCube]);
        KahanF row;  // sum of t at this hy
#pragma unroll
        for (int hz = -kEwCube; hz <= kEwCube; ++hz) {
          const float2 wgt = cw[(hy + kEwCube) * kEwCubeW + hz + kEwCube];
          if (wgt.x != 0.0f || wgt.y != 0.0f) {
            const float2 e = cmul(exy, ez[hz + kEwCube]);
            sp.add(wgt.x * e.x + wgt.y * e.y);
            const float t = wgt.x * e.y - wgt.y * e.x;
            row.add(t);
            if (hz != 0) sz.add((float)hz * t);
          }
        }
        st.add(row.s);
        st.c += row.c;
        if (hy != 0) {
          sy.add((float)hy * row.s);
          sy.c += (float)hy * row.c;
        }
      }
      pot += (double)sp.s - (double)sp.c;
      ax += (double)kf * (double)hx * ((double)st.s - (double)st.c);
      ay += (double)kf * ((double)sy.s - (double)sy.c);
      az += (double)kf * ((double)sz.s - (double)sz.c);
      ex = cmul(ex, e1x);
    }
  }
  // entries off the cube (a table cut beyond |h_i| = kEwCube): phase h.d / L
  // in revolutions (h integer), reduced exactly, then sin / cos of 2 pi that
  if (n_outside > 0) {
    for (int i = 0; i < p.nH; ++i) {
      const float4 e0 = sh[2 * i];
      const float4 e1 = sh[2 * i + 1];
      if (fabsf(e1.x) <= kEwCube && fabsf(e1.y) <= kEwCube && fabsf(e1.z) <= kEwCube) continue;
      const float hs = e1.w;
      float ph = e1.x * ux + e1.y * uy + e1.z * uz;
      ph -= rintf(ph);
      float s, c;
      sincospif(2.0f * ph, &s, &c);
      pot += (double)(e0.w * c + hs * s);
      float t = e0.w * s - hs * c;
      ax += (double)(e0.x * t);
      ay += (double)(e0.y * t);
      az += (double)(e0.z * t);
    }
  }
  if (live) {
    VariablePartData v = vars[id];
    v.a.x += (float)ax;
    v.a.y += (float)ay;
    v.a.z += (float)az;
    v.potential += (float)pot;
    vars[id] = v;
  }
}

// Builds the kernel parameters from the reference's read-only record; with
// d_root (a device record of changaEwaldRoot) the root's centre of mass, mass
// and moments come from there instead of ro and rootCm64.
int launch_ewald(const CompactPartData* parts, VariablePartData* vars, const int* markers,
                 int first, int n, const EwaldReadOnlyData* ro, const EwtData* d_ewt,
                 const double* pos64, const double* rootCm64, const double* d_root,
                 hipStream_t s) {
  if (n <= 0) return 0;
  EwaldParams p = make_params(ro, rootCm64);
  if (p.nEwReps > 3)
    return fail("Ewald: nEwReps > 3", hipErrorInvalidValue, __FILE__, __LINE__);
  size_t shm = sizeof(float4) * 2 * (size_t)(p.nH > 0 ? p.nH : 1);
  if (sizeof(EwLds) + shm > kEwLdsMax)
    return fail("Ewald: nEwhLoop too large (its table is staged in LDS)", hipErrorInvalidValue,
                __FILE__, __LINE__);
  int blocks = (n + kEwBlock - 1) / kEwBlock;
  hipLaunchKernelGGL(ewald_kernel, dim3(blocks), dim3(kEwBlock), shm, s, parts, vars, markers,
                     first, n, d_ewt, pos64, d_root, p);
  CGPU_CHECK(hipGetLastError());
  return 0;
}

// ---------------------------------------------------------------------------
// EwaldInit on the device (Ewald.cpp:285-383): the root record (centre of
// mass, mass, the 22 reduced moments brought to unit scale, the first 22
// MOMC components of momRescaleFmomr + momFmomr2Momc) and the h-loop table,
// from the root's node record node64[0] (cm.xyz, radius, soft, mass,
// lo.xyz, hi.xyz, 22 radius-scaled reduced moments). One block: each thread
// takes one lattice vector h of the cube |h_i| <= hreps, the valid ones
// (0 < |h|^2 <= hcut^2) are numbered in the host table's order (hx
// outermost, hz innermost) by a block scan, and each writes its entry:
//   k = 2 pi h / L,  w = exp(-k^2 / 4 alpha^2) / (pi h^2 L),  alpha = 2 / L,
//   hC = -w (M - (Q2:kk)/2 + (Q4:kkkk)/24),  hS = w (Q3:kkk)/6.
// ---------------------------------------------------------------------------
constexpr int kRootBlock = 512;

__global__ __launch_bounds__(kRootBlock) void ewald_root_kernel(const double* node64, double L,
                                                                double hcut2, int hreps,
                                                                double* root, EwtData* ewt) {
  __shared__ double q[22];
  __shared__ int wave_count[kRootBlock / kWave];
  __shared__ int base;
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wv = tid / kWave;
  if (tid < 22) {
    const int order = tid == 0 ? 0 : (tid < 6 ? 2 : (tid < 13 ? 3 : 4));
    const double u = node64[3];
    double s = 1.0;
    for (int k = 0; k < order; ++k) s *= u;
    q[tid] = node64[12 + tid] * s;
    root[4 + tid] = q[tid];
  }
  if (tid < 3) root[tid] = node64[tid];
  if (tid == 3) root[3] = node64[5];
  if (tid == 0) base = 0;
  __syncthreads();
  const double m = q[0], xx = q[1], yy = q[2], xy = q[3], xz = q[4], yz = q[5];
  const double zz = -(xx + yy);
  const double xxx = q[6], xyy = q[7], xxy = q[8], yyy = q[9], xxz = q[10], yyz = q[11],
               xyz = q[12];
  const double xzz = -(xxx + xyy), yzz = -(xxy + yyy), zzz = -(xxz + yyz);
  const double xxxx = q[13], xyyy = q[14], xxxy = q[15], yyyy = q[16], xxxz = q[17],
               yyyz = q[18], xxyy = q[19], xxyz = q[20], xyyz = q[21];
  const double xxzz = -(xxxx + xxyy), xyzz = -(xxxy + xyyy), xzzz = -(xxxz + xyyz),
               yyzz = -(xxyy + yyyy), yzzz = -(xxyz + yyyz), zzzz = -(xxzz + yyzz);
  const double alpha = 2.0 / L;
  const double k4 = M_PI * M_PI / (alpha * alpha * L * L);
  const double f = 2.0 * M_PI / L;
  const int W = 2 * hreps + 1, NC = W * W * W;
  for (int c0 = 0; c0 < NC; c0 += kRootBlock) {
    const int c = c0 + tid;
    const int hx = c / (W * W) - hreps, hy = (c / W) % W - hreps, hz = c % W - hreps;
    const int h2 = hx * hx + hy * hy + hz * hz;
    const bool valid = c < NC && h2 != 0 && (double)h2 <= hcut2;
    const unsigned long long mask = __ballot(valid);
    if (lane == 0) wave_count[wv] = __popcll(mask);
    __syncthreads();
    int idx = base + __popcll(mask & ((1ull << lane) - 1ull));
    for (int k = 0; k < wv; ++k) idx += wave_count[k];
    if (valid) {
      const double x = f * hx, y = f * hy, z = f * hz;
      const double w = exp(-k4 * h2) / (M_PI * h2 * L);
      const double q2 = xx * x * x + yy * y * y + zz * z * z +
                        2 * (xy * x * y + xz * x * z + yz * y * z);
      const double q3 = xxx * x * x * x + yyy * y * y * y + zzz * z * z * z +
                        3 * (xxy * x * x * y + xxz * x * x * z + xyy * x * y * y +
                             yyz * y * y * z + xzz * x * z * z + yzz * y * z * z) +
                        6 * xyz * x * y * z;
      const double q4 = xxxx * x * x * x * x + yyyy * y * y * y * y + zzzz * z * z * z * z +
                        4 * (xxxy * x * x * x * y + xxxz * x * x * x * z + xyyy * x * y * y * y +
                             yyyz * y * y * y * z + xzzz * x * z * z * z + yzzz * y * z * z * z) +
                        6 * (xxyy * x * x * y * y + xxzz * x * x * z * z + yyzz * y * y * z * z) +
                        12 * (xxyz * x * x * y * z + xyyz * x * y * y * z + xyzz * x * y * z * z);
      EwtData e;
      e.hx = (float)x;
      e.hy = (float)y;
      e.hz = (float)z;
      e.hCfac = (float)(-w * (m - 0.5 * q2 + q4 / 24.0));
      e.hSfac = (float)(w * q3 / 6.0);
      ewt[idx] = e;
    }
    __syncthreads();
    if (tid == 0)
      for (int k = 0; k < kRootBlock / kWave; ++k) base += wave_count[k];
    __syncthreads();
  }
}

int launch_ewald_root(const double* node64, const EwaldReadOnlyData* ro, double hcut,
                      double* root, EwtData* ewt, hipStream_t s) {
  if (!node64 || !ro || !root || (!ewt && ro->nEwhLoop > 0) || !(hcut >= 0.0) || ro->L <= 0.0f)
    return fail("changaEwaldRoot: missing argument", hipErrorInvalidValue, __FILE__, __LINE__);
  const int hreps = (int)ceil(hcut);
  const double hcut2 = hcut * hcut;
  int count = 0;
  for (int hx = -hreps; hx <= hreps; ++hx)
    for (int hy = -hreps; hy <= hreps; ++hy)
      for (int hz = -hreps; hz <= hreps; ++hz) {
        const int h2 = hx * hx + hy * hy + hz * hz;
        count += h2 != 0 && (double)h2 <= hcut2;
      }
  if (count != ro->nEwhLoop)
    return fail("changaEwaldRoot: ro->nEwhLoop is not the number of h with 0 < |h|^2 <= hCut^2",
                hipErrorInvalidValue, __FILE__, __LINE__);
  hipLaunchKernelGGL(ewald_root_kernel, dim3(1), dim3(kRootBlock), 0, s, node64, (double)ro->L,
                     hcut2, hreps, root, ewt);
  CGPU_CHECK(hipGetLastError());
  return 0;
}

}  // namespace cgpu
