// Per-bucket particle-cell and particle-particle kernels and their C-ABI
// launchers (changaNodeGravity, changaPartGravity, changaZeroVars,
// changaAddVars). The
// interaction bodies and the per-chunk loops are in gravity_body.h, shared
// with the persistent batched kernel of batch.hip.
#include "gravity_body.h"

namespace cgpu {

// float4 of LDS per wavefront
constexpr int kPcLds = (kPcTile + 1) * (kFwdRec / 4);
constexpr int kPpLds = (sizeof(PpFwdLds<kPpTile>) + 15) / 16;
static_assert(kPcLds * sizeof(float4) >= reduce_bytes<2>() &&
                  kPpLds * sizeof(float4) >= reduce_bytes<3>(),
              "reduction");

// ---------------------------------------------------------------------------
// Per-bucket particle-cell kernel: one workgroup per bucket, of one wavefront
// or, in launches of few buckets, of several that share its list (Team);
// buckets mapped to XCDs in contiguous ranges (xcd_bucket).
// ---------------------------------------------------------------------------
// REC: cells from the 128-byte cell records, else from the wire moments; in
// tiles of 64 either way (records in tiles of 32: 128^3 box 2.34 ms against
// 2.22, 256^3 box with a 10% rung 8.05 against 6.11). At most two targets
// per lane: no spills at four wavefronts per SIMD.
template <bool PRECISE, bool REC>
__global__ __launch_bounds__(kWave * kTeamWaves) __attribute__((amdgpu_waves_per_eu(4))) void
pc_kernel(ChangaGravityLaunch a) {
  // staged tile of each wavefront; reused for the slot reduction at the end
  // of each chunk
  extern __shared__ float4 lds[];
  const int lane = threadIdx.x & (kWave - 1);
  const Team team = block_team();
  float4* rec4 = lds + team.wave * kPcLds;

  const int b = xcd_bucket(blockIdx.x, a.numBuckets);
  const int start = a.marks[b], end = a.marks[b + 1];
  const int bstart = a.starts[b], n = a.sizes[b];
  double cx0, cy0, cz0;
  bucket_centre<PRECISE>(a.tpos64, bstart, n, cx0, cy0, cz0);

  for (int t0 = 0; t0 < n; t0 += kWave) {
    const int nt = min(kWave, n - t0);
    with_targets_per_lane<2, true>(nt, [&](auto kt) {
      constexpr int K = decltype(kt)::value;
      const Lanes l = lanes_for<K>(lane, nt);
      Target t[K];
      load_targets<PRECISE, K>(a, bstart + t0, l, cx0, cy0, cz0, t);
      Acc64 acc[K];
#pragma unroll
      for (int j = 0; j < K; ++j) acc[j] = {0.0, 0.0, 0.0, 0.0, 0.0f};
      pc_cells<PRECISE, kPcTile, true, K, REC>(a, team.share(start, end),
                                               team.share_end(start, end), cx0, cy0, cz0, t, l,
                                               rec4, acc);
      reduce_store<K>(reinterpret_cast<char*>(lds), kPcLds * sizeof(float4), team, l, acc,
                      a.vars + bstart + t0);
    });
  }
}

// ---------------------------------------------------------------------------
// Per-bucket particle-particle kernel (KIND: see pp_sources). TEAM: the build
// for several wavefronts per bucket. The one for a single wavefront has its
// tiles in a static array and no team arithmetic: 2^20 sphere 404 us against
// 419 for the TEAM build with one wavefront, 128^3 box 596 / 612, 2^22 halos
// 2,872 / 2,905 (half of it from the array: its LDS addresses are constants).
// ---------------------------------------------------------------------------
template <bool PRECISE, int KIND, bool TEAM>
__global__ __launch_bounds__(kWave * (TEAM ? kTeamWaves : 1))
__attribute__((amdgpu_waves_per_eu(4))) void pp_kernel(ChangaGravityLaunch a) {
  // staged tiles of each wavefront; reused for the slot reduction at the end
  // of each chunk
  extern __shared__ float4 team_lds[];
  __shared__ float4 own_lds[TEAM ? 1 : kPpLds];
  float4* lds = TEAM ? team_lds : own_lds;
  const int lane = threadIdx.x & (kWave - 1);
  const Team team = TEAM ? block_team() : Team{1, 0};
  PpFwdLds<kPpTile>& s = *reinterpret_cast<PpFwdLds<kPpTile>*>(lds + team.wave * kPpLds);

  const int b = xcd_bucket(blockIdx.x, a.numBuckets);
  const int start = a.marks[b], end = a.marks[b + 1];
  const int bstart = a.starts[b], n = a.sizes[b];
  double cx0, cy0, cz0;
  bucket_centre<PRECISE>(a.tpos64, bstart, n, cx0, cy0, cz0);

  for (int t0 = 0; t0 < n; t0 += kWave) {
    const int nt = min(kWave, n - t0);
    with_targets_per_lane<3, false>(nt, [&](auto kt) {
      constexpr int K = decltype(kt)::value;
      const Lanes l = lanes_for<K>(lane, nt);
      Target t[K];
      load_targets<PRECISE, K>(a, bstart + t0, l, cx0, cy0, cz0, t);
      Acc64 acc[K];
#pragma unroll
      for (int j = 0; j < K; ++j) acc[j] = {0.0, 0.0, 0.0, 0.0, 0.0f};
      pp_sources<PRECISE, KIND, kPpTile, true, K>(a, team.share(start, end),
                                                  team.share_end(start, end), cx0, cy0, cz0, t, l,
                                                  s, acc);
      reduce_store<K>(reinterpret_cast<char*>(lds), kPpLds * sizeof(float4), team, l, acc,
                      a.vars + bstart + t0);
    });
  }
}

template <bool TEAM>
static auto pick_pp(const ChangaGravityLaunch& a) {
  if (a.listKind == 0)
    return a.tpos64 ? pp_kernel<true, 0, TEAM> : pp_kernel<false, 0, TEAM>;
  return a.tpos64 ? pp_kernel<true, 1, TEAM> : pp_kernel<false, 1, TEAM>;
}

// 128-byte cell records (kCellRecFloats): centre of mass as 3 doubles, mass,
// softening, then the moments scaled as stage_cell_fwd scales them (same
// FP32 operations, so both staging paths give identical records).
__global__ void cell_records_kernel(const CudaMultipoleMoments* mom, const double* cm64, int n,
                                    float4* out) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* w = reinterpret_cast<const float*>(mom) + (size_t)i * kWireStride;
  float v[27];
#pragma unroll
  for (int k = 0; k < 27; ++k) v[k] = w[wire_float(k)];
  double c[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) c[k] = cm64 ? cm64[3 * (size_t)i + k] : (double)v[3 + k];
  float r[kCellRecFloats];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const long long b = __double_as_longlong(c[k]);
    r[2 * k] = __int_as_float((int)(unsigned)(b & 0xffffffffll));
    r[2 * k + 1] = __int_as_float((int)(unsigned)((unsigned long long)b >> 32));
  }
  r[F_M] = v[2];
  r[F_SOFT] = v[1];
  const float u = v[0], u2 = u * u;
  const float s2 = 3.0f * u2, s3 = 7.5f * u2 * u, s4 = 17.5f * u2 * u2;
#pragma unroll
  for (int k = 0; k < 5; ++k) r[F_Q2 + k] = s2 * v[6 + k];
  r[F_Q2 + 5] = -(r[F_Q2 + 0] + r[F_Q2 + 3]);
#pragma unroll
  for (int k = 0; k < 7; ++k) r[F_Q3 + k] = s3 * v[11 + k];
  r[F_Q3 + 7] = -(r[F_Q3 + 0] + r[F_Q3 + 1]);
  r[F_Q3 + 8] = -(r[F_Q3 + 2] + r[F_Q3 + 3]);
#pragma unroll
  for (int k = 0; k < 9; ++k) r[F_Q4 + k] = s4 * v[18 + k];
  float4* o = out + (size_t)i * (kCellRecFloats / 4);
#pragma unroll
  for (int k = 0; k < kCellRecFloats / 4; ++k)
    o[k] = make_float4(r[4 * k], r[4 * k + 1], r[4 * k + 2], r[4 * k + 3]);
}

__global__ void zero_vars_kernel(VariablePartData* v, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = VariablePartData{{0.f, 0.f, 0.f}, 0.f, 0.f};
}

// dst += src with the result array's semantics (+= for a and the potential,
// max for dtGrav)
__global__ void add_vars_kernel(VariablePartData* dst, const VariablePartData* src, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  VariablePartData d = dst[i];
  const VariablePartData s = src[i];
  d.a.x += s.a.x;
  d.a.y += s.a.y;
  d.a.z += s.a.z;
  d.potential += s.potential;
  d.dtGrav = fmaxf(d.dtGrav, s.dtGrav);
  dst[i] = d;
}

// A launch over no buckets (an empty rung) needs no arrays.
static int check_launch(const ChangaGravityLaunch* a) {
  if (!a || a->numBuckets < 0 ||
      (a->numBuckets > 0 && (!a->marks || !a->starts || !a->sizes || !a->vars || !a->targets)))
    return fail("gravity launch: missing argument", hipErrorInvalidValue, __FILE__, __LINE__);
  return 0;
}

}  // namespace cgpu

using namespace cgpu;

extern "C" int changaNodeGravity(const ChangaGravityLaunch* a, void* stream) {
  if (int e = check_launch(a)) return e;
  if (a->numBuckets == 0) return 0;
  if (!a->moments || !a->list)
    return fail("changaNodeGravity: moments/list", hipErrorInvalidValue, __FILE__, __LINE__);
  if (a->tpos64 && !a->cm64)
    return fail("changaNodeGravity: precision form needs cm64", hipErrorInvalidValue, __FILE__,
                __LINE__);
  if (a->variant != 0)
    return fail("changaNodeGravity: variant must be 0", hipErrorInvalidValue, __FILE__, __LINE__);
  if (reinterpret_cast<uintptr_t>(a->cellRecords) % CHANGA_CELL_RECORD_BYTES != 0)
    return fail("changaNodeGravity: cellRecords not 128-byte aligned", hipErrorInvalidValue,
                __FILE__, __LINE__);
  hipStream_t s = (hipStream_t)stream;
  // us with 1 / 2 / 4 wavefronts per bucket: 541 buckets 18 / 12 / 11, 2,074
  // 41 / 34 / 32, 7,985 136 / 129 / 136, 15,948 262 / 263 / 278, 20,185 of a
  // sparse rung 109 / 129 / 178. Four stop at 1,024 because requests also come
  // on several streams, which fill the card by themselves: cells and particles
  // of 8 requests on 8 streams took 264 / 333 us at 1,550 / 1,872 buckets with
  // four, 231 / 304 with two, 220 / 275 with one (a single one 57 / 66, 61 /
  // 66, 74 / 80).
  const int waves = team_waves(a->numBuckets, 1024, 8192);
  const auto kernel = a->cellRecords ? (a->tpos64 ? pc_kernel<true, true> : pc_kernel<false, true>)
                                     : (a->tpos64 ? pc_kernel<true, false> : pc_kernel<false, false>);
  hipLaunchKernelGGL(kernel, dim3(a->numBuckets), dim3(kWave * waves),
                     waves * kPcLds * sizeof(float4), s, *a);
  CGPU_CHECK(hipGetLastError());
  return 0;
}

extern "C" int changaCellRecords(const CudaMultipoleMoments* moments, const double* cm64,
                                 int numCells, void* records, void* stream) {
  if (numCells < 0 || (numCells > 0 && (!moments || !records)))
    return fail("changaCellRecords: missing argument", hipErrorInvalidValue, __FILE__, __LINE__);
  if (numCells > CHANGA_CELL_RECORD_MAX)
    return fail("changaCellRecords: more than CHANGA_CELL_RECORD_MAX cells", hipErrorInvalidValue,
                __FILE__, __LINE__);
  if (reinterpret_cast<uintptr_t>(records) % CHANGA_CELL_RECORD_BYTES != 0)
    return fail("changaCellRecords: records not 128-byte aligned", hipErrorInvalidValue,
                __FILE__, __LINE__);
  if (numCells == 0) return 0;
  hipLaunchKernelGGL(cell_records_kernel, dim3((numCells + 255) / 256), dim3(256), 0,
                     (hipStream_t)stream, moments, cm64, numCells, static_cast<float4*>(records));
  CGPU_CHECK(hipGetLastError());
  return 0;
}

extern "C" int changaPartGravity(const ChangaGravityLaunch* a, void* stream) {
  if (int e = check_launch(a)) return e;
  if (a->numBuckets == 0) return 0;
  if (!a->sources || !a->list)
    return fail("changaPartGravity: sources/list", hipErrorInvalidValue, __FILE__, __LINE__);
  if (a->tpos64 && !a->spos64)
    return fail("changaPartGravity: precision form needs spos64", hipErrorInvalidValue, __FILE__,
                __LINE__);
  hipStream_t s = (hipStream_t)stream;
  // the lists are a third of the cells' in time: 541 buckets 23 / 17 / 13 us
  // with 1 / 2 / 4 wavefronts per bucket, 2,074 25 / 23 / 25, 3,850 16 / 19 /
  // 30, 7,985 43 / 52 / 72. (Two of 1,550 / 1,872 buckets: 26 / 29 us against
  // 34 / 36 with one; 8 streams of them 108 / 128 against 95 / 104, which the
  // cells' kernels more than make up.)
  const int waves = team_waves(a->numBuckets, 1024, 2048);
  const auto kernel = waves > 1 ? pick_pp<true>(*a) : pick_pp<false>(*a);
  hipLaunchKernelGGL(kernel, dim3(a->numBuckets), dim3(kWave * waves),
                     waves > 1 ? waves * kPpLds * sizeof(float4) : 0, s, *a);
  CGPU_CHECK(hipGetLastError());
  return 0;
}

extern "C" int changaAddVars(VariablePartData* dst, const VariablePartData* src, int n,
                             void* stream) {
  if (n <= 0) return 0;
  if (!dst || !src)
    return fail("changaAddVars: missing argument", hipErrorInvalidValue, __FILE__, __LINE__);
  hipLaunchKernelGGL(add_vars_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     dst, src, n);
  CGPU_CHECK(hipGetLastError());
  return 0;
}

extern "C" int changaZeroVars(VariablePartData* vars, int n, void* stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(zero_vars_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream,
                     vars, n);
  CGPU_CHECK(hipGetLastError());
  return 0;
}
