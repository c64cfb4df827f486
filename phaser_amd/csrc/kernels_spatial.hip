// kernels_spatial.hip -- translation stage for gfx950: voxelisation,
// 3-D real FFT of the voxel means, Laplace channel fusion fused with the
// cross-power spectrum, inverse 3-D FFT and a signed first-maximum argmax.
//
// Restates PhaseAligner::discretizePointcloud (phase-aligner.cc:71-131,
// include/igl/histc.cpp:34-73) and SpatialCorrelationLaplace::
// correlateSignals (spatial-correlation-laplace.cc:17-89,
// spatial-correlation.cc:142-161): C = F conj(G) with no normalisation on the
// r2c half spectrum, c2r of the first N^2(N/2+1) entries.  Grid layout is
// the reference's: linear index x*N + y + N^2*z, i.e. [z][x][y].
#include "fft_reg.hpp"
#include "kernels.hpp"
#include "pose.hpp"
#include "spatial_dev.hpp"

namespace phz {

namespace {

__global__ void k_fill_u32(uint32_t* __restrict__ p, size_t n, uint32_t v) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// streaming 16-byte copy: the HBM reference (bandwidth, traffic counters)
__global__ void k_copy_f4(float4* __restrict__ dst, const float4* __restrict__ src, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}

// igl::histc bin of x against strictly increasing float edges E[0..N),
// N >= 2.  The reference's binary search returns, for E[0] <= x <= E[N-1],
// the largest k <= N-2 with E[k] <= x, or N-1 when x == E[N-1] (and N-2 for
// a NaN, which passes both range tests); -1 outside.  The same k is found
// from the uniform spacing (inv = (N-1) / (E[N-1] - E[0])) and corrected
// against the actual edges, one or two lookups instead of log2 N dependent
// ones.
__device__ __forceinline__ int histc_bin(float x, const float* E, int N, float inv) {
  if (x < E[0] || x > E[N - 1]) return -1;
  if (x != x) return N - 2;
  if (x == E[N - 1]) return N - 1;
  int k = (int)((x - E[0]) * inv);
  k = k < N - 2 ? k : N - 2;
  while (k > 0 && E[k] > x) --k;
  while (k < N - 2 && E[k + 1] <= x) ++k;
  return k;
}

// kClear = false: accumulate (phase-aligner.cc:98-120); true: zero the same
// voxels again after use.  Scans arrive in ring order, so neighbouring
// points of a wave often share a voxel: runs of equal voxels among adjacent
// lanes are summed with a segmented wave reduction and only the run's first
// lane touches memory (one atomic per run instead of per point).  The same
// lanes set (or reset) the occupancy bytes of the voxel's row and z plane.
// Clouds from first_posed on are transformed by their pose first (a batch's
// targets and sources in one launch).
// kExtra: the clouds also carry (reflectivity, ambient) per point, summed
// into sumF / sumA like the intensity (phase-aligner.cc:113-118).
template <bool kClear, bool kExtra>
__global__ void k_voxel_scatter(const float4* __restrict__ pts, const int* __restrict__ npts,
                                int64_t cap, const DevPose* __restrict__ pose, int first_posed,
                                int N, const float* __restrict__ edges, float* __restrict__ sumI,
                                float* __restrict__ sumR, uint32_t* __restrict__ cnt,
                                VoxelOcc occ, const float2* __restrict__ extra,
                                float* __restrict__ sumF, float* __restrict__ sumA) {
#pragma clang fp contract(off)
  // the grid covers cap points per cloud: workgroups past the cloud's
  // points leave before staging the edges (uniform over the workgroup)
  if ((int64_t)blockIdx.x * blockDim.x >= npts[blockIdx.y]) return;
  extern __shared__ float E[];
  for (int i = threadIdx.x; i < N; i += blockDim.x) E[i] = edges[i];
  __syncthreads();
  const float inv = (float)(N - 1) / (E[N - 1] - E[0]);
  const int c = blockIdx.y;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  // every lane of the wave takes part in the reduction; lanes without a
  // voxel carry a key no other lane has
  int64_t key = -1 - (int64_t)lane;
  float vi = 0.f, vr = 0.f, vf = 0.f, va = 0.f;
  if (i < npts[c]) {
    float4 p = pts[c * cap + i];
  if (pose && c >= first_posed) {
    const float* T = pose[c - first_posed].T;
    const float x = T[0] * p.x + T[1] * p.y + T[2] * p.z + T[3];
    const float y = T[4] * p.x + T[5] * p.y + T[6] * p.z + T[7];
    const float z = T[8] * p.x + T[9] * p.y + T[10] * p.z + T[11];
    p.x = x;
    p.y = y;
    p.z = z;
  }
    const uint32_t bx = (uint32_t)histc_bin(p.x, E, N, inv);
    const uint32_t by = (uint32_t)histc_bin(p.y, E, N, inv);
    const uint32_t bz = (uint32_t)histc_bin(p.z, E, N, inv);
    const uint32_t NN = (uint32_t)N;
    const uint32_t lin = (bx * NN + by) + (NN * NN * bz);  // Sub2Ind in uint32
    // the reference skips lin > nf and overruns at nf
    if (lin < NN * NN * NN) {
      key = (int64_t)c * NN * NN * NN + lin;
      vi = p.w;
      vr = sqrtf(p.x * p.x + p.y * p.y + p.z * p.z);
      if (kExtra) {
        const float2 e = extra[c * cap + i];
        vf = e.x;
        va = e.y;
      }
    }
  }
  // runs of equal keys in adjacent lanes: head flags, segment ids, then a
  // suffix sum within each segment that leaves the total in the head lane
  const int64_t prev = __shfl_up(key, 1, 64);
  const bool head = lane == 0 || prev != key;
  const unsigned long long heads = __ballot(head);
  const int seg = __popcll(heads & ((2ull << lane) - 1ull));
  float n = (key >= 0) ? 1.f : 0.f;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const float oi = __shfl_down(vi, d, 64), orr = __shfl_down(vr, d, 64),
                on = __shfl_down(n, d, 64);
    const int os = __shfl_down(seg, d, 64);
    float of = 0.f, oa = 0.f;
    if (kExtra) {
      of = __shfl_down(vf, d, 64);
      oa = __shfl_down(va, d, 64);
    }
    if (!kClear && lane + d < 64 && os == seg) {
      vi += oi;
      vr += orr;
      n += on;
      if (kExtra) {
        vf += of;
        va += oa;
      }
    }
  }
  if (!head || key < 0) return;
  const size_t off = (size_t)key;
  // key = cloud N^3 + z N^2 + x N + y: row (cloud, z, x) = key / N
  if (occ.row) occ.row[off / (size_t)N] = kClear ? 0 : 1;
  if (occ.plane) occ.plane[off / ((size_t)N * N)] = kClear ? 0 : 1;
  if (kClear) {
    sumI[off] = 0.f;
    sumR[off] = 0.f;
    cnt[off] = 0u;
    if (kExtra) {
      sumF[off] = 0.f;
      sumA[off] = 0.f;
    }
    return;
  }
  atomicAdd(&sumI[off], vi);
  atomicAdd(&sumR[off], vr);
  atomicAdd(&cnt[off], (uint32_t)n);
  if (kExtra) {
    atomicAdd(&sumF[off], vf);
    atomicAdd(&sumA[off], va);
  }
}

__global__ void k_reduce_keys(const unsigned long long* __restrict__ partials, int count,
                              unsigned long long* __restrict__ keys) {
  const int p = blockIdx.x;
  unsigned long long best = 0ull;
  for (int i = threadIdx.x; i < count; i += blockDim.x) {
    const unsigned long long k = partials[(int64_t)p * count + i];
    best = k > best ? k : best;
  }
  best = block_max_key(best);
  if (threadIdx.x == 0) keys[p] = best;
}

// pass 1: r2c along y of (mean I + i mean R) rows, split into the two
// half spectra.  spec[cloud][ch][row][k], row = z*N + x.  With row_occ (the
// clouds' row occupancy) rows without points are neither read nor written
// (their spectrum is zero; only the occupancy-skipping x pass reads it), and a
// workgroup without any ends at once.
template <bool kDense>
__global__ void k_spat_r2c(int N, const float* __restrict__ a0, const float* __restrict__ a1,
                           const uint32_t* __restrict__ cnt, int64_t cloud_stride,
                           const uint8_t* __restrict__ row_occ, FftPlan plan,
                           const float2* __restrict__ tw, float2* __restrict__ spec,
                           int64_t spec_stride0, int64_t spec_stride1) {
  constexpr int RT = 16;
  const int row0 = blockIdx.x * RT, c = blockIdx.y;
  const int rows = N * N, h = N / 2 + 1;
  extern __shared__ float2 sm[];
  float2* A = sm;
  float2* B = sm + RT * N;
  float2* tws = B + RT * N;
  uint32_t live = 0xffffu;  // rows of this workgroup to transform
  if (row_occ) {
    const int lane = threadIdx.x & 63;
    live = (uint32_t)__ballot(lane < RT && row0 + lane < rows &&
                              row_occ[(int64_t)c * rows + row0 + lane] != 0);
    if (live == 0u) return;  // the same in every wave
  }
  stage_plan_twiddles(tws, N, tw);
  for (int idx = threadIdx.x; idx < RT * N; idx += blockDim.x) {
    const int r = div_small(idx, plan.by_L), y = idx - r * N;
    float2 v = make_float2(0.f, 0.f);
    if (row0 + r < rows && ((live >> r) & 1u)) {
      const int64_t off = c * cloud_stride + (int64_t)(row0 + r) * N + y;
      if (kDense) {
        v.x = a0[off];
        v.y = a1 ? a1[off] : 0.f;
      } else {
        // empty voxels (the vast majority) never touch the sum arrays
        const uint32_t k = cnt[off];
        if (k) {
          v.x = a0[off] / (float)k;
          v.y = a1[off] / (float)k;
        }
      }
    }
    A[idx] = v;
  }
  __syncthreads();
  float2* R = lds_fft<-1>(A, B, RT, plan, tws);
  for (int idx = threadIdx.x; idx < RT * h; idx += blockDim.x) {
    const int r = div_small(idx, plan.by_h), k = idx - r * h;
    if (row0 + r >= rows || !((live >> r) & 1u)) continue;
    const float2 zk = R[r * N + k];
    const float2 zc = cconj(R[r * N + (k ? N - k : 0)]);
    const float2 s = cadd(zk, zc), d = csub(zk, zc);
    const int64_t o = (int64_t)(row0 + r) * h + k;
    spec[c * spec_stride0 + o] = make_float2(0.5f * s.x, 0.5f * s.y);
    if (spec_stride1 >= 0) spec[c * spec_stride0 + spec_stride1 + o] = make_float2(0.5f * d.y, -0.5f * d.x);
  }
}

// pass 1, plane form (N <= kPlaneMaxN): one workgroup per (z plane, cloud)
// keeps the whole complex plane Z = mean I + i mean R in LDS, transforms it
// along y and then x, and splits the 2-D spectrum into the two half spectra
// with Z(-k) = conj of the real parts' transforms:
//   I^(k) = (Z(k) + conj Z(-k)) / 2,  R^(k) = (Z(k) - conj Z(-k)) / 2i.
// Replaces k_spat_r2c plus the x column pass (one HBM round trip less).
constexpr int kPlaneMaxN = 128;
constexpr int kPlaneChunk = 8;  // lines per LDS FFT batch

size_t spat_plane_lds_bytes(int N) {
  return ((size_t)N * (N + 1) + 2 * (size_t)kPlaneChunk * (N + 1) + N) * sizeof(float2);
}

__global__ void __launch_bounds__(256) k_spat_plane_fwd(
    int N, const float* __restrict__ sumI, const float* __restrict__ sumR,
    const uint32_t* __restrict__ cnt, int64_t cloud_stride, FftPlan plan,
    const float2* __restrict__ tw, float2* __restrict__ spec, int64_t spec_stride0,
    int64_t spec_stride1) {
  const int z = blockIdx.x, c = blockIdx.y;
  const int h = N / 2 + 1, ls = N + 1;
  extern __shared__ float2 sm[];
  float2* P = sm;                     // N x ls: the plane, row x, column y
  float2* A = sm + (size_t)N * ls;    // kPlaneChunk x ls
  float2* Bf = A + kPlaneChunk * ls;  // kPlaneChunk x ls
  float2* tws = Bf + kPlaneChunk * ls;
  stage_plan_twiddles(tws, N, tw);
  const int64_t base = c * cloud_stride + (int64_t)z * N * N;
  // rows (x) in chunks: load means, FFT along y, park in P
  for (int x0 = 0; x0 < N; x0 += kPlaneChunk) {
    for (int idx = threadIdx.x; idx < kPlaneChunk * N; idx += blockDim.x) {
      const int r = idx / N, y = idx - r * N;
      float2 v = make_float2(0.f, 0.f);
      if (x0 + r < N) {
        const int64_t off = base + (int64_t)(x0 + r) * N + y;
        const uint32_t k = cnt[off];  // empty voxels never touch the sums
        if (k) {
          v.x = sumI[off] / (float)k;
          v.y = sumR[off] / (float)k;
        }
      }
      A[r * ls + y] = v;
    }
    __syncthreads();
    const float2* R = lds_fft<-1>(A, Bf, kPlaneChunk, plan, tws, ls);
    for (int idx = threadIdx.x; idx < kPlaneChunk * N; idx += blockDim.x) {
      const int r = idx / N, y = idx - r * N;
      if (x0 + r < N) P[(x0 + r) * ls + y] = R[r * ls + y];
    }
    __syncthreads();
  }
  // columns (ky) in chunks: FFT along x in place through A/Bf
  for (int k0 = 0; k0 < N; k0 += kPlaneChunk) {
    for (int idx = threadIdx.x; idx < kPlaneChunk * N; idx += blockDim.x) {
      const int x = idx / kPlaneChunk, j = idx - x * kPlaneChunk;
      A[j * ls + x] = (k0 + j < N) ? P[x * ls + k0 + j] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    const float2* R = lds_fft<-1>(A, Bf, kPlaneChunk, plan, tws, ls);
    for (int idx = threadIdx.x; idx < kPlaneChunk * N; idx += blockDim.x) {
      const int x = idx / kPlaneChunk, j = idx - x * kPlaneChunk;
      if (k0 + j < N) P[x * ls + k0 + j] = R[j * ls + x];
    }
    __syncthreads();
  }
  // split into the two half spectra, spec[cloud][ch][z][kx][ky], ky < h
  float2* o0 = spec + c * spec_stride0 + (int64_t)z * N * h;
  float2* o1 = o0 + spec_stride1;
  for (int idx = threadIdx.x; idx < N * h; idx += blockDim.x) {
    const int kx = idx / h, ky = idx - kx * h;
    const float2 zk = P[kx * ls + ky];
    const float2 zc = cconj(P[((N - kx) % N) * ls + (N - ky) % N]);
    const float2 sm2 = cadd(zk, zc), d = csub(zk, zc);
    o0[idx] = make_float2(0.5f * sm2.x, 0.5f * sm2.y);
    o1[idx] = make_float2(0.5f * d.y, -0.5f * d.x);
  }
}

// in-place FFT along the middle axis of [outer][L][inner] arrays; one
// workgroup per (inner tile, outer, batch array).  With row_occ / plane_occ
// (the forward x pass over what the sparse r2c left; outer = z plane, array b
// of cloud b / 2): planes without points are skipped and stay unwritten, rows
// without points are read as zero.
template <int DIR, int IT>
__global__ void k_fft_cols(float2* __restrict__ data, int64_t batch_stride, int L, int inner,
                           FftPlan plan, const float2* __restrict__ tw,
                           const uint8_t* __restrict__ row_occ,
                           const uint8_t* __restrict__ plane_occ) {
  const int i0 = blockIdx.x * IT, o = blockIdx.y;
  const int64_t plane = (int64_t)(blockIdx.z >> 1) * L + o;
  if (plane_occ && plane_occ[plane] == 0) return;
  if (row_occ) row_occ += plane * L;
  float2* base = data + blockIdx.z * batch_stride + (int64_t)o * L * inner;
  extern __shared__ float2 sm[];
  const int ls = L + 1;  // padded line stride: the transposed accesses hit distinct banks
  float2* A = sm;
  float2* B = sm + IT * ls;
  float2* tws = B + IT * ls;
  stage_plan_twiddles(tws, L, tw);
  for (int idx = threadIdx.x; idx < IT * L; idx += blockDim.x) {
    const int e = idx / IT, ii = idx - e * IT;
    A[ii * ls + e] = (i0 + ii < inner && (!row_occ || row_occ[e]))
                         ? base[(int64_t)e * inner + i0 + ii] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  float2* R = lds_fft<DIR>(A, B, IT, plan, tws, ls);
  for (int idx = threadIdx.x; idx < IT * L; idx += blockDim.x) {
    const int e = idx / IT, ii = idx - e * IT;
    if (i0 + ii < inner) base[(int64_t)e * inner + i0 + ii] = R[ii * ls + e];
  }
}

// inverse pass A: fused F, G -> C = F conj(G) (spatial-correlation.cc:158-159)
// -> inverse FFT along z.  work[z][x][k2].
template <int IT>
__global__ void k_spat_cross_z(int N, ChannelSet F, int64_t f_stride, ChannelSet G,
                               int64_t g_stride, FusionRuns runs, int fuse, FftPlan plan,
                               const float2* __restrict__ tw, float2* __restrict__ work) {
  const int h = N / 2 + 1, inner = N * h;
  const int i0 = blockIdx.x * IT;
  // pair blockIdx.y: its F and G channels and its work array
  const int64_t fo = blockIdx.y * f_stride, go = blockIdx.y * g_stride;
  work += blockIdx.y * (int64_t)N * inner;
  extern __shared__ float2 sm[];
  const int ls = N + 1;
  float2* A = sm;
  float2* B = sm + IT * ls;
  float2* tws = B + IT * ls;
  stage_plan_twiddles(tws, N, tw);
  for (int idx = threadIdx.x; idx < IT * N; idx += blockDim.x) {
    const int z = idx / IT, ii = idx - z * IT;
    float2 c = make_float2(0.f, 0.f);
    if (i0 + ii < inner) {
      const int64_t q = (int64_t)z * inner + i0 + ii;
      float2 f, g;
      if (fuse) {
        int mode = 0;
        for (int r = 0; r < runs.count; ++r)
          if ((uint64_t)q >= runs.start[r]) mode = (int)runs.mode[r];
        f = fuse_at(F, mode, q + fo);
        g = fuse_at(G, mode, q + go);
      } else {
        f = F.ch[0][q + fo];
        g = G.ch[0][q + go];
      }
      c.x = f.x * g.x - f.y * (-g.y);
      c.y = f.x * (-g.y) + f.y * g.x;
    }
    A[ii * ls + z] = c;
  }
  __syncthreads();
  float2* R = lds_fft<+1>(A, B, IT, plan, tws, ls);
  for (int idx = threadIdx.x; idx < IT * N; idx += blockDim.x) {
    const int z = idx / IT, ii = idx - z * IT;
    if (i0 + ii < inner) work[(int64_t)z * inner + i0 + ii] = R[ii * ls + z];
  }
}

// The forward z pass, the fusion, the cross spectrum and the inverse z pass of
// IT columns of a pair in LDS, for the lengths the register engine lacks
// (there k_spat_cross_zz_reg): each present channel's columns are transformed
// (occupied planes read, the others zero) and folded into the side's fused
// columns as fuse_at does, so that the z-transformed spectra are never stored.
// LDS: two transform buffers, the two fused sides and the twiddles.  Bound by
// VALU issue where the length has a large prime factor, else by LDS.
template <int IT>
__global__ void __launch_bounds__(256) k_spat_cross_zz(
    int N, ChannelSet F, int64_t f_stride, ChannelSet G, int64_t g_stride,
    const uint8_t* __restrict__ f_occ, int64_t f_occ_stride, const uint8_t* __restrict__ g_occ,
    int64_t g_occ_stride, FusionRuns runs, FftPlan plan, const float2* __restrict__ tw,
    float2* __restrict__ work) {
  constexpr int kPer = 8;  // entries of a thread: IT N / 256, N <= 256 at IT 8, 128 at 16
  const int h = N / 2 + 1, inner = N * h, ls = N + 1, p = blockIdx.y;
  const int i0 = blockIdx.x * IT;
  extern __shared__ float2 sm[];
  float2* A = sm;
  float2* B = A + IT * ls;
  float2* fused = B + IT * ls;  // both sides, IT x ls each
  float2* tws = fused + 2 * IT * ls;
  stage_plan_twiddles(tws, N, tw);
  work += p * (int64_t)N * inner;
  // entry i of a thread: frequency (or plane) e, column ii
  auto entry = [&](int i, int& e, int& ii) {
    const int idx = threadIdx.x + 256 * i;
    e = idx / IT;
    ii = idx - e * IT;
    return idx < IT * N;
  };
  uint32_t modes = 0u;  // two bits per entry
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    int e, ii;
    if (!entry(i, e, ii)) break;
    const uint32_t q = (uint32_t)(e * inner + i0 + ii);
    uint32_t m = 0u;
    for (int r = 0; r < runs.count; ++r) m = q >= runs.start[r] ? runs.mode[r] : m;
    modes |= (m & 3u) << (2 * i);
  }
  for (int side = 0; side < 2; ++side) {
    const ChannelSet& X = side ? G : F;
    const int64_t off = side ? p * g_stride : p * f_stride;
    const uint8_t* occ = side ? g_occ + p * g_occ_stride : f_occ + p * f_occ_stride;
    float2* acc = fused + side * IT * ls;
    bool first = true;
    for (int c = 0; c < X.C; ++c) {
      if (!X.ch[c]) continue;
      const float2* src = X.ch[c] + off + i0;
      float2 v[kPer];
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        int e, ii;
        const bool in = entry(i, e, ii);
        v[i] = in && i0 + ii < inner && occ[e] ? src[(int64_t)e * inner + ii]
                                              : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        int e, ii;
        if (entry(i, e, ii)) A[ii * ls + e] = v[i];
      }
      __syncthreads();
      const float2* R = lds_fft<-1>(A, B, IT, plan, tws, ls);
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        int e, ii;
        if (!entry(i, e, ii)) break;
        const float2 x = R[ii * ls + e];
        float2* a = &acc[ii * ls + e];
        if (first) {
          *a = x;
        } else {
          // the maximum is the first of equal energies, and a number before a NaN
          const float2 y = *a;
          const bool sum = ((modes >> (2 * i)) & 3u) == 1u;
          const float ey = y.x * y.x + y.y * y.y;
          const bool take = !(fmaxf(ey, x.x * x.x + x.y * x.y) == ey);
          *a = sum ? cadd(y, x) : (take ? x : y);
        }
      }
      first = false;
      __syncthreads();  // the result is read before the next channel's columns
    }
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    int e, ii;
    if (!entry(i, e, ii)) break;
    const uint32_t m = (modes >> (2 * i)) & 3u;
    float2 f = fused[ii * ls + e], g = fused[(IT + ii) * ls + e];
    if (m == 1u) {
      f = make_float2(f.x / (float)F.C, f.y / (float)F.C);
      g = make_float2(g.x / (float)G.C, g.y / (float)G.C);
    } else if (m != 0u) {
      f = g = make_float2(0.f, 0.f);
    }
    float2 c = make_float2(f.x * g.x - f.y * (-g.y), f.x * (-g.y) + f.y * g.x);
    if (c.x != c.x && m == 0u) {  // a side without a channel that is a number is zero
      const float ef = f.x * f.x + f.y * f.y, eg = g.x * g.x + g.y * g.y;
      if (ef != ef || eg != eg) {
        if (ef != ef) f = make_float2(0.f, 0.f);
        if (eg != eg) g = make_float2(0.f, 0.f);
        c = make_float2(f.x * g.x - f.y * (-g.y), f.x * (-g.y) + f.y * g.x);
      }
    }
    A[ii * ls + e] = c;
  }
  __syncthreads();
  const float2* R = lds_fft<+1>(A, B, IT, plan, tws, ls);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    int e, ii;
    if (!entry(i, e, ii)) break;
    if (i0 + ii < inner) work[(int64_t)e * inner + i0 + ii] = R[ii * ls + e];
  }
}

// last pass: c2r along y (real parts of k=0 and k=N/2, FFTW hc2r), two rows
// per complex line, signed argmax over x*N + y + N^2*z.
__global__ void k_spat_c2r(int N, const float2* __restrict__ work, FftPlan plan,
                           const float2* __restrict__ tw, float* __restrict__ corr,
                           unsigned long long* __restrict__ partials, uint32_t limit) {
  constexpr int RT = 16, NL = RT / 2;
  const int h = N / 2 + 1, rows = N * N;
  const int row0 = blockIdx.x * RT;
  // pair blockIdx.y: its half spectrum, output grid and argmax partials
  work += blockIdx.y * (int64_t)rows * h;
  if (corr) corr += blockIdx.y * (int64_t)rows * N;
  partials += blockIdx.y * (int64_t)gridDim.x;
  extern __shared__ float2 sm[];
  float2* X = sm;  // RT x h
  float2* A = sm + RT * h;
  float2* B = A + NL * N;
  float2* tws = B + NL * N;
  stage_plan_twiddles(tws, N, tw);
  for (int idx = threadIdx.x; idx < RT * h; idx += blockDim.x) {
    const int r = div_small(idx, plan.by_h), k = idx - r * h;
    X[idx] = (row0 + r < rows) ? work[(int64_t)(row0 + r) * h + k] : make_float2(0.f, 0.f);
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < NL * N; idx += blockDim.x) {
    const int p = div_small(idx, plan.by_L), m = idx - p * N;
    const float2* xa = X + (2 * p) * h;
    const float2* xb = X + (2 * p + 1) * h;
    float2 va, vb;
    if (m == 0 || 2 * m == N) {
      va = make_float2(xa[m].x, 0.f);
      vb = make_float2(xb[m].x, 0.f);
    } else if (m < h) {
      va = xa[m];
      vb = xb[m];
    } else {
      va = cconj(xa[N - m]);
      vb = cconj(xb[N - m]);
    }
    A[idx] = make_float2(va.x - vb.y, va.y + vb.x);
  }
  __syncthreads();
  float2* R = lds_fft<+1>(A, B, NL, plan, tws);
  unsigned long long best = 0ull;
  for (int idx = threadIdx.x; idx < RT * N; idx += blockDim.x) {
    const int r = div_small(idx, plan.by_L), y = idx - r * N;
    if (row0 + r >= rows) continue;
    const float2 z = R[(r >> 1) * N + y];
    const float v = (r & 1) ? z.y : z.x;
    const uint32_t lin = (uint32_t)((int64_t)(row0 + r) * N + y);
    if (corr) corr[lin] = v;
    if (lin >= limit) continue;  // past the correlation vector's length
    const unsigned long long kk = make_key(v, lin);
    best = kk > best ? kk : best;
  }
  best = block_max_key(best);
  if (threadIdx.x == 0) partials[blockIdx.x] = best;
}

// SpatialCorrelation::complexMulSeq (spatial-correlation.cc:142-161) on the
// fused (or, fuse = 0, single-channel) spectra without the inverse
// transform: work[pair][q] = F[q] conj(G[q]) over the H unshifted
// half-spectrum entries (the rest of the N^3 buffer is zero)
__global__ void k_spat_cross_product(int64_t H, ChannelSet F, int64_t f_stride, ChannelSet G,
                                     int64_t g_stride, FusionRuns runs, int fuse,
                                     float2* __restrict__ work) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= H) return;
  const int64_t fo = blockIdx.y * f_stride, go = blockIdx.y * g_stride;
  float2 f, g;
  if (fuse) {
    int mode = 0;
    for (int r = 0; r < runs.count; ++r)
      if ((uint64_t)q >= runs.start[r]) mode = (int)runs.mode[r];
    f = fuse_at(F, mode, q + fo);
    g = fuse_at(G, mode, q + go);
  } else {
    f = F.ch[0][q + fo];
    g = G.ch[0][q + go];
  }
  float2 c;
  c.x = f.x * g.x - f.y * (-g.y);
  c.y = f.x * (-g.y) + f.y * g.x;
  work[blockIdx.y * H + q] = c;
}

// The c2r input of the zero-padded correlation (spatial-correlation.cc:
// 142-161,221-230): the reference writes product entry i (i < T = N^3, in
// the product's own order) to Sub2Ind(x + pad, y + pad, z + pad, Np, Np) of a
// zeroed buffer, (x, y, z) = Ind2Sub(i, N, N); the Laplace class (shifted)
// then rotates the buffer's first T entries left by T/2 (IFFTShift,
// spatial-correlation-laplace.cc:36) and the c2r of size Np reads its first
// Hp = Np^2 (Np/2 + 1) entries.  Gathered per output q < Hp: the buffer
// entry r it holds, r's padded coordinates, the product index i, and, for
// the shifted order of the Laplace class, the unshifted half-spectrum entry
// u = (i + s) mod T (FFTShift rotates left by s = ceil(T/2), signal-utils.h:
// 29-37) that work holds when u < H.
// cube_lo <= cube_hi: SpatialCorrelationLowPass (spatial-correlation-low-pass.
// cc:39-94) multiplies only the product entries whose shifted index is
// Sub2Ind(i, j, k, N, N) with i, j, k in [cube_lo, cube_hi]; the rest stay zero
__global__ void k_spat_pad_gather(int N, int pad, int shifted, const float2* __restrict__ work,
                                  int64_t H, float2* __restrict__ out, int64_t Hp, int cube_lo,
                                  int cube_hi) {
  const int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (q >= Hp) return;
  const int64_t T = (int64_t)N * N * N;
  const int64_t Np = N + 2 * pad;
  int64_t r = q;
  if (shifted && q < T) {
    r = q + T / 2;
    if (r >= T) r -= T;
  }
  const int64_t zp = r / (Np * Np), rem = r - zp * Np * Np;
  const int64_t xp = rem / Np, yp = rem - xp * Np;
  float2 v = make_float2(0.f, 0.f);
  bool in = zp >= pad && zp < pad + N && xp >= pad && xp < pad + N && yp >= pad && yp < pad + N;
  if (in && cube_lo <= cube_hi)
    in = xp - pad >= cube_lo && xp - pad <= cube_hi && yp - pad >= cube_lo &&
         yp - pad <= cube_hi && zp - pad >= cube_lo && zp - pad <= cube_hi;
  if (in) {
    const int64_t i = (xp - pad) * N + (yp - pad) + (int64_t)N * N * (zp - pad);
    int64_t u = i;
    if (shifted) {
      u = i + (T % 2 ? T / 2 + 1 : T / 2);
      if (u >= T) u -= T;
    }
    if (u < H) v = work[blockIdx.y * H + u];
  }
  out[blockIdx.y * Hp + q] = v;
}

// The translation pose of pair blockIdx.x: its argmax from the `count` partial
// keys of the last pass, then, in one wavefront, the Gaussian fit
// to the +-k linear-index window around the argmax (GaussianPeakBasedEval,
// gaussian-peak-based-eval.cc:26-102; gaussian.cc:14-56): weights = the grid
// values normalised to sum 1 (CHECK_GT(sum, 0), :100), samples = the
// translations of the window's indices (translation-utils.cc:40-52,
// signal-utils.cc:11-19), mean = sum w t, covariance = sum w (t-mean)(t-mean)^T,
// NaN where the reference takes the root of a negative weight.
// The finished pose also goes to `result`, host memory the device writes: the
// caller needs no copy of its own once the stream is idle.
__global__ void __launch_bounds__(256) k_trans_pose(int N, int lower, int upper,
                                                   const unsigned long long* __restrict__ partials,
                                                   int count, const float* __restrict__ corr,
                                                   int64_t corr_stride, int k,
                                                   DevPose* __restrict__ pose, uint32_t n_corr,
                                                   int mixture, DevPose* __restrict__ result) {
  const int p = blockIdx.x, lane = threadIdx.x;
  const unsigned long long key = max_partial_key(partials + (int64_t)p * count, count);
  if (threadIdx.x >= 64) return;  // the fit is one wavefront's
  const uint32_t idx = key_index(key);
  const float value = unordered_value((uint32_t)(key >> 32));
  const double width = (double)(abs(lower) + abs(upper) + 1);
  // gaussian-peak-based-eval.cc:26-37
  const uint32_t uk = (uint32_t)k;
  const uint32_t start = uk > idx ? idx : idx - uk;
  // GmmPeakBasedEval (gmm-peak-based-eval.cc:58-68): end = idx only when
  // idx + k > n_corr, so an end of n_corr fails its CHECK_LT (:81)
  const uint32_t end = mixture ? (uk + idx > n_corr ? idx : idx + uk)
                               : (uk + idx >= n_corr ? idx : idx + uk);
  int32_t status = 0;
  double mean[3], cov[6] = {0, 0, 0, 0, 0, 0};  // upper triangle, row by row
  bool negative = false;
  if (end >= n_corr) {
    status |= kPoseTransWindow;
    translation_of_index(idx, N, width, mean);
  } else if (end == start || idx >= n_corr) {  // one sample (the default 0 neighbours): value / value
    if (!(value > 0.f)) status |= kPoseTransWeights;
    translation_of_index(idx, N, width, mean);
  } else {
    const float* g = corr + p * corr_stride;
    double sum = 0.0;
    for (uint32_t i = start + lane; i <= end; i += 64) sum += (double)g[i];
    sum = wave_sum(sum);
    if (!(sum > 0.0)) status |= kPoseTransWeights;
    double m[3] = {0, 0, 0};
    for (uint32_t i = start + lane; i <= end; i += 64) {
      const double w = (double)g[i] / sum;
      negative |= w < 0.0;
      double t[3];
      translation_of_index(i, N, width, t);
      for (int d = 0; d < 3; ++d) m[d] += w * t[d];
    }
    for (int d = 0; d < 3; ++d) mean[d] = wave_sum(m[d]);
    for (uint32_t i = start + lane; i <= end; i += 64) {
      const double w = (double)g[i] / sum;
      double t[3];
      translation_of_index(i, N, width, t);
      for (int d = 0; d < 3; ++d) t[d] -= mean[d];
      int e = 0;
      for (int r = 0; r < 3; ++r)
        for (int c = r; c < 3; ++c) cov[e++] += w * t[r] * t[c];
    }
    for (int e = 0; e < 6; ++e) cov[e] = wave_sum(cov[e]);
    negative = __any(negative);
  }
  if (lane == 0) {
  DevPose& P = pose[p];
  P.trans_index = idx;
  P.trans_value = value;
  for (int d = 0; d < 3; ++d) P.translation[d] = mean[d];
  int e = 0;
  for (int r = 0; r < 3; ++r)
    for (int c = r; c < 3; ++c) {
      const double v = cov[e++];
      P.trans_cov[r * 3 + c] = P.trans_cov[c * 3 + r] = negative ? __builtin_nan("") : v;
    }
  P.status |= status;
  }
  __threadfence();  // lane 0's entries are read back by the whole wave
  static_assert(sizeof(DevPose) % 4 == 0, "whole words");
  for (int i = lane; i < (int)(sizeof(DevPose) / 4); i += 64)
    ((uint32_t*)&result[p])[i] = ((const volatile uint32_t*)&pose[p])[i];
}

__global__ void k_apply_pose(const float4* __restrict__ pts, int64_t P,
                             const DevPose* __restrict__ pose, float4* __restrict__ out) {
#pragma clang fp contract(off)
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i >= P) return;
  const float* T = pose->T;
  const float4 p = pts[i];
  const float x = T[0] * p.x + T[1] * p.y + T[2] * p.z + T[3];
  const float y = T[4] * p.x + T[5] * p.y + T[6] * p.z + T[7];
  const float z = T[8] * p.x + T[9] * p.y + T[10] * p.z + T[11];
  out[i] = make_float4(x + (float)pose->translation[0], y + (float)pose->translation[1],
                       z + (float)pose->translation[2], p.w);
}

}  // namespace

void launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s) {
  if (n == 0) return;
  size_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
}

void launch_copy_f4(float4* dst, const float4* src, size_t n, hipStream_t s) {
  size_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  if (blocks == 0) return;
  hipLaunchKernelGGL(k_copy_f4, dim3((unsigned)blocks), dim3(256), 0, s, dst, src, n);
}

template <bool kClear>
static void voxel_pass(const float4* pts, const int* npts, int64_t cap, int nclouds,
                       const DevPose* pose, int first_posed, int N, const float* edges,
                       float* sumI, float* sumR, uint32_t* cnt, VoxelOcc occ, VoxelExtra ex,
                       hipStream_t s) {
  dim3 g((unsigned)((cap + 255) / 256), nclouds);
  if (ex.extra)
    hipLaunchKernelGGL((k_voxel_scatter<kClear, true>), g, dim3(256), N * sizeof(float), s, pts,
                       npts, cap, pose, first_posed, N, edges, sumI, sumR, cnt, occ, ex.extra,
                       ex.sumF, ex.sumA);
  else
    hipLaunchKernelGGL((k_voxel_scatter<kClear, false>), g, dim3(256), N * sizeof(float), s, pts,
                       npts, cap, pose, first_posed, N, edges, sumI, sumR, cnt, occ,
                       (const float2*)nullptr, (float*)nullptr, (float*)nullptr);
}

void launch_voxel_scatter(const float4* pts, const int* npts, int64_t cap, int nclouds,
                          const DevPose* pose, int first_posed, int N, const float* edges,
                          float* sumI, float* sumR, uint32_t* cnt, VoxelOcc occ, hipStream_t s,
                          VoxelExtra ex) {
  voxel_pass<false>(pts, npts, cap, nclouds, pose, first_posed, N, edges, sumI, sumR, cnt, occ,
                    ex, s);
}

void launch_voxel_clear(const float4* pts, const int* npts, int64_t cap, int nclouds,
                        const DevPose* pose, int first_posed, int N, const float* edges,
                        float* sumI, float* sumR, uint32_t* cnt, VoxelOcc occ, hipStream_t s,
                        VoxelExtra ex) {
  voxel_pass<true>(pts, npts, cap, nclouds, pose, first_posed, N, edges, sumI, sumR, cnt, occ,
                   ex, s);
}

void launch_reduce_keys(const unsigned long long* partials, int count, int npairs,
                        unsigned long long* keys, hipStream_t s) {
  hipLaunchKernelGGL(k_reduce_keys, dim3(npairs), dim3(256), 0, s, partials, count, keys);
}

int spatial_c2r_blocks(int N) { return (N * N + 15) / 16; }

// The forward x and z passes of both clouds' two channels, their Laplace
// fusion, C = F conj(G) and the inverse z pass for one pair at one y
// frequency k2, with the (z, x) plane of that frequency in LDS: the
// x-transformed spectra never go to memory (k_fft_x_occ followed by
// k_spat_cross_zz_reg store and reload them, two HBM round trips of every
// occupied plane).  Workgroup (pair, k2) of L R2 threads: line = thread % L,
// n2 = thread / L, so each wave holds 64 lines at one n2.
// Input: the half spectra of k_spat_r2c_rows (layout [z][x][k2]; only rows
// (z, x) that hold points were written), read with buffer loads whose
// masked lanes address past the buffer (no memory access, zero returned);
// the row bits come from the clouds' occupancy bytes.  x pass: over the z
// planes that hold points, listed ascending one per line (a wave whose
// lines are all past the list idles); the z pass reads every other plane
// row as zero.  Each line exchanges through its own row (x pass) or
// column (z pass) of the plane.  A thread's z-pass output k = n2 + R2 j +
// R1 k2' is the inverse transform's input n1 = j + (R1 / R2) k2' (as in
// k_spat_cross_zz_reg).  Output: work[pair][k2][z][x], one contiguous
// slab per workgroup (k_spat_inv_plane<L, TPB, true> reads it).
// f_shared: every pair reads target cloud 0.  xcd: workgroup b runs pair
// (b mod 8) + 8 (b / 8h) at k2 = (b / 8) mod h, so that the h workgroups of
// a pair run on one XCD and share its L2 (a 128-byte line of a spectrum
// row holds 16 consecutive k2); needs a multiple of 8 pairs.
// The fused F side waits in global memory (the workgroup's own output
// slab) while the G side runs, which keeps the registers of 1024 threads
// within 128.  Measured at L = 128, 64 pairs: 1.08 ms against 0.85 ms for
// k_fft_x_occ + k_spat_cross_zz_reg: with 138 KB of LDS one workgroup fills
// a CU, and its load latency, LDS phases and barriers have no other
// workgroup to overlap with; an option (phz_tuning.xz_slab), off by default.
template <int L>
__global__ void __launch_bounds__(L * RegSplit<L>::R2) k_spat_cross_slab(
    ChannelSet F, int64_t f_stride, ChannelSet G, int64_t g_stride,
    const uint8_t* __restrict__ f_rows, const uint8_t* __restrict__ f_planes, int f_shared,
    const uint8_t* __restrict__ g_rows, const uint8_t* __restrict__ g_planes, FusionRuns runs,
    int xcd, const float2* __restrict__ tw, float2* __restrict__ work) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, S = L + 1, h = L / 2 + 1;
  constexpr int TPB = L * R2, W = L / 32;  // W: bit words per plane row
  constexpr int64_t inner = (int64_t)L * h, H = inner * L;
  static_assert(32 % R2 == 0 && TPB >= 2 * L && L % 64 == 0, "thread layout");
  static_assert(H * 8 < 0x7fffffffLL, "one buffer resource per spectrum");
  extern __shared__ float2 P[];  // L rows (z) of S entries (x, padded)
  __shared__ uint32_t rowbits[2][L * W];
  __shared__ uint32_t planebits[2][W];
  __shared__ int zlist[2][L];
  __shared__ int nzs[2];
  __shared__ int wcnt[2 * L / 64];
  // n2 is uniform over a wave (L >= 64): the twiddles W_L^(n2 k1) are
  // scalar loads, kept out of the vector registers
  const int t = threadIdx.x, line = t % L, n2 = __builtin_amdgcn_readfirstlane(t / L);
  int p, k2;
  if (xcd) {
    const int b = blockIdx.x;
    p = (b & 7) + 8 * (b / (8 * h));
    k2 = (b >> 3) % h;
  } else {
    p = blockIdx.x / h;
    k2 = blockIdx.x - p * h;
  }
  const int fc = f_shared ? 0 : p;
  // row occupancy bytes -> bits: word r of a side covers bytes 32 r .. 32 r + 31
  for (int wi = t; wi < 2 * L * W; wi += TPB) {
    const int side = wi / (L * W), r = wi - side * (L * W);
    const uint4* src = (const uint4*)((side ? g_rows + (int64_t)p * L * L
                                            : f_rows + (int64_t)fc * L * L) + 32 * r);
    const uint4 a = src[0], b = src[1];
    const uint32_t wd[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t bits = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) bits |= (uint32_t)(((wd[k] >> (8 * j)) & 0xffu) != 0u) << (4 * k + j);
    rowbits[side][r] = bits;
  }
  // occupied planes of both sides: bits and ascending lists
  {
    const bool in = t < 2 * L;
    const int side = t / L, z = t % L, lane = t & 63, wv = t >> 6;
    const bool occ = in && (side ? g_planes[(int64_t)p * L + z] : f_planes[(int64_t)fc * L + z]) != 0;
    const unsigned long long m = __ballot(occ);
    if (in && lane == 0) {
      wcnt[wv] = __popcll(m);
      planebits[side][z >> 5] = (uint32_t)m;
      planebits[side][(z >> 5) + 1] = (uint32_t)(m >> 32);
    }
    __syncthreads();
    if (in) {
      int base = 0;
      for (int i = side * (L / 64); i < wv; ++i) base += wcnt[i];
      if (occ) zlist[side][base + __popcll(m & ((1ull << lane) - 1ull))] = z;
      if (z == 0) {
        int tot = 0;
        for (int i = 0; i < L / 64; ++i) tot += wcnt[side * (L / 64) + i];
        nzs[side] = tot;
      }
    }
    __syncthreads();
  }
  // forward x and z passes of one channel of one side; out[j R2 + k2'] =
  // X(kz = n2 + R2 j + R1 k2', kx = line)
  auto fwd2 = [&](int side, const float2* X, float2(&out)[R1]) {
    const int nz = nzs[side];
    const bool wave_on = (line & ~63) < nz, act = line < nz;
    const int z = act ? zlist[side][line] : 0;
    float2* row = P + z * S;
    float2 v[R1];
    if (wave_on) {
      // this thread's 16 row bits (x = n2 + R2 n1) in one register
      uint32_t xm = 0;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const uint32_t rw = act ? rowbits[side][z * W + i] : 0u;
#pragma unroll
        for (int n1 = 0; n1 < R1; ++n1)
          if (((R2 * n1) >> 5) == i) xm |= ((rw >> ((n2 + R2 * n1) & 31)) & 1u) << n1;
      }
      const __amdgpu_buffer_rsrc_t rs =
          __builtin_amdgcn_make_buffer_rsrc((void*)X, (short)0, (int)(H * 8), 0x00020000);
      // lane offset of x = n2 plus a scalar offset per n1; a masked lane's
      // offset lies past the buffer with or without the scalar part.  Two
      // 32-bit loads per entry (merged into one 64-bit load): this
      // compiler's 64-bit buffer-load builtin fetches one dword and returns
      // it in both halves.
      const uint32_t base = (uint32_t)(((z * L + n2) * h + k2) * 8);
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) {
        const uint32_t o = ((xm >> n1) & 1u) ? base : 0x80000000u;
        const int so = R2 * n1 * h * 8;
        v[n1] = make_float2(
            __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o, so, 0)),
            __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, o + 4u, so, 0)));
      }
      dft_reg<R1, -1>(v);
#pragma unroll
      for (int k1 = 1; k1 < R1; ++k1) v[k1] = cmul(v[k1], tw[n2 * k1]);
    }
    __syncthreads();  // the previous readers of the plane are done
    if (wave_on && act) {
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) row[k1 * R2 + n2] = v[k1];
    }
    __syncthreads();
    float2 r[R1];
    if (wave_on && act) {
#pragma unroll
      for (int j = 0; j < R1 / R2; ++j) {
        const int k1 = n2 + R2 * j;
        float2 u[R2];
#pragma unroll
        for (int m = 0; m < R2; ++m) u[m] = row[k1 * R2 + m];
        dft_reg<R2, -1>(u);
#pragma unroll
        for (int kk = 0; kk < R2; ++kk) r[j * R2 + kk] = u[kk];
      }
    }
    __syncthreads();  // the exchange is read before the results go back
    if (wave_on && act) {
#pragma unroll
      for (int j = 0; j < R1 / R2; ++j)
#pragma unroll
        for (int kk = 0; kk < R2; ++kk) row[(n2 + R2 * j) + R1 * kk] = r[j * R2 + kk];
    }
    __syncthreads();
    // z pass along column x = line; planes without points are zero
    uint32_t pw[W];  // uniform: scalar registers
#pragma unroll
    for (int i = 0; i < W; ++i) pw[i] = __builtin_amdgcn_readfirstlane(planebits[side][i]);
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
      const int zz = n2 + R2 * n1;
      const float2 e = P[zz * S + line];
      v[n1] = ((pw[(R2 * n1) >> 5] >> (zz & 31)) & 1u) ? e : make_float2(0.f, 0.f);
    }
    dft_reg<R1, -1>(v);
#pragma unroll
    for (int k1 = 1; k1 < R1; ++k1) v[k1] = cmul(v[k1], tw[n2 * k1]);
    __syncthreads();  // the columns are read before the exchanges overwrite them
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) P[(k1 * R2 + n2) * S + line] = v[k1];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < R1 / R2; ++j) {
      const int k1 = n2 + R2 * j;
      float2 u[R2];
#pragma unroll
      for (int m = 0; m < R2; ++m) u[m] = P[(k1 * R2 + m) * S + line];
      dft_reg<R2, -1>(u);
#pragma unroll
      for (int kk = 0; kk < R2; ++kk) out[j * R2 + kk] = u[kk];
    }
  };
  // fusion mode of this thread's frequencies (2 bits each)
  uint32_t modes = 0;
#pragma unroll
  for (int j = 0; j < R1 / R2; ++j)
#pragma unroll
    for (int kk = 0; kk < R2; ++kk) {
      const uint64_t idx = (uint64_t)(n2 + R2 * j + R1 * kk) * inner + (uint64_t)line * h + k2;
      uint32_t m = 0;
      for (int r = 0; r < runs.count; ++r)
        if (idx >= runs.start[r]) m = runs.mode[r];
      modes |= (m & 3u) << (2 * (j * R2 + kk));
    }
  // the fused F side waits in this workgroup's own output slab (rows kz,
  // column line) while the G side is transformed: every thread rereads and
  // finally overwrites exactly the entries it parked there, so no other
  // thread's accesses intervene
  float2* slab = work + ((int64_t)p * h + k2) * L * L + line;
  {
    float2 fa[R1], fb[R1];
    fwd2(0, F.ch[0] + p * f_stride, fa);
    fwd2(0, F.ch[1] + p * f_stride, fb);
#pragma unroll
    for (int j = 0; j < R1 / R2; ++j)
#pragma unroll
      for (int kk = 0; kk < R2; ++kk) {
        const int i = j * R2 + kk;
        slab[(int64_t)(n2 + R2 * j + R1 * kk) * L] =
            fuse_pair(fa[i], fb[i], F.C, (modes >> (2 * i)) & 3u);
      }
  }
  float2 ga[R1], xb[R1];
  fwd2(1, G.ch[0] + p * g_stride, ga);
  fwd2(1, G.ch[1] + p * g_stride, xb);
#pragma unroll
  for (int i = 0; i < R1; ++i) ga[i] = fuse_pair(ga[i], xb[i], G.C, (modes >> (2 * i)) & 3u);
  // the last z pass's exchange is read before the inverse one is written;
  // the parked F entries are loaded only after the G side has been fused
  __syncthreads();
  float2 v[R1];
#pragma unroll
  for (int j = 0; j < R1 / R2; ++j)
#pragma unroll
    for (int kk = 0; kk < R2; ++kk) {
      const int i = j * R2 + kk;
      const float2 f = slab[(int64_t)(n2 + R2 * j + R1 * kk) * L], g = ga[i];
      float2 cz;
      cz.x = f.x * g.x - f.y * (-g.y);
      cz.y = f.x * (-g.y) + f.y * g.x;
      v[j + (R1 / R2) * kk] = cz;
    }
  // inverse z pass along column line, straight to the slab
  dft_reg<R1, +1>(v);
#pragma unroll
  for (int k1 = 1; k1 < R1; ++k1) v[k1] = cmul(v[k1], cconj(tw[n2 * k1]));
#pragma unroll
  for (int k1 = 0; k1 < R1; ++k1) P[(k1 * R2 + n2) * S + line] = v[k1];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < R1 / R2; ++j) {
    const int k1 = n2 + R2 * j;
    float2 u[R2];
#pragma unroll
    for (int m = 0; m < R2; ++m) u[m] = P[(k1 * R2 + m) * S + line];
    dft_reg<R2, +1>(u);
#pragma unroll
    for (int kk = 0; kk < R2; ++kk) slab[(int64_t)(k1 + R1 * kk) * L] = u[kk];
  }
}

bool cross_zz_ok(const ChannelSet& F, const ChannelSet& G, int nch) {
  for (const ChannelSet* cs : {&F, &G}) {
    if (cs->C != 4) return false;
    for (int c = 0; c < cs->C; ++c)
      if ((cs->ch[c] != nullptr) != (c < nch)) return false;
  }
  return true;
}

bool spatial_cross_slab_ok(int N) { return N == 64 || N == 128; }

const SpatialReg* spatial_reg_a(int N);
const SpatialReg* spatial_reg_b(int N);
const SpatialReg* spatial_reg_c(int N);
const SpatialReg* spatial_reg_d(int N);
const SpatialReg* spatial_reg_e(int N);
const SpatialReg* spatial_reg(int N) {
  const SpatialReg* r = spatial_reg_a(N);
  if (!r) r = spatial_reg_b(N);
  if (!r) r = spatial_reg_c(N);
  if (!r) r = spatial_reg_d(N);
  if (!r) r = spatial_reg_e(N);
  return r;
}

template <int L>
static void launch_cross_slab_t(int npairs, ChannelSet F, int64_t fs, ChannelSet G, int64_t gs,
                                const uint8_t* f_rows, const uint8_t* f_planes, bool f_shared,
                                const uint8_t* g_rows, const uint8_t* g_planes,
                                const FusionRuns& runs, const float2* tw, float2* work,
                                hipStream_t s) {
  constexpr int h = L / 2 + 1, TPB = L * RegSplit<L>::R2;
  const int xcd = npairs % 8 == 0;
  const size_t lds = sizeof(float2) * L * (L + 1);
  hipLaunchKernelGGL(k_spat_cross_slab<L>, dim3(npairs * h), dim3(TPB), lds, s, F, fs, G, gs,
                     f_rows, f_planes, (int)f_shared, g_rows, g_planes, runs, xcd, tw, work);
}

void launch_spatial_cross_slab(int N, int npairs, ChannelSet F, int64_t f_stride, ChannelSet G,
                               int64_t g_stride, const uint8_t* f_rows, const uint8_t* f_planes,
                               bool f_shared, const uint8_t* g_rows, const uint8_t* g_planes,
                               const FusionRuns& runs, const float2* tw, float2* work,
                               hipStream_t s) {
  if (N == 64)
    launch_cross_slab_t<64>(npairs, F, f_stride, G, g_stride, f_rows, f_planes, f_shared, g_rows,
                            g_planes, runs, tw, work, s);
  else
    launch_cross_slab_t<128>(npairs, F, f_stride, G, g_stride, f_rows, f_planes, f_shared,
                             g_rows, g_planes, runs, tw, work, s);
}

// column tiles: IT columns per workgroup, two padded LDS line buffers
int fft_cols_default_tile(int L) { return spatial_reg(L) ? kRegisterEngine : (L <= 128 ? 16 : 8); }

SpatialTiles spatial_default_tiles(int N) {
  SpatialTiles t;
  t.fwd_x = t.fwd_z = t.inv_x = fft_cols_default_tile(N);
  t.fused_reg = spatial_reg(N) != nullptr;
  return t;
}

bool fft_cols_tile_ok(int L, int it) {
  if (it == kRegisterEngine) return spatial_reg(L) != nullptr;
  return (it == 8 || it == 16 || it == 32 || it == 64) &&
         (2 * (size_t)it * (L + 1) + L) * sizeof(float2) <= 160 * 1024;
}

template <int DIR, int IT>
static void fft_cols_it(float2* data, int nbatch, int64_t batch_stride, int outer, int L,
                        int inner, const FftPlan& plan, const float2* tw, hipStream_t s,
                        VoxelOcc occ = {}) {
  dim3 g((inner + IT - 1) / IT, outer, nbatch);
  const int threads = IT <= 16 ? 256 : (IT == 32 ? 512 : 1024);
  hipLaunchKernelGGL((k_fft_cols<DIR, IT>), g, dim3(threads),
                     (2 * IT * (L + 1) + L) * sizeof(float2), s, data, batch_stride, L, inner,
                     plan, tw, occ.row, occ.plane);
}

template <int DIR>
static void fft_cols_t(float2* data, int nbatch, int64_t batch_stride, int outer, int L,
                       int inner, int it, const FftPlan& plan, const float2* tw, hipStream_t s) {
  if (!fft_cols_tile_ok(L, it)) it = fft_cols_default_tile(L);
  if (it == kRegisterEngine) {
    spatial_reg(L)->lines(DIR, data, nbatch, batch_stride, outer, inner, tw, s);
    return;
  }
  switch (it) {
    case 8: fft_cols_it<DIR, 8>(data, nbatch, batch_stride, outer, L, inner, plan, tw, s); break;
    case 16: fft_cols_it<DIR, 16>(data, nbatch, batch_stride, outer, L, inner, plan, tw, s); break;
    case 32: fft_cols_it<DIR, 32>(data, nbatch, batch_stride, outer, L, inner, plan, tw, s); break;
    default: fft_cols_it<DIR, 64>(data, nbatch, batch_stride, outer, L, inner, plan, tw, s); break;
  }
}

static void fft_cols(float2* data, int nbatch, int64_t batch_stride, int outer, int L, int inner,
                     int dir, int it, const FftPlan& plan, const float2* tw, hipStream_t s) {
  if (dir < 0)
    fft_cols_t<-1>(data, nbatch, batch_stride, outer, L, inner, it, plan, tw, s);
  else
    fft_cols_t<+1>(data, nbatch, batch_stride, outer, L, inner, it, plan, tw, s);
}

void launch_spatial_r2c(int N, int nclouds, const float* sumI, const float* sumR,
                        const uint32_t* cnt, const FftPlan& plan, const float2* tw, float2* spec,
                        hipStream_t s, const uint8_t* row_occ) {
  const int h = N / 2 + 1;
  const int64_t H = (int64_t)N * N * h, T = (int64_t)N * N * N;
  dim3 g((N * N + 15) / 16, nclouds);
  hipLaunchKernelGGL(k_spat_r2c<false>, g, dim3(256), (2 * 16 + 1) * N * sizeof(float2), s, N,
                     sumI, sumR, cnt, T, row_occ, plan, tw, spec, 2 * H, H);
}

void launch_spatial_fft_x_occ(int N, int nbatch, float2* spec, VoxelOcc occ, int it,
                              const FftPlan& plan, const float2* tw, hipStream_t s) {
  const int h = N / 2 + 1;
  const int64_t H = (int64_t)N * N * h;
  if (!fft_cols_tile_ok(N, it)) it = fft_cols_default_tile(N);
  switch (it) {
    case kRegisterEngine: spatial_reg(N)->x_occ(nbatch, spec, occ, tw, s); break;
    case 8: fft_cols_it<-1, 8>(spec, nbatch, H, N, N, h, plan, tw, s, occ); break;
    case 16: fft_cols_it<-1, 16>(spec, nbatch, H, N, N, h, plan, tw, s, occ); break;
    case 32: fft_cols_it<-1, 32>(spec, nbatch, H, N, N, h, plan, tw, s, occ); break;
    default: fft_cols_it<-1, 64>(spec, nbatch, H, N, N, h, plan, tw, s, occ); break;
  }
}

void launch_spatial_cross_zz(int N, int npairs, ChannelSet F, int64_t f_stride, ChannelSet G,
                             int64_t g_stride, const uint8_t* f_occ, int64_t f_occ_stride,
                             const uint8_t* g_occ, int64_t g_occ_stride, const FusionRuns& runs,
                             int it, const FftPlan& plan, const float2* tw, float2* work,
                             hipStream_t s) {
  const int inner = N * (N / 2 + 1);
  // the kernel holds 16 columns up to N = 128, 8 beyond
  if (N <= 128 && it != 8)
    hipLaunchKernelGGL(k_spat_cross_zz<16>, dim3((inner + 15) / 16, npairs), dim3(256),
                       (4 * 16 * (N + 1) + N) * sizeof(float2), s, N, F, f_stride, G, g_stride,
                       f_occ, f_occ_stride, g_occ, g_occ_stride, runs, plan, tw, work);
  else
    hipLaunchKernelGGL(k_spat_cross_zz<8>, dim3((inner + 7) / 8, npairs), dim3(256),
                       (4 * 8 * (N + 1) + N) * sizeof(float2), s, N, F, f_stride, G, g_stride,
                       f_occ, f_occ_stride, g_occ, g_occ_stride, runs, plan, tw, work);
}

bool spatial_plane_ok(int N) { return N <= kPlaneMaxN && spat_plane_lds_bytes(N) <= 160 * 1024; }

void launch_spatial_plane_fwd(int N, int nclouds, const float* sumI, const float* sumR,
                              const uint32_t* cnt, const FftPlan& plan, const float2* tw,
                              float2* spec, hipStream_t s) {
  const int h = N / 2 + 1;
  const int64_t H = (int64_t)N * N * h, T = (int64_t)N * N * N;
  hipLaunchKernelGGL(k_spat_plane_fwd, dim3(N, nclouds), dim3(256), spat_plane_lds_bytes(N), s, N,
                     sumI, sumR, cnt, T, plan, tw, spec, 2 * H, H);
}

void launch_spatial_fft_pass(int N, int nbatch, float2* buf, int which, int it,
                             const FftPlan& plan, const float2* tw, hipStream_t s) {
  const int h = N / 2 + 1;
  const int64_t H = (int64_t)N * N * h;
  if (which == 0)  // forward along x: [z][x][k2], columns over (z, k2)
    fft_cols(buf, nbatch, H, N, N, h, -1, it, plan, tw, s);
  else if (which == 1)  // forward along z: columns over (x, k2)
    fft_cols(buf, nbatch, H, 1, N, N * h, -1, it, plan, tw, s);
  else if (which == 2)  // inverse along x
    fft_cols(buf, nbatch, H, N, N, h, +1, it, plan, tw, s);
  else  // inverse along z
    fft_cols(buf, nbatch, H, 1, N, N * h, +1, it, plan, tw, s);
}

void launch_spatial_fft_fwd(int N, int nspec, float2* spec, const FftPlan& plan,
                            const float2* tw, const SpatialTiles& tiles, hipStream_t s) {
  // x then z, over all nspec half spectra
  launch_spatial_fft_pass(N, nspec, spec, 0, tiles.fwd_x, plan, tw, s);
  launch_spatial_fft_pass(N, nspec, spec, 1, tiles.fwd_z, plan, tw, s);
}

// r2c of one or two real grids (b null: one)
static void r2c_dense(int N, const float* a, const float* b, const FftPlan& plan,
                      const float2* tw, float2* spec, const SpatialTiles& tiles, hipStream_t s) {
  const int64_t H = (int64_t)N * N * (N / 2 + 1), T = (int64_t)N * N * N;
  if (const SpatialReg* reg = tiles.fused_reg ? spatial_reg(N) : nullptr) {
    reg->r2c_dense(a, b, tw, spec, s);
    return;
  }
  hipLaunchKernelGGL(k_spat_r2c<true>, dim3((N * N + 15) / 16, 1), dim3(256),
                     (2 * 16 + 1) * N * sizeof(float2), s, N, a, b, (const uint32_t*)nullptr, T,
                     (const uint8_t*)nullptr, plan, tw, spec, 0, b ? H : (int64_t)-1);
}

void launch_spatial_forward_dense(int N, int nch, const float* chans, const FftPlan& plan,
                                  const float2* tw, float2* spec, const SpatialTiles& tiles,
                                  hipStream_t s) {
  const int64_t H = (int64_t)N * N * (N / 2 + 1), T = (int64_t)N * N * N;
  for (int c = 0; c < nch; c += 2)
    r2c_dense(N, chans + c * T, c + 1 < nch ? chans + (c + 1) * T : nullptr, plan, tw,
              spec + c * H, tiles, s);
  launch_spatial_fft_fwd(N, nch, spec, plan, tw, tiles, s);
}

void launch_spatial_forward_two(int N, const float* a, const float* b, const FftPlan& plan,
                                const float2* tw, float2* spec, hipStream_t s) {
  const SpatialTiles tiles = spatial_default_tiles(N);
  r2c_dense(N, a, b, plan, tw, spec, tiles, s);
  launch_spatial_fft_fwd(N, 2, spec, plan, tw, tiles, s);
}

void launch_spatial_cross_z(int N, int npairs, ChannelSet F, int64_t f_stride, ChannelSet G,
                            int64_t g_stride, const FusionRuns& runs, bool fuse,
                            const FftPlan& plan, const float2* tw, float2* work, hipStream_t s) {
  const int inner = N * (N / 2 + 1);
  if (N <= 128)
    hipLaunchKernelGGL(k_spat_cross_z<16>, dim3((inner + 15) / 16, npairs), dim3(256),
                       (2 * 16 * (N + 1) + N) * sizeof(float2), s, N, F, f_stride, G, g_stride, runs,
                       (int)fuse, plan, tw, work);
  else
    hipLaunchKernelGGL(k_spat_cross_z<8>, dim3((inner + 7) / 8, npairs), dim3(256),
                       (2 * 8 * (N + 1) + N) * sizeof(float2), s, N, F, f_stride, G, g_stride, runs,
                       (int)fuse, plan, tw, work);
}

void launch_spatial_fft_inv(int N, int npairs, float2* work, const FftPlan& plan,
                            const float2* tw, const SpatialTiles& tiles, hipStream_t s) {
  launch_spatial_fft_pass(N, npairs, work, 2, tiles.inv_x, plan, tw, s);
}

void launch_spatial_c2r(int N, int npairs, const float2* work, const FftPlan& plan,
                        const float2* tw, float* corr, unsigned long long* partials,
                        unsigned long long* keys, hipStream_t s, uint32_t limit) {
  const int h = N / 2 + 1;
  const size_t sh = (16 * h + (2 * 8 + 1) * N) * sizeof(float2);
  hipLaunchKernelGGL(k_spat_c2r, dim3(spatial_c2r_blocks(N), npairs), dim3(256), sh, s, N, work,
                     plan, tw, corr, partials, limit);
  if (keys) launch_reduce_keys(partials, spatial_c2r_blocks(N), npairs, keys, s);
}

void launch_spatial_inverse(int N, int npairs, ChannelSet F, int64_t f_stride, ChannelSet G,
                            int64_t g_stride, const FusionRuns& runs, bool fuse,
                            const FftPlan& plan, const float2* tw, float2* work, float* corr,
                            unsigned long long* partials, unsigned long long* keys,
                            const SpatialTiles& tiles, hipStream_t s) {
  const SpatialReg* reg = tiles.fused_reg ? spatial_reg(N) : nullptr;
  if (reg)
    reg->cross_z(npairs, F, f_stride, G, g_stride, runs, fuse, tw, work, s);
  else
    launch_spatial_cross_z(N, npairs, F, f_stride, G, g_stride, runs, fuse, plan, tw, work, s);
  if (reg && reg->inv_plane) {
    reg->inv_plane(npairs, work, tw, corr, partials, false, s);
    launch_reduce_keys(partials, N, npairs, keys, s);
    return;
  }
  launch_spatial_fft_inv(N, npairs, work, plan, tw, tiles, s);
  if (reg) {
    reg->c2r(npairs, work, tw, corr, partials, s);
    launch_reduce_keys(partials, reg->c2r_blocks, npairs, keys, s);
  } else {
    launch_spatial_c2r(N, npairs, work, plan, tw, corr, partials, keys, s);
  }
}

void launch_trans_pose(int N, int lower, int upper, int npairs,
                       const unsigned long long* partials, int count, const float* corr,
                       int64_t corr_stride, int k, DevPose* pose, DevPose* result, hipStream_t s,
                       uint32_t n_corr, bool mixture) {
  if (n_corr == 0) n_corr = (uint32_t)N * N * N;
  hipLaunchKernelGGL(k_trans_pose, dim3(npairs), dim3(256), 0, s, N, lower, upper, partials, count,
                     corr, corr_stride, k, pose, n_corr, (int)mixture, result);
}

void launch_spatial_cross_product(int N, int npairs, ChannelSet F, int64_t f_stride,
                                  ChannelSet G, int64_t g_stride, const FusionRuns& runs,
                                  bool fuse, float2* work, hipStream_t s) {
  const int64_t H = (int64_t)N * N * (N / 2 + 1);
  hipLaunchKernelGGL(k_spat_cross_product, dim3((unsigned)((H + 255) / 256), npairs), dim3(256),
                     0, s, H, F, f_stride, G, g_stride, runs, (int)fuse, work);
}

void launch_spatial_pad_gather(int N, int pad, bool shifted, int npairs, const float2* work,
                               float2* out, hipStream_t s, int cube_lo, int cube_hi) {
  const int64_t H = (int64_t)N * N * (N / 2 + 1);
  const int64_t Np = N + 2 * pad, Hp = Np * Np * (Np / 2 + 1);
  hipLaunchKernelGGL(k_spat_pad_gather, dim3((unsigned)((Hp + 255) / 256), npairs), dim3(256),
                     0, s, N, pad, (int)shifted, work, H, out, Hp, cube_lo, cube_hi);
}

void launch_apply_pose(const float4* pts, int64_t P, const DevPose* pose, float4* out,
                       hipStream_t s) {
  if (P <= 0) return;
  hipLaunchKernelGGL(k_apply_pose, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, s, pts, P,
                     pose, out);
}

}  // namespace phz
