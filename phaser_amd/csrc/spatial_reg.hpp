// spatial_reg.hpp -- the passes of the translation stage on the register
// engine (fft_reg.hpp), one set of launchers per length (spatial_reg(N)).
// Each spatial_reg_*.hip instantiates a group of lengths.
#pragma once

#include "fft_reg.hpp"
#include "kernels.hpp"
#include "spatial_dev.hpp"

namespace phz {

namespace {

// pass 1: rows (z, x) along y, contiguous; R2 threads per row, n2 fastest.
// kDense: the rows are given as two real channels (a1 may be null: one
// channel, one spectrum out) instead of sums and counts.
// A row without points (row_occ 0) is not read: its transform is zero.
template <int L, bool kDense>
__global__ void __launch_bounds__(RegSplit<L>::TPB) k_spat_r2c_reg(
    const float* __restrict__ sumI, const float* __restrict__ sumR,
    const uint32_t* __restrict__ cnt, int64_t cloud_stride, const uint8_t* __restrict__ row_occ,
    const float2* __restrict__ tw, float2* __restrict__ spec, int64_t spec_stride0,
    int64_t spec_stride1) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, LINES = RegSplit<L>::LINES, S = RegSplit<L>::kRowStride;
  constexpr int h = L / 2 + 1;
  __shared__ float2 buf[LINES * S];
  __shared__ float2 table[L];
  const int ln = threadIdx.x / R2, n2 = threadIdx.x % R2;
  const int row0 = blockIdx.x * LINES, c = blockIdx.y;
  const int nrow = L * L - row0 < LINES ? L * L - row0 : LINES;  // of this workgroup
  const uint8_t* occ = row_occ ? row_occ + (int64_t)c * L * L + row0 : nullptr;
  const bool live = ln < nrow && (!occ || occ[ln]);
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  const int64_t off = c * cloud_stride + (int64_t)(row0 + ln) * L;
  float2 v[R1];
  if (kDense && live) {
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
      const int64_t o = off + n2 + R2 * n1;
      v[n1] = make_float2(sumI[o], sumR ? sumR[o] : 0.f);
    }
  } else if (live) {
    // count and sums of every voxel of the row in one batch of loads (the
    // sums of empty voxels are zero), then the means
    uint32_t k[R1];
    float si[R1], sr[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
      const int64_t o = off + n2 + R2 * n1;
      k[n1] = cnt[o];
      si[n1] = sumI[o];
      sr[n1] = sumR[o];
    }
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1)
      v[n1] = k[n1] ? make_float2(si[n1] / (float)k[n1], sr[n1] / (float)k[n1])
                    : make_float2(0.f, 0.f);
  } else {
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) v[n1] = make_float2(0.f, 0.f);
  }
  __syncthreads();
  float2 out[RegSplit<L>::C * R2];
  fft_four_step_reg<-1, L, RegSplit<L>::kRowPitch>(v, n2, buf + ln * S, w, out);
  __syncthreads();
  for_outputs<L>(n2, [&](int i, int k) { buf[ln * S + k] = out[i]; });
  __syncthreads();
  // split Z = I^ + i R^ into the two half spectra, coalesced over the rows
  float2* o0 = spec + c * spec_stride0 + (int64_t)row0 * h;
  float2* o1 = o0 + spec_stride1;
  for (int idx = threadIdx.x; idx < nrow * h; idx += blockDim.x) {
    const int r = idx / h, k = idx - r * h;
    const float2 zk = buf[r * S + k];
    const float2 zc = cconj(buf[r * S + (L - k) % L]);
    const float2 sm = cadd(zk, zc), d = csub(zk, zc);
    o0[idx] = make_float2(0.5f * sm.x, 0.5f * sm.y);
    if (!kDense || spec_stride1 >= 0) o1[idx] = make_float2(0.5f * d.y, -0.5f * d.x);
  }
}

// pass 1 over the occupied rows only: gridDim.z workgroups per (z plane,
// cloud).  A plane without points ends at once; otherwise its occupied rows
// are listed (ascending) in LDS and transformed LINES at a time, every
// gridDim.z-th batch by this workgroup, so rows from different parts of the
// plane share a batch.  Rows without points are
// neither read nor written (their spectrum is zero; only
// launch_spatial_fft_x_occ reads the result).
template <int L>
__global__ void __launch_bounds__(RegSplit<L>::TPB) k_spat_r2c_rows(
    const float* __restrict__ sumI, const float* __restrict__ sumR,
    const uint32_t* __restrict__ cnt, int64_t cloud_stride, const uint8_t* __restrict__ row_occ,
    const uint8_t* __restrict__ plane_occ, const float2* __restrict__ tw,
    float2* __restrict__ spec, int64_t spec_stride0, int64_t spec_stride1) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, LINES = RegSplit<L>::LINES, S = RegSplit<L>::kRowStride;
  constexpr int h = L / 2 + 1;
  constexpr int NW = RegSplit<L>::TPB / 64;
  static_assert(L <= RegSplit<L>::TPB, "one row per thread when listing");
  __shared__ float2 buf[LINES * S];
  __shared__ float2 table[L];
  __shared__ int rows[L];
  __shared__ int nrows;
  const int z = blockIdx.x, c = blockIdx.y;
  if (plane_occ[(int64_t)c * L + z] == 0) return;  // uniform over the workgroup
  const int ln = threadIdx.x / R2, n2 = threadIdx.x % R2;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  // list the occupied rows x of the plane in ascending order
  {
    const int x = threadIdx.x;
    const bool occ = x < L && row_occ[((int64_t)c * L + z) * L + x] != 0;
    const unsigned long long m = __ballot(occ);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    __shared__ int wcount[NW];
    if (lane == 0) wcount[wv] = __popcll(m);
    __syncthreads();
    int base = 0;
    for (int i = 0; i < wv; ++i) base += wcount[i];
    if (occ) rows[base + __popcll(m & ((1ull << lane) - 1ull))] = x;
    if (threadIdx.x == 0) {
      int total = 0;
      for (int i = 0; i < NW; ++i) total += wcount[i];
      nrows = total;
    }
    __syncthreads();
  }
  const int nr = nrows;
  const int64_t plane_off = (int64_t)z * L;  // first row of the plane
  for (int r0 = blockIdx.z * LINES; r0 < nr; r0 += gridDim.z * LINES) {
    const bool live = r0 + ln < nr;
    const int x = live ? rows[r0 + ln] : 0;
    const int64_t off = c * cloud_stride + (plane_off + x) * L;
    float2 v[R1];
    if (live) {
      uint32_t k[R1];
      float si[R1], sr[R1];
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) {
        const int64_t o = off + n2 + R2 * n1;
        k[n1] = cnt[o];
        si[n1] = sumI[o];
        sr[n1] = sumR[o];
      }
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1)
        v[n1] = k[n1] ? make_float2(si[n1] / (float)k[n1], sr[n1] / (float)k[n1])
                      : make_float2(0.f, 0.f);
    } else {
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) v[n1] = make_float2(0.f, 0.f);
    }
    float2 out[RegSplit<L>::C * R2];
    fft_four_step_reg<-1, L, RegSplit<L>::kRowPitch>(v, n2, buf + ln * S, w, out);
    __syncthreads();
    for_outputs<L>(n2, [&](int i, int k) { buf[ln * S + k] = out[i]; });
    __syncthreads();
    // split Z = I^ + i R^ into the two half spectra, one row of h at a time
    float2* o0 = spec + c * spec_stride0 + plane_off * h;
    float2* o1 = o0 + spec_stride1;
    const int nlive = nr - r0 < LINES ? nr - r0 : LINES;
    for (int idx = threadIdx.x; idx < nlive * h; idx += blockDim.x) {
      const int r = idx / h, k = idx - r * h;
      const int64_t o = (int64_t)rows[r0 + r] * h + k;
      const float2 zk = buf[r * S + k];
      const float2 zc = cconj(buf[r * S + (L - k) % L]);
      const float2 sm = cadd(zk, zc), d = csub(zk, zc);
      o0[o] = make_float2(0.5f * sm.x, 0.5f * sm.y);
      o1[o] = make_float2(0.5f * d.y, -0.5f * d.x);
    }
    __syncthreads();  // buf is reused by the next batch
  }
}

// Forward x pass over the spectra a sparse r2c left (spectrum b of
// cloud b / 2, layout [z][x][k2], k2 < h = L/2+1): line q = (z, k2) along x
// (stride h).  When plane z holds no points the line is zero and is neither
// read nor written; otherwise row x is read only where row (z, x) holds
// points.  The row bytes of the (at most two) planes a workgroup's lines
// touch are staged in LDS first, so that the predicated data loads are all
// in flight together.
template <int L>
__global__ void __launch_bounds__(RegSplit<L>::TPB) k_fft_x_occ(
    float2* __restrict__ data, int64_t batch_stride, const uint8_t* __restrict__ row_occ,
    const uint8_t* __restrict__ plane_occ, const float2* __restrict__ tw) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, h = L / 2 + 1, S = L + 1;
  constexpr int nlines = L * h, kLines = RegSplit<L>::LINES;
  static_assert(kLines <= h, "a workgroup's lines span at most two planes");
  __shared__ float2 buf[kLines * S];
  __shared__ float2 table[L];
  __shared__ uint8_t ob[2 * L + 2] __attribute__((aligned(4)));
  const int c = threadIdx.x % kLines, n2 = threadIdx.x / kLines;
  const BlockXY blk = xcd_block_xy();
  const int q = blk.x * kLines + c;
  const int cloud = blk.y >> 1;
  const int z0 = (blk.x * kLines) / h;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  if constexpr (L % 4 == 0) {
    for (int i = threadIdx.x; i < 2 * L / 4; i += blockDim.x) {
      const int zz = z0 + (4 * i) / L;
      ((uint32_t*)ob)[i] =
          zz < L ? ((const uint32_t*)(row_occ + ((int64_t)cloud * L + zz) * L))[i % (L / 4)] : 0u;
    }
  } else {
    for (int i = threadIdx.x; i < 2 * L; i += blockDim.x)
      ob[i] = z0 + i / L < L ? row_occ[((int64_t)cloud * L + z0) * L + i] : (uint8_t)0;
  }
  if (threadIdx.x < 2)  // planes z0, z0 + 1
    ob[2 * L + threadIdx.x] = z0 + threadIdx.x < L
                                  ? plane_occ[(int64_t)cloud * L + z0 + threadIdx.x] : (uint8_t)0;
  __syncthreads();
  float2* base = data + blk.y * batch_stride;
  bool live = q < nlines;
  const uint8_t* rb = ob;
  if (live) {
    const int z = q / h;
    live = ob[2 * L + (z - z0)] != 0;
    base += (int64_t)z * L * h + (q - z * h);
    rb = ob + (z - z0) * L;
  }
  if (!__syncthreads_or(live)) return;  // uniform over the workgroup
  // predicated loads: masked buffer loads (SpectrumReader) measured slower
  // here (16 pairs: 106 against 94 us at L = 128, 163 against 140 at 144),
  // where nothing but these loads and the stores is left to overlap
  float2 v[R1];
#pragma unroll
  for (int n1 = 0; n1 < R1; ++n1) {
    const int e = n2 + R2 * n1;
    v[n1] = (live && rb[e]) ? base[(int64_t)e * h] : make_float2(0.f, 0.f);
  }
  fft_four_step<-1, L>(v, n2, buf + c * S, w, [&](int k, float2 x) {
    if (live) base[(int64_t)k * h] = x;
  });
}

// inverse pass A: fused F, G -> C = F conj(G) -> inverse FFT along z, for
// lines q = (x, k2) of stride inner = N h; pair blockIdx.y.
template <int L>
__global__ void __launch_bounds__(RegSplit<L>::TPB) k_spat_cross_z_reg(
    ChannelSet F, int64_t f_stride, ChannelSet G, int64_t g_stride, FusionRuns runs, int fuse,
    const float2* __restrict__ tw, float2* __restrict__ work) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, LINES = RegSplit<L>::LINES, S = L + 1;
  constexpr int inner = L * (L / 2 + 1);
  __shared__ float2 buf[LINES * S];
  __shared__ float2 table[L];
  const int cl = threadIdx.x % LINES, n2 = threadIdx.x / LINES;
  const int q = blockIdx.x * LINES + cl;
  const bool live = q < inner;
  const int64_t fo = blockIdx.y * f_stride, go = blockIdx.y * g_stride;
  float2* wp = work + blockIdx.y * (int64_t)L * inner + q;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  float2 v[R1];
#pragma unroll
  for (int n1 = 0; n1 < R1; ++n1) {
    float2 cz = make_float2(0.f, 0.f);
    if (live) {
      const int64_t idx = (int64_t)(n2 + R2 * n1) * inner + q;
      float2 f, g;
      if (fuse) {
        int mode = 0;
        for (int r = 0; r < runs.count; ++r)
          if ((uint64_t)idx >= runs.start[r]) mode = (int)runs.mode[r];
        f = fuse_at(F, mode, idx + fo);
        g = fuse_at(G, mode, idx + go);
      } else {
        f = F.ch[0][idx + fo];
        g = G.ch[0][idx + go];
      }
      cz.x = f.x * g.x - f.y * (-g.y);
      cz.y = f.x * (-g.y) + f.y * g.x;
    }
    v[n1] = cz;
  }
  __syncthreads();
  fft_four_step<+1, L>(v, n2, buf + cl * S, w, [&](int k, float2 x) {
    if (live) wp[(int64_t)k * inner] = x;
  });
}

// bit n1 of the result: plane z = n2 + R2 n1 holds points
template <int L>
__device__ __forceinline__ uint32_t plane_bits(const uint8_t* occ, int n2) {
  uint32_t m = 0u;
#pragma unroll
  for (int n1 = 0; n1 < RegSplit<L>::R1; ++n1)
    m |= occ[n2 + RegSplit<L>::R2 * n1] ? 1u << n1 : 0u;
  return m;
}

// One side (F or G) of the cross spectrum of NCH live channels: each
// channel's forward FFT along z (occupied planes only, bits planes), folded
// into acc in channel order as fuse_at does, but for its last step: mode 0
// keeps the first channel of largest energy, mode 1 sums ((c0 + c1) + c2) + c3.
template <int L, int NCH, class TW>
__device__ __forceinline__ void fused_side(const ChannelSet& X, int64_t off, uint32_t planes,
                                           int q, int n2, float2* lb, const TW& w, uint32_t sum,
                                           float2 (&acc)[RegSplit<L>::C * RegSplit<L>::R2]) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, E = RegSplit<L>::C * R2;
  constexpr int inner = L * (L / 2 + 1);
  float best[E];
  // a channel's loads are issued before the previous one is transformed
  float2 next[R1];
  const uint32_t base = (uint32_t)(n2 * inner + q) * 8u;
  auto load = [&](int c) {
    const SpectrumReader rd(X.ch[c] + off, (int64_t)inner * L);
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) next[n1] = rd.at(base, R2 * n1 * inner * 8, (planes >> n1) & 1u);
  };
  load(0);
  // no sum in any lane of the wave (most of the spectrum): the shorter fold
  const bool any_sum = __ballot(sum != 0u) != 0ull;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    float2 a[R1], xa[E];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) a[n1] = next[n1];
    if (c + 1 < NCH) load(c + 1);
    fft_four_step_reg<-1, L>(a, n2, lb, w, xa);
    __syncthreads();
    if (c == 0) {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        acc[i] = xa[i];
        best[i] = xa[i].x * xa[i].x + xa[i].y * xa[i].y;
      }
    } else if (!any_sum) {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float e = xa[i].x * xa[i].x + xa[i].y * xa[i].y;
        const bool take = e > best[i];
        acc[i].x = take ? xa[i].x : acc[i].x;
        acc[i].y = take ? xa[i].y : acc[i].y;
        best[i] = take ? e : best[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < E; ++i) {
        const float e = xa[i].x * xa[i].x + xa[i].y * xa[i].y;
        const bool add = (sum >> RegSplit<L>::order(i)) & 1u, take = e > best[i];
        const float2 t = cadd(acc[i], xa[i]);
        acc[i].x = add ? t.x : (take ? xa[i].x : acc[i].x);
        acc[i].y = add ? t.y : (take ? xa[i].y : acc[i].y);
        best[i] = take ? e : best[i];
      }
    }
  }
}

// Forward FFT along z of the NCH live channels of every x-transformed half
// spectrum of a pair (4: clouds with reflectivity and ambient, else 2), Laplace
// fusion, C = F conj(G) and the inverse FFT along z, all in registers (one LDS
// exchange per transform): the z-pass output is never stored.  Lines q = (x,
// k2) with stride inner = L h; pair blockIdx.y reads F.ch[c] + p f_stride and
// G.ch[c] + p g_stride (the other C - NCH channels are absent) and, where
// f_occ / g_occ are given (the clouds' z-plane occupancy, advanced by p
// f_occ_stride / p g_occ_stride), only the planes that hold points; the others
// are zero and were never written by the x pass.  A side's channels are
// transformed one after the other, each one's loads in flight during the
// previous transform, which bounds the registers held.
// Bound by memory: 16 pairs at L = 128 move 0.49 GB in 139 us, 3.5 TB/s of the
// copy kernel's 4.5 (the spectra of more than a few pairs do not stay in the
// cache); 64 pairs 2.1 GB at 4.4, 16 at 192 1.7 GB at 3.8, 8 at 256 2.2 GB at 3.7.
// At 150, 180 and 216 (960 and 576 threads: 128 and 168 registers) and with four
// channels at 200 the state spills: 53, 1 and 1 registers with two channels,
// 381, 342 and 409 with four, 126 at 200.  It is still well ahead of the LDS form
// there (whole calls with that form: 7 pairs at 150 575 against 960 us, with four
// channels 999 / 1514; 4 at 180 542 / 950 and 966 / 1502; 2 at 216 487 / 1039 and
// 873 / 1688; 3 at 200 with four 862 / 1496).  Masked buffer loads and branch-free fusion in place of predicated
// global loads and per-entry branches: 367 -> 263 us at L = 192, 87 -> 62 at 96.
template <int L, int NCH>
__global__ void __launch_bounds__(RegSplit<L>::TPB, 2) k_spat_cross_zz_reg(
    ChannelSet F, int64_t f_stride, ChannelSet G, int64_t g_stride,
    const uint8_t* __restrict__ f_occ, int64_t f_occ_stride, const uint8_t* __restrict__ g_occ,
    int64_t g_occ_stride, PlaneRuns runs, const float2* __restrict__ tw,
    float2* __restrict__ work) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, LINES = RegSplit<L>::LINES, S = L + 1;
  constexpr int inner = L * (L / 2 + 1), E = RegSplit<L>::C * R2;
  static_assert(RegSplit<L>::kOrdered, "entries at equal steps of frequency");
  __shared__ float2 buf[LINES * S];
  __shared__ float2 table[L];
  __shared__ uint8_t occ_b[2 * L];
  const int cl = threadIdx.x % LINES, n2 = threadIdx.x / LINES;
  const BlockXY blk = xcd_block_xy();
  const int q = blk.x * LINES + cl;
  const bool live = q < inner;
  const int p = blk.y;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  for (int i = threadIdx.x; i < 2 * L; i += blockDim.x) {
    const uint8_t* o = i < L ? f_occ : g_occ;
    const int64_t st = i < L ? f_occ_stride : g_occ_stride;
    occ_b[i] = o ? o[p * st + i % L] : (uint8_t)1;
  }
  __syncthreads();
  float2* lb = buf + cl * S;
  const FusionBits mode = fusion_bits<E, RegSplit<L>::kStep>(runs, n2, q);
  float2 ff[E], gf[E];
  fused_side<L, NCH>(F, p * f_stride, live ? plane_bits<L>(occ_b, n2) : 0u, q, n2, lb, w, mode.sum,
                     ff);
  fused_side<L, NCH>(G, p * g_stride, live ? plane_bits<L>(occ_b + L, n2) : 0u, q, n2, lb, w,
                     mode.sum, gf);
#pragma unroll
  for (int i = 0; i < E; ++i) {
    const float2 f = ff[i], g = gf[i];
    ff[i] = make_float2(f.x * g.x - f.y * (-g.y), f.x * (-g.y) + f.y * g.x);
  }
  if (__ballot((mode.sum | mode.zero) != 0u)) {
    // the mean over C = 4 channels on both sides: 1/16, a power of two, so the
    // same value as dividing each side; a zero stays one
#pragma unroll
    for (int i = 0; i < E; ++i) {
      const int e = RegSplit<L>::order(i);
      const bool mean = (mode.sum >> e) & 1u, zero = (mode.zero >> e) & 1u;
      const float2 m = cscale(ff[i], 0.0625f);
      ff[i].x = zero ? 0.f : (mean ? m.x : ff[i].x);
      ff[i].y = zero ? 0.f : (mean ? m.y : ff[i].y);
    }
  }
  float2* wp = work + p * (int64_t)L * inner + q;
  // inverse z: an even split's outputs are, reordered, the inputs of the
  // same split; otherwise the split with its factors swapped
  if constexpr (RegSplit<L>::kEven) {
    float2 v[R1];
#pragma unroll
    for (int j = 0; j < R1 / R2; ++j)
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) v[j + (R1 / R2) * k2] = ff[j * R2 + k2];
    fft_four_step<+1, L>(v, n2, lb, w, [&](int k, float2 x) {
      if (live) wp[(int64_t)k * inner] = x;
    });
  } else {
    fft_from_outputs<+1, L>(ff, n2, lb, table, [&](int k, float2 x) {
      if (live) wp[(int64_t)k * inner] = x;
    });
  }
}

// last pass: c2r along y (real parts of k = 0, N/2, FFTW hc2r), two rows per
// complex line, signed first-maximum argmax over x*N + y + N^2*z.
template <int L>
__global__ void __launch_bounds__(RegSplit<L>::TPB) k_spat_c2r_reg(const float2* __restrict__ work,
                                                      const float2* __restrict__ tw,
                                                      float* __restrict__ corr,
                                                      unsigned long long* __restrict__ partials) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, LINES = RegSplit<L>::LINES, S = RegSplit<L>::kRowStride;
  constexpr int h = L / 2 + 1, rows = L * L;
  // the workgroup's 2 LINES rows are contiguous: staged through LDS with
  // 16-byte loads, then the transform's line buffers reuse the space
  constexpr int kStage = 2 * LINES * h, kLds = kStage > LINES * S ? kStage : LINES * S;
  __shared__ __align__(16) float2 buf[kLds];
  __shared__ float2 table[L];
  const int ln = threadIdx.x / R2, n2 = threadIdx.x % R2;
  const int ra = (blockIdx.x * LINES + ln) * 2;  // rows ra, ra + 1 (rows is even)
  const bool live = ra < rows;  // the last workgroup may have idle lines
  work += blockIdx.y * (int64_t)rows * h;
  if (corr) corr += blockIdx.y * (int64_t)rows * L;
  partials += blockIdx.y * (int64_t)gridDim.x;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  {
    static_assert(kStage % 2 == 0, "whole float4s");
    const float4* src = (const float4*)(work + (int64_t)blockIdx.x * 2 * LINES * h);
    const int left = (rows - (int)blockIdx.x * 2 * LINES) * h;  // entries from here, even
    const int n4 = (left < kStage ? left : kStage) / 2;
    for (int i = threadIdx.x; i < n4; i += blockDim.x) ((float4*)buf)[i] = src[i];
  }
  __syncthreads();
  const float2* xa = buf + 2 * ln * h;
  const float2* xb = xa + h;
  float2 v[R1];
#pragma unroll
  for (int n1 = 0; n1 < R1; ++n1) {
    const int m = n2 + R2 * n1;
    float2 va = make_float2(0.f, 0.f), vb = va;
    if (!live) {
    } else if (m == 0 || 2 * m == L) {
      va = make_float2(xa[m].x, 0.f);
      vb = make_float2(xb[m].x, 0.f);
    } else if (m < h) {
      va = xa[m];
      vb = xb[m];
    } else {
      va = cconj(xa[L - m]);
      vb = cconj(xb[L - m]);
    }
    v[n1] = make_float2(va.x - vb.y, va.y + vb.x);
  }
  __syncthreads();  // the staged rows are read; the line buffers overwrite them
  float2 out[RegSplit<L>::C * R2];
  fft_four_step_reg<+1, L, RegSplit<L>::kRowPitch>(v, n2, buf + ln * S, w, out);
  // row ra's indices all lie below row ra + 1's
  FirstMax<true> ma, mb;
  const uint32_t la = (uint32_t)ra * L;
  if (live)
    for_outputs_ascending<L>(n2, [&](int i, int y, int e) {
      if (corr) {
        corr[la + y] = out[i].x;
        corr[la + L + y] = out[i].y;
      }
      ma.take(out[i].x, e);
      mb.take(out[i].y, e);
    });
  unsigned long long best = ma.key(la + place_frequency<L>(n2, ma.tag));
  const unsigned long long kb = mb.key(la + L + place_frequency<L>(n2, mb.tag));
  best = !live ? 0ull : (kb > best ? kb : best);
  best = block_max_key(best);
  if (threadIdx.x == 0) partials[blockIdx.x] = best;
}

// Inverse FFT along x and c2r along y of one z plane of a pair, with the
// plane in LDS (L h complex, 66.5 KB at L = 128): the x-transformed plane is
// never stored.  Workgroup (z, pair) of TPB threads: lines of R2 threads,
// LINES = TPB / R2 at a time (line = thread % LINES fastest, n2 = thread /
// LINES).  Pass x: L / 2 lines, one per column k2 = 1 .. L/2 - 1 and line 0
// for columns 0 and L/2 together: c2r reads only the real parts of those two,
// and Re IFFT(a) + i Re IFFT(b) = IFFT(a_h + i b_h) with the Hermitian parts
// a_h[k] = (a[k] + conj a[-k]) / 2.  Each line exchanges through its own
// column (stride h) and writes its results back there.  Pass y: row pairs
// (2r, 2r + 1) packed as one complex line (real parts of k = 0, L/2, FFTW
// hc2r), exchanging through the pair's own two rows; signed first-maximum
// argmax over x N + y + N^2 z into partials[pair][z]; the grid is written
// when corr is given.  kSlab: work is laid out [pair][k2][z][x] (the output
// of k_spat_cross_slab) instead of [pair][z][x][k2]; the plane's h rows of
// L entries are transposed into the same LDS layout as they are stored.
template <int L, int TPB, bool kSlab>
__global__ void __launch_bounds__(TPB) k_spat_inv_plane(const float2* __restrict__ work,
                                                        const float2* __restrict__ tw,
                                                        float* __restrict__ corr,
                                                        unsigned long long* __restrict__ partials) {
  constexpr int R1 = RegSplit<L>::R1, R2 = RegSplit<L>::R2, LINES = TPB / R2;
  constexpr int h = L / 2 + 1;
  static_assert(TPB % R2 == 0 && TPB % 64 == 0, "whole lines and waves");
  constexpr bool kWhole = (L / 2) % LINES == 0;  // no idle lines in the last pass
  __shared__ __align__(16) float2 P[L * h];
  __shared__ float2 table[L];
  const int c = threadIdx.x % LINES, n2 = threadIdx.x / LINES;
  const int z = blockIdx.x, pair = blockIdx.y;
  const LdsTwiddles<L> w = stage_twiddles<L>(table, n2, tw);
  if (kSlab) {
    // h rows (k2) of L contiguous entries (x), two per float4, all loads
    // of a thread in flight before its LDS stores
    constexpr int NV = h * L / 2, PER = (NV + TPB - 1) / TPB;
    const float4* src = (const float4*)(work + (int64_t)pair * h * L * L + (int64_t)z * L);
    float4 t[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = threadIdx.x + TPB * i, ic = idx < NV ? idx : NV - 1;
      const int k2 = ic / (L / 2), x2 = ic - k2 * (L / 2);
      t[i] = src[(int64_t)k2 * (L * L / 2) + x2];  // in bounds; the stores are predicated
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = threadIdx.x + TPB * i;
      if (idx < NV) {
        const int k2 = idx / (L / 2), x = 2 * (idx - k2 * (L / 2));
        P[x * h + k2] = make_float2(t[i].x, t[i].y);
        P[(x + 1) * h + k2] = make_float2(t[i].z, t[i].w);
      }
    }
  } else {
    // the plane (L h complex) in one batch of loads per thread, then into
    // LDS: a strided copy loop waits for each load before its LDS store,
    // one HBM round trip per iteration
    static_assert((L * h) % 2 == 0, "whole float4s");
    constexpr int NV = L * h / 2, PER = (NV + TPB - 1) / TPB;
    const float4* src = (const float4*)(work + ((int64_t)pair * L + z) * L * h);
    float4 t[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = threadIdx.x + TPB * i;
      t[i] = src[idx < NV ? idx : NV - 1];  // in bounds; the store below is predicated
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = threadIdx.x + TPB * i;
      if (idx < NV) ((float4*)P)[idx] = t[i];
    }
  }
  __syncthreads();
  // inverse FFT along x
  for (int g0 = 0; g0 < L / 2; g0 += LINES) {
    const int k2 = g0 + c;  // line 0: columns 0 and L/2
    const bool live = kWhole || k2 < L / 2;  // an idle line exchanges in no column
    float2 v[R1], out[RegSplit<L>::C * R2];
    if (k2 == 0) {
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) {
        const int x = n2 + R2 * n1, xm = x ? L - x : 0;
        const float2 a = P[x * h], ar = P[xm * h], b = P[x * h + L / 2], br = P[xm * h + L / 2];
        const float2 ah = make_float2(0.5f * (a.x + ar.x), 0.5f * (a.y - ar.y));
        const float2 bh = make_float2(0.5f * (b.x + br.x), 0.5f * (b.y - br.y));
        v[n1] = make_float2(ah.x - bh.y, ah.y + bh.x);
      }
    } else if (live) {
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) v[n1] = P[(n2 + R2 * n1) * h + k2];
    }
    __syncthreads();  // the columns are read before the exchanges overwrite them
    fft_four_step_reg<+1, L>(v, n2, P + k2, w, out, h, live);
    __syncthreads();  // the exchanges are read before the results go back
    if (live)
      for_outputs<L>(n2, [&](int i, int x) {
        const float2 o = out[i];
        if (k2 == 0) {
          P[x * h] = make_float2(o.x, 0.f);
          P[x * h + L / 2] = make_float2(o.y, 0.f);
        } else {
          P[x * h + k2] = o;
        }
      });
    __syncthreads();
  }
  // c2r along y, two rows per complex line; here the R2 threads of a line
  // are adjacent (n2 fastest) so that a line's grid stores are contiguous
  const int ln = threadIdx.x / R2, m2 = threadIdx.x % R2;
  const LdsTwiddles<L> wy{table + m2};
  unsigned long long best = 0ull;
  for (int r0 = 0; r0 < L / 2; r0 += LINES) {
    const int ra = 2 * (r0 + ln);
    const bool live = kWhole || ra < L;
    float2* xa = P + ra * h;
    const float2* xb = xa + h;
    float2 v[R1];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
      const int m = m2 + R2 * n1;
      float2 va = make_float2(0.f, 0.f), vb = va;
      if (!live) {
      } else if (m == 0 || 2 * m == L) {
        va = make_float2(xa[m].x, 0.f);
        vb = make_float2(xb[m].x, 0.f);
      } else if (m < h) {
        va = xa[m];
        vb = xb[m];
      } else {
        va = cconj(xa[L - m]);
        vb = cconj(xb[L - m]);
      }
      v[n1] = make_float2(va.x - vb.y, va.y + vb.x);
    }
    __syncthreads();  // the rows are read before the exchange overwrites them
    float2 out[RegSplit<L>::C * R2];
    fft_four_step_reg<+1, L>(v, m2, xa, wy, out, 1, live);
    if (live) {
      // row ra's indices all lie below row ra + 1's
      FirstMax<true> ma, mb;
      const uint32_t la = (uint32_t)(z * L + ra) * L;
      float* const ga = corr ? corr + (int64_t)pair * L * L * L + la : nullptr;
      for_outputs_ascending<L>(m2, [&](int i, int y, int e) {
        if (corr) {
          ga[y] = out[i].x;
          ga[L + y] = out[i].y;
        }
        ma.take(out[i].x, e);
        mb.take(out[i].y, e);
      });
      const unsigned long long ka = ma.key(la + place_frequency<L>(m2, ma.tag));
      const unsigned long long kb = mb.key(la + L + place_frequency<L>(m2, mb.tag));
      best = ka > best ? ka : best;
      best = kb > best ? kb : best;
    }
  }
  best = block_max_key(best);
  if (threadIdx.x == 0) partials[(int64_t)pair * L + z] = best;
}


// threads of the inverse plane pass: its lines in as few rounds as 1024
// threads allow, in whole lines and waves
constexpr int wave_lines(int r) {  // the least multiple of r that is whole waves
  int t = r;
  while (t % 64) t += r;
  return t;
}
constexpr int plane_threads(int L, int R2) {
  const int all = (L / 2) * R2, u = wave_lines(R2);
  for (int rounds = 1;; ++rounds) {
    const int t = ((all + rounds - 1) / rounds + u - 1) / u * u;
    if (t <= 1024) return t;
  }
}

template <int L>
struct SpatialRegT {
  static constexpr int LINES = RegSplit<L>::LINES, TPB = RegSplit<L>::TPB, h = L / 2 + 1;
  static constexpr int64_t H = (int64_t)L * L * h, T = (int64_t)L * L * L;
  // workgroups per plane of the sparse r2c in a small launch
  static constexpr int kRowSplit = (L + LINES - 1) / LINES < 4 ? (L + LINES - 1) / LINES : 4;
  static constexpr int kC2rBlocks = (L * L + 2 * LINES - 1) / (2 * LINES);

  static void lines(int dir, float2* data, int nbatch, int64_t batch_stride, int outer, int inner,
                    const float2* tw, hipStream_t s) {
    const int nl = outer * inner;
    const dim3 g((nl + LINES - 1) / LINES, nbatch);
    if (dir < 0)
      hipLaunchKernelGGL((k_fft_lines<-1, L>), g, dim3(TPB), 0, s, data, batch_stride, nl, inner, tw);
    else
      hipLaunchKernelGGL((k_fft_lines<+1, L>), g, dim3(TPB), 0, s, data, batch_stride, nl, inner, tw);
  }
  static void r2c(int nclouds, const float* sumI, const float* sumR, const uint32_t* cnt,
                  const uint8_t* row_occ, const float2* tw, float2* spec, hipStream_t s) {
    hipLaunchKernelGGL((k_spat_r2c_reg<L, false>), dim3((L * L + LINES - 1) / LINES, nclouds),
                       dim3(TPB), 0, s, sumI, sumR, cnt, T, row_occ, tw, spec, 2 * H, H);
  }
  static void r2c_dense(const float* a, const float* b, const float2* tw, float2* spec,
                        hipStream_t s) {
    hipLaunchKernelGGL((k_spat_r2c_reg<L, true>), dim3((L * L + LINES - 1) / LINES, 1), dim3(TPB),
                       0, s, a, b, (const uint32_t*)nullptr, T, (const uint8_t*)nullptr, tw, spec,
                       (int64_t)0, b ? H : (int64_t)-1);
  }
  static void r2c_rows(int nclouds, const float* sumI, const float* sumR, const uint32_t* cnt,
                       VoxelOcc occ, const float2* tw, float2* spec, hipStream_t s) {
    // a workgroup per batch of rows where the planes alone leave the chip idle
    // (one pair at L = 128: 14.8 -> 9.5 us), else one per plane (16 pairs at
    // L = 192: 128 us, split 143)
    const int split = L * nclouds < 2048 ? kRowSplit : 1;
    hipLaunchKernelGGL(k_spat_r2c_rows<L>, dim3(L, nclouds, split), dim3(TPB), 0, s, sumI, sumR,
                       cnt, T, occ.row, occ.plane, tw, spec, 2 * H, H);
  }
  static void x_occ(int nbatch, float2* spec, VoxelOcc occ, const float2* tw, hipStream_t s) {
    hipLaunchKernelGGL(k_fft_x_occ<L>, dim3((L * h + LINES - 1) / LINES, nbatch), dim3(TPB), 0, s,
                       spec, H, occ.row, occ.plane, tw);
  }
  static void cross_z(int npairs, ChannelSet F, int64_t fs, ChannelSet G, int64_t gs,
                      const FusionRuns& runs, bool fuse, const float2* tw, float2* work,
                      hipStream_t s) {
    hipLaunchKernelGGL(k_spat_cross_z_reg<L>, dim3((L * h + LINES - 1) / LINES, npairs), dim3(TPB),
                       0, s, F, fs, G, gs, runs, (int)fuse, tw, work);
  }
  static void cross_zz(int nch, int npairs, ChannelSet F, int64_t fs, ChannelSet G, int64_t gs,
                       const uint8_t* f_occ, int64_t f_occ_stride, const uint8_t* g_occ,
                       int64_t g_occ_stride, const FusionRuns& fusion, const float2* tw,
                       float2* work, hipStream_t s) {
    const PlaneRuns runs = plane_runs(fusion, L * h);
    const dim3 g((L * h + LINES - 1) / LINES, npairs);
    if (nch == 4) {
      hipLaunchKernelGGL((k_spat_cross_zz_reg<L, 4>), g, dim3(TPB), 0, s, F, fs, G, gs, f_occ,
                         f_occ_stride, g_occ, g_occ_stride, runs, tw, work);
      return;
    }
    hipLaunchKernelGGL((k_spat_cross_zz_reg<L, 2>), g, dim3(TPB), 0, s, F, fs, G, gs, f_occ,
                       f_occ_stride, g_occ, g_occ_stride, runs, tw, work);
  }
  static void c2r(int npairs, const float2* work, const float2* tw, float* corr,
                  unsigned long long* partials, hipStream_t s) {
    hipLaunchKernelGGL(k_spat_c2r_reg<L>, dim3(kC2rBlocks, npairs), dim3(TPB), 0, s, work, tw,
                       corr, partials);
  }
  static void inv_plane(int npairs, const float2* work, const float2* tw, float* corr,
                        unsigned long long* partials, bool slab, hipStream_t s) {
    if constexpr (L <= kInvPlaneMax) {
      constexpr int PT = plane_threads(L, RegSplit<L>::R2);
      if constexpr (L == 64 || L == 128) {
        if (slab) {
          hipLaunchKernelGGL((k_spat_inv_plane<L, PT, true>), dim3(L, npairs), dim3(PT), 0, s,
                             work, tw, corr, partials);
          return;
        }
      }
      hipLaunchKernelGGL((k_spat_inv_plane<L, PT, false>), dim3(L, npairs), dim3(PT), 0, s, work,
                         tw, corr, partials);
    }
  }
  static constexpr SpatialReg ops() {
    return SpatialReg{L,     lines,    r2c,  r2c_dense, r2c_rows,   x_occ, cross_z,
                      cross_zz, c2r, L <= kInvPlaneMax ? inv_plane : nullptr, kC2rBlocks};
  }
};

}  // namespace

// NAME(N): the passes of length N, or null, for the lengths of LIST
#define PHZ_SPATIAL_REG_OPS(LEN, A, B) SpatialRegT<LEN>::ops(),
#define PHZ_SPATIAL_REG_GROUP(NAME, LIST)                         \
  const SpatialReg* NAME(int N) {                                 \
    static constexpr SpatialReg ops[] = {LIST(PHZ_SPATIAL_REG_OPS)}; \
    for (const SpatialReg& o : ops)                               \
      if (o.N == N) return &o;                                    \
    return nullptr;                                               \
  }

}  // namespace phz
