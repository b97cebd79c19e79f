// Kaiser-Bessel interpolation kernels for CDNA4 (gfx950); the adjoint's
// spread is in spread.hip.
//
// interp (forward convolution, reference CUDA/src/gpu/atomic/
//   atomic_gpuNUFFT_kernels.cu:966-1400, texture_gpuNUFFT_kernels.cu:467-1039)
//
// Work decomposition: one workgroup per (sector chunk, coil block). A chunk
// is a contiguous run of at most `chunk` sorted samples of one sector, so
// heavy sectors near the k-space centre spread over many workgroups while
// ordinary sectors are one chunk each. Workgroup ids are remapped so that
// each of the 8 XCDs owns a contiguous range of chunks (neighbouring sectors
// share that XCD's L2).
//
// A chunk is processed in rounds of R samples (R sized to the LDS left over
// by the sub-grid). Each round first computes, once per sample, a tap record
// in LDS: the first tap index along each axis, whether the sample has kw+1
// taps along it, and the per-axis kernel weights (zero where the reference
// skips a tap). The tap loop then runs with lanes = (sample slot, coil);
// its trip counts are wave-uniform (kw, or kw+1 when any lane of the wave
// needs it), so no lane idles through masked iterations.
//
// Two kernel families: for kernel width 3 in 2-D the "lane" kernels form each
// sample's tap record in registers and share it across the four lanes of a
// quad (one lane per coil) with DPP moves; the round-based kernels stage tap
// records in LDS per round of samples.

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "gnufft_internal.hpp"

namespace gnufft {

constexpr int kThreads = 512;

// Chunk of workgroup bid: the (bid / 8)-th chunk of XCD (bid % 8)'s range,
// or ~0u past the end of that range.
__device__ inline uint32_t work_chunk(const WorkList& w, uint32_t bid) {
  const uint32_t x = bid & 7u;
  const uint32_t ci = w.xcd_begin[x] + (bid >> 3);
  return ci < w.xcd_begin[x + 1] ? ci : ~0u;
}

// Workgroups along x for a work list.
static inline uint32_t work_blocks(const WorkList& w) { return 8u * (w.max_range ? w.max_range : 1u); }

// Split n items of the given costs into 8 contiguous ranges of about equal
// total cost: begin[x] .. begin[x+1] is range x.
static void split_ranges(const uint32_t* costs, uint32_t n, uint32_t begin[9], uint32_t* max_range) {
  double total = 0.0;
  for (uint32_t i = 0; i < n; i++) total += (double)costs[i];
  uint32_t x = 0;
  double acc = 0.0;
  begin[0] = 0;
  for (uint32_t i = 0; i < n && x < 7; i++) {
    acc += (double)costs[i];
    while (x < 7 && acc >= total * (double)(x + 1) / 8.0) begin[++x] = i + 1;
  }
  while (x < 8) begin[++x] = n;
  *max_range = 0;
  for (int k = 0; k < 8; k++) *max_range = std::max(*max_range, begin[k + 1] - begin[k]);
}

void partition_work(const uint32_t* counts, uint32_t n, WorkList* w) {
  // Cost of a chunk: its samples plus a fixed share for staging and
  // storing the padded sub-grid (about 300 samples' worth on gfx950).
  std::vector<uint32_t> cost(n);
  for (uint32_t i = 0; i < n; i++) cost[i] = counts[i] + 300u;
  split_ranges(cost.data(), n, w->xcd_begin, &w->max_range);
  w->n_chunks = n;
}

void partition_items(const uint32_t* costs, uint32_t n, BatchList* l) {
  split_ranges(costs, n, l->xcd_begin, &l->max_range);
  l->n = n;
}

static inline uint32_t batch_blocks(const BatchList& l) { return 8u * (l.max_range ? l.max_range : 1u); }

template <int DIM>
__device__ inline void load_center(const Geom& g, uint32_t sector, int* c) {
  // the standard center layout (index * sw + sw / 2 per axis, the only one
  // plans accept, gpuNUFFT_operator_factory.cpp:207-214): computed, not
  // loaded, which saves a dependent memory round trip at workgroup start
  const uint32_t x = sector % (uint32_t)g.S[0];
  const uint32_t yz = sector / (uint32_t)g.S[0];
  const int half = g.sw / 2;
  c[0] = (int)x * g.sw + half;
  c[1] = (int)(yz % (uint32_t)g.S[1]) * g.sw + half;
  c[2] = DIM == 3 ? (int)(yz / (uint32_t)g.S[1]) * g.sw + half : 0;
}

// k-space positions of the padded sector's indices, per axis:
// kp[a * KPS + i] == map_grid_to_kspace(i, G[a], center[a], off).
template <int DIM, int NT>
__device__ inline void fill_kpos(const Geom& g, const int* c3, float* kp, int KPS) {
  for (int e = threadIdx.x; e < DIM * KPS; e += NT) {
    const int d = e / KPS;
    const int i = e - d * KPS;
    kp[e] = map_grid_to_kspace(i, g.G[d], c3[d], g.off);
  }
}

// ---------------------------------------------------------------------------
// Tap records. Word 0 packs the first tap index per axis (bits 8a..8a+7) and
// a flag per axis (bit 24+a) set when the sample has kw+1 taps along it;
// word 1 + a*NX + t holds the weight of tap first+t on axis a, zero for taps
// the reference does not apply (beyond the sample's range, or failing the
// nearest-mode radius test, atomic_gpuNUFFT_kernels.cu:343-368).
// ---------------------------------------------------------------------------
template <int NX>
struct Rec {
  static constexpr int W = ((1 + 3 * NX) + 3) & ~3;  // words, float4 aligned
};

template <int DIM, int NX>
__device__ inline void make_record(const Geom& g, const float* lut, const float* kp, int KPS,
                                   const int* c3, const float* p, float* rec) {
  constexpr int RW = Rec<NX>::W;
  float w[RW];
#pragma unroll
  for (int q = 0; q < RW; q++) w[q] = 0.0f;
  uint32_t packed = 0;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    const float u = map_kspace_to_grid(p[d], g.G[d], c3[d], g.off);
    int lo, hi;
    tap_range(u, g.Pmax, g.kradius, &lo, &hi);
    packed |= (uint32_t)lo << (8 * d);
    if (hi - lo + 1 > g.kw) packed |= 1u << (24 + d);
#pragma unroll
    for (int t = 0; t < NX; t++) {
      float wt = 0.0f;
      if (lo + t <= hi && axis_weight_kp(g, lut, d, kp[d * KPS + lo + t], p[d], &wt))
        w[1 + d * NX + t] = wt;
    }
  }
  w[0] = __uint_as_float(packed);
  float4* r4 = reinterpret_cast<float4*>(rec);
#pragma unroll
  for (int q = 0; q < RW / 4; q++) r4[q] = make_float4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
}

template <int NX>
__device__ inline void load_record(const float* rec, float* w) {
  const float4* r4 = reinterpret_cast<const float4*>(rec);
#pragma unroll
  for (int q = 0; q < Rec<NX>::W / 4; q++) {
    const float4 v = r4[q];
    w[4 * q] = v.x;
    w[4 * q + 1] = v.y;
    w[4 * q + 2] = v.z;
    w[4 * q + 3] = v.w;
  }
}

// Wave-uniform number of taps along axis a: kw, or kw+1 when any active
// lane's sample has kw+1 taps there.
__device__ inline int wave_trip(uint32_t packed, int a, int kw) {
  return kw + (__ballot((packed >> (24 + a)) & 1u) != 0ull ? 1 : 0);
}

// Sample coordinate of sorted sample s (SoA [DIM][M]).
template <int DIM>
__device__ inline void load_coord(const float* crds, int M, uint32_t s, float* p) {
  p[0] = crds[s];
  p[1] = crds[(size_t)M + s];
  p[2] = DIM == 3 ? crds[2 * (size_t)M + s] : 0.0f;
}

// Shared-memory layout of the round-based interp (offsets in bytes from the
// dynamic LDS base; identical on host and device).
struct InterpLayout {
  int kpad, kpw, sub_n;
  size_t kp_off, sub_off, rec_off, bytes;
  __host__ __device__ InterpLayout(const Geom& g, int nx, int cb, int R) {
    const int P = g.P;
    const int PD = g.dim == 3 ? P * P * P : P * P;
    const int rw = ((1 + 3 * nx) + 3) & ~3;
    kpad = (g.K + 3) & ~3;
    kpw = (3 * (P + nx) + 3) & ~3;
    sub_n = PD * cb + nx * cb;  // + slack for the last row's window overrun
    kp_off = (size_t)kpad * 4;
    sub_off = kp_off + (size_t)kpw * 4;
    rec_off = sub_off + (size_t)((sub_n + 1) & ~1) * 8;
    bytes = rec_off + (size_t)R * rw * 4;
  }
};

// Copy n floats to LDS with U loads in flight per thread (a plain loop
// waits for each load before its LDS write).
template <int NT, int U>
__device__ inline void copy_to_lds(float* dst, const float* __restrict__ src, int n) {
  for (int i0 = threadIdx.x; i0 < n; i0 += U * NT) {
    float t[U];
#pragma unroll
    for (int u = 0; u < U; u++) t[u] = i0 + u * NT < n ? src[i0 + u * NT] : 0.0f;
#pragma unroll
    for (int u = 0; u < U; u++)
      if (i0 + u * NT < n) dst[i0 + u * NT] = t[u];
  }
}

// ---------------------------------------------------------------------------
// Lane kernels: LDS layout. Taps run KW per axis with no clamping. A window
// starts at most at Pmax-1 (the clamps of the reference's tap range), so the
// last of KW+1 taps is at most index P+1; the sub-grid has a slack of
// 2P^2+2P+2 words (3-D; 2P+2 in 2-D) past its end for such indices, whose
// taps carry weight zero (they lie past the reference's last tap).
// ---------------------------------------------------------------------------
struct LaneLayout {
  int kpad, kpw, sub_n;
  size_t kp_off, sub_off, bytes;
  // lut: the kernel table is copied to LDS (else read from global memory)
  __host__ __device__ LaneLayout(const Geom& g, int kw, int cb, bool lut = true) {
    const int P = g.P;
    const int PD = g.dim == 3 ? P * P * P : P * P;
    const int slack = g.dim == 3 ? 2 * P * P + 2 * P + 2 : 2 * P + 2;
    kpad = lut ? (g.K + 3) & ~3 : 0;
    kpw = (3 * (P + kw + 1) + 3) & ~3;
    sub_n = (PD + slack) * cb;
    kp_off = (size_t)kpad * 4;
    sub_off = (kp_off + (size_t)kpw * 4 + 15) & ~(size_t)15;
    bytes = sub_off + (size_t)((sub_n + 1) & ~1) * 8;
  }
};

// Value of lane `src` of this lane's quad, for each of the four lanes of the
// quad (DPP quad_perm: a VALU move, no LDS).
template <int A, int B, int C, int D>
__device__ inline uint32_t quad_get(uint32_t v) {
  if (A == 0 && B == 1 && C == 2 && D == 3) return v;
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, A | (B << 2) | (C << 4) | (D << 6), 0xF, 0xF, false);
}

// Source lane pattern of pass p: lane qi of a quad works on the sample owned
// by lane p * (4 / CB) + qi / CB, coil qi % CB.
template <int CB, int PS>
__device__ inline uint32_t quad_pass(uint32_t v) {
  constexpr int SPQ = 4 / CB;
  return quad_get<PS * SPQ + 0 / CB, PS * SPQ + 1 / CB, PS * SPQ + 2 / CB, PS * SPQ + 3 / CB>(v);
}

template <int CB>
__device__ inline uint32_t quad_pass_rt(uint32_t v, int ps) {
  // passes are unrolled; this maps the runtime index onto the compile-time
  // patterns
  switch (ps) {
    case 0: return quad_pass<CB, 0>(v);
    case 1: return CB > 1 ? quad_pass<CB, (CB > 1 ? 1 : 0)>(v) : v;
    case 2: return CB > 2 ? quad_pass<CB, (CB > 2 ? 2 : 0)>(v) : v;
    default: return CB > 3 ? quad_pass<CB, (CB > 3 ? 3 : 0)>(v) : v;
  }
}

// ---------------------------------------------------------------------------
// Interp
// ---------------------------------------------------------------------------
// Interp taps of one (sample, coil): ny x nz rows (wave-uniform trip
// counts) of TX words each, read in one batch per row (taps past the
// sample's range have weight 0; the row window stays inside the sub-grid
// and its zeroed slack). Weight ((wz*wy)*wx) as the reference forms it.
template <int DIM, int NX, int CB, int TX>
__device__ inline void interp_rows(const float2* sub, int P, int Pmax, int bx, int by, int bz, int ny,
                                   int nz, const float* w, int c, float* accx, float* accy) {
  float ax = 0.0f, ay = 0.0f;
#pragma unroll
  for (int tz = 0; tz < (DIM == 3 ? NX : 1); tz++) {
    if (tz >= nz) break;
    const int iz = DIM == 3 ? min(bz + tz, Pmax) : 0;
    const float wz = DIM == 3 ? w[1 + 2 * NX + tz] : 1.0f;
#pragma unroll
    for (int ty = 0; ty < NX; ty++) {
      if (ty >= ny) break;
      const int iy = min(by + ty, Pmax);
      const float wzy = DIM == 3 ? wz * w[1 + NX + ty] : w[1 + NX + ty];
      const float2* row = sub + ((iz * P + iy) * P + bx) * CB + c;
      float2 v[TX];
#pragma unroll
      for (int tx = 0; tx < TX; tx++) v[tx] = row[tx * CB];
#pragma unroll
      for (int tx = 0; tx < TX; tx++) {
        const float val = wzy * w[1 + tx];
        ax += v[tx].x * val;
        ay += v[tx].y * val;
      }
    }
  }
  *accx = ax;
  *accy = ay;
}

// interp_rows with T rows per axis known at compile time (no branch per
// row, so the LDS reads of every row can be in flight together). Callers
// use it when no lane of the wave has more than T taps on any axis; the
// same operations in the same order as interp_rows with those trips.
template <int DIM, int NX, int CB, int T>
__device__ inline void interp_rows_fixed(const float2* sub, int P, int Pmax, int bx, int by, int bz,
                                         const float* w, int c, float* accx, float* accy) {
  float ax = 0.0f, ay = 0.0f;
#pragma unroll
  for (int tz = 0; tz < (DIM == 3 ? T : 1); tz++) {
    const int iz = DIM == 3 ? min(bz + tz, Pmax) : 0;
    const float wz = DIM == 3 ? w[1 + 2 * NX + tz] : 1.0f;
#pragma unroll
    for (int ty = 0; ty < T; ty++) {
      const int iy = min(by + ty, Pmax);
      const float wzy = DIM == 3 ? wz * w[1 + NX + ty] : w[1 + NX + ty];
      const float2* row = sub + ((iz * P + iy) * P + bx) * CB + c;
      float2 v[T];
#pragma unroll
      for (int tx = 0; tx < T; tx++) v[tx] = row[tx * CB];
#pragma unroll
      for (int tx = 0; tx < T; tx++) {
        const float val = wzy * w[1 + tx];
        ax += v[tx].x * val;
        ay += v[tx].y * val;
      }
    }
  }
  *accx = ax;
  *accy = ay;
}

constexpr size_t kInterpStaticLds = 4096;  // interp's static shared tables, rounded up

template <int DIM, int NX, int CB, int NT = kThreads>
__device__ inline void interp_body(const Geom& g, const InterpArgs& a, uint32_t ci, int coil_block,
                                   int R) {
  constexpr int NW = NT / 64;
  constexpr int SPW = 64 / CB;  // sample slots per wave; one lane per (slot, coil)
  constexpr int RW = Rec<NX>::W;

  extern __shared__ float4 smem4[];
  char* smem = reinterpret_cast<char*>(smem4);
  const InterpLayout L(g, NX, CB, R);
  float* lut = reinterpret_cast<float*>(smem);
  float* kp = reinterpret_cast<float*>(smem + L.kp_off);
  float2* sub = reinterpret_cast<float2*>(smem + L.sub_off);
  float* rec = reinterpret_cast<float*>(smem + L.rec_off);
  const int P = g.P;
  const int Pmax = g.Pmax;
  const int KPS = P + NX;
  const int PD = DIM == 3 ? P * P * P : P * P;

  const Chunk ch = a.work.chunks[ci];
  const int n = (int)(ch.end - ch.begin);
  const int coil0 = coil_block * CB;
  const int tid = threadIdx.x;
  int c3[3];
  load_center<DIM>(g, ch.sector, c3);

  // grid offset of padded index i along axis d (periodic wrap, FORWARD
  // fftshift folded in): the padded point (x, y, z) reads grid element
  // gix[0][x] + gix[1][y] + gix[2][z]
  __shared__ int gix[3][256];
  // round 0's coordinates first: their loads overlap the table set-up
  // (p0 then carries each next round's coordinates, loaded a round ahead)
  float p0[3] = {0.0f, 0.0f, 0.0f};
  if (tid < min(R, n)) load_coord<DIM>(a.crds, g.M, ch.begin + tid, p0);
  copy_to_lds<NT, 4>(lut, a.lut, g.K);
  fill_kpos<DIM, NT>(g, c3, kp, KPS);
  for (int e = tid; e < DIM * P; e += NT) {
    const int d = e >= 2 * P ? 2 : (e >= P ? 1 : 0);
    const int i = e - d * P;
    const int q = c3[d] - g.off + i + (a.fold_shift ? g.shift_fwd[d] : 0);
    const int stride = d == 0 ? 1 : (d == 1 ? g.G[0] : g.G[0] * g.G[1]);
    gix[d][i] = wrap(q, g.G[d]) * stride;
  }
  if (DIM == 2 && tid == 0) gix[2][0] = 0;
  __syncthreads();
  if (tid < min(R, n)) make_record<DIM, NX>(g, lut, kp, KPS, c3, p0, rec + tid * RW);
  // Stage the padded sector, element e = pt*CB + coil (the coil of thread
  // tid is tid % CB in every iteration); zero the overrun slack. Four
  // loads per thread in flight before their LDS writes.
  {
    constexpr int U = 4;
    const int cc = tid % CB;
    const bool coil_in = coil0 + cc < a.n_coils;
    const float2* gbase = a.grid + (size_t)(coil_in ? coil0 + cc : 0) * g.Ng;
    for (int e0 = tid; e0 < L.sub_n; e0 += U * NT) {
      float2 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int pt = (e0 + u * NT) / CB;
        v[u] = make_float2(0.0f, 0.0f);
        if (pt < PD && coil_in) {
          const int yz = (int)udiv((uint32_t)pt, g.mP);
          const int x = pt - yz * P;
          const int z = DIM == 3 ? (int)udiv((uint32_t)pt, g.mP2) : 0;
          const int y = yz - z * P;
          v[u] = gbase[(uint32_t)(gix[0][x] + gix[1][y] + gix[2][z])];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (e0 + u * NT < L.sub_n) sub[e0 + u * NT] = v[u];
    }
  }

  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int slot = lane / CB;
  const int c = lane % CB;
  const int cg = coil0 + c;

  for (int r0 = 0; r0 < n; r0 += R) {
    const int rn = min(R, n - r0);
    if (r0 > 0) {
      __syncthreads();  // previous round consumed
      // sample tid of this round (R <= NT); its coordinates were loaded
      // during the previous round's taps
      if (tid < rn) make_record<DIM, NX>(g, lut, kp, KPS, c3, p0, rec + tid * RW);
    }
    __syncthreads();  // sub-grid staged, the round's records ready
    // the next round's coordinates, in flight during this round's taps
    if (r0 + R + tid < n) load_coord<DIM>(a.crds, g.M, ch.begin + r0 + R + tid, p0);

    // consecutive samples per wave step: the scattered stores of one wave
    // cover runs of neighbouring k-space samples
    for (int b = wave * SPW; b < rn; b += NW * SPW) {
      const int ls = b + slot;
      if (ls >= rn || cg >= a.n_coils) continue;
      float w[RW];
      load_record<NX>(rec + ls * RW, w);
      const uint32_t packed = __float_as_uint(w[0]);
      const int bx = (int)(packed & 255u);
      const int by = (int)((packed >> 8) & 255u);
      const int bz = (int)((packed >> 16) & 255u);
      const int ny = wave_trip(packed, 1, g.kw);
      const int nz = DIM == 3 ? wave_trip(packed, 2, g.kw) : 1;
      float accx = 0.0f, accy = 0.0f;
      // x taps: NX, or 3 when NX is 4 and no lane of the wave has a fourth
      // (wave-uniform; one branch per sample, the rows unrolled); at kernel
      // width 3 with three taps on every axis the rows run without a branch
      // per row (narrower kernels keep their shorter trips)
      // the store's density weight and destination, loaded before the taps
      // so that their latency overlaps them
      const uint32_t s = ch.begin + r0 + ls;
      const float dn = a.dens ? a.dens[s] : 1.0f;
      const uint32_t dst = a.scatter ? a.scatter[s] : s;
      const int nxw = wave_trip(packed, 0, g.kw);
      if (NX == 4 && g.kw == 3 && nxw <= 3 && ny <= 3 && nz <= 3)
        interp_rows_fixed<DIM, NX, CB, 3>(sub, P, Pmax, bx, by, bz, w, c, &accx, &accy);
      else if (NX == 4 && nxw <= 3)
        interp_rows<DIM, NX, CB, (NX == 4 ? 3 : NX)>(sub, P, Pmax, bx, by, bz, ny, nz, w, c, &accx, &accy);
      else
        interp_rows<DIM, NX, CB, NX>(sub, P, Pmax, bx, by, bz, ny, nz, w, c, &accx, &accy);
      float rx = accx * a.scale, ry = accy * a.scale;
      if (a.dens) {
        const float sq = sqrtf(dn);
        rx = rx * sq;
        ry = ry * sq;
      }
      a.out[(size_t)cg * a.coil_stride + dst] = make_float2(rx, ry);
    }
  }
}

template <int DIM, int NX, int CB>
__global__ void __launch_bounds__(kThreads) interp_kernel(Geom g, InterpArgs a, int R) {
  const uint32_t ci = work_chunk(a.work, blockIdx.x);
  if (ci == ~0u) return;
  interp_body<DIM, NX, CB>(g, a, ci, blockIdx.y, R);
}

// ---------------------------------------------------------------------------
// Interp with tap records in registers (kernel width KW = 3): every thread
// forms the record of the samples it owns (sample j = round * NT + tid), the lanes of a quad share them with DPP moves, and each lane sums
// the KW^d taps of one (sample, coil) from the staged padded sector. The
// samples of a quad are consecutive (the scattered output stores of a wave
// cover runs of neighbouring samples). No LDS round trip of records and one
// barrier after the staging.
// ---------------------------------------------------------------------------
template <int DIM, int T, int CB>
__device__ inline void lane_gather(const float2* sub, int P, const int* b, const float (*w)[4],
                                   int cc, float* ax, float* ay) {
  const float2* base = sub + ((b[2] * P + b[1]) * P + b[0]) * CB + cc;
  float sx = 0.0f, sy = 0.0f;
#pragma unroll
  for (int tz = 0; tz < (DIM == 3 ? T : 1); tz++) {
    const float wz = DIM == 3 ? w[2][tz] : 1.0f;
#pragma unroll
    for (int ty = 0; ty < T; ty++) {
      const float wzy = DIM == 3 ? wz * w[1][ty] : w[1][ty];
      const float2* row = base + (tz * P + ty) * P * CB;
      float2 v[T];
#pragma unroll
      for (int tx = 0; tx < T; tx++) v[tx] = row[tx * CB];
#pragma unroll
      for (int tx = 0; tx < T; tx++) {
        const float val = wzy * w[0][tx];
        sx += v[tx].x * val;
        sy += v[tx].y * val;
      }
    }
  }
  *ax = sx;
  *ay = sy;
}

// LUTG: kernel table read from global memory (cached) instead of an LDS
// copy, for small workgroups whose few samples make fewer lookups than the
// copy has words.
template <int DIM, int KW, int CB, int NT = kThreads, bool LUTG = false>
__device__ inline void interp_lane_body(const Geom& g, const InterpArgs& a, uint32_t ci,
                                        int coil_block) {
  constexpr int NX = KW + 1;
  constexpr int RND = 2;
  constexpr int PASSES = CB;
  static_assert(CB == 1 || CB == 2 || CB == 4, "a sample's coils share one quad");

  extern __shared__ float4 smem4[];
  char* smem = reinterpret_cast<char*>(smem4);
  const LaneLayout L(g, KW, CB, !LUTG);
  float* lut = reinterpret_cast<float*>(smem);
  float* kp = reinterpret_cast<float*>(smem + L.kp_off);
  float2* sub = reinterpret_cast<float2*>(smem + L.sub_off);
  const int P = g.P;
  const int Pmax = g.Pmax;
  const int KPS = P + NX;
  const int PD = DIM == 3 ? P * P * P : P * P;

  const Chunk ch = a.work.chunks[ci];
  const int n = (int)(ch.end - ch.begin);
  const int coil0 = coil_block * CB;
  const int tid = threadIdx.x;
  const int qc = (tid & 3) % CB;
  const bool coil_ok = coil0 + qc < a.n_coils;
  int c3[3];
  load_center<DIM>(g, ch.sector, c3);

  // owned samples: j = r * NT + tid (a quad owns four consecutive samples)
  float p[RND][3];
  bool live[RND];
#pragma unroll
  for (int r = 0; r < RND; r++) {
    const int j = r * NT + tid;
    live[r] = j < n;
    p[r][0] = p[r][1] = p[r][2] = 0.0f;
    if (live[r]) load_coord<DIM>(a.crds, g.M, ch.begin + (uint32_t)j, p[r]);
  }

  if (!LUTG) copy_to_lds<NT, 4>(lut, a.lut, g.K);
  const float* wlut = LUTG ? a.lut : lut;
  fill_kpos<DIM, NT>(g, c3, kp, KPS);
  // Stage the padded sector as [point][coil] (periodic wrap and the FORWARD
  // fftshift folded into the grid index), zeros in the slack past it (its
  // words meet only zero weights, but must not hold NaNs). Four loads per
  // thread in flight before their LDS writes.
  {
    constexpr int U = 4;
    const int cc = tid % CB;
    const bool cin = coil0 + cc < a.n_coils;
    const float2* gbase = a.grid + (size_t)(cin ? coil0 + cc : 0) * g.Ng;
    int q0[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
      q0[d] = d < DIM ? c3[d] - g.off + (a.fold_shift ? g.shift_fwd[d] : 0) : 0;
    for (int e0 = tid; e0 < L.sub_n; e0 += U * NT) {
      float2 v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int pt = (e0 + u * NT) / CB;
        v[u] = make_float2(0.0f, 0.0f);
        if (pt < PD && cin) {
          const int yz = (int)udiv((uint32_t)pt, g.mP);
          const int x = pt - yz * P;
          const int z = DIM == 3 ? (int)udiv((uint32_t)pt, g.mP2) : 0;
          const int y = yz - z * P;
          const int gx = wrap(q0[0] + x, g.G[0]);
          const int gy = wrap(q0[1] + y, g.G[1]);
          const int gz = DIM == 3 ? wrap(q0[2] + z, g.G[2]) : 0;
          v[u] = gbase[(size_t)gx + (size_t)g.G[0] * ((size_t)gy + (size_t)g.G[1] * gz)];
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (e0 + u * NT < L.sub_n) sub[e0 + u * NT] = v[u];
    }
  }
  __syncthreads();

#pragma unroll
  for (int r = 0; r < RND; r++) {
    if (r * NT >= n) break;  // workgroup-uniform
    if (r * NT + (tid & ~63) >= n) continue;  // wave-uniform: this wave owns none
    uint32_t bp = 0;
    float w[3][4];
#pragma unroll
    for (int d = 0; d < 3; d++)
#pragma unroll
      for (int t = 0; t < 4; t++) w[d][t] = 0.0f;
    bool wide = false;
    if (live[r]) {
#pragma unroll
      for (int d = 0; d < DIM; d++) {
        const float u = map_kspace_to_grid(p[r][d], g.G[d], c3[d], g.off);
        int lo, hi;
        tap_range(u, Pmax, g.kradius, &lo, &hi);
        bp |= (uint32_t)lo << (8 * d);
        wide = wide || hi - lo + 1 > KW;
#pragma unroll
        for (int t = 0; t < NX; t++) {
          float wt = 0.0f;
          if (lo + t <= hi && axis_weight_kp(g, wlut, d, kp[d * KPS + lo + t], p[r][d], &wt))
            w[d][t] = wt;
        }
      }
    }
    const bool any_wide = __ballot(wide) != 0ull;
    const uint32_t lv = live[r] ? 1u : 0u;
#pragma unroll
    for (int ps = 0; ps < PASSES; ps++) {
      const uint32_t bo = quad_pass_rt<CB>(bp, ps);
      const bool lo_live = quad_pass_rt<CB>(lv, ps) != 0u;
      float wo[3][4];
#pragma unroll
      for (int d = 0; d < 3; d++)
#pragma unroll
        for (int t = 0; t < 4; t++)
          wo[d][t] = (d < DIM && t < (any_wide ? NX : KW))
                         ? __uint_as_float(quad_pass_rt<CB>(__float_as_uint(w[d][t]), ps))
                         : 0.0f;
      // the worked sample: owner lane (tid & ~3) + ps * (4 / CB) + qi / CB
      const int jo = r * NT + (tid & ~3) + ps * (4 / CB) + (tid & 3) / CB;
      if (!lo_live || !coil_ok) continue;
      const int b[3] = {(int)(bo & 255u), (int)((bo >> 8) & 255u), (int)((bo >> 16) & 255u)};
      // the store's density weight and destination, loaded before the taps
      const uint32_t s = ch.begin + (uint32_t)jo;
      const float dn = a.dens ? a.dens[s] : 1.0f;
      const uint32_t dst = a.scatter ? a.scatter[s] : s;
      float ax, ay;
      if (any_wide)
        lane_gather<DIM, NX, CB>(sub, P, b, wo, qc, &ax, &ay);
      else
        lane_gather<DIM, KW, CB>(sub, P, b, wo, qc, &ax, &ay);
      float rx = ax * a.scale, ry = ay * a.scale;
      if (a.dens) {
        const float sq = sqrtf(dn);
        rx = rx * sq;
        ry = ry * sq;
      }
      a.out[(size_t)(coil0 + qc) * a.coil_stride + dst] = make_float2(rx, ry);
    }
  }
}

template <int DIM, int KW, int CB>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(6))) interp_lane_kernel(Geom g, InterpArgs a) {
  const uint32_t ci = work_chunk(a.work, blockIdx.x);
  if (ci == ~0u) return;
  interp_lane_body<DIM, KW, CB>(g, a, ci, blockIdx.y);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// Dynamic LDS a workgroup may use on the current device (160 KB per CU on
// gfx950; queried, since launches above 64 KB need the device to allow it).
static size_t lds_limit() {
  static size_t limit = 0;
  if (limit == 0) {
    int dev = 0, v = 0;
    size_t l = 64 * 1024;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
        v > 0)
      l = (size_t)v;
    limit = l;
  }
  return limit;
}

template <typename K>
static hipError_t allow_lds(K kernel, size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

static int nx_of(const Geom& g) { return g.kw + 1 <= 4 ? 4 : 8; }

// Samples per round: as many as fit next to the sub-grid (budget `limit`),
// at most one per thread of a `threads`-thread workgroup and at most the
// chunk; multiple of 16.
template <typename Layout>
static int round_size(const Geom& g, int cb, int chunk, size_t limit, int threads = kThreads) {
  const int nx = nx_of(g);
  const size_t fixed = Layout(g, nx, cb, 0).bytes;
  const size_t per = Layout(g, nx, cb, 1).bytes - fixed;
  if (fixed + 16 * per > limit) return 0;
  size_t r = (limit - fixed) / per;
  r = r > (size_t)threads ? (size_t)threads : r;
  r &= ~(size_t)15;
  const int want = (chunk + 15) & ~15;
  return (int)r < want ? (int)r : want;
}

// Largest coil block (<= max_cb, not above the coil count) whose round size
// is at least min(64, chunk) samples.
template <typename Layout>
static int pick_cb(const Geom& g, int n_coils, int max_cb, int chunk, size_t limit, int* R) {
  const int need = chunk < 64 ? chunk : 64;
  for (int cb = max_cb; cb >= 1; cb /= 2) {
    if (cb > 1 && cb / 2 >= n_coils) continue;
    const int r = round_size<Layout>(g, cb, chunk, limit);
    if (r >= need || (cb == 1 && r > 0)) {
      *R = r;
      return cb;
    }
  }
  *R = 0;
  return 0;
}

template <int DIM, int NX, int CB>
static hipError_t interp_launch(const Geom& g, const InterpArgs& a, int R, hipStream_t s) {
  const uint32_t n_blocks = work_blocks(a.work);
  const int coil_blocks = (a.n_coils + CB - 1) / CB;
  const size_t lds = InterpLayout(g, NX, CB, R).bytes;
  hipError_t e = allow_lds(interp_kernel<DIM, NX, CB>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((interp_kernel<DIM, NX, CB>), dim3(n_blocks, coil_blocks), dim3(kThreads), lds,
                     s, g, a, R);
  return hipGetLastError();
}

// Lane interp: 2-D only by default (at 128^3 osf 1.5 the 3-D lane interp
// takes 0.81 ms against 0.65 ms for the round-based kernel; 2-D batches are
// faster with it). GNUFFT_INTERP=round / =lane override, for tuning.
static bool lane_interp_ok(const Geom& g, int chunk) {
  static int mode = -1;
  if (mode < 0) {
    const char* e = getenv("GNUFFT_INTERP");
    mode = e && strcmp(e, "round") == 0 ? 0 : (e && strcmp(e, "lane") == 0 ? 2 : 1);
  }
  const bool shape_ok = g.kw == 3 && g.P >= 4 && chunk <= 2 * kThreads;
  return shape_ok && (mode == 2 || (mode == 1 && g.dim == 2));
}

// Largest coil block (not above the coil count) whose footprint lets
// `per_cu` workgroups share a CU; 0 if none.
static int lane_cb(const Geom& g, int n_coils, int per_cu) {
  const size_t limit = lds_limit() / (size_t)per_cu - 1024;
  for (int cb = 4; cb >= 1; cb /= 2) {
    if (cb > 1 && cb / 2 >= n_coils) continue;
    if (LaneLayout(g, 3, cb).bytes <= limit) return cb;
  }
  return 0;
}

// Workgroups per CU the lane kernels' coil block is sized for (default 3:
// at 128^3 osf 1.5 three workgroups of 4 coils take the spread kernel
// 1.25 -> 0.72 ms against four of 2; GNUFFT_LANE_PER_CU overrides, for
// tuning).
static int lane_per_cu() {
  static int v = 0;
  if (v == 0) {
    const char* e = getenv("GNUFFT_LANE_PER_CU");
    v = e ? atoi(e) : 3;
    if (v < 1 || v > 8) v = 3;
  }
  return v;
}

template <int DIM, int NX>
static hipError_t interp_nx(const Geom& g, const InterpArgs& a, int chunk, hipStream_t s) {
  // Prefer a footprint that lets two workgroups share a CU.
  int R = 0;
  // three workgroups per CU if they fit, then two, then
  // one; room for the static tables (grid offsets, 3 KB) beside the
  // dynamic LDS
  int cb = pick_cb<InterpLayout>(g, a.n_coils, 8, chunk, lds_limit() / 3 - kInterpStaticLds, &R);
  if (cb == 0) cb = pick_cb<InterpLayout>(g, a.n_coils, 8, chunk, lds_limit() / 2 - kInterpStaticLds, &R);
  if (cb == 0) cb = pick_cb<InterpLayout>(g, a.n_coils, 8, chunk, lds_limit() - kInterpStaticLds, &R);
  switch (cb) {
    case 8: return interp_launch<DIM, NX, 8>(g, a, R, s);
    case 4: return interp_launch<DIM, NX, 4>(g, a, R, s);
    case 2: return interp_launch<DIM, NX, 2>(g, a, R, s);
    case 1: return interp_launch<DIM, NX, 1>(g, a, R, s);
    default: return hipErrorInvalidValue;
  }
}

// Room in LDS for the padded sector of `cb` coils beside a round of 16
// samples (kernel width 3 by itself: the lane layout, one coil): plans whose
// sectors are larger are refused, adjoint and forward alike.
bool padded_sector_fits(const Geom& g, int cb) {
  return InterpLayout(g, nx_of(g), cb, 16).bytes + 16 * (size_t)cb * sizeof(float2) <=
         lds_limit() - 1024;
}

bool spread_supported(const Geom& g) {
  if (g.kw > 7 || g.P > 255) return false;
  if (g.kw == 3 && g.P >= 4) return LaneLayout(g, 3, 1).bytes <= lds_limit() - 1024;
  return padded_sector_fits(g, 1);
}

template <int DIM, int CB>
static hipError_t interp_lane_launch(const Geom& g, const InterpArgs& a, hipStream_t s) {
  const uint32_t n_blocks = work_blocks(a.work);
  const int coil_blocks = (a.n_coils + CB - 1) / CB;
  const size_t lds = LaneLayout(g, 3, CB).bytes;
  hipError_t e = allow_lds(interp_lane_kernel<DIM, 3, CB>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((interp_lane_kernel<DIM, 3, CB>), dim3(n_blocks, coil_blocks), dim3(kThreads),
                     lds, s, g, a);
  return hipGetLastError();
}

template <int DIM>
static hipError_t interp_lane(const Geom& g, const InterpArgs& a, hipStream_t s) {
  int cb = 0;
  const int first = a.lane_per_cu > 0 ? a.lane_per_cu : lane_per_cu();
  for (int per = first; per >= 1 && cb == 0; per--) cb = lane_cb(g, a.n_coils, per);
  switch (cb) {
    case 4: return interp_lane_launch<DIM, 4>(g, a, s);
    case 2: return interp_lane_launch<DIM, 2>(g, a, s);
    case 1: return interp_lane_launch<DIM, 1>(g, a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_interp(const Geom& g, const InterpArgs& a, int chunk, hipStream_t s) {
  if (a.work.n_chunks == 0 || a.n_coils == 0) return hipSuccess;
  if (g.kw > 7 || g.P > 255) return hipErrorInvalidValue;
  if (lane_interp_ok(g, chunk)) return g.dim == 3 ? interp_lane<3>(g, a, s) : interp_lane<2>(g, a, s);
  InterpArgs b = a;
  if (a.work_runs.n_chunks > 0) b.work = a.work_runs;
  if (g.dim == 3) return nx_of(g) == 4 ? interp_nx<3, 4>(g, b, chunk, s) : interp_nx<3, 8>(g, b, chunk, s);
  return nx_of(g) == 4 ? interp_nx<2, 4>(g, b, chunk, s) : interp_nx<2, 8>(g, b, chunk, s);
}

// ---------------------------------------------------------------------------
// Batched launches: one launch per stage for a batch of operators
// ---------------------------------------------------------------------------
// Batch rounds are sized for kBatchPerCU workgroups of kBatchThreads per CU
// (eight waves per SIMD).
template <int DIM, int NX>
__global__ void __launch_bounds__(kBatchThreads) interp_batch_kernel(const BatchOp* __restrict__ ops,
                                                                     BatchList l) {
  uint4 it;
  if (!batch_item(l, blockIdx.x, &it)) return;
  const BatchOp& op = ops[it.x];
  interp_body<DIM, NX, kBatchCB, kBatchThreads>(op.g, op.i, it.y, (int)it.z, op.R_interp);
}

size_t lds_budget() { return lds_limit(); }

size_t interp_lds_bytes(const Geom& g, int cb, int R) {
  return InterpLayout(g, nx_of(g), cb, R).bytes;
}

int interp_round(const Geom& g, int cb, int chunk, size_t limit) {
  return round_size<InterpLayout>(g, cb, chunk, limit, kBatchThreads);
}

template <typename K>
static hipError_t launch_items(K kernel, const BatchOp* ops, const BatchList& l, int threads,
                               size_t lds, hipStream_t s) {
  if (l.n == 0) return hipSuccess;
  hipError_t e = allow_lds(kernel, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(batch_blocks(l)), dim3(threads), lds, s, ops, l);
  return hipGetLastError();
}

// Batched lane kernels (kernel width 3 in every plan): coil blocks of
// kBatchLaneCB, one sample's coils per quad.
template <int DIM>
__global__ void __launch_bounds__(kBatchThreads) __attribute__((amdgpu_waves_per_eu(6)))
    interp_batch_lane_kernel(const BatchOp* __restrict__ ops, BatchList l) {
  uint4 it;
  if (!batch_item(l, blockIdx.x, &it)) return;
  const BatchOp& op = ops[it.x];
  interp_lane_body<DIM, 3, kBatchLaneCB, kBatchThreads>(op.g, op.i, it.y, (int)it.z);
}

template <int DIM>
__global__ void __launch_bounds__(kBatchSmallThreads) __attribute__((amdgpu_waves_per_eu(6)))
    interp_batch_lane_small_kernel(const BatchOp* __restrict__ ops, BatchList l) {
  uint4 it;
  if (!batch_item(l, blockIdx.x, &it)) return;
  const BatchOp& op = ops[it.x];
  interp_lane_body<DIM, 3, kBatchLaneCB, kBatchSmallThreads, true>(op.g, op.i, it.y, (int)it.z);
}

hipError_t launch_interp_batch_small(int dim, const BatchOp* ops, const BatchList& l, size_t lds,
                                     hipStream_t s) {
  return dim == 3 ? launch_items(interp_batch_lane_small_kernel<3>, ops, l, kBatchSmallThreads, lds, s)
                  : launch_items(interp_batch_lane_small_kernel<2>, ops, l, kBatchSmallThreads, lds, s);
}

bool lane_batch_ok(const Geom& g) {
  return lane_interp_ok(g, 2 * kBatchThreads);
}

size_t lane_lds_bytes(const Geom& g, int cb, bool lut) { return LaneLayout(g, 3, cb, lut).bytes; }

hipError_t launch_interp_batch(int dim, int nx, const BatchOp* ops, const BatchList& l,
                               size_t lds, hipStream_t s) {
  if (nx == 3)
    return dim == 3 ? launch_items(interp_batch_lane_kernel<3>, ops, l, kBatchThreads, lds, s)
                    : launch_items(interp_batch_lane_kernel<2>, ops, l, kBatchThreads, lds, s);
  if (dim == 3)
    return nx == 4 ? launch_items(interp_batch_kernel<3, 4>, ops, l, kBatchThreads, lds, s)
                   : launch_items(interp_batch_kernel<3, 8>, ops, l, kBatchThreads, lds, s);
  return nx == 4 ? launch_items(interp_batch_kernel<2, 4>, ops, l, kBatchThreads, lds, s)
                 : launch_items(interp_batch_kernel<2, 8>, ops, l, kBatchThreads, lds, s);
}


}  // namespace gnufft
