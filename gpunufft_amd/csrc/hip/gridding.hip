// Kaiser-Bessel interpolation for CDNA4 (gfx950); the adjoint's spread is in
// spread.hip.
//
// interp (forward convolution, reference CUDA/src/gpu/atomic/
//   atomic_gpuNUFFT_kernels.cu:966-1400, texture_gpuNUFFT_kernels.cu:467-1039)
//
// One workgroup per (sector chunk, group of NC coils). A chunk is a contiguous
// run of sorted samples of one sector, so heavy sectors near the k-space
// centre spread over many workgroups. Workgroup ids are remapped so that each
// of the 8 XCDs owns a contiguous range of chunks (neighbouring sectors share
// that XCD's L2).
//
// The padded sector is staged in LDS as [point][coil], two points in x per
// load; the taps of the first samples are loaded from the plan's tap table
// meanwhile. Then every wave takes 64 / LP samples at a time, LP lanes of two
// coils each: a tap is one 16-byte LDS read per lane, the lanes of a sample
// read its 8 * NC bytes in a row, and the next samples' taps are in flight. The
// sums change lanes before the store (ds_bpermute), so that a store
// instruction writes runs of one coil's samples (neighbours of a sorted list
// are mostly neighbours on their trajectory).
//
// Bound: workgroups are short (a sector of a sparse 3-D trajectory holds some
// 30 samples) and mostly wait for a chain of loads (chunk, grid points, LDS,
// stores), so what counts is how many of them a CU holds: 64 registers and no
// LDS beside the sector. At 128^3 osf 1.5 the 268 MB of scattered results cost
// 0.14 of 0.45 ms, the staging 0.10 ms, the taps' reads nothing measurable.
// Against tap records formed in LDS per round of samples (3-D) or in registers
// (2-D): 0.58 -> 0.45 ms (128^3 koosh, 8 coils), 1.14 -> 0.76 ms (160^3 osf 2,
// 2.0 M samples, 8 coils), 0.30 -> 0.15 ms (168 x 160 x 44 stack, 6 coils),
// 66 -> 26 us (256^2 osf 2, 16 coils), 143 -> 17 us (224^2 kernel width 5,
// 12 coils), 5.3 -> 4.4 us (64^2, 1 coil).
// Eight staging loads in flight instead of four take 90 registers: 26 -> 30 us at
// 256^2.

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "gnufft_internal.hpp"

namespace gnufft {

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
  // Cost of a chunk: its samples plus a fixed share for staging the padded
  // sector (about 300 samples' worth on gfx950).
  std::vector<uint32_t> cost(n);
  for (uint32_t i = 0; i < n; i++) cost[i] = counts[i] + 300u;
  split_ranges(cost.data(), n, w->xcd_begin, &w->max_range);
  w->n_chunks = n;
}

void partition_items(const uint32_t* costs, uint32_t n, BatchList* l) {
  split_ranges(costs, n, l->xcd_begin, &l->max_range);
  l->n = n;
}

// ---------------------------------------------------------------------------
// Interp
// ---------------------------------------------------------------------------
// T: taps per axis read by a kernel; FULL: the kernel width is T, else
// the taps past it (weight zero) are left out on y and z.
template <int NC>
struct CoilLanes {
  static constexpr int CL = NC > 1 ? 2 : 1;  // coils per lane
  static constexpr int LP = NC / CL;         // lanes per sample
  static constexpr int SPW = 64 / LP;        // samples per wave and pass
};

// LDS: the padded sector and T - 1 points that the last row's taps may run
// into (zeros: their weights are zero), NC coils each.
static inline size_t interp_lds(const Geom& g, int nc, int t) {
  const size_t pd = (size_t)g.P * g.P * (g.dim == 3 ? g.P : 1);
  return (pd + t - 1) * nc * sizeof(float2);
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(8)));  // two complex values

// The padded sector at grid point q0 (in [0, G)) -> sub [point][coil]. Threads:
// (pair of points in x, 2^row_bits of them; coil; row), so that one instruction
// fetches whole rows (instructions on one cache line wait for each other while
// it is pending) and only the row changes from load to load.
template <int DIM, int NC, bool ONE_ROW>
__device__ __forceinline__ void stage_sector(const Geom& g, const InterpArgs& a, int coil0, const int* q0, int rows,
                                             bool small, float2* sub) {
  const int P = g.P;
  auto on_grid = [&](int i, int G) {  // i < G + P
    i -= i >= G ? G : 0;
    return small ? wrap(i, G) : i;
  };
  const int tid = threadIdx.x;
  const int x = 2 * (tid & ((1 << a.row_bits) - 1));
  const int cc = (tid >> a.row_bits) % NC;
  const bool live = x < P && coil0 + cc < a.n_coils, second = x + 1 < P;
  const int gx = x < P ? on_grid(q0[0] + x, g.G[0]) : 0, gx1 = second ? on_grid(gx + 1, g.G[0]) : 0;
  const bool pair = second && gx1 == gx + 1;
  const float2* gbase = a.grid + (size_t)(live ? coil0 + cc : 0) * g.Ng;
  int row = (tid >> a.row_bits) / NC;
  if (ONE_ROW) row = __builtin_amdgcn_readfirstlane(row);
  const int step = ((int)blockDim.x >> a.row_bits) / NC;
  int z = DIM == 3 ? row / P : 0, y = row - z * P;
  const int dz = DIM == 3 ? step / P : 0, dy = step - dz * P;
  constexpr int U = 4;
  while (row < rows) {
    f32x4 v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      v[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (row + u * step < rows) {
        const size_t yz = (size_t)on_grid(q0[1] + y, g.G[1]) +
                          (DIM == 3 ? (size_t)g.G[1] * on_grid(q0[DIM - 1] + z, g.G[2]) : 0);
        const float2* src = gbase + (size_t)g.G[0] * yz;
        if (live) {
          if (pair) {
            v[u] = *reinterpret_cast<const f32x4u*>(src + gx);
          } else {
            const float2 p = src[gx];
            v[u].x = p.x, v[u].y = p.y;
            if (second) {
              const float2 q = src[gx1];
              v[u].z = q.x, v[u].w = q.y;
            }
          }
        }
      }
      y += dy;
      z += dz;
      if (DIM == 3 && y >= P) y -= P, z++;
    }
    if (x < P) {
#pragma unroll
      for (int u = 0; u < U; u++)
        if (row + u * step < rows) {
          float2* to = sub + ((row + u * step) * P + x) * NC + cc;
          to[0] = make_float2(v[u].x, v[u].y);
          if (second) to[NC] = make_float2(v[u].z, v[u].w);
        }
    }
    row += U * step;
  }
}

template <int DIM, int NC, int T, bool FULL>
__device__ __forceinline__ void interp_body(const Geom& g, const InterpArgs& a, uint32_t ci, int group) {
  using C = CoilLanes<NC>;
  using V = std::conditional_t<C::CL == 2, f32x4, f32x2>;       // a lane's coils
  constexpr int NV = T == 3 ? 1 : 2;                            // float4 per tap table entry
  extern __shared__ float4 smem4[];
  float2* sub = reinterpret_cast<float2*>(smem4);
  const int P = g.P;
  const int PP = P * P;
  const Chunk ch = a.work.chunks[ci];
  const int coil0 = group * NC;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63;
  const uint32_t step = (uint32_t)(nt >> 6) * C::SPW;

  // first grid index of the padded sector (in [0, G); the standard centre
  // index * sw + sw / 2 per axis)
  int o3[3];
  {
    const uint32_t x = ch.sector % (uint32_t)g.S[0], yz = ch.sector / (uint32_t)g.S[0];
    const int first = g.sw / 2 - g.off;
    o3[0] = wrap((int)x * g.sw + first, g.G[0]);
    o3[1] = wrap((int)(yz % (uint32_t)g.S[1]) * g.sw + first, g.G[1]);
    o3[2] = DIM == 3 ? wrap((int)(yz / (uint32_t)g.S[1]) * g.sw + first, g.G[2]) : 0;
  }

  // Samples of this lane: `slot` of the pass whose taps it sums (coils 2 * part
  // ..), `out` of the pass whose result it stores (coils 2 * out_part ..).
  const int slot = lane / C::LP, part = lane % C::LP;
  const int out = lane % C::SPW, out_part = lane / C::SPW;
  uint32_t base = ch.begin + (uint32_t)(tid >> 6) * C::SPW;
  const uint32_t last = ch.end - 1;
  uint32_t js = 0, jo = 0;
  float4 tap[DIM][NV];
  auto load_index = [&](uint32_t b) {
    js = a.idx[min(b + slot, last)];
    if (C::LP > 1) jo = a.idx[min(b + out, last)];
    else jo = js;
  };
  auto load_taps = [&] {
#pragma unroll
    for (int d = 0; d < DIM; d++)
#pragma unroll
      for (int q = 0; q < NV; q++) tap[d][q] = a.taps[((size_t)d * g.M + js) * NV + q];
  };
  uint32_t jo_now = 0;
  if (base <= last) {
    load_index(base);
    load_taps();
    jo_now = jo;
    load_index(base + step);
  }

  // Stage the padded sector (periodic wrap, FORWARD fftshift folded in).
  const int rows = DIM == 3 ? PP : P;
  const bool small = P > g.G[0] || P > g.G[1] || (DIM == 3 && P > g.G[2]);
  int q0[3];
#pragma unroll
  for (int d = 0; d < DIM; d++) q0[d] = wrap(o3[d] + (a.fold_shift ? g.shift_fwd[d] : 0), g.G[d]);
  if (NC << a.row_bits >= 64)  // a wave is inside one row: its address in scalar registers
    stage_sector<DIM, NC, true>(g, a, coil0, q0, rows, small, sub);
  else
    stage_sector<DIM, NC, false>(g, a, coil0, q0, rows, small, sub);
  {
    const int pd = rows * P;
    for (int e = tid; e < (T - 1) * NC; e += nt) sub[pd * NC + e] = make_float2(0.f, 0.f);
  }
  __syncthreads();

  const V* mine = reinterpret_cast<const V*>(sub) + part;
  // (kernel width 1: a sample past the sector's last point keeps its tap second,
  // the reference's clamp of the first)
  const int kw = FULL ? T : g.kw == 1 ? 2 : g.kw;
  for (; base < ch.end; base += step) {
    // this pass's taps to scalars; the next one's on their way
    float w[DIM][T];
    int first[DIM];
#pragma unroll
    for (int d = 0; d < DIM; d++) {
      const int q = __float_as_int(tap[d][0].x) - o3[d];
      first[d] = min(q < 0 ? q + g.G[d] : q, P - 1);
      w[d][0] = tap[d][0].y, w[d][1] = tap[d][0].z, w[d][2] = tap[d][0].w;
      if constexpr (T > 3) w[d][3] = tap[d][NV - 1].x, w[d][4] = tap[d][NV - 1].y;
      if constexpr (T > 5) w[d][5] = tap[d][NV - 1].z, w[d][6] = tap[d][NV - 1].w;
    }
    const uint32_t j = jo_now;
    const float sq = a.dens ? a.dens[j] : 1.0f;
    if (base + step < ch.end) {
      load_taps();
      jo_now = jo;
      load_index(base + 2 * step);
    }
    float r[2 * C::CL];
#pragma unroll
    for (int q = 0; q < 2 * C::CL; q++) r[q] = 0.0f;
#pragma unroll
    for (int tz = 0; tz < (DIM == 3 ? T : 1); tz++) {
      if (DIM == 3 && tz >= kw) break;
      const int iz = DIM == 3 ? min(first[DIM - 1] + tz, P - 1) * PP : 0;
#pragma unroll
      for (int ty = 0; ty < T; ty++) {
        if (ty >= kw) break;
        const int iy = min(first[1] + ty, P - 1) * P;
        const float wzy = DIM == 3 ? w[DIM - 1][tz] * w[1][ty] : w[1][ty];
        const V* row = mine + (iz + iy + first[0]) * C::LP;
        V v[T];
#pragma unroll
        for (int tx = 0; tx < T; tx++) v[tx] = row[tx * C::LP];
#pragma unroll
        for (int tx = 0; tx < T; tx++) {
          const float val = wzy * w[0][tx];
#pragma unroll
          for (int q = 0; q < 2 * C::CL; q++) r[q] += v[tx][q] * val;
        }
        // the sums stay here: moved to the end, they would keep every tap's
        // value in a register
        if (DIM == 2 ? ty == T - 1 : T > 3 || ty == 2)
#pragma unroll
          for (int q = 0; q < 2 * C::CL; q++) asm volatile("" : "+v"(r[q]));
      }
    }
#pragma unroll
    for (int q = 0; q < 2 * C::CL; q++) {
      const float s = r[q] * a.scale;
      r[q] = C::LP > 1 ? __int_as_float(__builtin_amdgcn_ds_bpermute(4 * (out * C::LP + out_part), __float_as_int(s)))
                       : s;
      if (a.dens) r[q] *= sq;
    }
    if (base + out < ch.end) {
      const size_t dst = a.sorted_out ? base + out : j;
#pragma unroll
      for (int q = 0; q < C::CL; q++) {
        const int c = coil0 + C::CL * out_part + q;
        if (c < a.n_coils) a.out[(size_t)c * a.coil_stride + dst] = make_float2(r[2 * q], r[2 * q + 1]);
      }
    }
  }
}

template <int DIM, int NC, int T, bool FULL>
__global__ void __launch_bounds__(1024) interp_kernel(Geom g, InterpArgs a) {
  const uint32_t ci = work_chunk(a.work, blockIdx.x);
  if (ci == ~0u) return;
  interp_body<DIM, NC, T, FULL>(g, a, ci, blockIdx.y);
}

template <int DIM, int NC, int T, bool FULL>
__global__ void __launch_bounds__(1024) interp_batch_kernel(const BatchOp* __restrict__ ops, BatchList l) {
  uint4 it;
  if (!batch_item(l, blockIdx.x, &it)) return;
  const BatchOp& op = ops[it.x];
  interp_body<DIM, NC, T, FULL>(op.g, op.i, it.y, (int)it.z);
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
// Dynamic LDS a workgroup may use on the current device (160 KB per CU on
// gfx950; queried, since launches above 64 KB need the device to allow it).
size_t lds_limit() {
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

int default_per_cu(int built_in) {
  static const int set = [] {
    const char* e = getenv("GNUFFT_LANE_PER_CU");
    const int v = e ? atoi(e) : 0;
    return v >= 1 && v <= 8 ? v : 0;
  }();
  return set ? set : built_in;
}

template <typename K>
static hipError_t allow_lds(K kernel, size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

// What plans are accepted by: room in LDS for the padded sector of `cb` coils,
// a kernel table, and tap records of 16 samples or (kernel width 3: `lane`)
// rows for taps past the sector.
static size_t record_bytes(const Geom& g, int cb) {
  const int nx = g.kw + 1 <= 4 ? 4 : 8;
  const size_t pd = (size_t)g.P * g.P * (g.dim == 3 ? g.P : 1);
  const size_t kp = (size_t)((g.K + 3) & ~3) * 4 + (size_t)((3 * (g.P + nx) + 3) & ~3) * 4;
  return kp + (((pd + nx) * cb + 1) & ~(size_t)1) * 8 + (size_t)16 * (((1 + 3 * nx) + 3) & ~3) * 4;
}

size_t lane_bytes(const Geom& g, int cb) {
  const size_t P = (size_t)g.P, pd = P * P * (g.dim == 3 ? P : 1);
  const size_t slack = g.dim == 3 ? 2 * P * P + 2 * P + 2 : 2 * P + 2;
  const size_t kp = (size_t)((g.K + 3) & ~3) * 4 + (size_t)((3 * (g.P + 4) + 3) & ~3) * 4;
  return ((kp + 15) & ~(size_t)15) + (((pd + slack) * cb + 1) & ~(size_t)1) * 8;
}

bool padded_sector_fits(const Geom& g, int cb) {
  return record_bytes(g, cb) + 16 * (size_t)cb * sizeof(float2) <= lds_limit() - 1024;
}

bool batch_sector_fits(const Geom& g, int cb) {
  return padded_sector_fits(g, cb) && record_bytes(g, cb) <= lds_limit() - 4096;
}

bool spread_supported(const Geom& g) {
  if (g.kw > 7 || g.P > 255) return false;
  if (g.kw == 3 && g.P >= 4) return lane_bytes(g, 1) <= lds_limit() - 1024;
  return padded_sector_fits(g, 1);
}

static bool interp_supported(const Geom& g) {
  if (g.kw > 7 || g.P > 255) return false;
  if (g.dim == 2 && g.kw == 3 && g.P >= 4) return lane_bytes(g, 1) <= lds_limit() - 1024;
  return record_bytes(g, 1) <= lds_limit() - 4096;
}

int interp_row_bits(const Geom& g) {
  int b = 0;
  while ((2 << b) < g.P) b++;
  return b;
}

int interp_taps(int kw) { return kw <= 3 ? 3 : kw <= 5 ? 5 : 7; }

size_t interp_lds_bytes(const Geom& g, int nc, int taps) { return interp_lds(g, nc, taps); }

// Four workgroups per CU hide each other's loads: 8 coils in two workgroups
// take 0.79 ms at 160^3 osf 2 (4 in four: 0.76; 128^3 koosh: 0.445 and 0.45).
// Among the sizes that fit, the one that pads the coils least: six coils as
// three groups of two take 0.15 ms at a 168 x 160 x 44 stack, as one of eight
// 0.20 ms.
int interp_coils(const Geom& g, int n_coils, int per_cu) {
  const int t = interp_taps(g.kw);
  for (int per = per_cu > 0 ? per_cu : default_per_cu(4); per >= 1; per--) {
    int best = 0, least = 0;
    for (int nc = 8; nc >= 1; nc /= 2) {
      if (interp_lds(g, nc, t) > lds_limit() / per || (nc > 1 && nc / 2 >= n_coils)) continue;
      const int padded = (n_coils + nc - 1) / nc * nc;
      if (best && (padded >= least || nc == 1)) continue;
      best = nc;
      least = padded;
    }
    if (best) return best;
  }
  return 0;
}

// Threads of a workgroup: 32 waves per CU with the workgroups that its LDS
// allows.
static int interp_threads(size_t lds) {
  const size_t per = lds_limit() / lds;
  return per >= 5 ? 256 : 512;
}

template <int DIM, int NC, int T, bool FULL>
static hipError_t interp_launch(const Geom& g, const InterpArgs& a, hipStream_t s) {
  const size_t lds = interp_lds(g, NC, T);
  hipError_t e = allow_lds(interp_kernel<DIM, NC, T, FULL>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((interp_kernel<DIM, NC, T, FULL>), dim3(work_blocks(a.work), (a.n_coils + NC - 1) / NC),
                     dim3(interp_threads(lds)), lds, s, g, a);
  return hipGetLastError();
}

template <int DIM, int NC>
static hipError_t interp_width(const Geom& g, const InterpArgs& a, hipStream_t s) {
  if (g.kw == 3) return interp_launch<DIM, NC, 3, true>(g, a, s);
  if (g.kw < 3) return interp_launch<DIM, NC, 3, false>(g, a, s);
  if (g.kw == 5) return interp_launch<DIM, NC, 5, true>(g, a, s);
  return g.kw < 5 ? interp_launch<DIM, NC, 5, false>(g, a, s) : interp_launch<DIM, NC, 7, false>(g, a, s);
}

template <int DIM>
static hipError_t interp_dim(const Geom& g, const InterpArgs& args, hipStream_t s) {
  InterpArgs a = args;
  a.row_bits = interp_row_bits(g);
  switch (interp_coils(g, a.n_coils, a.per_cu)) {
    case 8: return interp_width<DIM, 8>(g, a, s);
    case 4: return interp_width<DIM, 4>(g, a, s);
    case 2: return interp_width<DIM, 2>(g, a, s);
    case 1: return interp_width<DIM, 1>(g, a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_interp(const Geom& g, const InterpArgs& a, hipStream_t s) {
  if (a.work.n_chunks == 0 || a.n_coils == 0) return hipSuccess;
  if (!interp_supported(g)) return hipErrorInvalidValue;
  return g.dim == 3 ? interp_dim<3>(g, a, s) : interp_dim<2>(g, a, s);
}

// Batches: one launch per coil-group size over (operator, chunk, group) items.
template <int DIM, int NC, int T, bool FULL>
static hipError_t interp_batch(const BatchOp* ops, const BatchList& l, size_t lds, hipStream_t s) {
  hipError_t e = allow_lds(interp_batch_kernel<DIM, NC, T, FULL>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((interp_batch_kernel<DIM, NC, T, FULL>), dim3(8u * (l.max_range ? l.max_range : 1u)),
                     dim3(interp_threads(lds)), lds, s, ops, l);
  return hipGetLastError();
}

template <int DIM, int NC>
static hipError_t interp_batch_width(int taps, bool full, const BatchOp* ops, const BatchList& l, size_t lds,
                                     hipStream_t s) {
  if (taps == 3) return full ? interp_batch<DIM, NC, 3, true>(ops, l, lds, s) : interp_batch<DIM, NC, 3, false>(ops, l, lds, s);
  if (taps == 5) return full ? interp_batch<DIM, NC, 5, true>(ops, l, lds, s) : interp_batch<DIM, NC, 5, false>(ops, l, lds, s);
  return interp_batch<DIM, NC, 7, false>(ops, l, lds, s);
}

template <int DIM>
static hipError_t interp_batch_nc(int nc, int taps, bool full, const BatchOp* ops, const BatchList& l, size_t lds,
                                  hipStream_t s) {
  switch (nc) {
    case 8: return interp_batch_width<DIM, 8>(taps, full, ops, l, lds, s);
    case 4: return interp_batch_width<DIM, 4>(taps, full, ops, l, lds, s);
    case 2: return interp_batch_width<DIM, 2>(taps, full, ops, l, lds, s);
    default: return interp_batch_width<DIM, 1>(taps, full, ops, l, lds, s);
  }
}

hipError_t launch_interp_batch(int dim, int nc, int taps, bool full, const BatchOp* ops, const BatchList& l,
                               size_t lds, hipStream_t s) {
  if (l.n == 0) return hipSuccess;
  return dim == 3 ? interp_batch_nc<3>(nc, taps, full, ops, l, lds, s)
                  : interp_batch_nc<2>(nc, taps, full, ops, l, lds, s);
}

}  // namespace gnufft
