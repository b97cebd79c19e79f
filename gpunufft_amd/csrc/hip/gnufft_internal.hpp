// Internal declarations shared by the HIP translation units of
// libgpunufft_hip.so. Not part of the public ABI (include/gpunufft_hip.h).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

namespace gnufft {

// Geometry and kernel constants of one operator, passed to kernels by value.
// Field meanings follow GpuNUFFTInfo (CUDA/inc/gpuNUFFT_types.hpp:230-311,
// derived in CUDA/src/gpuNUFFT_operator.cpp:53-146).
struct Geom {
  int dim;          // 2 or 3
  int G[3];         // grid dims; G[2] = 1 in 2-D
  int N[3];         // image dims; N[2] = 1 in 2-D
  int S[3];         // sectors per dim; S[2] = 1 in 2-D
  int sw;           // sector width
  int P;            // padded sector width sw + 2*floor(kw/2)
  int Pmax;         // P - 1
  int off;          // floor(P/2)
  int kw;           // kernel width
  int K;            // lookup table entries
  int lookup;       // GNUFFT_LOOKUP_*
  float kradius;    // kw/2
  float rsq;        // squared kernel radius relative to the largest grid dim
  float rsq_inv;
  float dist_mult;  // (K-1)/rsq
  float aniso[3];   // G_a / max(G)
  int shift_inv[3]; // floor(G/2): INVERSE fftshift offset
  int shift_fwd[3]; // ceil(G/2): FORWARD fftshift offset
  int crop[3];      // (int)(N*(osf-1)/2)
  long long Ng;     // grid points per coil
  long long Ni;     // image points per coil
  int M;            // samples
  float fft_scale;  // 1/sqrt(Ng)
};

// ceil(2^32 / d): exact quotient via __umulhi(n, m) for n*d < 2^32.
__host__ inline uint32_t udiv_magic(uint32_t d) {
  return (uint32_t)((0x100000000ull + d - 1) / d);
}

// One gridding work item: samples [begin, end) of a sector.
struct Chunk {
  uint32_t sector;
  uint32_t begin;
  uint32_t end;
  uint32_t pad;
};

// ---------------------------------------------------------------------------
// Tap table: per axis and sample (caller's order) the first grid index of the
// sample's taps, in [0, G), and its kw weights (zero where the reference skips a tap;
// the (kw + 1)-th tap of a position exactly half-way between grid points is
// at the kernel's edge and has weight zero). tap_vec(kw) float4 per entry:
// word 0 the index (as an int), then the weights, zeros past the last.
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int tap_vec(int kw) { return kw <= 3 ? 1 : 2; }

// ---------------------------------------------------------------------------
// Tiles of the adjoint gridding (spread.hip): the grid cut into tiles of
// tile_width(dim, axis) points, each with the list of the samples that have a
// tap of nonzero weight inside it. Sixteen points in x are whole 128-byte
// lines of the grid. A tile is worked on as sub-tiles of 4 points in x (3-D:
// by 4 in y).
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int tile_width(int dim, int axis) {
  return axis == 0 ? 16 : axis == 1 ? (dim == 3 ? 8 : 16) : (dim == 3 ? 4 : 1);
}
__host__ __device__ constexpr int tile_points(int dim) {
  return tile_width(dim, 0) * tile_width(dim, 1) * tile_width(dim, 2);
}
__host__ __device__ constexpr int tile_subs(int dim) { return dim == 3 ? 8 : 4; }
// Coils per workgroup of the spread: the block's 16 columns are 8 / NC
// points in x times NC coils.
__host__ __device__ constexpr int tile_coils(int n_coils) {
  return n_coils > 4 ? 8 : n_coils > 2 ? 4 : n_coils;
}
constexpr uint32_t kNoSlot = ~0u;

struct TileChunk {  // list entries [begin, begin + n) of a tile
  uint64_t begin;
  uint32_t n;  // 0: an empty tile
  uint32_t tile;
  uint32_t slot;  // scratch slot of a tile with several chunks, else kNoSlot
  uint32_t pad;
};

struct TileTask {  // a tile with several chunks: slots [slot, slot + count)
  uint32_t tile, slot, count, pad;
};

struct TileList {
  const uint32_t* entries;  // sample numbers, caller's order
  const TileChunk* chunks;  // every tile has at least one (an empty tile is cleared)
  const TileTask* tasks;
  uint32_t n_chunks, n_tasks;
  int nt[3];  // tiles per axis, rounded up to a multiple of 4 (1 on an unused axis)
};

struct TileTotals {
  uint32_t chunks, slots, tasks;
};

#if defined(__HIPCC__)
// First point of a tile. Tiles are numbered in blocks of 4 per axis (nt is a
// multiple of 4 on the axes in use), so that neighbouring numbers are
// neighbours on every axis; tiles past the grid's end are empty.
template <int DIM>
__device__ inline void tile_start(const TileList& l, uint32_t tile, int* t0) {
  constexpr uint32_t per = DIM == 3 ? 64 : 16;
  const uint32_t in = tile % per, b = tile / per;
  const uint32_t bx = (uint32_t)l.nt[0] / 4, by = (uint32_t)l.nt[1] / 4;
  t0[0] = (int)((b % bx) * 4 + (in & 3)) * tile_width(DIM, 0);
  t0[1] = (int)((DIM == 3 ? (b / bx) % by : b / bx) * 4 + ((in >> 2) & 3)) * tile_width(DIM, 1);
  t0[2] = DIM == 3 ? (int)((b / (bx * by)) * 4 + (in >> 4)) * tile_width(DIM, 2) : 0;
}

// Number of the tile at tile coordinates (x, y, z).
template <int DIM>
__device__ inline uint32_t tile_number(const TileList& l, uint32_t x, uint32_t y, uint32_t z) {
  const uint32_t bx = (uint32_t)l.nt[0] / 4, by = (uint32_t)l.nt[1] / 4;
  if (DIM == 2) return (x / 4 + bx * (y / 4)) * 16 + (x & 3) + 4 * (y & 3);
  return (x / 4 + bx * (y / 4 + by * (z / 4))) * 64 + (x & 3) + 4 * (y & 3) + 16 * (z & 3);
}

// Grid offset of point (x, y, z), at its INVERSE-fftshifted position when
// `shift` (std_gpuNUFFT_kernels.cu:629-654).
template <int DIM>
__device__ inline size_t tile_store_index(const Geom& g, int x, int y, int z, bool shift) {
  if (shift) {
    x = x < g.shift_inv[0] ? x - g.shift_inv[0] + g.G[0] : x - g.shift_inv[0];
    y = y < g.shift_inv[1] ? y - g.shift_inv[1] + g.G[1] : y - g.shift_inv[1];
    if (DIM == 3) z = z < g.shift_inv[2] ? z - g.shift_inv[2] + g.G[2] : z - g.shift_inv[2];
  }
  return (size_t)x + (size_t)g.G[0] * ((size_t)y + (DIM == 3 ? (size_t)g.G[1] * z : 0));
}
#endif

// ---------------------------------------------------------------------------
// Exact per-sample index / weight arithmetic. Contraction is disabled so the
// float rounding of every ceil/floor/round input matches the reference's
// separate multiply and add (CUDA/inc/gpuNUFFT_utils.hpp:89-104, 194-209).
// ---------------------------------------------------------------------------
#pragma clang fp contract(off)

__device__ __host__ inline float map_kspace_to_grid(float pos, int G, int center, int off) {
  return (pos * (float)G) + (0.5f * (float)G) - (float)center + (float)off;
}

__device__ __host__ inline float map_grid_to_kspace(int i, int G, int center, int off) {
  return ((float)i + (float)center - (float)off) / (float)G - 0.5f;
}

__device__ __host__ inline void tap_range(float u, int Pmax, float radius, int* lo, int* hi) {
  int mn = (int)ceilf(u - radius);
  int mx = (int)floorf(u + radius);
  if (mn < 0) mn = 0;
  if (mx < 0) mx = 0;
  if (mx >= Pmax) mx = Pmax;
  if (mn >= (float)Pmax) mn = (int)((float)Pmax - 2.0f * radius);
  if (mn < 0) mn = 0;  // only reachable when P < kw + 1 (reference reads out of bounds)
  *lo = mn;
  *hi = mx;
}

// Emulated clamp-addressed linear texture fetch of the 1-D table at the
// normalised coordinate u: texel coordinate u*K-0.5, fractional weight with
// 8 fractional bits (round to nearest).
__device__ __host__ inline float lerp_fetch(const float* tab, int K, float u) {
  float xb = u * (float)K - 0.5f;
  float fl = floorf(xb);
  int i0 = (int)fl;
  float a = xb - fl;
  a = rintf(a * 256.0f) * (1.0f / 256.0f);
  int i1 = i0 + 1;
  i0 = i0 < 0 ? 0 : (i0 > K - 1 ? K - 1 : i0);
  i1 = i1 < 0 ? 0 : (i1 > K - 1 ? K - 1 : i1);
  return (1.0f - a) * tab[i0] + a * tab[i1];
}

// roundf(x) as an integer for x >= 0 (half away from zero), without the sign
// handling of the library call.
__device__ __host__ inline int round_index(float x) {
  const int i = (int)x;
  return x - (float)i >= 0.5f ? i + 1 : i;
}

// Weight of one tap along one axis; returns false when the nearest-mode
// radius test rejects the tap (atomic_gpuNUFFT_kernels.cu:343-368); the
// linear mode has no radius test (texture_gpuNUFFT_kernels.cu:63-82).
__device__ __host__ inline bool axis_weight(const Geom& g, const float* lut, int a, int i,
                                            int center, float pos, float* w) {
  float kp = map_grid_to_kspace(i, g.G[a], center, g.off);
  float d = (kp - pos) * g.aniso[a];
  d *= d;
  if (g.lookup == 0) {
    if (!(d < g.rsq)) return false;
    int li = round_index(d * g.dist_mult);
    *w = lut[li < g.K - 1 ? li : g.K - 1];
    return true;
  }
  *w = lerp_fetch(lut, g.K, d * g.rsq_inv);
  return true;
}

// Sector index along one axis (CUDA/inc/precomp_utils.hpp:34-48): float
// product, double sum, round half away from zero in double, double
// quotient, floor, clamped to ceil((float)G/sw)-1 evaluated in float.
__device__ inline int sector_of(float coord, int G, int sw) {
  double v = (double)(coord * (float)G) + 0.5 * (double)(float)G;
  int sector = (int)floor(round(v) / (double)(float)sw);
  int smax = (int)ceilf((float)G / (float)sw);
  if (sector >= smax) sector = smax - 1;
  if (sector < 0) sector = 0;
  return sector;
}

#pragma clang fp contract(on)

// Periodic wrap into [0, G). Callers pass coordinates within a few grid
// lengths of the grid, so a short loop of +-G replaces a division.
__device__ __host__ inline int wrap(int p, int G) {
  while (p >= G) p -= G;
  while (p < 0) p += G;
  return p;
}

// Message returned by gnufft_last_error() on this thread (capi.hip).
void set_last_error(const std::string& msg);

}  // namespace gnufft

struct gnufft_plan_s;

namespace gnufft {

// Generation of a plan's device buffers (capi.hip): changes whenever memory
// that a captured graph or a batch may reference is freed or replaced.
uint64_t plan_generation(const gnufft_plan_s* p);

// Some grid length of the plan is odd: its two directions are not adjoint to
// each other (sector_spread.hip).
bool plan_odd_grid(const gnufft_plan_s* p);

// gnufft_adjoint; `sector_sums`: gridding by launch_sector_spread. The first such
// call after a trajectory was set builds tables (and waits for them).
int plan_adjoint(gnufft_plan_s* p, const void* kdata, void* out, uint32_t n_coils, int stop, bool sector_sums,
                 void* stream);

// ---------------------------------------------------------------------------
// Launchers implemented in the .hip translation units (all asynchronous on
// `stream`; return hipError_t).
// ---------------------------------------------------------------------------

// precompute.hip
hipError_t launch_assign_sectors(const Geom& g, const float* traj, uint32_t M, uint32_t* keys,
                                 uint32_t* vals, hipStream_t s);
hipError_t sort_pairs(void* temp, size_t* temp_bytes, const uint32_t* keys_in,
                      uint32_t* keys_out, const uint32_t* vals_in, uint32_t* vals_out,
                      uint32_t M, int key_bits, hipStream_t s);
hipError_t launch_sector_data_count(const uint32_t* sorted_keys, uint32_t M, uint32_t S,
                                    uint32_t* sdc, hipStream_t s);
hipError_t launch_sector_centers(const Geom& g, uint32_t* centers, hipStream_t s);
hipError_t launch_gather_traj(const float* traj, const float* dens, const uint32_t* idx,
                              uint32_t M, int dim, float* traj_sorted, float* dens_sorted,
                              hipStream_t s);
hipError_t count_chunks(const uint32_t* sdc, uint32_t S, uint32_t chunk, uint32_t* cnt,
                        uint32_t* chunk_off, void* temp, size_t* temp_bytes, hipStream_t s);
hipError_t launch_fill_chunks(const uint32_t* sdc, const uint32_t* chunk_off, uint32_t S,
                              uint32_t chunk, Chunk* chunks, hipStream_t s);

// Tap table of the sorted samples (s the caller's sample idx[s]), their sorted
// positions (pos[idx[s]] = s), the square roots of their density weights (dens
// NULL: none), all in the caller's order, and per caller's sample the number of
// tiles its taps reach (counts).
hipError_t launch_taps(const Geom& g, const float* crds, const float* dens, const uint32_t* idx, const float* lut,
                       float4* taps, uint32_t* pos, float* dens_sqrt, uint32_t* counts, hipStream_t s);
// Exclusive sums of n counts (n + 1 of them).
hipError_t scan_counts(void* temp, size_t* temp_bytes, const uint32_t* counts, uint64_t* offs, size_t n,
                       hipStream_t s);
// (tile, sample) pairs of every sample at its offset
hipError_t launch_emit_pairs(const Geom& g, const TileList& l, const float4* taps, const uint64_t* offs,
                             uint32_t* keys, uint32_t* vals, hipStream_t s);
hipError_t sort_tile_pairs(void* temp, size_t* temp_bytes, const uint32_t* keys_in, uint32_t* keys_out,
                           const uint32_t* vals_in, uint32_t* vals_out, size_t n, int key_bits, hipStream_t s);
// the tiles' offsets in the sorted pairs (tiles + 1)
hipError_t launch_tile_offsets(const uint32_t* keys, size_t n, uint32_t tiles, uint64_t* tile_off, hipStream_t s);
// chunks of at most `chunk` entries: per-tile exclusive sums (tiles + 1)
hipError_t scan_tile_chunks(void* temp, size_t* temp_bytes, const uint64_t* tile_off, uint32_t tiles,
                            uint32_t chunk, TileTotals* tot, hipStream_t s);
hipError_t fill_tile_chunks(const uint64_t* tile_off, uint32_t tiles, uint32_t chunk, const TileTotals* tot,
                            TileChunk* chunks, TileTask* tasks, hipStream_t s);

// All tables of a short trajectory (caller's order; short_tables_ok).
struct ShortTables {
  const float* traj;  // [dim][M]
  const float* dens;  // NULL: none
  const float* lut;
  uint32_t S, n_tiles, chunk;  // sectors, tiles, samples per interp chunk
  uint32_t max_slots;          // partial tiles
  // sector tables
  uint32_t *assigned, *idx, *sdc, *centers;
  float *traj_sorted, *dens_sorted;
  Chunk *chunks, *runs;  // room for S + M / chunk each
  // tap table and tile lists
  float4* taps;
  uint32_t* pos;
  float* dens_sqrt;
  uint32_t* entries;       // room for every pair (short_tables_entries)
  TileChunk* tile_chunks;  // room for n_tiles + entries / 128
  TileTask* tile_tasks;    // room for n_tiles
  uint32_t* host;          // pinned: sdc (S + 1 words), then chunks, runs, tile chunks, slots, tasks
  uint32_t *counts, *offs;  // short_tables_words each
};
constexpr uint32_t kShortTotals = 5;
bool short_tables_ok(uint32_t M, uint32_t S, uint32_t n_tiles);
size_t short_tables_entries(const Geom& g, uint32_t M);
size_t short_tables_words(uint32_t M, uint32_t S, uint32_t n_tiles);
// temp NULL: only sets *temp_bytes
hipError_t launch_short_tables(const Geom& g, const TileList& l, const ShortTables& t, void* temp,
                               size_t* temp_bytes, hipStream_t s);
// Entries per tile chunk for `pairs` list entries: enough chunks for the whole
// device (512 of them: a workgroup has 4 to 8 waves), between 128 and 512 (2-D)
// or 2048 (3-D). A batch of 24 2-D operators takes 1.90 ms with twice as many
// chunks (more partial tiles), CG at 240^2 1.46 instead of 1.36 ms with half.
__device__ __host__ inline uint32_t tile_chunk(int dim, uint64_t pairs) {
  const uint32_t most = dim == 3 ? 2048u : 512u;
  uint32_t chunk = 128;
  while (chunk < most && (uint64_t)chunk * 512 < pairs) chunk *= 2;
  return chunk;
}

// gridding.hip

// Chunks per 3-D interp run, which stages its sector once. Interp at 128^3 koosh /
// a 168 x 160 x 44 stack / 160^3: 459 / 140 / 759 us with 1, 450 / 143 / 757 with 2,
// 449 / 152 / 760 with 4, 469 / 155 / 754 with 8 (a tail of busy workgroups).
constexpr int kInterpRun = 2;

// Gridding work list: chunks in sector order, split into 8 contiguous
// ranges of about equal cost; range x is processed on XCD x (workgroups
// are dispatched round-robin over the XCDs), so neighbouring sectors share
// an L2 and no XCD is left with the dense k-space centre alone.
struct WorkList {
  const Chunk* chunks;
  uint32_t n_chunks;
  uint32_t xcd_begin[9];  // range x = [xcd_begin[x], xcd_begin[x+1])
  uint32_t max_range;     // longest range: workgroups per XCD
};

// Split `n` chunks of the given sample counts into the 8 ranges of `w`.
void partition_work(const uint32_t* counts, uint32_t n, WorkList* w);

struct SpreadArgs {
  const float2* data;      // [coil][...] samples, caller's order
  long long coil_stride;   // elements between coils of `data`
  const float* dens;       // square roots of the density weights, caller's order (NULL: none)
  const float4* taps;      // tap table [dim][M]
  const uint32_t* pos;     // data in sector order: sorted position of the caller's sample j (NULL: caller's order)
  TileList tiles;
  float2* scratch;         // partial tiles [slot][coil][tile point]
  float2* grid;            // [coil][Ng], every point written (no prior zeroing)
  int n_coils;
  bool fold_shift;         // store at INVERSE-fftshifted positions
};
hipError_t launch_spread(const Geom& g, const SpreadArgs& a, hipStream_t s);

// sector_spread.hip: the gridding of CG-SENSE on grids with an odd length.
constexpr uint32_t kSumsChunk = 1024;  // samples per chunk (two per thread)
struct SectorSpreadArgs {
  const float2* data;     // [coil][...] samples, caller's order
  long long coil_stride;  // elements between coils of `data`
  const float* dens;      // square roots of the density weights, caller's order (NULL: none)
  const float4* taps;     // tap table [dim][M]
  const uint32_t* idx;    // caller's number of sorted sample s
  const Chunk* chunks;    // the sectors' samples in runs of at most kSumsChunk
  const uint32_t* first;  // [sectors + 1] first chunk of a sector
  const uint32_t* cover_off[3];  // sector_cover of the axes in use
  const uint2* cover[3];
  float2* sub;   // [chunk][coil][padded point]
  float2* grid;  // [coil][Ng], every point written
  uint32_t n_chunks;
  int n_coils;
  bool fold_shift;  // store at INVERSE-fftshifted positions
};
// per_cu: workgroups per CU that coil blocks are sized for (0: default)
hipError_t launch_sector_spread(const Geom& g, const SectorSpreadArgs& a, int per_cu, hipStream_t s);
size_t sector_sub_elems(const Geom& g);  // of one chunk and coil
// Per grid index q of an axis, the (sector, padded index) pairs that fall on it:
// entries off[q] .. off[q + 1], by sector.
void sector_cover(const Geom& g, int axis, std::vector<uint32_t>* off, std::vector<uint2>* entries);

// gridding.hip
size_t lds_limit();
// Workgroups per CU that a plan without a target of its own sizes its coil groups
// for: the environment variable GNUFFT_LANE_PER_CU (1 .. 8, read once), else
// `built_in`.
int default_per_cu(int built_in);
// Padded sector of `cb` coils with room for taps past it, kernel table and positions.
size_t lane_bytes(const Geom& g, int cb);
// False for geometries whose padded sector does not fit the LDS of a CU (the
// interp stages padded sectors; gridding.hip).
bool spread_supported(const Geom& g);
bool padded_sector_fits(const Geom& g, int cb);
// False when the padded sectors covering one sector are more than 256 (sector
// widths far below the kernel width).
bool sector_cover_ok(const Geom& g);

struct InterpArgs {
  const float2* grid;      // [coil][Ng]
  WorkList work;
  const float4* taps;      // tap table [dim][M]
  const uint32_t* idx;     // caller's number of sorted sample s
  float2* out;             // [coil][...], caller's order
  long long coil_stride;
  bool sorted_out;         // write in sector order
  const float* dens;       // square roots of the density weights, caller's order (NULL: none)
  float scale;             // 1 (kernel only) or 1/sqrt(Ng)
  int n_coils;
  bool fold_shift;         // read grid at FORWARD-fftshifted positions
  int per_cu;              // workgroups per CU the coil group is sized for (0: default)
  int row_bits;            // interp_row_bits (launch_interp sets it)
};
hipError_t launch_interp(const Geom& g, const InterpArgs& a, hipStream_t s);

// prepost.hip
hipError_t launch_zero(void* p, size_t bytes, hipStream_t s);
// out[z][y][x] = norm / |sum_t B[t][y][x] E[t][z]| (double), t < T.
hipError_t launch_deapo_combine(const double2* B, const double2* E, int T, int Nx, int Ny, int Nz,
                                double norm, float* out, hipStream_t s);
hipError_t launch_adjoint_post(const Geom& g, const float2* grid, int n_coils,
                               const float* deapo, const float2* sens, float2* out,
                               bool accumulate, int stop, hipStream_t s);
hipError_t launch_forward_pre(const Geom& g, const float2* img, bool img_per_coil,
                              const float2* sens, const float* deapo, float2* grid, int n_coils,
                              hipStream_t s);
hipError_t launch_image_prep(const Geom& g, const float2* img, bool img_per_coil,
                             const float2* sens, const float* deapo, float2* out, int n_coils,
                             hipStream_t s);

// ---------------------------------------------------------------------------
// Batches of independent operators: every stage of every operator runs in
// one launch per stage. Workgroups take items (operator, index, coil block)
// from a flat list split into 8 XCD ranges of equal cost, and read their
// operator's geometry and arguments from a descriptor in device memory.
// ---------------------------------------------------------------------------
struct PostArgs {  // adjoint tail (crop, scale, deapo, coil combine)
  const float2* grid;
  int n_coils;
  const float* deapo;
  const float2* sens;  // NULL: per-coil output
  float2* out;
  int stop;
};

struct PreArgs {  // forward head (sens, deapo, pad, shift)
  const float2* img;
  int img_per_coil;
  const float2* sens;
  const float* deapo;
  float2* grid;
  int n_coils;
};

struct BatchOp {
  Geom g;
  SpreadArgs s;
  InterpArgs i;
  PostArgs post;
  PreArgs pre;
};

struct BatchList {
  const uint4* items;  // (operator, index, coil block, unused)
  uint32_t n;
  uint32_t xcd_begin[9];
  uint32_t max_range;
};

#if defined(__HIPCC__)
// Item of workgroup bid in a batch list (the XCD mapping of work_chunk);
// false past the end of its XCD's range.
__device__ inline bool batch_item(const BatchList& l, uint32_t bid, uint4* it) {
  const uint32_t x = bid & 7u;
  const uint32_t i = l.xcd_begin[x] + (bid >> 3);
  if (i >= l.xcd_begin[x + 1]) return false;
  const uint4 v = l.items[i];
  // workgroup-uniform: scalar registers, so the item's plan descriptor is
  // read with scalar loads (as vector values every descriptor field would
  // take VGPRs)
  *it = make_uint4(__builtin_amdgcn_readfirstlane(v.x), __builtin_amdgcn_readfirstlane(v.y),
                   __builtin_amdgcn_readfirstlane(v.z), __builtin_amdgcn_readfirstlane(v.w));
  return true;
}
#endif

// Split items of the given costs into the 8 XCD ranges of `l` (items stay in order).
void partition_items(const uint32_t* costs, uint32_t n, BatchList* l);

// gridding.hip (CB: coils per workgroup, the same for every operator).
// Coil block that a batch's padded sectors have to fit the LDS for.
constexpr int kBatchCB = 8;
// Spread of a batch: `items` (operator, chunk of its tile lists, coil group)
// by coils per workgroup nc (nx: taps per axis, 4 or 8); tasks (operator, task, coil, block) of the tiles
// with several chunks.
hipError_t launch_spread_batch(int dim, int nx, int nc, const BatchOp* ops, const BatchList& l,
                               size_t lds, hipStream_t s);
hipError_t launch_tile_reduce_batch(int dim, const BatchOp* ops, const BatchList& tasks, hipStream_t s);
size_t spread_lds_bytes(int dim, int nc);
// taps, full: interp_taps of the widest plan, and whether every plan's kernel
// width is that
hipError_t launch_interp_batch(int dim, int nc, int taps, bool full, const BatchOp* ops, const BatchList& l,
                               size_t lds, hipStream_t s);
int interp_taps(int kw);
// log2 of the threads per staged row: a power of two, two points each
int interp_row_bits(const Geom& g);
// Coils per group (8, 4, 2, 1) of an interp launch; 0: the sector does not fit
int interp_coils(const Geom& g, int n_coils, int per_cu);
size_t interp_lds_bytes(const Geom& g, int nc, int taps);
// The padded sector of `cb` coils fits a batch's LDS
bool batch_sector_fits(const Geom& g, int cb);

// prepost.hip: items (operator, block of 256 pixels / grid points, 0, 0)
hipError_t launch_post_batch(const BatchOp* ops, const BatchList& l, hipStream_t s);
hipError_t launch_pre_batch(const BatchOp* ops, const BatchList& l, hipStream_t s);

// Fused oversampled-grid FFT (fft.hip).
bool fused_fft_supported(const Geom& g);
bool fused_fft_preferred(const Geom& g);
// Some axis of g needs a prime stage (7 .. 19).
bool fused_fft_prime(const Geom& g);
size_t fused_fft_tmp_elems(const Geom& g);
std::vector<float2> fused_fft_twiddles(const Geom& g, size_t offsets[3][3]);
hipError_t fused_fft_adjoint(const Geom& g, float2* grid, float2* tmp, int coils,
                             const float* deapo, const float2* sens, float2* out, int stop,
                             bool accumulate, const float2* tw, const size_t tw_off[3][3],
                             hipStream_t s);
hipError_t fused_fft_forward(const Geom& g, const float2* img, bool img_per_coil,
                             const float2* sens, const float* deapo, float2* grid, float2* tmp,
                             int coils, const float2* tw, const size_t tw_off[3][3],
                             hipStream_t s);
// Batches: one opaque descriptor (fused_fft_desc_bytes) per operator in
// device memory; each pass of every operator is one launch over items
// (operator, block). Passes: adjoint ax[0 .. d-2] then x, forward x then
// ax[0 .. d-2] (fused_fft_pass_count(d) of each).
size_t fused_fft_desc_bytes();
bool fused_fft_desc_build(void* desc, const Geom& g, float2* grid, float2* tmp, int coils,
                          const float* deapo, const float2* sens, const float2* tw,
                          const size_t tw_off[3][3]);
void fused_fft_desc_set_io(void* desc, float2* adjoint_out, const float2* forward_img);
int fused_fft_pass_count(int dim);
uint32_t fused_fft_pass_blocks(const void* desc, bool adjoint, int pass);
size_t fused_fft_pass_lds(const void* desc, bool adjoint, int pass);
int fused_fft_pass_big(const void* desc, bool adjoint, int pass);
// prime: some operator's lengths need the prime stages 7 .. 19
hipError_t launch_fused_fft_batch(int dim, bool adjoint, int pass, bool big, bool prime,
                                  const void* descs_d, const uint2* items, uint32_t n_items,
                                  size_t lds, hipStream_t s);

}  // namespace gnufft
