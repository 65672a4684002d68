// Tile geometry shared by the tile sort, the window paint and the window
// gathers (16^3-cell tiles; particles sorted by the tile of their floor cell).
#pragma once

#include <vector>

#include "common.hpp"

namespace jpm {

constexpr int kTile = 16;                       // tile edge in cells
constexpr int kWin = kTile + 1;                 // window edge (CIC +1 corner)
constexpr int kWinCells = kWin * kWin * kWin;   // 4913
constexpr int kChunk = 8192;                    // default max particles per chunk
constexpr int kMaxKeysLds = 32768;              // LDS histogram limit (128 KiB)
constexpr uint32_t kSlice = 8192;               // particles per count / scatter workgroup of a large sort
// Accumulation / force-gather workgroup size: their LDS windows (38-39 KiB)
// allow 4 workgroups per CU, so 512 threads keep 32 waves resident.
constexpr int kWindowThreads = 512;

// Sort tuning carried in bits 16..26 of the pipeline flags (0 = default):
// chunk = 2^(9 + c) particles for c = bits 16..19 in 1..6 (1024..32768),
// slice = 2^(11 + s) particles for s = bits 20..23 in 1..7 (4096..262144).
inline uint32_t tuned_chunk(uint32_t flags) {
  const uint32_t c = (flags >> 16) & 0xfu;
  return (c >= 1 && c <= 6) ? (1u << (9 + c)) : uint32_t(kChunk);
}
// Bit 24: the force-VJP gather reads the density adjoint through the caches
// instead of an LDS window.
constexpr uint32_t kTuneRhoGlobal = 1u << 24;
inline bool tuned_rho_lds(uint32_t flags) { return !(flags & kTuneRhoGlobal); }
// Bit 25: XCD slabs.  The dispatcher deals workgroup b to XCD b mod 8; with
// slabs, the chunk (or tile) of workgroup b is (b mod 8) * per + b / 8, so
// each XCD walks one contiguous run of tiles and neighbouring tiles, whose
// windows overlap, share that XCD's L2.
constexpr uint32_t kTuneXcdSlabs = 1u << 25;
inline bool tuned_slabs(uint32_t flags) { return (flags & kTuneXcdSlabs) != 0; }
// Bit 26: the force evaluations' one-channel paint writes its finished
// low-face cells into the mesh, not into a buffer of their own that the
// potential solve's first pass reads (FaceCells); the same bits either way.
constexpr uint32_t kTuneFacesInMesh = 1u << 26;

// Workgroups for `items` work items and the per-XCD run length.
inline unsigned slab_grid(uint32_t items, bool slabs, uint32_t &per) {
  per = (items + 7u) / 8u;
  if (per == 0) per = 1;
  return slabs ? 8u * per : (items ? items : 1u);
}

__device__ __forceinline__ uint32_t slab_item(uint32_t b, uint32_t per, bool slabs) {
  return slabs ? (b & 7u) * per + (b >> 3) : b;
}

// XCD runs for the window gathers (without slabs): of each 8 R consecutive
// workgroups b = 8 R k + 8 q + x (the dispatcher deals b to XCD x), chunk
// 8 R k + R x + q, so each run of R consecutive chunks -- z-neighbouring
// tiles when single-chunk, two y-adjacent z rows of tiles at 256^3 -- runs
// on one XCD at once, and the 64-byte lines that their potential windows'
// rows overlap in (a window row of 21 floats spans three such lines) are
// fetched into its L2 once.  Runs still alternate over the XCDs, which keeps
// clustered tiles spread over them (the slab placement, one contiguous eighth
// of the tiles per XCD, does not).  At 256^3 with 512-thread gathers, against
// dispatch order: force+kick 0.239 -> 0.227 ms, force VJP 0.293 -> 0.280 ms
// (runs of 2: 0.235 / 0.286; of 8: 0.230 / 0.282; of 16: 0.229 / 0.280);
// with the 1024- and 768-thread gathers runs of 32 against 16 and 64:
// 0.2174 / 0.2693 ms against 0.2184 / 0.2703 and 0.2199 / 0.2715.
// Meshes of fewer than 256 tiles take shorter runs (powers of two, at most an
// eighth of their tiles), so that every XCD has some: runs of 32 put the 8
// tiles of a 32^3 mesh on one XCD and the 64 of a 64^3 mesh on two (its kick
// 15.0 -> 13.6 us, its force VJP 19.8 -> 18.8).
// `place` says which item a workgroup takes: with slabs the items per XCD,
// without them log2 of the run.
constexpr uint32_t kXcdRun = 32;
inline unsigned gather_grid(uint32_t items, uint32_t tiles, bool slabs, uint32_t &place) {
  const unsigned g = slab_grid(items, slabs, place);
  if (slabs) return g;
  uint32_t run = 0;
  while ((16u << run) <= tiles && (1u << run) < kXcdRun) ++run;
  place = run;
  return ((g + (8u << run) - 1u) >> (3u + run)) << (3u + run);
}

__device__ __forceinline__ uint32_t gather_item(uint32_t b, uint32_t place, bool slabs) {
  if (slabs) return slab_item(b, place, true);
  const uint32_t run = place, block = b >> (3u + run) << (3u + run), r = b - block;
  return block + ((r & 7u) << run) + (r >> 3);
}
// Particles per count / scatter workgroup of a sort of n particles.  Slices
// that narrow with n keep a few hundred workgroups on the chip (a slice of
// 8192 is 4 workgroups at 32^3, which take 11 us for a 2 us scatter); wide
// ones write longer runs per tile, which is what a paint of particles in no
// order needs.  The force pipelines (`forces`), whose particles are mostly in
// the order of their lattice or of their tiles, take slices of 4096 from 2^19
// particles on (192^3 relative forces 420 -> 402 us; pm_forces at 164^3, 224^3
// and 256^3, slices of 8192 and 4096 us: lattice order 457 and 442, 521 and
// 510, 538 and 522, no order 536 and 521, 739 and 729, 866 and 879).
inline uint32_t tuned_slice(uint32_t flags, int64_t n, bool forces = false) {
  const uint32_t v = (flags >> 20) & 0xfu;
  if (v >= 1 && v <= 7) return 1u << (11 + v);
  if (n < (int64_t(1) << 17)) return 1024;
  if (n < (int64_t(1) << 19)) return 2048;
  return forces || n < (int64_t(1) << 22) ? 4096 : kSlice;
}
// Bit 27, set inside the force pipelines.
constexpr uint32_t kSortForces = 1u << 27;

// A tile's low-face cells (lx = 0, or ly = 0, or lz = 0), numbered in face
// order: the lx = 0 plane (ly * 16 + lz), then ly = 0 with lx > 0
// (256 + (lx - 1) * 16 + lz), then lz = 0 with lx, ly > 0
// (496 + (lx - 1) * 15 + ly - 1) -- 721 cells.
constexpr int kFaces = kTile * kTile + (kTile - 1) * kTile + (kTile - 1) * (kTile - 1);

__host__ __device__ __forceinline__ int face_index(int a, int b, int c) {
  return a == 0 ? b * kTile + c
                : (b == 0 ? kTile * kTile + (a - 1) * kTile + c
                          : kTile * kTile + (kTile - 1) * kTile + (a - 1) * (kTile - 1) + (b - 1));
}

// The low-face cells of a paint kept apart from its mesh.  A tile's face
// cells take the lower neighbours' halos, which the face reduce adds; the
// force paths let it write the finished face values here, contiguous per
// tile, and the potential solve's first pass reads them in place of the
// mesh's (stale) face cells.  Written into the mesh, the lz = 0 face cells
// are single floats a mesh row apart, each write a partial 64-byte line.
// Channel ch, tile T at fb + ch * chan + T * kFaceStride, in face order.
// Needs one simulation whose mesh sides are multiples of 16 (every tile
// full), absolute positions and a paint that replaces the mesh.
constexpr int kFaceStride = 724;   // 721 cells, padded to 16 bytes
struct FaceCells {
  float *fb;            // null: the mesh holds every cell
  uint32_t ny, ty, tz;  // mesh cells along y; tiles along y and z
  size_t chan;          // floats per channel
  FastDiv div_ny;       // row -> (x, y)
};

// A load through the global address space.  For some pointers held in
// structs the compiler otherwise emits a flat load, which also counts
// against the LDS wait counter: every LDS wait after it would wait for the
// memory load too, and a load issued early to hide its latency would not.
__device__ __forceinline__ float4 load_global(const float4 *p) {
  const __attribute__((address_space(1))) float *q = (const __attribute__((address_space(1))) float *)(p);
  return make_float4(q[0], q[1], q[2], q[3]);
}

// Runs of equal keys among the 64 lanes of a wavefront: `heads` has bit l set
// when lane l starts a run (its key differs from lane l-1's, or l is lane 0);
// a head's run ends where the next head begins or at the last active lane
// (active lanes are always a prefix of the wavefront).
__device__ __forceinline__ unsigned long long run_heads(uint32_t key, bool active) {
  const int lane = threadIdx.x & 63;
  const uint32_t prev = __shfl_up(key, 1);
  const bool head = active && (lane == 0 || key != prev);
  return __ballot(head);
}

__device__ __forceinline__ uint32_t run_length(unsigned long long heads, unsigned long long act) {
  const int lane = threadIdx.x & 63;
  const unsigned long long above = heads & ~((2ull << lane) - 1ull);
  const int next = above ? __ffsll((long long)above) - 1 : 64;
  const int last_active = 63 - __clzll((long long)act);
  return uint32_t(min(next, last_active + 1) - lane);
}

struct TileGrid {
  int nx, ny, nz;   // mesh
  int tx, ty, tz;   // tiles per axis
  uint32_t K;       // tiles
  FastDiv div_nz, div_ny, div_tz, div_ty;
};

inline TileGrid make_tiles(int nx, int ny, int nz) {
  TileGrid t;
  t.nx = nx;
  t.ny = ny;
  t.nz = nz;
  t.tx = (nx + kTile - 1) / kTile;
  t.ty = (ny + kTile - 1) / kTile;
  t.tz = (nz + kTile - 1) / kTile;
  t.K = uint32_t(t.tx) * t.ty * t.tz;
  t.div_nz = FastDiv(uint32_t(nz));
  t.div_ny = FastDiv(uint32_t(ny));
  t.div_tz = FastDiv(uint32_t(t.tz));
  t.div_ty = FastDiv(uint32_t(t.ty));
  return t;
}

__device__ __forceinline__ int wrapi(int c, int n) {
  // cells already inside [0, n) (nearly all of them) skip the division
  if (uint32_t(c) < uint32_t(n)) return c;
  int r = c % n;
  return r < 0 ? r + n : r;
}

// Floor cell of a particle: absolute -> int32(floor(x)) mod n (painting.py:
// 23, 35-37); relative -> the low corner of enmesh (painting_utils.py:48-57),
// or, when that corner is dropped, the high corner minus one.
__device__ __forceinline__ int floor_cell_abs(float x, int n) { return wrapi(cell_int(floorf(x)), n); }

// The exact expressions below in float and double (and on the host, for their
// test).
__host__ __device__ __forceinline__ float fmod_of(float x, float L) { return fmodf(x, L); }
__host__ __device__ __forceinline__ double fmod_of(double x, double L) { return fmod(x, L); }
__host__ __device__ __forceinline__ float abs_of(float x) { return fabsf(x); }
__host__ __device__ __forceinline__ double abs_of(double x) { return fabs(x); }
__host__ __device__ __forceinline__ float rint_of(float x) { return rintf(x); }
__host__ __device__ __forceinline__ double rint_of(double x) { return rint(x); }
__host__ __device__ __forceinline__ float copysign_of(float x, float y) { return copysignf(x, y); }
__host__ __device__ __forceinline__ double copysign_of(double x, double y) { return copysign(x, y); }

// jnp.remainder(x, L) for L > 0.  Inside [0, 2 L) and (-L, 0) fmod is x, the
// exact difference x - L (Sterbenz) or x, so nearly every lattice node plus
// displacement skips its division loop; the rest, NaN among it, takes it.
template <class T>
__host__ __device__ __forceinline__ T jmod(T x, T L) {
  if (x >= T(0) && x < L) return x;
  if (x < T(0) && x > -L) return x + L;
  if (x >= L && x < T(2) * L) return x - L;
  T m = fmod_of(x, L);
  if (m != T(0) && m < T(0)) m = m + L;
  return m;
}

// nd - rint(nd / L) L for L > 0 (enmesh's periodic fold of a distance):
// a quarter of a period around 0 or +-L the quotient rounds to 0 or +-1
// without being formed.
template <class T>
__host__ __device__ __forceinline__ T fold_period(T nd, T L) {
  const T a = abs_of(nd);
  if (a <= T(0.25) * L) return nd;
  if (a >= T(0.75) * L && a <= T(1.25) * L) return nd - copysign_of(L, nd);
  return nd - rint_of(nd / L) * L;
}

__device__ __forceinline__ int floor_cell_rel(float p, int n) {
  const float L = float(n);
  float q = floorf(jmod(p, L));
  if (q >= 0.0f && q < L) return int(q);
  float q1 = floorf(jmod(p + 1.0f, L));
  if (q1 >= 0.0f && q1 < L) return wrapi(int(q1) - 1, n);
  return 0;  // NaN: every corner is dropped, any tile will do
}

// Two neighbouring mesh values in one load, aligned to a single one.
template <class T>
struct PairOf {
  typedef T type __attribute__((ext_vector_type(2), aligned(sizeof(T))));
};

// The 8 corner values of NC meshes (cstride apart) at cells {ix}, {iy}, {iz}
// (per axis the low and the high corner), v[c][bx | by << 1 | bz << 2].  The
// two z corners are neighbours in memory except across the periodic end and
// where a relative corner was dropped, so they come in one load per (x, y) row
// (PAIR; needs nz >= 2), at the low corner or, for the last cell, one before
// it, with loads of their own for a high corner elsewhere.  Every mesh's pairs
// are issued before the first is used.
template <bool PAIR, int NC, class T>
__device__ __forceinline__ void load_corners(const T *__restrict__ m, size_t cstride, const uint32_t ix[2],
                                             const uint32_t iy[2], const uint32_t iz[2], uint32_t ny, uint32_t nz,
                                             T v[NC][8]) {
  if (PAIR) {
    const uint32_t zc = iz[0] + 1 < nz ? iz[0] : nz - 2;
    typename PairOf<T>::type p[NC][4];
    uint32_t row[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) row[q] = (ix[q & 1] * ny + iy[q >> 1]) * nz;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        p[c][q] = *reinterpret_cast<const typename PairOf<T>::type *>(m + c * cstride + row[q] + zc);
    if (iz[1] != zc + 1) {
      // the low corner is the pair's second value in the last cell of a row
      T hi[NC][4];
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) hi[c][q] = m[c * cstride + row[q] + iz[1]];
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[c][q] = iz[0] == zc ? p[c][q].x : p[c][q].y;
          v[c][q | 4] = hi[c][q];
        }
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          v[c][q] = iz[0] == zc ? p[c][q].x : p[c][q].y;
          v[c][q | 4] = p[c][q].y;
        }
    }
  } else if (nz == 1) {
    // both z corners are the one cell: four loads (2^20 particles in no order on
    // 512 x 512 x 1: 23.4 -> 14.8 us, float64 29.7 -> 15.4)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[c][q] = v[c][q | 4] = m[c * cstride + ix[q & 1] * ny + iy[q >> 1]];
  } else {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int o = 0; o < 8; ++o) v[c][o] = m[c * cstride + (ix[o & 1] * ny + iy[(o >> 1) & 1]) * nz + iz[o >> 2]];
  }
}

// Workgroup b of a per-particle kernel takes the particles of block
// (b mod 8) per + b / 8: each XCD walks one contiguous eighth of them, so the
// mesh rows that neighbouring particles share come through one L2.
inline unsigned xcd_blocks(int64_t n, int block, uint32_t &per) {
  per = uint32_t(((n + block - 1) / block + 7) / 8);
  return 8u * per;
}

struct ChunkDesc {
  uint32_t tile, start, count, pad;
};

// The tile table of at most 32768 tile counts (bin.hip): tile starts, scatter
// cursors, chunks per tile and their offsets, totals [particles, chunks, 0]
// and the chunk descriptors.
int tile_table(hipStream_t s, const uint32_t *count, uint32_t K, uint32_t chunk, uint32_t *tstart, uint32_t *cursor,
               uint32_t *nchunk, uint32_t *choff, uint32_t *totals, ChunkDesc *desc, uint32_t groups = 1);

// One simulation as the tile-sort kernels see it.  A batch concatenates its
// simulations: particles [part0, part0 + n) of the positions, tiles
// [tile0, tile0 + t.K) of the tile arrays, cells [cell0, cell0 + M) of the
// meshes, count/scatter workgroups from blk0.
struct SimRef {
  TileGrid t;
  uint32_t tile0, part0, n, cell0, blk0, idx;
};

// A single simulation: the table is one entry held by value.
struct OneSim {
  SimRef s;
  __device__ __forceinline__ const SimRef &tile_sim(uint32_t) const { return s; }
  __device__ __forceinline__ const SimRef &block_sim(uint32_t) const { return s; }
};

// A batch: a device table of B entries, ordered by tile0 and blk0, looked up
// by binary search (the lookups are uniform across a workgroup).
struct SimTable {
  const SimRef *sims;
  int B;
  __device__ __forceinline__ const SimRef &tile_sim(uint32_t tile) const {
    int lo = 0, hi = B - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (sims[mid].tile0 <= tile) lo = mid; else hi = mid - 1;
    }
    return sims[lo];
  }
  __device__ __forceinline__ const SimRef &block_sim(uint32_t blk) const {
    int lo = 0, hi = B - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (sims[mid].blk0 <= blk) lo = mid; else hi = mid - 1;
    }
    return sims[lo];
  }
};

// The result of a tile sort: particles as float4 (x, y, z, global index
// bits) grouped by tile, chunked into runs of at most kChunk particles of one
// tile.  K, n and M are the batch totals.
template <class G>
struct BinsT {
  G g;
  uint32_t K, n, M, maxchunks, chunk;
  bool rel, slabs;
  const float4 *spos;
  const ChunkDesc *desc;
  const uint32_t *nchunk, *choff, *total_chunks;
  // set by a paint of these bins that met a NaN or +-Inf deposit; cleared by
  // the sort
  uint32_t *nonfinite;
};
using Bins = BinsT<OneSim>;
using BatchBins = BinsT<SimTable>;

// A batch of simulations: the host description and the device table.
// Simulations of one mesh shape are contiguous (a "class"), so each class's
// meshes and half spectra form one strided batch for hipFFT.
struct SimClass {
  int nx, ny, nz, first, count;
  uint32_t cell0, half0;
};

struct SimBatch {
  int B = 0;
  bool rel = false;
  uint32_t K = 0, N = 0, M = 0, H = 0, G = 0, maxK = 0, chunk = kChunk, slice = kSlice;
  bool rho_lds = true, slabs = false;
  std::vector<SimRef> host;
  std::vector<SimClass> classes;
  SimRef *dev = nullptr;
};

inline SimRef one_sim(int nx, int ny, int nz, int64_t n) {
  SimRef r;
  r.t = make_tiles(nx, ny, nz);
  r.tile0 = r.part0 = r.cell0 = r.blk0 = r.idx = 0;
  r.n = uint32_t(n);
  return r;
}

int bin_sort(hipStream_t s, int nx, int ny, int nz, const float *pos, int64_t n, uint32_t flags, void *ws,
             size_t ws_bytes, Bins &out, const uint32_t *counts_in = nullptr);
size_t bin_sort_workspace_size(int nx, int ny, int nz, int64_t n, uint32_t flags);
Bins bins_view(int nx, int ny, int nz, int64_t n, uint32_t flags, const void *ws);
template <class G>
int bins_order(hipStream_t s, const BinsT<G> &b, uint32_t *order);
size_t batch_sort_workspace_size(const SimBatch &bt);
size_t batch_paint_workspace_size(const SimBatch &bt, int nc);
int batch_sort(hipStream_t s, const SimBatch &bt, const float *pos, void *ws, size_t ws_bytes, BatchBins &out,
               const uint32_t *counts_in = nullptr);
int zero_u32(hipStream_t s, uint32_t *p, uint32_t n);
int bins_paint(hipStream_t s, const Bins &b, const float *weight, float wscalar, int nc, float *mesh, uint32_t flags,
               void *ws, size_t ws_bytes, const float *wmax_in = nullptr, const FaceCells *faces = nullptr,
               const float *base_mesh = nullptr);
// The potential solves (kspace.hip); faces: the painted mesh's face cells
// kept apart, on the shapes potential_faces_ok accepts, for a one-mesh solve.
bool potential_faces_ok(int nx, int ny, int nz);
int potential_solve(hipStream_t s, int nx, int ny, int nz, int batch, const float *in, void *spec, void *spec2,
                    float *out, float r_split, float scale, const float *scale_dev, uint32_t flags,
                    const FaceCells *faces = nullptr);
int potential_solve_div(hipStream_t s, int nx, int ny, int nz, int batch, const float *g3, size_t chan, float *rho,
                        void *spec, void *spec2, float *out, float r_split, float scale, const float *scale_dev,
                        uint32_t flags);
BatchBins batch_view(const SimBatch &bt, const void *ws);
int batch_paint(hipStream_t s, const SimBatch &bt, const BatchBins &b, const float *weight, int nc, float *mesh,
                void *ws, size_t ws_bytes, const float *wmax_in = nullptr);

// One corner axis of a particle relative to its tile origin: local window
// index (or -1 when the corner is dropped / outside the window) and weight.
struct LAxis {
  int l0, l1;
  float w0, w1;
};

__device__ __forceinline__ LAxis laxis_abs(float x, int origin, int n) {
  LAxis a;
  const float f = floorf(x);
  const float f1 = f + 1.0f;
  a.w0 = 1.0f - fabsf(x - f);
  a.w1 = 1.0f - fabsf(x - f1);
  const int c0 = wrapi(cell_int(f), n);
  a.l0 = c0 - origin;  // the floor cell lies in the tile by construction
  a.l1 = a.l0 + 1;
  return a;
}

// A tile as floats, for the floor cells of its absolute positions: origin,
// length - 1 and mesh edge per axis (exact below 2^22 cells; a longer axis
// gets a NaN origin, which sends every position to the general path).
struct TileFrame {
  float o[3], last[3], n[3];
};

__device__ __forceinline__ float window_edge(int n) { return n <= (1 << 22) ? float(n) : __builtin_nanf(""); }

// Window index (lx * kWin + ly) * kWin + lz of the floor cell f of an absolute
// position that the sort put in this tile.  Nearly all floors lie in the tile
// as they are, some one period away (a particle that left the box), and what
// is left (non-finite, far away) takes the wrap of floor_cell_abs; every path
// gives that cell.  far: set when the last path was taken; otherwise the
// position is finite, at most two periods from the box.
__device__ __forceinline__ uint32_t window_cell(const float f[3], const TileFrame &F, const TileGrid &t, int ox,
                                                int oy, int oz, bool &far) {
  float l[3];
  bool in = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    l[a] = f[a] - F.o[a];
    in = in && __builtin_amdgcn_fmed3f(l[a], 0.0f, F.last[a]) == l[a];
  }
  far = false;
  if (!in) {
    bool one = true;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      if (l[a] < 0.0f) l[a] += F.n[a];
      else if (l[a] > F.last[a]) l[a] -= F.n[a];
      one = one && __builtin_amdgcn_fmed3f(l[a], 0.0f, F.last[a]) == l[a];
    }
    if (!one) {
      far = true;
      l[0] = float(wrapi(cell_int(f[0]), t.nx) - ox);
      l[1] = float(wrapi(cell_int(f[1]), t.ny) - oy);
      l[2] = float(wrapi(cell_int(f[2]), t.nz) - oz);
    }
  }
  return uint32_t(fmaf(l[0], float(kWin * kWin), fmaf(l[1], float(kWin), l[2])));
}

// enmesh corner (painting_utils.py:48-69) mapped into the window; corners
// that land outside [origin, origin + 16] (rounding edge cases) report -1 and
// are deposited by the caller through the overflow path.
__device__ __forceinline__ void lcorner_rel(float p, float o, int n, int origin, int &l, float &w, int &cell,
                                            float &nd) {
  const float L = float(n);
  const float q = floorf(jmod(p + o, L));
  nd = fold_period(p - q, L);
  const bool ok = (q >= 0.0f) && (q < L);
  cell = ok ? int(q) : -1;
  w = ok ? 1.0f - fabsf(nd) : 0.0f;
  if (!ok) {
    l = -2;  // dropped: no deposit at all
    return;
  }
  int d = int(q) - origin;
  if (d < 0) d += n;  // window may wrap past the mesh end
  l = (d >= 0 && d < kWin) ? d : -1;
}

__device__ __forceinline__ int tile_len(int it, int ntile, int n) {
  return (it == ntile - 1) ? n - it * kTile : kTile;
}


// Tile origin of a tile index.
__device__ __forceinline__ void tile_origin(uint32_t tile, const TileGrid &t, int &itx, int &ity, int &itz) {
  const uint32_t txy = t.div_tz.div(tile);
  itz = int(tile - txy * uint32_t(t.tz));
  itx = int(t.div_ty.div(txy));
  ity = int(txy - uint32_t(itx) * uint32_t(t.ty));
}

__device__ __forceinline__ TileFrame tile_frame(const TileGrid &t, int itx, int ity, int itz) {
  TileFrame F;
  const int n[3] = {t.nx, t.ny, t.nz}, it[3] = {itx, ity, itz}, T[3] = {t.tx, t.ty, t.tz};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    F.n[a] = window_edge(n[a]);
    F.o[a] = float(it[a] * kTile) + 0.0f * F.n[a];
    F.last[a] = float(tile_len(it[a], T[a], n[a]) - 1);
  }
  return F;
}

}  // namespace jpm
