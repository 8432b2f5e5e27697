// Internal device-side descriptors shared by the kernels (kernels.hip) and the
// host engine (engine.cpp).  Not part of the public ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace ddx {

constexpr int NF = 19;
// the last six are the FWI accumulators (displacement, dt x velocity increment)
enum : int { VX = 0, VY, VZ, SXX, SYY, SZZ, SXY, SXZ, SYZ, SAU, VXP, VYP, VZP, UX, UY, UZ, VXRT, VYRT, VZRT };
enum : int { PURE_FORWARD = 0, RTM_FORWARD = 1, RTM_BACKWARD = 2, RTM_REVERSE = 3, FWI = 4 };
constexpr int kModes = 5;
// Tap n of the staggered first derivative of half order `half`
// (GEO/jarvis_device_geometry_bones.hpp:29-49, cu_cal_diff_coeff); 0 past it.
constexpr float fd_tap(int half, int n) {
  if (n >= half) return 0.f;
  double a1 = 1, a2 = 1, a3 = 1;
  for (int i = 0; i < half; i++) {
    if (i != n) a1 = a1 * (2 * i + 1) * (2 * i + 1);
    if (i < n) a2 = a2 * ((2 * n + 1) * (2 * n + 1) - (2 * i + 1) * (2 * i + 1));
    if (i > n) a3 = a3 * ((2 * i + 1) * (2 * i + 1) - (2 * n + 1) * (2 * n + 1));
  }
  return (float)((n & 1 ? -a1 : a1) / ((2 * n + 1) * a2 * a3));
}
// Wavefield storage formats (fields, CPML memory variables, VOWR store): FP32,
// or 16-bit codes of the value times a power-of-two scale per field class.
enum : int { STORE_F32 = 0, STORE_F16 = 1, STORE_BF16 = 2, STORE_BFP16 = 3 };
// STORE_BFP16 (VOWR store only): 16-bit codes (sign, 3-bit exponent, 12-bit
// mantissa) relative to one exponent shared by kRingBlock consecutive
// entries of a slice; each ring box starts on a run.
constexpr int kRingBlock = 16;
// the RTM modes update sau in the physical region
__host__ __device__ constexpr bool rtm_mode(int m) { return m == RTM_FORWARD || m == RTM_BACKWARD || m == RTM_REVERSE; }

// Threads per block of every grid-mapped kernel; the physical-region kernels
// use a 64 (x) by 4 (y) tile so one wavefront covers one contiguous x row.
constexpr int kBlock = 256;
constexpr int kTileX = 64;
constexpr int kTileY = 4;
// Work split of the CPML kernels (a context's pml_cz):
//   kPmlPairs: kBlock consecutive pairs of x cells of a slab
//     plane per block;
//   1, 2, 4, 8: kBlock consecutive cells of a slab plane per block, cz
//     planes per thread, the x and y stencil taps read through the caches;
//   kPmlTiled + p (p = 2, 4, 8): a tile of pml_tile_x(ni) x (kBlock /
//     pml_tile_x(ni)) plane cells per block, staged in LDS with its halo,
//     p planes marched per block (FP32 storage only).
constexpr int kPmlPairs = 0;
constexpr int kPmlTiled = 16;
// The split inside half steps that run as one launch.  FP32 has one cell per
// thread there: pairs take 120 registers where the bricks and one-cell CPML
// blocks take 85 to 110, and such grids live in the last-level cache, so the
// wavefronts in flight count for more than the loads saved (100^3 with 10
// layers: 75 us per step with one cell, 99 with pairs; 64^3 with 20: 51 and
// 53).  The 16-bit bricks take 136 registers or more anyway, and their pairs
// are ahead everywhere.
__host__ __device__ constexpr int pml_whole(int fmt) { return fmt == STORE_F32 ? 1 : kPmlPairs; }
__host__ __device__ constexpr bool pml_tiled(int cz) { return cz > kPmlTiled; }
__host__ __device__ constexpr int pml_planes(int cz) {
  return cz > kPmlTiled ? cz - kPmlTiled : cz == kPmlPairs ? 1 : cz;
}
// Tile width: the whole slab row when it is at most 64 cells (the 18-cell
// x slabs), else 64 (one wavefront per row).
__host__ __device__ constexpr int pml_tile_x(int ni) { return ni < 4 ? 4 : ni > 64 ? 64 : ni; }
// Plane tiles of one slab plane (ip: elements of a row of memory variables).
__host__ __device__ inline int pml_plane_tiles(int ni, int nj, int ip, int cz) {
  if (cz == kPmlPairs) return ((ip >> 1) * nj + kBlock - 1) / kBlock;
  if (!pml_tiled(cz)) return (ni * nj + kBlock - 1) / kBlock;
  const int tx = pml_tile_x(ni), ty = kBlock / tx;
  return ((ni + tx - 1) / tx) * ((nj + ty - 1) / ty);
}
// blocks of one CPML slab: plane tiles times chunks of pml_planes(cz) planes
inline int pml_blocks(int ni, int nj, int nk, int ip, int cz) {
  const int p = pml_planes(cz);
  return pml_plane_tiles(ni, nj, ip, cz) * ((nk + p - 1) / p);
}

// One physical region (gridphy) of the whole grid, all subdomains of the
// decomposition in it.  Field pointers address extended cell (0,0,0);
// strides sy, sz in elements.  Field elements are of the context's storage
// format.
struct PhyDesc {
  void *f[NF];
  const float *dtr;  // dt / rho, per cell
  const float *lam;
  const float *mu;
  long sy, sz;
  int ox, oy, oz;    // gridphy origin in extended coordinates
  int nx, ny, nz;    // gridphy size
  int R;             // VOWR ring width
  int tiles_x, tiles_y;
  float dt;          // time step (FWI accumulators)
  int io;            // member of a fused launch (StepIO)
  int blk0;
};

// One CPML slab of the whole grid (the reference's top/bottom, front/back,
// right/left PML frames, BASE/fdtd3d_base_6_pml_meat.hpp:29-93).
struct SlabDesc {
  void *f[NF];
  const float *dtr;
  const float *lam;
  const float *mu;
  long sy, sz;
  int i0, j0, k0, ni, nj, nk;        // box in extended coordinates
  int axes;                          // damped axes: 1 x, 2 y, 4 z
  int xlo, xhi, ylo, yhi, zlo, zhi;  // a cell is in an axis' damping range iff c < lo || c >= hi
  // rows of memory variables and coefficients hold ip elements, an even
  // number, cell i0 at element sh (0 or 1): pairs of elements 2q, 2q + 1 are
  // pairs of cells whose first lies on an even element of the fields' storage
  int ip, sh;
  unsigned mni, mnp;                 // (2^32 - 1) / ni, / (ip / 2), rounded down
  void *psi;                         // [6 * naxes][nk][nj][ip] memory variables (storage format)
  const float *coef;                 // [naxes][nk][nj][ip][4]: a, b, a_half, b_half per axis and cell
  float rdx, rdy, rdz;               // 1 / spacing
  int io;                            // member of a fused launch (StepIO)
  int blk0;
};

// XCD-partitioned block order of the CPML kernels.  Every slab is split
// into 8 parts, one per XCD: by z chunks when the slab is deeper (z) than it
// is long in y, else by plane tiles (kBlock cells of a plane).  Each XCD
// walks its parts chunk by chunk, so a block's z and y stencil taps were
// loaded into the XCD's own L2 by the blocks just before it.  Block b runs
// on XCD b % 8 as that XCD's (b / 8)-th block; a piece covers chunks
// [p0, p0 + n / tcnt) times tiles [t0, t0 + tcnt) of slab `desc`, from
// the XCD's block lstart on.
struct PmlPiece {
  int desc, lstart, p0, t0, tcnt;
};
struct PmlOrder {
  const PmlPiece *pieces = nullptr;  // nullptr: the group-interleaved launch order
  int xoff[9] = {0};                 // pieces of XCD x: [xoff[x], xoff[x + 1])
  int xn[8] = {0};                   // blocks of XCD x
  int grid = 0;                      // 8 x the largest xn
};

// One box copied between a field and a contiguous buffer (the VOWR boundary
// store).
struct CopyDesc {
  void *field;
  long sy, sz;
  int i0, j0, k0, ni, nj, nk;
  // the box is buffer elements buf_off .. , x fastest
  long buf_off;
  int cls;   // field class (0 velocity, 1 stress): the scale of a converting copy
  int fid;   // ring field index (0..9): the per-slice scale of a converting copy
  int io;    // member of a fused launch (StepIO)
  int blk0;
};
// How a boundary store holds its values (RING_F16, RING_BF16: converted, scaled).
enum : int { RING_COPY4, RING_COPY2, RING_F16, RING_BF16, RING_BFP };

// Imaging over one subdomain's gridphy.
struct ImgDesc {
  const void *b[6];   // backward (source) set: vx vy vz vxp vyp vzp
  const void *r[6];   // reverse (receiver) set
  long sy, sz;
  int ox, oy, oz, nx, ny, nz;
  void *img[9];       // Ip Ipp Ips Isp Iss and 4 Laplacians (float or double)
  int blk0;
};

// Brick of the z-blocked physical-region kernels: a block of tx*ty threads
// owns (px*tx) x (ty*cy) columns and kz consecutive planes (kz per thread);
// px = 2: every thread updates two neighbouring x cells; xl = 1: one cell
// per thread with the x arm taken from neighbouring lanes (tx = 64); xl = 2:
// that, and the y arm from LDS (cy = 1); kz == 0 selects the
// one-plane-per-block kernels.
struct Tiling {
  int tx, ty, cy, kz;
  int px = 1;
  int xl = 0;
  int whole = 1;  // the half step may run as one launch with the CPML cells (whole_half in engine.cpp)
};
// instantiated brick shapes (tx, ty, cy, kz) for a storage format
bool tiling_supported(const Tiling &t, int fmt = STORE_F32);
// the z-blocked shapes of a storage format (one-cell, paired, lane-exchange
// and y arm from LDS: xl = 2); returns how many there are and writes up to
// max of them
int tiling_list(int fmt, Tiling *out, int max);
// cy == 0 selects the LDS-tiled 2.5D kernels (tx = 64, ty = 8, kz planes per
// block).
inline int tiling_blocks(const Tiling &t, int nx, int ny, int nz) {
  const int rows = t.cy == 0 ? t.ty : t.ty * t.cy;
  const int cols = t.tx * t.px;
  return ((nx + cols - 1) / cols) * ((ny + rows - 1) / rows) * ((nz + t.kz - 1) / t.kz);
}

// One member of a fused batch of modelling shots: its source cell and
// wavelet, its receivers and seismograms, and the batch step at which its
// shot began (its time index is the batch step minus join).
struct MemberIO {
  void *sxx, *syy, *szz;  // source subdomain's fields; nullptr: the shot is outside gridext
  long src_off;
  int src_x, src_y, src_z;  // the source cell in the whole grid's extended coordinates (-1: none)
  const float *wavelet;
  int src_mode;
  float ss;               // stress-class scale (16-bit formats)
  void *const *vptr;      // receivers: per subdomain vx, vy, vz
  const int *rsub;
  const long *roff;
  int nrec;
  float *seis;            // [3][nrec][ntime]
  float inv_sv;
  float sv;               // velocity-class scale (receiver injection of the 16-bit formats)
  int join, ntime;
  int rev;                // 0: time index = batch step - join; 1: join - batch step (a reverse loop)
  // the member's boundary store (k_rev_vel, k_rev_stress)
  const float *store;     // [ring_slices][ring_slice], by ring_kind
  long ring_slice, ring_runs;
  int ring_slices, ring_kind;
  float ring_sv, ring_ss;         // class scales of a converted store
  const int *store_exp;           // per-slice scales instead (nullptr: the class scales)
  const signed char *store_bexp;  // run exponents of a block-scaled store
  int blk0;               // first block of this member's receivers
};

// Sources and receivers of a time step of the members of a launch (a shot on
// its own is the one member); a descriptor's member is its `io`.  Time index:
// gs, or *gsp when set (see launch_source_batch).  io null: no sources.
// nblk: receiver blocks (0: the step samples none here).
struct StepIO {
  const MemberIO *io = nullptr;
  const int *starts = nullptr;
  int n = 0, nblk = 0;
  int gs = 0;
  const int *gsp = nullptr;
  float sign = 1.f;  // of the sources
};

// A half step of the physical region and the CPML cells in one launch.
struct HalfStep {
  const PhyDesc *phy;
  const int *pstarts;
  int np, nphy;
  const SlabDesc *slabs;
  const int *sstarts;
  int ns, npml;
  float dx, dy, dz, sc;  // sc: as sign / dt of the separate kernels
  float sx, sy, sz;      // sc over dx, dy, dz
  int grp, pgrp;
  int cached;            // the bricks' own cells go through ordinary accesses (cached_limit in engine.cpp)
};
// The backward bricks of half a reverse iteration (sc, sx, sy, sz as HalfStep).
struct BackBricks {
  const PhyDesc *phy;
  const int *starts;
  int n, nblk;
  float sc, sx, sy, sz;
};
// Boundary-store boxes to inject, of the members of a StepIO.
struct RingBoxes {
  const CopyDesc *d;
  const int *starts;
  int n, nblk;
};

// ---- launchers (kernels.hip) ----
// fmt: storage format; the 16-bit formats fold their scale ratios into
// `sign` (velocity: sv/ss), `dt` (stress: ss/sv) and `rv` (CPML velocity:
// sv/ss); ss, sv, inv_sv: the class scales themselves.
// The physical-region launchers return false, launching nothing, when no
// kernel exists for the brick shape, storage format and mode.  grp: block
// order of the z-blocked bricks (0 contiguous per XCD, else groups of grp).
bool launch_vel_phy(const Tiling &t, int mode, int fmt, const PhyDesc *d, const int *starts, int n, int nblk,
                    float dx, float dy, float dz, float sign, int grp, hipStream_t st);
bool launch_stress_phy(const Tiling &t, int mode, int fmt, const PhyDesc *d, const int *starts, int n, int nblk,
                       float dx, float dy, float dz, float dt, int grp, hipStream_t st);
// One launch for a half step (CPML split pml_whole, group-interleaved orders); false,
// launching nothing, when no such kernel exists for the brick shape, format
// and mode (the backward mode has no CPML cells).  The stress step also adds
// the members' sources and samples their receivers (io).
bool whole_shape(const Tiling &t, int fmt);  // the shapes they exist for
bool launch_vel_all(const Tiling &t, int mode, int fmt, const HalfStep &a, hipStream_t st);
bool launch_stress_all(const Tiling &t, int mode, int fmt, const HalfStep &a, const StepIO &io, hipStream_t st);
// The halves of a reverse iteration, one launch each, in the shapes of
// whole_shape: the reverse set's half step a, the backward set's bricks q (of
// the same shape; stress next to the velocity half step and the other way
// round) and boxes rb; io: the members, their sources subtracted by the
// backward stress.  False, launching nothing, as launch_vel_all.
bool launch_rev_vel(const Tiling &t, int fmt, const HalfStep &a, const BackBricks &q, const StepIO &io,
                    const RingBoxes &rb, hipStream_t st);
bool launch_rev_stress(const Tiling &t, int fmt, const HalfStep &a, const BackBricks &q, const StepIO &io,
                       const RingBoxes &rb, hipStream_t st);
// grp: blocks per XCD group of the group-interleaved block order (0: launch order)
// ord (nullable): the XCD-partitioned block order of the table; without it
// (or with ord->pieces null) the blocks follow the table's own order.
void launch_vel_pml(int cz, int fmt, const SlabDesc *d, const int *starts, int n, int nblk, float dx, float dy,
                    float dz, float rv, int grp, const PmlOrder *ord, hipStream_t st);
void launch_stress_pml(int cz, int with_sau, int fmt, const SlabDesc *d, const int *starts, int n, int nblk,
                       float dx, float dy, float dz, float dt, int grp, const PmlOrder *ord, hipStream_t st);
// dir +1: field -> buffer (VOWR save); -1: buffer -> field (VOWR inject);
// esz: element size in bytes (4 or 2)
void launch_copy(int dir, int esz, const CopyDesc *d, const int *starts, int n, int nblk, void *buf, hipStream_t st);
// Converting copy between FP32 fields and a 16-bit buffer (fmt FP16 or
// BF16): saved values are scaled by sc[cls] and rounded; injected ones
// widened and scaled by 1 / sc[cls].
void launch_copy_conv(int dir, int fmt, const CopyDesc *d, const int *starts, int n, int nblk, void *buf, float sc_v,
                      float sc_s, hipStream_t st);
// Per-slice, per-field scaling of a 16-bit VOWR store over FP32 fields:
// launch_ring_max accumulates each field's largest |value| of the boxes into
// maxbits[fid] (float bits; the array starts at zero), launch_ring_exp turns
// them into the slice's scale exponents exps[0..nf) (e = 15 - the binary
// exponent of the maximum, clamped to [-100, 100]; 0 for an all-zero field)
// and clears maxbits again, launch_copy_dyn copies with scale 2^exps[fid]
// (dir +1 save, -1 inject).
void launch_ring_max(const CopyDesc *d, const int *starts, int n, int nblk, unsigned *maxbits, hipStream_t st);
void launch_ring_exp(unsigned *maxbits, int *exps, int nf, hipStream_t st);
void launch_copy_dyn(int dir, int fmt, const CopyDesc *d, const int *starts, int n, int nblk, void *buf,
                     const int *exps, hipStream_t st);
// The block-scaled VOWR store (STORE_BFP16): dir +1 saves the boxes of a
// save table (whole boxes on whole runs) into the slice buf and writes the
// runs' exponents to bexp, dir -1 injects the boxes of any ring table.
void launch_ring_bfp(int dir, const CopyDesc *d, const int *starts, int n, int nblk, void *buf, signed char *bexp,
                     hipStream_t st);
// itp (nullable): read the time index from this device int instead of it
void launch_source(int fmt, void *sxx, void *syy, void *szz, long off, const float *wavelet, int it, float sign,
                   int src_mode, float ss, const int *itp, hipStream_t st);
void launch_advance(int *p, int delta, hipStream_t st);
// Sources and receiver samples of every member of a fused batch at batch
// step gs, or *gsp when gsp is set (a device step counter: launches
// captured once in a graph and replayed every step); members outside
// [join, join + ntime) do nothing; nblk: receiver blocks over all members
// (starts[q] = io[q].blk0).
void launch_source_batch(int fmt, const MemberIO *io, int n, int gs, const int *gsp, hipStream_t st,
                         float sign = 1.f);
// Observed data of every member of a fused RTM batch injected at its
// receivers (io[q].vptr: the reverse set) at batch step gs.
void launch_inject_batch(int fmt, const MemberIO *io, const int *starts, int n, int nblk, int gs, hipStream_t st);
void launch_recv_batch(int fmt, const StepIO &io, hipStream_t st);
void launch_set_int(int *p, int v, hipStream_t st);
void launch_recv_sample(int fmt, void *const *vptr, const int *rsub, const long *roff, int nrec, int it, int ntime,
                        float *seis, float inv_sv, const int *itp, hipStream_t st);
void launch_recv_inject(int fmt, void *const *vptr, const int *rsub, const long *roff, int nrec, int it, int ntime,
                        const float *seis, float sv, hipStream_t st);
// v += obs - syn at the receivers (FWI adjoint source; FP32 storage)
void launch_recv_residual(void *const *vptr, const int *rsub, const long *roff, int nrec, int it, int ntime,
                          const float *obs, const float *syn, hipStream_t st);
void launch_image(int fp64, int fmt, const ImgDesc *d, const int *starts, int n, int nblk, float inv_sv, bool cached,
                  hipStream_t st);
void launch_image_post(int fp64, const ImgDesc *d, const int *starts, int n, int nblk, hipStream_t st);

// Sets *flag to 1 when any of the n elements of a field (storage format
// fmt) is infinite or NaN; leaves it alone otherwise.
void launch_nonfinite(int fmt, const void *field, long n, int *flag, hipStream_t st);

}  // namespace ddx
