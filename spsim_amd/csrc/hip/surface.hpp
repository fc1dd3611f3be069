// Structure factor of a smooth detector list by interpolation over the
// detector surface (surface.hip): descriptions shared with the batched plans.
#pragma once

#include "sf_kernels.hpp"

namespace spsim {

constexpr int kSurfDeg = 16;         // sample lines per axis of the list's surface (degree kSurfDeg - 1)
constexpr int kSurfLines = 31;       // lines per axis on which its slopes are measured
constexpr int kSurfMinSide = 64;     // shortest detector side that is tried
constexpr int kSurfMinNodes = 16;    // fewest and most nodes per axis, a multiple of 4
constexpr int kSurfMaxNodes = 512;
constexpr int kSurfMaxSplits = 128;  // atom ranges per node tile
constexpr int kSurfListBlocks = 448;  // with the atom blocks, two workgroups per CU
constexpr int kSurfAtomBlocks = 64;  // per molecule

// What one workgroup of the scan saw: the largest |q - surface| (list blocks), or
// the largest |r - r0|^2 and the range of B (atom blocks).
struct SurfRecord {
  double dev;
  double r2;
  float bmin, bmax;
  int bad;  // some value was not finite
  int pad;
};

// Steepest slopes of the surface along an axis: the largest |dq/du| and |dq_k/du|
// on the lines u = cos(pi j / (kSurfLines - 1)).
struct SurfSlopes {
  float all[kSurfLines], part[3][kSurfLines];
};

// The list's surface: Chebyshev coefficients of a polynomial through q at
// kSurfDeg x kSurfDeg pixels, in the pixel coordinates u, v in [-1, 1]
// (coef[n][m][k]: T_n(v) T_m(u), component k), and its slopes.
struct SurfFit {
  double coef[kSurfDeg][kSurfDeg][3];
  SurfSlopes slope_x, slope_y;
  float s2max;  // largest s^2 = (|q| 1e-10 / 2)^2 seen
  float normal[3];  // unit normal of the surface's middle
  int sym;          // 2: mirror- and transpose-symmetric, 1: mirror-symmetric, 0
};

// Nodes of one axis: u_i = asin(a cos t_i) / asin(a), t_i = (2 i + 1) pi / (2 n);
// n = 0: the axis needs more than kSurfMaxNodes.
struct SurfAxis {
  int n;
  double a, asin_a;
};

// One detector shape at one node count: node q [ax.n][ay.n][3], the
// interpolation weights, node-major (tx [ax.n][nx], ty [ay.n][ny]), and the same in
// FP32 with their derivatives in u and v.
struct SurfShape {
  SurfAxis ax, ay;
  double *nodes, *tx, *ty;
  float2 *tx32, *ty32;
};

// One cell of a molecule that is summed by cells: its atoms are `count` records
// from `start`, its sums `ranges` partial ones from `range0`.
struct SurfCell {
  double centre[3];
  int start, count, range0, ranges;
};

// Nodes at which a cell's sums are formed, and the weights that take them to the
// nodes fx x fy of the whole pattern: wx [ax.n][fx.n], wy [ay.n][fy.n].
struct SurfCoarse {
  SurfAxis ax, ay, fx, fy;
  double *nodes, *wx, *wy;
};

// A molecule summed by cells: g x g x gz boxes of the cube of half edge
// `extent` (g = 0: not). f and n are [range][ax.n][ay.n], tf and tn [cell][ay.n][fx.n].
struct SurfCells {
  int g, gz, per_lane, tiles;
  double extent;
  SurfCoarse co;
  unsigned short *id;  // of every atom, its cell
  int *order;          // the atoms by cell
  void *sorted;        // and their records
  SurfCell *cells;
  spsim_hip_segment *segs;  // [cell][nsegs], of the sorted records
  int *range_cell;          // cell of a range, or -1
  double2 *f, *tf;
  float2 *n, *tn;
};

// One pattern. The node sums f (F) and n (its derivative along the normal) are
// [ax.n][ay.n]; t64 (F) and t32 (dF/du, n) are fields along the detector's rows,
// [ay.n][nx].
struct SurfJob {
  int ok;
  int nx, ny;
  SurfShape sh;
  const spsim_hip_atom *atoms;
  const float *atom_b;
  const spsim_hip_segment *segs;
  int nsegs, natoms;
  int has_rot;
  double rot[9];
  double r0[3];  // subtracted from every atom
  float normal[3];
  int per_lane, tiles, splits;  // node tiles of 256 per_lane nodes (8: octants), atom ranges per tile
  double2 *f;
  float2 *n;
  void *prep;  // atom records of the node sums [natoms]
  double2 *slot_f;  // partial sums [tile * splits + split][256 per_lane]
  float2 *slot_n;
  double2 *t64;
  float4 *t32;
  long long pattern;  // index of the outputs
  int shape, coarse;  // of a plan
  SurfCells c;
};

struct SurfItem {
  int job, tile, split, pad;
};

// Everything about the molecule that the choice of nodes depends on.
struct SurfMol {
  double radius;     // largest |r - r0|
  double dev;        // largest |q - surface| of the list
  float b_smooth;    // largest Gaussian coefficient of the terms (form factor + B), A^2
  float weakest;     // smallest ratio of a term's amplitude at s2max to that at 0
  int bad;
  int ordered;       // the species' segments follow each other and are no more than species
};

// Host sizes only: is the pattern large enough to look at its list?
bool surf_worth(long long nx, long long ny, long long natoms, long long min_terms);

// One pattern on the device alone (no host decision). On return *ok_flag points
// to a device int that is non-zero when the outputs were written and zero when
// the list or molecule is not smooth enough, in which case nothing was.
size_t surf_single_bytes(int nx, int ny, int natoms, int nsegs, bool spectrum);
// sp: a wavelength spectrum, or null.
int launch_surface(const PatternLaunch &a, int nx, int ny, const Spectrum *sp, int cus, void *ws, const int **ok_flag,
                   hipStream_t s);

// ---- adjoint (adjoint.hip) ----

constexpr int kSurfAtomsPerLane = 2;

// A run of packed atoms of one species, at most 256 kSurfAtomsPerLane.
struct SurfAtomTile {
  int start, count, species, pad;
};

// Sums of the gradients over the detector a.hkl with the forward's a.F and
// g = dL/dI, by way of the nodes: partial[split][atom] as adjoint_kernel leaves
// them, `splits` node ranges per tile. *ok_flag as for launch_surface.
size_t surf_adjoint_bytes(int nx, int ny, int natoms);
int launch_surface_adjoint(const PatternLaunch &a, const float *gI, int nx, int ny, const SurfAtomTile *tiles,
                           int ntiles, int splits, bool want_b, double4 *partial, int cus, void *ws,
                           const int **ok_flag, hipStream_t s);

// ---- plans that decide on the host (batch.hip, nufft.hip) ----

// What the host reads of a list, and of a molecule seen on it.
struct SurfHead {
  SurfSlopes slope_x, slope_y;
  float s2max, normal[3];
  int sym, pad;
};
struct SurfDigest {
  SurfMol mol;
  double centre[3];
};

// A list and its patterns. Pattern p shows molecule pattern_mol[p] (null:
// molecule p, or 0 when there is only one) under the matrix rot9 + 9 p (null:
// none). All pointers but h_mols, pattern_mol, rot9 and limit are device memory;
// d_mols is null for one molecule h_mols[0].
struct SurfInput {
  const float *hkl;
  int nx, ny;
  const spsim_hip_atom *atoms;
  const float *atom_b;
  const spsim_hip_segment *segs;
  const MolInfo *d_mols, *h_mols;
  int nmol, npatterns;
  const int *pattern_mol;
  const double *rot9;
  const float *ff;
  float b_global;
  int cus;
  const double *limit;  // per molecule, cost above which its patterns are left; null: of the direct sum
};

// The scan's device memory (which a plan keeps using) and its digest: a SurfHead
// and a SurfDigest per molecule, for the host to copy.
size_t surf_scan_bytes(int nx, int ny, int nmol);
constexpr size_t surf_digest_bytes(int nmol) { return sizeof(SurfHead) + sizeof(SurfDigest) * (size_t)nmol; }
int surf_scan(const SurfInput &in, void *scan, void *digest, hipStream_t s);

struct SurfPlan;

// The patterns that are smooth enough and cheaper than in.limit, from the host
// copy of a digest; null when there is none. No device work.
SurfPlan *surf_plan_choose(const SurfInput &in, const void *digest);
// Device memory of its own that the plan needs, and the upload of its tables
// there. The plan has to outlast the upload: wait for s here, or synchronise it
// before surf_plan_destroy.
size_t surf_plan_bytes(const SurfPlan *p);
int surf_plan_bind(SurfPlan *p, const void *scan, void *mem, hipStream_t s, bool wait);

// All of it, in device memory that the plan owns. *out is null when no pattern
// is taken. Synchronises.
int surf_plan_create(const SurfInput &in, SurfPlan **out);
// Whether the plan takes pattern p.
bool surf_plan_takes(const SurfPlan *p, int pattern);
// Writes the outputs of the patterns it takes.
int surf_plan_run(const SurfPlan *p, float2 *F, float *I, hipStream_t s);
void surf_plan_destroy(SurfPlan *p);

}  // namespace spsim
