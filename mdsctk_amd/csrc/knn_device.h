// Internal interface between the C-ABI layer (api.cpp) and the gfx950
// kernels (knn_kernels.hip).  Not installed; include/mdsctk_knn.h is the
// public surface.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace mdsctk {

constexpr int kTile = 32;  // frames per MFMA tile edge (v_mfma_*_32x32xK)
// Contraction workgroup: one wave per 32x32 (ref x fit) frame tile,
// 2 reference tiles x contract_fit_tiles(prec) fit tiles.
constexpr int kRefTilesPerWG = 2;
// Frame sets are padded to a multiple of this many tiles.
constexpr int kTileAlign = 4;
// Symmetric self query: capacity of each frame's mirrored list (the scores
// it receives as the reference side of a pair), and the stride of the
// landmark pass (every kLandmarkStride-th reference tile pair).
constexpr int kMirrorCap = 8192;
constexpr int kLandmarkStride = 128;

enum Prec : int { kFP32 = 0, kBF16 = 1, kFP16 = 2, kExact = 3 };

// What a frame is and which distance the engine ranks by.
//   kMetricRMSD         frames of atoms: optimal-superposition RMSD (knn_rms)
//   kMetricEuclidean    data vectors: Euclidean distance (knn_data)
//   kMetricCorrelation  data vectors: correlation distance sqrt((1-r)/2)
//                       (knn_data -c)
// Data vectors run through the same contraction as frames with the QCP
// step replaced by the --nofit trace: a vector of length V is laid out as
// ceil(V/3) "atoms" of 3 values with unit masses, uncentred, so that the
// trace of the 3x3 block is the dot product.
enum Metric : int { kMetricRMSD = 0, kMetricEuclidean = 1, kMetricCorrelation = 2 };

// Atoms per operand K-group: split forms hold 16 atoms (one 32x32x16 MFMA
// step) per group, FP32 holds 8 atoms (four 32x32x2 MFMA steps).
inline int group_atoms(int prec) { return prec == kFP32 ? 8 : 16; }
// The split forms' K-loop walks K-groups four at a time (its four stage
// buffers), so their operand holds a multiple of four groups (the padding
// atoms are zero and contribute nothing).
constexpr int kSplitGroupAlign = 4;
inline int operand_groups(int prec, int natoms) {
  const int ga = group_atoms(prec);
  const int g = (natoms + ga - 1) / ga;
  return prec == kFP32 ? g : (g + kSplitGroupAlign - 1) / kSplitGroupAlign * kSplitGroupAlign;
}
// 16-byte operand blocks of 64 lanes per (tile, K-group): 3 planes x parts.
inline int blocks_per_group(int prec) { return prec == kFP32 ? 3 : 6; }
// K-groups of zero slack after a frame set's operand: the contraction's
// copy pipeline reads up to four groups past the end of the last tile.
constexpr int kOperandTailGroups = 4;

// A frame set resident in HBM.  Row counts are padded to a multiple of
// kTileAlign*kTile (the contraction walks reference tiles in pairs and fit
// tiles in fours); padded rows are zero.
struct DevFrames {
  int64_t n = 0;        // real frames
  int natoms = 0;
  int n_tiles = 0;      // padded tile count (multiple of kTileAlign)
  int cap_tiles = 0;    // tiles the derived arrays are allocated for (>= n_tiles)
  int n_groups = 0;     // operand K-groups
  int prec = kFP32;
  float* xyz = nullptr;   // [n][natoms][3] as given (nm)
  double* cen = nullptr;  // [n_tiles*32][3] FP64 mass-weighted centroid
  double* G = nullptr;    // [n_tiles*32] sum w |x-c|^2, FP64
  double* Gt = nullptr;   // [n_tiles*32] same sum over the rounded operand
  uint4* op = nullptr;    // contraction operand, fragment-major (see operand_kernel)
  bool owns_xyz = true;
  // data vectors only: the FP64 vectors [n][vdim] the exact scores use and,
  // for the correlation metric, [n][2] (mean, sample standard deviation)
  int vdim = 0;
  double* x64 = nullptr;
  double* aux = nullptr;
  // resident set only: one device double, max Gt over the set (the window's
  // reference term), computed once when the set is made resident
  double* gmax = nullptr;
  // resident set of a dithered split form only: its operand and G~ in the
  // query-side scaling, which a self query uses as its query operand
  uint4* op_q = nullptr;
  double* Gt_q = nullptr;
  // frames of fitted RMSD scores: each frame's principal axes, [rows][9],
  // written by the prep pass when it builds operands in those axes
  double* rot = nullptr;
};

// The resident set seen as a query set (self query): the query-side operand
// where the set has one.
inline DevFrames query_view(const DevFrames& ref) {
  DevFrames v = ref;
  if (ref.op_q) {
    v.op = ref.op_q;
    v.Gt = ref.Gt_q;
  }
  return v;
}

struct DevWeights {
  int natoms = 0;
  float* w = nullptr;   // masses
  float* sw = nullptr;  // sqrt(mass)
  // Output distance = out_scale * sqrt(s / W): for frames W is the sum of
  // masses and out_scale 10 (nm to Angstrom); for data vectors W is 1
  // (Euclidean) or 4 (correlation, s = 2(1-r)) and out_scale 1.
  double W = 0;
  double out_scale = 10.0;
  int metric = kMetricRMSD;
};

// Per-query candidate lists written by the contraction kernel.
struct Lists {
  int nl = 0;          // lists per query
  int cap = 0;         // entries per list
  uint2* ent = nullptr;       // [n_fit][nl][cap] (float key bits, ref index)
  int* cnt = nullptr;         // [n_fit][nl]
  float* ovf = nullptr;       // [n_fit][nl] smallest key dropped on overflow
  unsigned* thr = nullptr;    // [n_fit] shared threshold (float bits)
};

// What a query's kernels count: one small block, read back in one copy.
struct QuerySummary {
  int n_cand;     // candidates re-scored
  int n_flagged;  // rows the merge could not certify
  unsigned long long mirrored, mirrored_max;  // symmetric self query only
};

// The symmetric self query's second list per frame: the scores a frame
// receives as the reference side of a pair contracted only the other way
// round ([n][cap] entries, counters, smallest key dropped past cap).
struct Mirror {
  uint2* ent = nullptr;
  int* cnt = nullptr;
  float* ovf = nullptr;
  int cap = 0;
};

// ---- the tile filter (filter_kernels.hip): a proven test of which (fit
// block, reference pair) tiles of a fitted query can hold a pair below the
// thresholds, from one BF16 product of the frames' deviations from a mean
// structure.

// Extra operand slots at the end of each segment (the rank-one terms), and
// frames averaged into the mean structure.
constexpr int kFilterExtra = 12;
constexpr int kFilterSamples = 64;
// Fit tiles per filter block, and the smallest self query that takes it.
constexpr int kFilterFitTiles = 4;
constexpr int64_t kFilterMinFrames = 4096;
// Cross queries: resident frames (and frames x atoms) from which the set is
// ordered, query frames in all from which that is worth it, and the smallest
// query that takes the ordered form.  Measured at 100000 x 500 resident
// frames: ordering takes 4.6 ms and saves 3.8 ms per 4096 query frames, so it
// is even after about 5000 frames, whatever the size of the set (both grow
// with it); a query of one or two fit blocks would spend the saving on the
// extra launches.
constexpr int64_t kCrossMinRef = 8192;
constexpr int64_t kCrossMinWork = 1 << 22;
constexpr int64_t kCrossMinSeen = 8192;
constexpr int64_t kCrossMinFit = 256;
// Cells the rows are sorted into (13 bits of the sort key, above 19 bits of
// the distance).
constexpr int kFilterMaxCells = 8000;
// The ball test takes a self query's rows one by one up to this many frames
// (a contraction of 1/64 of its pairs), the middles of 64 beyond, where 64
// frames lie closer together and the rows would cost what they save.  30000 x
// 150, states: filter 1.60 ms without the test, 1.55 + .07 ms of test by
// middles, .59 + .27 by rows (one basin: .3 ms of 13 in vain); 200000 x 1000
// by middles: 91 -> 31 + 1.1 ms, where rows would take some 25.
constexpr int64_t kBallRowsMax = 65536;
constexpr int kFilterDistBits = 19;

// Rows up to which the merge takes 1024 threads a row.
constexpr int64_t kMergeWideRows = 256;

// How a frame's atoms are laid out: one or two segments, each a whole number
// of units of four stages of gps K-groups (16 slots each).
struct FilterShape {
  int natoms = 0;
  int gps = 1;
  int u0 = 0, u1 = 0;  // units of the first and second segment (u1 0: one segment)
  int n0 = 0;          // atoms of the first
  __host__ __device__ int groups0() const { return 4 * gps * u0; }
  __host__ __device__ int groups() const { return 4 * gps * (u0 + u1); }
  __host__ __device__ int slots() const { return 16 * groups(); }
  __host__ __device__ int segment_slots(int s) const { return 64 * gps * (s ? u1 : u0); }
};
FilterShape filter_shape(int natoms);
size_t filter_operand_bytes(const FilterShape& s, int n_tiles);

// C = sum m m^T of each segment (row-major), the norm of the mean structure
// over the first segment and over both.
struct FilterMean {
  float C[2][9];
  double norm0, norm;
};

// A frame set's filter operand and its rows' terms of the bound.
struct FilterSet {
  uint4* op = nullptr;
  float4* full = nullptr;   // [n_tiles * 32]
  float4* pre = nullptr;    // [n_tiles * 32]
  double* place = nullptr;  // [n_tiles * 32][12] rotation onto the mean, centroid
  ushort* extra = nullptr;  // [n_tiles * 32][segments][18]
};

// Reference pairs per fit block: flags [fit blocks][pairs], the flagged ones
// in ascending order (same shape) and their count; ctrl: two counters.
struct TileList {
  unsigned char* flags = nullptr;
  int* list = nullptr;
  int* count = nullptr;
  int* ctrl = nullptr;
  bool shared = false;  // one list for every block
};

// The test that comes before the filter (kOutBall): balls of the fit frames
// (or of their middles) and of the middles of every 64 reference frames: a
// radius and the square root of the largest threshold; twice the form's error
// bound; flags[fit / rows][pairs] is set where a candidate is possible.
struct BallTest {
  const float2* fit = nullptr;
  const float2* ref = nullptr;
  double kappa2 = 0;
  int rows = 1;
  int pairs = 0;
  unsigned char* flags = nullptr;
};

// Launchers (all asynchronous on `st`).
// mid[g] = the frame in the middle of the g-th 64 of the order.
hipError_t launch_middle(const int* order, int64_t n, int* mid, hipStream_t st);
// ball[g] = (radius of the g-th 64 frames of the order around mid[g]: an upper
// bound of sqrt(score); square root of the largest thr + eps2 / 2 of their
// rows).
hipError_t launch_balls(const DevFrames& f, const DevWeights& w, const int* order, const int* mid,
                        const unsigned* thr, const float* eps2, float2* ball, hipStream_t st);
hipError_t launch_row_balls(const unsigned* thr, const float* eps2, int64_t n, float2* ball,
                            hipStream_t st);
hipError_t launch_clear_flags(unsigned char* flags, int64_t n, hipStream_t st);
// The mean structure of the set (sqrt(w) scaled, [natoms][3]), its FilterMean
// and the slot map (shape.slots() ints); scratch: 12 kFilterSamples doubles.
hipError_t launch_filter_mean(const DevFrames& f, const DevWeights& w, const FilterShape& sh,
                              double* scratch, double* mean, FilterMean* mc, int* slots,
                              hipStream_t st);
// The set's filter operand and terms, row r from frame perm[r] (or r).
hipError_t launch_filter_prep(const DevFrames& f, const DevWeights& w, const FilterShape& sh,
                              const double* mean, const FilterMean* mc, const int* slots,
                              const int* perm, const FilterSet& out, hipStream_t st);
// The tiles with a pair that may lie within thr[fit] + eps2[fit] / 2 (sym: or
// the reference frame's), into tl.  test (if given): only the tiles flagged
// there, [fit blocks][pairs].
hipError_t launch_filter(const FilterSet& ref, const FilterSet& fit, int64_t n_ref, int64_t n_fit,
                         int ref_tiles, int fit_tiles, const FilterShape& sh, const FilterMean* mc,
                         const unsigned* thr, const float* eps2, bool sym, int grid,
                         const TileList& tl, const unsigned char* test, hipStream_t st);
// Each fit block of ft tiles against the `width` reference pairs around it.
hipError_t launch_band_list(int ref_tiles, int fit_tiles, int ft, int width, const TileList& tl,
                            hipStream_t st);
// The fit blocks of a cross query in the order of their keys (places in the
// ordered set, above dist_bits of the distance): `width` reference pairs around
// each row's place, or around every second, fourth ... row's where that makes
// more than `most` pairs.
hipError_t launch_place_band_list(const unsigned* keys, int dist_bits, const int* order, int64_t n,
                                  int ref_tiles, int fit_tiles, int width, int most,
                                  const TileList& tl, hipStream_t st);
// Every stride-th reference pair, as a list shared by every block.
hipError_t launch_stride_list(int ref_tiles, int stride, const TileList& tl, hipStream_t st);
// place[order[i]] = i.
hipError_t launch_places(const int* order, int64_t n, int* place, hipStream_t st);
// The resident set's order for cross queries, from each frame's nearest
// landmark (near: launch_contract): keys[q] = cell and distance, rows[q] = q.
hipError_t launch_fill_near(unsigned long long* near, int64_t n, hipStream_t st);
hipError_t launch_near_keys(const unsigned long long* near, int64_t n, int phases, unsigned* keys,
                            int* rows, hipStream_t st);
// order = rows sorted by key (stable); the rank form takes up to
// kRankSortMax rows and allocates and clears nothing (it may be captured).
constexpr int64_t kRankSortMax = 16384;
hipError_t launch_rank_sort(const unsigned* keys, int* order, int64_t n, hipStream_t st);
// order = rows (0, 1, ... n - 1) sorted by key (stable), the cells of the keys
// first put in the order of their leaders if given (rank: ncells ints of
// scratch).  keys_out: n more of scratch.
size_t sort_order_scratch(int64_t n);
hipError_t launch_sort_order(const int* leaders, int* rank, int ncells, unsigned* keys,
                             unsigned* keys_out, const int* rows, int* order, int64_t n, void* temp,
                             size_t temp_bytes, hipStream_t st);

// The prep pass: the FP64 centroids, G and G~ (one wave per frame), then,
// if f.op is set, the operand (one workgroup per tile and 4 K-groups).
// side 0: plain operand; +1 / -1: the dithered split's reference / query
// side (split forms only).  second (may be null): a view of the same frames
// whose op / Gt receive the operand and G~ of side2 as well (the resident
// set's query-side operand).  src_xyz (if given): the frames are read from
// it instead of f.xyz, row r from frame perm[r] when perm is given.  rot (if
// given, frames only): every frame is expressed in its principal axes,
// whose rotation is stored at rot[9 r] (frame_stats_kernel).
hipError_t launch_prep(const DevFrames& f, const DevWeights& w, int side,
                       const DevFrames* second, int side2, hipStream_t st,
                       const float* src_xyz = nullptr, const int* perm = nullptr,
                       double* rot = nullptr);
// reset_thr false keeps the shared thresholds (a landmark pass set them).
hipError_t launch_init_lists(const Lists& L, int64_t n_fit, hipStream_t st,
                             bool reset_thr = true);
// eps2[q] = 2 kappa (Gt_fit[q] + *ref.gmax); the merge's counters in *sum (if
// given) are set to 0.
hipError_t launch_eps(const DevFrames& fit, const DevFrames& ref, double kappa, float* eps2,
                      QuerySummary* sum, hipStream_t st);
// Approximate contraction into candidate lists.  When dbg_scores != nullptr
// it instead writes the approximate score of every pair to
// dbg_scores[fit*n_ref+ref] (small sizes).  With `mirror` (a self query: fit
// is the reference set's query view) it contracts the upper block triangle
// only: each pair joins the fit frame's lists and, contracted one way round
// only, the reference frame's mirrored list when it lies below that
// frame's shared threshold L.thr.  ph_run < ref_phases walks phases
// 0..ph_run-1 only (1: every ref_phases-th reference tile pair, the landmarks
// that the resident set is ordered around); 0 = all.  tiles: only the listed reference pairs of each block of
// kFilterFitTiles fit tiles, dealt out over the phases.  near: no lists, only
// each fit frame's smallest (key << 32 | reference) there (atomic minimum).
// ft 1: the one-fit-tile workgroup of short queries (contract_fit_tiles).
// ball: no lists, only the flags of that test.
hipError_t launch_contract(const DevFrames& ref, const DevFrames& fit, const Lists& L,
                           const float* eps2, int k1, int ref_phases, bool nofit,
                           double* dbg_scores, int grid_wgs, hipStream_t st,
                           const Mirror* mirror = nullptr, int ph_run = 0,
                           const TileList* tiles = nullptr,
                           unsigned long long* near = nullptr, int ft = 0,
                           const BallTest* ball = nullptr);
// The window of a symmetric self query (fit: the reference set's query
// view): eps2[r] = 2 kappa max(G~q[r] + max G~ref, G~ref[r] + max G~q);
// *gmax_q receives max G~q.
hipError_t launch_eps_sym(const DevFrames& fit, const DevFrames& ref, double kappa,
                          double* gmax_q, float* eps2, QuerySummary* sum, hipStream_t st);
// After the landmark pass (lists L of n rows, reference phases `phases`):
// thr[q] = the certified bound of row q's k1-th smallest key in the full
// query, label[q] = its nearest landmark (dense, < 64 ceil(pairs / phases)).
// keys (if given): keys[q] orders rows by their nearest landmark among every
// cell-th one, then by the distance to it, and rows[q] = q; leaders[cell] =
// the first cell whose landmark is among the leader_rank + 1 nearest of this
// cell's landmark.  place: keys[q] is its nearest landmark's place there, above
// dist_bits of the distance.
// label null: the lists are of a band or sample pass, and thr[q] is only
// lowered.
hipError_t launch_landmark_cap(const Lists& L, int64_t n, int k1, const float* eps2,
                               int phases, unsigned* thr, int* label, hipStream_t st,
                               int cell = 1, unsigned* keys = nullptr, int* rows = nullptr,
                               int* leaders = nullptr, int leader_rank = 0,
                               const int* place = nullptr, int dist_bits = kFilterDistBits);
// order[0..n) = rows grouped by label (counting sort; counts holds nlab ints).
hipError_t launch_row_order(const int* label, int64_t n, int nlab, int* counts, int* order,
                            hipStream_t st);
hipError_t launch_mirror_init(const Mirror& m, int64_t n, hipStream_t st);
// out->mirrored = total mirrored appends (including those dropped past cap),
// out->mirrored_max = most per frame.
hipError_t launch_mirror_sum(const Mirror& m, int64_t n, QuerySummary* out, hipStream_t st);
// dst[i] = frame rows[i] of src (natoms x 3 floats each).
hipError_t launch_gather_frames(const float* src, const int* rows, int nrows, int natoms,
                                float* dst, hipStream_t st);
// Output row i of (sd, si) to row rows[i] of (dd, di), k_out entries each.
hipError_t launch_scatter_rows(const double* sd, const int* si, const int* rows, int nrows,
                               int k_out, double* dd, int* di, hipStream_t st);
// order: the query rows in the order the merge workgroups take them
// (nullptr: 0..n_fit-1).  mirror: a symmetric self query's second list per
// row (nullptr: none).  perm (replaces order) and ref_perm: the lists,
// mirrored lists and eps2 were built over the frames in those orders (list
// row i is frame perm[i], entry index j reference ref_perm[j]); ref/fit and
// the outputs and fallback flags use the original indices.
hipError_t launch_merge(const DevFrames& ref, const DevFrames& fit, const DevWeights& w,
                        const Lists& L, const float* eps2, int k1, int k_out, int rank_off,
                        bool nofit, double* out_dist, int* out_idx, int* fallback,
                        QuerySummary* sum, const int* order, hipStream_t st,
                        const Mirror* mirror = nullptr, const int* perm = nullptr,
                        const int* ref_perm = nullptr);
// dst[i] = the float bits src[perm[i]] raised by add[i] (and one unit in the
// last place): the shared thresholds of a landmark pass moved to the
// permuted order, widened by the permuted frames' window.
hipError_t launch_permute_thresholds(const unsigned* src, const int* perm, const float* add,
                                     int64_t n, unsigned* dst, hipStream_t st);
// Exact FP64 scores s = G_a + G_b - 2 lambda for fit rows [row0,row0+nrows)
// against all refs.  Writes s into srow[(row-row0)*n_ref + ref] unless
// out_full is given, in which case it writes Angstrom distances into
// out_full[row*n_ref + ref] (the --sort false layout).
hipError_t launch_exact_rows(const DevFrames& ref, const DevFrames& fit, const DevWeights& w,
                             const int* rows, int nrows, bool nofit, double* srow,
                             double* out_full, int64_t out_ld, hipStream_t st);
// Top-k1 by (s, index) over exact score rows; writes ranks
// [rank_off, rank_off+k_out) of each listed fit row.
hipError_t launch_select_rows(const double* srow, int64_t n_ref, const int* rows, int nrows,
                              const DevWeights& w, int k1, int k_out, int rank_off,
                              double* out_dist, int* out_idx, hipStream_t st);
// Any k1 (the LDS select takes k1 <= 2048): the rows' k1 smallest (s, index)
// compacted in index order, then a stable segmented radix sort; `scratch`
// holds sort_rows_scratch(nrows, k1) bytes.
size_t sort_rows_scratch(int nrows, int k1);
hipError_t launch_select_rows_sorted(const double* srow, int64_t n_ref, const int* rows,
                                     int nrows, const DevWeights& w, int k1, int k_out,
                                     int rank_off, double* out_dist, int* out_idx, void* scratch,
                                     size_t scratch_bytes, hipStream_t st);
constexpr int kSelectLdsMaxK1 = 2048;
hipError_t launch_identity_rows(int64_t n_fit, int64_t n_ref, int* out_idx, hipStream_t st);
// Data vectors: mean[e] over the n vectors x[n][vdim] (FP64).
hipError_t launch_column_mean(const double* x, int64_t n, int vdim, double* mean, hipStream_t st);
// Data vectors to the frame layout of f (f.xyz, f.natoms * 3 >= f.vdim):
// Euclidean x - shift, correlation (x - mean) / |x - mean| with f.aux.
hipError_t launch_data_prep(const DevFrames& f, int metric, const double* shift, hipStream_t st);
hipError_t launch_max_gt(const DevFrames& f, double* out, hipStream_t st);

// Size of the per-GPU fixed workspace of the allocation-free query entry
// point, and its device address on `device` (which must be the current
// device on the first call for that device; later calls return the cached
// address).  Calls that overlap on one GPU share it.
constexpr size_t kScratchBytes = size_t(128) << 20;
hipError_t scratch_region(int device, void** addr);

// Fit tiles per contraction workgroup for a precision (2 or 4).
int contract_fit_tiles(int prec);
// The same for a query of n_fit frames: 1 for split forms and up to 32
// frames, where three of four fit tiles would be padding.  Two 2-wave
// workgroups per CU then stream the resident operand.  Measured, 1 frame
// against 100000 x 500 (614 MB of operand) with half the CUs, as a served
// batch gets: contraction 582 -> 199 us, 3.1 TB/s.
int contract_fit_tiles(int prec, int64_t n_fit);
// Queries of fewer frames than kCrossMinFit against this many resident frames
// or more bound their thresholds by a sample pass first: without a threshold
// every pair of a row enters its lists (no list fills up), and the merge of
// a few rows, a workgroup each, then walks n_ref entries a row in every
// radix pass.  Measured, 1 frame against 100000: merge 230 -> 98 us for a
// sample pass of 41 us and its cap of 22 us.
constexpr int64_t kSampleMinRef = 16384;
// Choose the per-list capacity for k1 (0 when the fused path cannot serve it).
int list_capacity_for(int k1);

}  // namespace mdsctk
