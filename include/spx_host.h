/*
 * spx_host.h -- C ABI of libspxhost.so, the host layer above libspx.
 *
 * libspxhost.so holds the C++ mirror of the reference's libs/core and
 * libs/ogs surface (platform_t, memory, settings_t, ogs_t, mesh_t).  C++
 * callers use those classes directly (streamparanumal_amd/libp/include);
 * this header exports the ogs_t and mesh pieces to non-C++ callers (the
 * Python package, ctypes).  Every function returns SPX_OK or a negative
 * SPX_ERR_* code with the message in spxh_last_error().
 */
#ifndef SPX_HOST_H
#define SPX_HOST_H

#include <stdint.h>

#include "spx.h"

#ifdef __cplusplus
extern "C" {
#endif

typedef struct spxh_ogs_s *spxh_ogs_t;

typedef struct {
  int32_t N;              /* local entries */
  int32_t Ngather;        /* positive gathered nodes (ogsBase.hpp:46) */
  int32_t NlocalT;        /* gathered nodes, all groups (ogsBase.hpp:48) */
  int32_t NlocalP;        /* gathered nodes with a positive member (ogsBase.hpp:50) */
  int32_t nnzT, nnzN;     /* CSR entries (ogsOperator.hpp:51-52) */
  int32_t NblocksT, NblocksN;
  int32_t block_nnz;      /* LDS tile of gather / scatter: max entries per row block */
  int32_t gs_block_nnz;   /* LDS tile of gather+scatter */
  int32_t Ngs_blocks;     /* row blocks of gather+scatter */
  int32_t gather_defined; /* ogsBase.hpp:57 */
  int32_t kind, unique;
  int64_t NgatherGlobal;
  double setup_seconds;
  int32_t scatter_by_rows; /* 1: rows are long enough (or the caller chose) to scatter by rows, 0: local
                              order.  spxh_ogs_scatter_path says which way a scatter goes and
                              what the caller chose. */
  int32_t mixed_tiles[2];  /* FP32 / BF16 gather+scatter on tiles of their own (1) or the FP64 one's (0) */
  int32_t gs_nontemporal;  /* spx_srb_t.nontemporal of the Sym gather+scatter's tiles */
} spxh_ogs_info_t;

const char *spxh_last_error(void);

/* platform_t on device `device_id` in HIP mode (libs/core/platformDeviceConfig.cpp) */
int spxh_platform_open(int device_id);

/* ogs_t::Setup(N, ids, comm, kind, Auto, unique, verbose, platform)
   (libs/ogs/ogsSetup.cpp:62-71).  ids (n entries) are updated in place when
   unique=1, as the reference writes the flags back (ogsSetup.cpp:149-151). */
int spxh_ogs_setup(int32_t n, int64_t *ids, int kind, int unique, int verbose, spxh_ogs_t *out);
int spxh_ogs_destroy(spxh_ogs_t ogs);
int spxh_ogs_info(spxh_ogs_t ogs, spxh_ogs_info_t *info);
/* ogs_t set up for the lexicographic GLL ids of an nx x ny x nz hex box at
   degree p (spxh_mesh_hex_ids) without the ids: the same operator and flags
   as spxh_ogs_setup over those ids, in closed form (meshSetupBoxHex3D.cpp
   and ogsSetup.cpp:87-290 give the operator this reproduces).  ids
   (optional, nx*ny*nz*(p+1)^3 entries) receives the ids as spxh_ogs_setup
   would leave them. */
int spxh_ogs_setup_hex(int32_t nx, int32_t ny, int32_t nz, int p, int kind, int unique, int64_t *ids,
                       spxh_ogs_t *out);
/* mesh_t's ogs_t of an element-type box (SPXH_TRIANGLES ... SPXH_HEXAHEDRA, 2-D types
   ignore nz; libs/mesh/meshGatherScatterSetup.cpp:31-44 over the ids of
   spxh_mesh_box_ids): the same operator as spxh_ogs_setup over those ids,
   with the gather+scatter tile order the mesh uses (lattice blocks for hex
   boxes, Tri / Quad boxes up to degree 3 and Tet boxes of degree 1 and 3).
   ids, when not NULL, has
   room for the box's elements x nodes per element (spxh_mesh_box_shape) and
   receives the sign-flagged ids. */
int spxh_ogs_setup_box(int type, int32_t nx, int32_t ny, int32_t nz, int p, int kind, int unique, int64_t *ids,
                       spxh_ogs_t *out);
/* The block-diagonal union of nparts set-up handles as one new handle (no
   reference counterpart): part i's local nodes follow parts 0..i-1's, so a
   batch of independent meshes is gathered in one launch.  The parts stay
   valid and independent. */
int spxh_ogs_setup_batch(const spxh_ogs_t *parts, int32_t nparts, spxh_ogs_t *out);
/* host copies of the operator: which = 0 (T-CSR) or 1 (N-CSR); arrays sized
   rows+1, nnz and blocks+1 (any may be NULL) */
int spxh_ogs_copy_csr(spxh_ogs_t ogs, int which, int32_t *rowStarts, int32_t *colIds, int32_t *blockStarts);
/* re-cut the row blocks for another LDS tile (autotuner): gather / scatter
   blocks, and gather+scatter blocks */
int spxh_ogs_set_block_nnz(spxh_ogs_t ogs, int32_t block_nnz);
int spxh_ogs_set_gs_block_nnz(spxh_ogs_t ogs, int32_t block_nnz);
/* scatter path: 1 (any positive value) = over the row blocks
   (ogsKernels.okl scatter), 0 = through the local->row map in local order,
   negative = as set up; results are identical.  The
   setup picks local order when the operator has fewer than 0.63 rows per
   local entry (short rows: there its coalesced stores win), else rows, of which up
   to 4 fields still go in local order, but for the Trans scatter of a Signed
   operator and for vectors whose alignment leaves whole words out
   (spx_ogs_scatter_inverse_streams).  A negative value also returns the rows to the layout set up
   (spxh_ogs_set_gather_format). */
int spxh_ogs_set_scatter_path(spxh_ogs_t ogs, int by_rows);
/* *chosen: the last value given to spxh_ogs_set_scatter_path as -1, 0 or 1 (-1 if none),
   which restores it; *runs: the way of a scatter of k fields from gv to
   v, 0 = T- or N-CSR row blocks, 1 = sorted-run row blocks, 2 = local order.
   Only the alignment of gv and v counts (NULL: aligned). */
int spxh_ogs_scatter_path(spxh_ogs_t ogs, int type, int trans, int k, const void *gv, const void *v,
                          int32_t *chosen, int32_t *runs);
/* layout of the Sym gather+scatter: 1 = sorted-run row blocks (spx_srb_t, the
   default), 0 = the T-CSR row blocks; results are identical.  xcd_remap is the
   sorted-run launch hint (negative: library default, 0 hardware order, 1 remap in
   the kernel's default blocks, a power of two 2..1024: blocks of that many
   tiles; as spx_srb_t.xcd_remap). */
int spxh_ogs_set_gs_format(spxh_ogs_t ogs, int sorted, int xcd_remap);
/* Row order of the sorted-run gather+scatter tiles (no reference counterpart):
   the T-CSR rows sorted by keys[r] (NlocalT keys; ties in row order), or the
   CSR's own order when keys is NULL.  The gather+scatter needs no row
   numbers, so results are identical; rows whose members share elements
   should share tiles.  A hex box's setup (spxh_ogs_setup_hex, mesh_t) orders
   its grid points in small 3-D blocks by itself; the gather and scatter keep
   the CSR's order. */
int spxh_ogs_set_gs_row_keys(spxh_ogs_t ogs, const int64_t *keys);
/* As spxh_ogs_set_gs_row_keys, and no tile holds rows of two different keys
   (rows of one key are cut into tiles by capacity only): each key names a
   group of rows meant to share tiles, e.g. the rows whose members fill whole
   memory lines of the vector.  No reference counterpart; results are
   identical. */
int spxh_ogs_set_gs_tiles(spxh_ogs_t ogs, const int64_t *keys);
/* The same for the tiles of the FP32 (storage SPX_STORE_F32) or BF16
   (SPX_STORE_BF16) gather+scatter (spxh_ogs_gather_scatter_mixed) alone;
   keys NULL returns them to the tiles of the other types.  A hex box's setup
   gives them line tiles of their own where those measured faster.  No
   reference counterpart; results are identical. */
int spxh_ogs_set_gs_mixed_tiles(spxh_ogs_t ogs, int storage, const int64_t *keys);
/* Non-temporal value loads and stores of the Sym gather+scatter, FP64 and
   FP32 / BF16 storage (spx_srb_t.nontemporal): -1 as the tiles' builder set them (node sizes
   whose 128-byte lines mostly lie whole in one tile), 0 never, 1 for every
   node size; kept when the tiles are rebuilt.  No reference counterpart;
   results are identical. */
int spxh_ogs_set_gs_nontemporal(spxh_ogs_t ogs, int mode);
/* layouts of the T-CSR gather (Trans) and scatter (NoTrans): 1 = the
   sorted-run blocks of the gather+scatter, 0 = T-CSR row blocks, -1 = keep;
   both sorted by default.  A scatter layout given here holds for every
   scatter that goes by rows, up to 4 fields included, until
   spxh_ogs_set_scatter_path is given a negative value.  Results are identical. */
int spxh_ogs_set_gather_format(spxh_ogs_t ogs, int gather_sorted, int scatter_sorted);
/* Autotuner (no reference counterpart; the reference's ogs::Auto times its
   halo exchange methods, ogsSetup.cpp:116-125, the same way): times every
   candidate launch shape of the Sym gather+scatter -- layout, block
   capacity, tile lanes, XCD remap -- on this operator for k fields of `type`
   (storage = -1) or of mixed storage `storage` (SPX_STORE_*), keeps the
   fastest and reports it.  Results never change with the shape. */
typedef struct {
  int32_t sorted, block_nnz, tile_lanes, xcd_remap;
  double ms;
  int32_t candidates;
} spxh_gs_tuning_t;
int spxh_ogs_autotune(spxh_ogs_t ogs, int type, int storage, int k, int reps, spxh_gs_tuning_t *best);
/* Times spx_cg_batch over plans of several sizes and unroll / streaming
   settings on the caller's vectors (alpha = 0: values unchanged); leaves
   the best in the "cg_batch" tuning and returns its plan (the caller
   destroys it). */
typedef struct {
  int32_t target_blocks, unroll, nontemporal;
  double ms;
  int32_t candidates;
} spxh_cg_tuning_t;
int spxh_cg_batch_autotune(int32_t nseg, const int64_t *segStarts, int storage, void *p, void *Ap, void *x,
                           void *r, double *rdotr, int reps, spx_cg_plan_t *plan, spxh_cg_tuning_t *best);
/* ogs_t::SetupGlobalToLocalMapping (ogsSetup.cpp:833-849) */
int spxh_ogs_global_to_local(spxh_ogs_t ogs, int32_t *g2l);

/* ogs_t device operations on device pointers, enqueued on the current stream
   (ogs.cpp:39-125, 205-301, 394-492) */
int spxh_ogs_gather_scatter(spxh_ogs_t ogs, int type, int op, int trans, int k, void *v);
int spxh_ogs_gather(spxh_ogs_t ogs, int type, int op, int trans, int k, const void *v, void *gv);
int spxh_ogs_scatter(spxh_ogs_t ogs, int type, int trans, int k, const void *gv, void *v);
/* Sym Add gatherScatter of v stored as SPX_STORE_F32 / SPX_STORE_BF16 (FP64
   row sums, one rounding; spx_ogs_gather_scatter_mixed); no reference
   counterpart, the reference gathers dfloat only (ogs.cpp:39-125) */
int spxh_ogs_gather_scatter_mixed(spxh_ogs_t ogs, int storage, int k, void *v);

/* The host half of the setup alone (no device needed): grouping, unique
   flagging (written back into ids), row numbering, T- and N-CSR. */
typedef struct spxh_csr_s *spxh_csr_t;
int spxh_csr_build(int32_t n, int64_t *ids, int kind, int unique, spxh_csr_t *out);
/* the same for a hex box in closed form (see spxh_ogs_setup_hex) */
int spxh_csr_build_hex(int32_t nx, int32_t ny, int32_t nz, int p, int kind, int unique, int64_t *ids,
                       spxh_csr_t *out);
/* sizes[0..4] = NrowsT, NrowsN, nnzT, nnzN, gather_defined */
int spxh_csr_sizes(spxh_csr_t csr, int32_t *sizes);
int spxh_csr_copy(spxh_csr_t csr, int which, int32_t *rowStarts, int32_t *colIds);
int spxh_csr_destroy(spxh_csr_t csr);
/* row blocks of at most cap entries (greedy); blockStarts holds nrows+2 */
int spxh_block_rows(int32_t nrows, const int32_t *rowStarts, int32_t cap, int32_t *nblocks,
                    int32_t *blockStarts);
/* Line-aligned gather+scatter tiles of an nx x ny x nz hex box at degree p
   (no reference counterpart): row_grid[r] is the lattice index (x fastest)
   of T-CSR row r's point.  order receives the rows tile by tile and cuts[i]
   is 1 where a tile starts (spxh_ogs_set_gs_tiles's form).  A tile holds the
   rows of one z plane, full x lines, and y points that never split a group
   of rows_per_line node rows of an element (the memory line of the vector),
   merged up to cap members; larger groups are cut along x at element
   boundaries. */
int spxh_hex_gs_tiles(int nx, int ny, int nz, int p, int rows_per_line, int cap, int32_t nrows,
                      const int64_t *row_grid, int32_t *order, uint8_t *cuts);
/* Sorted-run tiles (spx_srb_t) of a CSR and its row blocks, on the host (no
   device needed): sizes[0..5] = nblocks, nnz, nchunks (= nblocks *
   chunks_per_tile), nruns, nlinks, chunks_per_tile.  spxh_srb_copy fills
   host arrays of nchunks records, nruns run ids, nlinks + 1 links (the last a
   padding word) and nblocks + 1 CSR entry offsets of the tiles (any may be
   NULL); the caller uploads chunks, runIds and links and fills spx_srb_t. */
typedef struct spxh_srb_s *spxh_srb_t;
int spxh_srb_build(int32_t nrows, const int32_t *rowStarts, const int32_t *colIds, int32_t nblocks,
                   const int32_t *blockStarts, int32_t max_block_nnz, spxh_srb_t *out);
int spxh_srb_sizes(spxh_srb_t srb, int64_t *sizes);
int spxh_srb_copy(spxh_srb_t srb, spx_srb_chunk_t *chunks, int32_t *runIds, uint16_t *links, int32_t *entryStarts);
int spxh_srb_destroy(spxh_srb_t srb);
/* 1 when every tile's rows ascend by their first member's local index, as
   the layout's gather and scatter (which number rows by their leading
   positions) need; 0 otherwise, e.g. for the T-CSR of an ogs::Signed
   operator without unique flagging, whose groups with no positive member
   follow the others (ogsSetup.cpp:517-546).  The gather+scatter forms need
   no row numbers and run on any layout. */
int spxh_srb_rows_ascending(spxh_srb_t srb, int32_t *ascending);
/* The same for the T-CSR of an ogs::Signed operator (ncols local nodes)
   together with its N-CSR (ogsOperator.cpp:621-643), which must hold the
   members of the same T-CSR rows, in the same order, for its nrowsN rows
   (refused otherwise); spxh_srb_copy_members then fills the nchunks N-member
   masks of spx_ogs_*_srb_signed. */
int spxh_srb_build_signed(int32_t nrows, const int32_t *rowStarts, const int32_t *colIds, int32_t nblocks,
                          const int32_t *blockStarts, int32_t max_block_nnz, int32_t ncols, int32_t nrowsN,
                          const int32_t *rowStartsN, const int32_t *colIdsN, spxh_srb_t *out);
int spxh_srb_copy_members(spxh_srb_t srb, uint64_t *memberN);
/* spx_srb_t.nontemporal for the layout: bit e (e = 1..5) when at least 85 %
   of the (tile, 128-byte line) pairs of a vector of 2^e-byte nodes that hold
   an entry hold the whole line. */
int spxh_srb_nontemporal(spxh_srb_t srb, int32_t *mask);

/* mesh_t hex box ids: lexicographic GLL-grid ids of an nx x ny x nz box at
   degree p, n = nx*ny*nz*(p+1)^3 entries (meshSetupBoxHex3D.cpp:87-130) */
int spxh_mesh_hex_ids(int nx, int ny, int nz, int p, int64_t *ids);

/* element types of mesh_t (include/mesh.hpp:116-119) */
#define SPXH_TRIANGLES 3
#define SPXH_QUADRILATERALS 4
#define SPXH_TETRAHEDRA 6
#define SPXH_HEXAHEDRA 12

/* elements and nodes per element of a box of `type` (meshSetElementType.cpp,
   meshReferenceNodes*.cpp: Np = (p+1)(p+2)/2, (p+1)^2, (p+1)(p+2)(p+3)/6,
   (p+1)^3); 2-D types ignore nz (pass 1) */
int spxh_mesh_box_shape(int type, int nx, int ny, int nz, int p, int64_t *nelements, int *np);
/* mesh_t box ids for any element type: 1 + the lexicographic index of each
   node's point on the degree-p lattice of the box, in the reference's element
   and node order (meshSetupBoxTri2D.cpp:80-113, meshSetupBoxQuad2D.cpp:79-100,
   meshSetupBoxTet3D.cpp:87-189, meshBasisTri2D.cpp:81-92,
   meshBasisTet3D.cpp:81-94); the groups are those meshConnectNodes.cpp:32-82
   forms */
int spxh_mesh_box_ids(int type, int nx, int ny, int nz, int p, int64_t *ids);

#ifdef __cplusplus
}
#endif
#endif
