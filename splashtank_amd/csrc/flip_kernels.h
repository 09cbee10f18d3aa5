// flip_kernels.h - launch wrappers of the FLIP substep kernels (host side).
#pragma once
#include <hip/hip_runtime.h>

#include "flip_device.h"

// Everything one stage launch needs: the step's parameter block and collider
// records (device copies), the sim's device pointers, and launch sizes.
// entries of the per-step foam table (density sums 0 .. FOAM_TAB - 1)
#define FOAM_TAB 1024

// resident SOR: workgroup size, tiles resident per workgroup, and the largest
// grid its barrier serves (sorBar holds COOP_MAX_WG epochs, then the sequence
// number of the last solve it finished, a count of barrier time-outs, the
// barrier's release word, the path of the last solve: 0 launches per
// iteration or two, 1 resident, 2 streaming, and the sequence number of the last solve
// with a workgroup per tile)
#define COOP_WG 1024
#define COOP_TMAX 54
#define COOP_MAX_WG 1024
// most tiles in use of the one-per-tile solve: its exchange words are numbered in 20 bits
#define SOR_TILES_MAX 2048u
// its arrival words: one and TS_SUBS counters, a line of TS_LINE words each, in sorBar
// from SOR_HERE on (a batch: after its plan)
#define TS_SUBS 32u
#define TS_LINE 32u
#define SOR_HERE_WORDS (TS_LINE * (1u + TS_SUBS))
#define SOR_HERE (COOP_MAX_WG + 32u)
#define SOR_BAR_WORDS (SOR_HERE + SOR_HERE_WORDS)

struct LaunchCtx {
  const DParams* P;
  const DCols* C;
  DGrid G;
  uint32_t n;         // particles (host copy of P->n)
  uint32_t ntiles;
  uint32_t scap;
  uint32_t cellGrid;  // workgroups of grid-stride loops over active cells
  uint32_t tileGrid;  // workgroups of loops with one workgroup per tile in use
  uint32_t faceGrid;  // workgroups of the cell kernels that walk tiles in use (normFaces, divergence, project)
  uint32_t pipeGrid;  // persistent SOR workgroups (about eight per CU)
  uint32_t coopGrid;  // resident-SOR workgroups (one per CU), 0 when cooperative launches are unavailable
  uint32_t sorTiles;  // workgroups of the one-per-tile solve resident at once (0: not available)
  uint32_t sorSafe;   // as many are resident at once whatever other streams run
  uint32_t sorTag;    // tag of this solve's first exchange
  uint32_t sorSeq;    // sequence number of this pressure solve
  bool sorStream;     // the cooperative solve streams tile windows even when the tiles fit in LDS
  bool full;          // the whole substep follows the blocks stage (not a tile-only step)
  bool marksClean;    // need and binCount are zero
  bool barClean;      // the streaming SOR's barrier words are zero
  bool binned;        // blocks: need, binCount and binKey already hold A's marks and bins
  bool binNext;       // g2p: mark and bin the positions it writes, for the next substep
  bool nbOn;          // narrow band on this step
  bool ocean;         // ocean side boundary on this step
  uint32_t initStep;  // narrow-band start: 1 restart, 2 water added, 0 none
  uint32_t smax;      // whitewater slots (host copy of P->smax)
  uint32_t fullTiles; // tiles the particles would fill (n / particles of a full tile), for launch shapes
  uint32_t wetTiles;  // tiles that may hold water: fullTiles, or with a narrow band (water without particles) the pool's
  uint32_t extrap;    // opt-in face velocity extrapolation: layers (host copy of P->extrap)
  uint8_t* exMask;    // its face masks, two per pool cell (ping-pong)
};

// scratch of the narrow-band reseed: the dead slots' list over particles and the
// deficit scan over active cells (ncap = pool cells)
struct NbScratch {
  uint32_t* dead;       // N: by particle id, where the particle is stored if it is dead, else ST_NONE
  uint32_t* deadList;   // N
  uint32_t* deadCount;
  uint32_t* need;       // ncap
  uint32_t* needStart;  // ncap + 1
  uint32_t* entIdx;     // ncap
  uint32_t* entCount;
  uint64_t* sums;       // nb_sum_count() block totals of the two scans
  uint32_t ncap, nmax;
};
size_t nb_sum_count();

// Batched tanks.  Per tank: the device copies of the step's parameter block and
// collider records, and the tank's device pointers.
struct BTank {
  const DParams* P;
  const DCols* C;
  DGrid G;
  uint32_t split;  // g2p workgroups per tile
};
#define ST_BATCH_MAX 256
// per tank, what one batched substep launches for it
struct BTankPlan {
  uint32_t n;       // particles (0: the tank sits this substep out)
  uint32_t ntiles;
  uint32_t scap;
  uint32_t iters;   // SOR iterations
  bool binned;      // need, binCount and binKey already hold A's marks and bins
  bool marksClean;  // need and binCount are zero
  bool solid;       // rebuild the per-cell collider lookup
  uint32_t split;   // g2p workgroups per tile
};
// Block tables of a batched substep: table k holds nt + 1 workgroup starts, one
// range per tank (empty where the tank has no work in that launch).  Table
// BT_PIPE0 + it belongs to SOR iteration (or pass) it.
enum BatchTable {
  BT_FILL_MARK, BT_MARK, BT_SCAN, BT_PLACE, BT_FINISH, BT_CELL,
  BT_TILE, BT_SOLID, BT_COPY, BT_G2P, BT_PIPE0
};
size_t batch_table_words(uint32_t nt, uint32_t itersMax);
// fills the tables (host copy); full: tiles the tanks' particles would fill,
// sorResident = SOR workgroups resident at once; returns whether SOR launches that
// are not one cooperative launch take two iterations each
bool batch_tables(const BTankPlan* plan, uint32_t nt, uint32_t full, uint32_t itersMax, uint32_t sorResident, uint32_t* tab);
// every stage of one substep for all tanks, one launch per kernel: dT and dtab
// are the device copies of the tank records and tables, htab the host copy
// coopGrid > 0 (and a plan buffer of batch_plan_words): the SOR of every tank in
// one cooperative launch, with a workgroup per fluid tile where the device holds
// that many (sorTiles; most: tiles the tanks can have in use) or of coopGrid
// resident workgroups, else (or when the launch is refused) one launch per
// iteration, or per two where `passes` (batch_tables); returns whether it ran
// resident
inline __host__ __device__ uint32_t batch_here(uint32_t nt) { return (nt * 4u + 2u + TS_LINE - 1u) / TS_LINE * TS_LINE; }
inline size_t batch_plan_words(uint32_t nt) { return size_t(batch_here(nt)) + SOR_HERE_WORDS; }
bool launch_batch_step(hipStream_t st, const BTank* dT, const uint32_t* dtab, const uint32_t* htab, uint32_t nt, uint32_t itersMax,
                       uint32_t coopGrid, uint32_t sorTiles, uint32_t sorSafe, uint32_t most, uint32_t full, bool passes, uint32_t* dPlan);

// device-to-device copies made by one launch: whole words, starts aligned to 16
// bytes (allocations are), at most COPY_LIST_MAX
#define COPY_LIST_MAX 12
struct CopyList {
  void* dst[COPY_LIST_MAX];
  const void* src[COPY_LIST_MAX];
  size_t bytes[COPY_LIST_MAX];
  uint32_t first[COPY_LIST_MAX + 1] = {0};  // first workgroup of each copy
  uint32_t n = 0;
  void add(void* d, const void* s, size_t nbytes);
};
void launch_copies(hipStream_t st, const CopyList& L);
void launch_fill_u32(hipStream_t st, uint32_t* p, size_t n, uint32_t v);
void launch_blocks(hipStream_t st, const LaunchCtx& L);
void launch_clear(hipStream_t st, const LaunchCtx& L);
void launch_p2g(hipStream_t st, const LaunchCtx& L);
// counts: the fluid counts into ctl[0], ctl[1] now (normFaces does it too)
void launch_classify(hipStream_t st, const LaunchCtx& L, bool solid, bool counts);
// 64-bit words of DGrid.scanW
size_t scan_word_count(uint32_t ntiles);
void launch_narrowband(hipStream_t st, const LaunchCtx& L);
void launch_reseed(hipStream_t st, const LaunchCtx& L, const NbScratch& S);
void launch_norm_faces(hipStream_t st, const LaunchCtx& L);
void launch_divergence(hipStream_t st, const LaunchCtx& L);
// returns the error of the resident-SOR cooperative launch (the per-iteration
// launches still solve when it failed)
hipError_t launch_pressure(hipStream_t st, const LaunchCtx& L, int iters);
// workgroups of the persistent SOR launch that fit on `cus` CUs at once, a
// multiple of 8 (the XCD count)
uint32_t sor_resident_grid(uint32_t cus);
// workgroups of the resident SOR (one per CU when it fits there), 0 if it does not
uint32_t sor_coop_grid(uint32_t cus);
// workgroups of the one-per-tile SOR resident at once (at most SOR_TILES_MAX), 0 if none fits
uint32_t sor_tiles_grid(uint32_t cus);
// as many of them as are resident at once whatever other streams run
uint32_t sor_tiles_safe(uint32_t cus);
// tile indices in Morton order of their (ti, tj, tk) coordinates
void morton_tiles(uint32_t tx, uint32_t ty, uint32_t tz, uint32_t* out);
void launch_project(hipStream_t st, const LaunchCtx& L);
// table: make the foam table of this step's parameters first (tiles_finish has, of its step's)
void launch_g2p(hipStream_t st, const LaunchCtx& L, bool table);
// g2p workgroups per tile for particles that would fill this many tiles
uint32_t g2p_split(uint32_t fullTiles);
void launch_unsort(hipStream_t st, const float4* src, const uint32_t* pid, float4* out, uint32_t n);
// the same with *bad set when an id is not below n (that particle is left out)
void launch_unsort_checked(hipStream_t st, const float4* src, const uint32_t* pid, float4* out, uint32_t n, uint32_t* bad);
// the live view: what one packing needs (positions quantised to 16 bits across the box)
struct ViewParams {
  float x0, y0, z0, kx, ky, kz, vs, foamLife;  // kx = 65535 / (x1 - x0), ...
  uint32_t nW, nS, srcStride, fromPos;          // water points, whitewater capacity, water stride
  uint32_t oWp, oWs, oWf, oSp, oSk;             // word offsets of the parts
  uint32_t n;                                   // particles
};
// gathers the water (id order, every V.srcStride-th) and whitewater (sdMax sample slots,
// living ones compacted) samples and packs them into `out` (V's word offsets); flag and
// off hold sdMax (+1) words, sums sdMax / 1024 + 2, sdisp sdMax points
// deep water points of the narrow band look (at most DEEP_MAX, the reference's
// DEEPMAX); flags, scan and emit over the
// ncell = slots * 512 cells of the pool; all[0] counts every deep cell, off[ncell]
// the kept ones (at most ST_DEEP_MAX written to out)
#define DEEP_MAX 200000u
void launch_deep(hipStream_t st, const LaunchCtx& L, uint32_t ncell, uint32_t prev, uint32_t* flag, uint32_t* off, uint32_t* sums,
                 uint32_t* all, float4* out);
void launch_pack_view(hipStream_t st, const LaunchCtx& L, const ViewParams& V, uint32_t sdMax, uint32_t* flag, uint32_t* off,
                      uint32_t* sums, float4* sdisp, uint32_t* out);
// the spray stage (wgsl-whitewater.js): the air field when `air` (airN cells),
// then every whitewater point, then new points when `emit`, then the drops of
// ndrip drip samples (0: none)
void launch_spray(hipStream_t st, const LaunchCtx& L, uint32_t airN, bool air, bool emit, uint32_t ndrip);
// FP64 norms of the last pressure solve and projection (flip_norms.hip): part
// holds L.cellGrid x ST_NORM_WORDS doubles, out ST_NORM_WORDS (the st_norms fields)
#define ST_NORM_WORDS 8
void launch_norms(hipStream_t st, const LaunchCtx& L, double* part, double* out);
// the fixed scratch of the allocation-free norms on device `dev` (which must be
// current): room for the partials of NORMS_STATIC_WG workgroups and the results
#define NORMS_STATIC_WG 4096u
#define NORMS_STATIC_DEVICES 64
hipError_t norms_static_scratch(int dev, double** ptr, size_t* words);
