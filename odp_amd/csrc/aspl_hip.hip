// aspl_hip.hip -- host side of libodp_hip: the ODP_* lifecycle (the drop-in
// for aspl_cuda.cu), plan selection and autotuning, kernel timing, and the
// batched / looped evaluation paths.  Kernels live in kernels.hpp.
//
// Exact arithmetic (aspl.c:47-74, 81-118, 332-336): every block of l sources
// contributes sum_L (n*l - count_L) * s over its non-terminal levels, the
// diameter is max over blocks of (terminal level + 1), the ordered-pair sum
// starts at n*(n-1), ASPL = sum / ((n-1)*n) in double and the returned sum is
// (long)(sum / 2.0).  A block whose count stops growing before it reaches n*l
// marks the graph disconnected: diameter n+1, hence INT_MAX / LONG_MAX /
// DBL_MAX, exactly what the reference reaches after n levels.
#include <hip/hip_runtime.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <limits.h>
#include <float.h>
#include <math.h>
#include <time.h>
#include <unistd.h>
#include <sys/time.h>
#include <vector>
#include <atomic>
#include <algorithm>
#include <mutex>
#include "odp.h"
#include "odpx.h"
#include "kernels.hpp"

#define ODP_ERROR(...) do { fprintf(stderr, __VA_ARGS__); exit(1); } while (0)
#define HIPC(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) \
  ODP_ERROR("libodp_hip: %s failed: %s (%s:%d)\n", #x, hipGetErrorString(e_), __FILE__, __LINE__); } while (0)

static const int KIND_MATRIX = 1, KIND_SAVING = 2, KIND_BFS = 3;   // the reference's ASPL_* (common.h:39-41)
static const int GPU_CHUNK_WORDS = 64;          // column-block width of MATRIX_SAVING (parameter.h:13)
static const int SAVING_GROUP = 32;             // MATRIX_SAVING blocks resident at once (4 per XCD) ...
// ... unless the kind is the size's own choice (ODP_ASPL not set: who asks for
// MATRIX_SAVING asks for its bounded memory) and all blocks' buffers stay within
// this and an eighth of the free memory (so that eight processes that look at
// once all fit): the folded levels need them all resident, and k_direct walks the
// rows once instead of once per group (n = 100000, d = 8, 2.5 GB instead of 0.8:
// 4.99 -> 3.0 ms; n = 131072, d = 16: 10.8 -> 6.3 ms; n = 200000, d = 8, 10 GB: 28.4 -> 17.2 ms)
static const size_t SAVING_BYTES = 16ull << 30;
static const int LEVEL_BLOCK_WORDS = 16;        // default column-block width of the level plan
static const int RES_WB_MAX = 8;                // widest resident block: 256 sources
static const int BATCH_CLASSES = 5;             // size classes of the batch launch policy
static const int FRONTIER_MIN_LEVELS = 16;      // frontier-mode levels when the last evaluation needed more
static const u32 LIST_CAP = 1u << 22;           // unsaturated chunks a level may list (32 MiB)
static const int LIST_COUNTERS = 2 * LIST_SUBS * LIST_PAD;   // the counters of two lists
static const u32 THIN_CAP = 1u << 20;           // chunks a thin level may list (24 MiB),
static const u32 THIN2_CAP = 1u << 18;          // ... and k_thin leave unsaturated
static const double THIN_LEFT = 1.0 / 256;      // share of the chunks the thin neighbours should leave unsaturated
static const double THIN2_READS = 8e6;          // chunk reads k_thin2 may take (two steps from every chunk left)
static const double LIST_MAX_FRAC = 1.0 / 8;     // ... listed only when at most this share was left last time
static const double LIST_MAX_FRAC_PG = 1.0 / 32; // ... by k_pgather, whose count-only levels cost less
static const int LV_MISS_LEVELS = 64;            // levels whose missing pairs an evaluation records
// adjacency tables up to this size reach the device through the resident
// plan's table build reading pinned host memory (one kernel instead of a DMA
// command plus the kernel); larger ones are copied by DMA.  The kernel reads
// the link as fast as the copy and saves its command: an evaluation of n = 8192,
// d = 12 (384 KiB) 67.2 -> 53.0 us, 16384, 16 (1 MiB) 124 -> 108, 40000, 16
// (2.5 MiB) 538 -> 530.  A symmetric graph's build reads the base table once per
// copy of it and again for the device's: the smaller limit
static const size_t ZC_MAX_BYTES = 4096u << 10, ZC_MAX_BYTES_SYM = 256u << 10;
static const size_t LMAX_HOST_ENTRIES = 8192;   // adjacency entries whose longest edge the host measures itself
static const int TILE_MIN = 32;                 // smallest tile side of k_tile (halo 16)
static const int SPARSE_GRID = 2048;            // workgroups of a k_sparse launch (8 per CU)
static const long DIRECT_TREE_MAX = 8192;       // walk-tree nodes per row the automatic direct K allows
static const long DIRECT_TREE_CAP = 65536;      // ... and any requested K (larger K is lowered)
static const double MEM_THRESHOLD_MB = 2048.0;  // MATRIX -> MATRIX_SAVING switch (parameter.h:4)
static const size_t LDS_LIMIT = 163840;         // LDS a gfx950 workgroup may allocate
static const size_t LDS_STATIC = 512;           // k_resident's own __shared__ data, rounded up
static const size_t LDS_DYN_MAX = LDS_LIMIT - LDS_STATIC;
static const double RES_SPIN_S = 200e-6;         // a resident evaluation's wait watches its result this long
static const double LV_SPIN_S = 20e-3;           // a level batch's wait watches its sequence number this long
static const int LVFIN_MAX = 4096;               // counters k_lvfin hands over (more: copies, faster than one workgroup's writes to host memory)
static const int RING = 260;                    // per-level counter slots kept on the device
static const int MAX_BATCH_LEVELS = 256;        // levels launched between two host reads (< RING - 2)
static const size_t MALL_BYTES = 256u << 20;    // the last-level cache in front of HBM
static const int PG_PARTS = 4;                  // row parts of the XCD-phased gather (2 MiB of a 65536-row slab)
static const long long BATCH_PIPE_BYTES = 4 << 20;   // a batch handed over and run in one call is sent in chunks from here
static const int PG_MIN_ROWS = 24576;           // ... used by default from this many rows (a 3 MiB slab),
static const int PG_MIN_ROWS_NARROW = 20000;    // ... and from this many with tables of at most 16 ids

// ODP_HIP_TRACE=1 prints each host step to stderr (diagnostics)
static int g_trace = -1;
static void trace(const char* what)
{
  if (g_trace < 0) { const char* v = getenv("ODP_HIP_TRACE"); g_trace = v && atoi(v) == 1; }
  if (g_trace) { fprintf(stderr, "[libodp_hip] %s\n", what); fflush(stderr); }
}

static double wall_time()
{
  struct timeval t;
  gettimeofday(&t, NULL);
  return t.tv_sec + 1.0e-6 * t.tv_usec;
}

static inline int round_up(int x, int m) { return (x + m - 1) / m * m; }
static inline int ilog2(int x) { int r = 0; while ((1 << (r + 1)) <= x) r++; return r; }

// Annealing programs seed libc's generator once (ODP_Srand) and draw moves
// and acceptance tests from it between evaluations; the reference library
// draws nothing while it evaluates.  The HIP runtime does draw from it (its
// initialisation at least), which would shift such a program's trajectory.
// So every entry point that can reach the runtime runs with libc's
// random()/rand() switched to a private state and switches the caller's back
// on return (setstate keeps the caller's position; nested entries are fine).
// Entries may overlap (nested calls, or the serving calls from several
// threads): only the outermost switches, and the last one out switches back.
static char g_rand_private[256];
static bool g_rand_private_ready = false;
static std::mutex g_rand_mu;
static int g_rand_depth = 0;
static char* g_rand_caller = nullptr;
struct RandFence {
  RandFence()
  {
    std::lock_guard<std::mutex> lk(g_rand_mu);
    if (g_rand_depth++ > 0) return;
    if (!g_rand_private_ready) {
      g_rand_caller = initstate(1u, g_rand_private, sizeof g_rand_private);    // also makes it current
      g_rand_private_ready = true;
    } else {
      g_rand_caller = setstate(g_rand_private);
    }
  }
  ~RandFence()
  {
    std::lock_guard<std::mutex> lk(g_rand_mu);
    if (--g_rand_depth == 0) setstate(g_rand_caller);
  }
  RandFence(const RandFence&) = delete;
  RandFence& operator=(const RandFence&) = delete;
};

// ---------------------------------------------------------------------------
// device context: one stream (default priority) for everything

static struct { bool ready; hipStream_t stream; int ncu; } C;

static void ctx_init()
{
  if (C.ready) return;
  trace("ctx_init");
  int dev;
  HIPC(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  HIPC(hipGetDeviceProperties(&prop, dev));
  C.ncu = prop.multiProcessorCount;
  HIPC(hipStreamCreateWithFlags(&C.stream, hipStreamNonBlocking));
  HIPC(hipFuncSetAttribute((const void*)k_resident, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<2>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<4>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<2, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<4, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<8, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, false, RES_RPT_WIDE1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, true, RES_RPT_WIDE1>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, false, RES_RPT_WIDE1B>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, true, RES_RPT_WIDE1B>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, false, RES_RPT_WIDE1C>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<1, true, RES_RPT_WIDE1C>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<2, true, RES_RPT_WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_resident_w<2, false, RES_RPT_WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                           (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_anneal<1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_anneal<2>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_anneal<4>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  HIPC(hipFuncSetAttribute((const void*)k_anneal<8>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  for (auto k : {k_direct<true, true, true>, k_direct<true, false, true>, k_direct<true, false, false>,
                 k_direct<false, true, false>, k_direct<false, false, false>})
    HIPC(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS_DYN_MAX));
  C.ready = true;
  trace("ctx ready");
}

template <typename T> static void dalloc(T** p, size_t count)
{
  *p = nullptr;
  if (count) HIPC(hipMalloc((void**)p, count * sizeof(T)));
}
template <typename T> static void dfree(T** p) { if (*p) HIPC(hipFree(*p)); *p = nullptr; }
template <typename T> static void halloc(T** p, size_t count)
{
  *p = nullptr;
  if (count) HIPC(hipHostMalloc((void**)p, count * sizeof(T), hipHostMallocDefault));
}
template <typename T> static void hfree(T** p) { if (*p) HIPC(hipHostFree(*p)); *p = nullptr; }
// host memory that kernels write directly (coherent: not cached on the device side)
template <typename T> static void halloc_coherent(T** p, T** dev, size_t count)
{
  *p = nullptr; *dev = nullptr;
  if (!count) return;
  HIPC(hipHostMalloc((void**)p, count * sizeof(T), hipHostMallocCoherent));
  HIPC(hipHostGetDevicePointer((void**)dev, *p, 0));
}

// hipGraph capture and replay of repeated launch sequences (env ODP_HIP_GRAPH=0 turns it off)
static bool graphs_env()
{
  static int env = -1;
  if (env < 0) { const char* v = getenv("ODP_HIP_GRAPH"); env = v ? atoi(v) != 0 : 1; }
  return env != 0;
}

// the first pulled level of a resident block (res_walk_levels; env
// ODP_HIP_RES_WALK=0 builds level 0 from the table and pulls every later
// level, N walks the levels below N at most)
static int res_walk_cap()
{
  static int cap = -2;
  if (cap == -2) { const char* v = getenv("ODP_HIP_RES_WALK"); cap = v ? atoi(v) : -1; }
  return cap < 0 ? 1 << 20 : std::max(cap, 0);
}

static int res_walk_env(int n, int deg, int l)
{
  static double cost = -1;
  if (cost < 0) { const char* v = getenv("ODP_HIP_RES_WALK_COST"); cost = v ? atof(v) : 1.0; }
  return std::min(res_walk_levels(n, deg, l, cost), res_walk_cap());
}

// rows per thread a single-graph resident launch may take at width wb (the
// one- and two-word instances with RES_RPT_WIDE1(B, C) / RES_RPT_WIDE rows run past res_rpt's)
static int res_rows(int wb) { return wb == 1 ? RES_RPT_WIDE1C : wb == 2 ? RES_RPT_WIDE : res_rpt(wb); }

// Block width (32-bit words) of one graph's resident evaluation, up to wbmax:
// the width with the least work on the busiest CU -- blocks per CU
// (ceil(blocks / ncu): blocks that share a CU share its LDS and VALU issue)
// times a block's cost at that width relative to one word (measured on single
// graphs of n = 1024..16384, d = 6..24: two words 1.2, four 1.45, eight 2).
// Ties go to the narrower block (a lone block is latency-bound).  Giving every
// CU a block first had picked one-word blocks up to n = 16384: 1.6-1.8 x slower
// than two-word blocks from n = 8192 on (two blocks per CU against one).
static int res_width(int n, int nsrc, int wbmax, int ncu)
{
  static const double rel[4] = {1.0, 1.2, 1.45, 2.0};
  int wb = wbmax;
  double best = 1e300;
  for (int c = 1, i = 0; c <= wbmax && i < 4; c <<= 1, i++) {
    if (n > res_rows(c) * 1024) continue;          // too many rows for this width's instance
    const long blocks = (nsrc + 32L * c - 1) / (32L * c);
    const double t = (double)((blocks + ncu - 1) / ncu) * rel[i];
    if (t < best) { best = t; wb = c; }
  }
  return wb;
}

// ODP_HIP_FOLD=0: every unit of a gather level, whatever the table (diagnostics)
static bool pg_fold_env()
{
  const char* v = getenv("ODP_HIP_FOLD");
  return !v || atoi(v) != 0;
}

// ODP_HIP_THIN=0: no thin levels (diagnostics)
static bool pg_thin_env()
{
  const char* v = getenv("ODP_HIP_THIN");
  return !v || atoi(v) != 0;
}

// log2 of the pieces the units of k_pgather's last, partly filled round are cut
// into: `units` of an XCD's workgroups in rounds of `wgs`, `extra` more at the
// end.  A piece costs its share of a unit and about an eighth of one more (the
// fill of its gathers, its barriers).
static int pg_cut(double units, double extra, int wgs)
{
  const double rest = units - wgs * std::floor(units / wgs) + extra;
  int best = 0;
  double cost = 1e30;
  for (int c = 0; c <= PG_CUT_MAX; c++) {
    const double v = std::ceil(rest * (1 << c) / wgs - 1e-9) * (1.0 / (1 << c) + (c ? 0.125 : 0));
    if (v < cost - 1e-9) { cost = v; best = c; }
  }
  return best;
}

// the share of unsaturated chunks up to which a count-only last level lists
// them (env ODP_HIP_LIST_FRAC; a large value always lists)
static double list_frac_env(double dflt)
{
  const char* v = getenv("ODP_HIP_LIST_FRAC");
  const double f = v ? atof(v) : dflt;
  return f >= 0 ? f : dflt;
}

// capacity of the unsaturated-chunk list (env ODP_HIP_LIST_CAP lowers it; the
// sub-lists share it evenly, and a level that lists more chunks than a
// sub-list holds is counted by visiting every chunk)
static u32 list_cap_env()
{
  const char* v = getenv("ODP_HIP_LIST_CAP");
  if (!v) return LIST_CAP;
  const long c = atol(v);
  return c < 0 ? 0u : (c > (long)LIST_CAP ? LIST_CAP : (u32)c);
}

// ---------------------------------------------------------------------------
// kernel timing: HIP events recorded on the launch stream around launches

enum { T_OTHER = 0, T_LEVEL = 1, T_RESIDENT = 2 };
// nlev: levels the launch runs; wr: it writes the rows (0: a count-only level);
// fold: folded if the table is symmetric; nbrs: neighbours a row takes (-1: all)
struct TimedLaunch { hipEvent_t a, b; int kind, level, nlev = 1, wr = 1; bool fold = false; int nbrs = -1; };
static bool g_stats_on = false;
static bool g_stats_live = false;       // timed evaluations keep the untimed launch sequence
static ODPX_Stats g_stats;
// the ways evaluations went that results do not show (ODPX_Routes_get)
static struct { std::atomic<long long> folded{0}, thin{0}, thin_whole{0}, thin_late{0}, chunked{0}; } g_routes;
static std::vector<hipEvent_t> g_evpool;
static std::vector<TimedLaunch> g_pending;

static hipEvent_t ev_get()
{
  if (!g_evpool.empty()) { hipEvent_t e = g_evpool.back(); g_evpool.pop_back(); return e; }
  hipEvent_t e;
  HIPC(hipEventCreate(&e));
  return e;
}
// Only evaluations on the library's main stream (the ODP_* lifecycle, the
// batched and looped paths) are timed; the serving engine's slots run untimed.
static void timed_begin(TimedLaunch& t, int kind, int level, hipStream_t st = nullptr)
{
  t.kind = kind; t.level = level;
  if (!g_stats_on || (st && st != C.stream)) { t.a = nullptr; return; }
  t.a = ev_get(); t.b = ev_get();
  HIPC(hipEventRecord(t.a, C.stream));
}
static void timed_end(TimedLaunch& t)
{
  if (!t.a) return;
  HIPC(hipEventRecord(t.b, C.stream));
  g_pending.push_back(t);
}

// zero na words and *q (a kernel, so that sequences containing it can live in
// a hipGraph): the batch's per-graph accumulators and queue head, a list counter
__global__ void k_clear(u64* a, int na, int* q, int nq)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < na) a[i] = 0;
  if (i < nq) q[i] = 0;
}

// ---------------------------------------------------------------------------
// one graph on the device, the row-neighbour table and its plan

struct LevelRun {
  int n = 0, ntasks = 0, group = 0, kw = 0, kwp = 0, upw = 4, seg_major = 1, xcd = 0, urow = 0, per_task_wg = 0;
  int direct = 0, dnw = 4, dgrid = 0;   // levels done by k_direct (0: k_level0), its waves and grid
  int segs = 1;                         // 2 x lanes-per-row word segments per block row
  int batch = 4;                        // neighbour rows k_level gathers per batch
  size_t dlds = 0;
  size_t buf_words = 0;                 // capacity of bufs (64-bit words)
  size_t task_cap = 0;
  u64* bufs = nullptr; u64* cnt = nullptr; u32* done = nullptr;
  unsigned char* flags = nullptr;       // per block of the group 4 x segs x n bytes: changed flags, marks
  unsigned char* wgm = nullptr;         // per block of the group 2 x workgroups bytes: workgroup marks
  size_t wgm_bytes = 0;
  u32* tq = nullptr;                    // k_tile's unit list (tile mode): lengths, queue head, entries
  size_t tq_cap = 0;
  u64* list = nullptr;                  // unsaturated chunks of the level before a count-only one
  u32* list_n = nullptr;                // the two lists' counters (after the done flags)
  u32* asym = nullptr;                  // set unless the table is symmetric (after them)
  u32 list_cap = 0;
  // thin levels (k_thin): the chunks of a list with their bits, and the second list
  int thin = 0;                         // neighbours the pair lists mark thin
  u64x2* list_v = nullptr;
  u64* list2 = nullptr; u64x2* list2_v = nullptr;
  u64* h_acnt = nullptr;                // processed-unit counts on the host, then the asymmetry flag (kernel timing only)
  size_t flag_bytes = 0;
  // part-phased gather (k_pgather): row parts, sorted neighbour runs, persistent grid
  int parts = 0, psp = 0, pgrid = 0, pupt = 0;
  bool fold = false;                    // folded levels where the table is symmetric (k_pgather)
  int cut_full = 0, cut_fold = 0;       // log2 of the pieces its last round's units are cut into
  u32* plist = nullptr; int* ppoff = nullptr;  // per unit of PG_UNIT rows: pairs grouped by part, offsets
  size_t plist_cap = 0, ppoff_cap = 0;
  LevelTask* tasks = nullptr; int* wg_start = nullptr;
  u64* h_cnt = nullptr;                 // coherent host memory (k_lvfin writes it)
  u64* h_cnt_dev = nullptr;
  std::vector<int> l;                   // sources per task
};

struct ResRun {
  int ntasks = 0, wb = 1, threads = 1024, grid = 0;
  size_t lds = 0, task_cap = 0;
  ResTask* tasks = nullptr; ResOut* out = nullptr; int* qhead = nullptr;
  u32* done = nullptr;                  // the launch's arrival counter (left at zero by each launch)
  ResOut* part = nullptr;               // per-workgroup totals
  size_t part_cap = 0;
  ResHost* host = nullptr;              // pinned coherent host memory the launch writes its result to
  ResHost* host_dev = nullptr;          // its device address
  u32 seq = 0;                          // sequence number of the last launch
};

struct Evaluator {
  // graph
  int family = 0, n = 0, s = 1, degree = 0, dpad = 0, width = 0, height = 0, grid_s = 0, nsrc = 0;
  // source columns evaluated: [src_lo, src_hi) of [0, nsrc) (all but for one shard's share)
  int src_lo = 0, src_hi = 0;
  int has_numdeg = 0;
  double avg_deg = 0;
  size_t adj_cap = 0, nbr_cap = 0;
  int *d_adj = nullptr, *d_numdeg = nullptr, *d_itable = nullptr, *d_nbr = nullptr, *d_err = nullptr;
  unsigned short* d_nbr16 = nullptr;    // 16-bit row-neighbour table of the resident plan
  bool bfs = false;                     // the BFS kind: evaluations run k_bfs
  int* d_bfs_q = nullptr;               // [workgroups][2][n] frontier queues of k_bfs
  u32* d_bfs_vis = nullptr;             // [workgroups][n/32] visited bitmaps when LDS cannot hold one
  BfsOut *d_bfs_out = nullptr, *h_bfs_out = nullptr;
  int* d_bfs_next = nullptr;            // next source to take
  size_t bfs_q_cap = 0, bfs_vis_cap = 0;
  const int* ext_adj = nullptr;         // when set, the adjacency is read from this device copy
  int dp16 = 8;
  size_t nbr16_cap = 0;
  // grid geometry for k_tile (grid graphs whose rows are cells): cell <-> row
  int *d_xy2row = nullptr, *d_row2xy = nullptr;
  short* d_toff = nullptr;              // [n][dpad] cell offsets of the table entries
  size_t toff_cap = 0;
  int geo_lmax = -1;                    // largest |dx|, |dy| of an adjacency entry; -1: no geometry
  bool geo_stale = false;               // an upload changed it: measured on the device when an evaluation needs it
  int *d_lmax = nullptr, *h_lmax = nullptr;
  int *h_stage = nullptr, *h_err = nullptr;
  int* h_stage_dev = nullptr;           // device address of h_stage (coherent pinned memory)
  // the last upload is still only in h_stage: the resident plan's next table
  // build reads it there and copies it to d_adj (small tables: no DMA command)
  bool adj_on_host = false;
  size_t stage_cap = 0;
  // the current plan's table (the resident plan's 16-bit table; the level plan's
  // 32-bit table and its 16-bit copy) matches the adjacency at `table_src`: set
  // by its preparation, kept by device swaps (they patch the table as well),
  // cleared by an upload, a new shape or a new plan
  bool table_fresh = false;
  const int* table_src = nullptr;
  // the level plan's pair lists (k_plist) match its table (device swaps rebuild
  // the units of the rows they change); meaningful while table_fresh holds
  bool pl_fresh = false;
  // the level plan's asymmetry flag (after the done flags) is the current
  // table's: set by its check, outlived by device swaps (a swap of a symmetric
  // table leaves it symmetric) while table_fresh holds
  bool asym_fresh = false;
  // a batch of levels ends with k_lvfin: counters and error flag in host memory,
  // then its sequence number (lvseq: the last one enqueued; d_lvseq: the device's)
  LvHost* lvh = nullptr;
  LvHost* lvh_dev = nullptr;
  u32* d_lvseq = nullptr;
  u32 lvseq = 0;
  // table entries the next resident launch changes first (triples row, position, id)
  std::vector<int> pend_patch;
  // h_stage holds what the device copy holds (or will, once the pending entries are stored):
  // false after moves made on the device only
  bool stage_is_device = false;
  // h_mirror holds what the device copy holds once the enqueued work is done:
  // taken from h_stage by the first device swap after an upload and kept by
  // the swaps that follow, so they are checked on the host and launched
  // without waiting; anything else that changes the device copy clears it
  std::vector<int> h_mirror;
  bool mirror_ok = false;
  // the pending table entries as launch arguments (taken: the list is emptied)
  ResPatch make_patch()
  {
    ResPatch p{};
    p.n = (int)(pend_patch.size() / 3);
    if (p.n > RES_PATCH_MAX) ODP_ERROR("libodp_hip: internal error: too many pending table entries\n");
    for (int i = 0; i < p.n; i++)
      for (int k = 0; k < 3; k++) p.e[i][k] = pend_patch[3 * i + k];
    p.table = d_nbr16; p.tdp = dp16; p.adj = d_adj; p.degree = degree;
    pend_patch.clear();
    return p;
  }
  // stores the pending entries now (no evaluation follows)
  void apply_pending()
  {
    if (pend_patch.empty()) return;
    hipLaunchKernelGGL(k_patch, dim3(1), dim3(64), 0, st, make_patch());
    HIPC(hipGetLastError());
  }

  // the table a device swap patches along with the adjacency; null (and the
  // table no longer current) when there is none to keep
  unsigned short* swap_table()
  {
    if (table_fresh && table_src == d_adj && plan.plan == ODPX_PLAN_RESIDENT && s == 1 && !grid_s) return d_nbr16;
    table_fresh = false;
    return nullptr;
  }

  // The tables a change of the device adjacency patches along with it: the
  // resident plan's 16-bit table, or the level plan's 32-bit table and 16-bit
  // copy (whose pair lists the change's units then rebuild), when current;
  // otherwise none, and the next evaluation rebuilds the table.
  SwapTables patch_tables()
  {
    SwapTables tb{};
    const bool cur = table_fresh && table_src == d_adj && s == 1 && !grid_s;
    if (cur && plan.plan == ODPX_PLAN_RESIDENT) {
      tb.t16 = d_nbr16; tb.tdp = dp16;
    } else if (cur && plan.plan == ODPX_PLAN_LEVEL) {
      tb.t32 = d_nbr; tb.t16 = direct16() ? d_nbr16 : nullptr; tb.tdp = dpad;
    } else {
      table_fresh = false;
    }
    return tb;
  }

  // k_swap_at: the entries of mv (none: the units alone) into the adjacency and
  // the tables, and the pair lists of the units of rows[0..nrows) rebuilt when
  // the level plan's lists are current
  void entries_launch(const SwapTables& tb, const PlMove& mv, const int* rows, int nrows)
  {
    PlUnits units{};
    PlArgs pl{};
    if (tb.t32 && pl_fresh) {
      for (int q = 0; q < nrows; q++) {
        const int u = rows[q] / PG_UNIT;
        bool seen = false;
        for (int i = 0; i < units.cnt; i++) seen = seen || units.u[i] == u;
        if (!seen) units.u[units.cnt++] = u;
      }
      pl.nbr = d_nbr; pl.n = n; pl.dpad = dpad; pl.sp = lr.psp; pl.P = lr.parts; pl.thin = lr.thin; pl.list = lr.plist; pl.poff = lr.ppoff;
    }
    if (!mv.cnt && !units.cnt) return;
    auto kern = dpad + 1 <= 20 ? k_swap_at<20> : dpad + 1 <= 36 ? k_swap_at<36> : k_swap_at<64>;
    hipLaunchKernelGGL(kern, dim3(std::max(1, units.cnt)), dim3(PG_UNIT), 0, C.stream, d_adj, degree, tb, mv, units, pl);
    HIPC(hipGetLastError());
  }

  // A 2-opt move a-b, c-d -> a-c, b-d on the device copy, with the current
  // tables patched (patch_tables).  With the positions of the four entries
  // known (pos: found on the host copy by k_swap's rule, the move checked
  // there) one launch stores them and rebuilds the units (k_swap_at);
  // otherwise k_swap finds them (all or nothing) and k_swap_at rebuilds.
  void swap_launch(int a, int b, int c, int d, const int* pos = nullptr)
  {
    const SwapTables tb = patch_tables();
    if (has_numdeg) asym_fresh = false;    // an entry past num_degrees may change in the adjacency alone
    const int rows[4] = {a, b, c, d}, from[4] = {b, a, d, c}, to[4] = {c, d, a, b};
    PlMove mv{};
    if (pos) {
      for (int e = 0; e < 4; e++) { mv.row[e] = rows[e]; mv.pos[e] = pos[e]; mv.from[e] = from[e]; mv.to[e] = to[e]; }
      mv.cnt = 4;
    } else {
      hipLaunchKernelGGL(k_swap, dim3(1), dim3(64), 0, C.stream, d_adj, degree, a, b, c, d, d_err, tb);
      HIPC(hipGetLastError());
    }
    entries_launch(tb, mv, rows, 4);
  }
  ODPX_Plan plan{};
  LevelRun lr;
  ResRun rr;
  int guess_levels = 0;                 // levels the last level-plan evaluation needed
  // the count-only last level goes over a list of the chunks its level before
  // left unsaturated (k_sparse) while the last evaluations left few: their share
  // of the 16-byte chunks (bounded by the missing pairs over the chunks) at most
  // list_frac_env(), or after a dense one at most half that (no flip-flop of the
  // captured launch sequence between evaluations of similar graphs)
  bool list_on = true;
  // neighbours a thin level takes (0: the last level's predecessor runs whole),
  // from the last evaluation's reached pairs
  int thin_k = 0;
  int batch_cap = MAX_BATCH_LEVELS;     // gather levels launched between two host reads (serving: few)
  hipStream_t st = nullptr;             // launch stream (the library's main stream unless set)
  bool timed() const { return g_stats_on && st == C.stream; }

  // hipGraph of one evaluation's launch sequence: replayed while the plan, the
  // buffers, the adjacency pointer and (level plan) the first batch are unchanged
  hipGraphExec_t gexec = nullptr;
  long long g_key = -1;
  const int* g_adj = nullptr;
  long long g_seen = -1;                      // key of the last eager evaluation, for the repeat test
  const int* g_seen_adj = nullptr;
  void drop_graph()
  {
    if (gexec) HIPC(hipGraphExecDestroy(gexec));
    gexec = nullptr;
    g_key = -1;
    g_seen = -1;
    g_seen_adj = nullptr;
  }
  // Graphs are captured and replayed on the library's main stream only; the
  // serving engine's slots (their own streams) launch eagerly.
  bool graph_on() const { return graphs_env() && !timed() && st == C.stream; }
  const int* cur_adj() const { return ext_adj ? ext_adj : d_adj; }
  bool graph_ready(long long key) const { return gexec && g_key == key && g_adj == cur_adj(); }
  // Replay a graph only for a launch sequence that repeats: the first evaluation
  // of a key runs eagerly, the second captures, later ones replay.  One-off
  // evaluations (a new shape or plan every call) never pay for a capture.
  bool use_graph(long long key)
  {
    if (!graph_on()) return false;
    if (graph_ready(key) || (g_seen == key && g_seen_adj == cur_adj())) return true;
    g_seen = key;
    g_seen_adj = cur_adj();
    return false;
  }
  template <typename F> void capture(F enqueue, long long key)
  {
    drop_graph();
    hipGraph_t g;
    HIPC(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    enqueue();
    HIPC(hipStreamEndCapture(st, &g));
    HIPC(hipGraphInstantiate(&gexec, g, nullptr, nullptr, 0));
    HIPC(hipGraphDestroy(g));
    g_key = key;
    g_adj = cur_adj();
  }

  size_t adj_elems() const { return (size_t)(n / s) * degree; }

  void release()
  {
    if (st) HIPC(hipStreamSynchronize(st));    // a resident launch may still be finishing
    drop_graph();
    table_fresh = false;
    stage_is_device = false;
    mirror_ok = false;
    pend_patch.clear();
    dfree(&d_adj); dfree(&d_numdeg); dfree(&d_itable); dfree(&d_nbr); dfree(&d_err); dfree(&d_nbr16);
    dfree(&d_xy2row); dfree(&d_row2xy); dfree(&d_toff);
    dfree(&d_lmax); hfree(&h_lmax);
    nbr16_cap = 0; toff_cap = 0; geo_lmax = -1; geo_stale = false;
    hfree(&h_stage); hfree(&h_err); h_stage_dev = nullptr; adj_on_host = false;
    std::vector<int>().swap(h_mirror);
    dfree(&lr.bufs); dfree(&lr.cnt); dfree(&lr.done); dfree(&lr.tasks); dfree(&lr.wg_start); hfree(&lr.h_cnt);
    lr.h_cnt_dev = nullptr;
    hfree(&lvh); lvh_dev = nullptr; dfree(&d_lvseq); lvseq = 0;
    dfree(&lr.flags); hfree(&lr.h_acnt); dfree(&lr.wgm); dfree(&lr.list); dfree(&lr.tq);
    dfree(&lr.list_v); dfree(&lr.list2); dfree(&lr.list2_v);
    dfree(&lr.plist); dfree(&lr.ppoff);
    dfree(&rr.tasks); dfree(&rr.out); dfree(&rr.qhead); dfree(&rr.done); hfree(&rr.host); rr.host_dev = nullptr;
    dfree(&rr.part); rr.part_cap = 0;
    dfree(&d_bfs_q); dfree(&d_bfs_vis); dfree(&d_bfs_out); dfree(&d_bfs_next); hfree(&h_bfs_out);
    bfs_q_cap = bfs_vis_cap = 0; bfs = false;
    lr = LevelRun(); rr = ResRun();
    adj_cap = nbr_cap = stage_cap = 0;
    guess_levels = 0; list_on = true; thin_k = 0;
  }

  // shape of the graph; (re)allocates the graph buffers when they grow
  void shape(int fam, int nodes, int deg, int sym, int w, int h, const int* numdeg_full, int gs)
  {
    ctx_init();
    if (!st) st = C.stream;
    drop_graph();
    table_fresh = false;
    stage_is_device = false;
    mirror_ok = false;
    pend_patch.clear();
    family = fam; n = nodes; degree = deg; s = sym; width = w; height = h; grid_s = gs;
    nsrc = n / s;
    src_lo = 0; src_hi = nsrc;
    dpad = round_up(deg > 0 ? deg : 1, 4);
    has_numdeg = numdeg_full != nullptr;
    if (adj_elems() > adj_cap) { dfree(&d_adj); dalloc(&d_adj, adj_elems()); adj_cap = adj_elems(); }
    adj_on_host = false;
    if (adj_elems() > stage_cap) {
      hfree(&h_stage);
      halloc_coherent(&h_stage, &h_stage_dev, adj_elems());
      stage_cap = adj_elems();
    }
    size_t ne = (size_t)n * dpad;
    if (ne > nbr_cap) { dfree(&d_nbr); dalloc(&d_nbr, ne); nbr_cap = ne; }
    dp16 = round_up(deg > 0 ? deg : 1, 8);
    if (n <= 65536) {
      size_t ne16 = (size_t)n * dp16;
      if (ne16 > nbr16_cap) { dfree(&d_nbr16); dalloc(&d_nbr16, ne16); nbr16_cap = ne16; }
    }
    if (!d_err) { dalloc(&d_err, 1); halloc(&h_err, 1); HIPC(hipMemsetAsync(d_err, 0, sizeof(int), st)); }
    dfree(&d_numdeg);
    dfree(&d_itable);
    dfree(&d_xy2row); dfree(&d_row2xy);
    geo_lmax = -1; geo_stale = false;
    if (fam == 1 && s == 1) set_geometry(nullptr);    // rows are the cells themselves
    avg_deg = deg;
    if (numdeg_full) {
      dalloc(&d_numdeg, (size_t)n);
      HIPC(hipMemcpy(d_numdeg, numdeg_full, sizeof(int) * n, hipMemcpyHostToDevice));
      double t = 0;
      for (int i = 0; i < n; i++) t += numdeg_full[i];
      avg_deg = t / n;
    }
  }

  void set_itable(const int* itable)
  {
    drop_graph();                      // captured launches hold the old table's address
    table_fresh = false;               // the row-neighbour table follows the row order
    dfree(&d_itable);
    dalloc(&d_itable, (size_t)n);
    HIPC(hipMemcpy(d_itable, itable, sizeof(int) * n, hipMemcpyHostToDevice));
    set_geometry(itable);
  }

  // cell (x, y) = vertex x * height + y sits in row itable[vertex] (or row
  // vertex without a table); k_tile reads both directions
  void set_geometry(const int* itable)
  {
    std::vector<int> xy(n), rxy(n);
    for (int v = 0; v < n; v++) {
      const int r = itable ? itable[v] : v;
      xy[v] = r;
      rxy[r] = ((v / height) << 16) | (v % height);
    }
    dfree(&d_xy2row); dfree(&d_row2xy);
    dalloc(&d_xy2row, (size_t)n); dalloc(&d_row2xy, (size_t)n);
    HIPC(hipMemcpy(d_xy2row, xy.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    HIPC(hipMemcpy(d_row2xy, rxy.data(), sizeof(int) * n, hipMemcpyHostToDevice));
    const size_t ne = (size_t)n * dpad;
    if (ne > toff_cap) { dfree(&d_toff); dalloc(&d_toff, ne); toff_cap = ne; }
  }

  // largest |dx| or |dy| between a base row's cell and an entry's cell (entries
  // past num_degrees included: a larger value only turns k_tile off)
  int grid_lmax(const int* adj) const
  {
    const int based = n / s, bh = height / 2;
    int lm = 0;
    for (int i = 0; i < based; i++) {
      const int v = s == 4 ? (i / bh) * height + (i % bh) : i;
      const int vx = v / height, vy = v % height;
      for (int j = 0; j < degree; j++) {
        const int u = adj[(size_t)i * degree + j];
        if (u < 0 || u >= n) continue;
        lm = std::max(lm, std::max(abs(u / height - vx), abs(u % height - vy)));
      }
    }
    return lm;
  }

  // the change takes and adds as many entries u of row r as entries r of row u:
  // it leaves a symmetric table symmetric (and is checked on the device otherwise)
  static bool symmetric_change(const PlMove& mv)
  {
    auto delta = [&](int r, int u) {
      int c = 0;
      for (int e = 0; e < mv.cnt; e++) if (mv.row[e] == r) c += (mv.to[e] == u) - (mv.from[e] == u);
      return c;
    };
    for (int e = 0; e < mv.cnt; e++)
      for (int u : {mv.from[e], mv.to[e]})
        if (u != mv.row[e] && delta(mv.row[e], u) != delta(u, mv.row[e])) return false;
    return true;
  }

  // after an upload: small tables at once, larger ones on the device before the
  // next evaluation that needs it (256 x 256 grid, 131072 entries: 0.45 ms here, 0.03 there)
  void measure_lmax()
  {
    geo_stale = adj_elems() > LMAX_HOST_ENTRIES;
    if (!geo_stale) geo_lmax = grid_lmax(h_stage);
  }
  void settle_lmax()
  {
    if (!geo_stale) return;
    geo_stale = false;
    if (!d_lmax) { dalloc(&d_lmax, 1); halloc(&h_lmax, 1); }
    hipLaunchKernelGGL(k_clear, dim3(1), dim3(64), 0, st, (u64*)nullptr, 0, d_lmax, 1);
    const int grid = (int)std::min<size_t>((adj_elems() + 2047) / 2048, 256);
    hipLaunchKernelGGL(k_lmax, dim3(grid), dim3(256), 0, st, d_adj, n / s, degree, width, height, s, d_lmax);
    HIPC(hipGetLastError());
    HIPC(hipMemcpyAsync(h_lmax, d_lmax, sizeof(int), hipMemcpyDeviceToHost, st));
    HIPC(hipStreamSynchronize(st));
    geo_lmax = *h_lmax;
  }

  // a few changed entries against the last upload (at most RES_PATCH_MAX, of a
  // regular s = 1 table, every new id valid) under the resident plan with its
  // table current: queue them for the next launch (which stores them into the
  // table and the adjacency first) instead of sending and rebuilding the table.
  // The annealing pattern -- a 2-opt move, then ODP_Set_aspl on the same array
  // -- changes four entries.
  bool upload_as_patch(const int* a)
  {
    const bool lev = plan.plan == ODPX_PLAN_LEVEL && !bfs;   // the BFS kind rebuilds its table every run
    if ((plan.plan != ODPX_PLAN_RESIDENT && !lev) || s != 1 || grid_s || has_numdeg || ext_adj || adj_on_host)
      return false;
    if (!stage_is_device || !table_fresh || table_src != d_adj || !pend_patch.empty()) return false;
    const size_t m = adj_elems(), chunk = 64;
    int idx[RES_PATCH_MAX];
    int k = 0;
    for (size_t c = 0; c < m; c += chunk) {
      const size_t len = std::min(chunk, m - c);
      if (memcmp(a + c, h_stage + c, sizeof(int) * len) == 0) continue;
      for (size_t i = c; i < c + len; i++)
        if (a[i] != h_stage[i]) {
          if (k == RES_PATCH_MAX || a[i] < 0 || a[i] >= n) return false;
          idx[k++] = (int)i;
        }
    }
    mirror_ok = false;
    if (lev) {
      // the level plan stores them now (k_swap_at: adjacency, tables, units)
      static_assert(RES_PATCH_MAX <= PL_MOVE_MAX, "a small change fits one launch");
      PlMove mv{};
      int rows[RES_PATCH_MAX];
      for (int q = 0; q < k; q++) {
        const int i = idx[q];
        mv.row[q] = rows[q] = i / degree; mv.pos[q] = i % degree; mv.from[q] = h_stage[i]; mv.to[q] = a[i];
        h_stage[i] = a[i];
      }
      mv.cnt = k;
      if (!symmetric_change(mv)) asym_fresh = false;
      entries_launch(patch_tables(), mv, rows, k);
    } else {
      for (int q = 0; q < k; q++) {
        const int i = idx[q];
        h_stage[i] = a[i];
        const int e[3] = {i / degree, i % degree, a[i]};
        pend_patch.insert(pend_patch.end(), e, e + 3);
      }
    }
    if (d_xy2row && k) measure_lmax();
    return true;
  }

  void upload(const void* adjacency)
  {
    trace("upload");
    if (upload_as_patch((const int*)adjacency)) return;
    table_fresh = false;
    stage_is_device = true;
    mirror_ok = false;
    memcpy(h_stage, adjacency, sizeof(int) * adj_elems());
    if (plan.plan == ODPX_PLAN_RESIDENT && !ext_adj &&
        sizeof(int) * adj_elems() <= (s == 1 && !grid_s ? ZC_MAX_BYTES : ZC_MAX_BYTES_SYM)) {
      adj_on_host = true;          // the next table build reads it from host memory
    } else {
      adj_on_host = false;
      HIPC(hipMemcpyAsync(d_adj, h_stage, sizeof(int) * adj_elems(), hipMemcpyHostToDevice, st));
    }
    if (d_xy2row) measure_lmax();
  }

  // d_adj holds the last upload (copies it from host memory if it is still only there);
  // called outside stream capture before anything but the resident table build reads d_adj
  void flush_adj()
  {
    apply_pending();
    if (!adj_on_host) return;
    adj_on_host = false;
    HIPC(hipMemcpyAsync(d_adj, h_stage, sizeof(int) * adj_elems(), hipMemcpyHostToDevice, st));
  }

  // ---- plans ----
  // widest block the resident kernel can run for this graph with `threads`
  // threads: one LDS buffer of n*wb*4 bytes and n <= res_rows(wb)*threads rows
  int resident_wb_max(int threads = 1024) const
  {
    if (n > 65535 || !d_nbr16) return 0;
    for (int wb = RES_WB_MAX; wb >= 1; wb >>= 1)
      if ((size_t)n * wb * 4 <= LDS_DYN_MAX && n <= res_rows(wb) * threads) return wb;
    return 0;
  }

  // k_tile's tile side for this adjacency (env ODP_HIP_TILE_SIDE overrides)
  int tile_side() const
  {
    const char* v = getenv("ODP_HIP_TILE_SIDE");
    if (v) { const int t = atoi(v); if (t >= TILE_MIN && t <= 56 && t % 2 == 0) return t; }
    return TILE_MIN;
  }

  // k_tile applies to grid graphs whose rows are cells, with table width <= 16
  // and at least 4 cells per tile (its flags live in the changed-flag array)
  bool tile_capable() const
  {
    const int ntiles = ((width + TILE_MIN - 1) / TILE_MIN) * ((height + TILE_MIN - 1) / TILE_MIN);
    return d_xy2row && dpad <= 16 && 4 * ntiles <= n && !ext_adj;
  }

  int parts_default(int kw) const
  {
    return kw == LEVEL_BLOCK_WORDS && (n >= PG_MIN_ROWS || (n >= PG_MIN_ROWS_NARROW && dpad <= 16)) ? PG_PARTS : 0;
  }

  ODPX_Plan default_plan(int kind) const
  {
    ODPX_Plan p{};
    const char* env = getenv("ODP_HIP_PLAN");
    bool force_level = env && strcmp(env, "level") == 0;
    bool force_res = env && strcmp(env, "resident") == 0;
    int wbmax = resident_wb_max();
    if ((wbmax > 0 && !force_level) || (force_res && wbmax > 0)) {
      p.plan = ODPX_PLAN_RESIDENT;
      const int wb = res_width(n, nsrc, wbmax, C.ncu);
      p.wb = wb;
      // workgroup size: a row or two a thread up to n = 1024 (n = 1024, d = 6:
      // 22.9 us with 512 threads, 24.6 with 256, 23.3 with 1024; n = 512: the three
      // within 3 %), all 1024 threads from n = 2048 on (2048, d = 3: 31.9 against 34.2
      // with 512; 4096, d = 4, 8, 16: 35.2 / 32.1 / 35.1 against 37.8 / 33.6 / 36.4;
      // 5001, d = 10: 39.8 against 41.7)
      p.threads = 1024;
      for (int th : {256, 512, 1024})
        if (n <= res_rows(wb) * th && (n >= 2048 ? th == 1024 : (n > 512 ? th >= 512 : true))) { p.threads = th; break; }
      return p;
    }
    // Column blocks of 16 words (1024 sources), each stored as its own
    // contiguous n x 128 B slab, with each XCD owning whole slabs, so the rows
    // one XCD gathers from stay within a few MiB (its L2).  MATRIX
    // keeps every block resident and advances all of them per launch (the full
    // bit matrix, blocked); MATRIX_SAVING keeps SAVING_GROUP blocks resident
    // at a time, bounding memory as the reference does (aspl.c:77-119), where
    // ODP_ASPL asks for it or all blocks would take too much (SAVING_BYTES).
    p.plan = ODPX_PLAN_LEVEL;
    int W = (nsrc + 63) / 64;
    p.kw = std::min(LEVEL_BLOCK_WORDS, W);
    p.upw = 8;
    p.seg_major = 0;
    p.xcd = 1;
    p.group = (kind == KIND_MATRIX) ? 0 : SAVING_GROUP;
    p.direct = -1;
    // slabs larger than an XCD's L2 (n x 128 B > 4 MB): the XCD-phased gather
    // (measured against k_level at n = 16386-28000, d = 8, 16, 32: from n = 24576 the
    // part gather is 4-30 % faster at every degree but one (28000, d = 32: 2 % slower);
    // at n = 20000 it is 11-22 % faster for d <= 16 and 5 % slower for d = 32)
    p.parts = parts_default(p.kw);
    if (p.group && p.parts && s == 1 && !getenv("ODP_ASPL")) {
      const size_t bytes = (size_t)((W + p.kw - 1) / p.kw) * 2 * n * p.kw * 8;
      size_t avail = 0, total = 0;
      if (bytes <= SAVING_BYTES && hipMemGetInfo(&avail, &total) == hipSuccess && bytes <= avail / 8) p.group = 0;
    }
    if (tile_capable()) {
      // grid graphs: 2-word blocks and temporal tiles (k_tile); MATRIX_SAVING
      // keeps the same number of source words resident as with 16-word blocks
      p.kw = 2;
      p.tile = 1;
      p.parts = 0;
      if (p.group) p.group = SAVING_GROUP * LEVEL_BLOCK_WORDS / 2;
    }
    return p;
  }

  bool plan_valid(const ODPX_Plan& p) const
  {
    if (p.plan == ODPX_PLAN_RESIDENT) {
      if (p.wb != 1 && p.wb != 2 && p.wb != 4 && p.wb != 8) return false;
      if (p.threads != 256 && p.threads != 512 && p.threads != 1024) return false;
      return n <= 65535 && d_nbr16 && (size_t)n * p.wb * 4 <= LDS_DYN_MAX && n <= res_rows(p.wb) * p.threads;
    }
    if (p.plan == ODPX_PLAN_LEVEL) {
      if (!(p.kw >= 0 && p.upw >= 1 && p.upw <= 64 && p.group >= 0)) return false;
      if (p.tile != 0 && !(p.tile == 1 && p.kw == 2 && tile_capable())) return false;
      // direct K that does not apply to this graph's blocks falls back to k_level0
      if (p.batch != 0 && p.batch != 4 && p.batch != 8 && p.batch != 16) return false;
      if (p.parts != 0 && p.parts != 2 && p.parts != 4) return false;
      return p.direct == 0 || p.direct == -1 || (p.direct >= 2 && p.direct <= DIRECT_KMAX);
    }
    return false;
  }

  // ---- direct enumeration of the first levels (k_direct) ----
  // gather levels run k_pgather: a plan with parts, plain (not frontier, not tile) levels
  bool pg_on() const { return plan.plan == ODPX_PLAN_LEVEL && lr.parts > 0 && !lv.fr && !lv.tk; }
  // whether the gather levels' rows are streamed: the resident blocks' two buffers pass the last-level cache
  int pg_streamed() const { return (size_t)lr.group * 2 * n * lr.kwp * 8 > MALL_BYTES ? 1 : 0; }
  // k_direct reads the 16-bit table when it exists with the 32-bit table's width
  bool direct16() const
  {
    return plan.plan == ODPX_PLAN_LEVEL && lr.direct > 0 && d_nbr16 && dp16 == dpad;
  }
  long direct_tree(int K) const
  {
    long t = 0, m = 1;
    for (int i = 0; i <= K; i++) { t += m; m *= dpad; if (m > (1L << 40)) m = 1L << 40; }
    return t;
  }
  // ints k_direct's depth lists take per wave.  A launch over every source (all)
  // keeps breadth-first frontiers, at most degree^d ids at depth d, 16 bits each
  // when they fit; the others whole walk trees: 4 ints for depth 0, dpad^d for 0 < d < K
  long direct_list(int K, bool all) const
  {
    long t = all ? 1 : 4, m = 1;
    for (int i = 1; i < K; i++) { m *= all ? std::max(degree, 1) : dpad; t += m; }
    return all && n <= 65536 ? (t + 1) / 2 : t;
  }
  // every source in one launch of `group` blocks of kw words
  bool direct_all(int kw, int group) const
  {
    return src_lo == 0 && src_hi == n && (int64_t)group * kw * 64 >= n;
  }
  void (*direct_kernel(int kw, int group) const)(DirectArgs)
  {
    const bool id16 = direct16();
    if (!direct_all(kw, group)) return id16 ? k_direct<false, true, false> : k_direct<false, false, false>;
    return id16 ? k_direct<true, true, true> : n <= 65536 ? k_direct<true, false, true> : k_direct<true, false, false>;
  }
  size_t direct_lds(int K, int kw, int group, int nw) const
  {
    const size_t words = (size_t)group * kw, chunks = (words + 127) / 128;
    return (size_t)nw * (words * 8 + (size_t)direct_list(K, direct_all(kw, group)) * 4) + (size_t)K * chunks * 64 * 4;
  }
  // waves per workgroup k_direct can run with (0: not applicable): the block
  // rows must be a power of two of 2..128 words and one row bitmap must fit
  // LDS.  Each wave holds a row bitmap, so LDS bounds the waves per CU: take
  // the workgroup size (1..8 waves) that keeps the most of them (at n=65536,
  // d=16: 8 waves, 2 workgroups, 16 waves per CU against 12 with 4-wave
  // workgroups; the evaluation took 1.929 instead of 1.959 ms)
  int direct_waves(int K, int kw, int group) const
  {
    if (K < 2 || K > DIRECT_KMAX || kw < 2 || kw > 128 || (kw & (kw - 1)) || dpad > 1024) return 0;
    int best = 0, best_waves = 0;
    for (int nw = 1; nw <= 8; nw++) {
      const size_t l = direct_lds(K, kw, group, nw);
      if (l > LDS_DYN_MAX) break;
      const int waves = nw * (int)(LDS_LIMIT / l);
      if (waves > best_waves) { best = nw; best_waves = waves; }
    }
    return best;
  }
  int direct_auto(int kw, int group) const
  {
    int best = 0;
    for (int K = 2; K <= DIRECT_KMAX && K < n; K++)
      if (direct_tree(K) <= DIRECT_TREE_MAX && direct_waves(K, kw, group) > 0) best = K;
    return best;
  }

  // ---- level plan: buffers and task table ----
  void setup_level()
  {
    LevelRun& r = lr;
    int W = (src_hi - src_lo + 63) / 64;
    int kw = plan.kw > 0 ? std::min(plan.kw, W) : W;
    int kwp = kw <= 128 ? (1 << (ilog2(std::max(kw, 2) - 1) + 1)) : round_up(kw, 128);
    if (kwp < kw) kwp = kw;
    int ntasks = (W + kw - 1) / kw;
    int group = plan.group > 0 ? std::min(plan.group, ntasks) : ntasks;
    int lanes = std::min(64, kwp / 2);
    int lpr_log2 = ilog2(lanes);
    int rpw = 64 >> lpr_log2;
    int segs = kwp / (2 * lanes);
    int rgroups = (n + rpw - 1) / rpw;
    int units = rgroups * segs;
    // bit buffers for `group` column blocks; group g of blocks reuses them
    size_t words = (size_t)group * 2 * n * kwp;
    if (words > r.buf_words) { dfree(&r.bufs); dalloc(&r.bufs, words); r.buf_words = words; }
    const size_t fbytes = (size_t)group * 4 * segs * n;
    if (fbytes > r.flag_bytes) {
      dfree(&r.flags); dalloc(&r.flags, fbytes); r.flag_bytes = fbytes;
      HIPC(hipMemset(r.flags, 0, fbytes));           // marks start clear (later levels keep them so)
    }
    if ((size_t)ntasks > r.task_cap) {
      dfree(&r.cnt); dfree(&r.done); dfree(&r.tasks); dfree(&r.wg_start); hfree(&r.h_cnt);
      dalloc(&r.cnt, (size_t)3 * RING * ntasks);     // counts, changed, processed
      // done flags, the lists' counters (all cleared by the preparation), the table's asymmetry flag
      dalloc(&r.done, (size_t)ntasks + LIST_COUNTERS + 1);
      hfree(&r.h_acnt); halloc(&r.h_acnt, (size_t)RING * ntasks + 1);
      dalloc(&r.tasks, (size_t)ntasks); dalloc(&r.wg_start, (size_t)ntasks + 1);
      halloc_coherent(&r.h_cnt, &r.h_cnt_dev, (size_t)RING * ntasks);
      r.task_cap = ntasks;
    }
    // the previous contents are never read: level 0 rewrites every word it uses
    r.n = n; r.ntasks = ntasks; r.group = group; r.kw = kw; r.kwp = kwp; r.segs = segs;
    r.upw = plan.upw; r.seg_major = plan.seg_major; r.xcd = plan.xcd; r.urow = (lpr_log2 == 6);
    r.batch = plan.batch == 8 || plan.batch == 16 ? plan.batch : 4;
    r.per_task_wg = (units + 4 * r.upw - 1) / (4 * r.upw);
    if (!r.list) dalloc(&r.list, (size_t)LIST_CAP);
    r.list_n = r.done + ntasks;
    r.asym = r.list_n + LIST_COUNTERS;
    r.list_cap = (list_cap_env() + LIST_SUBS - 1) / LIST_SUBS;        // per sub-list
    if (plan.tile && tile_capable()) {
      const size_t cap = 3 + (size_t)group * ((width + TILE_MIN - 1) / TILE_MIN) * ((height + TILE_MIN - 1) / TILE_MIN);
      if (cap > r.tq_cap) { dfree(&r.tq); dalloc(&r.tq, cap); r.tq_cap = cap; }
    }
    const size_t wbytes = (size_t)group * 2 * r.per_task_wg;
    if (wbytes > r.wgm_bytes) {
      dfree(&r.wgm); dalloc(&r.wgm, wbytes); r.wgm_bytes = wbytes;
      HIPC(hipMemset(r.wgm, 0, wbytes));
    }
    r.fold = false;
    // the XCD-phased gather applies to 16-word rows, runs of at most 63 ids and
    // ids below 2^22 (the pair lists pack the row in the unit beside the id)
    r.parts = (plan.parts > 0 && kwp == 16 && dpad + 1 <= 63 && n <= (1 << 22)) ? plan.parts : 0;
    plan.parts = r.parts;              // the plan reports what runs
    if (r.parts) {
      r.psp = round_up(dpad + 1, 4);
      r.pupt = (n + PG_UNIT - 1) / PG_UNIT;
      const size_t nl = (size_t)r.pupt * PG_UNIT * r.psp, np = (size_t)r.pupt * PG_OFF;
      if (nl > r.plist_cap) { dfree(&r.plist); dalloc(&r.plist, nl); r.plist_cap = nl; }
      if (np > r.ppoff_cap) { dfree(&r.ppoff); dalloc(&r.ppoff, np); r.ppoff_cap = np; }
      if (!r.list_v) {
        dalloc(&r.list_v, (size_t)THIN_CAP);
        dalloc(&r.list2, (size_t)THIN2_CAP); dalloc(&r.list2_v, (size_t)THIN2_CAP);
      }
      // persistent grid: every workgroup the CUs hold at once, a multiple of the XCD count
      int occ = 0, occ_ls = 0;
      HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, k_pgather<false, true, true>, PG_WG, 0));
      HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ_ls, k_pgather<true, true, true>, PG_WG, 0));
      occ = std::max(1, std::min(occ, occ_ls));
      r.pgrid = ODP_NXCD * std::max(1, C.ncu / ODP_NXCD) * occ;
      // folded levels need the whole matrix resident, a task per PG_UNIT rows
      r.fold = s == 1 && !grid_s && src_lo == 0 && src_hi == n && group == ntasks && kw == LEVEL_BLOCK_WORDS &&
               pg_fold_env();
      const int T = ntasks;
      r.cut_full = pg_cut((double)T * r.pupt / ODP_NXCD, 0, r.pgrid / ODP_NXCD);
      r.cut_fold = pg_cut((double)T * ((T + (T & 1)) / 2) / ODP_NXCD, T & 1 ? 0 : T / 2.0 / ODP_NXCD,
                          r.pgrid / ODP_NXCD);
    }
    int K = plan.direct;
    while (K >= 2 && (direct_tree(K) > DIRECT_TREE_CAP || !direct_waves(K, kw, group))) K--;
    r.direct = plan.direct == -1 ? direct_auto(kw, group) : (K >= 2 ? K : 0);
    if (r.direct >= n) r.direct = 0;
    plan.direct = r.direct;            // the plan reports the K that runs
    if (r.direct) {
      // Over every source: the largest workgroup, up to 16 waves, that LDS holds --
      // every workgroup adds its counts with an atomic per block and level, so few
      // large ones beat more waves in small ones (n = 28000, d = 16: 16 waves 74 us,
      // 2 x 8 80, 2 x 10 93, 5 x 4 102, 20 x 1 240; n = 100000, d = 8: 10 waves).
      r.dnw = direct_waves(r.direct, kw, group);
      if (direct_all(kw, group))
        for (int nw = 16; nw >= 1; nw--)
          if (direct_lds(r.direct, kw, group, nw) <= LDS_DYN_MAX) { r.dnw = nw; break; }
      r.dlds = direct_lds(r.direct, kw, group, r.dnw);
      int per_cu = 0;
      HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, direct_kernel(kw, group), 64 * r.dnw, r.dlds));
      per_cu = std::max(1, std::min(per_cu, 32 / r.dnw));
      r.dgrid = std::max(1, std::min((n + r.dnw - 1) / r.dnw, per_cu * C.ncu));
    }
    std::vector<LevelTask> ht(ntasks);
    std::vector<int> ws(ntasks + 1);
    r.l.assign(ntasks, 0);
    for (int t = 0; t < ntasks; t++) {
      LevelTask& T = ht[t];
      T.nbr = d_nbr;
      T.buf0 = r.bufs + (size_t)(t % group) * 2 * n * kwp;
      T.buf1 = T.buf0 + (size_t)n * kwp;
      T.cnt = r.cnt + t;
      T.done = r.done + t;
      T.n = n; T.dpad = dpad; T.kwp = kwp;
      T.src0 = src_lo + t * kw * 64;
      T.l = std::min(kw * 64, src_hi - T.src0);
      T.lpr_log2 = lpr_log2; T.segs = segs; T.rgroups = rgroups; T.units = units;
      T.seg_major = r.seg_major; T.cstride = ntasks; T.pad = 0;
      T.ccnt = r.cnt + (size_t)RING * ntasks + t;
      T.acnt = r.cnt + (size_t)2 * RING * ntasks + t;
      T.chg0 = r.flags + (size_t)(t % group) * 4 * segs * n;
      T.chg1 = T.chg0 + (size_t)segs * n;
      T.act0 = T.chg0 + (size_t)2 * segs * n;
      T.act1 = T.chg0 + (size_t)3 * segs * n;
      T.asym = r.asym;
      T.wgm0 = r.wgm + (size_t)(t % group) * 2 * r.per_task_wg;
      T.wgm1 = T.wgm0 + r.per_task_wg;
      r.l[t] = T.l;
      ws[t] = t * r.per_task_wg;     // blocks are equal: the starts of a group rebase to 0
    }
    ws[ntasks] = ntasks * r.per_task_wg;
    HIPC(hipMemcpy(r.tasks, ht.data(), sizeof(LevelTask) * ntasks, hipMemcpyHostToDevice));
    HIPC(hipMemcpy(r.wg_start, ws.data(), sizeof(int) * (ntasks + 1), hipMemcpyHostToDevice));
  }

  // ---- resident plan: task table ----
  void setup_resident()
  {
    ResRun& r = rr;
    r.wb = plan.wb; r.threads = plan.threads;
    int b = 32 * r.wb;
    int ntasks = (src_hi - src_lo + b - 1) / b;
    if ((size_t)ntasks > r.task_cap) {
      dfree(&r.tasks);
      dalloc(&r.tasks, (size_t)ntasks);
      r.task_cap = ntasks;
    }
    if (!r.out) {
      // the queue head and the arrival counter are zeroed once here: every
      // launch leaves them at zero for the next (res_finish).  `out` is the
      // kernel's per-graph accumulator argument, unused by single-graph
      // launches (their totals go through the per-workgroup slots)
      dalloc(&r.out, 1); dalloc(&r.qhead, 1); dalloc(&r.done, 1);
      halloc_coherent(&r.host, &r.host_dev, 1);
      r.host->seq = r.seq;             // no launch has written it yet
      HIPC(hipMemsetAsync(r.out, 0, sizeof(ResOut), st));
      HIPC(hipMemsetAsync(r.qhead, 0, sizeof(int), st));
      HIPC(hipMemsetAsync(r.done, 0, sizeof(u32), st));
      HIPC(hipStreamSynchronize(st));
    }
    std::vector<ResTask> ht(ntasks);
    for (int t = 0; t < ntasks; t++) {
      ResTask& T = ht[t];
      T.nbr = d_nbr16; T.n = n; T.dp = dp16; T.src0 = src_lo + t * b; T.l = std::min(b, src_hi - T.src0);
      T.s = s; T.graph = 0; T.wb = r.wb; T.dq = (std::max(degree, 1) + 3) / 4;
      T.deg = std::max(degree, 1); T.walk = res_walk_env(n, T.deg, T.l);
    }
    HIPC(hipMemcpy(r.tasks, ht.data(), sizeof(ResTask) * ntasks, hipMemcpyHostToDevice));
    r.ntasks = ntasks;
    r.lds = (size_t)n * r.wb * 4;
    int per_cu = (int)std::max<size_t>(1, LDS_LIMIT / (r.lds + LDS_STATIC));
    per_cu = std::min(per_cu, 2048 / r.threads);
    r.grid = std::max(1, std::min(ntasks, per_cu * C.ncu));
    if ((size_t)r.grid > r.part_cap) { dfree(&r.part); dalloc(&r.part, (size_t)r.grid); r.part_cap = r.grid; }
  }

  void apply_plan(const ODPX_Plan& p)
  {
    flush_adj();
    drop_graph();
    table_fresh = false;
    plan = p;
    if (plan.plan == ODPX_PLAN_LEVEL) setup_level();
    else setup_resident();
    guess_levels = 0; list_on = true; thin_k = 0;
  }

  // ---- evaluation of the adjacency on the device ----
  // zeroes what it is given and (table) builds the current plan's table
  void prepare(u64* z64, int nz64, u32* z32, int nz32, bool table = true)
  {
    PrepArgs a;
    const bool res = plan.plan == ODPX_PLAN_RESIDENT;
    const bool from_host = adj_on_host && !ext_adj;     // set only under the resident plan
    a.adj = from_host ? h_stage_dev : (ext_adj ? ext_adj : d_adj);
    a.adj_copy = from_host ? d_adj : nullptr;
    a.adj_elems = from_host ? (int64_t)adj_elems() : 0;
    if (from_host) adj_on_host = false;
    a.numdeg = d_numdeg; a.itable = d_itable; a.err = d_err;
    a.nbr = res ? nullptr : d_nbr;
    a.nbr16 = res || direct16() ? d_nbr16 : nullptr;     // the level plan's k_direct reads 16-bit ids
    a.n = n; a.s = s; a.degree = degree; a.dpad = res ? dp16 : dpad;
    a.width = width; a.height = height; a.grid_s = grid_s;
    a.zero64 = z64; a.nzero64 = nz64; a.zero32 = z32; a.nzero32 = nz32;
    if (!table) { a.nbr = nullptr; a.nbr16 = nullptr; a.dpad = 0; }
    const int64_t total = std::max<int64_t>((int64_t)n * a.dpad, std::max(nz64, nz32));
    int grid = (int)std::min<int64_t>(std::max<int64_t>(1, (total + 255) / 256), 4096);
    TimedLaunch tl;
    timed_begin(tl, T_OTHER, -1, st);
    hipLaunchKernelGGL(k_prepare, dim3(grid), dim3(256), 0, st, a);
    HIPC(hipGetLastError());
    timed_end(tl);
  }

  void check_err()
  {
    if (*h_err) {
      int e = *h_err;
      *h_err = 0;
      HIPC(hipMemsetAsync(d_err, 0, sizeof(int), st));
      if (e & 2) ODP_ERROR("num_degrees holds a value outside [0, degree]\n");
      if (e & 8) ODP_ERROR("libodp_hip: internal error: a grid table entry is longer than measured\n");
      if (e & 4) ODP_ERROR("libodp_hip: internal error: a device swap found no such edge\n");
      ODP_ERROR("adjacency holds a vertex id outside [0, nodes) within num_degrees\n");
    }
  }

  // ---- level plan as a resumable sequence ----
  // lv_begin() enqueues prepare, the first levels and the first batch of
  // gather levels of the first group, ending with copies of the counter ring
  // and the error flag to the host.  Once the stream has passed those copies,
  // lv_step() examines the counters and enqueues the next batch (or the next
  // group), returning true when the evaluation is complete; lv_result() then
  // gives the ordered-pair excess over n(n-1), the diameter and whether the
  // graph is disconnected.  Column blocks run `group` at a time (all at once
  // for MATRIX); every launch advances each block of the group by one level.
  struct LvTask { int running; u64 sum, prev; int lwork; };
  struct LvState {
    int K = 0, L1 = 1, nzero = 0, be0 = 2;
    bool fr = false;                    // frontier-mode level kernel (graphs with many levels)
    int fr_from = 1;                    // ... from this level on (every row of it; >= L1)
    int tk = 0;                         // k_tile levels per launch (0: one k_level launch per level)
    int tside = TILE_MIN;               // k_tile's tile side (halo = (64 - side) / 2)
    bool thin = false;                  // the level before spec runs thin
    int spec = -1;                      // level of the current group launched count-only (expected last)
    bool graphed = false;
    bool pend_fin = false;              // the enqueued batch ends with k_lvfin (sequence number lvseq)
    bool fresh = false, plfresh = false; // the preparation keeps the table / the pair lists
    bool check = false;                  // ... and checks the table's symmetry
    int asym = -1;                       // whether it is not symmetric (where folded levels ask; -1: not handed over)
    int first = 0, cnt_t = 0;
    int launched = 0, examined = 0, running = 0, batch_end = 0;
    std::vector<LvTask> sts;
    bool any_disc = false;
    int max_d = 1, lmax = 0;
    double miss[LV_MISS_LEVELS] = {};   // pairs not reached after level L, over the tasks
  } lv;

  void lv_level0()
  {
    LevelRun& r = lr;
    const int K = lv.K, first = lv.first, cnt_t = lv.cnt_t;
    TimedLaunch tl;
    timed_begin(tl, T_OTHER, 0, st);
    if (K) {
      DirectArgs a;
      a.nbr = d_nbr;
      a.out = r.bufs + ((K & 1) ? (size_t)n * r.kwp : 0);     // the buffer level K reads
      a.tstride = (int64_t)2 * n * r.kwp;
      a.cnt = r.cnt + first; a.cstride = r.ntasks;
      a.n = n; a.dpad = dpad; a.kw = r.kw; a.kwl = ilog2(r.kw);
      a.src_lo = src_lo + first * r.kw * 64;
      a.nsrc = std::min(cnt_t * r.kw * 64, src_hi - a.src_lo);
      a.ntask = cnt_t; a.words = cnt_t * r.kw; a.chunks = (a.words + 127) / 128;
      a.K = K; a.list = (int)direct_list(K, direct_all(r.kw, r.group));
      // streamed stores when the row-part gather reads the rows next, by its own rule (measured:
      // n=65536 591 -> 600 evaluations/s); the tile plan re-reads them soon (the grid ran 2.7 % slower)
      a.nt = pg_on() ? pg_streamed() : 0;
      const bool id16 = direct16();
      const unsigned q = (unsigned)(dpad / (id16 ? 8 : 4));
      a.nbr16 = d_nbr16;
      a.qmul = q > 1 ? (unsigned)((1ULL << 32) / q + 1) : 0u;
      long m = 1;
      for (int i = 0; i < 8; i++) { a.pw[i] = (int)m; m = std::min<long>(m * dpad, 1L << 30); }
      hipLaunchKernelGGL(direct_kernel(r.kw, r.group), dim3(r.dgrid), dim3(64 * r.dnw), r.dlds, st, a);
    } else {
      hipLaunchKernelGGL(k_level0, dim3(cnt_t * r.per_task_wg), dim3(LEVEL_WG), 0, st,
                         r.tasks + first, r.wg_start, cnt_t, RING, r.upw, r.xcd);
    }
    HIPC(hipGetLastError());
    timed_end(tl);
  }

  // whether the level before a count-only level `spec` lists its unsaturated chunks
  bool listed_at(int spec) const
  {
    return spec >= 0 && !lv.fr && list_ok() && spec - 1 >= lv.L1 && lr.ntasks < 65536 && n < (1 << 24) && lr.kwp < (1 << 24);
  }

  // gather levels [from, to) of the current group, then the counter and error copies.
  // The count-only level counts just the chunks the level before it listed as
  // unsaturated (plain kernel variant, when that level is a gather level).
  void lv_levels(int from, int to)
  {
    LevelRun& r = lr;
    if (lv.tk) {
      for (int L = from; L < to; L += lv.tk) lv_tile(L);
      lv_copies(to);
      return;
    }
    const bool listed = listed_at(lv.spec) && from < lv.spec;   // the level before it is in this batch
    for (int L = from; L < to; L++) {
      int mode = LV_STORE | LV_COUNT;
      if (L == lv.spec) mode = listed ? LV_SPARSE : LV_COUNT;
      else if (listed && L == lv.spec - 1) {
        mode = lv.thin ? LV_LIST | LV_THIN : mode | LV_LIST;
        if (lv.first > 0) {            // the preparation cleared the first group's
          hipLaunchKernelGGL(k_clear, dim3(LIST_COUNTERS / 256), dim3(256), 0, st, (u64*)nullptr, 0, (int*)r.list_n,
                             LIST_COUNTERS);
          HIPC(hipGetLastError());
        }
      }
      lv_launch(L, mode);
    }
    lv_copies(to);
  }

  // levels L .. L+tk-1 of the current group by temporal tiles (k_tile)
  void lv_tile(int L)
  {
    LevelRun& r = lr;
    const int j = (L - lv.L1) / lv.tk;             // launch number of the group
    TileArgs g;
    g.xy2row = d_xy2row; g.toff = d_toff;
    g.width = width; g.height = height;
    g.tile = lv.tside; g.halo = (TILE_RW - lv.tside) / 2;
    g.tiles_x = (width + g.tile - 1) / g.tile; g.tiles_y = (height + g.tile - 1) / g.tile;
    g.lmax = std::max(1, geo_lmax); g.k = lv.tk;
    g.dpar = (lv.L1 + j) & 1;                      // launch 0 reads what level L1 - 1 wrote
    g.fpar = j & 1; g.first = j == 0; g.xcd = r.xcd;
    const int units = lv.cnt_t * g.tiles_x * g.tiles_y;
    auto kern = dpad == 4 ? k_tile<4> : dpad == 8 ? k_tile<8> : dpad == 12 ? k_tile<12> : k_tile<16>;
    TimedLaunch tl;
    tl.nlev = lv.tk;
    timed_begin(tl, T_LEVEL, L, st);
    if (j == 0) hipLaunchKernelGGL(k_clear, dim3(1), dim3(64), 0, st, (u64*)nullptr, 0, (int*)r.tq, 1);
    hipLaunchKernelGGL(k_tile_plan, dim3(std::min((units + 255) / 256, 1024)), dim3(256), 0, st,
                       r.tasks + lv.first, lv.cnt_t, L, RING, g, r.tq);
    const int per_cu = TILE_ONE(dpad) ? 2 : 1;
    hipLaunchKernelGGL(kern, dim3(std::min(units, per_cu * C.ncu)), dim3(TILE_THREADS(dpad)), 0, st, r.tasks + lv.first, L, RING, g,
                       r.tq);
    HIPC(hipGetLastError());
    timed_end(tl);
  }

  void lv_launch(int L, int mode)
  {
    LevelRun& r = lr;
    const int grid = lv.cnt_t * r.per_task_wg;
    const bool thin = (mode & LV_THIN) || ((mode & LV_SPARSE) && lv.thin);
    const u32* asym = pg_on() && r.fold ? r.asym : nullptr;
    const LvList lst{r.list, r.list_n, thin ? std::min(r.list_cap, THIN_CAP / LIST_SUBS) : r.list_cap,
                     thin ? r.list_v : nullptr};
    const LvList lst2{r.list2, r.list_n + LIST_SUBS * LIST_PAD, std::min(r.list_cap, THIN2_CAP / LIST_SUBS), r.list2_v};
    TimedLaunch tl;
    tl.wr = (mode & LV_STORE) ? 1 : 0;
    tl.fold = asym != nullptr;
    tl.nbrs = (mode & LV_THIN) ? r.thin : -1;
    // k_sparse is timed apart: its work is the listed chunks, not a level
    timed_begin(tl, (mode & LV_SPARSE) ? T_OTHER : T_LEVEL, L, st);
    if (thin && (mode & LV_SPARSE)) {
      hipLaunchKernelGGL(k_thin, dim3(std::min(grid, SPARSE_GRID)), dim3(LEVEL_WG), 0, st, r.tasks + lv.first,
                         lv.cnt_t, L - 1, RING, lst, lst2, asym, (int)((double)n * std::min(r.thin, degree) / std::max(degree, 1)));
      hipLaunchKernelGGL(k_thin2, dim3(std::min(grid, SPARSE_GRID)), dim3(LEVEL_WG), 0, st, r.tasks + lv.first,
                         lv.cnt_t, L, RING, lst, lst2, asym);
    } else if (mode & LV_SPARSE) {
      hipLaunchKernelGGL(k_sparse, dim3(std::min(grid, SPARSE_GRID)), dim3(LEVEL_WG), 0, st,
                         r.tasks + lv.first, lv.cnt_t, L, RING, lst, asym);
    } else if (pg_on()) {
      PgArgs a;
      a.list = r.plist; a.poff = r.ppoff; a.n = n; a.sp = r.psp; a.P = r.parts;
      a.upt = r.pupt; a.ntasks = lv.cnt_t;
      a.asym = asym;
      a.cut_full = r.cut_full; a.cut_fold = r.cut_fold;
      const bool ls = (mode & LV_LIST) != 0;
      const bool nt = pg_streamed() != 0;
      auto kern = asym ? (ls ? (nt ? k_pgather<true, true, true> : k_pgather<true, false, true>)
                             : (nt ? k_pgather<false, true, true> : k_pgather<false, false, true>))
                       : (ls ? (nt ? k_pgather<true, true, false> : k_pgather<true, false, false>)
                             : (nt ? k_pgather<false, true, false> : k_pgather<false, false, false>));
      hipLaunchKernelGGL(kern, dim3(r.pgrid), dim3(PG_WG), 0, st, r.tasks + lv.first, L, RING, mode, lst, a);
    } else {
      const bool ls = (mode & LV_LIST) != 0;
      auto kern = lv.fr
          ? (r.urow ? (r.batch == 16 ? k_level<true, 16, true, false> : r.batch == 8 ? k_level<true, 8, true, false> : k_level<true, 4, true, false>)
                    : (r.batch == 16 ? k_level<false, 16, true, false> : r.batch == 8 ? k_level<false, 8, true, false> : k_level<false, 4, true, false>))
          : ls
          ? (r.urow ? (r.batch == 16 ? k_level<true, 16, false, true> : r.batch == 8 ? k_level<true, 8, false, true> : k_level<true, 4, false, true>)
                    : (r.batch == 16 ? k_level<false, 16, false, true> : r.batch == 8 ? k_level<false, 8, false, true> : k_level<false, 4, false, true>))
          : (r.urow ? (r.batch == 16 ? k_level<true, 16, false, false> : r.batch == 8 ? k_level<true, 8, false, false> : k_level<true, 4, false, false>)
                    : (r.batch == 16 ? k_level<false, 16, false, false> : r.batch == 8 ? k_level<false, 8, false, false> : k_level<false, 4, false, false>));
      hipLaunchKernelGGL(kern, dim3(grid), dim3(LEVEL_WG), 0, st,
                         r.tasks + lv.first, r.wg_start, lv.cnt_t, L, RING, r.upw, r.xcd, lv.fr_from, mode, lst);
    }
    HIPC(hipGetLastError());
    timed_end(tl);
  }

  // Neighbours the level before the next evaluation's last one should take: with
  // a share p of the pairs missing before it, a chunk of 128 is unsaturated after
  // k neighbours with probability about 128 p^k (what the row itself holds, its
  // neighbours mostly hold too).  More than a row has: it takes them all and still
  // stores nothing.  Zero when the level leaves too many pairs for k_thin2's
  // two-step reads.
  int thin_choice() const
  {
    const int L = lv.lmax - 1;
    if (!lr.parts || L < 1 || L >= LV_MISS_LEVELS || !pg_thin_env()) return 0;
    const double pairs = (double)n * nsrc, p = lv.miss[L - 1] / pairs;
    if (p <= 0 || p >= 0.95) return 0;
    if (lv.miss[L] * dpad * (dpad + 1.0) * (lr.fold ? 0.5 : 1.0) > THIN2_READS) return 0;
    const int k = std::max(1, (int)std::ceil(std::log(THIN_LEFT / 128) / std::log(p)));
    // the lists keep their k while the choice stays near it (no rebuild per evaluation)
    const int kk = lr.thin > 0 && std::abs(k - lr.thin) <= 1 ? lr.thin : k;
    return std::min(kk, 63);
  }

  // the end of a batch that ends at level `to` (the counters of levels
  // lv.examined .. to-1 are read): k_lvfin on the library's stream, copies and a
  // stream synchronisation otherwise (timed passes, serving slots, long batches)
  bool lv_fin_ok(int from, int to) const
  {
    return !timed() && st == C.stream && lvh && (int64_t)(to - from) * lr.ntasks <= LVFIN_MAX;
  }
  void note_fin(bool fin)
  {
    lv.pend_fin = fin;
    if (fin) lvseq++;
  }
  void lv_copies(int to)
  {
    LevelRun& r = lr;
    if (lv_fin_ok(lv.examined, to)) {
      hipLaunchKernelGGL(k_lvfin, dim3(1), dim3(256), 0, st, r.cnt, r.ntasks, lv.examined, to, RING, r.h_cnt_dev,
                         d_err, r.asym, lvh_dev, d_lvseq);
      HIPC(hipGetLastError());
      note_fin(true);
      return;
    }
    note_fin(false);
    HIPC(hipMemcpyAsync(r.h_cnt, r.cnt, sizeof(u64) * RING * r.ntasks, hipMemcpyDeviceToHost, st));
    HIPC(hipMemcpyAsync(h_err, d_err, sizeof(int), hipMemcpyDeviceToHost, st));
    if (timed()) {
      HIPC(hipMemcpyAsync(r.h_acnt, r.cnt + (size_t)2 * RING * r.ntasks, sizeof(u64) * RING * r.ntasks,
                          hipMemcpyDeviceToHost, st));
      HIPC(hipMemcpyAsync(r.h_acnt + (size_t)RING * r.ntasks, r.asym, sizeof(u32), hipMemcpyDeviceToHost, st));
    }
  }

  // the first levels and the first batch of group lv.first
  void lv_group_start()
  {
    LevelRun& r = lr;
    lv.cnt_t = std::min(r.group, r.ntasks - lv.first);
    lv.launched = lv.L1; lv.examined = 0; lv.running = lv.cnt_t; lv.fr_from = lv.L1;
    lv.batch_end = lv.first == 0 ? lv.be0 : first_batch_end();
    // the last evaluation ended at level batch_end - 1: expect the same, and
    // launch that level count-only (timed passes keep every level whole)
    lv.spec = spec_at(lv.batch_end) ? lv.batch_end - 1 : -1;
    lv.thin = listed_at(lv.spec) && pg_on() && thin_k > 0;
    if (lv.thin) g_routes.thin++;
    if (lv.first == 0 && lv.graphed) {
      // prepare + the first levels + the first batch + the counter copies as one graph
      const int be = lv.batch_end, L1 = lv.L1;
      const long long key = lv_key(be);
      if (!graph_ready(key))
        capture([&]() { lv_prepare(); lv_level0(); lv_levels(L1, be); }, key);
      else
        note_fin(lv_fin_ok(0, be));       // the replay ends as the captured batch did
      HIPC(hipGraphLaunch(gexec, st));
    } else {
      lv_level0();
      lv_levels(lv.launched, lv.batch_end);
    }
    lv.launched = std::max(lv.launched, lv.batch_end);
  }

  // end of a group's first batch of levels: the last evaluation's level count
  // (8 without one), at most MAX_BATCH_LEVELS so that its counter-ring slots
  // are distinct (the ring holds RING >= MAX_BATCH_LEVELS levels)
  int first_batch_end() const
  {
    if (lv.tk) return tile_batch_end(lv.L1, guess_levels > 0 ? guess_levels - lv.L1 : 8);
    const int be = std::min(n, std::max(2, std::min(MAX_BATCH_LEVELS, guess_levels > 0 ? guess_levels : 8)));
    return capped_end(std::min(be, std::max(lv.L1 + batch_cap, 2)));
  }

  // a batch cut short (serving) that would end one level before the expected
  // last one takes that level too: the two run listed (thin) and sparse
  int capped_end(int be) const
  {
    return batch_cap < MAX_BATCH_LEVELS && be == guess_levels - 1 && be - 1 >= lv.L1 ? guess_levels : be;
  }

  // tile mode: batches are whole launches of lv.tk levels, short enough that
  // the slots a launch clears ahead (up to tk past the batch) are not slots the
  // host has yet to read
  int tile_batch_end(int from, int want) const
  {
    const int cap = (MAX_BATCH_LEVELS - 2 * TILE_KMAX) / lv.tk;
    const int m = std::max(1, std::min(cap, (std::max(want, 1) + lv.tk - 1) / lv.tk));
    return from + m * lv.tk;
  }

  // a first batch ending at be ends with a count-only level (the last
  // evaluation ended there; timed passes and tile mode keep every level whole)
  bool spec_at(int be) const
  {
    return guess_levels > 0 && be == guess_levels && be - 1 >= lv.L1 && !(timed() && !g_stats_live) && !lv.tk;
  }

  // neighbour table, zeroed rings and done flags; where the levels use it (folded,
  // frontier mode) and it is not known, whether the table is symmetric
  void lv_prepare()
  {
    LevelRun& r = lr;
    prepare(r.cnt, lv.nzero, r.done, r.ntasks + LIST_COUNTERS + (lv.check ? 1 : 0), !lv.fresh);
    if (lv.tk) {
      const int grid = std::min(std::max(1, (n + 255) / 256), 4096);     // a thread per cell
      hipLaunchKernelGGL(k_tgeom, dim3(grid), dim3(256), 0, st, d_nbr, n, dpad, d_row2xy, geo_lmax, d_toff, d_err);
      HIPC(hipGetLastError());
    }
    if (lv.check) {
      const int64_t total = (int64_t)n * dpad;
      const int grid = (int)std::min<int64_t>(std::max<int64_t>(1, (total + 255) / 256), 4096);
      auto kern = dpad == 4 ? k_symcheck<1> : dpad == 8 ? k_symcheck<2> : dpad == 12 ? k_symcheck<3>
                : dpad == 16 ? k_symcheck<4> : k_symcheck<0>;
      hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, st, d_nbr, n, dpad, r.asym);
      HIPC(hipGetLastError());
    }
    if (pg_on() && !lv.plfresh) {
      // the units' (row, neighbour) pairs grouped by part for k_pgather
      auto kern = dpad + 1 <= 20 ? k_plist<20> : dpad + 1 <= 36 ? k_plist<36> : k_plist<64>;
      hipLaunchKernelGGL(kern, dim3(r.pupt), dim3(PG_UNIT), 0, st, d_nbr, n, dpad, r.psp, r.parts, r.thin, r.plist, r.ppoff);
      HIPC(hipGetLastError());
    }
  }

  // graph key of a first batch ending at be: its length, the kernel variant,
  // whether its last level is count-only, which tables the preparation builds
  // and, in tile mode, the longest edge k_tgeom and the tiles' window take
  // listing many chunks serialises on the list's counter, and k_sparse's
  // scattered chunks then cost more than a plain count-only level
  bool list_ok() const { return list_on; }

  long long lv_key(int be) const
  {
    const long long key = 8 * (64 * (16 * (8 * be + (lv.fr ? 1 : 0) + (spec_at(be) ? 2 : 0) + (list_ok() ? 4 : 0)) +
                               lv.tk) + lv.tside) +
                    (lv.fresh ? 1 : 0) + (lv.plfresh ? 2 : 0) + (lv.check ? 4 : 0);
    return 64 * (64 * key + (lv.tk ? std::min(std::max(geo_lmax, 0), 63) : 0)) + thin_k;
  }

  void lv_begin()
  {
    flush_adj();
    if (plan.tile) settle_lmax();
    LevelRun& r = lr;
    trace("run_level");
    if (!lvh && st == C.stream) {
      halloc_coherent(&lvh, &lvh_dev, 1);
      dalloc(&d_lvseq, 1);
      HIPC(hipMemsetAsync(d_lvseq, 0, sizeof(u32), st));
      lvh->seq = 0; lvh->err = 0;
      lvseq = 0;
    }
    // the table (and the pair lists) the last evaluation built still match the
    // adjacency (never assumed of a caller's device array: it may have changed)
    lv.fresh = table_fresh && table_src == cur_adj() && !ext_adj;
    if (!lv.fresh) pl_fresh = false;
    lv.K = r.direct;                      // levels 0..K-1 come from k_direct (0: k_level0 does level 0)
    lv.L1 = lv.K ? lv.K : 1;              // first level the gather kernel runs
    lv.nzero = 3 * RING * r.ntasks;       // the rings (counts, changed, processed) start at zero
    // temporal tiles when the plan asks and this adjacency's entries are short
    // enough for at least one level per launch
    lv.tside = tile_side();
    const int halo = (TILE_RW - lv.tside) / 2;
    lv.tk = plan.tile && tile_capable() && r.kwp == 2 && geo_lmax >= 0 && geo_lmax <= halo
                ? std::min(TILE_KMAX, halo / std::max(1, geo_lmax)) : 0;
    lv.be0 = first_batch_end();
    // frontier mode pays off over long level sequences; with few levels every
    // level is dense and the plain kernel is faster.  Without a last evaluation
    // to tell, a plan with row parts runs its own levels and goes over when
    // FRONTIER_MIN_LEVELS of them were not enough (lv_step): a frontier level of
    // n = 65536, d = 16 takes 500 us, the row parts' 447; serving's first requests of
    // nine chains 14.3 -> 10.4 ms
    lv.fr = !lv.tk && (guess_levels == 0 ? r.parts == 0 : guess_levels > FRONTIER_MIN_LEVELS);
    if (thin_k > 0 && thin_k != r.thin) { r.thin = thin_k; pl_fresh = false; }
    lv.plfresh = lv.fresh && pl_fresh;
    lv.check = (lv.fr || (!lv.tk && guess_levels == 0) || (pg_on() && r.fold)) && !(lv.fresh && asym_fresh);
    lv.graphed = r.group == r.ntasks && use_graph(lv_key(lv.be0));
    if (!lv.graphed) lv_prepare();
    lv.sts.assign(r.ntasks, LvTask{1, 0, 0, 0});
    lv.asym = -1;
    lv.any_disc = false;
    lv.max_d = 1; lv.lmax = 0;
    for (double& m : lv.miss) m = 0;
    lv.first = 0;
    lv_group_start();
    // the preparation is enqueued: the table matches the adjacency, and the
    // pair lists when this evaluation's gather levels use them
    table_fresh = true;
    table_src = cur_adj();
    if (pg_on()) pl_fresh = true;
    asym_fresh = lv.check || (lv.fresh && asym_fresh);
  }

  bool lv_step()
  {
    LevelRun& r = lr;
    if (lv.thin && lv.spec >= 0 && r.h_cnt[(size_t)(lv.spec % RING) * r.ntasks + lv.first] == THIN_FAILED) {
      // more chunks than the lists hold: the thin level again, whole, and the next
      const int L = lv.spec - 1;
      for (int k : {L, L + 1}) {
        hipLaunchKernelGGL(k_clear, dim3((lv.cnt_t + 255) / 256), dim3(256), 0, st,
                           r.cnt + (size_t)(k % RING) * r.ntasks + lv.first, lv.cnt_t, (int*)nullptr, 0);
        HIPC(hipGetLastError());
      }
      g_routes.thin_whole++;
      lv.spec = -1; lv.thin = false; thin_k = 0;
      lv_levels(L, lv.batch_end);
      return false;
    }
    for (int t = lv.first; t < lv.first + lv.cnt_t; t++) {
      LvTask& q = lv.sts[t];
      if (!q.running) continue;
      const u64 target = (u64)n * (u64)r.l[t];
      for (int L = lv.examined; L < lv.launched; L++) {
        const u64 c = r.h_cnt[(size_t)(L % RING) * r.ntasks + t];
        if (c == target) { q.running = 0; q.lwork = L; lv.max_d = std::max(lv.max_d, L + 1); break; }
        if ((L >= 1 && c == q.prev) || L + 1 >= n) { q.running = 0; q.lwork = L; lv.any_disc = true; break; }
        q.sum += (target - c) * (u64)s;
        q.prev = c;
        if (L < LV_MISS_LEVELS) lv.miss[L] += (double)(target - c);
      }
      if (!q.running) lv.running--;
    }
    lv.examined = lv.launched;
    if (lv.running > 0 && lv.spec >= 0) {
      // the count-only level was not the last: write its rows now (its counts stand)
      // (after a thin level, that level's rows first)
      const bool thin = lv.thin;
      lv.thin = false;
      if (thin) { g_routes.thin_late++; lv_launch(lv.spec - 1, LV_STORE); }
      lv_launch(lv.spec, LV_STORE);
      lv.spec = -1;
    }
    if (lv.running > 0 && lv.launched < n) {
      if (guess_levels == 0 && !lv.tk && !lv.fr && lv.launched >= FRONTIER_MIN_LEVELS) {
        lv.fr = true;
        lv.fr_from = lv.launched;
      }
      const int step = std::min(batch_cap, std::min(MAX_BATCH_LEVELS, std::max(lv.launched, 8)));
      lv.batch_end = lv.tk ? tile_batch_end(lv.launched, step) : capped_end(std::min(n, lv.launched + step));
      if (batch_cap < MAX_BATCH_LEVELS && spec_at(lv.batch_end)) {
        lv.spec = lv.batch_end - 1;
        lv.thin = lv.launched < lv.spec && listed_at(lv.spec) && pg_on() && thin_k > 0;
        if (lv.thin) g_routes.thin++;
      }
      lv_levels(lv.launched, lv.batch_end);
      lv.launched = std::max(lv.launched, lv.batch_end);
      return false;
    }
    if (lv.running > 0) lv.any_disc = true;
    if (lv.any_disc) return true;          // the result is the sentinel whatever the other blocks give
    for (int t = lv.first; t < lv.first + lv.cnt_t; t++) lv.lmax = std::max(lv.lmax, lv.sts[t].lwork);
    guess_levels = lv.lmax + 1;
    if (lv.first + r.group >= r.ntasks) {         // the evaluation's last group
      const double frac = lv.lmax >= 1 && lv.lmax - 1 < LV_MISS_LEVELS
                              ? lv.miss[lv.lmax - 1] / ((double)n * (r.kwp / 2) * r.ntasks) : 0;
      list_on = frac <= (list_on ? 1.0 : 0.5) * list_frac_env(lr.parts ? LIST_MAX_FRAC_PG : LIST_MAX_FRAC);
      thin_k = thin_choice();
    }
    if (timed()) flush_level_stats(lv.sts.data(), lv.first, lv.cnt_t);
    lv.first += r.group;
    if (lv.first < r.ntasks) { lv_group_start(); return false; }
    return true;
  }

  void lv_result(u64* excess, int* diam, bool* disc)
  {
    u64 tot = 0;
    for (const LvTask& q : lv.sts) tot += q.sum;
    *excess = tot; *diam = lv.max_d; *disc = lv.any_disc;
    if (pg_on() && lv.asym == 0 && lv.launched > lv.L1) g_routes.folded++;
    if (timed()) flush_level_stats(lv.sts.data(), 0, 0);
  }

  // waits for the enqueued batch: its sequence number in host memory, watched
  // for up to LV_SPIN_S, else (and without one) a stream synchronisation
  void lv_wait()
  {
    bool seen = false;
    if (lv.pend_fin) {
      const volatile u32* sq = &lvh->seq;
      const double t0 = wall_time();
      for (int i = 0; !seen; i++) {
        seen = *sq == lvseq;
        if (!seen && (i & 255) == 255 && wall_time() - t0 > LV_SPIN_S) break;
      }
      if (seen) std::atomic_thread_fence(std::memory_order_acquire);
    }
    if (!seen) HIPC(hipStreamSynchronize(st));
    if (lv.pend_fin) *h_err = lvh->err;
    if (lr.fold && (lv.pend_fin || timed()))
      lv.asym = (lv.pend_fin ? lvh->asym : *(const u32*)(lr.h_acnt + (size_t)RING * lr.ntasks)) != 0;
  }

  void run_level(u64* excess, int* diam, bool* disc)
  {
    lv_begin();
    for (;;) {
      lv_wait();
      trace("level batch synchronized");
      check_err();
      if (lv_step()) break;
    }
    lv_result(excess, diam, disc);
  }

  template <typename St>
  void flush_level_stats(const St* stv, int first, int cnt_t)
  {
    LevelRun& r = lr;
    HIPC(hipStreamSynchronize(st));
    for (TimedLaunch& tl : g_pending) {
      float ms = 0;
      HIPC(hipEventElapsedTime(&ms, tl.a, tl.b));
      g_evpool.push_back(tl.a); g_evpool.push_back(tl.b);
      if (tl.kind == T_LEVEL) {
        double bytes = 0, minb = 0;
        // a level processes a share of the (row, segment) units: all of them, or
        // in frontier mode the active ones; bytes are that share of the full level's.
        // A folded level gathers for the units of one of each pair across the diagonal
        // and stores both; a thin one takes a part of the neighbours.
        // Compulsory bytes: each processed row of a working block read once and
        // (unless the launch only counts) written once, the neighbour ids once per launch
        const double fold = tl.fold && lv.asym == 0 ? (r.ntasks + 1) / (2.0 * r.ntasks) : 1.0;
        const double nbrs = tl.nbrs < 0 ? avg_deg : std::min((double)tl.nbrs, avg_deg);
        for (int t = first; t < first + cnt_t; t++)
          if (tl.level <= stv[t].lwork) {
            const double share = (lv.fr && tl.level >= lv.fr_from) || lv.tk
                                     ? (double)r.h_acnt[(size_t)(tl.level % RING) * r.ntasks + t] / ((double)n * r.segs)
                                     : 1.0;
            const double row = ((r.l[t] + 63) / 64) * 8.0;
            bytes += share * tl.nlev * (double)n * (fold * ((nbrs + 1.0) * row + 4.0 * nbrs) + tl.wr * row);
            minb += share * (double)n * ((r.l[t] + 63) / 64) * 8.0 * (1.0 + tl.wr);
          }
        if (minb > 0) minb += (double)n * avg_deg * 4.0;
        if (bytes > 0) {
          g_stats.level_launches++; g_stats.level_ms += ms; g_stats.level_bytes += bytes;
          g_stats.level_min_bytes += minb;
        }
        else { g_stats.idle_launches++; g_stats.idle_ms += ms; }
      } else {
        g_stats.other_launches++; g_stats.other_ms += ms;
      }
    }
    g_pending.clear();
  }

  void run_resident(u64* excess, int* diam, bool* disc)
  {
    ResRun& r = rr;
    trace("run_resident");
    // at most two launches (the table is rebuilt only when the adjacency changed
    // by other means than device swaps), no clears and no copies: the resident
    // kernel's last workgroup adds up the workgroups' totals, writes the result
    // and the error flag to host memory and re-zeroes its queue head and
    // arrival counter
    auto enqueue = [&]() {
      const int* src = ext_adj ? ext_adj : d_adj;
      if (!table_fresh || table_src != src) {
        prepare(nullptr, 0, nullptr, 0);
        table_fresh = true;
        table_src = src;
      }
      TimedLaunch tl;
      timed_begin(tl, T_RESIDENT, 0, st);
      const bool stop = degree > 8;
      auto kern = r.wb == 1 ? (n > RES_RPT_WIDE1B * r.threads
                                   ? (stop ? k_resident_w<1, true, RES_RPT_WIDE1C> : k_resident_w<1, false, RES_RPT_WIDE1C>)
                               : n > RES_RPT_WIDE1 * r.threads
                                   ? (stop ? k_resident_w<1, true, RES_RPT_WIDE1B> : k_resident_w<1, false, RES_RPT_WIDE1B>)
                               : n > res_rpt(1) * r.threads
                                   ? (stop ? k_resident_w<1, true, RES_RPT_WIDE1> : k_resident_w<1, false, RES_RPT_WIDE1>)
                                   : stop ? k_resident_w<1, true> : k_resident_w<1>)
                : r.wb == 2 ? (n > res_rpt(2) * r.threads
                                   ? (stop ? k_resident_w<2, true, RES_RPT_WIDE> : k_resident_w<2, false, RES_RPT_WIDE>)
                                   : stop ? k_resident_w<2, true> : k_resident_w<2>)
                : r.wb == 4 ? (stop ? k_resident_w<4, true> : k_resident_w<4>)
                : (stop ? k_resident_w<8, true> : k_resident_w<8>);
      ResFin fin;
      fin.done = r.done; fin.part = r.part; fin.host = r.host_dev; fin.err = d_err;
      fin.patch = make_patch();
      fin.seq = ++r.seq;
      hipLaunchKernelGGL(kern, dim3(r.grid), dim3(r.threads), r.lds, st, r.tasks, r.ntasks, r.qhead, r.out, fin);
      HIPC(hipGetLastError());
      timed_end(tl);
    };
    // launched directly: replaying these two launches as a captured graph took
    // longer (43.5 against 39.3 us per evaluation of n=1024, d=6)
    enqueue();
    trace("resident launched");
    // the kernel stores its sequence number after the result: watch for it a
    // while (cheaper than a stream synchronisation for small graphs), else, and
    // for timed launches, synchronize
    bool seen = false;
    if (!timed()) {
      const volatile u32* sq = &r.host->seq;
      const double t0 = wall_time();
      for (int i = 0; !seen; i++) {
        seen = *sq == r.seq;
        if (!seen && (i & 63) == 63 && wall_time() - t0 > RES_SPIN_S) break;
      }
      if (seen) std::atomic_thread_fence(std::memory_order_acquire);
    }
    if (!seen) HIPC(hipStreamSynchronize(st));
    trace("resident synchronized");
    const ResHost res = *r.host;      // written by the launch (its sequence number seen, or the stream synchronized)
    *h_err = res.err;
    check_err();
    *excess = res.out.sum;
    *diam = std::max(1, res.out.diam);
    *disc = (res.out.flags & 1) != 0;
    if (timed()) {
      for (TimedLaunch& t : g_pending) {
        float ms = 0;
        HIPC(hipEventElapsedTime(&ms, t.a, t.b));
        g_evpool.push_back(t.a); g_evpool.push_back(t.b);
        if (t.kind == T_RESIDENT) {
          double row = (avg_deg + 2.0) * (std::min(32 * r.wb, nsrc) / 8.0) + 4.0 * avg_deg;
          g_stats.resident_launches++; g_stats.resident_ms += ms;
          g_stats.resident_bytes += (double)res.out.levels * n * row;
        } else {
          g_stats.other_launches++; g_stats.other_ms += ms;
        }
      }
      g_pending.clear();
    }
  }

  // the reference's final arithmetic (aspl.c:73-74): ordered-pair sum, ASPL, halved sum;
  // a disconnected graph reports diameter n+1 (turned into the sentinels by the caller)
  void result_of(u64 excess, int d, bool disc, int* diameter, long* sum, double* ASPL) const
  {
    long lsum = (long)n * (n - 1) + (long)excess;
    if (disc) d = n + 1;
    *diameter = d;
    *ASPL = lsum / (((double)n - 1) * n);
    lsum /= 2.0;
    *sum = lsum;
  }

  // the evaluated sources' excess over their n-1 base distances (times s),
  // the largest terminal level + 1, and whether some block stalled
  void run_raw(u64* excess, int* d, bool* disc)
  {
    *excess = 0; *d = 1; *disc = false;
    if (plan.plan == ODPX_PLAN_LEVEL) run_level(excess, d, disc);
    else run_resident(excess, d, disc);
  }

  // ---- the BFS kind ----
  // the smallest level plan: one 1-word block resident, so the kind allocates
  // no bit matrix (its evaluations never run the level plan)
  ODPX_Plan bfs_plan() const
  {
    ODPX_Plan p{};
    p.plan = ODPX_PLAN_LEVEL; p.kw = 1; p.upw = 4; p.group = 1;
    return p;
  }

  // One breadth-first search per source row (k_bfs), over the 32-bit
  // row-neighbour table; the sources are rows [0, n/s), one per symmetry orbit
  // (circulant: vertices 0..n/s-1; grid: the base region's cells), so the
  // ordered-pair distance sum is s times theirs.  Returns what run_raw returns:
  // the excess over n(n-1), the diameter, whether some source missed a vertex.
  void run_bfs(u64* excess, int* d, bool* disc)
  {
    flush_adj();
    drop_graph();
    table_fresh = false;                       // the resident plan's 16-bit table is not kept current
    PrepArgs a{};
    a.adj = ext_adj ? ext_adj : d_adj;
    a.numdeg = d_numdeg; a.itable = d_itable; a.err = d_err;
    a.nbr = d_nbr; a.nbr16 = nullptr;
    a.n = n; a.s = s; a.degree = degree; a.dpad = dpad;
    a.width = width; a.height = height; a.grid_s = grid_s;
    const int64_t total = (int64_t)n * dpad;
    hipLaunchKernelGGL(k_prepare, dim3((int)std::min<int64_t>(std::max<int64_t>(1, (total + 255) / 256), 4096)),
                       dim3(256), 0, st, a);
    HIPC(hipGetLastError());
    const size_t words = ((size_t)n + 31) / 32;
    const bool vis_lds = words * 4 <= LDS_DYN_MAX;
    // workgroups: up to 8 per CU, fewer when the queues (and bitmaps) of that
    // many would pass 8 GiB
    const size_t per_wg = 8ull * n + (vis_lds ? 0 : words * 4);
    int G = (int)std::min<size_t>({(size_t)nsrc, (size_t)C.ncu * 8, std::max<size_t>(1, (8ull << 30) / per_wg)});
    if ((size_t)G * 2 * n > bfs_q_cap) { dfree(&d_bfs_q); dalloc(&d_bfs_q, (size_t)G * 2 * n); bfs_q_cap = (size_t)G * 2 * n; }
    if (!vis_lds && (size_t)G * words > bfs_vis_cap) {
      dfree(&d_bfs_vis); dalloc(&d_bfs_vis, (size_t)G * words); bfs_vis_cap = (size_t)G * words;
    }
    if (!d_bfs_out) { dalloc(&d_bfs_out, 1); dalloc(&d_bfs_next, 1); halloc(&h_bfs_out, 1); }
    hipLaunchKernelGGL(k_bfs_clear, dim3(1), dim3(64), 0, st, d_bfs_out, d_bfs_next);
    if (vis_lds)
      hipLaunchKernelGGL(k_bfs<true>, dim3(G), dim3(256), words * 4, st, d_nbr, n, dpad, nsrc, d_bfs_q,
                         (u32*)nullptr, d_bfs_next, d_bfs_out);
    else
      hipLaunchKernelGGL(k_bfs<false>, dim3(G), dim3(256), 0, st, d_nbr, n, dpad, nsrc, d_bfs_q, d_bfs_vis,
                         d_bfs_next, d_bfs_out);
    HIPC(hipGetLastError());
    HIPC(hipMemcpyAsync(h_bfs_out, d_bfs_out, sizeof(BfsOut), hipMemcpyDeviceToHost, st));
    HIPC(hipMemcpyAsync(h_err, d_err, sizeof(int), hipMemcpyDeviceToHost, st));
    HIPC(hipStreamSynchronize(st));
    check_err();
    const BfsOut o = *h_bfs_out;
    *disc = o.disc != 0;
    *d = std::max(1, o.ecc);
    *excess = o.sum * (u64)s - (u64)n * (u64)(n - 1);
  }

  // full evaluation of the adjacency on the device, reference arithmetic
  void evaluate(int* diameter, long* sum, double* ASPL)
  {
    double t0 = wall_time();
    u64 excess = 0;
    int d = 1;
    bool disc = false;
    if (bfs) run_bfs(&excess, &d, &disc);
    else run_raw(&excess, &d, &disc);
    result_of(excess, d, disc, diameter, sum, ASPL);
    if (timed()) { g_stats.evals++; g_stats.eval_ms += 1e3 * (wall_time() - t0); }
  }
};

// ---------------------------------------------------------------------------
// reference kind selection and memory estimate (utils.c:1206-1266, GPU branch)

static double ref_mem_mb(int kind, int nodes, int degree, int symmetries, bool numdeg, bool grid_s)
{
  double ab;
  if (kind == KIND_MATRIX) ab = nodes * ((double)nodes / (4.0 * symmetries));
  else if (kind == KIND_SAVING) ab = 16.0 * nodes * GPU_CHUNK_WORDS;
  else ab = nodes * (3.0 * sizeof(int) + 1.0);                // the BFS kind (utils.c:1220-1224)
  if (grid_s && kind != KIND_BFS) ab += 4.0 * nodes;
  double res = 8.0 * 448, adj = 4.0 * (nodes / symmetries) * degree, deg = numdeg ? 4.0 * nodes : 0;
  return (ab + res + adj + deg) / (1024.0 * 1024.0);
}

static int ref_kind(int nodes, int degree, int symmetries, bool numdeg, bool grid_s)
{
  const char* val = getenv("ODP_ASPL");
  if (!val) return ref_mem_mb(KIND_MATRIX, nodes, degree, symmetries, numdeg, grid_s) <= MEM_THRESHOLD_MB
                   ? KIND_MATRIX : KIND_SAVING;
  if (strcmp(val, "MATRIX") == 0) return KIND_MATRIX;
  if (strcmp(val, "MATRIX_SAVING") == 0) return KIND_SAVING;
  if (strcmp(val, "BFS") == 0) return KIND_BFS;   // the reference's GPU flavour refuses it (utils.c:1256-1259)
  ODP_ERROR("Unknown ASPL value (%s)\n", val);
  return 0;
}

extern "C" int ODPX_Get_kind(int nodes, int degree, int has_num_degrees, int symmetries, int grid_s)
{
  return ref_kind(nodes, degree, symmetries, has_num_degrees != 0, grid_s != 0);
}

extern "C" double ODPX_Get_mem_usage(int kind, int nodes, int degree, int has_num_degrees, int symmetries, int grid_s)
{
  return ref_mem_mb(kind, nodes, degree, symmetries, has_num_degrees != 0, grid_s != 0);
}

// ---------------------------------------------------------------------------
// the ODP_* lifecycle (aspl_cuda.cu:128-263)

static struct {
  bool active;
  int kind;
  Evaluator ev;
  bool profile;
  double elapsed;
  unsigned times;
} E;

static int rotate_host(int v, int width, int height, int s, int angle)
{
  int w = v / height, h = v % height;
  if (s == 2) return (width - w - 1) * height + (height - h - 1);
  if (angle == 90) return h * height + (height - w - 1);
  if (angle == 180) return (height - w - 1) * height + (height - h - 1);
  return (height - h - 1) * height + w;
}

// orbit-major row permutation of a 2/4-fold symmetric grid (utils.c:2103-2124)
// Position of each base vertex (local index x * bh + y of a bw x bh region)
// when the region is walked in GRID_TILE x GRID_TILE tiles: a column block of
// GRID_TILE^2 sources is then one compact patch of the grid, whose distances
// to any vertex span few levels (frontier-mode levels skip it sooner).
static const int GRID_TILE = 32;
static void tile_rank(int bw, int bh, std::vector<int>& rank)
{
  rank.assign((size_t)bw * bh, 0);
  int pos = 0;
  for (int tx = 0; tx < bw; tx += GRID_TILE)
    for (int ty = 0; ty < bh; ty += GRID_TILE)
      for (int x = tx; x < std::min(bw, tx + GRID_TILE); x++)
        for (int y = ty; y < std::min(bh, ty + GRID_TILE); y++) rank[(size_t)x * bh + y] = pos++;
}

// Row of every vertex of a 2/4-fold symmetric grid (utils.c:2103-2124): the base
// vertices (one per orbit) take rows [0, n/s), their rotations the same row plus
// k * n/s.  Within the base rows the order is tiled (tile_rank) instead of the
// reference's x-major order; results do not depend on it (rows and sources are
// relabelled together).
static void make_itable(int width, int height, int s, int* itable, bool tiled = true)
{
  int based = width * height / s;
  std::vector<int> rank;
  if (!tiled) {                // the reference's order: base vertex i takes row i
    rank.resize(based);
    for (int i = 0; i < based; i++) rank[i] = i;
  }
  if (s == 2) {
    if (tiled) tile_rank(width / 2, height, rank);
    for (int i = 0; i < based; i++) {
      itable[i] = rank[i];
      itable[rotate_host(i, width, height, 2, 180)] = rank[i] + based;
    }
  } else {
    int bh = height / 2;
    if (tiled) tile_rank(width / 2, bh, rank);
    for (int i = 0; i < based; i++) {
      int v = (i / bh) * height + (i % bh);
      itable[v] = rank[i];
      itable[rotate_host(v, width, height, 4, 90)] = rank[i] + based;
      itable[rotate_host(v, width, height, 4, 180)] = rank[i] + 2 * based;
      itable[rotate_host(v, width, height, 4, 270)] = rank[i] + 3 * based;
    }
  }
}

static bool profile_env()
{
  const char* v = getenv("ODP_PROFILE");
  return v && atoi(v) == 1;
}

static void lifecycle_init(int family, int nodes, int degree, const int* numdeg_full, int s,
                           int width, int height, bool grid_s, const int* itable)
{
  if (E.active) ODP_ERROR("ODP_Init_aspl_* called twice without ODP_Finalize_aspl\n");
  if (s < 1 || nodes % s != 0) ODP_ERROR("nodes(%d) must be divisible by symmetries(%d)\n", nodes, s);
  if (nodes < 1 || degree < 0) ODP_ERROR("Invalid nodes(%d) or degree(%d)\n", nodes, degree);
  E.kind = ref_kind(nodes, degree, s, numdeg_full != nullptr, grid_s);
  E.ev.shape(family, nodes, degree, s, width, height, numdeg_full, grid_s ? 1 : 0);
  if (grid_s) E.ev.set_itable(itable);
  E.ev.bfs = E.kind == KIND_BFS;
  E.ev.apply_plan(E.kind == KIND_BFS ? E.ev.bfs_plan() : E.ev.default_plan(E.kind));
  E.profile = profile_env();
  E.elapsed = 0;
  E.times = 0;
  E.active = true;
}

extern "C" void ODP_Init_aspl_general(int nodes, int degree, int* num_degrees)
{
  RandFence rand_fence;
  lifecycle_init(0, nodes, degree, num_degrees, 1, 0, -1, false, nullptr);
}

extern "C" void ODP_Init_aspl_general_s(int nodes, int degree, int* num_degrees, int symmetries)
{
  RandFence rand_fence;
  if (symmetries < 1 || nodes % symmetries != 0)
    ODP_ERROR("nodes(%d) must be divisible by symmetries(%d)\n", nodes, symmetries);
  std::vector<int> full;
  if (num_degrees) {          // aspl_cuda.cu:166-175: the base array repeated per orbit
    int based = nodes / symmetries;
    full.resize(nodes);
    for (int i = 0; i < symmetries; i++)
      for (int j = 0; j < based; j++) full[(size_t)i * based + j] = num_degrees[j];
  }
  lifecycle_init(0, nodes, degree, num_degrees ? full.data() : nullptr, symmetries, 0, -1, false, nullptr);
}

extern "C" void ODP_Init_aspl_grid(int width, int height, int degree, int* num_degrees)
{
  RandFence rand_fence;
  lifecycle_init(1, width * height, degree, num_degrees, 1, width, height, false, nullptr);
}

extern "C" void ODP_Init_aspl_grid_s(int width, int height, int degree, int* num_degrees, int symmetries)
{
  RandFence rand_fence;
  int nodes = width * height;
  bool gs = (symmetries == 2 || symmetries == 4);
  if (symmetries < 1 || nodes % symmetries != 0)
    ODP_ERROR("nodes(%d) must be divisible by symmetries(%d)\n", nodes, symmetries);
  if (symmetries == 2 && width % 2 != 0) ODP_ERROR("width(%d) must be divisible by 2\n", width);
  if (symmetries == 4 && (width % 2 != 0 || height % 2 != 0))
    ODP_ERROR("width(%d) and height(%d) must be divisible by 2\n", width, height);
  if (symmetries == 4 && width != height) ODP_ERROR("Must be the same as width(%d) and height(%d)\n", width, height);
  std::vector<int> itable;
  if (gs) { itable.resize(nodes); make_itable(width, height, symmetries, itable.data()); }
  std::vector<int> full;
  if (num_degrees) {          // aspl_cuda.cu:200-219: every orbit member gets its base vertex's degree
    int based = nodes / symmetries;
    full.resize(nodes);
    if (symmetries == 2) {
      for (int i = 0; i < based; i++) {
        full[i] = num_degrees[i];
        full[rotate_host(i, width, height, 2, 180)] = num_degrees[i];
      }
    } else if (symmetries == 4) {
      int bh = height / 2;
      for (int i = 0; i < based; i++) {
        int v = (i / bh) * height + (i % bh);
        full[v] = num_degrees[i];
        full[rotate_host(v, width, height, 4, 90)] = num_degrees[i];
        full[rotate_host(v, width, height, 4, 180)] = num_degrees[i];
        full[rotate_host(v, width, height, 4, 270)] = num_degrees[i];
      }
    } else {
      for (int i = 0; i < symmetries; i++)
        for (int j = 0; j < based; j++) full[(size_t)i * based + j] = num_degrees[j];
    }
  }
  lifecycle_init(1, nodes, degree, num_degrees ? full.data() : nullptr, symmetries, width, height, gs,
                 gs ? itable.data() : nullptr);
}

static void need_active(const char* fn)
{
  if (!E.active) ODP_ERROR("%s called before ODP_Init_aspl_*\n", fn);
}

static void finish_result(int* diameter, long* sum, double* ASPL)
{
  if (*diameter > E.ev.n) {   // aspl_cuda.cu:256-260
    *diameter = INT_MAX;
    *sum = LONG_MAX;
    *ASPL = DBL_MAX;
  }
}

extern "C" void ODP_Set_aspl(void* adjacency, int* diameter, long* sum, double* ASPL)
{
  RandFence rand_fence;
  need_active("ODP_Set_aspl");
  double t = wall_time();
  E.ev.upload(adjacency);
  E.ev.evaluate(diameter, sum, ASPL);
  E.elapsed += wall_time() - t;
  finish_result(diameter, sum, ASPL);
  E.times++;
}

extern "C" void ODP_Finalize_aspl(void)
{
  RandFence rand_fence;
  if (!E.active) return;
  if (E.profile) {             // utils.c:1268-1294, flavour "HIP"
    char host[256] = {0};
    gethostname(host, sizeof(host) - 1);
    time_t t = time(NULL);
    double mem = ref_mem_mb(E.kind, E.ev.n, E.ev.degree, E.ev.s, E.ev.has_numdeg != 0, E.ev.grid_s != 0);
    printf("------ Profile for SET_ASPL ------\n");
    printf("Date            = %s", ctime(&t));
    printf("Hostname        = %s\n", host);
    printf("Number of Times = %u\n", E.times);
    printf("Total Time      = %f sec.\n", E.elapsed);
    printf("Average Time    = %f sec.\n", E.elapsed / E.times);   // as utils.c:1284 (nan when never called)
    printf("Algorithm       = %s (HIP)\n", E.kind == KIND_MATRIX ? "MATRIX" : E.kind == KIND_SAVING ? "MATRIX_SAVING" : "BFS");
    printf("Symmetries      = %d\n", E.ev.s);
    printf("Memory Usage    = %.3f MB\n", mem);
    printf("Num of Procs    = 1\n");
    printf("Num of Threads  = 1\n");
    printf("--------- End of Profile ---------\n");
  }
  E.ev.release();
  E.active = false;
  E.kind = 0;
  E.times = 0;
  E.elapsed = 0;
}

// ---------------------------------------------------------------------------
// plans, autotuning, device-resident evaluation, timing

extern "C" int ODPX_Get_plan(ODPX_Plan* p)
{
  if (!E.active) return -1;
  *p = E.ev.plan;
  return 0;
}

extern "C" long long ODPX_Table_entries(void)
{
  return E.active ? (long long)E.ev.adj_elems() : 0;
}

extern "C" int ODPX_Set_plan(const ODPX_Plan* p)
{
  RandFence rand_fence;
  if (!E.active || !E.ev.plan_valid(*p)) return -1;
  E.ev.apply_plan(*p);
  return 0;
}

extern "C" void ODPX_Upload_adjacency(void* adjacency)
{
  RandFence rand_fence;
  need_active("ODPX_Upload_adjacency");
  E.ev.upload(adjacency);
  HIPC(hipStreamSynchronize(C.stream));
}

extern "C" void ODPX_Set_aspl_resident(int* diameter, long* sum, double* ASPL)
{
  RandFence rand_fence;
  need_active("ODPX_Set_aspl_resident");
  double t = wall_time();
  E.ev.evaluate(diameter, sum, ASPL);
  E.elapsed += wall_time() - t;
  finish_result(diameter, sum, ASPL);
  E.times++;
}

extern "C" int ODPX_Swap_device(int a, int b, int c, int d)
{
  RandFence rand_fence;
  need_active("ODPX_Swap_device");
  Evaluator& v = E.ev;
  if (v.s != 1) return -1;
  int ids[4] = {a, b, c, d};
  for (int x : ids) if (x < 0 || x >= v.n) return -1;
  if (a == b || a == c || a == d || b == c || b == d || c == d) return -1;   // not a 2-opt move
  v.flush_adj();
  if (!v.mirror_ok && v.stage_is_device && !v.ext_adj) {   // h_stage holds the device copy
    v.h_mirror.assign(v.h_stage, v.h_stage + v.adj_elems());
    v.mirror_ok = true;
  }
  if (v.mirror_ok) {
    // checked on the host copy with k_swap's rule (the first entry of each row
    // equal to the old neighbour), applied to it, and launched without waiting
    const int rows[4] = {a, b, c, d}, from[4] = {b, a, d, c}, to[4] = {c, d, a, b};
    int pos[4];
    for (int e = 0; e < 4; e++) {
      const int* r = v.h_mirror.data() + (size_t)rows[e] * v.degree;
      pos[e] = -1;
      for (int j = 0; j < v.degree; j++)
        if (r[j] == from[e]) { pos[e] = j; break; }
      if (pos[e] < 0) return -1;                   // nothing changed
    }
    for (int e = 0; e < 4; e++) v.h_mirror[(size_t)rows[e] * v.degree + pos[e]] = to[e];
    v.stage_is_device = false;
    v.swap_launch(a, b, c, d, pos);
  } else {
    v.stage_is_device = false;         // the device copy moves on its own
    v.swap_launch(a, b, c, d);
    HIPC(hipMemcpyAsync(v.h_err, v.d_err, sizeof(int), hipMemcpyDeviceToHost, C.stream));
    HIPC(hipStreamSynchronize(C.stream));
    if (*v.h_err & 4) {
      *v.h_err = 0;
      HIPC(hipMemsetAsync(v.d_err, 0, sizeof(int), C.stream));
      HIPC(hipStreamSynchronize(C.stream));
      return -1;
    }
  }
  if (v.geo_lmax >= 0) {
    // a grid's new edges a-c and b-d may be longer than any before (k_tile's halo)
    auto cheb = [&](int p, int q) { return std::max(abs(p / v.height - q / v.height), abs(p % v.height - q % v.height)); };
    v.geo_lmax = std::max(v.geo_lmax, std::max(cheb(a, c), cheb(b, d)));
  }
  return 0;
}

// ---------------------------------------------------------------------------
// one process's share of an evaluation, as the reference's MPI+CUDA flavour
// divides it (aspl_mpi_cuda.cu:44-123): the source columns of one rank

extern "C" int ODPX_Set_aspl_shard(int rank, int nranks, long long* excess, int* diameter, int* disconnected)
{
  RandFence rand_fence;
  need_active("ODPX_Set_aspl_shard");
  if (nranks < 1 || rank < 0 || rank >= nranks || !excess || !diameter || !disconnected) return -1;
  if (E.kind == KIND_BFS) return -1;               // the MPI flavours divide bit-matrix columns only
  Evaluator& v = E.ev;
  const int nsrc = v.nsrc, W = (nsrc + 63) / 64;
  // MATRIX: ceil(W / P)-word blocks, rank r the block r (aspl_mpi_cuda.cu:47-54);
  // MATRIX_SAVING: 64-word blocks r, r + P, ... (aspl_mpi_cuda.cu:92-94)
  std::vector<std::pair<int, int>> ranges;
  if (E.kind == KIND_MATRIX) {
    const int chunk = (W + nranks - 1) / nranks, parsize = (W + chunk - 1) / chunk;
    if (rank < parsize) ranges.push_back({64 * rank * chunk, std::min(nsrc, 64 * (rank + 1) * chunk)});
  } else {
    const int b = 64 * GPU_CHUNK_WORDS, parsize = (W + GPU_CHUNK_WORDS - 1) / GPU_CHUNK_WORDS;
    for (int t = rank; t < parsize; t += nranks) ranges.push_back({b * t, std::min(nsrc, b * (t + 1))});
  }
  // symmetric grids: the reference's row order, so that a source column is the
  // same base vertex as in the reference (utils.c:2103-2124)
  std::vector<int> itable;
  if (v.grid_s) {
    itable.resize(v.n);
    make_itable(v.width, v.height, v.s, itable.data(), false);
    v.set_itable(itable.data());
  }
  const ODPX_Plan saved = v.plan;
  u64 tot = 0;
  int dmax = 1;
  bool disc = false;
  for (const auto& r : ranges) {
    v.src_lo = r.first; v.src_hi = r.second;
    v.apply_plan(saved);
    u64 ex; int d; bool dc;
    v.run_raw(&ex, &d, &dc);
    tot += ex; dmax = std::max(dmax, d); disc = disc || dc;
  }
  v.src_lo = 0; v.src_hi = nsrc;
  if (v.grid_s) {
    make_itable(v.width, v.height, v.s, itable.data(), true);
    v.set_itable(itable.data());
  }
  v.apply_plan(saved);
  *excess = (long long)tot;
  *diameter = disc ? v.n + 1 : dmax;
  *disconnected = disc ? 1 : 0;
  return 0;
}

// ---------------------------------------------------------------------------
// simulated annealing of a general graph, the reference's SA loop
// (sample/SA/general.c:149-181) with the adjacency kept on the device

// acceptance test of sample/SA/common.c:15-43 with symmetries = 1; the uniform
// draw comes from the run's generator (the reference calls random())
static bool sa_accept(int nodes, int cur_d, int d, double cur_a, double a, double temp, bool hill, bool aspl_prio,
                      uint64_t rng[4])
{
  if (hill) return a <= cur_a;
  if (d < cur_d && !aspl_prio) return true;
  if (d > cur_d && !aspl_prio) return false;
  if (a <= cur_a) return true;
  const double diff = (cur_a - a) * nodes * (nodes - 1);
  const double u = ((double)(ODPX_Rng_next(rng) >> 11) + 0.5) / 9007199254740992.0;   // (0, 1)
  return exp(diff / temp) > u;
}

// The device loop (k_anneal) applies to a regular general graph under the
// resident plan whose block and whole 16-bit table fit one workgroup's LDS, with
// one workgroup per block and every block's workgroup resident at once
// (a cooperative launch).  ODP_HIP_ANNEAL=host keeps the host-stepped loop.
static size_t anneal_lds(const Evaluator& v)
{
  return (size_t)((v.n * v.rr.wb + 3) & ~3) * 4 + (size_t)v.n * v.dp16 * 2;
}

static bool anneal_device_ok(const Evaluator& v, const std::vector<int>& cur)
{
  const char* e = getenv("ODP_HIP_ANNEAL");
  if (e && strcmp(e, "host") == 0) return false;
  if (v.plan.plan != ODPX_PLAN_RESIDENT || v.s != 1 || v.family != 0 || v.has_numdeg || v.degree < 1) return false;
  for (int x : cur) if (x < 0 || x >= v.n) return false;
  const int G = v.rr.ntasks;
  if (G < 1 || G > C.ncu || anneal_lds(v) > LDS_DYN_MAX) return false;
  int dev = 0, coop = 0;
  HIPC(hipGetDevice(&dev));
  HIPC(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
  if (!coop) return false;
  int occ = 0;
  const int wb = v.rr.wb;
  const void* f = wb == 1 ? (const void*)k_anneal<1> : wb == 2 ? (const void*)k_anneal<2>
                : wb == 4 ? (const void*)k_anneal<4> : (const void*)k_anneal<8>;
  HIPC(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, f, v.rr.threads, anneal_lds(v)));
  return occ * C.ncu >= G;
}

static long long anneal_chunk_env()
{
  const char* e = getenv("ODP_HIP_ANNEAL_CHUNK");
  const long long c = e ? atoll(e) : 0;
  return c > 0 ? c : 4096;
}

static void anneal_on_device(Evaluator& v, int* adj_out, const std::vector<int>& start, const uint64_t rng[4],
                             long long ncalcs, double max_temp, double cooling, bool hill, bool prio, int low_d,
                             double low_a, int& cur_d, double& cur_a, int& best_d, long& best_sum, double& best_a,
                             long long& steps, long long& accepted, bool& optimum)
{
  const int n = v.n, deg = v.degree, G = v.rr.ntasks, wb = v.rr.wb;
  v.flush_adj();
  AnnealState S{};
  for (int i = 0; i < 4; i++) S.rng[i] = rng[i];
  S.cur_a = cur_a; S.best_a = best_a; S.temp = max_temp; S.cooling = cooling; S.low_a = low_a;
  S.steps = 0; S.accepted = 0; S.best_sum = best_sum;
  S.cur_d = cur_d; S.best_d = best_d; S.low_d = low_d;
  S.hill = hill ? 1 : 0; S.prio = prio ? 1 : 0;
  AnnealState* d_st = nullptr;
  u64* d_slots = nullptr;
  int* d_best = nullptr;
  dalloc(&d_st, 1); dalloc(&d_slots, (size_t)2 * G); dalloc(&d_best, (size_t)n * deg);
  HIPC(hipMemcpyAsync(d_st, &S, sizeof S, hipMemcpyHostToDevice, C.stream));
  const size_t lds = anneal_lds(v);
  const void* f = wb == 1 ? (const void*)k_anneal<1> : wb == 2 ? (const void*)k_anneal<2>
                : wb == 4 ? (const void*)k_anneal<4> : (const void*)k_anneal<8>;
  const long long chunk = anneal_chunk_env();
  const double t_dev = wall_time();
  while (S.steps < ncalcs && !S.optimum && !S.stop) {
    AnnealArgs aa;
    aa.adj = v.d_adj; aa.best = d_best; aa.st = d_st; aa.slots = d_slots;
    aa.n = n; aa.degree = deg; aa.dp = v.dp16; aa.ntasks = G;
    aa.steps = (int)std::min<long long>(chunk, ncalcs - S.steps);
    hipLaunchKernelGGL(k_clear, dim3((2 * G + 63) / 64), dim3(64), 0, C.stream, d_slots, 2 * G, (int*)nullptr, 0);
    void* args[] = {&aa};
    HIPC(hipLaunchCooperativeKernel(f, dim3(G), dim3(v.rr.threads), args, (unsigned)lds, C.stream));
    HIPC(hipMemcpyAsync(&S, d_st, sizeof S, hipMemcpyDeviceToHost, C.stream));
    HIPC(hipStreamSynchronize(C.stream));
    if (S.err) ODP_ERROR("libodp_hip: internal error: an annealing step's grid barrier timed out\n");
  }
  E.elapsed += wall_time() - t_dev;
  E.times += (unsigned)S.steps;
  // the caller's array receives the best graph (unchanged when nothing improved)
  if (S.best_d != best_d || S.best_a != best_a)
    HIPC(hipMemcpy(adj_out, d_best, sizeof(int) * (size_t)n * deg, hipMemcpyDeviceToHost));
  else
    memcpy(adj_out, start.data(), sizeof(int) * (size_t)n * deg);
  dfree(&d_st); dfree(&d_slots); dfree(&d_best);
  // the device copy now holds the chain's current graph; the 16-bit table is rebuilt from it
  v.stage_is_device = false;
  v.mirror_ok = false;
  v.table_fresh = false;
  steps = S.steps; accepted = S.accepted;
  cur_d = S.cur_d; cur_a = S.cur_a;
  best_d = S.best_d; best_sum = (long)S.best_sum; best_a = S.best_a;
  optimum = S.optimum != 0;
}

// acceptance test of sample/SA/common.c:15-43 (accept_s: the ASPL difference
// scaled by n(n-1)/symmetries); the uniform draw comes from the run's generator
static bool sa_accept_s(int nodes, int cur_d, int d, double cur_a, double a, double temp, bool hill, bool aspl_prio,
                        int symmetries, uint64_t rng[4])
{
  if (hill) return a <= cur_a;
  if (d < cur_d && !aspl_prio) return true;
  if (d > cur_d && !aspl_prio) return false;
  if (a <= cur_a) return true;
  const double diff = ((cur_a - a) * nodes * (nodes - 1)) / symmetries;
  const double u = ((double)(ODPX_Rng_next(rng) >> 11) + 0.5) / 9007199254740992.0;   // (0, 1)
  return exp(diff / temp) > u;
}

// Longest Manhattan length of a grid table's edges (base rows: the vertices
// ODP_Conv_edge2adjacency_grid_s keeps, utils.c:1116-1151)
static int grid_table_length(const Evaluator& v, const int* base)
{
  const int based = v.n / v.s, bh = v.height / 2;
  int len = 0;
  for (int i = 0; i < based; i++) {
    const int x = v.s == 4 ? (i / bh) * v.height + (i % bh) : i;
    for (int j = 0; j < v.degree; j++) {
      const int u = base[(size_t)i * v.degree + j];
      if (u < 0 || u >= v.n) continue;
      len = std::max(len, abs(u / v.height - x / v.height) + abs(u % v.height - x % v.height));
    }
  }
  return len;
}

// The annealing loop of sample/SA/general_s.c:160-194 and grid(_s).c:170-199 for
// symmetric general and grid Inits: each step one move of the reference's kind
// (ODPX_Mutate, drawn from the run's generator) on the host table, ODP_Set_aspl,
// the best graph kept, accept_s, and ODP_Restore_adjacency_* on a rejection.
// Grid moves keep every edge within the start graph's longest Manhattan length.
static int anneal_symmetric(int* adj, long long ncalcs, double max_temp, double min_temp, bool hill, bool prio,
                            uint64_t seed, ODPX_AnnealResult* res)
{
  Evaluator& v = E.ev;
  const double t0 = wall_time();
  const int n = v.n, deg = v.degree, s = v.s, based = n / s;
  const bool grid = v.family == 1;
  std::vector<int> cur(adj, adj + (size_t)based * deg);
  const int length = grid ? grid_table_length(v, cur.data()) : 0;
  uint64_t rng[4];
  ODPX_Rng_seed(seed, rng);
  int diameter; long sum; double ASPL;
  ODP_Set_aspl(cur.data(), &diameter, &sum, &ASPL);
  int cur_d = diameter, best_d = diameter;
  double cur_a = ASPL, best_a = ASPL;
  long best_sum = sum;
  int low_d; double low_a;
  if (grid) ODP_Set_lbounds_grid(v.width, v.height, deg, length, &low_d, &low_a);
  else ODP_Set_lbounds_general(n, deg, &low_d, &low_a);
  long long steps = 0, accepted = 0;
  bool optimum = diameter == low_d && ASPL == low_a;
  const double cooling = hill ? 0.0 : pow(min_temp / max_temp, 1.0 / (double)ncalcs);
  double temp = max_temp;
  for (long long i = 0; i < ncalcs && !optimum; i++) {
    ODP_Restore r;
    if (ODPX_Mutate(grid ? 1 : 0, grid ? v.width : n, v.height, deg, length, s, cur.data(), rng, &r) != 0) break;
    ODP_Set_aspl(cur.data(), &diameter, &sum, &ASPL);
    steps++;
    if (diameter < best_d || (diameter == best_d && ASPL < best_a)) {
      best_d = diameter; best_sum = sum; best_a = ASPL;
      memcpy(adj, cur.data(), sizeof(int) * (size_t)based * deg);
      if (diameter == low_d && ASPL == low_a) { optimum = true; break; }
    }
    if (sa_accept_s(n, cur_d, diameter, cur_a, ASPL, temp, hill, prio, s, rng)) {
      cur_d = diameter; cur_a = ASPL;
      accepted++;
    } else if (grid) {
      ODP_Restore_adjacency_grid(r, cur.data());
    } else {
      ODP_Restore_adjacency_general(r, cur.data());
    }
    temp *= cooling;
  }
  if (res) {
    res->steps = steps; res->accepted = accepted;
    res->best_diameter = best_d; res->best_sum = best_sum; res->best_ASPL = best_a;
    res->diameter = cur_d; res->ASPL = cur_a; res->optimum = optimum ? 1 : 0;
    res->seconds = wall_time() - t0;
  }
  return 0;
}

extern "C" int ODPX_Anneal(void* adjacency, long long ncalcs, double max_temp, double min_temp, int hill_climbing,
                           int ASPL_priority, uint64_t seed, ODPX_AnnealResult* res)
{
  RandFence rand_fence;
  need_active("ODPX_Anneal");
  Evaluator& v = E.ev;
  if (ncalcs < 0 || (!hill_climbing && (max_temp <= 0 || min_temp <= 0))) return -1;
  if (v.s != 1 || v.family != 0)
    return anneal_symmetric((int*)adjacency, ncalcs, max_temp, min_temp, hill_climbing != 0, ASPL_priority != 0, seed,
                            res);
  const double t0 = wall_time();
  const int n = v.n, deg = v.degree;
  int* adj = (int*)adjacency;
  std::vector<int> cur(adj, adj + (size_t)n * deg);
  uint64_t rng[4];
  ODPX_Rng_seed(seed, rng);
  int diameter; long sum; double ASPL;
  ODP_Set_aspl(cur.data(), &diameter, &sum, &ASPL);
  int cur_d = diameter, best_d = diameter;
  double cur_a = ASPL, best_a = ASPL;
  long best_sum = sum;
  int low_d; double low_a;
  ODP_Set_lbounds_general(n, deg, &low_d, &low_a);
  long long steps = 0, accepted = 0;
  bool optimum = diameter == low_d && ASPL == low_a;
  const double cooling = hill_climbing ? 0.0 : pow(min_temp / max_temp, 1.0 / (double)ncalcs);
  double temp = max_temp;
  v.flush_adj();
  v.stage_is_device = false;         // the moves change the device copy only
  v.mirror_ok = false;
  // Under the resident plan (its table current) a move is not a launch of its
  // own: its four table entries ride along with the next evaluation's launch
  // (the host copy gives their positions).  Otherwise k_swap applies it.
  const bool fold = v.plan.plan == ODPX_PLAN_RESIDENT && v.swap_table() != nullptr;
  auto pos_of = [&](int row, int id) {
    for (int j = 0; j < deg; j++) if (cur[(size_t)row * deg + j] == id) return j;
    ODP_ERROR("libodp_hip: internal error: a move's edge is not in the host copy\n");
    return -1;
  };
  // the move a-b, c-d -> a-c, b-d has been made on the host copy
  auto queue_move = [&](int a, int b, int c, int d) {
    const int e[12] = {a, pos_of(a, c), c, b, pos_of(b, d), d, c, pos_of(c, a), a, d, pos_of(d, b), b};
    v.pend_patch.insert(v.pend_patch.end(), e, e + 12);
  };
  if (!optimum && ncalcs > 0 && anneal_device_ok(v, cur)) {
    // every step on the device: a cooperative launch runs many of them
    anneal_on_device(v, adj, cur, rng, ncalcs, max_temp, cooling, hill_climbing != 0, ASPL_priority != 0, low_d, low_a,
                     cur_d, cur_a, best_d, best_sum, best_a, steps, accepted, optimum);
    if (res) {
      res->steps = steps; res->accepted = accepted;
      res->best_diameter = best_d; res->best_sum = best_sum; res->best_ASPL = best_a;
      res->diameter = cur_d; res->ASPL = cur_a; res->optimum = optimum ? 1 : 0;
      res->seconds = wall_time() - t0;
    }
    return 0;
  }
  for (long long i = 0; i < ncalcs && !optimum; i++) {
    int sw[4];
    if (ODPX_Two_opt(n, deg, cur.data(), rng, sw) != 0) break;      // no valid move left
    // the same move on the device copy (valid: the host copy mirrors it)
    if (fold) {
      queue_move(sw[0], sw[1], sw[2], sw[3]);
    } else {
      v.swap_launch(sw[0], sw[1], sw[2], sw[3]);
    }
    const double t = wall_time();
    v.evaluate(&diameter, &sum, &ASPL);
    E.elapsed += wall_time() - t;
    finish_result(&diameter, &sum, &ASPL);
    E.times++;
    steps++;
    if (diameter < best_d || (diameter == best_d && ASPL < best_a)) {
      best_d = diameter; best_sum = sum; best_a = ASPL;
      memcpy(adj, cur.data(), sizeof(int) * (size_t)n * deg);
      if (diameter == low_d && ASPL == low_a) { optimum = true; break; }
    }
    if (sa_accept(n, cur_d, diameter, cur_a, ASPL, temp, hill_climbing != 0, ASPL_priority != 0, rng)) {
      cur_d = diameter; cur_a = ASPL;
      accepted++;
    } else {
      // undo a-b, c-d -> a-c, b-d on both copies (the next launch on the stream follows it)
      ODPX_Swap_edges(n, deg, cur.data(), sw[0], sw[2], sw[1], sw[3]);
      if (fold) {
        queue_move(sw[0], sw[2], sw[1], sw[3]);
      } else {
        v.swap_launch(sw[0], sw[2], sw[1], sw[3]);
      }
    }
    temp *= cooling;
  }
  v.apply_pending();                 // a last undo, if the last move was rejected
  HIPC(hipStreamSynchronize(C.stream));
  if (res) {
    res->steps = steps; res->accepted = accepted;
    res->best_diameter = best_d; res->best_sum = best_sum; res->best_ASPL = best_a;
    res->diameter = cur_d; res->ASPL = cur_a; res->optimum = optimum ? 1 : 0;
    res->seconds = wall_time() - t0;
  }
  return 0;
}

extern "C" void ODPX_Stats_enable(int on)
{
  g_stats_on = on != 0;
  g_stats_live = on == 2;
}
extern "C" void ODPX_Stats_reset(void) { memset(&g_stats, 0, sizeof g_stats); }
extern "C" void ODPX_Stats_get(ODPX_Stats* out) { *out = g_stats; }
extern "C" void ODPX_Routes_get(ODPX_Routes* out)
{
  out->folded = g_routes.folded; out->thin = g_routes.thin; out->thin_whole = g_routes.thin_whole;
  out->thin_late = g_routes.thin_late; out->chunked = g_routes.chunked;
}

extern "C" int ODPX_Autotune(void* adjacency, int repeats)
{
  RandFence rand_fence;
  need_active("ODPX_Autotune");
  if (E.kind == KIND_BFS) return -1;               // the BFS kind runs no plan
  Evaluator& v = E.ev;
  std::vector<ODPX_Plan> cand;
  for (int wb = 1; wb <= RES_WB_MAX; wb <<= 1)
    for (int th : {256, 512, 1024}) {
      ODPX_Plan p{};
      p.plan = ODPX_PLAN_RESIDENT; p.wb = wb; p.threads = th;
      if (v.plan_valid(p)) cand.push_back(p);
    }
  int W = (v.nsrc + 63) / 64;
  std::vector<int> kws = {0};
  for (int k : {512, 256, 128, 64, 32, 16}) if (k < W) kws.push_back(k);
  for (int kw : kws)
    for (int sm = 0; sm < 2; sm++)
      for (int x = 0; x < 2; x++) {
        ODPX_Plan p{};
        p.plan = ODPX_PLAN_LEVEL; p.kw = kw; p.upw = kw == 0 ? 4 : 8; p.seg_major = sm; p.xcd = x;
        p.group = v.plan.plan == ODPX_PLAN_LEVEL ? v.plan.group : 0;
        p.direct = 0;
        cand.push_back(p);
        if (v.direct_auto(kw == 0 ? W : std::min(kw, W), 1) > 0) { p.direct = -1; cand.push_back(p); }
      }
  if (v.tile_capable()) {
    ODPX_Plan p{};
    p.plan = ODPX_PLAN_LEVEL; p.kw = 2; p.upw = 8; p.xcd = 1; p.direct = -1; p.tile = 1;
    p.group = E.kind == KIND_MATRIX ? 0 : SAVING_GROUP * LEVEL_BLOCK_WORDS / 2;
    cand.push_back(p);
  }
  if (repeats < 1) repeats = 1;
  v.upload(adjacency);
  double best = 1e30;
  ODPX_Plan bestp = v.plan;
  int rd = 0; long rs = 0; double ra = 0;
  bool have = false;
  for (const ODPX_Plan& p : cand) {
    v.apply_plan(p);
    int d; long sm; double as;
    v.evaluate(&d, &sm, &as);   // warm-up, also fixes the level guess
    double t0 = wall_time();
    for (int i = 0; i < repeats; i++) v.evaluate(&d, &sm, &as);
    double t = (wall_time() - t0) / repeats;
    if (!have) { rd = d; rs = sm; ra = as; have = true; }
    else if (d != rd || sm != rs || memcmp(&as, &ra, sizeof(double)) != 0)
      ODP_ERROR("libodp_hip: plans disagree (%d %ld vs %d %ld)\n", d, sm, rd, rs);
    if (t < best) { best = t; bestp = p; }
  }
  v.apply_plan(bestp);
  return (int)cand.size();
}

// ---------------------------------------------------------------------------
// batched evaluation: every graph small enough for LDS in one persistent launch

struct BatchGraph { long long adj_off, nbr_off, ent_start; int n, degree, dp, pad; };

// Orders each row's neighbour list so that the rows a wave reads in one LDS
// pass (g consecutive rows) fetch rows of different bank classes (id mod m,
// m = banks / words per row) at every list position: thread t takes group t
// of the concatenated graphs (gstart: first group of each graph, gstart[ng]
// the total) and fills the positions in turn, each row taking the id of its
// remaining ones whose class is the least used at that position so far.  A
// row's list only changes order, so every level ORs the same rows.
__global__ void k_balance(const BatchGraph* __restrict__ gs, const int* __restrict__ gstart, int ng, int g,
                          unsigned short* __restrict__ nbr)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= gstart[ng]) return;
  int lo = 0, hi = ng - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (gstart[mid] <= t) lo = mid; else hi = mid - 1;
  }
  const BatchGraph G = gs[lo];
  const u32 m = (u32)max(1, min(G.pad, 64));
  const int r0 = (t - gstart[lo]) * g, r1 = min(r0 + g, G.n);
  unsigned short* base = nbr + G.nbr_off;
  for (int j = 0; j < G.degree; j++) {
    u64 used[8] = {0, 0, 0, 0, 0, 0, 0, 0};          // used[k] bit c: class c taken more than k times
    for (int r = r0; r < r1; r++) {
      unsigned short* row = base + (int64_t)r * G.dp;
      int best = j, bc = 9;
      for (int q = j; q < G.degree; q++) {
        const u32 c = (u32)row[q] % m;
        int cnt = 0;
#pragma unroll
        for (int k = 0; k < 8; k++) cnt += (int)((used[k] >> c) & 1);
        if (cnt < bc) { bc = cnt; best = q; if (cnt == 0) break; }
      }
      const unsigned short x = row[best];
      row[best] = row[j];
      row[j] = x;
      const u32 c = (u32)x % m;
#pragma unroll
      for (int k = 0; k < 8; k++)
        if (!((used[k] >> c) & 1)) { used[k] |= 1ULL << c; break; }
    }
  }
}

// The tables of graphs gs[0, ng): a thread per 8 ids (one 16-byte store; a
// graph's rows are dp ids, dp a multiple of 8).  `first` is gs[0]'s first id
// among all graphs' tables, `total` the ids of these.
__global__ void k_prepare_batch(const BatchGraph* __restrict__ gs, int ng, long long first, long long total,
                                const int* __restrict__ adj, unsigned short* __restrict__ nbr, int* err)
{
  const long long tid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long stride = (long long)gridDim.x * blockDim.x;
  for (long long idx = first + 8 * tid; idx < first + total; idx += 8 * stride) {
    int lo = 0, hi = ng - 1;
    while (lo < hi) {
      int mid = (lo + hi + 1) >> 1;
      if (gs[mid].ent_start <= idx) lo = mid; else hi = mid - 1;
    }
    const BatchGraph G = gs[lo];
    const u32 e = (u32)(idx - G.ent_start);        // n dp < 2^32 (graphs here have n <= 65535)
    const int i = (int)(e / (u32)G.dp), j0 = (int)(e - (u32)i * (u32)G.dp);
    const int* row = adj + G.adj_off + (long long)i * G.degree;
    u32 out[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 8; k++) {
      int out_v = i;
      if (j0 + k < G.degree) {
        const int v = row[j0 + k];
        if (v >= 0 && v < G.n) out_v = v;
        else if (v != -1) atomicOr(err, 1);
      }
      out[k >> 1] |= (u32)(out_v & 0xffff) << (16 * (k & 1));
    }
    *(uint4*)(nbr + G.nbr_off + e) = make_uint4(out[0], out[1], out[2], out[3]);
  }
}

// chunks, at most, that a batch handed over and run in one call is sent in: a
// chunk's graphs are evaluated while the next chunk is on its way
#define BATCH_CHUNKS 8

static struct {
  // the loaded batch
  int ng = 0;
  std::vector<int> nodes, degrees;
  std::vector<long long> offsets;
  std::vector<int> small, large;        // graphs on the resident path / on the single-graph path
  std::vector<BatchGraph> hg;           // per small graph
  std::vector<int> wb;                  // per small graph
  int ntasks = 0;
  size_t lds = 0;
  // tasks are grouped by chunk (one, but for a call that loads and runs) and
  // block width (8, 4, 2, 1 words per row), one launch each; chunk c holds the
  // small graphs cfirst[c] .. cfirst[c + 1] - 1
  int chunks = 1, cfirst[BATCH_CHUNKS + 1] = {};
  int grp_start[BATCH_CHUNKS][4] = {}, grp_n[BATCH_CHUNKS][4] = {};
  size_t grp_lds[BATCH_CHUNKS][4] = {};
  bool balanced = false;                // the tables' lists are ordered for the current widths (k_balance)
  hipStream_t copies = nullptr;         // the chunks' way to the device
  hipEvent_t sent = nullptr;
  // device buffers (grow-only)
  size_t adj_cap = 0, nbr_cap = 0, g_cap = 0, t_cap = 0;
  int *d_adj = nullptr, *d_err = nullptr, *d_qhead = nullptr, *h_err = nullptr;
  unsigned short* d_nbr = nullptr;
  BatchGraph* d_g = nullptr;
  int* d_gstart = nullptr;   // [small graphs + 1] first balance group of each graph
  size_t gstart_cap = 0;
  ResOut *d_out = nullptr, *h_out = nullptr;
  ResTask* d_t = nullptr;
  Evaluator single;          // graphs too large for the LDS path, and the looped path
  // launch policy, set by ODPX_Batch_autotune: the widest block (32-bit words per
  // row) per size class, and resident workgroups per CU
  int wbcap[BATCH_CLASSES] = {RES_WB_MAX, RES_WB_MAX, RES_WB_MAX, RES_WB_MAX, RES_WB_MAX};
  int per_cu = 2;
  hipGraphExec_t gexec = nullptr;   // the resident launch sequence, captured once per load and policy
  int runs = 0;                     // runs since the task table was built (capture from the second)
} B;

static void batch_drop_graph()
{
  if (B.gexec) HIPC(hipGraphExecDestroy(B.gexec));
  B.gexec = nullptr;
  B.runs = 0;
}

// widest block for a graph of n rows in a 1024-thread resident workgroup; 0 if none
static int batch_wb(int n)
{
  if (n > 65535) return 0;
  for (int wb = RES_WB_MAX; wb >= 1; wb >>= 1)
    if ((size_t)n * wb * 4 <= LDS_DYN_MAX && n <= res_rpt(wb) * 1024) return wb;
  return 0;
}

// size class of a graph for the batch policy: n <= 2048, 4096, 8192, 16384, larger
static int batch_class(int n)
{
  return n <= 2048 ? 0 : n <= 4096 ? 1 : n <= 8192 ? 2 : n <= 16384 ? 3 : 4;
}

static void finish_one(int n, u64 excess, int d, bool disc, int* diameter, long* sum, double* ASPL)
{
  long lsum = (long)n * (n - 1) + (long)excess;
  if (disc) d = n + 1;
  double aspl = lsum / (((double)n - 1) * n);
  lsum /= 2.0;
  if (d > n) { d = INT_MAX; lsum = LONG_MAX; aspl = DBL_MAX; }
  *diameter = d; *sum = lsum; *ASPL = aspl;
}

// one graph through the single-graph path, its adjacency already on the device
static void single_eval_dev(Evaluator& v, int n, int degree, const int* dev_adj, int plan_kind,
                            int* diameter, long* sum, double* ASPL)
{
  v.shape(0, n, degree, 1, 0, -1, nullptr, 0);
  v.ext_adj = dev_adj;
  ODPX_Plan p = v.default_plan(KIND_MATRIX);
  if (plan_kind == ODPX_PLAN_LEVEL && p.plan != ODPX_PLAN_LEVEL) {
    p = ODPX_Plan{};
    p.plan = ODPX_PLAN_LEVEL; p.kw = LEVEL_BLOCK_WORDS; p.upw = 8; p.seg_major = 0; p.xcd = 1; p.group = 0;
  }
  v.apply_plan(p);
  v.evaluate(diameter, sum, ASPL);
  v.ext_adj = nullptr;
  if (*diameter > n) { *diameter = INT_MAX; *sum = LONG_MAX; *ASPL = DBL_MAX; }
}

// neighbour-list order of batched graphs (env ODP_HIP_BALANCE="banks,rows":
// LDS banks of 4 bytes and rows per LDS pass, default 64,32; "0" keeps the
// given order)
static void balance_env(int* banks, int* group)
{
  static int b = -1, g = 0;
  if (b < 0) {
    b = 64; g = 32;
    if (const char* v = getenv("ODP_HIP_BALANCE")) {
      g = 32;
      if (sscanf(v, "%d,%d", &b, &g) < 1) b = 0;
      if (b < 0 || b > 64 || (b & (b - 1)) || g < 1 || g > 64) b = 0;
    }
  }
  *banks = b; *group = g;
}

// the resident launches' task table under the current policy (per graph the
// widest block its size class allows): per chunk the widest blocks first, then
// each width's blocks longest first (short queue tails).  A graph's blocks cost
// the same, so the graphs are sorted, not the blocks.
static void batch_build_tasks()
{
  batch_drop_graph();
  const size_t ns = B.small.size();
  std::vector<double> cost(ns);
  size_t total = 0;
  B.lds = 0;
  for (size_t k = 0; k < ns; k++) {
    const BatchGraph& G = B.hg[k];
    int wb = batch_wb(G.n);
    while (wb > B.wbcap[batch_class(G.n)]) wb >>= 1;      // narrower blocks always fit
    B.wb[k] = wb;
    B.lds = std::max(B.lds, (size_t)G.n * wb * 4);
    cost[k] = (double)G.n * G.dp * (1.0 + log((double)G.n) / log(std::max(2.0, G.degree - 1.0)));
    total += (size_t)(G.n + 32 * wb - 1) / (32 * wb);
  }
  if (B.chunks == 1) { B.cfirst[0] = 0; B.cfirst[1] = (int)ns; }
  std::vector<ResTask> tasks;
  tasks.reserve(total);
  std::vector<int> ord;
  for (int c = 0; c < B.chunks; c++) {
    ord.clear();
    for (int k = B.cfirst[c]; k < B.cfirst[c + 1]; k++) ord.push_back(k);
    std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) {
      return B.wb[a] != B.wb[b] ? B.wb[a] > B.wb[b] : cost[a] > cost[b];
    });
    for (int g = 0; g < 4; g++) { B.grp_start[c][g] = 0; B.grp_n[c][g] = 0; B.grp_lds[c][g] = 0; }
    for (int k : ord) {
      const BatchGraph& G = B.hg[k];
      const int wb = B.wb[k], g = wb == 8 ? 0 : wb == 4 ? 1 : wb == 2 ? 2 : 3, b = 32 * wb;
      if (B.grp_n[c][g] == 0) B.grp_start[c][g] = (int)tasks.size();
      B.grp_lds[c][g] = std::max(B.grp_lds[c][g], (size_t)G.n * wb * 4);
      const int nt = (G.n + b - 1) / b, deg = std::max(G.degree, 1);
      const int walk = res_walk_env(G.n, deg, b), walk_last = res_walk_env(G.n, deg, G.n - (nt - 1) * b);
      for (int t = 0; t < nt; t++) {
        ResTask T;
        T.nbr = B.d_nbr + G.nbr_off; T.n = G.n; T.dp = G.dp; T.src0 = t * b; T.l = std::min(b, G.n - t * b);
        T.s = 1; T.graph = k; T.wb = wb; T.dq = (deg + 3) / 4;
        T.deg = deg; T.walk = t + 1 < nt ? walk : walk_last;
        tasks.push_back(T);
      }
      B.grp_n[c][g] += nt;
    }
  }
  if (tasks.size() > B.t_cap) { dfree(&B.d_t); dalloc(&B.d_t, tasks.size()); B.t_cap = tasks.size(); }
  B.ntasks = (int)tasks.size();
  B.balanced = false;
  HIPC(hipMemcpyAsync(B.d_t, tasks.data(), sizeof(ResTask) * tasks.size(), hipMemcpyHostToDevice, C.stream));
  HIPC(hipStreamSynchronize(C.stream));
}

// The neighbour lists ordered for the chosen block widths (bank classes id mod
// banks / wb).  It costs about four tenths of a run (256 graphs of up to 16384
// vertices: 2.2 ms against 5.4) and takes a tenth off every later one, so it
// comes with the second run of a loaded batch; a batch run once goes without.
static void batch_balance()
{
  if (B.balanced) return;
  B.balanced = true;
  int banks = 0, group = 0;
  balance_env(&banks, &group);
  if (banks <= 0) return;
  std::vector<int> gstart(B.small.size() + 1, 0);
  for (size_t k = 0; k < B.small.size(); k++) {
    B.hg[k].pad = std::max(1, banks / B.wb[k]);
    gstart[k + 1] = gstart[k] + (B.hg[k].n + group - 1) / group;
  }
  if (gstart.size() > B.gstart_cap) { dfree(&B.d_gstart); dalloc(&B.d_gstart, gstart.size()); B.gstart_cap = gstart.size(); }
  HIPC(hipMemcpyAsync(B.d_g, B.hg.data(), sizeof(BatchGraph) * B.hg.size(), hipMemcpyHostToDevice, C.stream));
  HIPC(hipMemcpyAsync(B.d_gstart, gstart.data(), sizeof(int) * gstart.size(), hipMemcpyHostToDevice, C.stream));
  const int total = gstart.back();
  hipLaunchKernelGGL(k_balance, dim3((total + 255) / 256), dim3(256), 0, C.stream, B.d_g, B.d_gstart,
                     (int)B.small.size(), group, B.d_nbr);
  HIPC(hipGetLastError());
  HIPC(hipStreamSynchronize(C.stream));
}

// the tables of small graphs [k0, k1) from their adjacency on the device
static void batch_prepare(int k0, int k1)
{
  if (k0 >= k1) return;
  const long long first = B.hg[k0].ent_start;
  const long long total = B.hg[k1 - 1].ent_start + (long long)B.hg[k1 - 1].n * B.hg[k1 - 1].dp - first;
  const int pgrid = (int)std::min<long long>(std::max<long long>(1, (total / 8 + 255) / 256), 8192);
  hipLaunchKernelGGL(k_prepare_batch, dim3(pgrid), dim3(256), 0, C.stream, B.d_g + k0, k1 - k0, first, total, B.d_adj,
                     B.d_nbr, B.d_err);
  HIPC(hipGetLastError());
}

// what a load keeps of the graphs, and room for them; returns the packed array's length
static long long batch_shape(int ngraphs, const int* nodes, const int* degrees, const long long* offsets)
{
  batch_drop_graph();
  ctx_init();
  B.ng = ngraphs;
  B.nodes.assign(nodes, nodes + ngraphs);
  B.degrees.assign(degrees, degrees + ngraphs);
  B.offsets.assign(offsets, offsets + ngraphs);
  B.small.clear(); B.large.clear(); B.hg.clear(); B.wb.clear();
  B.ntasks = 0; B.lds = 0; B.chunks = 1; B.balanced = false;
  if (ngraphs <= 0) return 0;
  long long adj_end = 0;
  for (int g = 0; g < ngraphs; g++) {
    if (nodes[g] < 1 || degrees[g] < 0 || offsets[g] < 0) ODP_ERROR("ODPX_Batch_load: invalid graph %d\n", g);
    adj_end = std::max(adj_end, offsets[g] + (long long)nodes[g] * degrees[g]);
    (batch_wb(nodes[g]) > 0 ? B.small : B.large).push_back(g);
  }
  if ((size_t)adj_end > B.adj_cap) { dfree(&B.d_adj); dalloc(&B.d_adj, (size_t)adj_end); B.adj_cap = adj_end; }
  if (!B.d_err) {
    dalloc(&B.d_err, 1); dalloc(&B.d_qhead, 4 * BATCH_CHUNKS); halloc(&B.h_err, 1);
    HIPC(hipMemsetAsync(B.d_err, 0, 4, C.stream));
  }
  if (!B.small.empty()) {
    long long nbr_tot = 0;
    B.hg.resize(B.small.size());
    B.wb.resize(B.small.size());
    for (size_t k = 0; k < B.small.size(); k++) {
      int g = B.small[k];
      BatchGraph& G = B.hg[k];
      G.adj_off = offsets[g]; G.n = nodes[g]; G.degree = degrees[g]; G.dp = round_up(std::max(1, degrees[g]), 8);
      G.nbr_off = nbr_tot; G.ent_start = nbr_tot; G.pad = 0;
      nbr_tot += (long long)G.n * G.dp;
    }
    if ((size_t)nbr_tot > B.nbr_cap) { dfree(&B.d_nbr); dalloc(&B.d_nbr, (size_t)nbr_tot); B.nbr_cap = nbr_tot; }
    if (B.small.size() > B.g_cap) {
      dfree(&B.d_g); dfree(&B.d_out); hfree(&B.h_out);
      dalloc(&B.d_g, B.small.size()); dalloc(&B.d_out, B.small.size()); halloc(&B.h_out, B.small.size());
      B.g_cap = B.small.size();
    }
    HIPC(hipMemcpyAsync(B.d_g, B.hg.data(), sizeof(BatchGraph) * B.hg.size(), hipMemcpyHostToDevice, C.stream));
  }
  return adj_end;
}

static void batch_check_err()
{
  if (*B.h_err) ODP_ERROR("ODPX_Batch_load: adjacency holds a vertex id outside [0, nodes)\n");
}

extern "C" int ODPX_Batch_load(int ngraphs, const int* nodes, const int* degrees, const long long* offsets,
                               const int* packed)
{
  RandFence rand_fence;
  const long long adj_end = batch_shape(ngraphs, nodes, degrees, offsets);
  if (ngraphs <= 0) return 0;
  HIPC(hipMemcpyAsync(B.d_adj, packed, sizeof(int) * adj_end, hipMemcpyHostToDevice, C.stream));
  if (!B.small.empty()) {
    batch_prepare(0, (int)B.small.size());
    batch_build_tasks();
  }
  HIPC(hipMemcpyAsync(B.h_err, B.d_err, sizeof(int), hipMemcpyDeviceToHost, C.stream));
  HIPC(hipStreamSynchronize(C.stream));
  batch_check_err();
  return 0;
}

static void batch_clear()
{
  const int na = (int)(B.small.size() * sizeof(ResOut) / 8);
  hipLaunchKernelGGL(k_clear, dim3((na + 255) / 256), dim3(256), 0, C.stream, (u64*)B.d_out, na, B.d_qhead,
                     4 * BATCH_CHUNKS);
  HIPC(hipGetLastError());
}

// the persistent resident launches over a chunk's graphs
static void batch_launch(int c)
{
  for (int g = 0; g < 4; g++) {
    if (!B.grp_n[c][g]) continue;
    // each width's launch holds only its own blocks' LDS: more workgroups per CU
    int per_cu = (int)std::max<size_t>(1, LDS_LIMIT / (B.grp_lds[c][g] + LDS_STATIC));
    per_cu = std::min(per_cu, B.per_cu);
    const int grid = std::max(1, std::min(B.grp_n[c][g], per_cu * C.ncu));
    auto kern = g == 0 ? k_resident_w<8, true> : g == 1 ? k_resident_w<4, true> : g == 2 ? k_resident_w<2, true>
                                                                                       : k_resident_w<1, true>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(1024), B.grp_lds[c][g], C.stream, B.d_t + B.grp_start[c][g],
                       B.grp_n[c][g], B.d_qhead + 4 * c + g, B.d_out, ResFin{});
    HIPC(hipGetLastError());
  }
}

// clear, the launches over every small graph, results to the host
static void batch_enqueue()
{
  batch_clear();
  TimedLaunch tr;
  timed_begin(tr, T_RESIDENT, 0);
  for (int c = 0; c < B.chunks; c++) batch_launch(c);
  timed_end(tr);
  HIPC(hipMemcpyAsync(B.h_out, B.d_out, sizeof(ResOut) * B.small.size(), hipMemcpyDeviceToHost, C.stream));
}

// the small graphs' results (their totals are in host memory), the others' evaluations
static void batch_results(int* diameter, long* sum, double* ASPL)
{
  for (size_t k = 0; k < B.small.size(); k++) {
    int g = B.small[k];
    const ResOut& o = B.h_out[k];
    finish_one(B.nodes[g], o.sum, std::max(1, o.diam), (o.flags & 1) != 0, &diameter[g], &sum[g], &ASPL[g]);
  }
}

static void batch_large(int* diameter, long* sum, double* ASPL)
{
  for (int g : B.large)
    single_eval_dev(B.single, B.nodes[g], B.degrees[g], B.d_adj + B.offsets[g], ODPX_PLAN_AUTO,
                    &diameter[g], &sum[g], &ASPL[g]);
}

extern "C" int ODPX_Batch_run(int* diameter, long* sum, double* ASPL)
{
  RandFence rand_fence;
  ctx_init();
  double t0 = wall_time();
  if (!B.small.empty()) {
    const bool again = B.runs++ > 0;
    if (again) {
      // from the second run on: one chunk, balanced tables
      if (B.chunks > 1) { B.chunks = 1; batch_build_tasks(); B.runs = 2; }
      batch_balance();
    }
    if (graphs_env() && !g_stats_on && again) {
      // replayed graph of the launch sequence, captured on the second run after a
      // load or policy change (a batch run once is launched eagerly)
      if (!B.gexec) {
        hipGraph_t g;
        HIPC(hipStreamBeginCapture(C.stream, hipStreamCaptureModeThreadLocal));
        batch_enqueue();
        HIPC(hipStreamEndCapture(C.stream, &g));
        HIPC(hipGraphInstantiate(&B.gexec, g, nullptr, nullptr, 0));
        HIPC(hipGraphDestroy(g));
      }
      HIPC(hipGraphLaunch(B.gexec, C.stream));
    } else {
      batch_enqueue();
    }
    HIPC(hipStreamSynchronize(C.stream));
    batch_results(diameter, sum, ASPL);
    if (g_stats_on) {
      for (TimedLaunch& t : g_pending) {
        float ms = 0;
        HIPC(hipEventElapsedTime(&ms, t.a, t.b));
        g_evpool.push_back(t.a); g_evpool.push_back(t.b);
        double bytes = 0;
        for (size_t k = 0; k < B.small.size(); k++) {
          const BatchGraph& G = B.hg[k];
          double row = (G.degree + 2.0) * (std::min(32 * B.wb[k], G.n) / 8.0) + 4.0 * G.degree;
          bytes += (double)B.h_out[k].levels * G.n * row;
        }
        g_stats.resident_launches++; g_stats.resident_ms += ms; g_stats.resident_bytes += bytes;
      }
      g_pending.clear();
    }
  }
  batch_large(diameter, sum, ASPL);
  if (g_stats_on) { g_stats.evals += B.ng; g_stats.eval_ms += 1e3 * (wall_time() - t0); }
  return 0;
}

extern "C" int ODPX_Loop_run(int plan, int* diameter, long* sum, double* ASPL)
{
  RandFence rand_fence;
  ctx_init();
  for (int g = 0; g < B.ng; g++)
    single_eval_dev(B.single, B.nodes[g], B.degrees[g], B.d_adj + B.offsets[g], plan, &diameter[g], &sum[g], &ASPL[g]);
  return 0;
}

extern "C" int ODPX_Batch_eval(int ngraphs, const int* nodes, const int* degrees, const long long* offsets,
                               const int* packed, int* diameter, long* sum, double* ASPL)
{
  RandFence rand_fence;
  // Sent in chunks of whole graphs, a chunk's tables built and its blocks run
  // while the next is on its way: four chunks, up to eight as the batch grows past
  // 28 MB (256 graphs of 1024 to 16384 vertices, 114 MB: 9.6 ms in one piece, 7.2 in
  // four, 7.05 in six to eight; 64 graphs, 28 MB: 1.91 in four, 2.12 in eight).  Graphs that lie in the packed
  // array in another order than their own, and small batches, are loaded whole.
  long long end = 0;
  bool pipe = !g_stats_on && ngraphs >= 8;
  for (int g = 0; g < ngraphs && pipe; g++) {
    pipe = nodes[g] >= 1 && degrees[g] >= 0 && offsets[g] >= end;
    if (pipe) end = offsets[g] + (long long)nodes[g] * degrees[g];
  }
  if (!pipe || end * (long long)sizeof(int) < BATCH_PIPE_BYTES) {
    ODPX_Batch_load(ngraphs, nodes, degrees, offsets, packed);
    return ODPX_Batch_run(diameter, sum, ASPL);
  }
  g_routes.chunked++;
  batch_shape(ngraphs, nodes, degrees, offsets);
  if (!B.copies) {
    HIPC(hipStreamCreateWithFlags(&B.copies, hipStreamNonBlocking));
    HIPC(hipEventCreateWithFlags(&B.sent, hipEventDisableTiming));
  }
  int glast[BATCH_CHUNKS + 1] = {0};              // chunk c: graphs glast[c] .. glast[c + 1] - 1
  const int nc = B.chunks = (int)std::max(4LL, std::min((long long)BATCH_CHUNKS, end * (long long)sizeof(int) / (14 << 20) + 2));
  for (int c = 0, g = 0, k = 0; c < nc; c++) {
    B.cfirst[c] = k;
    while (g < ngraphs && (c + 1 == nc || offsets[g] < end / nc * (c + 1)))
      k += batch_wb(nodes[g++]) > 0 ? 1 : 0;
    glast[c + 1] = g;
    B.cfirst[c + 1] = k;
  }
  if (!B.small.empty()) {
    batch_build_tasks();                          // (synchronizes: the buffers are free, the graphs' data there)
    batch_clear();
  } else {
    HIPC(hipStreamSynchronize(C.stream));
  }
  for (int c = 0; c < nc; c++) {
    if (glast[c] == glast[c + 1]) continue;
    const long long lo = offsets[glast[c]], hi = c + 1 < nc && glast[c + 1] < ngraphs ? offsets[glast[c + 1]] : end;
    HIPC(hipMemcpyAsync(B.d_adj + lo, packed + lo, sizeof(int) * (hi - lo), hipMemcpyHostToDevice, B.copies));
    HIPC(hipEventRecord(B.sent, B.copies));
    HIPC(hipStreamWaitEvent(C.stream, B.sent, 0));
    batch_prepare(B.cfirst[c], B.cfirst[c + 1]);
    batch_launch(c);
  }
  if (!B.small.empty())
    HIPC(hipMemcpyAsync(B.h_out, B.d_out, sizeof(ResOut) * B.small.size(), hipMemcpyDeviceToHost, C.stream));
  HIPC(hipMemcpyAsync(B.h_err, B.d_err, sizeof(int), hipMemcpyDeviceToHost, C.stream));
  HIPC(hipStreamSynchronize(C.stream));
  batch_check_err();
  if (!B.small.empty()) { B.runs = 1; batch_results(diameter, sum, ASPL); }
  batch_large(diameter, sum, ASPL);
  return 0;
}

extern "C" int ODPX_Loop_eval(int ngraphs, const int* nodes, const int* degrees, const long long* offsets,
                              const int* packed, int plan, int* diameter, long* sum, double* ASPL)
{
  RandFence rand_fence;
  ODPX_Batch_load(ngraphs, nodes, degrees, offsets, packed);
  return ODPX_Loop_run(plan, diameter, sum, ASPL);
}

extern "C" void ODPX_Batch_get_policy(int* wbcap, int* per_cu)
{
  for (int c = 0; c < BATCH_CLASSES; c++) wbcap[c] = B.wbcap[c];
  *per_cu = B.per_cu;
}

extern "C" int ODPX_Batch_set_policy(const int* wbcap, int per_cu)
{
  RandFence rand_fence;
  for (int c = 0; c < BATCH_CLASSES; c++)
    if (wbcap[c] != 1 && wbcap[c] != 2 && wbcap[c] != 4 && wbcap[c] != 8) return -1;
  if (per_cu != 1 && per_cu != 2) return -1;
  for (int c = 0; c < BATCH_CLASSES; c++) B.wbcap[c] = wbcap[c];
  B.per_cu = per_cu;
  B.chunks = 1;
  if (!B.small.empty()) batch_build_tasks();
  return 0;
}

// Times the loaded batch's resident launch under candidate policies --
// workgroups per CU, then per size class the widest block -- keeping each
// change that makes it faster (coordinate descent from the current policy).
// Every candidate must return identical results (exit(1) otherwise).
extern "C" int ODPX_Batch_autotune(int repeats)
{
  RandFence rand_fence;
  ctx_init();
  if (B.small.empty()) return 0;
  if (repeats < 1) repeats = 1;
  const int ng = B.ng;
  std::vector<int> d0(ng), d1(ng);
  std::vector<long> s0(ng), s1(ng);
  std::vector<double> a0(ng), a1(ng);
  if (B.chunks > 1) { B.chunks = 1; batch_build_tasks(); }
  const std::vector<int> large = B.large;
  B.large.clear();                          // time the resident launch alone
  auto timed_run = [&](std::vector<int>& d, std::vector<long>& sm, std::vector<double>& as) {
    for (int i = 0; i < 2; i++)                          // warm-up, then the balanced tables and the capture
      ODPX_Batch_run(d.data(), sm.data(), as.data());
    double t = wall_time();
    for (int i = 0; i < repeats; i++) ODPX_Batch_run(d.data(), sm.data(), as.data());
    return (wall_time() - t) / repeats;
  };
  double best = timed_run(d0, s0, a0);
  int tried = 1;
  auto consider = [&]() {
    batch_build_tasks();
    const double t = timed_run(d1, s1, a1);
    tried++;
    for (int k = 0; k < ng; k++)
      if (d1[k] != d0[k] || s1[k] != s0[k] || memcmp(&a1[k], &a0[k], sizeof(double)) != 0)
        ODP_ERROR("libodp_hip: batch policies disagree on graph %d\n", k);
    if (t < best) { best = t; return true; }
    return false;
  };
  for (int pc : {1, 2}) {
    if (pc == B.per_cu) continue;
    const int old = B.per_cu;
    B.per_cu = pc;
    if (!consider()) B.per_cu = old;
  }
  bool present[BATCH_CLASSES] = {false, false, false, false, false};
  for (int g : B.small) present[batch_class(B.nodes[g])] = true;
  for (int c = 0; c < BATCH_CLASSES; c++) {
    if (!present[c]) continue;
    for (int cap = RES_WB_MAX; cap >= 1; cap >>= 1) {
      if (cap == B.wbcap[c]) continue;
      const int old = B.wbcap[c];
      B.wbcap[c] = cap;
      if (!consider()) B.wbcap[c] = old;
    }
  }
  batch_build_tasks();
  B.large = large;
  return tried;
}

extern "C" void ODPX_Batch_release(void)
{
  RandFence rand_fence;
  batch_drop_graph();
  dfree(&B.d_adj); dfree(&B.d_nbr); dfree(&B.d_err); dfree(&B.d_qhead); hfree(&B.h_err); dfree(&B.d_gstart);
  dfree(&B.d_g); dfree(&B.d_out); hfree(&B.h_out); dfree(&B.d_t);
  if (B.copies) { HIPC(hipStreamDestroy(B.copies)); HIPC(hipEventDestroy(B.sent)); B.copies = nullptr; B.sent = nullptr; }
  B.chunks = 1;
  B.adj_cap = B.nbr_cap = B.g_cap = B.t_cap = B.gstart_cap = 0;
  B.ng = 0; B.small.clear(); B.large.clear();
  B.single.release();
}

// ---------------------------------------------------------------------------
// allocation-free evaluation: ODP_Set_aspl's result for a general graph, with
// every device buffer in one file-scope array (for callers that cannot allocate)

static const int NOALLOC_MAX_NODES = 16384;
static const int NOALLOC_MAX_DEGREE = 32;
static const size_t NA_ADJ = 0;                                                    // int32[n][degree]
static const size_t NA_TABLE = NA_ADJ + (size_t)NOALLOC_MAX_NODES * NOALLOC_MAX_DEGREE * 4;   // u16[n][dp16]
static const size_t NA_TASKS = NA_TABLE + (size_t)NOALLOC_MAX_NODES * NOALLOC_MAX_DEGREE * 2; // ResTask[n / 32]
static const size_t NA_PARTS = NA_TASKS + (size_t)(NOALLOC_MAX_NODES / 32) * 64;   // ResOut[grid <= n / 32]
static const size_t NA_CTRL = NA_PARTS + (size_t)(NOALLOC_MAX_NODES / 32) * 32;    // qhead, done, err, result
static const size_t NA_BYTES = NA_CTRL + 256;
static_assert(sizeof(ResTask) <= 64 && sizeof(ResOut) <= 32 && sizeof(ResHost) <= 128, "scratch layout");

// 3.1 MiB; each GPU the library runs on holds its own copy until the process ends
static __device__ __align__(256) unsigned char scratch[NA_BYTES];
static unsigned char* g_scratch_dev[64];          // hipGetSymbolAddress of `scratch` per device

// One grid: the 16-bit neighbour table (entry j of row r: adj[r][j] when it is
// a vertex id, r itself past the degree or for -1; other values set *err), the
// task list of 32 * wb-source blocks, and zeroed queue head, arrival counter
// and error flag.
__global__ void k_noalloc_prep(const int* __restrict__ adj, int n, int degree, int dp, int wb,
                               unsigned short* __restrict__ table, ResTask* __restrict__ tasks, int ntasks,
                               int* qhead, u32* done, int* err, int walk_cap)
{
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
  if (tid == 0) { *qhead = 0; *done = 0; }
  for (int64_t i = tid; i < (int64_t)n * dp; i += stride) {
    const int r = (int)(i / dp), j = (int)(i - (int64_t)r * dp);
    int v = r;
    if (j < degree) {
      const int a = adj[(int64_t)r * degree + j];
      if (a >= 0 && a < n) v = a;
      else if (a != -1) atomicOr(err, 1);
    }
    table[i] = (unsigned short)v;
  }
  const int b = 32 * wb;
  for (int64_t t = tid; t < ntasks; t += stride) {
    ResTask T;
    T.nbr = table; T.n = n; T.dp = dp; T.src0 = (int)t * b; T.l = min(b, n - (int)t * b);
    T.s = 1; T.graph = 0; T.wb = wb; T.dq = (max(degree, 1) + 3) / 4;
    T.deg = max(degree, 1); T.walk = min(res_walk_levels(n, T.deg, T.l), walk_cap);
    tasks[t] = T;
  }
}

__global__ void k_noalloc_clear(int* err) { if (threadIdx.x == 0) *err = 0; }

// the device address of `scratch` on the current device, looked up once per device
static unsigned char* noalloc_scratch()
{
  int dev = 0;
  HIPC(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) ODP_ERROR("ODPX_Set_aspl_noalloc: device %d out of range\n", dev);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    HIPC(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_dev[dev] = (unsigned char*)p;
  }
  return g_scratch_dev[dev];
}

extern "C" int ODPX_Set_aspl_noalloc(int nodes, int degree, const int* adjacency, int* diameter, long* sum,
                                     double* ASPL)
{
  RandFence rand_fence;
  if (nodes < 1 || nodes > NOALLOC_MAX_NODES || degree < 1 || degree > NOALLOC_MAX_DEGREE || !adjacency) {
    fprintf(stderr, "ODPX_Set_aspl_noalloc: nodes (%d) must be in [1, %d] and degree (%d) in [1, %d]\n", nodes,
            NOALLOC_MAX_NODES, degree, NOALLOC_MAX_DEGREE);
    return -1;
  }
  ctx_init();
  unsigned char* base = noalloc_scratch();
  int* d_adj = (int*)(base + NA_ADJ);
  unsigned short* d_table = (unsigned short*)(base + NA_TABLE);
  ResTask* d_tasks = (ResTask*)(base + NA_TASKS);
  ResOut* d_parts = (ResOut*)(base + NA_PARTS);
  int* d_qhead = (int*)(base + NA_CTRL);
  u32* d_done = (u32*)(base + NA_CTRL + 4);
  int* d_err = (int*)(base + NA_CTRL + 8);
  ResHost* d_res = (ResHost*)(base + NA_CTRL + 128);
  // block width and workgroup size as the resident plan picks them for this graph
  int wbmax = 0;
  for (int wb = RES_WB_MAX; wb >= 1 && !wbmax; wb >>= 1)
    if ((size_t)nodes * wb * 4 <= LDS_DYN_MAX && nodes <= res_rpt(wb) * 1024) wbmax = wb;
  const int wb = res_width(nodes, nodes, std::max(wbmax, 1), C.ncu);
  int threads = 1024;
  for (int th : {256, 512, 1024})
    if (nodes <= res_rpt(wb) * th && (nodes >= 4096 ? th == 1024 : (nodes > 512 ? th >= 512 : true))) {
      threads = th;
      break;
    }
  const int dp = round_up(degree, 8), ntasks = (nodes + 32 * wb - 1) / (32 * wb);
  const size_t lds = (size_t)nodes * wb * 4;
  const int per_cu = std::min((int)std::max<size_t>(1, LDS_LIMIT / (lds + LDS_STATIC)), 2048 / threads);
  const int grid = std::max(1, std::min(ntasks, per_cu * C.ncu));
  hipStream_t st = C.stream;
  HIPC(hipMemcpyAsync(d_adj, adjacency, sizeof(int) * (size_t)nodes * degree, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_noalloc_clear, dim3(1), dim3(64), 0, st, d_err);
  const int64_t work = std::max<int64_t>((int64_t)nodes * dp, ntasks);
  hipLaunchKernelGGL(k_noalloc_prep, dim3((int)std::min<int64_t>((work + 255) / 256, 1024)), dim3(256), 0, st,
                     d_adj, nodes, degree, dp, wb, d_table, d_tasks, ntasks, d_qhead, d_done, d_err, res_walk_cap());
  HIPC(hipGetLastError());
  ResFin fin{};
  fin.done = d_done; fin.part = d_parts; fin.host = d_res; fin.err = d_err;
  auto kern = wb == 1 ? k_resident_w<1> : wb == 2 ? k_resident_w<2> : wb == 4 ? k_resident_w<4> : k_resident_w<8>;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(threads), lds, st, d_tasks, ntasks, d_qhead, (ResOut*)nullptr, fin);
  HIPC(hipGetLastError());
  ResHost res;
  HIPC(hipMemcpyAsync(&res, d_res, sizeof res, hipMemcpyDeviceToHost, st));
  HIPC(hipStreamSynchronize(st));
  if (res.err) ODP_ERROR("adjacency holds a vertex id outside [0, nodes) within num_degrees\n");
  finish_one(nodes, res.out.sum, std::max(1, res.out.diam), (res.out.flags & 1) != 0, diameter, sum, ASPL);
  return 0;
}

// ---------------------------------------------------------------------------
// serving engine
#include "serve.hpp"
