// kernels.hpp -- gfx950 (CDNA4, wave64) kernels of the bit-matrix ASPL/diameter
// method.  Included once, by aspl_hip.hip.
//
// The method is the reference's (aspl.c:35-119, aspl_cuda.cu:53-126,
// utils_cuda.cu:97-211): bit c of row v says "source c reaches v"; each level
// computes next[v] = cur[v] | OR_{u in N(v)} cur[u] on 64-bit words and
// popcounts next.  Two kernel families implement it:
//
//  * level kernels (k_level0, k_level): one launch per BFS level for every
//    column block ("task") of one or more graphs.  A wave owns a segment of
//    64..128 words of a row (16 B per lane, so every neighbour gather is one
//    coalesced 512 B..1 KiB stream).  The popcount is fused and reduced per
//    wave into one 64-bit atomic; termination (count == n*l) is detected on
//    the device by the next level's workgroups, so the host needs no sync per
//    level (the reference syncs every level, aspl_cuda.cu:67).  Counts live in
//    a ring of `ring` slots per task; level L zeroes slot L+1 before level L+1
//    adds into it, and the host reads the ring between batches of levels.
//  * resident kernel (k_resident): for graphs small enough that a block of
//    32*wb sources of BOTH bit buffers fits in the 160 KiB LDS of a CU,
//    one workgroup runs every level of one block in LDS.  Workgroups pull
//    blocks from a work queue (one atomic counter), so many graphs of uneven
//    size are evaluated in one persistent launch.
//
// Neighbour ids reaching these kernels come from the row-neighbour table
// built by k_prepare: every entry is a valid row index (short rows are padded
// with the row's own index, which ORs in nothing new), so no gather can leave
// the bit buffers.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

typedef unsigned long long u64;
typedef unsigned int u32;

struct __attribute__((aligned(16))) u64x2 { u64 x, y; };
typedef u64 u64v2 __attribute__((ext_vector_type(2)));

#define ODP_NXCD 8          // XCDs of an MI355X; workgroups are dealt round-robin
#define LEVEL_WG 256        // threads per level-kernel workgroup (4 waves)
#define LV_STORE 1          // k_level mode bits: write the next rows
#define LV_COUNT 2          //   ... and add the level's counts (both: a normal level)
#define LV_LIST 4           //   ... and list the chunks left unsaturated (k_level's LS variant)
#define LV_SPARSE 8         // the count-only level as k_sparse over that list
#define LV_THIN 16          // k_pgather: a part of the neighbours, the unsaturated chunks listed with their bits

// chunks (task, row, 16-byte word pair) a level left unsaturated; only those
// can gain bits at the next level.  The list is LIST_SUBS sub-lists with a
// counter each (128 bytes apart), a workgroup appending to sub-list
// blockIdx.x % LIST_SUBS: one counter for the whole GPU serialised the appends
// (a listing level of n = 49152, d = 4 took 3.4 ms against 0.2 ms unlisted).
#define LIST_SUBS 64
#define LIST_PAD 32
struct LvList {
  u64* e;              // sub-list s at e + s * cap; entries: task << 48 | row << 24 | word
  u32* n;              // sub-list s's count at n[s * LIST_PAD] (may exceed cap: then no list is used)
  u32 cap;             // entries per sub-list
  u64x2* v;            // the entries' chunks (16 bytes each), or null
};

// ---------------------------------------------------------------------------
// shared helpers

// appends the wave's lanes with `unsat` set to the workgroup's sub-list: one
// atomic per wave.  Called by whole waves.  V: with the chunks' bits, where the
// list takes them.  k_level's lists never do, and it has an instance without the
// branch: four registers fewer, a listing level of n = 22000, d = 64 in 0.27 instead of 0.39 ms
template <bool V>
__device__ __forceinline__ void list_append(const LvList& lst, bool unsat, u64 val, u64 x = 0, u64 y = 0)
{
  const u64 m = __ballot(unsat);
  if (!m) return;
  const u32 sub = blockIdx.x % LIST_SUBS, lane = threadIdx.x & 63;
  u32 b = 0;
  if (lane == 0) b = atomicAdd(lst.n + sub * LIST_PAD, (u32)__popcll(m));
  b = __builtin_amdgcn_readfirstlane(b);
  if (unsat) {
    const u32 e = b + (u32)__popcll(m & ((1ULL << lane) - 1));
    if (e < lst.cap) {
      lst.e[(u64)sub * lst.cap + e] = val;
      if (V && lst.v) { u64x2 o; o.x = x; o.y = y; lst.v[(u64)sub * lst.cap + e] = o; }
    }
  }
}

// the wave's sum, by adds between lanes (DPP: no LDS trips, as shuffles make);
// the same value in every lane, in a scalar register
__device__ __forceinline__ u32 wave_sum_dpp(u32 v)
{
  v += __builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);   // row_shr:8
  v += __builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast:15
  v += __builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast:31
  return (u32)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ u64 wave_sum(u64 v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// valid-bit mask of word w of a block holding l sources
__device__ __forceinline__ u64 full_word(int l, int w)
{
  int v = l - 64 * w;
  return v >= 64 ? ~0ULL : (v <= 0 ? 0ULL : ((1ULL << v) - 1ULL));
}

// blockIdx -> logical index so that each XCD gets one contiguous range
__device__ __forceinline__ int remap_xcd(int b, int nb)
{
  int q = nb / ODP_NXCD, r = nb % ODP_NXCD, x = b % ODP_NXCD, i = b / ODP_NXCD;
  return x * q + (x < r ? x : r) + i;
}

// ---------------------------------------------------------------------------
// k_prepare: caller adjacency -> row-neighbour table.
//
//  s == 1              : row i, neighbour adj[i][j]                      (utils_cuda.cu:101-113)
//  general, s > 1      : row i = p*b+m, neighbour adj[m][j] + p*b (mod n) (utils_cuda.cu:133-151)
//  grid, s in {2, 4}   : vertex i lives in row itable[i]; neighbour is the
//                        rotated first-quadrant entry (utils_cuda.cu:3-59, 117-132)
// Entries j >= num_degrees[i] become the row itself.  Ids outside [0, n) set
// *err and are replaced by the row itself (the reference would read out of
// bounds; the host turns *err into the reference's print-and-exit).
// The first threads also reset the per-evaluation counters.

struct PrepArgs {
  const int* adj;        // [(n/s)][degree]
  const int* numdeg;     // [n] expanded, or null
  const int* itable;     // [n] or null
  int* nbr;              // [n][dpad] 32-bit ids, or null
  unsigned short* nbr16; // [n][dpad] 16-bit ids (n <= 65536), or null (both may be written)
  int* err;
  int n, s, degree, dpad, width, height, grid_s;
  u64* zero64; int nzero64;   // counters reset to 0 at the start of an evaluation
  u32* zero32; int nzero32;
  int* adj_copy; int64_t adj_elems;   // adj is in host memory: also copy it here (or null)
};

__device__ __forceinline__ int grid_rotate(int v, int width, int height, int s, int angle)
{
  int w = v / height, h = v % height;
  if (s == 2) return (width - w - 1) * height + (height - h - 1);
  if (angle == 90) return h * height + (height - w - 1);
  if (angle == 180) return (height - w - 1) * height + (height - h - 1);
  return (height - h - 1) * height + w;
}

// neighbour d of vertex v of a 2/4-fold symmetric grid; -1 when the table
// entry is not a vertex id
__device__ __forceinline__ int grid_nbr(const int* adj, int width, int height, int degree, int s, int v, int d)
{
  int n = width * height, bw = width / 2, bh = height / 2, w = v / height, h = v % height;
  int base, back = 0;
  if (s == 2) {
    if (w < bw) base = v;
    else { base = grid_rotate(v, width, height, 2, 180); back = 180; }
  } else {
    int x = v, lx;
    if (w < bw && h < bh) back = 0;
    else if (w < bw) { x = grid_rotate(v, width, height, 4, 270); back = 90; }
    else if (h >= bh) { x = grid_rotate(v, width, height, 4, 180); back = 180; }
    else { x = grid_rotate(v, width, height, 4, 90); back = 270; }
    lx = (x / height) * bh + (x % height);
    base = lx;
  }
  int y = adj[(int64_t)base * degree + d];
  if (y < 0 || y >= n) return -1;
  return back ? grid_rotate(y, width, height, s, back) : y;
}

__global__ void k_prepare(PrepArgs a)
{
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = tid; i < a.nzero64; i += stride) a.zero64[i] = 0;
  for (int64_t i = tid; i < a.nzero32; i += stride) a.zero32[i] = 0;
  const int64_t total = (int64_t)a.n * a.dpad;
  const bool plain = a.s == 1 && !a.grid_s;
  // a table in host memory is bound by the link: an entry is read once, for the
  // copy and the table together (n = 1024, d = 6: 5.3 -> 4.6 us; n = 5001, d = 10: 11 -> 7.1)
  const bool both = a.adj_copy && plain && total > 0;
  if (a.adj_copy && !both)
    for (int64_t i = tid; i < a.adj_elems; i += stride) a.adj_copy[i] = a.adj[i];
  const int b = a.n / a.s;
  for (int64_t idx = tid; idx < total; idx += stride) {
    const int i = total <= 0xffffffffLL ? (int)((u32)idx / (u32)a.dpad) : (int)(idx / a.dpad);
    const int j = (int)(idx - (int64_t)i * a.dpad);
    int e = 0;
    if (plain && j < a.degree) {
      e = a.adj[(int64_t)i * a.degree + j];
      if (both) a.adj_copy[(int64_t)i * a.degree + j] = e;
    }
    const int row = a.grid_s ? a.itable[i] : i;
    int d = a.numdeg ? a.numdeg[i] : a.degree;
    if (d < 0 || d > a.degree) { atomicOr(a.err, 2); d = d < 0 ? 0 : a.degree; }
    int out = row;
    if (j < d) {
      int v;
      if (a.grid_s) {
        v = grid_nbr(a.adj, a.width, a.height, a.degree, a.s, i, j);
      } else if (plain) {
        v = e < a.n ? e : -1;
      } else {
        const int p = i / b, m = i - p * b;
        v = a.adj[(int64_t)m * a.degree + j];
        if (v >= a.n) v = -1;
        if (v >= 0) { v += p * b; if (v >= a.n) v -= a.n; }
      }
      if (v < 0) atomicOr(a.err, 1);
      else out = a.grid_s ? a.itable[v] : v;
    }
    if (a.nbr16) a.nbr16[(int64_t)row * a.dpad + j] = (unsigned short)out;
    if (a.nbr) a.nbr[(int64_t)row * a.dpad + j] = out;
  }
}

// the row-neighbour tables a device swap patches along with the adjacency
struct SwapTables {
  int* t32;                 // 32-bit table or null
  unsigned short* t16;      // 16-bit table or null
  int tdp;                  // their row stride
};

// 2-opt swap a-b, c-d -> a-c, b-d on the device adjacency (s = 1), all or
// nothing: one thread finds the four entries first (rows a, b, c, d holding b,
// a, d, c) and writes only when all four exist; otherwise it changes nothing
// and sets bit 4 of *err.  The ids must be distinct (the host checks), so the
// four entries are four different cells.  The tables set in `tb` are patched
// entry for entry: a table row holds the adjacency's entry where it is a
// neighbour and the row itself where it is padding, so an entry equal to
// `from` is the same edge.
__global__ void k_swap(int* adj, int degree, int a, int b, int c, int d, int* err, SwapTables tb)
{
  __shared__ int spos[4];
  auto row = [&](int e) { return e == 0 ? a : e == 1 ? b : e == 2 ? c : d; };
  auto from = [&](int e) { return e == 0 ? b : e == 1 ? a : e == 2 ? d : c; };
  auto to = [&](int e) { return e == 0 ? c : e == 1 ? d : e == 2 ? a : b; };
  if (threadIdx.x < 4) spos[threadIdx.x] = INT_MAX;
  __syncthreads();
  // the four rows' entries are read at once; a row's first match wins
  for (int i = threadIdx.x; i < 4 * degree; i += blockDim.x) {
    const int e = i / degree, j = i - e * degree;
    if (adj[(int64_t)row(e) * degree + j] == from(e)) atomicMin(&spos[e], j);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int e = 0; e < 4; e++)
    if (spos[e] == INT_MAX) { atomicOr(err, 4); return; }
  for (int e = 0; e < 4; e++) {
    adj[(int64_t)row(e) * degree + spos[e]] = to(e);
    const int64_t k = (int64_t)row(e) * tb.tdp + spos[e];
    if (tb.t16 && tb.t16[k] == (unsigned short)from(e)) tb.t16[k] = (unsigned short)to(e);
    if (tb.t32 && tb.t32[k] == from(e)) tb.t32[k] = to(e);
  }
}

// Sets *asym unless the table is symmetric: row u holds row r as many times as
// row r holds u (entries equal to the row itself are padding).  Counting the
// repeats makes the property outlive 2-opt swaps: each removes and adds one
// entry of both directions.  A thread per entry, 16 bytes a load, a row's loads
// in flight together (Q of them; 0: any width): 12 us at n = 65536, d = 16, 21 with
// the loads one after the other, 41 over single ids.
template <int Q>
__global__ void k_symcheck(const int* __restrict__ nbr, int n, int dpad, u32* asym)
{
  const int64_t total = (int64_t)n * dpad;
  bool bad = false;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int r = (int)((u32)(idx >> 2) / (u32)(dpad >> 2));     // dpad is a multiple of 4; n dpad < 2^33
    const int u = nbr[idx];
    if (u == r) continue;
    const int4* own = (const int4*)(nbr + (int64_t)r * dpad);
    const int4* his = (const int4*)(nbr + (int64_t)u * dpad);
    int c = 0;
    auto add = [&](const int4& o, const int4& h) {
      c += (o.x == u) + (o.y == u) + (o.z == u) + (o.w == u);
      c -= (h.x == r) + (h.y == r) + (h.z == r) + (h.w == r);
    };
    if (Q) {
      int4 o[Q ? Q : 1], h[Q ? Q : 1];
#pragma unroll
      for (int k = 0; k < Q; k++) { o[k] = own[k]; h[k] = his[k]; }
#pragma unroll
      for (int k = 0; k < Q; k++) add(o[k], h[k]);
    } else {
      for (int k = 0; k < dpad >> 2; k++) add(own[k], his[k]);
    }
    bad = bad || c != 0;
  }
  // a wave adds once, and not where the flag is set: a thread each, as a table of
  // n = 65536, d = 16 directed entries did, queued a million adds on one word (180 us)
  if (__ballot(bad) && (threadIdx.x & 63) == 0 &&
      __hip_atomic_load(asym, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    atomicOr(asym, 1u);
}

// ---------------------------------------------------------------------------
// level kernels

struct LevelTask {
  const int* nbr;      // [n][dpad]
  u64* buf0;           // [n][kwp]  level L reads buf[L&1], writes buf[(L+1)&1]
  u64* buf1;
  u64* cnt;            // per-level popcount of this task: cnt[(L % ring) * cstride]
  u32* done;           // set once the task has terminated
  int n, dpad, kwp;    // rows, neighbour-table width, words per row in the buffers
  int src0, l;         // first source (row index) of the block, sources in it
  int lpr_log2;        // log2(lanes per row): 6 -> one row per wave
  int segs;            // 2*64-word segments per row (kwp / (2 * lanes per row))
  int rgroups;         // ceil(n / rows per wave)
  int units;           // rgroups * segs wave-units
  int seg_major;       // unit order: segment-major (1) or row-major (0)
  int cstride;         // level stride of cnt and ccnt
  int pad;
  u64* ccnt;           // per-level count of changed (row, segment) units: ccnt[(L % ring) * cstride]
  u64* acnt;           // per-level count of processed (row, segment) units, same layout
  unsigned char* chg0; // changed flag of (segment s, row r) at [s * n + r]: levels of even parity
  unsigned char* chg1; //   ... and of odd parity
  unsigned char* act0; // "may change" marks of (segment, row) for levels of even parity (push mode)
  unsigned char* act1; //   ... and of odd parity
  const u32* asym;     // nonzero when the table is not symmetric (push mode needs u in N(r) <=> r in N(u))
  unsigned char* wgm0; // per workgroup of the task: some row of it is marked (push mode), even levels
  unsigned char* wgm1; //   ... odd levels
};

// workgroup (within its task) that processes segment seg of row r, for upw
// units per wave and 4 waves per workgroup
__device__ __forceinline__ int unit_wg(const LevelTask& T, int r, int seg, int upw)
{
  const int rg = r >> (6 - T.lpr_log2);
  const int u = T.seg_major ? seg * T.rgroups + rg : rg * T.segs + seg;
  return u / (4 * upw);
}

__device__ __forceinline__ int find_task(const int* __restrict__ wg_start, int ntasks, int g)
{
  int lo = 0, hi = ntasks - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (wg_start[mid] <= g) lo = mid; else hi = mid - 1;
  }
  return lo;
}

struct UnitGeom { int r, w, seg; };

__device__ __forceinline__ UnitGeom unit_geom(const LevelTask& T, int u, int lane)
{
  int seg, rg;
  if (T.seg_major) { seg = u / T.rgroups; rg = u - seg * T.rgroups; }
  else { rg = u / T.segs; seg = u - rg * T.segs; }
  const int lpr = 1 << T.lpr_log2;
  UnitGeom g;
  g.r = (rg << (6 - T.lpr_log2)) + (lane >> T.lpr_log2);
  g.w = seg * (2 * lpr) + 2 * (lane & (lpr - 1));
  g.seg = seg;
  return g;
}

__device__ __forceinline__ void put_bit(u64& x0, u64& x1, int c, int l, int w)
{
  if ((unsigned)c < (unsigned)l) {
    const int cw = c >> 6;
    const u64 bit = 1ULL << (c & 63);
    if (cw == w) x0 |= bit;
    else if (cw == w + 1) x1 |= bit;
  }
}

// Level 0 of every task straight from the identity: next[r] holds the bits of
// r itself and of its neighbours (cur = identity needs no reads).
__global__ __launch_bounds__(LEVEL_WG) void k_level0(const LevelTask* __restrict__ tasks,
                                                     const int* __restrict__ wg_start, int ntasks,
                                                     int ring, int upw, int xcd)
{
  int g = blockIdx.x;
  if (xcd) g = remap_xcd(g, gridDim.x);
  const int t = ntasks > 1 ? find_task(wg_start, ntasks, g) : 0;
  const LevelTask T = tasks[t];
  const int wg = g - wg_start[t];
  if (wg == 0 && threadIdx.x == 0) T.cnt[(int64_t)(1 % ring) * T.cstride] = 0;   // level 1's slot
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  u64 pop = 0;
  const int base = wg * 4 * upw;
  for (int i = 0; i < upw; i++) {
    const int u = base + i * 4 + wave;
    if (u >= T.units) break;
    const UnitGeom q = unit_geom(T, u, lane);
    if (q.r < T.n) {
      u64 x0 = 0, x1 = 0;
      put_bit(x0, x1, q.r - T.src0, T.l, q.w);
      const int* nb = T.nbr + (int64_t)q.r * T.dpad;
      for (int j = 0; j < T.dpad; j += 4) {
        const int4 v = *(const int4*)(nb + j);
        put_bit(x0, x1, v.x - T.src0, T.l, q.w);
        put_bit(x0, x1, v.y - T.src0, T.l, q.w);
        put_bit(x0, x1, v.z - T.src0, T.l, q.w);
        put_bit(x0, x1, v.w - T.src0, T.l, q.w);
      }
      u64x2 o; o.x = x0; o.y = x1;
      *(u64x2*)(T.buf1 + (int64_t)q.r * T.kwp + q.w) = o;
      pop += (u64)(__popcll(x0) + __popcll(x1));
    }
  }
  pop = wave_sum(pop);
  if (lane == 0 && pop) atomicAdd(T.cnt, pop);
}

// One gather level L >= 1 of every task.  UROW: one row per wave, so the row's
// neighbour ids are wave-uniform (scalar loads).  G: neighbour rows gathered
// per batch (in flight together) before the wave checks for saturation.
//
// FR (chosen per evaluation, for graphs with many levels): every level records,
// per (row, segment), whether the segment changed and how many did.  For a
// symmetric table (push mode) a changed segment also marks itself and its
// neighbours' segments for level L+1, so the next level tests one byte per
// row; otherwise it tests the row's and its neighbours' changed flags (pull).
// When fewer than half changed at level L-1 (and L-1 was not the first
// gathered level, which wrote every row), level L runs in frontier
// mode: a segment whose row and neighbours all stayed unchanged at L-1 cannot
// change at L, and the buffer level L writes already holds its value (the
// level L-2 value, equal to L-1's), so it is skipped -- no reads, no write.
// The count of level L is the count of L-1 plus each processed segment's
// gain, which equals the popcount of the whole level.
//
// mode: LV_STORE | LV_COUNT for a normal level; LV_COUNT alone for a level
// expected to be the last one (its rows are never read again, so they are not
// written); LV_STORE alone to write the rows of such a level after all when
// it turned out not to be the last (its counts are already in place).  The
// LS variant (plain mode only) also appends every chunk it leaves unsaturated
// to lst (LV_LIST), for k_sparse to count the next level from.
template <bool UROW, int G, bool FR, bool LS>
__global__ __launch_bounds__(LEVEL_WG) void k_level(const LevelTask* __restrict__ tasks,
                                                    const int* __restrict__ wg_start, int ntasks,
                                                    int level, int ring, int upw, int xcd, int first_level,
                                                    int mode, LvList lst)
{
  int g = blockIdx.x;
  if (xcd) g = remap_xcd(g, gridDim.x);
  const int t = ntasks > 1 ? find_task(wg_start, ntasks, g) : 0;
  const LevelTask T = tasks[t];
  if (*T.done) return;
  const u64 target = (u64)T.n * (u64)T.l;
  const u64 c1 = T.cnt[(int64_t)((level - 1) % ring) * T.cstride];
  {
    const bool stop = (c1 == target) || (level >= 2 && c1 == T.cnt[(int64_t)((level - 2) % ring) * T.cstride]);
    if (stop) {
      if (threadIdx.x == 0) *T.done = 1;
      return;
    }
  }
  const int wg = g - wg_start[t];
  const bool count = (mode & LV_COUNT) != 0, store = (mode & LV_STORE) != 0;
  if (count && wg == 0 && threadIdx.x == 0) {
    T.cnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
    if (FR) {
      T.ccnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
      T.acnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
      atomicAdd(&T.cnt[(int64_t)(level % ring) * T.cstride], c1);    // the gains below add to it
    }
  }
  const bool fr = FR && level > first_level &&
                  2 * T.ccnt[(int64_t)((level - 1) % ring) * T.cstride] < (u64)T.n * (u64)T.segs;
  const unsigned char* __restrict__ chr = (level & 1) ? T.chg0 : T.chg1;   // written by level L-1
  unsigned char* __restrict__ chw = (level & 1) ? T.chg1 : T.chg0;
  const bool push = FR && *T.asym == 0;
  unsigned char* actr = (level & 1) ? T.act1 : T.act0;    // marks for this level
  unsigned char* actw = (level & 1) ? T.act0 : T.act1;    // marks for level L+1
  unsigned char* wgmw = (level & 1) ? T.wgm0 : T.wgm1;
  if (fr && push) {
    // a workgroup none of whose rows is marked has nothing to do at this level
    unsigned char* wgmr = (level & 1) ? T.wgm1 : T.wgm0;
    if (wgmr[wg] == 0) return;
    __syncthreads();                                   // every thread has read the mark
    if (store && threadIdx.x == 0) wgmr[wg] = 0;       // cleared like the row marks
  }
  const u64* __restrict__ cur = (level & 1) ? T.buf1 : T.buf0;
  u64* __restrict__ nxt = (level & 1) ? T.buf0 : T.buf1;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int lpr = 1 << T.lpr_log2;
  const u64 gmask = lpr == 64 ? ~0ULL : ((1ULL << lpr) - 1);
  const int64_t kwp = T.kwp;
  u64 pop = 0, nch = 0, nact = 0;
  const int base = wg * 4 * upw;
  for (int i = 0; i < upw; i++) {
    const int u = base + i * 4 + wave;
    if (u >= T.units) break;
    UnitGeom q = unit_geom(T, u, lane);
    if (UROW) q.r = __builtin_amdgcn_readfirstlane(q.r);
    bool unsat = false;
    if (q.r < T.n) {
      const int64_t so = (int64_t)q.seg * T.n;
      const int* nb = T.nbr + (int64_t)q.r * T.dpad;
      bool act = true;
      if (fr && push) {
        // marked by level L-1 for a change of this row or a neighbour; the pass
        // that writes the rows clears the mark (a count-only pass leaves it for
        // its store-only re-run), so the array is clean when level L+1 marks it
        act = actr[so + q.r] != 0;
        if (act && store && (lane & (lpr - 1)) == 0) actr[so + q.r] = 0;
      } else if (fr) {
        act = chr[so + q.r] != 0;
        for (int j = 0; j < T.dpad && !act; j += 4) {
          const int4 v = *(const int4*)(nb + j);
          act = (chr[so + v.x] | chr[so + v.y] | chr[so + v.z] | chr[so + v.w]) != 0;
        }
      }
      bool changed = false;
      if (act) {
        const u64 f0 = full_word(T.l, q.w), f1 = full_word(T.l, q.w + 1);
        const u64x2 x0 = *(const u64x2*)(cur + q.r * kwp + q.w);
        u64x2 x = x0;
        // Once a lane's words are saturated the remaining neighbours cannot add
        // a bit (OR is monotone): the lane stops gathering (its loads are masked
        // off, so they cost no memory requests) and the wave stops once every
        // lane has.
        bool need = !(x.x == f0 && x.y == f1);
        if (__any(need)) {
          for (int j = 0; j < T.dpad; j += G) {
            int id[G];
#pragma unroll
            for (int k = 0; k < G; k += 4) {
              int4 v;
              if (need && (k == 0 || j + k < T.dpad)) v = *(const int4*)(nb + j + k);
              else { v.x = q.r; v.y = q.r; v.z = q.r; v.w = q.r; }
              id[k] = v.x; id[k + 1] = v.y; id[k + 2] = v.z; id[k + 3] = v.w;
            }
            u64x2 gv[G];
#pragma unroll
            for (int k = 0; k < G; k++) {
              if (need) gv[k] = *(const u64x2*)(cur + (int64_t)id[k] * kwp + q.w);
              else { gv[k].x = 0; gv[k].y = 0; }
            }
#pragma unroll
            for (int k = 0; k < G; k++) { x.x |= gv[k].x; x.y |= gv[k].y; }
            need = !(x.x == f0 && x.y == f1);
            if (!__any(need)) break;
          }
        }
        if (store) *(u64x2*)(nxt + q.r * kwp + q.w) = x;
        if (LS) unsat = !(x.x == f0 && x.y == f1);
        if (FR) {
          changed = x.x != x0.x || x.y != x0.y;
          pop += (u64)(__popcll(x.x) + __popcll(x.y) - __popcll(x0.x) - __popcll(x0.y));
        } else {
          pop += (u64)(__popcll(x.x) + __popcll(x.y));
        }
      }
      if (FR && count) {
        // the segment changed if any of its lanes did
        const u64 m = __ballot(changed);
        const bool any = ((m >> (lane & ~(lpr - 1))) & gmask) != 0;
        if ((lane & (lpr - 1)) == 0) {
          if (!push) chw[so + q.r] = any ? 1 : 0;     // push mode reads marks, not flags
          nch += any ? 1 : 0;
          nact += act ? 1 : 0;
        }
        if (push && any) {
          // mark the row and its neighbours for level L+1 (the table is symmetric:
          // the rows that gather this one are its neighbours), and their
          // workgroups; the row's lanes share the neighbours
          if ((lane & (lpr - 1)) == 0) {
            actw[so + q.r] = 1;
            wgmw[unit_wg(T, q.r, q.seg, upw)] = 1;
          }
          for (int j = lane & (lpr - 1); j < T.dpad; j += lpr) {
            const int x = nb[j];
            actw[so + x] = 1;
            wgmw[unit_wg(T, x, q.seg, upw)] = 1;
          }
        }
      }
    }
    if (LS) list_append<false>(lst, unsat, ((u64)t << 48) | ((u64)q.r << 24) | (u64)q.w);   // a slot per unsaturated chunk
  }
  if (!count) return;
  pop = wave_sum(pop);
  if (lane == 0 && pop) atomicAdd(&T.cnt[(int64_t)(level % ring) * T.cstride], pop);
  if (FR) {
    nch = wave_sum(nch);
    nact = wave_sum(nact);
    if (lane == 0 && nch) atomicAdd(&T.ccnt[(int64_t)(level % ring) * T.cstride], nch);
    if (lane == 0 && nact) atomicAdd(&T.acnt[(int64_t)(level % ring) * T.cstride], nact);
  }
}

// ---------------------------------------------------------------------------
// part-phased gather level (k_pgather): the plain level of k_level for blocks
// of 16 words (128-byte rows), arranged so that one XCD's L2 holds what its
// workgroups gather from.
//
// A block's input slab (n rows x 128 B: 8 MiB at n = 65536) does not fit the
// 4 MB L2 of an XCD, and random neighbours spread the gathers over all of it.
// So the rows of the slab are cut into P parts (rows [p n / P, (p+1) n / P)).
// Rows are taken in units of PG_UNIT consecutive rows; for every unit and part
// a list holds the unit's (row, neighbour) pairs whose neighbour lies in that
// part (the row itself counts as a neighbour; repeats are dropped), built by
// k_plist with the table (a device swap rebuilds the units of the rows it
// changes).  Workgroups are persistent and grouped
// by XCD (workgroup b runs on XCD b % 8): the workgroups of one XCD take
// consecutive units -- the same block -- and sweep the parts in order, with
// their rows' next values accumulated in LDS (ds_or) across the sweep.  While
// they are in part p, the XCD's gathers fall into one n/P-row piece of the slab
// (2 MiB at P = 4), which its L2 keeps.  The gathers need no masking (every
// pair is a 128-byte row read) and none waits for another.  Counts, stop test
// and listing are k_level's (the plain variant): every result is bit-identical.
//
// Folded levels.  With a symmetric table the bit matrix of every level is
// symmetric: 1024 rows of a 1024-column block are the transpose of the rows
// and block across the diagonal.  When every block of the matrix is resident
// (s = 1, 16-word blocks), a level runs the units of one of each such pair and
// stores both: a unit's rows and, transposed in LDS, its mirror's.  Its bits count
// for both blocks.  Half the gathers for 6 us of mirroring a unit of 50:
// a level of n = 65536, d = 16 went from 677 to 459 us.  Of a block t the rows
// of blocks t, t + 1, ..., t + (T - 1) / 2 (mod T, T blocks) run, so every block has
// as many and an XCD still works on one block's slab at a time; for even T the
// rows t + T / 2 of the first half of the blocks come last.  Whether the table is
// symmetric is read on the device (k_symcheck); other tables run every unit.

#define PG_MAXP 4
#define PG_SUB 8             // pieces of a unit's rows in its offsets (128 rows each)
#define PG_OFF (2 * PG_MAXP * PG_SUB + 1)   // offsets of a unit's pair list: per part, its thin pairs and the
                             // others, per piece; then its end
#ifndef PG_SLOTS
#define PG_SLOTS 12          // gathers a wave keeps in flight (registers: 4 per slot)
#endif
#define PG_CH (8 * PG_SLOTS) // pairs of a chunk
#define PG_NL ((PG_CH + 63) / 64)
#define PG_UNIT 1024         // rows of a unit (and sources of a 16-word block, which a folded unit mirrors to):
                             // 128 KiB of LDS rows, one workgroup per CU.  With 512 rows and two workgroups, whose
                             // phases drift apart, the XCD's L2 holds more than one part: 762 against 665 us a level
#define PG_WG PG_UNIT        // threads of the workgroup: 64 rows a wave at the end
#define PG_CUT_MAX 3         // log2 of the pieces of a unit: two waves' rows are the smallest

struct PgArgs {
  const u32* list;       // per unit, parts in order: (row in unit) << 22 | neighbour
  const int* poff;       // per unit PG_OFF offsets into its list (relative to unit * PG_UNIT * sp): piece k of
                         // part p's thin pairs starts at [2 p * PG_SUB + k], of its others at [(2 p + 1) * PG_SUB + k],
                         // the list ends at [2 P * PG_SUB]
  int n, sp, P;
  int upt;               // units per task: ceil(n / PG_UNIT)
  int ntasks;
  const u32* asym;       // folded levels unless *asym (null: never; needs one task per PG_UNIT rows)
  int cut_full, cut_fold;  // log2 of the pieces a unit of the last, partly filled round is cut into (<= PG_CUT_MAX)
};

// One workgroup of PG_UNIT threads per unit, a thread per row: the row's
// distinct neighbours and the row itself (padding entries are the row), their
// parts, a scan of the rows' run lengths per part, and the unit's pairs
// grouped by part with the part offsets.  A part's thin pairs come first: the
// row itself and its first `thin` neighbours, in the order of the parts (a thin
// level, LV_THIN, takes those alone); rows ascend within either group.
// DMAX >= dpad + 1 bounds the ids a row holds in registers (DMAX = 64: 22 of 150
// spilled since the pairs have a thin part, 92 bytes a lane; with the levels it
// serves, a move and an evaluation of n = 50000, d = 60 went 2563 -> 1463 us).
//
// A device swap (or a small change of an uploaded table) hands the changed
// entries to the units it rebuilds (rows, positions in the row, old and new
// ids), so that they see them whether or not the table already holds them.
#define PL_MOVE_MAX 8
struct PlMove { int row[PL_MOVE_MAX], pos[PL_MOVE_MAX], from[PL_MOVE_MAX], to[PL_MOVE_MAX]; int cnt; };

// one unit's pair lists (a workgroup of PG_UNIT threads, unit u)
template <int DMAX>
__device__ __forceinline__ void plist_unit(const int* __restrict__ nbr, int n, int dpad, int sp, int P,
                                           int thin, u32* __restrict__ list, int* __restrict__ poff, int u,
                                           const PlMove& mv)
{
  __shared__ u64 wtot[2][PG_UNIT / 64];
  const int t = threadIdx.x, r = u * PG_UNIT + t, lane = t & 63, wave = t >> 6;
  // the row's table entries, 16 bytes a load (dpad is a multiple of 4), every
  // thread loading (a row past n reads the last row's): a load under a lane
  // mask would make the compiler wait for each one before the next
  int id[DMAX];
  const int4* src = (const int4*)(nbr + (int64_t)(r < n ? r : n - 1) * dpad);
#pragma unroll
  for (int j4 = 0; j4 < DMAX / 4; j4++) {
    int4 v = make_int4(-1, -1, -1, -1);
    if (4 * j4 < dpad) v = src[j4];                 // uniform
    id[4 * j4] = v.x; id[4 * j4 + 1] = v.y; id[4 * j4 + 2] = v.z; id[4 * j4 + 3] = v.w;
  }
#pragma unroll
  for (int j = 0; j < DMAX; j++)
    if (r >= n || j > dpad) id[j] = -1;
    else if (j == dpad) id[j] = r;
  for (int e = 0; e < mv.cnt; e++)
    if (r == mv.row[e]) {
#pragma unroll
      for (int j = 0; j < DMAX; j++)
        if (j == mv.pos[e] && id[j] == mv.from[e]) id[j] = mv.to[e];
    }
  // part of an id: floor(id P / n), the number of cuts ceil(p n / P) (0 < p < P) at or below it
  int cut[PG_MAXP - 1];
#pragma unroll
  for (int p = 1; p < PG_MAXP; p++) cut[p - 1] = p < P ? (int)(((int64_t)p * n + P - 1) / P) : INT_MAX;
  auto part = [&](int v) {
    int q = 0;
#pragma unroll
    for (int p = 0; p < PG_MAXP - 1; p++) q += v >= cut[p] ? 1 : 0;
    return q;
  };
  // drop repeats (an id equal to an earlier one), count the rest per part
#pragma unroll
  for (int j = 1; j < DMAX; j++) {
    bool dup = false;
#pragma unroll
    for (int k = 0; k < j; k++) dup = dup || id[k] == id[j];
    if (dup) id[j] = -1;
  }
  // per part, how many of the row's ids are thin: its own (once), and the first
  // `thin` neighbours in the order of the parts
  u64 all = 0, own = 0;                             // four 16-bit counts each (a unit holds < 65536 pairs of a part)
#pragma unroll
  for (int j = 0; j < DMAX; j++)
    if (id[j] >= 0) {
      const u64 one = 1ULL << (16 * part(id[j]));
      if (id[j] == r) own += one; else all += one;
    }
  u64 run[2] = {own, all};
  int left = thin;
#pragma unroll
  for (int p = 0; p < PG_MAXP; p++) {
    const int k = min((int)((all >> (16 * p)) & 0xffff), left);
    left -= k;
    run[0] += (u64)k << (16 * p);
    run[1] -= (u64)k << (16 * p);
  }
  const u64 quota = run[0] - own;
  // inclusive scans over the unit's rows: within the wave, then the waves before
  u64 inc[2] = {run[0], run[1]}, tot[2] = {0, 0};
#pragma unroll
  for (int c = 0; c < 2; c++) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const u64 v = __shfl_up(inc[c], o, 64);
      if (lane >= o) inc[c] += v;
    }
    if (lane == 63) wtot[c][wave] = inc[c];
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < 2; c++)
    for (int i = 0; i < PG_UNIT / 64; i++) {
      const u64 v = wtot[c][i];
      if (i < wave) inc[c] += v;
      tot[c] += v;
    }
  __syncthreads();                                  // wtot is free for the next unit
  u32* ul = list + (int64_t)u * PG_UNIT * sp;
  int pos[PG_MAXP][2], base = 0;
#pragma unroll
  for (int p = 0; p < PG_MAXP; p++)
#pragma unroll
    for (int c = 0; c < 2; c++) {
      pos[p][c] = base + (int)((inc[c] >> (16 * p)) & 0xffff) - (int)((run[c] >> (16 * p)) & 0xffff);
      if (t % (PG_UNIT / PG_SUB) == 0 && p < P)
        poff[u * PG_OFF + (2 * p + c) * PG_SUB + t / (PG_UNIT / PG_SUB)] = pos[p][c];
      base += p < P ? (int)((tot[c] >> (16 * p)) & 0xffff) : 0;
    }
  if (t == 0) poff[u * PG_OFF + 2 * P * PG_SUB] = base;
  int need[PG_MAXP];                                // thin neighbours still to place
#pragma unroll
  for (int p = 0; p < PG_MAXP; p++) need[p] = (int)((quota >> (16 * p)) & 0xffff);
#pragma unroll
  for (int j = 0; j < DMAX; j++)
    if (id[j] >= 0) {
      const int q = part(id[j]);
      const bool mine = id[j] == r;
      int at = 0;
#pragma unroll
      for (int p = 0; p < PG_MAXP; p++)
        if (p == q) {
          const bool th = mine || need[p] > 0;
          at = th ? pos[p][0]++ : pos[p][1]++;
          need[p] -= th && !mine ? 1 : 0;
        }
      ul[at] = ((u32)t << 22) | (u32)id[j];
    }
}

// every unit (workgroup u builds unit u)
template <int DMAX>
__global__ __launch_bounds__(PG_UNIT) void k_plist(const int* __restrict__ nbr, int n, int dpad, int sp, int P,
                                                   int thin, u32* __restrict__ list, int* __restrict__ poff)
{
  PlMove none;
  none.cnt = 0;
  plist_unit<DMAX>(nbr, n, dpad, sp, P, thin, list, poff, blockIdx.x, none);
}

// Entries at positions the host found (a 2-opt move, checked with k_swap's
// rule on the host's copy of the adjacency, or the entries an upload changed):
// workgroup 0 stores the mv.cnt entries into the adjacency and the tables;
// workgroup i < units.cnt rebuilds the pair lists of unit units.u[i],
// applying the entries to its rows as it reads them.  With mv.cnt = 0 it only
// rebuilds the units.
struct PlUnits { int u[PL_MOVE_MAX]; int cnt; };
struct PlArgs { const int* nbr; int n, dpad, sp, P, thin; u32* list; int* poff; };

template <int DMAX>
__global__ __launch_bounds__(PG_UNIT) void k_swap_at(int* adj, int degree, SwapTables tb, PlMove mv, PlUnits units,
                                                     PlArgs pl)
{
  if (blockIdx.x == 0 && (int)threadIdx.x < mv.cnt) {
    const int e = threadIdx.x;
    adj[(int64_t)mv.row[e] * degree + mv.pos[e]] = mv.to[e];
    const int64_t k = (int64_t)mv.row[e] * tb.tdp + mv.pos[e];
    if (tb.t16 && tb.t16[k] == (unsigned short)mv.from[e]) tb.t16[k] = (unsigned short)mv.to[e];
    if (tb.t32 && tb.t32[k] == mv.from[e]) tb.t32[k] = mv.to[e];
  }
  if ((int)blockIdx.x < units.cnt)
    plist_unit<DMAX>(pl.nbr, pl.n, pl.dpad, pl.sp, pl.P, pl.thin, pl.list, pl.poff, units.u[blockIdx.x], mv);
}

typedef u32 u32x4v __attribute__((ext_vector_type(4)));
typedef u32 u32x2v __attribute__((ext_vector_type(2)));

// Bits (i, j) of a 64 x 64 bit block swapped, for the block's word w and w + 1:
// before, x[g] of lane l holds row 8 g + l / 8 of the word pair l % 8; after, it
// holds column 8 g + l / 8 of the pair's words as 64 bits of rows.  Six
// exchanges of an index bit with a bit position: row bits 5, 4 and 3 lie in g
// (registers: a renaming and byte permutes), bits 2, 1 and 0 in lane bits 5, 4
// and 3.
__device__ __forceinline__ void swap_bits(u32& p, u32& q, u32 m, int sh)   // q's bits under m with p's sh above
{
  const u32 a = (p & m) | ((q & m) << sh), b = ((p >> sh) & m) | (q & ~m);
  p = a; q = b;
}
__device__ __forceinline__ void transpose64(u32 (&lo)[8], u32 (&hi)[8], int lane)
{
#pragma unroll
  for (int g = 0; g < 4; g++) { const u32 t = hi[g]; hi[g] = lo[g + 4]; lo[g + 4] = t; }
  auto perm2 = [](u32& p, u32& q, u32 s0, u32 s1) {
    const u32 a = __builtin_amdgcn_perm(q, p, s0), b = __builtin_amdgcn_perm(q, p, s1);
    p = a; q = b;
  };
#pragma unroll
  for (int g = 0; g < 8; g++)
    if (!(g & 2)) {
      perm2(lo[g], lo[g + 2], 0x05040100u, 0x07060302u);
      perm2(hi[g], hi[g + 2], 0x05040100u, 0x07060302u);
    }
#pragma unroll
  for (int g = 0; g < 8; g += 2) {
    perm2(lo[g], lo[g + 1], 0x06020400u, 0x07030501u);
    perm2(hi[g], hi[g + 1], 0x06020400u, 0x07030501u);
  }
  // a pair of registers: the swap brings both rows of an exchange into one
  // lane, and back
  auto lanes32 = [](u32& p, u32& q) {
    auto r = __builtin_amdgcn_permlane32_swap(p, q, false, false);
    p = r[0]; q = r[1];
  };
  auto lanes16 = [](u32& p, u32& q) {
    auto r = __builtin_amdgcn_permlane16_swap(p, q, false, false);
    p = r[0]; q = r[1];
  };
#pragma unroll
  for (int g = 0; g < 8; g++) {
    lanes32(lo[g], hi[g]); swap_bits(lo[g], hi[g], 0x0f0f0f0fu, 4); lanes32(lo[g], hi[g]);
    lanes16(lo[g], hi[g]); swap_bits(lo[g], hi[g], 0x33333333u, 2); lanes16(lo[g], hi[g]);
  }
  const bool odd = (lane & 8) != 0;
  const u32 keep = odd ? 0xaaaaaaaau : 0x55555555u, rot = odd ? 1u : 31u;
  auto lanes8 = [&](u32& p) {                          // lane ^ 8: a rotation by 8 within 16 lanes
    const u32 y = (u32)__builtin_amdgcn_update_dpp(0, (int)p, 0x128, 0xf, 0xf, false);
    p = (p & keep) | (__builtin_amdgcn_alignbit(y, y, rot) & ~keep);
  };
#pragma unroll
  for (int g = 0; g < 8; g++) { lanes8(lo[g]); lanes8(hi[g]); }
}

// the stop test of k_level at this level
__device__ __forceinline__ bool task_stops(const LevelTask& T, int level, int ring)
{
  const u64 c1 = T.cnt[(int64_t)((level - 1) % ring) * T.cstride];
  return c1 == (u64)T.n * (u64)T.l || (level >= 2 && c1 == T.cnt[(int64_t)((level - 2) % ring) * T.cstride]);
}

// A workgroup barrier that orders LDS alone: __syncthreads also waits for the
// global stores, and k_pgather's rows, which nothing in the launch reads, may
// drain while the next unit gathers.
__device__ __forceinline__ void lds_barrier()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A level's rows are streamed past the caches (nt) unless both levels' rows
// fit the 256 MB last-level cache, from which the next level then gathers
// (n = 30002, d = 16: an evaluation 281 -> 247 us; n = 65536: 952 streamed, 1026 not)
template <bool NT>
__device__ __forceinline__ void row_store(u64v2 o, u64v2* p)
{
  if (NT) __builtin_nontemporal_store(o, p);
  else *p = o;
}

// Persistent: workgroup b runs on XCD b % 8 and takes every (gridDim.x / 8)-th
// unit of its XCD's contiguous range of units (a unit: PG_UNIT rows of one
// task), so the XCD's workgroups sweep that range together; any grid that is a
// multiple of 8 works.  The units of the last round, when they do not fill it,
// are cut into pieces of their rows (2^cut of them) dealt over the workgroups.
// The gathers are buffer loads bounded by the slab (out-of-range offsets read
// zero).  LS: listing; NT: rows streamed past the caches; FOLD: folds where the
// table is symmetric (128 registers, four more spilled to 20 bytes a lane; the
// others, for launches that never fold, 111 without a spill: general_s n = 100000,
// d = 6, s = 2 3190 -> 3084 us a call).
template <bool LS, bool NT, bool FOLD>
__global__ __launch_bounds__(PG_WG) void k_pgather(const LevelTask* __restrict__ tasks, int level, int ring,
                                                   int mode, LvList lst, PgArgs a)
{
  __shared__ u64x2 acc[PG_UNIT * 8];                  // row r of the unit at [8 r, 8 r + 8)
  __shared__ u64 s_pop[PG_WG / 64];
  __shared__ int s_off[PG_OFF], s_next;
  __shared__ int2 s_chunk[PG_UNIT * 64 / PG_CH + 2 * PG_MAXP];   // chunks of a unit (at most 64 pairs a row, rounded up per group)
  const int x = blockIdx.x % ODP_NXCD, wi = blockIdx.x / ODP_NXCD, nwx = gridDim.x / ODP_NXCD;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane_ = tid & 63, lane = lane_;
  const int nw = PG_WG / 64;
  static_assert(PG_UNIT / (PG_WG / 64) == 64, "a wave stores and transposes 64 rows of a unit");
  const bool count = (mode & LV_COUNT) != 0, store = (mode & LV_STORE) != 0;
  const int w = 2 * (lane & 7);                       // the lane's two words of a row
  const bool fold = FOLD && __builtin_amdgcn_readfirstlane(*a.asym) == 0;
  if (fold) {
    // a unit stands for two blocks, so all run until none has to
    bool run = false;
    for (int t = lane; t < a.ntasks; t += 64) {
      const LevelTask& T = tasks[t];
      const bool stop = *T.done || task_stops(T, level, ring);
      run = run || !stop;
      if (blockIdx.x == 0 && wave == 0) {
        if (stop) *T.done = 1;
        if (count) T.cnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
      }
    }
    if (!__any(run)) return;                          // the same in every wave of the launch
  }
  const int T2 = a.ntasks, hs = (T2 + (T2 & 1)) / 2;  // folded: blocks of rows a block runs in the rounds
  const int main_n = fold ? T2 * hs : a.ntasks * a.upt, extra_n = fold && !(T2 & 1) ? T2 / 2 : 0;
  const int u_lo = (int)((int64_t)main_n * x / ODP_NXCD), u_hi = (int)((int64_t)main_n * (x + 1) / ODP_NXCD);
  const int e_lo = extra_n * x / ODP_NXCD, e_hi = extra_n * (x + 1) / ODP_NXCD;
  const int rounds = (u_hi - u_lo) / nwx, rest = (u_hi - u_lo) - rounds * nwx;
  const int cut = fold ? a.cut_fold : a.cut_full, pieces = (rest + e_hi - e_lo) << cut;
  for (int it = 0;; it++) {                           // uniform
    int u, s0 = 0, s1 = PG_SUB;                       // the unit and its piece [s0, s1) in PG_SUB-ths
    if (it < rounds) {
      u = u_lo + it * nwx + wi;
    } else {
      const int p = (it - rounds) * nwx + wi, k = p >> cut;
      if (p >= pieces) break;
      u = k < rest ? u_lo + rounds * nwx + k : main_n + e_lo + (k - rest);
      s0 = (p & ((1 << cut) - 1)) * (PG_SUB >> cut);
      s1 = s0 + (PG_SUB >> cut);
    }
    int t, ur;
    if (!fold) { t = u / a.upt; ur = u - t * a.upt; }
    else if (u < main_n) { t = u / hs; ur = t + (u - t * hs); if (ur >= T2) ur -= T2; }
    else { t = u - main_n; ur = t + T2 / 2; }
    const LevelTask& T = tasks[t];
    if (!fold) {
      if (*T.done) continue;
      if (task_stops(T, level, ring)) {
        if (tid == 0) *T.done = 1;
        continue;
      }
      if (count && ur == 0 && tid == 0) T.cnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
    }
    const bool mirror = fold && ur != t;
    const u64* __restrict__ cur = (level & 1) ? T.buf1 : T.buf0;
    u64* __restrict__ nxt = (level & 1) ? T.buf0 : T.buf1;
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc((void*)cur, 0, a.n * 128, 0x00020000);
    const u64 f0 = full_word(T.l, w), f1 = full_word(T.l, w + 1);
    for (int i = s0 * 128 * 8 + tid; i < s1 * 128 * 8; i += PG_WG) { acc[i].x = 0; acc[i].y = 0; }
    const u32* __restrict__ ul = a.list + (int64_t)ur * PG_UNIT * a.sp;
    const int* po = a.poff + ur * PG_OFF;
    // the parts in order; the waves take the chunks of PG_CH pairs of all parts
    // from a counter, two chunks ahead (dealt in turn, wave 0, which the SIMD
    // prefers, waited 11 us of a unit's 57 for the others at the barrier: a folded
    // level 478 -> 459 us).  A chunk's PG_SLOTS gathers (eight rows each) are in
    // flight while the wave ORs in the previous chunk's rows: a slot's next gather is issued
    // as soon as its rows are ORed in, and a chunk's pairs are loaded a chunk
    // ahead.  (Waiting slot by slot instead of once per chunk was measured
    // slower.)  The in-flight rows live in registers: PG_SLOTS sets how many.
    const u32 SENT = 0xffffffffu;
    // The chunks of the piece, part after part, listed in LDS (a chunk's pairs
    // [first, end)); no table read from memory in the chunk loop, which would
    // make the wave wait for the gathers in flight.  The XCD's workgroups take
    // its units in rounds; every other round sweeps the parts backwards, so it
    // starts with the part the round before ended with, whose rows are still in
    // L2.
    if (tid < PG_OFF) s_off[tid] = po[tid];               // (entries past 2 P * PG_SUB are not used)
    if (tid == 0) s_next = 3 * nw;
    lds_barrier();
    int nch = 0;
    for (int pp = 0; pp < 2 * a.P; pp++) {                // uniform
      const int p = it & 1 ? 2 * a.P - 1 - pp : pp;
      if ((p & 1) && (mode & LV_THIN)) continue;
      const int lo = __builtin_amdgcn_readfirstlane(s_off[p * PG_SUB + s0]);
      const int hi = __builtin_amdgcn_readfirstlane(s_off[p * PG_SUB + s1]);
      const int nc = (int)((u32)(hi - lo + PG_CH - 1) / PG_CH);
      for (int k = tid; k < nc; k += PG_WG) {
        s_chunk[nch + k].x = lo + k * PG_CH;
        s_chunk[nch + k].y = min(lo + (k + 1) * PG_CH, hi);
      }
      nch += nc;
    }
    lds_barrier();                                      // acc is clear, the chunks are listed
    // a chunk's pairs, 64 per register (every lane loads: an idle one the unit's
    // first entry).  Lane group g (eight lanes, one row) takes the chunk's pairs
    // [g PG_SLOTS, (g + 1) PG_SLOTS), one per slot: a row's pairs of a part are
    // consecutive in the list, so the eight groups of a slot meet eight
    // different rows and their ORs no two lanes' same LDS word.  Register h,
    // lane l holds the pair of slot 8 h + l / 8, group l % 8.
    struct Pairs { u32 v[PG_NL]; };
    auto pairs = [&](int k) -> Pairs {
      Pairs r;
      // past the last chunk (a piece may have none, and s_chunk[0] is then unwritten): no pair
      const int2 c = s_chunk[k < nch ? k : 0];
      const int cc = k < nch ? c.x : 0, ce = k < nch ? c.y : 0;
#pragma unroll
      for (int h = 0; h < PG_NL; h++) {
        const int q = 8 * h + (lane >> 3);
        const int i = cc + (lane & 7) * PG_SLOTS + q;
        const bool ok = q < PG_SLOTS && i < ce;
        const u32 v = ul[ok ? i : 0];
        r.v[h] = ok ? v : SENT;
      }
      return r;
    };
    u64x2 gv[PG_SLOTS];
    int lr[PG_SLOTS];
    // Every lane loads (a pair-less lane past the slab's end, which reads zero):
    // loads under a lane mask would make the compiler wait for all of them.
    auto issue = [&](const Pairs& chunk, int q) {
      const u32 e = (u32)__shfl((int)chunk.v[q >> 3], (q & 7) * 8 + (lane >> 3), 64);
      lr[q] = e == SENT ? -1 : (int)(e >> 22);
      const u32 off = e == SENT ? 0xfffffff0u : (e & 0x3fffff) * 128u + w * 8u;
      const u32x4v v = __builtin_amdgcn_raw_buffer_load_b128(src, (int)off, 0, 0);
      gv[q].x = ((u64)v.y << 32) | v.x; gv[q].y = ((u64)v.w << 32) | v.z;
    };
    const Pairs first = pairs(wave);
    Pairs next = pairs(wave + nw);
#pragma unroll
    for (int q = 0; q < PG_SLOTS; q++) issue(first, q);
    int k0 = wave, k1 = wave + nw, k2 = wave + 2 * nw;    // this chunk, the next (its pairs loaded) and the one after
    while (k0 < nch) {                                    // wave-uniform: this chunk's gathers are in flight
      const Pairs after = pairs(k2);
      int k3 = 0;
      if (lane == 0) k3 = atomicAdd(&s_next, 1);
      // Rows are 128 bytes apart: a row's eight lanes meet 16 of the 64 banks
      // with the first word of their pieces, the other 16 of the row's half of
      // the banks with the second.  A row with bit 1 set ORs its second word
      // first, so the rows of an instruction spread over four classes of 16
      // banks (row mod 4) instead of two.
#pragma unroll
      for (int q = 0; q < PG_SLOTS; q++) {
        if (lr[q] >= 0) {
          u64* d = (u64*)&acc[lr[q] * 8 + (w >> 1)];
          const int sw = (lr[q] >> 1) & 1;
          const u64 f = sw ? gv[q].y : gv[q].x, g = sw ? gv[q].x : gv[q].y;
          if (f) atomicOr(d + sw, f);
          if (g) atomicOr(d + (sw ^ 1), g);
        }
        issue(next, q);                                     // all SENT past the last chunk
      }
      next = after;
      k0 = k1; k1 = k2; k2 = __builtin_amdgcn_readfirstlane(k3);
    }
    lds_barrier();
    // the unit's rows: written, counted, listed; wave w takes rows [64 w, 64 w + 64)
    u32 pop = 0;                                    // at most 64 rows of 1024 bits a wave
    // the lane's addresses of this part are computed here: hoisted out of the
    // unit loop they would take the registers of the gathers in flight
    int lane = lane_;
    asm volatile("" : "+v"(lane));
    const int w = 2 * (lane & 7);
    const bool mine = (wave >> 1) >= s0 && (wave >> 1) < s1;   // two waves' rows are a piece
    u32 lo0[8], hi0[8], lo1[8], hi1[8];
    if (mine) {
#pragma unroll
      for (int g = 0; g < 8; g++) {
        const int lr = wave * 64 + g * 8 + (lane >> 3), r = ur * PG_UNIT + lr;
        const bool valid = r < a.n;
        const u64x2 v = acc[lr * 8 + (w >> 1)];
        lo0[g] = (u32)v.x; hi0[g] = (u32)(v.x >> 32); lo1[g] = (u32)v.y; hi1[g] = (u32)(v.y >> 32);
        if (valid) {
          if (store) {
            u64v2 o; o.x = v.x; o.y = v.y;
            row_store<NT>(o, (u64v2*)(nxt + (int64_t)r * 16 + w));
          }
          pop += (u32)(__popcll(v.x) + __popcll(v.y));
        }
        if (LS) list_append<true>(lst, valid && !(v.x == f0 && v.y == f1), ((u64)t << 48) | ((u64)r << 24) | (u64)w, v.x, v.y);
      }
    }
    if (count) {
      const u32 sum = wave_sum_dpp(pop);
      if (lane == 0) s_pop[wave] = sum;
    }
    lds_barrier();                                  // acc is read, s_pop written
    if (count && tid == 0) {
      u64 sum = 0;
      for (int i = 0; i < nw; i++) sum += s_pop[i];
      if (sum) {
        atomicAdd(&T.cnt[(int64_t)(level % ring) * T.cstride], sum);
        if (mirror) atomicAdd(&tasks[ur].cnt[(int64_t)(level % ring) * T.cstride], sum);
      }
    }
    if (mirror && store) {                            // uniform
      // The mirror's row c (column c of this unit) holds wave j's 64 rows as its
      // word j, at position j ^ swz(c) of the row in LDS: the 64 lanes of a store
      // have one j and rows that differ in bits 0-2 and 7-9, and bit 0 and swz
      // spread them over all banks.
      auto swz = [](int c) { return ((c >> 1) & 3) | (((c >> 7) & 3) << 2); };
      if (mine) {
        transpose64(lo0, hi0, lane);
        transpose64(lo1, hi1, lane);
        u64* words = (u64*)acc;
#pragma unroll
        for (int g = 0; g < 8; g++) {
          const int c = 64 * w + 8 * g + (lane >> 3);
          words[c * 16 + (wave ^ swz(c))] = ((u64)hi0[g] << 32) | lo0[g];
          words[(c + 64) * 16 + (wave ^ swz(c + 64))] = ((u64)hi1[g] << 32) | lo1[g];
        }
      }
      lds_barrier();
      u64* __restrict__ mnxt = (level & 1) ? tasks[ur].buf0 : tasks[ur].buf1;
      const int kq = lane & 7;                        // the lane's word pair of a row: waves 2 kq, 2 kq + 1
      if (kq >= s0 && kq < s1) {
#pragma unroll
        for (int g = 0; g < 8; g++) {
          const int c = wave * 64 + g * 8 + (lane >> 3), r = t * PG_UNIT + c, f = swz(c);
          const u64x2 v = acc[c * 8 + (kq ^ (f >> 1))];
          u64v2 o;
          o.x = f & 1 ? v.y : v.x; o.y = f & 1 ? v.x : v.y;
          if (r < a.n) row_store<NT>(o, (u64v2*)(mnxt + (int64_t)r * 16 + w));
        }
      }
      lds_barrier();                                // acc is free for the next unit
    }
  }
}

// ---------------------------------------------------------------------------
// The BFS kind (the reference's CPU-only aspl_bfs, aspl.c:166-221, with the
// top-down step of utils.c:1999-2100): one breadth-first search per source
// over the row-neighbour table.  Workgroups are persistent and take sources
// from a counter; each keeps its visited bitmap in LDS (VIS_LDS) or in its own
// slice of device memory, and its two frontier queues (n ids each) in device
// memory.  A level's frontier entries (vertex, table position) are dealt over
// the threads; a test-and-set on the bitmap admits each new vertex once.  Per
// source the distances' sum, the eccentricity and the number reached are
// folded into per-workgroup totals, added into the result once at the end.
struct BfsOut {
  u64 sum;          // sum over the sources of sum_v dist(source, v)
  int ecc;          // largest eccentricity
  int disc;         // a source did not reach every vertex
};

__global__ void k_bfs_clear(BfsOut* out, int* next_src)
{
  if (threadIdx.x == 0) { out->sum = 0; out->ecc = 0; out->disc = 0; *next_src = 0; }
}

template <bool VIS_LDS>
__global__ __launch_bounds__(256) void k_bfs(const int* __restrict__ nbr, int n, int dpad, int nsrc,
                                             int* __restrict__ queues, u32* __restrict__ gvis,
                                             int* __restrict__ next_src, BfsOut* __restrict__ out)
{
  extern __shared__ u32 dyn_vis[];
  __shared__ int s_src, s_cnt;
  const int tid = threadIdx.x, nth = blockDim.x;
  const int words = (n + 31) >> 5;
  u32* vis = VIS_LDS ? dyn_vis : gvis + (size_t)blockIdx.x * words;
  int* fq = queues + (size_t)blockIdx.x * 2 * n;
  int* nq = fq + n;
  u64 tot = 0;
  int ecc_max = 0, disc = 0;
  for (;;) {                                            // uniform: s_src is read after a barrier
    if (tid == 0) s_src = atomicAdd(next_src, 1);
    __syncthreads();
    const int src = __builtin_amdgcn_readfirstlane(s_src);
    if (src >= nsrc) break;
    for (int i = tid; i < words; i += nth) vis[i] = 0;
    __syncthreads();
    if (tid == 0) { vis[src >> 5] = 1u << (src & 31); fq[0] = src; }
    int fcount = 1, level = 0, reached = 1;
    u64 dsum = 0;
    while (fcount > 0) {                                // uniform
      level++;
      if (tid == 0) s_cnt = 0;
      __syncthreads();                                  // the frontier, the bitmap and s_cnt are set
      const int entries = fcount * dpad;
      for (int e = tid; e < entries; e += nth) {
        const int f = e / dpad, j = e - f * dpad;
        const int u = nbr[(size_t)fq[f] * dpad + j];
        const u32 b = 1u << (u & 31);
        if (!(atomicOr(&vis[u >> 5], b) & b)) nq[atomicAdd(&s_cnt, 1)] = u;
      }
      __syncthreads();                                  // every new vertex is queued and counted
      fcount = __builtin_amdgcn_readfirstlane(s_cnt);
      dsum += (u64)level * (u64)fcount;
      reached += fcount;
      int* t = fq; fq = nq; nq = t;
      __syncthreads();                                  // s_cnt is read before it is reset
    }
    tot += dsum;
    ecc_max = max(ecc_max, level - 1);
    if (reached < n) disc = 1;
  }
  if (tid == 0) {
    if (tot) atomicAdd(&out->sum, tot);
    atomicMax(&out->ecc, ecc_max);
    if (disc) atomicOr(&out->disc, 1);
  }
}

// ---------------------------------------------------------------------------
// k_sparse: the count of a level expected to be the last one (LV_SPARSE), from
// the list of chunks the level before it left unsaturated.  A chunk saturated
// at level L-1 keeps its bits at level L, so the count of level L is that of
// L-1 plus, over the listed chunks, the bits their neighbours' words add.  As
// for a count-only k_level launch nothing is written but the counts and the
// done flags.  When a sub-list overflowed its capacity every chunk of every
// running task is visited instead.  Any grid size works.

// the bits row r's 16-byte chunk at word w gains at this level (0 if saturated)
__device__ __forceinline__ int chunk_gain(const LevelTask& T, int level, int r, int w)
{
  const u64* __restrict__ cur = (level & 1) ? T.buf1 : T.buf0;
  const int64_t kwp = T.kwp;
  const u64 f0 = full_word(T.l, w), f1 = full_word(T.l, w + 1);
  const u64x2 x0 = *(const u64x2*)(cur + r * kwp + w);
  if (x0.x == f0 && x0.y == f1) return 0;
  u64x2 x = x0;
  const int* nb = T.nbr + (int64_t)r * T.dpad;
  for (int j = 0; j < T.dpad; j += 4) {            // dpad is a multiple of 4
    const int4 v = *(const int4*)(nb + j);
    const u64x2 a = *(const u64x2*)(cur + (int64_t)v.x * kwp + w);
    const u64x2 b = *(const u64x2*)(cur + (int64_t)v.y * kwp + w);
    const u64x2 c = *(const u64x2*)(cur + (int64_t)v.z * kwp + w);
    const u64x2 d = *(const u64x2*)(cur + (int64_t)v.w * kwp + w);
    x.x |= a.x | b.x | c.x | d.x;
    x.y |= a.y | b.y | c.y | d.y;
    if (x.x == f0 && x.y == f1) break;
  }
  return __popcll(x.x) + __popcll(x.y) - __popcll(x0.x) - __popcll(x0.y);
}

// adds each lane's gain (or, negative, loss) to its task's count of the level: one wave sum and one
// atomic per task among the lanes with a gain (listed chunks next to each
// other in the list can come from several tasks; an atomic per lane on the
// few task counters had serialised, 15 ms for 3 M chunks at n = 20000).
// Called by whole waves.
__device__ __forceinline__ void add_gains(const LevelTask* __restrict__ tasks, int level, int ring,
                                          int t, int gain)
{
  bool left = gain != 0;
  for (u64 m = __ballot(left); m; m = __ballot(left)) {   // wave-uniform
    const int t0 = __shfl(t, __ffsll((long long)m) - 1, 64);
    const bool mine = left && t == t0;
    const u64 s = wave_sum(mine ? (u64)(long long)gain : 0ULL);
    if ((threadIdx.x & 63) == 0) atomicAdd(&tasks[t0].cnt[(int64_t)(level % ring) * tasks[t0].cstride], s);
    left = left && !mine;
  }
}

// A list's sub-lists read as one: lane s holds sub-list s's count (LIST_SUBS is
// the wave size) and the count of the sub-lists before it; entry e is in the
// last sub-list that starts at or below e.
struct ListView {
  u32 excl, total, cap;
  bool over;                                          // a sub-list passed its capacity
  __device__ __forceinline__ ListView(const LvList& lst, int lane)
  {
    static_assert(LIST_SUBS == 64, "one sub-list per lane");
    const u32 cnt = lst.n[lane * LIST_PAD];
    over = __any(cnt > lst.cap);
    u32 inc = cnt;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const u32 v = (u32)__shfl_up((int)inc, o, 64);
      if (lane >= o) inc += v;
    }
    excl = inc - cnt;
    total = (u32)__shfl((int)inc, 63, 64);
    cap = lst.cap;
  }
  // where entry e lies; called by whole waves (the shuffles read all lanes)
  __device__ __forceinline__ u64 at(u32 e) const
  {
    int sub = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1)
      if ((u32)__shfl((int)excl, sub + step, 64) <= e) sub += step;
    return (u64)sub * cap + (e - (u32)__shfl((int)excl, sub, 64));
  }
};

// asym: the list is a folded k_pgather's unless *asym (null: not folded): a listed
// chunk's gain counts for its block and, off the diagonal, for the block of its
// row's sources too, whose mirrored chunks gain the same pairs.
__global__ __launch_bounds__(LEVEL_WG) void k_sparse(const LevelTask* __restrict__ tasks, int ntasks,
                                                     int level, int ring, LvList lst, const u32* asym)
{
  const bool fold = asym && __builtin_amdgcn_readfirstlane(*asym) == 0;
  const u32 tid = blockIdx.x * blockDim.x + threadIdx.x, nth = gridDim.x * blockDim.x;
  const int lane = threadIdx.x & 63;
  // per running task: the count of level L starts from L-1's (slot L was
  // cleared by level L-1), and slot L+1 is cleared for level L+1
  for (u32 t = tid; t < (u32)ntasks; t += nth) {
    const LevelTask& T = tasks[t];
    if (*T.done) continue;
    if (task_stops(T, level, ring)) { *T.done = 1; continue; }
    T.cnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
    atomicAdd(&T.cnt[(int64_t)(level % ring) * T.cstride], T.cnt[(int64_t)((level - 1) % ring) * T.cstride]);
  }
  const u32 wbase = tid & ~63u;                       // the wave's first thread; loops are wave-uniform
  const ListView lv(lst, lane);
  if (!lv.over) {
    // A task that stops at this level gains nothing: it stops because level
    // L-1 reached every pair (nothing listed) or added no bit (no chunk can
    // gain one now), so its listed chunks need no test.
    for (u32 b = wbase; b < lv.total; b += nth) {
      const u32 e = b + lane;
      const u64 k = lv.at(e);
      int t = 0, t2 = 0, gain = 0;
      if (e < lv.total) {
        const u64 v = lst.e[k];
        t = (int)(v >> 48);
        t2 = (int)((v >> 24) & 0xffffff) / PG_UNIT;
        gain = chunk_gain(tasks[t], level, (int)((v >> 24) & 0xffffff), (int)(v & 0xffffff));
      }
      add_gains(tasks, level, ring, t, gain);
      if (fold) add_gains(tasks, level, ring, t2, t2 == t ? 0 : gain);
    }
  } else {
    for (int t = 0; t < ntasks; t++) {
      const LevelTask& T = tasks[t];
      if (*T.done || task_stops(T, level, ring)) continue;
      const int chunks = T.segs << T.lpr_log2;       // 16-byte chunks per row of the block
      const u64 total = (u64)T.n * (u64)chunks;
      for (u64 b = wbase; b < total; b += nth) {
        const u64 i = b + lane;
        int gain = 0;
        if (i < total) gain = chunk_gain(T, level, (int)(i / chunks), 2 * (int)(i % chunks));
        add_gains(tasks, level, ring, t, gain);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Thin levels.  When a level L is expected to leave hardly a pair (the level
// after it the last), most of its gathers find their chunk saturated: at
// n = 65536, d = 16 level 4 meets rows 59 % full, and twelve of a row's sixteen
// neighbours fill 99.6 % of the chunks.  So k_pgather takes those neighbours
// alone (LV_THIN) and lists the chunks left unsaturated with their bits; k_thin
// completes the listed chunks from the rows' other neighbours; and level L + 1 is
// done by k_thin2 from level L - 1's rows, two steps away, for the few chunks
// still unsaturated.  Level L's rows are never written.  The counts are all pairs
// less what the listed chunks still miss.  When the guess is wrong the host
// stores levels L and L + 1 (their counts stand); when a list overflows, both
// kernels leave the counts alone and k_thin2 marks level L + 1 (THIN_FAILED) for the
// host, which runs level L whole.  n = 65536, d = 16: a folded level 4 of 459 us
// and k_sparse's 30 become 310 of k_pgather, 24 of k_thin and 26 of k_thin2.
#define THIN_FAILED (~0ULL)

__device__ __forceinline__ bool chunk_full(const u64x2& x, u64 f0, u64 f1) { return x.x == f0 && x.y == f1; }

// all pairs of every running task, into its count of the level (a slot that is
// zero), from which k_thin and k_thin2 take the missing ones
__device__ __forceinline__ void thin_counts(const LevelTask* __restrict__ tasks, int ntasks, int level, int ring,
                                            u32 tid, u32 nth, bool clear_next)
{
  for (u32 t = tid; t < (u32)ntasks; t += nth) {
    const LevelTask& T = tasks[t];
    if (*T.done) continue;
    if (task_stops(T, level, ring)) { *T.done = 1; continue; }
    if (clear_next) T.cnt[(int64_t)((level + 1) % ring) * T.cstride] = 0;
    atomicAdd(&T.cnt[(int64_t)(level % ring) * T.cstride], (u64)T.n * (u64)T.l);
  }
}

// the listed chunks completed; those still unsaturated counted as missing and
// listed in lst2
__global__ __launch_bounds__(LEVEL_WG) void k_thin(const LevelTask* __restrict__ tasks, int ntasks, int level,
                                                   int ring, LvList lst, LvList lst2, const u32* asym, int cut)
{
  const bool fold = asym && __builtin_amdgcn_readfirstlane(*asym) == 0;
  const u32 tid = blockIdx.x * blockDim.x + threadIdx.x, nth = gridDim.x * blockDim.x;
  const int lane = threadIdx.x & 63;
  const u32 wbase = tid & ~63u;
  const ListView lv(lst, lane);
  if (lv.over) return;                                // uniform
  thin_counts(tasks, ntasks, level, ring, tid, nth, false);
  for (u32 b = wbase; b < lv.total; b += nth) {       // wave-uniform
    const u32 e = b + lane;
    const u64 k = lv.at(e);
    int t = 0, t2 = 0, miss = 0;
    u64 id = 0;
    u64x2 x;
    x.x = x.y = 0;
    bool unsat = false;
    if (e < lv.total) {
      id = lst.e[k];
      x = lst.v[k];
      t = (int)(id >> 48);
      const int r = (int)((id >> 24) & 0xffffff), w = (int)(id & 0xffffff);
      t2 = r / PG_UNIT;
      const LevelTask& T = tasks[t];
      const u64* __restrict__ cur = ((level & 1) ? T.buf1 : T.buf0) + w;
      const u64 f0 = full_word(T.l, w), f1 = full_word(T.l, w + 1);
      const int* nb = T.nbr + (int64_t)r * T.dpad;
      // the row's ids from `cut` on first: the thin pairs are its first ones in
      // the order of the parts.  Sixteen ids at a time, their reads in flight
      // together (one id group after the other took 116 us for 100 k chunks)
      for (int pass = 0; pass < 2 && !chunk_full(x, f0, f1); pass++)
        for (int j = 0; j < T.dpad && !chunk_full(x, f0, f1); j += 16) {
          int4 q[4];
#pragma unroll
          for (int i = 0; i < 4; i++) {
            q[i] = make_int4(r, r, r, r);
            if (j + 4 * i < T.dpad) q[i] = *(const int4*)(nb + j + 4 * i);
          }
          u64x2 o[16];
#pragma unroll
          for (int i = 0; i < 16; i++) {
            const int v = i % 4 == 0 ? q[i / 4].x : i % 4 == 1 ? q[i / 4].y : i % 4 == 2 ? q[i / 4].z : q[i / 4].w;
            o[i].x = o[i].y = 0;
            if ((v >= cut) == (pass == 0) && v != r) o[i] = *(const u64x2*)(cur + (int64_t)v * 16);
          }
#pragma unroll
          for (int i = 0; i < 16; i++) { x.x |= o[i].x; x.y |= o[i].y; }
        }
      miss = __popcll(f0 & ~x.x) + __popcll(f1 & ~x.y);
      unsat = miss != 0;
    }
    add_gains(tasks, level, ring, t, -miss);
    if (fold) add_gains(tasks, level, ring, t2, t2 == t ? 0 : -miss);
    list_append<true>(lst2, unsat, id, x.x, x.y);
  }
}

// level L + 1 (`level`) from level L - 1's rows: a wave per chunk of lst2, its lanes
// over the pairs of a neighbour and a neighbour's neighbour
__global__ __launch_bounds__(LEVEL_WG) void k_thin2(const LevelTask* __restrict__ tasks, int ntasks, int level,
                                                    int ring, LvList lst, LvList lst2, const u32* asym)
{
  const bool fold = asym && __builtin_amdgcn_readfirstlane(*asym) == 0;
  const u32 tid = blockIdx.x * blockDim.x + threadIdx.x, nth = gridDim.x * blockDim.x;
  const int lane = threadIdx.x & 63;
  const ListView la(lst, lane), lv(lst2, lane);
  if (la.over || lv.over) {                           // uniform
    if (tid == 0) tasks[0].cnt[(int64_t)(level % ring) * tasks[0].cstride] = THIN_FAILED;
    return;
  }
  thin_counts(tasks, ntasks, level, ring, tid, nth, true);
  const u32 nwaves = nth >> 6;
  for (u32 e = __builtin_amdgcn_readfirstlane(tid >> 6); e < lv.total; e += nwaves) {
    const u64 k = lv.at(e);                           // the same in every lane
    const u64 id = lst2.e[k];
    const u64x2 x0 = lst2.v[k];
    const int t = (int)(id >> 48), r = (int)((id >> 24) & 0xffffff), w = (int)(id & 0xffffff);
    const LevelTask& T = tasks[t];
    const u64* __restrict__ cur = ((level & 1) ? T.buf0 : T.buf1) + w;   // what level L read
    const int* __restrict__ nbr = T.nbr;
    const int dp = T.dpad, m = dp * (dp + 1);
    u64x2 x = x0;
    for (int i0 = lane; i0 < m; i0 += 64 * 4) {       // four pairs a lane in flight (past the last: the first neighbour's row, which counts anyway)
      int u[4], q[4], v[4];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int i = i0 + 64 * c, j = i / (dp + 1);
        q[c] = i < m ? i - j * (dp + 1) : dp;
        u[c] = nbr[(int64_t)r * dp + (i < m ? j : 0)];
      }
#pragma unroll
      for (int c = 0; c < 4; c++) v[c] = nbr[(int64_t)u[c] * dp + (q[c] == dp ? 0 : q[c])];
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const u64x2 o = *(const u64x2*)(cur + (int64_t)(q[c] == dp ? u[c] : v[c]) * 16);
        x.x |= o.x; x.y |= o.y;
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { x.x |= __shfl_xor(x.x, o, 64); x.y |= __shfl_xor(x.y, o, 64); }
    const int miss = __popcll(full_word(T.l, w) & ~x.x) + __popcll(full_word(T.l, w + 1) & ~x.y);
    const int t2 = r / PG_UNIT;
    if (lane == 0 && miss) {
      atomicAdd(&T.cnt[(int64_t)(level % ring) * T.cstride], 0 - (u64)miss);
      if (fold && t2 != t) atomicAdd(&tasks[t2].cnt[(int64_t)(level % ring) * T.cstride], 0 - (u64)miss);
    }
  }
}

// ---------------------------------------------------------------------------
// k_tile: k levels of a grid graph per launch (temporal tiles)
//
// The table entries of a grid graph join cells at most lmax apart in x and in
// y, so a row's value k levels later depends only on the rows within k * lmax
// cells of it.  A workgroup loads one 16-byte chunk (128 sources, a 2-word
// column block) of a square tile of cells plus a ring of halo cells around it
// (tile + 2 * halo = 64 cells a side) into LDS, runs k <= halo / lmax levels
// there and writes the tile's rows back.  Level i of the launch updates the cells at least
// (i + 1) * lmax inside the ring: those are the cells later levels read, and
// every neighbour they read was updated at level i - 1.  Levels alternate
// between two LDS copies of the region (128 KiB, one barrier per level).
//
// A tile is skipped when it cannot change in this launch and its rows in the
// output buffer are already current: none of its rows changed in the previous
// launch, and none of its or its 8 neighbour tiles' rows changed at the
// previous launch's last level (a row changes at level L only if a row it
// gathers from changed at L-1, so changes spread at most lmax cells per
// level, and halo <= tile).  Counts are k_level's: level L+i's count is
// L-1's plus the gains of the tiles' rows up to level L+i.
#define TILE_RW 64                                // region side: tile + 2 * halo = one wave
#define TILE_SLOTS (TILE_RW * TILE_RW)
// threads of a k_tile workgroup: tables of at most 8 ids keep one copy of the
// region (64 KiB, the next values in registers until a level is read) and two
// workgroups of 512 a CU; wider ones two copies and one workgroup of 1024, since
// their cells' offsets leave no registers for the next values
#define TILE_ONE(DP) ((DP) <= 8)
#define TILE_THREADS(DP) (TILE_ONE(DP) ? 512 : 1024)
#define TILE_KMAX 8
#define TILE_DPMAX 16                             // widest table k_tile takes

struct TileArgs {
  const int* xy2row;     // cell x * height + y -> row
  const short* toff;     // [n][dpad]: entry j of row r as the cell offset dx * TILE_RW + dy (0: r itself)
  int width, height, tiles_x, tiles_y;
  int tile, halo;        // tile side and halo width in cells, tile + 2 * halo = TILE_RW, halo <= tile
  int lmax;              // largest |dx| or |dy| of an entry (>= 1)
  int k;                 // levels of this launch, k * lmax <= halo
  int dpar;              // the launch reads buf1 (1) or buf0 (0) and writes the other
  int fpar;              // parity of the tile flags it writes (it reads the other)
  int first;             // first launch of the evaluation: every tile runs
  int xcd;
};

// cell offsets of the row-neighbour table for k_tile; an entry longer than
// lmax (which the host measured on the adjacency) is an internal error
// One thread per cell.  A cell's offsets are stored in order of their y
// offset: k_tile's lanes are consecutive y of one region column and read
// neighbour j together, and a region slot's LDS banks follow its y (rows are
// TILE_RW slots apart), so lanes whose j-th neighbours share a y offset read
// distinct banks; random order put several lanes on one bank.
__global__ void k_tgeom(const int* __restrict__ nbr, int n, int dpad, const int* __restrict__ row2xy, int lmax,
                        short* __restrict__ toff, int* err)
{
  for (int r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
    const int a = row2xy[r];
    int o[TILE_DPMAX], key[TILE_DPMAX];
#pragma unroll
    for (int j = 0; j < TILE_DPMAX; j++) {
      o[j] = 0;
      key[j] = INT_MAX;                                      // past the width: sorts last
      if (j < dpad) {
        const int b = row2xy[nbr[(int64_t)r * dpad + j]];
        int dx = (b >> 16) - (a >> 16), dy = (b & 0xffff) - (a & 0xffff);
        if (dx > lmax || dx < -lmax || dy > lmax || dy < -lmax) { atomicOr(err, 8); dx = 0; dy = 0; }
        o[j] = dx * TILE_RW + dy;
        key[j] = dy;
      }
    }
    // odd-even transposition sort by y offset (every index fixed: registers only)
#pragma unroll
    for (int pass = 0; pass < TILE_DPMAX; pass++)
#pragma unroll
      for (int j = pass & 1; j + 1 < TILE_DPMAX; j += 2)
        if (key[j] > key[j + 1]) {
          const int tk = key[j]; key[j] = key[j + 1]; key[j + 1] = tk;
          const int to = o[j]; o[j] = o[j + 1]; o[j + 1] = to;
        }
#pragma unroll
    for (int j = 0; j < TILE_DPMAX; j++)
      if (j < dpad) toff[(int64_t)r * dpad + j] = (short)o[j];
  }
}

// the longest |dx| or |dy| of an adjacency entry (ids outside the grid skipped),
// into *lmax (zero before the launch).  Row i is base vertex i, or (s = 4) the
// i-th vertex of the first quadrant.  Bound by the waves' adds to one word: eight
// entries a thread and a look at the word first (131072 entries: 25.6 -> 7.4 us).
__global__ void k_lmax(const int* __restrict__ adj, int rows, int degree, int width, int height, int s, int* lmax)
{
  const int bh = height / 2, n = width * height;
  int m = 0;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < rows * degree; i += gridDim.x * blockDim.x) {
    const int r = i / degree, u = adj[i];
    const int v = s == 4 ? (r / bh) * height + (r % bh) : r;
    if (u >= 0 && u < n) m = max(m, max(abs(u / height - v / height), abs(u % height - v % height)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0 && m > __hip_atomic_load(lmax, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(lmax, m);
}

// k_tile_plan: per (task, tile) unit of the launch: k_level's stop test, the
// count slots of levels L..L+k-1 (tile 0 of a task), and the activity test;
// the active units go to a list that k_tile's workgroups drain.
// tq: [0..1] list lengths by flag parity, [2] queue head, [3..] the list.
__global__ void k_tile_plan(const LevelTask* __restrict__ tasks, int ntasks, int level, int ring, TileArgs g,
                            u32* __restrict__ tq)
{
  const int ntiles = g.tiles_x * g.tiles_y;
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid == 0) { tq[g.fpar ^ 1] = 0; tq[2] = 0; }    // the next launch's list, this launch's queue
  for (int u = gid; u < ntasks * ntiles; u += gridDim.x * blockDim.x) {
    const int t = u / ntiles, tile = u - t * ntiles;
    const LevelTask& T = tasks[t];
    const int64_t cs = T.cstride;
    if (*T.done) continue;
    const u64 c1 = T.cnt[(int64_t)((level - 1) % ring) * cs];
    if (c1 == (u64)T.n * (u64)T.l || (level >= 2 && c1 == T.cnt[(int64_t)((level - 2) % ring) * cs])) {
      if (tile == 0) *T.done = 1;
      continue;
    }
    if (tile == 0) {
      // levels L..L+k-1 start from L-1's count; the next launch's slots are cleared
      for (int i = 0; i < g.k; i++) {
        atomicAdd(&T.cnt[(int64_t)((level + i) % ring) * cs], c1);
        T.cnt[(int64_t)((level + g.k + i) % ring) * cs] = 0;
        T.acnt[(int64_t)((level + g.k + i) % ring) * cs] = 0;
      }
    }
    // tile flags of the task: [parity][changed in the launch, changed at its last level][tile]
    const unsigned char* fr = T.chg0 + (g.fpar ^ 1) * 2 * ntiles;
    unsigned char* fw = T.chg0 + g.fpar * 2 * ntiles;
    const int tx = tile / g.tiles_y, ty = tile - tx * g.tiles_y;
    // the tile and the 8 around it, read together (past the edge: the nearest)
    u32 any = (u32)g.first | fr[tile];
#pragma unroll
    for (int d = 0; d < 9; d++) {
      const int ax = min(max(tx + d / 3 - 1, 0), g.tiles_x - 1), ay = min(max(ty + d % 3 - 1, 0), g.tiles_y - 1);
      any |= fr[ntiles + ax * g.tiles_y + ay];
    }
    const bool active = any != 0;
    if (active) tq[3 + atomicAdd(&tq[g.fpar], 1u)] = (u32)u;
    else { fw[tile] = 0; fw[ntiles + tile] = 0; }
  }
}

// k_tile: persistent workgroups pull units from the list until it is drained.
// While a unit runs its levels, the workgroup already claims the next unit and
// looks up its cells' rows (after levels 0 and 1), so most of the chain of
// dependent global loads a unit starts with overlaps the previous unit's levels.
// Bound by LDS reads (10.8 cycles a 16-byte neighbour read of a wave, conflicts
// included); with two region copies and one workgroup a CU, nothing ran while a
// unit was loaded, written back or waited at a barrier, 16 us a unit against the
// 8 its reads take.  256 x 256 grid, d = 8: 144 -> 122 us a launch, 118 with the
// offsets of cells outside a level's window read from one row and the gains added between lanes.
// (The instance for 8 ids spills five registers, 24 bytes a lane, at the 128 that
// two workgroups a CU leave it; the two-copy one of 99 had none.)

// cell (lx, ly) of the region of a tile: thread tid owns (wave + waves m, lane),
// a wave whole region columns
struct TileUnit {
  int t, tile, tx, ty;
  __device__ TileUnit(u32 u, int ntiles, int tiles_y)
  {
    t = (int)(u / ntiles); tile = (int)(u - (u32)t * ntiles);
    tx = tile / tiles_y; ty = tile - tx * tiles_y;
  }
};

template <int DP>
__global__ __launch_bounds__(TILE_THREADS(DP), 4) void k_tile(const LevelTask* __restrict__ tasks, int level, int ring,
                                                              TileArgs g, u32* __restrict__ tq)
{
  constexpr bool ONE = TILE_ONE(DP);
  constexpr int NW = TILE_THREADS(DP) / 64, PER = TILE_SLOTS / TILE_THREADS(DP);
  __shared__ u64x2 rows[ONE ? 1 : 2][TILE_SLOTS];   // the region's chunks, cell (lx, ly) at lx * TILE_RW + ly
  __shared__ u64 red[NW][TILE_KMAX];                // per wave and level: gains of the tile's rows
  __shared__ u32 claim_s;
  const int ntiles = g.tiles_x * g.tiles_y;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const u32 nunits = tq[g.fpar];
  // rows of the unit's cells (-1: outside the grid) and their chunks
  auto cell_rows = [&](const TileUnit& U, int* rr) {
#pragma unroll
    for (int m = 0; m < PER; m++) {
      const int x = U.tx * g.tile - g.halo + wave + m * NW, y = U.ty * g.tile - g.halo + lane;
      rr[m] = (x >= 0 && x < g.width && y >= 0 && y < g.height) ? g.xy2row[x * g.height + y] : -1;
    }
  };
  auto cell_chunks = [&](const TileUnit& U, const int* rr, u64x2* vv) {
    const LevelTask& T = tasks[U.t];
    const u64* __restrict__ in = g.dpar ? T.buf1 : T.buf0;
#pragma unroll
    for (int m = 0; m < PER; m++) {
      vv[m].x = 0; vv[m].y = 0;
      if (rr[m] >= 0) vv[m] = *(const u64x2*)(in + (int64_t)rr[m] * T.kwp);
    }
  };
  if (tid == 0) claim_s = atomicAdd(&tq[2], 1u);
  __syncthreads();
  const u32 q0 = __builtin_amdgcn_readfirstlane(claim_s);
  if (q0 >= nunits) return;                          // uniform
  u32 u = tq[3 + q0];
  int rid[PER];
  cell_rows(TileUnit(u, ntiles, g.tiles_y), rid);
  for (;;) {
    u32 claim = 0;
    if (tid == 0) claim = atomicAdd(&tq[2], 1u);    // the following unit, published after level 0
    const TileUnit U(u, ntiles, g.tiles_y);
    const LevelTask& T = tasks[U.t];
    const int64_t cs = T.cstride;
    unsigned char* fw = T.chg0 + g.fpar * 2 * ntiles;
    u64* __restrict__ out = g.dpar ? T.buf0 : T.buf1;
    const int64_t kwp = T.kwp;
    u32 off[ONE ? 2 : PER][DP / 2];                  // the cells' offsets (one copy: read again each level, a cell ahead)
    const u64 f0 = full_word(T.l, 0), f1 = full_word(T.l, 1);   // a saturated chunk
    bool nzv = false, usv = false;                   // some cell of the thread's is nonzero / unsaturated
    {
      u64x2 val[PER];
      cell_chunks(U, rid, val);
#pragma unroll
      for (int m = 0; m < PER; m++) {
        rows[0][(wave + m * NW) * TILE_RW + lane] = val[m];
        nzv = nzv || (val[m].x | val[m].y) != 0;
        usv = usv || (rid[m] >= 0 && !(val[m].x == f0 && val[m].y == f1));
      }
    }
    // cell m's offsets; a cell outside the grid or not in [lo, hi) reads row 0's
    // (it is not updated): one line instead of a line every four cells
    auto offsets = [&](int m, u32* w, int lo, int hi) {
      const int lx = wave + m * NW;
      const bool in = rid[m] >= 0 && lx >= lo && lx < hi && lane >= lo && lane < hi;
      const unsigned short* o = (const unsigned short*)g.toff + (int64_t)(in ? rid[m] : 0) * DP;
      if constexpr (DP % 8 == 0) {
#pragma unroll
        for (int j = 0; j < DP / 8; j++) {
          const uint4 v = ((const uint4*)o)[j];
          w[4 * j] = v.x; w[4 * j + 1] = v.y; w[4 * j + 2] = v.z; w[4 * j + 3] = v.w;
        }
      } else {
#pragma unroll
        for (int j = 0; j < DP / 4; j++) { const uint2 v = ((const uint2*)o)[j]; w[2 * j] = v.x; w[2 * j + 1] = v.y; }
      }
    };
    if (!ONE)
#pragma unroll
      for (int m = 0; m < PER; m++) offsets(m, off[ONE ? 0 : m], g.lmax, TILE_RW - g.lmax);
    // a region whose cells are all zero, or all saturated, stays so for the k
    // levels: its tile is written back as loaded without running them (most
    // units of a first launch, and tiles the BFS front has just left)
    const bool any_nz = __syncthreads_or(nzv) != 0;
    const bool live = any_nz && __syncthreads_or(usv) != 0;
    u32 qn = nunits, un = 0;
    int nrid[PER];
#pragma unroll
    for (int m = 0; m < PER; m++) nrid[m] = -1;
    if (!live) {
      if (tid == 0) claim_s = claim;
      __syncthreads();
      qn = __builtin_amdgcn_readfirstlane(claim_s);
      if (qn < nunits) un = tq[3 + qn];
    }
    for (int i = 0; i < (live ? g.k : 0); i++) {
      // level i reads copy i & 1 (level i - 1) and writes the other, or (one
      // copy) writes it once every wave has read it; cells it leaves out are
      // never read again
      const u64x2* src = rows[ONE ? 0 : i & 1];
      u64x2* dst = rows[ONE ? 0 : (i + 1) & 1];
      u64x2 nx[ONE ? PER : 1];
      const int lo = (i + 1) * g.lmax, hi = TILE_RW - lo;
      u32 gain = 0;                                  // at most 8 * 128 bits a thread
      if (ONE) offsets(0, off[0], lo, hi);
#pragma unroll
      for (int m = 0; m < PER; m++) {
        if (ONE && m + 1 < PER) offsets(m + 1, off[ONE ? (m + 1) & 1 : 0], lo, hi);
        const int lx = wave + m * NW, sl = lx * TILE_RW + lane;
        if (rid[m] >= 0 && lx >= lo && lx < hi && lane >= lo && lane < hi) {
          const u64x2 o = src[sl];
          u64x2 x = o;
          // a saturated chunk gains nothing: its neighbours are not read
          if (!(o.x == f0 && o.y == f1)) {
            const u32* w = off[ONE ? m & 1 : m];
#pragma unroll
            for (int j = 0; j < DP / 2; j++) {
              // the window keeps every neighbour inside the region: a cell at least
              // (i + 1) lmax from its edges, and no offset longer than lmax cells
              // (k_tgeom flags longer ones, which end the run)
              const int s0 = sl + (int)(short)(w[j] & 0xffff);
              const int s1 = sl + (int)(short)(w[j] >> 16);
              const u64x2 a = src[s0], c = src[s1];
              x.x |= a.x | c.x;
              x.y |= a.y | c.y;
            }
          }
          if (ONE) nx[ONE ? m : 0] = x;
          else dst[sl] = x;
          if (lx >= g.halo && lx < g.halo + g.tile && lane >= g.halo && lane < g.halo + g.tile)
            gain += (u32)(__popcll(x.x ^ o.x) + __popcll(x.y ^ o.y));   // x holds o: its new bits
        }
      }
      if (ONE) {
        __syncthreads();                             // level i - 1 is read
#pragma unroll
        for (int m = 0; m < PER; m++) {
          const int lx = wave + m * NW;
          if (rid[m] >= 0 && lx >= lo && lx < hi && lane >= lo && lane < hi) dst[lx * TILE_RW + lane] = nx[ONE ? m : 0];
        }
      }
      const u32 wgain = wave_sum_dpp(gain);
      if (lane == 0) red[wave][i] = wgain;
      if (i == 0 && tid == 0) claim_s = claim;
      __syncthreads();                               // level i is in LDS
      // the next unit's loads, one dependent step per level
      if (i == 0) {
        qn = __builtin_amdgcn_readfirstlane(claim_s);
        if (qn < nunits) un = tq[3 + qn];
      } else if (i == 1) {
        if (qn < nunits) cell_rows(TileUnit(un, ntiles, g.tiles_y), nrid);
      }
    }
    if ((!live || g.k < 2) && qn < nunits) cell_rows(TileUnit(un, ntiles, g.tiles_y), nrid);   // not yet
    // the tile's rows, its counts and flags
#pragma unroll
    for (int m = 0; m < PER; m++) {
      const int lx = wave + m * NW;
      if (rid[m] >= 0 && lx >= g.halo && lx < g.halo + g.tile && lane >= g.halo && lane < g.halo + g.tile)
        *(u64x2*)(out + (int64_t)rid[m] * kwp) = rows[live && !ONE ? (g.k & 1) : 0][lx * TILE_RW + lane];
    }
    if (tid < g.k) {
      u64 cum = 0, last = 0;
      for (int i = 0; live && i <= tid; i++)
        for (int w = 0; w < NW; w++) { cum += red[w][i]; if (i == tid) last += red[w][i]; }
      if (cum) atomicAdd(&T.cnt[(int64_t)((level + tid) % ring) * cs], cum);
      if (tid == g.k - 1) {
        fw[U.tile] = cum != 0;
        fw[ntiles + U.tile] = last != 0;
        const int cx = min(g.tile, g.width - U.tx * g.tile), cy = min(g.tile, g.height - U.ty * g.tile);
        atomicAdd(&T.acnt[(int64_t)(level % ring) * cs], (u64)(cx * cy));   // rows processed (timing)
      }
    }
    __syncthreads();                                 // red and the region are free for the next unit
    if (qn >= nunits) break;                         // uniform
    u = un;
#pragma unroll
    for (int m = 0; m < PER; m++) rid[m] = nrid[m];
  }
}

// ---------------------------------------------------------------------------
// direct kernel: the first K levels of a group of column blocks in one launch
//
// Row v of level L holds the sources reachable from v by a walk of at most
// L+1 steps through the row-neighbour table (level 0: v and its neighbours;
// each level ORs in the neighbours' rows).  While those sets are small they
// are cheaper to enumerate than to gather.  One wave per row expands the walk
// tree of v breadth-first: the ids at depth d-1 sit in an LDS list, the wave
// loads their table rows (16 B per load, DIRECT_UNROLL independent loads per
// lane in flight), sets the bits in an LDS bitmap of the group's row and, for
// d < K, appends the ids to the depth-d list.  After each depth the bitmap is
// popcounted per block (the count of level d-1); after depth K the row is
// written to the buffer level K reads.  The sets are exactly those the level
// kernels build, so every count and every word equals k_level0 followed by
// levels 1..K-1.
//
// A launch over every source (ALL) drops the ids its bitmap already holds: the
// walks on from a vertex met before end where its first occurrence's end, so a
// depth's list is the breadth-first frontier (485 instead of 1365 expanded ids
// at d = 4, K = 6), its length the level's count, and only the last depth's
// bitmap is popcounted.  Bound by LDS atomics and the latency of a row's K
// dependent table reads.  n = 49999, d = 4: 332 -> 135 us; n = 100000, d = 8:
// 678 -> 389; n = 65536, d = 16 (4112 of 4368 ids): 170 -> 147.

struct DirectArgs {
  const int* nbr;        // [n][dpad] row-neighbour table
  const unsigned short* nbr16;   // the same with 16-bit ids (n <= 65536), read when ID16
  u64* out;              // block t, row v, word w: out[t * tstride + v * kw + w]
  int64_t tstride;       // words between the slabs of consecutive blocks
  u64* cnt;              // count of block t at level L: cnt[L * cstride + t], L < K
  int cstride;
  int n, dpad, kw, kwl;  // kw: words per block row, a power of two in [2, 128]; kwl = log2(kw)
  int src_lo, nsrc;      // sources of the group: [src_lo, src_lo + nsrc)
  int ntask, words;      // blocks in the group; words = ntask * kw
  int chunks;            // ceil(words / 128): 128-word chunks a wave sweeps per row
  int K;                 // levels computed (2..DIRECT_KMAX)
  int list;              // ints a wave's depth lists take (Evaluator::direct_list)
  unsigned qmul;         // floor(2^32 / q) + 1 for q = 16-byte loads per table row > 1:
                         // idx / q == umulhi(idx, qmul) for idx < 2^32 / q (idx < 2^24, q <= 256 here)
  int pw[8];             // dpad^i
  int nt;                // the rows of level K are streamed past L2 (the next level gathers from other XCDs)
};

#define DIRECT_KMAX 6
#define DIRECT_UNROLL 8
#define DIRECT_UNROLL_BFS 4

// ALL: every id is a source of the group (src_lo == 0, nsrc == n), no range test
template <bool ALL>
__device__ __forceinline__ void direct_set(u32* bm, int id, int src_lo, int nsrc)
{
  const int c = id - src_lo;
  if (ALL || (unsigned)c < (unsigned)nsrc) atomicOr(&bm[c >> 5], 1u << (c & 31));
}

// ID16: the 16-bit table (eight ids per 16-byte load) instead of the 32-bit one
// L16: the depth lists hold 16-bit ids (ALL, n <= 65536): less LDS, more waves
template <bool ALL, bool ID16, bool L16>
__global__ __launch_bounds__(1024) void k_direct(DirectArgs a)
{
  extern __shared__ __attribute__((aligned(16))) u64 dlds[];
  const int nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  u64* bm = dlds + (int64_t)wave * a.words;
  u32* bm32 = (u32*)bm;
  // LDS: nw row bitmaps, nw id lists, then per-lane counts lc[K][chunks][64] of
  // the workgroup (lane l of chunk j holds words 128 j + 2 l, 128 j + 2 l + 1).
  // Depth 0 takes 4 ints of a list and depth d >= 1 dpad^d, so every depth
  // starts 16-byte aligned (dpad is a multiple of 4).
  static_assert(ALL || !L16, "16-bit depth lists");
  typedef typename std::conditional<L16, unsigned short, int>::type lid;
  lid* list = (lid*)((int*)(dlds + (int64_t)nw * a.words) + wave * a.list);
  u32* lc = (u32*)((int*)(dlds + (int64_t)nw * a.words) + nw * a.list);
  const int ncnt = a.K * a.chunks * 64;
  for (int i = threadIdx.x; i < ncnt; i += blockDim.x) lc[i] = 0;
  __syncthreads();
  const int IPL = ID16 ? 8 : 4;                    // ids per 16-byte load
  const int Q = a.dpad / IPL;                      // 16-byte loads per table row
  // Each wave works on its own rows, bitmap and lists: between the phases of a
  // row only the wave's own LDS accesses must be ordered, which LDS guarantees
  // for one wave's instructions, so a wavefront fence (compiler ordering) is
  // enough and the waves of a workgroup never wait for each other.
  for (int v = blockIdx.x * nw + wave; v < a.n; v += gridDim.x * nw) {   // wave-uniform
    for (int w = 2 * lane; w < a.words; w += 128) { u64x2 z; z.x = 0; z.y = 0; *(u64x2*)(bm + w) = z; }
    if (lane == 0) list[0] = (lid)v;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane == 0) direct_set<ALL>(bm32, v, a.src_lo, a.nsrc);
    int off = 0, m_last = 0;                       // start of the depth d-1 list; its ids (ALL, d = K)
    if (ALL) {
      // the bitmap holds every id, so it tells a new id from one met before,
      // whose walks on from here end where its first occurrence's do: the depth
      // lists are breadth-first frontiers, and their entries the level's count
      if (lane == 0) atomicAdd(&lc[v >> 7], 1u);
      int m = 1;
      for (int d = 1; d < a.K; d++) {
        const int jobs = m * Q;
        const lid* from = list + off;
        lid* to = list + off + m;
        u32* lcd = lc + (d - 1) * a.chunks * 64;
        int got = 0;                               // ids appended (uniform)
        for (int j0 = 0; j0 < jobs; j0 += 64 * DIRECT_UNROLL_BFS) {
          uint4 q[DIRECT_UNROLL_BFS];
#pragma unroll
          for (int u = 0; u < DIRECT_UNROLL_BFS; u++) {
            const unsigned idx = j0 + u * 64 + lane;
            if (idx < (unsigned)jobs) {
              const unsigned r = Q == 1 ? idx : __umulhi(idx, a.qmul);
              const int64_t e = (int64_t)from[r] * a.dpad + IPL * (idx - r * Q);
              q[u] = ID16 ? *(const uint4*)(a.nbr16 + e) : *(const uint4*)(a.nbr + e);
            }
          }
#pragma unroll
          for (int u = 0; u < DIRECT_UNROLL_BFS; u++) {
            if (j0 + u * 64 < jobs) {              // uniform
              const bool act = j0 + u * 64 + lane < jobs;
              const u32 w4[4] = {q[u].x, q[u].y, q[u].z, q[u].w};
              int id[ID16 ? 8 : 4];
              u32 old[ID16 ? 8 : 4];
#pragma unroll
              for (int i = 0; i < (ID16 ? 8 : 4); i++) {
                id[i] = ID16 ? (int)(i & 1 ? w4[i >> 1] >> 16 : w4[i >> 1] & 0xffff) : (int)w4[i];
                old[i] = ~0u;
                if (act) old[i] = atomicOr(&bm32[id[i] >> 5], 1u << (id[i] & 31));
              }
#pragma unroll
              for (int i = 0; i < (ID16 ? 8 : 4); i++) {
                const bool fresh = !((old[i] >> (id[i] & 31)) & 1);
                const u64 mask = __ballot(fresh);
                if (fresh) {
                  to[got + __popcll(mask & ((1ULL << lane) - 1))] = (lid)id[i];
                  atomicAdd(&lcd[id[i] >> 7], 1u);
                }
                got += __popcll(mask);
              }
            }
          }
        }
        off += m;
        m = got;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      }
      m_last = m;
    }
    for (int d = ALL ? a.K : 1; d <= a.K; d++) {
      const int m = ALL ? m_last : a.pw[d - 1];    // ids at depth d-1
      const int jobs = m * Q;
      const lid* from = list + off;
      const int step = d == 1 ? 4 : m;             // ints the depth d-1 list takes
      lid* to = list + off + step;                 // the depth-d list follows
      for (int j0 = 0; j0 < jobs; j0 += 64 * DIRECT_UNROLL) {
        uint4 q[DIRECT_UNROLL];
#pragma unroll
        for (int u = 0; u < DIRECT_UNROLL; u++) {
          const unsigned idx = j0 + u * 64 + lane;
          if (idx < (unsigned)jobs) {
            const unsigned r = Q == 1 ? idx : __umulhi(idx, a.qmul);
            const int64_t e = (int64_t)from[r] * a.dpad + IPL * (idx - r * Q);
            q[u] = ID16 ? *(const uint4*)(a.nbr16 + e) : *(const uint4*)(a.nbr + e);
          }
        }
#pragma unroll
        for (int u = 0; u < DIRECT_UNROLL; u++) {
          const int idx = j0 + u * 64 + lane;
          if (idx < jobs) {
            if (ID16) {
              int4 lo, hi;
              lo.x = q[u].x & 0xffff; lo.y = q[u].x >> 16; lo.z = q[u].y & 0xffff; lo.w = q[u].y >> 16;
              hi.x = q[u].z & 0xffff; hi.y = q[u].z >> 16; hi.z = q[u].w & 0xffff; hi.w = q[u].w >> 16;
              direct_set<ALL>(bm32, lo.x, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, lo.y, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, lo.z, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, lo.w, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, hi.x, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, hi.y, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, hi.z, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, hi.w, a.src_lo, a.nsrc);
              if (!ALL && d < a.K) { *(int4*)(to + 8 * idx) = lo; *(int4*)(to + 8 * idx + 4) = hi; }
            } else {
              int4 v;
              v.x = (int)q[u].x; v.y = (int)q[u].y; v.z = (int)q[u].z; v.w = (int)q[u].w;
              direct_set<ALL>(bm32, v.x, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, v.y, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, v.z, a.src_lo, a.nsrc);
              direct_set<ALL>(bm32, v.w, a.src_lo, a.nsrc);
              if (!ALL && d < a.K) *(int4*)(to + 4 * idx) = v;
            }
          }
        }
      }
      off += step;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      // level d-1: popcounts into the lane's counters; after the last depth, the row itself
      u32* lcd = lc + (d - 1) * a.chunks * 64 + lane;
      for (int j = 0; j < a.chunks; j++) {
        const int w = 128 * j + 2 * lane;
        if (w < a.words) {
          const u64x2 x = *(const u64x2*)(bm + w);
          const u32 c = (u32)(__popcll(x.x) + __popcll(x.y));
          if (c) atomicAdd(&lcd[64 * j], c);
          if (d == a.K) {
            u64* dst = a.out + (int64_t)(w >> a.kwl) * a.tstride + (int64_t)v * a.kw + (w & (a.kw - 1));
            if (a.nt) {
              u64v2 o; o.x = x.x; o.y = x.y;
              __builtin_nontemporal_store(o, (u64v2*)dst);
            } else {
              *(u64x2*)dst = x;
            }
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
  }
  __syncthreads();
  // per block: the kw/2 lanes of a chunk that share a block row add up
  const int half = a.kw >> 1;
  for (int e = wave; e < a.K * a.chunks; e += nw) {            // wave-uniform
    const int L = e / a.chunks, j = e - L * a.chunks;
    u64 c = lc[e * 64 + lane];
    if (ALL && L < a.K - 1)                                    // the ids first met at each depth so far
      for (int i = 0; i < L; i++) c += lc[(i * a.chunks + j) * 64 + lane];
    for (int o = 1; o < half; o <<= 1) c += __shfl_xor(c, o, 64);
    const int w = 128 * j + 2 * lane;
    if (w < a.words && (lane & (half - 1)) == 0 && c)
      atomicAdd(&a.cnt[(int64_t)L * a.cstride + (w >> a.kwl)], c);
  }
}

// ---------------------------------------------------------------------------
// resident kernel
//
// One workgroup runs every level of one block of sources with the block's
// bit matrix in LDS: u32[n][WB], a single buffer.  Each thread owns rows
// tid, tid+nth, ... (at most RPT of them) and keeps their next values in
// registers until the whole workgroup has read the level, then writes them
// back, so one buffer of n*WB*4 bytes suffices (two barriers per level).
// Neighbour ids are read as 16-bit row indices, eight per 16-byte load.
// The pulled levels of a large block are bound by LDS reads of random rows: 9 to
// 9.5 cycles a wave's read of 4 or 8 bytes a lane, bank conflicts included (n =
// 30002, d = 7: 34k cycles a level of 3750 reads), so the block is as wide as
// LDS allows.  Small blocks are bound by the chain from one level to the next;
// what lay on it besides the reads: the own row's read and the wait for its ids
// (kept in registers, and fetched a row ahead, across the barrier too), the
// count's trips through LDS shuffles (now adds between lanes, 32 bits), and the
// passes over empty rows of the unrolled loops (now left at the last row).  A
// pulled level of n = 1024, d = 6 takes 2300 cycles of 6000 before; one
// evaluation n = 1024 26.8 -> 24.0 us, n = 5001, d = 10 49.2 -> 41.0,
// n = 30002, d = 7 375 -> 342.

struct ResTask {
  const unsigned short* nbr;   // [n][dp] 16-bit row indices, padded with the row itself
  int n, dp;                   // rows; ids per row (multiple of 8)
  int src0, l;                 // first source row of the block, sources in it (<= 32*wb)
  int s;                       // symmetry factor of the graph
  int graph;                   // index into the per-graph outputs
  int wb;                      // 32-bit words per row of the block: 1, 2, 4 or 8
  int dq;                      // groups of 4 ids a row reads: ceil(table width / 4) <= dp / 4
  int deg;                     // table width (entries a row holds, padding included)
  int walk;                    // levels 0 .. walk - 1 from walks out of the block's sources (0: none)
};

// Levels a block builds from walks out of its l sources instead of pulling
// every row's neighbours: level L (sources within L + 1 hops) adds the walks
// of exactly L + 1 steps, l * deg^(L+1) LDS bit-sets (each decoded prefix of L
// steps reads one table row for its deg last steps), against n * (deg + 1) row
// reads for a pulled level; a level is walked while cost * (L + 1) times its
// walks stay below a pulled level's row reads (cost 1: measured best for the
// 1024-graph batch, 20.2 ms against 20.3 at 2, 20.55 at 4, 20.5 at 0.5).
// Returns the first pulled level (1: level 0 alone, whose l * (deg + 1) walks
// of at most one step always beat reading the table).  A level's prefixes
// (l * deg^L) stay below 2^24 whatever the cost: res_run's FastDiv decodes them.
__host__ __device__ inline int res_walk_levels(int n, int deg, int l, double cost = 1.0)
{
  int K = 1;
  double w = (double)l * deg;                        // walks of one step
  for (int L = 1; L < 8; L++) {
    w *= deg;                                        // walks of L + 1 steps
    if (w * cost * (L + 1) > (double)n * (deg + 1) || w >= 16777216.0 * deg) break;
    K = L + 1;
  }
  return K;
}

struct ResOut {     // per-graph accumulators
  u64 sum;          // sum over blocks of sum_L (n*l - count_L) * s   (the n(n-1) base excluded)
  int diam;         // max over blocks of (terminal level + 1)
  u32 flags;        // bit 0: a block found no new bits before completing (disconnected)
  u32 levels;       // levels run, summed over the graph's blocks (for byte accounting)
  u32 pad;
};

// rows per thread held in registers for each width (at most 32 u32 of next rows)
// rows per thread of a resident block: with 4-word rows, 10 (10240 rows, as
// many as LDS holds: graphs of 8192 < n <= 10208 take 4-word blocks, 23.5 ms
// against 24.6 for the 1024-graph batch)
__host__ __device__ constexpr int res_rpt(int wb) { return wb == 1 ? 16 : wb == 2 ? 16 : wb == 4 ? 10 : 2; }
// rows per thread of the single-graph instances past 16384 rows, for two-word
// blocks (their LDS buffer holds up to 20416 rows) and one-word blocks (up to
// 40832 rows; 62 to 74 registers): instantiations of their own, so that the
// other launches keep their registers
#define RES_RPT_WIDE 20
#define RES_RPT_WIDE1 28
#define RES_RPT_WIDE1B 32
#define RES_RPT_WIDE1C 40

template <int WB> struct RowT { u32 w[WB]; };

template <int WB>
__device__ __forceinline__ RowT<WB> lds_row(const u32* p)
{
  RowT<WB> r;
  if constexpr (WB == 1) {
    r.w[0] = p[0];
  } else if constexpr (WB == 2) {
    const uint2 v = *(const uint2*)p;
    r.w[0] = v.x; r.w[1] = v.y;
  } else {
#pragma unroll
    for (int k = 0; k < WB; k += 4) {
      const uint4 v = *(const uint4*)(p + k);
      r.w[k] = v.x; r.w[k + 1] = v.y; r.w[k + 2] = v.z; r.w[k + 3] = v.w;
    }
  }
  return r;
}

template <int WB>
__device__ __forceinline__ void lds_store(u32* p, const RowT<WB>& r)
{
  if constexpr (WB == 1) {
    p[0] = r.w[0];
  } else if constexpr (WB == 2) {
    *(uint2*)p = make_uint2(r.w[0], r.w[1]);
  } else {
#pragma unroll
    for (int k = 0; k < WB; k += 4) *(uint4*)(p + k) = make_uint4(r.w[k], r.w[k + 1], r.w[k + 2], r.w[k + 3]);
  }
}

template <int WB>
__device__ __forceinline__ void row_bit(RowT<WB>& r, int c, int l)
{
  if ((unsigned)c < (unsigned)l) {
    const int k = c >> 5;
    const u32 bit = 1u << (c & 31);
#pragma unroll
    for (int i = 0; i < WB; i++) r.w[i] |= (i == k) ? bit : 0u;
  }
}

template <int WB>
__device__ __forceinline__ void row_or(RowT<WB>& r, const u32* cur, int v)
{
  const RowT<WB> a = lds_row<WB>(cur + v * WB);
#pragma unroll
  for (int k = 0; k < WB; k++) r.w[k] |= a.w[k];
}

// The two rows a 32-bit word of 16-bit ids names, ORed into r: their LDS byte
// addresses id * 4 WB + base each take one v_mad_u32_u16 (op_sel picks the
// high half), where the compiler's own extract, shift and add took two or
// three instructions -- the pulled levels are bound by VALU and LDS issue.
typedef __attribute__((address_space(3))) const u32 lds_u32_t;
template <int WB>
__device__ __forceinline__ RowT<WB> lds_row_at(u32 addr)
{
  typedef __attribute__((address_space(3))) const u32x2v lds_u32x2_t;
  typedef __attribute__((address_space(3))) const u32x4v lds_u32x4_t;
  RowT<WB> r;
  if constexpr (WB == 1) {
    r.w[0] = *(lds_u32_t*)(uintptr_t)addr;
  } else if constexpr (WB == 2) {
    const u32x2v v = *(lds_u32x2_t*)(uintptr_t)addr;
    r.w[0] = v.x; r.w[1] = v.y;
  } else {
#pragma unroll
    for (int k = 0; k < WB; k += 4) {
      const u32x4v v = *(lds_u32x4_t*)(uintptr_t)(addr + 4u * k);
      r.w[k] = v.x; r.w[k + 1] = v.y; r.w[k + 2] = v.z; r.w[k + 3] = v.w;
    }
  }
  return r;
}

template <int WB>
__device__ __forceinline__ void row_or2(RowT<WB>& r, u32 base, u32 word)
{
  u32 lo, hi;
  asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(lo) : "v"(word), "v"((u32)(4 * WB)), "v"(base));
  asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(hi) : "v"(word), "v"((u32)(4 * WB)), "v"(base));
  const RowT<WB> a = lds_row_at<WB>(lo), b = lds_row_at<WB>(hi);
#pragma unroll
  for (int k = 0; k < WB; k++) r.w[k] |= a.w[k] | b.w[k];
}

// No divergent branch may sit in a loop that contains a barrier.  With an
// `if (lane == 0)` around the queue pop, the compiler structurized the block
// loop per lane: lane 0 left the loop to pop the next block while the other
// lanes re-entered the barrier and re-read the old block id -- a livelock.  So
// every loop-control value is made wave-uniform with readfirstlane, and
// single-lane side effects are done by whole waves with zero contributions
// from the other lanes.
__device__ __forceinline__ u64 uniform_u64(u64 v)
{
  const u32 lo = __builtin_amdgcn_readfirstlane((u32)v);
  const u32 hi = __builtin_amdgcn_readfirstlane((u32)(v >> 32));
  return ((u64)hi << 32) | lo;
}

// part: 16 words a wave each, those past the workgroup's waves zero
__device__ __forceinline__ u32 block_total(u32 v, u32* part, int wave)
{
  part[wave] = wave_sum_dpp(v);      // every lane writes the same value
  __syncthreads();
  u32 s = 0;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint4 q = ((const uint4*)part)[i];
    s += q.x + q.y + q.z + q.w;
  }
  return (u32)__builtin_amdgcn_readfirstlane((int)s);
}

// v again, as far as the compiler can tell a new value: what is computed from
// it is not kept in registers across the loop around it
__device__ __forceinline__ int again(int v)
{
  asm volatile("" : "+s"(v));
  return v;
}

// Division of numbers below 2^24 by one divisor: the float quotient is at most
// one off.
struct FastDiv {
  u32 d;
  float inv;
  __device__ __forceinline__ explicit FastDiv(u32 v) : d(v), inv(1.0f / (float)v) {}
  __device__ __forceinline__ u32 div(u32 x, u32& rem) const
  {
    u32 q = (u32)((float)x * inv);
    int r = (int)(x - q * d);
    if (r < 0) { q--; r += (int)d; }
    else if (r >= (int)d) { q++; r -= (int)d; }
    rem = (u32)r;
    return q;
  }
};

// All levels of one block of T.l <= 32*WB sources; returns the block's totals
// (the same value in every thread).
// The counts fit 32 bits: a block is at most 160 KiB of them.
template <int WB, bool STOP = false, bool WALK = true, int RPT = res_rpt(WB)>
__device__ __forceinline__ ResOut res_run(const ResTask& T, u32* cur, u32 (*s_part)[16],
                                          int tid, int nth, int wave)
{
  const u32 target = (u32)T.n * (u32)T.l;
  const u32 cbase = (u32)(uintptr_t)(__attribute__((address_space(3))) u32*)cur;   // cur's LDS byte address
  RowT<WB> full;
#pragma unroll
  for (int k = 0; k < WB; k++) {
    const int v = T.l - 32 * k;
    full.w[k] = v >= 32 ? ~0u : (v <= 0 ? 0u : ((1u << v) - 1u));
  }
  // level 0 straight from the identity: row r holds r and its neighbours
  u32 pop = 0;
  if (WALK && T.walk >= 1) {
    // from the sources' side: clear every row, then each source sets its bit
    // in its own row and in its neighbours' rows (the table is symmetric);
    // whoever finds a bit clear counts it
    const int words = T.n * WB;
    for (int w = 4 * tid; w < (words & ~3); w += 4 * nth) *(uint4*)(cur + w) = make_uint4(0, 0, 0, 0);
    if (tid < (words & 3)) cur[(words & ~3) + tid] = 0;
    __syncthreads();
    const FastDiv per((u32)T.deg + 1);
    for (u32 it = (u32)tid; it < (u32)T.l * per.d; it += (u32)nth) {
      u32 j;
      const u32 c0 = per.div(it, j);
      const int src = T.src0 + (int)c0;
      const int v = j == (u32)T.deg ? src : (int)T.nbr[src * T.dp + (int)j];
      const u32 b = 1u << (c0 & 31);
      pop += (atomicOr(&cur[v * WB + (int)(c0 >> 5)], b) & b) == 0;
    }
  } else
  for (int r = tid; r < T.n; r += nth) {
    RowT<WB> row;
#pragma unroll
    for (int k = 0; k < WB; k++) row.w[k] = 0;
    row_bit<WB>(row, r - T.src0, T.l);
    // 8 ids per 16-byte load, then 4 more when the table width leaves them
    // (the padding past the width is not read)
    const uint4* ids = (const uint4*)T.nbr;     // uniform base, 32-bit offsets
    const u32 off = (u32)r * (u32)(T.dp >> 3);
    for (int j = 0; j < (T.dq >> 1); j++) {
      const uint4 v = ids[off + j];
      row_bit<WB>(row, (int)(v.x & 0xffff) - T.src0, T.l); row_bit<WB>(row, (int)(v.x >> 16) - T.src0, T.l);
      row_bit<WB>(row, (int)(v.y & 0xffff) - T.src0, T.l); row_bit<WB>(row, (int)(v.y >> 16) - T.src0, T.l);
      row_bit<WB>(row, (int)(v.z & 0xffff) - T.src0, T.l); row_bit<WB>(row, (int)(v.z >> 16) - T.src0, T.l);
      row_bit<WB>(row, (int)(v.w & 0xffff) - T.src0, T.l); row_bit<WB>(row, (int)(v.w >> 16) - T.src0, T.l);
    }
    if (T.dq & 1) {
      const uint2 v = ((const uint2*)T.nbr)[2 * off + (T.dq - 1)];
      row_bit<WB>(row, (int)(v.x & 0xffff) - T.src0, T.l); row_bit<WB>(row, (int)(v.x >> 16) - T.src0, T.l);
      row_bit<WB>(row, (int)(v.y & 0xffff) - T.src0, T.l); row_bit<WB>(row, (int)(v.y >> 16) - T.src0, T.l);
    }
    lds_store<WB>(cur + r * WB, row);
#pragma unroll
    for (int k = 0; k < WB; k++) pop += (u32)__popc(row.w[k]);
  }
  int par = 0;
  u32 c = block_total(pop, s_part[par], wave);
  u32 prev = 0;
  u64 sum = 0;
  int L = 0, D = 0;
  bool disc = false;
  // (n = 30002, d = 7: level 0 8.4k -> 3.2k cycles, the walked third 11.5k -> 5.7k,
  // with the counts taken from the bit-sets instead of a pass over the rows)
  // levels 1 .. T.walk - 1: the walks of exactly L + 1 steps from each source
  // set its bit in the rows they end at (the rows already hold level L - 1,
  // every shorter walk); the exits are left to the pulled levels' loop below
  while (WALK && L + 1 < T.walk && c != target && !(L >= 1 && c == prev) && L + 1 < T.n) {
    sum += (u64)(target - c) * (u64)T.s;
    prev = c;
    L++;
    const u32 steps = (u32)L + 1;
    // a thread takes a walk's first steps - 1 steps (its prefix, decoded with
    // divisions) and then every last step at once: the whole table row of the
    // vertex reached, 8 ids a load -- deg walks per decoded prefix
    u32 all = 1;
    for (u32 i = 0; i + 1 < steps; i++) all *= (u32)T.deg;
    const FastDiv per(all), deg((u32)T.deg);
    pop = 0;
    for (u32 it = (u32)tid; it < (u32)T.l * all; it += (u32)nth) {
      u32 rem;
      const u32 c0 = per.div(it, rem);
      int v = T.src0 + (int)c0;
      for (u32 i = 0; i + 1 < steps; i++) {
        u32 j;
        rem = deg.div(rem, j);
        v = T.nbr[v * T.dp + (int)j];
      }
      u32* col = cur + (int)(c0 >> 5);
      const u32 b = 1u << (c0 & 31);
      auto set2 = [&](u32 g) {
        const u32 x = atomicOr(col + (g & 0xffff) * WB, b), y = atomicOr(col + (g >> 16) * WB, b);
        pop += ((x & b) == 0) + ((y & b) == 0);
      };
      const uint4* ids = (const uint4*)(T.nbr + v * T.dp);
      for (int q = 0; q < (T.dq >> 1); q++) {
        const uint4 g = ids[q];
        set2(g.x); set2(g.y); set2(g.z); set2(g.w);
      }
      if (T.dq & 1) {
        const uint2 g = ((const uint2*)ids)[T.dq - 1];
        set2(g.x); set2(g.y);
      }
    }
    par ^= 1;
    c += block_total(pop, s_part[par], wave);
  }
  // the pulled levels: a thread's own rows stay in registers from level to level
  RowT<WB> own[RPT];
  uint4 w0 = make_uint4(0, 0, 0, 0), w1 = w0;      // the first 16 ids of the row fetched last
  bool live = false;                               // ... which has bits to gain
  auto is_full = [&](const RowT<WB>& q) {
    bool f = true;
#pragma unroll
    for (int k = 0; k < WB; k++) f = f && q.w[k] == full.w[k];
    return f;
  };
  auto ids_at = [&](int i, int nl) { return (const uint4*)(T.nbr + (int64_t)(i * nl) * T.dp) + (u32)tid * (u32)(T.dp >> 3); };
  auto fetch = [&](int i, int nl) {
    live = tid + i * nl < T.n && !is_full(own[i]);
    if (live) {
      const uint4* ids = ids_at(i, nl);
      w0 = ids[0];
      if (T.dq > 2) w1 = ids[1];
    }
  };
  if (c != target) {
    const int nl = again(nth);
#pragma unroll
    for (int i = 0; i < RPT; i++) {
      const int r = tid + i * nl;
      if (r < T.n) own[i] = lds_row<WB>(cur + r * WB);
      else
#pragma unroll
        for (int k = 0; k < WB; k++) own[i].w[k] = 0;
    }
    fetch(0, nl);
  }
  for (;;) {
    if (c == target) { D = L + 1; break; }
    if ((L >= 1 && c == prev) || L + 1 >= T.n) { disc = true; break; }
    sum += (u64)(target - c) * (u64)T.s;
    prev = c;
    L++;
    pop = 0;
    const int nl = again(nth);
#pragma unroll
    for (int i = 0; i < RPT; i++) {
      if (i > 0 && i * nl >= T.n) break;           // uniform
      // the next row's ids are on their way while this row's neighbours are read
      const uint4 v0 = w0, v1 = w1;
      const bool need = live;
      live = false;
      if (i + 1 < RPT) fetch(i + 1, nl);
      if (need) {
        row_or2<WB>(own[i], cbase, v0.x); row_or2<WB>(own[i], cbase, v0.y);
        if (T.dq > 1) { row_or2<WB>(own[i], cbase, v0.z); row_or2<WB>(own[i], cbase, v0.w); }
        if (T.dq > 2 && !(STOP && is_full(own[i]))) {        // STOP: a row filled by 8 neighbours reads no more
          uint4 v2 = make_uint4(0, 0, 0, 0);           // ids past the sixteenth: a group ahead
          if (T.dq > 4) v2 = ids_at(i, nl)[2];
          row_or2<WB>(own[i], cbase, v1.x); row_or2<WB>(own[i], cbase, v1.y);
          if (T.dq > 3) { row_or2<WB>(own[i], cbase, v1.z); row_or2<WB>(own[i], cbase, v1.w); }
          for (int j = 4; j < T.dq && !(STOP && is_full(own[i])); j += 2) {
            const uint4 v = v2;
            if (j + 2 < T.dq) v2 = ids_at(i, nl)[(j >> 1) + 1];
            row_or2<WB>(own[i], cbase, v.x); row_or2<WB>(own[i], cbase, v.y);
            if (j + 1 < T.dq) { row_or2<WB>(own[i], cbase, v.z); row_or2<WB>(own[i], cbase, v.w); }
          }
        }
      }
#pragma unroll
      for (int k = 0; k < WB; k++) pop += (u32)__popc(own[i].w[k]);
    }
    fetch(0, nl);                                // the next level's first row, ahead of the barriers
    par ^= 1;
    c = block_total(pop, s_part[par], wave);   // every read of this level is done
    {
      const int nl = again(nth);
#pragma unroll
      for (int i = 0; i < RPT; i++) {
        if (i > 0 && i * nl >= T.n) break;
        const int r = tid + i * nl;
        if (r < T.n) lds_store<WB>(cur + r * WB, own[i]);
      }
    }
    __syncthreads();                               // the new level is visible
  }
  ResOut r;
  r.sum = sum; r.diam = D; r.flags = disc ? 1u : 0u; r.levels = (u32)(L + 1); r.pad = 0;
  return r;
}

// adds a block's totals into its graph's accumulators
__device__ __forceinline__ void res_commit(ResOut* out, int graph, const ResOut& b, int lane, int wave)
{
  if (wave == 0) {       // wave-uniform branch; only lane 0 contributes
    const bool first = lane == 0;
    atomicAdd(&out[graph].sum, first ? b.sum : 0ULL);
    atomicMax(&out[graph].diam, b.diam);
    atomicOr(&out[graph].flags, b.flags);
    atomicAdd(&out[graph].levels, first ? b.levels : 0u);
  }
}

// End of a batch of levels as the host reads it (pinned, coherent host memory).
struct LvHost {
  int err;          // the device error flag as it stood at the end of the batch
  u32 asym;         // the table's asymmetry flag (k_symcheck)
  u32 seq;          // the batch's sequence number, written after these and the counters
};

// The counters of levels [from, to) (ring slots L % ring of every task), the
// error flag and the table's asymmetry flag, stored into host memory; then the next sequence number
// (kept on the device, so that a replayed graph advances it too), which the
// host watches for instead of synchronising the stream.
__global__ __launch_bounds__(256) void k_lvfin(const u64* __restrict__ cnt, int ntasks, int from, int to, int ring,
                                              u64* hcnt, const int* err, const u32* asym, LvHost* host,
                                              u32* dseq)
{
  const int m = (to - from) * ntasks;
  for (int i = threadIdx.x; i < m; i += blockDim.x) {
    const int L = from + i / ntasks, t = i - (i / ntasks) * ntasks;
    const int64_t k = (int64_t)(L % ring) * ntasks + t;
    hcnt[k] = cnt[k];
  }
  __threadfence_system();                          // each thread's stores reach host memory first
  __syncthreads();
  if (threadIdx.x == 0) {
    host->err = *err;
    host->asym = *asym;
    const u32 sq = *dseq + 1;
    *dseq = sq;
    __threadfence_system();
    __hip_atomic_store(&host->seq, sq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Result of a single-graph launch as the host reads it (pinned, coherent host memory).
struct ResHost {
  ResOut out;
  int err;          // the device error flag as it stood at the end of the launch
  u32 seq;          // the launch's sequence number, written after out and err
};

// Finishing step of a single-graph launch.  Each workgroup stores its totals
// (over the blocks it ran) in its own slot; the last one to arrive adds the
// slots up, hands the result and the error flag to host memory and leaves the
// queue head and the arrival counter at zero for the next launch, so a launch
// needs no clear before it and no copy after it.
// Entries to change (2-opt moves): row, position, new id, applied in order to
// the 16-bit table and the adjacency of one graph.
#define RES_PATCH_MAX 8
struct ResPatch {
  int n;
  int e[RES_PATCH_MAX][3];
  unsigned short* table; int tdp;
  int* adj; int degree;
};

// one thread: in order, since a later entry may overwrite an earlier one
__device__ __forceinline__ void res_patch(const ResPatch& p, bool adj_too)
{
  for (int i = 0; i < p.n; i++) {
    const int r = p.e[i][0], c = p.e[i][1], val = p.e[i][2];
    p.table[(int64_t)r * p.tdp + c] = (unsigned short)val;
    if (adj_too) p.adj[(int64_t)r * p.degree + c] = val;
  }
}

__global__ void k_patch(ResPatch p)
{
  if (threadIdx.x == 0) res_patch(p, true);
}

struct ResFin {
  u32* done;           // workgroups finished; null: no finishing step (batched launches)
  ResOut* part;        // [gridDim.x] per-workgroup totals
  ResHost* host;       // device address of the host result
  const int* err;      // device error flag
  // applied before the levels: every workgroup stores the entries into the
  // table it reads (the same values: no conflict), workgroup 0 also into the
  // adjacency -- a move folded into the evaluation's launch
  ResPatch patch;
  u32 seq;             // stored into host->seq once the result is in host memory
};

__device__ __forceinline__ u32 wave_or(u32 v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v |= __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ int wave_max(int v)
{
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// run by wave 0 of the last workgroup
__device__ __forceinline__ void res_finish(const ResFin& fin, int* qhead, int lane)
{
  __threadfence();
  u64 sum = 0, levels = 0;
  u32 flags = 0;
  int diam = 0;
  for (int i = lane; i < (int)gridDim.x; i += 64) {
    const ResOut* p = fin.part + i;
    sum += __hip_atomic_load(&p->sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    diam = max(diam, __hip_atomic_load(&p->diam, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    flags |= __hip_atomic_load(&p->flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    levels += __hip_atomic_load(&p->levels, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  sum = wave_sum(sum);
  levels = wave_sum(levels);
  flags = wave_or(flags);
  diam = wave_max(diam);
  if (lane == 0) {
    ResOut o;
    o.sum = sum; o.diam = diam; o.flags = flags; o.levels = (u32)levels; o.pad = 0;
    fin.host->out = o;
    fin.host->err = __hip_atomic_load(fin.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence_system();                           // the result before its sequence number
    __hip_atomic_store(&fin.host->seq, fin.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(qhead, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(fin.done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __threadfence_system();
  }
}

// The same loop for blocks of one width only: its register allocation is that
// width's alone (k_resident holds all four, and the widest pressure makes every
// width spill), and a launch can size its LDS to its own blocks.  STOP: a pulled
// row stops reading neighbours once full (measured: the 1024-graph batch 25.05
// -> 24.6 ms; one n=1024 graph 39.6k -> 36.0k evaluations/s, so only batches use it).
template <int WB, bool STOP = false, int RPT = res_rpt(WB)>
__global__ __launch_bounds__(1024) void k_resident_w(const ResTask* __restrict__ tasks, int ntasks,
                                                     int* __restrict__ qhead, ResOut* __restrict__ out, ResFin fin)
{
  extern __shared__ __attribute__((aligned(16))) u32 lds[];
  __shared__ int s_task, s_last;
  __shared__ __attribute__((aligned(16))) u32 s_part[2][16];
  const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 32 && (tid & 15) >= (nth + 63) / 64) s_part[tid >> 4][tid & 15] = 0;
  ResOut mine;           // this workgroup's totals (single-graph launches)
  mine.sum = 0; mine.diam = 0; mine.flags = 0; mine.levels = 0; mine.pad = 0;
  if (fin.patch.n) {     // uniform: a kernel argument
    if (tid == 0) {
      res_patch(fin.patch, blockIdx.x == 0);
      __threadfence();   // stored at L2 before any of this workgroup's table loads
    }
    __syncthreads();
  }
  // the first gridDim.x blocks are dealt by workgroup index, the rest popped
  // from *qhead (which then counts past gridDim.x)
  int t = blockIdx.x;
  while (t < ntasks) {
    const ResTask T = tasks[t];
    const ResOut b = res_run<WB, STOP, true, RPT>(T, lds, s_part, tid, nth, wave);
    if (fin.done) {
      mine.sum += b.sum; mine.diam = max(mine.diam, b.diam); mine.flags |= b.flags; mine.levels += b.levels;
    } else {
      res_commit(out, T.graph, b, lane, wave);
    }
    if ((int)gridDim.x >= ntasks) break;          // nothing left to pop
    if (wave == 0) {       // wave-uniform: lane 0 adds 1, the others add 0
      const int got = atomicAdd(qhead, lane == 0 ? 1 : 0);
      s_task = __builtin_amdgcn_readfirstlane(got);
    }
    __syncthreads();
    t = (int)gridDim.x + __builtin_amdgcn_readfirstlane(s_task);
  }
  if (fin.done) {        // uniform: a kernel argument
    if (tid == 0) {
      fin.part[blockIdx.x] = mine;
      __threadfence();   // the slot precedes the arrival
      s_last = atomicAdd(fin.done, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (s_last && wave == 0) res_finish(fin, qhead, lane);
  }
}

// Persistent: every workgroup pulls blocks from *qhead until none is left, so
// the grid drains once the queue is exhausted.  Blocks of any width run in the
// same launch (T.wb picks the instantiation).  The launch's dynamic LDS must
// hold n * wb * 4 bytes for its largest block, and blockDim.x * res_rpt(wb)
// must cover n for every block.
__global__ __launch_bounds__(1024) void k_resident(const ResTask* __restrict__ tasks, int ntasks,
                                                   int* __restrict__ qhead, ResOut* __restrict__ out)
{
  extern __shared__ __attribute__((aligned(16))) u32 lds[];
  __shared__ int s_task;
  __shared__ __attribute__((aligned(16))) u32 s_part[2][16];
  const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 32 && (tid & 15) >= (nth + 63) / 64) s_part[tid >> 4][tid & 15] = 0;
  for (;;) {
    if (wave == 0) {       // wave-uniform: lane 0 adds 1, the others add 0
      const int got = atomicAdd(qhead, lane == 0 ? 1 : 0);
      s_task = __builtin_amdgcn_readfirstlane(got);
    }
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(s_task);
    if (t >= ntasks) break;
    const ResTask T = tasks[t];
    ResOut b;
    switch (T.wb) {
      case 1: b = res_run<1>(T, lds, s_part, tid, nth, wave); break;
      case 2: b = res_run<2>(T, lds, s_part, tid, nth, wave); break;
      case 4: b = res_run<4>(T, lds, s_part, tid, nth, wave); break;
      default: b = res_run<8>(T, lds, s_part, tid, nth, wave); break;
    }
    res_commit(out, T.graph, b, lane, wave);
  }
}

// ---------------------------------------------------------------------------
// annealing on the device (k_anneal): many steps of the annealing loop of
// sample/SA/general.c:149-181 in one cooperative launch, for a regular general
// graph (s = 1) whose blocks fit LDS together with its neighbour table.
//
// Every workgroup holds the whole 16-bit neighbour table in LDS (the first
// `degree` entries of a row are its adjacency row) and evaluates one block of
// 32 * WB sources.  Wave 0 of every workgroup keeps the same copy of the
// chain's state -- generator, current and best results, temperature -- and
// draws the same 2-opt move the host's ODPX_Two_opt would draw from it, so the
// tables stay identical without any exchange.  Each step every workgroup
// publishes its block's totals in one word, watches for all the others', adds
// them up in the same order and makes the same acceptance decision (the test of
// sample/SA/common.c:15-43); a rejected move is undone in every table.
// Bound by the chain of a step: move, levels, totals across the XCDs, decision.
// One thread that searched the rows entry by entry, an arrival counter with a
// second read of the totals after it, and six workgroup barriers took 12.6 us a
// step at n = 1024, d = 6; rows searched by the wave's lanes, totals that carry
// their own arrival and two barriers 10.5.

struct AnnealState {
  uint64_t rng[4];
  double cur_a, best_a, temp, cooling, low_a;
  long long steps, accepted, best_sum;
  int cur_d, best_d, low_d;
  int optimum;          // the lower bounds were reached
  int stop;             // no valid move was found
  int hill, prio;
  int err;              // a grid barrier timed out
};

struct AnnealArgs {
  int* adj;             // [n][degree]: the chain's current graph (read at start, written at the end)
  int* best;            // [n][degree]: the best graph, written on every improvement
  AnnealState* st;
  u64* slots;           // [2][ntasks] packed block totals of a step (by step parity; zero at launch)
  int n, degree, dp, ntasks, steps;
};

#define ANNEAL_SPIN_LIMIT (1ull << 24)

__device__ __forceinline__ u32 anneal_rnd(uint64_t s[4], u32 bound)
{
  // xoshiro256** step and Lemire's multiply-shift, as odp_gen.c's rnd()
  const uint64_t r = ((s[1] * 5) << 7 | (s[1] * 5) >> 57) * 9, t = s[1] << 17;
  s[2] ^= s[0]; s[3] ^= s[1]; s[1] ^= s[2]; s[0] ^= s[3]; s[2] ^= t; s[3] = (s[3] << 45) | (s[3] >> 19);
  return (u32)(((r >> 32) * (uint64_t)bound) >> 32);
}

__device__ __forceinline__ uint64_t anneal_next(uint64_t s[4])
{
  const uint64_t r = ((s[1] * 5) << 7 | (s[1] * 5) >> 57) * 9, t = s[1] << 17;
  s[2] ^= s[0]; s[3] ^= s[1]; s[1] ^= s[2]; s[0] ^= s[3]; s[2] ^= t; s[3] = (s[3] << 45) | (s[3] >> 19);
  return r;
}

// first position of id among a row's entries, -1 if none; the wave's lanes look
// at 64 entries together, every lane returns the same value
__device__ __forceinline__ int anneal_find(const unsigned short* tab, int dp, int degree, int row, int id, int lane)
{
  for (int j = 0; j < degree; j += 64) {
    const u64 hit = __ballot(j + lane < degree && tab[row * dp + j + lane] == id);
    if (hit) return j + __ffsll((unsigned long long)hit) - 1;
  }
  return -1;
}

__device__ __forceinline__ void anneal_replace(unsigned short* tab, int dp, int degree, int row, int from, int to, int lane)
{
  const int j = anneal_find(tab, dp, degree, row, from, lane);
  if (j >= 0) tab[row * dp + j] = (unsigned short)to;
}

// a-b, c-d -> a-c, b-d in the table (ODPX_Swap_edges' order of replacements), by one wave
__device__ __forceinline__ void anneal_swap(unsigned short* tab, int dp, int degree, int a, int b, int c, int d, int lane)
{
  anneal_replace(tab, dp, degree, a, b, c, lane);
  anneal_replace(tab, dp, degree, b, a, d, lane);
  anneal_replace(tab, dp, degree, c, d, a, lane);
  anneal_replace(tab, dp, degree, d, c, b, lane);
}

// A block's totals of one step in one word, so that a workgroup's slot is
// complete whenever it is read: sum (bits 0..39: at most n levels of the 1.3 M
// bits a block's LDS holds), diameter (40..53: n <= 10240), flag (54), and the
// step's tag (55..63; a slot is rewritten two steps later at the earliest).
__device__ __forceinline__ u64 anneal_pack(const ResOut& b, int step)
{
  return b.sum | (u64)(u32)b.diam << 40 | (u64)(b.flags & 1) << 54 | (u64)((step + 1) & 511) << 55;
}

template <int WB>
__global__ __launch_bounds__(1024) void k_anneal(AnnealArgs a)
{
  extern __shared__ __attribute__((aligned(16))) u32 lds[];
  __shared__ __attribute__((aligned(16))) u32 s_part[2][16];
  __shared__ int s_mv[5], s_dec[3];
  __shared__ AnnealState S;          // the chain's state: wave 0 reads it, its lane 0 writes it
  const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (tid < 32 && (tid & 15) >= (nth + 63) / 64) s_part[tid >> 4][tid & 15] = 0;
  const int g = blockIdx.x, G = gridDim.x, n = a.n, deg = a.degree, dp = a.dp;
  u32* bits = lds;
  unsigned short* tab = (unsigned short*)(lds + ((n * WB + 3) & ~3));
  for (int i = tid; i < n * dp; i += nth) {
    const int r = i / dp, j = i - r * dp;
    tab[i] = (unsigned short)(j < deg ? a.adj[(int64_t)r * deg + j] : r);
  }
  if (tid == 0) S = *a.st;
  __syncthreads();
  ResTask T;
  T.nbr = tab; T.n = n; T.dp = dp; T.src0 = g * 32 * WB; T.l = min(32 * WB, n - T.src0);
  T.s = 1; T.graph = 0; T.wb = WB; T.dq = (max(deg, 1) + 3) / 4;
  T.deg = deg; T.walk = 0;                            // res_run below is built without walks
  for (int k = 0; k < a.steps; k++) {                 // uniform: every exit below is uniform
    if (wave == 0) {                                  // every lane holds the same values
      uint64_t rng[4] = {S.rng[0], S.rng[1], S.rng[2], S.rng[3]};
      int found = 0, ma = 0, mb = 0, mc = 0, md = 0;
      for (int tries = 0; tries < 1000000 && !found; tries++) {
        const int x = (int)anneal_rnd(rng, (u32)n), y = (int)anneal_rnd(rng, (u32)n);
        const u32 jx = anneal_rnd(rng, (u32)deg), jy = anneal_rnd(rng, (u32)deg);
        const int bx = tab[x * dp + jx], dy = tab[y * dp + jy];
        if (x == y || x == dy || bx == y || bx == dy) continue;
        if (anneal_find(tab, dp, deg, x, y, lane) >= 0 || anneal_find(tab, dp, deg, bx, dy, lane) >= 0) continue;
        anneal_swap(tab, dp, deg, x, bx, y, dy, lane);
        found = 1; ma = x; mb = bx; mc = y; md = dy;
      }
      if (lane == 0) {
        S.rng[0] = rng[0]; S.rng[1] = rng[1]; S.rng[2] = rng[2]; S.rng[3] = rng[3];
        if (!found) S.stop = 1;
        s_mv[0] = found; s_mv[1] = ma; s_mv[2] = mb; s_mv[3] = mc; s_mv[4] = md;
      }
    }
    __syncthreads();
    if (!s_mv[0]) break;
    const ResOut b = res_run<WB, false, false>(T, bits, s_part, tid, nth, wave);   // no walks (measured faster)
    if (wave == 0) {
      // publish this block's totals, then watch for every block's; they are
      // added in the same order in every workgroup
      u64* slots = a.slots + (k & 1) * G;
      __hip_atomic_store(&slots[g], anneal_pack(b, k), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      u64 sum = 0, spins = 0;
      u32 diam = 0, flags = 0;
      int abort = 0;
      for (int i0 = 0; i0 < G && !abort; i0 += 64) {
        const int i = min(i0 + lane, G - 1);
        u64 v;
        for (;;) {
          v = __hip_atomic_load(&slots[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          if (__ballot((int)(v >> 55) != ((k + 1) & 511)) == 0) break;
          if (++spins > ANNEAL_SPIN_LIMIT) { abort = 1; break; }
          __builtin_amdgcn_s_sleep(1);
        }
        if (i0 + lane < G) {
          sum += v & ((1ull << 40) - 1);
          diam = max(diam, (u32)(v >> 40) & 0x3fff);
          flags |= (u32)(v >> 54) & 1;
        }
      }
      if (abort) {
        if (lane == 0) { atomicOr(&a.st->err, 1); s_dec[2] = 1; }
      } else {
        sum = (u64)wave_sum_dpp((u32)(sum & 0xffffff)) + ((u64)wave_sum_dpp((u32)(sum >> 24)) << 24);
        diam = (u32)wave_max((int)diam);
        const bool disc = __ballot(flags != 0) != 0;
        // the result as ODP_Set_aspl reports it (aspl.c:73-74, 332-336)
        long lsum = (long)n * (n - 1) + (long)sum;
        int d = max(1, (int)diam);
        if (disc) d = n + 1;
        double aspl = lsum / (((double)n - 1) * n);
        lsum /= 2.0;
        if (d > n) { d = INT_MAX; lsum = LONG_MAX; aspl = DBL_MAX; }
        // every lane reads the state and decides alike; lane 0 stores what changed
        AnnealState q = S;
        q.steps++;
        int improved = 0, accept, drawn = 0;
        if (d < q.best_d || (d == q.best_d && aspl < q.best_a)) {
          improved = 1;
          q.best_d = d; q.best_sum = lsum; q.best_a = aspl;
          if (d == q.low_d && aspl == q.low_a) q.optimum = 1;
        }
        if (q.optimum) accept = 1;              // the loop ends here; the move stays
        else if (q.hill) accept = aspl <= q.cur_a;
        else if (d < q.cur_d && !q.prio) accept = 1;
        else if (d > q.cur_d && !q.prio) accept = 0;
        else if (aspl <= q.cur_a) accept = 1;
        else {
          const double diff = (q.cur_a - aspl) * n * (n - 1);
          const double u = ((double)(anneal_next(q.rng) >> 11) + 0.5) / 9007199254740992.0;
          accept = exp(diff / q.temp) > u;
          drawn = 1;
        }
        if (!q.optimum) {
          if (accept) { q.cur_d = d; q.cur_a = aspl; q.accepted++; }
          q.temp *= q.cooling;
        }
        if (lane == 0) {
          S.steps = q.steps; S.temp = q.temp; S.optimum = q.optimum;
          if (improved) { S.best_d = q.best_d; S.best_sum = q.best_sum; S.best_a = q.best_a; }
          if (accept) { S.cur_d = q.cur_d; S.cur_a = q.cur_a; S.accepted = q.accepted; }
          if (drawn) for (int i = 0; i < 4; i++) S.rng[i] = q.rng[i];
          s_dec[0] = improved; s_dec[1] = accept; s_dec[2] = 2 * q.optimum;
        }
      }
    }
    __syncthreads();
    if (s_dec[2] & 1) break;
    if (s_dec[0]) {                                    // the best graph: workgroup 0's table
      if (g == 0)
        for (int i = tid; i < n * deg; i += nth) a.best[i] = tab[(i / deg) * dp + (i % deg)];
      __syncthreads();
    }
    if (!s_dec[1] && wave == 0) anneal_swap(tab, dp, deg, s_mv[1], s_mv[3], s_mv[2], s_mv[4], lane);   // undo
    if (s_dec[2] & 2) break;                           // the lower bounds were reached
  }
  __syncthreads();
  if (g == 0) {
    for (int i = tid; i < n * deg; i += nth) a.adj[i] = tab[(i / deg) * dp + (i % deg)];
    if (tid == 0) {
      S.err = __hip_atomic_load(&a.st->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *a.st = S;
    }
  }
}
