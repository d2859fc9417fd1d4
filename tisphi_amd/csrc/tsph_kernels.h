// tsph_kernels.h — HIP kernels of the SPH step (gfx950).
//
// Launch model: every particle kernel runs over a fixed grid of 64-particle
// tiles; tiles[w] = (scene slot, first particle) for wave w, or slot -1 for
// an unused tile.  A wave therefore always belongs to one scene, and the
// scene parameters are read with wave-uniform (scalar) loads.  The grid is
// sized from the engine capacity, so one captured hipGraph serves any set
// of resident scenes.
#pragma once
#include <type_traits>

#include "tsph_device.h"

namespace tsph {

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own
// L2.  A grid that the chip holds at once (about 2048 threads per CU) is
// remapped so that every XCD walks one contiguous stretch of tiles:
// neighbouring particles (and their shared neighbour data) stay in one L2.
// A larger grid is remapped into kXcdStretches stretches per XCD, stretch c
// going to XCD c % 8: locality within a stretch, and an even share of the
// work per XCD when the work is not uniform along the tile range.  (One
// stretch per XCD left the 3D dam break's last two XCDs with 4 % of the
// fluid work: its water sits in the first 70 % of the particle order, and
// the busiest XCD set the pass time at 1.33x the even share.)  Both maps
// are bijections of [0, gridDim.x).  Stretched: block b on XCD x = b % 8 at
// position i = b / 8 takes logical block ((i / S) * 8 + x) * S + i % S for
// b below the largest multiple of 8 S, and b itself above it.
constexpr int kXcds = 8;
constexpr int kXcdStretches = 32;  // measured: 4 / 8 / 16 / 32 / 64 -> 4.03 / 3.99 / 3.96 / 3.94 / 3.95 ms per 3D step
constexpr int kOneRoundThreads = 256 * 2048;
__device__ __forceinline__ int xcd_block() {
  const int nb = gridDim.x, b = blockIdx.x;
  if (nb * (int)blockDim.x <= kOneRoundThreads) {
    const int q = nb / kXcds, r = nb % kXcds, x = b % kXcds;
    return x * q + (x < r ? x : r) + b / kXcds;
  }
  // blocks per stretch S = 2^sh: shifts instead of divisions
  const int sh = max(0, 31 - __clz(nb / (kXcds * kXcdStretches)));
  const int nmain = nb & ~((kXcds << sh) - 1);
  if (b >= nmain) return b;
  const int x = b % kXcds, i = b / kXcds;
  return ((((i >> sh) * kXcds) + x) << sh) + (i & ((1 << sh) - 1));
}
__device__ __forceinline__ int wave_id() {
  return __builtin_amdgcn_readfirstlane((int)((xcd_block() * blockDim.x + threadIdx.x) >> 6));
}

// Thread -> (slot, particle).  False for idle lanes.
__device__ __forceinline__ bool tile_thread(const KArgs& a, int& s, int& p) {
  const int w = wave_id();
  const int2 t = a.tiles[w];
  if (t.x < 0) return false;
  s = __builtin_amdgcn_readfirstlane(t.x);
  p = t.y + (int)(threadIdx.x & 63);
  const SceneDev S = a.scenes[s];
  return p < S.pbase + S.n;
}

// What a tile holds, set by the list build: solid particles with pairs (or
// rigid ones), boundary particles without, and flow or rigid particles.
constexpr int kTileWall = 1, kTileBare = 2, kTileFlow = 4;

// Particle p with the start of its list (any p below the capacity).
template <bool NL>
__device__ __forceinline__ Own own_of(const KArgs& a, int p) {
  Own o;
  o.P = a.cur.pos[p];
  o.n = 0;
  o.e0 = o.e1 = 0;
  if (NL) {
    o.n = a.w.nlc[p];
    const uint32_t* __restrict__ li = a.w.nl + nl_base(p, a.nl_cap) + (threadIdx.x & 3);
    o.e0 = li[0];
    o.e1 = li[nl_at(4)];
  }
  return o;
}

// Work distribution of the pair passes: four waves per tile, a quad of lanes
// per particle.  pred(s, p) says whether particle p has pairs to sum and, if
// not, stores what it gets instead.  Tiles without any of `flags` are left
// at once (the chain tile -> scene -> types of an idle wave costs more than
// its work: 26 k of the 3D dam break's 71 k tiles are wall).  PACK: the
// tile's particles with pairs are packed into groups of 16 first (boundary
// tiles: 26 % of their particles have any).  Without lists (NL false) a lane
// walks the stencil of its own particle.
template <bool NL, bool PACK, class Pred, class Body>
__device__ __forceinline__ void for_work(const KArgs& a, int flags, Pred&& pred, Body&& body) {
  const int lane = (int)(threadIdx.x & 63);
  const int w = wave_id();
  const int tile = NL ? w >> 2 : w, sub = w & 3;
  const int2 t = a.tiles[tile];
  if (NL && (a.w.tflag[tile] & flags) == 0) return;
  if (t.x < 0) return;
  const int s = __builtin_amdgcn_readfirstlane(t.x);
  const int end = a.scenes[s].pbase + a.scenes[s].n;
  if (!NL || !PACK) {
    const int p = t.y + (NL ? sub * 16 + (lane >> 2) : lane);
    if (p < end && pred(s, p, !NL || (lane & 3) == 0)) body(s, p, own_of<NL>(a, p));
    return;
  }
  const int p = t.y + lane;
  const bool work = p < end && pred(s, p, (lane >> 4) == sub);
  const unsigned long long mask = __ballot(work);
  const int cnt = __popcll(mask), g = sub * 16 + (lane >> 2);
  if (sub * 16 >= cnt) return;
  __shared__ uint8_t packed[kMaxBlock / 64][64];
  uint8_t* __restrict__ pk = packed[threadIdx.x >> 6];
  if (work)
    pk[__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0))] =
        (uint8_t)lane;
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (g < cnt) {
    const int q = t.y + (int)pk[g];
    body(s, q, own_of<NL>(a, q));
  }
}
// The lane that stores a particle's results.
template <int L>
__device__ __forceinline__ bool group_head() {
  return L == 1 || threadIdx.x % L == 0;
}

__device__ __forceinline__ int32_t scene_shift(const KArgs& a, const SceneDev& S) {
  return S.pbase - a.w.start[S.cbase];
}

// ===================================================================== sort
// update_grid_id (particle_system.py:228-236): renormalise the offset,
// flattened cell id, histogram with an arrival slot per particle.
//
// Cell of particle p, its cell id and offset brought up to date.  A particle
// that is still inside its cell (all but ~1 % of them in a step) keeps both
// as they are: renorm() changes nothing for an offset in [0, grid), since
// there floor(o / grid) = 0 exactly (-0, which it turns into +0, is not taken
// to be inside, nor is a NaN).  That leaves out the FP64 divisions, the
// decoding of the cell id and the stores (3D dam break: 52 -> 36 us).
template <int DIM>
__device__ __forceinline__ int32_t hash_one(const KArgs& a, const SceneDev& S, int s, int p, int32_t c, float4 P) {
  auto inside = [&](float o) { return __float_as_int(o) >= 0 && (double)o < S.grid; };
  if (inside(P.x) && inside(P.y) && (DIM == 3 ? inside(P.z) : __float_as_int(P.z) == 0)) return c;
  int cx, cy, cz;
  decode_cell(S, c, cx, cy, cz);
  renorm(cx, P.x, S.grid);
  renorm(cy, P.y, S.grid);
  if (DIM == 3) {
    renorm(cz, P.z, S.grid);
  } else {
    cz = 0;
    P.z = 0.0f;
  }
  int esc = 0;
  int* cc[3] = {&cx, &cy, &cz};
  float* oo[3] = {&P.x, &P.y, &P.z};
#pragma unroll
  for (int ax = 0; ax < DIM; ++ax) {
    int k = *cc[ax];
    if (k < 0 || k >= S.gn[ax]) {
      int cl = k < 0 ? 0 : S.gn[ax] - 1;
      *oo[ax] = (float)((double)*oo[ax] + (double)(k - cl) * S.grid);
      *cc[ax] = cl;
      esc = 1;
    }
  }
  if (esc) atomicAdd(&a.w.status[2 * s], 1ull);
  c = (cx * S.gn[1] + cy) * S.gn[2] + cz;
  a.cur.cell[p] = c;
  a.cur.pos[p] = P;
  return c;
}

// Arrival slot of a lane's particle among those of its key in `count`.  Runs
// of equal keys among consecutive lanes share one atomic: the run's first
// lane adds the run length and hands out its slots.  The live lanes of a
// wave are a prefix, and some lane is live.
__device__ __forceinline__ int arrival_slot(int32_t* count, int32_t key, bool live) {
  const int lane = (int)(threadIdx.x & 63);
  const int prev = __shfl_up(key, 1, 64);
  const bool head = live && (lane == 0 || prev != key);
  const unsigned long long heads = __ballot(head);
  const unsigned long long upto = (lane == 63) ? ~0ull : ((2ull << lane) - 1);
  const int first = 63 - __clzll(heads & upto);
  const unsigned long long above = heads & ~upto;
  const int nlive = __popcll(__ballot(live));
  const int next = above ? (__ffsll((long long)above) - 1) : nlive;
  int base = 0;
  if (head) base = atomicAdd(&count[key], next - lane);
  base = __shfl(base, first, 64);
  return base + (lane - first);
}

template <int DIM>
__global__ __launch_bounds__(256) void k_hash(KArgs a) {
  int s, p;
  const bool live = tile_thread(a, s, p);
  if (!__any(live)) return;  // before any cross-lane operation
  int32_t key = -1;
  if (live) {
    const SceneDev S = a.scenes[s];
    key = S.cbase + hash_one<DIM>(a, S, s, p, a.cur.cell[p], a.cur.pos[p]);
    a.w.key[p] = key;
  }
  const int slot = arrival_slot(a.w.count, key, live);
  if (live) a.w.slot[p] = slot;
}

// Exclusive scan of the cell histogram (the inclusive prefix sum of
// particle_system.py:256, stored shifted by one cell).  Two phases over
// blocks of kScanBlock*kScanItems cells: block sums, then every block adds
// up the sums before its own (at most kScanTile of them, 208 on the 3D dam
// break, one read per thread) and scans its cells; the down-sweep also clears
// the histogram for the next step.
constexpr int kScanBlock = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanBlock * kScanItems;

__device__ __forceinline__ int wave_incl_scan(int v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    int u = __shfl_up(v, d, 64);
    if (lane >= d) v += u;
  }
  return v;
}

// Block-wide exclusive scan of one int per thread; returns the total.
__device__ __forceinline__ int block_excl_scan(int v, int& total) {
  __shared__ int wsum[kScanBlock / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int inc = wave_incl_scan(v);
  if (lane == 63) wsum[wid] = inc;
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int k = 0; k < kScanBlock / 64; ++k) {
    if (k < wid) off += wsum[k];
    tot += wsum[k];
  }
  __syncthreads();
  total = tot;
  return off + inc - v;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_reduce(const int32_t* __restrict__ count,
                                                            int32_t* __restrict__ bsum, int n) {
  const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int i = base + k;
    if (i < n) s += count[i];
  }
  int total;
  block_excl_scan(s, total);
  if (threadIdx.x == 0) bsum[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_down(int32_t* __restrict__ count,
                                                          const int32_t* __restrict__ bsum,
                                                          int32_t* __restrict__ start,
                                                          uint8_t* __restrict__ cflow, int n) {
  const int base = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
  int loc[kScanItems];
  int s = 0;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int i = base + k;
    loc[k] = i < n ? count[i] : 0;
    s += loc[k];
  }
  int before = 0, total;
  for (int k = threadIdx.x; k < (int)blockIdx.x; k += kScanBlock) before += bsum[k];
  block_excl_scan(before, total);
  const int first = total;
  int off = block_excl_scan(s, total) + first;
  if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) start[n] = first + total;
#pragma unroll
  for (int k = 0; k < kScanItems; ++k) {
    int i = base + k;
    if (i < n) {
      start[i] = off;
      count[i] = 0;
      cflow[i] = 0;
    }
    off += loc[k];
  }
}

// The hash, scan and scatter of one small scene by one workgroup, with the
// histogram in LDS: one launch for four.  A workgroup takes a scene slot, so a
// batch of small scenes fills the chip.  Bounded by what a thread's registers
// hold (kSmallItems particles) and by 64 KiB of LDS, the wave sums included
// (kSmallCells); at these registers a CU holds one such workgroup, so the LDS
// costs no occupancy (9.1 k particles in 2D: 11.0 us, as with the LDS sized by
// the scene's cells).  Up to there it is the faster route: per step against
// the four launches, 1.5 k particles in 1.8 k cells 51 against 60 us, 9.4 k in
// 14.0 k cells 64 against 68, 15.0 k in 1.8 k cells 60.5 against 61.6, 16.1 k
// in 7.7 k cells 67 and 67, 16.1 k in 3D 95 against 96; 64 scenes of 14 k
// particles and cells 297 against 315, 256 of them 1257 against 1334.
constexpr int kSmallBlock = 1024;
constexpr int kSmallItems = 16;
constexpr int kSmallParticles = kSmallBlock * kSmallItems;
constexpr int kSmallWaves = kSmallBlock / 64;
constexpr int kSmallCells = 65536 / 4 - kSmallWaves;

// Workgroups of a launch at most; beyond, one takes several slots.  With one
// of 65,536 slots in use, a workgroup per slot took 196 us per step against
// the general sort's 158, this 145; of 16,384 slots 72, 70 and 61.
constexpr int kSmallGrid = 2048;  // at least a 64th of the slots an engine may have

template <int DIM>
__device__ __forceinline__ void sort_small_one(const KArgs& a, int s, int32_t* __restrict__ cnt,
                                               int32_t* __restrict__ wsum) {
  const SceneDev S = a.scenes[s];
  const int tid = (int)threadIdx.x, lane = tid & 63, wid = tid >> 6;
  for (int c = tid; c < S.ncell; c += kSmallBlock) cnt[c] = 0;
  __syncthreads();
  int32_t cell[kSmallItems], slot[kSmallItems];
  constexpr int kAhead = 8;  // particles whose loads are in flight together
#pragma unroll
  for (int k0 = 0; k0 < kSmallItems; k0 += kAhead) {
    if (k0 > 0 && k0 * kSmallBlock >= S.n) {
#pragma unroll
      for (int k = k0; k < k0 + kAhead; ++k) cell[k] = -1;
      continue;
    }
    float4 P[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int i = (k0 + k) * kSmallBlock + tid;
      cell[k0 + k] = i < S.n ? a.cur.cell[S.pbase + i] : -1;
      P[k] = a.cur.pos[S.pbase + min(i, max(S.n - 1, 0))];
    }
#pragma unroll
    for (int k = 0; k < kAhead; ++k) {
      const int i = (k0 + k) * kSmallBlock + tid;
      const bool live = i < S.n;
      if (!__any(live)) continue;
      int32_t& c = cell[k0 + k];
      if (live) {
        c = hash_one<DIM>(a, S, s, S.pbase + i, c, P[k]);
        a.w.key[S.pbase + i] = S.cbase + c;
      }
      slot[k0 + k] = arrival_slot(cnt, c, live);
    }
  }
  __syncthreads();
  // exclusive scan in place: a run of cells per thread, then the runs' sums
  const int per = (S.ncell + kSmallBlock - 1) / kSmallBlock, lo = min(tid * per, S.ncell), hi = min(lo + per, S.ncell);
  int sum = 0;
  for (int c = lo; c < hi; ++c) sum += cnt[c];
  const int inc = wave_incl_scan(sum);
  if (lane == 63) wsum[wid] = inc;
  __syncthreads();
  int off = S.sbase + inc - sum;
  for (int k = 0; k < wid; ++k) off += wsum[k];
  for (int c = lo; c < hi; ++c) {
    const int n = cnt[c];
    cnt[c] = off;
    off += n;
  }
  __syncthreads();
  for (int c = tid; c < S.ncell; c += kSmallBlock) {
    a.w.start[S.cbase + c] = cnt[c];
    a.w.cflow[S.cbase + c] = 0;
  }
  if (tid == 0) {
    // equal to the first entry of the scene above, if one follows directly
    a.w.start[S.cbase + S.ncell] = S.sbase + S.n;
    a.w.start[a.ccap] = S.total;
  }
#pragma unroll
  for (int k = 0; k < kSmallItems; ++k)
    if (cell[k] >= 0) a.w.tmp[cnt[cell[k]] + slot[k]] = S.pbase + k * kSmallBlock + tid;
}
template <int DIM>
__global__ __launch_bounds__(kSmallBlock) void k_sort_small(KArgs a, int nslots) {
  __shared__ int32_t cnt[kSmallCells];
  __shared__ int32_t wsum[kSmallWaves];
  const int grid = (int)gridDim.x;
  unsigned long long turns = 1;  // those of this workgroup with a scene
  if (nslots > grid) {
    const int s = (int)blockIdx.x + (int)(threadIdx.x & 63) * grid;
    turns = __ballot(s < nslots && a.scenes[min(s, nslots - 1)].active);
  } else if (!a.scenes[blockIdx.x].active) {
    return;
  }
  while (turns) {
    sort_small_one<DIM>(a, (int)blockIdx.x + __builtin_ctzll(turns) * grid, cnt, wsum);
    turns &= turns - 1;
    if (turns) __syncthreads();  // the cells are read to the end, the next slot's follow
  }
}

// The cells [cb, ce) of a scene just added, which no sort has filled yet,
// hold nothing: its first entry stays (the end of the scene below, if one
// ends there) and the others take its value.  A sort of small scenes writes
// their own entries only, so a range that a removed scene held keeps that
// scene's counts, and a pass run before the next sort would walk them.
// next: entry ce is the first of another scene.  It is too high by `excess`,
// the particles of scenes removed since the last sort, by which it and all
// above then move down: the others' ranges stay as they are, for only
// differences of entries are used.
__global__ __launch_bounds__(256) void k_empty_cells(int32_t* __restrict__ start, int cb, int ce, int next,
                                                     int32_t* __restrict__ excess) {
  const int i = cb + 1 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int32_t v = start[cb];
  if (i < ce || (i == ce && !next)) start[i] = v;
  if (i == ce && next) *excess = start[ce] - v;
}
__global__ __launch_bounds__(256) void k_close_cells(int32_t* __restrict__ start, int ce, int n,
                                                     const int32_t* __restrict__ excess) {
  const int i = ce + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i < n) start[i] -= *excess;
}

__global__ __launch_bounds__(256) void k_scatter(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const int32_t key = a.w.key[p];
  a.w.tmp[a.w.start[key] + a.w.slot[p]] = p;
}

// counting_sort (particle_system.py:238-252) with a deterministic slot:
// rank among the particles of the same cell by previous index (the serial
// reference order), then move the persistent state to the other buffer.
// The slots of a workgroup lie in the cells of its first and last slot;
// those cells' arrival slots are staged in LDS once, so the rank count of
// every thread reads LDS (lanes of one cell read the same words) instead
// of the texture path (the global-memory count kept the TD unit ~94 % busy).
constexpr int kRankStage = 1024;
__device__ __forceinline__ float wc_eos(const SceneDev& S, float rt);
__device__ __forceinline__ void dp_adapt_store(const KArgs& a, const SceneDev& S, int p, double (&t)[6], float rt);
template <bool DPN>
__global__ __launch_bounds__(256) void k_rank_move(KArgs a, int move_vtmp, int move_mui,
                                                   int move_dp, int fuse_init) {
  __shared__ int32_t win[kRankStage];
  __shared__ int32_t wlo, whi;
  const int total = a.w.start[a.ccap];
  const int k0 = blockIdx.x * blockDim.x;
  if (k0 >= total) return;  // workgroup-uniform
  const int k = k0 + (int)threadIdx.x;
  const bool live = k < total;
  int p = 0, b = 0, e = 0;
  int32_t key = 0;
  if (live) {
    p = a.w.tmp[k];
    key = a.w.key[p];
    b = a.w.start[key];
    e = a.w.start[key + 1];
  }
  const int klast = min(k0 + (int)blockDim.x, total) - 1;
  if (k == k0) wlo = b;
  if (k == klast) whi = e;
  __syncthreads();
  const int lo = wlo, nw = whi - lo;
  const bool staged = nw <= kRankStage;  // workgroup-uniform
  if (staged) {
    for (int q = (int)threadIdx.x; q < nw; q += (int)blockDim.x) win[q] = a.w.tmp[lo + q];
    __syncthreads();
  }
  if (!live) return;
  int rank = 0;
  if (staged) {
    for (int q = b; q < e; ++q) rank += (win[q - lo] < p) ? 1 : 0;
  } else {
    for (int q = b; q < e; ++q) rank += (a.w.tmp[q] < p) ? 1 : 0;
  }
  const int s = a.w.sid[p];
  const SceneDev S = a.scenes[s];
  const int d = S.pbase + (b - a.w.start[S.cbase]) + rank;
  a.alt.cell[d] = key - S.cbase;
  if (is_flow(a.cur.type[p])) a.w.cflow[key] = 1;  // same value from every writer
  a.alt.pos[d] = a.cur.pos[p];
  a.alt.vel[d] = a.cur.vel[p];
  a.alt.mass[d] = a.cur.mass[p];
  a.alt.type[d] = a.cur.type[p];
  a.alt.id0[d] = a.cur.id0[p];
  a.alt.obj[d] = a.cur.obj[p];
  // (HBM-bound: 842 MB in 160 us for 4.5 M particles before v_tmp, formed
  // anew, was left out; now 146 us)
  if (move_vtmp && !(fuse_init && is_real(a.cur.type[p]))) a.alt.vtmp[d] = a.cur.vtmp[p];
  const int st = a.stride;
  if (move_mui) {
    // a soil particle's stress is not read in a step, whose regularisation
    // writes it anew
    if (!(fuse_init && a.cur.type[p] == kSoil))
#pragma unroll
      for (int c = 0; c < 6; ++c) a.alt.sig_f[c * st + d] = a.cur.sig_f[c * st + p];
    a.alt.seq[d] = a.cur.seq[p];
  }
  if (move_dp) {
#pragma unroll
    for (int c = 0; c < 6; ++c) a.alt.sig_d[c * st + d] = a.cur.sig_d[c * st + p];
    a.alt.seq[d] = a.cur.seq[p];
    a.alt.seqp[d] = a.cur.seqp[p];
    a.alt.flag[d] = a.cur.flag[p];
  }
  if (fuse_init) {
    // init_real2tmp (solver_sph_base.py:67-74) at the new position, and the
    // Tait pressure the first one_step starts with (solver_sph_wc.py:88).
    const int t = a.cur.type[p];
    if (is_real(t)) {
      const float4 v = a.cur.vel[p];
      a.alt.vtmp[d] = v;
      if (S.method == kWC && t == kFluid) {
        const float pv = wc_eos(S, v.w);
        a.w.p[d] = pv;
        a.w.vp[d] = make_float4(v.x, v.y, v.z, pv / (v.w * v.w));
      }
    }
    // muI: stress_tmp is formed by the first soil loop.  DP: with the return
    // mapping that starts the first one_step.
    if (DPN && t == kSoil) {
      double q[6];
#pragma unroll
      for (int c = 0; c < 6; ++c) q[c] = a.cur.sig_d[c * st + p];
      dp_adapt_store(a, S, d, q, a.cur.vel[p].w);
    }
  }
}

// ============================================================ pair helpers
// Walk the stencil around particle p's own (renormalised) cell.
template <int DIM, class Fn>
__device__ __forceinline__ void walk_c(const SceneDev& S, const KArgs& a, int p, const float4& P,
                                       Fn&& fn) {
  int cx, cy, cz;
  decode_cell(S, a.cur.cell[p], cx, cy, cz);
  walk<DIM>(S, a.w.start, a.cur.pos, scene_shift(a, S), p, cx, cy, cz, cx, cy, cz, P.x, P.y, P.z, fn);
}

// The stencil walk by a quad of lanes: lane q tests every fourth candidate
// and the hits' terms are added in walk order, as in sum_list().
template <int DIM, int NT, class Fn>
__device__ __forceinline__ void walk_quad(const SceneDev& S, const KArgs& a, int i, const float4& P,
                                          float (&acc)[NT], Fn&& fn) {
  int cx, cy, cz;
  decode_cell(S, a.cur.cell[i], cx, cy, cz);
  const int32_t shift = scene_shift(a, S);
  const int q = (int)threadIdx.x & 3;
#pragma unroll 1
  for (int k = 0; k < (DIM == 3 ? 27 : 9); ++k) {
    const int dx = k / (DIM == 3 ? 9 : 3) - 1, dy = (DIM == 3 ? k / 3 : k) % 3 - 1, dz = DIM == 3 ? k % 3 - 1 : 0;
    const int nx = cx + dx, ny = cy + dy, nz = cz + dz;
    if (nx < 0 || nx >= S.gn[0] || ny < 0 || ny >= S.gn[1] || nz < 0 || nz >= S.gn[2]) continue;
    const float bx = P.x + (float)(-dx) * S.g, by = P.y + (float)(-dy) * S.g;
    const float bz = DIM == 3 ? P.z + (float)(-dz) * S.g : 0.0f;
    const int32_t key = S.cbase + (nx * S.gn[1] + ny) * S.gn[2] + nz;
    const int32_t je = a.w.start[key + 1] + shift;
    for (int32_t j0 = a.w.start[key] + shift; j0 < je; j0 += 4) {
      const int32_t j = j0 + q;
      const float4 pj = a.cur.pos[min(j, je - 1)];
      const float x = bx - pj.x, y = by - pj.y, z = DIM == 3 ? bz - pj.z : 0.0f;
      const float r2 = fmaf(z, z, fmaf(y, y, x * x));
      const bool hit = j < je && r2 < S.rs2 && j != i;
      if (!__any(hit)) continue;
      float t[NT];
#pragma unroll
      for (int c = 0; c < NT; ++c) t[c] = 0.0f;
      if (hit) fn(j, x, y, z, r2, pj.w, t);
      ordered_add<4>(acc, t);
    }
  }
}

// acc[c] += term c of every neighbour of p: over the stored list when the
// step has lists, by the stencil walk when p's is longer than nl_cap or there
// are none.  All visit the same pairs in the same order.
template <int DIM, bool NL, int L, int NT, class Fn>
__device__ __forceinline__ void sum_pairs(const SceneDev& S, const KArgs& a, int p, const Own& o,
                                          float (&acc)[NT], Fn&& fn) {
  if (NL) {
    if (o.n <= a.nl_cap) sum_list<DIM>(S, a.w.nl, a.nl_cap, a.cur.pos, p, o, acc, fn);
    else walk_quad<DIM>(S, a, p, o.P, acc, fn);
    return;
  }
  walk_c<DIM>(S, a, p, o.P, [&](int j, float x, float y, float z, float r2, float mVj, int) {
    float t[NT];
    fn(j, x, y, z, r2, mVj, t);
    ordered_add<1>(acc, t);
  });
}

// Appends of one particle's list, four entries per 16-byte store: a quarter
// of the write transactions of one store per entry.
struct ListAppender {
  uint32_t* __restrict__ li;
  int cap, n = 0;
  // the last three entries, oldest first (a shift register: no per-lane
  // compare picks the slot)
  uint32_t b0 = 0, b1 = 0, b2 = 0;
  __device__ __forceinline__ void add(uint32_t e) {
    if ((n & 3) == 3 && n < cap) *reinterpret_cast<uint4*>(li + nl_at(n - 3)) = make_uint4(b0, b1, b2, e);
    b0 = b1;
    b1 = b2;
    b2 = e;
    ++n;
  }
  // the last 1-3 entries, padded with the null particle's
  __device__ __forceinline__ int finish(uint32_t pad) {
    const int r = n & 3;
    if (n <= cap && r > 0) {
      const uint4 v = r == 3 ? make_uint4(b0, b1, b2, pad)
                             : (r == 2 ? make_uint4(b1, b2, pad, pad) : make_uint4(b2, pad, pad, pad));
      *reinterpret_cast<uint4*>(li + nl_at(n - r)) = v;
    }
    return n;
  }
};

// sum_pairs() with the scene's kernel type as a compile-time tag: fn gets
// KTag<1> (Wendland C2) or KTag<0> (cubic) first, so its kernel values
// come from kernel_W_t / kernel_gradfac_t (straight-line code).
template <int K>
struct KTag {
  static constexpr int v = K;
};
template <int DIM, bool NL, int L, int NT, class Fn>
__device__ __forceinline__ void sum_pairs_k(const SceneDev& S, const KArgs& a, int p,
                                            const Own& o, float (&acc)[NT], Fn&& fn) {
  if (S.kernel == 1)
    sum_pairs<DIM, NL, L>(S, a, p, o, acc, [&](int j, float x, float y, float z, float r2, float mVj,
                                               float (&t)[NT]) { fn(KTag<1>{}, j, x, y, z, r2, mVj, t); });
  else
    sum_pairs<DIM, NL, L>(S, a, p, o, acc, [&](int j, float x, float y, float z, float r2, float mVj,
                                               float (&t)[NT]) { fn(KTag<0>{}, j, x, y, z, r2, mVj, t); });
}
// A term that no neighbour of another kind adds: +0 leaves a sum's bits.
template <int NT>
__device__ __forceinline__ void no_terms(float (&t)[NT]) {
#pragma unroll
  for (int c = 0; c < NT; ++c) t[c] = 0.0f;
}

// Whether any of the 3^DIM stencil cells around (cx, cy, cz) holds a flow
// particle (per-cell flags set by the last sort).  Stops at the first one:
// cheaper than loading all flags together (measured).
template <int DIM>
__device__ __forceinline__ bool flow_in_reach(const SceneDev& S, const uint8_t* __restrict__ cflow,
                                              int cx, int cy, int cz) {
  const int gx = S.gn[0], gy = S.gn[1], gz = S.gn[2];
  for (int dx = -1; dx <= 1; ++dx) {
    const int nx = cx + dx;
    if (nx < 0 || nx >= gx) continue;
    for (int dy = -1; dy <= 1; ++dy) {
      const int ny = cy + dy;
      if (ny < 0 || ny >= gy) continue;
      for (int dz = (DIM == 3 ? -1 : 0); dz <= (DIM == 3 ? 1 : 0); ++dz) {
        const int nz = cz + dz;
        if (nz < 0 || nz >= gz) continue;
        if (cflow[S.cbase + (nx * gy + ny) * gz + nz]) return true;
      }
    }
  }
  return false;
}

// The tile's flags (every lane of the wave that owns it; n: list length, < 0
// for a lane without a particle).
__device__ __forceinline__ void set_tile_flags(const KArgs& a, int tile, int n, bool bdy, bool rig) {
  const bool some = n >= 0;
  const int f = (__any(some && (rig || (bdy && n > 0))) ? kTileWall : 0) |
                (__any(some && bdy && n == 0) ? kTileBare : 0) | (__any(some && !bdy) ? kTileFlow : 0);
  if ((threadIdx.x & 63) == 0) a.w.tflag[tile] = f;
}

// Neighbour-list build: one stencil walk per particle per step, recording
// (j << 6 | stencil code) for every neighbour; boundary particles keep only
// their flow neighbours (the only ones their passes read).  The candidate
// loop does nothing else, so the rarely taken append is the only divergent
// work in it.
template <int DIM>
__device__ __forceinline__ int nl_build_one(const KArgs& a, int s, int p, bool bdy, bool rig, int use_cflow,
                                            int cull) {
  const SceneDev S = a.scenes[s];
  const float4 P = a.cur.pos[p];
  const int8_t* __restrict__ type = a.cur.type;
  const int cap = a.nl_cap;
  uint32_t* __restrict__ li = a.w.nl + nl_base(p, cap);
  int cx, cy, cz;
  decode_cell(S, a.cur.cell[p], cx, cy, cz);
  // A boundary particle only records flow neighbours: none can exist if
  // no stencil cell holds a flow particle.
  if (bdy && use_cflow && !flow_in_reach<DIM>(S, a.w.cflow, cx, cy, cz)) return 0;
  ListAppender ap{li, cap};
  auto rec = [&](int j, float x, float y, float z, float r2, float mVj, int code) {
    if ((bdy && !is_flow(type[j])) || (rig && !(is_flow(type[j]) || type[j] == kRigid))) return;
    ap.add(nl_entry(j, code));
  };
  if (cull)
    walk<DIM, true>(S, a.w.start, a.cur.pos, scene_shift(a, S), p, cx, cy, cz, cx, cy, cz, P.x, P.y,
                    P.z, rec);
  else
    walk_c<DIM>(S, a, p, P, rec);
  return ap.finish(a.nl_pad);
}
template <int DIM>
__global__ __launch_bounds__(256) void k_nl_build(KArgs a, int use_cflow, int cull) {
  const int w = wave_id();
  if (a.tiles[w].x < 0) return;
  int s, p, n = -1;
  bool bdy = false, rig = false;
  if (tile_thread(a, s, p)) {
    // Boundary particles record flow neighbours only; rigid ones flow and
    // rigid neighbours (the XSPH sum of a rigid particle runs over rigid
    // ones); flow particles record all.
    bdy = is_bdy(a.cur.type[p]);
    rig = a.cur.type[p] == kRigid;
    n = nl_build_one<DIM>(a, s, p, bdy, rig, use_cflow, cull);
    a.w.nlc[p] = n;
  }
  set_tile_flags(a, w, n, bdy, rig);
}

// ------------------------------------------------ LDS-staged list build
// The same lists from candidates staged in LDS.  A workgroup of three waves
// owns one tile; wave v takes the stencil's dx = v - 1 plane for the tile's
// 64 particles, a lane each, so a tile's work is three independent pieces
// (a small scene has few tiles).  Cell keys run (row, fast) with the fast
// axis z in 3D and y in 2D.  The lanes of one row (a tile holds one or two)
// have their candidates of one row offset (dy in 3D) in one contiguous
// particle range, which the wave copies into LDS (STAGE candidates, the cell
// tile, at a time).
//
// Test: every lane walks its own three fast-axis cells there in the order of
// walk() and shifts one bit per candidate, hit or not, into a word per 32:
// 8 vector instructions per candidate (6 in 2D) and nothing else in the
// loop, so no lane waits for another's append.  Words with a hit go to LDS.
// Record: when all three waves have counted, each knows where its hits start
// in the list; a lane pops one hit per turn from its words, all lanes in the
// same turn, so four turns fill one aligned quad of every list and a wave's
// store is a contiguous kilobyte.  A quad that holds hits of two waves is
// written by the first of them.  A tile with a lane whose words do not fit
// (many cells of over 32 particles) is tested a second time and records its
// hits one by one; the counts, and so the places, are known by then.
//
// Bound by vector issue (the tests; 85-90 % busy in 3D).  Against one wave per
// tile that appended hit by hit: 4.5 M particles in 3D 1107 -> 1030 us; 191 k
// with the flow developed 172 -> 61; 307 k of soil in 3D 94.
constexpr int kStageDefault = 256;
constexpr int kBuildWaves = 3;
// per lane and wave: a word per cell and 1 to spare (30 KiB of LDS in 3D with
// 256 candidates staged: five workgroups per CU)
template <int DIM>
constexpr int kHitWords = DIM == 3 ? 10 : 5;

// Hit words of one lane in list order: rows [v NW, v NW + nw_v) of wave v.
template <int NW>
struct HitWords {
  const uint2 (*__restrict__ words)[64];
  const int32_t (*__restrict__ count)[64];  // words << 16 | hits, per wave
  int lane, v, k, end;
  uint32_t w = 0, eb = 0;
  __device__ __forceinline__ HitWords(const uint2 (*wd)[64], const int32_t (*ct)[64], int ln, int wave)
      : words(wd), count(ct), lane(ln), v(wave), k(wave * NW), end(wave * NW + (ct[wave][ln] >> 16)) {}
  // the next hit's entry; at least one is left in this wave's words
  __device__ __forceinline__ uint32_t pop() {
    if (w == 0) {
      const uint2 x = words[k++][lane];
      w = x.x;
      eb = x.y;
    }
    const int b = __builtin_clz(w);
    w ^= 0x80000000u >> b;
    return eb + ((uint32_t)b << kNlShift);
  }
  // as pop(), going on to the next waves' words; `pad` past the last
  __device__ __forceinline__ uint32_t pop_on(uint32_t pad) {
    while (w == 0 && k == end && v < kBuildWaves - 1) {
      ++v;
      k = v * NW;
      end = k + (count[v][lane] >> 16);
    }
    return (w == 0 && k == end) ? pad : pop();
  }
};

template <int DIM, int STAGE>
__global__ __launch_bounds__(64 * kBuildWaves) void k_nl_build_lds(KArgs a, int use_cflow) {
  constexpr int NW = kHitWords<DIM>;
  __shared__ float4 stage[kBuildWaves][STAGE + 32];  // read up to 31 past the window
  __shared__ uint2 words[kBuildWaves * NW][64];
  __shared__ int32_t count[kBuildWaves][64];  // words (at most NW + 1) << 16 | hits
  __shared__ int32_t flow[kBuildWaves][64];   // a flow particle in the wave's reach of the lane
  const int tile = __builtin_amdgcn_readfirstlane(xcd_block());
  const int2 t = a.tiles[tile];
  if (t.x < 0) return;  // unused tile: the whole workgroup leaves
  const int s = __builtin_amdgcn_readfirstlane(t.x);
  const int v = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int lane = (int)(threadIdx.x & 63), dx = v - 1;
  const SceneDev S = a.scenes[s];
  const int8_t* __restrict__ type = a.cur.type;
  const float4* __restrict__ pos = a.cur.pos;
  const int32_t* __restrict__ start = a.w.start;
  const int32_t shift = scene_shift(a, S);
  const int gx = S.gn[0], gy = DIM == 3 ? S.gn[1] : 1;  // rows: gx * gy
  const int gf = DIM == 3 ? S.gn[2] : S.gn[1];          // cells of a row
  const int p = t.y + lane;
  const bool live = p < S.pbase + S.n;
  int row = -1, f = 0, tp = 0;
  float4 P = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
    const int32_t c = a.cur.cell[p];
    row = c / gf;
    f = c - row * gf;
    P = pos[p];
    tp = type[p];
  }
  // boundary particles record flow neighbours only, rigid ones flow and rigid
  // neighbours (the XSPH sum of a rigid particle runs over rigid ones)
  const bool bdy = live && is_bdy(tp), rig = live && tp == kRigid;
  const int need = bdy ? 2 : (rig ? 1 : 0);
  float4* __restrict__ sp = stage[v];
  uint2(*__restrict__ wd)[64] = words + v * NW;
  // found(w, eb): hit bits (from the top) of up to 32 consecutive candidates,
  // the first of which has entry eb, in list order
  auto scan = [&](auto&& found) {
    unsigned long long todo = __ballot(live);
#pragma unroll 1
    while (todo) {
      // the lanes of the next row (consecutive in cell order)
      const int l0 = __builtin_ctzll(todo);
      const int R = __builtin_amdgcn_readlane(row, l0);
      bool act = row == R;
      const unsigned long long mine = __ballot(act);
      todo &= ~mine;
      const int l1 = 63 - __builtin_clzll(mine);
      int f0 = __builtin_amdgcn_readlane(f, l0), f1 = __builtin_amdgcn_readlane(f, l1);
      // Uploads since the sort (no flags then) may leave particles out of cell
      // order: the row's window is that of its outermost lanes, and a particle
      // may stand among the candidates of another cell than its own.
      if (!use_cflow) {
        f0 = act ? f : INT32_MAX;
        f1 = act ? f : -1;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
          f0 = min(f0, __shfl_xor(f0, d, 64));
          f1 = max(f1, __shfl_xor(f1, d, 64));
        }
      }
      const int wlo = max(f0 - 1, 0), whi = min(f1 + 1, gf - 1);
      const int rx = DIM == 3 ? R / gy : R, ry = DIM == 3 ? R - rx * gy : 0;
      const bool inx = rx + dx >= 0 && rx + dx < gx;
      // A boundary particle records nothing if no stencil cell holds a flow
      // particle.  The flags of a row offset's window are one load; each lane
      // picks its three from the wave's mask.
      if (use_cflow && __any(act && bdy)) {
        bool reach = whi - wlo >= 64;
        if (inx && !reach) {
#pragma unroll
          for (int dy = (DIM == 3 ? -1 : 0); dy <= (DIM == 3 ? 1 : 0); ++dy) {
            if (ry + dy < 0 || ry + dy >= gy) continue;
            const int32_t nk = S.cbase + ((rx + dx) * gy + ry + dy) * gf + wlo;
            const unsigned long long m = __ballot(lane <= whi - wlo && a.w.cflow[nk + min(lane, whi - wlo)] != 0);
            const int sh = act ? f - 1 - wlo : 0;  // bit of the lane's first cell
            reach = reach || ((sh >= 0 ? m >> sh : m << 1) & 7ull) != 0;
          }
        }
        flow[v][lane] = reach;
        __syncthreads();
        act = act && (!bdy || flow[0][lane] | flow[1][lane] | flow[2][lane]);
        __syncthreads();  // before the next row's flags
      }
      if (!inx || !__any(act)) continue;
      const bool filter = __any(act && need != 0);
      const float bx = P.x + (float)(-dx) * S.g;
#pragma unroll 1
      for (int dy0 = (DIM == 3 ? -1 : 0); dy0 <= (DIM == 3 ? 1 : 0); ++dy0) {
        if (ry + dy0 < 0 || ry + dy0 >= gy) continue;
        const int32_t nk = S.cbase + ((rx + dx) * gy + ry + dy0) * gf;
        const int32_t jlo = start[nk + wlo] + shift, cnt = start[nk + whi + 1] + shift - jlo;
        // the lane's cells: candidates [c[k], c[k + 1]) at fast offset k - 1
        int c[4] = {0, 0, 0, 0};
        if (act) {
          c[1] = start[nk + f] + shift - jlo;
          c[2] = start[nk + f + 1] + shift - jlo;
          c[0] = f > 0 ? start[nk + f - 1] + shift - jlo : c[1];
          c[3] = f < gf - 1 ? start[nk + f + 2] + shift - jlo : c[2];
        }
#pragma unroll 1
        for (int w0 = 0; w0 < cnt; w0 += STAGE) {
          const int wn = min(cnt - w0, STAGE);
          __builtin_amdgcn_wave_barrier();  // the last window's reads are done (one wave, in order)
          for (int q = lane; q < wn; q += 64) {
            float4 r = pos[jlo + w0 + q];
            const int tq = type[jlo + w0 + q];
            r.w = is_flow(tq) ? 2.0f : (tq == kRigid ? 1.0f : 0.0f);
            sp[q] = r;
          }
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          __builtin_amdgcn_wave_barrier();
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const int dy = DIM == 3 ? dy0 : k - 1, dz = DIM == 3 ? k - 1 : 0;
            const float by = P.y + (float)(-dy) * S.g;
            const float bz = DIM == 3 ? P.z + (float)(-dz) * S.g : 0.0f;
            // the sign bit of |r2| - rs2 (a NaN's is clear) is the hit
            auto dist = [&](const float4& r) {
              const float x = bx - r.x, y = by - r.y;
              float r2;
              if (DIM == 3) {
                const float z = bz - r.z;
                r2 = fmaf(z, z, fmaf(y, y, x * x));
              } else {
                r2 = fmaf(y, y, x * x);
              }
              return __float_as_uint(fabsf(r2) - S.rs2);
            };
            auto shift_in = [&](uint32_t w, const float4& r) {
              return __builtin_amdgcn_alignbit(w, dist(r), 31);
            };
            // as shift_in, for candidates the lane records (kind >= need) only
            auto shift_in_kind = [&](uint32_t w, const float4& r) {
              return __builtin_amdgcn_alignbit(w, dist(r) & ~__float_as_uint(r.w - (float)need), 31);
            };
            int lo = max(c[k] - w0, 0);
            const int hi = min(c[k + 1] - w0, wn);
#pragma unroll 1
            for (; __any(lo < hi); lo += 32) {
              const int m = min(hi - lo, 32);  // <= 0 for a lane that is done
              uint32_t w = 0;
              const float4* __restrict__ q = sp + min(lo, wn);
              int done = 0;
              if (!filter) {
#pragma unroll 1
                do {
                  const float4 r0 = q[0], r1 = q[1], r2 = q[2], r3 = q[3];
                  w = shift_in(shift_in(shift_in(shift_in(w, r0), r1), r2), r3);
                  done += 4;
                  q += 4;
                } while (__any(done < m));
              } else {
#pragma unroll 1
                do {
                  const float4 r0 = q[0], r1 = q[1], r2 = q[2], r3 = q[3];
                  w = shift_in_kind(shift_in_kind(shift_in_kind(shift_in_kind(w, r0), r1), r2), r3);
                  done += 4;
                  q += 4;
                } while (__any(done < m));
              }
              w <<= (32 - done) & 31;
              // candidates past the lane's cell, and the particle itself
              if (m < 32) w &= m > 0 ? ~(0xFFFFFFFFu >> m) : 0u;
              const int32_t j = jlo + w0 + lo;
              if (!use_cflow || (dx == 0 && dy == 0 && dz == 0)) {
                const int i = p - j;
                if (i >= 0 && i < 32) w &= ~(0x80000000u >> i);
              }
              if (w) found(w, nl_entry(j, ((dx + 1) << 4) | ((dy + 1) << 2) | (dz + 1)));
            }
          }
        }
      }
    }
  };
  int nw = 0, h = 0;
  scan([&](uint32_t w, uint32_t eb) {
    if (nw < NW) wd[nw][lane] = make_uint2(w, eb);
    ++nw;
    h += __popc(w);
  });
  // at most 2^16 - 1 hits can be recorded, and a list is far shorter
  count[v][lane] = min(nw, NW + 1) << 16 | min(h, 0xFFFF);
  __syncthreads();
  const int c0 = count[0][lane], c1 = count[1][lane], c2 = count[2][lane];
  const int cap = a.nl_cap;
  const int h0 = c0 & 0xFFFF, h1 = c1 & 0xFFFF, n = h0 + h1 + (c2 & 0xFFFF);
  if (v == 0) {
    if (live) a.w.nlc[p] = n;
    set_tile_flags(a, tile, live ? n : -1, bdy, rig);
  }
  // this wave's hits are [o, o + h) of the list
  const int o = (v > 0 ? h0 : 0) + (v > 1 ? h1 : 0);
  if (__any(max(c0, max(c1, c2)) >> 16 > NW)) {  // workgroup-uniform
    int k = o;
    uint32_t* __restrict__ li = a.w.nl + nl_base(live ? p : t.y, cap);
    scan([&](uint32_t w, uint32_t eb) {
      while (w) {
        const int b = __builtin_clz(w);
        w ^= 0x80000000u >> b;
        if (n <= cap) li[nl_at(k)] = eb + ((uint32_t)b << kNlShift);
        ++k;
      }
    });
    if (v == 2 && live && n <= cap)
      for (; k & (kNlPad - 1); ++k) li[nl_at(k)] = a.nl_pad;
    return;
  }
  if (n > cap) return;  // walked by the pair passes
  // the quads that start in it
  const int skip = -o & 3;
  if (h <= skip) return;
  uint32_t* __restrict__ li = a.w.nl + nl_base(p, cap) + nl_at(o + skip);
  HitWords<NW> hw(words, count, lane, v);
  for (int i = 0; i < skip; ++i) hw.pop();
  int left = h - skip;
  for (; left >= 4; left -= 4) {
    const uint32_t e0 = hw.pop(), e1 = hw.pop(), e2 = hw.pop(), e3 = hw.pop();
    *reinterpret_cast<uint4*>(li) = make_uint4(e0, e1, e2, e3);
    li += nl_at(4);
  }
  if (left > 0) {
    const uint32_t e0 = hw.pop(), e1 = hw.pop_on(a.nl_pad), e2 = hw.pop_on(a.nl_pad), e3 = hw.pop_on(a.nl_pad);
    *reinterpret_cast<uint4*>(li) = make_uint4(e0, e1, e2, e3);
  }
}

// calc_CSPM_f (solver_sph_base.py:386-398) over the recorded lists.
template <int DIM>
__global__ __launch_bounds__(256) void k_shepard_list(KArgs a, int skip_fluid) {
  const int8_t* __restrict__ type = a.cur.type;
  for_work<true, false>(
      a, ~0,
      [&](int, int p, bool mine) {
        if (skip_fluid && type[p] == kFluid) return false;  // formed by the fluid pass
        if (a.w.nlc[p] != 0) return true;
        if (mine) a.w.cspm[p] = 1.0f;
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        float acc[1] = {0.0f};
        sum_pairs_k<DIM, true, kLanes>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z,
                                                                       float r2, float mVj, float (&t)[1]) {
          // straight-line: a non-flow neighbour adds +0 (the sum's bits stay)
          const bool fl = is_flow(type[j]);
          const float w = kernel_W_t<decltype(kt)::v>(S, pair_dist(r2));
          t[0] = term_if(fl, mVj * w);
        });
        if (group_head<kLanes>()) a.w.cspm[p] = acc[0] != 0.0f ? 1.0f / acc[0] : 1.0f;
      });
}

// calc_CSPM_L (solver_sph_base.py:400-423) for scenes with
// kernelCorrection 1: L = sum_{j same type} m_V_j (x_j - x_i) (x) grad W_ij
// over a flow particle's neighbours, stored inverted; every other particle
// stores I.  With kernelCorrection 2 (the MLS switch) calc_kernel_corr
// computes no matrix (:363-368) and kernel_deriv_corr's branch for it is
// empty, so the corrected gradient is the zero vector (:375-384): the
// stored matrix is 0 (the untouched field), and the passes that apply it
// get a zero gradient.
template <int DIM, bool NL>
__global__ __launch_bounds__(256) void k_cspm_L(KArgs a) {
  constexpr int L = NL ? kLanes : 1;
  const int8_t* __restrict__ type = a.cur.type;
  auto store = [&](int p, const float M[9]) {
#pragma unroll
    for (int c = 0; c < 9; ++c) a.w.Lc[(size_t)c * a.stride + p] = M[c];
  };
  for_work<NL, false>(
      a, ~0,
      [&](int s, int p, bool mine) {
        const int kc = a.scenes[s].kcorr;
        if (kc == 0) return false;
        if (kc == 1 && is_flow(type[p])) return true;
        if (!mine) return false;
        const float one = kc == 1 ? 1.f : 0.f;
        const float M[9] = {one, 0.f, 0.f, 0.f, one, 0.f, 0.f, 0.f, one};
        store(p, M);
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        const int ti = type[p];
        float M[9] = {1.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f, 0.f, 1.f};
        float acc[9] = {};
        sum_pairs_k<DIM, NL, L>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z, float r2,
                                                                float mVj, float (&t)[9]) {
          const bool same = type[j] == ti;
          const float f = kernel_gradfac_t<decltype(kt)::v>(S, pair_dist(r2));
          const float g[3] = {f * x, f * y, f * z};
          const float c[3] = {mVj * (-x), mVj * (-y), mVj * (-z)};
#pragma unroll
          for (int k = 0; k < 9; ++k) t[k] = term_if(same, c[k / 3] * g[k % 3]);
        });
        const float Lm[3][3] = {{acc[0], acc[1], acc[2]}, {acc[3], acc[4], acc[5]}, {acc[6], acc[7], acc[8]}};
        corr_invert<DIM>(Lm, S.eps, M);
        if (group_head<L>()) store(p, M);
      });
}

// =================================================================== Shepard
// calc_CSPM_f (solver_sph_base.py:386-398)
template <int DIM>
__global__ __launch_bounds__(256) void k_shepard(KArgs a, int skip_fluid) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (skip_fluid && a.cur.type[p] == kFluid) return;  // formed by the fluid pass
  const SceneDev S = a.scenes[s];
  const float4 P = a.cur.pos[p];
  const int8_t* __restrict__ type = a.cur.type;
  float sum = 0.0f;
  walk_c<DIM>(S, a, p, P, [&](int j, float x, float y, float z, float r2, float mVj, int) {
    if (is_flow(type[j])) sum += mVj * kernel_W(S, pair_dist(r2));
  });
  a.w.cspm[p] = sum != 0.0f ? 1.0f / sum : 1.0f;
}

// init_real2tmp (solver_sph_base.py:67-74)
__global__ __launch_bounds__(256) void k_init_tmp(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  if (is_real(t)) a.cur.vtmp[p] = a.cur.vel[p];
  if (t == kSoil) {
    const int st = a.stride;
    if (S.method == kMUI) {
      float q[6];
#pragma unroll
      for (int c = 0; c < 6; ++c) q[c] = a.cur.sig_f[c * st + p];
      rec6_store(a.w.sigt_f, p, q);
    } else if (S.method == kDP) {
#pragma unroll
      for (int c = 0; c < 6; ++c) a.w.sigt_d[c * st + p] = a.cur.sig_d[c * st + p];
    }
  }
}

// ===================================================================== WCSPH
__global__ __launch_bounds__(256) void k_wc_eos(KArgs a) {  // solver_sph_wc.py:86-88
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (a.cur.type[p] == kFluid) {
    const float4 vt = a.cur.vtmp[p];
    const float pv = wc_eos(a.scenes[s], vt.w);
    a.w.p[p] = pv;
    a.w.vp[p] = make_float4(vt.x, vt.y, vt.z, pv / (vt.w * vt.w));
  }
}

// Dummy extrapolation (solver_sph_wc.py:90-103; solver_sph_base.py:653-663).
// With SHEP the same walk first forms the particle's Shepard sum
// (calc_CSPM_f, solver_sph_base.py:386-398: flow neighbours, list order),
// which the fused step then leaves out of the Shepard pass: bitwise equal.
// acc: sums of v (3), p and, with SHEP, W.
template <bool SHEP>
__device__ __forceinline__ void wc_wall_store(const KArgs& a, const SceneDev& S, int p, const float* acc) {
  const float4 v = a.cur.vel[p];
  float cs;
  if (SHEP) {
    cs = acc[4] != 0.0f ? 1.0f / acc[4] : 1.0f;
    a.w.cspm[p] = cs;
  } else {
    cs = a.w.cspm[p];
  }
  const float4 vt = make_float4(2.0f * v.x - acc[0] * cs, 2.0f * v.y - acc[1] * cs,
                                2.0f * v.z - acc[2] * cs, S.rho0);
  a.cur.vtmp[p] = vt;
  const float pv = acc[3] * cs;
  const float pc = pv > 0.0f ? pv : 0.0f;
  a.w.p[p] = pc;
  // sign bit marks the boundary particle for the fluid pass
  a.w.vp[p] = make_float4(vt.x, vt.y, vt.z,
                          __int_as_float(__float_as_int(pc / (S.rho0 * S.rho0)) | (int)0x80000000));
}
// again: a later one_step of the same fused step.  Most dummy particles have
// no flow particle in reach (an empty list): their sums are +0 in every
// one_step, so the first stores their extrapolation and the later ones skip
// them (1.41 M of the 1.65 M dummy particles of the 3D dam break).
template <int DIM, bool NL, bool SHEP>
__global__ __launch_bounds__(256) void k_wc_bdy(KArgs a, int again) {
  constexpr int L = NL ? kLanes : 1;
  const int8_t* __restrict__ type = a.cur.type;
  const float4* __restrict__ vtmp = a.cur.vtmp;
  const float* __restrict__ pr = a.w.p;
  for_work<NL, true>(
      a, again ? kTileWall : kTileWall | kTileBare,
      [&](int s, int p, bool mine) {
        const int tp = type[p];
        if (!is_solid(tp)) return false;  // boundary and rigid (solver_sph_wc.py:90-103)
        if (!NL || a.w.nlc[p] != 0) return true;
        if (mine && !(again && is_bdy(tp))) {
          const float none[5] = {};
          wc_wall_store<SHEP>(a, a.scenes[s], p, none);
        }
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        const float gy = S.grav[1];
        constexpr int NT = SHEP ? 5 : 4;
        float acc[NT] = {};
        // Straight-line pair terms (a non-flow neighbour adds +0, which leaves
        // every sum's bits unchanged: the sums start at +0 and never become -0
        // in round-to-nearest), so the loads of a batch of neighbours are
        // issued together instead of one branch at a time.
        sum_pairs_k<DIM, NL, L>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z, float r2,
                                                                float mVj, float (&t)[NT]) {
          const bool fl = is_flow(type[j]);
          const float4 vj = vtmp[j];
          const float prj = pr[j];
          const float w = kernel_W_t<decltype(kt)::v>(S, pair_dist(r2));
          t[0] = term_if(fl, mVj * vj.x * w);
          t[1] = term_if(fl, mVj * vj.y * w);
          t[2] = term_if(fl, mVj * vj.z * w);
          t[3] = term_if(fl, mVj * (prj + vj.w * gy * y) * w);
          if (SHEP) t[NT - 1] = term_if(fl, mVj * w);
        });
        if (group_head<L>()) wc_wall_store<SHEP>(a, S, p, acc);
      });
}

// Fluid loop B (solver_sph_wc.py:108-123; tasks solver_sph_base.py:195-203,
// solver_sph_wc.py:33-71): d_density and d_vel in one walk.  With SHEP
// the same walk also forms the particle's Shepard sum (calc_CSPM_f,
// solver_sph_base.py:386-398: flow neighbours, list order), which the fused
// step then leaves out of the Shepard pass: in WC only boundary particles
// read CSPM_f within the step, so fluid particles get it here, bitwise equal.
// The pair terms: d_density (solver_sph_base.py:195-203, by the corrected
// gradient with KC), viscosity and pressure force (solver_sph_wc.py:33-71,
// by the plain one) and, with SHEP, the Shepard sum.  A WC scene holds fluid,
// boundary and rigid particles only (checked at upload), and rigid ones are
// walls to the fluid: a neighbour's pair record q (v_tmp, p / rho_tmp^2,
// written by the EOS or the boundary pass, sign bit set for a wall) says
// which it is, so the pass reads position + m_V and q per neighbour and
// nothing else.
//
// In 2D z = g_z = 0, so the third components' terms are +-0, and the list
// replay, whose additions are most of its work, leaves them out (Z false).
// But 0 times an infinity, or a NaN, is not a number, which d_vel and
// d_density then carry.  So `odd` gathers the bits of the neighbours' v_z (an
// "or" of two of them with what is there is one instruction), a force that is
// not finite shows in d_vel, and wc_fluid_one() then forms the sums with all
// terms.  Batch of 256 in 2D, 1.31 M particles: passes of 91.1 and 80.5 us,
// without the check 93.1 and 79.0.
template <int DIM, bool Z, bool NL, bool SHEP, int KT, bool KC, int L, int NT>
__device__ __forceinline__ void wc_fluid_sums(const KArgs& a, const SceneDev& S, int p, const Own& o, const float4& vi,
                                              float pri, const float (&M)[9], float (&acc)[NT], uint32_t& odd) {
  static_assert(NT == (Z ? 4 : 3) + (SHEP ? 1 : 0), "d_density, d_vel, Shepard");
  const float4* __restrict__ vp = a.w.vp;
  const float c1 = S.visc_c1, c2 = S.visc_c2, rho0 = S.rho0;
  const float rr = rho0 / vi.w;  // rho0 / rho_i of the boundary viscosity
  sum_pairs<DIM, NL, L>(S, a, p, o, acc, [&](int j, float x, float y, float z, float r2, float mVj,
                                             float (&t)[NT]) {
    const float rn = pair_dist(r2);
    const float f = kernel_gradfac_t<KT>(S, rn);
    const float gx = f * x, gy = f * y, gz = f * z;
    float4 q = vp[j];
    if (DIM == 2) asm volatile("" : "+v"(q.z));  // one 16-byte load
    const bool bj = __float_as_int(q.w) < 0;  // boundary neighbour
    const float ux = vi.x - q.x, uy = vi.y - q.y, uz = vi.z - q.z;
    float cg[3] = {gx, gy, gz};
    if (KC) corr_apply(M, cg);
    t[0] = (mVj * ux) * cg[0] + (mVj * uy) * cg[1];
    if (Z || KC) t[0] += (mVj * uz) * cg[2];
    if (SHEP) t[NT - 1] = term_if(!bj, mVj * kernel_W_t<KT>(S, rn));
    // viscosity_force: fluid and boundary neighbours (solver_sph_wc.py:33-45)
    const float vx_ = Z ? ux * x + uy * y + uz * z : ux * x + uy * y;
    const float mn = vx_ < 0.0f ? vx_ : 0.0f;
    const float a0 = c1 * mVj;
    const float aa = bj ? a0 * rr : a0;
    const float vis = aa * mn / (r2 + c2);
    const float pc = (-rho0 * mVj) * (pri + fabsf(q.w));
    const float sc = vis + pc;
    t[1] = sc * gx;
    t[2] = sc * gy;
    if (Z) t[3] = sc * gz;
    else odd |= __float_as_uint(q.z);
  });
  if (S.rep) {
    // calc_rep_force_task (solver_sph_wc.py:74-76, 118-121): a second sweep
    // adding the repulsive particles' force after the pair forces
    const int8_t* __restrict__ type = a.cur.type;
    constexpr int NV = Z ? 3 : 2;
    float dv[NV];
#pragma unroll
    for (int c = 0; c < NV; ++c) dv[c] = acc[1 + c];
    sum_pairs<DIM, NL, L>(S, a, p, o, dv, [&](int j, float x, float y, float z, float r2, float,
                                              float (&t)[NV]) {
      if (type[j] != kRep) return no_terms(t);
      const float f = rep_fac(S, sqrtf(r2));
      t[0] = f * x;
      t[1] = f * y;
      if (Z) t[NV - 1] = f * z;
    });
#pragma unroll
    for (int c = 0; c < NV; ++c) acc[1 + c] = dv[c];
  }
}
template <int DIM, bool NL, bool SHEP, int KT, bool KC, int L>
__device__ __forceinline__ void wc_fluid_one(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  const float4 vi = a.cur.vtmp[p];
  const float pri = a.w.vp[p].w;
  float M[9];
  if (KC) corr_load(a.w.Lc, a.stride, p, M);
  constexpr int SH = SHEP ? 1 : 0;
  float sum[4 + SH] = {};  // d_density, d_vel, Shepard
  constexpr bool kFlat = DIM == 2 && NL;
  uint32_t odd = 0;
  if (kFlat) {
    float acc[3 + SH] = {};
    wc_fluid_sums<DIM, false, NL, SHEP, KT, KC, L>(a, S, p, o, vi, pri, M, acc, odd);
#pragma unroll
    for (int c = 0; c < 3; ++c) sum[c] = acc[c];
    if (SHEP) sum[3 + SH] = acc[2 + SH];
    odd |= __float_as_uint(vi.z);
  }
  // a lane has seen its own neighbours only: the quad's lanes go together
  // (exponents that only together have all bits cost the second sums' time)
  constexpr uint32_t kInf = 0x7F800000u;
  if (!kFlat || __any((odd & kInf) == kInf || !(fabsf(sum[1] + sum[2]) < INFINITY))) {
    float acc[4 + SH] = {};
    wc_fluid_sums<DIM, true, NL, SHEP, KT, KC, L>(a, S, p, o, vi, pri, M, acc, odd);
#pragma unroll
    for (int c = 0; c < 4 + SH; ++c) sum[c] = acc[c];
  }
  if (!group_head<L>()) return;
  a.w.drho[p] = sum[0] * vi.w;
  a.w.dv[p] = make_float4(sum[1] + S.grav[0], sum[2] + S.grav[1], sum[3] + S.grav[2], 0.0f);
  if (SHEP) a.w.cspm[p] = sum[3 + SH] != 0.0f ? 1.0f / sum[3 + SH] : 1.0f;
}

// d_vel of a dynamic rigid particle j: g (loop A, solver_sph_wc.py:105-106)
// minus the pair force of every fluid neighbour i (loop B, :68-71, where
// fluid i subtracts its calc_d_vel_task term from j).  The reference
// scatters with atomic updates in no fixed order; here j gathers the same
// terms, formed from i's side (x_ij = x_i - x_j, i's density_tmp in the
// wall viscosity), in its own neighbour order.
template <int DIM, bool NL, int KT, int L>
__device__ __forceinline__ float4 wc_rigid_force(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  const int8_t* __restrict__ type = a.cur.type;
  const float4* __restrict__ vtmp = a.cur.vtmp;
  const float4* __restrict__ vp = a.w.vp;
  const float4 vj = vtmp[p];
  const float mVj = o.P.w;
  const float prj = fabsf(vp[p].w);  // p_j / rho_j^2 of the wall record
  const float c1 = S.visc_c1, c2 = S.visc_c2, rho0 = S.rho0;
  float dv[3] = {S.grav[0], S.grav[1], S.grav[2]};
  sum_pairs<DIM, NL, L>(S, a, p, o, dv, [&](int i, float x, float y, float z, float r2, float,
                                            float (&t)[3]) {
    if (type[i] != kFluid) return no_terms(t);
    const float xi = -x, yi = -y, zi = -z;  // x_i - x_j
    const float rn = pair_dist(r2);
    const float f = kernel_gradfac_t<KT>(S, rn);
    const float gx = f * xi, gy = f * yi, gz = f * zi;
    const float4 vi = vtmp[i];
    const float ux = vi.x - vj.x, uy = vi.y - vj.y, uz = vi.z - vj.z;
    const float vx_ = ux * xi + uy * yi + uz * zi;
    const float mn = vx_ < 0.0f ? vx_ : 0.0f;
    const float rr = rho0 / vi.w;
    const float vis = ((c1 * mVj) * rr) * mn / (r2 + c2);
    const float pc = (-rho0 * mVj) * (vp[i].w + prj);
    const float sc = vis + pc;
    t[0] = -(sc * gx);
    t[1] = -(sc * gy);
    t[2] = -(sc * gz);
  });
  return make_float4(dv[0], dv[1], dv[2], 0.0f);
}

// Rates of other particles are never written by the reference: zero (by the
// step's first pass; again: a later one); a static rigid particle's d_vel is
// zero too (solver_sph_wc.py:125-126).
//
// The second sums of the 2D replay hardly ever run and may not cost the first
// their waves per SIMD (72 registers for seven, 96 for five).
constexpr int fluid_waves(int dim, bool nl, bool kc) {
  return dim == 3 || !nl ? 1 : (kc ? 5 : 7);
}
template <int DIM, bool NL, bool SHEP, bool KC>
__global__ __launch_bounds__(256, fluid_waves(DIM, NL, KC)) void k_wc_fluid(KArgs a, int again) {
  constexpr int L = NL ? kLanes : 1;
  for_work<NL, false>(
      a, again ? kTileFlow : ~0,
      [&](int s, int p, bool mine) {
        const int tp = a.cur.type[p];
        if (tp == kFluid) return true;
        if (tp == kRigid && rigid_slot(a.scenes[s], tp, a.cur.obj[p]) >= 0) return true;
        if (mine && !again) {
          a.w.drho[p] = 0.0f;
          a.w.dv[p] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        if (a.cur.type[p] == kRigid) {
          const float4 dv = S.kernel == 1 ? wc_rigid_force<DIM, NL, 1, L>(a, S, p, o)
                                          : wc_rigid_force<DIM, NL, 0, L>(a, S, p, o);
          if (!group_head<L>()) return;
          a.w.drho[p] = 0.0f;
          a.w.dv[p] = dv;
          return;
        }
        if (KC && S.kcorr != 0) {
          if (S.kernel == 1) wc_fluid_one<DIM, NL, SHEP, 1, true, L>(a, S, p, o);
          else wc_fluid_one<DIM, NL, SHEP, 0, true, L>(a, S, p, o);
        } else {
          if (S.kernel == 1) wc_fluid_one<DIM, NL, SHEP, 1, false, L>(a, S, p, o);
          else wc_fluid_one<DIM, NL, SHEP, 0, false, L>(a, S, p, o);
        }
      });
}

// ======================================================================= muI
// Velocity gradient L and d_density terms of a soil pair (calc_v_grad_task,
// d_density): t[0..8] = m_V (v_j - v_i) (x) grad W, t[9] = d_density.
__device__ __forceinline__ void soil_grad_terms(const float4& vi, const float4& vj, float mVj,
                                                const float gw[3], float* t) {
  const float u[3] = {mVj * (vj.x - vi.x), mVj * (vj.y - vi.y), mVj * (vj.z - vi.z)};
#pragma unroll
  for (int k = 0; k < 9; ++k) t[k] = u[k / 3] * gw[k % 3];
  t[9] = (mVj * (vi.x - vj.x)) * gw[0] + (mVj * (vi.y - vj.y)) * gw[1] +
         (mVj * (vi.z - vj.z)) * gw[2];
}

// stress_tmp of particle p and what the force pass takes from it, the
// quotients by density_tmp^2: formed here once per particle, not once per
// pair (six divisions each; the same quotients).  Both as records, two loads
// per neighbour instead of six or seven.  muI force pass: 108 -> 54 us at
// 120 k soil particles in 3D (wall pass 33 -> 26), 22 -> 14 us at 85 k in 2D;
// DP pass 35 -> 28 us at 85 k in 2D.
__device__ __forceinline__ void soil_stress_store(const KArgs& a, int p, const float (&sg)[6], float rt) {
  const float rt2 = rt * rt;
  float q[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) q[c] = sg[c] / rt2;
  rec6_store(a.w.sigt_f, p, sg);
  rec6_store(a.w.sigq, p, q, rt);
}

// Soil loop 1 (solver_sph_muI.py:200-225).
template <int DIM, bool NL, bool KC>
__device__ __forceinline__ void mui_soil1_one(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  constexpr int LN = NL ? kLanes : 1;
  const float4* __restrict__ vtmp = a.cur.vtmp;
  const float4 vi = vtmp[p];
  const bool kc = KC && S.kcorr != 0;
  float M[9];
  if (kc) corr_load(a.w.Lc, a.stride, p, M);
  float acc[10] = {};
  sum_pairs_k<DIM, NL, LN>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z, float r2,
                                                float mVj, float (&t)[10]) {
    const float f = kernel_gradfac_t<decltype(kt)::v>(S, pair_dist(r2));
    float gw[3] = {f * x, f * y, f * z};
    if (kc) corr_apply(M, gw);
    soil_grad_terms(vi, vtmp[j], mVj, gw, t);
  });
  if (!group_head<LN>()) return;
  const float L[3][3] = {{acc[0], acc[1], acc[2]}, {acc[3], acc[4], acc[5]}, {acc[6], acc[7], acc[8]}};
  const float dd = acc[9];
  a.w.drho[p] = dd * vi.w;
  float pp = S.vsound2 * (a.cur.vel[p].w - S.rho0);
  pp = pp > 0.0f ? pp : 0.0f;
  a.w.p[p] = pp;
  float e[3][3];
  float ss = 0.f;
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) e[aa][bb] = 0.5f * (L[aa][bb] + L[bb][aa]);
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) ss += e[aa][bb] * e[aa][bb];
  const float en = sqrtf(0.5f * ss) + S.eps;
  const float fac = 0.0f + (S.coh + pp * S.mu) / en;
  float sg[6];
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = aa; bb < 3; ++bb) sg[sidx(aa, bb)] = fac * e[aa][bb] - (aa == bb ? pp : 0.0f);
  soil_stress_store(a, p, sg, vi.w);
  const float tr3 = (e[0][0] + e[1][1] + e[2][2]) / 3.0f;
  float sd = 0.f;
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
      const float dlt = e[aa][bb] - (aa == bb ? tr3 : 0.0f);
      sd += dlt * dlt;
    }
  a.w.dseq[p] = (double)sqrtf(sd * 2.0f / 3.0f);
}
template <int DIM, bool NL, bool KC>
__global__ __launch_bounds__(256) void k_mui_soil1(KArgs a, int again) {
  for_work<NL, false>(
      a, again ? kTileFlow : ~0,
      [&](int, int p, bool mine) {
        if (a.cur.type[p] == kSoil) return true;
        if (mine && !again) {
          a.w.drho[p] = 0.0f;
          a.w.p[p] = 0.0f;
          a.w.dseq[p] = 0.0;
        }
        return false;
      },
      [&](int s, int p, const Own& o) { mui_soil1_one<DIM, NL, KC>(a, a.scenes[s], p, o); });
}

// Dummy loop of muI (:228-242) and DP (:220-231).
// acc: sums of the stress (6), v (3) and the density.
template <bool EXTRAP_DENSITY>
__device__ __forceinline__ void soil_wall_store(const KArgs& a, const SceneDev& S, int p, const float* acc) {
  const int st = a.stride;
  const float cs = a.w.cspm[p];
  const float4 v = a.cur.vel[p];
  float rt = S.rho0;
  if (EXTRAP_DENSITY) {
    const float r = acc[9] * cs;
    rt = r > S.rho0 ? r : S.rho0;
  }
  a.cur.vtmp[p] = make_float4(2.0f * v.x - acc[6] * cs, 2.0f * v.y - acc[7] * cs,
                              2.0f * v.z - acc[8] * cs, rt);
  float sg[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    sg[c] = acc[c] * cs;
    if (!EXTRAP_DENSITY) a.w.sigt_d[c * st + p] = (double)sg[c];
  }
  soil_stress_store(a, p, sg, rt);
}
template <int DIM, bool EXTRAP_DENSITY, bool NL>
__global__ __launch_bounds__(256) void k_soil_bdy(KArgs a, int again) {
  constexpr int L = NL ? kLanes : 1;
  const int8_t* __restrict__ type = a.cur.type;
  const float4* __restrict__ vtmp = a.cur.vtmp;
  const float* __restrict__ sgt = a.w.sigt_f;
  for_work<NL, true>(
      a, again ? kTileWall : kTileWall | kTileBare,
      [&](int s, int p, bool mine) {
        const int tp = type[p];
        if (!is_solid(tp)) return false;  // boundary and rigid (muI :96, DP :221)
        if (!NL || a.w.nlc[p] != 0) return true;
        if (mine && !(again && is_bdy(tp))) {  // as in k_wc_bdy
          const float none[10] = {};
          soil_wall_store<EXTRAP_DENSITY>(a, a.scenes[s], p, none);
        }
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        float acc[10] = {};
        // straight-line pair terms, as in k_wc_bdy
        sum_pairs_k<DIM, NL, L>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z, float r2,
                                                                float mVj, float (&t)[10]) {
          const bool fl = is_flow(type[j]);
          const float w = kernel_W_t<decltype(kt)::v>(S, pair_dist(r2));
          const float4 vj = vtmp[j];
          float sj[6];
          rec6_load(sgt, j, sj);
          const float xr[3] = {x, y, z};
#pragma unroll
          for (int c = 0; c < 3; ++c) t[c] = term_if(fl, mVj * (sj[c] + (vj.w * S.grav[c]) * xr[c]) * w);
#pragma unroll
          for (int c = 3; c < 6; ++c) t[c] = term_if(fl, mVj * sj[c] * w);
          t[6] = term_if(fl, mVj * vj.x * w);
          t[7] = term_if(fl, mVj * vj.y * w);
          t[8] = term_if(fl, mVj * vj.z * w);
          t[9] = term_if(fl, mVj * vj.w * w);
        });
        if (group_head<L>()) soil_wall_store<EXTRAP_DENSITY>(a, S, p, acc);
      });
}

// Acceleration from stress (muI :248-261; DP :260-270) + viscous damping
// (solver_sph_base.py:713-715).
// qi, qj: the stresses over their density_tmp^2; rtj: j's density_tmp.
__device__ __forceinline__ void soil_dv_pair(const float (&qi)[6], const float (&qj)[6], float mVj,
                                             float rtj, const float gw[3], float* t) {
  const float sc = mVj * rtj;
#pragma unroll
  for (int aa = 0; aa < 3; ++aa) {
    float acc = 0.f;
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
      const int c = sidx(aa, bb);
      acc += (sc * (qj[c] + qi[c])) * gw[bb];
    }
    t[aa] = acc;
  }
}

// d_vel of a dynamic rigid particle p of a soil scene: g (muI :111-112, DP
// :233-234) minus the calc_d_vel_from_stress_task term of every soil
// neighbour i (muI :38-46, DP :158-165), formed from i's side (x_ip, i's
// corrected gradient) and gathered in p's neighbour order (the reference
// subtracts them with atomic updates in no fixed order).
template <int DIM, bool NL, int KT, int L>
__device__ __forceinline__ float4 soil_rigid_force(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  const int8_t* __restrict__ type = a.cur.type;
  const float* __restrict__ sgq = a.w.sigq;
  const int st = a.stride;
  float qp[6];
  const float rtp = rec7_load(sgq, p, qp), mVp = o.P.w;
  const bool kc = S.kcorr != 0;
  float dv[3] = {S.grav[0], S.grav[1], S.grav[2]};
  sum_pairs<DIM, NL, L>(S, a, p, o, dv, [&](int i, float x, float y, float z, float r2, float,
                                            float (&t)[3]) {
    if (type[i] != kSoil) return no_terms(t);
    const float f = kernel_gradfac_t<KT>(S, pair_dist(r2));
    float gw[3] = {f * -x, f * -y, f * -z};
    if (kc) {
      float M[9];
      corr_load(a.w.Lc, st, i, M);
      corr_apply(M, gw);
    }
    float qi[6];
    rec6_load(sgq, i, qi);
    soil_dv_pair(qi, qp, mVp, rtp, gw, t);
#pragma unroll
    for (int c = 0; c < 3; ++c) t[c] = -t[c];
  });
  return make_float4(dv[0], dv[1], dv[2], 0.0f);
}
// The other particles of the soil force passes: zero rates, or the gathered
// force of a dynamic rigid particle (a static one keeps 0, muI :130-132, DP
// :272-274).
__device__ __forceinline__ bool soil_has_force(const KArgs& a, int s, int p) {
  const int tp = a.cur.type[p];
  return tp == kSoil || (tp == kRigid && rigid_slot(a.scenes[s], tp, a.cur.obj[p]) >= 0);
}
template <int DIM, bool NL, int L>
__device__ __forceinline__ float4 soil_nonsoil_dv(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  return S.kernel == 1 ? soil_rigid_force<DIM, NL, 1, L>(a, S, p, o)
                       : soil_rigid_force<DIM, NL, 0, L>(a, S, p, o);
}

__device__ __forceinline__ float4 soil_dv_finish(const SceneDev& S, const float dv[3], float4 vi) {
  const float damp = -5e-5f * sqrtf(S.young / (vi.w * S.h2));
  return make_float4(dv[0] + S.grav[0] + damp * vi.x, dv[1] + S.grav[1] + damp * vi.y,
                     dv[2] + S.grav[2] + damp * vi.z, 0.0f);
}

template <int DIM, bool NL, bool KC>
__device__ __forceinline__ void mui_soil3_one(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  constexpr int L = NL ? kLanes : 1;
  const float* __restrict__ sgq = a.w.sigq;
  const float4 vi = a.cur.vtmp[p];
  float qi[6];
  rec6_load(sgq, p, qi);
  float dv[3] = {};
  const bool kc = KC && S.kcorr != 0;
  float M[9];
  if (kc) corr_load(a.w.Lc, a.stride, p, M);
  sum_pairs_k<DIM, NL, L>(S, a, p, o, dv, [&](auto kt, int j, float x, float y, float z, float r2,
                                              float mVj, float (&t)[3]) {
    const float f = kernel_gradfac_t<decltype(kt)::v>(S, pair_dist(r2));
    float gw[3] = {f * x, f * y, f * z};
    if (kc) corr_apply(M, gw);
    float qj[6];
    const float rtj = rec7_load(sgq, j, qj);
    soil_dv_pair(qi, qj, mVj, rtj, gw, t);
  });
  if (S.rep) {
    // calc_rep_force_task (solver_sph_muI.py:34-36, 121-123), after the
    // stress forces and before gravity and damping
    const int8_t* __restrict__ type = a.cur.type;
    sum_pairs<DIM, NL, L>(S, a, p, o, dv, [&](int j, float x, float y, float z, float r2, float,
                                              float (&t)[3]) {
      if (type[j] != kRep) return no_terms(t);
      const float f = rep_fac(S, sqrtf(r2));
      t[0] = f * x;
      t[1] = f * y;
      t[2] = f * z;
    });
  }
  if (group_head<L>()) a.w.dv[p] = soil_dv_finish(S, dv, vi);
}
template <int DIM, bool NL, bool KC>
__global__ __launch_bounds__(256) void k_mui_soil3(KArgs a, int again) {
  constexpr int L = NL ? kLanes : 1;
  for_work<NL, false>(
      a, again ? kTileFlow : ~0,
      [&](int s, int p, bool mine) {
        if (soil_has_force(a, s, p)) return true;
        if (mine && !again) a.w.dv[p] = make_float4(0.f, 0.f, 0.f, 0.f);
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        if (a.cur.type[p] == kSoil) return mui_soil3_one<DIM, NL, KC>(a, S, p, o);
        const float4 d = soil_nonsoil_dv<DIM, NL, L>(a, S, p, o);
        if (group_head<L>()) a.w.dv[p] = d;
      });
}

// advect_something_func, muI (:267-289), phase 1 of D2.  The stress it sets
// to stress_tmp is read there by phase 2, which writes every soil particle's.
__global__ __launch_bounds__(256) void k_mui_adv1(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (a.cur.type[p] != kSoil) return;
  const SceneDev S = a.scenes[s];
  float4 v = a.cur.vel[p];
  v.w = v.w > S.rho0 ? v.w : S.rho0;
  a.cur.vel[p] = v;
  a.cur.pos[p].w = a.cur.mass[p] / v.w;
  a.cur.seq[p] = (double)((float)a.cur.seq[p] + S.dt * (float)a.w.dseq[p]);
}

// Phase 2 of D2: stress regularisation from the post-advect positions; the
// stencil centre is the cell of the new position, the pair vectors use the
// stored (pre-advect) cells.  The step's lists hold the pairs of the
// positions before, so the stencil is walked again: a quad of lanes per
// particle tests four candidates of a stencil column at a time (the cells of
// a column are adjacent in the particle order) and queues the hits in LDS,
// and the terms are formed from the queue, four entries at a time, in walk
// order.  (Formed where a candidate hits, they cost every candidate of the
// wave their time: one of sixteen particles' hits nearly always.)  It reads
// stress_tmp, which phase 1 makes the stress, and writes the stress.
// Bound: vector issue (66 % busy) and L1 data return (72 %), of ~730
// candidates per particle in 3D.  120 k soil particles in 3D (307 k with
// walls): 278 -> 193 us, 85 k in 2D: 41 -> 24 us, against a
// lane per particle with the terms where a candidate hits and a copy after.
// A queue of 16: 220 and 27 us; one quad of candidates per turn: 225 and 24.
constexpr int kReguQueue = 32;  // hits held per particle, a multiple of 4
struct ReguHit {
  int j;
  float r2;
};
// rows an odd number of entries apart: the quads' rows start in different banks
__device__ __forceinline__ ReguHit* regu_queue() {
  __shared__ ReguHit queue[kMaxBlock / 4 * (kReguQueue + 1)];
  return queue;
}
template <int DIM, int KT>
__device__ __forceinline__ void mui_regu_one(const KArgs& a, const SceneDev& S, int p) {
  ReguHit* __restrict__ queue = regu_queue() + (threadIdx.x >> 2) * (kReguQueue + 1);
  const float4 P = a.cur.pos[p];
  const float4* __restrict__ pos = a.cur.pos;
  const int32_t* __restrict__ start = a.w.start;
  const int8_t* __restrict__ type = a.cur.type;
  const float* __restrict__ sgt = a.w.sigt_f;
  const int st = a.stride;
  const int lane = (int)(threadIdx.x & 63), q = lane & 3, quad = lane & 28;
  const bool upper = lane >= 32;
  const float rs2 = S.rs2;
  const uint32_t below = (1u << q) - 1u;
  const int32_t shift = scene_shift(a, S);
  int cx, cy, cz;
  decode_cell(S, a.cur.cell[p], cx, cy, cz);
  int sx = cx, sy = cy, sz = cz;
  float tx = P.x, ty = P.y, tz = P.z;
  renorm(sx, tx, S.grid);
  renorm(sy, ty, S.grid);
  if (DIM == 3) renorm(sz, tz, S.grid);
  // the column's axis: z in 3D, y in 2D (one cell in z)
  const int cf = DIM == 3 ? cz : cy, gf = DIM == 3 ? S.gn[2] : S.gn[1];
  const int f0 = max((DIM == 3 ? sz : sy) - 1, 0), f1 = min((DIM == 3 ? sz : sy) + 1, gf - 1);
  const float of = DIM == 3 ? P.z : P.y;
  float b0 = of + (float)(cf - f0) * S.g;
  float b1 = of + (float)(cf - (f0 + 1)) * S.g;
  float b2 = of + (float)(cf - (f0 + 2)) * S.g;
  // kept, or they are formed again for every candidate
  asm("" : "+v"(b0), "+v"(b1), "+v"(b2));
  constexpr int U = DIM == 3 ? 2 : 1;  // quads of candidates per turn
  float acc[6] = {};
  int cnt = 0;
  // the terms of the first `n` queued hits (a multiple of 4, or all)
  auto drain = [&](int n) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int k = 0; k < n; k += 4) {
      const bool in = k + q < n;
      ReguHit h = queue[in ? k + q : 0];
      const bool same = in && h.j != p && type[h.j] == kSoil;
      const float mVj = pos[h.j].w;
      const float w = kernel_W_t<KT>(S, pair_dist(h.r2));
      float t[6];
      rec6_load(sgt, h.j, t);
#pragma unroll
      for (int c = 0; c < 6; ++c) t[c] = term_if(same, mVj * t[c] * w);
      ordered_add<4>(acc, t);
    }
  };
  if (f0 <= f1) {
#pragma unroll 1
    for (int k = 0; k < (DIM == 3 ? 9 : 3); ++k) {
      const int nx = sx + (DIM == 3 ? k / 3 : k) - 1, ny = DIM == 3 ? sy + k % 3 - 1 : 0;
      if (nx < 0 || nx >= S.gn[0] || (DIM == 3 && (ny < 0 || ny >= S.gn[1]))) continue;
      const float bx = P.x + (float)(cx - nx) * S.g;
      const float by = P.y + (float)(cy - ny) * S.g;  // 3D
      const int32_t* __restrict__ sk = start + S.cbase + (DIM == 3 ? (nx * S.gn[1] + ny) : nx) * gf + f0;
      const int nf = f1 - f0 + 1;
      const int32_t e1 = sk[1] + shift, e2 = sk[min(2, nf)] + shift, je = sk[nf] + shift;
      // up to seven records past the column are read (the state ends in a
      // tile of null particles)
      for (int32_t j = sk[0] + shift + q; j - q < je; j += 4 * U) {
        float4 pj[U];
#pragma unroll
        for (int u = 0; u < U; ++u) pj[u] = pos[j + 4 * u];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int32_t ju = j + 4 * u;
          float bf = b2;
          bf = ju < e2 ? b1 : bf;
          bf = ju < e1 ? b0 : bf;
          const float x = bx - pj[u].x;
          const float y = DIM == 3 ? by - pj[u].y : bf - pj[u].y;
          const float z = DIM == 3 ? bf - pj[u].z : 0.0f;
          const float r2 = fmaf(z, z, fmaf(y, y, x * x));
          const bool hit = ju < je && r2 < rs2;
          const uint64_t m = __builtin_amdgcn_ballot_w64(hit);
          const uint32_t half = upper ? (uint32_t)(m >> 32) : (uint32_t)m;
          const uint32_t four = (half >> quad) & 15u;
          if (hit) queue[cnt + __popc(four & below)] = {ju, r2};
          cnt += __popc(four);
        }
        if (__any(cnt > kReguQueue - 4 * U)) {
          const int full = cnt & ~3, rest = cnt & 3;
          drain(full);
          const ReguHit h = queue[min(full + q, kReguQueue)];
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          if (q < rest) queue[q] = h;
          cnt = rest;
        }
      }
    }
  }
  drain(cnt);
  if (q != 0) return;
  const float cs = a.w.cspm[p];
#pragma unroll
  for (int c = 0; c < 6; ++c) a.cur.sig_f[c * st + p] = acc[c] * cs;
}
// Four waves per tile; `flagged`: the tiles' flags are those of this step.
template <int DIM>
__global__ __launch_bounds__(256) void k_mui_regu(KArgs a, int flagged) {
  const int w = wave_id(), tile = w >> 2;
  if (flagged && (a.w.tflag[tile] & kTileFlow) == 0) return;
  const int2 t = a.tiles[tile];
  if (t.x < 0) return;
  const int s = __builtin_amdgcn_readfirstlane(t.x);
  const SceneDev& S = a.scenes[s];
  const int p = t.y + (w & 3) * 16 + (int)((threadIdx.x & 63) >> 2);
  if (p >= S.pbase + S.n || a.cur.type[p] != kSoil) return;
  if (S.kernel == 1) mui_regu_one<DIM, 1>(a, S, p);
  else mui_regu_one<DIM, 0>(a, S, p);
}

// ======================================================================== DP
struct Inv {
  double s[6], I1, sJ2, f;
};
__device__ __forceinline__ Inv dp_invariants(const SceneDev& S, const double st[6]) {
  Inv v;
  v.I1 = st[0] + st[1] + st[2];
  const double m = v.I1 / 3.0;
#pragma unroll
  for (int c = 0; c < 6; ++c) v.s[c] = st[c] - (c < 3 ? m : 0.0);
  double ss = 0.0;
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) ss += v.s[sidx(aa, bb)] * v.s[sidx(aa, bb)];
  v.sJ2 = sqrt(0.5 * ss);
  v.f = v.sJ2 + S.alpha * v.I1 - S.kc;
  return v;
}
// adapt_stress (solver_sph_dp.py:73-96), FP64.
__device__ __forceinline__ void dp_adapt(const SceneDev& S, double st[6]) {
  Inv v = dp_invariants(S, st);
  if (v.f > S.eps_f) {
    if (v.f > v.sJ2) {
      const double t = (v.I1 - S.kc / S.alpha) / 3.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) st[c] -= t;
    }
    v = dp_invariants(S, st);
    const double r = (-v.I1 * S.alpha + S.kc) / v.sJ2;
#pragma unroll
    for (int c = 0; c < 6; ++c) st[c] = r * v.s[c] + (c < 3 ? v.I1 / 3.0 : 0.0);
  }
}
__device__ __forceinline__ int dp_flag(const SceneDev& S, const double st[6]) {
  const Inv v = dp_invariants(S, st);
  if (v.f < -S.eps_f) return 0;
  if (v.f > S.eps_f) return v.f >= v.sJ2 ? 3 : 2;
  return 1;
}

// one_step loop 1 of particle p: stress_tmp t mapped back and stored; rt: its
// density_tmp.
__device__ __forceinline__ void dp_adapt_store(const KArgs& a, const SceneDev& S, int p, double (&t)[6], float rt) {
  dp_adapt(S, t);
  float sg[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) {
    a.w.sigt_d[c * a.stride + p] = t[c];
    sg[c] = (float)t[c];
  }
  soil_stress_store(a, p, sg, rt);
}
__global__ __launch_bounds__(256) void k_dp_adapt(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (a.cur.type[p] != kSoil) return;
  double t[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) t[c] = a.w.sigt_d[c * a.stride + p];
  dp_adapt_store(a, a.scenes[s], p, t, a.cur.vtmp[p].w);
}

// calc_d_stress_Bui2008 (solver_sph_dp.py:171-208), FP64.
__device__ void dp_bui2008(const SceneDev& S, const double L[3][3], const double st[6],
                           double ds_out[6], double& dseq, double& dseqp) {
  const Inv v = dp_invariants(S, st);
  double e[3][3], w[3][3], Sg[3][3], s3[3][3];
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
      e[aa][bb] = 0.5 * (L[aa][bb] + L[bb][aa]);
      w[aa][bb] = 0.5 * (L[aa][bb] - L[bb][aa]);
      Sg[aa][bb] = st[sidx(aa, bb)];
      s3[aa][bb] = v.s[sidx(aa, bb)];
    }
  const double tr = e[0][0] + e[1][1] + e[2][2];
  double ed[3][3];
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) ed[aa][bb] = e[aa][bb] - (aa == bb ? tr / 3.0 : 0.0);
  const bool plastic = v.f >= -S.eps_f && v.sJ2 > 1e-8;
  double lam = 0.0;
  if (plastic) {
    double se = 0.0;
#pragma unroll
    for (int aa = 0; aa < 3; ++aa)
#pragma unroll
      for (int bb = 0; bb < 3; ++bb) se += s3[aa][bb] * e[aa][bb];
    lam = (3.0 * S.alpha * S.K * tr + (S.G / v.sJ2) * se) /
          (27.0 * S.alpha * S.K * S.sin_psi + S.G);
  }
  double ds[3][3];
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
      const double J = Sg[aa][0] * w[bb][0] + Sg[aa][1] * w[bb][1] + Sg[aa][2] * w[bb][2] +
                       Sg[0][bb] * w[aa][0] + Sg[1][bb] * w[aa][1] + Sg[2][bb] * w[aa][2];
      const double gt =
          plastic ? lam * ((aa == bb ? 9.0 * S.K * S.sin_psi : 0.0) + S.G / v.sJ2 * s3[aa][bb])
                  : 0.0;
      ds[aa][bb] = J + (2.0 * S.G * ed[aa][bb] + (aa == bb ? S.K * tr : 0.0)) - gt;
    }
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = aa; bb < 3; ++bb) ds_out[sidx(aa, bb)] = ds[aa][bb];
  double sd = 0.0;
#pragma unroll
  for (int aa = 0; aa < 3; ++aa)
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) sd += ed[aa][bb] * ed[aa][bb];
  dseq = sqrt(sd * 2.0 / 3.0);
  dseqp = 0.0;
  if (plastic) {
    const double gp = v.sJ2 + 3.0 * v.I1 * S.sin_psi;
    double ep[3][3];
#pragma unroll
    for (int aa = 0; aa < 3; ++aa)
#pragma unroll
      for (int bb = 0; bb < 3; ++bb)
        ep[aa][bb] = (fabs(ds[aa][bb]) > 1e-8 ? gp / ds[aa][bb] : 0.0) * lam;
    const double t3 = (ep[0][0] + ep[1][1] + ep[2][2]) / 3.0;
    double q = 0.0;
#pragma unroll
    for (int aa = 0; aa < 3; ++aa)
#pragma unroll
      for (int bb = 0; bb < 3; ++bb) {
        const double d = ep[aa][bb] - (aa == bb ? t3 : 0.0);
        q += d * d;
      }
    dseqp = sqrt(q * 2.0 / 3.0);
  }
}

// DP soil loop (solver_sph_dp.py:237-270): velocity gradient, d_density
// and the stress acceleration in one walk, then the FP64 stress rate.
template <int DIM, bool NL, bool KC>
__device__ __forceinline__ void dp_soil_one(const KArgs& a, const SceneDev& S, int p, const Own& o) {
  constexpr int LN = NL ? kLanes : 1;
  const float4* __restrict__ vtmp = a.cur.vtmp;
  const float* __restrict__ sgq = a.w.sigq;
  const int st = a.stride;
  const float4 vi = vtmp[p];
  float qi[6];
  rec6_load(sgq, p, qi);
  const bool kc = KC && S.kcorr != 0;
  float M[9];
  if (kc) corr_load(a.w.Lc, a.stride, p, M);
  float acc[13] = {};  // velocity gradient (9), d_density, d_vel (3)
  sum_pairs_k<DIM, NL, LN>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z, float r2,
                                                float mVj, float (&t)[13]) {
    const float f = kernel_gradfac_t<decltype(kt)::v>(S, pair_dist(r2));
    float gw[3] = {f * x, f * y, f * z};
    if (kc) corr_apply(M, gw);
    const float4 vj = vtmp[j];
    soil_grad_terms(vi, vj, mVj, gw, t);
    float qj[6];
    rec6_load(sgq, j, qj);
    soil_dv_pair(qi, qj, mVj, vj.w, gw, t + 10);
  });
  if (!group_head<LN>()) return;
  const float dv[3] = {acc[10], acc[11], acc[12]};
#pragma unroll
  for (int c = 0; c < 9; ++c) a.w.gradv[c * a.stride + p] = acc[c];
  a.w.drho[p] = acc[9] * vi.w;
  a.w.dv[p] = soil_dv_finish(S, dv, vi);
}
// The stress rate of the velocity gradient that dp_soil_one() left, by a
// pass (or part of one) of a lane per particle: as the pair pass's epilogue a
// quarter of its lanes ran these ~500 FP64 instructions, at the registers
// they take (128, four waves per SIMD).  85 k in 2D: the pass 28 -> 21 us; in
// a fused step the rate joins the half step and the last update (3 us each)
// and the return mapping before it (8 us, twice) the pass ahead of it.
__device__ __forceinline__ void dp_rate(const KArgs& a, const SceneDev& S, int p, double (&ds)[6]) {
  const int st = a.stride;
  double Ld[3][3], sd[6], dq, dqp;
#pragma unroll
  for (int c = 0; c < 9; ++c) Ld[c / 3][c % 3] = (double)a.w.gradv[c * st + p];
#pragma unroll
  for (int c = 0; c < 6; ++c) sd[c] = a.w.sigt_d[c * st + p];
  dp_bui2008(S, Ld, sd, ds, dq, dqp);
#pragma unroll
  for (int c = 0; c < 6; ++c) a.w.dsig_d[c * st + p] = ds[c];
  a.w.dseq[p] = dq;
  a.w.dseqp[p] = dqp;
}
__global__ __launch_bounds__(256) void k_dp_rate(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (a.cur.type[p] != kSoil) return;
  double ds[6];
  dp_rate(a, a.scenes[s], p, ds);
}
template <int DIM, bool NL, bool KC>
__global__ __launch_bounds__(256) void k_dp_soil(KArgs a, int again) {
  constexpr int L = NL ? kLanes : 1;
  const int st = a.stride;
  auto other = [&](int p, const float4& d) {
    a.w.drho[p] = 0.0f;
    a.w.dv[p] = d;
#pragma unroll
    for (int c = 0; c < 6; ++c) a.w.dsig_d[c * st + p] = 0.0;
    a.w.dseq[p] = 0.0;
    a.w.dseqp[p] = 0.0;
  };
  for_work<NL, false>(
      a, again ? kTileFlow : ~0,
      [&](int s, int p, bool mine) {
        if (soil_has_force(a, s, p)) return true;
        if (mine && !again) other(p, make_float4(0.f, 0.f, 0.f, 0.f));
        return false;
      },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        if (a.cur.type[p] == kSoil) return dp_soil_one<DIM, NL, KC>(a, S, p, o);
        const float4 d = soil_nonsoil_dv<DIM, NL, L>(a, S, p, o);
        if (group_head<L>()) other(p, d);
      });
}

// advect_something_func, DP (:276-296).
__global__ __launch_bounds__(256) void k_dp_adv(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (a.cur.type[p] != kSoil) return;
  const SceneDev S = a.scenes[s];
  float4 v = a.cur.vel[p];
  v.w = v.w > S.rho0 ? v.w : S.rho0;
  a.cur.vel[p] = v;
  a.cur.pos[p].w = a.cur.mass[p] / v.w;
  const int st = a.stride;
  double t[6];
#pragma unroll
  for (int c = 0; c < 6; ++c) t[c] = a.cur.sig_d[c * st + p];
  a.cur.flag[p] = dp_flag(S, t);
  dp_adapt(S, t);
#pragma unroll
  for (int c = 0; c < 6; ++c) a.cur.sig_d[c * st + p] = t[c];
  a.cur.seq[p] += S.dt_d * a.w.dseq[p];
  a.cur.seqp[p] += S.dt_d * a.w.dseqp[p];
}

// =============================================================== integrators
// advect_LF_half (solver_sph_base.py:96-104).
// DPN: in a fused DP step, with the stress rate before and the return mapping
// of the next one_step after.
template <bool DPN>
__global__ __launch_bounds__(256) void k_lf_half(KArgs a, int eos) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  float rt = 0.0f;
  if (is_real(t)) {
    float4 vt = a.cur.vtmp[p];
    const float4 d = a.w.dv[p];
    vt.w += S.half_dt * a.w.drho[p];
    a.cur.pos[p].w = a.cur.mass[p] / vt.w;
    vt.x += S.half_dt * d.x;
    vt.y += S.half_dt * d.y;
    vt.z += S.half_dt * d.z;
    a.cur.vtmp[p] = vt;
    rt = vt.w;
    // the EOS of the next one_step (solver_sph_wc.py:88), fused
    if (eos && S.method == kWC && t == kFluid) {
      const float pv = wc_eos(S, vt.w);
      a.w.p[p] = pv;
      a.w.vp[p] = make_float4(vt.x, vt.y, vt.z, pv / (vt.w * vt.w));
    }
  }
  if (t == kSoil && S.method == kDP) {
    const int st = a.stride;
    const double h = 0.5 * S.dt_d;
    if (DPN) {
      double ds[6], q[6];
      dp_rate(a, S, p, ds);
      for (int c = 0; c < 6; ++c) q[c] = a.w.sigt_d[c * st + p] + h * ds[c];
      dp_adapt_store(a, S, p, q, rt);
    } else {
      for (int c = 0; c < 6; ++c) a.w.sigt_d[c * st + p] += h * a.w.dsig_d[c * st + p];
    }
  }
}

// advect_LF (:106-114); advect_SE (:79-87) is the same update.
// DPN: in a fused DP step, with the stress rate before.
template <bool DPN>
__global__ __launch_bounds__(256) void k_lf_full(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  if (is_real(t)) {
    float4 v = a.cur.vel[p];
    const float4 d = a.w.dv[p];
    v.w += S.dt * a.w.drho[p];
    a.cur.pos[p].w = a.cur.mass[p] / v.w;
    v.x += S.dt * d.x;
    v.y += S.dt * d.y;
    v.z += S.dt * d.z;
    a.cur.vel[p] = v;
    if (isnan(v.x) || isnan(v.y) || isnan(v.z) || isnan(v.w)) atomicAdd(&a.w.status[2 * s + 1], 1ull);
  }
  if (t == kSoil && S.method == kDP) {
    const int st = a.stride;
    double ds[6];
    if (DPN) dp_rate(a, S, p, ds);
#pragma unroll
    for (int c = 0; c < 6; ++c) a.cur.sig_d[c * st + p] += S.dt_d * (DPN ? ds[c] : a.w.dsig_d[c * st + p]);
  }
}

// End of step, fused: advect_LF (unless already run, XSPH case) ->
// advect_pos -> the elementwise part of advect_something (WC chk_density,
// DP return mapping, muI phase 1).  Same per-particle arithmetic as the
// separate passes.
// DPN: in a fused DP step, with the stress rate before.
template <bool DPN>
__global__ __launch_bounds__(256) void k_finish(KArgs a, int do_lf, int use_xsph) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  if (!is_real(t)) return;  // walls stay as they are (4.5 M particles, 1.65 M of them: 61 -> 50 us)
  const int st = a.stride;
  float4 v = a.cur.vel[p];
  float mv = a.cur.pos[p].w;
  if (do_lf) {
    const float4 d = a.w.dv[p];
    v.w += S.dt * a.w.drho[p];
    mv = a.cur.mass[p] / v.w;
    v.x += S.dt * d.x;
    v.y += S.dt * d.y;
    v.z += S.dt * d.z;
    if (isnan(v.x) || isnan(v.y) || isnan(v.z) || isnan(v.w)) atomicAdd(&a.w.status[2 * s + 1], 1ull);
    if (t == kSoil && S.method == kDP) {
      double ds[6];
      if (DPN) dp_rate(a, S, p, ds);
#pragma unroll
      for (int c = 0; c < 6; ++c) a.cur.sig_d[c * st + p] += S.dt_d * (DPN ? ds[c] : a.w.dsig_d[c * st + p]);
    }
  }
  float4 P = a.cur.pos[p];
  if (use_xsph && S.xsph) {
    const float4 xs = a.w.xs[p];
    P.x += S.dt * (v.x + 0.5f * xs.x);
    P.y += S.dt * (v.y + 0.5f * xs.y);
    P.z += S.dt * (v.z + 0.5f * xs.z);
  } else {
    P.x += S.dt * v.x;
    P.y += S.dt * v.y;
    P.z += S.dt * v.z;
  }
  if (S.dim == 2) P.z = 0.0f;
  if ((S.method == kWC && t == kFluid) || (S.method != kWC && t == kSoil)) {
    v.w = v.w > S.rho0 ? v.w : S.rho0;
    mv = a.cur.mass[p] / v.w;
  }
  P.w = mv;
  a.cur.vel[p] = v;
  a.cur.pos[p] = P;
  if (t != kSoil) return;
  if (S.method == kMUI) {
    a.cur.seq[p] = (double)((float)a.cur.seq[p] + S.dt * (float)a.w.dseq[p]);
  } else if (S.method == kDP) {
    double q[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) q[c] = a.cur.sig_d[c * st + p];
    a.cur.flag[p] = dp_flag(S, q);
    dp_adapt(S, q);
#pragma unroll
    for (int c = 0; c < 6; ++c) a.cur.sig_d[c * st + p] = q[c];
    a.cur.seq[p] += S.dt_d * a.w.dseq[p];
    a.cur.seqp[p] += S.dt_d * a.w.dseqp[p];
  }
}

// XSPH sum (solver_sph_base.py:223-226), from pre-advect positions (D3).
template <int DIM, bool NL>
__global__ __launch_bounds__(256) void k_xsph(KArgs a) {
  constexpr int L = NL ? kLanes : 1;
  const int8_t* __restrict__ type = a.cur.type;
  const float4* __restrict__ vel = a.cur.vel;
  for_work<NL, false>(
      a, kTileFlow, [&](int, int p, bool) { return is_real(type[p]); },
      [&](int s, int p, const Own& o) {
        const SceneDev S = a.scenes[s];
        const int ti = type[p];
        const float4 vi = vel[p];
        float acc[3] = {};
        sum_pairs_k<DIM, NL, L>(S, a, p, o, acc, [&](auto kt, int j, float x, float y, float z, float r2,
                                                                float mVj, float (&t)[3]) {
          // straight-line: a neighbour of another type adds +0
          const bool same = type[j] == ti;
          const float w = kernel_W_t<decltype(kt)::v>(S, pair_dist(r2));
          const float4 vj = vel[j];
          t[0] = term_if(same, mVj * (vj.x - vi.x) * w);
          t[1] = term_if(same, mVj * (vj.y - vi.y) * w);
          t[2] = term_if(same, mVj * (vj.z - vi.z) * w);
        });
        if (group_head<L>()) a.w.xs[p] = make_float4(acc[0], acc[1], acc[2], 0.f);
      });
}

// advect_pos (solver_sph_base.py:228-238): offsets move, cells are
// re-derived by the next hash.
__global__ __launch_bounds__(256) void k_advect_pos(KArgs a, int use_xsph) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (!is_real(a.cur.type[p])) return;
  const SceneDev S = a.scenes[s];
  const float4 v = a.cur.vel[p];
  float4 P = a.cur.pos[p];
  if (use_xsph && S.xsph) {
    const float4 xs = a.w.xs[p];
    P.x += S.dt * (v.x + 0.5f * xs.x);
    P.y += S.dt * (v.y + 0.5f * xs.y);
    P.z += S.dt * (v.z + 0.5f * xs.z);
  } else {
    P.x += S.dt * v.x;
    P.y += S.dt * v.y;
    P.z += S.dt * v.z;
  }
  if (S.dim == 2) P.z = 0.0f;
  a.cur.pos[p] = P;
}

// chk_density for fluid (WC advect_something, solver_sph_wc.py:129-133).
__global__ __launch_bounds__(256) void k_chk_density(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (a.cur.type[p] != kFluid) return;
  const SceneDev S = a.scenes[s];
  float4 v = a.cur.vel[p];
  v.w = v.w > S.rho0 ? v.w : S.rho0;
  a.cur.vel[p] = v;
  a.cur.pos[p].w = a.cur.mass[p] / v.w;
}

// enforce_boundary_2D/3D (solver_sph_base.py:540-601) for boundary == 1.
__global__ __launch_bounds__(256) void k_enforce_boundary(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  // judge_enforce_bdy (solver_sph_base.py:532-538): flow particles with the
  // collision boundary, dynamic rigid particles always
  const int t = a.cur.type[p];
  const bool dyn = rigid_slot(S, t, a.cur.obj[p]) >= 0;
  if (!((S.boundary == 1 && is_flow(t)) || dyn)) return;
  int cc[3];
  decode_cell(S, a.cur.cell[p], cc[0], cc[1], cc[2]);
  float4 P = a.cur.pos[p];
  float* o[3] = {&P.x, &P.y, &P.z};
  double pos[3];
  for (int ax = 0; ax < 3; ++ax)
    pos[ax] = (ax == 2 && S.dim == 2) ? 0.0 : S.vds[ax] + (double)cc[ax] * S.grid + (double)*o[ax];
  const double dist = S.radius - 1e-8;
  double nrm[3] = {0.0, 0.0, 0.0};
  auto setp = [&](int ax, double x) { *o[ax] = (float)(x - S.vds[ax] - (double)cc[ax] * S.grid); };
  if (pos[0] > S.dend[0] - dist) { nrm[0] += 1.0; setp(0, S.dend[0] - dist); }
  if (pos[0] <= S.dstart[0] + dist) { nrm[0] -= 1.0; setp(0, S.dstart[0] + dist); }
  if (pos[1] <= S.dstart[1] + dist) { nrm[1] -= 1.0; setp(1, S.dstart[1] + dist); }
  if (S.dim == 3) {
    if (pos[2] > S.dend[2] - dist) { nrm[2] += 1.0; setp(2, S.dend[2] - dist); }
    if (pos[2] <= S.dstart[2] + dist) { nrm[2] -= 1.0; setp(2, S.dstart[2] + dist); }
  }
  a.cur.pos[p] = P;
  const double len = sqrt(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
  if (len > 1e-8) {
    const float u[3] = {(float)(nrm[0] / len), (float)(nrm[1] / len), (float)(nrm[2] / len)};
    float4 v = a.cur.vel[p];
    const float k = 1.3f * (v.x * u[0] + v.y * u[1] + v.z * u[2]);
    v.x -= k * u[0];
    v.y -= k * u[1];
    v.z -= k * u[2];
    a.cur.vel[p] = v;
  }
}

// ======================================================================= RK4
// substep_RK (solver_sph_base.py:134-180).
__global__ __launch_bounds__(256) void k_rk_init(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const int t = a.cur.type[p];
  if (is_real(t)) {
    a.w.drho_rk[p] = 0.f;
    a.w.dv_rk[p] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  if (t == kSoil && a.w.dsig_rk) {  // DP
    const int st = a.stride;
    for (int c = 0; c < 6; ++c) a.w.dsig_rk[c * st + p] = 0.0;
  }
}
__global__ __launch_bounds__(256) void k_rk_update(KArgs a, int m) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  const float mf = (float)m;
  if (is_real(t)) {
    a.w.drho_rk[p] += a.w.drho[p] * mf;
    float4 r = a.w.dv_rk[p];
    const float4 d = a.w.dv[p];
    r.x += d.x * mf;
    r.y += d.y * mf;
    r.z += d.z * mf;
    a.w.dv_rk[p] = r;
  }
  if (t == kSoil && S.method == kDP) {
    const int st = a.stride;
    for (int c = 0; c < 6; ++c) a.w.dsig_rk[c * st + p] += a.w.dsig_d[c * st + p] * m;
  }
}
__global__ __launch_bounds__(256) void k_rk_advect4(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  if (is_real(t)) {
    const float4 v = a.cur.vel[p];
    const float4 d = a.w.dv[p];
    float4 vt;
    vt.w = S.half_dt * a.w.drho[p] + v.w;
    a.cur.pos[p].w = a.cur.mass[p] / vt.w;
    vt.x = S.half_dt * d.x + v.x;
    vt.y = S.half_dt * d.y + v.y;
    vt.z = S.half_dt * d.z + v.z;
    a.cur.vtmp[p] = vt;
  }
  if (t == kSoil && S.method == kDP) {
    const int st = a.stride;
    for (int c = 0; c < 6; ++c)
      a.w.sigt_d[c * st + p] = 0.5 * S.dt_d * a.w.dsig_d[c * st + p] + a.cur.sig_d[c * st + p];
  }
}
__global__ __launch_bounds__(256) void k_rk_advect(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  if (is_real(t)) {
    float4 v = a.cur.vel[p];
    const float4 d = a.w.dv_rk[p];
    v.w += S.dt6 * a.w.drho_rk[p];
    a.cur.pos[p].w = a.cur.mass[p] / v.w;
    v.x += S.dt6 * d.x;
    v.y += S.dt6 * d.y;
    v.z += S.dt6 * d.z;
    a.cur.vel[p] = v;
    // the NaN status of k_lf_full, for the RK4 update of the same state
    if (isnan(v.x) || isnan(v.y) || isnan(v.z) || isnan(v.w)) atomicAdd(&a.w.status[2 * s + 1], 1ull);
  }
  if (t == kSoil && S.method == kDP) {
    const int st = a.stride;
    for (int c = 0; c < 6; ++c)
      a.cur.sig_d[c * st + p] += S.dt_d / 6.0 * a.w.dsig_rk[c * st + p];
  }
}
// In a fused step, all that lies between one_step k (0..3) and the next: the
// update of the sums (0 + the first rates, as the passes one by one form it),
// the advance of v_tmp or, last, of v, and the EOS (DPN: the stress rate and
// the return mapping) around them.  Bound by launches at the sizes RK4 is
// used at: 4 of these in place of 13 launches (1 + 4 + 3 + 1 here, 4 EOS),
// 25 k particles in 2D 132 -> 113 us per step.
template <bool DPN>
__global__ __launch_bounds__(256) void k_rk_stage(KArgs a, int k) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  const int m = k == 1 || k == 2 ? 2 : 1;
  const float mf = (float)m;
  float rt = 0.0f;
  if (is_real(t)) {
    const float dr = a.w.drho[p];
    const float4 d = a.w.dv[p];
    float4 R = make_float4(0.f, 0.f, 0.f, 0.f);  // w: the density's
    if (k > 0) {
      R = a.w.dv_rk[p];
      R.w = a.w.drho_rk[p];
    }
    R.x += d.x * mf;
    R.y += d.y * mf;
    R.z += d.z * mf;
    R.w += dr * mf;
    float4 v = a.cur.vel[p];
    if (k < 3) {
      a.w.drho_rk[p] = R.w;
      a.w.dv_rk[p] = R;
      float4 vt;
      vt.w = S.half_dt * dr + v.w;
      a.cur.pos[p].w = a.cur.mass[p] / vt.w;
      vt.x = S.half_dt * d.x + v.x;
      vt.y = S.half_dt * d.y + v.y;
      vt.z = S.half_dt * d.z + v.z;
      a.cur.vtmp[p] = vt;
      rt = vt.w;
      if (S.method == kWC && t == kFluid) {
        const float pv = wc_eos(S, vt.w);
        a.w.p[p] = pv;
        a.w.vp[p] = make_float4(vt.x, vt.y, vt.z, pv / (vt.w * vt.w));
      }
    } else {
      v.w += S.dt6 * R.w;
      a.cur.pos[p].w = a.cur.mass[p] / v.w;
      v.x += S.dt6 * R.x;
      v.y += S.dt6 * R.y;
      v.z += S.dt6 * R.z;
      a.cur.vel[p] = v;
      if (isnan(v.x) || isnan(v.y) || isnan(v.z) || isnan(v.w)) atomicAdd(&a.w.status[2 * s + 1], 1ull);
    }
  }
  if (DPN && t == kSoil) {
    const int st = a.stride;
    double ds[6], q[6];
    dp_rate(a, S, p, ds);
#pragma unroll
    for (int c = 0; c < 6; ++c) {
      const double r = (k > 0 ? a.w.dsig_rk[c * st + p] : 0.0) + ds[c] * m;
      if (k < 3) {
        a.w.dsig_rk[c * st + p] = r;
        q[c] = 0.5 * S.dt_d * ds[c] + a.cur.sig_d[c * st + p];
      } else {
        a.cur.sig_d[c * st + p] += S.dt_d / 6.0 * r;
      }
    }
    if (k < 3) dp_adapt_store(a, S, p, q, rt);
  }
}

// Neighbour-set digest for tests: count, sum and sum of squares of the
// neighbours' id0 (for_all_neighbors membership, particle_system.py:268).
// only_slot < 0: every particle, output at its engine index; else only the
// particles of that slot, output at (index - base).
template <int DIM>
__global__ __launch_bounds__(256) void k_neighbor_stats(KArgs a, int32_t* __restrict__ cnt,
                                                        long long* __restrict__ s1,
                                                        long long* __restrict__ s2, int only_slot,
                                                        int32_t base) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  if (only_slot >= 0 && s != only_slot) return;
  const SceneDev S = a.scenes[s];
  const float4 P = a.cur.pos[p];
  const int32_t* __restrict__ id0 = a.cur.id0;
  int n = 0;
  long long a1 = 0, a2 = 0;
  walk_c<DIM>(S, a, p, P, [&](int j, float x, float y, float z, float r2, float mVj, int) {
    const long long id = id0[j];
    ++n;
    a1 += id;
    a2 += id * id;
  });
  const int o = p - base;
  cnt[o] = n;
  s1[o] = a1;
  s2[o] = a2;
}

// Exhaustive check of pair_dist against the correctly rounded sqrtf over
// the float bit patterns [lo, hi): out[0] counts differences at arguments
// >= 2^-96 (bit pattern 0x0F800000), out[1] results outside [0, 1e-8)
// below it.  Grid-stride over a fixed grid; no memory is read.
__global__ __launch_bounds__(256) void k_check_pair_dist(uint32_t lo, uint32_t hi,
                                                         unsigned long long* __restrict__ out) {
  const uint32_t stride = gridDim.x * blockDim.x;
  unsigned long long bad = 0, small = 0;
  for (uint64_t i = (uint64_t)lo + blockIdx.x * blockDim.x + threadIdx.x; i < hi; i += stride) {
    const float x = __uint_as_float((uint32_t)i);
    const float r = pair_dist(x);
    if (i >= 0x0F800000u) bad += __float_as_uint(r) != __float_as_uint(sqrtf(x));
    else small += !(r >= 0.0f && r < 1e-8f);
  }
  if (bad) atomicAdd(&out[0], bad);
  if (small) atomicAdd(&out[1], small);
}

// =================================================================== globals
// FP64 front / potential / kinetic / mass over flow particles.  Partials per
// 64-particle tile with a fixed shuffle tree, then one block per scene sums
// the scene's tiles in a fixed order: results do not depend on where the
// scene sits in the engine or on what else is resident.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmax(v, __shfl_xor(v, d, 64));
  return v;
}
__global__ __launch_bounds__(256) void k_globals_tile(KArgs a, int slot) {
  const SceneDev S = a.scenes[slot];
  const int k = wave_id();
  if (k >= S.n_tiles) return;
  const int w = S.tile_first + k;
  const int p = a.tiles[w].y + (int)(threadIdx.x & 63);
  double fr = -INFINITY, pe = 0.0, ke = 0.0, m = 0.0;
  if (p < S.pbase + S.n && is_flow(a.cur.type[p])) {
    int cc[3];
    decode_cell(S, a.cur.cell[p], cc[0], cc[1], cc[2]);
    const float4 P = a.cur.pos[p];
    const double x = S.vds[0] + (double)cc[0] * S.grid + (double)P.x;
    const double y = S.vds[1] + (double)cc[1] * S.grid + (double)P.y;
    const double z = S.dim == 3 ? S.vds[2] + (double)cc[2] * S.grid + (double)P.z : 0.0;
    const float4 v = a.cur.vel[p];
    const double mi = (double)a.cur.mass[p];
    fr = x;
    pe = mi * -((double)S.grav[0] * x + (double)S.grav[1] * y + (double)S.grav[2] * z);
    ke = 0.5 * mi * ((double)v.x * v.x + (double)v.y * v.y + (double)v.z * v.z);
    m = mi;
  }
  fr = wave_max(fr);
  pe = wave_sum(pe);
  ke = wave_sum(ke);
  m = wave_sum(m);
  if ((threadIdx.x & 63) == 0) {
    double* o = a.w.gpart + 4 * (size_t)w;
    o[0] = fr;
    o[1] = pe;
    o[2] = ke;
    o[3] = m;
  }
}
// out: the four, in pinned host memory.
__global__ __launch_bounds__(256) void k_globals_scene(KArgs a, int slot, double* __restrict__ out) {
  const SceneDev S = a.scenes[slot];
  double fr = -INFINITY, pe = 0.0, ke = 0.0, m = 0.0;
  for (int k = threadIdx.x; k < S.n_tiles; k += blockDim.x) {
    const double* o = a.w.gpart + 4 * (size_t)(S.tile_first + k);
    fr = fmax(fr, o[0]);
    pe += o[1];
    ke += o[2];
    m += o[3];
  }
  __shared__ double red[4][256 / 64];
  fr = wave_max(fr);
  pe = wave_sum(pe);
  ke = wave_sum(ke);
  m = wave_sum(m);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wid] = fr;
    red[1][wid] = pe;
    red[2][wid] = ke;
    red[3][wid] = m;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
      fr = fmax(fr, red[0][k]);
      pe += red[1][k];
      ke += red[2][k];
      m += red[3][k];
    }
    out[0] = fr;
    out[1] = pe;
    out[2] = ke;
    out[3] = m;
  }
}

// ============================================================== rigid bodies
// solve_rigid_body / solve_constraints (solver_sph_base.py:472-510): shape
// matching of every dynamic rigid object after advect_something, in FP64
// (the reference's default_fp): centre of mass cm = sum m x / sum m,
// A = sum m_V rho (x - cm) (x0 - cm0)^T, R the rotation of A's polar
// decomposition, then x += (cm + R (x0 - cm0) - x).  One pass of per-tile
// partial sums (sum m, m x, w x q^T, w q with w = m_V rho, q = x0 - cm0;
// A = sum w x q^T - cm (sum w q)^T), one block per object in a fixed order,
// then the per-particle move.
__device__ __forceinline__ void abs_position(const SceneDev& S, int32_t cell, const float4& P,
                                             double x[3]) {
  int cc[3];
  decode_cell(S, cell, cc[0], cc[1], cc[2]);
  x[0] = S.vds[0] + (double)cc[0] * S.grid + (double)P.x;
  x[1] = S.vds[1] + (double)cc[1] * S.grid + (double)P.y;
  x[2] = S.dim == 3 ? S.vds[2] + (double)cc[2] * S.grid + (double)P.z : 0.0;
}
constexpr int kRigidSums = 16;
__global__ __launch_bounds__(256) void k_rigid_tile(KArgs a) {
  const int w = wave_id();
  const int2 t = a.tiles[w];
  if (t.x < 0) return;
  const SceneDev S = a.scenes[t.x];
  if (S.nrig == 0) return;  // wave-uniform
  const int lane = (int)(threadIdx.x & 63);
  const int p = t.y + lane;
  int k = -1;
  double v[kRigidSums];
  for (int c = 0; c < kRigidSums; ++c) v[c] = 0.0;
  if (p < S.pbase + S.n) k = rigid_slot(S, a.cur.type[p], a.cur.obj[p]);
  if (k >= 0) {
    double x[3];
    const float4 P = a.cur.pos[p];
    abs_position(S, a.cur.cell[p], P, x);
    const double m = (double)a.cur.mass[p];
    const double wv = (double)P.w * (double)a.cur.vel[p].w;
    const size_t id = (size_t)S.pbase + (size_t)a.cur.id0[p];
    const int st = a.stride;
    double q[3];
    // the initial centre read from the scene table (a runtime index into
    // the local copy S would put S on the stack)
    const double* cm0 = a.scenes[t.x].rig_cm0[k];
    for (int c = 0; c < 3; ++c) q[c] = a.w.x0[(size_t)c * st + id] - cm0[c];
    v[0] = m;
    for (int c = 0; c < 3; ++c) v[1 + c] = m * x[c];
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c) v[4 + 3 * r + c] = wv * x[r] * q[c];
    for (int c = 0; c < 3; ++c) v[13 + c] = wv * q[c];
  }
  for (int o = 0; o < S.nrig; ++o) {
    double* out = a.w.rigpart + ((size_t)w * kMaxRigid + o) * kRigidSums;
    const bool any = __any(k == o);
    for (int c = 0; c < kRigidSums; ++c) {
      double u = (k == o) ? v[c] : 0.0;
      if (any) u = wave_sum(u);
      if (lane == 0) out[c] = any ? u : 0.0;
    }
  }
}

// Orthogonal factor of the polar decomposition A = R S.  2D (the xy block;
// R_zz = 1): the nearest rotation, (a + d, c - b) normalised.  3D: Newton's
// iteration X <- (X + X^-T) / 2 (Higham 1986) from X = A.  A singular A
// gives I.
__device__ __forceinline__ void polar_rotation(const double A[9], int dim, double R[9]) {
  for (int c = 0; c < 9; ++c) R[c] = (c % 4 == 0) ? 1.0 : 0.0;
  if (dim == 2) {
    const double s = A[0] + A[4], t = A[3] - A[1];
    const double nrm = sqrt(s * s + t * t);
    if (nrm == 0.0) return;
    R[0] = s / nrm;
    R[1] = -t / nrm;
    R[3] = t / nrm;
    R[4] = s / nrm;
    return;
  }
  double X[9];
  for (int c = 0; c < 9; ++c) X[c] = A[c];
  for (int it = 0; it < 100; ++it) {
    // cofactors: X^-T = cof(X) / det(X)
    double cf[9];
    cf[0] = X[4] * X[8] - X[5] * X[7];
    cf[1] = X[5] * X[6] - X[3] * X[8];
    cf[2] = X[3] * X[7] - X[4] * X[6];
    cf[3] = X[2] * X[7] - X[1] * X[8];
    cf[4] = X[0] * X[8] - X[2] * X[6];
    cf[5] = X[1] * X[6] - X[0] * X[7];
    cf[6] = X[1] * X[5] - X[2] * X[4];
    cf[7] = X[2] * X[3] - X[0] * X[5];
    cf[8] = X[0] * X[4] - X[1] * X[3];
    const double det = X[0] * cf[0] + X[1] * cf[1] + X[2] * cf[2];
    if (det == 0.0) return;
    double d = 0.0;
    for (int c = 0; c < 9; ++c) {
      const double xn = 0.5 * (X[c] + cf[c] / det);
      const double e = fabs(xn - X[c]);
      d = e > d ? e : d;
      X[c] = xn;
    }
    if (d <= 1e-15) break;
  }
  for (int c = 0; c < 9; ++c) R[c] = X[c];
}

__global__ __launch_bounds__(256) void k_rigid_solve(KArgs a, int nslots) {
  const int s = blockIdx.x / kMaxRigid, o = blockIdx.x % kMaxRigid;
  if (s >= nslots) return;
  const SceneDev S = a.scenes[s];
  if (!S.active || o >= S.nrig) return;
  double v[kRigidSums];
  for (int c = 0; c < kRigidSums; ++c) v[c] = 0.0;
  for (int k = threadIdx.x; k < S.n_tiles; k += blockDim.x) {
    const double* in = a.w.rigpart + ((size_t)(S.tile_first + k) * kMaxRigid + o) * kRigidSums;
    for (int c = 0; c < kRigidSums; ++c) v[c] += in[c];
  }
  __shared__ double red[kRigidSums][256 / 64];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  for (int c = 0; c < kRigidSums; ++c) {
    v[c] = wave_sum(v[c]);
    if (lane == 0) red[c][wid] = v[c];
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int c = 0; c < kRigidSums; ++c)
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) v[c] += red[c][k];
  double cm[3], A[9], R[9];
  for (int c = 0; c < 3; ++c) cm[c] = v[1 + c] / v[0];
  for (int r = 0; r < 3; ++r)
    for (int c = 0; c < 3; ++c) A[3 * r + c] = v[4 + 3 * r + c] - cm[r] * v[13 + c];
  polar_rotation(A, S.dim, R);
  double* out = a.w.rigout + ((size_t)s * kMaxRigid + o) * 12;
  for (int c = 0; c < 3; ++c) out[c] = cm[c];
  for (int c = 0; c < 9; ++c) out[3 + c] = R[c];
}

__global__ __launch_bounds__(256) void k_rigid_apply(KArgs a) {
  int s, p;
  if (!tile_thread(a, s, p)) return;
  const SceneDev S = a.scenes[s];
  const int k = rigid_slot(S, a.cur.type[p], a.cur.obj[p]);
  if (k < 0) return;
  const double* cr = a.w.rigout + ((size_t)s * kMaxRigid + k) * 12;
  const size_t id = (size_t)S.pbase + (size_t)a.cur.id0[p];
  const int st = a.stride;
  double q[3], x[3];
  const double* cm0 = a.scenes[s].rig_cm0[k];  // as in k_rigid_tile
  for (int c = 0; c < 3; ++c) q[c] = a.w.x0[(size_t)c * st + id] - cm0[c];
  float4 P = a.cur.pos[p];
  abs_position(S, a.cur.cell[p], P, x);
  int cc[3];
  decode_cell(S, a.cur.cell[p], cc[0], cc[1], cc[2]);
  float o[3] = {P.x, P.y, P.z};
#pragma unroll
  for (int r = 0; r < 3; ++r) {  // constant indices: no stack array
    if (r >= S.dim) continue;
    const double goal = cr[r] + (cr[3 + 3 * r] * q[0] + cr[4 + 3 * r] * q[1] + cr[5 + 3 * r] * q[2]);
    const double xn = x[r] + (goal - x[r]) * 1.0;
    o[r] = (float)(xn - S.vds[r] - (double)cc[r] * S.grid);
  }
  P.x = o[0];
  P.y = o[1];
  P.z = o[2];
  a.cur.pos[p] = P;
}

// ============================================================== colour feed
// assign_value_color (solver_sph_base.py:721-789): the colour value of one
// colorTitle in FP64 (the reference's default_fp), for real particles and,
// with show_bdy, dummy particles; 0 for the rest.
__device__ __forceinline__ double norm3(double x, double y, double z) {
  return sqrt(x * x + y * y + z * z);
}
// SplitMix64 (Steele, Lea & Flood, OOPSLA 2014) of (seed, id0) -> [0, 1),
// standing in for ti.random() of title 101.
__device__ __forceinline__ double uniform01(uint32_t seed, int32_t id) {
  uint64_t z = ((uint64_t)seed << 32 | (uint32_t)id) + 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z ^= z >> 31;
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}
__global__ __launch_bounds__(256) void k_color_val(KArgs a, int slot, int title, int show_bdy,
                                                   uint32_t seed) {
  int s, p;
  if (!tile_thread(a, s, p) || s != slot) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  double v = 0.0;
  if (is_real(t) || (show_bdy && t == kDummy)) {
    const int st = a.stride;
    auto stress = [&](int c) -> double {
      if (a.cur.sig_d) return a.cur.sig_d[c * st + p];
      if (a.cur.sig_f) return (double)a.cur.sig_f[c * st + p];
      return 0.0;  // WC: the fluid's stress field stays zero
    };
    auto position = [&](double x[3]) {
      int cc[3];
      decode_cell(S, a.cur.cell[p], cc[0], cc[1], cc[2]);
      const float4 P = a.cur.pos[p];
      x[0] = S.vds[0] + (double)cc[0] * S.grid + (double)P.x;
      x[1] = S.vds[1] + (double)cc[1] * S.grid + (double)P.y;
      x[2] = S.dim == 3 ? S.vds[2] + (double)cc[2] * S.grid + (double)P.z : 0.0;
    };
    const float4 vel = a.cur.vel[p];
    const float4 dv = a.w.dv[p];
    double x[3];
    switch (title) {
      case 1: v = (double)a.cur.id0[p]; break;
      case 2: v = (double)vel.w; break;
      case 21: v = (double)a.w.drho[p]; break;
      case 3: v = norm3(vel.x, vel.y, vel.z); break;
      case 31: v = (double)vel.x; break;
      case 32: v = -(double)vel.y; break;
      case 33: v = (double)vel.z; break;
      case 34: v = norm3(dv.x, dv.y, dv.z); break;
      case 35: v = (double)dv.x; break;
      case 36: v = (double)dv.y; break;
      case 37: v = (double)dv.z; break;
      case 4: position(x); v = norm3(x[0], x[1], x[2]); break;
      case 41: position(x); v = x[0]; break;
      case 42: position(x); v = x[1]; break;
      case 43: position(x); v = x[2]; break;
      case 44: {
        position(x);
        const size_t k = (size_t)S.pbase + (size_t)a.cur.id0[p];
        v = norm3(x[0] - a.w.x0[k], x[1] - a.w.x0[st + k], x[2] - a.w.x0[2 * (size_t)st + k]);
        break;
      }
      case 51: v = stress(0); break;
      case 52: v = -stress(1); break;
      case 53: v = -stress(2); break;
      case 54: v = stress(3); break;
      case 55: v = stress(4); break;
      case 56: v = stress(5); break;
      case 57: v = -(stress(0) + stress(1) + stress(2)) / 3.0; break;
      case 61: v = a.cur.seq ? a.cur.seq[p] : 0.0; break;
      case 62: v = a.cur.seqp ? a.cur.seqp[p] : 0.0; break;
      case 7: v = (double)a.w.p[p]; break;
      case 8: v = a.cur.flag ? (double)a.cur.flag[p] : 0.0; break;
      case 100: v = (double)a.cur.cell[p]; break;
      case 101: v = uniform01(seed, a.cur.id0[p]); break;
      case 102: v = S.kcorr == 1 ? (double)a.w.Lc[p] : 0.0; break;
      case 103: {
        const float4 vt = a.cur.vtmp[p];
        v = norm3(vt.x, vt.y, vt.z);
        break;
      }
      default: v = 0.0;
    }
  }
  a.w.val[p] = v;
}

// v_maxmin (particle_system.py:387-397): max / min of val over flow
// particles; per-tile partials, then one block per scene, then the
// givenMax / givenMin / fixMax / fixMin rule.  max / min do not depend on the
// reduction order.
__device__ __forceinline__ double wave_min(double v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmin(v, __shfl_xor(v, d, 64));
  return v;
}
__global__ __launch_bounds__(256) void k_color_range_tile(KArgs a, int slot) {
  const int w = wave_id();
  const int2 t = a.tiles[w];
  if (t.x != slot) return;  // wave-uniform
  const SceneDev S = a.scenes[t.x];
  const int p = t.y + (int)(threadIdx.x & 63);
  double hi = -INFINITY, lo = INFINITY;
  if (p < S.pbase + S.n && is_flow(a.cur.type[p])) hi = lo = a.w.val[p];
  hi = wave_max(hi);
  lo = wave_min(lo);
  if ((threadIdx.x & 63) == 0) {
    a.w.gpart[4 * (size_t)w] = hi;
    a.w.gpart[4 * (size_t)w + 1] = lo;
  }
}
__global__ __launch_bounds__(256) void k_color_range_scene(KArgs a, int slot, double given_max,
                                                           double given_min, int fix_max,
                                                           int fix_min, double* __restrict__ out) {
  const SceneDev S = a.scenes[slot];
  double hi = -INFINITY, lo = INFINITY;
  for (int k = threadIdx.x; k < S.n_tiles; k += blockDim.x) {
    const double* o = a.w.gpart + 4 * (size_t)(S.tile_first + k);
    hi = fmax(hi, o[0]);
    lo = fmin(lo, o[1]);
  }
  __shared__ double red[2][256 / 64];
  hi = wave_max(hi);
  lo = wave_min(lo);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wid] = hi;
    red[1][wid] = lo;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) {
      hi = fmax(hi, red[0][k]);
      lo = fmin(lo, red[1][k]);
    }
    // vmax if givenmax == -1 or (vmax < givenmax and not fixmax) else givenmax
    const double vmax = (given_max == -1.0 || (hi < given_max && !fix_max)) ? hi : given_max;
    const double vmin = (given_min == -1.0 || (lo > given_min && !fix_min)) ? lo : given_min;
    a.w.crange[2 * slot] = out[0] = vmax;
    a.w.crange[2 * slot + 1] = out[1] = vmin;
  }
}

// set_color (particle_system.py:399-407) with the jet map of colormap.py:
// map(x) = clamp((w - |clamp(x) - c|) / w * h), w = wl below c, wr above,
// clamp to [0, 1]; (h, wl, wr, c) = (1.5, .37, .37, .75 / .5 / .25) for
// R / G / B.  FP64 as the reference's Python constants, stored as f32.
__device__ __forceinline__ double clamp01(double x) { return fmax(0.0, fmin(1.0, x)); }
__device__ __forceinline__ double jet_channel(double x, double c) {
  const double h = 1.5, wl = 0.37, wr = 0.37;
  const double w = x < c ? wl : wr;
  return clamp01((w - fabs(clamp01(x) - c)) / w * h);
}
__global__ __launch_bounds__(256) void k_set_color(KArgs a, int slot, int group, int show_bdy) {
  int s, p;
  if (!tile_thread(a, s, p) || s != slot) return;
  const SceneDev S = a.scenes[s];
  const int t = a.cur.type[p];
  const bool member = (group == 0 && is_flow(t)) || (group == 1 && is_real(t)) ||
                      (group == 2 && (is_real(t) || (show_bdy && t == kDummy)));
  float4 c;
  if (member) {
    const double vmax = a.w.crange[2 * slot], vmin = a.w.crange[2 * slot + 1];
    const double vrange1 = 1.0 / (vmax - vmin);
    const double x = (a.w.val[p] - vmin) * vrange1;
    c = make_float4((float)jet_channel(x, 0.75), (float)jet_channel(x, 0.5),
                    (float)jet_channel(x, 0.25), 0.0f);
  } else {
    c = a.w.c0[(size_t)S.pbase + (size_t)a.cur.id0[p]];
  }
  a.w.rgb[p] = c;
}

// ================================================================= read-out
// A field of one scene in the layout its caller reads: `comps` values per
// particle, double or int32.  Written straight into pinned host memory, in
// whole lines; the reads are of the engine's own layout.
enum PackKind { kPackF4, kPackPos, kPackF, kPackD, kPackI, kPackB, kPackRec, kPackStart };
struct Pack {
  const void* src;      // the scene's first entry
  const int32_t* cell;  // kPackPos
  int kind, comps;
  int lane0;            // kPackF4: first of the float4's
  int64_t st;           // kPackF, kPackD: stride between the components
  int dim, gn1, gn2;    // kPackPos
  double vds[3], grid;
};
__global__ __launch_bounds__(256) void k_pack(Pack k, int64_t first, int m, void* __restrict__ out) {
  const int e = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (e >= m) return;
  const int q = e / k.comps, c = e - q * k.comps;
  const int64_t i = first + q;
  double v = 0.0;
  switch (k.kind) {
    case kPackF4: v = (double)((const float*)k.src)[4 * i + k.lane0 + c]; break;
    case kPackPos: {
      const int32_t key = k.cell[i];
      const int yz = k.gn1 * k.gn2;
      const int x = key / yz, y = (key - x * yz) / k.gn2, z = key - x * yz - y * k.gn2;
      const int cc = c == 0 ? x : (c == 1 ? y : z);
      if (!(c == 2 && k.dim == 2)) v = k.vds[c] + (double)cc * k.grid + (double)((const float*)k.src)[4 * i + c];
      break;
    }
    case kPackF: v = (double)((const float*)k.src)[c * k.st + i]; break;
    case kPackD: v = ((const double*)k.src)[c * k.st + i]; break;
    case kPackRec: v = (double)((const float*)k.src)[kRec * i + c]; break;
    case kPackI: ((int32_t*)out)[e] = ((const int32_t*)k.src)[i]; return;
    case kPackB: ((int32_t*)out)[e] = ((const int8_t*)k.src)[i]; return;
    case kPackStart: ((int32_t*)out)[e] = ((const int32_t*)k.src)[i] - ((const int32_t*)k.src)[0]; return;
  }
  ((double*)out)[e] = v;
}

}  // namespace tsph
