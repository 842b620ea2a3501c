// pbf_tiles.h -- list passes over LDS tiles (included by pbf_kernels.hip).
//
// What bounds the per-lane list passes of a chip-filling state is the path of
// their gathers through the L1: a wave-wide gather touches ~41 cache lines, a
// λ launch of 4,096,000 particles 112M of them, nearly one per cycle and CU,
// while its arithmetic alone would take ~130 us of the 244.  Here a workgroup
// takes the particles of a block of 5 x 4 x 3 cells (~480 at rest, 7.5 waves of
// 8), copies the records of the block and of the cells around it (7 x 6 x 5,
// ~1,690 records of 16 bytes) into LDS, row by row and coalesced, and gathers
// from there: one 16-byte LDS read per neighbour.  A compact block is what
// makes that fit: the same particles taken in row order have 9.8 records of
// halo each instead of 3.5.  The lists hold LDS byte offsets, 16 bits per
// entry, so each pass also reads half the list bytes.  The memory order of
// the particles, their cells and the order of every list stay as they are,
// and with them every bit of the result.
//
// Measured, 4,096,000 particles at rest density (steps 1-20; per-lane passes /
// tiles, us per launch): build + first λ 927 / 670, λ 244 / 193, delta-p
// 275 / 209, XSPH 440 / 262, vorticity + next prediction 377 / 260, sort (with
// the tiles laid out) 117 / 135; the step 3.71 / 2.77 ms, over the whole run
// through both impacts 3.99 / 3.24.  1,000,000 particles 0.95 / 0.76 ms,
// 400,000 0.451 / 0.417, 300,000 0.341 / 0.345: below ~350,000 there are too few
// blocks for the card's 256 CUs (Ctx::tile_min).
//
// What a λ launch still spends: ~58 us on filling the tiles (latency: record
// of the tile, rows, barrier), ~30 us on LDS bank conflicts, the rest on the
// arithmetic of its pairs.  Tried and slower: blocks of 5 x 3 x 2 cells with 256
// threads (the same within 2%), quads in LDS tiles for mid-size and dense
// states (λ at 70,000 particles 15.3 us against 13.2, the compressed dam break
// 98 against 67), the next tile's rows prefetched into registers, and the
// prediction fused into the vorticity pass (the waves of a tile then wait for
// histogram atomics while they hold its LDS: 288 us against 260).
//
// Blocks that do not fit (more than kTileCap - 1 records) are cut into parts,
// level after level.  Particles of sparse blocks (fewer than kTileMin) go to a
// queue that workgroups without a tile take, a lane per particle, with the
// per-lane passes' lists and gathers; those of blocks that fit at no level, and
// particles whose cell or list stands out of its tile, to the queue of the
// dense split, a quad per particle.
#pragma once

constexpr int kTX = 5, kTY = 4, kTZ = 3;   // cells of a block
constexpr int kTRY = kTY + 2, kTRows = kTRY * (kTZ + 2);
constexpr int kTileBlock = 512;
constexpr uint32_t kTileWaves = kTileBlock / 64;
// Records of a tile, the padding record included: 40 KB of 16-byte records,
// so four workgroups (all 32 waves) share a CU's 160 KB.
constexpr uint32_t kTileCap = 2556;
// Particles of a tiled block: below, a workgroup's fill and its idle waves cost
// more than a lane per particle with global gathers (1,000,000 particles, ms per
// step, per-lane passes / this line / 24: random at 20 a block 0.34 / 0.42 / 1.04,
// at 100 0.50 / 0.61 / 1.07, at 200 0.64 / 0.80 / 0.80, at 480 0.98 / 0.74 / 0.74;
// the dam's first and last 30 of 120 steps 0.94, 1.40 / 0.75, 1.35 / 0.75, 1.39;
// lines of 200 and 256 are slower at 480 a block, 0.78 and 0.80).
constexpr uint32_t kTileMin = 128;
constexpr uint32_t kTileFew = 24;  // sparse blocks that one thread stores
// Particles from which a block is worth its tile in a state full of its like
// (Ctx::tile_sparse).
constexpr uint32_t kTileFull = 300;
constexpr int kTileLevels = 6;
constexpr unsigned kTileQuads = 256;      // workgroups of a pass that take the queue
constexpr unsigned kQueueBuildGrid = 2048;
constexpr uint32_t kTileRun = 8;          // consecutive tiles per XCD
// How far above its tile's mean a cell or list may stand before its particles
// go to the queue (measured, 1,000,000-particle dam over 150 steps, whose
// column compresses: 1.49 ms per step without, 1.24 at 2.5, 1.23 at 4, 1.29
// at 6; the 4,096,000-particle run 3.20, 3.36, 3.24, 3.24).
constexpr float kTileSpike = 4.0f;
// Cells up to kTileCrowd and lists up to kTileLong never stand out.
constexpr uint32_t kTileCrowd = 32, kTileLong = 128;
static_assert(kTRows <= kTileRows && kTX <= 5 && kTX * kTY * kTZ <= 64 && kTileCap <= 4096 &&
                  kTileMin <= 128,
              "tile");

__device__ __forceinline__ uint32_t tile_blocks(const SceneGrid& g, uint32_t* nbx, uint32_t* nby) {
  *nbx = (uint32_t)(g.dims[0] + kTX - 1) / kTX;
  *nby = (uint32_t)(g.dims[1] + kTY - 1) / kTY;
  return *nbx * *nby * ((uint32_t)(g.dims[2] + kTZ - 1) / kTZ);
}

// Cells of the parts of a block at a level.
__device__ __forceinline__ void tile_sub(int level, int* sx, int* sy, int* sz) {
  *sx = level <= 3 ? kTX : (level == 4 ? (kTX + 1) / 2 : 1);
  *sy = level <= 1 ? kTY : (level == 2 && kTY % 2 == 0 ? kTY / 2 : 1);
  *sz = level == 0 ? kTZ : 1;
}

// The tiles of the step: a thread per base block.  Most blocks fit as a
// whole; the lanes of a wave size the others together, block by block: every
// lane takes one part, level after level of finer parts, until all parts of
// a level fit.  A block's parts take consecutive items and units.
struct TileParts {
  int level;
  int px, py, pz, sx, sy, sz;  // this lane's part
  uint32_t pn;                 // its particles (0: none)
};
__device__ __forceinline__ TileParts tile_parts(const TileDev& d, const SceneGrid& g, int x0, int y0,
                                                int z0, uint32_t (*cs)[8], int level) {
  const uint32_t lane = threadIdx.x & 63u;
  for (uint32_t t = lane; t < kTRows * 8u; t += 64u) {
    const int r = (int)(t >> 3), k = (int)(t & 7u);
    const int y = y0 - 1 + r % kTRY, z = z0 - 1 + r / kTRY;
    uint32_t v = 0;
    if (y >= 0 && y < g.dims[1] && z >= 0 && z < g.dims[2])
      v = d.cellStart[g.cell_base +
                      ((uint32_t)z * (uint32_t)g.dims[1] + (uint32_t)y) * (uint32_t)g.dims[0] +
                      (uint32_t)min(max(x0 - 1 + k, 0), g.dims[0])];
    cs[r][k] = v;
  }
  __builtin_amdgcn_wave_barrier();
  TileParts p;
  p.level = -1;
  p.pn = 0;
  for (int l = level < 0 ? 1 : level; l < kTileLevels && p.level < 0; l++) {
    tile_sub(l, &p.sx, &p.sy, &p.sz);
    const int mx = (kTX + p.sx - 1) / p.sx, my = kTY / p.sy, mz = kTZ / p.sz;
    const int q = (int)lane;
    p.px = (q % mx) * p.sx;
    p.py = ((q / mx) % my) * p.sy;
    p.pz = (q / (mx * my)) * p.sz;
    p.pn = 0;
    uint32_t h = 0;
    if (q < mx * my * mz) {
      const int ex = min(p.px + p.sx, kTX);
      for (int z = p.pz; z < p.pz + p.sz + 2; z++)
        for (int y = p.py; y < p.py + p.sy + 2; y++) {
          const uint32_t* c = cs[z * kTRY + y];
          h += c[ex + 2] - c[p.px];
          if (z > p.pz && z <= p.pz + p.sz && y > p.py && y <= p.py + p.sy)
            p.pn += c[ex + 1] - c[p.px + 1];
        }
      if (!p.pn) h = 0;
    }
    if (!__ballot(h >= kTileCap)) p.level = l;
  }
  __builtin_amdgcn_wave_barrier();
  return p;
}

__device__ __forceinline__ TileItem tile_item(int x, int y, int z, int sx, int sy, int sz,
                                              uint32_t unit, uint32_t n) {
  TileItem it;
  it.x0 = x;
  it.y0 = y;
  it.z0 = z;
  it.dims = (uint32_t)sx | ((uint32_t)sy << 4) | ((uint32_t)sz << 8);
  it.unit = unit;
  it.n = n;
  return it;
}

__global__ __launch_bounds__(kBlock) void k_tile_items(TileDev d, SceneGrid g) {
  __shared__ uint32_t cs_all[kBlock / 64][kTRows][8];
  uint32_t (*cs)[8] = cs_all[threadIdx.x >> 6];
  const int lane = (int)(threadIdx.x & 63u);
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
  uint32_t nbx, nby;
  const uint32_t nb = tile_blocks(g, &nbx, &nby);
  const int x0 = (int)(b % nbx) * kTX, y0 = (int)((b / nbx) % nby) * kTY,
            z0 = (int)(b / (nbx * nby)) * kTZ;
  uint32_t N = 0, H = 0;
  uint32_t first[kTY * kTZ], len[kTY * kTZ];  // its rows
#pragma unroll
  for (int r = 0; r < kTY * kTZ; r++) first[r] = len[r] = 0;
  if (b < nb) {
    const int xs = max(x0 - 1, 0), xa = min(x0 + kTX, g.dims[0]),
              xe = min(x0 + kTX + 1, g.dims[0]);
#pragma unroll
    for (int r = 0; r < kTY * kTZ; r++) {
      const int y = y0 + r % kTY, z = z0 + r / kTY;
      if (y >= g.dims[1] || z >= g.dims[2]) continue;
      const uint32_t* c = d.cellStart + g.cell_base +
                          ((uint32_t)z * (uint32_t)g.dims[1] + (uint32_t)y) * (uint32_t)g.dims[0];
      first[r] = c[x0];
      len[r] = c[xa] - first[r];
      N += len[r];
    }
    if (N >= kTileMin) {
#pragma unroll
      for (int r = 0; r < kTRows; r++) {
        const int y = y0 - 1 + r % kTRY, z = z0 - 1 + r / kTRY;
        if (y < 0 || y >= g.dims[1] || z < 0 || z >= g.dims[2]) continue;
        const uint32_t* c = d.cellStart + g.cell_base +
                            ((uint32_t)z * (uint32_t)g.dims[1] + (uint32_t)y) * (uint32_t)g.dims[0];
        H += c[xe] - c[xs];
      }
    }
  }
  int level = N >= kTileMin && H < kTileCap ? 0 : -1;
  uint32_t m = level == 0 ? 1u : 0u, w = level == 0 ? (N + 63u) >> 6 : 0u;
  for (unsigned long long s = __ballot(N >= kTileMin && level < 0); s; s &= s - 1ull) {
    const int l = __ffsll((long long)s) - 1;
    const TileParts p =
        tile_parts(d, g, __shfl(x0, l), __shfl(y0, l), __shfl(z0, l), cs, -1);
    const uint32_t has = p.level >= 0 && p.pn ? 1u : 0u;
    const uint32_t t = __shfl(wave_incl_scan((has << 16) | (has ? (p.pn + 63u) >> 6 : 0u)), 63);
    if (lane == l) {
      level = p.level;
      m = t >> 16;
      w = t & 0xffffu;
    }
  }
  const uint32_t im = wave_incl_scan(m), iw = wave_incl_scan(w);
  const uint32_t tm = __shfl(im, 63), tw = __shfl(iw, 63);
  unsigned long long base = 0;
  if (lane == 0 && tm)
    base = atomicAdd(reinterpret_cast<unsigned long long*>(d.flags + kTileUnitsSlot),
                     ((unsigned long long)tm << 32) | tw);
  const uint32_t bi = __shfl((uint32_t)(base >> 32), 0) + im - m;
  const uint32_t bu = __shfl((uint32_t)base, 0) + iw - w;
  const bool tiled = level >= 0 && bi + m <= d.tile_items && bu + w <= d.tile_units;
  if (level == 0 && bi < d.tile_items)
    d.titem[bi] = tile_item(x0, y0, z0, kTX, kTY, kTZ, bu, tiled ? N : 0u);
  const uint32_t thin = wave_incl_scan(N < kTileFull ? N : 0u);
  if (lane == 63 && thin) atomicAdd(&d.flags[kTileSparseSlot], thin);
  // Particles of sparse blocks, in block order, to the queue of the lanes.
  const uint32_t sn = N < kTileMin ? N : 0u, is = wave_incl_scan(sn), ts = __shfl(is, 63);
  uint32_t sb = 0;
  if (lane == 0 && ts) sb = atomicAdd(&d.flags[kDenseBuildSlot], ts);
  uint32_t slot = __shfl(sb, 0) + is - sn;
  // (Each particle once per step, so the slots stay below n.)  A thread stores
  // the few of its own block; the lanes of the wave store the others together.
  if (sn && sn < kTileFew) {
#pragma unroll
    for (int r = 0; r < kTY * kTZ; r++)
      for (uint32_t k = 0; k < len[r]; k++, slot++)
        if (slot < d.n) d.dense_b[slot] = first[r] + k;
  }
  for (unsigned long long s = __ballot(sn >= kTileFew); s; s &= s - 1ull) {
    const int l = __ffsll((long long)s) - 1;
    const uint32_t q = __shfl(slot, l) + (uint32_t)lane, end = __shfl(slot + sn, l);
    uint32_t o = (uint32_t)lane, j0 = 0, j1 = 0;  // places lane and lane + 64 of the block
#pragma unroll
    for (int r = 0; r < kTY * kTZ; r++) {
      const uint32_t j = __builtin_amdgcn_readlane(first[r], l), m = __builtin_amdgcn_readlane(len[r], l);
      if (o < m) j0 = j + o;
      if (o + 64u < m) j1 = j + o + 64u;
      o -= m;
    }
    if (q < end && q < d.n) d.dense_b[q] = j0;
    if (q + 64u < end && q + 64u < d.n) d.dense_b[q + 64u] = j1;
  }
  // Those of blocks that fit at no level, or beyond the capacity, to the
  // queue of the quads, a wave per block.
  for (unsigned long long s = __ballot(N >= kTileMin && !tiled); s; s &= s - 1ull) {
    const int l = __ffsll((long long)s) - 1;
    const int bx = __shfl(x0, l), by = __shfl(y0, l), bz = __shfl(z0, l);
    const uint32_t all = __shfl(N, l);
    uint32_t q = 0;
    if (lane == 0) q = atomicAdd(&d.flags[kDenseSlot], all);
    q = __shfl(q, 0);
    for (int r = 0; r < kTY * kTZ; r++) {
      const int y = by + r % kTY, z = bz + r / kTY;
      if (y >= g.dims[1] || z >= g.dims[2]) continue;
      const uint32_t* c = d.cellStart + g.cell_base +
                          ((uint32_t)z * (uint32_t)g.dims[1] + (uint32_t)y) * (uint32_t)g.dims[0];
      const uint32_t j = c[bx], m = c[min(bx + kTX, g.dims[0])] - j;
      for (uint32_t k = (uint32_t)lane; k < m; k += 64u)
        if (q + k < d.n) d.dense[q + k] = j + k;
      q += m;
    }
  }
  for (unsigned long long s = __ballot(level > 0); s; s &= s - 1ull) {
    const int l = __ffsll((long long)s) - 1;
    const int bx = __shfl(x0, l), by = __shfl(y0, l), bz = __shfl(z0, l);
    const TileParts p = tile_parts(d, g, bx, by, bz, cs, __shfl(level, l));
    const uint32_t has = p.pn ? 1u : 0u, pk = (has << 16) | (has ? (p.pn + 63u) >> 6 : 0u);
    const uint32_t ex = wave_incl_scan(pk) - pk;
    const uint32_t i = __shfl(bi, l) + (ex >> 16), first = __shfl(bu, l);
    const bool ok = __shfl((int)tiled, l) != 0;
    if (has && i < d.tile_items)
      d.titem[i] = tile_item(bx + p.px, by + p.py, bz + p.pz, min(p.px + p.sx, kTX) - p.px, p.sy,
                             p.sz, first + (ex & 0xffffu), ok ? p.pn : 0u);
  }
}

// Every kCensusStep-th particle of every base block (block has to be zero),
// then an estimate of the particles of the thin ones together
// (flags[kTileSparseSlot] likewise).  The first step after a load waits for it:
// 218 us with all of 4,096,000 particles, 43 with these.
constexpr uint32_t kCensusStep = 7;  // odd: lattices are loaded row by row
__global__ __launch_bounds__(kBlock) void k_tile_census(const float4* __restrict__ pos, uint32_t n,
                                                        SceneGrid g, uint32_t* __restrict__ block) {
  const uint32_t i = (blockIdx.x * kBlock + threadIdx.x) * kCensusStep;
  if (i >= n) return;
  uint32_t nbx, nby;
  tile_blocks(g, &nbx, &nby);
  const float4 x = pos[i];
  int c[3];
  cell_lin(g, make_float3(x.x, x.y, x.z), c);
  atomicAdd(block + ((uint32_t)(c[2] / kTZ) * nby + (uint32_t)(c[1] / kTY)) * nbx + (uint32_t)(c[0] / kTX),
            1u);
}
__global__ __launch_bounds__(kBlock) void k_tile_sparse(const uint32_t* __restrict__ block,
                                                        uint32_t nb, uint32_t* __restrict__ sum) {
  const uint32_t b = blockIdx.x * kBlock + threadIdx.x;
  const uint32_t c = b < nb ? block[b] * kCensusStep : 0u;
  const uint32_t t = wave_incl_scan(c < kTileFull ? c : 0u);
  if ((threadIdx.x & 63u) == 63u && t) atomicAdd(sum, t);
}

// Appends i to a queue (count in flags[slot]) for the lanes with q set (every
// lane of the wave calls).
__device__ __forceinline__ void wave_queue(const TileDev& d, uint32_t* queue, int counter, uint32_t i,
                                           bool q) {
  const unsigned long long mask = __ballot(q);
  if (!mask) return;
  const uint32_t lane = __lane_id();
  const int lead = __ffsll((long long)mask) - 1;
  uint32_t base = 0;
  if ((int)lane == lead) base = atomicAdd(&d.flags[counter], (uint32_t)__popcll(mask));
  base = __shfl(base, lead);
  const uint32_t slot = base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
  if (q && slot < d.n) queue[slot] = i;
}

// Consecutive workgroups go to the XCDs in turn: a run of kTileRun consecutive
// pieces of work for each.
__device__ __forceinline__ uint32_t tile_order(uint32_t b) {
  return (b & ~(8u * kTileRun - 1u)) + (b & 7u) * kTileRun + ((b >> 3) & (kTileRun - 1u));
}
__device__ __forceinline__ uint32_t tile_span(uint32_t ni) {
  return (ni + 8u * kTileRun - 1u) & ~(8u * kTileRun - 1u);
}
__device__ __forceinline__ uint32_t tile_count(const TileDev& d) {
  return min(d.flags[kTileItemsSlot], d.tile_items);
}
// The work of a pass: the particles of sparse blocks, a lane each, in chunks of
// kTileBlock, then the tiles.  Workgroup b of G takes every G-th piece, the
// XCDs runs of kTileRun consecutive ones.  Chunks come first: as the last
// workgroups to start, their gathers would run on after the tiles (two spheres
// of 500,009 particles 0.45 ms per step, 0.49 in that order).
template <class Lane, class Tile>
__device__ __forceinline__ void tile_work(const TileDev& d, uint32_t b, uint32_t G, Lane lane,
                                          Tile tile) {
  const uint32_t ni = tile_count(d), nq = min(d.flags[kDenseBuildSlot], d.n);
  const uint32_t sc = tile_span((nq + (uint32_t)kTileBlock - 1u) / (uint32_t)kTileBlock);
  uint32_t w = b;
  for (; w < sc; w += G) {
    const uint32_t q = tile_order(w) * (uint32_t)kTileBlock + threadIdx.x;
    if (q < nq) lane(d.dense_b[q]);
  }
  for (w -= sc; w < tile_span(ni); w += G) {
    const uint32_t item = tile_order(w);
    if (item < ni) tile(item);
  }
}
// The wave's index in its workgroup, known to be uniform: what it addresses
// comes through scalar loads into scalar registers.
__device__ __forceinline__ uint32_t tile_wave() {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}
__device__ __forceinline__ uint32_t* tile_list(const TileDev& d, uint32_t unit) {
  return reinterpret_cast<uint32_t*>(
      d.tnbr + ((size_t)unit * kTileChunks * 64u + (threadIdx.x & 63u)) * 8u);
}

// What a pass reads of its tile before the barrier: the lanes of this wave's
// first unit and their first list chunks, and the tile's rows through
// load/store.
struct TileHead {
  uint32_t unit, nu;
  uint2 own;
  uint4 q0;
};
template <class Load, class Store>
__device__ __forceinline__ TileHead tile_fill(const TileDev& d, uint32_t item, Load load, Store store) {
  const uint32_t wave = tile_wave(), lane = threadIdx.x & 63u;
  using V = decltype(load(0u));
  constexpr int Q = (kTRows + (int)kTileWaves - 1) / (int)kTileWaves;
  static_assert(Q * (int)kTileWaves <= kTileRows, "rows");
  const TileRec* rec = d.trec + item;
  uint2 rw[Q];
  V v[Q];
  const uint2 head = rec->head;
#pragma unroll
  for (int q = 0; q < Q; q++) rw[q] = rec->row[wave + kTileWaves * q];
#pragma unroll
  for (int q = 0; q < Q; q++)
    if (lane < (rw[q].y >> 16)) v[q] = load(rw[q].x + lane);
  TileHead h;
  h.unit = head.x;
  h.nu = (head.y + 63u) >> 6;
  h.own = make_uint2(0xffffffffu, 0u);
  h.q0 = make_uint4(0u, 0u, 0u, 0u);
  if (wave < h.nu) {
    h.own = d.town[(size_t)(h.unit + wave) * 64u + lane];
    h.q0 = load_chunk(tile_list(d, h.unit + wave));
  }
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const uint32_t len = rw[q].y >> 16, off = rw[q].y & 0xffffu;
    if (lane < len) store(off + lane, v[q]);
    for (uint32_t k = lane + 64u; k < len; k += 64u) store(off + k, load(rw[q].x + k));
  }
  return h;
}
// The lanes and first chunks of unit u of the tile (those of the wave's first
// unit are there already).
__device__ __forceinline__ void tile_next(const TileDev& d, TileHead& h, uint32_t u) {
  if (u == tile_wave()) return;
  h.own = d.town[(size_t)(h.unit + u) * 64u + (threadIdx.x & 63u)];
  h.q0 = load_chunk(tile_list(d, h.unit + u));
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(3))) char* lds_ptr;
__device__ __forceinline__ lds_ptr lds_of(const void* p) { return (lds_ptr)p; }
// One record: a single 16-byte LDS read (volatile keeps it whole where w is
// not used: three narrower reads meet five times the bank conflicts).
__device__ __forceinline__ float4 lds_rec(lds_ptr p) {
  const f32x4 q = *(const volatile __attribute__((address_space(3))) f32x4*)p;
  return make_float4(q.x, q.y, q.z, q.w);
}
struct TileGet {
  lds_ptr p;
  __device__ __forceinline__ float4 operator()(uint32_t o) const { return lds_rec(p + o); }
};
struct TileXV {
  float4 a;
  float2 b;
};
struct TileGetXV {
  lds_ptr p, p2;
  __device__ __forceinline__ TileXV operator()(uint32_t o) const {
    TileXV q;
    q.a = lds_rec(p + o);
    const f32x2 t = *(const __attribute__((address_space(3))) f32x2*)(p2 + (o >> 1));
    q.b = make_float2(t.x, t.y);
    return q;
  }
};
__device__ __forceinline__ float4 rec_pos(const float4& q) { return q; }
__device__ __forceinline__ float4 rec_pos(const TileXV& q) { return q.a; }

// The step constants of a tiled pass: the short sequences are on (tile_step
// requires it), and the constants that the terms use most sit in vector
// registers (an instruction with a scalar operand issues at half rate).
__device__ __forceinline__ float in_vgpr(float a) {
  asm("" : "+v"(a));
  return a;
}
__device__ __forceinline__ SimConst tile_const(const SimConst& c0) {
  SimConst c = c0;
  c.fast_div = c.fast_rcp = c.fast_sqrt = 1;
  c.r9s = in_vgpr(c.r9s);
  c.h9s = in_vgpr(c.h9s);
  c.inv_rho0 = in_vgpr(c.inv_rho0);
  return c;
}

// Slot 0 pads the lists: a record at rest beyond h of every particle, whose
// terms are zero: its factors of the particle's own values, which plan_tiles
// and tile_step hold finite, are.
__device__ __forceinline__ float4 tile_sentinel(const TileDev& d) {
  return make_float4(d.tile_far, 0.0f, 0.0f, 0.0f);
}

struct TilePair {
  float rx, ry, rz, r2;
};
template <class R>
__device__ __forceinline__ TilePair tile_pair(const float3& xi, const R& q) {
  TilePair p;
  const float4 x = rec_pos(q);
  p.rx = xi.x - x.x;
  p.ry = xi.y - x.y;
  p.rz = xi.z - x.z;
  p.r2 = p.rx * p.rx + p.ry * p.ry + p.rz * p.rz;
  return p;
}

// poly6 and the spiky gradient without selections: the bits of poly6_sel and
// spiky_sel for |r| >= EPS_D, except for the sign of zero terms.  Beyond h
// the clamped difference is 0 and so are the terms.  A NaN distance would give
// 0 here; there is none, as every position is finite: a load refuses others
// and each move ends in a clamp to the box (smin and smax let NaN become hi_e),
// and plan_tiles bounds the squares.
__device__ __forceinline__ float tile_w(const SimConst& c, float r2) {
  const float t = fmaxf(c.h2 - r2, 0.0f);
  return div_seq(c.c1s * ((t * t) * t), c.h9s, c.r9s);
}
__device__ __forceinline__ float3 tile_g(const SimConst& c, const TilePair& p) {
  const float rl = sqrt_rn(p.r2);
  const float q = fmaxf(c.h - rl, 0.0f);
  const float coef = c.m3c2 * (q * q);
  const float rc = rcp_seq(c.h6 * rl);
  return make_float3(rc * (coef * p.rx), rc * (coef * p.ry), rc * (coef * p.rz));
}

// Visits the list of one lane, 8 entries a chunk, G at a time: get(offset)
// reads a record, fast(pair, record) and slow(pair, record) add its terms.  The
// fast terms hold where |r|^2 >= c.r2_min; the rare group with a closer (or
// coincident) pair takes the general terms.
template <int G, class Get, class Fast, class Slow>
__device__ __forceinline__ void tile_visit(const uint32_t* lp, uint4 q, int cnt, float r2_min,
                                           const float3& xi, Get get, Fast fast, Slow slow) {
  const int ng = (cnt + 3) >> 2, nc = (cnt + 7) >> 3;
  auto two = [&](uint32_t a) {
    const auto r0 = get(a & 0xffffu), r1 = get(a >> 16);
    const TilePair p0 = tile_pair(xi, r0), p1 = tile_pair(xi, r1);
    if (__ballot(fminf(p0.r2, p1.r2) < r2_min)) {
      slow(p0, r0);
      slow(p1, r1);
    } else {
      fast(p0, r0);
      fast(p1, r1);
    }
  };
  auto group = [&](uint32_t a, uint32_t b) {
    if (G == 2) {
      two(a);
      two(b);
      return;
    }
    const auto r0 = get(a & 0xffffu), r1 = get(a >> 16), r2 = get(b & 0xffffu), r3 = get(b >> 16);
    const TilePair p0 = tile_pair(xi, r0), p1 = tile_pair(xi, r1), p2 = tile_pair(xi, r2),
                   p3 = tile_pair(xi, r3);
    const float m = fminf(fminf(fminf(p0.r2, p1.r2), p2.r2), p3.r2);
    if (__ballot(m < r2_min)) {
      slow(p0, r0);
      slow(p1, r1);
      slow(p2, r2);
      slow(p3, r3);
    } else {
      fast(p0, r0);
      fast(p1, r1);
      fast(p2, r2);
      fast(p3, r3);
    }
  };
  for (int ch = 0; ch < nc; ch++) {
    uint4 qn = q;
    if (ch + 1 < nc) qn = load_chunk(lp + (size_t)(ch + 1) * 256u);
    group(q.x, q.y);
    if (2 * ch + 1 < ng) group(q.z, q.w);
    q = qn;
  }
}

// newtonStepCalculateLambda of one lane (lambda_terms).
__device__ __forceinline__ float tile_lambda(const SimConst& c, const uint32_t* lp,
                                                 uint4 q0, int cnt, lds_ptr rec, const float3& xi) {
  float dens = 0.0f, denom = 0.0f, Gx = 0.0f, Gy = 0.0f, Gz = 0.0f;
  auto add = [&](float w, float3 gr) {
    gr.x = gr.x * c.inv_rho0;
    gr.y = gr.y * c.inv_rho0;
    gr.z = gr.z * c.inv_rho0;
    dens = dens + w;
    Gx = Gx + gr.x;
    Gy = Gy + gr.y;
    Gz = Gz + gr.z;
    denom = denom + (gr.x * gr.x + gr.y * gr.y + gr.z * gr.z);
  };
  tile_visit<2>(
      lp, q0, cnt, c.r2_min, xi, TileGet{rec},
      [&](const TilePair& p, const float4&) { add(tile_w(c, p.r2), tile_g(c, p)); },
      [&](const TilePair& p, const float4&) {
        add(poly6_sel(c, p.r2), spiky_sel(c, p.rx, p.ry, p.rz, p.r2));
      });
  return lambda_of(c, dens, denom, Gx, Gy, Gz);
}

// The particles whose lists overflow a tile's, a quad each.
__global__ __launch_bounds__(kBlock) void k_queue_build(TileDev d, SimConst c, SceneGrid g,
                                                        float4* out) {
  const uint32_t qn = min(d.flags[kDenseSlot], d.n);
  const uint32_t stride = gridDim.x * (kBlock / 4);
  for (uint32_t q = blockIdx.x * (kBlock / 4) + (threadIdx.x >> 2); q < qn; q += stride) {
    const uint32_t i = d.dense[q];
    nbr_quad_one<16>(i, d, c.h2, g);
    __threadfence_block();
    lambda_quad_one<false>(i, d, c, d.predQ, out);
  }
}

// nbr_one and the first λ of a tile's particles, a lane each: the rows, the
// pruning and the order of nbr_one over the tile's records, so the lists are
// nbr_one's.  Also writes the tile's rows and lanes for the later passes.
__global__ __launch_bounds__(kTileBlock, 6) void k_tile_build(TileDev d, SimConst c0, SceneGrid g,
                                                              float4* out) {
  __shared__ float4 rec[kTileCap + 4];
  __shared__ uint32_t cs[kTRows][8];
  __shared__ uint32_t rowO[kTRows];
  __shared__ uint32_t intr[kTY * kTZ + 1];
  const SimConst c = tile_const(c0);
  const uint32_t tid = threadIdx.x, wave = tile_wave(), lane = tid & 63u;
  const auto tile = [&](uint32_t item) {
    const TileItem it = d.titem[item];
    const int bx = (int)(it.dims & 15u), by = (int)((it.dims >> 4) & 15u), bz = (int)(it.dims >> 8);
    const int ry = by + 2, R = ry * (bz + 2), wx = bx + 2;
    if (tid < kTRows * 8u) {
      const int r = (int)(tid >> 3), k = (int)(tid & 7u);
      uint32_t v = 0;
      if (r < R) {
        const int y = it.y0 - 1 + r % ry, z = it.z0 - 1 + r / ry;
        if (y >= 0 && y < g.dims[1] && z >= 0 && z < g.dims[2]) {
          const int x = min(max(it.x0 - 1 + min(k, wx), 0), g.dims[0]);
          v = d.cellStart[g.cell_base + ((uint32_t)z * (uint32_t)g.dims[1] + (uint32_t)y) *
                                            (uint32_t)g.dims[0] + (uint32_t)x];
        }
      }
      cs[r][k] = v;
    }
    if (tid == 0) rec[0] = tile_sentinel(d);
    __syncthreads();
    if (tid < 64u) {
      const uint32_t len = lane < (uint32_t)kTRows ? cs[lane][7] - cs[lane][0] : 0u;
      const uint32_t off = 1u + wave_incl_scan(len) - len;
      if (lane < (uint32_t)kTRows) {
        rowO[lane] = off;
        d.trec[item].row[lane] = make_uint2(cs[lane][0], off | (len << 16));
      } else if (lane < (uint32_t)kTileRows) {
        d.trec[item].row[lane] = make_uint2(0u, 0u);
      }
      if (lane == 0) d.trec[item].head = make_uint2(it.unit, it.n);
      const int l = (int)lane;
      uint32_t il = 0;
      if (l < by * bz) {
        const int r = (1 + l / by) * ry + 1 + l % by;
        il = cs[r][bx + 1] - cs[r][1];
      }
      const uint32_t ii = wave_incl_scan(il);
      if (l < kTY * kTZ) intr[l + 1] = ii;
      if (l == 0) intr[0] = 0;
    }
    __syncthreads();
    for (uint32_t r = wave; r < (uint32_t)R; r += kTileWaves) {
      const uint32_t s = cs[r][0], len = cs[r][7] - s, off = rowO[r];
      for (uint32_t k = lane; k < len; k += 64u) {
        const float4 q = d.predQ[s + k];
        if (off + k < kTileCap) rec[off + k] = q;
      }
    }
    __syncthreads();
    const float cell = 1.0f / g.inv_cell;
    const float h2 = in_vgpr(c.h2), hm2 = h2 * 1.0201f;
    // Lanes of a wave and waves of a tile wait for their longest list, so
    // what stands out of its tile goes to the queue: particles of cells that
    // hold kTileSpike times the tile's mean, and lists as much longer than
    // the mean cell suggests (a cell of the size of h and its neighbours
    // hold 3.9 neighbours per particle of the mean cell).
    const float mean = (float)(rowO[R - 1] + (cs[R - 1][7] - cs[R - 1][0])) / (float)(wx * R);
    const uint32_t crowd = max(kTileCrowd, (uint32_t)(kTileSpike * mean));
    const uint32_t cap = min(min((uint32_t)d.K4 * kChunk, 8u * (uint32_t)kTileChunks),
                             max(kTileLong, (uint32_t)(kTileSpike * 3.9f * mean)));
    const uint32_t nu = (it.n + 63u) >> 6;
    for (uint32_t u = wave; u < nu; u += kTileWaves) {
      const uint32_t p = u * 64u + lane, unit = it.unit + u;
      const bool act = p < it.n;
      uint32_t i = 0xffffffffu, self = 0, cnt = 0;
      uint32_t* lp = tile_list(d, unit);
      float3 xi = make_float3(0.f, 0.f, 0.f);
      if (act) {
        int l = 0;
        for (int q = 1; q < by * bz; q++) l += p >= intr[q] ? 1 : 0;
        const int r0 = (1 + l / by) * ry + 1 + l % by;
        i = cs[r0][1] + (p - intr[l]);
        self = rowO[r0] + (i - cs[r0][0]);
        const float4 x4 = rec[self];
        xi = make_float3(x4.x, x4.y, x4.z);
        int cc[3];
        cell_lin(g, xi, cc);
        auto dist = [&](uint32_t j) {
          const float4 xj = lds_rec(lds_of(&rec[j]));
          const float rx = xi.x - xj.x, ry_ = xi.y - xj.y, rz = xi.z - xj.z;
          return rx * rx + ry_ * ry_ + rz * rz;
        };
        const float gxl = face_gap(xi.x, g.lo[0], cell, cc[0], -1);
        const float gxr = face_gap(xi.x, g.lo[0], cell, cc[0], 1);
        const int kx = cc[0] - (it.x0 - 1), ky = cc[1] - (it.y0 - 1), kz = cc[2] - (it.z0 - 1);
        const uint32_t* own = cs[kz * ry + ky];
        if (own[kx + 1] - own[kx] > crowd) cnt = 0xffffffffu;
        // The candidate rows of nbr_one, as slot ranges [s, e) of the tile.
        auto rows = [&](auto walk) {
          for (int dz = -1; dz <= 1; dz++) {
            const float gz = face_gap(xi.z, g.lo[2], cell, cc[2], dz);
            for (int dy = -1; dy <= 1; dy++) {
              const float gy = face_gap(xi.y, g.lo[1], cell, cc[1], dy);
              const float yz2 = gy * gy + gz * gz;
              if (yz2 > hm2) continue;
              const int r = (kz + dz) * ry + ky + dy;
              const int k0 = gxl * gxl + yz2 <= hm2 ? kx - 1 : kx;
              const int k1 = gxr * gxr + yz2 <= hm2 ? kx + 1 : kx;
              const uint32_t c0_ = cs[r][0], ro = rowO[r];
              walk(ro + (cs[r][k0] - c0_), ro + (cs[r][k1 + 1] - c0_));
            }
          }
        };
        if (cnt == 0u) {
          uint32_t b0 = 0, b1 = 0, b2 = 0, b3 = 0;
          auto push = [&](uint32_t slot) {
            b0 = __builtin_amdgcn_alignbit(b1, b0, 16);
            b1 = __builtin_amdgcn_alignbit(b2, b1, 16);
            b2 = __builtin_amdgcn_alignbit(b3, b2, 16);
            b3 = __builtin_amdgcn_alignbit(slot << 4, b3, 16);
            cnt++;
            if ((cnt & 7u) == 0u) {
              const uint32_t ch = (cnt >> 3) - 1u;
              if (ch < (uint32_t)kTileChunks)
                *reinterpret_cast<uint4*>(lp + (size_t)ch * 256u) = make_uint4(b0, b1, b2, b3);
            }
          };
          rows([&](uint32_t s, uint32_t e) {
            for (uint32_t jb = s; jb < e; jb += 32u) {
              const uint32_t len = min(e - jb, 32u);
              uint32_t mask = 0;
              const uint32_t len4 = (len + 3u) & ~3u;
              for (uint32_t o = 0; o < len4; o += 4u) {
                const uint32_t j = jb + o;
                const float d0 = dist(j), d1 = dist(j + 1u), d2 = dist(j + 2u), d3 = dist(j + 3u);
                // Four times mask = 2 mask + (d <= h2); a carry is read two
                // instructions after its compare at the earliest.
                unsigned long long k1, k2, k3;
                asm("v_cmp_ge_f32 vcc, %4, %5\n\t"
                    "v_cmp_ge_f32 %1, %4, %6\n\t"
                    "v_cmp_ge_f32 %2, %4, %7\n\t"
                    "v_cmp_ge_f32 %3, %4, %8\n\t"
                    "v_addc_co_u32 %0, vcc, %0, %0, vcc\n\t"
                    "v_addc_co_u32 %0, vcc, %0, %0, %1\n\t"
                    "v_addc_co_u32 %0, vcc, %0, %0, %2\n\t"
                    "v_addc_co_u32 %0, vcc, %0, %0, %3"
                    : "+v"(mask), "=&s"(k1), "=&s"(k2), "=&s"(k3)
                    : "v"(h2), "v"(d0), "v"(d1), "v"(d2), "v"(d3)
                    : "vcc");
              }
              // Candidate jb + q sits at bit len4 - 1 - q; the first comes to bit 31.
              mask <<= 32u - len4;
              mask &= 0xffffffffu << (32u - len);
              const uint32_t me = self - jb;
              if (me < 32u) mask &= ~(0x80000000u >> me);
              while (mask) {
                const uint32_t q = (uint32_t)__builtin_clz(mask);
                mask &= ~(0x80000000u >> q);
                push(jb + q);
              }
            }
          });
          const uint32_t real = cnt;
          while (cnt & 7u) push(0u);
          cnt = real;
        }
      }
      const bool over = cnt > cap;
      wave_queue(d, d.dense, kDenseSlot, i, act && over);
      if (over) cnt = 0;
      d.town[(size_t)unit * 64u + lane] =
          make_uint2(act && !over ? i : 0xffffffffu, (self << 4) | (cnt << 16));
      if (act && !over) {
        d.ncnt[i] = cnt;
        const float lam = tile_lambda(c, lp, load_chunk(lp), (int)cnt, lds_of(rec), xi);
        out[i] = make_float4(xi.x, xi.y, xi.z, lam);
      }
    }
    __syncthreads();
  };
  tile_work(
      d, blockIdx.x, gridDim.x,
      [&](uint32_t i) {
        nbr_one(i, d, c0.h2, g);
        lambda_one<false, 0>(i, d, c0, d.predQ, out);
      },
      tile);
}

// The first kTileQuads workgroups of a pass take the queue of long lists, a
// quad each.
template <class F>
__device__ __forceinline__ bool tile_queue(const TileDev& d, F f) {
  if (blockIdx.x >= kTileQuads) return false;
  const uint32_t nl = min(d.flags[kDenseSlot], d.n);
  for (uint32_t q = blockIdx.x * (kTileBlock / 4) + (threadIdx.x >> 2); q < nl;
       q += kTileQuads * (kTileBlock / 4))
    f(d.dense[q]);
  return true;
}

// Runs lane(i) for this workgroup's particles of sparse blocks and unit(head)
// for every unit of its tiles.
template <class Load, class Store, class Unit, class Lane>
__device__ __forceinline__ void tile_run(const TileDev& d, Load load, Store store, Unit unit,
                                         Lane lane) {
  const uint32_t wave = tile_wave();
  tile_work(d, blockIdx.x - kTileQuads, gridDim.x - kTileQuads, lane, [&](uint32_t item) {
    TileHead h = tile_fill(d, item, load, store);
    __syncthreads();
    for (uint32_t u = wave; u < h.nu; u += kTileWaves) {
      tile_next(d, h, u);
      if (h.own.x != 0xffffffffu) unit(h, tile_list(d, h.unit + u));
    }
    __syncthreads();  // the next tile's fill
  });
}

// The passes after the build: lambda_one<true>, deltap_one, xsph_one and
// vort_one over tiles.  64 VGPRs keep four workgroups of λ on a CU (two
// records in flight per lane; four need 78 VGPRs, 198 us against 189), the
// others run three (delta-p, at 80 VGPRs, of which it spills 8 to 16 bytes a
// lane) or two (XSPH, whose records take 60 KB).
__global__ __launch_bounds__(kTileBlock, 8) void k_tile_lambda(TileDev d, SimConst c0, float4* out) {
  __shared__ float4 rec[kTileCap + 4];
  if (tile_queue(d, [&](uint32_t i) { lambda_quad_one<true>(i, d, c0, nullptr, out); })) return;
  const SimConst c = tile_const(c0);
  if (threadIdx.x == 0) rec[0] = tile_sentinel(d);
  const lds_ptr rb = lds_of(rec);
  tile_run(
      d, [&](uint32_t j) { return at(d.xs3, j); },
      [&](uint32_t s, const float3& v) { *reinterpret_cast<float3*>(&rec[s]) = v; },
      [&](const TileHead& h, const uint32_t* lp) {
        const float4 x4 = lds_rec(rb + (h.own.y & 0xffffu));
        const float3 xi = make_float3(x4.x, x4.y, x4.z);
        const float lam = tile_lambda(c, lp, h.q0, (int)(h.own.y >> 16), rb, xi);
        out[h.own.x] = make_float4(xi.x, xi.y, xi.z, lam);
      },
      [&](uint32_t i) { lambda_one<true, 0>(i, d, c0, nullptr, out); });
}

template <bool LAST, int NT>
__global__ __launch_bounds__(kTileBlock, 6) void k_tile_deltap(TileDev d, SimConst c0, SceneGrid g,
                                                               const float4* in) {
  __shared__ float4 rec[kTileCap + 4];
  if (tile_queue(d, [&](uint32_t i) { deltap_quad_one<LAST, NT>(i, d, c0, g, in); })) return;
  const SimConst c = tile_const(c0);
  if (threadIdx.x == 0) rec[0] = tile_sentinel(d);
  const lds_ptr rb = lds_of(rec);
  tile_run(
      d, [&](uint32_t j) { return at(in, j); },
      [&](uint32_t s, const float4& v) { rec[s] = v; },
      [&](const TileHead& h, const uint32_t* lp) {
        const float4 xi = lds_rec(rb + (h.own.y & 0xffffu));
        float dx = 0.0f, dy = 0.0f, dz = 0.0f;
        auto add = [&](float w, const float3& gr, float lj) {
          const float t = c.negk * ipow_n<NT>(w * c.S, c.n_tensile);
          const float sc = (xi.w + lj) + t;
          dx = dx + sc * gr.x;
          dy = dy + sc * gr.y;
          dz = dz + sc * gr.z;
        };
        tile_visit<4>(
            lp, h.q0, (int)(h.own.y >> 16), c.r2_min, make_float3(xi.x, xi.y, xi.z), TileGet{rb},
            [&](const TilePair& p, const float4& q) { add(tile_w(c, p.r2), tile_g(c, p), q.w); },
            [&](const TilePair& p, const float4& q) {
              add(poly6_sel(c, p.r2), spiky_sel(c, p.rx, p.ry, p.rz, p.r2), q.w);
            });
        deltap_finish<LAST>(h.own.x, d, c, g, xi, dx, dy, dz);
      },
      [&](uint32_t i) { deltap_one<LAST, NT, 0>(i, d, c0, g, in, nullptr); });
}

__global__ __launch_bounds__(kTileBlock) void k_tile_xsph(TileDev d, SimConst c0, float4* out) {
  __shared__ float4 rec[kTileCap + 4];
  __shared__ float2 rec2[kTileCap + 4];
  if (tile_queue(d, [&](uint32_t i) { xsph_quad_one(i, d, c0, out); })) return;
  const SimConst c = tile_const(c0);
  if (threadIdx.x == 0) {
    rec[0] = tile_sentinel(d);
    rec2[0] = make_float2(0.0f, 0.0f);
  }
  const float3* __restrict__ xv = reinterpret_cast<const float3*>(d.xv);
  const TileGetXV get{lds_of(rec), lds_of(rec2)};
  tile_run(
      d, [&](uint32_t j) { return XVRec{at(xv, 2 * j), at(xv, 2 * j + 1)}; },
      [&](uint32_t s, const XVRec& v) {
        rec[s] = make_float4(v.x.x, v.x.y, v.x.z, v.v.x);
        rec2[s] = make_float2(v.v.y, v.v.z);
      },
      [&](const TileHead& h, const uint32_t* lp) {
        const TileXV o = get(h.own.y & 0xffffu);
        const float3 xi = make_float3(o.a.x, o.a.y, o.a.z);
        const float3 vi = make_float3(o.a.w, o.b.x, o.b.y);
        float ox = 0.0f, oy = 0.0f, oz = 0.0f, sx = 0.0f, sy = 0.0f, sz = 0.0f, dens = 0.0f;
        auto add = [&](float w, const float3& gr, const TileXV& q) {
          const float u0 = q.a.w - vi.x, u1 = q.b.x - vi.y, u2 = q.b.y - vi.z;
          ox = ox + (u1 * gr.z - u2 * gr.y);
          oy = oy + (u2 * gr.x - u0 * gr.z);
          oz = oz + (u0 * gr.y - u1 * gr.x);
          sx = sx + u0 * w;
          sy = sy + u1 * w;
          sz = sz + u2 * w;
          dens = dens + w;
        };
        tile_visit<4>(
            lp, h.q0, (int)(h.own.y >> 16), c.r2_min, xi, get,
            [&](const TilePair& p, const TileXV& q) { add(tile_w(c, p.r2), tile_g(c, p), q); },
            [&](const TilePair& p, const TileXV& q) {
              add(poly6_sel(c, p.r2), spiky_sel(c, p.rx, p.ry, p.rz, p.r2), q);
            });
        xsph_finish(h.own.x, d, c, xi, vi, ox, oy, oz, sx, sy, sz, dens, out);
      },
      [&](uint32_t i) { xsph_one<0>(i, d, c0, out); });
}

__global__ __launch_bounds__(kTileBlock) void k_tile_vort(TileDev d, SimConst c0, const float4* in) {
  __shared__ float4 rec[kTileCap + 4];
  if (tile_queue(d, [&](uint32_t i) {
        const float4 xi = in[i];
        float s[3];
        quad_sums<3>(
            i, (int)d.ncnt[i], d.K4, d.nbr, [&](uint32_t j) { return at(in, j); },
            [&](uint32_t, const float4& xj, float* t) { vort_terms(c0, xi, xj, t); }, s);
        if ((threadIdx.x & 3u) == 0)
          vort_finish(i, d, c0, xi, s[0], s[1], s[2], nullptr, nullptr, true);
      }))
    return;
  const SimConst c = tile_const(c0);
  if (threadIdx.x == 0) rec[0] = tile_sentinel(d);
  const lds_ptr rb = lds_of(rec);
  tile_run(
      d, [&](uint32_t j) { return at(in, j); },
      [&](uint32_t s, const float4& v) { rec[s] = v; },
      [&](const TileHead& h, const uint32_t* lp) {
        const float4 xi = lds_rec(rb + (h.own.y & 0xffffu));
        float ex = 0.0f, ey = 0.0f, ez = 0.0f;
        auto add = [&](const float3& gr, float wj) {
          ex = ex + wj * gr.x;
          ey = ey + wj * gr.y;
          ez = ez + wj * gr.z;
        };
        tile_visit<4>(
            lp, h.q0, (int)(h.own.y >> 16), c.r2_min, make_float3(xi.x, xi.y, xi.z), TileGet{rb},
            [&](const TilePair& p, const float4& q) { add(tile_g(c, p), q.w); },
            [&](const TilePair& p, const float4& q) {
              add(spiky_sel(c, p.rx, p.ry, p.rz, p.r2), q.w);
            });
        vort_finish(h.own.x, d, c, xi, ex, ey, ez, nullptr, nullptr, true);
      },
      [&](uint32_t i) { vort_one<0>(i, d, c0, in); });
}

// The lists of the tiles by load id (k_nbr_export's output): slots back to
// particles through the tile's rows.
__global__ __launch_bounds__(kTileBlock) void k_tile_export(TileDev d, uint32_t* __restrict__ counts,
                                                            uint32_t* __restrict__ out, int stride) {
  const uint32_t ni = tile_count(d), lane = threadIdx.x & 63u;
  for (uint32_t item = blockIdx.x; item < ni; item += gridDim.x) {
    const TileRec* rec = d.trec + item;
    const uint32_t nu = (rec->head.y + 63u) >> 6;
    for (uint32_t u = tile_wave(); u < nu; u += kTileWaves) {
      const uint2 own = d.town[(size_t)(rec->head.x + u) * 64u + lane];
      if (own.x == 0xffffffffu) continue;
      const uint32_t id = id_of(d.posB[own.x]);
      const int cnt = (int)(own.y >> 16);
      counts[id] = (uint32_t)cnt;
      const uint16_t* lp = reinterpret_cast<const uint16_t*>(tile_list(d, rec->head.x + u));
      for (int k = 0; k < min(cnt, stride); k++) {
        const uint32_t slot = lp[(size_t)(k >> 3) * 512u + (uint32_t)(k & 7)] >> 4;
        uint32_t j = 0;
        for (int r = 0; r < kTRows; r++) {
          const uint2 row = rec->row[r];
          const uint32_t o = slot - (row.y & 0xffffu);
          if (o < (row.y >> 16)) j = row.x + o;
        }
        out[(size_t)id * stride + k] = id_of(d.posB[j]);
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_queue_export(TileDev d, uint32_t* __restrict__ counts,
                                                         uint32_t* __restrict__ out, int stride) {
  const uint32_t nb = min(d.flags[kDenseBuildSlot], d.n), nl = min(d.flags[kDenseSlot], d.n);
  for (uint32_t q = flat_index(); q < nb + nl; q += gridDim.x * kBlock)
    nbr_export_one(q < nb ? d.dense_b[q] : d.dense[q - nb], d, counts, out, stride);
}
