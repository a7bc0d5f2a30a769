// Deposit of a bunch in the caller's (random) order through bricks of cells.
//
// In random order every particle's charge is an atomic of its own at the
// memory side, and those are what the plain deposit waits for: 15 per
// nanosecond on the whole card, 652 us for 10M particles whose rows stream in
// 100 us.  Here each particle's (charge, cell) is first moved to the run of
// its brick, and a workgroup then adds a run up in LDS, with one atomic per
// cell of the brick, neighbouring cells in one request:
//
//   k_bin_keys     cell of every particle (48 bytes read), key = brick and cell
//                  inside it (4 written), histogram of the tile's bricks
//   k_rs_scan      per brick: offsets of the tiles (sort.hpp)
//   k_bin_base     offsets of the bricks, list of (brick, chunk) work items
//   k_bin_scatter  (charge, cell) to its place: 12 bytes read, 16 written
//   k_bin_deposit  one workgroup per chunk of a brick: 16 bytes read, LDS sums
//
// 96 bytes per particle, sequential but for one run of entries per tile and
// brick, against 56 bytes and an atomic.  The order inside a brick's run
// depends on timing; the sums are integers, so the grid does not.
//
// Moving the whole particle instead (a 64-byte record, deposit and kick on the
// records, rows gathered back) was measured: 10M / 127^3 443 us for the scatter
// and 224 for the way back against 226 us saved in the kick.
#pragma once
#include "particles.hpp"
#include "sort.hpp"

namespace ocsc {

constexpr int kBinYZ = 16;         // cells of a brick along y and z
constexpr int kBinMax = 4096;      // bricks of a mesh at most (LDS histogram of a tile)
constexpr int kBinTilePT = 512;    // threads of the key and scatter passes
constexpr int kBinChunk = 8192;    // entries per work item of the deposit
constexpr int kBinPT = 512;        // its threads
constexpr uint32_t kBinNone = 0xFFFFFFFFu;
constexpr int kBinLocalBits = 12;  // cells of a brick: at most 16^3

// bricks of 16 x 16 x 16 cells in the one-word form, 8 x 16 x 16 in the
// two-word form (32 KB of LDS in both) unless that gives more than kBinMax
struct BinShape {
  int sx;          // log2 of the cells along x
  int cx, cy, cz;  // bricks per axis
};
__host__ __device__ inline BinShape bin_shape(int nx, int ny, int nz, int nword) {
  BinShape s;
  s.cy = (ny + kBinYZ - 1) / kBinYZ;
  s.cz = (nz + kBinYZ - 1) / kBinYZ;
  s.sx = nword == 2 && (int64_t)((nx + 7) / 8) * s.cy * s.cz <= kBinMax ? 3 : 4;
  s.cx = (nx + (1 << s.sx) - 1) >> s.sx;
  return s;
}
__host__ __device__ inline int64_t bin_count(const BinShape& s) { return (int64_t)s.cx * s.cy * s.cz; }

struct alignas(16) BinEntry {
  double q;
  uint32_t cell;  // inside the brick
  uint32_t pad;
};

// entries of chunk number `chunk` of a brick with `total` entries (one brick
// can hold all of a bunch of up to 2^32 - 1 particles, so the rest of its
// entries is compared unsigned)
__host__ __device__ constexpr int bin_chunk_entries(uint32_t total, int chunk) {
  const uint32_t left = total - (uint32_t)chunk * kBinChunk;
  return left < (uint32_t)kBinChunk ? (int)left : kBinChunk;
}

// device buffers of one binned deposit
struct BinBufs {
  uint32_t* keys;    // n
  uint32_t* hist;    // bricks x tiles, brick-major, then the bricks' totals
  uint32_t* start;   // bricks: first entry
  int* nwork;        // work items
  int2* work;        // (brick, chunk of its entries), at most n / kBinChunk + bricks
  BinEntry* ent;     // n
  int items;         // particles per thread of a tile
  int64_t ntiles;
};

template <bool FAST>
__global__ void __launch_bounds__(kBinTilePT) k_bin_keys(Rows R, KickScalars* __restrict__ scp, uint32_t* __restrict__ keys,
                                                 uint32_t* __restrict__ H, int64_t ntiles, BinShape b, int items) {
  constexpr int PT = kBinTilePT;
  __shared__ uint32_t h[kBinMax];
  const KickScalars& s0 = *scp;
  if (s0.err) return;  // uniform across the grid
  const KickScalars s = s0;
  const int nb = b.cx * b.cy * b.cz;
  for (int i = threadIdx.x; i < nb; i += PT) h[i] = 0;
  __syncthreads();
  const int64_t base = (int64_t)blockIdx.x * (PT * items);
  int bad = 0;
  double cur[6], nxt[6] = {0, 0, 0, 0, 0, 0};
  int64_t p = base + threadIdx.x;
  if (p < s.n)
#pragma unroll
    for (int k = 0; k < 6; ++k) cur[k] = ldnt(R.r + k * R.ld + p);
  for (int it = 0; it < items && p < s.n; ++it, p += PT) {
    if (it + 1 < items && p + PT < s.n)
#pragma unroll
      for (int k = 0; k < 6; ++k) nxt[k] = ldnt(R.r + k * R.ld + p + PT);
    int c[3];
    uint32_t key = kBinNone;
    if (ngp_node<FAST>(cur, s, c)) {
      const int bin = ((c[0] >> b.sx) * b.cy + c[1] / kBinYZ) * b.cz + c[2] / kBinYZ;
      key = (uint32_t)bin << kBinLocalBits |
            (uint32_t)(((c[0] & ((1 << b.sx) - 1)) * kBinYZ + c[1] % kBinYZ) * kBinYZ + c[2] % kBinYZ);
      atomicAdd(&h[bin], 1u);
    } else {
      bad = 1;
    }
    keys[p] = key;
#pragma unroll
    for (int k = 0; k < 6; ++k) cur[k] = nxt[k];
  }
  if (bad) atomicOr(&scp->err, (int)kErrCell);
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += PT) H[(int64_t)i * ntiles + blockIdx.x] = h[i];
}

// first entries and work items of the bricks from their totals, one workgroup
__global__ void __launch_bounds__(1024) k_bin_base(const KickScalars* __restrict__ scp, const uint32_t* __restrict__ T,
                                                   int nb, uint32_t* __restrict__ start, int* __restrict__ nwork,
                                                   int2* __restrict__ work) {
  constexpr int kPer = kBinMax / 1024;
  __shared__ uint32_t we[16], wc[16], first[kBinMax];
  if (scp->err) {
    if (threadIdx.x == 0) *nwork = 0;
    return;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  uint32_t tot[kPer], e = 0, c = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = threadIdx.x * kPer + k;
    tot[k] = i < nb ? T[i] : 0u;
    e += tot[k];
    c += (tot[k] + kBinChunk - 1) / kBinChunk;
  }
  uint32_t xe = e, xc = c;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t ye = __shfl_up(xe, off), yc = __shfl_up(xc, off);
    if (lane >= off) {
      xe += ye;
      xc += yc;
    }
  }
  if (lane == 63) {
    we[w] = xe;
    wc[w] = xc;
  }
  __syncthreads();
  uint32_t pe = xe - e, pc = xc - c, all = 0;
  for (int k = 0; k < 16; ++k) {
    if (k < w) {
      pe += we[k];
      pc += wc[k];
    }
    all += wc[k];
  }
  if (threadIdx.x == 0) *nwork = (int)all;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = threadIdx.x * kPer + k;
    first[i] = pc;  // bricks past nb: all
    if (i < nb) start[i] = pe;
    pe += tot[k];
    pc += (tot[k] + kBinChunk - 1) / kBinChunk;
  }
  __syncthreads();
  // work item j belongs to the last brick whose first item is <= j
  for (int j = threadIdx.x; j < (int)all; j += 1024) {
    int lo = 0;
#pragma unroll
    for (int d = kBinMax / 2; d > 0; d >>= 1)
      if ((int)first[lo + d] <= j) lo += d;
    work[j] = make_int2(lo, j - (int)first[lo]);
  }
}

__global__ void __launch_bounds__(kBinTilePT) k_bin_scatter(const double* __restrict__ q,
                                                            const KickScalars* __restrict__ scp,
                                                            const uint32_t* __restrict__ keys,
                                                            const uint32_t* __restrict__ H, int64_t ntiles, int nb,
                                                            const uint32_t* __restrict__ start,
                                                            BinEntry* __restrict__ ent, int items) {
  constexpr int PT = kBinTilePT, U = 4;  // loads of U particles in flight per thread
  __shared__ uint32_t next[kBinMax];
  if (scp->err) return;  // uniform across the grid
  const int64_t n = scp->n;
  const int64_t base = (int64_t)blockIdx.x * (PT * items);
  const int64_t end = base + PT * items < n ? base + PT * items : n;
  for (int i = threadIdx.x; i < nb; i += PT) next[i] = start[i] + H[(int64_t)i * ntiles + blockIdx.x];
  __syncthreads();
  for (int64_t p0 = base + threadIdx.x; p0 < end; p0 += U * PT) {
    uint32_t key[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t p = p0 + u * PT;
      key[u] = p < end ? keys[p] : kBinNone;
      v[u] = p < end ? ldnt(q + p) : 0.0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (key[u] == kBinNone) continue;
      const uint32_t dst = atomicAdd(&next[key[u] >> kBinLocalBits], 1u);
      ent[dst] = BinEntry{v[u], key[u] & ((1u << kBinLocalBits) - 1), 0u};
    }
  }
}

// LDS: NWORD words per cell of a brick
template <int NWORD>
__global__ void __launch_bounds__(kBinPT) k_bin_deposit(const KickScalars* __restrict__ scp,
                                                        const uint32_t* __restrict__ T,
                                                        const uint32_t* __restrict__ start,
                                                        const int* __restrict__ nwork, const int2* __restrict__ work,
                                                        const BinEntry* __restrict__ ent,
                                                        unsigned long long* __restrict__ grid, BinShape b) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  unsigned long long* h = (unsigned long long*)smem_raw;
  if (scp->err || (int)blockIdx.x >= *nwork) return;  // uniform across the workgroup
  const int2 wk = work[blockIdx.x];
  const int words = (kBinYZ * kBinYZ * NWORD) << b.sx;
  for (int i = threadIdx.x; i < words; i += kBinPT) h[i] = 0ull;
  const int cnt = bin_chunk_entries(T[wk.x], wk.y);
  const BinEntry* e0 = ent + start[wk.x] + (uint32_t)wk.y * kBinChunk;
  const double qscale = scp->qscale;
  __syncthreads();
#pragma unroll 4
  for (int i = threadIdx.x; i < cnt; i += kBinPT) {
    const BinEntry e = e0[i];
    const double v = e.q * qscale;  // exact: qscale is a power of two
    const double hi = __builtin_rint(v);
    atomicAdd(&h[e.cell * NWORD], (unsigned long long)(long long)hi);
    if constexpr (NWORD == 2)
      atomicAdd(&h[e.cell * NWORD + 1], (unsigned long long)(long long)__builtin_rint((v - hi) * 0x1p30));
  }
  __syncthreads();
  const int nx = scp->nmesh[0], ny = scp->nmesh[1], nz = scp->nmesh[2];
  const int bz = wk.x % b.cz, t = wk.x / b.cz, by = t % b.cy, bx = t / b.cy;
  for (int i = threadIdx.x; i < words; i += kBinPT) {
    const unsigned long long v = h[i];
    if (!v) continue;
    const int c = i / NWORD, z = bz * kBinYZ + c % kBinYZ, y = by * kBinYZ + (c / kBinYZ) % kBinYZ,
              x = (bx << b.sx) + c / (kBinYZ * kBinYZ);
    if (x < nx && y < ny && z < nz) atomicAdd(&grid[(((int64_t)x * ny + y) * nz + z) * NWORD + i % NWORD], v);
  }
}

}  // namespace ocsc
