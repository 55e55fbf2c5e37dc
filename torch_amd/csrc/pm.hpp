// Particle-mesh pieces beside the bridge kick, on guarded FLASH leaf blocks, FP64:
// cloud-in-cell mass deposit, the finite-difference acceleration (optionally fused with the
// grid kick v += g dt) and cloud-in-cell interpolation to particles.
//
// Block layout: one variable of nblk blocks of nbg^3 cells (nbg = nb + 2 ng: nb interior
// cells per axis, ng guard layers), block b at b * nbg^3, cell (i, j, k) at
// (k * nbg + j) * nbg + i -- x fastest, as solnData(VAR, i, j, k) of one variable.  Block b
// has interior lower corner (ox, oy, oz)[b] and cubic physical size bs[b]; the cell width is
// del = bs / nb and guarded cell i has centre o + ((i - ng) + 0.5) del.
//
// All three are HBM / latency-bound elementwise work (no MFMA shape): one lane per cell for
// the gradient (x-fastest lanes, so each neighbour load of a wave is one or two contiguous
// segments), one lane per particle for the deposit and the interpolation.
//
// The deposit is deterministic: every contribution c = (m / del^3) w is split exactly into
// 64-bit integers, c 2^S = H 2^32 + L (0 <= L < 2^32; S per cell, from the largest |c| the
// cell receives), and H and L are summed with integer atomics, which do not depend on the
// order of the adds.  A cell's density (H 2^32 + L) 2^-S is then within an ulp of the exact
// sum of its contributions (each is truncated to ~2^-66 of the cell's largest one).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

struct PmBlocks {
  const double *ox, *oy, *oz, *bs;
  int64_t nblk;
  int nb, ng, nbg;
  int64_t nc;   // nbg^3
};

// Cloud-in-cell weights along one axis (the oracle's cic_axis, same operations in the same
// order): u = (x - o) / del - 0.5 + ng, base cell floor(u), weights (1 - f, f).
__device__ __forceinline__ bool pm_axis(double x, double o, double del, int ng, int nbg, int& i0,
                                        double& w0, double& w1) {
  double u;
  {
#pragma clang fp contract(off)
    u = (x - o) / del - 0.5 + (double)ng;
  }
  const double fl = floor(u);
  if (!(fl >= 0.0 && fl + 1.0 < (double)nbg)) return false;
  i0 = (int)fl;
  w1 = u - fl;
  w0 = 1.0 - w1;
  return true;
}

// Scale exponent of one cell's fixed-point sum from cmax = bits of the largest |c| among the
// cell's contributions: np * cmax < 2^e, S = 94 - e keeps every partial sum of H below 2^62
// and resolves each contribution to 2^-66 of that cell's largest one.
__device__ __forceinline__ int pm_scale(unsigned long long cmax, int64_t np) {
  const double mx = __longlong_as_double((long long)cmax);
  if (!(mx > 0.0 && mx < 1e300)) return 0;
  int e;
  frexp(mx * (double)np, &e);
  return 94 - e;
}

// c 2^S = H 2^32 + L exactly, 0 <= L < 2^32, and back from the sums of H and L.
__device__ __forceinline__ void pm_split(double c, int S, unsigned long long& H, unsigned long long& L) {
  const double t = ldexp(c, S - 32);
  const double h = floor(t);
  H = (unsigned long long)(long long)h;
  L = (unsigned long long)ldexp(t - h, 32);
}
__device__ __forceinline__ double pm_value(unsigned long long H, unsigned long long L, int S) {
  return ldexp((double)(long long)H, 32 - S) + ldexp((double)L, -S);
}

// Particle p's block, densities and weights; false if the block index or the CIC stencil
// is outside the guarded block.
__device__ __forceinline__ bool pm_particle(const PmBlocks& B, const int64_t* blk, int64_t p,
                                            double x, double y, double z, int64_t& b, double& del,
                                            int (&c0)[3], double (&w)[3][2]) {
  b = blk[p];
  if (b < 0 || b >= B.nblk) return false;
  del = B.bs[b] / (double)B.nb;
  return pm_axis(x, B.ox[b], del, B.ng, B.nbg, c0[0], w[0][0], w[0][1]) &&
         pm_axis(y, B.oy[b], del, B.ng, B.nbg, c0[1], w[1][0], w[1][1]) &&
         pm_axis(z, B.oz[b], del, B.ng, B.nbg, c0[2], w[2][0], w[2][1]);
}

// The 8 contributions of particle p: c = (m / del^3) ((wx wy) wz) with the oracle's
// roundings, corners dk slowest, di fastest.  Calls f(cell index, c).
template <class F>
__device__ __forceinline__ bool pm_corners(const PmBlocks& B, const double* x, const double* y,
                                           const double* z, const double* m, const int64_t* blk,
                                           int64_t p, F f) {
  int64_t b;
  double del;
  int c0[3];
  double w[3][2];
  if (!pm_particle(B, blk, p, x[p], y[p], z[p], b, del, c0, w)) return false;
  const double md = m[p] / ((del * del) * del);
  const int64_t base = b * B.nc;
#pragma unroll
  for (int dk = 0; dk < 2; ++dk)
#pragma unroll
    for (int dj = 0; dj < 2; ++dj)
#pragma unroll
      for (int di = 0; di < 2; ++di) {
#pragma clang fp contract(off)
        const double c = md * ((w[0][di] * w[1][dj]) * w[2][dk]);
        f(base + ((int64_t)(c0[2] + dk) * B.nbg + (c0[1] + dj)) * B.nbg + (c0[0] + di), c);
      }
  return true;
}

// Pass 1: cmax[cell] = max |c| over the cell's contributions (as non-negative double bits,
// whose unsigned order is the numeric order); a bad particle sets *err (may be null).
__global__ void k_pm_cell_max(int64_t np, const double* __restrict__ x, const double* __restrict__ y,
                              const double* __restrict__ z, const double* __restrict__ m,
                              const int64_t* __restrict__ blk, PmBlocks B, unsigned long long* cmax,
                              unsigned long long* err) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  const bool ok = pm_corners(B, x, y, z, m, blk, p, [&](int64_t idx, double c) {
    const unsigned long long bits = (unsigned long long)__double_as_longlong(fabs(c));
    if (bits) atomicMax(&cmax[idx], bits);
  });
  if (!ok && err) *err = 1ULL;   // every writer stores the same value
}

// Pass 2: accH / accL += the exact integer split c 2^S = H 2^32 + L of every contribution,
// S from the cell's bound.
__global__ void k_pm_deposit(int64_t np, const double* __restrict__ x, const double* __restrict__ y,
                             const double* __restrict__ z, const double* __restrict__ m,
                             const int64_t* __restrict__ blk, PmBlocks B,
                             const unsigned long long* __restrict__ cmax, unsigned long long* accH,
                             unsigned long long* accL) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  pm_corners(B, x, y, z, m, blk, p, [&](int64_t idx, double c) {
    unsigned long long h, l;
    pm_split(c, pm_scale(cmax[idx], np), h, l);
    atomicAdd(&accH[idx], h);
    atomicAdd(&accL[idx], l);
  });
}

// Pass 3: rho = (H 2^32 + L) 2^-S (or rho += that with accumulate).
__global__ void k_pm_finalize(int64_t n, const unsigned long long* __restrict__ accH,
                              const unsigned long long* __restrict__ accL,
                              const unsigned long long* __restrict__ cmax, int64_t np,
                              double* __restrict__ rho, int accumulate) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double v = pm_value(accH[i], accL[i], pm_scale(cmax[i], np));
  rho[i] = accumulate ? rho[i] + v : v;
}

// ---- the deposit block by block, in LDS (guarded blocks of at most TG_PM_LDS_CELLS cells) ----
// The passes above move 56 B per cell through memory (zero three words, read them back, write rho) for
// particles that touch a few cells of some blocks.  Here the particles are binned by block, and one
// workgroup per block keeps the three words of its cells in LDS, TG_PM_LDS_SLICE cells at a time, and
// writes each cell's density once: 8 B per cell.  The sums are integers (and a maximum), so the order
// of a block's particles does not matter and the densities are the ones above, bit for bit.
// 8.2 million cells, 10,000 particles: 89 us for the passes above, 30 us here and 14 for the binning.
#define TG_PM_LDS_CELLS 8192
#define TG_PM_LDS_SLICE 2048     // 48 KB: three workgroups per CU

// n zeroes (counts, then the offsets' total and the error word).
__global__ void k_zero_u32(int64_t n, unsigned int* a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0u;
}

// rank[p] = particle p's place among its block's particles (any order); ~0u and *err for a bad particle.
// The lanes of a wave that share a block take one atomic, for up to 8 blocks.
__global__ __launch_bounds__(256) void k_pm_bin(int64_t np, const double* __restrict__ x, const double* __restrict__ y,
                                                const double* __restrict__ z, const int64_t* __restrict__ blk,
                                                PmBlocks B, unsigned int* cnt, int cs,
                                                unsigned int* __restrict__ rank, unsigned long long* err) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool in = p < np;        // every lane stays for the wave's shuffle
  int64_t b = 0;
  double del, w[3][2];
  int c0[3];
  const bool ok = in && pm_particle(B, blk, p, x[p], y[p], z[p], b, del, c0, w);
  const unsigned int mine = ok ? (unsigned int)b : ~0u;
  unsigned long long left = __builtin_amdgcn_ballot_w64(ok);
  int lead = lane;               // the lane that counts for this one, for how many, and this one's place
  unsigned int n = 1u, r = 0u;
  for (int i = 0; i < 8 && left; ++i) {
    const int first = __builtin_ctzll(left);
    const bool same = mine == (unsigned int)__builtin_amdgcn_readlane((int)mine, first);
    const unsigned long long group = __builtin_amdgcn_ballot_w64(same);
    if (same) {
      lead = first;
      n = (unsigned int)__builtin_popcountll(group);
      r = (unsigned int)__builtin_popcountll(group & ((1ULL << lane) - 1ULL));
    }
    left &= ~group;
  }
  unsigned int base = 0u;
  if (ok && lead == lane) base = atomicAdd(&cnt[b * cs], n);
  base = (unsigned int)__shfl((int)base, lead);
  if (!in) return;
  rank[p] = ok ? base + r : ~0u;
  if (!ok && err) *err = 1ULL;   // every writer stores the same value
}

// Blocks of more than TG_PM_HEAVY particles ("heavy") are summed by several workgroups, TG_PM_SEG particles
// each (k_pm_heavy_max, k_pm_heavy_sum), into words in memory: one workgroup takes ~30 ns per particle, and a
// cluster inside one or a few blocks left the rest of the chip idle.  A call of 2,000 blocks of 16^3 cells with
// all of its particles in one: 10,000 86 us (315 by one workgroup, 118 by the passes over memory), 100,000 91
// (3,248; 311), 1,000,000 357 (33,000; 2,306); in eight of them 86 (75; 111), 92 (475; 212), 405 (4,645;
// 1,288).  The line at 512: 1,000 particles in one block 86 us against 50; at 2,048: 2,000 in one 53 against 40.
#define TG_PM_HEAVY 1024
#define TG_PM_SEG 1024
struct PmHeavy {
  unsigned int block, seg;       // its first workgroup among all heavy blocks'
  unsigned int off, cnt;         // its stretch of perm
};

// off[b]: a stretch of perm for each block with particles, in whatever order the workgroups come.  slot[b]: a
// heavy block's place in `list` (ascending in seg: one counter, blocks in its high word and workgroups in its
// low word, gives both), else ~0u; *any (may be null) is set if there is one.
__global__ __launch_bounds__(256) void k_pm_offsets(int64_t nblk, const unsigned int* __restrict__ cnt, int cs,
                                                    unsigned int* __restrict__ off, unsigned int* total,
                                                    unsigned int* __restrict__ slot, unsigned long long* nheavy,
                                                    PmHeavy* __restrict__ list, unsigned long long* any) {
  __shared__ unsigned int wsum[4], start;
  const int64_t b = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const unsigned int n = b < nblk ? cnt[b * cs] : 0u;
  unsigned int s = n;            // inclusive sum over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned int t = __shfl_up(s, o);
    if (lane >= o) s += t;
  }
  if (lane == 63) wsum[w] = s;
  __syncthreads();
  if (threadIdx.x == 0) start = atomicAdd(total, wsum[0] + wsum[1] + wsum[2] + wsum[3]);
  __syncthreads();
  unsigned int at = start + s - n;
  for (int q = 0; q < w; ++q) at += wsum[q];
  if (b >= nblk) return;
  off[b] = at;
  unsigned int h = ~0u;
  if (n > TG_PM_HEAVY) {
    const unsigned long long r = atomicAdd(nheavy, (1ULL << 32) | ((n + TG_PM_SEG - 1) / TG_PM_SEG));
    h = (unsigned int)(r >> 32);
    list[h] = {(unsigned int)b, (unsigned int)r, at, n};
    if (any) *any = 1ULL;        // every writer stores the same value
  }
  slot[b] = h;
}

// perm from the ranks; workgroups from nscatter on clear one heavy block's words each (block h's at h * nc).
__global__ __launch_bounds__(256) void k_pm_scatter(int64_t np, const int64_t* __restrict__ blk,
                                                    const unsigned int* __restrict__ rank,
                                                    const unsigned int* __restrict__ off,
                                                    unsigned int* __restrict__ perm, unsigned int nscatter,
                                                    const unsigned long long* __restrict__ nheavy, int64_t nc,
                                                    unsigned long long* M, unsigned long long* H,
                                                    unsigned long long* L) {
  if (blockIdx.x >= nscatter) {
    const unsigned int h = blockIdx.x - nscatter;
    if (h >= (unsigned int)(*nheavy >> 32)) return;
    const int64_t at = (int64_t)h * nc;
    for (int64_t i = at + threadIdx.x; i < at + nc; i += 256) M[i] = H[i] = L[i] = 0ULL;
    return;
  }
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= np) return;
  const unsigned int r = rank[p];
  if (r != ~0u) perm[off[blk[p]] + r] = (unsigned int)p;
}

// The cells [lo, lo + len) of block b in LDS: M = max |c|, then H and L += the split of every contribution
// of particles perm[q0 ... q1).  512 lanes.
__device__ __forceinline__ void pm_lds_max(unsigned long long* M, int lo, int len, int64_t base, unsigned int q0,
                                           unsigned int q1, const unsigned int* __restrict__ perm,
                                           const double* __restrict__ x, const double* __restrict__ y,
                                           const double* __restrict__ z, const double* __restrict__ m,
                                           const int64_t* __restrict__ blk, const PmBlocks& B) {
  for (unsigned int q = q0 + threadIdx.x; q < q1; q += 512)
    pm_corners(B, x, y, z, m, blk, (int64_t)perm[q], [&](int64_t idx, double c) {
      const int i = (int)(idx - base) - lo;
      const unsigned long long bits = (unsigned long long)__double_as_longlong(fabs(c));
      if (bits && i >= 0 && i < len) atomicMax(&M[i], bits);
    });
}
__device__ __forceinline__ void pm_lds_sum(const unsigned long long* M, unsigned long long* H, unsigned long long* L,
                                           int lo, int len, int64_t base, unsigned int q0, unsigned int q1,
                                           const unsigned int* __restrict__ perm, int64_t np,
                                           const double* __restrict__ x, const double* __restrict__ y,
                                           const double* __restrict__ z, const double* __restrict__ m,
                                           const int64_t* __restrict__ blk, const PmBlocks& B) {
  for (unsigned int q = q0 + threadIdx.x; q < q1; q += 512)
    pm_corners(B, x, y, z, m, blk, (int64_t)perm[q], [&](int64_t idx, double c) {
      const int i = (int)(idx - base) - lo;
      if (i < 0 || i >= len) return;
      unsigned long long h, l;
      pm_split(c, pm_scale(M[i], np), h, l);
      atomicAdd(&H[i], h);
      atomicAdd(&L[i], l);
    });
}

// Workgroup i of the heavy blocks': its block's entry and its particles perm[q0 ... q1); false past the last.
__device__ __forceinline__ bool pm_heavy_part(const unsigned long long* __restrict__ nheavy,
                                              const PmHeavy* __restrict__ list, unsigned int i, unsigned int& h,
                                              PmHeavy& e, unsigned int& q0, unsigned int& q1) {
  const unsigned long long n = *nheavy;
  if (i >= (unsigned int)n) return false;
  unsigned int lo = 0, hi = (unsigned int)(n >> 32);   // list[lo].seg <= i < list[hi].seg
  while (hi - lo > 1) {
    const unsigned int mid = (lo + hi) / 2;
    if (list[mid].seg <= i) lo = mid;
    else hi = mid;
  }
  h = lo;
  e = list[lo];
  q0 = e.off + (i - e.seg) * TG_PM_SEG;
  q1 = e.off + e.cnt;
  if (q1 - q0 > TG_PM_SEG) q1 = q0 + TG_PM_SEG;
  return true;
}

// blockIdx.x = workgroup of the heavy blocks', blockIdx.y = slice of TG_PM_LDS_SLICE cells.
__global__ __launch_bounds__(512) void k_pm_heavy_max(const unsigned long long* __restrict__ nheavy,
                                                      const PmHeavy* __restrict__ list, const double* __restrict__ x,
                                                      const double* __restrict__ y, const double* __restrict__ z,
                                                      const double* __restrict__ m, const int64_t* __restrict__ blk,
                                                      PmBlocks B, const unsigned int* __restrict__ perm,
                                                      unsigned long long* Mg) {
  __shared__ unsigned long long M[TG_PM_LDS_SLICE];
  unsigned int h, q0, q1;
  PmHeavy e;
  if (!pm_heavy_part(nheavy, list, blockIdx.x, h, e, q0, q1)) return;   // uniform over the workgroup
  const int lo = (int)blockIdx.y * TG_PM_LDS_SLICE, nc = (int)B.nc;
  const int len = nc - lo < TG_PM_LDS_SLICE ? nc - lo : TG_PM_LDS_SLICE;
  for (int i = threadIdx.x; i < len; i += 512) M[i] = 0ULL;
  __syncthreads();
  pm_lds_max(M, lo, len, (int64_t)e.block * B.nc, q0, q1, perm, x, y, z, m, blk, B);
  __syncthreads();
  for (int i = threadIdx.x; i < len; i += 512)
    if (M[i]) atomicMax(&Mg[(int64_t)h * B.nc + lo + i], M[i]);
}

__global__ __launch_bounds__(512) void k_pm_heavy_sum(const unsigned long long* __restrict__ nheavy,
                                                      const PmHeavy* __restrict__ list, int64_t np,
                                                      const double* __restrict__ x, const double* __restrict__ y,
                                                      const double* __restrict__ z, const double* __restrict__ m,
                                                      const int64_t* __restrict__ blk, PmBlocks B,
                                                      const unsigned int* __restrict__ perm,
                                                      const unsigned long long* __restrict__ Mg,
                                                      unsigned long long* Hg, unsigned long long* Lg) {
  __shared__ unsigned long long M[TG_PM_LDS_SLICE], H[TG_PM_LDS_SLICE], L[TG_PM_LDS_SLICE];
  unsigned int h, q0, q1;
  PmHeavy e;
  if (!pm_heavy_part(nheavy, list, blockIdx.x, h, e, q0, q1)) return;
  const int lo = (int)blockIdx.y * TG_PM_LDS_SLICE, nc = (int)B.nc;
  const int len = nc - lo < TG_PM_LDS_SLICE ? nc - lo : TG_PM_LDS_SLICE;
  const int64_t at = (int64_t)h * B.nc + lo;
  for (int i = threadIdx.x; i < len; i += 512) {
    M[i] = Mg[at + i];
    H[i] = L[i] = 0ULL;
  }
  __syncthreads();
  pm_lds_sum(M, H, L, lo, len, (int64_t)e.block * B.nc, q0, q1, perm, np, x, y, z, m, blk, B);
  __syncthreads();
  for (int i = threadIdx.x; i < len; i += 512)
    if (M[i]) {
      if (H[i]) atomicAdd(&Hg[at + i], H[i]);
      if (L[i]) atomicAdd(&Lg[at + i], L[i]);
    }
}

// One workgroup of 512 lanes per block; a heavy block's sums are in memory already (Mg, Hg, Lg).
__global__ __launch_bounds__(512) void k_pm_block(int64_t np, const double* __restrict__ x,
                                                  const double* __restrict__ y, const double* __restrict__ z,
                                                  const double* __restrict__ m, const int64_t* __restrict__ blk,
                                                  PmBlocks B, const unsigned int* __restrict__ cnt, int cs,
                                                  const unsigned int* __restrict__ off,
                                                  const unsigned int* __restrict__ perm,
                                                  const unsigned int* __restrict__ slot,
                                                  const unsigned long long* __restrict__ Mg,
                                                  const unsigned long long* __restrict__ Hg,
                                                  const unsigned long long* __restrict__ Lg,
                                                  double* __restrict__ rho, int accumulate) {
  __shared__ unsigned long long M[TG_PM_LDS_SLICE], H[TG_PM_LDS_SLICE], L[TG_PM_LDS_SLICE];
  const int64_t b = blockIdx.x, base = b * B.nc;
  const int nc = (int)B.nc;
  const unsigned int n = cnt[b * cs];
  if (n == 0u) {                 // uniform over the workgroup, as the next test
    for (int i = threadIdx.x; i < nc; i += 512) rho[base + i] = accumulate ? rho[base + i] + 0.0 : 0.0;
    return;
  }
  if (n > TG_PM_HEAVY) {
    const int64_t at = (int64_t)slot[b] * B.nc;
    for (int i = threadIdx.x; i < nc; i += 512) {
      const unsigned long long mx = Mg[at + i];
      const double v = mx ? pm_value(Hg[at + i], Lg[at + i], pm_scale(mx, np)) : 0.0;
      rho[base + i] = accumulate ? rho[base + i] + v : v;
    }
    return;
  }
  const unsigned int o = off[b];
  for (int lo = 0; lo < nc; lo += TG_PM_LDS_SLICE) {
    const int len = nc - lo < TG_PM_LDS_SLICE ? nc - lo : TG_PM_LDS_SLICE;
    for (int i = threadIdx.x; i < len; i += 512) M[i] = H[i] = L[i] = 0ULL;
    __syncthreads();
    pm_lds_max(M, lo, len, base, o, o + n, perm, x, y, z, m, blk, B);
    __syncthreads();
    pm_lds_sum(M, H, L, lo, len, base, o, o + n, perm, np, x, y, z, m, blk, B);
    __syncthreads();
    for (int i = threadIdx.x; i < len; i += 512) {
      const double v = M[i] ? pm_value(H[i], L[i], pm_scale(M[i], np)) : 0.0;
      const int64_t t = base + lo + i;
      rho[t] = accumulate ? rho[t] + v : v;
    }
    __syncthreads();
  }
}

__global__ void k_zero_u64(int64_t n, unsigned long long* a, unsigned long long* b,
                           unsigned long long* c) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  a[i] = 0ULL;
  if (b) b[i] = 0ULL;
  if (c) c[i] = 0ULL;
}

// g = -grad(phi) by the row rule delxinv (phi(i-1) - phi(i+1)), delxinv = 0.5 (nb / bs), the
// two ends of each row copying their neighbour; any of gx/gy/gz may be null.  With vx != null
// also the grid kick v += g dt (product and sum rounded separately).
// Grid: x = slice * 8 + (b mod 8), y = b / 8 - grp0, where a slice is 256 consecutive cells of
// a block.  Workgroups are dealt to the 8 XCDs round-robin by linear id (x fastest, gridDim.x a
// multiple of 8), so all slices of block b run on XCD (b mod 8) and a block's z-neighbour reads
// hit the L2 that its other slices filled.  Cell (i, j, k) comes from the slice offset r by two
// divisions by nbg done as multiply-high with m = ceil(2^32 / nbg), exact for r < 2^32 / nbg
// (nbg <= 128 and r < 2^21 here).
__global__ __launch_bounds__(256) void k_pm_gradient(PmBlocks B, uint32_t magic, int64_t grp0,
                                                     const double* __restrict__ phi,
                                                     double* __restrict__ gx, double* __restrict__ gy,
                                                     double* __restrict__ gz, double dt,
                                                     double* __restrict__ vx, double* __restrict__ vy,
                                                     double* __restrict__ vz) {
  const int64_t b = (grp0 + blockIdx.y) * 8 + (blockIdx.x & 7u);
  if (b >= B.nblk) return;
  const uint32_t r = (blockIdx.x >> 3) * 256u + threadIdx.x;
  if (r >= (uint32_t)B.nc) return;
  const int n = B.nbg;
  const uint32_t q = __umulhi(r, magic);        // r / n
  const uint32_t k = __umulhi(q, magic);        // r / n^2
  const int c[3] = {(int)(r - q * (uint32_t)n), (int)(q - k * (uint32_t)n), (int)k};
  const int stride[3] = {1, n, n * n};
  double delxinv = (double)B.nb / B.bs[b];
  delxinv = 0.5 * delxinv;
  const double* f = phi + b * B.nc;
  double g[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int ii = c[a] < 1 ? 1 : (c[a] > n - 2 ? n - 2 : c[a]);
    const int ctr = (int)r + (ii - c[a]) * stride[a];
    g[a] = delxinv * (f[ctr - stride[a]] - f[ctr + stride[a]]);
  }
  const int64_t t = b * B.nc + r;
  if (gx) gx[t] = g[0];
  if (gy) gy[t] = g[1];
  if (gz) gz[t] = g[2];
  if (vx) {
#pragma clang fp contract(off)
    vx[t] = vx[t] + g[0] * dt;
    vy[t] = vy[t] + g[1] * dt;
    vz[t] = vz[t] + g[2] * dt;
  }
}

// a_p = sum over the 8 corners of w g (corner order and roundings of the oracle).  A
// particle outside its guarded block gets NaN and sets *err (may be null).
__global__ void k_pm_interpolate(int64_t np, const double* __restrict__ x,
                                 const double* __restrict__ y, const double* __restrict__ z,
                                 const int64_t* __restrict__ blk, PmBlocks B,
                                 const double* __restrict__ gx, const double* __restrict__ gy,
                                 const double* __restrict__ gz, double* __restrict__ ax,
                                 double* __restrict__ ay, double* __restrict__ az,
                                 unsigned long long* err) {
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= np) return;
  int64_t b;
  double del;
  int c0[3];
  double w[3][2];
  if (!pm_particle(B, blk, p, x[p], y[p], z[p], b, del, c0, w)) {
    if (err) *err = 1ULL;        // every writer stores the same value
    ax[p] = ay[p] = az[p] = __longlong_as_double(0x7ff8000000000000LL);
    return;
  }
  const int64_t base = b * B.nc;
  double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
  for (int dk = 0; dk < 2; ++dk)
#pragma unroll
    for (int dj = 0; dj < 2; ++dj)
#pragma unroll
      for (int di = 0; di < 2; ++di) {
#pragma clang fp contract(off)
        const int64_t idx = base + ((int64_t)(c0[2] + dk) * B.nbg + (c0[1] + dj)) * B.nbg + (c0[0] + di);
        const double wt = (w[0][di] * w[1][dj]) * w[2][dk];
        sx = sx + wt * gx[idx];
        sy = sy + wt * gy[idx];
        sz = sz + wt * gz[idx];
      }
  ax[p] = sx;
  ay[p] = sy;
  az[p] = sz;
}

// Particle accelerations straight from the potential: the row rule of k_pm_gradient at the 8 corners of
// each particle's cloud, then the CIC sum of k_pm_interpolate, with the same operations in the same
// order (same bits) and without the three block arrays between them: a whole gradient writes 24 B and
// reads 8 B per cell (62 us for 8.2 million cells) for the few cells that particles touch.  8 lanes per
// particle, one per corner (6 loads each instead of 48 in a chain): 10,000 particles in 6 us.
__global__ __launch_bounds__(256) void k_pm_long_range(int64_t np, const double* __restrict__ x,
                                                       const double* __restrict__ y, const double* __restrict__ z,
                                                       const int64_t* __restrict__ blk, PmBlocks B,
                                                       const double* __restrict__ phi, double* __restrict__ ax,
                                                       double* __restrict__ ay, double* __restrict__ az,
                                                       unsigned long long* err) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, p = i >> 3;
  const int corner = (int)(i & 7), first = (int)(threadIdx.x & 63) & ~7;
  const bool in = p < np;        // whole groups of 8 lanes
  int64_t b = 0;
  double del = 1.0, w[3][2] = {{0.0, 0.0}, {0.0, 0.0}, {0.0, 0.0}};
  int c0[3] = {0, 0, 0};
  const bool ok = in && pm_particle(B, blk, p, x[p], y[p], z[p], b, del, c0, w);
  double q[3] = {0.0, 0.0, 0.0};   // weight times the corner's acceleration
  if (ok) {
    const int n = B.nbg, d[3] = {corner & 1, (corner >> 1) & 1, corner >> 2};
    const int c[3] = {c0[0] + d[0], c0[1] + d[1], c0[2] + d[2]};
    const int stride[3] = {1, n, n * n};
    const int r = (c[2] * n + c[1]) * n + c[0];
    const double* f = phi + b * B.nc;
    double delxinv = (double)B.nb / B.bs[b];
    delxinv = 0.5 * delxinv;
    const double wt = ((d[0] ? w[0][1] : w[0][0]) * (d[1] ? w[1][1] : w[1][0])) * (d[2] ? w[2][1] : w[2][0]);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int ii = c[a] < 1 ? 1 : (c[a] > n - 2 ? n - 2 : c[a]);
      const int ctr = r + (ii - c[a]) * stride[a];
      q[a] = wt * (delxinv * (f[ctr - stride[a]] - f[ctr + stride[a]]));
    }
  }
  double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 8; ++k)    // corners di fastest, dk slowest
#pragma unroll
    for (int a = 0; a < 3; ++a) s[a] = s[a] + __shfl(q[a], first + k);
  if (!in || corner != 0) return;
  if (!ok) {
    if (err) *err = 1ULL;
    s[0] = s[1] = s[2] = __longlong_as_double(0x7ff8000000000000LL);
  }
  ax[p] = s[0];
  ay[p] = s[1];
  az[p] = s[2];
}

}  // namespace tg
