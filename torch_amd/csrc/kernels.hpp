// Device code of the direct-sum field: target loaders, the per-tile interaction loops
// (FP64 and mixed precision), the per-workgroup driver shared by the grid kernels and
// the persistent batch kernel, and the small elementwise kernels around them.
//
// Execution model (gfx950, wave64):
//   * a workgroup of NT lanes owns a target tile of K*NT targets (K per lane, held in
//     VGPRs; target t = tile0 + k*NT + lane, so every load/store is coalesced);
//   * sources stream through LDS in tiles of NT (one source staged per lane per tile);
//     every lane then reads the same LDS word (broadcast, no bank conflicts) and updates
//     its K targets;
//   * the source range may be a chunk of the full set (split over blockIdx.y or over
//     work items); chunk partial sums then go to a scratch array and a second kernel
//     sums them in fixed order, so results are deterministic (no float atomics).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tg {

// ----------------------------------------------------------------- descriptors ----
struct Tgt {
  const double *x, *y, *z, *eps;           // explicit targets (eps may be null)
  const double *ox, *oy, *oz, *bdx, *beps; // block-structured targets
  int64_t n;
  int nb;
  int blocks;
};

struct Out {
  double *ax, *ay, *az, *phi;   // final outputs (any may be null)
  double *vx, *vy, *vz;         // fused kick v += dt * a (null = no kick)
  double dt;
  double *part;                 // non-null: write unscaled chunk sums to part[q*pstride + t]
  int64_t pstride;
  double G;
  int nopot = 0;                // 1: the potential is not wanted (its accumulator is skipped)
  int noacc = 0;                // 1: only the potential is wanted (no acceleration, no kick)
  const int* gate = nullptr;    // non-null: the kernel runs only if *gate == gate_on, else it
  int gate_on = 0;              //   returns at once (one of several launches picked on the device)
};

// Uniform across the grid: every workgroup of a gated-off launch returns before any barrier.
__device__ __forceinline__ bool gated_off(const Out& O) { return O.gate && *O.gate != O.gate_on; }

// Cell centre of block-structured target t: o + (idx + 1/2) dx with the multiply and the
// add rounded separately (no FMA contraction) so the centres are bit-identical to the
// host-side construction (numpy / C: o + (i + 0.5) * dx).
__device__ __forceinline__ void load_target(const Tgt& T, int64_t t, double& x, double& y,
                                            double& z, double& e2) {
  if (!T.blocks) {
    x = T.x[t];
    y = T.y[t];
    z = T.z[t];
    const double e = T.eps ? T.eps[t] : 0.0;
    e2 = e * e;
  } else {
    const int nb = T.nb;
    const int64_t nb3 = (int64_t)nb * nb * nb;
    const int64_t b = t / nb3;
    const int c = (int)(t - b * nb3);
    const int i = c / (nb * nb), j = (c / nb) % nb, k = c % nb;
    const double d = T.bdx[b];
    {
#pragma clang fp contract(off)
      x = T.ox[b] + ((double)i + 0.5) * d;
      y = T.oy[b] + ((double)j + 0.5) * d;
      z = T.oz[b] + ((double)k + 0.5) * d;
    }
    const double e = T.beps ? T.beps[b] : 0.0;
    e2 = e * e;
  }
}

// Min/max over the workgroup of NV values per lane: xor-shuffle within the wave, then
// one LDS slot per wave.  `red` holds 2*NV*(NT/64) doubles and is private to this call.
template <int NT, int NV>
__device__ __forceinline__ void block_minmax(double (&mn)[NV], double (&mx)[NV], double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      mn[v] = fmin(mn[v], __shfl_xor(mn[v], off));
      mx[v] = fmax(mx[v], __shfl_xor(mx[v], off));
    }
  }
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      red[(w * NV + v) * 2] = mn[v];
      red[(w * NV + v) * 2 + 1] = mx[v];
    }
  }
  __syncthreads();
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    mn[v] = red[v * 2];
    mx[v] = red[v * 2 + 1];
  }
#pragma unroll
  for (int w2 = 1; w2 < NT / 64; ++w2) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      mn[v] = fmin(mn[v], red[(w2 * NV + v) * 2]);
      mx[v] = fmax(mx[v], red[(w2 * NV + v) * 2 + 1]);
    }
  }
  __syncthreads();
}

// --------------------------------------------------------------- inner-loop flags ----
// Per-tile code path, chosen at run time once per workgroup (a uniform branch), compiled
// as separate loops:
//   F_GUARD  the tile's smallest possible eps^2 is 0: zero r2 -> the pair contributes 0
//   F_UNIF   all targets of the tile share eps_t^2: folded into the staged source eps^2
//   F_NOPOT  the caller did not ask for the potential
//   F_NOACC  the caller asked for the potential only (never together with F_NOPOT)
enum { F_GUARD = 1, F_UNIF = 2, F_NOPOT = 4, F_NOACC = 8 };

// --------------------------------------------------------------- FP64 tile loop ----
// 1/sqrt(r2) in FP64: a hardware estimate refined by one third-order Newton/Householder
// step  y <- y + y e (1/2 + 3/8 e),  e = 1 - r2 y^2  (the Taylor series of (1-e)^(-1/2);
// an estimate with relative error d leaves ~2.5 d^3, below FP64 rounding for d ~ 2^-24).
__device__ __forceinline__ double refine_rsqrt(double r2, double y) {
  const double t = r2 * y;
  const double e = fma(-t, y, 1.0);
  const double p = fma(e, 0.375, 0.5);
  const double q = y * e;
  return fma(q, p, y);
}
template <int FL>
__device__ __forceinline__ double rsqrt_f64(double r2) {
  double y = __builtin_amdgcn_rsq(r2);
  if (FL & F_GUARD) y = r2 > 0.0 ? y : 0.0;   // |d|^2 + eps^2 == 0: the pair contributes 0
  return refine_rsqrt(r2, y);
}

// Pairs per group of the FP64 tile loop (their v_rsq_f64 first, then the refinements): 20,011
// points x 5,003 sources 149 us per call in groups of 8 against 153 of 4.
#define TG_FP64_GROUP 8
// F_GUARD for a group of pairs: y[q] = 0 where r2[q] == 0.  Zero pairs are rare (a point on an unsoftened
// source), so the group is tested at once -- the smallest of its r2's high words, which no r2 >= 2^-1042
// has zero -- and the selects are in a branch the wave takes only then: 5 instructions for 8 pairs instead
// of 24.
template <int N>
__device__ __forceinline__ void guard_zero(const double (&r2)[N], double (&y)[N]) {
  unsigned h = (unsigned)__double2hiint(r2[0]);
#pragma unroll
  for (int q = 1; q < N; ++q) h = min(h, (unsigned)__double2hiint(r2[q]));
  if (__builtin_expect(__builtin_amdgcn_ballot_w64(h == 0u) != 0ULL, 0)) {
    asm volatile("");             // keeps the selects inside the branch
#pragma unroll
    for (int q = 0; q < N; ++q) y[q] = r2[q] > 0.0 ? y[q] : 0.0;
  }
}

// Sources 0 .. cnt - 1 of the staged tile, rounded up to a multiple of 8 (the padding adds nothing).
template <int K, int NT, int FL>
__device__ __forceinline__ void fp64_tile(const double4* __restrict__ s4,
                                          const double* __restrict__ se2, int cnt,
                                          const double (&tx)[K], const double (&ty)[K],
                                          const double (&tz)[K], const double (&te2)[K],
                                          double (&ax)[K], double (&ay)[K], double (&az)[K],
                                          double (&ap)[K]) {
  // K = 8 fills a group by itself and has no registers left for one: pair by pair (10^6 points x 8,193
  // unsoftened sources 6,040 us per call against 6,360, 8,193 x 10^6 softened 5,795 against 6,305).
  if constexpr (K >= 8) {
#pragma unroll 2
    for (int j = 0; j < cnt; ++j) {
      const double4 s = s4[j];
      const double e2 = se2[j];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const double dx = s.x - tx[k], dy = s.y - ty[k], dz = s.z - tz[k];
        const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, (FL & F_UNIF) ? e2 : e2 + te2[k])));
        const double y = rsqrt_f64<FL>(r2);
        if constexpr (FL & F_NOACC) {
          ap[k] = fma(s.w, y, ap[k]);
          continue;
        }
        const double mr = s.w * y;
        if (!(FL & F_NOPOT)) ap[k] += mr;
        const double w = mr * (y * y);
        ax[k] = fma(w, dx, ax[k]);
        ay[k] = fma(w, dy, ay[k]);
        az[k] = fma(w, dz, az[k]);
      }
    }
    return;
  }
  constexpr int J = K >= TG_FP64_GROUP ? 1 : TG_FP64_GROUP / K;   // sources per group
#pragma unroll 1
  for (int j = 0; j < cnt; j += J) {
    double4 s[J];
    double dx[J * K], dy[J * K], dz[J * K], r2[J * K], y[J * K];
#pragma unroll
    for (int i = 0; i < J; ++i) {
      s[i] = s4[j + i];
      const double e2 = se2[j + i];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int q = i * K + k;
        dx[q] = s[i].x - tx[k];
        dy[q] = s[i].y - ty[k];
        dz[q] = s[i].z - tz[k];
        r2[q] = fma(dx[q], dx[q], fma(dy[q], dy[q], fma(dz[q], dz[q], (FL & F_UNIF) ? e2 : e2 + te2[k])));
        y[q] = __builtin_amdgcn_rsq(r2[q]);
      }
    }
    if constexpr (FL & F_GUARD) guard_zero(r2, y);
#pragma unroll
    for (int i = 0; i < J; ++i)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int q = i * K + k;
        const double yr = refine_rsqrt(r2[q], y[q]);
        if constexpr (FL & F_NOACC) {
          ap[k] = fma(s[i].w, yr, ap[k]);
          continue;
        }
        const double mr = s[i].w * yr;
        if (!(FL & F_NOPOT)) ap[k] += mr;
        const double w = mr * (yr * yr);
        ax[k] = fma(w, dx[q], ax[k]);
        ay[k] = fma(w, dy[q], ay[k]);
        az[k] = fma(w, dz[q], az[k]);
      }
  }
}

// ------------------------------------------------------ mixed-precision tile loop ----
// y[k] <- v_rsq_f32(y[k]) for a run of N, with the wave's issue priority raised for the run.
// A SIMD issues FP32 multiplies and FMAs of two of its waves together, 2.1 cycles per wave64
// instruction against 4.1 for one wave alone; one v_rsq_f32 takes the transcendental unit 8.1 cycles.
// Streams of 9 FMAs per v_rsq_f32 (registers only, 3 waves per SIMD) lost the pairing behind every
// v_rsq_f32: 43 cycles per group, 34 with 8 v_rsq_f32 in a row.  With the run at priority 1 a wave's
// transcendentals finish before the other waves' arithmetic resumes, and that resumes paired: 27.2-27.7
// cycles for any run length, against 26.7 for 9 FMAs + 1 v_rsq_f32 issued back to back without loss.
// Same instructions, same results, bit for bit.  Column kernel, 10,000 stars onto 1,024,000 cells:
// 2.42 -> 2.13 ms; 16 uneven problems of 3.7e10 pairs: 7.98 -> 7.02 ms (34 -> 30 cycles per pair).
template <int N>
__device__ __forceinline__ void rsq_run(float (&y)[N]) {
  static_assert(N == 2 || N == 4 || N == 8 || N == 16, "");
  if constexpr (N == 2)
    asm("s_setprio 1\n\tv_rsq_f32 %0, %0\n\tv_rsq_f32 %1, %1\n\ts_setprio 0" : "+v"(y[0]), "+v"(y[1]));
  else if constexpr (N == 4)
    asm("s_setprio 1\n\tv_rsq_f32 %0, %0\n\tv_rsq_f32 %1, %1\n\tv_rsq_f32 %2, %2\n\tv_rsq_f32 %3, %3\n\ts_setprio 0"
        : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]));
  else if constexpr (N == 8)
    asm("s_setprio 1\n\tv_rsq_f32 %0, %0\n\tv_rsq_f32 %1, %1\n\tv_rsq_f32 %2, %2\n\tv_rsq_f32 %3, %3\n\t"
        "v_rsq_f32 %4, %4\n\tv_rsq_f32 %5, %5\n\tv_rsq_f32 %6, %6\n\tv_rsq_f32 %7, %7\n\ts_setprio 0"
        : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7]));
  else
    asm("s_setprio 1\n\tv_rsq_f32 %0, %0\n\tv_rsq_f32 %1, %1\n\tv_rsq_f32 %2, %2\n\tv_rsq_f32 %3, %3\n\t"
        "v_rsq_f32 %4, %4\n\tv_rsq_f32 %5, %5\n\tv_rsq_f32 %6, %6\n\tv_rsq_f32 %7, %7\n\t"
        "v_rsq_f32 %8, %8\n\tv_rsq_f32 %9, %9\n\tv_rsq_f32 %10, %10\n\tv_rsq_f32 %11, %11\n\t"
        "v_rsq_f32 %12, %12\n\tv_rsq_f32 %13, %13\n\tv_rsq_f32 %14, %14\n\tv_rsq_f32 %15, %15\n\ts_setprio 0"
        : "+v"(y[0]), "+v"(y[1]), "+v"(y[2]), "+v"(y[3]), "+v"(y[4]), "+v"(y[5]), "+v"(y[6]), "+v"(y[7]),
          "+v"(y[8]), "+v"(y[9]), "+v"(y[10]), "+v"(y[11]), "+v"(y[12]), "+v"(y[13]), "+v"(y[14]), "+v"(y[15]));
}

template <int K, int NT, int FL>
__device__ __forceinline__ void f32_tile(const float4* __restrict__ s4,
                                         const float* __restrict__ se2,
                                         const float (&tx)[K], const float (&ty)[K],
                                         const float (&tz)[K], const float (&te2)[K],
                                         float (&ax)[K], float (&ay)[K], float (&az)[K],
                                         float (&ap)[K]) {
  // Sources per run of 16 v_rsq_f32 (K a power of two, at most 16): 100,000 scattered points, K = 2:
  // 499 us per call with the v_rsq_f32 spread over the loop, 483 in runs of 4, 469 of 8, 453 of 16.
  constexpr int J = 16 / K;
#pragma unroll 1
  for (int j = 0; j < NT; j += J) {
    float4 s[J];
    float dx[J * K], dy[J * K], dz[J * K], r2[J * K], y[J * K];
#pragma unroll
    for (int i = 0; i < J; ++i) {
      s[i] = s4[j + i];
      const float e2 = se2[j + i];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int q = i * K + k;
        dx[q] = s[i].x - tx[k];
        dy[q] = s[i].y - ty[k];
        dz[q] = s[i].z - tz[k];
        y[q] = r2[q] = fmaf(dx[q], dx[q], fmaf(dy[q], dy[q], fmaf(dz[q], dz[q], (FL & F_UNIF) ? e2 : e2 + te2[k])));
      }
    }
    rsq_run(y);
#pragma unroll
    for (int i = 0; i < J; ++i)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int q = i * K + k;
        if (FL & F_GUARD) y[q] = r2[q] > 0.0f ? y[q] : 0.0f;
        if constexpr (FL & F_NOACC) {
          ap[k] = fmaf(s[i].w, y[q], ap[k]);
          continue;
        }
        const float mr = s[i].w * y[q];
        if (!(FL & F_NOPOT)) ap[k] = fmaf(s[i].w, y[q], ap[k]);
        const float w = (mr * y[q]) * y[q];
        ax[k] = fmaf(w, dx[q], ax[k]);
        ay[k] = fmaf(w, dy[q], ay[k]);
        az[k] = fmaf(w, dz[q], az[k]);
      }
  }
}

// Knuth two-sum: (hi, lo) += v with the rounding error of hi + v kept in lo.
__device__ __forceinline__ void two_sum(float& hi, float& lo, float v) {
  const float s = hi + v;
  const float bp = s - hi;
  const float err = (hi - (s - bp)) + (v - bp);
  hi = s;
  lo += err;
}

// ------------------------------------------------------------------ LDS layout ----
template <int NT>
struct LdsF64 {
  double4 s4[NT];
  double se2[NT];
  double red[2 * 4 * (NT / 64)];
};
template <int NT>
struct LdsF32 {
  float4 s4[NT];
  float se2[NT];
  double red[2 * 4 * (NT / 64)];
};

// Threshold on the smallest possible eps^2 of a tile below which the FP32 loop guards
// r2 == 0 (and keeps rsq far from overflow).
#define TG_F32_TINY_E2 1e-30

// Statistics of a packed source set, device words written by the pack kernels: doubles stored as
// their bits (non-negative, so integer atomicMin / atomicMax order them like the values).
enum {
  ST_E2MIN = 0,   // smallest eps^2 (read by every kernel)
  ST_BAD = 1,     // non-zero: a NaN/Inf input (validation)
  ST_RMAX = 2,    // largest |x|, |y|, |z|
  ST_E2MAX = 3,   // largest eps^2
  ST_MMAX = 4,    // largest |m|
  ST_WORDS = 5
};

__device__ __forceinline__ double max_abs3(double x, double y, double z) {
  return fmax(fabs(x), fmax(fabs(y), fabs(z)));
}

// v + dt*a with the product and the sum rounded separately (no FMA contraction), as the
// reference's FP64 kick loops compute it (interface.F90:1793-1795).
__device__ __forceinline__ void kick_one(const Out& O, int64_t t, double gx, double gy, double gz) {
#pragma clang fp contract(off)
  O.vx[t] = O.vx[t] + O.dt * gx;
  O.vy[t] = O.vy[t] + O.dt * gy;
  O.vz[t] = O.vz[t] + O.dt * gz;
}

__device__ __forceinline__ void store_result(const Out& O, int64_t t, double sx, double sy,
                                             double sz, double sp) {
  if (O.part) {                 // components that nobody wants are neither written nor read back
    if (!O.noacc) {
      O.part[t] = sx;
      O.part[O.pstride + t] = sy;
      O.part[2 * O.pstride + t] = sz;
    }
    if (!O.nopot) O.part[3 * O.pstride + t] = sp;
    return;
  }
  const double gx = O.G * sx, gy = O.G * sy, gz = O.G * sz;
  if (O.ax) O.ax[t] = gx;
  if (O.ay) O.ay[t] = gy;
  if (O.az) O.az[t] = gz;
  if (O.phi) O.phi[t] = -O.G * sp;
  if (O.vx) kick_one(O, t, gx, gy, gz);
}

// Code path of a tile from its smallest/largest target eps^2 and the sources' smallest.
__device__ __forceinline__ int tile_flags(double e2s_min, double e2t_min, double e2t_max,
                                          const Out& O, bool f32) {
  int fl = 0;
  if (e2t_min == e2t_max) fl |= F_UNIF;
  const double lo = e2s_min + e2t_min;
  if (!(lo > (f32 ? TG_F32_TINY_E2 : 0.0))) fl |= F_GUARD;
  if (O.nopot) fl |= F_NOPOT;
  else if (O.noacc) fl |= F_NOACC;
  return fl;
}

// ------------------------------------------------------- per-workgroup drivers ----
template <int K, int NT, int FL>
__device__ __forceinline__ void fp64_sources(LdsF64<NT>& L, const double4* __restrict__ src4,
                                          const double* __restrict__ srce2, int64_t s_begin,
                                          int64_t s_end, double e2u, const double (&tx)[K],
                                          const double (&ty)[K], const double (&tz)[K],
                                          const double (&te2)[K], double (&ax)[K],
                                          double (&ay)[K], double (&az)[K], double (&ap)[K]) {
  const int tid = threadIdx.x;
  for (int64_t base = s_begin; base < s_end; base += NT) {
    __syncthreads();
    const int64_t j = base + tid;
    if (j < s_end) {
      L.s4[tid] = src4[j];
      L.se2[tid] = srce2[j] + e2u;
    } else {   // padding source: zero mass, eps^2 = 1 -> contributes exactly 0
      L.s4[tid] = make_double4(0.0, 0.0, 0.0, 0.0);
      L.se2[tid] = 1.0;
    }
    __syncthreads();
    const int cnt = (int)(s_end - base < NT ? s_end - base : NT);
    // each tile's sum on its own, then onto the total: rounding errors grow with a tile's length and the
    // number of tiles, not with the chunk's length (20,011 x 5,003 in one chunk: 2e-15 against 5e-16)
    double sx[K], sy[K], sz[K], sp[K];
#pragma unroll
    for (int k = 0; k < K; ++k) sx[k] = sy[k] = sz[k] = sp[k] = 0.0;
    fp64_tile<K, NT, FL>(L.s4, L.se2, cnt, tx, ty, tz, te2, sx, sy, sz, sp);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      ax[k] += sx[k];
      ay[k] += sy[k];
      az[k] += sz[k];
      ap[k] += sp[k];
    }
  }
}

#define TG_DISPATCH(FN, fl, ...)                                              \
  switch (fl) {                                                               \
    case 0: FN<0>(__VA_ARGS__); break;                                        \
    case F_GUARD: FN<F_GUARD>(__VA_ARGS__); break;                            \
    case F_UNIF: FN<F_UNIF>(__VA_ARGS__); break;                              \
    case F_UNIF | F_GUARD: FN<F_UNIF | F_GUARD>(__VA_ARGS__); break;          \
    case F_NOPOT: FN<F_NOPOT>(__VA_ARGS__); break;                            \
    case F_NOPOT | F_GUARD: FN<F_NOPOT | F_GUARD>(__VA_ARGS__); break;        \
    case F_NOPOT | F_UNIF: FN<F_NOPOT | F_UNIF>(__VA_ARGS__); break;          \
    case F_NOPOT | F_UNIF | F_GUARD: FN<F_NOPOT | F_UNIF | F_GUARD>(__VA_ARGS__); break; \
    case F_NOACC: FN<F_NOACC>(__VA_ARGS__); break;                            \
    case F_NOACC | F_GUARD: FN<F_NOACC | F_GUARD>(__VA_ARGS__); break;        \
    case F_NOACC | F_UNIF: FN<F_NOACC | F_UNIF>(__VA_ARGS__); break;          \
    default: FN<F_NOACC | F_UNIF | F_GUARD>(__VA_ARGS__); break;              \
  }

template <int K, int NT>
struct Fp64Run {
  template <int FL>
  static __device__ __forceinline__ void run(LdsF64<NT>& L, const double4* src4, const double* srce2,
                                             int64_t sb, int64_t se, double e2u,
                                             const double (&tx)[K], const double (&ty)[K],
                                             const double (&tz)[K], const double (&te2)[K],
                                             double (&ax)[K], double (&ay)[K], double (&az)[K],
                                             double (&ap)[K]) {
    fp64_sources<K, NT, FL>(L, src4, srce2, sb, se, (FL & F_UNIF) ? e2u : 0.0, tx, ty, tz, te2,
                            ax, ay, az, ap);
  }
};

// sst: the source statistics (ST_*).
template <int K, int NT>
__device__ void process_fp64(LdsF64<NT>& L, const Tgt& T, int64_t tile0,
                             const double4* __restrict__ src4, const double* __restrict__ srce2,
                             int64_t s_begin, int64_t s_end, const double* sst, const Out& O) {
  const int tid = threadIdx.x;
  double tx[K], ty[K], tz[K], te2[K];
  double mn[1] = {INFINITY}, mx[1] = {-INFINITY};   // eps^2
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t t = tile0 + (int64_t)k * NT + tid;
    load_target(T, t < T.n ? t : T.n - 1, tx[k], ty[k], tz[k], te2[k]);
    if (t < T.n) {
      mn[0] = fmin(mn[0], te2[k]);
      mx[0] = fmax(mx[0], te2[k]);
    }
  }
  block_minmax<NT, 1>(mn, mx, L.red);
  const int fl = tile_flags(sst[ST_E2MIN], mn[0], mx[0], O, false);
  double ax[K], ay[K], az[K], ap[K];
#pragma unroll
  for (int k = 0; k < K; ++k) ax[k] = ay[k] = az[k] = ap[k] = 0.0;
  typedef Fp64Run<K, NT> R;
  TG_DISPATCH(R::template run, fl, L, src4, srce2, s_begin, s_end, mn[0], tx, ty, tz,
              te2, ax, ay, az, ap)
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t t = tile0 + (int64_t)k * NT + tid;
    if (t < T.n) store_result(O, t, ax[k], ay[k], az[k], ap[k]);
  }
}

// Mixed precision.  The tile's FP64 anchor c is the centre of its targets' bounding box.
// Sources are staged as fp32(x_s - c) (the FP64 difference rounded once), targets are held
// as fp32(x_t - c); the FP32 difference of the two is exact whenever they are within a
// factor of two of each other (Sterbenz), i.e. for exactly the close pairs where a
// difference of raw FP32 coordinates would cancel catastrophically.  The FP32 partial sums
// of each LDS tile (NT sources) are folded into per-target two-sum (hi, lo) accumulators.
template <int K, int NT, int FL>
__device__ __forceinline__ void f32_sources(LdsF32<NT>& L, const double4* __restrict__ src4,
                                         const double* __restrict__ srce2, int64_t s_begin,
                                         int64_t s_end, double e2u, double cx, double cy,
                                         double cz, const float (&tx)[K], const float (&ty)[K],
                                         const float (&tz)[K], const float (&te2)[K],
                                         float (&hx)[K], float (&hy)[K], float (&hz)[K],
                                         float (&hp)[K], float (&lx)[K], float (&ly)[K],
                                         float (&lz)[K], float (&lp)[K]) {
  const int tid = threadIdx.x;
  for (int64_t base = s_begin; base < s_end; base += NT) {
    __syncthreads();
    const int64_t j = base + tid;
    if (j < s_end) {
      const double4 s = src4[j];
      L.s4[tid] = make_float4((float)(s.x - cx), (float)(s.y - cy), (float)(s.z - cz), (float)s.w);
      L.se2[tid] = (float)(srce2[j] + e2u);
    } else {
      L.s4[tid] = make_float4(0.f, 0.f, 0.f, 0.f);
      L.se2[tid] = 1.0f;
    }
    __syncthreads();
    float ax[K], ay[K], az[K], ap[K];
#pragma unroll
    for (int k = 0; k < K; ++k) ax[k] = ay[k] = az[k] = ap[k] = 0.f;
    f32_tile<K, NT, FL>(L.s4, L.se2, tx, ty, tz, te2, ax, ay, az, ap);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      two_sum(hx[k], lx[k], ax[k]);
      two_sum(hy[k], ly[k], ay[k]);
      two_sum(hz[k], lz[k], az[k]);
      if (!(FL & F_NOPOT)) two_sum(hp[k], lp[k], ap[k]);
    }
  }
}

template <int K, int NT>
struct MixRun {
  template <int FL>
  static __device__ __forceinline__ void run(LdsF32<NT>& L, const double4* src4, const double* srce2,
                                             int64_t sb, int64_t se, double e2u, double cx,
                                             double cy, double cz, const float (&tx)[K],
                                             const float (&ty)[K], const float (&tz)[K],
                                             const float (&te2)[K], float (&hx)[K], float (&hy)[K],
                                             float (&hz)[K], float (&hp)[K], float (&lx)[K],
                                             float (&ly)[K], float (&lz)[K], float (&lp)[K]) {
    f32_sources<K, NT, FL>(L, src4, srce2, sb, se, (FL & F_UNIF) ? e2u : 0.0, cx, cy,
                                       cz, tx, ty, tz, te2, hx, hy, hz, hp, lx, ly, lz, lp);
  }
};

template <int K, int NT>
__device__ void process_mixed(LdsF32<NT>& L, const Tgt& T, int64_t tile0,
                              const double4* __restrict__ src4, const double* __restrict__ srce2,
                              int64_t s_begin, int64_t s_end, const double* sst, const Out& O) {
  const int tid = threadIdx.x;
  double px[K], py[K], pz[K], pe2[K];
  double mn[4] = {INFINITY, INFINITY, INFINITY, INFINITY};
  double mx[4] = {-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t t = tile0 + (int64_t)k * NT + tid;
    load_target(T, t < T.n ? t : T.n - 1, px[k], py[k], pz[k], pe2[k]);
    if (t < T.n) {
      mn[0] = fmin(mn[0], px[k]); mx[0] = fmax(mx[0], px[k]);
      mn[1] = fmin(mn[1], py[k]); mx[1] = fmax(mx[1], py[k]);
      mn[2] = fmin(mn[2], pz[k]); mx[2] = fmax(mx[2], pz[k]);
      mn[3] = fmin(mn[3], pe2[k]); mx[3] = fmax(mx[3], pe2[k]);
    }
  }
  block_minmax<NT, 4>(mn, mx, L.red);
  const double cx = 0.5 * (mn[0] + mx[0]), cy = 0.5 * (mn[1] + mx[1]), cz = 0.5 * (mn[2] + mx[2]);
  const int fl = tile_flags(sst[ST_E2MIN], mn[3], mx[3], O, true);
  float tx[K], ty[K], tz[K], te2[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    tx[k] = (float)(px[k] - cx);
    ty[k] = (float)(py[k] - cy);
    tz[k] = (float)(pz[k] - cz);
    te2[k] = (float)pe2[k];
  }
  float hx[K], hy[K], hz[K], hp[K], lx[K], ly[K], lz[K], lp[K];
#pragma unroll
  for (int k = 0; k < K; ++k) hx[k] = hy[k] = hz[k] = hp[k] = lx[k] = ly[k] = lz[k] = lp[k] = 0.f;
  typedef MixRun<K, NT> R;
  TG_DISPATCH(R::template run, fl, L, src4, srce2, s_begin, s_end, mn[3], cx, cy, cz, tx,
              ty, tz, te2, hx, hy, hz, hp, lx, ly, lz, lp)
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t t = tile0 + (int64_t)k * NT + tid;
    if (t < T.n)
      store_result(O, t, (double)hx[k] + (double)lx[k], (double)hy[k] + (double)ly[k],
                   (double)hz[k] + (double)lz[k], (double)hp[k] + (double)lp[k]);
  }
}

// ------------------------------------------------------------------ grid kernels ----
// blockIdx.x = target tile, blockIdx.y = source chunk [c*chunk, min((c+1)*chunk, ns)).
template <int K, int NT>
__global__ __launch_bounds__(NT) void k_eval_fp64(Tgt T, const double4* __restrict__ src4,
                                                  const double* __restrict__ srce2, int64_t ns,
                                                  int64_t chunk, const double* sst, Out O) {
  __shared__ LdsF64<NT> L;
  if (gated_off(O)) return;
  const int64_t tile0 = (int64_t)blockIdx.x * (K * NT);
  const int64_t sb = (int64_t)blockIdx.y * chunk;
  const int64_t se = sb + chunk < ns ? sb + chunk : ns;
  Out o = O;
  if (o.part) o.part += (int64_t)blockIdx.y * 4 * o.pstride;
  process_fp64<K, NT>(L, T, tile0, src4, srce2, sb, se, sst, o);
}

template <int K, int NT>
__global__ __launch_bounds__(NT) void k_eval_mixed(Tgt T, const double4* __restrict__ src4,
                                                   const double* __restrict__ srce2, int64_t ns,
                                                   int64_t chunk, const double* sst, Out O) {
  __shared__ LdsF32<NT> L;
  if (gated_off(O)) return;
  const int64_t tile0 = (int64_t)blockIdx.x * (K * NT);
  const int64_t sb = (int64_t)blockIdx.y * chunk;
  const int64_t se = sb + chunk < ns ? sb + chunk : ns;
  Out o = O;
  if (o.part) o.part += (int64_t)blockIdx.y * 4 * o.pstride;
  process_mixed<K, NT>(L, T, tile0, src4, srce2, sb, se, sst, o);
}

// s += the partials of target t from chunks [c0, c1), in chunk order: the components that somebody wants
// (the others are not written).  The choice is made once, around the loop: tests inside it kept the loads of
// successive chunks from being in flight together (10 targets, 1,000,001 sources in FP64, 485 us per call
// against 398; 512 cells, 300,000 sources 201 against 156).
template <int Q0, int Q1>
__device__ __forceinline__ void sum_chunks_of(const double* __restrict__ part, int64_t pstride, int64_t t, int c0,
                                              int c1, double (&s)[4]) {
#pragma unroll 4
  for (int c = c0; c < c1; ++c) {
    const double* p = part + (int64_t)c * 4 * pstride + t;
#pragma unroll
    for (int q = Q0; q < Q1; ++q) s[q] += p[q * pstride];
  }
}
__device__ __forceinline__ void sum_chunks(const double* __restrict__ part, int64_t pstride, int64_t t, int c0,
                                           int c1, bool noacc, bool nopot, double (&s)[4]) {
  if (noacc) sum_chunks_of<3, 4>(part, pstride, t, c0, c1, s);
  else if (nopot) sum_chunks_of<0, 3>(part, pstride, t, c0, c1, s);
  else sum_chunks_of<0, 4>(part, pstride, t, c0, c1, s);
}

// Sum of the nsplit chunk partials of each target in chunk order, then the G scaling,
// the stores and the fused kick.
__global__ void k_reduce_chunks(const double* __restrict__ part, int64_t pstride, int nsplit,
                                int64_t n, Out O) {
  if (gated_off(O)) return;
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  sum_chunks(part, pstride, t, 0, nsplit, O.noacc, O.nopot, s);
  Out o = O;
  o.part = nullptr;
  store_result(o, t, s[0], s[1], s[2], s[3]);
}

// The same reduction for few targets and many chunks (k_reduce_chunks would run a handful of
// workgroups, each thread walking every chunk): a workgroup of 16 waves takes 64 targets, wave
// w sums chunks [w*per, (w+1)*per) in order, and wave 0 adds the 16 wave sums in wave order,
// so the result does not depend on scheduling.  Grid: ceil(n / 64) workgroups of 1024 lanes.
__global__ __launch_bounds__(1024) void k_reduce_chunks_wide(const double* __restrict__ part,
                                                             int64_t pstride, int nsplit, int64_t n,
                                                             Out O) {
  __shared__ double red[16][4][64];
  if (gated_off(O)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t t = (int64_t)blockIdx.x * 64 + lane;
  const int per = (nsplit + 15) / 16;
  const int c0 = w * per, c1 = min(nsplit, c0 + per);
  double s[4] = {0.0, 0.0, 0.0, 0.0};
  if (t < n) sum_chunks(part, pstride, t, c0, c1, O.noacc, O.nopot, s);
#pragma unroll
  for (int q = 0; q < 4; ++q) red[w][q][lane] = s[q];
  __syncthreads();
  if (w == 0 && t < n) {
    double a0 = red[0][0][lane], a1 = red[0][1][lane], a2 = red[0][2][lane], a3 = red[0][3][lane];
    for (int q = 1; q < 16; ++q) {
      a0 += red[q][0][lane];
      a1 += red[q][1][lane];
      a2 += red[q][2][lane];
      a3 += red[q][3][lane];
    }
    Out o = O;
    o.part = nullptr;
    store_result(o, t, a0, a1, a2, a3);
  }
}

// Bits of a non-negative double: their unsigned-integer order is the numeric order.
__device__ __forceinline__ unsigned long long dbits(double v) {
  return (unsigned long long)__double_as_longlong(v);
}

__device__ __forceinline__ unsigned long long shfl_xor_u64(unsigned long long v, int off) {
  return (unsigned long long)__shfl_xor((long long)v, off);
}

// Folds one lane's source statistics (ST_* words) into `stat`: reduced within each wave by
// shuffles, across the workgroup's (at most 4) waves through LDS, then at most one atomic per
// word.  Every lane of the workgroup (<= 256 lanes) must call it.
__device__ __forceinline__ void fold_source_stats(unsigned long long e2min, unsigned long long rmax,
                                                  unsigned long long e2max, unsigned long long mmax,
                                                  unsigned long long* stat) {
  __shared__ unsigned long long sm[4][4];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    e2min = min(e2min, shfl_xor_u64(e2min, off));
    rmax = max(rmax, shfl_xor_u64(rmax, off));
    e2max = max(e2max, shfl_xor_u64(e2max, off));
    mmax = max(mmax, shfl_xor_u64(mmax, off));
  }
  const int t = threadIdx.x, w = t >> 6, nw = (blockDim.x + 63) >> 6;
  if ((t & 63) == 0) {
    sm[0][w] = e2min;
    sm[1][w] = rmax;
    sm[2][w] = e2max;
    sm[3][w] = mmax;
  }
  __syncthreads();
  if (t == 0) {
    for (int q = 1; q < nw; ++q) {
      sm[0][0] = min(sm[0][0], sm[0][q]);
      sm[1][0] = max(sm[1][0], sm[1][q]);
      sm[2][0] = max(sm[2][0], sm[2][q]);
      sm[3][0] = max(sm[3][0], sm[3][q]);
    }
  }
  __syncthreads();
  // One lane per word; the atomic only where the workgroup's value improves on what the word
  // already holds (a plain read, possibly stale, which only costs an atomic): with thousands of
  // workgroups on the same five words, most then skip their atomics instead of queueing on them.
  if (t < ST_WORDS) {
    volatile unsigned long long* w = stat + t;
    if (t == ST_E2MIN) {
      if (sm[0][0] < *w) atomicMin(&stat[ST_E2MIN], sm[0][0]);
    } else if (t == ST_RMAX) {
      if (sm[1][0] > *w) atomicMax(&stat[ST_RMAX], sm[1][0]);
    } else if (t == ST_E2MAX) {
      if (sm[2][0] > *w) atomicMax(&stat[ST_E2MAX], sm[2][0]);
    } else if (t == ST_MMAX) {
      if (sm[3][0] > *w) atomicMax(&stat[ST_MMAX], sm[3][0]);
    }
  }
}

// ---- one-pass reductions of an input set, read by the host ----
// The pack and check kernels reduce their set's statistics (ST_*) and one violation bit over the whole
// grid in the same launch: each workgroup writes its six words to its slot, takes a ticket, and the
// last one reduces the slots, writes the results (device words for later kernels, pinned host words for
// a caller that waits) and returns the ticket to 0.  No reset launch before it, no copy after it, and
// no queue of atomics on five shared words, which took 75 of 85 us on a million cells.
#define TG_PUB_WG 512            // most workgroups of such a launch (slots)
struct Publish {
  unsigned long long* slots;     // TG_PUB_WG x 8 words
  unsigned int* ticket;          // 0 between launches
  unsigned long long* stat;      // device result: ST_WORDS words (may be null)
  int* flag;                     // device result: 1 if nothing was violated, else 0 (may be null)
  unsigned long long* host;      // pinned result: ST_WORDS words, then the violation bit (may be null)
  const unsigned long long* src_stat;   // non-null: host[8 ...] = these ST_WORDS words of the source set,
  const int* src_flag;                  //   host[13] = *src_flag (null: 0)
};

// One lane's (e2min, rmax, e2max, mmax, bad | viol << 1) -> the workgroup's, in every lane.  256 lanes.
__device__ __forceinline__ void wg_stats(unsigned long long (&v)[4], int& bits, unsigned long long (*sm)[5]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    v[0] = min(v[0], shfl_xor_u64(v[0], off));
#pragma unroll
    for (int q = 1; q < 4; ++q) v[q] = max(v[q], shfl_xor_u64(v[q], off));
    bits |= __shfl_xor(bits, off);
  }
  __syncthreads();               // an earlier use of sm is over
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) sm[threadIdx.x >> 6][q] = v[q];
    sm[threadIdx.x >> 6][4] = (unsigned long long)bits;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    v[0] = min(v[0], sm[w][0]);
#pragma unroll
    for (int q = 1; q < 4; ++q) v[q] = max(v[q], sm[w][q]);
    bits |= (int)sm[w][4];
  }
}

// Every lane of every workgroup (256 lanes, at most TG_PUB_WG workgroups) calls it once, last.
__device__ __forceinline__ void publish_stats(unsigned long long e2min, unsigned long long rmax,
                                              unsigned long long e2max, unsigned long long mmax, int bad,
                                              int viol, const Publish& P) {
  __shared__ unsigned long long sm[4][5];
  __shared__ int last;
  unsigned long long v[4] = {e2min, rmax, e2max, mmax};
  int bits = (bad ? 1 : 0) | (viol ? 2 : 0);
  wg_stats(v, bits, sm);
  if (gridDim.x > 1) {
    if (threadIdx.x == 0) {
      unsigned long long* s = P.slots + (size_t)blockIdx.x * 8;
      // agent-scope stores go through to where every XCD sees them; the wait completes them before the
      // ticket is taken, so whoever takes the last ticket reads every slot whole
#pragma unroll
      for (int q = 0; q < 4; ++q) __hip_atomic_store(s + q, v[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(s + 4, (unsigned long long)bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      last = __hip_atomic_fetch_add(P.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    asm volatile("" ::: "memory");
    for (unsigned int b = threadIdx.x; b < gridDim.x; b += 256) {
      unsigned long long* s = P.slots + (size_t)b * 8;
      v[0] = min(v[0], __hip_atomic_load(s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
      for (int q = 1; q < 4; ++q)
        v[q] = max(v[q], __hip_atomic_load(s + q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      bits |= (int)__hip_atomic_load(s + 4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    wg_stats(v, bits, sm);
    if (threadIdx.x == 0) __hip_atomic_store(P.ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (threadIdx.x != 0) return;
  const unsigned long long st[ST_WORDS] = {v[0], (unsigned long long)(bits & 1), v[1], v[2], v[3]};
  static_assert(ST_E2MIN == 0 && ST_BAD == 1 && ST_RMAX == 2 && ST_E2MAX == 3 && ST_MMAX == 4, "");
#pragma unroll
  for (int q = 0; q < ST_WORDS; ++q) {
    if (P.stat) P.stat[q] = st[q];
    if (P.host) P.host[q] = st[q];
  }
  if (P.flag) *P.flag = (bits & 2) ? 0 : 1;
  if (P.host) {
    P.host[ST_WORDS] = (unsigned long long)(bits >> 1);
    if (P.src_stat) {
#pragma unroll
      for (int q = 0; q < ST_WORDS; ++q) P.host[8 + q] = P.src_stat[q];
      P.host[8 + ST_WORDS] = P.src_flag ? (unsigned long long)*P.src_flag : 0ULL;
    }
    __threadfence_system();
  }
}

__device__ __forceinline__ bool finite5(double a, double b, double c, double d, double e) {
  return isfinite(a) && isfinite(b) && isfinite(c) && isfinite(d) && isfinite(e);
}

// Packs SoA FP64 sources into {x,y,z,m} + eps^2 with their statistics.  nb8 > 0 (n = 512 nb8): the
// sources may be 8^3 leaf blocks in C order (cell c = 64 i + 8 j + k of block b at b * 512 + c): x
// depends on i only, y on j only, z on k only, and eps^2 is the block's.  Each source is compared with
// the first of its line (any difference is a violation: P.flag = 0), and the block-source form is
// written too: the axes sax, the block eps^2 be2 and the contiguous cell masses sm.  With `check`, a
// NaN/Inf input sets ST_BAD.
__global__ __launch_bounds__(256) void k_pack_sources(int64_t n, const double* __restrict__ x,
                                                      const double* __restrict__ y,
                                                      const double* __restrict__ z,
                                                      const double* __restrict__ m,
                                                      const double* __restrict__ eps,
                                                      double4* __restrict__ s4,
                                                      double* __restrict__ se2, int64_t nb8,
                                                      double* __restrict__ sax, double* __restrict__ be2,
                                                      double* __restrict__ sm, int check, Publish P) {
  unsigned long long e2min = 0x7ff0000000000000ULL, rmax = 0ULL, e2max = 0ULL, mmax = 0ULL;
  int bad = 0, viol = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const double4 v = make_double4(x[i], y[i], z[i], m[i]);
    const double e = eps ? eps[i] : 0.0;
    s4[i] = v;
    const double e2 = e * e;
    se2[i] = e2;
    e2min = min(e2min, dbits(e2));
    e2max = max(e2max, dbits(e2));
    rmax = max(rmax, dbits(max_abs3(v.x, v.y, v.z)));
    mmax = max(mmax, dbits(fabs(v.w)));
    if (check && !finite5(v.x, v.y, v.z, v.w, e)) bad = 1;
    if (nb8 > 0) {
      const int64_t b = i >> 9, base = b * 512;
      const int c = (int)(i & 511), ci = c >> 6, cj = (c >> 3) & 7, ck = c & 7;
      const double eb = eps ? eps[base] : 0.0;
      if (!(v.x == x[base + ci * 64] && v.y == y[base + cj * 8] && v.z == z[base + ck] && e2 == eb * eb)) viol = 1;
      sm[i] = v.w;
      if (cj == 0 && ck == 0) sax[b * 24 + ci] = v.x;
      if (ci == 0 && ck == 0) sax[b * 24 + 8 + cj] = v.y;
      if (ci == 0 && cj == 0) sax[b * 24 + 16 + ck] = v.z;
      if (c == 0) be2[b] = e2;
    }
  }
  publish_stats(e2min, rmax, e2max, mmax, bad, viol, P);
}

// Column structure of explicit targets, the C order of 8^3 leaf blocks
// (.deprecated/bridge_multiples.py:566-575 flattens each block's meshgrid this way): every
// aligned group of 8 consecutive targets shares x and y, and every aligned group of 512 shares
// eps.  One lane per target, compared with the first of its group (coalesced reads).
__device__ __forceinline__ bool column_ok(const double* x, const double* y, const double* eps, int64_t t) {
  const int64_t g = t & ~(int64_t)7;
  bool ok = x[t] == x[g] && y[t] == y[g];
  if (eps) ok = ok && eps[t] == eps[t & ~(int64_t)511];
  return ok;
}

// Checks a point set (x, y, z, eps per point; dx == null) or a set of 8^3 blocks (x, y, z the lower
// corners and dx the cell widths, so the centres lie within [x, x + 8 dx]; eps per block), with nm masses
// m (may be null): NaN/Inf (ST_BAD), the range statistics (ST_*) and, with `cols`, the points' column
// structure (a violation: not columns).
__global__ __launch_bounds__(256) void k_check_set(int64_t n, const double* __restrict__ x,
                                                   const double* __restrict__ y, const double* __restrict__ z,
                                                   const double* __restrict__ dx, const double* __restrict__ e,
                                                   int64_t nm, const double* __restrict__ m, int cols, Publish P) {
  unsigned long long e2min = 0x7ff0000000000000ULL, rmax = 0ULL, e2max = 0ULL, mmax = 0ULL;
  int bad = 0, viol = 0;
  const int64_t most = m && nm > n ? nm : n;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < most; i += (int64_t)gridDim.x * 256) {
    if (i < n) {
      const double px = x[i], py = y[i], pz = z[i], ei = e ? e[i] : 0.0, d = dx ? dx[i] : 0.0;
      double r = max_abs3(px, py, pz);
      if (dx) r = fmax(r, max_abs3(px + 8.0 * d, py + 8.0 * d, pz + 8.0 * d));
      rmax = max(rmax, dbits(r));
      e2min = min(e2min, dbits(ei * ei));
      e2max = max(e2max, dbits(ei * ei));
      if (!finite5(px, py, pz, ei, d)) bad = 1;
      if (cols && !column_ok(x, y, e, i)) viol = 1;
    }
    if (m && i < nm) {
      const double mi = m[i];
      mmax = max(mmax, dbits(fabs(mi)));
      if (!isfinite(mi)) bad = 1;
    }
  }
  publish_stats(e2min, rmax, e2max, mmax, bad, viol, P);
}

__global__ void k_kick(int64_t n, double dt, const double* __restrict__ ax,
                       const double* __restrict__ ay, const double* __restrict__ az,
                       double* __restrict__ vx, double* __restrict__ vy, double* __restrict__ vz) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  {
#pragma clang fp contract(off)
    vx[i] = vx[i] + dt * ax[i];
    vy[i] = vy[i] + dt * ay[i];
    vz[i] = vz[i] + dt * az[i];
  }
}

// Gate value of an explicit-target evaluation whose structure the host does not know: 2 if the sources
// are explicit 8^3 blocks (*sflag, written when they were packed; sflag null: they are not), else
// `tcand` (1: the targets may have column structure, which k_check_cols then tests; 0: they do not).
__global__ void k_eval_gate(int* gate, const int* sflag, int tcand) {
  if (blockIdx.x == 0 && threadIdx.x == 0) gate[0] = (sflag && sflag[0] == 1) ? 2 : tcand;
}

// The column test for such an evaluation: any violation clears flag[0] (1 before; 2, the block-source
// path, is left alone); all writers store the same value.
__global__ void k_check_cols(Tgt T, int* flag) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T.n || flag[0] != 1) return;   // 2: the block-source kernel runs; nothing to test
  if (!column_ok(T.x, T.y, T.eps, t)) flag[0] = 0;
}

__global__ void k_fill(int64_t n, double v, double* a, double* b, double* c, double* d) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  if (a) a[i] = v;
  if (b) b[i] = v;
  if (c) c[i] = v;
  if (d) d[i] = v;
}

}  // namespace tg
