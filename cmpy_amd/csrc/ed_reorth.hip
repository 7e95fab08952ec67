// Fully reorthogonalised Lanczos steps in three launches.
//
// A step orthogonalises w = H v_j against v_0..v_j by classical Gram-Schmidt,
// twice.  The basis vectors are stored unnormalised (v_i = s_i V_i, s_i =
// 1/beta_i) one after another, so a pass is two products with the basis:
// dots d_i = <V_i, w> (a sum over all states) and w -= sum_i s_i^2 d_i V_i.  A
// block owns 64 S consecutive states of every vector, 64 at a time in LDS, so
// a pass's combination and the next pass's dots share one read of the basis:
//   k_reorth_hv    beta_j from the previous step's |w|^2 partials, w = s_j H V_j
//                  for the block's states, its share of every d_i
//   k_reorth_pass  d_i summed, alpha_j = s_j d_j, w -= sum (first pass), the
//                  block's share of the second pass's dots; then the same
//                  kernel for the second pass, leaving partials of |w|^2
// The recurrence's own terms alpha_j v_j and beta_j v_{j-1} are among the
// first pass's components.  Every block sums the partials of all blocks in the
// same order, so all hold the same coefficients and runs repeat bit for bit.
//
// At these sizes a launch costs as much as its code is long: a kernel's
// instructions are fetched anew on every launch, about 0.9 us per KB of
// straight-line code (a form with the tile in registers and its loops unrolled
// took 4 us at 2 KB and 17 us at 19 KB for the same work).  So the tile is
// held in LDS and every loop stays rolled.
#include "ed_internal.h"

#include <algorithm>
#include <mutex>

namespace ed {

constexpr int kReorthThreads = 1024;
constexpr int kReorthWaves = kReorthThreads / 64;
constexpr int kReorthBlocks = 256;  // at most; the partials each block sums grow with it
constexpr int kPre = 8;             // vectors of a tile each wave loads together

// LDS of both kernels: per-thread partial sums, one value per state of the
// tile, the coefficients, and (dynamic) the tile, tile[i * 64 + state].
struct ReorthLds {
  double* red;   // [kReorthThreads]
  double* tot;   // [64]
  double* tile;  // [(j + 1) * 64]
};

// Loads of the wave's first kPre vectors i = wave + 16 r of the tile at k0;
// clamped past the last vector and the last state (what the clamped ones bring
// is not stored, or meets w = 0).
__device__ __forceinline__ void tile_request(double (&v)[kPre], const double* __restrict__ V, int D, int k,
                                             int i0, int j) {
  const int kc = k < D ? k : D - 1;
#pragma unroll
  for (int r = 0; r < kPre; ++r) {
    const int i = i0 + kReorthWaves * r;
    v[r] = (V + (uint32_t)((i <= j ? i : j) * D))[kc];
  }
}

__device__ __forceinline__ void tile_store(const double (&v)[kPre], double* tile, int i0, int lane, int j) {
#pragma unroll
  for (int r = 0; r < kPre; ++r) {
    const int i = i0 + kReorthWaves * r;
    if (i <= j) tile[i * 64 + lane] = v[r];
  }
}

// The tile at k into LDS: v holds its first kPre vectors a wave.
__device__ __forceinline__ void tile_fill(double (&v)[kPre], double* tile, const double* __restrict__ V, int D,
                                          int k, int wave, int lane, int j) {
  tile_store(v, tile, wave, lane, j);
  for (int i0 = wave + kReorthWaves * kPre; i0 <= j; i0 += kReorthWaves * kPre) {
    tile_request(v, V, D, k, i0, j);
    tile_store(v, tile, i0, lane, j);
  }
}

// One value per lane and wave -> its sum over the waves, the same on every
// wave, and in tot[lane].
__device__ __forceinline__ double wave_total(double v, const ReorthLds& L, int wave, int lane) {
  L.red[wave * 64 + lane] = v;
  __syncthreads();
  if (wave == 0) {
    double s = 0.0;
#pragma unroll 4
    for (int w = 0; w < kReorthWaves; ++w) s += L.red[w * 64 + lane];
    L.tot[lane] = s;
  }
  __syncthreads();
  return L.tot[lane];
}

// Dots of the tile with w (in L.tot): thread t takes vector t mod 2^lg over
// 64 / (1024 / 2^lg) of the states, each lane starting at a state of its own
// (the tile's rows are 64 doubles apart).
__device__ __forceinline__ double tile_dots(double acc, const ReorthLds& L, int lg, int j) {
  const int i = threadIdx.x & ((1 << lg) - 1), g = threadIdx.x >> lg;
  const int per = 1 << (lg - 4);
  const double* row = L.tile + (i <= j ? i : j) * 64;
#pragma unroll 4
  for (int q = 0; q < per; ++q) {
    const int k = (g * per + q + i) & 63;
    acc = fma(row[k], L.tot[k], acc);
  }
  return acc;
}

// Sum over the threads of a vector, in order; valid on threads t <= 2^lg.
__device__ __forceinline__ double group_sum(double v, const ReorthLds& L, int lg) {
  __syncthreads();
  L.red[threadIdx.x] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x < (1u << lg))
    for (int t = threadIdx.x; t < kReorthThreads; t += 1 << lg) s += L.red[t];
  return s;
}

// S subtiles of 64 states per block.
__global__ __launch_bounds__(kReorthThreads) void k_reorth_hv(HvArgs a, int hops_up, int hops_dn,
                                                              const double* __restrict__ V, int D, int j, LzCoef c,
                                                              HvBeta prev, double* __restrict__ w,
                                                              double* __restrict__ part, int S, int lg) {
  extern __shared__ double tile[];
  __shared__ double red[kReorthThreads];
  __shared__ double tot[64];
  const ReorthLds L{red, tot, tile};
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int k = (int)blockIdx.x * S * 64 + lane;
  double v[kPre];
  tile_request(v, V, D, k, wave, j);
  double cp;
  const double sx = prev.j >= 0 ? form_beta(prev, blockIdx.x == 0, &cp) : c.scale[j];
  const double* __restrict__ u = V + (uint32_t)(j * D);
  const uint32_t nd = (uint32_t)a.num_dn;
  double acc = 0.0;
#pragma unroll 1
  for (int s = 0; s < S; ++s, k += 64) {
    if (k - lane >= D) break;  // uniform over the block
    double h = 0.0;
    if (k < D) {
      const uint32_t iu = (uint32_t)k / nd, id = (uint32_t)k - iu * nd;
      // the hop slots dealt over the waves: the first half takes the up hops
      // (slots past a state's count hold target 0 and value 0)
      const bool up = wave < kReorthWaves / 2;
      const int32_t* cp = up ? a.up_col + (int64_t)iu * a.up_w : a.dn_col + id;
      const double* vp = up ? a.up_val + (int64_t)iu * a.up_w : a.dn_val + id;
      const uint32_t es = up ? 1u : nd;       // table entries between slots
      const uint32_t mul = up ? nd : 1u;      // source = base + target * mul
      const double* ub = up ? u + id : u + (int64_t)iu * nd;
      const int hops = up ? hops_up : hops_dn;
#pragma unroll 2
      for (int e = wave & (kReorthWaves / 2 - 1); e < hops; e += kReorthWaves / 2)
        h = fma(vp[(uint32_t)e * es], ub[(uint32_t)cp[(uint32_t)e * es] * mul], h);
      if (wave == kReorthWaves - 1) h += (a.d_up[iu] + a.d_dn[id] + hv_u_term(a, a.st_up[iu] & a.st_dn[id])) * u[k];
    }
    if (s > 0) __syncthreads();  // the previous tile's dots are done
    tile_fill(v, tile, V, D, k, wave, lane, j);
    if (s + 1 < S) tile_request(v, V, D, k + 64, wave, j);
    const double wk = wave_total(sx * h, L, wave, lane);  // 0 past the last state
    if (wave == 0 && k < D) w[k] = wk;
    acc = tile_dots(acc, L, lg, j);
  }
  const double d = group_sum(acc, L, lg);
  if ((int)threadIdx.x <= j) part[(int64_t)blockIdx.x * kReorthMaxVectors + threadIdx.x] = d;
}

// One Gram-Schmidt pass from the dots in part.  first: alpha_j is set and the
// next pass's dots go to out; else partials of |w|^2.
__global__ __launch_bounds__(kReorthThreads) void k_reorth_pass(const double* __restrict__ V, int64_t D, int j,
                                                                LzCoef c, const double* __restrict__ part,
                                                                double* __restrict__ w, double* __restrict__ out,
                                                                int S, int lg, int first) {
  extern __shared__ double tile[];
  __shared__ double red[kReorthThreads];
  __shared__ double tot[64];
  __shared__ double cs[kReorthMaxVectors];
  const ReorthLds L{red, tot, tile};
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  int k = (int)blockIdx.x * S * 64 + lane;
  const int nblk = (int)gridDim.x;
  double v[kPre];
  tile_request(v, V, D, k, wave, j);
  double wk = k < D ? w[k] : 0.0;
  {
    // coefficients: thread t sums vector t mod 2^lg over the blocks t >> lg, ...
    const int i = threadIdx.x & ((1 << lg) - 1);
    const int gs = kReorthThreads >> lg;
    const double* p = part + (i <= j ? i : j);
    double d = 0.0;
    for (int b = threadIdx.x >> lg; b < nblk; b += gs * kPre) {
      double t[kPre];
#pragma unroll
      for (int r = 0; r < kPre; ++r) t[r] = p[min(b + gs * r, nblk - 1) * kReorthMaxVectors];
#pragma unroll
      for (int r = 0; r < kPre; ++r)
        if (b + gs * r < nblk) d += t[r];
    }
    d = group_sum(d, L, lg);
    if ((int)threadIdx.x <= j) {
      const double s = c.scale[threadIdx.x], sd = s * d;
      cs[threadIdx.x] = sd * s;  // (s * s may overflow: the start vector's length is the caller's)
      if (first && (int)threadIdx.x == j && blockIdx.x == 0) c.alpha[j] = sd;
    }
  }
  double acc = 0.0;
#pragma unroll 1
  for (int s = 0; s < S; ++s, k += 64) {
    if (k - lane >= D) break;  // uniform over the block
    __syncthreads();           // the coefficients are set, the previous tile's dots done
    tile_fill(v, tile, V, D, k, wave, lane, j);
    const double w0 = wk;
    if (s + 1 < S) {
      tile_request(v, V, D, k + 64, wave, j);
      wk = k + 64 < D ? w[k + 64] : 0.0;
    }
    double t = 0.0;
#pragma unroll 4
    for (int i = wave; i <= j; i += kReorthWaves) t = fma(cs[i], tile[i * 64 + lane], t);
    // w - sum, through the total so that the dots see it too; 0 past the last state
    if (wave == 0) t -= w0;
    if (k >= D) t = 0.0;
    const double wn = -wave_total(t, L, wave, lane);
    if (wave == 0 && k < D) w[k] = wn;
    if (first)
      acc = tile_dots(acc, L, lg, j);
    else
      acc = fma(wn, wn, acc);
  }
  if (first) {
    // the tile held -w
    const double d = -group_sum(acc, L, lg);
    if ((int)threadIdx.x <= j) out[(int64_t)blockIdx.x * kReorthMaxVectors + threadIdx.x] = d;
  } else if (wave == 0) {
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if (lane == 0) out[blockIdx.x] = acc;
  }
}

ReorthGrid reorth_grid(int64_t D) {
  const int64_t tiles = (D + 63) / 64;
  ReorthGrid g;
  g.sub = (int)((tiles + kReorthBlocks - 1) / kReorthBlocks);
  g.blocks = (int)((tiles + g.sub - 1) / g.sub);
  return g;
}

bool grant_lds(const void* kernel, size_t bytes) {
  struct Grant {
    int device;
    const void* kernel;
    size_t bytes;
  };
  static std::mutex mu;
  static std::vector<Grant> granted;
  if (bytes <= 65536) return true;
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::lock_guard<std::mutex> lk(mu);
  for (const Grant& g : granted)
    if (g.device == dev && g.kernel == kernel && g.bytes >= bytes) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  granted.push_back({dev, kernel, bytes});
  return true;
}

bool reorth_available() {
  const size_t bytes = kReorthMaxVectors * 64 * sizeof(double);
  return grant_lds((const void*)k_reorth_hv, bytes) && grant_lds((const void*)k_reorth_pass, bytes);
}

int launch_reorth_step(const ed_op* op, const double* V, int64_t D, int j, LzCoef c, double* part, double* part2,
                       const HvBeta& prev, double* nout, hipStream_t s) {
  const ReorthGrid g = reorth_grid(D);
  double* w = const_cast<double*>(V) + (int64_t)(j + 1) * D;
  const dim3 grid((unsigned)g.blocks), block(kReorthThreads);
  const int lg = j < 64 ? 6 : (j < 128 ? 7 : 8);
  const size_t lds = sizeof(double) * 64 * (size_t)(j + 1);
  hipLaunchKernelGGL(k_reorth_hv, grid, block, lds, s, make_hv_args(op), op->max_hops_up, op->max_hops_dn, V, (int)D, j, c,
                     prev, w, part, g.sub, lg);
  hipLaunchKernelGGL(k_reorth_pass, grid, block, lds, s, V, (int)D, j, c, part, w, part2, g.sub, lg, 1);
  hipLaunchKernelGGL(k_reorth_pass, grid, block, lds, s, V, (int)D, j, c, part2, w, nout, g.sub, lg, 0);
  ED_HIP(hipGetLastError());
  return ED_OK;
}

}  // namespace ed
