// Con2prim kernels for gfx950: AsterX_Con2Prim on a patch (optionally fused
// with ComputedBstagFromA + ComputedBFromdBstag) and Con2PrimFactory solves
// on independent zones.  One work-item per cell; flag and iteration
// histograms are reduced in LDS per block before one atomic per bin.
#include <algorithm>

#include "asx_zone.hpp"

namespace asx {

struct HistLDS {
  unsigned int flags[8];
  unsigned int iters[64];
};

ASX_DEV void hist_init(HistLDS &h) {
  for (int q = threadIdx.x; q < 72; q += blockDim.x) {
    if (q < 8) h.flags[q] = 0;
    else h.iters[q - 8] = 0;
  }
}
ASX_DEV void hist_flush(HistLDS &h, unsigned long long *g) {
  for (int q = threadIdx.x; q < 71; q += blockDim.x) {
    const unsigned v = q < 7 ? h.flags[q] : h.iters[q - 7];
    if (v) atomicAdd(&g[q], (unsigned long long)v);
  }
}

// Pass 1: every zone through the primary solver (Palenzuela, the only one a
// table takes; compiled alone, so the backup costs no registers here).  Where
// there is a backup, zones whose primary solve fails store nothing; a wavefront
// ballot packs their indices into `queue` with one atomic per wavefront.
// Without one they end here, and the queue stays empty.
template <bool FROM_A, class E>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(c2p_waves<E>())))
void k_c2p_main(KPatch P, Box B, E eos, C2PArgs a, unsigned long long *hist, int *queue,
                unsigned *qcount) {
  __shared__ HistLDS h;
  if (hist) {
    hist_init(h);
    __syncthreads();
  }
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = t < B.total();
  bool fail = false;
  if (live) {
    int i, j, k;
    B.ijk(t, i, j, k);
    C2PIn in;
    load_zone<FROM_A>(P, i, j, k, a, in);
    C2POut o;
    if (con2prim_zone<ASX_C2P_PALENZUELA>(eos, a, in, o)) {
      store_zone(P, off(P, 0, i, j, k), o);
      if (hist) {
        atomicAdd(&h.flags[(int)o.flag], 1u);
        atomicAdd(&h.iters[o.iters < 63 ? o.iters : 63], 1u);
      }
    } else {
      fail = true;
    }
  }
  queue_push(fail, (int)t, queue, qcount);
  if (hist) {
    __syncthreads();
    hist_flush(h, hist);
  }
}

// Pass 2: the queued zones through the reference's full chain (primary
// again, then the backup), grid-stride over the device-side count.
template <bool FROM_A, class E>
__global__ __launch_bounds__(256) void k_c2p_rest(KPatch P, Box B, E eos, C2PArgs a,
                                                  unsigned long long *hist, const int *queue,
                                                  const unsigned *qcount) {
  __shared__ HistLDS h;
  if (hist) {
    hist_init(h);
    __syncthreads();
  }
  const unsigned nq = *qcount;
  for (unsigned q = blockIdx.x * blockDim.x + threadIdx.x; q < nq;
       q += gridDim.x * blockDim.x) {
    int i, j, k;
    B.ijk(queue[q], i, j, k);
    C2PIn in;
    load_zone<FROM_A>(P, i, j, k, a, in);
    C2POut o;
    con2prim_cell(eos, a, in, o);
    store_zone(P, off(P, 0, i, j, k), o);
    if (hist) {
      atomicAdd(&h.flags[(int)o.flag], 1u);
      atomicAdd(&h.iters[o.iters < 63 ? o.iters : 63], 1u);
    }
  }
  if (hist) {
    __syncthreads();
    hist_flush(h, hist);
  }
}

// Every zone through the full chain: a zone whose primary fails goes on to
// the backup in its own lane.  Bound by memory on the ideal gas (60 fields a
// zone), whose full chain fits the two wavefronts per SIMD that the primary
// alone takes; so the backup costs the wavefronts that hold a failed zone, and
// on a patch those are few: they lie together, at a shock or the edge of the
// atmosphere.  A second pass over queued zones repeats the failed primary in
// a few wavefronts (253 x 231 x 246 torus, MP5, after 70 substeps: 11.6 ms a
// substep with the queue, 8.73 so; 64^3 WENO-Z 0.219 -> 0.192 ms; 22 x 17 x 13
// con2prim 50 -> 26 us; 192^3, no failed zones: the same), and where they are
// scattered too (con2prim of 128^3, a twentieth of the primaries failed at
// random: 0.80 -> 0.61 ms).
template <bool FROM_A, class E>
__global__ __launch_bounds__(256) void k_c2p_one(KPatch P, Box B, E eos, C2PArgs a,
                                                 unsigned long long *hist) {
  __shared__ HistLDS h;
  if (hist) {
    hist_init(h);
    __syncthreads();
  }
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < B.total()) {
    int i, j, k;
    B.ijk(t, i, j, k);
    C2PIn in;
    load_zone<FROM_A>(P, i, j, k, a, in);
    C2POut o;
    con2prim_cell(eos, a, in, o);
    store_zone(P, off(P, 0, i, j, k), o);
    if (hist) {
      atomicAdd(&h.flags[(int)o.flag], 1u);
      atomicAdd(&h.iters[o.iters < 63 ? o.iters : 63], 1u);
    }
  }
  if (hist) {
    __syncthreads();
    hist_flush(h, hist);
  }
}

__global__ void k_zero_u32(unsigned *p) { *p = 0u; }

// k_c2p_one over the patches of a batch
__global__ __launch_bounds__(256) void k_c2p_patches(const KPatch *__restrict__ tab, IdealGas eos,
                                                     C2PArgs a, const BatchRef *__restrict__ map,
                                                     int nmap) {
  const BatchRef r = map[xcd_tile((int)blockIdx.x, nmap)];
  const KPatch &P = tab[r.pid];
  const int t = r.chunk * 256 + (int)threadIdx.x;
  if (t >= P.n[0] * P.n[1] * P.n[2]) return;
  int i, j, k;
  interior_ijk(P, t, i, j, k);
  C2PIn in;
  load_zone<true>(P, i, j, k, a, in);
  C2POut o;
  con2prim_cell(eos, a, in, o);
  store_zone(P, off(P, 0, i, j, k), o);
}

// Independent zones (layout of asx_c2p_batch in include/asterx.h) in two
// passes without scratch memory: every zone through the primary solver, which
// alone sets the register budget (124 VGPRs for Noble and 114 for Palenzuela,
// 4 waves per SIMD; 241 and 2 for the full chain); a zone it fails gets the
// flag kZoneFailed, which the second pass looks for, and in iters the steps
// of a Newton chain that did not converge, which is not repeated then (-1
// for any other failure).  Bound by the latency of the Newton
// steps' dependent square roots and reciprocals: 4 000 037 zones from the
// previous step's primitives 0.770 -> 0.427 ms (0.10 of them the second pass).
constexpr double kZoneFailed = -1.0;
template <int PRIME>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void k_c2p_zones(int64_t nz, const double *cons, const double *g, const double *seed,
                 double *prim, double *flag, int32_t *iters, IdealGas eos, C2PArgs a) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= nz) return;
  C2PIn in;
  batch_zone_in(z, nz, cons, g, seed, a, in);
  C2POut o;
  if (con2prim_zone<PRIME>(eos, a, in, o)) {
    batch_zone_out(z, nz, o, prim, flag);
    iters[z] = o.iters;
  } else {
    flag[z] = kZoneFailed;
    iters[z] = PRIME == ASX_C2P_NOBLE && o.failed == ST_ROOT_FAIL_CONV ? o.iters : -1;
  }
}
// The failed zones among each wavefront's `per` <= kRestZones, gathered in
// LDS, through the rest of the chain: the latency of the backup's
// iterations, so what counts is that the few zones spread over all SIMDs
// (4 000 037 zones, the failed Newton steps repeated as well: 0.19 ms with
// workgroups of 256 for 4096 zones, 0.13 with a wavefront each; 0.10 without
// the Newton steps).
constexpr int kRestZones = 4096;
__global__ __launch_bounds__(64)
void k_c2p_zones_rest(int64_t nz, int per, const double *cons, const double *g,
                      const double *seed, double *prim, double *flag, int32_t *iters,
                      IdealGas eos, C2PArgs a) {
  __shared__ int list[kRestZones];
  __shared__ int n;
  if (threadIdx.x == 0) n = 0;
  __syncthreads();
  const int64_t z0 = (int64_t)blockIdx.x * per;
#pragma unroll 16
  for (int q = threadIdx.x; q < per; q += 64)
    if (z0 + q < nz && flag[z0 + q] == kZoneFailed) list[atomicAdd(&n, 1)] = q;
  __syncthreads();
  const int nq = n;
  for (int q = threadIdx.x; q < nq; q += 64) {
    const int64_t z = z0 + list[q];
    C2PIn in;
    batch_zone_in(z, nz, cons, g, seed, a, in);
    C2POut o;
    con2prim_cell(eos, a, in, o, -1.0, -1.0, iters[z]);
    batch_zone_out(z, nz, o, prim, flag);
    iters[z] = o.iters;
  }
}
// In one pass, for few zones.
__global__ __launch_bounds__(256) void k_c2p_batch(int64_t nz, const double *cons,
                                                   const double *g, const double *seed,
                                                   double *prim, double *flag,
                                                   int32_t *iters, IdealGas eos,
                                                   C2PArgs a) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= nz) return;
  C2PIn in;
  batch_zone_in(z, nz, cons, g, seed, a, in);
  C2POut o;
  con2prim_cell(eos, a, in, o);
  batch_zone_out(z, nz, o, prim, flag);
  iters[z] = o.iters;
}

template <class E>
static void c2p_one_t(const KPatch &P, const Box &b, const E &eos, const C2PArgs &a,
                      bool from_A, unsigned long long *hist, hipStream_t s) {
  if (from_A) hipLaunchKernelGGL((k_c2p_one<true, E>), b.grid(), dim3(256), 0, s, P, b, eos, a, hist);
  else hipLaunchKernelGGL((k_c2p_one<false, E>), b.grid(), dim3(256), 0, s, P, b, eos, a, hist);
}

static Box c2p_box(const KPatch &P) {
  Box b;
  for (int d = 0; d < 3; ++d) {
    b.lo[d] = P.ng;
    b.cnt[d] = P.n[d];
  }
  return b;
}

hipError_t launch_con2prim_one(const KPatch &P, const IdealGas &eos, const C2PArgs &a,
                               bool from_A, unsigned long long *hist, hipStream_t s) {
  c2p_one_t(P, c2p_box(P), eos, a, from_A, hist, s);
  return hipGetLastError();
}
hipError_t launch_con2prim_one(const KPatch &P, const TabEOS &eos, const C2PArgs &a,
                               bool from_A, unsigned long long *hist, hipStream_t s) {
  c2p_one_t(P, c2p_box(P), eos, a, from_A, hist, s);
  return hipGetLastError();
}

hipError_t launch_con2prim_main(const KPatch &P, const TabEOS &eos, const C2PArgs &a,
                                bool from_A, unsigned long long *hist, int *queue,
                                unsigned *qcount, hipStream_t s) {
  const Box b = c2p_box(P);
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(1), 0, s, qcount);
  if (from_A)
    hipLaunchKernelGGL((k_c2p_main<true, TabEOS>), b.grid(), dim3(256), 0, s, P, b, eos, a, hist, queue, qcount);
  else
    hipLaunchKernelGGL((k_c2p_main<false, TabEOS>), b.grid(), dim3(256), 0, s, P, b, eos, a, hist, queue, qcount);
  return hipGetLastError();
}
hipError_t launch_con2prim_rest(const KPatch &P, const TabEOS &eos, const C2PArgs &a,
                                bool from_A, unsigned long long *hist, const int *queue,
                                const unsigned *qcount, hipStream_t s) {
  const Box b = c2p_box(P);
  // enough work-items for a few percent of the zones; more stride
  const dim3 grid((unsigned)std::min<int64_t>((b.htotal() + 255) / 256, 2048));
  if (from_A)
    hipLaunchKernelGGL((k_c2p_rest<true, TabEOS>), grid, dim3(256), 0, s, P, b, eos, a, hist, queue, qcount);
  else
    hipLaunchKernelGGL((k_c2p_rest<false, TabEOS>), grid, dim3(256), 0, s, P, b, eos, a, hist, queue, qcount);
  return hipGetLastError();
}

hipError_t launch_con2prim_patches(const KPatch *tab, const IdealGas &eos, const C2PArgs &a,
                                   const BatchRef *map, int nmap, hipStream_t s) {
  if (nmap <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_c2p_patches, dim3((unsigned)nmap), dim3(256), 0, s, tab, eos, a, map, nmap);
  return hipGetLastError();
}

hipError_t launch_c2p_batch(int64_t nz, const double *cons, const double *g,
                            const double *seed, double *prim, double *flag,
                            int32_t *iters, const IdealGas &eos, const C2PArgs &a,
                            hipStream_t s) {
  if (nz <= 0) return hipSuccess;
  const dim3 grid((unsigned)((nz + 255) / 256)), block(256);
  if (nz <= kOnePassZones) {
    hipLaunchKernelGGL(k_c2p_batch, grid, block, 0, s, nz, cons, g, seed, prim, flag, iters, eos, a);
    return hipGetLastError();
  }
  if (a.prime == ASX_C2P_NOBLE)
    hipLaunchKernelGGL(k_c2p_zones<ASX_C2P_NOBLE>, grid, block, 0, s, nz, cons, g, seed, prim, flag, iters, eos, a);
  else if (a.prime == ASX_C2P_ENTROPY)
    hipLaunchKernelGGL(k_c2p_zones<ASX_C2P_ENTROPY>, grid, block, 0, s, nz, cons, g, seed, prim, flag, iters, eos, a);
  else
    hipLaunchKernelGGL(k_c2p_zones<ASX_C2P_PALENZUELA>, grid, block, 0, s, nz, cons, g, seed, prim, flag, iters, eos, a);
  // one wavefront for each of the 1024 SIMDs
  const int per = (int)std::min<int64_t>(kRestZones, (nz / 1024 + 64) / 64 * 64);
  hipLaunchKernelGGL(k_c2p_zones_rest, dim3((unsigned)((nz + per - 1) / per)), dim3(64), 0, s,
                     nz, per, cons, g, seed, prim, flag, iters, eos, a);
  return hipGetLastError();
}

} // namespace asx
