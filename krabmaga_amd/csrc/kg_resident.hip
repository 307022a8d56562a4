// kg_resident.hip -- the resident kernel (kg_resident.hpp): one work-group
// per run, many schedule steps to a launch.
#include "kg_launch.hpp"
#include "kg_resident.hpp"

namespace kg {

// tab[0..n) (counts) becomes its exclusive prefix and tab[n] the total, by
// the whole work-group.
template <int kT>
__device__ __forceinline__ void res_scan(uint32_t* tab, uint32_t n, uint32_t* s_warp) {
  const uint32_t per = (n + kT - 1) / kT;
  const uint32_t lo = min(n, threadIdx.x * per), hi = min(n, lo + per);
  uint32_t sum = 0;
  for (uint32_t b = lo; b < hi; ++b) sum += tab[b];
  uint32_t total;
  uint32_t run = block_exclusive_scan<kT>(sum, s_warp, &total);
  for (uint32_t b = lo; b < hi; ++b) {
    const uint32_t v = tab[b];
    tab[b] = run;
    run += v;
  }
  if (threadIdx.x == 0) tab[n] = total;
}

// kT threads, up to kB birds each.  What bounds it: one CU's VALU issue (16
// waves, about 1,200 instructions per bird and step in a field of 0.025
// birds per unit^2), not memory: a step touches nothing but LDS.
template <int kT, int kB>
__global__ __launch_bounds__(kT) void k_resident(const RepDev* __restrict__ reps,
                                                 const uint32_t* __restrict__ list, Buf R,
                                                 uint32_t* __restrict__ offset,
                                                 const uint64_t* __restrict__ gstep,
                                                 uint32_t koff, uint32_t nsteps,
                                                 uint32_t* __restrict__ err, uint32_t cap,
                                                 uint32_t bins) {
  extern __shared__ __align__(16) uint8_t smem_raw[];
  __shared__ uint32_t s_warp[kT / kWave];
  __shared__ uint32_t s_bad;
  const uint32_t t = threadIdx.x;
  const RepDev& rp = reps[list ? list[blockIdx.x] : blockIdx.x];
  if (rp.dead) return;
  const Geom& g = rp.g;
  const uint32_t base = offset[rp.bin_base];
  const uint32_t n = offset[rp.bin_base + g.nbins] - base;
  // the host has planned for every run's count
  if (n > cap || n > (uint32_t)(kT * kB) || g.nbins > bins) {
    if (t == 0) atomicOr(err, 4u);
    return;
  }
  const ResSmem S = res_carve(smem_raw, cap);
  const ResBins rb = res_bins(g, bins);
  const CellFind find{S.b.z, S.tab, rb.rows, rb.shift};
  const uint64_t step0 = rp.step_base + *gstep + koff;

  ResBird b[kB];
#pragma unroll
  for (int j = 0; j < kB; ++j) {
    const uint32_t i = (uint32_t)j * kT + t;
    if (i < n) {
      b[j].x = R.x[base + i];
      b[j].y = R.y[base + i];
      b[j].hx = R.hx[base + i];
      b[j].hy = R.hy[base + i];
      b[j].id = R.id[base + i];
    }
  }
  for (uint32_t k = 0;; ++k) {
    // the birds into (bin, row, id) order; after the last step in the read
    // buffer's bins
    const bool last = k == nsteps;
    const uint32_t nb = last ? g.nbins : rb.n;
    for (uint32_t q = t; q < nb; q += kT) S.tab[q] = 0u;
    if (t == 0) s_bad = rp.near ? 0u : 1u;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      if ((uint32_t)j * kT + t < n) {
        res_place(rp, rb, last, &b[j], err);
        b[j].slot = atomicAdd(&S.tab[b[j].bin], 1u);
        if (near_bad(g, b[j].x, b[j].y, b[j].hx, b[j].hy)) s_bad = 1u;
      }
    }
    __syncthreads();
    res_scan<kT>(S.tab, nb, s_warp);
    __syncthreads();
    uint64_t* const key = (uint64_t*)S.b.rec;
#pragma unroll
    for (int j = 0; j < kB; ++j)
      if ((uint32_t)j * kT + t < n) key[S.tab[b[j].bin] + b[j].slot] = res_key(b[j]);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      if ((uint32_t)j * kT + t < n) {
        const uint32_t lo = S.tab[b[j].bin], hi = S.tab[b[j].bin + 1];
        b[j].slot = lo + (hi - lo > 1u
                              ? gather_rank(key, lo, hi, lo + b[j].slot, res_key(b[j]))
                              : 0u);
      }
    }
    if (last) break;
    __syncthreads();  // the keys have been read: the birds take their place
#pragma unroll
    for (int j = 0; j < kB; ++j) {
      if ((uint32_t)j * kT + t < n) {
        S.b.rec[b[j].slot] = NearRec{b[j].x, b[j].y, b[j].hx, b[j].hy};
        S.b.z[b[j].slot] = b[j].z;
        S.b.id[b[j].slot] = b[j].id;
      }
    }
    if (t == 0) S.b.z[n] = ~0u;
    __syncthreads();
    const bool near = s_bad == 0u;
    // bird i of the sorted order: neighbouring lanes walk neighbouring windows
    for (int j = 0; j < kB && (uint32_t)j * kT < n; ++j) {
      const uint32_t i = (uint32_t)j * kT + t;
      NearRec r{0.0f, 0.0f, 0.0f, 0.0f};
      uint32_t id = 0;
      if (i < n) {
        id = S.b.id[i];
        if (near) near_step<true>(rp, 0, step0 + k, i, find, S.b, &r);
        else full_step(rp, step0 + k, i, find, S.b, &r);
      }
      // j is the same on every lane: the birds stay in registers
#pragma unroll
      for (int q = 0; q < kB; ++q) {
        if (q == j) {
          b[q].x = r.x;
          b[q].y = r.y;
          b[q].hx = r.hx;
          b[q].hy = r.hy;
          b[q].id = id;
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kB; ++j) {
    if ((uint32_t)j * kT + t < n) {
      const uint32_t pos = base + b[j].slot;
      R.x[pos] = b[j].x;
      R.y[pos] = b[j].y;
      R.hx[pos] = b[j].hx;
      R.hy[pos] = b[j].hy;
      R.id[pos] = b[j].id;
    }
  }
  for (uint32_t q = t; q < g.nbins; q += kT) offset[rp.bin_base + q] = base + S.tab[q];
}

hipError_t launch_resident(const RepDev* reps, const uint32_t* list, uint32_t nruns, Buf R,
                           uint32_t* offset, const uint64_t* gstep, uint32_t koff,
                           uint32_t nsteps, uint32_t* err, uint32_t cap, uint32_t bins,
                           hipStream_t s) {
  if (nruns == 0 || nsteps == 0) return hipSuccess;
  if (cap > kResidentMaxAgents || nsteps > kResidentSteps) return hipErrorInvalidValue;
  auto go = [&](auto kern, int threads) {
    hipLaunchKernelGGL(kern, dim3(nruns), dim3(threads), res_smem_bytes(cap, bins), s, reps, list,
                       R, offset, gstep, koff, nsteps, err, cap, bins);
  };
  if (cap <= 256) go(k_resident<256, 1>, 256);
  else if (cap <= 512) go(k_resident<512, 1>, 512);
  else if (cap <= 1024) go(k_resident<1024, 1>, 1024);
  else if (cap <= 2048) go(k_resident<1024, 2>, 1024);
  else go(k_resident<1024, 4>, 1024);
  return hipGetLastError();
}

}  // namespace kg
