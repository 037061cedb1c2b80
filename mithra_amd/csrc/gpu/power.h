// Radiation power P(z) (Solver::powerSample, reference src/radiation.cpp:127-232).
//
// One thread per (plane, transverse node) interpolates E/B to the plane, transforms them to the
// lab frame, stores them in ring slot n_time % Nf and evaluates the Nf-point DFT of the node's ring
// for every frequency; a workgroup reduces its nodes to one partial sum per (plane, frequency), and
// the last workgroup of a plane to finish adds the plane's partials in a fixed order, so P is
// deterministic.
//
// The DFT of a slot does not depend on the step, only the one slot's values change: each
// frequency keeps its eight sums per node and exchanges the slot's old products for the new ones.
// The products are exact (Dekker's two-product by FMA) and the sums are pairs of doubles (Knuth's
// two-sum), so what is taken out is what was put in and the sums carry some 100 bits, more than the
// plain sum over the ring has.  They are summed afresh at slot 0 and whenever a slot does not lie behind the
// one sampled before it (sampler_slot), so that no more than one pass over the ring collects rounding or
// keeps what is left of a value far larger than those after it, however the samples are spaced.  A node whose
// sums are not finite is summed afresh too, and plainly while its ring holds an infinity or a NaN.
//
// Walking the ring of 139-152 slots at every step, with one workgroup per 256 nodes, was bound by the
// latency of those reads on small planes and by the bytes (32 a slot and node) on large ones.  A sample
// of one frequency, launches back to back: 32 x 32 nodes 24 -> 6.7 us, 128 x 128 35 -> 7.9; in a step of
// 256 x 256 nodes 89 -> 19 us between events.
#pragma once

#include "common.h"

namespace mithra {

namespace {

constexpr int kPowerBlock = 256;

struct Sum2 {  // a sum as a pair of doubles
  double hi, lo;
};

// s + x c, the product taken exactly
__device__ inline Sum2 add_product(Sum2 s, double x, double c) {
  const double p = x * c, e = fma(x, c, -p);
  const double t = s.hi + p, b = t - s.hi;
  const double r = ((s.hi - (t - b)) + (p - b)) + (s.lo + e);
  const double h = t + r;
  return {h, r - (h - t)};
}

// The eight sums of one node and frequency, q = 2 field + (0: cos, 1: sin): Ex, Ey, Bx, By of the ring
// times the phases.
struct PowerBufs {
  double* ring;              // [Nf][4][Nz][N1N0]
  double* sums;              // [Nz][Nl][16][N1N0]: hi, lo of the eight sums; nullptr: none are kept
  const double* dft;         // [Nl][Nf][2]
  const int* plane_k;        // [Nz], and after it plane_of[N]
  const double* plane_dzr;
  double* partial;           // [Nz][blocks][Nl]
  unsigned* done;            // [Nz] workgroups of the plane that have finished, zero between launches
  unsigned N, Nz, Nl, Nf;
  double gamma, beta, c0, pc;
};

// The phases are the same for every lane and no kernel writes them: scalar loads, no vector registers.
typedef const double __attribute__((address_space(4))) * Phases;

// The slots of a node's ring in order: use(x, cos, sin) takes a slot's four fields.  Bound by latency, with one
// wavefront to a SIMD, so the loads of U slots and of their phases go out before the first use.  Left to
// itself the compiler keeps one load in flight and waits for each in turn, and it advances a pointer for every
// load; here one pointer steps through the fields, which lie evenly.  A launch of 40 frequencies, 140
// slots, 128 x 128 nodes: 6.4 ms with the loads one by one, 1.1 ms with the phases' loads after the ring's, 0.74 so.
template <int U, class Use>
__device__ inline void walk_ring(gptr<const double> ring, size_t field, Phases w, unsigned Nf, Use use) {
  double x[4 * U], p[2 * U];
  auto load = [&](unsigned m, int n) {
#pragma unroll
    for (int i = 0; i < 2 * n; ++i) p[i] = w[2 * m + i];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4 * n; ++i) {
      x[i] = *ring;
      ring += field;
      asm("" : "+v"(ring));
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  unsigned m = 0;
  for (; m + U <= Nf; m += U) {
    load(m, U);
#pragma unroll
    for (int u = 0; u < U; ++u) use(x + 4 * u, p[2 * u], p[2 * u + 1]);
  }
  for (; m < Nf; ++m) {
    load(m, 1);
    use(x, p[0], p[1]);
  }
}

__device__ inline double power_of(const double* f) {
  // ew1 = sum fdt0 ep, bw1 = sum fdt3 em, ew2 = sum fdt1 ep, bw2 = sum fdt2 em; ep = cos + i sin, em
  // its conjugate
  return (f[0] * f[6] - f[1] * -f[7]) - (f[2] * f[4] - f[3] * -f[5]);
}

// Workgroup bx of nbx of inside plane pz; row receives the plane's N x Nl powers.  fresh: the sums are
// taken from the whole ring.
__device__ inline void power_body(const float* __restrict__ eb, const PowerBufs& B, double* __restrict__ row, int N0,
                                  int N1, unsigned slot, bool fresh, int bx, int nbx, unsigned pz) {
  const long ni_count = (long)(N0 - 4) * (N1 - 4);
  const long t = (long)bx * blockDim.x + threadIdx.x;
  const long N1N0 = (long)N1 * N0;
  const size_t ring_slot = (size_t)4 * B.Nz * N1N0, field = (size_t)B.Nz * N1N0;  // doubles per slot and field
  __shared__ double red[kPowerBlock];
  __shared__ unsigned last;
  const bool own = t < ni_count;
  const long i = own ? 2 + t / (N1 - 4) : 0, j = own ? 2 + t % (N1 - 4) : 0;
  const long node = (long)N1 * i + j;
  const gptr<double> ring = G(B.ring) + (size_t)pz * N1N0 + node;  // of this node: slot m, field f at m ring_slot + f field
  double put[4], old[4] = {0.0, 0.0, 0.0, 0.0};
  if (own) {
    const gptr<const f2> ebg = G(reinterpret_cast<const f2*>(eb));
    const long mi = (long)G(B.plane_k)[pz] * N1N0 + node;
    const double dzr = G(B.plane_dzr)[pz];
    const long na = kEBPairs * mi, nb = kEBPairs * (mi + N1N0);
    const f2 a0 = ebg[na], a1 = ebg[na + 1], a2 = ebg[na + 2];  // {Ex, Ey}, {Ez, Bx}, {By, Bz}
    const f2 b0 = ebg[nb], b1 = ebg[nb + 1], b2 = ebg[nb + 2];
    const double et0 = (1.0 - dzr) * (double)a0.x + dzr * (double)b0.x;
    const double et1 = (1.0 - dzr) * (double)a0.y + dzr * (double)b0.y;
    const double bt0 = (1.0 - dzr) * (double)a1.y + dzr * (double)b1.y;
    const double bt1 = (1.0 - dzr) * (double)a2.x + dzr * (double)b2.x;
    put[0] = B.gamma * (et0 + B.c0 * B.beta * bt1);
    put[1] = B.gamma * (et1 - B.c0 * B.beta * bt0);
    put[2] = B.gamma * (bt0 - B.beta / B.c0 * et1);
    put[3] = B.gamma * (bt1 + B.beta / B.c0 * et0);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      const gptr<double> r = ring + slot * ring_slot + f * field;
      if (B.sums && !fresh) old[f] = *r;
      *r = put[f];
    }
  }
  for (unsigned l = 0; l < B.Nl; ++l) {
    double v = 0.0;
    if (own) {
      const Phases w = (Phases)B.dft + (size_t)l * B.Nf * 2;
      const gptr<double> S = G(B.sums) + ((size_t)pz * B.Nl + l) * 16 * N1N0 + node;
      double sum[8];
      bool finite = false;
      if (B.sums) {
        Sum2 q[8];
        auto settled = [&]() {
          bool ok = true;
#pragma unroll
          for (int k = 0; k < 8; ++k) ok = ok && isfinite(q[k].hi) && isfinite(q[k].lo);
          return ok;
        };
        if (!fresh) {
          const double cs = w[2 * slot], sn = w[2 * slot + 1];
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            q[k] = {S[2 * k * N1N0], S[(2 * k + 1) * N1N0]};
            q[k] = add_product(q[k], put[k >> 1], k & 1 ? sn : cs);
            q[k] = add_product(q[k], -old[k >> 1], k & 1 ? sn : cs);
          }
          finite = settled();
        }
        if (!finite) {
#pragma unroll
          for (int k = 0; k < 8; ++k) q[k] = {0.0, 0.0};
          walk_ring<2>(ring, field, w, B.Nf, [&](const double* x, double cs, double sn) {
#pragma unroll
            for (int f = 0; f < 4; ++f) {
              q[2 * f] = add_product(q[2 * f], x[f], cs);
              q[2 * f + 1] = add_product(q[2 * f + 1], x[f], sn);
            }
          });
          finite = settled();
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          sum[k] = q[k].hi;
          S[2 * k * N1N0] = q[k].hi;
          S[(2 * k + 1) * N1N0] = q[k].lo;
        }
      }
      if (!finite) {
#pragma unroll
        for (int k = 0; k < 8; ++k) sum[k] = 0.0;
        walk_ring<8>(ring, field, w, B.Nf, [&](const double* x, double cs, double sn) {
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            sum[2 * f] += x[f] * cs;
            sum[2 * f + 1] += x[f] * sn;
          }
        });
      }
      v = B.pc * power_of(sum);
    }
    red[threadIdx.x] = v;
    __syncthreads();
    for (int s = kPowerBlock / 2; s > 0; s >>= 1) {
      if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) B.partial[((size_t)pz * nbx + bx) * B.Nl + l] = red[0];
    __syncthreads();
  }
  // The last workgroup of the plane adds its partials.  Thread 0 wrote this workgroup's: its
  // release makes them visible to whoever acquires the count after it.
  if (threadIdx.x == 0)
    last = __hip_atomic_fetch_add(&B.done[pz], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)nbx - 1;
  __syncthreads();
  if (!last) return;  // uniform over the workgroup
  const int* plane_of = B.plane_k + B.Nz;
  const int lane = threadIdx.x & 63;
  for (unsigned l = threadIdx.x >> 6; l < B.Nl; l += kPowerBlock / 64) {  // a frequency to a wavefront
    double s = 0.0;  // every 64th partial, then the lanes' sums in a fixed tree
    for (int b = lane; b < nbx; b += 64)
      s += __hip_atomic_load(&B.partial[((size_t)pz * nbx + b) * B.Nl + l], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) s += __shfl_xor(s, h);
    for (unsigned k = lane; k < B.N; k += 64)
      if (plane_of[k] == (int)pz) row[k * B.Nl + l] = s;
  }
  if (threadIdx.x == 0) B.done[pz] = 0;  // for the next launch
}

// The slot a domain samples at n_time, and whether its sums start afresh there.
inline unsigned sampler_slot(Domain* d, unsigned n_time, bool* fresh) {
  const unsigned slot = n_time % d->pNf;
  *fresh = slot == 0 || (long)slot <= d->pslot;
  d->pslot = slot;
  return slot;
}

// Of a Domain or a BatchView (their members are named alike)
template <typename D>
__host__ __device__ inline PowerBufs power_bufs(const D& d) {
  return {d.ring, d.psums, d.dft, d.pk, d.pdzr, d.partial, d.pdone, d.pN, d.pNz, d.pNl, d.pNf, d.pgamma, d.pbeta,
          d.pc0, d.pc};
}

}  // namespace

}  // namespace mithra
