// Whole Jacobi-CG solves in one launch, with the solve's vectors resident on the compute units.
//
// For operators of up to about a million rows (see Krylov::resident_plan) an iteration moves so little that
// the two kernels of the streaming solver (k_spmv, k_cg_update) are bound by their launches and by the time a
// few blocks take to fill. Here each block keeps a box of the grid for the whole solve: x, z = D^-1 r, D and the
// couplings of its cells in registers, p with a one-cell halo in LDS. Nothing but one value per halo cell
// and five partial sums leave a block per iteration, and no memory is streamed inside the loop.
//
// Blocks meet once per iteration, in an all-to-all exchange of partial sums that is also the barrier: a
// block stores its sums, waits for those of every block, and adds them in block order, so all blocks
// hold the same bits and take the same decisions. One exchange is enough because everything an iteration
// needs follows from p and z at its start: with q = A p and w = D^-1 q,
//   alpha = r.z / p.q,  x += alpha p,  z -= alpha w  (r = D z is not kept),
//   r.z of the next iterate = r.z - alpha (2 z.q - alpha q.w)   (for beta only),
// and r.z, z.z themselves are summed again from z in the next exchange, so that alpha and the
// convergence test use sums of the actual residual; a relative error e of the predicted r.z only turns
// the next direction by about e. The halo value that travels is w: a block updates z and p at its halo
// cells by the owner's formulas with the owner's operands (explicit fma), so the copies stay equal
// to the owner's bit for bit.
//
// Every 8-byte word that crosses blocks carries its own 32-bit tag (launch and exchange number) beside 32
// bits of payload and is stored and loaded at device scope: a reader waits until the word it needs carries
// the expected tag, so no fence orders payload against flag, and no buffer is cleared between exchanges.
// Mailbox and halo words alternate between two halves from exchange to exchange: a block writes a word of
// exchange k + 2 only after it has seen every block's sums of exchange k + 1, which each block posts after its
// last look at the words of exchange k.
//
// The grid is at most one block per compute unit (a compute unit holds one: 512 threads of up to 252 registers),
// so all blocks of a launch that has the device to itself are resident together. Another process's launches of this
// kind, or any kernel that holds compute units, can keep some of them from starting, and two such launches that
// hold a part of the device each would wait for one another. So a block reports at its gate as it starts and, once
// its part of the operator is loaded, looks whether all have; it closes the gate of a block that has not
// reported within kCgGateTicks. A gate is either passed or closed for good, so all blocks see the same and with
// a closed one all leave, x as it was. Behind the gates every block is on the device and the waits are short; a
// bound on them (kCgWaitTicks and kCgWaitLooks) is left so that they end whatever happens. Either way the
// launch reports that it gave up, and the caller solves with the streaming kernels.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "krylov.hpp"

namespace frehg {

constexpr int kCgNT = 512;          // threads per block
constexpr int kCgHalo = 4;          // halo cells per thread, at most
constexpr int kCgMailWords = 10;    // 8-byte words that one block posts per exchange
constexpr int kCgMaxBlocks = 512;   // one polling thread per block
constexpr int kCgMailFront = kCgMaxBlocks / 2;  // words before the posted ones: the gates, 32 bits per block
constexpr int kCgMaxLds = 62 * 1024;        // dynamic LDS with the operator in registers
constexpr int kCgMaxLdsOp = 158 * 1024;     // and with the operator in LDS (the rest is for the reductions)
// Looks before kCgWaitTicks may end a wait (tens of milliseconds): the clock also runs while the device has
// switched the waves out for another process's.
constexpr unsigned int kCgWaitLooks = 1u << 16;

template <typename T>
struct CgResidentArgs {
  Geo g;
  StencilView<T> A;
  const T* b;
  const T* bn;               // null: b
  T* x;
  const unsigned char* fixed;  // 2D only, may be null
  const T* r0;               // started by a refinement sweep: its residual (b, bn unused, x0 = 0)
  const KrylovCtl* ctl;      // and its control block
  KrylovCtl* out;            // result (device or pinned host memory)
  int* gave_up;              // set to 1 when a wait ends without its word
  int* refused;              // null, or a device word: not 0 on entry when the operator is not to be solved (one
                             // block: cleared again)
  int* failed;               // device word for kernels queued behind: set to 1 unless the solve converges
  double rtol, atol;
  int max_it, guard, x0_zero;
  int tx, ty, tz, ntx, nty, ntz;  // cells per tile, tiles
  unsigned long long *lo[2], *hi[2];  // a tagged word per cell and half (hi: FP64 only)
  unsigned long long* mail;  // 2 x kCgMailWords x blocks, the gates before them
  unsigned int launch;       // 1 .. 2^19 - 1
  // see kCgGateTicks; for tests of the recovery, 0: block 0 closes its own gate / leaves after the first iteration
  long long gate_ticks, wait_ticks;
};

__device__ __forceinline__ void cg_put(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long cg_get(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void cg_fail(int* failed) {
  __hip_atomic_store(failed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void cg_give_up(int* gave_up, int* failed) {
  __hip_atomic_store(gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  cg_fail(failed);
}
__device__ __forceinline__ unsigned long long cg_tagged(unsigned int tag, unsigned int v) {
  return ((unsigned long long)tag << 32) | v;
}
// The gates, a 32-bit word per block before the posted words: 2 launch once the block has started, 2 launch + 1 if
// another block closed it before that.
__device__ __forceinline__ unsigned int* cg_gate(unsigned long long* mail, unsigned int blk) {
  return reinterpret_cast<unsigned int*>(mail - kCgMailFront) + blk;
}
// Waits until block `blk` has started, or closes its gate after `ticks`; whether the gate is closed.
__device__ __forceinline__ bool cg_closed(unsigned int* p, unsigned int launch, long long ticks) {
  const long long t0 = wall_clock64();
  for (;;) {
    unsigned int was = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (was == 2 * launch || was == 2 * launch + 1) return was & 1u;
    if (wall_clock64() - t0 > ticks &&
        __hip_atomic_compare_exchange_strong(p, &was, 2 * launch + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT))
      return true;
  }
}

// Sum over a wave by DPP moves (within rows of 16, then across rows), valid in lane 63: a fixed
// order, and a tenth of the latency of the LDS-permute form, which a solve of a few hundred rows per
// block feels at every exchange.
template <int CTRL, int ROWS>
__device__ __forceinline__ double cg_dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xF, false);
  return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double cg_wave_sum(double v) {
  v = cg_dpp_add<0x111, 0xF>(v);  // row_shr:1
  v = cg_dpp_add<0x112, 0xF>(v);  // row_shr:2
  v = cg_dpp_add<0x114, 0xF>(v);  // row_shr:4
  v = cg_dpp_add<0x118, 0xF>(v);  // row_shr:8
  v = cg_dpp_add<0x142, 0xA>(v);  // row_bcast:15 to rows 1 and 3
  return cg_dpp_add<0x143, 0xC>(v);  // row_bcast:31 to rows 2 and 3
}

// N sums over the block, valid in every thread, with one barrier: consecutive calls alternate between
// the two halves of `red` (2 x 5 sums x waves), so a half is written again only after the barrier of the
// call in between.
template <int N>
__device__ __forceinline__ void cg_block_sums(double (&v)[N], double* red, unsigned int flip) {
  constexpr int NW = kCgNT / kWave;
  double* h = red + (flip & 1u) * 5 * NW;
#pragma unroll
  for (int q = 0; q < N; ++q) v[q] = cg_wave_sum(v[q]);
  if ((threadIdx.x & (kWave - 1)) == kWave - 1) {
#pragma unroll
    for (int q = 0; q < N; ++q) h[q * NW + threadIdx.x / kWave] = v[q];
  }
  __syncthreads();
  // the N x 8 wave sums in the lanes of every wave, added within groups of eight lanes
  static_assert(NW == 8 && N * NW <= kWave, "a lane per wave sum");
  const int lane = threadIdx.x & (kWave - 1);
  double t = lane < N * NW ? h[lane] : 0.0;
  t = cg_dpp_add<0x111, 0xF>(t);
  t = cg_dpp_add<0x112, 0xF>(t);
  t = cg_dpp_add<0x114, 0xF>(t);  // lanes 7 mod 8 hold their group's sum
#pragma unroll
  for (int q = 0; q < N; ++q)
    v[q] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(t), q * NW + NW - 1),
                            __builtin_amdgcn_readlane(__double2loint(t), q * NW + NW - 1));
}

// base[byte offset]: a scalar base and a 32-bit offset, so that no 64-bit address is kept per cell (the
// fields of at most a few million cells stay below 2^32 bytes).
template <typename U>
__device__ __forceinline__ U& cg_at(U* base, unsigned int off) {
  return *reinterpret_cast<U*>(reinterpret_cast<char*>(base) + off);
}
template <typename U>
__device__ __forceinline__ const U& cg_at(const U* base, unsigned int off) {
  return *reinterpret_cast<const U*>(reinterpret_cast<const char*>(base) + off);
}

// z = D^-1 (b - A x) at in-domain cell c (b where x0 = 0; 0 at fixed rows), without contraction: the owner
// of a cell and the blocks that hold it in their halo get the same bits.
template <typename T, bool THREE_D>
__device__ __forceinline__ T cg_start_z(const CgResidentArgs<T>& P, long long c) {
#pragma clang fp contract(off)
  const Geo& g = P.g;
  const double d = (double)P.A.D[c];
  if (P.r0) return (T)((double)P.r0[c] / d);
  if (P.fixed != nullptr && P.fixed[c] != 0) return (T)0;
  double ax = 0.0;
  if (!P.x0_zero) {
    ax = d * (double)P.x[c] + (double)P.A.ax[c] * (double)P.x[c + 1] + (double)P.A.ax[c - 1] * (double)P.x[c - 1] +
         (double)P.A.ay[c] * (double)P.x[c + g.sy] + (double)P.A.ay[c - g.sy] * (double)P.x[c - g.sy];
    if (THREE_D) ax += (double)P.A.az[c] * (double)P.x[c + g.sz] + (double)P.A.az[c - g.sz] * (double)P.x[c - g.sz];
  }
  const T r = (T)((double)P.b[c] - ax);
  return (T)((double)r / d);
}

// CPT cells per thread. T state, double arithmetic (as the streaming kernels).
template <typename T, bool THREE_D, int CPT>
__global__ __launch_bounds__(kCgNT) void k_cg_resident(CgResidentArgs<T> P) {
  extern __shared__ __align__(16) unsigned char cg_lds[];
  __shared__ double red[2 * 5 * (kCgNT / kWave)];
  __shared__ int dead;
  __shared__ long long bound;  // P.wait_ticks (looked at now and then: not worth registers)
  T* sp = reinterpret_cast<T*>(cg_lds);  // p on the tile and its halo
  const Geo& g = P.g;
  const int tid = threadIdx.x;
  const unsigned int nblk = gridDim.x, blk = blockIdx.x;
  // neighbouring tiles on one XCD (workgroups go round-robin over the XCDs)
  const int tile = (int)xcd_remap(blk, nblk);
  const int bx = tile % P.ntx, brest = tile / P.ntx, by = brest % P.nty, bz = brest / P.nty;
  const int i0 = bx * P.tx, j0 = by * P.ty, k0 = bz * P.tz;
  const int px = P.tx + 2, py = px * (P.ty + 2);
  const int ncell = P.tx * P.ty * P.tz;
  auto gidx = [&](int i, int j, int k) -> long long { return THREE_D ? g.idx(i, j, k) : g.sidx(i, j); };
  const bool first = blk == 0 && tid == 0;
  if (P.r0 && P.ctl->done) {  // the sweep met the tolerance: the correction is zero
    for (int l = tid; l < ncell; l += kCgNT) {
      const int lx = l % P.tx, lr = l / P.tx, i = i0 + lx, j = j0 + lr % P.ty, k = k0 + lr / P.ty;
      if (i < g.nx && j < g.ny && (!THREE_D || k < g.nz)) P.x[gidx(i, j, k)] = (T)0;
    }
    if (first) {
      KrylovCtl o = *P.ctl;
      *P.out = o;
    }
    return;
  }
  const int refused =
      P.refused ? __hip_atomic_load(P.refused, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;  // (used below)
  if (tid == 0) {
    dead = 0;
    bound = P.wait_ticks;
    if (nblk > 1)
      (void)__hip_atomic_fetch_max(cg_gate(P.mail, blk), 2 * P.launch + (first && P.gate_ticks == 0 ? 1u : 0u),
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  const int nsp = py * (THREE_D ? P.tz + 2 : 1);
  for (int q = tid; q < nsp; q += kCgNT) sp[q] = (T)0;
  __syncthreads();

  // Up to four cells per thread the operator stays in registers; with eight it is staged in LDS behind p
  // (D; the couplings of the tile and of the row of cells before it).
  constexpr bool KEEP = CPT < 8;
  T* lD = sp + nsp;
  T* lax = lD + ncell;
  T* lay = lax + (P.tx + 1) * P.ty * P.tz;
  T* laz = lay + P.tx * (P.ty + 1) * P.tz;
  const int txy = P.tx * P.ty;
  enum : int { kVal = 1, kEdge = 2, kFixed = 4 };
  // this thread's cells: byte offset in the fields of T, index in sp, kind
  unsigned int off[CPT];
  int ls[CPT], kind[CPT];  // (kind with the cell's row (bits 4-15) and layer (16-27) in the tile)
  T x[CPT], z[CPT], d[CPT], axp[CPT], axm[CPT], ayp[CPT], aym[CPT], azp[CPT], azm[CPT], w[CPT];
  double bb = 0.0;
#pragma unroll
  for (int m = 0; m < CPT; ++m) {
    const int l = tid + m * kCgNT;
    const int lx = l % P.tx, lr = l / P.tx, ly = lr % P.ty, lz = lr / P.ty;
    const int i = i0 + lx, j = j0 + ly, k = k0 + lz;
    const bool val = l < ncell && i < g.nx && j < g.ny && (!THREE_D || k < g.nz);
    const bool edge = val && ((lx == 0 && i > 0) || (lx == P.tx - 1 && i + 1 < g.nx) || (ly == 0 && j > 0) ||
                              (ly == P.ty - 1 && j + 1 < g.ny) ||
                              (THREE_D && ((lz == 0 && k > 0) || (lz == P.tz - 1 && k + 1 < g.nz))));
    ls[m] = val ? (lx + 1) + (ly + 1) * px + (THREE_D ? (lz + 1) * py : 0) : px + 1 + (THREE_D ? py : 0);
    const long long c = val ? gidx(i, j, k) : gidx(0, 0, 0);
    off[m] = (unsigned int)c * (unsigned int)sizeof(T);
    kind[m] = (val ? kVal : 0) | (edge ? kEdge : 0) | (KEEP ? 0 : ((lr & 4095) << 4) | ((lz & 4095) << 16));
    x[m] = z[m] = w[m] = axp[m] = axm[m] = ayp[m] = aym[m] = azp[m] = azm[m] = (T)0;
    d[m] = (T)1;
    if (val) {
      if (KEEP) {
        d[m] = P.A.D[c];
        axp[m] = P.A.ax[c];
        axm[m] = P.A.ax[c - 1];
        ayp[m] = P.A.ay[c];
        aym[m] = P.A.ay[c - g.sy];
        if (THREE_D) {
          azp[m] = P.A.az[c];
          azm[m] = P.A.az[c - g.sz];
        }
      } else {
        lD[l] = P.A.D[c];
        lax[l + lr + 1] = P.A.ax[c];
        if (lx == 0) lax[l + lr] = P.A.ax[c - 1];
        lay[l + lz * P.tx + P.tx] = P.A.ay[c];
        if (ly == 0) lay[l + lz * P.tx] = P.A.ay[c - g.sy];
        if (THREE_D) {
          laz[l + txy] = P.A.az[c];
          if (lz == 0) laz[l] = P.A.az[c - g.sz];
        }
      }
      z[m] = cg_start_z<T, THREE_D>(P, c);
      if (!P.r0) {
        if (P.fixed != nullptr && P.fixed[c] != 0) kind[m] |= kFixed;
        if (!P.x0_zero) x[m] = P.x[c];
        const double bz2 = (double)(P.bn ? P.bn[c] : P.b[c]) / (double)P.A.D[c];
        bb += bz2 * bz2;
      }
      sp[ls[m]] = z[m];  // p = z
    }
    if (CPT >= 4) __builtin_amdgcn_sched_barrier(0);  // (all cells' loads at once would spill)
  }
  // this thread's halo cells: faces x-, x+, y-, y+, z-, z+ of the tile
  unsigned int ho[kCgHalo];  // byte offset in the halo words, or ~0
  int hs[kCgHalo];
  T hz[kCgHalo], hw[kCgHalo];
  {
    const int fxy = P.ty * P.tz, fyx = P.tx * P.tz, fz = THREE_D ? P.tx * P.ty : 0;
    const int e1 = fxy, e2 = 2 * fxy, e3 = e2 + fyx, e4 = e3 + fyx, e5 = e4 + fz, e6 = e5 + fz;
#pragma unroll
    for (int e = 0; e < kCgHalo; ++e) {
      const int h = tid + e * kCgNT;
      ho[e] = ~0u;
      hs[e] = 0;
      hz[e] = hw[e] = (T)0;
      if (nblk > 1 && h < e6) {
        int lx, ly, lz;
        if (h < e2) {
          const int q = h < e1 ? h : h - e1;
          lx = h < e1 ? -1 : P.tx;
          ly = q % P.ty;
          lz = q / P.ty;
        } else if (h < e4) {
          const int q = h < e3 ? h - e2 : h - e3;
          ly = h < e3 ? -1 : P.ty;
          lx = q % P.tx;
          lz = q / P.tx;
        } else {
          const int q = h < e5 ? h - e4 : h - e5;
          lz = h < e5 ? -1 : P.tz;
          lx = q % P.tx;
          ly = q / P.tx;
        }
        const int i = i0 + lx, j = j0 + ly, k = k0 + lz;
        if (i >= 0 && i < g.nx && j >= 0 && j < g.ny && (!THREE_D || (k >= 0 && k < g.nz))) {
          const long long c = gidx(i, j, k);
          ho[e] = (unsigned int)c * 8u;
          hs[e] = (lx + 1) + (ly + 1) * px + (THREE_D ? (lz + 1) * py : 0);
          hz[e] = cg_start_z<T, THREE_D>(P, c);
          sp[hs[e]] = hz[e];
        }
      }
    }
  }
  __syncthreads();
  if (nblk > 1) {
    if (tid < (int)nblk && cg_closed(cg_gate(P.mail, tid), P.launch, P.gate_ticks)) dead = 1;
    __syncthreads();
    if (dead) {
      if (tid == 0) cg_give_up(P.gave_up, P.failed);
      return;
    }
  }

  if (refused) {
    if (first) {
      if (nblk == 1) *P.refused = 0;
      cg_fail(P.failed);
    }
    return;
  }

  // Pause between posting and the first look, in units of 64 clocks: a look that comes too early costs
  // more than the pause (measured, us per iteration at pauses 0 / 8 / 14 / 20 / 26 / 34: 80 thousand rows 5.9 /
  // 4.6 / 4.0 / 3.7 / 3.9 / 4.1; 512 thousand, four cells per thread: 8.2 / 7.7 / 7.1 / 6.7 / 6.2 / 5.7).
  constexpr int kWait = CPT <= 2 ? 22 : (CPT == 4 ? 34 : 44);
  unsigned int flip = 0;
  // Exchange `phase`: sums the N values of v over all blocks, sends w at this block's edge cells and
  // receives it at its halo cells. False when a wait ran out.
  auto exchange = [&](auto& v, unsigned int phase) -> bool {
    constexpr int N = sizeof(v) / sizeof(double);
    const unsigned int tag = (P.launch << 12) | (phase & 4095u);
    unsigned long long* const lo = (phase & 1u) ? P.lo[1] : P.lo[0];
    unsigned long long* const hi = (phase & 1u) ? P.hi[1] : P.hi[0];
    if (nblk > 1) {
#pragma unroll
      for (int m = 0; m < CPT; ++m)
        if (kind[m] & kEdge) {
          if constexpr (sizeof(T) == 8) {
            cg_put(&cg_at(lo, off[m]), cg_tagged(tag, (unsigned int)__double2loint((double)w[m])));
            cg_put(&cg_at(hi, off[m]), cg_tagged(tag, (unsigned int)__double2hiint((double)w[m])));
          } else {
            cg_put(&cg_at(lo, 2 * off[m]), cg_tagged(tag, __float_as_uint((float)w[m])));
          }
        }
    }
    cg_block_sums<N>(v, red, flip++);
    if (nblk == 1) return true;
    // word q of block t at (half kCgMailWords + q) nblk + t
    const unsigned int half = (phase & 1u) * (unsigned int)kCgMailWords;
    if (tid < 2 * N) {
      double s = v[0];
#pragma unroll
      for (int q = 1; q < N; ++q) s = tid >= 2 * q ? v[q] : s;
      cg_put(&cg_at(P.mail, 8u * ((half + tid) * nblk + blk)),
             cg_tagged(tag, (unsigned int)((tid & 1) ? __double2hiint(s) : __double2loint(s))));
    }
    const bool reader = tid < (int)nblk;
    __builtin_amdgcn_s_sleep(kWait);
#pragma unroll
    for (int q = 0; q < N; ++q) v[q] = 0.0;
    long long t0 = 0;
    for (unsigned int spin = 0;; ++spin) {
      bool all = true;
      unsigned long long h0[kCgHalo], h1[kCgHalo], u[2 * N];
      if (reader) {
#pragma unroll
        for (int q = 0; q < 2 * N; ++q) u[q] = cg_get(&cg_at(P.mail, 8u * ((half + q) * nblk) + 8u * tid));
      }
#pragma unroll
      for (int e = 0; e < kCgHalo; ++e)
        if (ho[e] != ~0u) {
          h0[e] = cg_get(&cg_at(lo, ho[e]));
          if (sizeof(T) == 8) h1[e] = cg_get(&cg_at(hi, ho[e]));
        }
      if (reader) {
#pragma unroll
        for (int q = 0; q < N; ++q) {
          all = all && (unsigned int)(u[2 * q] >> 32) == tag && (unsigned int)(u[2 * q + 1] >> 32) == tag;
          v[q] = __hiloint2double((int)(unsigned int)u[2 * q + 1], (int)(unsigned int)u[2 * q]);
        }
      }
#pragma unroll
      for (int e = 0; e < kCgHalo; ++e)
        if (ho[e] != ~0u) {
          all = all && (unsigned int)(h0[e] >> 32) == tag;
          if constexpr (sizeof(T) == 8) {
            all = all && (unsigned int)(h1[e] >> 32) == tag;
            hw[e] = (T)__hiloint2double((int)(unsigned int)h1[e], (int)(unsigned int)h0[e]);
          } else {
            hw[e] = (T)__uint_as_float((unsigned int)h0[e]);
          }
        }
      if (all) break;
      if ((spin & 63u) == 63u) {
        const long long now = wall_clock64();
        if (t0 == 0) t0 = now;
        else if (now - t0 > bound && spin > (bound > 0 ? kCgWaitLooks : 0u)) {
          dead = 1;
          break;
        }
      }
    }
    cg_block_sums<N>(v, red, flip++);  // its barrier also makes `dead` visible
    if (dead) {
      if (tid == 0) cg_give_up(P.gave_up, P.failed);
      return false;
    }
    return true;
  };

  double rz = 0.0, zz = 0.0, pq = 0.0, ttol2 = 0.0;
  int iters = 0, conv = 0, breakdown = 0, rejected = 0;
  if (P.r0) ttol2 = P.ctl->ttol2;
  const bool leave = nblk > 1 && blk == 0 && P.wait_ticks == 0;
  const int max_it = leave ? 1 : P.max_it;
  for (;;) {
    // q = A p, w = D^-1 q, and the sums p.q, z.q, q.w, r.z, z.z
    double v[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < CPT; ++m) {
      // (the addresses of a cell's neighbours in sp are formed here, not kept for every cell)
      if (CPT >= 4) asm volatile("" : "+v"(ls[m]));
      if (!KEEP) asm volatile("" : "+v"(kind[m]));
      const T* c = sp + ls[m];
      const double pc = (double)c[0];
      double y, dd;
      if constexpr (KEEP) {
        dd = (double)d[m];
        y = dd * pc + (double)axp[m] * (double)c[1] + (double)axm[m] * (double)c[-1] + (double)ayp[m] * (double)c[px] +
            (double)aym[m] * (double)c[-px];
        if (THREE_D) y += (double)azp[m] * (double)c[py] + (double)azm[m] * (double)c[-py];
      } else {
        const int l = (kind[m] & kVal) ? tid + m * kCgNT : 0;
        const T* fx = lax + l + ((kind[m] >> 4) & 4095);
        const T* fy = lay + l + ((kind[m] >> 16) & 4095) * P.tx;
        dd = (double)lD[l];
        y = dd * pc + (double)fx[1] * (double)c[1] + (double)fx[0] * (double)c[-1] + (double)fy[P.tx] * (double)c[px] +
            (double)fy[0] * (double)c[-px];
        if (THREE_D) y += (double)laz[l + txy] * (double)c[py] + (double)laz[l] * (double)c[-py];
      }
      if (kind[m] & kVal) {
        w[m] = (T)(y / dd);
        const double zc = (double)z[m];
        v[0] += pc * y;
        v[1] += zc * y;
        v[2] += y * (double)w[m];
        v[3] += dd * zc * zc;
        v[4] += zc * zc;
      }
      if (!KEEP && (m & 3) == 3) __builtin_amdgcn_sched_barrier(0);
    }
    // (p = z at the start, so z.q = p.q there and its place is free for ||D^-1 bn||^2)
    if (iters == 0) v[1] = bb;
    if (!exchange(v, (unsigned int)iters)) return;
    if (iters == 0) {
      if (!P.r0) {
        bb = v[1];
        const double ttol = fmax(P.rtol * sqrt(bb), P.atol);
        ttol2 = ttol * ttol;
        rejected = (P.guard && !P.x0_zero && !(v[4] < bb)) ? 1 : 0;
      }
      v[1] = v[0];
    }
    rz = v[3];
    zz = v[4];
    conv = (zz <= ttol2) ? 1 : 0;
    if (conv || rejected || iters >= max_it) break;
    pq = v[0];
    if (!(pq > 0.0) || !isfinite(pq)) {
      breakdown = 1;
      break;
    }
    const double alpha = rz / pq;
    const double next = rz - alpha * (2.0 * v[1] - alpha * v[2]);
    const double beta = next > 0.0 ? next / rz : 0.0;
#pragma unroll
    for (int m = 0; m < CPT; ++m)
      if (kind[m] & kVal) {
        const double pc = (double)sp[ls[m]];
        x[m] = (T)fma(alpha, pc, (double)x[m]);
        z[m] = (T)fma(-alpha, (double)w[m], (double)z[m]);
        sp[ls[m]] = (T)fma(beta, pc, (double)z[m]);
      }
#pragma unroll
    for (int e = 0; e < kCgHalo; ++e)
      if (ho[e] != ~0u) {
        hz[e] = (T)fma(-alpha, (double)hw[e], (double)hz[e]);
        sp[hs[e]] = (T)fma(beta, (double)sp[hs[e]], (double)hz[e]);
      }
    ++iters;
    __syncthreads();
  }
  if (leave && iters == 1) {
    if (tid == 0) cg_give_up(P.gave_up, P.failed);
    return;
  }
  if (!rejected) {
#pragma unroll
    for (int m = 0; m < CPT; ++m)
      if ((kind[m] & kVal) && !(kind[m] & kFixed)) cg_at(P.x, off[m]) = x[m];
  }
  if (first) {
    KrylovCtl o{};
    o.rz = rz;
    o.zz = zz;
    o.ttol2 = ttol2;
    o.bb = P.r0 ? P.ctl->bb : bb;
    o.pq = pq;
    o.iters = iters;
    o.done = 1;
    o.converged = conv;
    o.breakdown = breakdown;
    o.max_it = P.max_it;
    o.guess_rejected = rejected;
    *P.out = o;
    if (!conv) cg_fail(P.failed);
  }
}

}  // namespace frehg
