// Resident solves of small systems (gfx950).
//
// A system of up to 2^21 cells needs a few microseconds of work per iteration
// while launching an iteration's kernels costs tens: at 64^3 the reference CG
// took 31 us per iteration in four graph-replayed launches, each mostly launch
// gap and dependent memory round trips.  Here one cooperative launch runs
// hundreds of iterations: a workgroup owns a box of whole rows, keeps the
// box's coefficients and vectors in registers and the stencil's vector in LDS
// (own rows and one row of halo on each side), and the workgroups meet twice
// per iteration in an all-gather of their partial sums (gather()).
//
// Exchange between workgroups.  L2 is per XCD, so what another workgroup
// reads goes through agent-scope relaxed atomics (written through, read past
// L2).  A partial sum is published as tagged 64-bit words (32 bits of data, 32
// of tag), so a reader needs no flag besides the data, and one round trip both
// reduces and synchronises: 64 workgroups 2.6 us, 256 3.9 us per gather, where
// release / acquire fences (which write back and invalidate L2) cost 6.7 and
// 20 us.  Boundary rows of the residual are stored before the partial sum
// that follows them (s_waitcnt vmcnt(0), then the workgroup barrier, then the
// sum's words), so a workgroup that has gathered every sum finds its
// neighbours' rows in memory.  Each row buffer is overwritten only after a
// gather that its readers reach after reading it.
//
// Microseconds per iteration, iteration kernels in graph replays -> resident:
// reference CG 64^3 31.0 -> 6.4; reference Jacobi 60 x 45 x 52 16.4 -> 4.7;
// PCG mixed 101 x 75 x 93 46 -> 10.5 (with a mass term 11.1), FP64 128^3 52.9 ->
// 22 (mixed 128^3 14).  What bounds an iteration is waiting, 70 to 78 % of the
// wavefronts' time by counters: its two gathers and the halo rows behind one of
// them; then the stencil's LDS reads (0.35 us per cell and thread); at 16 cells
// per thread in FP64 also the x and y conductances, read again in every
// iteration (67 MB at 128^3, 3.4 TB/s).
//
// Every workgroup sums the partials in the same order, so all of them hold
// the same scalars and take the same branches, and the result depends neither
// on scheduling nor on the other systems of the launch.
//
// The launch is cooperative (all workgroups resident).  Every wait ends all the
// same: a workgroup that has waited too long (another process's resident
// launch may hold half of the device and wait for the other half) asks for the
// launch to be given up.  Whether a system's launch counts is decided once, in
// one word that the first workgroup to ask sets (decide()): one that has all
// sums of the last gather asks to keep the launch, one whose wait has passed to
// give it up, and all follow that word.  No workgroup writes any state before a
// launch is kept; a given-up launch leaves the state as it was, and the host
// goes on with the iteration kernels.
#include "persist.h"

#include "kernels.h"
#include "reduce.h"

namespace aph {

namespace {

constexpr int kT = kPersThreads;
constexpr int kWaves = kT / 64;
using u64 = unsigned long long;
template <typename T>
using gp = const __attribute__((address_space(1))) T*;

template <typename T>
__device__ __forceinline__ T ld_agent(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_agent(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Makes a register opaque at this point of a loop, so that what is computed
// from it (addresses, conversions) is not hoisted into registers of its own.
template <typename T>
__device__ __forceinline__ void opaque(T& v) {
  asm volatile("" : "+v"(v));
}

constexpr long long kPersAgain = 200000000;  // ticks; values known to be there
constexpr int kGroups = kPersMaxBlocks / 64;  // slot groups, one wave reads each

struct Shared {
  double red[2][kWaves];
  double out[2][kGroups];
  int bad[kGroups];
  int flag;  // what one thread read for all
};

// Keeps (keep) a system's launch, whose first tag is `launch`, or gives it up:
// true if it is kept.  The first workgroup's answer holds for all.
__device__ __forceinline__ bool decide(u64* word, unsigned launch, bool keep, Shared& sh) {
  if (threadIdx.x == 0) {
    u64 w = ld_agent(word);
    // (other launches' words have other tags; this one's is never replaced, so
    // a failed exchange has found it)
    if ((unsigned)(w >> 32) != launch) {
      const u64 mine = ((u64)launch << 32) | (keep ? 1u : 0u);
      if (__hip_atomic_compare_exchange_strong(word, &w, mine, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT))
        w = mine;
    }
    sh.flag = (int)(w & 1u);
  }
  __syncthreads();
  const bool kept = sh.flag != 0;
  __syncthreads();
  return kept;
}

__device__ __forceinline__ u64* pers_word(const PersRec& rc) {
  return rc.slots + kPersPhases * kPersMaxBlocks * kPersWords;
}

// Whether a system takes no part in this launch, read once for the workgroup
// (one that gives up stores pers_fail while others may just start).
__device__ __forceinline__ bool passed_by(bool skip, Shared& sh) {
  if (threadIdx.x == 0) sh.flag = skip ? 1 : 0;
  __syncthreads();
  const bool out = sh.flag != 0;
  __syncthreads();
  return out;
}

// The second half of gather(): waits for the values of all workgroups.
template <int NV, unsigned MaxMask>
__device__ __forceinline__ bool collect(double (&v)[NV], const u64* slots, int nblk, unsigned tag,
                                        long long wait, Shared& sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ngrp = (nblk + 63) >> 6;
  if (wave < ngrp) {
    // wave w reads the slots 64 w .. 64 w + 63, one per lane
    const int i = lane + 64 * wave;
    const u64* s = slots + (long long)i * kPersWords;
    u64 w[2 * NV];
    bool need = i < nblk, bad = false;
    const long long t0 = wall_clock64();
    for (int n = 1;; ++n) {
      if (need) {
#pragma unroll
        for (int k = 0; k < 2 * NV; ++k) w[k] = ld_agent(s + k);
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 2 * NV; ++k) ok = ok && (unsigned)w[k] == tag;
        need = !ok;
      }
      if (!__any(need)) break;
      if (((n & 255) == 0 && wall_clock64() - t0 > wait) || wait < 0) {
        bad = true;
        break;
      }
    }
    double t[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k)
      t[k] = i < nblk ? __longlong_as_double((long long)((w[2 * k + 1] & 0xffffffff00000000ull) |
                                                         (w[2 * k] >> 32)))
                      : 0.0;
    wave_reduce<NV, MaxMask>(t);
    if (lane == 0) {
#pragma unroll
      for (int k = 0; k < NV; ++k) sh.out[k][wave] = t[k];
      sh.bad[wave] = bad ? 1 : 0;
    }
  }
  __syncthreads();
  bool ok = sh.bad[0] == 0;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = sh.out[k][0];
  for (int w = 1; w < ngrp; ++w) {
    ok = ok && sh.bad[w] == 0;
#pragma unroll
    for (int k = 0; k < NV; ++k)
      v[k] = ((MaxMask >> k) & 1u) ? fmax(v[k], sh.out[k][w]) : v[k] + sh.out[k][w];
  }
  return ok;
}

// All-gather reduction of NV values (sums, or maxima where flagged in MaxMask)
// over the nblk workgroups of a system; the result is valid in every thread of
// every workgroup, summed in workgroup order.  Every global store this thread
// issued before the call is complete before the workgroup's values appear.
// meanwhile(): run by every wavefront once the workgroup's values are on their
// way, before it waits for the others'.
// Returns false if some workgroup's values did not appear in time.
template <int NV, unsigned MaxMask, class F>
__device__ __forceinline__ bool gather(double (&v)[NV], u64* slots, int nblk, int me,
                                       unsigned tag, long long wait, Shared& sh,
                                       F meanwhile) {
  wave_reduce<NV, MaxMask>(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) sh.red[k][wave] = v[k];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (wave == 0 && lane < 2 * NV) {
    // lane 2 k publishes the low half of value k, lane 2 k + 1 the high half
    const int k = NV > 1 ? lane >> 1 : 0;
    double t = sh.red[k][0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) {
      const double x = sh.red[k][w];
      t = ((MaxMask >> k) & 1u) ? fmax(t, x) : t + x;
    }
    const u64 b = (u64)__double_as_longlong(t);
    st_agent(slots + (long long)me * kPersWords + lane,
             ((lane & 1) ? (b & 0xffffffff00000000ull) : (b << 32)) | tag);
  }
  meanwhile();
  return collect<NV, MaxMask>(v, slots, nblk, tag, wait, sh);
}

// The box of a workgroup and its place in LDS: rows of nx values, (bz + 2) x
// (by + 2) of them (own rows and the halo rows around; the four edge rows are
// not used).
struct Box {
  int nx, ny, nz;
  int y0, z0, by, bz;  // own rows
  int nhalo, nhrow;
  int ly;              // rows per LDS plane
  float inv_nx;
  __device__ Box(const SysDev& s, const PersRec& rc, int lb)
      : nx(s.nx), ny(s.ny), nz(s.nz) {
    y0 = (lb % rc.py) * rc.by;
    z0 = (lb / rc.py) * rc.bz;
    by = min(rc.by, ny - y0);
    bz = min(rc.bz, nz - z0);
    nhrow = 2 * (by + bz);
    nhalo = nx * nhrow;
    ly = by + 2;
    inv_nx = 1.0f / (float)nx;
  }
  // row of linear cell i (exact: i < 2^20, and i + 0.5 keeps the quotient
  // 0.5 / nx away from the next row)
  __device__ int row_of(int i) const { return (int)(((float)i + 0.5f) * inv_nx); }
  __device__ int lds_row(int yy, int zz) const { return ((zz + 1) * ly + yy + 1) * nx; }
};

// flags of a column's LDS offset
constexpr int kXm = 1 << 20, kXp = 1 << 21, kEdge = 1 << 22, kOn = 1 << 23;
constexpr int kOfs = (1 << 20) - 1;

// Own columns: thread t holds the columns t + c * kT of the box's (x, y)
// plane, each bz <= ZC cells in z (so z neighbours are in the thread).
// d: LDS offset of the column's first cell and flags (x wraps on either side;
// the column borders another box in y; the column exists); g: the global
// index of that cell.
template <int CC>
__device__ __forceinline__ void own_columns(const Box& b, int (&d)[CC], int (&g)[CC]) {
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const int i = (int)threadIdx.x + c * kT;
    const bool on = i < b.nx * b.by;
    const int ii = on ? i : 0;
    const int yy = b.row_of(ii), x = ii - yy * b.nx;
    d[c] = (b.lds_row(yy, 0) + x) | (x == 0 ? kXm : 0) | (x == b.nx - 1 ? kXp : 0) |
           (yy == 0 || yy == b.by - 1 ? kEdge : 0) | (on ? kOn : 0);
    g[c] = (b.z0 * b.ny + b.y0 + yy) * b.nx + x;
  }
}

// Table of the halo rows: global index of the row's first cell and its LDS
// offset.  Rows: y-minus and y-plus of every plane, z-minus and z-plus of
// every row.
__device__ __forceinline__ void halo_table(const Box& b, int2* tab) {
  for (int r = threadIdx.x; r < b.nhrow; r += kT) {
    int yy, zz;
    if (r < 2 * b.bz) {
      zz = r >> 1;
      yy = (r & 1) ? b.by : -1;
    } else {
      yy = (r - 2 * b.bz) >> 1;
      zz = (r & 1) ? b.bz : -1;
    }
    int y = b.y0 + yy, z = b.z0 + zz;
    y = y < 0 ? b.ny - 1 : (y >= b.ny ? 0 : y);
    z = z < 0 ? b.nz - 1 : (z >= b.nz ? 0 : z);
    tab[r] = make_int2((z * b.ny + y) * b.nx, b.lds_row(yy, zz));
  }
}

// f(h, value(g), lds offset) over this thread's halo cells from the skip-th on,
// four loads of value(g) in flight
template <class V, class F>
__device__ __forceinline__ void for_halo(const Box& b, const int2* tab, V value, F f,
                                         int skip = 0) {
  constexpr int U = 4;
  for (int h0 = threadIdx.x + skip * kT; h0 < b.nhalo; h0 += U * kT) {
    decltype(value(0)) v[U];
    int o[U];
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int h = h0 + k * kT;
      if (h < b.nhalo) {
        const int row = b.row_of(h), x = h - row * b.nx;
        const int2 t = tab[row];
        o[k] = t.y + x;
        v[k] = value(t.x + x);
      }
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
      const int h = h0 + k * kT;
      if (h < b.nhalo) f(h, v[k], o[k]);
    }
  }
}

// Halo values a thread loads early, by the bytes of one vector of its cells:
// what the registers left over hold.
constexpr int early_halo(int bytes) { return bytes >= 128 ? 0 : (bytes >= 64 ? 2 : 4); }

// The first HR halo values of a thread, loaded while the gather that follows
// their stores is under way: a neighbour's values in that gather say that its
// rows are in memory.  A wavefront that has waited too long for a neighbour
// (late) loads them again when they are used, behind the gather, whose result
// says the same of every neighbour.
template <typename T, int HR>
struct EarlyHalo {
  T v[HR > 0 ? HR : 1];
  bool late = false;  // (the same in every lane)
  int nb;             // slot of the neighbour in y-, y+, z-, z+ (lane % 4)
  __device__ EarlyHalo(const PersRec& rc, int lb) {
    const int pz = rc.nblk / rc.py, jy = lb % rc.py, jz = lb / rc.py;
    const int q = threadIdx.x & 3;
    const int y = q == 0 ? (jy == 0 ? rc.py - 1 : jy - 1)
                         : (q == 1 ? (jy == rc.py - 1 ? 0 : jy + 1) : jy);
    const int z = q == 2 ? (jz == 0 ? pz - 1 : jz - 1)
                         : (q == 3 ? (jz == pz - 1 ? 0 : jz + 1) : jz);
    nb = (z * rc.py + y) * kPersWords;
  }
  __device__ __forceinline__ void rows(const Box& b, const int2* tab, const T* src) {
#pragma unroll
    for (int k = 0; k < HR; ++k) {
      const int h = (int)threadIdx.x + k * kT;
      if (h < b.nhalo) {
        const int row = b.row_of(h);
        v[k] = ld_agent(src + tab[row].x + (h - row * b.nx));
      }
    }
  }
  // waits for the neighbours' values of gather `tag` in `slots`, then starts the
  // loads of rows of src
  __device__ __forceinline__ void load(const Box& b, const int2* tab, const T* src,
                                       const u64* slots, unsigned tag, long long wait) {
    if (HR == 0) return;
    late = wait < 0;
    const long long t0 = wall_clock64();
    for (int n = 1;; ++n) {
      if (!__any((unsigned)ld_agent(slots + nb) != tag)) break;
      if (((n & 255) == 0 && wall_clock64() - t0 > wait) || wait < 0) {
        late = true;
        break;
      }
    }
    rows(b, tab, src);
  }
  // f(h, global index, value, lds offset) of the cells loaded, behind the gather
  // that load() ran ahead of
  template <class F>
  __device__ __forceinline__ void use(const Box& b, const int2* tab, const T* src, F f) {
    if (HR == 0) return;
    if (late) rows(b, tab, src);
#pragma unroll
    for (int k = 0; k < HR; ++k) {
      const int h = (int)threadIdx.x + k * kT;
      if (h < b.nhalo) {
        const int row = b.row_of(h), x = h - row * b.nx;
        const int2 t = tab[row];
        f(h, t.x + x, v[k], t.y + x);
      }
    }
  }
};

// distance in LDS to a column's x neighbours
__device__ __forceinline__ int step_xm(int d, int nx) { return (d & kXm) ? nx - 1 : -1; }
__device__ __forceinline__ int step_xp(int d, int nx) { return (d & kXp) ? 1 - nx : 1; }

#pragma clang fp contract(off)

// Reference CG (k_ref_spmv, k_fin_ref_spmv, k_ref_update, k_fin_ref_update):
// the same operations per cell in the same order; p of the own and halo rows
// in LDS, r, u, q and the first NR of the seven coefficients of the own cells
// in registers (all seven up to 8 cells per thread; the others are read from
// memory in every iteration).
template <int CC, int ZC, int NR>
__global__ __launch_bounds__(kT) void k_pers_cg(const SysDev* __restrict__ sds,
                                                const PersRec* __restrict__ recs,
                                                const int* __restrict__ b2r, int iters,
                                                unsigned tag, PersWait wait) {
  extern __shared__ __align__(16) double sp[];
  __shared__ Shared sh;
  const PersRec rc = recs[b2r[blockIdx.x]];
  const SysDev& s = sds[rc.sys];
  Scalars* sc = s.sc;
  if (passed_by(sc->done || sc->pers_fail, sh)) return;
  const int lb = (int)blockIdx.x - rc.blk0;
  const Box b(s, rc, lb);
  const int nx = b.nx, zs = b.ly * nx, pl = nx * b.ny, bz = b.bz;
  int2* tab = (int2*)(sp + (long long)(bz + 2) * zs);
  const int fs = s.f7sh;
  double* __restrict__ rg = s.rr;
  double* __restrict__ pg = s.pp[sc->cur];
  double* __restrict__ ug = s.u[0];
  double* hg = (double*)s.halo[0];
  halo_table(b, tab);
  int d[CC], g[CC];
  own_columns<CC>(b, d, g);
  double r[CC][ZC], u[CC][ZC], q[CC][ZC], e[CC][ZC][NR];
#pragma unroll
  for (int c = 0; c < CC; ++c) {
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      const bool on = (d[c] & kOn) && j < bz;
      const long long i = g[c] + j * pl;
      r[c][j] = on ? rg[i] : 0.0;
      u[c][j] = on ? ug[i] : 0.0;
      if (on) sp[(d[c] & kOfs) + j * zs] = pg[i];
#pragma unroll
      for (int k = 0; k < NR; ++k) e[c][j][k] = on ? s.f7[k][i << fs] : 0.0;
    }
  }
  __syncthreads();
  for_halo(b, tab, [&](int gi) { return pg[gi]; },
           [&](int, double v, int o) { sp[o] = v; });
  double rho = sc->rho, beta = sc->beta, res = sc->residual;
  const double tol = sc->tol, h3 = sc->h3;
  int first = sc->first, iter = sc->iter, done = 0, conv = 0;
  const int miniter = sc->miniter, maxiter = sc->maxiter, rmode = sc->resmode;
  __syncthreads();
  u64* const sl0 = rc.slots;
  u64* const sl1 = rc.slots + kPersMaxBlocks * kPersWords;
  constexpr int HR = early_halo(8 * CC * ZC);
  EarlyHalo<double, HR> eh(rc, lb);
  bool ok = true;
  // the iteration's end, from the sum of r^2 and the largest |r|
  auto step = [&](const double (&v)[2]) {
    const double dot_r = v[0];
    res = rmode == 1 ? v[1] / h3 : sqrt(dot_r / h3);
    iter += 1;
    beta = dot_r / (rho + 1e-100);
    rho = dot_r;
    first = 0;
    if (iter >= miniter && (iter > maxiter || res < tol)) {
      conv = res < tol ? 1 : 0;
      done = 1;
    }
  };
  int it = 0;
  for (; it < iters && !done; ++it) {
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      opaque(d[c]);
      opaque(g[c]);
    }
    if (!first) {
      const double* hs = it == 0 ? rg : hg;
      if (it > 0)
        eh.use(b, tab, hs, [&](int, int, double v, int o) { sp[o] = v + beta * sp[o]; });
      for_halo(b, tab, [&](int gi) { return ld_agent(hs + gi); },
               [&](int, double v, int o) { sp[o] = v + beta * sp[o]; }, it > 0 ? HR : 0);
#pragma unroll
      for (int c = 0; c < CC; ++c) {
        if (d[c] & kOn) {
#pragma unroll
          for (int j = 0; j < ZC; ++j) {
            const int o = (d[c] & kOfs) + j * zs;
            if (j < bz) sp[o] = r[c][j] + beta * sp[o];
          }
        }
      }
      __syncthreads();
    }
    double acc[1] = {0.0};
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if (!(d[c] & kOn)) continue;
      const int o0 = d[c] & kOfs, xm = step_xm(d[c], nx), xp = step_xp(d[c], nx);
      double pm = sp[o0 - zs], pc = sp[o0];
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if (j < bz) {
          const int o = o0 + j * zs;
          const double pn = sp[o + zs];
          double k[7];
#pragma unroll
          for (int f = 0; f < 7; ++f)
            k[f] = f < NR ? e[c][j][f < NR ? f : 0] : s.f7[f][(long long)(g[c] + j * pl) << fs];
          double v = pc * k[0];
          v += sp[o + xm] * k[1];
          v += sp[o + xp] * k[2];
          v += sp[o - nx] * k[3];
          v += sp[o + nx] * k[4];
          v += pm * k[5];
          v += pn * k[6];
          q[c][j] = v;
          acc[0] += pc * v;
          pm = pc;
          pc = pn;
        }
      }
    }
    ok = gather<1, 0u>(acc, sl0, rc.nblk, lb, tag + 2 * it, wait.gather, sh, [] {});
    if (!ok) break;
    const double alpha = rho / (acc[0] + 1e-100);
    double ac2[2] = {0.0, 0.0};
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if (!(d[c] & kOn)) continue;
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if (j < bz) {
          u[c][j] += alpha * sp[(d[c] & kOfs) + j * zs];
          const double rv = r[c][j] - alpha * q[c][j];
          r[c][j] = rv;
          if ((d[c] & kEdge) || j == 0 || j == bz - 1) st_agent(hg + g[c] + j * pl, rv);
          ac2[0] += rv * rv;
          ac2[1] = fmax(ac2[1], fabs(rv));
        }
      }
    }
    ok = gather<2, 2u>(ac2, sl1, rc.nblk, lb, tag + 2 * it + 1, wait.gather, sh,
                       [&] { eh.load(b, tab, hg, sl1, tag + 2 * it + 1, wait.early); });
    if (!ok) break;
    step(ac2);
  }
  if (!decide(pers_word(rc), tag, ok, sh)) {
    if (threadIdx.x == 0) st_agent(&sc->pers_fail, 1);
    return;
  }
  if (!ok) {
    // kept by a workgroup that found this gather, the last, complete
    double v[2];
    collect<2, 2u>(v, sl1, rc.nblk, tag + 2 * it + 1, kPersAgain, sh);
    step(v);
  }
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    if (!(d[c] & kOn)) continue;
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      if (j < bz) {
        const int i = g[c] + j * pl;
        ug[i] = u[c][j];
        rg[i] = r[c][j];
        pg[i] = sp[(d[c] & kOfs) + j * zs];
      }
    }
  }
  if (lb == 0 && threadIdx.x == 0) {
    sc->rho = rho;
    sc->beta = beta;
    sc->residual = res;
    sc->first = first;
    sc->iter = iter;
    sc->converged = conv;
    sc->done = done;
  }
}

// Jacobi sweeps (k_jacobi, k_fin_jacobi), the same operations per cell: one
// gather per sweep (the largest change).  Boundary rows alternate between two
// arrays: a workgroup that is one sweep ahead must not overwrite rows its
// neighbours still read.  The iterate starts and ends in u[0].
// NR: of the eight terms, those held in registers.
template <int CC, int ZC, int NR>
__global__ __launch_bounds__(kT) void k_pers_jacobi(const SysDev* __restrict__ sds,
                                                    const PersRec* __restrict__ recs,
                                                    const int* __restrict__ b2r, int iters,
                                                    unsigned tag, PersWait wait) {
  extern __shared__ __align__(16) double sp[];
  __shared__ Shared sh;
  const PersRec rc = recs[b2r[blockIdx.x]];
  const SysDev& s = sds[rc.sys];
  Scalars* sc = s.sc;
  if (passed_by(sc->done || sc->pers_fail, sh)) return;
  const int lb = (int)blockIdx.x - rc.blk0;
  const Box b(s, rc, lb);
  const int nx = b.nx, zs = b.ly * nx, pl = nx * b.ny, bz = b.bz;
  int2* tab = (int2*)(sp + (long long)(bz + 2) * zs);
  const int fs = s.f7sh;
  double* ug = s.u[0];
  halo_table(b, tab);
  int d[CC], g[CC];
  own_columns<CC>(b, d, g);
  double e[CC][ZC][NR], v[CC][ZC];
#pragma unroll
  for (int c = 0; c < CC; ++c) {
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      const bool on = (d[c] & kOn) && j < bz;
      const long long i = g[c] + j * pl;
      v[c][j] = on ? ug[i] : 0.0;
      if (on) sp[(d[c] & kOfs) + j * zs] = v[c][j];
#pragma unroll
      for (int k = 0; k < NR; ++k) e[c][j][k] = on ? s.f7[k][i << fs] : 0.0;
    }
  }
  __syncthreads();
  for_halo(b, tab, [&](int gi) { return ug[gi]; },
           [&](int, double w, int o) { sp[o] = w; });
  double res = sc->residual;
  const double tol = sc->tol;
  int iter = sc->iter, done = 0, conv = 0;
  const int miniter = sc->miniter, maxiter = sc->maxiter;
  u64* const sl0 = rc.slots;
  u64* const sl1 = rc.slots + kPersMaxBlocks * kPersWords;
  constexpr int HR = early_halo(8 * CC * ZC);
  EarlyHalo<double, HR> eh(rc, lb);
  bool ok = true;
  // the sweep's end, from its largest change
  auto step = [&](const double (&v)[1]) {
    res = v[0];
    iter += 1;
    if (iter >= miniter && (iter > maxiter || res < tol)) {
      conv = res < tol ? 1 : 0;
      done = 1;
    }
  };
  __syncthreads();
  int it = 0;
  for (; it < iters && !done; ++it) {
    double* const ub = (double*)s.halo[it & 1];
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      opaque(d[c]);
      opaque(g[c]);
    }
    double acc[1] = {0.0};
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if (!(d[c] & kOn)) continue;
      const int o0 = d[c] & kOfs, xm = step_xm(d[c], nx), xp = step_xp(d[c], nx);
      double um = sp[o0 - zs];
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if (j < bz) {
          const int o = o0 + j * zs;
          const double uc = v[c][j];
          const double un = j + 1 < bz ? v[c][j + 1 < ZC ? j + 1 : j] : sp[o + zs];
          double k[8];
#pragma unroll
          for (int f = 0; f < 8; ++f)
            k[f] = f < NR ? e[c][j][f < NR ? f : 0] : s.f7[f][(long long)(g[c] + j * pl) << fs];
          double nd = k[7];
          nd += sp[o + xm] * k[1];
          nd += sp[o + xp] * k[2];
          nd += sp[o - nx] * k[3];
          nd += sp[o + nx] * k[4];
          nd += um * k[5];
          nd += un * k[6];
          const double w = -nd / k[0];
          acc[0] = fmax(acc[0], fabs(w - uc));
          if ((d[c] & kEdge) || j == 0 || j == bz - 1) st_agent(ub + g[c] + j * pl, w);
          um = uc;
          v[c][j] = w;
        }
      }
    }
    // (the gather's barriers separate these reads of LDS from the writes below)
    u64* const sl = (it & 1) ? sl1 : sl0;
    ok = gather<1, 1u>(acc, sl, rc.nblk, lb, tag + it, wait.gather, sh,
                       [&] { eh.load(b, tab, ub, sl, tag + it, wait.early); });
    if (!ok) break;
    step(acc);
    eh.use(b, tab, ub, [&](int, int, double w, int o) { sp[o] = w; });
    for_halo(b, tab, [&](int gi) { return ld_agent(ub + gi); },
             [&](int, double w, int o) { sp[o] = w; }, HR);
#pragma unroll
    for (int c = 0; c < CC; ++c) {
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if ((d[c] & kOn) && j < bz) sp[(d[c] & kOfs) + j * zs] = v[c][j];
      }
    }
    __syncthreads();
  }
  if (!decide(pers_word(rc), tag, ok, sh)) {
    if (threadIdx.x == 0) st_agent(&sc->pers_fail, 1);
    return;
  }
  if (!ok) {
    // kept by a workgroup that found this gather, the last, complete
    double v[1];
    collect<1, 1u>(v, (it & 1) ? sl1 : sl0, rc.nblk, tag + it, kPersAgain, sh);
    step(v);
  }
#pragma unroll
  for (int c = 0; c < CC; ++c) {
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      if ((d[c] & kOn) && j < bz) ug[g[c] + j * pl] = v[c][j];
    }
  }
  if (lb == 0 && threadIdx.x == 0) {
    sc->residual = res;
    sc->iter = iter;
    sc->converged = conv;
    sc->cur = 0;
    sc->done = done;
  }
}

#pragma clang fp contract(on)

// Jacobi-scaled PCG (k_pcg_spmv<T, VX, true, true>, k_fin_pcg_spmv,
// k_pcg_update, k_fin_pcg_update): the same operations per cell, with the
// same rounding of the stored p, q, r and x^ to T.  u = S p (FP64) of the own
// and halo rows in LDS, beside the halo's p; r, p, q, x^, S and the face
// conductances of the own cells in registers (kz of the face below a cell is
// that of the cell below, in the same thread).  KXY = false: the x and y
// conductances are read from memory in every iteration (FP64 boxes of more
// than 8 cells per thread).  Ends early when a reliable update is due
// (sc->ru), with the state that k_ru_accum expects.
// WG: workgroups that a compute unit is to hold, as far as registers go.
template <typename T, int CC, int ZC, bool HM, bool KXY, int WG = 1>
__global__ __launch_bounds__(kT, WG * kT / 256) void k_pers_pcg(const SysDev* __restrict__ sds,
                                                 const PersRec* __restrict__ recs,
                                                 const int* __restrict__ b2r, int iters,
                                                 unsigned tag, PersWait wait) {
  extern __shared__ __align__(16) double sp[];
  __shared__ Shared sh;
  const PersRec rc = recs[b2r[blockIdx.x]];
  const SysDev& s = sds[rc.sys];
  Scalars* sc = s.sc;
  if (passed_by(sc->done || sc->ru || sc->pers_fail, sh)) return;
  const int lb = (int)blockIdx.x - rc.blk0;
  const Box b(s, rc, lb);
  const int nx = b.nx, ny = b.ny, zs = b.ly * nx, pl = nx * b.ny, bz = b.bz;
  T* ph = (T*)(sp + (long long)(bz + 2) * zs);  // p of the halo cells
  int2* tab = (int2*)(ph + ((b.nhalo + 1) & ~1));
  T* __restrict__ rg = (T*)s.r;
  T* __restrict__ pg = (T*)s.p[sc->cur];
  T* __restrict__ xg = (T*)s.xh;
  T* hg = (T*)s.halo[0];
  const T* __restrict__ Sg = (const T*)s.S;
  const T* __restrict__ kxg = (const T*)s.kx;
  const T* __restrict__ kyg = (const T*)s.ky;
  const T* __restrict__ kzg = (const T*)s.kz;
  const T* __restrict__ mg = (const T*)s.m;
  halo_table(b, tab);
  int d[CC], g[CC];
  own_columns<CC>(b, d, g);
  // FP64 at 8 cells per thread has no registers left for the mass term
  constexpr bool MREG = HM && sizeof(T) * CC * ZC < 64;
  constexpr int CK = KXY ? CC : 1, ZK = KXY ? ZC : 1;
  T r[CC][ZC], p[CC][ZC], q[CC][ZC], S[CC][ZC], x[CC][ZC], kz[CC][ZC], kz0[CC];
  T kx[CK][ZK], kw[CK][ZK], ky[CK][ZK], ks[CK][ZK];  // own and minus x and y faces
  T m[MREG ? CC : 1][MREG ? ZC : 1];
  const int fold0 = sc->xh_fold;
  // global index of a column's y-minus neighbour relative to the column
  auto step_ym = [&](int gc) {
    const int y = (gc / nx) % ny;
    return y == 0 ? (ny - 1) * nx : -nx;
  };
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    const bool con = d[c] & kOn;
    kz0[c] = con ? kzg[b.z0 == 0 ? g[c] + (b.nz - 1) * pl : g[c] - pl] : (T)0;
    const int ym = step_ym(g[c]), xm = step_xm(d[c], nx);
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      const bool on = con && j < bz;
      const int i = g[c] + j * pl;
      r[c][j] = on ? rg[i] : (T)0;
      p[c][j] = on ? pg[i] : (T)0;
      S[c][j] = on ? Sg[i] : (T)0;
      x[c][j] = on && fold0 == 0 ? xg[i] : (T)0;
      kz[c][j] = on ? kzg[i] : (T)0;
      if constexpr (KXY) {
        kx[c][j] = on ? kxg[i] : (T)0;
        kw[c][j] = on ? kxg[i + xm] : (T)0;
        ky[c][j] = on ? kyg[i] : (T)0;
        ks[c][j] = on ? kyg[i + ym] : (T)0;
      }
      if constexpr (MREG) m[c][j] = on ? mg[i] : (T)0;
    }
  }
  __syncthreads();
  for_halo(b, tab, [&](int gi) { return pg[gi]; }, [&](int h, T v, int) { ph[h] = v; });
  double rho = sc->rho, beta = sc->beta, alpha = sc->alpha, rho_pend = 0.0;
  const double tol = sc->tol, delta = sc->delta, gamma = sc->gamma, rmax2 = sc->rmax2;
  int iter = sc->iter, fold = fold0, status = sc->status, done = 0, ru = 0;
  const int maxiter = sc->maxiter;
  u64* const sl0 = rc.slots;
  u64* const sl1 = rc.slots + kPersMaxBlocks * kPersWords;
  constexpr int HR = early_halo((int)sizeof(T) * CC * ZC);
  EarlyHalo<T, HR> eh(rc, lb);
  bool ok = true;
  struct RS {
    T r, S;
  };
  // (r, r) says that a reliable update is due
  auto due = [&](double rn) {
    const double est = gamma * sqrt(rn);
    return !isfinite(rn) || sqrt(rn) < delta * sqrt(rmax2) || est <= 0.9 * tol || iter > maxiter;
  };
  int it = 0, half = 0;  // half: the iteration's gathers passed
  for (; it < iters && !done && !ru; ++it) {
    half = 0;
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      opaque(d[c]);
      opaque(g[c]);
      if constexpr (sizeof(T) == 4) {  // or their FP64 values would be kept too
#pragma unroll
        for (int j = 0; j < ZC; ++j) {
          opaque(S[c][j]);
          opaque(kz[c][j]);
          if constexpr (KXY) {
            opaque(kx[c][j]);
            opaque(kw[c][j]);
            opaque(ky[c][j]);
            opaque(ks[c][j]);
          }
          if constexpr (MREG) opaque(m[c][j]);
        }
      }
    }
    // p = r + beta p; x^ += alpha p_old as in k_pcg_spmv (fold 0 and 2)
    const T* hs = it == 0 ? rg : hg;
    auto halo_p = [&](int h, T rh, T Sh, int o) {
      const T pn = (T)((double)rh + beta * (double)ph[h]);
      ph[h] = pn;
      sp[o] = (double)Sh * (double)pn;
    };
    if (it > 0)
      eh.use(b, tab, hs, [&](int h, int gi, T rh, int o) { halo_p(h, rh, Sg[gi], o); });
    for_halo(
        b, tab, [&](int gi) { return RS{ld_agent(hs + gi), Sg[gi]}; },
        [&](int h, RS v, int o) { halo_p(h, v.r, v.S, o); }, it > 0 ? HR : 0);
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if (!(d[c] & kOn)) continue;
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if (j < bz) {
          const double po = (double)p[c][j];
          if (fold == 0) {
            if (alpha != 0.0) x[c][j] = (T)((double)x[c][j] + alpha * po);
          } else if (fold == 2) {
            x[c][j] = (T)(0.0 + alpha * po);
          }
          p[c][j] = (T)((double)r[c][j] + beta * po);
          sp[(d[c] & kOfs) + j * zs] = (double)S[c][j] * (double)p[c][j];
        }
      }
    }
    __syncthreads();
    double acc[1] = {0.0};
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if (!(d[c] & kOn)) continue;
      const int o0 = d[c] & kOfs, xm = step_xm(d[c], nx), xp = step_xp(d[c], nx);
      const int ym = KXY ? 0 : step_ym(g[c]);
      double um = sp[o0 - zs], uc = (double)S[c][0] * (double)p[c][0];
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if (j < bz) {
          const int o = o0 + j * zs, i = g[c] + j * pl;
          const int jn = j + 1 < ZC ? j + 1 : j;
          const double un =
              j + 1 < bz ? (double)S[c][jn] * (double)p[c][jn] : sp[o + zs];
          const T kzm = j > 0 ? kz[c][j > 0 ? j - 1 : 0] : kz0[c];
          double l = (double)kz[c][j] * (uc - un) + (double)kzm * (uc - um);
          const int ck = KXY ? c : 0, jk = KXY ? j : 0;
          const T kyc = KXY ? ky[ck][jk] : kyg[i], kym = KXY ? ks[ck][jk] : kyg[i + ym];
          const T kxc = KXY ? kx[ck][jk] : kxg[i], kxm = KXY ? kw[ck][jk] : kxg[i + xm];
          l += (double)kym * (uc - sp[o - nx]);
          l += (double)kyc * (uc - sp[o + nx]);
          l += (double)kxc * (uc - sp[o + xp]) + (double)kxm * (uc - sp[o + xm]);
          if constexpr (HM) l += (double)(MREG ? m[MREG ? c : 0][MREG ? j : 0] : mg[i]) * uc;
          q[c][j] = (T)((double)S[c][j] * l);
          acc[0] += (double)p[c][j] * (double)q[c][j];
          um = uc;
          uc = un;
        }
      }
    }
    ok = gather<1, 0u>(acc, sl0, rc.nblk, lb, tag + 2 * it, wait.gather, sh, [] {});
    if (!ok) break;
    const double pq = acc[0];
    fold = fold == 1 ? 2 : 0;
    if (!(pq != 0.0) || !isfinite(pq)) {
      status = 6;
      done = 1;
      break;
    }
    alpha = rho / pq;
    half = 1;
    double ac2[1] = {0.0};
#pragma unroll
    for (int c = 0; c < CC; ++c) {
      if (!(d[c] & kOn)) continue;
#pragma unroll
      for (int j = 0; j < ZC; ++j) {
        if (j < bz) {
          const T rv = (T)((double)r[c][j] - alpha * (double)q[c][j]);
          r[c][j] = rv;
          if ((d[c] & kEdge) || j == 0 || j == bz - 1) st_agent(hg + g[c] + j * pl, rv);
          ac2[0] += (double)rv * (double)rv;
        }
      }
    }
    ok = gather<1, 0u>(ac2, sl1, rc.nblk, lb, tag + 2 * it + 1, wait.gather, sh,
                       [&] { eh.load(b, tab, hg, sl1, tag + 2 * it + 1, wait.early); });
    if (!ok) break;
    const double rn = ac2[0];
    iter += 1;
    if (due(rn)) {
      ru = 1;
      rho_pend = rn;
    } else {
      beta = rn / rho;
      rho = rn;
    }
  }
  if (!decide(pers_word(rc), tag, ok, sh)) {
    if (threadIdx.x == 0) st_agent(&sc->pers_fail, 1);
    return;
  }
  if (!ok) {
    // kept by a workgroup that found this gather, the last, complete: the second
    // of an iteration, or the first of one whose operator ends the solve
    double v[1];
    collect<1, 0u>(v, half ? sl1 : sl0, rc.nblk, tag + 2 * it + half, kPersAgain, sh);
    const double rn = v[0];
    if (!half) {
      fold = fold == 1 ? 2 : 0;
      status = 6;
      done = 1;
    } else {
      iter += 1;
      if (due(rn)) {
        ru = 1;
        rho_pend = rn;
      } else {
        beta = rn / rho;
        rho = rn;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < CC; ++c) {
    if (!(d[c] & kOn)) continue;
#pragma unroll
    for (int j = 0; j < ZC; ++j) {
      if (j < bz) {
        const int i = g[c] + j * pl;
        rg[i] = r[c][j];
        pg[i] = p[c][j];
        if (fold == 0) xg[i] = x[c][j];
      }
    }
  }
  if (lb == 0 && threadIdx.x == 0) {
    sc->rho = rho;
    sc->beta = beta;
    sc->alpha = alpha;
    sc->iter = iter;
    sc->xh_fold = fold;
    sc->status = status;
    sc->done = done;
    if (ru) {
      sc->rho_pend = rho_pend;
      sc->ru = 1;
    }
  }
}

// LDS of a box: u or p of the own and halo rows, the halo's p (PCG), the
// halo row table
long long lds_bytes(int method, int fp32, int nx, int by, int bz) {
  long long b = 8LL * nx * (by + 2) * (bz + 2) + 8LL * 2 * (by + bz);
  if (method == kPcg) {
    const long long nh = 2LL * nx * (by + bz);
    b += (fp32 ? 4 : 8) * ((nh + 1) & ~1LL);
  }
  return b;
}

// The kernel instances: columns per thread and cells per column.
constexpr int kShapes[][2] = {{1, 1}, {1, 2}, {1, 4}, {1, 8}, {2, 8}};
constexpr int kNumShapes = sizeof(kShapes) / sizeof(kShapes[0]);

}  // namespace

int pers_units(int device) {
  int coop = 0, ncu = 0;
  if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, device) != hipSuccess ||
      !coop ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess)
    return 0;
  return ncu;
}

bool pers_plan(int method, int fp32, int nx, int ny, int nz, int ncu, PersPlan* out) {
  const long long n = (long long)nx * ny * nz;
  const int nbmax = ncu < kPersMaxBlocks ? ncu : kPersMaxBlocks;
  if (n > (1LL << 21) || nbmax < 1) return false;
  // Of the boxes that fit, the one with the smallest estimate.  Measured (us
  // per iteration): CG 64^3 with 64 / 128 / 256 workgroups 8.1 / 7.2 / 9.2,
  // 32^3 with 16 / 32 / 64 / 128 5.9 / 5.7 / 5.5 / 6.0; PCG mixed 101 x 75 x
  // 93 with 96 / 128 / 180 / 240 14.4 / 13.1 / 11.6 / 11.6.  2^21 cells are
  // what 256 workgroups of 16 cells per thread hold.
  auto each = [&](auto f) {
    for (int pz = 1; pz <= nz && pz <= nbmax; ++pz) {
      const int bz = (nz + pz - 1) / pz;
      if ((nz + bz - 1) / bz != pz) continue;
      for (int py = 1; py <= ny && py * pz <= nbmax; ++py) {
        const int by = (ny + py - 1) / py;
        if ((ny + by - 1) / by != py) continue;
        int shape = 0;
        while (shape < kNumShapes &&
               ((long long)nx * by > (long long)kShapes[shape][0] * kPersThreads ||
                bz > kShapes[shape][1]))
          ++shape;
        if (shape == kNumShapes) continue;
        const long long lds = lds_bytes(method, fp32, nx, by, bz);
        if (lds > 156 * 1024) continue;
        const int nb = py * pz;
        const int cpt = kShapes[shape][0] * kShapes[shape][1];
        // gathers, own cells (twice the price with two columns per thread:
        // fewer wavefronts' worth of latency hidden per cell), halo cells
        const double cost = 4.2 + (nb <= 64 ? 0.04 * nb : 2.56 + 0.02 * (nb - 64)) +
                            0.4 * kShapes[shape][0] * bz * (cpt == 16 ? 2.0 : 1.0) +
                            0.0007 * (2.0 * nx * (by + bz));
        f(cost, PersPlan{by, bz, py, pz, nb, shape, (int)lds});
      }
    }
  };
  double best = -1;
  each([&](double cost, const PersPlan& p) {
    if (best < 0 || cost < best) {
      best = cost;
      *out = p;
    }
  });
  if (best < 0) return false;
  // PCG systems come in batches, whose launches hold more of them the fewer
  // workgroups each takes.  Up to 2^13 cells the fewest within 2 % of the best
  // (16^3 with 16 / 8 alone 0.97 / 0.98 ms, 400 in a batch mixed 12.9 / 7.2, FP64
  // 13.2 / 8.2); above, half the device's within 2.5 % (mixed 72^3 with 132 / 121
  // alone 5.73 / 5.86 ms, 24 in a batch 133 / 71).
  if (method != kPcg) return true;
  if (n <= (1LL << 13)) {
    double bc = best;
    each([&](double cost, const PersPlan& p) {
      if (cost > 1.02 * best || p.nblk > out->nblk || (p.nblk == out->nblk && cost >= bc)) return;
      bc = cost;
      *out = p;
    });
  } else if (out->nblk > nbmax / 2) {
    double bc = 1.025 * best;
    each([&](double cost, const PersPlan& p) {
      if (p.nblk > nbmax / 2 || cost > bc) return;
      bc = cost;
      *out = p;
    });
  }
  return true;
}

namespace {

// The kernel instance of a system; crowded: of a launch with more workgroups
// than compute units.  PCG at 4 cells per thread in FP32 and 2 in FP64 then has
// an instance of its own with the registers that let a unit hold two
// workgroups (fewer cells fit two anyway; mixed at 8 cells would spill 300 and
// more, 80^3 x 24 166 -> 178 ms).  The registers it spills cost a lone solve
// (mixed 64^3 4.60 -> 4.76 ms), two workgroups per unit shorten a batch: mixed
// 64^3 x 96 225 -> 147 ms, FP64 24^3 x 200 27.1 -> 19.3, 32^3 x 96 22.9 -> 17.0.
const void* pers_kernel(int method, int fp32, int has_m, int shape, bool crowded) {
#define APH_K(...) return (const void*)(__VA_ARGS__)
  if (method == kConjugate) {
    switch (shape) {
      case 0: APH_K(k_pers_cg<1, 1, 7>);
      case 1: APH_K(k_pers_cg<1, 2, 7>);
      case 2: APH_K(k_pers_cg<1, 4, 7>);
      case 3: APH_K(k_pers_cg<1, 8, 7>);
      default: APH_K(k_pers_cg<2, 8, 2>);
    }
  }
  if (method == kJacobi) {
    switch (shape) {
      case 0: APH_K(k_pers_jacobi<1, 1, 8>);
      case 1: APH_K(k_pers_jacobi<1, 2, 8>);
      case 2: APH_K(k_pers_jacobi<1, 4, 8>);
      case 3: APH_K(k_pers_jacobi<1, 8, 8>);
      default: APH_K(k_pers_jacobi<2, 8, 4>);
    }
  }
#define APH_PCG(T, HM)                                                 \
  switch (shape) {                                                     \
    case 0: APH_K(k_pers_pcg<T, 1, 1, HM, true>);                      \
    case 1:                                                            \
      if (crowded) APH_K(k_pers_pcg<T, 1, 2, HM, true, 2>);            \
      APH_K(k_pers_pcg<T, 1, 2, HM, true>);                            \
    case 2:                                                            \
      if (crowded) APH_K(k_pers_pcg<T, 1, 4, HM, true, (sizeof(T) == 4 ? 2 : 1)>);  \
      APH_K(k_pers_pcg<T, 1, 4, HM, true>);                            \
    case 3: APH_K(k_pers_pcg<T, 1, 8, HM, true>);                      \
    default: APH_K(k_pers_pcg<T, 2, 8, HM, (sizeof(T) == 4)>);         \
  }
  if (fp32) {
    if (has_m) {
      APH_PCG(float, true)
    } else {
      APH_PCG(float, false)
    }
  } else {
    if (has_m) {
      APH_PCG(double, true)
    } else {
      APH_PCG(double, false)
    }
  }
#undef APH_PCG
#undef APH_K
}

}  // namespace

int pers_per_unit(int method, int fp32, int has_m, int shape, int lds) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
          &n, pers_kernel(method, fp32, has_m, shape, true), kT, (size_t)lds) != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  return n < 1 ? 1 : n;
}

hipError_t launch_pers(int method, int fp32, int has_m, int shape, int lds, const SysDev* sds,
                       const PersRec* recs, const int* b2r, int nblk, bool crowded, int iters,
                       unsigned tag, PersWait wait, hipStream_t st) {
  if (wait.gather == kPersRefuse) return hipErrorCooperativeLaunchTooLarge;
  void* args[] = {(void*)&sds,   (void*)&recs, (void*)&b2r,
                  (void*)&iters, (void*)&tag,  (void*)&wait};
  return hipLaunchCooperativeKernel(pers_kernel(method, fp32, has_m, shape, crowded), dim3(nblk),
                                    dim3(kT), args, (unsigned)lds, st);
}

}  // namespace aph
