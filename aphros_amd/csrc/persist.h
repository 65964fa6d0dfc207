// Resident solves of small systems (persist.hip): one cooperative launch runs
// many iterations of CONJUGATE, JACOBI or Jacobi-scaled PCG with the system's
// coefficients and vectors held on the chip.
#pragma once

#include "common.h"

namespace aph {

constexpr int kPersThreads = 512;
constexpr int kPersMaxBlocks = 256;  // workgroups of one launch (slots per phase)
constexpr int kPersPhases = 2;
constexpr int kPersWords = 4;        // 64-bit words of one slot (two tagged doubles)
// slots of one system: phases x workgroups x words, and the word in which a
// launch is kept or given up
constexpr long long kPersSlotBytes = 8LL * kPersPhases * kPersMaxBlocks * kPersWords + 256;

// How one system runs in a resident launch (a property of the system and the
// device alone): boxes of by x bz whole rows, py x pz of them, one workgroup
// each; shape: the kernel instance (columns per thread, cells per column).
struct PersPlan {
  int by, bz, py, pz, nblk;
  int shape;
  int lds;  // dynamic LDS bytes
};

// One system of a resident launch.
struct PersRec {
  int sys, blk0, nblk;
  int by, bz, py;
  unsigned long long* slots;  // kPersSlotBytes, zeroed once
};

// Ticks of the 100 MHz counter (negative: none at all) after which a workgroup
// stops waiting for the others' sums (gather) and a wavefront for its
// neighbours' before it loads their rows early (early; it then loads them
// behind the gather).
struct PersWait {
  long long gather = 200000000, early = 200000000;
};
// a wait (gather) with which launch_pers() answers as the runtime does when it
// cannot place a cooperative launch
constexpr long long kPersRefuse = -0x7fffffffffffffffLL - 1;

// Plan of a system of method (Method), element type and size on a device of
// ncu compute units; false: the system is not for a resident launch.
bool pers_plan(int method, int fp32, int nx, int ny, int nz, int ncu, PersPlan* out);

// Runs up to `iters` iterations of every system of recs (all of one kernel
// instance: shape and, for PCG, has_m) in one cooperative launch of nblk
// workgroups with `lds` bytes of dynamic LDS; crowded: nblk is more than the
// device's compute units (at most pers_per_unit() times as many).  recs and b2r
// (workgroup -> record) are device arrays; tag: the launch's first tag, larger
// than every tag the slots have seen (a launch uses fewer than 2 * iters + 2).
// A system whose workgroups did not meet keeps the state it had before the
// launch and gets pers_fail = 1.  An error of the launch itself leaves
// everything as it was.
hipError_t launch_pers(int method, int fp32, int has_m, int shape, int lds, const SysDev* sds,
                       const PersRec* recs, const int* b2r, int nblk, bool crowded, int iters,
                       unsigned tag, PersWait wait, hipStream_t st);

// Workgroups of a kernel instance (of a crowded launch) that one compute unit of
// the current device holds at once, with `lds` bytes of dynamic LDS each.
int pers_per_unit(int method, int fp32, int has_m, int shape, int lds);

// Compute units of a device for pers_plan: 0 if it cannot launch
// cooperatively.
int pers_units(int device);

}  // namespace aph
