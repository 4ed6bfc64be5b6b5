// pgk_rules.h - launch choices that follow from a call's sizes alone.
#pragma once
#include <stdint.h>

// Whether the reciprocal chain forks onto the second stream beside the pair
// kernel.  on: pgk_tune has not switched it off; chosen: pgk_tune has switched
// it on; step: the call is a step of a trajectory, queued far ahead of the
// device; bonded: bonded terms are due in the call as well, and every step has
// such a call; work: list entries + grid points.
//
// Such a step pays about 12 us for the fork and the join, which the shorter
// side of a small system of rigid molecules does not earn back.  us per step
// of rigid water, beside / one after the other, by work:
//   mixed  159 k 103/99  300 k 113/108  419 k 130/125  512 k 132/130
//          546 k 132/131  594 k 134/136  710 k 123/137
//   FP32   159 k 102/96  300 k 110/106  419 k 124/121  512 k 126/124
//          546 k 128/130  594 k 130/134
//   FP64   159 k 102/97  300 k 119/114  349 k 144/150  419 k 141/140
//          512 k 136/138  546 k 137/151
// One line for the three: around it they differ by 2 % either way.
// A fork now and then costs more: with the steps that sample energies alone
// forked, 200 steps of 90 k took 96 us each instead of 87; with RESPA's long
// calls forked (their bonded terms are torsions and 1-4 pairs, the short calls
// between do not fork), an FP64 slab of 378 k 349 us a step instead of 340.
// With bonded terms in the call the fork pays at every size: water and
// 1-propanol 43 k 128/140 (mixed) and 125/140 (FP64), 180 k 112/120 and
// 116/128, 352 k 145/157 and 153/172; butane 52 k 80/91 and 84/96; a slab of
// 198 k 109/115 and 110/116; 16 replicas of water and 1-propanol together 1000
// against 1087.  So it does in single calls, waited for or queued (queued and
// read, water: 44 k 111/121, 159 k 99/102, 419 k 126/132).
static inline bool pgk_pme_beside(bool on, bool chosen, bool step, bool bonded, int64_t work) {
  if (!on) return false;
  if (chosen || !step || bonded) return true;
  return work >= 450000;
}
