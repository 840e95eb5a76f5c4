// The schedule of the record ring of the LU-SGS sweeps (k_sweep_wg): when a record is copied to
// its slot and when it is read from there.  Plain C++ as well, so that a model of the ring on
// the CPU can run the copy waves' own loop.
//
// A step has two phases, with a barrier of the workgroup after each and one barrier before the
// first step; record s is that of step s and takes slot s mod RS.  A wave's LDS reads are
// complete before its next barrier, its copies only where it has waited for them.
#pragma once

namespace ff {

// Slots: what the LDS holds beside the exchange buffers (FWD: the corrector, with the
// increments beside its records; F32: FP32 records).
template <bool FWD, bool F32>
constexpr int ring_slots() { return FWD ? (F32 ? 6 : 3) : (F32 ? 8 : 5); }

// Loads of a copy wave per record (1 KiB each; two waves share a record of 48 fields of 64
// lanes, the corrector's with 8 rows of increments).
template <bool FWD, bool F32>
constexpr int ring_loads() { return (48 * 64 * (F32 ? 4 : 8) + (FWD ? 8 * 64 * 8 : 0)) / 1024 / 2; }

// The phase of step s in which compute wave w reads its face's fields of record s.  Wave 0
// reads the increments' fields a step ahead, in the second phase of the step before.
constexpr int ring_face_phase(int w) { return w > 0 ? 1 : 2; }

// What is in flight, as a type, where a copy wave waits until no more than N loads are.
template <int N>
struct RingLoads { static constexpr int value = N; };

// A copy wave: copy(s) issues its NLD loads of record s, wait(RingLoads<N>()) waits until N of
// its loads are in flight (they complete in order), sync() is the barrier.
//
// The last read of record s is in the second phase of step s (wave 0's face), the first one of
// record s + 1 there too: slot s is free after the second barrier of step s, so its next copy
// starts in the first phase of step s + 1; before the first barrier of step s record s + 1
// must have arrived, and of the copies issued by then (up to record s - 1 + RS) the last RS - 2
// may still be in flight.  (A copy started a phase earlier overtakes wave 0's reads if that
// wave is held up, as by the instruction fetches of a first launch.)
template <int RS, int NLD, typename Copy, typename Wait, typename Sync>
__attribute__((always_inline)) constexpr void ring_copy_wave(int nsteps, Copy copy, Wait wait, Sync sync)
{
    for (int s = 0; s < RS && s < nsteps; s++) copy(s);
    if (RS <= nsteps) wait(RingLoads<NLD * (RS - 1)>()); else wait(RingLoads<0>());
    sync();
    for (int s = 0; s < nsteps; s++) {
        if (s > 0 && s - 1 + RS < nsteps) copy(s - 1 + RS);
        if (s - 1 + RS < nsteps) wait(RingLoads<NLD * (RS - 2)>()); else wait(RingLoads<0>());
        sync();
        sync();
    }
    wait(RingLoads<0>());
}

}  // namespace ff
