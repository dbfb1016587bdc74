// Internal: host-side validation and pack of a j-set upload (regf_pack.cpp).
// Not part of the public ABI.
#pragma once

#include <functional>

namespace abyss {

constexpr int kPackBadState = 1;    // non-finite position or velocity
constexpr int kPackBadMass = 2;     // non-finite or negative mass
constexpr int kPackBadRadius = 3;   // NaN or negative r_nb^2
// Below this many particles the pack runs on the calling thread alone.
constexpr int kPackParallelMin = 16384;

// The lowest-indexed invalid particle (index -1: every particle is valid)
// and what is wrong with it.
struct PackStatus {
    int index = -1;
    int kind = 0;
};

// Validates particles [j0, j1) of n (x, v: [n][3]; m, r2: [n]) and packs
// them into the device layout: soa = 8 arrays of n doubles
// [x|y|z|vx|vy|vz|m|r2], m32 = the masses rounded to FP32.  After a failure
// soa / m32 hold partial contents.
PackStatus pack_jset(int n, int j0, int j1, const double *m, const double *x, const double *v,
                     const double *r2, double *soa, float *m32);

// The same over all n particles, positions first: once every position is
// packed and valid, `positions_done` runs (once, on the calling thread)
// while the other threads pack the rest (velocities, masses, radii), so a
// caller can copy the three position arrays meanwhile.  It does not run
// when a position is invalid.  Returns the first invalid particle as
// pack_jset does.
PackStatus pack_jset_staged(int n, const double *m, const double *x, const double *v,
                            const double *r2, double *soa, float *m32,
                            const std::function<void()> &positions_done);

// Host threads a job can run on, the caller's included (1: none started).
int host_parts();
// Runs f(0) on the caller and f(1) ... f(parts - 1) on the pool's threads
// (parts <= host_parts()); returns when all are done.  False, with nothing
// run, when another caller's job holds the pool.
bool host_run(int parts, const std::function<void(int)> &f);

// Copies `steps` pieces that arrive one after the other: wait(k) returns once
// piece k is there (false: it will not be), here(k) tells without waiting, and
// copy(k0, k1, p, parts) copies part p of the pieces [k0, k1).  Only the
// calling thread waits, and the pool is free meanwhile: a job on up to `parts`
// threads copies the pieces that have arrived.  False when a wait failed.
bool copy_arriving(int steps, int parts, const std::function<bool(int)> &wait,
                   const std::function<bool(int)> &here,
                   const std::function<void(int, int, int, int)> &copy);

// Copies the populated entries (min(|counts[k]|, cap)) of list rows [k0, k1)
// from `rows` (row stride `stride`) to `list` (row stride cap).
void unpack_rows(int k0, int k1, const int *counts, const int *rows, size_t stride, int cap,
                 int *list);

}  // namespace abyss
