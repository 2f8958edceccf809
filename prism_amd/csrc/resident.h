// resident.h -- the resident BiCGSTAB kernel (resident.hip): many iterations in one launch, the
// matrix rows and the vectors in registers.
#pragma once

#include "krylov.h"

namespace prism_hip {

constexpr int RES_BS = 512;  // threads per block
constexpr int RES_MAX_BLOCKS = 255;

// Shape of a resident launch: `blocks` blocks of RES_BS threads with up to R rows each, and one
// more block when there are several (at most one block per compute unit in all); blocks == 0:
// the system does not qualify.
struct ResidentPlan {
    int blocks{0}, R{0};
    int rows{0};  // rows of a block, a multiple of 64
    int W{0};  // entries per row held in registers
};

// Exchange buffers of a solve: every word starts, and is left between launches, as the mark
// (see resident.hip): 5 n words of the iteration's type, and two sets (one per launch, in turn)
// of resident_sums(blocks) partial sums and totals, a 128-byte line for each block.
constexpr int RES_LINE = 16;
constexpr int RES_COPIES = 8;  // of the totals, one for each XCD's blocks
inline size_t resident_sums(int blocks) { return (size_t)RES_LINE * (blocks + RES_COPIES); }
template <typename T>
struct ResidentView {
    T* pub;                     // published p by iteration modulo 3, then s by iteration parity: 5 n
    unsigned long long* slots;  // this launch's partial sums
    unsigned long long* stale;  // the previous launch's, marked again by this one
    int blocks, rows;
    int quota;                  // iterations of this launch at most
    unsigned spin;              // polls of one wait at most
    double* x64;                // mixed precision: x is added here (and cleared) when the launch ends on a flag
};

// Plan for an n-row system (wmax: the longest stored row) on a device of n_cu compute units.
template <typename T>
ResidentPlan resident_plan(int64_t n, bool dia, int wmax, int n_cu);
// Marks `count` words at p and `more` words at q as unwritten.
template <typename T>
void launch_resident_mark(const Launch& L, T* p, size_t count, unsigned long long* q, size_t more);
// Up to rv.quota iterations from the state in kv (p_new, r, r0, rhat, x and kv.ks, as the
// three-kernel iteration keeps them) and back into it, to the next event at most.  A wait
// that runs out (the blocks were not resident together) sets ks->stuck and ends the launch
// without a consistent state: x stays a valid guess, all else is to be seeded again.
template <typename T>
void launch_resident(const Launch& L, const KView<T>& kv, const ResidentView<T>& rv, const ResidentPlan& plan);

}  // namespace prism_hip
