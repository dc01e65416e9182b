// The resident Krylov engine: a whole solve in one launch, every right-hand side (or segmented
// piece) held by a team of workgroups with its matrix rows and vectors in registers. See
// pp_resident.hip.
#pragma once

#include "pp_krylov.hpp"
#include "pp_patience.hpp"

namespace pp {

constexpr int RES_WG = 512;        // threads of a multi-workgroup team's workgroups
constexpr int RES_LOCAL_WG = 1024; // threads at most of a one-workgroup team
constexpr int RES_TOLS = 8;        // tolerances passed by value
constexpr int RES_SPINS = 1 << 21; // polls a thread spends on one exchange before it gives up, about a microsecond each

// Several right-hand sides are set to x = 0 if all of them are zero, and solved as any other if one is not: a
// zero one is held (SolveRec::zero = ZERO_HELD) until all are known.
enum { ZERO_RUNS = 0, ZERO_SOLVED = 1, ZERO_HELD = 2 };

// Pieces of a segmented solve: piece k has len[k] rows at vector offset base[k], its matrix rows
// start at mrow[k]; workgroup w of the launch works on piece wgPiece[w], whose workgroups are
// wg0[k] .. wg0[k] + G[k] - 1. All null for a plain solve.
struct ResPieces {
    const int32_t *base, *len, *mrow, *wg0, *G, *wgPiece;
};

template <typename T>
struct ResArgs {
    Csr<T> A;
    const T *b;
    T *x, *xbest;                // xbest: null without return-best
    T *x0;                       // gets the start guess, for the host to put back when a team gave up
    const T *dinv;               // Jacobi preconditioner (null: none)
    int dinvStride;
    unsigned long long *zbuf;    // exchanged vectors: [2][vecLen] values in tagged words
    unsigned long long *slots;   // partial sums: [2][3][wgs] values in tagged words
    size_t vecLen, zorigin;      // values per parity; vector offset of the first of them
    SolveRec *recs;              // final records
    unsigned *status;            // per right-hand side: `done` from the team that finished it
    unsigned *failed;            // `done` from a workgroup that gave up waiting
    unsigned *declined;          // `done`: a row is longer than the kernel takes, nothing is solved
    unsigned tag, done;          // the exchanges' first tag less one; the launch's word
    int spins;                   // RES_SPINS, less where a test wants teams to give up
    int n, rpm, G, team0;        // plain solve: rows, right-hand sides per matrix, workgroups per team, first team
    int wgs;                     // workgroups of the launch
    int maxit, returnBest, project, resetEvery;
    int zeroStops;               // a zero right-hand side ends at once: ZERO_SOLVED (x = 0) or ZERO_HELD (x kept)
    int onlyHeld;                // run the right-hand sides held by the launch before, as any other
    double scale;                // 1 / sqrt(n) or 1 (a plain solve)
    double tols[RES_TOLS];       // per right-hand side when tolsDev is null (one: tols[0])
    int ntols;
    const double *tolsDev;
    ResPieces P;
};

// Largest one-workgroup system, in rows, for stencil rows of `ew` entries.
inline int resident_local_rows(int ew) { return (ew == 5 ? 4 : 3) * RES_LOCAL_WG; }

// *declined = word if one of the n CSR rows has more than ew entries; run before the launches that look at it.
int launch_row_check(const int32_t *row, int n, int ew, unsigned *declined, unsigned word, hipStream_t s);

// Launch on `wgs` workgroups: local = every team is one workgroup of `threads` threads with up
// to R rows per thread; otherwise teams of RES_WG-thread workgroups with R rows per thread.
template <typename T>
int launch_resident_cg(const ResArgs<T> &a, int ew, int R, int threads, bool local, hipStream_t s);

} // namespace pp
