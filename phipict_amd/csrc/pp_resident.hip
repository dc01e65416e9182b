// Krylov solvers of the gfx950 library, part 3: the resident engine. One launch runs a whole CG
// solve of systems whose rows fit the register files: a team of workgroups per right-hand side,
// R rows per thread with their matrix entries, x, r and p in registers for the whole solve.
//
// Why: the multi-launch engine takes 13 us per CG iteration at 108 k rows, of which the memory traffic
// is ~4 us; the rest is the chain of cold loads after every kernel boundary, the fold, the launch. Here
// an iteration is two all-gathers of partial sums through memory (~2 us each) and one exchange of the
// preconditioned residual with the neighbour rows: 7.2 us.
//
// Exchange without fences: every 64-bit word that crosses workgroups carries its own 32-bit tag
// next to 32 bits of payload (a double takes two words), written and read with relaxed agent-scope
// atomics, which go past the L2 caches of the XCDs. A reader polls the word itself until it shows
// the tag of this exchange, so no ordering between different words is needed and no cache is
// written back or invalidated (an agent-scope fence in every wave of 256 workgroups measured 30 us).
// Tags grow from exchange to exchange and from solve to solve, so stale words never match.
// Every tag has exactly one all-gather, of the sums of that exchange (of nothing where only a vector
// is exchanged, at a residual replacement). A word is rewritten two tags later at the earliest (two
// parities). Its writer has then passed the all-gather of the tag between, to which every member
// contributes only when it is done with the words of the tag before: it has passed that tag's
// all-gather and read the vector published with it. Without the all-gather at a replacement a member that
// waits for its stencil neighbours' x alone would overwrite sums that a member farther away still polls.
//
// A team member that waits too long (some other process or a fault keeps a workgroup of the team from
// running) gives up, and says so in the launch's `failed` word: the host then puts the start guess back,
// which teams that finished have overwritten, and runs the solve on the multi-launch engine. A thread
// spends RES_SPINS polls at most on the words of one vector and, in the wave that folds, as many on the
// sums; polls left after a workgroup has given up anywhere in the launch are not made, and a workgroup
// whose vector did not arrive does not wait for sums. The launches of several-workgroup teams that a
// process has on a device have at most one workgroup per CU together (pp_gate.hpp), so that all members
// are resident together.
//
// Recurrences and stopping rules are those of the other engines (pp_krylov.hpp); every thread
// applies them to its own copy of the record, from sums folded in one fixed order by every workgroup.
#include "pp_resident.hpp"

#include <algorithm>

namespace pp {

typedef unsigned long long word_t;
constexpr int RES_WAVES = 16;
constexpr int RES_POLL = 2; // members a lane of the deciding wave polls at a time

__device__ __forceinline__ void put_word(word_t *p, word_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ word_t get_word(const word_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Values in tagged words.
template <typename T> struct Tagged;
template <> struct Tagged<double> {
    static constexpr int W = 2;
    word_t w[2];
    __device__ __forceinline__ void load(const word_t *p) { w[0] = get_word(p); w[1] = get_word(p + 1); }
    __device__ __forceinline__ bool is(unsigned tag) const { return unsigned(w[0] >> 32) == tag && unsigned(w[1] >> 32) == tag; }
    __device__ __forceinline__ double value() const { return __hiloint2double(int(unsigned(w[1])), int(unsigned(w[0]))); }
    __device__ static __forceinline__ void store(word_t *p, double v, unsigned tag) {
        const word_t t = word_t(tag) << 32;
        put_word(p, t | unsigned(__double2loint(v)));
        put_word(p + 1, t | unsigned(__double2hiint(v)));
    }
};
template <> struct Tagged<float> {
    static constexpr int W = 1;
    word_t w;
    __device__ __forceinline__ void load(const word_t *p) { w = get_word(p); }
    __device__ __forceinline__ bool is(unsigned tag) const { return unsigned(w >> 32) == tag; }
    __device__ __forceinline__ float value() const { return __uint_as_float(unsigned(w)); }
    __device__ static __forceinline__ void store(word_t *p, float v, unsigned tag) {
        put_word(p, (word_t(tag) << 32) | __float_as_uint(v));
    }
};

// The value unchanged, opaque to the compiler.
__device__ __forceinline__ int hide(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A workgroup's view of its team.
struct Team {
    word_t *slots;       // [2][3][wgs] tagged doubles
    int wg, wg0, G, wgs; // this workgroup, the team's first, their number, all workgroups of the launch
    unsigned tag;        // of the latest exchange
    Patience fresh;      // what a wait starts with
};
// What wave 0 tells the workgroup after a decision.
struct Verdict {
    double step; // alpha, beta, omega or mean
    int active, fresh, keep, half;
};
struct TeamLds {
    double part[3][RES_WAVES]; // per wave: this workgroup's sums
    SolveRec S;
    Verdict out;
    int bad;  // a word of a vector did not arrive
    int quit; // as of the latest decision: `bad`, or sums that did not arrive (written by the first wave
              // between the barriers of a decision, so that all threads read the same)
};

// The team's totals of v[q], handed to `decide` in wave 0 (all its lanes hold them, the same bits in
// every member: the waves of a workgroup, then the members lane by lane), whose updates of the
// record and verdict every thread sees on return. One wave decides: the rules' square roots
// and divisions in all 16 waves would take longer than the extra barrier. False: a member did not answer.
// `meanwhile` runs in every wave while the sums travel.
template <int NQ, bool LOCAL, typename F, typename G>
__device__ __forceinline__ bool team_decide(Team &tm, const double (&v)[NQ], TeamLds &L, F decide, G meanwhile) {
    const int t = threadIdx.x, waves = (int)blockDim.x >> 6;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const double s = wave_sum0(v[q]);
        if ((t & 63) == 0) L.part[q][t >> 6] = s;
    }
    __syncthreads();
    ++tm.tag;
    word_t *S = tm.slots + (size_t)(tm.tag & 1) * 3 * tm.wgs * 2;
    double tot[NQ];
    if (t < 64) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) tot[q] = wave_total(t < waves ? L.part[q][t] : 0.0);
        if (!LOCAL && t == 0)
#pragma unroll
            for (int q = 0; q < NQ; ++q) Tagged<double>::store(S + ((size_t)q * tm.wgs + tm.wg) * 2, tot[q], tm.tag);
    }
    meanwhile();
    if (t < 64) {
        if (!LOCAL) {
            double got[NQ];
#pragma unroll
            for (int q = 0; q < NQ; ++q) got[q] = 0.0;
            bool late = L.bad != 0;
            Patience left = tm.fresh;
            if (late) left.left = 0;
            for (int g0 = 0; g0 < tm.G; g0 += 64 * RES_POLL) {
                Tagged<double> m[RES_POLL][NQ];
                bool ok;
                do {
                    ok = true;
#pragma unroll
                    for (int u = 0; u < RES_POLL; ++u)
#pragma unroll
                        for (int q = 0; q < NQ; ++q)
                            if (g0 + 64 * u + t < tm.G)
                                m[u][q].load(S + ((size_t)q * tm.wgs + tm.wg0 + g0 + 64 * u + t) * 2);
#pragma unroll
                    for (int u = 0; u < RES_POLL; ++u)
#pragma unroll
                        for (int q = 0; q < NQ; ++q)
                            if (g0 + 64 * u + t < tm.G) ok = ok && m[u][q].is(tm.tag);
                } while (!ok && left.more());
                late = late || !ok;
#pragma unroll
                for (int u = 0; u < RES_POLL; ++u)
#pragma unroll
                    for (int q = 0; q < NQ; ++q)
                        if (g0 + 64 * u + t < tm.G) got[q] += m[u][q].value();
            }
            if (late) L.quit = 1;
#pragma unroll
            for (int q = 0; q < NQ; ++q) tot[q] = wave_total(got[q]);
        }
        SolveRec rec = L.S;
        Verdict o = L.out;
        decide(tot, rec, o);
        if (t == 0) {
            L.S = rec;
            L.out = o;
        }
    }
    __syncthreads();
    return LOCAL || L.quit == 0;
}
template <int NQ, bool LOCAL, typename F>
__device__ __forceinline__ bool team_decide(Team &tm, const double (&v)[NQ], TeamLds &L, F decide) {
    return team_decide<NQ, LOCAL>(tm, v, L, decide, [] {});
}

// What a workgroup works on.
struct Share {
    int piece, n, mrow, row0; // result index, rows, matrix row offset, first own row
    size_t vbase;             // vector offset
    int m;                    // matrix of a batch
    double scale;
};
template <typename T>
__device__ __forceinline__ Share share_of(const ResArgs<T> &a, Team &tm, int rowsPerWg) {
    Share s;
    tm.wg = blockIdx.x;
    tm.wgs = a.wgs;
    if (a.P.base) {
        s.piece = a.P.wgPiece[blockIdx.x];
        tm.wg0 = a.P.wg0[s.piece];
        tm.G = a.P.G[s.piece];
        s.n = a.P.len[s.piece];
        s.vbase = a.P.base[s.piece];
        s.mrow = a.P.mrow[s.piece];
        s.m = 0;
        s.scale = 1.0 / sqrt(double(s.n));
    } else {
        const int team = blockIdx.x / a.G;
        tm.wg0 = team * a.G;
        tm.G = a.G;
        s.piece = a.team0 + team;
        s.n = a.n;
        s.vbase = (size_t)s.piece * a.n;
        s.mrow = 0;
        s.m = s.piece / a.rpm;
        s.scale = a.scale;
    }
    s.row0 = (tm.wg - tm.wg0) * rowsPerWg;
    return s;
}
template <typename T>
__device__ __forceinline__ double tol_of(const ResArgs<T> &a, int piece) {
    if (a.tolsDev) return a.tolsDev[piece];
    double t = a.tols[0];
#pragma unroll
    for (int k = 1; k < RES_TOLS; ++k)
        if (a.ntols > k && piece == k) t = a.tols[k];
    return t;
}

// The rows of a thread: row k is row0 + t + k * blockDim. Entry codes: a row of this workgroup as
// its LDS index, another row as -1 - (its row). Rows past the end and missing entries: value 0, code
// of the thread's own slot. False if a row has more than EW entries.
template <typename T, int EW, int R>
struct Rows {
    T a[R][EW];
    int c[R][EW];
    __device__ __forceinline__ bool load(const Csr<T> &A, const Share &s) {
        const int blk = blockDim.x, t = threadIdx.x;
        const size_t N = A.n;
        const T *ellv = A.ell_w > 0 ? A.ell_val + (A.valStride ? (size_t)s.m * A.ell_w * N : 0) : nullptr;
        const T *val = A.val + (size_t)s.m * A.valStride;
        bool fits = true;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int own = t + k * blk, i = s.row0 + own;
            const size_t gr = (size_t)s.mrow + i;
            const bool in = i < s.n;
            int first = 0, len = 0;
            if (in && A.ell_w == 0) {
                first = A.row[gr];
                len = A.row[gr + 1] - first;
                fits = fits && len <= EW;
            }
#pragma unroll
            for (int j = 0; j < EW; ++j) {
                int col = -1;
                T v = T(0);
                if (in) {
                    if (A.ell_w > 0) {
                        col = A.ell_col[j * N + gr];
                        v = ellv[j * N + gr];
                    } else if (j < len) {
                        col = A.col[first + j];
                        v = val[first + j];
                    }
                }
                const int local = col - s.mrow - s.row0;
                c[k][j] = col < 0 ? own : (local >= 0 && local < blk * R ? local : -1 - (col - s.mrow));
                a[k][j] = v;
            }
        }
        return fits;
    }
};

// Past the L2 cache of the workgroup's XCD, like the exchanged words: workgroups on other XCDs look at it.
template <typename T>
__device__ __forceinline__ void give_up(const ResArgs<T> &a) {
    if (threadIdx.x == 0) __hip_atomic_store(a.failed, a.done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Rows longer than the resident kernels take. They are looked for before anything is solved: pieces that
// found one in their own rows while the others solved theirs would leave x half done for the engine
// that takes over. Right-hand sides of one workgroup each look for themselves (they share the pattern, so
// all of them find it): the launch takes 4 us, the solve of 4 k rows 900.
__global__ void __launch_bounds__(256) k_row_check(const int32_t *__restrict__ row, int n, int ew, unsigned *declined,
                                                   unsigned word) {
    bool lng = false;
    for (int i = blockIdx.x * 256 + (int)threadIdx.x; i < n; i += gridDim.x * 256) lng |= row[i + 1] - row[i] > ew;
    if (lng) *declined = word;
}
int launch_row_check(const int32_t *row, int n, int ew, unsigned *declined, unsigned word, hipStream_t s) {
    hipLaunchKernelGGL(k_row_check, dim3(std::min(512, (n + 255) / 256)), dim3(256), 0, s, row, n, ew, declined, word);
    PP_LAUNCH_CHECK();
    return PP_OK;
}

// CG (with dinv its Jacobi variant), a team per right-hand side.
template <typename T, int EW, int R, bool LOCAL>
__global__ void __launch_bounds__(LOCAL ? RES_LOCAL_WG : RES_WG) k_resident_cg(ResArgs<T> a) {
    constexpr int TW = Tagged<T>::W;
    extern __shared__ __align__(16) char res_lds[];
    T *zs = reinterpret_cast<T *>(res_lds); // exchanged values of the workgroup's own rows
    __shared__ TeamLds L;
    const int t = threadIdx.x, blk = blockDim.x;
    if (*a.declined == a.done) return;
    Team tm;
    const Share sh = share_of(a, tm, blk * R);
    if (a.onlyHeld && a.recs[sh.piece].zero != ZERO_HELD) return;
    tm.slots = a.slots;
    tm.tag = a.tag;
    tm.fresh = Patience{a.spins, a.failed, a.done};
    if (t == 0) {
        L.bad = L.quit = 0;
        L.S = rec_init(tol_of(a, sh.piece), a.maxit);
        L.out = Verdict{0.0, 1, 1, 0, 0};
    }
    Rows<T, EW, R> M;
    const bool fits = M.load(a.A, sh);
    if constexpr (LOCAL)
        if (__syncthreads_or(!fits)) {
            if (t == 0) *a.declined = a.done;
            return;
        }
    const T *dv = a.dinv ? a.dinv + (size_t)sh.m * a.dinvStride + sh.row0 : nullptr;
    const int own = sh.n - sh.row0; // rows k with t + k * blk < own belong to this thread
    const size_t v0 = sh.vbase + sh.row0 + t; // vector offset of the thread's first row
    T x[R], r[R], p[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        x[k] = T(0);
        if (t + k * blk < own) a.x0[v0 + k * blk] = x[k] = a.x[v0 + k * blk];
    }
    T mean = T(0);
    __syncthreads();
    if (a.project) {
        // the mean of b
        double s[1] = {0.0};
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (t + k * blk < own) s[0] += double(a.b[v0 + k * blk]);
        if (!team_decide<1, LOCAL>(tm, s, L, [&](const double (&tot)[1], SolveRec &, Verdict &o) {
                o.step = tot[0] / double(sh.n);
            }))
            return give_up(a);
        mean = T(L.out.step);
    }
    auto rhs = [&](int k) { return a.project ? a.b[v0 + k * blk] - mean : a.b[v0 + k * blk]; };
    auto zof = [&](int k) { return dv && t + k * blk < own ? r[k] * dv[t + k * blk] : r[k]; };
    auto zpar = [&](unsigned tag) { return a.zbuf + (tag & 1 ? a.vecLen * TW : size_t(0)); };
    // own values to the team: LDS, and tagged words under the tag of the next exchange
    auto publish = [&](const T (&z)[R]) {
        const unsigned tag = tm.tag + 1;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            zs[t + k * blk] = z[k];
            if (!LOCAL && t + k * blk < own) Tagged<T>::store(zpar(tag) + (v0 - a.zorigin + k * blk) * TW, z[k], tag);
        }
    };
    // the values published under `tag` for the entries of row k (the codes pass through `hide`, so
    // that no address derived from them is kept in registers over the iterations)
    auto gather = [&](int k, unsigned tag, T (&out)[EW], Patience &left) {
        Tagged<T> g[EW];
        int c[EW];
        const word_t *Z = zpar(tag) + (sh.vbase - a.zorigin) * TW;
#pragma unroll
        for (int j = 0; j < EW; ++j) {
            c[j] = hide(M.c[k][j]);
            if (!LOCAL && c[j] < 0) g[j].load(Z + unsigned(-1 - c[j]) * TW);
        }
#pragma unroll
        for (int j = 0; j < EW; ++j) {
            if (LOCAL || c[j] >= 0) out[j] = zs[c[j]];
            else {
                while (!g[j].is(tag) && left.more()) g[j].load(Z + unsigned(-1 - c[j]) * TW);
                if (!g[j].is(tag)) L.bad = 1;
                out[j] = g[j].value();
            }
        }
    };
    // With few rows per thread the neighbours' z are fetched while the sums of the same exchange
    // travel; with more rows they would not fit the registers next to the directions.
    constexpr bool EARLY = !LOCAL && R <= 2;
    T zn[EARLY ? R : 1][EW];
    auto fetch = [&] {
        if constexpr (EARLY) {
            Patience left = tm.fresh;
#pragma unroll
            for (int k = 0; k < R; ++k) gather(k, tm.tag, zn[k], left);
        }
    };
    {
        // r = b - A x
        double s[3] = {0.0, 0.0, 0.0};
        T z[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const bool in = t + k * blk < own;
            p[k] = r[k] = T(0);
            if (in) {
                T ax = T(0);
#pragma unroll
                for (int j = 0; j < EW; ++j) {
                    const int c = M.c[k][j] >= 0 ? sh.row0 + M.c[k][j] : -1 - M.c[k][j];
                    ax += M.a[k][j] * a.x[sh.vbase + c];
                }
                const T bi = rhs(k);
                r[k] = bi - ax;
                s[0] += double(r[k]) * double(r[k]);
                s[1] += double(bi) * double(bi);
            }
            z[k] = zof(k);
            s[2] += double(r[k]) * double(z[k]);
        }
        publish(z);
        if (!team_decide<3, LOCAL>(tm, s, L, [&](const double (&tot)[3], SolveRec &S, Verdict &o) {
                rule_open(S, tot[0], sh.scale, false);
                S.zero = tot[1] == 0.0;
                if (dv) S.rho = tot[2];
                if (S.zero && a.zeroStops && rec_active(S)) {
                    S.fate = F_MET;
                    S.report = 0;
                    S.crit = 0.0;
                    S.zero = a.zeroStops;
                }
                o.active = rec_active(S);
                o.fresh = 1;
                o.half = 0; // residual replacement due
            }, fetch))
            return give_up(a);
    }
    T pn[LOCAL ? 1 : R][EW]; // the neighbours' directions, formed here from their residuals
    if constexpr (!LOCAL)
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int j = 0; j < EW; ++j) pn[k][j] = T(0);
    unsigned ztag = tm.tag;
    while (L.out.active) {
        T beta = T(L.out.step);
        bool fresh = L.out.fresh;
        if (L.out.half) {
            // residual replacement: r = b - A x, a fresh direction
            // (an all-gather of nothing under the tag of the published x, see the top of the file)
            publish(x);
            const double none[1] = {0.0};
            if (!team_decide<1, LOCAL>(tm, none, L, [](const double (&)[1], SolveRec &, Verdict &) {})) return give_up(a);
            const unsigned xtag = tm.tag;
            Patience left = tm.fresh;
            double s[2] = {0.0, 0.0};
            T z[R];
#pragma unroll
            for (int k = 0; k < R; ++k) {
                T xn[EW], ax = T(0);
                gather(k, xtag, xn, left);
#pragma unroll
                for (int j = 0; j < EW; ++j) ax += M.a[k][j] * xn[j];
                if (t + k * blk < own) r[k] = rhs(k) - ax;
                z[k] = zof(k);
                s[0] += double(r[k]) * double(r[k]);
                s[1] += double(r[k]) * double(z[k]);
            }
            __syncthreads();
            publish(z);
            if (!team_decide<2, LOCAL>(tm, s, L, [&](const double (&tot)[2], SolveRec &S, Verdict &) {
                    S.rho = dv ? tot[1] : tot[0];
                }, fetch))
                return give_up(a);
            ztag = tm.tag;
            fresh = true;
        }
        T q[R];
        double pq[1] = {0.0};
        if constexpr (LOCAL) {
            // p in LDS, then q = A p
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const T z = zof(k);
                p[k] = fresh ? z : z + beta * p[k];
                zs[t + k * blk] = p[k];
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < R; ++k) {
                T s = T(0);
#pragma unroll
                for (int j = 0; j < EW; ++j) s += M.a[k][j] * zs[hide(M.c[k][j])];
                q[k] = s;
                pq[0] += double(p[k]) * double(s);
            }
        } else {
            // p' = z + beta p at every neighbour as its z arrives, q = A p'
            Patience left = tm.fresh;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                T zk[EW], s = T(0);
                if constexpr (!EARLY) gather(k, ztag, zk, left);
#pragma unroll
                for (int j = 0; j < EW; ++j) {
                    const T z = EARLY ? zn[k][j] : zk[j];
                    pn[k][j] = fresh ? z : z + beta * pn[k][j];
                    s += M.a[k][j] * pn[k][j];
                }
                const T z = zof(k);
                p[k] = fresh ? z : z + beta * p[k];
                q[k] = s;
                pq[0] += double(p[k]) * double(s);
            }
        }
        if (!team_decide<1, LOCAL>(tm, pq, L, [&](const double (&tot)[1], SolveRec &S, Verdict &o) {
                o.step = rule_alpha(S, tot[0]);
                S.flags &= ~R_FRESH;
                o.active = rec_active(S);
                o.keep = a.xbest && (S.flags & R_KEEP);
            }))
            return give_up(a);
        if (!L.out.active) break;
        const T alpha = T(L.out.step);
        if (L.out.keep)
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (t + k * blk < own) a.xbest[v0 + k * blk] = x[k];
        double s[2] = {0.0, 0.0};
        T z[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            x[k] += alpha * p[k];
            r[k] -= alpha * q[k];
            z[k] = zof(k);
            s[0] += double(r[k]) * double(r[k]);
            if (dv) s[1] += double(r[k]) * double(z[k]);
        }
        if (!LOCAL) publish(z);
        if (!team_decide<2, LOCAL>(tm, s, L, [&](const double (&tot)[2], SolveRec &S, Verdict &o) {
                rule_step(S, tot[0], sh.scale, a.returnBest != 0);
                if (rec_active(S)) o.step = rule_cg_beta(S, dv ? tot[1] : tot[0]);
                o.active = rec_active(S);
                o.fresh = 0;
                o.half = a.resetEvery > 0 && S.iter > 0 && S.iter % a.resetEvery == 0;
            }, fetch))
            return give_up(a);
        ztag = tm.tag;
    }
    const SolveRec &S = L.S;
    const bool best = a.xbest && (S.fate == F_EXHAUSTED || S.fate == F_STALLED) && S.bestAt >= 0 && S.best < S.crit;
    const bool zero = S.zero && a.zeroStops == ZERO_SOLVED;
#pragma unroll
    for (int k = 0; k < R; ++k)
        if (t + k * blk < own) a.x[v0 + k * blk] = zero ? T(0) : (best ? a.xbest[v0 + k * blk] : x[k]);
    if (t == 0 && tm.wg == tm.wg0) {
        a.recs[sh.piece] = S;
        a.status[sh.piece] = a.done;
    }
}

template <typename T>
int launch_resident_cg(const ResArgs<T> &a, int ew, int R, int threads, bool local, hipStream_t s) {
    const dim3 grid(a.wgs), block(threads);
    const size_t lds = sizeof(T) * (size_t)threads * R;
#define PP_RES_GO(EWV, RV, LOC)                                                                     \
    if (ew == EWV && R == RV && local == LOC) {                                                     \
        hipLaunchKernelGGL((k_resident_cg<T, EWV, RV, LOC>), grid, block, lds, s, a);               \
        PP_LAUNCH_CHECK();                                                                          \
        return PP_OK;                                                                               \
    }
#define PP_RES_BOTH(RV, LOC) PP_RES_GO(5, RV, LOC) PP_RES_GO(7, RV, LOC)
    PP_RES_BOTH(1, false)
    PP_RES_BOTH(2, false)
    PP_RES_BOTH(4, false)
    PP_RES_BOTH(1, true)
    PP_RES_BOTH(2, true)
    PP_RES_BOTH(3, true)
    PP_RES_GO(5, 4, true)
#undef PP_RES_BOTH
#undef PP_RES_GO
    set_error("launch_resident_cg: no such kernel");
    return PP_ERR_ARG;
}
template int launch_resident_cg<float>(const ResArgs<float> &, int, int, int, bool, hipStream_t);
template int launch_resident_cg<double>(const ResArgs<double> &, int, int, int, bool, hipStream_t);

} // namespace pp
