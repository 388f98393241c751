// LAMMPS pair style chimesFF (etc/lmp/src/pair_chimes.cpp) on the GPU, one
// process's local and ghost atoms per call:
//   k_lmp_pair      1- and 2-body loops of PairCHIMES::compute (567-656)
//   k_lmp_lists, k_lmp_lists_short  PairCHIMES::build_mb_neighlists (321-478)
//   k_lmp_near, k_lmp_clusters      3- and 4-body loops (673-829) over those lists
//   k_lmp_out       fixed-point accumulators -> forces and tallies
// Every tally of Pair::ev_tally_mb (etc/lmp/etc/pair.cpp:1425-1482) is added
// in the exact fixed-point form of the batch pipeline, so results do not
// depend on the order of the lists or on the kernel schedule.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "chx_cluster.h"
#include "chx_dev.h"
#include "chx_lmp.h"
#include "chx_tab.h"

namespace chx {

// get_dist (pair_chimes.cpp:303-312): dr = x_b - x_a, same operation order
__device__ __forceinline__ double lmp_dist(const double *a, const double *b, double (&dr)[3])
{
    dr[0] = b[0] - a[0];
    dr[1] = b[1] - a[1];
    dr[2] = b[2] - a[2];
    return sqrt(dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
}

// ChIMES stress (xx xy xz yy yz zz) -> LAMMPS virial order (xx yy zz xy xz yz)
__device__ __forceinline__ void lmp_order(const double (&s)[6], double (&v)[6])
{
    v[0] = s[0]; v[1] = s[3]; v[2] = s[5];
    v[3] = s[1]; v[4] = s[2]; v[5] = s[4];
}

// Per-workgroup LDS table of the atoms a tile adds to, the pair style's form
// of fx_table: three force components per atom and, when the step asks for
// per-atom tallies, its energy and six virial terms, as (hi, lo) words in
// dynamic LDS.  An atom that finds no slot within LMP_PROBES goes straight to
// memory.
constexpr int LMP_PROBES = 32;
constexpr int LMP_SHORT_ROW = 64;   // candidates of an owner the one-wavefront list form holds
constexpr int LMP_BRIEF_MEAN = 80;  // mean row length up to which it goes first

struct lmp_table {
    int cap, nw;               // slots (a power of two), words per slot: 6 or 20
    int *key;
    unsigned long long *val;   // [cap][nw]: 3 forces, energy, 6 virial terms
    __host__ __device__ static size_t bytes(int cap, int nw) { return (size_t)cap * (8 * nw + 4); }
    __device__ __forceinline__ lmp_table(char *lds, int cap_, bool tally) : cap(cap_), nw(tally ? 20 : 6)
    {
        val = reinterpret_cast<unsigned long long *>(lds);
        key = reinterpret_cast<int *>(val + (size_t)cap * nw);
    }
    // all threads; a barrier must follow before use
    __device__ __forceinline__ void clear()
    {
        for (int s = threadIdx.x; s < cap; s += blockDim.x) key[s] = -1;
        for (int s = threadIdx.x; s < cap * nw; s += blockDim.x) val[s] = 0ull;
    }
    // force F and (tallying) energy share e and virial share w * v of an atom
    __device__ __forceinline__ void add(int atom, const double (&F)[3], double e, const double (&v)[6],
                                        const chx_lmp_args &A, bool &bad)
    {
        if (atom < 0) return;
        int s = (int)((((unsigned)atom * 2654435761u) >> 8) & (cap - 1));
        bool found = false;
        for (int probe = 0; probe < LMP_PROBES; probe++) {
            const int prev = atomicCAS(&key[s], -1, atom);
            if (prev == -1 || prev == atom) { found = true; break; }
            s = (s + 1) & (cap - 1);
        }
        if (!found) {
            for (int k = 0; k < 3; k++) fx_atomic(A.Facc + 2L * (3L * atom + k), F[k], bad);
            if (A.Eacc) fx_atomic(A.Eacc + 2L * atom, e, bad);
            if (A.Vacc)
                for (int k = 0; k < 6; k++) fx_atomic(A.Vacc + 2L * (6L * atom + k), v[k], bad);
            return;
        }
        unsigned long long *a = val + s * nw;
#pragma unroll
        for (int k = 0; k < 3; k++) fx_atomic(a + 2 * k, F[k], bad);
        if (A.Eacc) fx_atomic(a + 6, e, bad);
        if (A.Vacc)
#pragma unroll
            for (int k = 0; k < 6; k++) fx_atomic(a + 8 + 2 * k, v[k], bad);
    }
    // all threads, after a barrier
    __device__ __forceinline__ void flush(const chx_lmp_args &A)
    {
        for (int t = threadIdx.x; t < cap * nw; t += blockDim.x) {
            const int s = t / nw, k = t - s * nw;
            const unsigned long long w = val[t];
            if (key[s] < 0 || !w) continue;
            const long atom = key[s];
            unsigned long long *g = k < 6 ? A.Facc + 6 * atom + k
                                          : (k < 8 ? A.Eacc + 2 * atom + (k - 6) : A.Vacc + 12 * atom + (k - 8));
            atomicAdd(g, w);
        }
    }
};

// Adds the wavefront's energies and virials (lanes of on) into copy `slot` of
// the global sums: fourteen integer parts summed over the lanes at once.
__device__ __forceinline__ void lmp_global_add(const chx_lmp_args &A, bool on, double E, const double (&v)[6],
                                               int slot, bool &bad)
{
    if (!A.Gacc || __ballot(on) == 0) return;
    long long x[16];
#pragma unroll
    for (int k = 0; k < 16; k++) x[k] = 0;
    if (on) {
        if (A.eflag_global) fx_split(E, x[0], x[1], bad);
        if (A.vflag_global)
#pragma unroll
            for (int k = 0; k < 6; k++) fx_split(v[k], x[2 + 2 * k], x[3 + 2 * k], bad);
    }
    const long long t = fx_wave_sums16(x);
    const int l = threadIdx.x & 63;
    if (l < 14 && t) atomicAdd(A.Gacc + (long)slot * 16 + l, (unsigned long long)t);
}

// Sum of a double over the wavefront, in one fixed order.
__device__ __forceinline__ double lmp_wave_sum(double x)
{
    const long long r = __double_as_longlong(group_sum<16>(x));  // each row's total on its last lane
    const double s0 = __longlong_as_double(readlane_i64(r, 15)), s1 = __longlong_as_double(readlane_i64(r, 31)),
                 s2 = __longlong_as_double(readlane_i64(r, 47)), s3 = __longlong_as_double(readlane_i64(r, 63));
    return (s0 + s1) + (s2 + s3);
}

// ---------------------------------------------------------------------------
// 1- and 2-body: one wavefront per owner ilist[ii], four owners per
// workgroup.  Pairs with tag[j] > tag[i] only (pair_chimes.cpp:603).  A row
// reaches one skin past the cutoff and half of it has lower tags, so three
// quarters of its entries are skipped: the wavefront queues the entries that
// count, in row order, and evaluates 64 at a time, where lanes striding over
// the row each did a few of many passes.  The owner's force and tallies are
// summed over its lanes in double in that fixed order and added exactly once;
// the partners' go through the workgroup's table.  2744 carbon atoms, order
// 20, energy and virial: 22 us with rows of 161 entries and 13 with rows of 27,
// where sixteen striding lanes per owner and atomics to memory took 54 and 15.
// (With 112 bytes of scratch per lane, 23 and 15.)  TAB: the pair's energy and force scalar
// come from its table (compute_2B_tab, chimesFF.cpp:1782-1856: cutoff test,
// table lookups, no penalty term).
// ---------------------------------------------------------------------------
constexpr int LMP_PAIR_SLOTS = 256;

template <bool TAB>
__global__ __launch_bounds__(256) void k_lmp_pair(chx_lmp_args A, chx_model_dev M, chx_tabs_dev T)
{
    extern __shared__ __attribute__((aligned(16))) char lds[];
    __shared__ int queue[4][128];
    const bool tally = A.Eacc || A.Vacc;
    lmp_table tab(lds, LMP_PAIR_SLOTS, tally);
    tab.clear();
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    const int ii = (int)(blockIdx.x * 4 + wv);
    bool bad = false, tab_err = false;
    if (ii < A.inum) {
        const int i = A.ilist[ii];
        const int itag = A.tag[i], ti = A.ctype[i];
        const double xi[3] = {A.x[3L * i], A.x[3L * i + 1], A.x[3L * i + 2]};
        // owner force, energy and virial of the pairs (halves go to each atom)
        double acc[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        int flags = 0, nq = 0;
        // the first cnt queued partners, one per lane
        auto batch = [&](int cnt) {
            double E = 0.0, v[6] = {0, 0, 0, 0, 0, 0};
            if (lane < cnt) {
                const int j = queue[wv][lane];
                const double xj[3] = {A.x[3L * j], A.x[3L * j + 1], A.x[3L * j + 2]};
                double dr[3], fs;
                const double r = lmp_dist(xi, xj, dr);
                const int pt = M.pairmap[ti * M.nt + A.ctype[j]];
                if constexpr (TAB) tab2_lookup(T, pt, r, E, fs, tab_err);
                else
                    eval_pair(r, M.slots2[pt], M.c2 + (long)pt * (M.order[0] + 1), M.order[0], M.tersoff, M.fcut_var,
                              M.pen_dist, M.pen_scale, E, fs, flags);
                const double F[3] = {fs * dr[0], fs * dr[1], fs * dr[2]};
                const double s[6] = {-(fs * (dr[0] * dr[0])), -(fs * (dr[0] * dr[1])), -(fs * (dr[0] * dr[2])),
                                     -(fs * (dr[1] * dr[1])), -(fs * (dr[1] * dr[2])), -(fs * (dr[2] * dr[2]))};
                lmp_order(s, v);
                const double Fj[3] = {-F[0], -F[1], -F[2]};
                const double vj[6] = {v[0] / 2, v[1] / 2, v[2] / 2, v[3] / 2, v[4] / 2, v[5] / 2};
                tab.add(j, Fj, E / 2, vj, A, bad);
#pragma unroll
                for (int k = 0; k < 3; k++) acc[k] += F[k];
                acc[3] += E;
#pragma unroll
                for (int k = 0; k < 6; k++) acc[4 + k] += v[k];
            }
        };
        const int beg = A.nbr_off[ii], end = A.nbr_off[ii + 1];
        for (int q0 = beg; q0 < end; q0 += 64) {
            bool in = false;
            int j = 0;
            if (q0 + lane < end) {
                j = A.nbr[q0 + lane];
                if (A.tag[j] > itag) {
                    const double xj[3] = {A.x[3L * j], A.x[3L * j + 1], A.x[3L * j + 2]};
                    double dr[3];
                    in = !(lmp_dist(xi, xj, dr) >= M.slots2[M.pairmap[ti * M.nt + A.ctype[j]]].rout);
                }
            }
            const unsigned long long b = __ballot(in);
            if (in) queue[wv][nq + __popcll(b & below)] = j;
            nq += __popcll(b);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (nq >= 64) {
                batch(64);
                nq -= 64;
                const int rest = lane < nq ? queue[wv][64 + lane] : 0;
                __builtin_amdgcn_wave_barrier();
                if (lane < nq) queue[wv][lane] = rest;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        }
        if (nq) batch(nq);
        double tot[10];
#pragma unroll
        for (int k = 0; k < 10; k++) tot[k] = lmp_wave_sum(acc[k]);
        const double e1 = M.eoff[ti];  // compute_1B, tallied for one atom
        const double v[6] = {tot[4], tot[5], tot[6], tot[7], tot[8], tot[9]};
        if (lane == 0) {
            for (int k = 0; k < 3; k++) fx_atomic(A.Facc + 2L * (3L * i + k), tot[k], bad);
            if (A.Eacc) {
                fx_atomic(A.Eacc + 2L * i, e1, bad);
                fx_atomic(A.Eacc + 2L * i, tot[3] / 2, bad);
            }
            if (A.Vacc)
                for (int k = 0; k < 6; k++) fx_atomic(A.Vacc + 2L * (6L * i + k), v[k] / 2, bad);
        }
        // lane 0 the pairs' energy and virial, lane 1 the 1-body energy
        const double ev = lane ? e1 : tot[3];
        double gv[6];
#pragma unroll
        for (int k = 0; k < 6; k++) gv[k] = lane ? 0.0 : v[k];  // an array of zeros here would put both in scratch
        lmp_global_add(A, lane < 2, ev, gv, blockIdx.x & (CHX_LMP_GSLOTS - 1), bad);
    }
    __syncthreads();
    tab.flush(A);
    if (bad) atomicOr(&A.status[CHX_LMP_ST_FLAGS], CHX_LMP_BAD_RANGE);
    if (tab_err) atomicOr(&A.status[CHX_LMP_ST_FLAGS], CHX_LMP_BAD_TAB2);
}

// ---------------------------------------------------------------------------
// Many-body lists, four wavefronts per owner ilist[ii].  The owner's row is
// filtered to J = {j : j != i, tag[j] >= tag[i], d_ij below either padded
// cutoff}, kept in row order in LDS; every k and l of the reference's loops
// lies in J.  For each a of J a bit row holds the b of J that may follow it
// (another atom, tag[b] >= tag[a], every distance of (i, a, b) below the
// padded cutoff).  The triplets are then the set bits of the 3-body rows in
// row-major order, and the l of a pair (a, b) are the common bits of the
// 4-body rows of a and b: tag[l] >= tag[b] >= tag[a], both distances and both
// atoms checked once per pair instead of once per quadruplet, and counting is
// a population count.  Positions come from the rows' counts, so the lists are
// written in the reference's loop order.
//
// MODE 0 counts per owner, MODE 1 writes at the scanned offsets.  CAP bounds
// |J|: the small form (32 KB of LDS, four owners a CU) takes owners with at
// most CAP, the large one those above `lo`; it is launched only when a row is
// long enough, and neither where the one-wavefront form below took every
// owner.  1728 atoms at 3.2 g/cc, pads 5.5 / 4.625 A: 67 us
// to count and 147 us to write, where one wavefront per owner testing every l
// of every pair took 1286 and 1465 us; the writes are now 53 MB in runs of a
// few entries per lane.
// ---------------------------------------------------------------------------
template <int CAP, int MODE>
__global__ __launch_bounds__(256) void k_lmp_lists(chx_lmp_args A, int lo, double pad3, double pad4, int has4,
                                                   int *cnt3, int *cnt4, const long long *off3,
                                                   const long long *off4, int *trips, int *quads)
{
    constexpr int W = CAP / 64, LD = W + 1;  // odd row stride: lanes' rows lie in different banks
    __shared__ double cx[CAP][3], cd[CAP];
    __shared__ int cj[CAP], ctag[CAP];
    __shared__ unsigned long long r3[CAP][LD], r4[CAP][LD];
    __shared__ int row3[CAP], row4[CAP], wsum[4];
    const int ii = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    const int i = A.ilist[ii], itag = A.tag[i];
    const double xi[3] = {A.x[3L * i], A.x[3L * i + 1], A.x[3L * i + 2]};
    const int beg = A.nbr_off[ii], n = A.nbr_off[ii + 1] - beg;
    int m = 0;
    for (int b0 = 0; b0 < n; b0 += 256) {
        bool v = false;
        int j = 0, tj = 0;
        double xj[3] = {0, 0, 0}, d = 0.0;
        if (b0 + tid < n) {
            j = A.nbr[beg + b0 + tid];
            tj = A.tag[j];
            if (j != i && tj >= itag) {
                xj[0] = A.x[3L * j]; xj[1] = A.x[3L * j + 1]; xj[2] = A.x[3L * j + 2];
                double dr[3];
                d = lmp_dist(xi, xj, dr);
                v = !(d >= pad3 && d >= pad4);
            }
        }
        const unsigned long long bal = __ballot(v);
        if (lane == 0) wsum[wv] = __popcll(bal);
        __syncthreads();
        int r = m + __popcll(bal & below);
#pragma unroll
        for (int w = 0; w < 4; w++) {
            r += w < wv ? wsum[w] : 0;
            m += wsum[w];
        }
        if (v && r < CAP) {
            cj[r] = j;
            ctag[r] = tj;
            cx[r][0] = xj[0]; cx[r][1] = xj[1]; cx[r][2] = xj[2];
            cd[r] = d;
        }
        __syncthreads();
    }
    if (m <= lo) return;
    if (m > CAP) {
        if (CAP == CHX_LMP_CAND && tid == 0) {
            atomicOr(&A.status[CHX_LMP_ST_FLAGS], CHX_LMP_BAD_CAND);
            atomicMax(&A.status[CHX_LMP_ST_MAXCAND], m);
        }
        return;
    }
    const int mw = (m + 63) >> 6;
    for (int a = wv; a < m; a += 4) {
        const double da = cd[a];
        for (int w = 0; w < mw; w++) {
            const int b = w * 64 + lane;
            bool v3 = false, v4 = false;
            if (b < m && cj[a] != cj[b] && ctag[b] >= ctag[a]) {
                double dr[3];
                const double dab = lmp_dist(cx[a], cx[b], dr);
                const double db = cd[b];
                v3 = da < pad3 && db < pad3 && dab < pad3;
                v4 = has4 && da < pad4 && db < pad4 && dab < pad4;
            }
            const unsigned long long b3 = __ballot(v3), b4 = __ballot(v4);
            if (lane == 0) {
                r3[a][w] = b3;
                r4[a][w] = b4;
            }
        }
    }
    __syncthreads();
    // quadruplets of the pair (a, b): the common followers of a and b
    auto common = [&](int a, int b) {
        int c = 0;
        for (int w = 0; w < mw; w++) c += __popcll(r4[a][w] & r4[b][w]);
        return c;
    };
    // clusters of each row
    for (int a = wv; a < m; a += 4) {
        int c3 = 0, c4 = 0;
        for (int w = 0; w < mw; w++) {
            c3 += __popcll(r3[a][w]);
            const unsigned long long b4 = r4[a][w];
            if (b4 == 0) continue;
            if ((b4 >> lane) & 1) c4 += common(a, w * 64 + lane);
        }
        for (int s = 1; s < 64; s <<= 1) c4 += __shfl_xor(c4, s, 64);
        if (lane == 0) {
            row3[a] = c3;
            row4[a] = c4;
        }
    }
    __syncthreads();
    // rows' offsets (exclusive) and totals, by the first wavefront
    if (wv == 0) {
        int t3 = 0, t4 = 0;
        for (int w = 0; w < mw; w++) {
            const int a = w * 64 + lane;
            const int c3 = a < m ? row3[a] : 0, c4 = a < m ? row4[a] : 0;
            int s3 = c3, s4 = c4;
            for (int s = 1; s < 64; s <<= 1) {
                const int u3 = __shfl_up(s3, s, 64), u4 = __shfl_up(s4, s, 64);
                if (lane >= s) {
                    s3 += u3;
                    s4 += u4;
                }
            }
            if (a < m) {
                row3[a] = t3 + s3 - c3;
                row4[a] = t4 + s4 - c4;
            }
            t3 += __shfl(s3, 63, 64);
            t4 += __shfl(s4, 63, 64);
        }
        if (MODE == 0 && lane == 0) {
            cnt3[ii] = t3;
            cnt4[ii] = t4;
        }
    }
    if (MODE == 0) return;
    __syncthreads();
    const long long o3 = off3[ii], o4 = off4[ii];
    for (int a = wv; a < m; a += 4) {
        const int ja = cj[a];
        int p3 = row3[a], p4 = row4[a];
        for (int w = 0; w < mw; w++) {
            const int b = w * 64 + lane;
            const unsigned long long b3 = r3[a][w], b4 = r4[a][w];
            if ((b3 >> lane) & 1) {
                int *t = trips + 3 * (o3 + p3 + __popcll(b3 & below));
                t[0] = i; t[1] = ja; t[2] = cj[b];
            }
            p3 += __popcll(b3);
            if (b4 == 0) continue;
            const bool on = (b4 >> lane) & 1;
            const int c = on ? common(a, b) : 0;
            int s4 = c;
            for (int s = 1; s < 64; s <<= 1) {
                const int u4 = __shfl_up(s4, s, 64);
                if (lane >= s) s4 += u4;
            }
            // each lane writes its pair's quadruplets, one consecutive run
            if (c) {
                int4 *u = reinterpret_cast<int4 *>(quads) + (o4 + p4 + s4 - c);
                const int jb = cj[b];
                for (int y = 0; y < mw; y++) {
                    unsigned long long l = r4[a][y] & r4[b][y];
                    while (l) {
                        *u++ = make_int4(i, ja, jb, cj[y * 64 + __ffsll((long long)l) - 1]);
                        l &= l - 1;
                    }
                }
            }
            p4 += __shfl(s4, 63, 64);
        }
    }
}

// The same lists for owners with at most 64 candidates, one wavefront per
// owner.  The row-wise form above gives a wavefront one row of at most m pairs
// at a time, a few lanes' worth where rows are short; here the m^2 pairs of
// (a, b) are taken 64 at a time in list order, the 3-body entries come straight
// from the ballots, and only the 4-body bits are kept as rows.  Bound by its
// dependent loads and LDS reads.  Both passes, 8000 carbon atoms at 0.5 g/cc:
// 25 us against 98 us with the row-wise form (20 and 94 without 4-body terms).
template <int MODE>
__global__ __launch_bounds__(64) void k_lmp_lists_short(chx_lmp_args A, double pad3, double pad4, int has4,
                                                        int *cnt3, int *cnt4, const long long *off3,
                                                        const long long *off4, int *trips, int *quads)
{
    constexpr int CAP = LMP_SHORT_ROW;
    static_assert(CAP == 64, "a 4-body row is one word");
    __shared__ double cx[CAP][3], cd[CAP];
    __shared__ int cj[CAP], ctag[CAP];
    __shared__ unsigned long long r4[CAP];
    const int ii = blockIdx.x, lane = threadIdx.x;
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
    const int i = A.ilist[ii], itag = A.tag[i];
    const double xi[3] = {A.x[3L * i], A.x[3L * i + 1], A.x[3L * i + 2]};
    const int beg = A.nbr_off[ii], n = A.nbr_off[ii + 1] - beg;
    r4[lane] = 0ull;
    int m = 0;
    for (int b0 = 0; b0 < n; b0 += 64) {
        bool v = false;
        int j = 0, tj = 0;
        double xj[3] = {0, 0, 0}, d = 0.0;
        if (b0 + lane < n) {
            j = A.nbr[beg + b0 + lane];
            tj = A.tag[j];
            if (j != i && tj >= itag) {
                xj[0] = A.x[3L * j]; xj[1] = A.x[3L * j + 1]; xj[2] = A.x[3L * j + 2];
                double dr[3];
                d = lmp_dist(xi, xj, dr);
                v = !(d >= pad3 && d >= pad4);
            }
        }
        const unsigned long long bal = __ballot(v);
        const int r = m + __popcll(bal & below);
        if (v && r < CAP) {
            cj[r] = j;
            ctag[r] = tj;
            cx[r][0] = xj[0]; cx[r][1] = xj[1]; cx[r][2] = xj[2];
            cd[r] = d;
        }
        m += __popcll(bal);
    }
    if (m > CAP) return;  // the row-wise form takes it
    __syncthreads();
    const int total = m * m;
    const float rm = 1.0f / (float)m;  // (p + 1/2) rm is at least 1/128 from a whole number, p < 4096: its floor is p / m
    long long o3 = MODE ? off3[ii] : 0, o4 = MODE ? off4[ii] : 0;
    int c3 = 0;
    for (int p0 = 0; p0 < total; p0 += 64) {
        const int p = p0 + lane;
        bool v3 = false, v4 = false;
        int a = 0, b = 0;
        if (p < total) {
            a = (int)(((float)p + 0.5f) * rm);
            b = p - a * m;
            if (cj[a] != cj[b] && ctag[b] >= ctag[a]) {
                double dr[3];
                const double dab = lmp_dist(cx[a], cx[b], dr), da = cd[a], db = cd[b];
                v3 = da < pad3 && db < pad3 && dab < pad3;
                v4 = has4 && da < pad4 && db < pad4 && dab < pad4;
            }
        }
        const unsigned long long b3 = __ballot(v3);
        if (MODE && v3) {
            int *t = trips + 3 * (o3 + c3 + __popcll(b3 & below));
            t[0] = i; t[1] = cj[a]; t[2] = cj[b];
        }
        c3 += __popcll(b3);
        if (v4) atomicOr(&r4[a], 1ull << b);
    }
    __syncthreads();
    int c4 = 0;
    if (has4) {
        for (int p0 = 0; p0 < total; p0 += 64) {
            const int p = p0 + lane;
            unsigned long long l = 0ull;
            int a = 0, b = 0;
            if (p < total) {
                a = (int)(((float)p + 0.5f) * rm);
                b = p - a * m;
                if ((r4[a] >> b) & 1) l = r4[a] & r4[b];
            }
            if (__ballot(l != 0ull) == 0) continue;
            const int c = __popcll(l);
            int s4 = c;
            for (int s = 1; s < 64; s <<= 1) {
                const int u4 = __shfl_up(s4, s, 64);
                if (lane >= s) s4 += u4;
            }
            if (MODE && c) {
                int4 *u = reinterpret_cast<int4 *>(quads) + (o4 + c4 + s4 - c);
                const int ja = cj[a], jb = cj[b];
                while (l) {
                    *u++ = make_int4(i, ja, jb, cj[__ffsll((long long)l) - 1]);
                    l &= l - 1;
                }
            }
            c4 += __shfl(s4, 63, 64);
        }
    }
    if (MODE == 0 && lane == 0) {
        cnt3[ii] = c3;
        cnt4[ii] = c4;
    }
}

// ---------------------------------------------------------------------------
// 3- and 4-body: one thread per listed cluster.  Pair distances and vectors
// as the reference forms them (ij, ik, jk / ij, ik, il, jk, jl, kl; x_b - x_a),
// the terms of compute_3B / compute_4B, then the forces of every member and
// the tallies of ev_tally_mb (energy and virial shared equally by the
// members; the global part in CHX_LMP_GSLOTS copies).
// ---------------------------------------------------------------------------
// compute_3B_tab (chimesFF.cpp:2183-2313): exclusion and the cutoffs of the
// mapped slots as compute_3B, then the table at the runtime pair distances
// (ij, ik, jk; get_tab_3B's sort is not executed, 2459-2470); forces and
// stress of ij, ik, jk with the distance-tensor products, in that order.
__device__ __forceinline__ void tab3_cluster(const chx_model_dev &M, const chx_tabs_dev &T, const int (&ty)[3],
                                             const double (&dist)[3], const double (&dr)[3][3], double &E,
                                             double (&fo)[3][3], double (&S)[6], bool &evaluated, bool &err)
{
    E = 0.0;
    for (int a = 0; a < 3; a++) fo[a][0] = fo[a][1] = fo[a][2] = 0.0;
    for (int k = 0; k < 6; k++) S[k] = 0.0;
    evaluated = false;
    const int tau = M.tripmap[(ty[0] * M.nt + ty[1]) * M.nt + ty[2]];
    if (tau < 0 || !cluster_inside<3>(M, ty, dist)) return;
    if (tau >= T.ntab3) {
        err = true;
        return;
    }
    double v[4];
    tab3_lookup(T, tau, dist[0], dist[1], dist[2], v, err);
    evaluated = true;
    E = v[0];
    const int ma[3] = {0, 0, 1}, mb[3] = {1, 2, 2};
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const double f = v[1 + q];
        const double *d = dr[q];
        for (int k = 0; k < 3; k++) {
            fo[ma[q]][k] += f * d[k];
            fo[mb[q]][k] -= f * d[k];
        }
        S[0] -= f * (d[0] * d[0]);
        S[1] -= f * (d[0] * d[1]);
        S[2] -= f * (d[0] * d[2]);
        S[3] -= f * (d[1] * d[1]);
        S[4] -= f * (d[1] * d[2]);
        S[5] -= f * (d[2] * d[2]);
    }
}

// ---------------------------------------------------------------------------
// The listed clusters that may be evaluated this step: every pair distance
// within the largest cutoff of the body order.  The lists reach one skin
// further, so most of their entries are outside (97% of the quadruplets and
// 85% of the triplets of a 3.2 g/cc carbon box at 3.125 / 4 A with a 1.5 A
// skin); evaluated one entry per lane, nearly every wavefront paid for the
// whole polynomial with a few lanes active.  The test is on squared lengths
// with a relative margin of 2^-40 on the limit (lim2), far above the rounding
// of either form, so every cluster the exact test of the evaluation accepts
// is kept.  Each workgroup takes NEAR_SPAN consecutive entries and appends its
// survivors' list indices as one run, so neighbouring clusters stay together
// for the force table; every sum is exact, so their order decides nothing.
// Bound by the gathers of the members' positions (L2).
// ---------------------------------------------------------------------------
constexpr int NEAR_SPAN = 2048;
constexpr int LMP_TILE_SLOTS = 256;

template <int NB>
__global__ __launch_bounds__(256) void k_lmp_near(long n, const int *__restrict__ list,
                                                  const double *__restrict__ x, double lim2, int *near, int *count)
{
    constexpr int PER = NEAR_SPAN / 256;
    __shared__ int wtot[PER][4];
    __shared__ int base_s;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const long b0 = (long)blockIdx.x * NEAR_SPAN;
    unsigned long long bal[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
        const long c = b0 + u * 256 + threadIdx.x;
        bool in = false;
        if (c < n) {
            int m[NB];
            if constexpr (NB == 4) {
                const int4 q = reinterpret_cast<const int4 *>(list)[c];
                m[0] = q.x; m[1] = q.y; m[2] = q.z; m[3] = q.w;
            } else {
#pragma unroll
                for (int a = 0; a < NB; a++) m[a] = list[c * NB + a];
            }
            double p[NB][3];
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int k = 0; k < 3; k++) p[a][k] = x[3L * m[a] + k];
            in = true;
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int b = a + 1; b < NB; b++) {
                    const double d0 = p[b][0] - p[a][0], d1 = p[b][1] - p[a][1], d2 = p[b][2] - p[a][2];
                    in = in && d0 * d0 + d1 * d1 + d2 * d2 < lim2;
                }
        }
        bal[u] = __ballot(in);
        if (lane == 0) wtot[u][wv] = __popcll(bal[u]);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
#pragma unroll
        for (int u = 0; u < PER; u++)
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const int v = wtot[u][w];
                wtot[u][w] = t;
                t += v;
            }
        base_s = t ? atomicAdd(count, t) : 0;
    }
    __syncthreads();
    const unsigned long long below = lane ? (~0ull >> (64 - lane)) : 0ull;
#pragma unroll
    for (int u = 0; u < PER; u++)
        if ((bal[u] >> lane) & 1)
            near[base_s + wtot[u][wv] + __popcll(bal[u] & below)] = (int)(b0 + u * 256 + threadIdx.x);
}

// One thread per cluster of near[0 .. *count) (k_lmp_near); a fixed grid walks
// them 128 at a time, since the host does not know their number.  4096 carbon
// atoms at 3.2 g/cc, orders 5 / 3: one entry per lane over the whole lists took
// 269 us (triplets) and 890 us (quadruplets), and a step of the pair style
// 1426 us; selection and evaluation together leave a step of 504 us.  With the
// per-atom tallies through the table too, 1728 atoms take 66 and 57 us (337 and
// 172 us with those in atomics to memory).
template <int NB, int D, bool TAB>
__global__ __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(2))) void k_lmp_clusters(const int *__restrict__ count, const int *__restrict__ near, const int *__restrict__ list, chx_lmp_args A,
                                                      chx_model_dev M, chx_tabs_dev T)
{
    // forces and per-atom tallies of the workgroup's clusters, merged per atom
    // (a tile of consecutive clusters touches one or two hundred atoms)
    extern __shared__ __attribute__((aligned(16))) char lds[];
    lmp_table tab(lds, LMP_TILE_SLOTS, A.Eacc || A.Vacc);
    const int nc = *count;
    bool bad = false;
    for (int c0 = blockIdx.x * 128; c0 < nc; c0 += gridDim.x * 128) {
        tab.clear();
        __syncthreads();
        const bool valid = c0 + (int)threadIdx.x < nc;
        const long c = valid ? near[c0 + threadIdx.x] : 0;
        constexpr int P = NB * (NB - 1) / 2;
        int mem[NB], ty[NB];
        double xm[NB][3];
#pragma unroll
        for (int a = 0; a < NB; a++) {
            mem[a] = valid ? list[c * NB + a] : 0;
            ty[a] = A.ctype[mem[a]];
            for (int k = 0; k < 3; k++) xm[a][k] = A.x[3L * mem[a] + k];
        }
        double dist[P], dr[P][3];
        {
            int q = 0;
#pragma unroll
            for (int a = 0; a < NB; a++)
#pragma unroll
                for (int b = a + 1; b < NB; b++, q++) dist[q] = lmp_dist(xm[a], xm[b], dr[q]);
        }
        double Ec = 0.0, fo[NB][3], So[6];
        int flags = 0;
        bool evaluated = false, tab_err = false;
        if constexpr (TAB) {
            if (valid) tab3_cluster(M, T, ty, dist, dr, Ec, fo, So, evaluated, tab_err);
        } else {
            if (valid) explicit_cluster<NB, D>(M, ty, dist, dr, Ec, fo, So, flags, evaluated, nullptr);
        }
        if (tab_err) atomicOr(&A.status[CHX_LMP_ST_FLAGS], CHX_LMP_BAD_TAB3);
        double v[6];
        lmp_order(So, v);
        // every member's force and share of the tallies (ev_tally_mb), the
        // owner's included, through the LDS table
        const double e = Ec / NB, vs[6] = {v[0] / NB, v[1] / NB, v[2] / NB, v[3] / NB, v[4] / NB, v[5] / NB};
#pragma unroll
        for (int a = 0; a < NB; a++) tab.add(evaluated ? mem[a] : -1, fo[a], e, vs, A, bad);
        lmp_global_add(A, evaluated, Ec, v, blockIdx.x & (CHX_LMP_GSLOTS - 1), bad);
        __syncthreads();
        tab.flush(A);
        __syncthreads();
    }
    if (bad) atomicOr(&A.status[CHX_LMP_ST_FLAGS], CHX_LMP_BAD_RANGE);
}

// ---------------------------------------------------------------------------
// Accumulators -> doubles: one thread per atom; block 0 first sums the
// CHX_LMP_GSLOTS copies of the global energy and virial, one per thread
// (integer sums, exact).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_lmp_out(chx_lmp_args A, double *F, double *eatom, double *vatom,
                                                 double *glob)
{
    static_assert(CHX_LMP_GSLOTS == 256, "one copy per thread");
    if (A.Gacc && blockIdx.x == 0) {
        __shared__ long long part[4][16];
        long long x[16];
        const unsigned long long *g = A.Gacc + 16L * threadIdx.x;
#pragma unroll
        for (int k = 0; k < 7; k++) {
            fx_sum t;
            t.add(g + 2 * k);
            x[2 * k] = t.hi;
            x[2 * k + 1] = t.lo;
        }
        x[14] = x[15] = 0;
        const long long t = fx_wave_sums16(x);
        const int l = threadIdx.x & 63;
        if (l < 16) part[threadIdx.x >> 6][l] = t;
        __syncthreads();
        if (threadIdx.x < 7) {
            fx_sum r;
            for (int w = 0; w < 4; w++) {
                r.hi += part[w][2 * threadIdx.x];
                r.lo += part[w][2 * threadIdx.x + 1];
            }
            glob[threadIdx.x] = r.value();
        }
    }
    const long a = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= A.nall) return;
    for (int k = 0; k < 3; k++) {
        fx_sum t;
        t.add(A.Facc + 2 * (3 * a + k));
        F[3 * a + k] = t.value();
    }
    if (A.Eacc) {
        fx_sum t;
        t.add(A.Eacc + 2 * a);
        eatom[a] = t.value();
    }
    if (A.Vacc)
        for (int k = 0; k < 6; k++) {
            fx_sum t;
            t.add(A.Vacc + 2 * (6 * a + k));
            vatom[6 * a + k] = t.value();
        }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
// ---------------------------------------------------------------------------
// Cluster rows of the FINGERPRINT build (pair_chimes.cpp:526-535, 625-640,
// 703-714, 777-790, recorded by chimesFF.cpp:1694-1703, 2013-2022,
// 2603-2613): a cluster of the pair style's loops is recorded when its
// members are in order (2-body: i < j by atom index, on pairs with tag[j] >
// tag[i]; 3-body: tag[i] < tag[j], tag[i] < tag[k], tag[j] < tag[k]; 4-body:
// tag[i] < tag[j] < tag[k] < tag[l]) and compute_nB evaluates it (type not
// excluded, every pair below its slot's outer cutoff).  Row: the pair
// distances in runtime order (get_dist's arithmetic), then the member types
// as doubles.  One thread per loop entry (2-body: per packed neighbour-row
// entry), 256 entries per block: MODE 0 counts each block's rows, MODE 1
// writes them from the block's offset in entry order, so rows come in the
// loops' order.
// ---------------------------------------------------------------------------
template <int NB, int MODE>
__global__ __launch_bounds__(256) void k_lmp_fp_rows(long n, const int *__restrict__ list, chx_lmp_args A,
                                                     chx_model_dev M, int *blk_cnt, const long long *blk_off,
                                                     double *rows)
{
    constexpr int P = NB * (NB - 1) / 2;
    constexpr int pa[6] = {0, 0, 0, 1, 1, 2}, pb[6] = {1, 2, 3, 2, 3, 3};
    constexpr int pa3[3] = {0, 0, 1}, pb3[3] = {1, 2, 2};
    __shared__ int wsum[4];
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    bool keep = false;
    int ty[NB];
    double dist[P];
    if (e < n) {
        int m[NB];
        if constexpr (NB == 2) {
            int lo = 0, hi = A.inum - 1;  // owner: the last row starting at or before e
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (A.nbr_off[mid] <= e) lo = mid; else hi = mid - 1;
            }
            m[0] = A.ilist[lo];
            m[1] = A.nbr[e];
            keep = A.tag[m[1]] > A.tag[m[0]] && m[0] < m[1];
        } else {
#pragma unroll
            for (int a = 0; a < NB; a++) m[a] = list[e * NB + a];
            const int *t = A.tag;
            if constexpr (NB == 3) keep = t[m[0]] < t[m[1]] && t[m[0]] < t[m[2]] && t[m[1]] < t[m[2]];
            else keep = t[m[0]] < t[m[1]] && t[m[1]] < t[m[2]] && t[m[2]] < t[m[3]];
        }
        if (keep) {
#pragma unroll
            for (int a = 0; a < NB; a++) ty[a] = A.ctype[m[a]];
#pragma unroll
            for (int q = 0; q < P; q++) {
                const int a = NB == 3 ? pa3[q] : pa[q], b = NB == 3 ? pb3[q] : pb[q];
                double dr[3];
                dist[q] = lmp_dist(A.x + 3L * m[a], A.x + 3L * m[b], dr);
            }
            keep = cluster_inside<NB>(M, ty, dist);
        }
    }
    const unsigned long long bal = __ballot(keep);
    const int before = __popcll(bal & (lane ? (~0ull >> (64 - lane)) : 0ull));
    if (lane == 0) wsum[wv] = __popcll(bal);
    __syncthreads();
    int base = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 4; w++) {
        base += w < wv ? wsum[w] : 0;
        total += wsum[w];
    }
    if (MODE == 0) {
        if (threadIdx.x == 0) blk_cnt[blockIdx.x] = total;
        return;
    }
    if (!keep) return;
    double *row = rows + (blk_off[blockIdx.x] + base + before) * (P + NB);
#pragma unroll
    for (int q = 0; q < P; q++) row[q] = dist[q];
#pragma unroll
    for (int a = 0; a < NB; a++) row[P + a] = (double)ty[a];
}

void launch_lmp_fp_rows(int nb, int mode, long n, const int *list, const chx_lmp_args &A, const chx_model_dev &M,
                        int *blk_cnt, const long long *blk_off, double *rows, hipStream_t st)
{
    if (n <= 0) return;
    const dim3 grid((unsigned)((n + 255) / 256)), block(256);
#define L(NB_, MODE_) \
    hipLaunchKernelGGL((k_lmp_fp_rows<NB_, MODE_>), grid, block, 0, st, n, list, A, M, blk_cnt, blk_off, rows)
    if (nb == 2) { if (mode) L(2, 1); else L(2, 0); }
    else if (nb == 3) { if (mode) L(3, 1); else L(3, 0); }
    else { if (mode) L(4, 1); else L(4, 0); }
#undef L
}

void launch_lmp_pair(const chx_lmp_args &A, const chx_model_dev &M, const chx_tabs_dev *T, hipStream_t st)
{
    if (A.inum <= 0) return;
    const dim3 grid((unsigned)((A.inum + 3) / 4)), block(256);
    const size_t lds = lmp_table::bytes(LMP_PAIR_SLOTS, A.Eacc || A.Vacc ? 20 : 6);
    if (T && T->ntab2) hipLaunchKernelGGL(k_lmp_pair<true>, grid, block, lds, st, A, M, *T);
    else hipLaunchKernelGGL(k_lmp_pair<false>, grid, block, lds, st, A, M, chx_tabs_dev{});
}

void launch_lmp_lists(int mode, const chx_lmp_args &A, int max_row, long entries, double pad3, double pad4, int has4,
                      int *cnt3, int *cnt4, const long long *off3, const long long *off4, int *trips, int *quads,
                      hipStream_t st)
{
    if (A.inum <= 0) return;
    constexpr int SMALL = CHX_LMP_CAND / 2;
    const dim3 grid((unsigned)A.inum), block(256);
    // Rows of up to 80 entries on average hold 64 candidates or fewer for
    // nearly every owner.  2744 atoms, both passes, row-wise form alone against
    // one wavefront per owner first: rows of 27 entries 43 against 18 us, 53:
    // 60 and 36, 77: 71 and 64, 85: 102 and 128 (without 4-body terms 41 and
    // 14, 53 and 21, 60 and 41, 87 and 76, but rows of 110 134 and 154).
    const bool brief = entries <= (long)LMP_BRIEF_MEAN * A.inum;
    const int lo = brief ? LMP_SHORT_ROW : -1;
#define SHORT(MODE_)                                                                                           \
    hipLaunchKernelGGL(k_lmp_lists_short<MODE_>, grid, dim3(64), 0, st, A, pad3, pad4, has4, cnt3, cnt4, off3, off4, \
                       trips, quads)
#define L(CAP_, MODE_, LO_)                                                                                    \
    hipLaunchKernelGGL((k_lmp_lists<CAP_, MODE_>), grid, block, 0, st, A, LO_, pad3, pad4, has4, cnt3, cnt4, off3, \
                       off4, trips, quads)
    if (mode == 0) {
        if (brief) SHORT(0);
        if (max_row > lo) L(SMALL, 0, lo);
        if (max_row > SMALL) L(CHX_LMP_CAND, 0, SMALL);
    } else {
        if (brief) SHORT(1);
        if (max_row > lo) L(SMALL, 1, lo);
        if (max_row > SMALL) L(CHX_LMP_CAND, 1, SMALL);
    }
#undef SHORT
#undef L
}

void launch_lmp_clusters(int nb, int D, long n, const int *list, double rc, int *near, int *count,
                         const chx_lmp_args &A, const chx_model_dev &M, const chx_tabs_dev *T, hipStream_t st)
{
    if (n <= 0) return;
    const double lim2 = rc * rc * (1.0 + 0x1p-40);
    const dim3 ngrid((unsigned)((n + NEAR_SPAN - 1) / NEAR_SPAN));
    if (nb == 3) hipLaunchKernelGGL(k_lmp_near<3>, ngrid, dim3(256), 0, st, n, list, A.x, lim2, near, count);
    else hipLaunchKernelGGL(k_lmp_near<4>, ngrid, dim3(256), 0, st, n, list, A.x, lim2, near, count);
    // two workgroups for each of the 1024 the device holds at once (two
    // wavefronts on each of a CU's SIMDs), fewer for short lists
    const dim3 grid((unsigned)std::min<long>((n + 127) / 128, 2048)), block(128);
    const size_t lds = lmp_table::bytes(LMP_TILE_SLOTS, A.Eacc || A.Vacc ? 20 : 6);
    if (nb == 3 && T && T->ntab3) {
        hipLaunchKernelGGL((k_lmp_clusters<3, 0, true>), grid, block, lds, st, count, near, list, A, M, *T);
        return;
    }
#define X(d)                                                                                                  \
    if (D == d) {                                                                                             \
        hipLaunchKernelGGL((k_lmp_clusters<3, d, false>), grid, block, lds, st, count, near, list, A, M, chx_tabs_dev{}); \
        return;                                                                                               \
    }
    if (nb == 3) { CHX_D3_CASES(X) }
#undef X
#define X(d)                                                                                                  \
    if (D == d) {                                                                                             \
        hipLaunchKernelGGL((k_lmp_clusters<4, d, false>), grid, block, lds, st, count, near, list, A, M, chx_tabs_dev{}); \
        return;                                                                                               \
    }
    if (nb == 4) { CHX_D4_CASES(X) }
#undef X
}

void launch_lmp_out(const chx_lmp_args &A, double *F, double *eatom, double *vatom, double *glob, hipStream_t st)
{
    if (A.nall > 0)
        hipLaunchKernelGGL(k_lmp_out, dim3((unsigned)((A.nall + 255) / 256)), dim3(256), 0, st, A, F, eatom, vatom,
                           glob);
}

}  // namespace chx
