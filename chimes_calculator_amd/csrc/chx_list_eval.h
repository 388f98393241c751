// Device code shared by the kernels that evaluate the 3-/4-body lists: pair
// vectors, a list slot's group, the members of a cluster record in canonical
// order with their geometry, and the members' forces.
#pragma once
#include <hip/hip_runtime.h>

#include "chx_dev.h"
#include "chx_types.h"
#include "eval_math.h"

namespace chx {

__device__ __forceinline__ void mv3(const double *m, const double *d, double *o)
{
    o[0] = m[0] * d[0] + m[1] * d[1] + m[2] * d[2];
    o[1] = m[3] * d[0] + m[4] * d[1] + m[5] * d[2];
    o[2] = m[6] * d[0] + m[7] * d[1] + m[8] * d[2];
}

// dr = h (b - a) and its length (serial_chimes_interface.h:176-208)
__device__ __forceinline__ double pair_vec(const double *h, const double *a, const double *b, double *dr)
{
    const double d[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
    mv3(h, d, dr);
    return sqrt(dr[0] * dr[0] + dr[1] * dr[1] + dr[2] * dr[2]);
}

__device__ __forceinline__ void note_flags(int *cfg_stat, int cfg, int flags)
{
    if (!flags) return;
    atomicMax(&cfg_stat[4 * cfg + 0], (flags & FLAG_BELOW_RIN) ? 2 : ((flags & FLAG_PENALTY) ? 1 : 0));
    if (flags & FLAG_PENALTY) atomicAdd(&cfg_stat[4 * cfg + 1], 1);
    if (flags & FLAG_OUT_OF_RANGE) atomicAdd(&cfg_stat[4 * cfg + 2], 1);
}

// Group of list slot t: the last group whose aligned base is <= t.
__device__ __forceinline__ int find_group(const int *__restrict__ gbase, int G, long t)
{
    int lo = 0, hi = G - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (gbase[mid] <= t) lo = mid; else hi = mid - 1;
    }
    return lo;
}

// Member positions, types and replicated atom indices of a cluster record.
template <int NB>
__device__ __forceinline__ void load_members(const int2 rec, const chx_atom_s *__restrict__ as,
                                             int nb_cap, const chx_entry_s *__restrict__ es,
                                             double (&p)[NB][3], int (&t)[NB], int (&par)[NB], int &cfg)
{
    const int i = rec.x;
    const chx_atom_s ai = as[i];
    cfg = ai.cfg;
    p[0][0] = ai.u[0]; p[0][1] = ai.u[1]; p[0][2] = ai.u[2];
    t[0] = ai.type;
    par[0] = i;
    const long off = (long)i * nb_cap - 1;  // owner i's slab
#pragma unroll
    for (int m = 1; m < NB; m++) {
        const int s = (rec.y >> (10 * (m - 1))) & 1023;
        const chx_entry_s g = es[off + s];
        p[m][0] = g.v[0]; p[m][1] = g.v[1]; p[m][2] = g.v[2];
        t[m] = g.type;
        par[m] = g.parent;
    }
}

// Reorders the members into parameter-file atom order: canonical member a is
// runtime member perm[a] (the first matching permutation, chimesFF.h:480-526).
template <int NB>
__device__ __forceinline__ void canonical(const int *__restrict__ perm_tab, int tup, double (&p)[NB][3],
                                          int (&par)[NB], int (&pm)[NB])
{
#pragma unroll
    for (int a = 0; a < NB; a++) pm[a] = perm_tab[tup * NB + a];
    double q[NB][3];
    int c[NB];
#pragma unroll
    for (int a = 0; a < NB; a++) {
        c[a] = par[0];
        q[a][0] = p[0][0]; q[a][1] = p[0][1]; q[a][2] = p[0][2];
#pragma unroll
        for (int b = 1; b < NB; b++) {
            const bool s = pm[a] == b;
            c[a] = s ? par[b] : c[a];
            q[a][0] = s ? p[b][0] : q[a][0];
            q[a][1] = s ? p[b][1] : q[a][1];
            q[a][2] = s ? p[b][2] : q[a][2];
        }
    }
#pragma unroll
    for (int a = 0; a < NB; a++) {
        par[a] = c[a];
        p[a][0] = q[a][0]; p[a][1] = q[a][1]; p[a][2] = q[a][2];
    }
}

template <int NB>
struct pairs_of;
template <>
struct pairs_of<3> {
    static constexpr int P = 3;
    static constexpr int a[3] = {0, 0, 1};
    static constexpr int b[3] = {1, 2, 2};
};
template <>
struct pairs_of<4> {
    static constexpr int P = 6;
    static constexpr int a[6] = {0, 0, 0, 1, 1, 2};
    static constexpr int b[6] = {1, 2, 3, 2, 3, 3};
};

// Cluster geometry in canonical order: members, pair vectors and distances,
// and whether every pair is inside its cutoff (rout(q) of slot q); canonical
// member a is runtime member pm[a] (runtime member 0 is the owner).
template <int NB, class ROUT>
__device__ __forceinline__ bool cluster_geometry(int nt, const int *__restrict__ perm, const ROUT &rout,
                                                 const int2 rec, const chx_cfg *__restrict__ cfgs,
                                                 const chx_atom_s *__restrict__ as, int nb_cap,
                                                 const chx_entry_s *__restrict__ es, double (&p)[NB][3],
                                                 int (&par)[NB], double (&r)[pairs_of<NB>::P], int &cfg,
                                                 int (&pm)[NB], double (&dr)[pairs_of<NB>::P][3])
{
    using PQ = pairs_of<NB>;
    int t[NB];
    load_members<NB>(rec, as, nb_cap, es, p, t, par, cfg);
    int tup = 0;
#pragma unroll
    for (int a = 0; a < NB; a++) tup = tup * nt + t[a];
    canonical<NB>(perm, tup, p, par, pm);
    const chx_cfg &C = cfgs[cfg];
    bool in = true;
#pragma unroll
    for (int q = 0; q < PQ::P; q++) {
        r[q] = pair_vec(C.h, p[PQ::a[q]], p[PQ::b[q]], dr[q]);
        in = in && (r[q] < rout(q));
    }
    return in;
}

template <int NB>
__device__ __forceinline__ bool cluster_geometry(const chx_group &grp, const int2 rec,
                                                 const chx_cfg *__restrict__ cfgs,
                                                 const chx_atom_s *__restrict__ as, int nb_cap,
                                                 const chx_entry_s *__restrict__ es, double (&p)[NB][3],
                                                 int (&par)[NB], double (&r)[pairs_of<NB>::P], int &cfg,
                                                 int (&pm)[NB], double (&dr)[pairs_of<NB>::P][3])
{
    return cluster_geometry<NB>(grp.nt, grp.perm, [&](int q) { return grp.s[q].rout; }, rec, cfgs, as, nb_cap, es, p,
                                par, r, cfg, pm, dr);
}

// The same without the pair vectors.
template <int NB>
__device__ __forceinline__ bool cluster_geometry(const chx_group &grp, const int2 rec,
                                                 const chx_cfg *__restrict__ cfgs,
                                                 const chx_atom_s *__restrict__ as, int nb_cap,
                                                 const chx_entry_s *__restrict__ es, double (&p)[NB][3],
                                                 int (&par)[NB], double (&r)[pairs_of<NB>::P], int &cfg,
                                                 int (&pm)[NB])
{
    double dr[pairs_of<NB>::P][3];
    return cluster_geometry<NB>(grp, rec, cfgs, as, nb_cap, es, p, par, r, cfg, pm, dr);
}

// Forces of one cluster from its pair force scalars: F_a += fs dr, F_b -= fs
// dr for pair (a, b) of canonical members; virial -= fs dr dr into the q7
// owner accumulator slots 1..6.
template <int NB>
__device__ __forceinline__ void cluster_forces(const double (&drq)[pairs_of<NB>::P][3],
                                               const double (&fs)[pairs_of<NB>::P], double (&F)[NB][3],
                                               double (&q7)[7])
{
    using PQ = pairs_of<NB>;
#pragma unroll
    for (int m = 0; m < NB; m++) F[m][0] = F[m][1] = F[m][2] = 0.0;
#pragma unroll
    for (int q = 0; q < PQ::P; q++) {
        const double (&dr)[3] = drq[q];
        const double f = fs[q];
#pragma unroll
        for (int k = 0; k < 3; k++) {
            F[PQ::a[q]][k] += f * dr[k];
            F[PQ::b[q]][k] -= f * dr[k];
        }
        q7[1] -= f * (dr[0] * dr[0]);
        q7[2] -= f * (dr[0] * dr[1]);
        q7[3] -= f * (dr[0] * dr[2]);
        q7[4] -= f * (dr[1] * dr[1]);
        q7[5] -= f * (dr[1] * dr[2]);
        q7[6] -= f * (dr[2] * dr[2]);
    }
}

}  // namespace chx
