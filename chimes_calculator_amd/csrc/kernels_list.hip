// 3- and 4-body evaluation with one cluster per lane: in FP32-mixed precision
// with the coefficient contraction on the matrix cores (k_lane), in FP64 and
// for larger 4-body dimensions on the vector units (k_evalv).
//
// v_mfma_f32_4x4x1 multiplies sixteen independent 4x1 by 1x4 blocks: lane l
// holds column l of B and gets column l of D, four rows in four registers.
// With one block of A broadcast to all sixteen (cbsz = 4, abid = its number)
// an instruction is four FMAs of the lane's own B value with four
// coefficients, so each lane contracts its own cluster, with no staging, no
// exchange and no barrier, and one register of A holds sixteen such blocks.
// The vector ALU, which issues one unpacked FP32 FMA per lane in four cycles,
// bounded the vector form of these kernels (86-100% busy); here four FMAs take
// one issue slot and eight cycles of a matrix core that works beside it.
//
// The matrix instructions are reached by whole wavefronts only (lanes without
// a cluster carry a harmless one), since they ignore the execution mask.
//
// Compiled with -ffp-contract=off, as the other list kernels: the geometry
// reproduces the reference's get_dist bit for bit.
#include <hip/hip_runtime.h>

#include <utility>

#include "chx_cluster.h"
#include "chx_dev.h"
#include "chx_engine.h"
#include "chx_eval.h"
#include "chx_lane.h"
#include "chx_list_eval.h"
#include "eval_math.h"

namespace chx {

typedef float flt4 __attribute__((ext_vector_type(4)));

// f(integral_constant<int, 0>) ... f(integral_constant<int, N - 1>)
template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// acc[i] += (row i of block BLK of a) * b, each lane with its own b
template <int BLK>
__device__ __forceinline__ flt4 lane_fma4(float a, float b, flt4 acc)
{
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, acc, 4, BLK, 0);
}

// Dense contraction of the 3-body form, the arithmetic of contract3 (FP32
// sums over the last pair's index, in index order, FP64 above): the D^2 rows
// (a0, a1) in blocks of four.  A: the image's registers.
template <int D>
__device__ __forceinline__ void lane_contract3(const float (&A)[lane3_shape<D>::NV], const float (&T)[3][D],
                                               const float (&dT)[3][D], double &S, double (&G)[3])
{
    using SH = lane3_shape<D>;
    double t1[D], d1[D];
#pragma unroll
    for (int u = 0; u < D; u++) { t1[u] = T[1][u]; d1[u] = dT[1][u]; }
    double s0 = 0, g00 = 0, g01 = 0, g02 = 0, s1 = 0, g11 = 0, g12 = 0;
    // two blocks at a time: four independent chains of matrix instructions
    static_for<(SH::NQ + 1) / 2>([&](auto Hc) {
        constexpr int H = 2 * Hc, N = SH::NQ - H < 2 ? 1 : 2;
        flt4 z[2] = {}, w[2] = {};
        static_for<D>([&](auto Kc) {
            constexpr int k = Kc;
            static_for<N>([&](auto Jc) {
                constexpr int j = Jc, idx = (H + j) * D + k;
                z[j] = lane_fma4<idx % 16>(A[idx / 16], k == 0 ? 1.f : T[2][k], z[j]);
            });
            static_for<N>([&](auto Jc) {
                constexpr int j = Jc, idx = (H + j) * D + k;
                if constexpr (k > 0) w[j] = lane_fma4<idx % 16>(A[idx / 16], dT[2][k], w[j]);
            });
        });
        static_for<4 * N>([&](auto Ic) {
            constexpr int r = 4 * H + Ic, a0 = r / D, a1 = r % D;
            if constexpr (r < D * D) {
                const double zr = z[Ic / 4][r % 4], wr = w[Ic / 4][r % 4];
                if constexpr (a1 == 0) {
                    s1 = zr;
                    g11 = 0;
                    g12 = wr;
                } else {
                    s1 = fma(t1[a1], zr, s1);
                    g11 = fma(d1[a1], zr, g11);
                    g12 = fma(t1[a1], wr, g12);
                }
                if constexpr (a1 == D - 1) {
                    if constexpr (a0 == 0) {
                        s0 = s1;
                        g01 = g11;
                        g02 = g12;
                    } else {
                        const double t0 = T[0][a0], dt0 = dT[0][a0];
                        s0 = fma(t0, s1, s0);
                        g00 = fma(dt0, s1, g00);
                        g01 = fma(t0, g11, g01);
                        g02 = fma(t0, g12, g02);
                    }
                }
            }
        });
        __builtin_amdgcn_sched_barrier(0);
    });
    S = s0;
    G[0] = g00; G[1] = g01; G[2] = g02;
}

// Fold of a D^3 vector V[(x, y, z)] against T_x T_y T_z of three pairs and
// against the products with one factor's derivative, in FP64.
template <int D>
__device__ __forceinline__ void lane_fold(const flt4 (&V)[lane4_shape<D>::NQ], const float (&T)[6][D],
                                          const float (&dT)[6][D], int q0, double &S, double (&G)[3])
{
    double s0 = 0, g00 = 0, g01 = 0, g02 = 0;
#pragma unroll
    for (int x = 0; x < D; x++) {
        double s1 = 0, g11 = 0, g12 = 0;
#pragma unroll
        for (int y = 0; y < D; y++) {
            const int b = (x * D + y) * D;
            double s2 = V[b / 4][b % 4], g22 = 0;
#pragma unroll
            for (int z = 1; z < D; z++) {
                const double v = V[(b + z) / 4][(b + z) % 4];
                s2 = fma((double)T[q0 + 2][z], v, s2);
                g22 = fma((double)dT[q0 + 2][z], v, g22);
            }
            if (y == 0) {
                s1 = s2;
                g12 = g22;
            } else {
                const double t = T[q0 + 1][y], d = dT[q0 + 1][y];
                s1 = fma(t, s2, s1);
                g11 = fma(d, s2, g11);
                g12 = fma(t, g22, g12);
            }
        }
        if (x == 0) {
            s0 = s1;
            g01 = g11;
            g02 = g12;
        } else {
            const double t = T[q0][x], d = dT[q0][x];
            s0 = fma(t, s1, s0);
            g00 = fma(d, s1, g00);
            g01 = fma(t, g11, g01);
            g02 = fma(t, g12, g02);
        }
        __builtin_amdgcn_sched_barrier(0);  // conversions of V not ahead of their use
    }
    S = s0;
    G[0] = g00; G[1] = g01; G[2] = g02;
}

// V[m] = sum_k M[k][m] T_x T_y T_z (k = (x, y, z) of pairs q0 .. q0 + 2), from
// the image at img (row blocks of k = D^3 - 1 first).  The terms of high
// degree, the smaller ones, are added first.
template <int D>
__device__ __forceinline__ void lane_product(const float *__restrict__ img, const float (&T)[6][D], int q0,
                                             flt4 (&V)[lane4_shape<D>::NQ])
{
    using SH = lane4_shape<D>;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < SH::NQ; q++) V[q] = flt4{0.f, 0.f, 0.f, 0.f};
    if constexpr (D < 4) {
        float A[SH::NV];
#pragma unroll
        for (int v = 0; v < SH::NV; v++) A[v] = img[64 * v + lane];
        static_for<SH::ROWS>([&](auto Kc) {
            constexpr int kk = Kc, k = SH::ROWS - 1 - kk, x = k / (D * D), y = k / D % D, z = k % D;
            float b = 1.f;
            if constexpr (x > 0) b = T[q0][x];
            if constexpr (y > 0) b = x > 0 ? b * T[q0 + 1][y] : T[q0 + 1][y];
            if constexpr (z > 0) b = x + y > 0 ? b * T[q0 + 2][z] : T[q0 + 2][z];
            static_for<SH::NQ>([&](auto Qc) {
                constexpr int q = Qc, idx = kk * SH::NQ + q;
                V[q] = lane_fma4<idx % 16>(A[idx / 16], b, V[q]);
            });
        });
    } else {
        // one register of the image per k; a loop over the first index (code
        // size), its factor consumed from the back of a rotating copy
        static_assert(SH::NQ == 16, "one image register per k");
        float t0[D];
#pragma unroll
        for (int u = 0; u < D; u++) t0[u] = T[q0][u];
#pragma unroll 1
        for (int x = D - 1; x >= 0; x--) {
            const float *p = img + (D - 1 - x) * D * D * 64 + lane;
            float A[D * D];
#pragma unroll
            for (int v = 0; v < D * D; v++) A[v] = p[64 * v];
            const float tx = t0[D - 1];
            static_for<D * D>([&](auto Kc) {
                constexpr int kk = Kc, k = D * D - 1 - kk, y = k / D, z = k % D;
                float b = tx;
                if constexpr (y > 0) b *= T[q0 + 1][y];
                if constexpr (z > 0) b *= T[q0 + 2][z];
                static_for<16>([&](auto Qc) {
                    constexpr int q = Qc;
                    V[q] = lane_fma4<q>(A[kk], b, V[q]);
                });
            });
#pragma unroll
            for (int u = D - 1; u > 0; u--) t0[u] = t0[u - 1];
        }
    }
}

// Dense contraction of the 4-body form: with X = T_01 (x) T_02 (x) T_03 and
// Y = T_12 (x) T_13 (x) T_23, Z = C^T X gives the energy form and the
// derivatives of the last three pairs as folds of Z, W = C Y those of the
// first three as folds of W.
template <int D>
__device__ __forceinline__ void lane_contract4(const float *__restrict__ img, const float (&T)[6][D],
                                               const float (&dT)[6][D], double &S, double (&G)[6])
{
    using SH = lane4_shape<D>;
    double g[3], s;
    {
        flt4 Z[SH::NQ];
        lane_product<D>(img, T, 0, Z);
        __builtin_amdgcn_sched_barrier(0);
        lane_fold<D>(Z, T, dT, 3, S, g);
        G[3] = g[0]; G[4] = g[1]; G[5] = g[2];
        // the first fold ends before the second product begins, or both
        // vectors are alive together (D = 4: 485 registers spilled, 0.54
        // against 0.17 ms)
        asm volatile("" : "+v"(S), "+v"(G[3]), "+v"(G[4]), "+v"(G[5]));
    }
    {
        flt4 W[SH::NQ];
        lane_product<D>(img + 64 * SH::NV, T, 3, W);
        __builtin_amdgcn_sched_barrier(0);
        lane_fold<D>(W, T, dT, 0, s, g);
        G[0] = g[0]; G[1] = g[1]; G[2] = g[2];
    }
}

// ---------------------------------------------------------------------------
// 3- and 4-body, FP32-mixed: one cluster per lane, one wavefront per
// 64-cluster tile of one group, the contraction on the matrix cores.
//
// A workgroup takes `tiles` consecutive tiles per wavefront.  With the
// contraction there, the kernel waits on dependent gathers (record, atom and
// images, type permutation) and on the accumulation's atomics more than it
// computes, so what a workgroup does once (status, group search, clearing the
// force table, barriers, the table's flush) is spread over more clusters, its
// wavefronts drift apart and hide each other's waits, and an atom that
// consecutive tiles share is flushed once.  C/O batch of 4096 configurations
// (26.3 M triplets, 13.2 M quadruplets): 3-body D = 7 1.60 ms on the vector
// ALU, 1.63 ms here with one tile, 1.43 with four, 1.41 with eight; 4-body
// D = 3 1.33 ms on the vector ALU, 1.27 with four, 1.29 with eight (1.17 since
// the exact splits were shortened).  Carbon,
// 32768 atoms: 3-body D = 10 156 -> 129 us, 4-body D = 4 202 -> 167 us.
//
// The file is compiled without the hoisting of constants out of that loop
// (-disable-machine-licm): the FP64 literals of the exponentials in registers
// across the loop made every kernel here spill (3-body D = 7: 43 registers,
// 1.64 against 1.43 ms).
// ---------------------------------------------------------------------------
// Wavefronts per SIMD.  The targets hold the 3-body kernels for D <= 8 to 128
// registers and for D <= 11 to 168; at D = 8 and 11 a few spill (32 and 12 bytes
// of scratch), which costs less than a wavefront: 22 M carbon triplets, D = 8
// 1.31 ms at four wavefronts, 1.45 at three without scratch; D = 11 2.17 ms at
// three, 2.54 at two.
template <int NB, int D>
constexpr int lane_waves()
{
    return NB == 3 ? (D <= 8 ? 4 : (D <= 11 ? 3 : 2)) : (D <= 3 ? 3 : 2);
}

template <int NB, int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(lane_waves<NB, D>()))) void k_lane(
    int tiles, int G, const int *__restrict__ gbase, const int *__restrict__ gend,
    const chx_group *__restrict__ groups, int total_word, const int2 *__restrict__ list,
    const chx_cfg *__restrict__ cfgs, const chx_atom_s *__restrict__ as, int nb_cap,
    const chx_entry_s *__restrict__ es, unsigned long long *Facc, unsigned long long *Cacc, int *cfg_stat,
    int *status)
{
    using PQ = pairs_of<NB>;
    constexpr int P = PQ::P;
    // the workgroup's member forces merged per atom; the table holds the
    // distinct atoms of a typical workgroup (a few hundred) with room to
    // spare, and anything past it goes straight to memory
    __shared__ fx_table<512> tab;
    // status read overlapped with the table clear; one barrier for both
    __shared__ int flags_s;
    if (threadIdx.x == 0) flags_s = __atomic_load_n(&status[CHX_ST_FLAGS], __ATOMIC_RELAXED);
    tab.clear();
    __syncthreads();
    if (flags_s & CHX_STOP) return;
    const int lane = threadIdx.x & 63;
    // wave index made explicitly uniform, so the group, its slots and its
    // coefficients are read through the scalar unit
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const long total = __builtin_amdgcn_readfirstlane(status[total_word]);
    const long first = ((long)blockIdx.x * 4 + wave) * tiles * 64;
    bool bad = false;
    int g = first < total ? find_group(gbase, G, first) : 0;
#pragma unroll 1
    for (int u = 0; u < tiles; u++) {
        const long t0 = first + u * 64;
        if (t0 >= total) break;
        while (g + 1 < G && uniform_load(gbase, g + 1) <= t0) g++;
        g = __builtin_amdgcn_readfirstlane(g);
        // read through the constant address space, field by field where they
        // are used: past the first tile's atomics the compiler would not use
        // scalar loads by itself, and a copy of the whole group spilled
        // scalar registers
        const const_ptr<chx_group> grp = (const_ptr<chx_group>)(groups + g);
        auto slot = [&](int q) {
            chx_slot s;
            s.rin = grp->s[q].rin; s.rout = grp->s[q].rout;
            s.xavg = grp->s[q].xavg; s.ilam = grp->s[q].ilam; s.ixdiff = grp->s[q].ixdiff;
            s.irout = grp->s[q].irout; s.iramp = grp->s[q].iramp;
            return s;
        };
        if (!(grp->type >= 0 && grp->D == D)) continue;
        const int end = uniform_load(gend, g);
        const long c = t0 + lane;
        int ckey = -1;
        double q7[7] = {0, 0, 0, 0, 0, 0, 0};
        double Fr[NB][3];   // force on each member (canonical order)
        int key[NB];        // replicated atom of each member, -1 none
#pragma unroll
        for (int m = 0; m < NB; m++) { key[m] = -1; Fr[m][0] = Fr[m][1] = Fr[m][2] = 0.0; }
        double p[NB][3], r[P], dr[P][3], S, Gq[P];
        int par[NB], cfg = 0, pm[NB], flags = 0;
        bool act = false;
        if (c < end)
            act = cluster_geometry<NB>(grp->nt, grp->perm, [&](int q) { return grp->s[q].rout; }, list[c], cfgs, as,
                                       nb_cap, es, p, par, r, cfg, pm, dr);
        auto finish = [&]() {
            double f[P], fd[P], E, fs[P];
#pragma unroll
            for (int q = 0; q < P; q++) fcut(r[q], slot(q), grp->tersoff, grp->fcut_var, f[q], fd[q]);
            cluster_scalars<P, double>(r, f, fd, S, Gq, E, fs);
            q7[0] = E;
            cluster_forces<NB>(dr, fs, Fr, q7);
#pragma unroll
            for (int a = 0; a < NB; a++) key[a] = par[a];
            ckey = cfg;
            note_flags(cfg_stat, cfg, flags);
        };
        if (__ballot(act) == 0) continue;
        // whole wavefront: lanes without a cluster at the cutoffs
#pragma unroll
        for (int q = 0; q < P; q++) r[q] = act ? r[q] : grp->s[q].rout;
        float T[P][D], dT[P][D];
#pragma unroll
        for (int q = 0; q < P; q++) cheby<D, float>(r[q], slot(q), T[q], dT[q], flags);
        if constexpr (NB == 3) {
            float A[lane3_shape<D>::NV];
#pragma unroll
            for (int v = 0; v < lane3_shape<D>::NV; v++) A[v] = grp->Cl[64 * v + lane];
            lane_contract3<D>(A, T, dT, S, Gq);
        } else {
            lane_contract4<D>(grp->Cl, T, dT, S, Gq);
        }
        // the folds stay here: moved into the branch below, where their
        // results are used, they would keep every product alive
        asm volatile("" : "+v"(S));
#pragma unroll
        for (int q = 0; q < P; q++) asm volatile("" : "+v"(Gq[q]));
        if (act) finish();
        // every member's force through the LDS table; energy and virial go to
        // the configuration
#pragma unroll
        for (int m = 0; m < NB; m++) tab.add(key[m], Fr[m], Facc, bad);
        fx_cfg_sums(Cacc, ckey, blockIdx.x & (CHX_CACC_SLOTS - 1), q7, bad);
    }
    __syncthreads();
    tab.flush(Facc);
    if (bad) atomicOr(&status[CHX_ST_FLAGS], CHX_BAD_RANGE);
}

// ---------------------------------------------------------------------------
// 3- and 4-body on the vector units: one thread per cluster, one wavefront per
// 64-cluster tile of one group (any supported D); the workgroup's member
// forces are merged per atom in an LDS table before they reach memory.
// Occupancy targets, measured: the FP64 4-body kernels for D <= 3 are held to
// two wavefronts per SIMD (left alone the compiler gives them one; at two
// they need no scratch), the FP64 3-body kernels for D <= 8 to three.
// ---------------------------------------------------------------------------
template <int NB, int D, typename R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NB == 4 && D <= 3 ? 2 : (NB == 3 && D <= 8 ? 3 : 1)))) void k_evalv(int G, const int *__restrict__ gbase, const int *__restrict__ gend,
                                                const chx_group *__restrict__ groups, int total_word,
                                                const int2 *__restrict__ list, const chx_cfg *__restrict__ cfgs,
                                                const chx_atom_s *__restrict__ as, int nb_cap,
                                                const chx_entry_s *__restrict__ es, unsigned long long *Facc,
                                                unsigned long long *Cacc, int *cfg_stat, int *status)
{
    using PQ = pairs_of<NB>;
    constexpr int P = PQ::P;
    // the workgroup's member forces merged per atom; the table holds the
    // distinct atoms of a typical tile (a few hundred) with room to spare,
    // and anything past it goes straight to memory, so the workgroup stays
    // small enough for five per CU
    __shared__ fx_table<512> tab;
    // status read overlapped with the table clear; one barrier for both
    __shared__ int flags_s;
    if (threadIdx.x == 0) flags_s = __atomic_load_n(&status[CHX_ST_FLAGS], __ATOMIC_RELAXED);
    tab.clear();
    __syncthreads();
    if (flags_s & CHX_STOP) return;
    const int lane = threadIdx.x & 63;
    // wave index made explicitly uniform, so the group, its slots and its
    // coefficients are read through the scalar unit
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const long t0 = ((long)blockIdx.x * 4 + wave) * 64;
    bool wave_on = t0 < status[total_word];
    const int g = wave_on ? find_group(gbase, G, t0) : 0;
    const chx_group &grp = groups[g];
    wave_on = wave_on && grp.type >= 0 && grp.D == D;
    const long c = t0 + lane;
    int ckey = -1;
    double q7[7] = {0, 0, 0, 0, 0, 0, 0};
    double Fr[NB][3];   // force on each member (canonical order)
    int key[NB];        // replicated atom of each member, -1 none
#pragma unroll
    for (int m = 0; m < NB; m++) { key[m] = -1; Fr[m][0] = Fr[m][1] = Fr[m][2] = 0.0; }
    bool bad = false;
    if (wave_on && c < gend[g]) {
        const int2 rec = list[c];
        double p[NB][3], r[P], dr[P][3];
        int par[NB], cfg, pm[NB];
        if (cluster_geometry<NB>(grp, rec, cfgs, as, nb_cap, es, p, par, r, cfg, pm, dr)) {
            R T[P][D], dT[P][D];
            double f[P], fd[P];
            int flags = 0;
#pragma unroll
            for (int q = 0; q < P; q++) {
                cheby<D, R>(r[q], grp.s[q], T[q], dT[q], flags);
                fcut(r[q], grp.s[q], grp.tersoff, grp.fcut_var, f[q], fd[q]);
            }
            const R *Cd = sizeof(R) == 8 ? (const R *)grp.C : (const R *)grp.Cf;
            double S, Gq[P], E, fs[P];
            if constexpr (NB == 3) contract3<D, R, double>(Cd, T, dT, S, Gq);
            else contract4<D, R, double>(Cd, T, dT, S, Gq);
            cluster_scalars<P, double>(r, f, fd, S, Gq, E, fs);
            q7[0] = E;
            double F[NB][3];
            cluster_forces<NB>(dr, fs, F, q7);
#pragma unroll
            for (int a = 0; a < NB; a++) {
                key[a] = par[a];
                Fr[a][0] = F[a][0]; Fr[a][1] = F[a][1]; Fr[a][2] = F[a][2];
            }
            ckey = cfg;
            note_flags(cfg_stat, cfg, flags);
        }
    }
    // every member's force through the LDS table (the owner's too: its
    // lanes' LDS atomics cost fewer instructions than six wavefront scans);
    // energy and virial go to the configuration
#pragma unroll
    for (int m = 0; m < NB; m++) tab.add(key[m], Fr[m], Facc, bad);
    fx_cfg_sums(Cacc, ckey, blockIdx.x & (CHX_CACC_SLOTS - 1), q7, bad);
    __syncthreads();
    tab.flush(Facc);
    if (bad) atomicOr(&status[CHX_ST_FLAGS], CHX_BAD_RANGE);
}

// Tiles per wavefront of the lane kernels: four where that leaves 4096
// workgroups (four for each of the 1024 the device holds at once), else one,
// so that a short list still reaches every compute unit.  One, two and four
// tiles, us: 1.3 M slots (C/O 4-body) 145, 129, 129; 2.1 M 227, 205, 208;
// 4.7 M (C/O 3-body) 295, 281, 281; 5.1 M (C/O 4-body) 530, 472, 436; but 0.2 M
// 25, 28, 35, and 0.4 to 0.8 M 52, 58, 63 and 100, 94, 108.  Two or four tiles
// from 1.3 M slots would be 3-18% shorter than the one that the line gives
// lists up to 4.2 M.
constexpr long LANE_TILES = 4;

void launch_evalv(int nb, int D, int prec, const chx_list_args &la, hipStream_t st)
{
    if (la.cap <= 0 || la.G <= 0) return;
    const int word = nb == 3 ? CHX_ST_N3 : CHX_ST_N4;
    const dim3 grid((unsigned)((la.cap + 255) / 256)), block(256);
    const int tiles = la.cap >= 256 * 4096 * LANE_TILES ? (int)LANE_TILES : 1;
    const dim3 lgrid((unsigned)((la.cap + 256 * tiles - 1) / (256 * tiles)));
#define LANE(NB_, d)                                                                                           \
    if (D == d) {                                                                                              \
        hipLaunchKernelGGL((k_lane<NB_, d>), lgrid, block, 0, st, tiles, la.G, la.gbase, la.gend, la.groups,     \
                           word, la.list, la.cfgs, la.as, la.nb_cap, la.es, la.Facc, la.Cacc, la.cfg_stat,     \
                           la.status);                                                                         \
        return;                                                                                                \
    }
#define VEC(NB_, d, R)                                                                                         \
    if (D == d) {                                                                                              \
        hipLaunchKernelGGL((k_evalv<NB_, d, R>), grid, block, 0, st, la.G, la.gbase, la.gend, la.groups, word,   \
                           la.list, la.cfgs, la.as, la.nb_cap, la.es, la.Facc, la.Cacc, la.cfg_stat, la.status); \
        return;                                                                                                \
    }
    const bool f32 = prec != CHX_FP64;
    if (f32 && nb == 3) {
#define X(d) LANE(3, d)
        CHX_D3_CASES(X)
#undef X
    } else if (f32) {
        LANE(4, 2) LANE(4, 3) LANE(4, 4) VEC(4, 5, float) VEC(4, 6, float)
    } else if (nb == 3) {
#define X(d) VEC(3, d, double)
        CHX_D3_CASES(X)
#undef X
    } else {
#define X(d) VEC(4, d, double)
        CHX_D4_CASES(X)
#undef X
    }
#undef LANE
#undef VEC
}

}  // namespace chx
