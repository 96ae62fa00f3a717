// Compact line-operator kernels for gfx950 (wave64).
//
// One thread owns one chunk (<= MC points) of one line and keeps it in
// registers: it forms the compact RHS from a register window of f
// (src/operators.jl:113-174 fill), runs the chunk-local Thomas / banded LU
// sweeps (src/tridiag.jl:46-57, src/banded.jl:63-80), exchanges its 2q end
// values with the other chunks of the same line, solves the
// reduced interface system by block parallel cyclic reduction (coefficients
// precomputed by the plan), and applies the spike correction
// x = y - V tail_prev - W head_next (src/tridiag.jl:159-168,
// src/banded.jl:371-382) before handing each value to a fused epilogue.
//
//  * y/z sweeps: 64 (or fewer) consecutive x-lanes per chunk row; every load
//    and store of a row is a contiguous 512-byte segment; no transposes.
//  * x sweeps: a wave (lines of at most 64 chunks) or a block (longer ones)
//    stages whole lines in LDS with coalesced loads, each lane reads its chunk
//    window from LDS, results return through the same tile for coalesced stores.
// No MFMA: the work is banded and HBM-bound.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "cles_internal.h"

// Multiply-adds in the line kernels are written as explicit fma where they
// matter and are otherwise not contracted: the compiler's choice of which
// product to fuse can differ between instantiations of the same arithmetic
// (chunk capacities, epilogues), and every kernel must round alike.
#pragma clang fp contract(off)

namespace cles {

constexpr int MC = 32;     // maximum chunk length (points per thread)
constexpr int YZU_THREADS = 1024;   // threads of a one-chunk-per-wave y / z block at most
constexpr int NCMAX = 4;   // closure rows per edge handled by the kernels

// Plan tables live in global memory; a pointer read out of memory (the ragged
// kernel's per-instance plans) is otherwise a flat pointer, whose loads also
// wait on the LDS counter.
template <typename T> __device__ __forceinline__ T gload(const T *ptr)
{
    return *(const __attribute__((address_space(1))) T *)ptr;
}

template <typename T> __device__ __forceinline__ const T *coefp(const LineDev &p);
template <> __device__ __forceinline__ const double *coefp<double>(const LineDev &p) { return p.coef64; }
template <> __device__ __forceinline__ const float *coefp<float>(const LineDev &p) { return p.coef32; }
template <typename T> __device__ __forceinline__ const T *rowsp(const LineDev &p);
template <> __device__ __forceinline__ const double *rowsp<double>(const LineDev &p) { return p.rows64; }
template <> __device__ __forceinline__ const float *rowsp<float>(const LineDev &p) { return p.rows32; }

// Loads through the constant address space: wave-uniform addresses become
// scalar loads wherever they stand (tables are never written by a kernel).
template <typename T> __device__ __forceinline__ T cload(const T *ptr)
{
    return *(const __attribute__((address_space(4))) T *)ptr;
}

// One chunk's block of row constants (LineDev::rows64): row t of field f, read
// by scalar loads (UNI: the wave has one chunk) or per lane (the lanes of a wave
// share a few blocks, so a load is a few broadcasts at constant offsets).
// fence(v) makes per-lane loads that follow wait for v: an empty asm statement
// through which the base pointer depends on it, which keeps the compiler from
// issuing every group of rows at once (and spilling them).
template <typename T, int CAP, bool UNI> struct Rows {
    const T *base;
    __device__ __forceinline__ T operator()(int f, int t) const
    {
        if constexpr (UNI) return cload(base + f * CAP + t);
        else return gload(base + f * CAP + t);
    }
    template <typename D> __device__ __forceinline__ void fence(const D &dep)
    {
        if constexpr (!UNI) asm volatile("" : "+v"(base) : "v"(dep));
    }
};

// ---------------------------------------------------------------------------
// Epilogues
// ---------------------------------------------------------------------------
template <typename T, int EPI>
__device__ __forceinline__ void epilogue(const EpiArgs &e, int64_t o, double v)
{
    if constexpr (EPI == EPI_ART_MULTI) {   // e is the field's own ART_* epilogue (select_field)
        if (e.kind == EPI_ART_MUBETA) epilogue<T, EPI_ART_MUBETA>(e, o, v);
        else if (e.kind == EPI_ART_KAPPA) epilogue<T, EPI_ART_KAPPA>(e, o, v);
        else epilogue<T, EPI_ART_D>(e, o, v);
        return;
    }
    // gated kinds: one flag and dt, or (ipts > 0: instances of ipts points side
    // by side) the flag and dt of the point's instance
    [[maybe_unused]] unsigned ii = 0;
    if constexpr (EPI == EPI_STORE_GATE || EPI == EPI_LSRK_DEV) {
        if (e.ipts) ii = (unsigned)o / e.ipts;
        if (!e.gate[ii]) return;
    }
    if constexpr (EPI == EPI_STORE || EPI == EPI_STORE_GATE || EPI == EPI_STORE_NEG) {
        ((T *)e.out)[o] = EPI == EPI_STORE_NEG ? (T)(-v) : (T)v;
    } else if constexpr (EPI == EPI_SUB) {
        T *out = (T *)e.out;
        out[o] = out[o] - (T)v;
    } else if constexpr (EPI == EPI_LSRK || EPI == EPI_LSRK_DEV) {
        // rhs.jl:665-667 dQ -= D_z F_z, then timestep.jl:85-94 on the FP64 state
        // acc == NULL: this is the only active dimension, dQ = 0 - v
        const T *acc = (const T *)e.a0;
        const double dq = acc ? (double)(acc[o] - (T)v) : -v;
        const double dt = EPI == EPI_LSRK_DEV ? e.dtp[ii] : e.dt;
        double nv = fma(dt, dq, e.c0 != 0.0 ? e.c0 * e.du[o] : 0.0);
        e.du[o] = nv;
        e.Q[o] = fma(e.c1, nv, e.Q[o]);
    } else if constexpr (EPI == EPI_ART_MUBETA) {
        // artificial.jl:296-304
        const T *rho = (const T *)e.a0;
        T s = (T)v;
        T rs = rho[o] * (s > T(0) ? s : T(0));
        ((T *)e.out)[o] = (T)e.c0 * rs;
        ((T *)e.out2)[o] = (T)e.c1 * rs;
    } else if constexpr (EPI == EPI_ART_KAPPA) {
        // artificial.jl:331-339 with physics.jl:155-156
        const T *rho = (const T *)e.a0, *c = (const T *)e.a1, *Tt = (const T *)e.a2;
        T s = (T)v;
        T tt = Tt[o];
        const T eps = sizeof(T) == 8 ? (T)2.220446049250313e-16 : (T)1.1920929e-07f;
        T scale = rho[o] * c[o] / (tt > eps ? tt : eps);
        ((T *)e.out)[o] = (T)e.c0 * scale * (s > T(0) ? s : T(0));
    } else if constexpr (EPI == EPI_ART_D) {
        // artificial.jl:349-355
        const T *c = (const T *)e.a1;
        T s = (T)v;
        ((T *)e.out)[o] = (T)e.c0 * c[o] * (s > T(0) ? s : T(0));
    }
}

// Batched epilogue: every input of NB points is loaded before any output is
// stored, so the loads of a batch are in flight together (the compiler cannot
// reorder them across stores through pointers that may alias).
template <typename T, int EPI, int NB>
__device__ __forceinline__ void epilogue_batch(const EpiArgs &e, const int64_t (&o)[NB], const T (&v)[NB],
                                               const bool (&ok)[NB])
{
    if constexpr (EPI == EPI_ART_MULTI) {
        if (e.kind == EPI_ART_MUBETA) epilogue_batch<T, EPI_ART_MUBETA, NB>(e, o, v, ok);
        else if (e.kind == EPI_ART_KAPPA) epilogue_batch<T, EPI_ART_KAPPA, NB>(e, o, v, ok);
        else epilogue_batch<T, EPI_ART_D, NB>(e, o, v, ok);
        return;
    }
    // gated kinds: one flag and dt for the launch, or (ipts > 0) those of
    // each point's instance
    bool okk[NB];
    double dtv[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        okk[i] = ok[i];
        dtv[i] = e.dt;
    }
    if constexpr (EPI == EPI_STORE_GATE || EPI == EPI_LSRK_DEV) {
        if (e.ipts) {
#pragma unroll
            for (int i = 0; i < NB; i++) {
                const unsigned ii = ok[i] ? (unsigned)o[i] / e.ipts : 0u;
                okk[i] = ok[i] && e.gate[ii] != 0;
                if constexpr (EPI == EPI_LSRK_DEV) dtv[i] = e.dtp[ii];
            }
        } else {
            if (!*e.gate) return;
            if constexpr (EPI == EPI_LSRK_DEV) {
                const double d = *e.dtp;
#pragma unroll
                for (int i = 0; i < NB; i++) dtv[i] = d;
            }
        }
    }
    if constexpr (EPI == EPI_STORE || EPI == EPI_STORE_NEG || EPI == EPI_STORE_GATE) {
        constexpr int E1 = EPI == EPI_STORE_GATE ? (int)EPI_STORE : EPI;   // the gate is applied
#pragma unroll
        for (int i = 0; i < NB; i++)
            if (okk[i]) epilogue<T, E1>(e, o[i], (double)v[i]);
    } else if constexpr (EPI == EPI_SUB) {
        T *out = (T *)e.out;
        T a[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) a[i] = ok[i] ? out[o[i]] : T(0);
#pragma unroll
        for (int i = 0; i < NB; i++)
            if (ok[i]) out[o[i]] = a[i] - v[i];
    } else if constexpr (EPI == EPI_LSRK || EPI == EPI_LSRK_DEV) {
        const T *acc = (const T *)e.a0;
        T a[NB];
        double du[NB], q[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            a[i] = (okk[i] && acc) ? acc[o[i]] : T(0);
            du[i] = okk[i] && e.c0 != 0.0 ? e.du[o[i]] : 0.0;
            q[i] = okk[i] ? e.Q[o[i]] : 0.0;
        }
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!okk[i]) continue;
            const double dq = acc ? (double)(a[i] - v[i]) : -(double)v[i];
            const double nv = fma(dtv[i], dq, e.c0 * du[i]);
            e.du[o[i]] = nv;
            e.Q[o[i]] = fma(e.c1, nv, q[i]);
        }
    } else if constexpr (EPI == EPI_ART_MUBETA) {
        const T *rho = (const T *)e.a0;
        T r[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) r[i] = ok[i] ? rho[o[i]] : T(0);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
            const T rs = r[i] * (v[i] > T(0) ? v[i] : T(0));
            ((T *)e.out)[o[i]] = (T)e.c0 * rs;
            ((T *)e.out2)[o[i]] = (T)e.c1 * rs;
        }
    } else if constexpr (EPI == EPI_ART_KAPPA) {
        const T *rho = (const T *)e.a0, *c = (const T *)e.a1, *Tt = (const T *)e.a2;
        T r[NB], cc[NB], tt[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            r[i] = ok[i] ? rho[o[i]] : T(0);
            cc[i] = ok[i] ? c[o[i]] : T(0);
            tt[i] = ok[i] ? Tt[o[i]] : T(1);
        }
        const T eps = sizeof(T) == 8 ? (T)2.220446049250313e-16 : (T)1.1920929e-07f;
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
            const T scale = r[i] * cc[i] / (tt[i] > eps ? tt[i] : eps);
            ((T *)e.out)[o[i]] = (T)e.c0 * scale * (v[i] > T(0) ? v[i] : T(0));
        }
    } else if constexpr (EPI == EPI_ART_D) {
        const T *c = (const T *)e.a1;
        T cc[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) cc[i] = ok[i] ? c[o[i]] : T(0);
#pragma unroll
        for (int i = 0; i < NB; i++)
            if (ok[i]) ((T *)e.out)[o[i]] = (T)e.c0 * cc[i] * (v[i] > T(0) ? v[i] : T(0));
    }
}

// Field of a multi-field launch (grid y): field 0 keeps the launch's own input
// and epilogue, field i >= 1 takes its input and output from the table.
// PAIR: grid z = 1 is the second direction of a paired launch, whose fields
// follow the first direction's in the table.
template <typename T, int EPI, bool PAIR = false>
__device__ __forceinline__ void select_field(const LineFields &mf, const T *__restrict__ &f, EpiArgs &e)
{
    const int i = PAIR ? blockIdx.y + gridDim.y * blockIdx.z : blockIdx.y;
    if constexpr (EPI == EPI_ART_MULTI) e = e.multi[i];
    if (i == 0) return;
    f = (const T *)mf.in[i];
    if constexpr (EPI == EPI_LSRK || EPI == EPI_LSRK_DEV) {
        const int64_t o = mf.eoff[i];
        if (e.a0) e.a0 = (const T *)e.a0 + o;
        e.du += o;
        e.Q += o;
    } else if constexpr (EPI != EPI_ART_MULTI) {
        e.out = mf.out[i];
    }
}

// ---------------------------------------------------------------------------
// Per-thread chunk machinery
// ---------------------------------------------------------------------------
// Interior RHS of one row from the window fv (centre index c):
// a0 f_c + sum_m c_m (f_{c+m} + f_{c-m}) (symmetric) or
// sum_m c_m (f_{c+m} - f_{c-m}), summed left to right, one fma per term.
template <typename T, int M, int SYM, int W>
__device__ __forceinline__ T rhs_row(const T (&fv)[W], int c, const T (&ci)[M], T a0)
{
    T acc;
    if constexpr (SYM) {
        acc = a0 * fv[c];
#pragma unroll
        for (int m = 1; m <= M; m++) acc = fma(ci[m - 1], fv[c + m] + fv[c - m], acc);
    } else {
        acc = ci[0] * (fv[c + 1] - fv[c - 1]);
#pragma unroll
        for (int m = 2; m <= M; m++) acc = fma(ci[m - 1], fv[c + m] - fv[c - m], acc);
    }
    return acc;
}

// RHS of every row of a chunk from its window fv[t + M] = f[s + t]; rows past
// the chunk's length are zero.  At a closed line's ends (first, last: the lane
// holds that chunk) the closure rows replace the first and last nc rows, from
// fv and from fe[kap] = f[n - 1 - kap].  tmin: the fewest points of a chunk of
// this launch that the compiler may count on.  MUNI: p.m is wave-uniform (the
// last chunk holds p.m points, so its closure rows sit at wave-uniform t).
template <typename T, int M, int SYM, int CL, bool FULL, bool MUNI, int TMIN>
__device__ __forceinline__ void chunk_rhs(const LineDev &p, const T (&fv)[CL + 2 * M], const T (&fe)[8], bool first,
                                          bool last, int len, T (&d)[CL])
{
    const T *cf = coefp<T>(p);
    auto ld = [](const T *q) {
        if constexpr (MUNI) return cload(q);
        else return gload(q);
    };
    T ci[M];
#pragma unroll
    for (int m = 0; m < M; m++) ci[m] = ld(cf + COEF_CI + m);
    const T a0 = ld(cf + COEF_A0);
#pragma unroll
    for (int t = 0; t < CL; t++) {
        d[t] = rhs_row<T, M, SYM>(fv, t + M, ci, a0);
        if (!FULL && t >= TMIN) d[t] = t < len ? d[t] : T(0);
    }
    if (!p.closed) return;
#pragma unroll
    for (int t = 0; t < NCMAX; t++) {
        if (t >= p.nc) continue;
        const T *cr = cf + COEF_CLO + t * 8;
        T acc = ld(cr) * fv[M];
#pragma unroll
        for (int kap = 1; kap < 8; kap++) {
            // points past a line shorter than the stencil take a zero weight
            const T fk = kap < p.n ? fv[kap + M] : T(0);
            acc = fma(ld(cr + kap), fk, acc);
        }
        d[t] = first ? acc : d[t];
    }
    if constexpr (MUNI) {
#pragma unroll
        for (int t = 0; t < CL; t++) {
            const int jr = p.m - 1 - t;
            if (jr < 0 || jr >= p.nc) continue;
            const T *cr = cf + COEF_CHI + jr * 8;
            T acc = ld(cr) * fe[0];
#pragma unroll
            for (int kap = 1; kap < 8; kap++) acc = fma(ld(cr + kap), fe[kap], acc);
            d[t] = last ? acc : d[t];
        }
    } else {
#pragma unroll
        for (int jr = 0; jr < NCMAX; jr++) {
            if (jr >= p.nc) continue;
            const T *cr = cf + COEF_CHI + jr * 8;
            T acc = ld(cr) * fe[0];
#pragma unroll
            for (int kap = 1; kap < 8; kap++) acc = fma(ld(cr + kap), fe[kap], acc);
            const int at = last ? len - 1 - jr : -1;
#pragma unroll
            for (int t = 0; t < CL; t++) d[t] = t == at ? acc : d[t];
        }
    }
}

// Chunk sweeps (src/tridiag.jl:46-57, src/banded.jl:63-80) over all CL rows:
// rows past the chunk's length hold zeros and multiply by zeros.  The row
// constants are read G rows at a time: the loads of group g + 1 are issued once
// the arithmetic of group g - 1 is done and before that of group g, so each
// group waits for one round trip while two groups are held in registers.
template <typename T, int Q, int CL, int G, typename Rows>
__device__ __forceinline__ void solve_padded(T (&d)[CL], Rows R)
{
    constexpr int NG = CL / G;
    constexpr int NL = Q, NU = Q == 1 ? 2 : 3;
    const int fl[2] = {Q == 1 ? (int)R1_L : (int)R2_L1, (int)R2_L2};
    const int fu[3] = {Q == 1 ? (int)R1_DINV : (int)R2_U0INV, Q == 1 ? (int)R1_C : (int)R2_U1, (int)R2_U2};
    T c[NL][G], nx[NL][G];
#pragma unroll
    for (int f = 0; f < NL; f++)
#pragma unroll
        for (int i = 0; i < G; i++) c[f][i] = R(fl[f], i);
#pragma unroll
    for (int g = 0; g < NG; g++) {
        if (g + 1 < NG) {
            if (g > 0) R.fence(d[g * G - 1]);
#pragma unroll
            for (int f = 0; f < NL; f++)
#pragma unroll
                for (int i = 0; i < G; i++) nx[f][i] = R(fl[f], (g + 1) * G + i);
        }
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int t = g * G + i;
            if constexpr (Q == 1) {
                if (t >= 1) d[t] = fma(-c[0][i], d[t - 1], d[t]);
            } else {
                if (t + 1 < CL) d[t + 1] = fma(-c[0][i], d[t], d[t + 1]);
                if (t + 2 < CL) d[t + 2] = fma(-c[1][i], d[t], d[t + 2]);
            }
        }
        if (g + 1 < NG) {
#pragma unroll
            for (int f = 0; f < NL; f++)
#pragma unroll
                for (int i = 0; i < G; i++) c[f][i] = nx[f][i];
        }
    }
    T u[NU][G], nu[NU][G];
    R.fence(d[CL - 1]);
#pragma unroll
    for (int f = 0; f < NU; f++)
#pragma unroll
        for (int i = 0; i < G; i++) u[f][i] = R(fu[f], (NG - 1) * G + i);
#pragma unroll
    for (int g = NG - 1; g >= 0; g--) {
        if (g > 0) {
            if (g < NG - 1) R.fence(d[(g + 1) * G]);
#pragma unroll
            for (int f = 0; f < NU; f++)
#pragma unroll
                for (int i = 0; i < G; i++) nu[f][i] = R(fu[f], (g - 1) * G + i);
        }
#pragma unroll
        for (int i = G - 1; i >= 0; i--) {
            const int t = g * G + i;
            T acc = d[t];
            if (t + 1 < CL) acc = fma(-u[1][i], d[t + 1 < CL ? t + 1 : t], acc);
            if constexpr (Q == 2)
                if (t + 2 < CL) acc = fma(-u[2][i], d[t + 2 < CL ? t + 2 : t], acc);
            d[t] = acc * u[0][i];
        }
        if (g > 0) {
#pragma unroll
            for (int f = 0; f < NU; f++)
#pragma unroll
                for (int i = 0; i < G; i++) u[f][i] = nu[f][i];
        }
    }
}

// The 2Q end values of a chunk of len points (TMIN as in chunk_rhs).
template <typename T, int Q, int CL, bool FULL, int TMIN>
__device__ __forceinline__ void chunk_ends(const T (&d)[CL], int len, double (&r)[2 * Q])
{
#pragma unroll
    for (int i = 0; i < Q; i++) {
        r[i] = (double)d[i];
        if constexpr (FULL) {
            r[Q + i] = (double)d[CL - Q + i];
        } else {
            constexpr int T0 = TMIN - Q > 0 ? TMIN - Q : 0;
            T x = d[T0];
#pragma unroll
            for (int t = T0 + 1; t < CL; t++) {
                // the value is read before the choice: a choice between
                // addresses would put the whole chunk into scratch memory
                const T y = d[t];
                x = t == len - Q + i ? y : x;
            }
            r[Q + i] = (double)x;
        }
    }
}

// x = y - V tail_prev - W head_next (src/tridiag.jl:159-168, src/banded.jl:
// 371-382) for every row, the FP64 spike rows read G at a time; put(t, value)
// takes each row.
template <typename T, int Q, int CL, int G, typename R64, typename Put>
__device__ __forceinline__ void correct_padded(T (&d)[CL], R64 R, const double (&tp)[Q], const double (&hn)[Q], Put put)
{
#pragma unroll
    for (int g = 0; g < CL / G; g++) {
        if (g > 0) R.fence(d[g * G - 1]);
        double c[2 * Q][G];
#pragma unroll
        for (int i = 0; i < G; i++) {
            c[0][i] = R(Q == 1 ? (int)R1_V : (int)R2_V0, g * G + i);
            c[1][i] = R(Q == 1 ? (int)R1_W : (int)R2_W0, g * G + i);
            if constexpr (Q == 2) {
                c[2][i] = R(R2_V1, g * G + i);
                c[3][i] = R(R2_W1, g * G + i);
            }
        }
#pragma unroll
        for (int i = 0; i < G; i++) {
            const int t = g * G + i;
            double acc = fma(c[1][i], hn[0], c[0][i] * tp[0]);
            if constexpr (Q == 2) {
                acc = fma(c[2][i], tp[1], acc);
                acc = fma(c[3][i], hn[1], acc);
            }
            d[t] = (T)((double)d[t] - acc);
            put(t, d[t]);
        }
    }
}

// Reduced interface system: block PCR across the P chunks of each line
// (slot = chunk * nl + line-in-block), then fetch the previous chunk's tail
// and the next chunk's head.  Every thread of the block must call this.
// PF: each step's coefficient blocks are loaded one step ahead, before the
// exchange through LDS (the barriers wait for LDS traffic only), so their
// latency overlaps the exchange; for per-lane chunk indices (the x sweep).
// UNI: k is wave-uniform (scalar loads).  The blocks of inner chunks are the
// same block of the table (LineDev::pcr), so the lanes of a wave read a few.
//
// The plan leaves out steps whose coefficients are below rounding, but a NaN or
// an infinity still has to reach its whole line: a chunk whose values are not
// finite (they reach its ends, and z[0] sums every end value) raises its line's
// flag (*bad, which every thread cleared before the first step's barrier: a line
// of several chunks takes one step at least), and a raised flag makes the line
// NaN; bad[64] takes what the others write.  No branch, and nothing kept in
// registers for it: flags per wave and a branch to look for the line cost the
// y / z sweeps a block per CU (C6 derivative of 160^3 FP32 11.8 / 16.0 us).
constexpr int XCH_FLAGS = 64;   // doubles of flags before a block's exchange buffers

template <int Q, bool PF = false, bool UNI = false>
__device__ __forceinline__ void reduced_solve(const LineDev &p, double *buf, int NT, int nl, int k, int li,
                                              double (&r)[2 * Q], double (&tp)[Q], double (&hn)[Q], int *bad)
{
    constexpr int B = 2 * Q;
    const int P = p.P;
    const int slot = k * nl + li;
    const double *pc = p.pcr;
    auto ld = [](const auto *q) {
        if constexpr (UNI) return cload(q);
        else return gload(q);
    };
    // offsets of this chunk's blocks, one per step and the final one
    const int *ix = p.pidx + k;
    const int last = p.nsteps - 1;
    int at = ld(ix);
    if constexpr (PF) {
        constexpr int C = 2 * B * B;
        // one PCR step: multiplies by the blocks in cur and loads the next
        // step's into nxt (this step's again on the last step: in bounds, unused)
        auto step = [&](int st, double (&cur)[C], double (&nxt)[C]) {
            const int dd = 1 << st;
            // at: the next step's block (this step's again on the last step)
            const double *an = pc + at;
#pragma unroll
            for (int c = 0; c < C; c++) nxt[c] = ld(an + c);
            at = ld(ix + (st + 2 < last ? st + 2 : last) * P);
            double *bf = buf + (st & 1) * B * NT;
#pragma unroll
            for (int c = 0; c < B; c++) bf[c * NT + slot] = r[c];
            __syncthreads();
            int km = k - dd, kp = k + dd;
            bool hm = true, hp = true;
            if (p.periodic) {
                km &= (P - 1);
                kp &= (P - 1);
            } else {
                hm = km >= 0;
                hp = kp < P;
            }
            double rm[B], rp[B];
#pragma unroll
            for (int c = 0; c < B; c++) {
                rm[c] = hm ? bf[c * NT + km * nl + li] : 0.0;
                rp[c] = hp ? bf[c * NT + kp * nl + li] : 0.0;
            }
#pragma unroll
            for (int i = 0; i < B; i++) {
                double acc = r[i];
#pragma unroll
                for (int j = 0; j < B; j++) {
                    acc = fma(cur[i * B + j], rm[j], acc);
                    acc = fma(cur[B * B + i * B + j], rp[j], acc);
                }
                r[i] = acc;
            }
        };
        double ca[C], cb[C];
        if (p.nsteps > 0) {
            const double *a0 = pc + at;
#pragma unroll
            for (int c = 0; c < C; c++) ca[c] = ld(a0 + c);
            at = ld(ix + (last > 0 ? 1 : 0) * P);
        }
        // two steps per trip, so the prefetch buffers alternate without copies
        for (int st = 0; st < p.nsteps; st += 2) {
            step(st, ca, cb);
            if (st + 1 < p.nsteps) step(st + 1, cb, ca);
        }
    } else {
        for (int st = 0, dd = 1; st < p.nsteps; st++, dd <<= 1) {
            double *bf = buf + (st & 1) * B * NT;
#pragma unroll
            for (int c = 0; c < B; c++) bf[c * NT + slot] = r[c];
            __syncthreads();
            int km = k - dd, kp = k + dd;
            bool hm = true, hp = true;
            if (p.periodic) {
                km &= (P - 1);
                kp &= (P - 1);
            } else {
                hm = km >= 0;
                hp = kp < P;
            }
            double rm[B], rp[B];
#pragma unroll
            for (int c = 0; c < B; c++) {
                rm[c] = hm ? bf[c * NT + km * nl + li] : 0.0;
                rp[c] = hp ? bf[c * NT + kp * nl + li] : 0.0;
            }
            const double *al = pc + at;
            const double *be = al + B * B;
            at = ld(ix + (st + 1) * P);
#pragma unroll
            for (int i = 0; i < B; i++) {
                double acc = r[i];
#pragma unroll
                for (int j = 0; j < B; j++) {
                    acc = fma(ld(al + i * B + j), rm[j], acc);
                    acc = fma(ld(be + i * B + j), rp[j], acc);
                }
                r[i] = acc;
            }
        }
    }
    const double *mi = pc + (PF ? ld(ix + p.nsteps * P) : at);
    double z[B];
#pragma unroll
    for (int i = 0; i < B; i++) {
        double acc = 0.0;
#pragma unroll
        for (int j = 0; j < B; j++) acc = fma(ld(mi + i * B + j), r[j], acc);
        z[i] = acc;
    }
    double *bf = buf + (p.nsteps & 1) * B * NT;
#pragma unroll
    for (int c = 0; c < B; c++) bf[c * NT + slot] = z[c];
    bad[__builtin_isfinite(z[0]) ? 64 : 0] = 1;
    __syncthreads();
    int kprev = k - 1, knext = k + 1;
    bool hasp = true, hasn = true;
    if (p.periodic) {
        kprev &= (P - 1);
        knext &= (P - 1);
    } else {
        hasp = kprev >= 0;
        hasn = knext < P;
    }
#pragma unroll
    for (int i = 0; i < Q; i++) {
        tp[i] = hasp ? bf[(Q + i) * NT + kprev * nl + li] : 0.0;
        hn[i] = hasn ? bf[i * NT + knext * nl + li] : 0.0;
    }
    tp[0] = *bad ? (double)__builtin_nanf("") : tp[0];
}

// ---------------------------------------------------------------------------
// y / z sweeps, one chunk per wave: 64 lanes along x with V adjacent lines per
// lane, so a row is one contiguous segment of 64 V values and every per-row
// constant is wave-uniform.
//
// Bound: HBM for FP64 and large FP32 grids, instruction issue before that.  The
// row constants come from chunk blocks padded with zeros (LineDev::rows64),
// so the sweeps run CL unconditional steps: a row past the chunk's length only
// multiplies by zeros, and the last row's coupling is stored as zero.  Every
// window load is unconditional too, from the row wrapped or clamped into the
// line (scalar arithmetic), and the closure rows, the zero halo of a closed
// line and the ends of a chunk shorter than CL are fixed up in branches that
// only their own waves take.  FULL: every chunk holds CL points.
//
// V = 2 (float): two lines per lane make the row segments 512 bytes, as for
// double, and halve the instructions per point.
//
// The C6 store kernel of 32-point chunks went from 4777 to 1237 instructions
// (2375 with uneven chunks).  Measured before / after, one pass: C6 gradient of
// 384^3 FP32 665 / 578 us, in-place C8 filter of 256 x 255 x 257 FP64 185 / 176
// us, C10 gradient of 250 x 199 x 180 FP32 256 / 224 us; 40 Taylor-Green steps
// at 64^3 FP64 31.9 / 28.7 ms, 120 x 97 x 81 FP32 81.8 / 73.4 ms.  The
// capacities 12 and 24 (LineDev::cap) between 8, 16 and 32 save the steps and
// registers of half-empty chunks: C6 gradient of 384^3 FP32 (24-point chunks)
// 384 / 342 us.
// ---------------------------------------------------------------------------
// Blocks are dispatched round-robin over the 8 XCDs, each with its own L2;
// renumbered so that every XCD sweeps one contiguous slab.  For y sweeps, whose
// blocks share memory rows, this is the better order (four-field C6 derivative
// at 256^3 FP64: 226 us round-robin, 201 us in slabs); z sweeps, whose
// neighbouring blocks are adjacent in memory, keep the dispatch order (a copy
// with their access pattern takes 196 us so and 208 us in slabs).
__device__ __forceinline__ unsigned xcd_slab(unsigned b, unsigned nb)
{
    const unsigned nfull = nb & ~7u;
    return b < nfull ? (b & 7u) * (nfull >> 3) + (b >> 3) : b;
}

// V adjacent values as one access; elements are only element-aligned (odd
// strides and halos), which the memory unit takes for global accesses.
template <typename T, int V> struct Pack {
    typedef T type __attribute__((ext_vector_type(V), aligned(sizeof(T))));
};
template <int V, typename T> __device__ __forceinline__ void vload(const T *ptr, T (&v)[V])
{
    if constexpr (V == 1) {
        v[0] = *ptr;
    } else {
        const typename Pack<T, V>::type x = *(const typename Pack<T, V>::type *)ptr;
#pragma unroll
        for (int i = 0; i < V; i++) v[i] = x[i];
    }
}
template <int V, typename T> __device__ __forceinline__ void vstore(T *ptr, const T (&v)[V])
{
    if constexpr (V == 1) {
        *ptr = v[0];
    } else {
        typename Pack<T, V>::type x;
#pragma unroll
        for (int i = 0; i < V; i++) x[i] = v[i];
        *(typename Pack<T, V>::type *)ptr = x;
    }
}

// The epilogue of NB rows of V adjacent points: element o[i] .. o[i] + V - 1
// takes v[.][i].  Every input is loaded before any output is stored.  Row i is
// stored where ok[i] (wave-uniform); the offsets of other rows are in bounds.
template <typename T, int EPI, int NB, int V>
__device__ __forceinline__ void epilogue_rows(const EpiArgs &e, const int64_t (&o)[NB], const T (&v)[V][NB],
                                              const bool (&ok)[NB])
{
    if constexpr (EPI == EPI_ART_MULTI) {
        if (e.kind == EPI_ART_MUBETA) epilogue_rows<T, EPI_ART_MUBETA, NB, V>(e, o, v, ok);
        else if (e.kind == EPI_ART_KAPPA) epilogue_rows<T, EPI_ART_KAPPA, NB, V>(e, o, v, ok);
        else epilogue_rows<T, EPI_ART_D, NB, V>(e, o, v, ok);
        return;
    }
    if constexpr (EPI == EPI_STORE || EPI == EPI_STORE_NEG) {
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
            T x[V];
#pragma unroll
            for (int j = 0; j < V; j++) x[j] = EPI == EPI_STORE_NEG ? -v[j][i] : v[j][i];
            vstore<V>((T *)e.out + o[i], x);
        }
    } else if constexpr (EPI == EPI_SUB) {
        T a[NB][V];
#pragma unroll
        for (int i = 0; i < NB; i++) vload<V>((const T *)e.out + o[i], a[i]);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
#pragma unroll
            for (int j = 0; j < V; j++) a[i][j] = a[i][j] - v[j][i];
            vstore<V>((T *)e.out + o[i], a[i]);
        }
    } else if constexpr (EPI == EPI_LSRK) {
        const T *acc = (const T *)e.a0;
        T a[NB][V];
        double du[NB][V], q[NB][V];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (acc) vload<V>(acc + o[i], a[i]);
            if (e.c0 != 0.0) {
                vload<V>((const double *)e.du + o[i], du[i]);
            } else {   // the first stage (A = 0) does not read the register
#pragma unroll
                for (int j = 0; j < V; j++) du[i][j] = 0.0;
            }
            vload<V>((const double *)e.Q + o[i], q[i]);
        }
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
#pragma unroll
            for (int j = 0; j < V; j++) {
                const double dq = acc ? (double)(a[i][j] - v[j][i]) : -(double)v[j][i];
                du[i][j] = fma(e.dt, dq, e.c0 * du[i][j]);
                q[i][j] = fma(e.c1, du[i][j], q[i][j]);
            }
            vstore<V>(e.du + o[i], du[i]);
            vstore<V>(e.Q + o[i], q[i]);
        }
    } else if constexpr (EPI == EPI_ART_MUBETA) {
        T r[NB][V];
#pragma unroll
        for (int i = 0; i < NB; i++) vload<V>((const T *)e.a0 + o[i], r[i]);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
            T mu[V], be[V];
#pragma unroll
            for (int j = 0; j < V; j++) {
                const T rs = r[i][j] * (v[j][i] > T(0) ? v[j][i] : T(0));
                mu[j] = (T)e.c0 * rs;
                be[j] = (T)e.c1 * rs;
            }
            vstore<V>((T *)e.out + o[i], mu);
            vstore<V>((T *)e.out2 + o[i], be);
        }
    } else if constexpr (EPI == EPI_ART_KAPPA) {
        T r[NB][V], cc[NB][V], tt[NB][V];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            vload<V>((const T *)e.a0 + o[i], r[i]);
            vload<V>((const T *)e.a1 + o[i], cc[i]);
            vload<V>((const T *)e.a2 + o[i], tt[i]);
        }
        const T eps = sizeof(T) == 8 ? (T)2.220446049250313e-16 : (T)1.1920929e-07f;
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
            T ka[V];
#pragma unroll
            for (int j = 0; j < V; j++) {
                const T scale = r[i][j] * cc[i][j] / (tt[i][j] > eps ? tt[i][j] : eps);
                ka[j] = (T)e.c0 * scale * (v[j][i] > T(0) ? v[j][i] : T(0));
            }
            vstore<V>((T *)e.out + o[i], ka);
        }
    } else if constexpr (EPI == EPI_ART_D) {
        T cc[NB][V];
#pragma unroll
        for (int i = 0; i < NB; i++) vload<V>((const T *)e.a1 + o[i], cc[i]);
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (!ok[i]) continue;
            T dd[V];
#pragma unroll
            for (int j = 0; j < V; j++) dd[j] = (T)e.c0 * cc[i][j] * (v[j][i] > T(0) ? v[j][i] : T(0));
            vstore<V>((T *)e.out + o[i], dd);
        }
    } else {
        // gated kinds: the flag and dt of the launch, or of each point's instance
#pragma unroll
        for (int j = 0; j < V; j++) {
            int64_t oj[NB];
            T vj[NB];
#pragma unroll
            for (int i = 0; i < NB; i++) {
                oj[i] = o[i] + j;
                vj[i] = v[j][i];
            }
            epilogue_batch<T, EPI, NB>(e, oj, vj, ok);
        }
    }
}

//
// One block; nb: the blocks of its direction.
template <typename T, int Q, int M, int SYM, int EPI, int CL, bool FULL, int V>
__device__ __forceinline__ void line_yzu(const LineDev &p, const T *__restrict__ f, int sd, int64_t so, int nlane,
                                         int nxb, int slabs, unsigned nb, const EpiArgs &e)
{
    extern __shared__ double smem[];
    constexpr int B = 2 * Q;
    const int P = p.P, n = p.n;
    const int NT = 64 * P;
    const int lane = (int)(threadIdx.x & 63);
#pragma unroll
    for (int j = 0; j < V; j++) ((int *)(smem + XCH_FLAGS * j))[lane] = 0;
    const int k = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned blk = slabs ? xcd_slab(blockIdx.x, nb) : blockIdx.x;
    const int xb = blk % nxb;
    const int64_t ob = blk / nxb;
    const int x0 = (xb * 64 + lane) * V;
    const bool valid = x0 < nlane;                  // nlane is a multiple of V
    const int xi = valid ? x0 : nlane - V;
    const int64_t off = ob * so;
    const T *fl = f + off;
    const int s = FULL ? k * CL : k * p.m + min(k, p.extra);
    const int len = FULL ? CL : p.m + (k < p.extra ? 1 : 0);
    const bool lo = p.closed && k == 0, hi = p.closed && k == P - 1;

    T fv[V][CL + 2 * M];
#pragma unroll
    for (int t = -M; t < CL + M; t++) {
        // the wrapped row, or for a closed line any row of it (fixed up below)
        int r = s + t;
        if (t < 0) r = r < 0 ? r + n : r;
        if (!FULL || t >= CL) r = r >= n ? r - n : r;
        if (!FULL) r = r >= n ? n - 1 : r;          // rows past a short last chunk
        T x[V];
        vload<V>(fl + (int64_t)r * sd + xi, x);
#pragma unroll
        for (int j = 0; j < V; j++) fv[j][t + M] = x[j];
    }
    if (lo) {
#pragma unroll
        for (int t = 0; t < M; t++)
#pragma unroll
            for (int j = 0; j < V; j++) fv[j][t] = T(0);
    }
    if (hi) {
#pragma unroll
        for (int t = 0; t < CL + M; t++)
#pragma unroll
            for (int j = 0; j < V; j++) fv[j][t + M] = t >= len ? T(0) : fv[j][t + M];
    }

    const T *cf = coefp<T>(p);
    T d[V][CL];
    {
        T ci[M];
#pragma unroll
        for (int m = 0; m < M; m++) ci[m] = cload(cf + COEF_CI + m);
        const T a0 = cload(cf + COEF_A0);
#pragma unroll
        for (int j = 0; j < V; j++)
#pragma unroll
            for (int t = 0; t < CL; t++) d[j][t] = rhs_row<T, M, SYM>(fv[j], t + M, ci, a0);
    }
    if (lo) {
#pragma unroll
        for (int t = 0; t < NCMAX; t++) {
            if (t >= p.nc) continue;
            const T *cr = cf + COEF_CLO + t * 8;
#pragma unroll
            for (int j = 0; j < V; j++) {
                T acc = cload(cr) * fv[j][M];
#pragma unroll
                for (int kap = 1; kap < 8; kap++) acc = fma(cload(cr + kap), fv[j][kap + M], acc);
                d[j][t] = acc;
            }
        }
    }
    if (hi) {
        T fe[V][8];
#pragma unroll
        for (int kap = 0; kap < 8; kap++) {
            T x[V];
            vload<V>(fl + (int64_t)(kap < n ? n - 1 - kap : 0) * sd + xi, x);
#pragma unroll
            for (int j = 0; j < V; j++) fe[j][kap] = kap < n ? x[j] : T(0);
        }
#pragma unroll
        for (int jr = 0; jr < NCMAX; jr++) {
            if (jr >= p.nc) continue;
            const T *cr = cf + COEF_CHI + jr * 8;
#pragma unroll
            for (int j = 0; j < V; j++) {
                T acc = cload(cr) * fe[j][0];
#pragma unroll
                for (int kap = 1; kap < 8; kap++) acc = fma(cload(cr + kap), fe[j][kap], acc);
#pragma unroll
                for (int t = 0; t < CL; t++) d[j][t] = t == len - 1 - jr ? acc : d[j][t];
            }
        }
    }

    // chunk sweeps (src/tridiag.jl:46-57, src/banded.jl:63-80)
    const int rows = cload(p.blk + k);
    const T *rw = rowsp<T>(p) + rows;
    if constexpr (Q == 1) {
        const T *rl = rw + R1_L * CL, *rdi = rw + R1_DINV * CL, *rc = rw + R1_C * CL;
#pragma unroll
        for (int t = 1; t < CL; t++)
#pragma unroll
            for (int j = 0; j < V; j++) d[j][t] = fma(-cload(rl + t), d[j][t - 1], d[j][t]);
#pragma unroll
        for (int j = 0; j < V; j++) d[j][CL - 1] *= cload(rdi + CL - 1);
#pragma unroll
        for (int t = CL - 2; t >= 0; t--)
#pragma unroll
            for (int j = 0; j < V; j++) d[j][t] = fma(-cload(rc + t), d[j][t + 1], d[j][t]) * cload(rdi + t);
    } else {
        const T *l1 = rw + R2_L1 * CL, *l2 = rw + R2_L2 * CL, *u0 = rw + R2_U0INV * CL, *u1 = rw + R2_U1 * CL,
                *u2 = rw + R2_U2 * CL;
#pragma unroll
        for (int t = 0; t < CL - 1; t++)
#pragma unroll
            for (int j = 0; j < V; j++) {
                d[j][t + 1] = fma(-cload(l1 + t), d[j][t], d[j][t + 1]);
                if (t + 2 < CL) d[j][t + 2] = fma(-cload(l2 + t), d[j][t], d[j][t + 2]);
            }
#pragma unroll
        for (int t = CL - 1; t >= 0; t--)
#pragma unroll
            for (int j = 0; j < V; j++) {
                T acc = d[j][t];
                if (t + 1 < CL) acc = fma(-cload(u1 + t), d[j][t + 1], acc);
                if (t + 2 < CL) acc = fma(-cload(u2 + t), d[j][t + 2], acc);
                d[j][t] = acc * cload(u0 + t);
            }
    }

    // the reduced system, each of the V lines in its own part of the flags and buffers
    double tp[V][Q], hn[V][Q];
#pragma unroll
    for (int j = 0; j < V; j++) {
        double r[B];
#pragma unroll
        for (int i = 0; i < Q; i++) {
            r[i] = (double)d[j][i];
            r[Q + i] = (double)d[j][CL - Q + i];
        }
        if constexpr (!FULL) {
#pragma unroll
            for (int i = 0; i < Q; i++) {
                T x = d[j][0];
#pragma unroll
                for (int t = 1; t < CL; t++) x = t == len - Q + i ? d[j][t] : x;
                r[Q + i] = (double)x;
            }
        }
        reduced_solve<Q, false, true>(p, smem + XCH_FLAGS * V + (size_t)j * 2 * B * NT, NT, 64, k, lane, r, tp[j],
                                      hn[j], (int *)(smem + XCH_FLAGS * j) + lane);
    }
    if (!valid) return;

    // spike correction, FP64 as the reduced system
    const double *rv = p.rows64 + rows;
    // the Runge-Kutta epilogues hold three inputs per point: four rows at a
    // time where eight would spill
    constexpr int NB = CL % 8 != 0 || ((EPI == EPI_LSRK || EPI == EPI_LSRK_DEV) && (CL > 16 || V > 1)) ? 4 : 8;
#pragma unroll
    for (int b = 0; b < CL; b += NB) {
        int64_t o[NB];
        T v[V][NB];
        bool ok[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int t = b + i;
            ok[i] = FULL || t < len;
            const int r = FULL ? s + t : min(s + t, n - 1);
            o[i] = off + (int64_t)r * sd + xi;
#pragma unroll
            for (int j = 0; j < V; j++) {
                double acc;
                if constexpr (Q == 1) {
                    acc = fma(cload(rv + R1_W * CL + t), hn[j][0], cload(rv + R1_V * CL + t) * tp[j][0]);
                } else {
                    acc = cload(rv + R2_V0 * CL + t) * tp[j][0];
                    acc = fma(cload(rv + R2_W0 * CL + t), hn[j][0], acc);
                    acc = fma(cload(rv + R2_V1 * CL + t), tp[j][1], acc);
                    acc = fma(cload(rv + R2_W1 * CL + t), hn[j][1], acc);
                }
                v[j][i] = (T)((double)d[j][t] - acc);
            }
        }
        epilogue_rows<T, EPI, NB, V>(e, o, v, ok);
    }
}

// Waves per SIMD that a variant is held to: those of uneven 24-point chunks lie
// at 78 to 84 registers, and 80 still let a CU take three blocks instead of two
// (C4 derivative of 192^3 FP64: 20.0 us at 79, 22.9 at 81).
template <typename T, int Q, int M, int EPI, int CL, bool FULL, int V> constexpr int yzu_waves()
{
    constexpr bool store24 = CL == 24 && !FULL && (EPI == EPI_STORE || EPI == EPI_STORE_NEG);
    if (Q == 2) return store24 ? 6 : 4;
    return store24 && M <= 2 && sizeof(T) * V == 8 ? 6 : 1;
}

template <typename T, int Q, int M, int SYM, int EPI, int CL, bool FULL, int V>
__global__ void __launch_bounds__(1024, (yzu_waves<T, Q, M, EPI, CL, FULL, V>()))
k_line_yzu(LineDev p, const T *__restrict__ f, int sd, int64_t so, int nlane, int nxb, int slabs, EpiArgs e,
           LineFields mf)
{
    select_field<T, EPI>(mf, f, e);
    line_yzu<T, Q, M, SYM, EPI, CL, FULL, V>(p, f, sd, so, nlane, nxb, slabs, gridDim.x, e);
}

// The y (grid z = 0) and z (1) directions in one launch, store epilogue.  A
// kernel of its own, so that plain launches carry neither the second plan's
// arguments nor the choice between the plans (C6 gradient of 33 x 29 x 31 FP64,
// three plain launches: 21.2 us a pass with one kernel for both, 20.5 so).
template <typename T, int Q, int M, int SYM, int CL, bool FULL, int V>
__global__ void __launch_bounds__(1024, (yzu_waves<T, Q, M, EPI_STORE, CL, FULL, V>()))
k_line_yzu_pair(LineDev p1, const T *__restrict__ f, int sd, int64_t so, int nlane, int nxb, int slabs, EpiArgs e,
                LineFields mf, LineSecond two)
{
    select_field<T, EPI_STORE, true>(mf, f, e);
    const bool second = blockIdx.z;
    // the two directions may differ in lines, hence in blocks
    const unsigned nb = (unsigned)nxb * (unsigned)(second ? two.nouter : two.nouter1);
    if (blockIdx.x >= nb) return;
    LineDev p = p1;
    if (second) {
        p = two.p;
        sd = two.sd;
        so = two.so;
        slabs = two.slabs;
    }
    line_yzu<T, Q, M, SYM, EPI_STORE, CL, FULL, V>(p, f, sd, so, nlane, nxb, slabs, nb, e);
}

// ---------------------------------------------------------------------------
// y / z sweeps on narrow blocks: lanes along x.
// Line dimension stride sd, outer dimension stride so; block = Lx lanes x P
// chunks, several chunks per wave: narrow x extents (2-D grids), and lines
// with too many chunks for 64 lanes.
// ---------------------------------------------------------------------------
template <typename T, int Q, int M, int SYM, int EPI, int CL>
__device__ __forceinline__ void line_yz(const LineDev &p, const T *__restrict__ f, int sd, int64_t so, int nlane, int nxb,
                                        int Lx, const EpiArgs &e)
{
    extern __shared__ double smem[];
    const int NT = Lx * p.P;
    const int lane = (int)(threadIdx.x % Lx);
    const int k = (int)(threadIdx.x / Lx);
    ((int *)smem)[lane] = 0;
    const int xb = blockIdx.x % nxb;
    const int64_t ob = blockIdx.x / nxb;
    const int xi = xb * Lx + lane;
    const bool valid = xi < nlane;
    const int64_t off = (int64_t)xi + ob * so;
    const int n = p.n;
    const int s = k * p.m + min(k, p.extra);
    const int len = p.m + (k < p.extra ? 1 : 0);

    T fv[CL + 2 * M];
    // lanes of one wave own different chunks, so branching per load
    // would diverge: every load is unconditional, from the wrapped row
    // clamped into the line (and the last lane of the row set for lanes
    // past it), and its value selected afterwards.  Rows of the line past the
    // chunk's own window stay: the low closure reads up to eight points from
    // the edge, however short the first chunk is
    const T *fa = f + (int64_t)(valid ? xi : nlane - 1) + ob * so;
#pragma unroll
    for (int t = -M; t < CL + M; t++) {
        int r = s + t;
        bool ok = valid;
        if (r < 0) {
            ok = ok && p.periodic;
            r += n;
        } else if (r >= n) {
            ok = ok && p.periodic;
            r -= n;
        }
        const int rc = r < 0 ? 0 : (r > n - 1 ? n - 1 : r);
        const T val = fa[(int64_t)rc * sd];
        fv[t + M] = ok ? val : T(0);
    }
    T fe[8];
#pragma unroll
    for (int kap = 0; kap < 8; kap++) fe[kap] = T(0);
    if (p.closed) {
#pragma unroll
        for (int kap = 0; kap < 8; kap++)
            if (kap < n) fe[kap] = fa[(int64_t)(n - 1 - kap) * sd];
    }

    constexpr int TMIN = CL == 8 ? 1 : CL / 2;
    constexpr int G = CL <= 8 ? CL : 4;
    T d[CL];
    chunk_rhs<T, M, SYM, CL, false, true, TMIN>(p, fv, fe, k == 0, k == p.P - 1, len, d);
    const int blk = p.blk[k];
    solve_padded<T, Q, CL, G>(d, Rows<T, CL, false>{rowsp<T>(p) + blk});
    double r[2 * Q], tp[Q], hn[Q];
    chunk_ends<T, Q, CL, false, TMIN>(d, len, r);
    reduced_solve<Q, Q == 1 && sizeof(T) == 8>(p, smem + XCH_FLAGS, NT, Lx, k, lane, r, tp, hn, (int *)smem + lane);
    if (!valid) return;
    correct_padded<T, Q, CL, G>(d, Rows<double, CL, false>{p.rows64 + blk}, tp, hn, [](int, T) {});
    // the device-dt LSRK epilogue (per-point gate and dt beside three
    // inputs) goes four points at a time at the full capacity (no spills)
    constexpr int NB = EPI == EPI_LSRK_DEV && CL > 16 ? 4 : 8;
#pragma unroll
    for (int b = 0; b < CL; b += NB) {
        int64_t o[NB];
        T v[1][NB];
        bool ok[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            ok[i] = b + i < len;
            o[i] = off + (int64_t)(ok[i] ? s + b + i : s) * sd;
            v[0][i] = d[b + i];
        }
        epilogue_rows<T, EPI, NB, 1>(e, o, v, ok);
    }
}

// Waves per SIMD: three, but the pentadiagonal sweep of 32-point chunks spills 160
// registers there and 64 at two (C10 of 100 x 2000 FP64 along y 42.7 / 28.6 us).
template <int Q, int CL> constexpr int yz_waves() { return Q == 2 && CL > 16 ? 2 : 3; }

template <typename T, int Q, int M, int SYM, int EPI, int CL>
__global__ void __launch_bounds__(512, (yz_waves<Q, CL>())) k_line_yz(LineDev p, const T *__restrict__ f, int sd, int64_t so, int nlane,
                                                    int nxb, int Lx, EpiArgs e, LineFields mf)
{
    select_field<T, EPI>(mf, f, e);
    line_yz<T, Q, M, SYM, EPI, CL>(p, f, sd, so, nlane, nxb, Lx, e);
}

// The y and z directions in one launch, as k_line_yzu_pair.
template <typename T, int Q, int M, int SYM, int CL>
__global__ void __launch_bounds__(512, (yz_waves<Q, CL>())) k_line_yz_pair(LineDev p1, const T *__restrict__ f, int sd, int64_t so,
                                                         int nlane, int nxb, int Lx, EpiArgs e, LineFields mf,
                                                         LineSecond two)
{
    select_field<T, EPI_STORE, true>(mf, f, e);
    const bool second = blockIdx.z;
    if (blockIdx.x >= (unsigned)nxb * (unsigned)(second ? two.nouter : two.nouter1)) return;
    LineDev p = p1;
    if (second) {
        p = two.p;
        sd = two.sd;
        so = two.so;
    }
    line_yz<T, Q, M, SYM, EPI_STORE, CL>(p, f, sd, so, nlane, nxb, Lx, e);
}

// ---------------------------------------------------------------------------
// x sweep, block-wide: lines of more than 64 chunks (or of chunks longer than
// 16 points).  The block stages Lt whole lines in LDS with the M halo points at
// both ends; thread li P + k owns chunk k of line li, so the lanes of a wave
// hold adjacent chunks; results return through the tile.  As in the wave-local
// sweep, no element index is divided by the line length, window reads need no
// wrap test and the sweeps run on zero-padded rows.  60 steps of the 1024 x 512
// shock / interface FP64 and the state's return, this kernel and the narrow y
// sweep on row-major tables / on shared chunk blocks: 84.6 / 80.5 ms.
// ---------------------------------------------------------------------------
template <int XC> __device__ __forceinline__ int xw_slot(int x) { return x + x / XC; }

template <typename T, int Q, int M, int SYM, int EPI, int CL>
__global__ void __launch_bounds__(512, CL <= 8 ? 4 : 1)
k_line_x(LineDev p, const T *__restrict__ f, int64_t sy, int64_t sz, int ny, int64_t nlines, int Lt, int TS, bool overlay,
         EpiArgs e, LineFields mf)
{
    select_field<T, EPI>(mf, f, e);
    extern __shared__ double smem[];
    const int n = p.n, P = p.P;
    const int NT = Lt * P;
    T *tile = (T *)smem;
    // overlay: the exchange buffers share the tile's memory, between barriers
    // of their own (lines that leave no room for both)
    double *buf = overlay ? smem : smem + (((size_t)Lt * TS * sizeof(T) + 7) / 8);
    const int tid = threadIdx.x;
    const int64_t l0 = (int64_t)blockIdx.x * Lt;
    const int left = (int)(nlines - l0 < Lt ? nlines - l0 : Lt);   // lines that exist, >= 1
    const int seg = (n + NT - 1) / NT;
    // element i of this thread: point x = tid + q NT of line lj, segment by segment
    struct Walk {
        int q, lj;
    };
    auto next = [&](Walk &w) {
        const bool turn = w.q + 1 == seg;
        w.q = turn ? 0 : w.q + 1;
        w.lj += turn ? 1 : 0;
    };
    // a launch holds fewer than 2^32 threads, hence fewer lines
    auto line_off = [&](int lj) -> int64_t {
        const uint32_t l = (uint32_t)l0 + (uint32_t)(lj < left ? lj : 0);
        const uint32_t kk = l / (uint32_t)ny;
        return (int64_t)(l - kk * (uint32_t)ny) * sy + (int64_t)kk * sz;
    };
    {
        Walk w{0, 0};
        for (int e0 = 0; e0 < Lt * seg; e0 += CL) {
            T tmp[CL];
            Walk u = w;
#pragma unroll
            for (int i = 0; i < CL; i++) {
                const int x = tid + u.q * NT;
                tmp[i] = f[line_off(u.lj) + (x < n ? x : n - 1)];
                next(u);
            }
#pragma unroll
            for (int i = 0; i < CL; i++) {
                const int x = tid + w.q * NT;
                if (w.lj < Lt && x < n) tile[w.lj * TS + xw_slot<CL>(x + M)] = tmp[i];
                next(w);
            }
        }
        for (int h = tid; h < Lt * 2 * M; h += NT) {
            const int lj = h / (2 * M), hx = h % (2 * M);
            T v = T(0);
            if (p.periodic) v = f[line_off(lj) + (hx < M ? n - M + hx : hx - M)];
            tile[lj * TS + xw_slot<CL>(hx < M ? hx : hx + n)] = v;
        }
    }
    __syncthreads();

    const int k = tid & (P - 1), li = tid / P;
    const int s = k * p.m + min(k, p.extra);
    const int len = p.m + (k < p.extra ? 1 : 0);
    T *trow = tile + li * TS;
    constexpr int TMIN = CL == 8 ? 1 : CL / 2;
    constexpr int G = CL <= 8 ? 8 : 4;
    T d[CL];
    {
        T fv[CL + 2 * M], fe[8];
#pragma unroll
        for (int t = 0; t < CL + 2 * M; t++) fv[t] = trow[xw_slot<CL>(s + t)];
#pragma unroll
        for (int kap = 0; kap < 8; kap++)
            fe[kap] = p.closed && kap < n ? trow[xw_slot<CL>(n - 1 - kap + M)] : T(0);
        chunk_rhs<T, M, SYM, CL, false, true, TMIN>(p, fv, fe, k == 0, k == P - 1, len, d);
    }
    const int blk = p.blk[k];
    solve_padded<T, Q, CL, G>(d, Rows<T, CL, false>{rowsp<T>(p) + blk});
    double r[2 * Q], tp[Q], hn[Q];
    chunk_ends<T, Q, CL, false, TMIN>(d, len, r);
    if (overlay) __syncthreads();
    ((int *)buf)[li] = 0;
    reduced_solve<Q, Q == 1>(p, buf + XCH_FLAGS, NT, Lt, k, li, r, tp, hn, (int *)buf + li);
    // every thread has finished reading the tile before the reduced solve's barrier
    if (overlay) __syncthreads();
    correct_padded<T, Q, CL, G>(d, Rows<double, CL, false>{p.rows64 + blk}, tp, hn, [&](int t, T v) {
        if (t < TMIN || t < len) trow[xw_slot<CL>(s + t + M)] = v;
    });
    __syncthreads();

    Walk w{0, 0};
    for (int e0 = 0; e0 < Lt * seg; e0 += 8) {
        int64_t o[8];
        T v[1][8];
        bool ok[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int x = tid + w.q * NT, xc = x < n ? x : n - 1;
            ok[i] = w.lj < left && x < n;
            o[i] = line_off(w.lj) + xc;
            v[0][i] = tile[(w.lj < Lt ? w.lj : 0) * TS + xw_slot<CL>(xc + M)];
            next(w);
        }
        epilogue_rows<T, EPI, 8, 1>(e, o, v, ok);
    }
}

// ---------------------------------------------------------------------------
// x sweep, wave-local: a line of n <= 64*XCL points is split into P <= 64
// chunks of <= XCL contiguous points; lane (li, k) of a wave owns chunk k of
// line li (64/P lines per wave).  The reduced interface system is solved by
// block PCR through cross-lane shuffles (no LDS tile, no barrier).
// UNIROW: periodic line with equal chunks, so every chunk has the same
// factors, spikes and PCR blocks (those of chunk 0): all per-row constants are
// wave-uniform.
// ---------------------------------------------------------------------------
constexpr int XCL = 16;

// PF: each step's coefficient blocks are loaded one step ahead (per-lane
// chunk indices kc, whose blocks are vector loads), so their latency overlaps
// the previous step's shuffles and products.
// UNI: kc is wave-uniform (scalar loads).
template <int Q, bool PF = false, bool UNI = false>
__device__ __forceinline__ void reduced_solve_wave(const LineDev &p, int k, int kc, int base, double (&r)[2 * Q],
                                                   double (&tp)[Q], double (&hn)[Q])
{
    constexpr int B = 2 * Q;
    const int P = p.P;
    const double *pc = p.pcr;
    auto ld = [](const auto *q) {
        if constexpr (UNI) return cload(q);
        else return gload(q);
    };
    // offsets of this chunk's blocks, one per step and the final one
    const int *ix = p.pidx + kc;
    const int last = p.nsteps - 1;
    int at = ld(ix);
    if constexpr (PF) {
        constexpr int C = 2 * B * B;
        // one PCR step: multiplies by the blocks in cur and loads the next
        // step's into nxt (this step's again on the last step: in bounds, unused)
        auto step = [&](int st, double (&cur)[C], double (&nxt)[C]) {
            const int dd = 1 << st;
            // at: the next step's block (this step's again on the last step)
            const double *an = pc + at;
#pragma unroll
            for (int c = 0; c < C; c++) nxt[c] = ld(an + c);
            at = ld(ix + (st + 2 < last ? st + 2 : last) * P);
            int km = k - dd, kp = k + dd;
            bool hm = true, hp = true;
            if (p.periodic) {
                km &= (P - 1);
                kp &= (P - 1);
            } else {
                hm = km >= 0;
                hp = kp < P;
                km = hm ? km : k;
                kp = hp ? kp : k;
            }
            double rm[B], rp[B];
#pragma unroll
            for (int c = 0; c < B; c++) {
                rm[c] = __shfl(r[c], base + km, 64);
                rp[c] = __shfl(r[c], base + kp, 64);
                if (!hm) rm[c] = 0.0;
                if (!hp) rp[c] = 0.0;
            }
#pragma unroll
            for (int i = 0; i < B; i++) {
                double acc = r[i];
#pragma unroll
                for (int j = 0; j < B; j++) {
                    acc = fma(cur[i * B + j], rm[j], acc);
                    acc = fma(cur[B * B + i * B + j], rp[j], acc);
                }
                r[i] = acc;
            }
        };
        double ca[C], cb[C];
        if (p.nsteps > 0) {
            const double *a0 = pc + at;
#pragma unroll
            for (int c = 0; c < C; c++) ca[c] = ld(a0 + c);
            at = ld(ix + (last > 0 ? 1 : 0) * P);
        }
        // two steps per trip, so the prefetch buffers alternate without copies
        for (int st = 0; st < p.nsteps; st += 2) {
            step(st, ca, cb);
            if (st + 1 < p.nsteps) step(st + 1, cb, ca);
        }
    } else {
        for (int st = 0, dd = 1; st < p.nsteps; st++, dd <<= 1) {
            int km = k - dd, kp = k + dd;
            bool hm = true, hp = true;
            if (p.periodic) {
                km &= (P - 1);
                kp &= (P - 1);
            } else {
                hm = km >= 0;
                hp = kp < P;
                km = hm ? km : k;
                kp = hp ? kp : k;
            }
            double rm[B], rp[B];
#pragma unroll
            for (int c = 0; c < B; c++) {
                rm[c] = __shfl(r[c], base + km, 64);
                rp[c] = __shfl(r[c], base + kp, 64);
                if (!hm) rm[c] = 0.0;
                if (!hp) rp[c] = 0.0;
            }
            const double *al = pc + at;
            const double *be = al + B * B;
            at = ld(ix + (st + 1) * P);
#pragma unroll
            for (int i = 0; i < B; i++) {
                double acc = r[i];
#pragma unroll
                for (int j = 0; j < B; j++) {
                    acc = fma(ld(al + i * B + j), rm[j], acc);
                    acc = fma(ld(be + i * B + j), rp[j], acc);
                }
                r[i] = acc;
            }
        }
    }
    const double *mi = pc + (PF ? ld(ix + p.nsteps * P) : at);
    double z[B];
#pragma unroll
    for (int i = 0; i < B; i++) {
        double acc = 0.0;
#pragma unroll
        for (int j = 0; j < B; j++) acc = fma(ld(mi + i * B + j), r[j], acc);
        z[i] = acc;
    }
    int kprev = k - 1, knext = k + 1;
    bool hasp = true, hasn = true;
    if (p.periodic) {
        kprev &= (P - 1);
        knext &= (P - 1);
    } else {
        hasp = kprev >= 0;
        hasn = knext < P;
        kprev = hasp ? kprev : k;
        knext = hasn ? knext : k;
    }
#pragma unroll
    for (int i = 0; i < Q; i++) {
        const double a = __shfl(z[Q + i], base + kprev, 64);
        const double b = __shfl(z[i], base + knext, 64);
        tp[i] = hasp ? a : 0.0;
        hn[i] = hasn ? b : 0.0;
    }
    // a NaN or an infinity reaches its whole line (see reduced_solve)
    const uint64_t bad = (uint64_t)__ballot(!__builtin_isfinite(z[0]));
    if (bad && (bad >> base & (~(uint64_t)0 >> (64 - P)))) tp[0] = __builtin_nan("");
}

// One wave per block, 64/P lines staged in LDS (a pad slot after every XC
// points keeps the chunk-strided reads conflict-free), so global loads and
// stores are contiguous.  XC is the chunk capacity (8, 12 or 16).
//
// Bound: instruction issue before HBM, so every row costs as few instructions
// as it can.  A line's points are dealt to LPL = 8..64 lanes (the power of two
// that holds the line, at most a wave), 64 / LPL lines at a time, so no element
// index is divided by the line length; WIDE (LPL = 64): one line at a time,
// its offset in scalar registers.  The tile row holds the M halo points at both
// ends (wrapped copies, or zeros at closed ends), so window reads need no wrap
// test.  The row constants are zero-padded to XC rows (LineDev::rows64), so the
// sweeps run without length tests.  UNIROW: periodic line of equal
// chunks, whose factors, spikes and PCR blocks are those of chunk 0 (scalar
// loads).  FULL: those chunks hold XC points, which fixes every LDS offset at
// compile time.
//
// The FP32 C6 kernel of equal 12-point chunks went from 7416 to 2224
// instructions.  Measured before / after, one pass (three sweeps): C6 gradient
// of 384^3 FP32 578 / 390 us, C10 gradient of 250 x 199 x 180 FP32 between
// walls 224 / 126 us; 40 Taylor-Green steps at 64^3 FP64 28.7 / 25.6 ms, at
// 120 x 97 x 81 FP32 73.4 / 62.4 ms.
template <typename T, int Q, int M, int SYM, int EPI, bool UNIROW, int XC, bool FULL, bool WIDE>
__global__ void __launch_bounds__(64, 4) k_line_xw(LineDev p, const T *__restrict__ f, int64_t sy, int64_t sz, int ny,
                                                int64_t nlines, int TS, int lsh, EpiArgs e, LineFields mf)
{
    select_field<T, EPI>(mf, f, e);
    extern __shared__ double smem[];
    T *tile = (T *)smem;
    const int P = p.P, n = p.n;
    const int lane = threadIdx.x;
    const int nl = 64 / P;                       // lines of the wave
    // element i of this lane: point x = xl + q lpl of line lj < nl, walked
    // segment by segment (at most XC elements)
    const int lpl = WIDE ? 64 : 1 << lsh, grp = 64 / lpl;
    const int seg = (n + lpl - 1) / lpl;
    const int lsub = WIDE ? 0 : lane >> lsh, xl = lane & (lpl - 1);
    // lane l holds the offset of line l (the first one's for lines that do not
    // exist); WIDE reads it into scalar registers
    const int64_t l0 = (int64_t)blockIdx.x * nl;
    const int left = (int)(nlines - l0 < nl ? nlines - l0 : nl);   // lines that exist, >= 1
    int olo, ohi;
    {
        // a launch holds fewer than 2^32 threads, hence fewer lines
        const uint32_t l = (uint32_t)l0 + (uint32_t)(lane < left ? lane : 0);
        const uint32_t kk = l / (uint32_t)ny;
        const int64_t off = (int64_t)(l - kk * (uint32_t)ny) * sy + (int64_t)kk * sz;
        olo = (int)(uint32_t)off;
        ohi = (int)(off >> 32);
    }
    auto line_off = [&](int lj) -> int64_t {
        uint32_t a;
        int b;
        if constexpr (WIDE) {
            a = (uint32_t)__builtin_amdgcn_readlane(olo, lj);
            b = __builtin_amdgcn_readlane(ohi, lj);
        } else {
            a = (uint32_t)__shfl(olo, lj, 64);
            b = __shfl(ohi, lj, 64);
        }
        return (int64_t)(((uint64_t)(uint32_t)b << 32) | a);
    };
    struct Walk {
        int q, lj;
    };
    auto next = [&](Walk &w) {
        const bool turn = w.q + 1 == seg;
        w.q = turn ? 0 : w.q + 1;
        w.lj += turn ? grp : 0;
    };
    {
        T tmp[XC];
        Walk w{0, lsub};
#pragma unroll
        for (int i = 0; i < XC; i++) {
            const int x = xl + w.q * lpl;
            tmp[i] = f[line_off(w.lj) + (x < n ? x : n - 1)];
            next(w);
        }
        // the M halo points at both ends of each line: wrapped copies, or zeros
        for (int h0 = 0; h0 < nl * 2 * M; h0 += 64) {
            const int h = h0 + lane;
            const int lj = h / (2 * M), hx = h % (2 * M);
            T v = T(0);
            if (p.periodic) {
                const uint32_t a = (uint32_t)__shfl(olo, lj & 63, 64);
                const uint32_t b = (uint32_t)__shfl(ohi, lj & 63, 64);
                v = f[(int64_t)(((uint64_t)b << 32) | a) + (hx < M ? n - M + hx : hx - M)];
            }
            if (lj < nl) tile[lj * TS + xw_slot<XC>(hx < M ? hx : hx + n)] = v;
        }
        w = Walk{0, lsub};
#pragma unroll
        for (int i = 0; i < XC; i++) {
            const int x = xl + w.q * lpl;
            if (w.lj < nl && x < n) tile[w.lj * TS + xw_slot<XC>(x + M)] = tmp[i];
            next(w);
        }
    }
    __syncthreads();
    const int k = lane & (P - 1);
    const int li = lane / P;
    const int s = FULL ? k * XC : k * p.m + min(k, p.extra);
    const int len = FULL ? XC : p.m + (k < p.extra ? 1 : 0);
    T *trow = tile + li * TS;
    // slot of window point t (halo included), t = 0 .. XC + 2 M - 1
    auto slot = [&](int t) { return FULL ? k * (XC + 1) + t + t / XC : xw_slot<XC>(s + t); };
    constexpr int TMIN = XC <= 12 ? 1 : 8;   // the next smaller capacity is 12 (8 for other plans)
    T d[XC];
    {
        T fv[XC + 2 * M], fe[8];
#pragma unroll
        for (int t = 0; t < XC + 2 * M; t++) fv[t] = trow[slot(t)];
#pragma unroll
        for (int kap = 0; kap < 8; kap++)
            fe[kap] = !UNIROW && p.closed && kap < n ? trow[xw_slot<XC>(n - 1 - kap + M)] : T(0);
        LineDev pr = p;
        if constexpr (UNIROW) pr.closed = 0;   // periodic: no closure code
        chunk_rhs<T, M, SYM, XC, FULL, true, TMIN>(pr, fv, fe, k == 0, k == P - 1, len, d);
    }
    // rows per group of per-lane loads: four where two groups of eight spill
    constexpr int G = XC == 12 || (!UNIROW && XC > 8 && (Q == 2 || sizeof(T) == 8)) ? 4 : 8;
    const int blk = UNIROW ? cload(p.blk) : p.blk[k];
    solve_padded<T, Q, XC, G>(d, Rows<T, XC, UNIROW>{rowsp<T>(p) + blk});
    double r[2 * Q], tp[Q], hn[Q];
    chunk_ends<T, Q, XC, FULL, TMIN>(d, len, r);
    reduced_solve_wave<Q, !UNIROW && Q == 1 && sizeof(T) == 8, UNIROW>(p, k, UNIROW ? 0 : k, li * P, r, tp, hn);
    // spike correction; each result goes back to the tile (every window read
    // of the wave is done: the wave runs in step)
    __syncthreads();
    correct_padded<T, Q, XC, G>(d, Rows<double, XC, UNIROW>{p.rows64 + blk}, tp, hn, [&](int t, T v) {
        if (FULL || t < TMIN || t < len) trow[slot(t + M)] = v;
    });
    __syncthreads();
    Walk w{0, lsub};
    constexpr int NB = XC % 8 == 0 ? 8 : 4;
#pragma unroll
    for (int b = 0; b < XC; b += NB) {
        int64_t o[NB];
        T v[1][NB];
        bool ok[NB];
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const int x = xl + w.q * lpl, xc = x < n ? x : n - 1;
            ok[i] = w.lj < left && x < n;
            o[i] = line_off(w.lj) + xc;
            v[0][i] = tile[(w.lj < nl ? w.lj : 0) * TS + xw_slot<XC>(xc + M)];
            next(w);
        }
        epilogue_rows<T, EPI, NB, 1>(e, o, v, ok);
    }
}

// x sweep for periodic lines of 256 points in 16 chunks of 16 (the production
// grids): the same algorithm as k_line_xw with the line length, chunk length,
// lines per wave (NL = 4) and the element-to-line map fixed at compile time, line
// offsets computed once per wave and a mask for the periodic wrap.  Lines of 256
// points between walls take k_line_xw: C6 of 256^3 FP64 109 us with a closed
// variant of this kernel and 106 so, FP32 67 / 50, 256 x 256 FP32 5.4 / 5.8.
template <typename T, int Q, int M, int SYM, int EPI, int NL>
__global__ void __launch_bounds__(64) k_line_xwf(LineDev p, const T *__restrict__ f, int64_t sy, int64_t sz, int ny,
                                                 int64_t nlines, EpiArgs e, LineFields mf)
{
    select_field<T, EPI>(mf, f, e);
    constexpr int P = 64 / NL;            // chunks (lanes) per line
    constexpr int N = XCL * P;            // points per line
    constexpr int TS = N + N / XCL + 1;   // padded tile row
    constexpr int EPL = N / 64;           // staged elements per lane and line
    __shared__ T tile[NL * TS];
    const int lane = threadIdx.x;
    const int64_t l0 = (int64_t)blockIdx.x * NL;
    int64_t loff[NL];
    bool lval[NL];
#pragma unroll
    for (int lj = 0; lj < NL; lj++) {
        const int64_t l = l0 + lj;
        lval[lj] = l < nlines;
        loff[lj] = (l % ny) * sy + (l / ny) * sz;
    }
    {
        T tmp[NL * EPL];
#pragma unroll
        for (int lj = 0; lj < NL; lj++)
#pragma unroll
            for (int q = 0; q < EPL; q++) tmp[lj * EPL + q] = lval[lj] ? f[loff[lj] + lane + 64 * q] : T(0);
#pragma unroll
        for (int lj = 0; lj < NL; lj++)
#pragma unroll
            for (int q = 0; q < EPL; q++) tile[lj * TS + xw_slot<XCL>(lane + 64 * q)] = tmp[lj * EPL + q];
    }
    __syncthreads();
    const int li = lane / P, k = lane % P;
    const int s = k * XCL;
    T *trow = tile + li * TS;
    T fv[XCL + 2 * M];
#pragma unroll
    for (int t = -M; t < XCL + M; t++) {
        fv[t + M] = trow[xw_slot<XCL>((s + t) & (N - 1))];
    }
    T d[XCL];
    {
        const T *cf = coefp<T>(p);
        T ci[M];
#pragma unroll
        for (int m = 0; m < M; m++) ci[m] = cload(cf + COEF_CI + m);
        const T a0 = cload(cf + COEF_A0);
#pragma unroll
        for (int t = 0; t < XCL; t++) d[t] = rhs_row<T, M, SYM>(fv, t + M, ci, a0);
    }
    const int blk = cload(p.blk);
    solve_padded<T, Q, XCL, 8>(d, Rows<T, XCL, true>{rowsp<T>(p) + blk});
    double r[2 * Q], tp[Q], hn[Q];
    chunk_ends<T, Q, XCL, true, XCL>(d, XCL, r);
    reduced_solve_wave<Q, false, true>(p, k, 0, li * P, r, tp, hn);
    __syncthreads();   // all window reads done before the tile is overwritten
    correct_padded<T, Q, XCL, 8>(d, Rows<double, XCL, true>{p.rows64 + blk}, tp, hn,
                                 [&](int t, T v) { trow[xw_slot<XCL>(s + t)] = v; });
    __syncthreads();
#pragma unroll
    for (int lj = 0; lj < NL; lj++) {
#pragma unroll
        for (int q0 = 0; q0 < EPL; q0 += 8) {
            int64_t o[8];
            T v[8];
            bool ok[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int q = q0 + i;
                const bool in = q < EPL && lval[lj];
                const int x = lane + 64 * (q < EPL ? q : 0);
                ok[i] = in;
                o[i] = loff[lj] + x;
                v[i] = tile[lj * TS + xw_slot<XCL>(x)];
            }
            epilogue_batch<T, EPI, 8>(e, o, v, ok);
        }
    }
}

// ---------------------------------------------------------------------------
// Dispatch
// ---------------------------------------------------------------------------
inline size_t lds_limit()
{
    static size_t lim = 0;
    if (!lim) {
        int dev = 0, v = 0;
        (void)hipGetDevice(&dev);
        if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess || v <= 0)
            v = 64 * 1024;
        lim = (size_t)v;
    }
    return lim;
}

template <typename K>
inline void allow_lds(K kern, size_t shm)
{
    if (shm > 64 * 1024)
        CLES_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
}

template <typename T, int Q, int M, int SYM, int EPI>
void launch_variant(const HostPlan &hp, int dim, const View3 &v, const T *f, const EpiArgs &e,
                           hipStream_t st, const LineFields &mf, const HostPlan *hp2)
{
    const unsigned nf = (unsigned)mf.nf;
    const LineDev &p = hp.dev;

    const int P = p.P;
    const size_t lim = lds_limit();
    if (dim == 1 && p.extra == 0 && p.m == XCL && P == 16 && p.periodic) {
        // 256-point lines: four per wave
        const int64_t nlines = v.n[1] * v.n[2];
        const int64_t nblk = (nlines + 3) / 4;
        hipLaunchKernelGGL((k_line_xwf<T, Q, M, SYM, EPI, 4>), dim3((unsigned)nblk, nf), dim3(64), 0, st, p, f,
                           v.s[1], v.s[2], (int)v.n[1], nlines, e, mf);
    } else if (dim == 1 && P <= 64 && p.cap <= XCL) {
        const int64_t nlines = v.n[1] * v.n[2];
        const int nl = 64 / P;
        const int64_t nblk = (nlines + nl - 1) / nl;
        const bool uni = p.periodic && p.extra == 0;
        int lsh = 3;   // lanes per line: the power of two that holds it, 8 .. 64
        while ((1 << lsh) < p.n && lsh < 6) lsh++;
        auto go = [&](auto kern, int xc) {
            const int y = p.n + 2 * M + xc;
            const int TS = y + y / xc + 1;
            const size_t shm = (size_t)nl * TS * sizeof(T);
            hipLaunchKernelGGL(kern, dim3((unsigned)nblk, nf), dim3(64), shm, st, p, f, v.s[1], v.s[2], (int)v.n[1],
                               nlines, TS, lsh, e, mf);
        };
        auto pick = [&](auto xcv) {
            constexpr int XC = xcv.value;
            // plans take capacity 12 from 16 chunks on, hence lines of 129 points or more
            constexpr bool WIDE_ONLY = XC == 12;
            if (uni && lsh == 6 && p.m == XC) go(k_line_xw<T, Q, M, SYM, EPI, true, XC, true, true>, XC);
            else if (uni && (WIDE_ONLY || lsh == 6)) go(k_line_xw<T, Q, M, SYM, EPI, true, XC, false, true>, XC);
            else if (uni) go(k_line_xw<T, Q, M, SYM, EPI, true, XC, false, WIDE_ONLY>, XC);
            else if (WIDE_ONLY || lsh == 6) go(k_line_xw<T, Q, M, SYM, EPI, false, XC, false, true>, XC);
            else go(k_line_xw<T, Q, M, SYM, EPI, false, XC, false, WIDE_ONLY>, XC);
        };
        if (p.cap == 8) pick(std::integral_constant<int, 8>{});
        else if (p.cap == 12) pick(std::integral_constant<int, 12>{});
        else pick(std::integral_constant<int, XCL>{});
    } else if (dim == 1) {
        const int64_t nlines = v.n[1] * v.n[2];
        const int y = p.n + 2 * M + p.cap;
        const int TS = y + y / p.cap + 1;
        auto shm_of = [&](int Lt, bool over = false) {
            const size_t tile = (((size_t)Lt * TS * sizeof(T) + 7) / 8) * 8;
            const size_t bufs = ((size_t)4 * Q * Lt * P + XCH_FLAGS) * sizeof(double);
            return over ? std::max(tile, bufs) : tile + bufs;
        };
        int Lt = 1;
        while (Lt * 2 * P <= 512 && shm_of(Lt * 2) <= 48 * 1024 && Lt < 32) Lt *= 2;
        const bool overlay = shm_of(Lt) > lim;
        if (Lt * P > 512 || shm_of(Lt, overlay) > lim)
            throw Error{CLES_ERR_UNSUPPORTED, "line too long for the x-sweep kernel"};
        const int NT = Lt * P;
        const size_t shm = shm_of(Lt, overlay);
        const int64_t nblk = (nlines + Lt - 1) / Lt;
        auto go = [&](auto kern) {
            allow_lds(kern, shm);
            hipLaunchKernelGGL(kern, dim3((unsigned)nblk, nf), dim3(NT), shm, st, p, f, v.s[1], v.s[2], (int)v.n[1],
                               nlines, Lt, TS, overlay, e, mf);
        };
        if (p.cap == 8)
            go(k_line_x<T, Q, M, SYM, EPI, 8>);
        else if (p.cap == 16)
            go(k_line_x<T, Q, M, SYM, EPI, 16>);
        else
            go(k_line_x<T, Q, M, SYM, EPI, MC>);
    } else {
        const int64_t nlane = v.n[0];
        const int64_t sd = dim == 2 ? v.s[1] : v.s[2];
        const int64_t so = dim == 2 ? v.s[2] : v.s[1];
        // hp2: the z direction (dim is 2) in the same launch, grid z = 1
        // (pairable_lines has checked that it takes the same kernel)
        LineSecond two{};
        if (hp2) {
            two.p = hp2->dev;
            two.sd = (int)v.s[2];
            two.so = v.s[1];
            two.slabs = 0;
            two.nouter = (int)v.n[1];
            two.nouter1 = (int)v.n[2];
        }
        const unsigned nz = hp2 ? 2 : 1;
        const int64_t nouter = dim == 2 ? (hp2 ? std::max(v.n[1], v.n[2]) : v.n[2]) : v.n[1];
        if ((int64_t)(p.n - 1) * sd > INT32_MAX) throw Error{CLES_ERR_UNSUPPORTED, "array too large for 32-bit line offsets"};
        if (nlane >= 48 && 64 * P <= YZU_THREADS) {
            const int NT = 64 * P;
            const bool full = p.extra == 0 && p.m == p.cap && (!hp2 || (two.p.extra == 0 && two.p.m == two.p.cap));
            auto go = [&](auto kern, int V, auto... second) {
                const int nxb = (int)((nlane + 64 * V - 1) / (64 * V));
                const size_t shm = ((size_t)4 * Q * NT + XCH_FLAGS) * V * sizeof(double);
                allow_lds(kern, shm);
                hipLaunchKernelGGL(kern, dim3((unsigned)(nxb * nouter), nf, nz), dim3(NT), shm, st, p, f, (int)sd, so,
                                   (int)nlane, nxb, dim == 2 ? 1 : 0, e, mf, second...);
            };
            auto pick = [&](auto cl, auto vv) {
                if constexpr (EPI == EPI_STORE && !SYM) {
                    if (hp2 && full) return go(k_line_yzu_pair<T, Q, M, SYM, cl.value, true, vv.value>, vv.value, two);
                    if (hp2) return go(k_line_yzu_pair<T, Q, M, SYM, cl.value, false, vv.value>, vv.value, two);
                }
                if (full) go(k_line_yzu<T, Q, M, SYM, EPI, cl.value, true, vv.value>, vv.value);
                else go(k_line_yzu<T, Q, M, SYM, EPI, cl.value, false, vv.value>, vv.value);
            };
            using std::integral_constant;
            auto capd = [&](auto vv) {
                switch (p.cap) {
                case 8: return pick(integral_constant<int, 8>{}, vv);
                case 12: return pick(integral_constant<int, 12>{}, vv);
                case 16: return pick(integral_constant<int, 16>{}, vv);
                case 24: return pick(integral_constant<int, 24>{}, vv);
                default: return pick(integral_constant<int, MC>{}, vv);
                }
            };
            // two lines per lane in FP32 where the launch still has two blocks
            // per CU (the row width must be even)
            bool pairs = false;
            if constexpr (sizeof(T) == 4 && Q == 1) {
                pairs = nlane % 2 == 0 && ((nlane + 127) / 128) * nouter * (int64_t)nf * nz >= 512;
                if (pairs) capd(integral_constant<int, 2>{});
            }
            if (!pairs) capd(integral_constant<int, 1>{});
        } else {
            int Lx = 64;
            while (Lx * P > 512 && Lx > 1) Lx /= 2;
            while (Lx / 2 >= nlane && Lx > 1) Lx /= 2;   // narrow x extents (2-D / 1-D grids)
            // few lines (2-D grids): narrower blocks, down to 8 lanes (64-byte
            // rows), until the launch has two blocks per CU
            while (Lx > 8 && ((nlane + Lx - 1) / Lx) * nouter * (int64_t)nf * nz < 512) Lx /= 2;
            if (Lx * P > 512) throw Error{CLES_ERR_UNSUPPORTED, "line too long for the y/z-sweep kernel"};
            if (p.cap == 12 || p.cap == 24) throw Error{CLES_ERR_INVALID, "plan built for another line kernel"};
            const int NT = Lx * P;
            const int nxb = (int)((nlane + Lx - 1) / Lx);
            const size_t shm = ((size_t)4 * Q * NT + XCH_FLAGS) * sizeof(double);
            auto go = [&](auto kern, auto... second) {
                hipLaunchKernelGGL(kern, dim3((unsigned)(nxb * nouter), nf, nz), dim3(NT), shm, st, p, f, (int)sd, so,
                                   (int)nlane, nxb, Lx, e, mf, second...);
            };
            auto pick = [&](auto cl) {
                if constexpr (EPI == EPI_STORE && !SYM) {
                    if (hp2) return go(k_line_yz_pair<T, Q, M, SYM, cl.value>, two);
                }
                go(k_line_yz<T, Q, M, SYM, EPI, cl.value>);
            };
            if (p.cap == 8) pick(std::integral_constant<int, 8>{});
            else if (p.cap == 16) pick(std::integral_constant<int, 16>{});
            else pick(std::integral_constant<int, MC>{});
        }
    }
    CLES_HIP(hipGetLastError());
}

template <typename T, int Q, int M, int SYM>
void launch_epi(const HostPlan &hp, int dim, const View3 &v, const T *f, const EpiArgs &e, hipStream_t st,
                const LineFields &mf, const HostPlan *hp2)
{
    if constexpr (SYM) {
        switch (e.kind) {
        case EPI_STORE: return launch_variant<T, Q, M, SYM, EPI_STORE>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_STORE_GATE: return launch_variant<T, Q, M, SYM, EPI_STORE_GATE>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_ART_MUBETA: return launch_variant<T, Q, M, SYM, EPI_ART_MUBETA>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_ART_KAPPA: return launch_variant<T, Q, M, SYM, EPI_ART_KAPPA>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_ART_D: return launch_variant<T, Q, M, SYM, EPI_ART_D>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_ART_MULTI: return launch_variant<T, Q, M, SYM, EPI_ART_MULTI>(hp, dim, v, f, e, st, mf, hp2);
        default: break;
        }
    } else {
        switch (e.kind) {
        case EPI_STORE: return launch_variant<T, Q, M, SYM, EPI_STORE>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_STORE_NEG: return launch_variant<T, Q, M, SYM, EPI_STORE_NEG>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_SUB: return launch_variant<T, Q, M, SYM, EPI_SUB>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_LSRK: return launch_variant<T, Q, M, SYM, EPI_LSRK>(hp, dim, v, f, e, st, mf, hp2);
        case EPI_LSRK_DEV: return launch_variant<T, Q, M, SYM, EPI_LSRK_DEV>(hp, dim, v, f, e, st, mf, hp2);
        default: break;
        }
    }
    throw Error{CLES_ERR_UNSUPPORTED, "epilogue not available for this scheme kind"};
}

}  // namespace cles
