// Ragged batch of independent compact lines (one line per instance of a
// batch of one-dimensional problems, each with its own length and plan).
//
// One wave per work item.  The item's 64/P lines (all with P chunks of at
// most RAG_MAX_CHUNK points) are staged in LDS with coalesced loads; lane
// (line, chunk) forms its chunk's RHS from the tile, runs the chunk sweeps,
// solves the reduced interface system by block PCR over cross-lane shuffles
// and applies the spike correction (the same machinery as the x sweep); the
// results return through the tile for coalesced, per-instance epilogues.
// Every line is computed from its own data and plan only, so an instance's
// result does not depend on the other instances of the batch.
#pragma once
#include "cles_line.hpp"

namespace cles {

// Blocks are dispatched round-robin over the 8 XCDs; renumbering them so that
// each XCD takes one contiguous range keeps the nf blocks of one work item
// (same lines, different fields) on one XCD's L2.
__device__ __forceinline__ unsigned rag_block(unsigned b, unsigned nb)
{
    const unsigned nfull = nb & ~7u;
    return b < nfull ? (b & 7u) * (nfull >> 3) + (b >> 3) : b;
}

// One launch for both classes up to this many blocks (waves), four times what
// the long class's registers let run at once (from there on the two launches
// fill the card by themselves and the results are equal): 512 tubes FP64, 1392 to 2784 blocks
// per launch, 131.0 ms per 96 steps with two launches and 105.8 with one for up
// to 2048 blocks; 1024 tubes 1.76 / 1.73 ms per step, 4096 tubes 6.34 / 6.36.
constexpr int64_t RAG_BOTH_BLOCKS = 8192;

// Tile row of a line of at most CL P points with its halo, a pad slot after
// every CL points (xw_slot) and room for the last chunk's window overrun.
template <int CL, int M> __host__ __device__ constexpr int rag_row(int P)
{
    return (CL * P + 2 * M + CL) + (CL * P + 2 * M + CL) / CL + 1;
}

// CL: chunk capacity of the launch's items (RAG_SHORT_CHUNK for the short
// class, RAG_MAX_CHUNK otherwise).
//
// Bound: the latency of one wave's chain (a few thousand lines fill the chip
// less than twice over), so what is waited for counts: the row constants of
// all instances share one pool of distinct chunk blocks (LineDev::rows64), a
// few KB that stay in the nearest cache instead of 40 bytes of tables per
// point; each tile row carries the halo points, so window reads have no wrap
// tests; the sweeps run on zero-padded rows.  96 steps of 512 tubes and their
// states FP64, tables per instance / shared: 163.8 / 133.5 ms.
template <typename T, int Q, int M, int SYM, int EPI, int CL>
__device__ __forceinline__ void rag_item(const RagLines &r, unsigned logical, const T *__restrict__ f, EpiArgs e,
                                         T *tile)
{
    const int lane = threadIdx.x;
    const int item = (int)(logical / (unsigned)r.nf), fld = (int)(logical % (unsigned)r.nf);
    const int64_t fo = (int64_t)fld * r.fstride;
    f += fo;
    if constexpr (EPI == EPI_ART_MULTI) e = e.multi[fld];   // its own outputs: no field offset
    const int *it = r.items + 3 * item;
    const int P = cload(it), start = cload(it + 1), count = cload(it + 2);
    const int TS = rag_row<CL, M>(P);

    // stage the item's lines
    for (int lj = 0; lj < count; lj++) {
        const int inst = cload(r.order + start + lj);
        const int n = r.plans[inst].n;
        const bool per = r.plans[inst].periodic;
        const T *src = f + r.off[inst];
        T *row = tile + lj * TS;
        // a line of up to 64 CL points in one round of CL loads per lane (the
        // registers of the sweeps are not live yet)
        for (int x0 = 0; x0 < n; x0 += 64 * CL) {
            T v[CL];
#pragma unroll
            for (int i = 0; i < CL; i++) {
                const int x = x0 + lane + 64 * i;
                v[i] = x < n ? src[x] : T(0);
            }
#pragma unroll
            for (int i = 0; i < CL; i++) {
                const int x = x0 + lane + 64 * i;
                if (x < n) row[xw_slot<CL>(x + M)] = v[i];
            }
        }
        if (lane < 2 * M) {   // the halo: wrapped copies, or zeros
            const T v = per ? src[lane < M ? n - M + lane : lane - M] : T(0);
            row[xw_slot<CL>(lane < M ? lane : lane + n)] = v;
        }
    }
    __syncthreads();

    // lanes of empty line slots repeat line 0 and store nothing
    const int li = lane / P, k = lane & (P - 1);
    const bool live = li < count;
    const int inst = r.order[start + (live ? li : 0)];
    const LineDev p = r.plans[inst];
    const int n = p.n;
    const int s = k * p.m + min(k, p.extra);
    const int len = p.m + (k < p.extra ? 1 : 0);
    T *trow = tile + (live ? li : 0) * TS;
    constexpr int TMIN = 1;   // a line may be one chunk of a few points
    T d[CL];
    {
        T fv[CL + 2 * M], fe[8];
#pragma unroll
        for (int t = 0; t < CL + 2 * M; t++) fv[t] = trow[xw_slot<CL>(s + t)];
#pragma unroll
        for (int kap = 0; kap < 8; kap++)
            fe[kap] = (p.closed && kap < n) ? trow[xw_slot<CL>(n - 1 - kap + M)] : T(0);
        chunk_rhs<T, M, SYM, CL, false, false, TMIN>(p, fv, fe, k == 0, k == P - 1, len, d);
    }
    const int blk = p.blk[k];
    solve_padded<T, Q, CL, 8>(d, Rows<T, CL, false>{rowsp<T>(p) + blk});
    double ends[2 * Q], tp[Q], hn[Q];
    chunk_ends<T, Q, CL, false, TMIN>(d, len, ends);
    reduced_solve_wave<Q, Q == 1>(p, k, k, li * P, ends, tp, hn);
    __syncthreads();   // every window read is done before the tile is overwritten
    correct_padded<T, Q, CL, 8>(d, Rows<double, CL, false>{p.rows64 + blk}, tp, hn, [&](int t, T v) {
        if (live && t < len) trow[xw_slot<CL>(s + t + M)] = v;
    });
    __syncthreads();

    for (int lj = 0; lj < count; lj++) {
        const int ij = cload(r.order + start + lj);
        if (r.mask && !r.mask[ij]) continue;
        const int nj = r.plans[ij].n;
        const int64_t oj = r.off[ij];
        EpiArgs ej = e;
        if (EPI != EPI_ART_MULTI && fo) {
            if (ej.out) ej.out = (T *)ej.out + fo;
            if (ej.du) ej.du += fo;
            if (ej.Q) ej.Q += fo;
        }
        if (r.dt) ej.dt = r.dt[ij];
        const T *row = tile + lj * TS;
        // at capacity 32, 16 points per lane per batch (the sweeps' registers
        // are free here; at capacity 16 that would raise the allocation)
        constexpr int NB = CL > 16 ? 16 : 8;
        for (int x0 = 0; x0 < nj; x0 += 64 * NB) {
            int64_t o[NB];
            T v[1][NB];
            bool ok[NB];
#pragma unroll
            for (int i = 0; i < NB; i++) {
                const int x = x0 + lane + 64 * i;
                ok[i] = x < nj;
                o[i] = oj + (ok[i] ? x : 0);
                v[0][i] = row[xw_slot<CL>((ok[i] ? x : 0) + M)];
            }
            epilogue_rows<T, EPI, NB, 1>(ej, o, v, ok);
        }
    }
}

template <typename T, int Q, int M, int SYM, int EPI, int CL>
__global__ void __launch_bounds__(64) k_line_rag(RagLines r, const T *__restrict__ f, EpiArgs e)
{
    extern __shared__ double smem[];
    rag_item<T, Q, M, SYM, EPI, CL>(r, rag_block(blockIdx.x, gridDim.x), f, e, (T *)smem);
}

// Both classes in one launch, the longer lines' blocks first (they take
// longest): batches too small to fill the chip with one class at a time run the
// two side by side instead of one after the other.  The short class then has
// the long one's registers and LDS, which is why large batches keep two launches.
template <typename T, int Q, int M, int SYM, int EPI>
__global__ void __launch_bounds__(64) k_line_rag_both(RagLines rs, RagLines rl, const T *__restrict__ f, EpiArgs e)
{
    extern __shared__ double smem[];
    const unsigned nbl = (unsigned)rl.nitems * (unsigned)rl.nf;
    if (blockIdx.x < nbl)
        rag_item<T, Q, M, SYM, EPI, RAG_MAX_CHUNK>(rl, rag_block(blockIdx.x, nbl), f, e, (T *)smem);
    else
        rag_item<T, Q, M, SYM, EPI, RAG_SHORT_CHUNK>(rs, rag_block(blockIdx.x - nbl, gridDim.x - nbl), f, e, (T *)smem);
}

template <typename T, int Q, int M, int SYM, int EPI>
void launch_rag_variant(const RagLines &r, const T *f, const EpiArgs &e, hipStream_t st)
{
    if (r.nshort < 0 || r.nshort > r.nitems) throw Error{CLES_ERR_INVALID, "short items out of range"};
    if (r.nitems <= 0 || r.nf <= 0) return;
    if (r.nf > 1 && e.kind != EPI_STORE && e.kind != EPI_STORE_NEG && e.kind != EPI_LSRK && e.kind != EPI_ART_MULTI)
        throw Error{CLES_ERR_INVALID, "several fields per launch need a store, LSRK or multi epilogue"};
    if (e.kind == EPI_ART_MULTI && !e.multi) throw Error{CLES_ERR_INVALID, "the multi epilogue needs its table"};
    if (e.kind == EPI_LSRK && e.a0 && r.nf > 1)
        throw Error{CLES_ERR_INVALID, "the ragged LSRK epilogue takes no accumulator with several fields"};
    // the short items, then the rest, each with its own chunk capacity
    RagLines rs = r, rl = r;
    rs.nitems = r.nshort;
    rl.items = r.items + 3 * r.nshort;
    rl.nitems = r.nitems - r.nshort;
    const size_t shm_s = (size_t)(64 / r.pmin[0]) * rag_row<RAG_SHORT_CHUNK, M>(r.pmin[0]) * sizeof(T);
    const size_t shm_l = (size_t)(64 / r.pmin[1]) * rag_row<RAG_MAX_CHUNK, M>(r.pmin[1]) * sizeof(T);
    const int64_t blocks = (int64_t)r.nitems * r.nf;
    if (rs.nitems > 0 && rl.nitems > 0 && blocks <= RAG_BOTH_BLOCKS) {
        hipLaunchKernelGGL((k_line_rag_both<T, Q, M, SYM, EPI>), dim3((unsigned)blocks), dim3(64),
                           std::max(shm_s, shm_l), st, rs, rl, f, e);
        CLES_HIP(hipGetLastError());
        return;
    }
    if (rs.nitems > 0) {
        const int64_t nb = (int64_t)rs.nitems * r.nf;
        hipLaunchKernelGGL((k_line_rag<T, Q, M, SYM, EPI, RAG_SHORT_CHUNK>), dim3((unsigned)nb), dim3(64), shm_s, st, rs, f,
                           e);
        CLES_HIP(hipGetLastError());
    }
    if (rl.nitems > 0) {
        const int64_t nb = (int64_t)rl.nitems * r.nf;
        hipLaunchKernelGGL((k_line_rag<T, Q, M, SYM, EPI, RAG_MAX_CHUNK>), dim3((unsigned)nb), dim3(64), shm_l, st, rl, f,
                           e);
        CLES_HIP(hipGetLastError());
    }
}

template <typename T, int Q, int M, int SYM>
void launch_rag_epi(const RagLines &r, const T *f, const EpiArgs &e, hipStream_t st)
{
    if constexpr (SYM) {
        switch (e.kind) {
        case EPI_STORE: return launch_rag_variant<T, Q, M, SYM, EPI_STORE>(r, f, e, st);
        case EPI_ART_MUBETA: return launch_rag_variant<T, Q, M, SYM, EPI_ART_MUBETA>(r, f, e, st);
        case EPI_ART_KAPPA: return launch_rag_variant<T, Q, M, SYM, EPI_ART_KAPPA>(r, f, e, st);
        case EPI_ART_D: return launch_rag_variant<T, Q, M, SYM, EPI_ART_D>(r, f, e, st);
        case EPI_ART_MULTI: return launch_rag_variant<T, Q, M, SYM, EPI_ART_MULTI>(r, f, e, st);
        default: break;
        }
    } else {
        switch (e.kind) {
        case EPI_STORE: return launch_rag_variant<T, Q, M, SYM, EPI_STORE>(r, f, e, st);
        case EPI_STORE_NEG: return launch_rag_variant<T, Q, M, SYM, EPI_STORE_NEG>(r, f, e, st);
        case EPI_LSRK: return launch_rag_variant<T, Q, M, SYM, EPI_LSRK>(r, f, e, st);
        default: break;
        }
    }
    throw Error{CLES_ERR_UNSUPPORTED, "epilogue not available for the ragged line kernel"};
}

}  // namespace cles
