// The conjugate gradient of kernels_cg.hip as one launch: the same preconditioned single-reduction
// recurrence (Chronopoulos and Gear), stopping rule, precision and two-level correction, with the
// iterations run inside a persistent kernel instead of as five launches each.
//
// What bounds a solve of a small or middle-sized system is not the matrix but the chain of dependent
// steps: five kernels of 3-10 us per iteration whose work is a microsecond or two each, and every
// launch starts with cold caches. Here a workgroup of eight wavefronts owns the same 64-row slices for
// the whole solve. Its threads hold their rows' x, r, p, s and diagonal in registers, its part of the
// matrix stays in the XCD's L2 while all of it fits the eight (28 MB; a larger one is streamed past them), and only
// these travel between workgroups, once per iteration
// each: the aggregates' shares of P^T r and the coarse correction, the preconditioned residual u (read by the neighbours' SpMV)
// with the partial sums of (r, u) and (r, r), and the partial sums of (K u, u).
//
// Exchange between workgroups. The eight L2 caches are not coherent with each other, and a fence
// that writes back and invalidates them costs more than a launch. So everything that another
// workgroup reads is stored and loaded at agent scope (relaxed atomics, or buffer loads with the same
// sc1 policy), which goes past the L2, and nothing else is exchanged. A partial sum and the signal
// that it is there are one 8-byte word: slots start as PCG_EMPTY, a workgroup publishes its value
// into its own slot, and readers poll until the word is something else. Before a publication that
// also stands for other data (u, or reset slots), every wavefront waits for its own stores
// (s_waitcnt vmcnt(0)) and the workgroup passes a barrier. Slots come in two sets, used in turn
// by iteration parity; a set is emptied again once every workgroup is known to have read it:
//   C (P^T r)    of iteration k-1 after C of k, since every workgroup published U of k-1 after it,
//   Y (Ac^-1 P^T r) of iteration k-1 before Y of k, for the same reason,
//   U (u, sums)  of iteration k-1 after U of k, since every workgroup published D of k-1 after it,
//   D (K u, u)   of iteration k-1 after D of k, since every workgroup published U of k after it,
// and each emptying is complete before the owner's next publication, which every reader of the
// emptied set waits for first.
//
// Every workgroup adds the same words in the same order, so all reach the same alpha, beta and stop
// decision, and a result does not depend on scheduling.
//
// Time per iteration, launched and here (two-level unless marked; FP32 unless marked):
//   SC 12^3      25.8 -> 14.2 us      hex 200 x 231   26.8 -> 19.7 us    SC 48^3       67.4 -> 61.3 us
//   SC 20^3      30.5 -> 17.7 us      hex 350 x 370   37.2 -> 29.7 us    FCC 24^3      47.4 -> 38.9 us
//   SC 28^3      31.7 -> 23.9 us      SC 16^3 Jacobi  18.5 ->  9.6 us    SC 36^3 FP64  63.8 -> 50.8 us
//   hex 100 x 115, FP64, Jacobi       14.9 -> 9.8 us                     SC 45^3 FP64  91.8 -> 89.4 us
//   SC 50 x 51 x 51 (130,050)         73.9 -> 65.5 us    in FP64 125 -> 114 us, FP64 Jacobi 112 -> 103 us
// The bound of 131,072 rows is that of one row per thread. In 3D in FP64 with Jacobi the two come level at 83,000 to
// 97,000 rows (FCC 27^3 78.1 and 78.4, SC 45^3 77.6 and 80.1, SC 46^3 83.1 and 82.1, BCC 36^3 64.7 and 58.9).
// Of the 19.7 us at hex 200 x 231 (241 workgroups): shares of P^T r 1.3, waiting for them and Ac^-1 6.6,
// correction 0.9, u 1.3, its exchange 4.1, SpMV 2.7, its exchange 2.7. Eight wavefronts of up to
// 256 registers hold a row's state and eight slots in flight; with sixteen of 128 the compiler spilled
// 70-150 registers and the kernel lost to the launches (hex 200 x 231: 31.9-42.6 us).
//
// The grid has at most one workgroup per CU, so all of it is resident: the solves that contexts run at the same time
// from several threads share the CUs out (ResidentCus), and other kernels end. Cooperative launches give the
// same promise, but run one after the other on the device. us per iteration over all of four contexts in threads
// of their own, launch by launch, cooperative, and with the CUs shared out: SC 12^3 8.3, 15.3, 4.0; hex 60 x 60 6.9,
// 12.4, 3.2; SC 20^3 10.5, 17.7, 9.8; SC 40^3, whose grid takes every CU, 29.7, 40.4, 40.9 (one context: 47.2, 40.4, 40.3).
// Every wait is bounded all the same: a workgroup that has polled for cg_wait_ms sets SC_ABORT and
// leaves, the others see it and leave, and the host solves the system again launch by launch, as it does all
// later ones of the context until cg_persist or cg_wait_ms is set again.
#include <algorithm>
#include <cfloat>
#include <condition_variable>
#include <map>
#include <mutex>
#include <vector>

#include "lpm_internal.h"
#include "reduce.h"

namespace {

typedef unsigned long long u64;
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x3 __attribute__((ext_vector_type(3)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr u64 PCG_EMPTY = ~0ull;            // no value yet (a NaN pattern that is never published)
constexpr int PCG_NT = 512, PCG_NW = 8;   // threads and wavefronts of a workgroup
constexpr int PCG_WG = 256;                 // most workgroups: one per CU
constexpr int PCG_SPW = 8;                 // most slices of a workgroup: one row per thread
constexpr int PCG_CZ = 2048;                // most coarse DoFs a workgroup reads
constexpr int PCG_LA = 64;                  // most aggregates of a workgroup's rows
constexpr int PCG_SHARES = 32768;           // most shares of P^T r that a workgroup polls
constexpr int PCG_LAUNCH_ITERS = 1024;      // iterations of one launch (longer solves are continued)

struct PcgArgs {
    int64_t n, nslice;
    int spw, block_pre, coarse, it0, itmax;
    double tol, maxit;
    const int64_t *sp;
    const int32_t *cptr;
    const void *scol, *aval, *invd;
    uint32_t scol_bytes, aval_bytes, u_bytes;
    const double *b64;
    void *x, *r, *u, *p, *s;
    double *scal;
    u64 *slot_c, *slot_y, *slot_u, *slot_d;  // two sets each
    int nslot_c, ncoarse, ndof_wg;  // words of one set of slot_c and of slot_y; coarse DoFs whose rows a workgroup forms
    int ainv_lds;                   // row length of the copy of its rows of Ac^-1 that a workgroup keeps in LDS (0: none)
    u64 wait_ticks;
    const double *agg_d, *Ainv;
    const uint8_t *mask;
    const int32_t *agg_grp, *cb, *ca_cnt;  // ca_cnt: workgroups that share each aggregate
    const int64_t *off;
    // rows of each workgroup by aggregate: its aggregates, its rank among their workgroups, where their
    // rows begin in aggregate order; per row that position and the aggregate's rank, (rank << 16) | position
    const int32_t *wl_ptr, *wl_agg, *wl_slot, *wl_beg, *wpos;
    const int32_t *order;  // slices in the order in which the workgroups take them
};

// Word i of the U and D slots: four words together, 256 B (the interleave of the memory channels)
// from the next four. Every workgroup polls all of them; packed together they are served by few
// channels (wait and sum of D with 241 workgroups: packed 6.1 us, eight words per 256 B 3.1, four
// 2.8; eight words per 4 KB + 256 B 4.3).
constexpr int PCG_LINE = 256 / 8;
__host__ __device__ __forceinline__ constexpr int slot_at(int i) { return (i >> 2) * PCG_LINE + (i & 3); }
constexpr int PCG_SET = slot_at(PCG_WG);  // words of one set of one sum

__device__ __forceinline__ u64 ld_agent(const u64 *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_agent(u64 *p, u64 v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 word_of(double v) {
    const u64 b = (u64)__double_as_longlong(v);
    return b == PCG_EMPTY ? 0x7ff8000000000000ull : b;
}
__device__ __forceinline__ double value_of(u64 b) { return __longlong_as_double((long long)b); }
// this wavefront's stores have reached the agent's point of coherence
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Polls N words until each holds a value (word u is at p + u * stride, for u < have); false when
// the wait was given up (see above).
template <int N>
__device__ __forceinline__ bool slot_wait(const u64 *p, int stride, int have, u64 (&v)[N], const PcgArgs &a) {
    u64 t0 = 0;
    for (int k = 0;; ++k) {
        bool all = true;
#pragma unroll
        for (int u = 0; u < N; ++u) v[u] = u < have ? ld_agent(p + u * stride) : 0ull;
#pragma unroll
        for (int u = 0; u < N; ++u) all = all && v[u] != PCG_EMPTY;
        if (all) return true;
        if ((k & 31) == 31 || a.wait_ticks == 0) {
            u64 *stop = (u64 *)&a.scal[SC_ABORT];
            if (ld_agent(stop) != 0) return false;
            const u64 t = (u64)wall_clock64();
            if (t0 == 0) t0 = t;
            if (t - t0 >= a.wait_ticks) {
                st_agent(stop, word_of(1.0));
                return false;
            }
        }
    }
}

// Buffer loads: an offset past the buffer returns zero, which stands for "no block here".
constexpr uint32_t NO_ELEM = 0xffff0000u;  // stays past every buffer with an element's offset added
constexpr int AUX_SC1 = 16, AUX_NT = 2;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, (int)bytes, 0x00027000);
}

template <typename T, int AUX>
__device__ __forceinline__ T ld_elem(__amdgpu_buffer_rsrc_t b, uint32_t o) {
    if constexpr (sizeof(T) == 4) return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, (int)o, 0, AUX));
    else {
        const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(b, (int)o, 0, AUX);
        return value_of(((u64)w.y << 32) | w.x);
    }
}

// the D entries of a particle in u, past the L2
template <typename T, int D>
__device__ __forceinline__ void ld_u(__amdgpu_buffer_rsrc_t b, uint32_t o, T (&v)[D]) {
    if constexpr (sizeof(T) == 4 && D == 2) {
        const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(b, (int)o, 0, AUX_SC1);
        v[0] = __uint_as_float(w.x);
        v[1] = __uint_as_float(w.y);
    } else if constexpr (sizeof(T) == 4) {
        const u32x3 w = __builtin_amdgcn_raw_buffer_load_b96(b, (int)o, 0, AUX_SC1);
        v[0] = __uint_as_float(w.x);
        v[1] = __uint_as_float(w.y);
        v[2] = __uint_as_float(w.z);
    } else {
        const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(b, (int)o, 0, AUX_SC1);
        v[0] = value_of(((u64)w.y << 32) | w.x);
        v[1] = value_of(((u64)w.w << 32) | w.z);
        if constexpr (D == 3) v[2] = ld_elem<T, AUX_SC1>(b, o + 16);
    }
}

// P^T r and P y of one particle (rigid_modes in reduce.h), written out so that P is never held
template <int D>
__device__ __forceinline__ void modes_t(const double (&d)[D], const double (&r)[D], double (&t)[D == 3 ? 6 : 3]) {
    if constexpr (D == 3) {
        t[0] = r[0];
        t[1] = r[1];
        t[2] = r[2];
        t[3] = d[1] * r[2] - d[2] * r[1];
        t[4] = d[2] * r[0] - d[0] * r[2];
        t[5] = d[0] * r[1] - d[1] * r[0];
    } else {
        t[0] = r[0];
        t[1] = r[1];
        t[2] = d[0] * r[1] - d[1] * r[0];
    }
}

template <int D>
__device__ __forceinline__ void modes(const double (&d)[D], const double *y, double (&t)[D]) {
    if constexpr (D == 3) {
        t[0] = y[0] + d[2] * y[4] - d[1] * y[5];
        t[1] = y[1] + d[0] * y[5] - d[2] * y[3];
        t[2] = y[2] + d[1] * y[3] - d[0] * y[4];
    } else {
        t[0] = y[0] - d[1] * y[2];
        t[1] = y[1] + d[0] * y[2];
    }
}

template <typename T>
__device__ __forceinline__ void st_u(T *p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sums NV values over the workgroup in a fixed order; every thread gets the sums.
template <int NV>
__device__ __forceinline__ void wg_sum(double (&v)[NV], double (*red)[PCG_NW + 1]) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int k = 0; k < NV; ++k) {
        for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_xor(v[k], o, 64);
        if (lane == 0) red[k][wv] = v[k];
    }
    __syncthreads();
    for (int k = 0; k < NV; ++k) {
        double t = 0.0;
        for (int w = 0; w < PCG_NW; ++w) t += red[k][w];
        v[k] = t;
    }
}

template <typename T, int D, typename IX, bool NT>
__global__ __launch_bounds__(PCG_NT) void k_pcg(PcgArgs a) {
    constexpr int M = D == 3 ? 6 : 3, EB = D * D;
    constexpr int UNR = sizeof(T) * EB > 36 ? 4 : 8;  // slots in flight per lane: what the registers hold
    constexpr int AUX = NT ? AUX_NT : 0;
    extern __shared__ double lds[];
    __shared__ double red0[2][PCG_NW + 1], red1[2][PCG_NW + 1], red2[2][PCG_NW + 1], red3[2][PCG_NW + 1];
    __shared__ int gave_up;  // set by a thread whose wait was given up, read behind the next barrier
    if (threadIdx.x == 0) gave_up = 0;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = gridDim.x, wg = (int)xcd_major_block();
    const int64_t k0 = (int64_t)wg * a.spw;
    const int nsl = (int)(a.nslice - k0 < a.spw ? a.nslice - k0 : a.spw);  // >= 1 by the grid's size
    const int nrow_lds = 64 * a.spw;
    // LDS: the SpMV's partial row sums and the rows' shares of P^T r (never live together), cz, y
    T *part = (T *)lds;
    double *share = lds;
    const size_t un = sizeof(T) * PCG_NW * D * 64 > sizeof(double) * M * nrow_lds ? sizeof(T) * PCG_NW * D * 64
                                                                                  : sizeof(double) * M * nrow_lds;
    double *cz = (double *)((char *)lds + un), *ycor = cz + PCG_CZ, *arow = ycor + PCG_LA * M;

    // ---- this thread's row in the vector updates
    const int64_t row = wv < nsl ? (int64_t)a.order[k0 + wv] * 64 + lane : a.n;
    const bool own = row < a.n;
    T x[D], r[D], p[D], s[D], dinv[D];
    double d[D];
    unsigned mk = 0;
    int pos = 0, rank = 0;
    for (int k = 0; k < D; ++k) x[k] = r[k] = p[k] = s[k] = dinv[k] = (T)0, d[k] = 0.0;
    if (own) {
        for (int k = 0; k < D; ++k) {
            if (a.it0 == 0) {
                r[k] = (T)a.b64[D * row + k];
            } else {
                x[k] = ((T *)a.x)[D * row + k];
                r[k] = ((T *)a.r)[D * row + k];
                p[k] = ((T *)a.p)[D * row + k];
                s[k] = ((T *)a.s)[D * row + k];
            }
            if (!a.block_pre) dinv[k] = ((const T *)a.invd)[D * row + k];
        }
        if (a.coarse) {
            for (int k = 0; k < D; ++k) d[k] = a.agg_d[D * row + k];
            mk = a.mask[row];
            const int w = a.wpos[row];
            pos = w & 0xffff;
            rank = w >> 16;
        }
    }
    // ---- its part of the SpMV: wps wavefronts share each slice, taking every wps-th slot
    const int wps = PCG_NW / nsl, sl = wv / wps, part0 = wv - sl * wps;
    const bool spmv = sl < nsl;
    const int64_t slice = spmv ? a.order[k0 + sl] : 0, srow = slice * 64 + lane;
    int W = 0, len = 0;
    uint32_t cbase = 0;
    if (spmv) {
        const int64_t base = a.sp[slice];
        W = (int)((a.sp[slice + 1] - base) >> 6);
        len = srow < a.n ? a.cptr[srow + 1] - a.cptr[srow] : 0;
        cbase = (uint32_t)base;
    }
    const __amdgpu_buffer_rsrc_t bc = rsrc_of(a.scol, a.scol_bytes), bv = rsrc_of(a.aval, a.aval_bytes),
                                 bu = rsrc_of(a.u, a.u_bytes);
    // ---- its aggregates
    const int l0 = a.coarse ? a.wl_ptr[wg] : 0, nl = a.coarse ? a.wl_ptr[wg + 1] - l0 : 0;
    // ---- the coarse DoFs whose rows of Ac^-1 it applies, and the range of P^T r these take
    const int y0 = a.coarse ? min(a.ncoarse, wg * a.ndof_wg) : 0, ny = a.coarse ? min(a.ncoarse, y0 + a.ndof_wg) - y0 : 0;
    int cz0 = 0, ncz = 0;
    if (ny > 0) {
        cz0 = a.cb[a.agg_grp[y0 / M]];
        ncz = a.cb[a.agg_grp[(y0 + ny - 1) / M] + 1] - cz0;
    }
    if (a.ainv_lds)
        for (int q = wv; q < ny; q += PCG_NW) {
            const int b = a.agg_grp[(y0 + q) / M], nc = a.cb[b + 1] - a.cb[b];
            const double *A = a.Ainv + a.off[b] + (int64_t)(y0 + q - a.cb[b]) * nc;
            for (int c = lane; c < nc; c += 64) arow[(size_t)q * a.ainv_lds + c] = A[c];
        }
    double thr = a.scal[SC_THR], rhs2 = a.scal[SC_RHS2], gprev = a.scal[SC_GAMMA_P], aprev = a.scal[SC_ALPHA_P];
    double rr = 0.0, done = 0.0;
    int it = a.it0;
    for (;; ++it) {
        const int set = it & 1;
        if (it == a.itmax) break;
        if (a.coarse) {
            // ---- C: this workgroup's shares of P^T r
            if (own) {
                double rf[D], t[M];
                for (int k = 0; k < D; ++k) rf[k] = (mk >> k) & 1 ? 0.0 : (double)r[k];
                modes_t<D>(d, rf, t);
                for (int m = 0; m < M; ++m) share[m * nrow_lds + pos] = t[m];
            }
            __syncthreads();
            u64 *sc = a.slot_c + (size_t)set * a.nslot_c, *sc_old = a.slot_c + (size_t)(set ^ 1) * a.nslot_c;
            const int q0 = threadIdx.x >> 3, sub = threadIdx.x & 7;
            for (int q = q0; q < nl * M; q += PCG_NT / 8) {  // 8 lanes per (aggregate, mode)
                const int l = q / M, m = q - l * M;
                double t = 0.0;
                for (int e = a.wl_beg[l0 + wg + l] + sub; e < a.wl_beg[l0 + wg + l + 1]; e += 8) t += share[m * nrow_lds + e];
                for (int o = 4; o > 0; o >>= 1) t += __shfl_xor(t, o, 8);
                if (sub == 0) st_agent(&sc[(size_t)a.wl_slot[l0 + l] * a.ncoarse + a.wl_agg[l0 + l] * M + m], word_of(t));
            }
            bool ok = true;
            for (int j = threadIdx.x; j < ncz; j += PCG_NT) {
                const int c = cz0 + j, cnt = a.ca_cnt[c / M];
                double t = 0.0;
                for (int e = 0; e < cnt; e += 8) {
                    u64 v[8];
                    ok = slot_wait<8>(&sc[(size_t)e * a.ncoarse + c], a.ncoarse, cnt - e, v, a) && ok;
#pragma unroll
                    for (int u = 0; u < 8; ++u) t += value_of(v[u]);
                }
                cz[j] = t;
            }
            if (!ok) gave_up = 1;
            __syncthreads();
            if (gave_up) return;
            for (int q = q0; q < nl * M; q += PCG_NT / 8)
                if (sub == 0)
                    st_agent(&sc_old[(size_t)a.wl_slot[l0 + q / M] * a.ncoarse + a.wl_agg[l0 + q / M] * M + q % M], PCG_EMPTY);
            // ---- Y: Ac^-1 P^T r of its coarse DoFs, a wavefront per row, all of the row in flight
            u64 *sy = a.slot_y + (size_t)set * a.ncoarse, *sy_old = a.slot_y + (size_t)(set ^ 1) * a.ncoarse;
            for (int q = wv; q < ny; q += PCG_NW) {
                const int b = a.agg_grp[(y0 + q) / M], bse = a.cb[b], nc = a.cb[b + 1] - bse;
                const double *A = a.ainv_lds ? arow + (size_t)q * a.ainv_lds
                                             : a.Ainv + a.off[b] + (int64_t)(y0 + q - bse) * nc;
                double ar[16], t = 0.0;
#pragma unroll
                for (int u = 0; u < 16; ++u) ar[u] = lane + 64 * u < nc ? A[lane + 64 * u] : 0.0;
#pragma unroll
                for (int u = 0; u < 16; ++u)
                    if (lane + 64 * u < nc) t += ar[u] * cz[bse - cz0 + lane + 64 * u];
                for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
                if (lane == 0) {
                    st_agent(&sy_old[y0 + q], PCG_EMPTY);
                    st_agent(&sy[y0 + q], word_of(t));
                }
            }
            for (int q = threadIdx.x; q < nl * M; q += PCG_NT) {
                u64 v[1];
                ok = slot_wait<1>(&sy[a.wl_agg[l0 + q / M] * M + q % M], 0, 1, v, a) && ok;
                ycor[q] = value_of(v[0]);
            }
            if (!ok) gave_up = 1;
            __syncthreads();
            if (gave_up) return;
        }
        // ---- U: u = M^-1 r, (r, r) and (r, u)
        T uu[D];
        double vu[2] = {0.0, 0.0};
        for (int k = 0; k < D; ++k) uu[k] = (T)0;
        if (own) {
            if (a.block_pre) {
                const T *B = (const T *)a.invd + (int64_t)EB * row;
                for (int k = 0; k < D; ++k)
                    for (int q = 0; q < D; ++q) uu[k] += B[k * D + q] * r[q];
            } else {
                for (int k = 0; k < D; ++k) uu[k] = dinv[k] * r[k];
            }
            if (a.coarse) {
                double t[D];
                modes<D>(d, ycor + rank * M, t);
                for (int k = 0; k < D; ++k)
                    if (!((mk >> k) & 1)) uu[k] += (T)t[k];
            }
            for (int k = 0; k < D; ++k) {
                st_u((T *)a.u + D * row + k, uu[k]);
                vu[0] += (double)r[k] * (double)r[k];
                vu[1] += (double)r[k] * (double)uu[k];
            }
        }
        stores_done();
        wg_sum<2>(vu, red0);  // its barrier follows every wavefront's stores
        u64 *su = a.slot_u + (size_t)set * 2 * PCG_SET, *su_old = a.slot_u + (size_t)(set ^ 1) * 2 * PCG_SET;
        if (threadIdx.x == 0) {
            st_agent(&su[slot_at(wg)], word_of(vu[0]));
            st_agent(&su[PCG_SET + slot_at(wg)], word_of(vu[1]));
        }
        double vs[2] = {0.0, 0.0};
        bool ok = true;
        if ((int)threadIdx.x < G) {
            u64 v[2];
            ok = slot_wait<2>(&su[slot_at(threadIdx.x)], PCG_SET, 2, v, a);
            vs[0] = value_of(v[0]);
            vs[1] = value_of(v[1]);
        }
        if (!ok) gave_up = 1;
        wg_sum<2>(vs, red1);
        if (gave_up) return;
        if (threadIdx.x == 0) {
            st_agent(&su_old[slot_at(wg)], PCG_EMPTY);
            st_agent(&su_old[PCG_SET + slot_at(wg)], PCG_EMPTY);
        }
        rr = vs[0];
        const double gamma = vs[1];
        if (it == 0) {
            rhs2 = rr;
            thr = fmax(a.tol * a.tol * rr, DBL_MIN);
            done = (rr == 0.0) ? 3.0 : ((rr < thr) ? 1.0 : (a.maxit <= 0 ? 2.0 : 0.0));
        } else if (rr < thr) {
            done = 1.0;
        } else if ((double)it >= a.maxit) {
            done = 2.0;
        }
        if (done != 0.0) break;
        // ---- D: w = K u and (w, u)
        if (spmv) {
            T acc[D];
            for (int k = 0; k < D; ++k) acc[k] = (T)0;
            for (int s0 = part0; s0 < W; s0 += wps * UNR) {
                T e[UNR][EB], uj[UNR][D];
                uint32_t o[UNR];
#pragma unroll
                for (int q = 0; q < UNR; ++q) {
                    const int sq = s0 + q * wps;
                    const bool in = sq < len;
                    const uint32_t b = cbase + (uint32_t)sq * 64 + lane;
                    if constexpr (sizeof(IX) == 2)
                        o[q] = (uint32_t)((int)srow + (int)(int16_t)__builtin_amdgcn_raw_buffer_load_b16(
                                                          bc, in ? (int)(2 * b) : (int)NO_ELEM, 0, AUX));
                    else
                        o[q] = __builtin_amdgcn_raw_buffer_load_b32(bc, in ? (int)(4 * b) : (int)NO_ELEM, 0, AUX);
                    const uint32_t vb = in ? (EB * (cbase + (uint32_t)sq * 64) + lane) * (uint32_t)sizeof(T) : NO_ELEM;
#pragma unroll
                    for (int c = 0; c < EB; ++c) e[q][c] = ld_elem<T, AUX>(bv, vb + c * 64 * (uint32_t)sizeof(T));
                }
#pragma unroll
                for (int q = 0; q < UNR; ++q)
                    ld_u<T, D>(bu, s0 + q * wps < len ? o[q] * (uint32_t)(D * sizeof(T)) : NO_ELEM, uj[q]);
#pragma unroll
                for (int q = 0; q < UNR; ++q)
                    for (int rw = 0; rw < D; ++rw)
                        for (int c = 0; c < D; ++c) acc[rw] += e[q][rw * D + c] * uj[q][c];
            }
            for (int k = 0; k < D; ++k) part[(wv * D + k) * 64 + lane] = acc[k];
        }
        __syncthreads();
        T w[D];
        double vd[1] = {0.0};
        for (int k = 0; k < D; ++k) w[k] = (T)0;
        if (own) {
            for (int k = 0; k < D; ++k) {
                for (int q = 0; q < wps; ++q) w[k] += part[((wv * wps + q) * D + k) * 64 + lane];
                vd[0] += (double)uu[k] * (double)w[k];
            }
        }
        wg_sum<1>(vd, red2);
        u64 *sd = a.slot_d + (size_t)set * PCG_SET, *sd_old = a.slot_d + (size_t)(set ^ 1) * PCG_SET;
        if (threadIdx.x == 0) {
            stores_done();
            st_agent(&sd[slot_at(wg)], word_of(vd[0]));
        }
        double vt[1] = {0.0};
        if ((int)threadIdx.x < G) {
            u64 v[1];
            ok = slot_wait<1>(&sd[slot_at(threadIdx.x)], 0, 1, v, a);
            vt[0] = value_of(v[0]);
        }
        if (!ok) gave_up = 1;
        wg_sum<1>(vt, red3);
        if (gave_up) return;
        if (threadIdx.x == 0) st_agent(&sd_old[slot_at(wg)], PCG_EMPTY);
        const double delta = vt[0];
        double alpha, beta = 0.0;
        if (it == 0) {
            alpha = gamma / delta;
        } else {
            beta = gamma / gprev;
            alpha = gamma / (delta - beta * gamma / aprev);
        }
        gprev = gamma;
        aprev = alpha;
        const T ta = (T)alpha, tb = (T)beta;
        for (int k = 0; k < D; ++k) {
            p[k] = uu[k] + tb * p[k];
            s[k] = w[k] + tb * s[k];
            x[k] += ta * p[k];
            r[k] -= ta * s[k];
        }
    }
    if (own) {
        for (int k = 0; k < D; ++k) {
            ((T *)a.x)[D * row + k] = x[k];
            if (done == 0.0) {  // continued by the next launch
                ((T *)a.r)[D * row + k] = r[k];
                ((T *)a.p)[D * row + k] = p[k];
                ((T *)a.s)[D * row + k] = s[k];
            }
        }
    }
    if (wg == 0 && threadIdx.x == 0) {
        a.scal[SC_RHS2] = rhs2;
        a.scal[SC_THR] = thr;
        a.scal[SC_RR] = rr;
        a.scal[SC_ITER] = (double)it;
        a.scal[SC_GAMMA_P] = gprev;
        a.scal[SC_ALPHA_P] = aprev;
        a.scal[SC_DONE] = done;
    }
}

// empties every slot and clears the abort word before a launch
__global__ __launch_bounds__(256) void k_pcg_clear(int64_t words, u64 *slots, double *scal) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < words) slots[i] = PCG_EMPTY;
    if (i == 0) scal[SC_ABORT] = 0.0;
}

}  // namespace

// Coarse DoFs whose rows of Ac^-1 a workgroup forms: at least one row per wavefront, since every
// workgroup that forms any polls all shares of its group
static int dofs_per_wg(int ncoarse, int G) { return std::max(PCG_NW, (ncoarse + G - 1) / G); }

// whether a runtime call succeeded; the error of one that did not is cleared, since the launches take over
static bool hip_done(hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();
    return e == hipSuccess;
}

// Whether neighbouring rows have neighbouring columns: over the rows of eight slices, the groups of 16 particles
// that the q-th columns of a slice's rows fall into, against the rows (a lattice in its own order 0.1-0.3, a
// shuffled one 0.9). False when the device could not be read.
static bool pcg_scattered(lpm_ctx *c, bool *scattered) {
    constexpr int NS = 8;
    int32_t ptr[NS][65];
    int64_t row[NS], rows[NS];
    for (int k = 0; k < NS; ++k) {
        row[k] = 64 * (c->nslice * k / NS);
        rows[k] = std::min<int64_t>(64, c->n - row[k]);
        if (!hip_done(hipMemcpyAsync(ptr[k], c->cptr + row[k], sizeof(int32_t) * (rows[k] + 1), hipMemcpyDeviceToHost, c->stream)))
            return false;
    }
    if (!hip_done(hipStreamSynchronize(c->stream))) return false;
    std::vector<int32_t> col[NS];
    for (int k = 0; k < NS; ++k) {
        col[k].resize(ptr[k][rows[k]] - ptr[k][0]);
        if (!col[k].empty() && !hip_done(hipMemcpyAsync(col[k].data(), c->cidx + ptr[k][0], sizeof(int32_t) * col[k].size(),
                                                        hipMemcpyDeviceToHost, c->stream)))
            return false;
    }
    if (!hip_done(hipStreamSynchronize(c->stream))) return false;
    int64_t lanes = 0, groups = 0;
    std::vector<int32_t> g;
    for (int k = 0; k < NS; ++k)
        for (int q = 0; q < c->maxconn; ++q) {
            g.clear();
            for (int64_t i = 0; i < rows[k]; ++i)
                if (q < ptr[k][i + 1] - ptr[k][i]) g.push_back(col[k][ptr[k][i] - ptr[k][0] + q] >> 4);
            lanes += (int64_t)g.size();
            std::sort(g.begin(), g.end());
            groups += std::unique(g.begin(), g.end()) - g.begin();
        }
    *scattered = 2 * groups > lanes;
    return true;
}

// Slots and, for the two-level preconditioner, the rows of each workgroup by aggregate: built once for each of
// the two kinds and kept, since a caller may switch between them from solve to solve (SC 40^3: 0.5 ms a time).
// Sets the plan's state: 1 usable, -1 not. No failure in here ends the solve: the launches need none of this.
static void pcg_prepare(lpm_ctx *c, PcgPlan &P, bool coarse) {
    if (P.state != 0) return;
    P.state = -1;
    const int spw = (int)((c->nslice + PCG_WG - 1) / PCG_WG);
    if (spw > PCG_SPW) return;  // more than one row per thread
    const int G = (int)((c->nslice + spw - 1) / spw), D = c->dim, M = D == 3 ? 6 : 3;
    // 32-bit buffer offsets, FP64 values at most
    if ((double)c->nslots * D * D * 8 > 4.0e9) return;
    int64_t nctr = 0;
    // Slices in id order, or, with the coarse space, by the aggregate of their middle row: slices that
    // lie side by side across the numbering direction then meet in one workgroup, which so
    // touches fewer aggregates (hex 200 x 231: 6 instead of 15).
    std::vector<int32_t> order(c->nslice), lptr(1, 0), lagg, slot, lbeg, wpos, cnt;
    for (int64_t k = 0; k < c->nslice; ++k) order[k] = (int32_t)k;
    if (coarse) {
        const int64_t n = c->n;
        std::vector<int32_t> agg(n), grp(c->nagg), cb(c->ncgrp + 1);
        if (!hip_done(hipMemcpyAsync(agg.data(), c->agg_of, sizeof(int32_t) * n, hipMemcpyDeviceToHost, c->stream)) ||
            !hip_done(hipMemcpyAsync(grp.data(), c->agg_grp, sizeof(int32_t) * c->nagg, hipMemcpyDeviceToHost, c->stream)) ||
            !hip_done(hipMemcpyAsync(cb.data(), c->cgrp_cb, sizeof(int32_t) * (c->ncgrp + 1), hipMemcpyDeviceToHost, c->stream)) ||
            !hip_done(hipStreamSynchronize(c->stream)))
            return;
        if (spw > 1)
            std::stable_sort(order.begin(), order.end(), [&](int32_t x, int32_t y) {
                return agg[std::min<int64_t>(n - 1, 64LL * x + 32)] < agg[std::min<int64_t>(n - 1, 64LL * y + 32)];
            });
        std::vector<int32_t> rank(c->nagg, -1), fill;
        wpos.resize(n);
        for (int w = 0; w < G; ++w) {
            std::vector<int64_t> rows;
            for (int64_t q = (int64_t)w * spw; q < std::min<int64_t>(c->nslice, (int64_t)(w + 1) * spw); ++q)
                for (int64_t i = 64LL * order[q]; i < std::min<int64_t>(n, 64LL * order[q] + 64); ++i) rows.push_back(i);
            std::vector<int32_t> mine;
            for (int64_t i : rows) mine.push_back(agg[i]);
            std::sort(mine.begin(), mine.end());
            mine.erase(std::unique(mine.begin(), mine.end()), mine.end());
            if ((int)mine.size() > PCG_LA) return;
            fill.assign(mine.size() + 1, 0);
            for (size_t q = 0; q < mine.size(); ++q) rank[mine[q]] = (int32_t)q;
            for (int64_t i : rows) ++fill[rank[agg[i]] + 1];
            for (size_t q = 0; q < mine.size(); ++q) fill[q + 1] += fill[q];
            lbeg.insert(lbeg.end(), fill.begin(), fill.end());  // one entry more than aggregates
            for (int64_t i : rows) {
                const int q = rank[agg[i]];
                wpos[i] = (q << 16) | fill[q]++;
            }
            lagg.insert(lagg.end(), mine.begin(), mine.end());
            lptr.push_back((int32_t)lagg.size());
        }
        const int per = dofs_per_wg(c->ncoarse, G);
        for (int y = 0; y < c->ncoarse; y += per)
            if (cb[grp[(std::min(c->ncoarse, y + per) - 1) / M] + 1] - cb[grp[y / M]] > PCG_CZ) return;
        // share u of coarse DoF d lies at u * ncoarse + d, so that a wavefront's polls are contiguous
        cnt.assign(c->nagg, 0);
        slot.resize(lagg.size());
        for (size_t q = 0; q < lagg.size(); ++q) slot[q] = cnt[lagg[q]]++;
        // Where the numbering scatters the rows of a workgroup over many aggregates, every aggregate has shares of
        // many workgroups, and polling them takes longer than the launches' restriction. Launched against persistent
        // time by shares: lattices in their own order up to 12,000: 1.08-1.37; shuffled in part or in full: 20,000
        // to 27,000 1.00-1.23, 32,000 1.05-1.12, 37,000 0.85-0.98, 50,000 0.87, 77,000 0.78, 88,000 0.68-0.70.
        std::vector<int64_t> upto(c->nagg + 1, 0);
        for (int g = 0; g < c->nagg; ++g) upto[g + 1] = upto[g] + (int64_t)M * cnt[g];
        for (int y = 0; y < c->ncoarse; y += per)
            if (upto[cb[grp[(std::min(c->ncoarse, y + per) - 1) / M] + 1] / M] - upto[cb[grp[y / M]] / M] > PCG_SHARES) return;
        nctr = (int64_t)*std::max_element(cnt.begin(), cnt.end()) * c->ncoarse;
    }
    if (!c->scol16 && !pcg_scattered(c, &P.scattered)) return;
    P.words = 2 * (nctr + (coarse ? c->ncoarse : 0) + 3 * (int64_t)PCG_SET);
    P.nslot_c = (int)nctr;
    Slab slab;
    slab.add(&P.slots, P.words);
    const std::vector<int32_t> *src[7] = {&order, &lptr, &lagg, &slot, &lbeg, &wpos, &cnt};
    int32_t **dst[7] = {&P.order, &P.lptr, &P.lagg, &P.lslot, &P.lbeg, &P.wpos, &P.cnt};
    for (int k = 0; k < 7; ++k) slab.add(dst[k], (int64_t)src[k]->size());
    if (!hip_done(slab.alloc(&P.base))) return;
    for (int k = 0; k < 7; ++k)
        if (!src[k]->empty() && !hip_done(hipMemcpyAsync(*dst[k], src[k]->data(), sizeof(int32_t) * src[k]->size(),
                                                         hipMemcpyHostToDevice, c->stream)))
            return;
    if (!hip_done(hipStreamSynchronize(c->stream))) return;
    P.spw = spw;
    P.grid = G;
    P.state = 1;
    c->st_pcg_plans++;
}

void pcg_free(lpm_ctx *c) {
    for (PcgPlan &P : c->pcg_plan) {
        if (P.base) hipFree(P.base);
        P = PcgPlan();
    }
}

namespace {

// The CUs of each device, dealt out to the persistent solves in flight, in the order in which they ask. Workgroups
// go round the eight XCDs, so a grid takes ceil(grid / 8) CUs of each.
class ResidentCus {
public:
    ResidentCus(int device, int cus, int grid) : d_(of(device)) {
        const int all = std::max(1, cus / 8);
        n_ = std::min(all, (grid + 7) / 8);
        std::unique_lock<std::mutex> lock(d_.m);
        const uint64_t turn = d_.next++;
        d_.cv.wait(lock, [&] { return d_.serving == turn && d_.used + n_ <= all; });
        d_.used += n_;
        d_.serving++;
        d_.cv.notify_all();
    }
    ~ResidentCus() {
        std::lock_guard<std::mutex> lock(d_.m);
        d_.used -= n_;
        d_.cv.notify_all();
    }
    ResidentCus(const ResidentCus &) = delete;
    ResidentCus &operator=(const ResidentCus &) = delete;

private:
    struct Device {
        std::mutex m;
        std::condition_variable cv;
        int used = 0;
        uint64_t next = 0, serving = 0;
    };
    static Device &of(int device) {
        // never destroyed: a thread may still solve while the process ends
        static std::mutex &m = *new std::mutex;
        static std::map<int, Device> &all = *new std::map<int, Device>;
        std::lock_guard<std::mutex> lock(m);
        return all[device];
    }
    Device &d_;
    int n_ = 0;
};

}  // namespace

template <typename T, int D, typename IX, bool NT>
static int pcg_go(lpm_ctx *c, PcgPlan &P, PcgArgs &a, int64_t maxit, bool *ran) {
    const int M = D == 3 ? 6 : 3;
    const size_t un = std::max(sizeof(T) * PCG_NW * D * 64, sizeof(double) * M * 64 * (size_t)P.spw);
    size_t lds = un + sizeof(double) * (PCG_CZ + PCG_LA * M);
    auto kern = k_pcg<T, D, IX, NT>;
    if (P.kern != (const void *)kern) {
        // The device's LDS less the kernel's own. Every context asks for this same limit, as the attribute belongs
        // to the kernel and not to the context.
        hipFuncAttributes fa;
        int most = 0;
        P.kern = (const void *)kern;
        P.lds = 0;
        P.lds_most = 0;
        if (hip_done(hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, c->device)) &&
            hip_done(hipFuncGetAttributes(&fa, (const void *)kern)) && (size_t)most > fa.sharedSizeBytes &&
            hip_done(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, most - (int)fa.sharedSizeBytes)))
            P.lds_most = most - fa.sharedSizeBytes;
    }
    if (lds > P.lds_most) return LPM_OK;
    // a workgroup's rows of Ac^-1 stay in its LDS where they fit beside the rest
    a.ainv_lds = 0;
    const size_t rows = sizeof(double) * (size_t)a.ndof_wg * std::max(c->cgrp_nbmax, 1);
    if (a.coarse && lds + rows <= P.lds_most) {
        a.ainv_lds = c->cgrp_nbmax;
        lds += rows;
    }
    if (P.lds != lds) {  // all workgroups must be resident at once
        int per = 0, cus = 0, khz = 0;
        P.fits = hip_done(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kern, PCG_NT, lds)) &&
                 hip_done(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device)) &&
                 hip_done(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device)) &&
                 (int64_t)per * cus >= P.grid;
        P.lds = lds;
        P.cus = cus;
        P.khz = khz;
    }
    if (!P.fits) return LPM_OK;
    a.wait_ticks = (u64)(c->cg_wait_ms * P.khz);
    const ResidentCus held(c->device, P.cus, P.grid);  // until the solve has ended
    for (int64_t it = 0;;) {
        hipLaunchKernelGGL(k_pcg_clear, dim3(blocks_for(P.words, 256)), dim3(256), 0, c->stream, P.words,
                           P.slots, c->scal);
        a.it0 = (int)it;
        a.itmax = (int)std::min<int64_t>(it + PCG_LAUNCH_ITERS, 0x7fffffff);
        void *args[] = {&a};
        if (!hip_done(hipLaunchKernel((const void *)kern, dim3(P.grid), dim3(PCG_NT), args, lds, c->stream))) {
            P.fits = false;  // the caller solves launch by launch
            return LPM_OK;
        }
        LPM_HIP(c, hipMemcpyAsync(c->h_scal, c->scal, sizeof(double) * SC_COUNT, hipMemcpyDeviceToHost, c->stream));
        LPM_HIP(c, hipStreamSynchronize(c->stream));
        if (c->h_scal[SC_ABORT] != 0.0) {  // what holds the device may hold it for long: no further wait in this context
            c->pcg_given_up = true;
            c->st_pcg_given_up++;
            return LPM_OK;
        }
        if (c->h_scal[SC_DONE] != 0.0) {
            *ran = true;
            return LPM_OK;
        }
        it = a.itmax;
        if (it > maxit + 2 * PCG_LAUNCH_ITERS) return lpm_fail(c, LPM_E_HIP, "k_pcg passed its iteration limit");
    }
}

// The whole solve in one launch (see the head of this file). *ran is false, with nothing done,
// where the rule below keeps the launch-by-launch solve, or where the launch was given up.
int pcg_solve(lpm_ctx *c, int64_t maxit, bool *ran) {
    *ran = false;
    // a caller that fixes the SpMV launch shape, replays batches from a graph or times single SpMVs
    // asks for the launches themselves
    if (!c->cg_persist || c->cg_graph || !c->spmv_tune || c->timing > 0 || c->pcg_given_up) return LPM_OK;
    const bool coarse = two_level(c);
    PcgPlan &P = c->pcg_plan[coarse ? 1 : 0];
    pcg_prepare(c, P, coarse);
    if (P.state != 1) return LPM_OK;
    const size_t es = c->precision == 0 ? 4 : 8;
    const int D = c->dim;
    const bool idx16 = c->scol16 && c->spmv_idx16;
    // u is read past the L2s here, an entry of its own for almost every block where the columns are scattered,
    // while the launched SpMV finds u in them. That costs more than the launches do from 28 MB of such reads per
    // product on, until at 250 MB the matrix leaves the MALL and its bytes bound both. Launched against persistent
    // time of shuffled lattices, Jacobi, by MB of u read (MB of matrix): 18 (44) 1.08, 19 (48) 1.12, 25 (63) 1.04, 25 (82)
    // 1.00, 32 (80) 0.94, 32 (107) 0.95, 35 (79) 0.96, 38 (86) 1.04, 39 (125) 0.87, 49 (156) 0.84, 61 (202) 0.77, 64
    // (204) 0.80, 66 (209) 0.83; 80 (255) 1.00, 87 (290) 1.09, 88 (280) 1.05, 121 (384) 1.12, 174 (551) 1.11.
    if (P.scattered && (double)c->nconn * D * es > 28e6 && (double)c->nslots * (D * D * es + 4) < 250e6) return LPM_OK;
    PcgArgs a = {};
    a.n = c->n;
    a.nslice = c->nslice;
    a.spw = P.spw;
    a.block_pre = block_jacobi(c);
    a.coarse = coarse;
    a.tol = c->cg_tol;
    a.maxit = (double)maxit;
    a.sp = c->sp;
    a.cptr = c->cptr;
    a.scol = idx16 ? (const void *)c->scol16 : (const void *)c->scol;
    a.aval = c->aval;
    a.invd = c->invdiag;
    a.scol_bytes = (uint32_t)(c->nslots * (idx16 ? 2 : 4));
    a.aval_bytes = (uint32_t)(c->nslots * D * D * es);
    a.u_bytes = (uint32_t)(c->n * D * es);
    a.b64 = c->residual;
    a.x = c->v_x;
    a.r = c->v_r;
    a.u = c->v_u;
    a.p = c->v_p;
    a.s = c->v_s;
    a.scal = c->scal;
    u64 *w = P.slots;
    a.slot_u = w;
    a.slot_d = w + 4 * PCG_SET;
    a.slot_c = w + 6 * PCG_SET;
    a.nslot_c = P.nslot_c;
    a.slot_y = a.slot_c + 2 * (int64_t)a.nslot_c;
    a.ncoarse = coarse ? c->ncoarse : 0;
    a.ndof_wg = dofs_per_wg(a.ncoarse, P.grid);
    a.agg_d = c->agg_d;
    a.Ainv = c->Ainv;
    a.mask = c->dofmask;
    a.agg_grp = c->agg_grp;
    a.cb = c->cgrp_cb;
    a.off = c->cgrp_off;
    a.ca_cnt = P.cnt;
    a.wl_ptr = P.lptr;
    a.wl_agg = P.lagg;
    a.wl_slot = P.lslot;
    a.wl_beg = P.lbeg;
    a.wpos = P.wpos;
    a.order = P.order;
    // the matrix is kept in the L2s while it fits them (8 x 4 MB) and streamed past them otherwise
    const bool nt = (double)c->nslots * (D * D * es + (idx16 ? 2 : 4)) > 28e6 && c->spmv_nt;
#define PCG_GO(T, D_, IX) (nt ? pcg_go<T, D_, IX, true>(c, P, a, maxit, ran) : pcg_go<T, D_, IX, false>(c, P, a, maxit, ran))
    if (c->precision == 0) {
        if (D == 3) return idx16 ? PCG_GO(float, 3, int16_t) : PCG_GO(float, 3, int32_t);
        return idx16 ? PCG_GO(float, 2, int16_t) : PCG_GO(float, 2, int32_t);
    }
    if (D == 3) return idx16 ? PCG_GO(double, 3, int16_t) : PCG_GO(double, 3, int32_t);
    return idx16 ? PCG_GO(double, 2, int16_t) : PCG_GO(double, 2, int32_t);
#undef PCG_GO
}
