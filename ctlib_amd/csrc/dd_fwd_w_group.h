// Weighted line -> bin work item (backprojection_t and its exact adjoint form) with wave-private
// line tables, over a group of slices (gfx950).
#pragma once
#include "dd_device.h"

namespace ctlib {
namespace dd {

// Entries of a wave-private line table sit at j + j/8 (one 16-byte pad every 8):
// lane L writes entries 8L+1 .. 8L+8, and with the pad consecutive lanes land
// 9 entries apart, so each ds_write_b128 of 16 lanes covers all 64 banks.
__host__ __device__ inline int wtab_slots(int n) { return n + 2 + (n + 2) / 8 + 1; }
__device__ __forceinline__ int wtab_slot(int j) { return j + (j >> 3); }

// LDS bytes of one fwd_group_w: one wave-private table per wave.
__host__ __device__ inline size_t fwd_w_block_lds(int nmax) { return (size_t)4 * wtab_slots(nmax) * 16; }

// For lines of at most 64*PPL pixels: G = 4 views per block, one per wave, and each wave builds the
// weighted cumulative table of its own view for every line by itself: lane L owns pixels L*PPL ..
// L*PPL+PPL-1 (one serial sum and one wave scan per line) and writes them into its wave's private
// table, so no barrier is needed anywhere.  The kernel is VALU-bound; the pixel weights, tau and the
// entries' addresses (some 130 of its 220 instructions per line and view) depend on the geometry
// alone and can be formed once for NS slices b0 .. b0 + NS - 1 (one past the batch repeats the last and
// is not stored), whose tables follow each other in the wave's buffer (LDS operations of a wave stay
// in order).  As in the unweighted kernel, lane L takes the bin edge at position b128_pos(L) of its
// slot, so that the reads are free of bank conflicts, and at most four reads are under way, which keeps
// the registers within four waves per SIMD (fan-ED 512^2 B=8 1.42 -> 1.38 ms, fan-EA B=16 3.97 -> 3.60,
// fan-ED 1024^2 B=4 6.13 -> 5.51).  The line's pixels and coefficients are loaded
// one line ahead into registers.  FULL: every line has exactly 64*PPL pixels, so no lane needs a bounds
// predicate.  The pixel weight 1/(s ((w0 + w1 p)^2 + w2)) is formed in the data precision (fp32 data:
// fp32 arithmetic with a fp32 reciprocal, about 1e-7 relative; fp64 data: fp64 arithmetic with a
// Newton-refined reciprocal), and the weighted value is rounded to the data type before the fp64
// prefix sum, as in fwd_block with WEIGHTED.  Lines [lb, le) of the axis contribute
// (at least one).
template <typename T, int NS, int NEM, int PPL, bool FULL>
__device__ __forceinline__ void fwd_group_w(const DevPlan& P, const T* __restrict__ src, T* __restrict__ y, int b0,
                                            int B, int mode, int grp, const double* __restrict__ post,
                                            unsigned char* __restrict__ smem, int lb, int le) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int* vlist = mode == MODE_Y ? P.yviews : P.xviews;
    const int nv = mode == MODE_Y ? P.ny : P.nx;
    const int nlines = mode == MODE_Y ? P.W : P.H;
    const int n = FULL ? 64 * PPL : (mode == MODE_Y ? P.H : P.W);
    const int D = P.D;

    int vw[1];
    {
        const int idx = grp * 4 + wave;
        vw[0] = vlist[idx < nv ? idx : nv - 1];
    }
    double e[NEM], S[NS][1][NEM];
#pragma unroll
    for (int i = 0; i < NEM; i++) {
        const int k = b128_pos(lane) + 64 * i;
        e[i] = P.edges[(size_t)vw[0] * (D + 1) + (k <= D ? k : D)];
#pragma unroll
        for (int s = 0; s < NS; s++) S[s][0][i] = 0.0;
    }

    double2* tb = reinterpret_cast<double2*>(smem) + (size_t)wave * wtab_slots(n);
    const T* base = src + (size_t)b0 * nlines * n;
    const size_t next_slice = b0 + 1 < B ? (size_t)nlines * n : 0;  // NS <= 2
    const int p0 = lane * PPL;
    const int hi = n + 1;
    // LineCoef word `lane` (lanes 0..7) of this wave's view, one line ahead
    const double* crow = reinterpret_cast<const double*>(P.lines + (size_t)vw[0] * P.max_lines) + (lane & 7);
    // fp32 data: the line's pre-scaled weight coefficients {., c w1, c w0, c^2 w2} (uniform)
    const float4* wrow = P.adj_wk + (size_t)vw[0] * P.max_lines;
    auto load_pixels = [&](int l, int s, T (&x)[PPL]) {
        const T* row = base + s * next_slice + (size_t)l * n;
#pragma unroll
        for (int k = 0; k < PPL; k++) x[k] = (FULL || p0 + k < n) ? row[p0 + k] : T(0);
    };
    T xv[NS][PPL];
    double cw = 0.0;
    float4 wk = make_float4(0.f, 0.f, 0.f, 1.f);
    auto load_coef = [&](int l) {
        cw = crow[(size_t)l * LC_WORDS];
        if (sizeof(T) == 4) wk = wrow[l];
    };
#pragma unroll
    for (int s = 0; s < NS; s++) load_pixels(lb, s, xv[s]);
    load_coef(lb);

    for (int l = lb; l < le; l++) {
        const double s = readlane_d(cw, LC_S), A = readlane_d(cw, LC_A), Bc = readlane_d(cw, LC_B);
        const double w0 = readlane_d(cw, LC_W0), w1 = readlane_d(cw, LC_W1);
        const double w2 = readlane_d(cw, LC_W2), is = readlane_d(cw, LC_INVS);
        T w[PPL];  // pixel weights
        if constexpr (sizeof(T) == 4) {
            // weight (1/s) / ((w0 + w1 p)^2 + w2) = 1 / (u^2 + c^2 w2), u = k c w1 + (p0 c w1 + c w0)
            const float u0 = __builtin_fmaf(wk.y, (float)p0, wk.z);
#pragma unroll
            for (int k = 0; k < PPL; k++) {
                const float u = k == 0 ? u0 : __builtin_fmaf((float)k, wk.y, u0);
                w[k] = __builtin_amdgcn_rcpf(__builtin_fmaf(u, u, wk.w));
            }
        } else {
#pragma unroll
            for (int k = 0; k < PPL; k++) {
                const double u = __builtin_fma(w1, (double)(p0 + k), w0);
                w[k] = is * rcp_refined(__builtin_fma(u, u, w2));
            }
        }
        load_coef(min(l + 1, le - 1));
        const char* at[NEM];  // NS > 1: the entries' addresses, for every slice
        auto tau = [&](int i) { return __builtin_fma(A, e[i], Bc); };
        auto address = [&](int i) { return reinterpret_cast<const char*>(tb) + 16 * wtab_slot(table_index_u(tau(i), hi)); };
        if (NS > 1)
#pragma unroll
            for (int i = 0; i < NEM; i++) at[i] = address(i);
        if (FULL) __builtin_amdgcn_sched_barrier(0);
        // One slice's table after the other: the wave's reads of the table before were consumed
        // (in-order LDS within a wave), so it can be overwritten.
#pragma unroll
        for (int q = 0; q < NS; q++) {
            T val[PPL];
            double run = 0.0;
#pragma unroll
            for (int k = 0; k < PPL; k++) {
                val[k] = (FULL || p0 + k < n) ? xv[q][k] * w[k] : T(0);
                run += (double)val[k];
            }
            load_pixels(min(l + 1, le - 1), q, xv[q]);
            const double inc = wave_scan_incl(run, lane);
            double pref = inc - run;
#pragma unroll
            for (int k = 0; k < PPL; k++) {
                const int p = p0 + k;
                const double v = (double)val[k];
                if (FULL || p < n) tb[wtab_slot(p + 1)] = make_double2(__builtin_fma(-(double)(p + 1), v, pref), v);
                pref += v;
            }
            if (lane == 0) tb[0] = make_double2(0.0, 0.0);
            if (lane == 63) tb[wtab_slot(n + 1)] = make_double2(inc, 0.0);
            if constexpr (FULL) {
                __builtin_amdgcn_sched_barrier(0);
                // four reads under way, and no further: registers
                constexpr int AHEAD = 4;
                double2 ent[AHEAD];
#pragma unroll
                for (int i = 0; i < AHEAD && i < NEM; i++) ent[i] = *reinterpret_cast<const double2*>(NS > 1 ? at[i] : address(i));
#pragma unroll
                for (int i = 0; i < NEM; i++) {
                    const double2 g = ent[i % AHEAD];
                    S[q][0][i] = __builtin_fma(s, __builtin_fma(tau(i), g.y, g.x), S[q][0][i]);
                    asm volatile("" : "+v"(S[q][0][i]));
                    if (i + AHEAD < NEM)
                        ent[i % AHEAD] = *reinterpret_cast<const double2*>(NS > 1 ? at[i + AHEAD] : address(i + AHEAD));
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                // the bounds predicates leave the compiler's own order the faster one
#pragma unroll
                for (int i = 0; i < NEM; i++) {
                    const double2 g = *reinterpret_cast<const double2*>(NS > 1 ? at[i] : address(i));
                    S[q][0][i] = __builtin_fma(s, __builtin_fma(tau(i), g.y, g.x), S[q][0][i]);
                }
            }
        }
    }
    const int from = 4 * b128_pos(lane);
#pragma unroll
    for (int q = 0; q < NS; q++) {
        if (b0 + q >= B) break;
#pragma unroll
        for (int i = 0; i < NEM; i++) {  // the sums back in lane order
            int2 w = __builtin_bit_cast(int2, S[q][0][i]);
            w.x = __builtin_amdgcn_ds_bpermute(from, w.x);
            w.y = __builtin_amdgcn_ds_bpermute(from, w.y);
            S[q][0][i] = __builtin_bit_cast(double, w);
        }
        fwd_store<T, 1, NEM, false>(P, S[q], vw, grp, b0 + q, mode, lane, wave, y, post, nullptr, nullptr);
    }
}

}  // namespace dd
}  // namespace ctlib
