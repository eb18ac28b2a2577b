// Line -> bin kernel (projection) over the prebuilt line tables of a group of slices (gfx950).
//
// Which table entry a bin edge falls on depends on the view and the line, not on the slice: one work
// item evaluates tau and the entry's address once (one FMA, conversion, clamp, shift) and reads the
// tables of NS slices with it, two FMAs per slice.  That leaves the LDS reads as the bound, so four
// slices of fp32 data share packed tables: per entry {C_0, C_1}, {C_2, C_3} and the four slopes, which
// are pixels, in fp32 - three 16-byte reads for four lookups, and a quarter less to copy.
//
// Lane L of a wave takes the bin edge at position b128_pos(L) of its slot, so that each of the four
// passes in which ds_read_b128 serves a wave (16 lanes over 16 slots of 16 bytes) holds 16
// consecutive edges.  A bin is 0.6 to 0.85 pixels wide at the measured geometries: their entries span
// fewer than 16 and a read costs 5 cycles; in plain lane order a pass spans 28 edges and costs 8.
//
// Measured (k_fwd_lt alone, fp32 unless marked; before = one slice per block, lanes in order):
//   fan-ED 512^2, 736 x 736     B=32 2.40 -> 1.78 ms   B=8 0.60 -> 0.48   B=8 fp64 0.64 -> 0.58
//   fan-EA 512^2, 1024 x 888    B=16 1.96 -> 1.40 ms
//   fan-ED 1024^2, 1440 x 1536  B=4  2.57 -> 2.00 ms (pairs)
// and level at B=1.  At B=32 the VALU is busy 64 % and the LDS reads 50 %; the copies into LDS cost
// 0.10 ms, the barriers 0.06 (left out where the tables do not change).
#pragma once
#include "dd_device.h"

namespace ctlib {
namespace dd {

// Waves per block and lines per barrier (two buffers): two blocks to a CU's LDS for several slices,
// small blocks at NS = 1 (small batches).  One block of 16 waves and twice the lines instead measured
// 1.72 against 1.75 ms at fan-ED 512^2 B=32, but 0.54 against 0.47 ms at B=8 (fewer, larger blocks).
template <int NS>
__host__ __device__ constexpr int fwg_waves() { return NS == 1 ? 4 : 8; }
template <int NS, int M>
__host__ __device__ constexpr int fwg_lines() { return M == 1 ? (NS == 1 ? 4 : 2) : M == 2 && NS == 2 ? 2 : 1; }
// A step's tables are rows of n + 2 entries of 16 bytes (of ltab_n<M>() in memory and LDS): per line and
// slice one, per line of a packed group three.  A row is copied in chunks of 64, the last masked: rows
// of whole chunks in LDS leave 256-pixel lines three blocks a CU where four fit (fan-ED 200^2, 500 views,
// B=3: 68 us).
template <int NS>
__host__ __device__ constexpr int fwg_line_rows() { return NS == 4 ? 3 : NS; }
template <int NS, int M>
__host__ __device__ constexpr int fwg_rows() { return fwg_lines<NS, M>() * fwg_line_rows<NS>(); }
template <int M>
__host__ __device__ constexpr int fwg_pitch() { return ltab_n<M>(); }
template <int NS, int M>
inline size_t fwg_lds() { return (size_t)2 * fwg_rows<NS, M>() * fwg_pitch<M>() * 16; }
// Slots of 64 edges a wave can have (NS sums and the edge per slot) in 128 registers; 168 from 17 on.
template <int NS>
__host__ __device__ constexpr int fwg_most() { return NS == 4 ? 7 : NS == 2 ? 12 : 24; }
template <int NS, int NE>
__host__ __device__ constexpr int fwg_waves_per_simd() { return NS == 1 && NE > 16 ? 3 : 4; }

// One work item: slices b0 .. b0 + NS - 1 (one past the batch repeats the last and is not stored),
// sweep axis `mode`, views vlist[grp*G .. grp*G+G-1] of that axis, G = waves / EH, image lines [lb, le).
// Wave w has view w % G and its edges half*64*NE + 64 i + b128_pos(lane), half = w / G < EH: a view's
// edges are split over EH waves where one wave's registers do not hold them.  `lt` points at line 0
// of the axis in slice b0 (NS = 4: in the packed group), slices `stride` entries apart.  Per step of LB lines the tables are copied
// global -> LDS one step ahead (copy_to_lds16; the allocation ends with a chunk to spare), with one
// wait for this wave's copies and one bare barrier.  EXTRA: D == EH*64*NE, so that
// edge D has no slot; the last wave of each view evaluates it as one slot more, in all lanes alike.
template <typename T, int NS, int NE, int M, bool RESID, bool EXTRA>
__device__ __forceinline__ void fwd_group(const DevPlan& P, const double2* __restrict__ lt, size_t stride,
                                          T* __restrict__ y, int b0, int B, int mode, int grp, int EH,
                                          const double* __restrict__ post, const T* __restrict__ m,
                                          double2* __restrict__ tabs, unsigned char* __restrict__ smem, int lb, int le,
                                          double* __restrict__ rowsq) {
    constexpr int NW = fwg_waves<NS>(), LB = fwg_lines<NS, M>(), TABN = ltab_n<M>(), PITCH = fwg_pitch<M>();
    constexpr int LROWS = fwg_line_rows<NS>(), ROWS = fwg_rows<NS, M>();
    constexpr bool PACKED = NS == 4;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // a caller's loop over work items keeps nothing derived from it in registers
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = NW / EH, half = wave / G, vi = wave % G;
    const int* vlist = mode == MODE_Y ? P.yviews : P.xviews;
    const int nv = mode == MODE_Y ? P.ny : P.nx;
    const int n = mode == MODE_Y ? P.H : P.W;
    const int D = P.D;
    const int hi = n + 1;
    const bool extra = EXTRA && half == EH - 1;  // uniform
    const int view = __builtin_amdgcn_readfirstlane(vlist[min(grp * G + vi, nv - 1)]);
    const char* lines = scalar_ptr(reinterpret_cast<const char*>(P.lines + (size_t)view * P.max_lines));

    double e[NE], S[NS][NE];
    const int k0 = half * 64 * NE + b128_pos(lane);
#pragma unroll
    for (int i = 0; i < NE; i++) {
        e[i] = P.edges[(size_t)view * (D + 1) + min(k0 + 64 * i, D)];
#pragma unroll
        for (int s = 0; s < NS; s++) S[s][i] = 0.0;
    }
    const double ex = EXTRA ? P.edges[(size_t)view * (D + 1) + D] : 0.0;
    double Sx[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) Sx[s] = 0.0;

    const unsigned lds0 = lds_address(smem);
    // row r of a line: packed, row r of the line's three; else the line's table of slice b0 + r
    const char* tsrc = reinterpret_cast<const char*>(lt);
    const size_t row_step = 16 * (PACKED ? (size_t)TABN : B - 1 > b0 ? stride : 0);
    auto issue = [&](int l, int buf) {
#pragma unroll
        for (int r = 0; r < ROWS; r++) {
            const int ln = r / LROWS;
            if (ln && l + ln >= le) break;
            const char* src = tsrc + (size_t)(l + ln) * ((PACKED ? 3 : 1) * TABN * 16) + (r % LROWS) * row_step;
            const unsigned dst = lds0 + 16 * (buf * ROWS + r) * PITCH;
            // chunks of 64 entries, the first at a wave of the row's own, so that every wave has its share
            const int first = (wave + 3 * r) % NW;
#pragma unroll
            for (int c = 0; c < (PITCH + 63) / 64; c += NW) {
                if ((c + first) * 64 >= n + 2) break;
                if (lane < n + 2 - 64 * (c + first)) copy_to_lds16(scalar_ptr(src + 1024 * (c + first)), 16 * lane, dst + 1024 * (c + first));
            }
        }
    };

    // Line coefficients s and {A, B}, loaded one line ahead, by vector loads of one address: after scalar
    // ones the first wait for an LDS read waits for all of them (8 % of the time, measured).
    unsigned zero = 0;
    asm("" : "+v"(zero));
    double ns = 0.0;
    double2 nab = make_double2(0.0, 0.0);
    auto load_coef = [&](int l) {
        const char* c = lines + (size_t)l * sizeof(LineCoef);
        asm("" : "+s"(c));  // uniform base, lane offset zero
        ns = *reinterpret_cast<const double*>(c + zero + 8 * LC_S);
        nab = *reinterpret_cast<const double2*>(c + zero + 8 * LC_A);
    };
    if (lb < le) {
        issue(lb, 0);
        load_coef(lb);
    }
    for (int l = lb; l < le; l++) {
        const int q = (l - lb) % LB, buf = (l - lb) / LB & 1;  // line q of buffer buf
        const double sc = ns, A = nab.x, Bc = nab.y;
        const char* t0 = reinterpret_cast<const char*>(smem) + (size_t)(buf * ROWS + q * LROWS) * PITCH * 16;
        // the reads of AHEAD slots are under way while one is used
        constexpr int AHEAD = NS == 1 ? 3 : NS == 4 || (EXTRA && NE > 8) ? 1 : 2;
        double tau[AHEAD + 1];
        const char* at[AHEAD + 1];
        struct Entries {
            double2 e[PACKED ? 2 : NS];
            float4 s;
        } ent[AHEAD + 1];
        auto address = [&](int i) {
            const int r = i % (AHEAD + 1);
            tau[r] = __builtin_fma(A, e[i], Bc);
            at[r] = t0 + 16 * table_index_u(tau[r], hi);
        };
        auto entries_at = [&](const char* a) {
            Entries t;
            if constexpr (PACKED) {
                t.e[0] = *reinterpret_cast<const double2*>(a);
                t.e[1] = *reinterpret_cast<const double2*>(a + PITCH * 16);
                t.s = *reinterpret_cast<const float4*>(a + 2 * PITCH * 16);
            } else {
#pragma unroll
                for (int s = 0; s < NS; s++) t.e[s] = *reinterpret_cast<const double2*>(a + (size_t)s * PITCH * 16);
            }
            return t;
        };
        auto read = [&](int i) { ent[i % (AHEAD + 1)] = entries_at(at[i % (AHEAD + 1)]); };
        auto integral = [&](const Entries& t, int s, double u) {  // F at u pixels of slice s
            if constexpr (PACKED) {
                const float sl = s == 0 ? t.s.x : s == 1 ? t.s.y : s == 2 ? t.s.z : t.s.w;
                return __builtin_fma(u, (double)sl, s & 1 ? t.e[s / 2].y : t.e[s / 2].x);
            } else {
                return __builtin_fma(u, t.e[s].y, t.e[s].x);
            }
        };
#pragma unroll
        for (int i = 0; i < AHEAD; i++) address(i);
        if (q == 0) {
            // this wave's copies of these lines have landed; after the barrier everybody's
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            if (l + LB < le) issue(l + LB, buf ^ 1);
        }
#pragma unroll
        for (int i = 0; i < AHEAD; i++) read(i);
        load_coef(min(l + 1, le - 1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NE; i++) {
            if (i + AHEAD < NE) {
                address(i + AHEAD);
                read(i + AHEAD);
            }
            const int r = i % (AHEAD + 1);
#pragma unroll
            for (int s = 0; s < NS; s++) {
                S[s][i] = __builtin_fma(sc, integral(ent[r], s, tau[r]), S[s][i]);
                asm volatile("" : "+v"(S[s][i]));  // keeps the sums in the loop
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (extra) {
            const double tx = __builtin_fma(A, ex, Bc);
            const Entries t = entries_at(t0 + 16 * table_index_u(tx, hi));
#pragma unroll
            for (int s = 0; s < NS; s++) Sx[s] = __builtin_fma(sc, integral(t, s, tx), Sx[s]);
        }
    }

    // Bin values.  The sums back in lane order; the edge right of a wave's last one is the next wave's
    // first, exchanged through LDS (or edge D); RESID: the running sum of the residual table goes from
    // wave to wave of a view.
    double* first_edge = reinterpret_cast<double*>(smem);  // [NW][NS]
    double* carry_at = first_edge + NW * NS;               // [G][NS][2]: running sum, sum of squares
    if (EH > 1) __syncthreads();
    const int src = 4 * b128_pos(lane);
#pragma unroll
    for (int s = 0; s < NS; s++) {
#pragma unroll
        for (int i = 0; i < NE; i++) {
            int2 w = __builtin_bit_cast(int2, S[s][i]);
            w.x = __builtin_amdgcn_ds_bpermute(src, w.x);
            w.y = __builtin_amdgcn_ds_bpermute(src, w.y);
            S[s][i] = __builtin_bit_cast(double, w);
        }
        if (EH > 1 && lane == 0) first_edge[wave * NS + s] = S[s][0];
    }
    if (EH > 1) __syncthreads();
    const bool valid = grp * G + vi < nv;
    const bool rev = P.vp[view].rev;
    const double* pr = post + (size_t)view * D;
    const double* ev = P.edges + (size_t)view * (D + 1);
    for (int h = 0; h < (RESID ? EH : 1); h++) {
        if (valid && (!RESID || half == h)) {
#pragma unroll
            for (int s = 0; s < NS; s++) {
                const int b = b0 + s;
                if (b >= B) break;
                const size_t row = (size_t)b * P.V + view;
                const double beyond = half + 1 < EH ? first_edge[(wave + G) * NS + s] : Sx[s];
                double2* tb = RESID ? tabs + row * (D + 2) : nullptr;
                double carry = 0.0, rsq = 0.0;
                if (RESID && h) carry = carry_at[(vi * NS + s) * 2];
#pragma unroll
                for (int i = 0; i < NE; i++) {
                    const int k = half * 64 * NE + 64 * i + lane;
                    double nxt = shfl_next_d(S[s][i]);
                    const double r0 = i + 1 < NE ? readlane_d(S[s][i + 1 < NE ? i + 1 : i], 0) : beyond;
                    if (lane == 63) nxt = r0;
                    double yk = nxt - S[s][i];
                    if (k < D) yk *= pr[k];
                    const int o = rev ? D - 1 - k : k;
                    if (!RESID) {
                        if (k < D) y[row * D + o] = (T)yk;
                    } else {
                        double gk = 0.0, ek = 0.0, wg = 0.0;
                        if (k < D) {
                            if (y) y[row * D + o] = (T)yk;
                            const double mk = (double)m[row * D + o];
                            gk = (yk - mk) * pr[k];
                            const double rk = (double)(T)yk - mk;
                            rsq = __builtin_fma(rk, rk, rsq);
                            ek = ev[k];
                            wg = (ev[k + 1] - ek) * gk;
                        }
                        const double inc = wave_scan_incl(wg, lane);
                        if (k < D) tb[k + 1] = make_double2(carry + (inc - wg) - ek * gk, gk);
                        carry += readlane_d(inc, 63);
                        __builtin_amdgcn_sched_barrier(0);  // one slot's loads at a time: registers
                    }
                }
                if (RESID) {
                    double tot = readlane_d(wave_scan_incl(rsq, lane), 63);
                    if (h) tot += carry_at[(vi * NS + s) * 2 + 1];
                    if (lane == 0) {
                        if (h == 0) tb[0] = make_double2(0.0, 0.0);
                        if (h == EH - 1) {
                            tb[D + 1] = make_double2(carry, 0.0);
                            if (rowsq) rowsq[row] = tot;
                        } else {
                            carry_at[(vi * NS + s) * 2] = carry;
                            carry_at[(vi * NS + s) * 2 + 1] = tot;
                        }
                    }
                }
            }
        }
        if (RESID && EH > 1) __syncthreads();
    }
}

}  // namespace dd

namespace {

// One launch covers both sweep axes: work items [0, ngrp*ngx) are (slice group, G X-axis views), the
// rest (slice group, G Y-axis views); with nch > 1 each is split into nch chunks of its axis's lines,
// chunk k writing its partial sinogram k*B*V*D elements into y.
template <typename T, int NS, int NE, int M, bool RESID, bool EXTRA>
__global__ __launch_bounds__((64 * dd::fwg_waves<NS>()), (dd::fwg_waves_per_simd<NS, NE>())) void k_fwd_lt(DevPlan P, const double2* __restrict__ lt, T* __restrict__ y,
                                                                 int B, int ngrp, int ngx, int ngy, int EH,
                                                                 const double* __restrict__ post, const T* __restrict__ m,
                                                                 double2* __restrict__ tabs, int nch,
                                                                 double* __restrict__ rowsq) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int nwx = ngrp * ngx;
    int w = dd::xcd_remap(blockIdx.x, gridDim.x, (nwx + ngrp * ngy) * nch);
    if (w < 0) return;
    const int ch = w % nch;
    w /= nch;
    const int mode = w < nwx ? MODE_X : MODE_Y;
    if (mode == MODE_Y) w -= nwx;
    const int ngroups = mode == MODE_Y ? ngy : ngx;
    const int sg = w / ngroups, grp = w - sg * ngroups;
    const int nl = mode == MODE_Y ? P.W : P.H;
    const int hx = P.nx ? P.H : 0, wy = P.ny ? P.W : 0;
    const size_t stride = (size_t)(hx + wy) * ((NS == 4 ? 3 : 1) * dd::ltab_n<M>());  // of a slice, or of a packed group
    const int b0 = sg * NS;
    const double2* lts = lt + (NS == 4 ? sg : b0) * stride + (size_t)(mode == MODE_Y ? hx : 0) * ((NS == 4 ? 3 : 1) * dd::ltab_n<M>());
    T* yc = y ? y + (size_t)ch * B * P.V * P.D : nullptr;
    dd::fwd_group<T, NS, NE, M, RESID, EXTRA>(P, lts, stride, yc, b0, B, mode, grp, EH, post, m, tabs, smem, ch * nl / nch,
                                       (ch + 1) * nl / nch, rowsq);
}

template <typename T, int NS, int NE, int M, bool RESID, bool EXTRA>
hipError_t fwg_launch(const DevPlan& P, const FwdGroupArgs& a, int EH, hipStream_t s) {
    const int G = dd::fwg_waves<NS>() / EH;
    const int ngx = (P.nx + G - 1) / G, ngy = (P.ny + G - 1) / G, ngrp = (a.B + NS - 1) / NS;
    const long long nw = (long long)(ngx + ngy) * ngrp * a.nch;
    if (nw > (1LL << 30)) return hipErrorInvalidValue;  // grid size (one block per work item)
    const size_t lds = dd::fwg_lds<NS, M>();
    auto kern = k_fwd_lt<T, NS, NE, M, RESID, EXTRA>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(dd::grid_for((int)nw)), dim3((unsigned)(64 * dd::fwg_waves<NS>())), lds, s, P, a.lt, (T*)a.y, a.B, ngrp,
                       ngx, ngy, EH, a.post, (const T*)a.m, a.tabs, a.nch, a.rowsq);
    return hipGetLastError();
}

// Slots per wave: as many as the registers hold, beyond that a view's edges go over two or four waves.
// Detectors of whole slots have their edge D taken apart instead of opening another slot.
template <typename T, int NS, int M, bool RESID, bool EXTRA, int NE = 3>
hipError_t fwg_edges(const DevPlan& P, const FwdGroupArgs& a, int per, int EH, hipStream_t s) {
    if constexpr (NE > dd::fwg_most<NS>()) {
        return hipErrorInvalidValue;
    } else if constexpr ((NE > 8 && NE % 2) || (NE > 16 && NE % 4)) {
        return fwg_edges<T, NS, M, RESID, EXTRA, NE + 1>(P, a, per, EH, s);
    } else {
        if (per <= NE) return fwg_launch<T, NS, NE, M, RESID, EXTRA>(P, a, EH, s);
        return fwg_edges<T, NS, M, RESID, EXTRA, NE + 1>(P, a, per, EH, s);
    }
}

template <typename T, int NS, int M>
hipError_t fwg_detector(const DevPlan& P, const FwdGroupArgs& a, hipStream_t s) {
    const bool whole = whole_slots(P);
    const int ne = edge_slots(P);
    int EH = 1;
    while ((ne + EH - 1) / EH > dd::fwg_most<NS>()) EH *= 2;
    if (EH > dd::fwg_waves<NS>()) return hipErrorInvalidValue;
    const int per = (ne + EH - 1) / EH;
    if (whole)
        return a.tabs ? fwg_edges<T, NS, M, true, true>(P, a, per, EH, s) : fwg_edges<T, NS, M, false, true>(P, a, per, EH, s);
    return a.tabs ? fwg_edges<T, NS, M, true, false>(P, a, per, EH, s) : fwg_edges<T, NS, M, false, false>(P, a, per, EH, s);
}

template <typename T, int M>
hipError_t fwg_slices(const DevPlan& P, const FwdGroupArgs& a, hipStream_t s) {
    switch (fwd_slices(P, sizeof(T) == 4 ? DT_F32 : DT_F64, a.B, a.nch)) {
    case 4:
        if constexpr (sizeof(T) == 4 && M <= 2) return fwg_detector<T, 4, M>(P, a, s);
        return hipErrorInvalidValue;
    case 2: return fwg_detector<T, 2, M>(P, a, s);
    default: return fwg_detector<T, 1, M>(P, a, s);
    }
}

template <typename T>
hipError_t fwg_px(const DevPlan& P, const FwdGroupArgs& a, hipStream_t s) {
    switch (line_table_px(P)) {
    case 1: return fwg_slices<T, 1>(P, a, s);
    case 2: return fwg_slices<T, 2>(P, a, s);
    case 4: return fwg_slices<T, 4>(P, a, s);
    case 8: return fwg_slices<T, 8>(P, a, s);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace
}  // namespace ctlib
