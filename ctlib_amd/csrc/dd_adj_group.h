// Bin -> pixel kernel (projection_t / backprojection) over a group of slices (gfx950).
//
// The bin that a pixel edge falls into depends on the view and the line, not on the slice, so one
// work item evaluates the lookup once and reads the tables of NS slices with it: per edge 9 VALU
// cycles for the lookup (two FMAs, reciprocal, product, clamp, conversion, address, the fp64 edge
// coordinate) and two FP64 operations and one 16-byte ds_read per slice.  fan-EA's polynomial
// arctangent adds 9 to the shared part.
//
// Lane layout.  ds_read_b128 serves a wave in four passes of 16 lanes, lanes {0-3, 12-15, 20-27},
// {4-11, 16-19, 28-31} and the same 32 lanes further, over 16 slots of 16 bytes; lanes of one pass
// that hit different entries of one slot cost another pass.  A pixel is 1.2 to 1.7 bins wide at the
// measured geometries, so 16 neighbouring pixel edges span 20 to 28 entries and collide (8 to 12
// cycles per read, measured).  Here each pass holds 8 neighbouring edges of two neighbouring lines,
// whose edges fall into nearly the same bins: its span stays within 16 entries up to about 1.8 bins
// per pixel and a read costs 5.1 cycles, the conflict-free rate.
//
// Measured (k_adj alone, fp32 unless marked; before = one slice per block, lanes along one line):
//   projection_t   fan-ED 512^2, 736 x 736, B=32   2.30 -> 1.35 ms
//                  fan-EA 512^2, 1024 x 888, B=16  2.38 -> 1.15 ms
//                  fan-ED 1024^2, 1440 x 1536, B=4 2.65 -> 1.50 ms (two slices per block)
//                  fan-ED 512^2, B=8, fp64         0.87 -> 0.42 ms
//   backprojection fan-ED 512^2, B=8               0.87 -> 0.60 ms
//                  fan-EA 512^2, B=16              3.21 -> 1.98 ms
//                  fan-EA 512^2, B=4, fp64         2.33 -> 1.06 ms
// Of the 1.35 ms at B=32 the VALU is busy 60 %, the LDS reads 55 %; the copies of the tables into LDS
// (1.4 bytes per 16 read) cost 0.18 ms and the barrier per view 0.09 ms (both measured by leaving
// them out where the tables do not change).
#pragma once
#include "dd_device.h"

namespace ctlib {
namespace dd {

// Waves per block, and the slots a wave can have: 64 accumulator registers at 16 waves (128 VGPRs
// each), 128 at 8, 32 at NS = 1 (more blocks per CU).  Four waves per SIMD hide the reads best
// (projection_t at fan-ED 512^2, B=32: 1.33 ms against 1.47 with two), but the weighted and fp64
// indices take too many registers for that: what spills waits for the copies under way.
template <typename T, int NS, bool WEIGHTED>
__host__ __device__ constexpr int adjg_waves() { return NS > 1 && sizeof(T) == 4 && !WEIGHTED ? 16 : 8; }
template <typename T, int NS, bool WEIGHTED>
__host__ __device__ constexpr int adjg_most(bool arctan) {
    if (NS == 1) return 16;
    if (sizeof(T) == 4) return 32 / NS;
    if (WEIGHTED) return NS == 4 ? 4 : arctan ? 8 : 10;
    return (arctan ? 40 : 64) / NS;
}
// Slots with a kernel of their own: from half of the most on (fewer slots per wave: more waves along
// the line instead), even ones in steps of an eighth, and 4 and 6.
__host__ __device__ constexpr int adjg_slot_step(int most) { return most >= 32 ? 4 : 2; }
__host__ __device__ constexpr bool adjg_has_slots(int most, int SL) {
    return SL <= most && ((SL >= most / 2 && SL % adjg_slot_step(most) == 0) || SL == 4 || SL == 6);
}
// The distance of the slices' tables in LDS (entries), fixed for NS > 1, which makes the slice an
// immediate offset of the read.
template <int NS>
__host__ __device__ constexpr int adjg_pitch(int D) { return NS == 4 ? 1024 : NS == 2 ? 2048 : (D + 2 + 63) / 64 * 64; }
// Largest number of bins of a group of NS slices (table of D + 2 entries within the pitch).
template <int NS>
__host__ __device__ constexpr int adjg_max_bins() { return NS == 4 ? 1022 : 2046; }

// Bytes of one line's coefficients in LDS: {a, s}; fp32 data: composed lookup {64 c0, c1, 64 c2, c3}
// [and pre-scaled weight]; fp64 data, weighted: the whole LineCoef.  Before them the view's: fan-EA's
// angle -> bin scale and offset (fp32 data) or the lookup (fp64 data).
constexpr int ADJG_HEAD = 48;
template <typename T, bool WEIGHTED>
__host__ __device__ constexpr int adjg_side() { return sizeof(T) == 4 ? (WEIGHTED ? 48 : 32) : (WEIGHTED ? 64 : 16); }

// LDS bytes: double-buffered tables and coefficients, reused for the edge sums at the end; then the
// sums of the lines' edges past the slots, [L][NS].
template <typename T, int NS, bool WEIGHTED>
__host__ __device__ inline size_t adjg_lds_loop(int D, int L, int cover) {
    const size_t loop = 2 * NS * (size_t)adjg_pitch<NS>(D) * 16 + 2 * (ADJG_HEAD + (size_t)L * adjg_side<T, WEIGHTED>());
    const size_t sums = ((size_t)L * (cover + 1) + 1) / 2 * 16;
    return loop > sums ? loop : sums;
}
template <typename T, int NS, bool WEIGHTED>
inline size_t adjg_lds(int D, int L, int cover) {
    return adjg_lds_loop<T, NS, WEIGHTED>(D, L, cover) + (size_t)L * NS * 8;
}

// One work item: slices b0 .. b0 + NS - 1 (those past the batch repeat the last one and are not
// stored), sweep axis `mode`, image lines [tile*L, tile*L + L) (rows for X, columns bottom-to-top
// for Y), views [vb, ve) of the axis list.  The block's waves form LP = waves / PH line pairs
// (L = 2 LP) times PH pixel parts of 32*SL edges each: wave w owns lines 2 (w % LP) + {0, 1} and
// edges (w / LP)*32*SL + 32 i + 8 g + k, with lane position q = b128_pos(lane) = 16 g + 8 line + k.
// X lines are written to outX [B][H][W], Y lines to outYT [B][W][H].
//
// Unweighted: acc = sum_v G_v(edge), pixel p = acc_{p+1} - acc_p.  Weighted: with the pixel weight
// w_v(p) the pixel is sum_v w_v(p) G_v(p+1) - sum_v w_v(p) G_v(p); each edge accumulates both its
// terms, w_v(p) G and w_v(p-1) G, so that only the weight, which the slices share, crosses lanes
// (exchanging the edges' values cost five instructions per edge and slice).  w_v is a function of
// the pixel index alone, so the two products of a pixel carry the same weight to the bit.
// With n == PH*32*SL the last edge n has no slot: lanes < L evaluate it for line `lane`, the waves
// taking the views in turn, into sums in LDS (one wave between two barriers).
//
// Per view the next view's tables are copied global -> LDS (copy_to_lds16) into the other buffer,
// whole 64-entry chunks (entries past the row are never looked up; the table allocation ends with a
// chunk to spare), and the next view's coefficients beside them: one wait for this wave's copies and
// one bare barrier per view.  Nothing in the loop is read by scalar loads, which would have the wave
// wait for all its LDS reads.
template <typename T, int NS, int SL, bool WEIGHTED, int GEO, int NW = adjg_waves<T, NS, WEIGHTED>()>
__device__ __forceinline__ void adj_group(const DevPlan& P, const double2* __restrict__ tabs, T* __restrict__ outX,
                                          T* __restrict__ outYT, int b0, int B, int mode, int tile, int PH,
                                          double wscale, unsigned char* __restrict__ smem, int vb, int ve) {
    constexpr bool F32 = sizeof(T) == 4;
    constexpr int NA = WEIGHTED ? 2 : 1;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // a caller's loop over work items keeps nothing derived from it in registers
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int LP = NW / PH, L = 2 * LP;
    const int* vlist = mode == MODE_Y ? P.yviews : P.xviews;
    const int nlines = mode == MODE_Y ? P.W : P.H;
    const int n = mode == MODE_Y ? P.H : P.W;
    const int D = P.D;
    const float hi = (float)(D + 1);
    const int tabn = D + 2;
    const int pitch = adjg_pitch<NS>(D);
    const int cover = PH * 32 * SL;

    double2* stab = reinterpret_cast<double2*>(smem);  // [2][NS][pitch]
    const int SIDE_BUF = ADJG_HEAD + L * adjg_side<T, WEIGHTED>();
    unsigned char* side = smem + (size_t)2 * NS * pitch * 16;  // [2] of the coefficients
    const unsigned lds0 = lds_address(smem), side0 = lds0 + 2 * NS * pitch * 16;
    // wave w copies slice w % NS, chunks w / NS, w / NS + NW / NS, ...
    const char* tsrc = reinterpret_cast<const char*>(tabs + (size_t)min(b0 + wave % NS, B - 1) * P.V * tabn +
                                                     (wave / NS) * 64);
    auto issue = [&](int v, int buf) {
        const char* src = tsrc + (size_t)v * tabn * sizeof(double2);
        const unsigned dst = lds0 + 16 * ((buf * NS + wave % NS) * pitch + (wave / NS) * 64);
        constexpr int STEP = 64 * (NW / NS), MOST = (NS == 4 ? 1024 : 2048) / STEP;
#pragma unroll
        for (int r = 0; r < MOST; r++) {
            if ((wave / NS) * 64 + r * STEP >= tabn) break;
            copy_to_lds16(src, 16 * (lane + r * STEP), dst + 16 * r * STEP);
        }
        const unsigned sd = side0 + buf * SIDE_BUF;
        const size_t row = (size_t)v * P.max_lines;
        const unsigned l = min(tile * L + lane, nlines - 1);
        if (wave == 0) {
            if (!F32 && lane < 3) copy_to_lds16(P.lookup_d + (size_t)v * 6, 16 * lane, sd);
            if (F32 && (GEO == GEO_EA || GEO == GEO_EAP) && lane < 1) copy_to_lds16(&P.vp[v].ea_sc, 0, sd);
        }
        if constexpr (!F32 && WEIGHTED) {
            const unsigned l4 = min(tile * L + (tid >> 2), nlines - 1);
            if (tid < 4 * L) copy_to_lds16(P.lines + row, 64 * l4 + 16 * (tid & 3), sd + ADJG_HEAD + 1024 * wave);
        } else if (lane < L) {
            if (wave == 1) copy_to_lds16(P.lines + row, 64 * l, sd + ADJG_HEAD);
            if (F32 && wave == 2) copy_to_lds16(P.adj_lk + row, 16 * l, sd + ADJG_HEAD + 16 * L);
            if (F32 && WEIGHTED && wave == 3) copy_to_lds16(P.adj_wk + row, 16 * l, sd + ADJG_HEAD + 32 * L);
        }
    };

    const int pos = b128_pos(lane);
    const int lq = 2 * (wave % LP) + ((pos >> 3) & 1);                      // this lane's line of the tile
    const int px0 = (wave / LP) * 32 * SL + ((pos >> 4) << 3) + (pos & 7);  // and its edge of slot 0
    const bool extra = n == cover;
    float h[(SL + 1) / 2];  // uniform: 64-edge group of slots 2k and 2k + 1 (SL is even where PH > 1)
#pragma unroll
    for (int k = 0; k < (SL + 1) / 2; k++)
        h[k] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (float)((wave / LP) * (SL / 2) + k))));

    struct Coef {
        double2 as;
        float4 lk, wk;
        float2 ea;
        double4 wd;
        double lkd[6];
    };
    // coefficients of line l of the tile from side buffer sd
    auto load_coef = [&](const unsigned char* sd, int l) {
        Coef c;
        const unsigned char* ls = sd + ADJG_HEAD;
        c.as = *reinterpret_cast<const double2*>(ls + (!F32 && WEIGHTED ? 64 : 16) * l);
        if constexpr (F32) {
            c.lk = *reinterpret_cast<const float4*>(ls + 16 * L + 16 * l);
            if constexpr (WEIGHTED) c.wk = *reinterpret_cast<const float4*>(ls + 32 * L + 16 * l);
            if constexpr (GEO == GEO_EA || GEO == GEO_EAP) c.ea = *reinterpret_cast<const float2*>(sd);
        } else {
            if constexpr (WEIGHTED) c.wd = *reinterpret_cast<const double4*>(ls + 64 * l + 32);
#pragma unroll
            for (int k = 0; k < (GEO == GEO_PARA ? 2 : GEO == GEO_ED ? 4 : 6); k++)
                c.lkd[k] = reinterpret_cast<const double*>(sd)[k];
        }
        return c;
    };
    // pixel weight as a function of the pixel index alone
    auto weight = [](const Coef& c, float p) -> T {
        if constexpr (F32) {
            const float u = __builtin_fmaf(p, c.wk.y, c.wk.z);
            return __builtin_amdgcn_rcpf(__builtin_fmaf(u, u, c.wk.w));
        } else {
            const double u = __builtin_fma(c.wd.y, (double)p, c.wd.x);
            return c.wd.w * rcp_refined(__builtin_fma(u, u, c.wd.z));
        }
    };

    // The weight of the pixel left of this lane's edge: the neighbouring lane's, for the first lane of
    // a run of 8 that of the last lane of the run before - of the slot before if it is the last run.
    const int left_pos = (pos & 7) ? pos - 1 : ((pos - 16) & 0x30) | (pos & 8) | 7;
    const int left_lane = 4 * b128_pos(left_pos);
    const bool last = (pos & 0x37) == 0x37;
    auto from_left = [&](T here, T before) -> T {
        const T give = last ? before : here;
        if constexpr (F32) {
            return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(left_lane, __builtin_bit_cast(int, give)));
        } else {
            int2 w = __builtin_bit_cast(int2, give);
            w.x = __builtin_amdgcn_ds_bpermute(left_lane, w.x);
            w.y = __builtin_amdgcn_ds_bpermute(left_lane, w.y);
            return __builtin_bit_cast(double, w);
        }
    };

    double acc[NA][NS][SL];
#pragma unroll
    for (int k = 0; k < NA; k++)
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int i = 0; i < SL; i++) acc[k][s][i] = 0.0;
    double* xs = reinterpret_cast<double*>(smem + adjg_lds_loop<T, NS, WEIGHTED>(D, L, cover));  // [L][NS]
    if (tid < L * NS) xs[tid] = 0.0;

    int ahead = vlist[min(vb + lane, ve - 1)];  // the next 64 views, one per lane
    issue(__builtin_amdgcn_readfirstlane(ahead), 0);

    for (int iv = vb; iv < ve; iv++) {
        const int buf = (iv - vb) & 1;
        // this wave's copies of view iv have landed; after the barrier everybody's
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const unsigned char* sd = side + buf * SIDE_BUF;
        const Coef c = load_coef(sd, lq);
        if (iv + 1 < ve) {
            if (((iv + 1 - vb) & 63) == 0) ahead = vlist[min(iv + 1 + lane, ve - 1)];
            issue(__builtin_amdgcn_readlane(ahead, (iv + 1 - vb) & 63), buf ^ 1);
        }
        // table index of the edge with lookup argument num / den (fp32 data)
        auto index_f = [&](float num, float den) {
            float q = num;
            if (GEO != GEO_PARA) q = num * __builtin_amdgcn_rcpf(den);
            if (GEO == GEO_EA) q = __builtin_fmaf(atanf(q), c.ea.x, c.ea.y);
            if (GEO == GEO_EAP) {
                const float tc = __builtin_amdgcn_fmed3f(q, -P.ea_T, P.ea_T);
                const float s2 = tc * tc;
                float z = P.ea_c[5];
#pragma unroll
                for (int k = 4; k >= 0; k--) z = __builtin_fmaf(z, s2, P.ea_c[k]);
                q = __builtin_fmaf(tc * z, c.ea.x, c.ea.y);
            }
            return table_index(q, hi);
        };
        // of the edge at axis coordinate pi (fp64 data)
        auto index_d = [&](double pi) {
            double q;
            if (GEO == GEO_PARA) {
                q = __builtin_fma(c.lkd[0], pi, c.lkd[1]);
            } else {
                q = __builtin_fma(c.lkd[0], pi, c.lkd[1]) * rcp_refined(__builtin_fma(c.lkd[2], pi, c.lkd[3]));
                if (GEO == GEO_EA || GEO == GEO_EAP) q = __builtin_fma(atan(q), c.lkd[4], c.lkd[5]);
            }
            return table_index_d(q, D + 1);
        };
        const double pi0 = __builtin_fma(c.as.y, (double)px0, c.as.x), s32 = 32.0 * c.as.y;
        // lookup argument of edge p: p = 64 h + r with r < 64, numerator (c0 r + c1) + h (64 c0); even
        // slots have this lane's r < 32, odd ones r + 32
        float n0[2] = {0.f, 0.f}, d0[2] = {0.f, 0.f};
        if constexpr (F32) {
#pragma unroll
            for (int o = 0; o < 2; o++) {
                const float r64 = (float)((px0 & 31) + 32 * o) * (1.0f / 64.0f);  // exact
                n0[o] = __builtin_fmaf(c.lk.x, r64, c.lk.y);
                d0[o] = __builtin_fmaf(c.lk.z, r64, c.lk.w);
            }
        }
        auto edge_pi = [&](int i) { return i == 0 ? pi0 : __builtin_fma((double)i, s32, pi0); };
        const char* t0 = reinterpret_cast<const char*>(stab + (size_t)buf * NS * pitch);
        auto table_at = [&](int i) {
            int j;
            if constexpr (F32)
                j = index_f(__builtin_fmaf(h[i / 2], c.lk.x, n0[i & 1]), __builtin_fmaf(h[i / 2], c.lk.z, d0[i & 1]));
            else
                j = index_d(edge_pi(i));
            return t0 + 16 * j;
        };
        // U slots (4 reads) per step; the reads of a step are issued before the step ahead of it is used,
        // and no further: more in flight costs more registers than four waves per SIMD have
        constexpr int U = 4 / NS;
        double2 e[2][U][NS];
        auto read = [&](int i0, const char* const (&t)[U]) {
            const int q = (i0 / U) & 1;
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u < SL)
#pragma unroll
                    for (int k = 0; k < NS; k++) e[q][u][k] = *reinterpret_cast<const double2*>(t[u] + (size_t)k * pitch * 16);
        };
        auto indices = [&](int i0, const char* (&t)[U]) {
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u < SL) t[u] = table_at(i0 + u);
        };
        const char* t[U];
        indices(0, t);
        read(0, t);
        if (extra && (iv - vb) % NW == wave) {  // wave-uniform
            const int lx = min(lane, L - 1);
            const Coef cx = load_coef(sd, lx);
            const double px = __builtin_fma(cx.as.y, (double)n, cx.as.x);
            int j;
            if constexpr (F32) {
                const float p64 = (float)n * (1.0f / 64.0f);
                j = index_f(__builtin_fmaf(cx.lk.x, p64, cx.lk.y), __builtin_fmaf(cx.lk.z, p64, cx.lk.w));
            } else {
                j = index_d(px);
            }
            const double w = WEIGHTED ? (double)weight(cx, (float)(n - 1)) : 1.0;
            if (lane < L)
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    const double2 g = *reinterpret_cast<const double2*>(t0 + 16 * j + (size_t)k * pitch * 16);
                    double* x = xs + lane * NS + k;
                    *x = __builtin_fma(w, __builtin_fma(px, g.y, g.x), *x);
                }
        }
        indices(U, t);
        __builtin_amdgcn_sched_barrier(0);
        double pi = pi0;
        // weights of the pixels right and left of the step's edges, one step ahead
        T wr[2][U], wl[2][U], wbefore = T(0);
        auto weights = [&](int i0) {
            const int q = (i0 / U) & 1;
#pragma unroll
            for (int u = 0; u < U; u++)
                if (i0 + u < SL) {
                    wr[q][u] = weight(c, (float)px0 + 32.0f * (i0 + u));
                    wl[q][u] = from_left(wr[q][u], wbefore);
                    wbefore = wr[q][u];
                }
        };
        if constexpr (WEIGHTED) {
            wbefore = weight(c, (float)px0 - 32.0f);
            weights(0);
        }
#pragma unroll
        for (int i0 = 0; i0 < SL; i0 += U) {
            const int q = (i0 / U) & 1;
            if (i0 + U < SL) read(i0 + U, t);
            if (i0 + 2 * U < SL) indices(i0 + 2 * U, t);
            if (WEIGHTED && i0 + U < SL) weights(i0 + U);
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u;
                if (i >= SL) break;
                if (i) pi += s32;
                const double wp = WEIGHTED ? (double)wr[(i0 / U) & 1][u] : 1.0, wm = WEIGHTED ? (double)wl[(i0 / U) & 1][u] : 1.0;
#pragma unroll
                for (int k = 0; k < NS; k++) {
                    const double G = __builtin_fma(pi, e[q][u][k].y, e[q][u][k].x);
                    if constexpr (WEIGHTED) {
                        acc[0][k][i] = __builtin_fma(wp, G, acc[0][k][i]);
                        acc[NA - 1][k][i] = __builtin_fma(wm, G, acc[NA - 1][k][i]);
                    } else {
                        acc[0][k][i] += G;
                    }
                    // holds the sums here: the compiler otherwise sinks them below the last slot
                    asm volatile("" : "+v"(acc[0][k][i]));
                    if constexpr (WEIGHTED) asm volatile("" : "+v"(acc[1][k][i]));
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // The right edge's sum of pixel p sits with edge p + 1, another lane: exchange through LDS.
    double* sums = reinterpret_cast<double*>(smem);  // [L][cover + 1]
    __syncthreads();
    const int l = tile * L + lq;
#pragma unroll
    for (int k = 0; k < NS; k++) {
        const int b = b0 + k;
        if (b >= B) break;  // uniform
        if (k) __syncthreads();
#pragma unroll
        for (int i = 0; i < SL; i++) sums[(size_t)lq * (cover + 1) + px0 + 32 * i] = acc[NA - 1][k][i];
        if (extra && tid < L) sums[(size_t)tid * (cover + 1) + n] = xs[tid * NS + k];
        __syncthreads();
        T* dst = mode == MODE_Y ? outYT + ((size_t)b * P.W + l) * P.H : outX + ((size_t)b * P.H + l) * P.W;
#pragma unroll
        for (int i = 0; i < SL; i++) {
            const int p = px0 + 32 * i;
            if (l < nlines && p < n) {
                dst[p] = (T)((sums[(size_t)lq * (cover + 1) + p + 1] - acc[0][k][i]) * wscale);
            }
        }
    }
}

}  // namespace dd

namespace {

// One launch covers both sweep axes: work items [0, ngrp*ntx) are (slice group, tile of L image rows)
// over the X-axis views, the rest (slice group, tile of columns) over the Y-axis views, written
// bottom-to-top to outYT.  With nch > 1 every item is split into nch chunks of its axis's views;
// chunk k writes its partial image k*B*H*W elements into outX / outYT.
template <typename T, int NS, int SL, bool WEIGHTED, int GEO>
__global__ __launch_bounds__((64 * dd::adjg_waves<T, NS, WEIGHTED>())) void k_adj(DevPlan P, const double2* __restrict__ tabs,
                                                                   T* __restrict__ outX, T* __restrict__ outYT, int B,
                                                                   int ngrp, int ntx, int nty, int PH, double wscale,
                                                                   int nch) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int nwx = ngrp * ntx;
    int w = dd::xcd_remap(blockIdx.x, gridDim.x, (nwx + ngrp * nty) * nch);
    if (w < 0) return;
    const int ch = w % nch;
    w /= nch;
    const int mode = w < nwx ? MODE_X : MODE_Y;
    if (mode == MODE_Y) w -= nwx;
    const int ntiles = mode == MODE_Y ? nty : ntx;
    const int grp = w / ntiles, tile = w - grp * ntiles;
    const int nv = mode == MODE_Y ? P.ny : P.nx;
    const size_t part = (size_t)ch * B * P.H * P.W;
    dd::adj_group<T, NS, SL, WEIGHTED, GEO>(P, tabs, outX + part, outYT + part, grp * NS, B, mode, tile, PH, wscale,
                                            smem, ch * nv / nch, (ch + 1) * nv / nch);
}

template <typename T, int NS, int SL, bool WEIGHTED, int GEO>
hipError_t adj_launch_t(const DevPlan& P, const AdjArgs& a, hipStream_t s) {
    const AdjShape& sh = a.sh;
    if (sh.NS != NS || sh.SL != SL) return hipErrorInvalidValue;
    const int L = sh.L, cover = sh.PH * 32 * SL;
    const int ngrp = (a.B + NS - 1) / NS;
    const int ntx = P.nx ? (P.H + L - 1) / L : 0;
    const int nty = P.ny ? (P.W + L - 1) / L : 0;
    const long long nw = (long long)(ntx + nty) * ngrp * sh.nch;
    if (nw > (1LL << 30)) return hipErrorInvalidValue;  // grid size (one block per work item)
    const size_t lds = dd::adjg_lds<T, NS, WEIGHTED>(P.D, L, cover);
    auto kern = k_adj<T, NS, SL, WEIGHTED, GEO>;
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kern, dim3(dd::grid_for((int)nw)), dim3((unsigned)(64 * dd::adjg_waves<T, NS, WEIGHTED>())), lds, s, P, a.tabs,
                       (T*)a.outX, (T*)a.outYT, a.B, ngrp, ntx, nty, sh.PH, a.wscale, sh.nch);
    return hipGetLastError();
}

template <typename T, int NS, bool WEIGHTED, int GEO, int SL = 2>
hipError_t adj_slots(const DevPlan& P, const AdjArgs& a, hipStream_t s) {
    constexpr int most = dd::adjg_most<T, NS, WEIGHTED>(GEO == dd::GEO_EA || GEO == dd::GEO_EAP);
    if constexpr (SL > most) {
        return hipErrorInvalidValue;
    } else {
        if constexpr (dd::adjg_has_slots(most, SL))
            if (a.sh.SL == SL) return adj_launch_t<T, NS, SL, WEIGHTED, GEO>(P, a, s);
        return adj_slots<T, NS, WEIGHTED, GEO, SL + 1>(P, a, s);
    }
}

template <typename T, bool WEIGHTED, int GEO>
hipError_t adj_slices(const DevPlan& P, const AdjArgs& a, hipStream_t s) {
    switch (a.sh.NS) {
    case 1: return adj_slots<T, 1, WEIGHTED, GEO>(P, a, s);
    case 2: return adj_slots<T, 2, WEIGHTED, GEO>(P, a, s);
    case 4: return adj_slots<T, 4, WEIGHTED, GEO>(P, a, s);
    default: return hipErrorInvalidValue;
    }
}

template <typename T, bool WEIGHTED>
hipError_t adj_geo(const DevPlan& P, const AdjArgs& a, hipStream_t s) {
    if (P.scan_type == dd::GEO_ED) return adj_slices<T, WEIGHTED, dd::GEO_ED>(P, a, s);
    if (P.scan_type != dd::GEO_EA) return adj_slices<T, WEIGHTED, dd::GEO_PARA>(P, a, s);
    // fp64 data takes the arctangent with atan either way
    if (sizeof(T) == 8 || !P.ea_poly) return adj_slices<T, WEIGHTED, dd::GEO_EA>(P, a, s);
    if constexpr (sizeof(T) == 4) return adj_slices<T, WEIGHTED, dd::GEO_EAP>(P, a, s);
    return hipErrorInvalidValue;
}

}  // namespace
}  // namespace ctlib
