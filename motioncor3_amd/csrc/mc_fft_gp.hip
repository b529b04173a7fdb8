// mc_fft_gp.hip -- row and column passes for lengths without a compile-time
// schedule: in-place FFT passes of run-time radices, and Bluestein's
// convolution where a length has a prime factor above 31 (mc_fft_gp.h).
//
// What bounds these kernels: vector arithmetic and its index work, not
// memory.  Smooth lengths run at 5-7 ns per thousand points and pass against
// 8-75 for a stage per small factor; lengths with a large prime at 8-14
// against 40-370 for the direct prime sums they replace, and depend on the
// prime no more.
#define MC_PRIME_LITERALS
#include <algorithm>
#include <cmath>
#include <complex>
#include <type_traits>
#include <vector>

#include "mc_fft.h"
#include "mc_fft_args.h"
#include "mc_fft_ct.h"
#include "mc_fft_gp.h"

namespace {

// Radices of plain lengths (31-smooth) and of convolution lengths (a dense
// enough set of cheap ones).
#define MC_GP_RADICES(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(15) X(16) \
    X(17) X(19) X(20) X(23) X(24) X(25) X(29) X(31) X(32)
#define MC_GP_CONV_RADICES(X) X(4) X(5) X(6) X(8) X(9) X(10) X(12) X(15) X(16) X(20) X(24)

enum { GP_FWD, GP_MID, GP_INV };  // forward pass, turning pass of a convolution, inverse pass

__device__ __forceinline__ cfloat cswap(cfloat a) { return cmk(a.y, a.x); }

// One pass over the `cnt` transforms in LDS.  Forward: butterfly, then the
// twiddles; inverse: conjugate twiddles, then the inverse butterfly (the
// forward one with real and imaginary parts exchanged).  Pass 0 of a
// convolution reads zeros past the n inputs, and its inverse leaves only the
// n results, times the chirp.  An item's LDS position and trailing index come
// from a table: forming them by run-time divisions cost as many instructions
// as a third of the butterfly.
template <int R, int MODE, bool CONV>
__device__ __forceinline__ void gp_pass_r(cfloat* lds, const GpPlan& P, int p, int cnt) {
    const int J = P.J[p], inner = P.inner[p], S = P.S[p], total = cnt * J, n = P.n;
    const float rJ = P.rJ[p];
    const cfloat* __restrict__ tw = P.tw[p];
    const unsigned int* __restrict__ item = P.item[p];
    for (int e = threadIdx.x; e < total; e += blockDim.x) {
        const int c = fdiv(e, J, rJ);
        const int i = e - c * J;
        const unsigned int d = item[i];
        const int j = d >> 16;
        cfloat* x = lds + c * P.ld + (d & 0xffffu);
        cfloat v[R];
        if (CONV && MODE == GP_FWD && p == 0) {
#pragma unroll
            for (int t = 0; t < R; t++) {
                v[t] = x[t * S];
                if (j + t * inner >= n) v[t] = cmk(0.f, 0.f);
            }
        } else {
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = x[t * S];
        }
        if (MODE == GP_INV) {
#pragma unroll
            for (int t = 1; t < R; t++) v[t] = cmul(v[t], cconj(tw[(t - 1) * inner + j]));
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = cswap(v[t]);
        }
        RegDft<R>::run(v);
        if (MODE == GP_MID) {
            const cfloat* __restrict__ kn = P.kern;
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = cswap(cmul(v[t], kn[t * J + i]));
            RegDft<R>::run(v);
        }
        if (MODE != GP_FWD) {
#pragma unroll
            for (int t = 0; t < R; t++) v[t] = cswap(v[t]);
        }
        if (MODE == GP_FWD && inner > 1) {
#pragma unroll
            for (int t = 1; t < R; t++) v[t] = cmul(v[t], tw[(t - 1) * inner + j]);
        }
        if (MODE != GP_FWD && p == 0) {
            const cfloat* __restrict__ ch = P.chirp;
#pragma unroll
            for (int t = 0; t < R; t++) {
                const int k = j + t * inner;
                if (k < n) x[t * S] = cmul(v[t], ch[k]);
            }
        } else {
#pragma unroll
            for (int t = 0; t < R; t++) x[t * S] = v[t];
        }
    }
    __syncthreads();
}

template <int MODE, bool CONV>
__device__ __forceinline__ void gp_pass(cfloat* lds, const GpPlan& P, int p, int cnt) {
    if constexpr (CONV) {
        switch (P.R[p]) {
#define X(RR) case RR: gp_pass_r<RR, MODE, CONV>(lds, P, p, cnt); break;
            MC_GP_CONV_RADICES(X)
#undef X
        }
    } else {
        switch (P.R[p]) {
#define X(RR) case RR: gp_pass_r<RR, MODE, CONV>(lds, P, p, cnt); break;
            MC_GP_RADICES(X)
#undef X
        }
    }
}

// The transforms held in LDS at natural positions (CONV: times the chirp):
// results at P.frq positions.  Ends with a barrier.
template <bool CONV>
__device__ __forceinline__ void gp_fft(cfloat* lds, const GpPlan& P, int cnt) {
    if constexpr (CONV) {
        for (int p = 0; p < P.np - 1; p++) gp_pass<GP_FWD, true>(lds, P, p, cnt);
        gp_pass<GP_MID, true>(lds, P, P.np - 1, cnt);
        for (int p = P.np - 2; p >= 0; p--) gp_pass<GP_INV, true>(lds, P, p, cnt);
    } else {
        for (int p = 0; p < P.np; p++) gp_pass<GP_FWD, false>(lds, P, p, cnt);
    }
}

// Transforms per workgroup and chunk widths are powers of two, so every
// thread keeps one row (or column) and steps along it: no index arithmetic
// per element beyond the two position tables.  Loads go out MC_GP_U at a time.
#define MC_GP_U 4
// four waves per SIMD: the LDS of two 512-thread workgroups allows no more
#define MC_GP_BOUNDS __launch_bounds__(512, 4)

__device__ __forceinline__ int ilog2(int v) { return __ffs(v) - 1; }

template <bool CONV>
__global__ MC_GP_BOUNDS void k_rows_r2c_gp(RowR2CArgs a, const GpPlan* __restrict__ plan) {
    const GpPlan& P = *plan;
    extern __shared__ cfloat lds[];
    const int nrb = (a.H + a.R - 1) / a.R;
    const int tt = xcd_tile(blockIdx.x, gridDim.x);
    const int b = tt / nrb;
    const int row0 = (tt - b * nrb) * a.R;
    const int nrows = min(a.R, a.H - row0);
    const int n = P.n, NT = blockDim.x, lr = ilog2(a.R), lc = ilog2(a.C);
    const unsigned short* __restrict__ nat = P.nat;
    const unsigned short* __restrict__ frq = P.frq;
    const cfloat* __restrict__ chirp = P.chirp;
    const int img = a.in_mod > 0 ? b % a.in_mod : b;
    const int wi = a.in_mod > 0 ? b / a.in_mod : b;
    int x0 = 0, y0 = 0;
    if (a.win) {
        x0 = a.win[2 * wi];
        y0 = a.win[2 * wi + 1];
    }
    const bool vec = ((x0 | (int)(a.pitch & 1) | (int)(a.in_bstride & 1)) & 1) == 0 &&
                     (((uintptr_t)a.in) & 7) == 0;
    {
        const int tpr = NT >> lr, r = threadIdx.x / tpr, i0 = threadIdx.x % tpr;
        const float* src = a.in + (long long)img * a.in_bstride + (long long)(y0 + row0 + r) * a.pitch + x0;
        cfloat* row = lds + r * P.ld;
        auto load = [&](auto pairs) {
            for (int i = i0; i < n; i += tpr * MC_GP_U) {
                float2 v[MC_GP_U];
                cfloat w[MC_GP_U];
                int d[MC_GP_U];
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    const int iu = min(i + u * tpr, n - 1);
                    if constexpr (decltype(pairs)::value) v[u] = reinterpret_cast<const float2*>(src)[iu];
                    else v[u] = make_float2(src[2 * iu], src[2 * iu + 1]);
                    d[u] = nat[iu];
                    if (CONV) w[u] = chirp[iu];
                }
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    cfloat z = cmk(v[u].x, v[u].y);
                    if (CONV) z = cmul(z, w[u]);
                    if (i + u * tpr < n) row[d[u]] = z;
                }
            }
        };
        if (r < nrows) {
            if (vec) load(std::true_type{});
            else load(std::false_type{});
        }
    }
    __syncthreads();
    gp_fft<CONV>(lds, P, nrows);
    // Post-processing as in k_rows_r2c_rp, the pair X[k], X[n-k] at a time;
    // consecutive lanes write the C values of a row's staging chunk, then
    // the next row's.  Steps along k are whole chunks, so both offsets move
    // by a constant.
    const int c = threadIdx.x & (a.C - 1), r = (threadIdx.x >> lc) & (a.R - 1);
    if (r >= nrows) return;
    const int dkb = NT >> (lc + lr);
    const int kb0 = threadIdx.x >> (lc + lr);
    const int kbs = a.H << lc, step = dkb * kbs;
    const int k0 = (kb0 << lc) + c, m0 = n - k0;
    const cfloat* row = lds + r * P.ld;
    cfloat* tb = a.T + (long long)b * a.t_bstride + (long long)(row0 + r) * a.C;
    // (offsets wrap harmlessly where k or m is out of range: not used there)
    unsigned int ok = (unsigned)kb0 * kbs + c, om = (unsigned)(m0 >> lc) * kbs + (m0 & (a.C - 1));
    for (int k = k0; 2 * k <= n; k += (dkb << lc) * MC_GP_U) {
        cfloat zk[MC_GP_U], zm[MC_GP_U], tk[MC_GP_U], tm[MC_GP_U];
        int fk[MC_GP_U], fm[MC_GP_U];
#pragma unroll
        for (int u = 0; u < MC_GP_U; u++) {
            const int ku = min(k + u * (dkb << lc), n / 2), mu = n - ku;
            tk[u] = a.post_tw[ku];
            tm[u] = a.post_tw[mu];
            fk[u] = frq[ku];
            fm[u] = frq[ku == 0 ? 0 : mu];
        }
#pragma unroll
        for (int u = 0; u < MC_GP_U; u++) {
            zk[u] = row[fk[u]];
            zm[u] = row[fm[u]];
        }
#pragma unroll
        for (int u = 0; u < MC_GP_U; u++) {
            const int ku = k + u * (dkb << lc);
            const cfloat E = cmk(0.5f * (zk[u].x + zm[u].x), 0.5f * (zk[u].y - zm[u].y));
            const cfloat D = cmk(zk[u].x - zm[u].x, zk[u].y + zm[u].y);
            const cfloat O = cmk(0.5f * D.y, -0.5f * D.x);
            if (2 * ku <= n) tb[ok] = cscale(cadd(E, cmul(tk[u], O)), a.scale);
            if (2 * ku < n) tb[om] = cscale(cadd(cconj(E), cmul(tm[u], cconj(O))), a.scale);
            ok += step;
            om -= step;
        }
    }
}

// Z[k] of the half-length packing (see c2r_pre in mc_fft.hip) from X[k], its
// partner X[n-k] and the post-twiddle of k.
__device__ __forceinline__ cfloat gp_c2r_pre(cfloat p, cfloat q, cfloat w) {
    const cfloat t = cmul(cconj(w), cmk(p.x - q.x, p.y + q.y));
    return cconj(cmk(p.x + q.x - t.y, p.y - q.y + t.x));
}

template <bool CONV>
__global__ MC_GP_BOUNDS void k_rows_c2r_gp(RowC2RArgs a, const GpPlan* __restrict__ plan) {
    const GpPlan& P = *plan;
    extern __shared__ cfloat lds[];
    const int nrb = (a.H + a.R - 1) / a.R;
    const int tt = xcd_tile(blockIdx.x, gridDim.x);
    const int b = tt / nrb;
    const int row0 = (tt - b * nrb) * a.R;
    const int nrows = min(a.R, a.H - row0);
    const int n = P.n, NT = blockDim.x, lr = ilog2(a.R), lc = ilog2(a.C);
    const unsigned short* __restrict__ nat = P.nat;
    const unsigned short* __restrict__ frq = P.frq;
    const cfloat* __restrict__ chirp = P.chirp;
    {
        // one item per Hermitian pair (k, n - k), in the staging layout's order
        const int c = threadIdx.x & (a.C - 1), r = (threadIdx.x >> lc) & (a.R - 1);
        const int dkb = NT >> (lc + lr), kb0 = threadIdx.x >> (lc + lr);
        const int kbs = a.H << lc, step = dkb * kbs;
        const int k0 = (kb0 << lc) + c, m0 = n - k0;
        const cfloat* tb = a.T + (long long)b * a.t_bstride + (long long)(row0 + min(r, nrows - 1)) * a.C;
        cfloat* row = lds + r * P.ld;
        unsigned int ok = (unsigned)kb0 * kbs + c, om = (unsigned)(m0 >> lc) * kbs + (m0 & (a.C - 1));
        if (r < nrows) {
            for (int k = k0; 2 * k <= n; k += (dkb << lc) * MC_GP_U) {
                cfloat xp[MC_GP_U], xq[MC_GP_U], tk[MC_GP_U], tm[MC_GP_U], wk[MC_GP_U], wm[MC_GP_U];
                int fk[MC_GP_U], fm[MC_GP_U];
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    const bool in = 2 * (k + u * (dkb << lc)) <= n;
                    const int ku = in ? k + u * (dkb << lc) : 0, mu = n - ku;
                    xp[u] = tb[in ? ok : 0u];
                    xq[u] = tb[in ? om : 0u];
                    ok += step;
                    om -= step;
                    tk[u] = a.post_tw[ku];
                    tm[u] = a.post_tw[mu];
                    fk[u] = nat[ku];
                    fm[u] = nat[ku == 0 ? 0 : mu];
                    if (CONV) {
                        wk[u] = chirp[ku];
                        wm[u] = chirp[ku == 0 ? 0 : mu];
                    }
                }
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    const int ku = k + u * (dkb << lc);
                    cfloat zk = gp_c2r_pre(xp[u], xq[u], tk[u]), zm = gp_c2r_pre(xq[u], xp[u], tm[u]);
                    if (ku == 0) zk = cconj(cmk(xp[u].x + xq[u].x, xp[u].x - xq[u].x));
                    if (CONV) {
                        zk = cmul(zk, wk[u]);
                        zm = cmul(zm, wm[u]);
                    }
                    if (2 * ku <= n) row[fk[u]] = zk;
                    if (ku > 0 && 2 * ku < n) row[fm[u]] = zm;
                }
            }
        }
    }
    __syncthreads();
    gp_fft<CONV>(lds, P, nrows);
    const int tpr = NT >> lr, r = threadIdx.x / tpr, j0 = threadIdx.x % tpr;
    if (r >= nrows) return;
    float* ob = a.out + (long long)b * a.out_bstride + (long long)(row0 + r) * a.pitch;
    const cfloat* row = lds + r * P.ld;
    const bool clamp = a.clamp != 0;
    auto store = [&](auto pairs) {
#pragma unroll 4
        for (int j = j0; j < n; j += tpr) {
            const cfloat z = row[frq[j]];
            float v0 = z.x, v1 = -z.y;
            v0 = clamp ? fmaxf(v0, 0.f) : v0;
            v1 = clamp ? fmaxf(v1, 0.f) : v1;
            if constexpr (decltype(pairs)::value) {
                reinterpret_cast<float2*>(ob)[j] = make_float2(v0, v1);
            } else {
                ob[2 * j] = v0;
                ob[2 * j + 1] = v1;
            }
        }
    };
    if (((a.pitch | a.out_bstride) & 1) == 0 && (((uintptr_t)a.out) & 7) == 0) store(std::true_type{});
    else store(std::false_type{});
}

// Columns: cw of the staging chunk's C columns per workgroup.
template <bool CONV>
__global__ MC_GP_BOUNDS void k_cols_fwd_gp(ColFwdArgs a, const GpPlan* __restrict__ plan, int cw) {
    const GpPlan& P = *plan;
    extern __shared__ cfloat lds[];
    const int ncb = (a.ncols + cw - 1) / cw;
    const int tt = xcd_tile(blockIdx.x, gridDim.x);
    const int b = tt / ncb, c0 = (tt - b * ncb) * cw;
    const int kb = c0 / a.C, coff = c0 - kb * a.C;
    const int nc = min(cw, a.ncols - c0);
    const int NT = blockDim.x, H = a.H, lw = ilog2(cw);
    const unsigned short* __restrict__ nat = P.nat;
    const unsigned short* __restrict__ frq = P.frq;
    const cfloat* __restrict__ chirp = P.chirp;
    {
        const int c = threadIdx.x & (cw - 1), y0 = threadIdx.x >> lw, dy = NT >> lw;
        const cfloat* src = a.T + (long long)b * a.t_bstride + (long long)kb * H * a.C + coff + c;
        cfloat* col = lds + c * P.ld;
        if (c < nc) {
            for (int y = y0; y < H; y += dy * MC_GP_U) {
                cfloat v[MC_GP_U], w[MC_GP_U];
                int d[MC_GP_U];
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    const int yu = min(y + u * dy, H - 1);
                    v[u] = src[yu * a.C];
                    d[u] = nat[yu];
                    if (CONV) w[u] = chirp[yu];
                }
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++)
                    if (y + u * dy < H) col[d[u]] = CONV ? cmul(v[u], w[u]) : v[u];
            }
        }
    }
    __syncthreads();
    gp_fft<CONV>(lds, P, nc);
    const int tpc = NT >> lw, c = threadIdx.x / tpc, i0 = threadIdx.x % tpc;
    if (c >= nc) return;
    const cfloat* col = lds + c * P.ld;
    if (a.S) {
        cfloat* dst = a.S + (long long)b * a.s_bstride + (long long)(c0 + c) * H;
#pragma unroll 4
        for (int y = i0; y < H; y += tpc) dst[y] = col[frq[y]];
    }
    if (a.X && c0 + c < a.xcx) {
        cfloat* xd = a.X + (long long)b * a.x_bstride + (long long)(c0 + c) * a.xcy;
#pragma unroll 4
        for (int yo = i0; yo < a.xcy; yo += tpc) {
            const int yi = resize_row(yo, a.xcy, H);
            if (yi >= 0) xd[yo] = col[frq[yi]];
        }
    }
}

template <bool CONV>
__global__ MC_GP_BOUNDS void k_cols_inv_gp(ColInvArgs a, const GpPlan* __restrict__ plan, int cw) {
    const GpPlan& P = *plan;
    extern __shared__ cfloat lds[];
    const int ncb = (a.ncols + cw - 1) / cw;
    const int tt = xcd_tile(blockIdx.x, gridDim.x);
    const int b = tt / ncb, c0 = (tt - b * ncb) * cw;
    const int kb = c0 / a.C, coff = c0 - kb * a.C;
    const int nc = min(cw, a.ncols - c0);
    const int NT = blockDim.x, H = a.H, lw = ilog2(cw);
    const unsigned short* __restrict__ nat = P.nat;
    const unsigned short* __restrict__ frq = P.frq;
    const cfloat* __restrict__ chirp = P.chirp;
    {
        const int tpc = NT >> lw, c = threadIdx.x / tpc, i0 = threadIdx.x % tpc;
        const int kx = c0 + c;
        const bool same = a.src_cx == a.ncols && a.src_cy == H;
        // a column of a crop or pad that has no source is zero
        const bool has = c < nc && kx < a.src_cx;
        const cfloat* sc = a.S + (long long)b * a.s_bstride + (long long)(has ? kx : 0) * a.src_cy;
        const cfloat* pb = a.phB ? a.phB + (long long)b * H : nullptr;
        const cfloat pa = a.phA && c < nc ? a.phA[(long long)b * a.ncols + kx] : cmk(1.f, 0.f);
        cfloat* col = lds + c * P.ld;
        // one straight-line copy of the load per form: with the choices
        // inside the unrolled loop every load waited for the one before it
        // (8.4 against 6.5 ns per thousand points, columns of 512)
        auto load = [&](auto crop, auto shift) {
            for (int y = i0; y < H; y += tpc * MC_GP_U) {
                cfloat v[MC_GP_U], w[MC_GP_U], ph[MC_GP_U];
                int d[MC_GP_U];
                bool in[MC_GP_U];
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    const int yu = min(y + u * tpc, H - 1);
                    int yi = yu;
                    in[u] = true;
                    if constexpr (decltype(crop)::value) {
                        // Fourier crop or pad from a src_cx x src_cy spectrum
                        yi = resize_row(yu, H, a.src_cy);
                        in[u] = has && yi >= 0;
                        yi = in[u] ? yi : 0;
                    }
                    v[u] = sc[yi];
                    if constexpr (decltype(shift)::value) ph[u] = pb[yu];
                    d[u] = nat[yu];
                    if (CONV) w[u] = chirp[yu];
                }
#pragma unroll
                for (int u = 0; u < MC_GP_U; u++) {
                    cfloat z = in[u] ? v[u] : cmk(0.f, 0.f);
                    if constexpr (decltype(shift)::value) z = cmul(z, cmul(pa, ph[u]));
                    z = cconj(z);
                    if (y + u * tpc < H) col[d[u]] = CONV ? cmul(z, w[u]) : z;
                }
            }
        };
        if (c < nc) {
            if (same) {
                if (a.phA) load(std::false_type{}, std::true_type{});
                else load(std::false_type{}, std::false_type{});
            } else {
                if (a.phA) load(std::true_type{}, std::true_type{});
                else load(std::true_type{}, std::false_type{});
            }
        }
    }
    __syncthreads();
    gp_fft<CONV>(lds, P, nc);
    const int c = threadIdx.x & (cw - 1), y0 = threadIdx.x >> lw, dy = NT >> lw;
    if (c >= nc) return;
    cfloat* dst = a.T + (long long)b * a.t_bstride + (long long)kb * H * a.C + coff + c;
    const cfloat* col = lds + c * P.ld;
#pragma unroll 4
    for (int y = y0; y < H; y += dy) dst[y * a.C] = cconj(col[frq[y]]);
}

// ---- plans ----------------------------------------------------------------
// Operations of one radix-r butterfly as RegDft forms it.
double bfly_ops(int r) {
    if (r == 1) return 0;
    if (r == 2) return 4;
    if (r == 4) return 16;
    if (r == 8) return 60;
    if (rp_leaf(r)) {
        const double h = (r - 1) / 2;
        return h * (4 * h + 4) + 6 * h;
    }
    const int a = rp_first(r), b = r / a;
    return b * bfly_ops(a) + a * bfly_ops(b) + 4.0 * (a - 1) * (b - 1);
}

// Cost of a pass per point: the butterfly, twiddles, LDS accesses, and about
// 30 instructions of index work per item.
double pass_cost(int r) { return (bfly_ops(r) + 8.0 * r + 30.0) / r; }

void search(const std::vector<int>& rads, int np, int lo, int hi, long long prod, double cost,
            std::vector<int>& cur, std::vector<int>& best, double& best_cost) {
    if (!cur.empty() && prod >= lo && prod <= hi) {
        const double c = cost * (double)prod;
        if (c < best_cost) {
            best_cost = c;
            best = cur;
        }
    }
    if ((int)cur.size() == np) return;
    for (int r : rads) {
        if (!cur.empty() && r < cur.back()) continue;
        if (prod * r > hi || (lo == hi && lo % (prod * r))) continue;
        cur.push_back(r);
        search(rads, np, lo, hi, prod * r, cost + pass_cost(r), cur, best, best_cost);
        cur.pop_back();
    }
}

// In-place double FFT of any length by its smallest prime factors (host).
void host_fft(std::vector<std::complex<double>>& x) {
    const int n = (int)x.size();
    if (n == 1) return;
    int p = 2;
    while (n % p) p++;
    const int m = n / p;
    std::vector<std::vector<std::complex<double>>> s(p, std::vector<std::complex<double>>(m));
    for (int i = 0; i < n; i++) s[i % p][i / p] = x[i];
    for (auto& v : s) host_fft(v);
    for (int k = 0; k < n; k++) {
        std::complex<double> a = 0;
        for (int t = 0; t < p; t++) a += s[t][k % m] * std::polar(1.0, -2.0 * M_PI * ((long long)t * k % n) / n);
        x[k] = a;
    }
}

bool g_gp_attr_done = false;

template <class F>
bool gp_attr(F* f) {
    return hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, MC_GP_LDS_MAX) ==
           hipSuccess;
}

}  // namespace

static bool gp_build(int n, GpPlan* P, GpTables* T) {
    static const std::vector<int> plain = {
#define X(R) R,
        MC_GP_RADICES(X)
#undef X
    };
    static const std::vector<int> conv = {
#define X(R) R,
        MC_GP_CONV_RADICES(X)
#undef X
    };
    if (n < 2 || n > MC_LDS_ELEMS) return false;
    std::vector<int> cur, rad;
    double best = 1e300;
    search(plain, MC_GP_MAXP, n, n, 1, 0.0, cur, rad, best);
    *P = GpPlan();
    P->n = n;
    P->conv = rad.empty();
    if (P->conv) search(conv, MC_GP_MAXP, 2 * n - 1, 4 * n, 1, 0.0, cur, rad, best);
    if (rad.empty()) return false;
    // largest radix first, but last the smallest odd one (no padding), else
    // the smallest that keeps the padding below an eighth
    std::sort(rad.rbegin(), rad.rend());
    size_t last = 0;
    for (size_t i = 1; i < rad.size(); i++) {
        const bool odd = rad[i] % 2 && rad[i] >= 5, podd = rad[last] % 2 && rad[last] >= 5;
        if (odd || (!podd && rad[i] >= 8)) last = i;
    }
    std::rotate(rad.begin() + last, rad.begin() + last + 1, rad.end());
    const int np = P->np = (int)rad.size();
    int M = 1;
    for (int r : rad) M *= r;
    P->M = M;
    for (int p = np - 1, in = 1; p >= 0; in *= rad[p], p--) {
        P->R[p] = rad[p];
        P->inner[p] = in;
        P->J[p] = M / rad[p];
        P->rJ[p] = 1.0f / P->J[p];
        P->S[p] = p == np - 1 ? 1 : P->S[p + 1] * rad[p + 1];
        if (p == np - 2 || p == 0) P->S[p] |= 1;
    }
    P->ld = np > 1 ? P->S[0] * rad[0] : M;
    if ((size_t)P->ld * sizeof(cfloat) > MC_GP_LDS_MAX || P->ld > 65535) return false;
    // LDS positions
    std::vector<unsigned short> pos(M + n);
    for (int i = 0; i < M; i++) {
        int a = 0;
        for (int p = 0; p < np; p++) a += (i / P->inner[p]) % rad[p] * P->S[p];
        pos[i] = (unsigned short)a;
    }
    for (int k = 0; k < n; k++) {
        int a = 0, q = k;
        for (int p = 0; p < np; p++) {
            a += q % rad[p] * P->S[p];
            q /= rad[p];
        }
        pos[M + k] = P->conv ? pos[k] : (unsigned short)a;
    }
    // items of each pass: digits before p packed k_0 fastest, then those after
    // p in natural order; LDS position of output 0 | trailing index << 16
    std::vector<unsigned int> items;
    std::vector<size_t> ioff(np);
    for (int p = 0; p < np; p++) {
        ioff[p] = items.size();
        const int in = P->inner[p];
        for (int i = 0; i < P->J[p]; i++) {
            int q = i / in, a = 0;
            const int j = i % in;
            for (int d = 0; d < p; d++) {
                a += q % rad[d] * P->S[d];
                q /= rad[d];
            }
            for (int d = p + 1; d < np; d++) a += (j / P->inner[d]) % rad[d] * P->S[d];
            items.push_back((unsigned int)a | (unsigned int)j << 16);
        }
    }
    // tables
    std::vector<cfloat> h;
    std::vector<size_t> off(np, 0);
    for (int p = 0; p + 1 < np; p++) {
        off[p] = h.size();
        const int in = P->inner[p], L = in * rad[p];
        for (int t = 1; t < rad[p]; t++)
            for (int j = 0; j < in; j++) {
                const double g = -2.0 * M_PI * ((long long)j * t % L) / L;
                h.push_back(cfloat{(float)std::cos(g), (float)std::sin(g)});
            }
    }
    size_t okern = 0, ochirp = 0;
    if (P->conv) {
        std::vector<std::complex<double>> b(M);
        ochirp = h.size();
        for (int i = 0; i < n; i++) {
            const double g = M_PI * (double)((long long)i * i % (2 * n)) / n;
            h.push_back(cfloat{(float)std::cos(g), (float)-std::sin(g)});
            b[i] = std::polar(1.0, g);
            if (i) b[M - i] = b[i];
        }
        host_fft(b);
        okern = h.size();
        // item i of the last pass holds the digits k_0, k_1, ... (k_0
        // fastest); its output t is frequency i + J t
        const int J = P->J[np - 1];
        for (int t = 0; t < rad[np - 1]; t++)
            for (int i = 0; i < J; i++) {
                const std::complex<double> v = b[i + J * t] / (double)M;
                h.push_back(cfloat{(float)v.real(), (float)v.imag()});
            }
    }
    if (h.empty()) h.push_back(cfloat{1.f, 0.f});
    const size_t hb = h.size() * sizeof(cfloat), pb = pos.size() * sizeof(pos[0]);
    const size_t ib = items.size() * sizeof(items[0]);
    if (hipMalloc(&T->tab, hb) != hipSuccess || hipMalloc(&T->pos, pb) != hipSuccess ||
        hipMalloc(&T->item, ib) != hipSuccess ||
        hipMemcpy(T->item, items.data(), ib, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(T->tab, h.data(), hb, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(T->pos, pos.data(), pb, hipMemcpyHostToDevice) != hipSuccess) {
        gp_free(T);
        return false;
    }
    for (int p = 0; p < np; p++) {
        P->tw[p] = T->tab + off[p];
        P->item[p] = T->item + ioff[p];
    }
    P->kern = T->tab + okern;
    P->chirp = T->tab + ochirp;
    P->nat = T->pos;
    P->frq = T->pos + M;
    if (hipMalloc(&T->plan, sizeof(GpPlan)) != hipSuccess ||
        hipMemcpy(T->plan, P, sizeof(GpPlan), hipMemcpyHostToDevice) != hipSuccess) {
        gp_free(T);
        return false;
    }
    P->dev = T->plan;
    return true;
}

bool gp_plan(int n, GpPlan* P, GpTables* T) {
    if (gp_build(n, P, T)) return true;
    *P = GpPlan();  // n = 0: callers take the stage kernels
    return false;
}

void gp_free(GpTables* T) {
    if (T->tab) (void)hipFree(T->tab);
    if (T->pos) (void)hipFree(T->pos);
    if (T->item) (void)hipFree(T->item);
    if (T->plan) (void)hipFree(T->plan);
    *T = GpTables();
}

int mc_fft_gp_init() {
    if (g_gp_attr_done) return 0;
    const bool ok = gp_attr(k_rows_r2c_gp<false>) && gp_attr(k_rows_r2c_gp<true>) &&
                    gp_attr(k_rows_c2r_gp<false>) && gp_attr(k_rows_c2r_gp<true>) &&
                    gp_attr(k_cols_fwd_gp<false>) && gp_attr(k_cols_fwd_gp<true>) &&
                    gp_attr(k_cols_inv_gp<false>) && gp_attr(k_cols_inv_gp<true>);
    g_gp_attr_done = ok;
    return ok ? 0 : -1;
}

// Transforms per workgroup: as many as fill about 36 KB of LDS (four
// 256-thread workgroups per CU), at least `want` where 70 KB hold them (short
// runs of the staging layout cost more than occupancy), at most `cap`, and
// few enough that `all` transforms give every CU a workgroup.
static int gp_group(const GpPlan& P, int cap, int want, long long all) {
    const size_t b = (size_t)P.ld * sizeof(cfloat);
    int g = 1;
    while (2 * g <= cap && (2 * g * b <= 36 * 1024 || (2 * g <= want && 2 * g * b <= MC_GP_LDS_WG))) g *= 2;
    while (g > 1 && all / g < 256) g /= 2;
    return g;
}
static int gp_threads(const GpPlan& P, int g) { return (long long)g * P.M <= 5120 ? 256 : 512; }

hipError_t gp_rows_r2c(const GpPlan& P, const RowR2CArgs& args, int batch, hipStream_t s) {
    RowR2CArgs a = args;
    a.R = gp_group(P, 256 / a.C, 2, (long long)a.H * batch);
    const dim3 grid(mc_div_up(a.H, a.R) * batch), blk(gp_threads(P, a.R));
    const size_t lds = (size_t)a.R * P.ld * sizeof(cfloat);
    if (P.conv) hipLaunchKernelGGL(k_rows_r2c_gp<true>, grid, blk, lds, s, a, P.dev);
    else hipLaunchKernelGGL(k_rows_r2c_gp<false>, grid, blk, lds, s, a, P.dev);
    return hipGetLastError();
}

hipError_t gp_rows_c2r(const GpPlan& P, const RowC2RArgs& args, int batch, hipStream_t s) {
    RowC2RArgs a = args;
    a.R = gp_group(P, 256 / a.C, 2, (long long)a.H * batch);
    const dim3 grid(mc_div_up(a.H, a.R) * batch), blk(gp_threads(P, a.R));
    const size_t lds = (size_t)a.R * P.ld * sizeof(cfloat);
    if (P.conv) hipLaunchKernelGGL(k_rows_c2r_gp<true>, grid, blk, lds, s, a, P.dev);
    else hipLaunchKernelGGL(k_rows_c2r_gp<false>, grid, blk, lds, s, a, P.dev);
    return hipGetLastError();
}

hipError_t gp_cols_fwd(const GpPlan& P, const ColFwdArgs& a, int batch, hipStream_t s) {
    const int cw = gp_group(P, a.C, 4, (long long)a.ncols * batch);
    const dim3 grid(mc_div_up(a.ncols, cw) * batch), blk(gp_threads(P, cw));
    const size_t lds = (size_t)cw * P.ld * sizeof(cfloat);
    if (P.conv) hipLaunchKernelGGL(k_cols_fwd_gp<true>, grid, blk, lds, s, a, P.dev, cw);
    else hipLaunchKernelGGL(k_cols_fwd_gp<false>, grid, blk, lds, s, a, P.dev, cw);
    return hipGetLastError();
}

hipError_t gp_cols_inv(const GpPlan& P, const ColInvArgs& a, int batch, hipStream_t s) {
    const int cw = gp_group(P, a.C, 4, (long long)a.ncols * batch);
    const dim3 grid(mc_div_up(a.ncols, cw) * batch), blk(gp_threads(P, cw));
    const size_t lds = (size_t)cw * P.ld * sizeof(cfloat);
    if (P.conv) hipLaunchKernelGGL(k_cols_inv_gp<true>, grid, blk, lds, s, a, P.dev, cw);
    else hipLaunchKernelGGL(k_cols_inv_gp<false>, grid, blk, lds, s, a, P.dev, cw);
    return hipGetLastError();
}
