// mc_fft_args.h -- kernel arguments of the row and column passes.
#pragma once
#include "mc_common.h"

struct RowR2CArgs {
    FftPlan1 plan;
    int H, m, C, R;
    const float* in;
    long long pitch, in_bstride;
    int in_mod;            // transform b reads image b % in_mod (0: b)
    const int* win;        // (x0, y0) per b / in_mod, or null
    cfloat* T;
    long long t_bstride;
    const cfloat* post_tw;
    float scale;
    float* dc;             // |row DC| per (transform, row) of the output, or null
};

struct RowC2RArgs {
    FftPlan1 plan;
    int H, m, C, R;
    const cfloat* T;
    long long t_bstride;
    float* out;
    long long pitch, out_bstride;
    const cfloat* post_tw;
    int clamp;
};

struct ColFwdArgs {
    FftPlan1 plan;
    int H, ncols, C;
    const cfloat* T;
    long long t_bstride;
    cfloat* S;
    long long s_bstride;
    cfloat* X;
    int xcx, xcy;
    long long x_bstride;
    const float* s_g;      // store factors of a reduced S format (per transform)
    const float* x_g;      // store factors of a reduced X format
};

struct ColInvArgs {
    FftPlan1 plan;
    int H, ncols, C;
    const cfloat* S;
    long long s_bstride;
    int src_cx, src_cy;
    const cfloat* phA;
    const cfloat* phB;
    cfloat* T;
    long long t_bstride;
    const float* s_inv;    // load factors of a reduced S format (per transform)
};

// Util/GFourierResize2D.cu:15-35 row map: output row yo of a spectrum with
// `outy` rows taken from a spectrum with `iny` rows, -1 if unmapped.
__device__ __forceinline__ int resize_row(int yo, int outy, int iny) {
    int y = yo;
    if (y > outy / 2) {
        y -= outy;
        if (y <= -iny / 2) return -1;
        return y + iny;
    }
    return (y > iny / 2) ? -1 : y;
}

// Output row of a cropped (xcy-row) spectrum that input row y maps to, or -1
// (the inverse of resize_row for xcy < H).
__device__ __forceinline__ int crop_row(int y, int xcy, int H) {
    if (y <= xcy / 2) return y;
    const int d = H - xcy;
    return (y > xcy / 2 + d) ? y - d : -1;
}
