// mc_fft_gp.h -- in-place FFT passes for lengths known at run time.
//
// Lengths without a compile-time schedule (mc_fft_rp.h, mc_fft_ct.h) are
// transformed in LDS by at most four passes of radix R_p <= 32 (M = R_0 R_1
// ...).  A work item holds one radix-R_p butterfly in registers (RegDft), so
// a length like 2000 = 10 * 10 * 20 needs three passes where a stage per
// small factor needs five.  The passes run in place (decimation in
// frequency): an item reads and writes the same LDS words, so a pass costs
// one barrier and no second buffer, and any number of items can be looped
// over by any number of threads.
//
// Element i (digits d_0 .. d_{np-1}, d_0 slowest) lies at sum d_p S_p, with
// S_{np-2} and S_0 made odd: the last pass (lanes step over S_{np-2} or S_0)
// and the reads in frequency order (lanes step over S_0) then spread over all
// LDS banks.  Pass p turns digit d_p into k_p: over the later digits' natural
// index j, output t is multiplied by W_{L_p}^{j t}, L_p = R_p R_{p+1} ....
// Frequency k = k_0 + R_0 k_1 + R_0 R_1 k_2 + ... ends at sum k_p S_p.  Two
// tables give the LDS position of a natural index and of a frequency.
//
// A length n with a prime factor above 31 becomes a convolution of length
// M >= 2n - 1 (Bluestein's chirp transform): X_k = c_k sum_i (x_i c_i)
// conj(c)_{k-i}, c_i = e^{-i pi i^2 / n}.  The forward passes leave the
// product's operand in digit order, its last pass multiplies by the
// transformed kernel in registers and starts the inverse passes at once, and
// these end in natural order, so no reordering is needed.
#pragma once
#include <vector>
#include "mc_common.h"

#define MC_GP_MAXP 4
// LDS bytes a workgroup may take (two of 70 KB share a CU's 160 KB), and the
// most a single transform may need
#define MC_GP_LDS_WG (70 * 1024)
#define MC_GP_LDS_MAX (152 * 1024)

struct RowR2CArgs;  // mc_fft_args.h
struct RowC2RArgs;
struct ColFwdArgs;
struct ColInvArgs;

struct GpPlan {
    int n;                     // transform length
    int M;                     // length of the passes (n, or the convolution's)
    int np;
    int conv;                  // 1: chirp convolution
    int ld;                    // LDS elements of one transform
    int R[MC_GP_MAXP];
    int S[MC_GP_MAXP];         // LDS stride of digit p
    int J[MC_GP_MAXP];         // items of pass p (M / R_p)
    int inner[MC_GP_MAXP];     // product of the later radices
    float rJ[MC_GP_MAXP];      // 1 / J for fdiv
    const unsigned int* item[MC_GP_MAXP];  // per item: LDS position of input 0 | trailing index << 16
    const cfloat* tw[MC_GP_MAXP];  // [t-1][j] twiddles of pass p
    const cfloat* kern;        // conv: transformed kernel / M, [t][item] of the last pass
    const cfloat* chirp;       // conv: c_i, i < n
    const unsigned short* nat; // LDS position of natural index i < M
    const unsigned short* frq; // LDS position of output k < n (conv: nat)
    const GpPlan* dev;         // this plan in device memory: the kernels index it
                               // by pass, which a by-value argument would put in scratch
};

struct GpTables {              // device memory of a plan (owned by the Fft2D)
    cfloat* tab = nullptr;
    unsigned short* pos = nullptr;
    unsigned int* item = nullptr;
    GpPlan* plan = nullptr;
};

// A plan for length n, or false and P->n = 0 when it has none (too long for LDS).
bool gp_plan(int n, GpPlan* P, GpTables* T);
void gp_free(GpTables* T);
int mc_fft_gp_init();
// The passes (mc_fft.h) by run-time radices, FP32 spectra.
hipError_t gp_rows_r2c(const GpPlan& P, const RowR2CArgs& a, int batch, hipStream_t s);
hipError_t gp_rows_c2r(const GpPlan& P, const RowC2RArgs& a, int batch, hipStream_t s);
hipError_t gp_cols_fwd(const GpPlan& P, const ColFwdArgs& a, int batch, hipStream_t s);
hipError_t gp_cols_inv(const GpPlan& P, const ColInvArgs& a, int batch, hipStream_t s);
