// mc_sums.h -- dose-weighted sums from a few node images (host).
//
// A frame whose accumulated dose counts c raw frames has the weight q^c,
// q = exp(-a), a in [0, amax] over the frequencies.  Over a class of frames
// (those in and out of -SumRange, even and odd ones under -SplitSum) every
// q^c_i is fitted by the weights of `nodes` of its frames, q^c_i = sum_j lam_ij
// q^c_j, by least squares over a.  A class takes the fewest nodes whose
// residual, relative to the weights' normaliser sqrt(sum q^2c) and summed in
// squares over the class, stays below 2e-8 at every frequency: under the
// rounding of one FP32 weight (6e-8).  A class that would need more than
// `rank` nodes is cut in two.
#pragma once
#include <algorithm>
#include <cmath>
#include <vector>

struct SumPlan {
    struct Class {
        std::vector<int> frames, nodes;  // frame numbers; nodes: positions in frames
        std::vector<double> lam;         // [frame][node]
        int half = -1;                   // 0 even, 1 odd frames (split sums), else -1
    };
    std::vector<Class> classes;
    int images = 0;                      // nodes of all classes

    // Least-squares coefficients of the columns of E (weights over m values of
    // a, n frames) over its columns `nodes`, by Householder QR.
    static bool fit(std::vector<double> E, int m, int n, const std::vector<int>& nodes, std::vector<double>* lam) {
        const int r = (int)nodes.size();
        std::vector<double> B((size_t)m * r);
        for (int k = 0; k < m; k++)
            for (int j = 0; j < r; j++) B[(size_t)k * r + j] = E[(size_t)k * n + nodes[j]];
        for (int j = 0; j < r; j++) {
            double s = 0;
            for (int k = j; k < m; k++) s += B[(size_t)k * r + j] * B[(size_t)k * r + j];
            s = std::sqrt(s);
            if (!(s > 1e-300)) return false;
            if (B[(size_t)j * r + j] > 0) s = -s;
            std::vector<double> v(m - j);
            for (int k = j; k < m; k++) v[k - j] = B[(size_t)k * r + j];
            v[0] -= s;
            double vv = 0;
            for (double x : v) vv += x * x;
            if (!(vv > 0)) return false;
            auto reflect = [&](std::vector<double>& M, int w, int c0) {
                std::vector<double> d(w, 0.0);
                for (int k = j; k < m; k++)
                    for (int col = c0; col < w; col++) d[col] += v[k - j] * M[(size_t)k * w + col];
                for (int k = j; k < m; k++)
                    for (int col = c0; col < w; col++) M[(size_t)k * w + col] -= 2.0 / vv * d[col] * v[k - j];
            };
            reflect(B, r, j);
            reflect(E, n, 0);
        }
        lam->assign((size_t)n * r, 0.0);
        for (int i = 0; i < n; i++)
            for (int j = r - 1; j >= 0; j--) {
                double x = E[(size_t)j * n + i];
                for (int k = j + 1; k < r; k++) x -= B[(size_t)j * r + k] * (*lam)[(size_t)i * r + k];
                const double d = B[(size_t)j * r + j];
                if (d == 0) return false;
                (*lam)[(size_t)i * r + j] = x / d;
            }
        return true;
    }

    // The class `frames` with the fewest nodes, or its two halves.
    void add(const std::vector<int>& frames, const std::vector<int>& cum, const std::vector<double>& a,
             const std::vector<double>& rs, int rank, int half) {
        const int n = (int)frames.size();
        if (n == 0) return;
        std::vector<int> c(n);
        for (int i = 0; i < n; i++) c[i] = cum[frames[i]];
        const int m = (int)a.size();
        std::vector<double> E((size_t)m * n);
        for (int k = 0; k < m; k++)
            for (int i = 0; i < n; i++) E[(size_t)k * n + i] = std::exp(-a[k] * c[i]) * rs[k];
        // (five nodes serve about six frames at 1 e-/px: fewer are not tried)
        for (int r = std::min(n, 5); r <= std::min(rank, n); r++) {
            Class k;
            k.frames = frames;
            k.half = half;
            // nodes spread as the extrema of a Chebyshev polynomial
            for (int j = 0; j < r; j++) {
                int p = r == 1 ? 0 : (int)std::lround((n - 1) * 0.5 * (1 - std::cos(M_PI * j / (r - 1))));
                if (!k.nodes.empty()) p = std::max(p, k.nodes.back() + 1);
                k.nodes.push_back(std::min(p, n - r + j));
            }
            if (r == n) {
                k.lam.assign((size_t)n * n, 0.0);
                for (int i = 0; i < n; i++) k.lam[(size_t)i * n + i] = 1.0;
            } else {
                if (!fit(E, m, n, k.nodes, &k.lam)) continue;
                double worst = 0, big = 0;
                for (int q = 0; q < m; q++) {
                    const double* row = E.data() + (size_t)q * n;
                    double s = 0;
                    for (int i = 0; i < n; i++) {
                        double e = row[i];
                        for (int j = 0; j < r; j++) e -= k.lam[(size_t)i * r + j] * row[k.nodes[j]];
                        s += e * e;
                    }
                    worst = std::max(worst, std::sqrt(s));
                }
                for (int i = 0; i < n; i++) {
                    double s = 0;
                    for (int j = 0; j < r; j++) s += std::fabs(k.lam[(size_t)i * r + j]);
                    big = std::max(big, s);
                }
                // (coefficients that cancel would cost the sums digits)
                if (!(worst <= 2e-8) || !(big <= 4.0)) continue;
            }
            images += r;
            classes.push_back(k);
            return;
        }
        // cut at a gap of the doses, else in the middle
        int cut = n / 2, gap = 0;
        for (int i = 1; i < n; i++)
            if (c[i] - c[i - 1] > gap) {
                gap = c[i] - c[i - 1];
                cut = i;
            }
        if (gap < 4 * std::max(1, (c[n - 1] - c[0]) / n)) cut = n / 2;
        add(std::vector<int>(frames.begin(), frames.begin() + cut), cum, a, rs, rank, half);
        add(std::vector<int>(frames.begin() + cut, frames.end()), cum, a, rs, rank, half);
    }

    // cum: increasing raw-frame counts; in: frames in -SumRange (null: one
    // class); dw 0: plain sums only.
    SumPlan(int N, const std::vector<int>& cum, bool dw, double amax, const std::vector<char>* in, bool split,
            int rank) {
        // Chebyshev points of [0, amax], both ends among them
        std::vector<double> a(129), rs(129);
        for (int k = 0; k < 129; k++) {
            a[k] = 0.5 * amax * (1 - std::cos(M_PI * k / 128));
            double s = 0;
            for (int i = 0; i < N; i++) s += std::exp(-2 * a[k] * cum[i]);
            rs[k] = 1 / std::sqrt(s);
        }
        for (int h = 0; h < (split ? 2 : 1); h++)
            for (int q = 0; q < (dw && in ? 2 : 1); q++) {
                std::vector<int> f;
                for (int i = 0; i < N; i++)
                    if ((!split || (i & 1) == h) && (!(dw && in) || ((*in)[i] != 0) == (q == 0))) f.push_back(i);
                if (dw) {
                    add(f, cum, a, rs, rank, -1);
                } else if (!f.empty()) {
                    Class k;
                    k.frames = f;
                    k.half = split ? h : -1;
                    classes.push_back(k);
                }
            }
    }
};

// Everything a plan depends on.
struct SumPlanKey {
    std::vector<int> cum;
    std::vector<char> in;
    bool dw = false, split = false;
    double amax = 0;
    bool operator==(const SumPlanKey& o) const {
        return cum == o.cum && in == o.in && dw == o.dw && split == o.split && amax == o.amax;
    }
};
