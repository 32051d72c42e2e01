// Device side of the mixed-radix FFT used by the screen filter and the
// objective refocus: Stockham autosort stages over C lines held together in
// LDS, ping-ponging between two buffers.  Element k of line i sits at
// k*C + i, so the C lines of a block are read from HBM as rows of C
// consecutive complex values (columns of a plane) and the threads of a wave
// touch consecutive LDS words.  Stage with radix r after sub-transforms of
// length L:
//   y'[j + L p + L r k] = sum_q w_r^{pq} ( w_{Lr}^{jq} y[j + L k + (n/r) q] )
// Twiddles tw[t] = exp(-2 pi i t / n); sign < 0 is the forward transform
// (exp(-i)), sign > 0 the unnormalised backward one.
#pragma once

#include "device_common.h"
#include "kernels.h"

namespace nmk {

// t / d for 0 <= t < 2^16 and d >= 1: (t + 1/2) / d lies at least 1 / (2 d)
// from a whole number, 2^-18 of itself, which the float product cannot cross (a 32-bit
// division by a run-time value is a chain of some twenty instructions)
struct SmallDiv {
    float inv;
    __device__ explicit SmallDiv(int d) : inv(1.0f / (float)d) {}
    __device__ int operator()(int t) const { return (int)(((float)t + 0.5f) * inv); }
};

// one stage of radix R over the C lines of the block.  LM selects the LDS
// layout: line-major (element k of line i at i*n + k, rows) or interleaved
// (k*C + i, column tiles); work items run along the contiguous direction.
// P2: n is a power of two (there 512 lines of 256 points took 347 us a pass
// with the shorter divisions, 315 without: those waves are bound by memory).
template <int C, bool LM, int R, bool P2>
__device__ __forceinline__ void fft_stage(const c64 *__restrict__ b0, c64 *__restrict__ b1, int n, int L,
                                          const c64 *__restrict__ tw, int sign) {
    const int Lr = L * R, nb = n / R, tstep = n / Lr, rstep = n / R;
    auto W = [&](int idx) -> c64 {
        const c64 w = tw[idx];
        return sign > 0 ? conj(w) : w;
    };
    // R-th roots of unity of the butterfly
    c64 wr[R];
#pragma unroll
    for (int m = 0; m < R; m++) wr[m] = (R == 2 || R == 4) ? mk(1.0, 0.0) : W(m * rstep);
    const int step = LM ? 1 : C;          // LDS distance of consecutive elements of a line
    const SmallDiv by_nb(nb), by_L(L);
    for (int t = threadIdx.x; t < nb * C; t += blockDim.x) {
        const int i = LM ? (P2 ? t / nb : by_nb(t)) : t % C;
        const int b = LM ? t - i * nb : t / C;
        const int base = LM ? i * n : i;
        const int k = P2 ? b / L : by_L(b), j = P2 ? b % L : b - k * L;
        c64 u[R];
#pragma unroll
        for (int q = 0; q < R; q++) {
            const c64 v = b0[base + (j + L * k + rstep * q) * step];
            u[q] = (q == 0 || j == 0) ? v : v * W(j * q * tstep);
        }
        c64 *o = b1 + base + (j + Lr * k) * step;
        const int os = L * step;
        if constexpr (R == 2) {
            o[0] = u[0] + u[1];
            o[os] = u[0] - u[1];
        } else if constexpr (R == 4) {
            // w_4 = -i (forward) or +i (backward)
            const c64 t0 = u[0] + u[2], t1 = u[0] - u[2], t2 = u[1] + u[3], d = u[1] - u[3];
            const c64 t3 = sign > 0 ? mk(-d.y, d.x) : mk(d.y, -d.x);
            o[0] = t0 + t2;
            o[os] = t1 + t3;
            o[2 * os] = t0 - t2;
            o[3 * os] = t1 - t3;
        } else if constexpr (R == 8) {
            // two 4-point transforms of the even and odd inputs, joined by
            // w_8^k (k = 0..3; w_8^2 = -+i, w_8^1 and w_8^3 from the table)
            auto dft4 = [&](c64 a, c64 b, c64 c, c64 d, c64 (&y)[4]) {
                const c64 t0 = a + c, t1 = a - c, t2 = b + d, e = b - d;
                const c64 t3 = sign > 0 ? mk(-e.y, e.x) : mk(e.y, -e.x);
                y[0] = t0 + t2;
                y[1] = t1 + t3;
                y[2] = t0 - t2;
                y[3] = t1 - t3;
            };
            c64 ev[4], od[4];
            dft4(u[0], u[2], u[4], u[6], ev);
            dft4(u[1], u[3], u[5], u[7], od);
            const c64 o1 = od[1] * wr[1], o3 = od[3] * wr[3];
            const c64 o2 = sign > 0 ? mk(-od[2].y, od[2].x) : mk(od[2].y, -od[2].x);
            o[0] = ev[0] + od[0];
            o[os] = ev[1] + o1;
            o[2 * os] = ev[2] + o2;
            o[3 * os] = ev[3] + o3;
            o[4 * os] = ev[0] - od[0];
            o[5 * os] = ev[1] - o1;
            o[6 * os] = ev[2] - o2;
            o[7 * os] = ev[3] - o3;
        } else {
            // odd: outputs k and R - k share the products of the folded inputs
            // s_q = u_q + u_{R-q} with the cosines and d_q = u_q - u_{R-q}
            // with the sines (a quarter of the direct sum's multiplications)
            constexpr int H = R / 2;
            c64 sum = u[0];
#pragma unroll
            for (int q = 1; q <= H; q++) {
                const c64 d = u[q] - u[R - q];
                u[q] = u[q] + u[R - q];
                u[R - q] = d;
                sum = sum + u[q];
            }
            o[0] = sum;
#pragma unroll
            for (int k1 = 1; k1 <= H; k1++) {
                c64 a = u[0], e = mk(0.0, 0.0);
#pragma unroll
                for (int q = 1; q <= H; q++) {
                    const int m = (k1 * q) % R;  // (the second half mirrors the first: fewer registers)
                    const c64 w = m <= H ? wr[m] : conj(wr[R - m]);
                    a = mk(fma(u[q].x, w.x, a.x), fma(u[q].y, w.x, a.y));
                    e = mk(fma(u[R - q].x, w.y, e.x), fma(u[R - q].y, w.y, e.y));
                }
                o[k1 * os] = mk(a.x - e.y, a.y + e.x);
                o[(R - k1) * os] = mk(a.x + e.y, a.y - e.x);
            }
        }
    }
}

// One stage of any odd radix R (primes above 13), as a product with the
// matrix of cosines and sines.  The inputs of a butterfly are folded first,
// s_q = u_q + u_{R-q} and d_q = u_q - u_{R-q}, so that
//   X_k, X_{R-k} = (u_0 + sum_q s_q cos) -+ i (sum_q d_q sin),  q, k <= R / 2
// are two real products for both outputs, a quarter of the multiplications of
// the direct sum.  They run on the FP64 matrix cores (16 outputs k x 16
// columns, four terms q a step): a column is the real or imaginary part of one
// butterfly, so that neither operand needs more than one LDS word per lane and
// step.  Waves take the tiles in turn; rows past R / 2 and terms past it are
// padding.  161 points (7 x 23), 532 planes of 161 lines: rows 144-180 us and the
// refocus columns 280 us a pass, where the direct sum over the whole length
// took 844 us for each of their transforms; the bound is latency (two blocks
// of waves a CU, a barrier between the short stages), not the matrix cores,
// busy about a tenth of it.
template <int C, bool LM>
__device__ __forceinline__ void fft_stage_any(c64 *__restrict__ b0, c64 *__restrict__ b1, int n, int L, int R,
                                              const c64 *__restrict__ tw, int sign) {
    typedef double v4d __attribute__((ext_vector_type(4)));
    const int nb = n / R, H = R / 2, cols = nb * C, tstep = n / (L * R);
    const int step = LM ? 1 : C, qs = nb * step;  // LDS distances of consecutive elements, and of inputs of a butterfly
    const SmallDiv by_cols(cols), by_nb(nb), by_L(L);
    for (int t = threadIdx.x; t < H * cols; t += blockDim.x) {
        const int q = 1 + by_cols(t), c = t - (q - 1) * cols;
        const int i = LM ? by_nb(c) : c % C, b = LM ? c - i * nb : c / C;
        c64 *x = b0 + (LM ? i * n + b : c);
        c64 u = x[q * qs], v = x[(R - q) * qs];
        const int j = b - by_L(b) * L;
        if (j) {
            const c64 wu = tw[j * q * tstep], wv = tw[j * (R - q) * tstep];
            u = u * (sign > 0 ? conj(wu) : wu);
            v = v * (sign > 0 ? conj(wv) : wv);
        }
        x[q * qs] = u + v;
        x[(R - q) * qs] = u - v;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int nct = (cols + 7) / 8, nkt = (H + 16) / 16;
    const SmallDiv by_nct(nct), by_R(R);
    for (int tile = threadIdx.x >> 6; tile < nct * nkt; tile += blockDim.x >> 6) {
        const int kt = by_nct(tile), ct = tile - kt * nct;
        const int c = min(ct * 8 + (r >> 1), cols - 1), part = r & 1;
        const int i = LM ? by_nb(c) : c % C, b = LM ? c - i * nb : c / C;
        const double *x = reinterpret_cast<const double *>(b0 + (LM ? i * n + b : c)) + part;
        const int k = min(kt * 16 + r, H), inc = 4 * k - by_R(4 * k) * R;
        int idx = k * (1 + g) - by_R(k * (1 + g)) * R;
        v4d sc = {x[0], x[0], x[0], x[0]}, sd = {0.0, 0.0, 0.0, 0.0};
        for (int q = 1 + g; q - g <= H; q += 4) {
            const bool in = q <= H;
            const int qq = in ? q : 1;
            const c64 w = tw[idx * nb];
            const double s = x[2 * qq * qs], d = x[2 * (R - qq) * qs];
            sc = __builtin_amdgcn_mfma_f64_16x16x4f64(w.x, in ? s : 0.0, sc, 0, 0, 0);
            sd = __builtin_amdgcn_mfma_f64_16x16x4f64(w.y, in ? d : 0.0, sd, 0, 0, 0);
            idx += inc;
            if (idx >= R) idx -= R;
        }
        // w.y is the forward -sin: X_k = sc + i sd of the complex columns
        const int kk = by_L(b);
        double *o = reinterpret_cast<double *>(b1 + (LM ? i * n : i) + (b - kk * L + L * R * kk) * step) + part;
        const bool mine = ct * 8 + (r >> 1) < cols;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const double other = __shfl_xor(sd[e], 1);
            double term = part ? other : -other;
            if (sign > 0) term = -term;
            const int ko = kt * 16 + 4 * e + g;  // row of the product held here
            if (mine && ko <= H) o[2 * ko * L * step] = sc[e] + term;
            if (mine && ko <= H && ko) o[2 * (R - ko) * L * step] = sc[e] - term;
        }
    }
}

// radices a plan may hold: 2, 4 and 8; those and the primes to 13; any
enum { FFT_POW2 = 0, FFT_SMALL = 1, FFT_ANY = 2 };

// runs every stage of plan pl on the C lines in b0 (all threads of the block
// take part; the caller has synchronised after filling b0 and the twiddle
// table tw, normally an LDS copy) and returns the buffer that holds the result
// (MODE: the radices compiled, which keeps the power-of-two kernels small)
template <int C, bool LM, int MODE>
__device__ c64 *fft_stages(c64 *b0, c64 *b1, const FftPlan &pl, const c64 *__restrict__ tw, int sign) {
    const int n = pl.n;
    int L = 1;
    for (int st = 0; st < pl.nst; st++) {
        int r = (int)((pl.radices >> (4 * st)) & 15);
        if (r == 4) fft_stage<C, LM, 4, MODE == FFT_POW2>(b0, b1, n, L, tw, sign);
        else if (r == 8) fft_stage<C, LM, 8, MODE == FFT_POW2>(b0, b1, n, L, tw, sign);
        else if (r == 2) fft_stage<C, LM, 2, MODE == FFT_POW2>(b0, b1, n, L, tw, sign);
        else if constexpr (MODE >= FFT_SMALL) {
            switch (r) {
            case 3: fft_stage<C, LM, 3, MODE == FFT_POW2>(b0, b1, n, L, tw, sign); break;
            case 5: fft_stage<C, LM, 5, MODE == FFT_POW2>(b0, b1, n, L, tw, sign); break;
            case 7: fft_stage<C, LM, 7, MODE == FFT_POW2>(b0, b1, n, L, tw, sign); break;
            case 11: fft_stage<C, LM, 11, MODE == FFT_POW2>(b0, b1, n, L, tw, sign); break;
            case 13: fft_stage<C, LM, 13, MODE == FFT_POW2>(b0, b1, n, L, tw, sign); break;
            default:
                if constexpr (MODE == FFT_ANY) {
                    r = pl.big[st];
                    fft_stage_any<C, LM>(b0, b1, n, L, r, tw, sign);
                }
            }
        }
        __syncthreads();
        c64 *tmp = b0;
        b0 = b1;
        b1 = tmp;
        L *= r;
    }
    return b0;
}

__host__ inline int fft_mode(const FftPlan &pl) {
    int mode = FFT_POW2;
    for (int st = 0; st < pl.nst; st++) {
        const int r = (int)((pl.radices >> (4 * st)) & 15);
        if (r == 15) return FFT_ANY;
        if (r != 2 && r != 4 && r != 8) mode = FFT_SMALL;
    }
    return mode;
}

// lines per block: at least 1024 values per block of 256 threads (one
// radix-4 butterfly per thread and stage); with a matrix-core stage, whose
// tiles are eight columns wide, twice as many, and as many as LDS holds
// beyond 1024 points
__host__ __device__ constexpr int fft_lines_per_block(int n, int cap, bool any) {
    int c = 1;
    while (2 * c <= cap && 2 * c * n <= (any ? 2048 : 1024)) c *= 2;
    while (any && c < 4 && 2 * c * n <= 4096) c *= 2;
    return c;
}
// LDS bytes of a block: two line buffers and the twiddle table
__host__ __device__ constexpr size_t fft_lds_bytes(int n, int C) { return (size_t)(2 * C + 1) * n * 16; }

}  // namespace nmk
