// PME grid transforms of any length as dense products on the FP64 matrix cores.
//
// A length-m DFT folded about its middle is two real products: with
// s_r = v_r + v_(m-r) and d_r = v_r - v_(m-r) (r = 0 .. m/2; at r = 0 and r = m/2
// s = v, d = 0),
//   A_q = sum_r s_r cos(2 pi r q / m),   B_q = sum_r d_r sin(2 pi r q / m),
//   X_q = A_q -+ i B_q,   X_(m-q) = A_q +- i B_q   (q = 0 .. m/2),
// so a batch of lines is an (m/2+1) x (m/2+1) cosine and a sine matrix times a
// block of 16 columns: v_mfma_f64_16x16x4 tiles of 16 outputs by 16 columns (8
// complex columns -- a 128-byte segment of the half spectrum's rows, copied
// without transposing -- or 16 real lines), 4 inputs a step.  The matrix elements
// are gathered from the m roots of unity in LDS.  The x and y passes first split a
// length N = F m by an F-point stage in registers (F <= 4), which leaves F
// products of length m: F times fewer multiplications.  One block takes 16
// columns; its waves take the tiles of outputs in turn.  The same five passes as
// kernels_fft.hip, over the same arrays.
//
// What bounds them: one round trip of the grid through the cache and HBM, and
// after it the matrix products (their phases overlap little within a block).  At
// 182^3 the y pass takes 29 us, 18 of them without any product (97.5 MB, 5.3
// TB/s) and 8 the products at the FP64 matrix rate; the mixed radix took 103 us
// (16-byte segments, one line a block).  Without the front stage it is 41 us,
// with one of 7 points (28 products a tile column instead of 72) 40 us: too few
// threads have work in that stage.
#include <algorithm>

#include "device_common.h"
#include "fft_kernels.h"
#include "fft_roots.h"

namespace mbpol {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

constexpr int kCol = 16;     // columns of a tile
constexpr int kColPad = 17;  // row length of the z passes' LDS block (transposed on the way in: no bank conflicts)
constexpr int kMaxWaves = 8;
constexpr int kMaxThreads = 64 * kMaxWaves;

// (cos, sin)(2 pi t / m) into LDS for m = n / step, and a zero entry for t = m
__device__ __forceinline__ void load_roots(double2* roots, const FftAxis& ax, int m, int step) {
    for (int t = threadIdx.x; t <= m; t += blockDim.x)
        roots[t] = t < m ? make_double2(ax.tw[t * step].x, -ax.tw[t * step].y) : make_double2(0.0, 0.0);
}

// One tile of outputs q0 .. q0 + 15 from the folded inputs r = 0 .. N/2 of 16
// columns: A = sum s_r cos, B = sum d_r sin, with s_r at s[r * LD + column] and
// d_r at d[r * DLD + column].
// DATA_ROWS: the data is the left operand (result rows = columns of the data,
// result columns = q), else the right one (result rows = q).
// Operand layout of the 16x16x4 product: lane l holds row/column l % 16 at k = l / 16; the result's
// element v of lane l is row 4 v + l / 16, column l % 16.
template <bool DATA_ROWS, int LD, int DLD>
__device__ __forceinline__ void dft_tile(int N, int q0, const double2* roots, const double* s, const double* d, d4& A,
                                         d4& B) {
    const int lane = threadIdx.x & 63, i = lane & 15, k = lane >> 4;
    const int q = min(q0 + i, N >> 1);  // outputs beyond the middle repeat it and are not stored
    unsigned idx = q * k, inc = 4 * q;  // root of (r, q): r q mod N
    while (idx >= (unsigned)N) idx -= N;
    while (inc >= (unsigned)N) inc -= N;
    const int K = (N >> 1) + 1, full = K >> 2;
    s += k * LD + i;
    d += k * DLD + i;
    A = d4{0.0, 0.0, 0.0, 0.0};
    B = d4{0.0, 0.0, 0.0, 0.0};
    auto step = [&](double2 w, double sv, double dv) {
        if constexpr (DATA_ROWS) {
            A = __builtin_amdgcn_mfma_f64_16x16x4f64(sv, w.x, A, 0, 0, 0);
            B = __builtin_amdgcn_mfma_f64_16x16x4f64(dv, w.y, B, 0, 0, 0);
        } else {
            A = __builtin_amdgcn_mfma_f64_16x16x4f64(w.x, sv, A, 0, 0, 0);
            B = __builtin_amdgcn_mfma_f64_16x16x4f64(w.y, dv, B, 0, 0, 0);
        }
    };
    auto next = [&]() {
        const unsigned t = idx;
        idx = min(idx + inc, idx + inc - N);  // the smaller of the two as unsigned numbers: reduced mod N
        return t;
    };
    int t = 0;
    constexpr int U = 4;
    for (; t + U <= full; t += U) {
        double2 w[U];
        double sv[U], dv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            w[u] = roots[next()];
            sv[u] = s[u * 4 * LD];
            dv[u] = d[u * 4 * DLD];
        }
        s += U * 4 * LD;
        d += U * 4 * DLD;
#pragma unroll
        for (int u = 0; u < U; ++u) step(w[u], sv[u], dv[u]);
    }
    for (; t < full; ++t) {
        step(roots[next()], s[0], d[0]);
        s += 4 * LD;
        d += 4 * DLD;
    }
    if (K & 3) {  // the last inputs: the rows past N/2 meet the zero root
        const bool in = 4 * full + k < K;
        step(roots[in ? idx : N], in ? s[0] : 0.0, in ? d[0] : 0.0);
    }
}

// value of the neighbouring lane (lane ^ 1)
__device__ __forceinline__ double swap_pair(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_mov_dpp(lo, 0xB1, 0xf, 0xf, true);  // quad_perm 1,0,3,2
    hi = __builtin_amdgcn_mov_dpp(hi, 0xB1, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// F-point DFT of v in place (inv: the conjugate roots)
template <int F>
__device__ __forceinline__ void small_dft(double (&x)[F], double (&y)[F], bool inv) {
    if constexpr (F == 1) return;
    if constexpr (F == 2) {
        const double ax = x[0] - x[1], ay = y[0] - y[1];
        x[0] += x[1];
        y[0] += y[1];
        x[1] = ax;
        y[1] = ay;
    }
    if constexpr (F == 4) {
        const double ax = x[0] + x[2], ay = y[0] + y[2], bx = x[0] - x[2], by = y[0] - y[2];
        const double cx = x[1] + x[3], cy = y[1] + y[3];
        const double dx = inv ? y[3] - y[1] : y[1] - y[3], dy = inv ? x[1] - x[3] : x[3] - x[1];  // -+ i (v1 - v3)
        x[0] = ax + cx;
        y[0] = ay + cy;
        x[2] = ax - cx;
        y[2] = ay - cy;
        x[1] = bx + dx;
        y[1] = by + dy;
        x[3] = bx - dx;
        y[3] = by - dy;
    }
    if constexpr (F % 2 == 1 && F > 1) {
        constexpr int H = F / 2;
        double sx[H], sy[H], dx[H], dy[H], x0 = x[0], y0 = y[0];
        const double sg = inv ? -1.0 : 1.0;
#pragma unroll
        for (int r = 1; r <= H; ++r) {
            sx[r - 1] = x[r] + x[F - r];
            sy[r - 1] = y[r] + y[F - r];
            dx[r - 1] = sg * (x[r] - x[F - r]);
            dy[r - 1] = sg * (y[r] - y[F - r]);
        }
#pragma unroll
        for (int r = 0; r < H; ++r) {
            x[0] += sx[r];
            y[0] += sy[r];
        }
#pragma unroll
        for (int q = 1; q <= H; ++q) {
            double ax = x0, ay = y0, bx = 0.0, by = 0.0;
#pragma unroll
            for (int r = 1; r <= H; ++r) {
                const double c = Roots<F>::c[(r * q) % F], sn = Roots<F>::s[(r * q) % F];
                ax += sx[r - 1] * c;
                ay += sy[r - 1] * c;
                bx += dx[r - 1] * sn;
                by += dy[r - 1] * sn;
            }
            x[q] = ax + by;
            y[q] = ay - bx;
            x[F - q] = ax - by;
            y[F - q] = ay + bx;
        }
    }
}

// Front stage of 8 complex columns of length N = F m: the F-point DFTs over the
// rows n + j m, their twiddles, and the fold about the middle of each of the F
// sequences of length m that are left: sequence p's s_r in row p m + r of v, its
// d_r in row p m + m - r.  src(row, column) reads the input.
template <int F, typename Src>
__device__ __forceinline__ void front_stage(double* v, const FftAxis& ax, bool inv, Src&& src) {
    double2* v2 = reinterpret_cast<double2*>(v);
    constexpr int R = kCol / 2;
    const int N = ax.n, m = N / F, items = ((m >> 1) + 1) * R;
    for (int e = threadIdx.x; e < items; e += blockDim.x) {
        const int n = e / R, c = e % R;
        const bool self = n == 0 || 2 * n == m;
        const int n2 = self ? n : m - n;
        double x[2][F], y[2][F];
#pragma unroll
        for (int j = 0; j < F; ++j) {
            src(n + j * m, c, x[0][j], y[0][j]);
            src(n2 + j * m, c, x[1][j], y[1][j]);
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            small_dft<F>(x[h], y[h], inv);
#pragma unroll
            for (int p = 1; p < F; ++p) {
                const double2 w = ax.tw[(h ? n2 : n) * p];
                const double wy = inv ? -w.y : w.y, t = x[h][p] * w.x - y[h][p] * wy;
                y[h][p] = x[h][p] * wy + y[h][p] * w.x;
                x[h][p] = t;
            }
        }
#pragma unroll
        for (int p = 0; p < F; ++p) {
            double2* seq = v2 + p * m * R;
            if (self) {
                seq[e] = make_double2(x[0][p], y[0][p]);
            } else {
                seq[e] = make_double2(x[0][p] + x[1][p], y[0][p] + y[1][p]);
                seq[(m - n) * R + c] = make_double2(x[0][p] - x[1][p], y[0][p] - y[1][p]);
            }
        }
    }
    if (threadIdx.x < kCol) v[N * kCol + threadIdx.x] = 0.0;
}

// The products of 8 complex columns (16 interleaved doubles) after the front
// stage; out(k, X_k, k2, X_k2) receives this lane's column of every pair of outputs
// k = F q + p, k2 = F (m - q) + p (k2 = -1: none)
template <int F, typename Out>
__device__ __forceinline__ void complex_columns(const double* v, int N, const double2* roots, bool inv, Out&& out) {
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6, m = N / F, tiles = ((m >> 1) + 16) >> 4;
    const bool imag = lane & 1;
    // X_q = A -+ i B on interleaved columns: the other component's B with a sign
    const double sg = imag != inv ? -1.0 : 1.0;
    for (int t = threadIdx.x >> 6; t < F * tiles; t += nw) {
        const int p = t / tiles, q0 = 16 * (t - p * tiles);
        d4 A, B;
        dft_tile<false, kCol, -kCol>(m, q0, roots, v + p * m * kCol, v + (p + 1) * m * kCol, A, B);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int q = q0 + 4 * e + (lane >> 4);
            const double b = sg * swap_pair(B[e]);
            if (2 * q <= m) out(F * q + p, A[e] + b, q != 0 && 2 * q != m ? F * (m - q) + p : -1, A[e] - b);
        }
    }
}

// y pass, either direction, in place: block = (x, 8 consecutive kz)
template <int F>
__global__ void __launch_bounds__(kMaxThreads) k_dft_y(double2* __restrict__ H, int ntile, int Khp, FftAxis ay, int inv,
                                                       const int* __restrict__ stop) {
    critical_path_wave();
    extern __shared__ double2 lds[];
    if (stop && *stop) return;
    const int N = ay.n, m = N / F, x = blockIdx.x / ntile, kz0 = (blockIdx.x - x * ntile) * 8;
    double2* roots = lds;
    double* v = reinterpret_cast<double*>(lds + m + 1);
    double2* col = H + (size_t)x * N * Khp + kz0;
    front_stage<F>(v, ay, inv != 0, [&](int row, int c, double& re, double& im) {
        const double2* p = col + (size_t)row * Khp + c;
        re = p->x;
        im = p->y;
    });
    load_roots(roots, ay, m, F);
    __syncthreads();
    double* dst = reinterpret_cast<double*>(col) + (threadIdx.x & 15);
    complex_columns<F>(v, N, roots, inv != 0, [&](int k, double a, int k2, double b) {
        dst[(size_t)k * 2 * Khp] = a;
        if (k2 >= 0) dst[(size_t)k2 * 2 * Khp] = b;
    });
}

// x pass in place: forward, influence function, inverse; block = (y, 8 consecutive kz)
template <int F>
__global__ void __launch_bounds__(kMaxThreads) k_dft_x_conv(double2* __restrict__ H, const double* __restrict__ influence,
                                                            int ntile, int K1, int Khp, FftAxis ax,
                                                            const int* __restrict__ stop) {
    critical_path_wave();
    extern __shared__ double2 lds[];
    if (stop && *stop) return;
    const int N = ax.n, m = N / F, y = blockIdx.x / ntile, kz0 = (blockIdx.x - y * ntile) * 8;
    double2* roots = lds;
    double* v = reinterpret_cast<double*>(lds + m + 1);
    double* w = v + (N + 1) * kCol;
    const size_t stride = (size_t)K1 * Khp;
    double2* col = H + (size_t)y * Khp + kz0;
    front_stage<F>(v, ax, false, [&](int row, int c, double& re, double& im) {
        const double2* p = col + (size_t)row * stride + c;
        re = p->x;
        im = p->y;
    });
    load_roots(roots, ax, m, F);
    __syncthreads();
    const int c = threadIdx.x & 15;
    const double* inf = influence + (size_t)y * Khp + kz0 + (c >> 1);
    complex_columns<F>(v, N, roots, false, [&](int k, double a, int k2, double b) {
        w[k * kCol + c] = a * inf[(size_t)k * stride];
        if (k2 >= 0) w[k2 * kCol + c] = b * inf[(size_t)k2 * stride];
    });
    __syncthreads();
    const double2* w2 = reinterpret_cast<const double2*>(w);
    front_stage<F>(v, ax, true, [&](int row, int cc, double& re, double& im) {
        re = w2[row * (kCol / 2) + cc].x;
        im = w2[row * (kCol / 2) + cc].y;
    });
    __syncthreads();
    double* dst = reinterpret_cast<double*>(col) + c;
    complex_columns<F>(v, N, roots, true, [&](int k, double a, int k2, double b) {
        dst[(size_t)k * 2 * stride] = a;
        if (k2 >= 0) dst[(size_t)k2 * 2 * stride] = b;
    });
}

// s and d of points z and N - z of one line into rows z and N - z
__device__ __forceinline__ void store_folded(double* v, int N, int z, int l, double a, double b) {
    if (z == 0 || 2 * z == N) {
        v[z * kColPad + l] = a;
    } else {
        v[z * kColPad + l] = a + b;
        v[(N - z) * kColPad + l] = a - b;
    }
}

// forward z transform of the block's 16 real lines, folded in v -> half spectrum rows
__device__ __forceinline__ void z_forward(const double* v, const double2* roots, double2* __restrict__ H, int L0,
                                          int nlines, int N, int Khp) {
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    for (int q0 = 16 * (threadIdx.x >> 6); q0 <= N >> 1; q0 += 16 * nw) {
        d4 A, B;
        dft_tile<true, kColPad, -kColPad>(N, q0, roots, v, v + N * kColPad, A, B);
        const int q = q0 + (lane & 15);
        if (2 * q <= N) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int l = L0 + 4 * e + (lane >> 4);
                if (l < nlines) {
                    double2* dst = H + (size_t)l * Khp + q;
                    dst->x = A[e];
                    dst->y = -B[e];
                }
            }
        }
    }
}

// z pass, forward: 16 lines of the real grid a block
__global__ void __launch_bounds__(kMaxThreads) k_dft_z_r2c(const double* __restrict__ real, double2* __restrict__ H,
                                                           int nlines, FftAxis az, int Khp,
                                                           const int* __restrict__ stop) {
    critical_path_wave();
    extern __shared__ double2 lds[];
    if (stop && *stop) return;
    const int N = az.n, L0 = blockIdx.x * kCol, m = min(kCol, nlines - L0);
    double2* roots = lds;
    double* v = reinterpret_cast<double*>(lds + N + 1);
    const double* src = real + (size_t)L0 * N;
    for (int l = threadIdx.x >> 4; l < kCol; l += blockDim.x >> 4)  // 16 lanes a line
        for (int z = threadIdx.x & 15; 2 * z <= N; z += 16) {
            const double* p = src + (size_t)l * N;
            store_folded(v, N, z, l, l < m ? p[z] : 0.0, l < m && z > 0 ? p[N - z] : 0.0);
        }
    if (threadIdx.x < kCol) v[N * kColPad + threadIdx.x] = 0.0;
    load_roots(roots, az, N, 1);
    __syncthreads();
    z_forward(v, roots, H, L0, nlines, N, Khp);
}

// Adds the entries b .. e - 1 of one grid line to the points z0 .. z0 + len - 1 in
// v[(z - z0) * kColPad + l] (WHOLE: z0 = 0 and len = N, every point of an entry
// falls in), with 16 lanes, 3 entries at a time: lane 5 t + z adds point z of entry
// t, the entries one after the other (entries of a line may overlap, so their order
// is kept within the wave).  The loads of 12 entries are in flight together:
// latency, not the table's bytes, is what the kernel waits for.
// Before: a table by grid point, one thread summing 8 points' rows, 18.4 us at 99^3
// (6591 sites) and 25 us at 121^3 (12288 sites), z pass included; now 16.9 and 22.2.
template <bool CHARGES, bool WHOLE>
__device__ __forceinline__ void spread_entries(double* v, const LineTable& T, const double* __restrict__ w, int b, int e,
                                               int l, int z0, int len) {
    const int N = T.nz, lane = threadIdx.x & 15, t = lane / 5, z = lane - 5 * t;
    constexpr int U = 4;
    for (int k = b; k < e; k += 3 * U) {
        double val[U];
        int at[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int en = k + 3 * u + t;
            at[u] = -1;
            val[u] = 0.0;
            if (t < 3 && en < e) {
                const int2 s = T.sz[en];
                int p = s.y + z;
                p = p >= N ? p - N : p;
                if (WHOLE || (unsigned)(p - z0) < (unsigned)len) {
                    const double* sp = T.sptab + 30 * (size_t)s.x + 20 + z;
                    const double* c = T.coef + 3 * (size_t)en;
                    const double c2 = c[2];
                    if constexpr (CHARGES)
                        val[u] = w[s.x] * c2 * sp[0];
                    else
                        val[u] = (w[3 * s.x] * c[0] + w[3 * s.x + 1] * c[1]) * sp[0] +
                                 w[3 * s.x + 2] * T.scale_z * c2 * sp[5];
                    at[u] = (WHOLE ? p : p - z0) * kColPad + l;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int o = 0; o < 3; ++o) {
                if (t == o && at[u] >= 0) v[at[u]] += val[u];
                // the next entry's lanes read after this one's have written (LDS keeps a wave's order)
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
    }
}

// The block's 16 whole lines from the spreading table into v[z * kColPad + line] (zeroed here; unfolded)
template <bool CHARGES>
__device__ __forceinline__ void spread_lines(double* v, const LineTable& T, const double* __restrict__ w, int L0, int m) {
    const int N = T.nz;
    for (int e = threadIdx.x; e < N * kColPad; e += blockDim.x) v[e] = 0.0;
    __syncthreads();
    for (int l = threadIdx.x >> 4; l < m; l += blockDim.x >> 4)
        for (int part = 0; part < (CHARGES ? 2 : 1); ++part) {
            const int* row = T.start + (size_t)(L0 + l + part * T.nlines) * T.nseg;
            spread_entries<CHARGES, true>(v, T, w, row[0], row[T.nseg], l, 0, N);
        }
}

// spreading fused with the forward z pass: the real grid is neither written nor read back
template <bool CHARGES>
__global__ void __launch_bounds__(kMaxThreads) k_spread_dft_z_r2c(LineTable T, const double* __restrict__ w,
                                                                  double2* __restrict__ H, FftAxis az, int Khp,
                                                                  const int* __restrict__ stop) {
    critical_path_wave();
    extern __shared__ double2 lds[];
    if (stop && *stop) return;
    const int N = az.n, L0 = blockIdx.x * kCol, m = min(kCol, T.nlines - L0);
    double2* roots = lds;
    double* v = reinterpret_cast<double*>(lds + N + 1);
    spread_lines<CHARGES>(v, T, w, L0, m);
    __syncthreads();
    for (int e = threadIdx.x; e < kCol * ((N >> 1) + 1); e += blockDim.x) {
        const int z = e >> 4, l = e & 15;
        if (z > 0 && 2 * z < N) store_folded(v, N, z, l, v[z * kColPad + l], v[(N - z) * kColPad + l]);
    }
    if (threadIdx.x < kCol) v[N * kColPad + threadIdx.x] = 0.0;
    load_roots(roots, az, N, 1);
    __syncthreads();
    z_forward(v, roots, H, L0, T.nlines, N, Khp);
}

// Spreading onto the real grid, for the other transforms: a block takes one segment
// of 16 lines, whose entries start in it or reach over from the segment before (the
// one before the first is the last).  Segments bound the LDS of a block whatever the
// length of the axis (whole lines end at 1204 points), and share the entries of a
// long line, which its 16 lanes add one after the other, among several blocks.
// Electrostatics of 3430 waters on 52 x 52 x 512 points: 2.66 ms with whole lines,
// 2.28 now; of 6370 waters on 52 x 52 x 1000: 4.90, 4.09.
constexpr int kSpreadThreads = 256;
template <bool CHARGES>
__global__ void __launch_bounds__(kSpreadThreads) k_spread_lines(LineTable T, const double* __restrict__ w,
                                                                 double* __restrict__ real,
                                                                 const int* __restrict__ stop) {
    critical_path_wave();
    extern __shared__ double2 lds[];
    if (stop && *stop) return;
    const int seg = blockIdx.x % T.nseg, L0 = (int)(blockIdx.x / T.nseg) * kCol, m = min(kCol, T.nlines - L0);
    const int z0 = segment_start(seg, T.nz, T.nseg), len = segment_start(seg + 1, T.nz, T.nseg) - z0;
    double* v = reinterpret_cast<double*>(lds);
    for (int e = threadIdx.x; e < len * kColPad; e += blockDim.x) v[e] = 0.0;
    __syncthreads();
    const int before = seg == 0 ? T.nseg - 1 : seg - 1;
    for (int l = threadIdx.x >> 4; l < m; l += blockDim.x >> 4)
        for (int part = 0; part < (CHARGES ? 2 : 1); ++part) {
            const int* row = T.start + (size_t)(L0 + l + part * T.nlines) * T.nseg;
            spread_entries<CHARGES, false>(v, T, w, row[seg], row[seg + 1], l, z0, len);
            if (before != seg) spread_entries<CHARGES, false>(v, T, w, row[before], row[before + 1], l, z0, len);
        }
    __syncthreads();
    for (int l = threadIdx.x >> 4; l < m; l += blockDim.x >> 4)
        for (int z = threadIdx.x & 15; z < len; z += 16)
            real[(size_t)(L0 + l) * T.nz + z0 + z] = v[z * kColPad + l];
}

// z pass, inverse: half spectrum -> 16 real lines a block:
// v_n = E_n - O_n, v_(N-n) = E_n + O_n with E = sum_k w_k Re X_k cos, O = sum_k w_k Im X_k sin,
// w = 1 at k = 0 and k = N/2, else 2
__global__ void __launch_bounds__(kMaxThreads) k_dft_z_c2r(const double2* __restrict__ H, double* __restrict__ real,
                                                           int nlines, FftAxis az, int Khp,
                                                           const int* __restrict__ stop) {
    critical_path_wave();
    extern __shared__ double2 lds[];
    if (stop && *stop) return;
    const int N = az.n, Kh = (N >> 1) + 1, L0 = blockIdx.x * kCol, m = min(kCol, nlines - L0);
    double2* roots = lds;
    double* xr = reinterpret_cast<double*>(lds + N + 1);
    double* xi = xr + Kh * kColPad;
    for (int l = threadIdx.x >> 4; l < kCol; l += blockDim.x >> 4)
        for (int k = threadIdx.x & 15; k < Kh; k += 16) {
            double re = 0.0, im = 0.0;
            if (l < m) {
                const double2* p = H + (size_t)(L0 + l) * Khp + k;
                const double w = (k == 0 || 2 * k == N) ? 1.0 : 2.0;
                re = w * p->x;
                im = w * p->y;
            }
            xr[k * kColPad + l] = re;
            xi[k * kColPad + l] = im;
        }
    load_roots(roots, az, N, 1);
    __syncthreads();
    const int lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    for (int q0 = 16 * (threadIdx.x >> 6); q0 <= N >> 1; q0 += 16 * nw) {
        d4 A, B;
        dft_tile<true, kColPad, kColPad>(N, q0, roots, xr, xi, A, B);
        const int q = q0 + (lane & 15);
        if (2 * q <= N) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int l = L0 + 4 * e + (lane >> 4);
                if (l < nlines) {
                    double* dst = real + (size_t)l * N;
                    dst[q] = A[e] - B[e];
                    if (q != 0 && 2 * q != N) dst[N - q] = A[e] + B[e];
                }
            }
        }
    }
}

}  // namespace

static inline int nblk(long long n, int b) { return (int)((n + b - 1) / b); }
// one wave per tile of 16 outputs, at most kMaxWaves
static int threads(const FftAxis& a, int f) { return 64 * std::min(kMaxWaves, f * nblk(a.n / f / 2 + 1, 16)); }
static size_t roots_bytes(const FftAxis& a, int f) { return sizeof(double2) * (size_t)(a.n / f + 1); }
static size_t columns_bytes(const FftAxis& a) { return sizeof(double) * kCol * (size_t)(a.n + 1); }
static size_t z_bytes(const FftAxis& a) { return roots_bytes(a, 1) + sizeof(double) * kColPad * (size_t)(a.n + 1); }

hipError_t dft_allow_lds() {
    for (const void* kern : {(const void*)k_dft_z_r2c, (const void*)k_spread_dft_z_r2c<true>,
                             (const void*)k_spread_dft_z_r2c<false>, (const void*)k_dft_z_c2r, (const void*)k_dft_y<1>,
                             (const void*)k_dft_y<2>, (const void*)k_dft_y<3>, (const void*)k_dft_y<4>,
                             (const void*)k_dft_x_conv<1>, (const void*)k_dft_x_conv<2>, (const void*)k_dft_x_conv<3>,
                             (const void*)k_dft_x_conv<4>}) {
        const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

void launch_dft_z_r2c(hipStream_t s, const PmeFft& F, const double* real, double2* H, const KEvents& ev,
                      const int* stop) {
    const int nl = F.ax[0].n * F.ax[1].n;
    MBPOL_LAUNCH(ev, k_dft_z_r2c, nblk(nl, kCol), threads(F.ax[2], 1), z_bytes(F.ax[2]), s, real, H, nl, F.ax[2], F.khp,
                 stop);
}
void launch_spread_dft_z_r2c(hipStream_t s, const PmeFft& F, const LineTable& T, bool charges, const double* w,
                             double2* H, const KEvents& ev, const int* stop) {
    const int blocks = nblk(T.nlines, kCol), nt = threads(F.ax[2], 1);
    if (charges)
        MBPOL_LAUNCH(ev, k_spread_dft_z_r2c<true>, blocks, nt, z_bytes(F.ax[2]), s, T, w, H, F.ax[2], F.khp, stop);
    else
        MBPOL_LAUNCH(ev, k_spread_dft_z_r2c<false>, blocks, nt, z_bytes(F.ax[2]), s, T, w, H, F.ax[2], F.khp, stop);
}
void launch_spread_lines(hipStream_t s, const LineTable& T, bool charges, const double* w, double* real,
                         const KEvents& ev, const int* stop) {
    const long long blocks = (long long)nblk(T.nlines, kCol) * T.nseg;
    const size_t bytes = sizeof(double) * kColPad * (size_t)nblk(T.nz, T.nseg);  // the longest segment
    if (charges)
        MBPOL_LAUNCH(ev, k_spread_lines<true>, (unsigned)blocks, kSpreadThreads, bytes, s, T, w, real, stop);
    else
        MBPOL_LAUNCH(ev, k_spread_lines<false>, (unsigned)blocks, kSpreadThreads, bytes, s, T, w, real, stop);
}
// the front radix as a template argument
#define MBPOL_DFT_LAUNCH(kern, f, ...)                             \
    switch (f) {                                                   \
        case 2: MBPOL_LAUNCH(ev, kern<2>, __VA_ARGS__); break;     \
        case 3: MBPOL_LAUNCH(ev, kern<3>, __VA_ARGS__); break;     \
        case 4: MBPOL_LAUNCH(ev, kern<4>, __VA_ARGS__); break;     \
        default: MBPOL_LAUNCH(ev, kern<1>, __VA_ARGS__); break;    \
    }
void launch_dft_y(hipStream_t s, const PmeFft& F, double2* H, int inverse, const KEvents& ev, const int* stop) {
    const FftAxis& a = F.ax[1];
    const int nt = nblk(F.ax[2].n / 2 + 1, 8), f = a.front;
    MBPOL_DFT_LAUNCH(k_dft_y, f, F.ax[0].n * nt, threads(a, f), roots_bytes(a, f) + columns_bytes(a), s, H, nt, F.khp,
                     a, inverse, stop)
}
void launch_dft_x_conv(hipStream_t s, const PmeFft& F, double2* H, const double* influence, const KEvents& ev,
                       const int* stop) {
    const FftAxis& a = F.ax[0];
    const int nt = nblk(F.ax[2].n / 2 + 1, 8), f = a.front;
    MBPOL_DFT_LAUNCH(k_dft_x_conv, f, F.ax[1].n * nt, threads(a, f), roots_bytes(a, f) + 2 * columns_bytes(a), s, H,
                     influence, nt, F.ax[1].n, F.khp, a, stop)
}
#undef MBPOL_DFT_LAUNCH
void launch_dft_z_c2r(hipStream_t s, const PmeFft& F, const double2* H, double* real, const KEvents& ev,
                      const int* stop) {
    const int nl = F.ax[0].n * F.ax[1].n;
    const FftAxis& a = F.ax[2];
    MBPOL_LAUNCH(ev, k_dft_z_c2r, nblk(nl, kCol), threads(a, 1),
                 roots_bytes(a, 1) + 2 * sizeof(double) * kColPad * (size_t)(a.n / 2 + 1), s, H, real, nl, a, F.khp, stop);
}

}  // namespace mbpol
