// PME grid transforms (kernels_fft.hip).
#pragma once
#include "kernels.h"

namespace mbpol {

constexpr int kFftThreads = 128;  // threads per workgroup of the grid transforms

// One axis of the grid: length n = fac[0] * ... * fac[nfac-1] (radices 2, 3,
// 4, 5, 7, 11, 13); stage s has ns[s] = fac[0] ... fac[s-1], nb[s] = n / fac[s]
// butterflies and twiddle step n / (ns[s] fac[s]).  2^lgP threads work on one
// line (lgP <= 7); tw[t] = exp(-2 pi i t / n) in device memory.
struct FftAxis {
    int n;
    int nfac;
    int fac[12], ns[12], nb[12], step[12];
    float inv_ns[12];
    int lgP;
    int inplace;  // every stage has at most 2^lgP butterflies: stages run in place (one LDS buffer)
    const double2* tw;
    int dense;  // the axis runs as dense products (kernels_dft.hip), after a front stage of radix `front`
    int front;
};

struct PmeFft {
    FftAxis ax[3];  // x, y, z
    int khp;        // padded kz row length of the half spectrum (>= n_z / 2 + 1, multiple of 8)
};

// longest axis the LDS transforms take: one line per workgroup, two buffers in 32 KB
constexpr int kFftMaxLength = 1024;
// real grid -> half spectrum H -> (x pass) times influence -> real grid, as five passes:
// z_r2c, y (forward), x_conv, y (inverse), z_c2r
// stop: when non-null and *stop != 0 at launch, the pass does nothing (a dipole solve that has converged)
void launch_fft_z_r2c(hipStream_t s, const PmeFft& F, const double* real, double2* H, const KEvents& ev,
                      const int* stop = nullptr);
// The spreading table by grid line (kernels_elec.hip): rows 0 .. nseg nlines - 1 the polarisable sites of the
// lines' segments, line by line, rows nseg nlines .. 2 nseg nlines - 1 the other charged sites
struct LineTable {
    int nlines, nz;  // lines (x, y), points of a line
    int nseg;        // segments a line's points are cut into
    const int* start;
    const int2* sz;      // site, first z
    const double* coef;  // 3 per entry
    const double* sptab; // z splines: sptab[30 site + 20 ..]
    double scale_z;      // K_z / L_z
};
// first point of segment s of nz points in nseg segments whose lengths differ by at most one
__host__ __device__ inline int segment_start(int s, int nz, int nseg) { return (int)((long long)s * nz / nseg); }
// the segment that point z lies in: the last one that starts at or before it
__host__ __device__ inline int segment_of(int z, int nz, int nseg) {
    return (int)(((long long)(z + 1) * nseg - 1) / nz);
}
// Segments of a line of nz points: none shorter than 64 points (a site's 5 then
// reach into the next one at most), none longer than 127 (17 KB of LDS).
constexpr int kSegmentPoints = 64;
inline int spread_segments(int nz) { return nz < 2 * kSegmentPoints ? 1 : nz / kSegmentPoints; }
// spreads charges (w = q) or dipoles (w = mu) onto the real grid, or straight into the forward z pass (dense z only)
void launch_spread_lines(hipStream_t s, const LineTable& T, bool charges, const double* w, double* real,
                         const KEvents& ev, const int* stop = nullptr);
void launch_spread_dft_z_r2c(hipStream_t s, const PmeFft& F, const LineTable& T, bool charges, const double* w,
                             double2* H, const KEvents& ev, const int* stop = nullptr);
void launch_fft_y(hipStream_t s, const PmeFft& F, double2* H, int inverse, const KEvents& ev,
                  const int* stop = nullptr);
void launch_fft_x_conv(hipStream_t s, const PmeFft& F, double2* H, const double* influence, const KEvents& ev,
                       const int* stop = nullptr);
void launch_fft_z_c2r(hipStream_t s, const PmeFft& F, const double2* H, double* real, const KEvents& ev,
                      const int* stop = nullptr);
// the same passes as dense products on the FP64 matrix cores, for lengths up to kDftMaxLength (kernels_dft.hip)
constexpr int kDftMaxLength = 512;
// lets their kernels use more than 64 KB of LDS on the current device: once before their launches
hipError_t dft_allow_lds();
void launch_dft_z_r2c(hipStream_t s, const PmeFft& F, const double* real, double2* H, const KEvents& ev,
                      const int* stop);
void launch_dft_y(hipStream_t s, const PmeFft& F, double2* H, int inverse, const KEvents& ev, const int* stop);
void launch_dft_x_conv(hipStream_t s, const PmeFft& F, double2* H, const double* influence, const KEvents& ev,
                       const int* stop);
void launch_dft_z_c2r(hipStream_t s, const PmeFft& F, const double2* H, double* real, const KEvents& ev,
                      const int* stop);
// z and y passes of one direction as one kernel per x plane (plane in LDS);
// fft_plane_ok: the plane fits in LDS and every stage has at most one butterfly per thread
bool fft_plane_ok(const PmeFft& F);
void launch_fft_plane_fwd(hipStream_t s, const PmeFft& F, const double* real, double2* H, const KEvents& ev,
                          const int* stop = nullptr);
void launch_fft_plane_inv(hipStream_t s, const PmeFft& F, const double2* H, double* real, const KEvents& ev,
                          const int* stop = nullptr);

}  // namespace mbpol
