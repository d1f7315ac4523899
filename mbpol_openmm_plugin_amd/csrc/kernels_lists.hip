// O-O cell lists and the stream-compacted dimer / chain-trimer lists.
//
// Set semantics follow the reference exactly, with FP64 distances computed in
// the same operation order (no contraction) so that boundary cases fall the
// same way:
//  * dimers: every pair i<j with d^2 <= rc^2 (minimum image when periodic) --
//    OpenMM's computeNeighborListVoxelHash as called at
//    platforms/reference/src/MBPolReferenceKernels.cpp:379-383;
//  * trimers: the "chain" rule of ReferenceThreeNeighborList.cpp:181-226 --
//    (i, j, k) with j in lo(i), k in lo(j), lo(i) = {j < i : d(i,j) <= rc},
//    d(i,k) never tested; a molecule whose wrapped coordinate rounds into the
//    voxel index nv is invisible to later molecules there (:86-97, :140-146),
//    which is reproduced.
// The pair passes are bound by the latency of their loads (a cell range, a member,
// its position), not by their few thousand distances a wave: so the positions are
// copied in cell order, a wave takes a molecule and lays the 27 cells' members end
// to end, and 64 candidates are in flight at once (2700 waters: dimer pass 50 us with
// 16 lanes walking range by range, 8.6 us now; lower pass of 3000 38 -> 5.2 us).  The trimer pass takes the pairs (i, j)
// of the lower lists, 8 lanes each, instead of walking all pairs of one i in turn
// (512 clusters of up to 64 waters: 2 x 310 us -> 2 x 107; 3000 waters 2 x 29 -> 2 x 6.5).
// Lists are built in two passes (count, exclusive scan, fill); the fill pass
// recomputes the same predicate, so it writes exactly `count` entries -- those
// below the list's capacity: the host learns the totals after the evaluation
// and runs it again with larger lists when one did not fit, so that no host
// wait sits between the passes.
#include <algorithm>

#include "device_common.h"
#include "kernels.h"

namespace mbpol {

#pragma clang fp contract(off)

// periodicDifference (ReferenceThreeNeighborList.cpp:14-18)
__device__ __forceinline__ double pdiff(double a, double b, double L) {
    const double diff = a - b;
    const double base = floor(diff / L + 0.5) * L;
    return diff - base;
}

// squared distance p1 -> p2 (ReferenceThreeNeighborList.cpp:21-34)
__device__ __forceinline__ double dist2(const d3& p1, const d3& p2, const d3& L, int periodic) {
    double dx, dy, dz;
    if (!periodic) {
        dx = p2.x - p1.x;
        dy = p2.y - p1.y;
        dz = p2.z - p1.z;
    } else {
        dx = pdiff(p2.x, p1.x, L.x);
        dy = pdiff(p2.y, p1.y, L.y);
        dz = pdiff(p2.z, p1.z, L.z);
    }
    return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ d3 opos(const double* pos, const int* idx, int m) { return load_d3(pos, idx[3 * m]); }

__device__ __forceinline__ int wrap_cell(int c, int n) { return c < 0 ? c + n : (c >= n ? c - n : c); }

// ---- cell binning (periodic, nc >= 3 per dimension) ----
__global__ void k_cell_count(int n, const int* __restrict__ idx, const double* __restrict__ pos, d3 L, int3 nc,
                             int* __restrict__ cell_of, int* __restrict__ cell_count) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const d3 p = opos(pos, idx, m);
    const double q[3] = {p.x - L.x * floor(p.x / L.x), p.y - L.y * floor(p.y / L.y), p.z - L.z * floor(p.z / L.z)};
    const double Ld[3] = {L.x, L.y, L.z};
    const int ncd[3] = {nc.x, nc.y, nc.z};
    int c[3];
    for (int d = 0; d < 3; ++d) {
        int v = (int)floor(q[d] * ncd[d] / Ld[d]);
        c[d] = v < 0 ? 0 : (v >= ncd[d] ? ncd[d] - 1 : v);
    }
    const int cell = (c[0] * nc.y + c[1]) * nc.z + c[2];
    cell_of[m] = cell;
    atomicAdd(&cell_count[cell], 1);
}

// members of every cell (in arbitrary order within a cell), packed: the oxygen's
// position and the molecule's index; with `phantoms` the index of a molecule in a
// phantom voxel (see phantom_voxel) is stored as -1 - index
__device__ __forceinline__ bool phantom_voxel(const d3& p, const ListGeom& g);
__global__ void k_cell_fill(int n, const int* __restrict__ idx, const double* __restrict__ pos, ListGeom g, int phantoms,
                            const int* __restrict__ cell_of, const int* __restrict__ cell_start,
                            int* __restrict__ cell_fill, double4* __restrict__ cpos) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= n) return;
    const int c = cell_of[m];
    const int slot = atomicAdd(&cell_fill[c], 1);
    const d3 p = opos(pos, idx, m);
    cpos[cell_start[c] + slot] = make_double4(p.x, p.y, p.z, (double)(phantoms && phantom_voxel(p, g) ? -1 - m : m));
}

// Lanes of one G-lane group share molecule m; these helpers give the group's
// lane bits and the bits of the lanes below this one, for ballot compaction.
template <int G>
__device__ __forceinline__ unsigned long long group_bits() {
    const int lane = threadIdx.x & 63;
    return G == 64 ? ~0ull : (((1ull << G) - 1ull) << (lane & ~(G - 1)));
}
__device__ __forceinline__ unsigned long long lanes_below() { return (1ull << (threadIdx.x & 63)) - 1ull; }

// Visit the members of the 27 cells around cell c, packed in cell order, with the
// 64 lanes of a wave: f(member, active) is called by all lanes in step, so that it
// may use wavefront ballots.  The cells along z of each (X, Y) column are
// consecutive in the cell order, so there are one or two member ranges a column,
// found by lanes 0 .. 17 together and then laid end to end.
template <typename F>
__device__ __forceinline__ void for_cell_members(int c, const int3& nc, const int* __restrict__ cell_start,
                                                 const double4* __restrict__ cpos, F&& f) {
    const int lane = threadIdx.x & 63;
    int b = 0, e = 0;
    if (lane < 18) {
        const int cz = c % nc.z, cy = (c / nc.z) % nc.y, cx = c / (nc.z * nc.y), col = lane >> 1;
        const int base = (wrap_cell(cx + col / 3 - 1, nc.x) * nc.y + wrap_cell(cy + col % 3 - 1, nc.y)) * nc.z;
        int za = cz - 1, zb = cz + 1;
        if (lane & 1) {  // the part of the column across the boundary
            if (za < 0) {
                za += nc.z;
                zb = nc.z - 1;
            } else if (zb >= nc.z) {
                za = 0;
                zb -= nc.z;
            } else {
                zb = za - 1;
            }
        } else {
            za = max(za, 0);
            zb = min(zb, nc.z - 1);
        }
        if (za <= zb) {
            b = cell_start[base + za];
            e = cell_start[base + zb + 1];
        }
    }
    int end = e - b;  // end of this lane's range among the members laid end to end
#pragma unroll
    for (int off = 1; off < 32; off <<= 1) {
        const int o = __shfl_up(end, off, 64);
        if (lane >= off) end += o;
    }
    const int shift = b - (end - (e - b));  // position of a member minus its place end to end
    const int total = __builtin_amdgcn_readlane(end, 17);
    for (int k0 = 0; k0 < total; k0 += 64) {
        const int k = k0 + lane;
        int r = 0;
#pragma unroll
        for (int s = 0; s < 17; ++s) r += k >= __builtin_amdgcn_readlane(end, s) ? 1 : 0;
        const int at = k + __shfl(shift, r, 64);
        const bool act = k < total;
        f(act ? cpos[at] : make_double4(0.0, 0.0, 0.0, 0.0), act);
    }
}

// every molecule (of the group) as a candidate of molecule m, with G lanes (PHANTOMS: those in a phantom
// voxel with the index -1 - j)
template <int G, bool PHANTOMS, typename F>
__device__ __forceinline__ void for_all(int m, int lane, int n, const int* __restrict__ idx, const double* __restrict__ pos,
                                        const ListGeom& g, F&& f) {
    const int b0 = g.gs ? g.gs[m] : 0, b1 = g.gs ? g.ge[m] : n;
    for (int b = b0; b < b1; b += G) {
        const int j = b + lane;
        const bool act = j < b1;
        const d3 p = act ? opos(pos, idx, j) : d3{0.0, 0.0, 0.0};
        f(make_double4(p.x, p.y, p.z, (double)(PHANTOMS && act && phantom_voxel(p, g) ? -1 - j : j)), act);
    }
}

constexpr int kGL = 16;  // lanes per molecule in the pair passes without cells

// ---- dimer list: count pass (pairs == nullptr) and fill pass ----
// G lanes per molecule: 64 with cells, kGL without
template <int G>
__global__ void __launch_bounds__(256) k_dimer_pass(int n, const int* __restrict__ idx, const double* __restrict__ pos,
                                                    ListGeom g, const int* __restrict__ cell_of,
                                                    const int* __restrict__ cell_start, const double4* __restrict__ cpos,
                                                    long long* __restrict__ count, const long long* __restrict__ offset,
                                                    int2* __restrict__ pairs, long long cap) {
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) / G, lane = threadIdx.x % G;
    if (i >= n) return;  // uniform over the group
    const d3 pi = opos(pos, idx, i);
    const double rc2 = g.rc * g.rc;
    const unsigned long long gb = group_bits<G>(), below = lanes_below();
    long long c = 0;
    const long long o = offset ? offset[i] : 0;
    auto consider = [&](const double4& q, bool act) {
        const int j = (int)q.w;
        const bool ok = act && j > i && dist2(pi, d3{q.x, q.y, q.z}, g.L, g.periodic) <= rc2;
        const unsigned long long bits = __ballot(ok) & gb;
        if (ok && pairs) {
            const long long t = o + c + __popcll(bits & below);
            if (t < cap) pairs[t] = make_int2(i, j);  // beyond the capacity: counted, reported, not written
        }
        c += __popcll(bits);
    };
    if constexpr (G == 64)
        for_cell_members(__builtin_amdgcn_readfirstlane(cell_of[i]), g.nc, cell_start, cpos, consider);
    else
        for_all<G, false>(i, lane, n, idx, pos, g, consider);
    if (count && lane == 0) {
        count[i] = c;
        if (i == 0) count[n] = 0;
    }
}

// ---- chain trimer list ----
// voxel index of the reference's ThreeVoxelHash (ReferenceThreeNeighborList.cpp:86-97); a molecule whose
// index equals nv in some dimension is never found from a later molecule
__device__ __forceinline__ bool phantom_voxel(const d3& p, const ListGeom& g) {
    if (!g.periodic) return false;
    const double Ld[3] = {g.L.x, g.L.y, g.L.z}, pd[3] = {p.x, p.y, p.z};
    for (int d = 0; d < 3; ++d) {
        const double edge = Ld[d] / floor(Ld[d] / g.rc);
        const int nv = (int)floor(Ld[d] / edge + 0.5);
        const double q = pd[d] - Ld[d] * floor(pd[d] / Ld[d]);
        if ((int)floor(q / edge) >= nv) return true;
    }
    return false;
}

// lo(i) = {j < i : d(i,j) <= rc, j not in a phantom voxel}: count pass (lower == nullptr) and fill pass
// (lower[t] = (i, j))
template <int G>
__global__ void __launch_bounds__(256) k_lower_pass(int n, const int* __restrict__ idx, const double* __restrict__ pos,
                                                    ListGeom g, const int* __restrict__ cell_of,
                                                    const int* __restrict__ cell_start, const double4* __restrict__ cpos,
                                                    int* __restrict__ count, const int* __restrict__ offset,
                                                    int2* __restrict__ lower, int cap) {
    const int i = (blockIdx.x * blockDim.x + threadIdx.x) / G, lane = threadIdx.x % G;
    if (i >= n) return;
    const d3 pi = opos(pos, idx, i);
    const double rc2 = g.rc * g.rc;
    const unsigned long long gb = group_bits<G>(), below = lanes_below();
    int c = 0;
    const int o = offset ? offset[i] : 0;
    auto consider = [&](const double4& q, bool act) {
        const int j = (int)q.w;  // negative in a phantom voxel
        const bool ok = act && j >= 0 && j < i && dist2(pi, d3{q.x, q.y, q.z}, g.L, g.periodic) <= rc2;
        const unsigned long long bits = __ballot(ok) & gb;
        if (ok && lower) {
            const int t = o + c + __popcll(bits & below);
            if (t < cap) lower[t] = make_int2(i, j);
        }
        c += __popcll(bits);
    };
    if constexpr (G == 64)
        for_cell_members(__builtin_amdgcn_readfirstlane(cell_of[i]), g.nc, cell_start, cpos, consider);
    else
        for_all<G, true>(i, lane, n, idx, pos, g, consider);
    if (count && lane == 0) {
        count[i] = c;
        if (i == 0) count[n] = 0;
    }
}

// O-O distances of a triplet after the reference's imaging (every O imaged to Oa,
// MBPolReferenceTwoBodyForce.cpp:78-109), in Angstrom.
__device__ __forceinline__ void trimer_oo(const d3& a, d3 b, d3 c, const ListGeom& g, double& rab, double& rac, double& rbc) {
    if (g.periodic) {
        b = image_to(a, b, g.L);
        c = image_to(a, c, g.L);
    }
    auto d = [](const d3& u, const d3& v) {
        const double x = (u.x - v.x) * 10., y = (u.y - v.y) * 10., z = (u.z - v.z) * 10.;
        return sqrt(x * x + y * y + z * z);
    };
    rab = d(a, b);
    rac = d(a, c);
    rbc = d(b, c);
}

// A triplet contributes nothing when an O-O distance is below 2 A
// (MBPolReferenceThreeBodyForce.cpp:165-166) or when fewer than two of the
// three switches are non-zero (the switch is 0 for r >= 4.5 A, :103-120).
__device__ __forceinline__ bool trimer_active(const d3& a, const d3& b, const d3& c, const ListGeom& g) {
    double rab, rac, rbc;
    trimer_oo(a, b, c, g, rab, rac, rbc);
    if (rab < 2 || rac < 2 || rbc < 2) return false;
    const double rf = mbpol_params::th_r3f;
    const int on = (rab < rf) + (rac < rf) + (rbc < rf);
    return on >= 2;
}

constexpr int kGT = 8;  // lanes per pair in the trimer pass

// trimers (i, j, k) with (i, j) in the lower lists and k in lo(j): the lanes of a
// pair's group take its k, compacting the active ones by ballot.  count and offset
// are per pair; the pairs are in list order, so the trimers of i are too.
__global__ void __launch_bounds__(256) k_trimer_pass(int n, const int* __restrict__ idx, const double* __restrict__ pos,
                                                     ListGeom g, const int* __restrict__ lo_start,
                                                     const int2* __restrict__ lower, int full_list,
                                                     long long* __restrict__ count, const long long* __restrict__ offset,
                                                     int* __restrict__ trip, int lower_cap, long long cap) {
    const int lane = threadIdx.x % kGT, nl = lo_start[n];
    const unsigned long long gb = group_bits<kGT>(), below = lanes_below();
    const long long step = (long long)gridDim.x * blockDim.x / kGT;
    for (long long a = ((long long)blockIdx.x * blockDim.x + threadIdx.x) / kGT; a <= lower_cap;
         a += step) {  // uniform over the group
        // past the list's end, or an incomplete lower list (it overflowed its capacity):
        // nothing to read; the evaluation is then run again with a larger one
        if (a >= nl || nl > lower_cap) {
            if (count && lane == 0) count[a] = 0;
            continue;
        }
        const int2 ij = lower[a];
        const d3 pi = opos(pos, idx, ij.x), pj = opos(pos, idx, ij.y);
        long long c = 0;
        const long long o = offset ? offset[a] : 0;
        const int e = lo_start[ij.y + 1];
        for (int b = lo_start[ij.y]; b < e; b += kGT) {
            const bool act = b + lane < e;
            const int k = act ? lower[b + lane].y : 0;
            const bool ok = act && (full_list || trimer_active(pi, pj, opos(pos, idx, k), g));
            const unsigned long long bits = __ballot(ok) & gb;
            if (ok && trip) {
                const long long t = o + c + __popcll(bits & below);
                if (t < cap) {
                    trip[3 * t] = ij.x;
                    trip[3 * t + 1] = ij.y;
                    trip[3 * t + 2] = k;
                }
            }
            c += __popcll(bits);
        }
        if (count && lane == 0) count[a] = c;
    }
}

// out[i] = off[start[i]], i <= n: offsets per molecule from those per lower pair
__global__ void k_offsets_of(int n, const int* __restrict__ start, int limit, const long long* __restrict__ off,
                             long long* __restrict__ out) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i <= n) out[i] = off[min(start[i], limit)];
}

}  // namespace mbpol

namespace mbpol {
static inline int nblk(long long n, int b) { return (int)((n + b - 1) / b); }
void launch_cell_count(hipStream_t s, int n, const int* idx, const double* pos, d3 L, int3 nc, int* cell_of,
                       int* cell_count) {
    if (n > 0) hipLaunchKernelGGL(k_cell_count, nblk(n, 256), 256, 0, s, n, idx, pos, L, nc, cell_of, cell_count);
}
void launch_cell_fill(hipStream_t s, int n, const int* idx, const double* pos, const ListGeom& g, int phantoms,
                      const int* cell_of, const int* cell_start, int* cell_fill, double4* cpos) {
    if (n > 0)
        hipLaunchKernelGGL(k_cell_fill, nblk(n, 256), 256, 0, s, n, idx, pos, g, phantoms, cell_of, cell_start, cell_fill,
                           cpos);
}
// a wave per molecule with cells, kGL lanes without
#define MBPOL_PAIR_PASS(kern, ...)                                                                      \
    do {                                                                                                \
        if (n <= 0) return;                                                                             \
        if (g.use_cells)                                                                                \
            hipLaunchKernelGGL(kern<64>, nblk((long long)n * 64, 256), 256, 0, s, __VA_ARGS__);         \
        else                                                                                            \
            hipLaunchKernelGGL(kern<kGL>, nblk((long long)n * kGL, 256), 256, 0, s, __VA_ARGS__);       \
    } while (0)
void launch_dimer_pass(hipStream_t s, int n, const int* idx, const double* pos, ListGeom g, const int* cell_of,
                       const int* cell_start, const double4* cpos, long long* count, const long long* offset,
                       int2* pairs, long long cap) {
    MBPOL_PAIR_PASS(k_dimer_pass, n, idx, pos, g, cell_of, cell_start, cpos, count, offset, pairs, cap);
}
void launch_lower_pass(hipStream_t s, int n, const int* idx, const double* pos, ListGeom g, const int* cell_of,
                       const int* cell_start, const double4* cpos, int* count, const int* offset, int2* lower,
                       int cap) {
    MBPOL_PAIR_PASS(k_lower_pass, n, idx, pos, g, cell_of, cell_start, cpos, count, offset, lower, cap);
}
#undef MBPOL_PAIR_PASS
void launch_trimer_pass(hipStream_t s, int n, const int* idx, const double* pos, ListGeom g, const int* lo_start,
                        const int2* lower, int full_list, long long* count, const long long* offset, int* trip,
                        int lower_cap, long long cap) {
    // at most 2^17 blocks, whose groups stride over longer lists (from 2^29 pairs on a thread's index would not fit
    // the 32 bits of blockIdx.x * blockDim.x)
    const int blocks = std::min(nblk((lower_cap + 1LL) * kGT, 256), 1 << 17);
    if (n > 0)
        hipLaunchKernelGGL(k_trimer_pass, blocks, 256, 0, s, n, idx, pos, g, lo_start, lower, full_list, count, offset,
                           trip, lower_cap, cap);
}
void launch_offsets_of(hipStream_t s, int n, const int* start, int limit, const long long* off, long long* out) {
    if (n > 0) hipLaunchKernelGGL(k_offsets_of, nblk(n + 1, 256), 256, 0, s, n, start, limit, off, out);
}
}  // namespace mbpol
