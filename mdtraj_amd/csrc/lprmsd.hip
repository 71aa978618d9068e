// LP-RMSD (gfx950): the RMSD minimised over rotations and over relabellings
// of atoms inside permute groups (rmsd/_lprmsd.pyx:72-228).  Per target frame:
//   (1) gather the selection and centre it (FP64 centroid, float coordinates
//       rounded once);
//   (2) if some selected atoms are in no group ("distinguishable"), fit them
//       alone, each set centred on its own centroid, and rotate the whole
//       centred selection by that rotation, x' = x R1 in float as
//       rot_atom_major;
//   (3) for each group, the assignment of reference atoms (rows) to target
//       atoms (columns) minimising the summed squared distances, the costs
//       formed as euclidean_permutation.cpp:28-35 does (float differences
//       and squares, summed in double), solved exactly by the Hungarian
//       method in its shortest-augmenting-path form (row potentials u,
//       column potentials v, one Dijkstra-like search per row);
//   (4) the QCP RMSD of the relabelled selection against the reference; with
//       superpose, the frame (every atom, centred) is rotated by R1 R2.
// Two waves per frame.  Most rows of a group need no search: every row's
// nearest column is found first, on the matrix cores and by both waves, and
// rows whose nearest columns differ are matched at once.  The first wave does
// all else (and groups of up to 32 atoms alone); the columns of a search are spread over its lanes, and the
// search's minimum is a wave reduction (ties to the lowest column).  The
// group's reference coordinates, potentials and search state sit in LDS (sized
// to keep eight frames per CU for groups of a few hundred atoms).
// What bounds it (20,000 frames x 400 atoms, one group of 300; 8.05 ms a call
// when every row was searched for, 0.60 ms now): the latency of a frame's
// serial steps, about 119,000 cycles (gather 17, fit 16, nearest columns 41,
// two searches of two passes 25, the rest 20 thousand) with eight frames
// resident per CU.  That is with atoms near their reference places; what a
// diffused liquid costs is the searches themselves, which the start hardly
// shortens (4,000 frames x (100 + 300), every row searched for / now: 0.02 nm of
// noise 1.63 / 0.12 ms, 0.1 nm 2.05 / 0.66, 0.2 nm 12.7 / 10.1, independent places
// 26.3 / 23.7).
#include <type_traits>

#include "common.h"

namespace hr {
namespace {

constexpr int kLpBlock = kWave;
constexpr int kLpFrameBlock = 2 * kWave;
constexpr int kLpBatch = 5;  // atoms or columns a lane handles at a time
constexpr size_t kLpLdsMax = 64 * 1024;

size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

__host__ __device__ inline size_t lp_lds_bytes(int n_sel, int kmax) {
    const size_t k1 = (size_t)kmax + 1;
    return 3 * 8 * k1      // u, v, minv
           + 2 * 4 * k1    // p, way
           + 4 * (size_t)kmax  // the group's atoms
           + 12 * (size_t)kmax  // the group's reference coordinates
           + 12 * (size_t)n_sel  // target selection, x, y, z
           + k1;           // used
}

// What only the lead wave touches: a wave's LDS accesses complete in program
// order, so ordering them needs only a wavefront fence that keeps the compiler
// from moving them, not a workgroup barrier (which would also wait for memory).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Sum of the wave, in every lane: rows of 16 by DPP moves, then two lane
// exchanges (six exchanges of both halves of a double cost about 800 cycles of
// latency, and a frame takes some thirty sums).
__device__ __forceinline__ double lp_sum(double v) {
    v = row16_sum(v);
    v += __shfl_xor(v, 16, kWave);
    v += __shfl_xor(v, 32, kWave);
    return v;
}

// Index arrays live on the device, where the host cannot check them: every
// index is clamped into its array, so malformed input gives wrong numbers,
// never an access outside the buffers.
__device__ __forceinline__ int clamp_index(int i, int n) { return (unsigned)i < (unsigned)n ? i : 0; }

__device__ __forceinline__ int ref_atom(const int* idx, const int* dis, int part, int a, int n_sel,
                                        int n_atoms) {
    const int s = part == 0 ? a : clamp_index(dis[a], n_sel);
    return clamp_index(idx[s], n_atoms);
}

// Prepared reference: the selection centred (x, y, z planes of n_sel
// floats), the distinguishable subset centred on its own centroid (planes of
// n_dis), and their traces.
__global__ __launch_bounds__(kLpBlock) void lp_ref_kernel(const float* __restrict__ ref,
                                                          int n_atoms,
                                                          const int* __restrict__ idx, int n_sel,
                                                          const int* __restrict__ dis, int n_dis,
                                                          float* __restrict__ rsel,
                                                          float* __restrict__ rdis,
                                                          double* __restrict__ traces) {
    const int lane = threadIdx.x;
    for (int part = 0; part < 2; ++part) {
        const int n = part == 0 ? n_sel : n_dis;
        if (n == 0) {
            if (lane == 0) traces[part] = 0.0;
            continue;
        }
        float* out = part == 0 ? rsel : rdis;
        double s[3] = {0.0, 0.0, 0.0};
        for (int a = lane; a < n; a += kWave) {
            const int at = ref_atom(idx, dis, part, a, n_sel, n_atoms);
#pragma unroll
            for (int c = 0; c < 3; ++c) s[c] += (double)ref[3LL * at + c];
        }
        double mu[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) mu[c] = wave_sum(s[c]) / n;
        double g = 0.0;
        for (int a = lane; a < n; a += kWave) {
            const int at = ref_atom(idx, dis, part, a, n_sel, n_atoms);
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const float v = (float)((double)ref[3LL * at + c] - mu[c]);
                out[(size_t)c * n + a] = v;
                g += (double)v * v;
            }
        }
        g = wave_sum(g);
        if (lane == 0) traces[part] = g;
    }
}

struct LpArgs {
    float* xyz;  // (n_frames, n_atoms, 3); rotated in place with superpose
    long long n_frames;
    int n_atoms;
    const int* idx;
    int n_sel;
    const int* dis;  // selection positions of the distinguishable atoms
    int n_dis;
    const int* group_atoms;  // selection positions, group g at [off[g], off[g + 1])
    const int* group_off;
    int n_groups;
    int kmax;
    const float* rsel;  // prepared reference (lp_ref_kernel)
    const float* rdis;
    const double* traces;
    int superpose;
    float* out;
};

// (value, column) pairs ordered by value, then by the lower column; a NaN
// never beats a number, and any valid column beats none (INT_MAX).  The
// order is total on the pairs that occur, so any reduction tree gives the
// same minimum.
__device__ __forceinline__ void take_min(double& best, int& col, double ob, int oc) {
    if (ob < best || (!(ob > best) && oc < col)) {
        best = ob;
        col = oc;
    }
}

template <int kCtrl>
__device__ __forceinline__ void argmin_dpp(double& best, int& col) {
    const double ob = dpp_move<kCtrl>(best);
    const int oc = __builtin_amdgcn_mov_dpp(col, kCtrl, 0xF, 0xF, false);
    take_min(best, col, ob, oc);
}

// Minimum of the wave, in every lane: within rows of 16 lanes by DPP moves
// (xor 1, xor 2, half mirror, mirror: a few cycles each), then across rows
// by two lane exchanges.
__device__ __forceinline__ void wave_argmin(double& best, int& col) {
    argmin_dpp<0xB1>(best, col);
    argmin_dpp<0x4E>(best, col);
    argmin_dpp<0x141>(best, col);
    argmin_dpp<0x140>(best, col);
#pragma unroll
    for (int m = 16; m <= 32; m <<= 1) take_min(best, col, __shfl_xor(best, m, kWave),
                                                __shfl_xor(col, m, kWave));
}

// euclidean_permutation.cpp: squares of float differences, summed in double
__device__ __forceinline__ double lp_cost(float dx, float dy, float dz) {
    return (double)__fmul_rn(dx, dx) + (double)__fmul_rn(dy, dy) + (double)__fmul_rn(dz, dz);
}

// The two least of two disjoint sets, and the place of the least.
__device__ __forceinline__ void lp_merge(float& best, float& second, int& arg, float o_best,
                                         float o_second, int o_arg) {
    second = fminf(fmaxf(best, o_best), fminf(second, o_second));
    arg = o_best < best ? o_arg : arg;
    best = fminf(best, o_best);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Start of a group's assignment: u[i] = the least cost of row i (v = 0, so
// the duals are feasible) and col[i] its column, rows i = 1 .. k.  All k^2
// pairs are compared once, on the matrix cores: |b|^2 - 2 a.b, the squared
// distance less the row's own |a|^2, is a product over four terms, two
// v_mfma_f32_32x32x2_f32 for 32 targets (rows of the tile) by 32 reference
// atoms (its columns, one per lane of each half wave), and what is left for
// the vector units is three instructions a pair: the place into the value's
// last bits, the least and the second least.  (Costing each pair in float
// there, ten instructions a pair, measured 759 us a call of 20,000 frames with
// 300 interchangeable atoms; this, 601 us.)  A row whose two least values are
// further apart than rounding can move them takes the double cost of the
// nearer target; one that is closer (or not finite) is scanned again in double
// by the whole wave, ties to the lowest column.  With m the largest |a|^2 or
// |b|^2 a value (below 3 m) is off by 3 m 2^-19 for its last four bits, by
// 1.2 m 2^-20 for the product's roundings, and the double cost, of float
// squares, by m 2^-20: two values by 16.4 m 2^-20 together; tol is twice that.
// That holds while nothing overflows or goes below float's normal numbers, and
// the places that fill up the last tile (1e30, less 2 m at most) are farther
// than any target while 3 m is below 1e30 - 2 m: rows with m outside 2^-96 ..
// 2^96 (8e28) are all scanned in double.
// Returns whether every row of the lane has a finite least cost.
//   q   the group's target atoms as x, z, y, |b|^2, 16-byte aligned
//   biggest   the largest |b|^2
//   first   0 or 32: the wave's first row
__device__ __forceinline__ bool lp_row_minima(const float* q, int k, const float* grx,
                                              const float* gry, const float* grz, float biggest,
                                              double* u, int* col, int lane, int first) {
    bool finite = true;
    // -inf, unknown to the compiler: as a minimum it would first quiet both
    // operands, an instruction each
    float lowest = -__builtin_huge_valf();
    asm("" : "+v"(lowest));
    const int half = lane >> 5, in = lane & 31;
    for (int r0 = first; r0 < k; r0 += 64) {
        const int r = min(r0 + in, k - 1);
        const float x = grx[r], y = gry[r], z = grz[r];
        const float aa = fmaf(x, x, fmaf(y, y, z * z));
        const float b0 = -2.0f * (half ? y : x), b1 = half ? 1.0f : -2.0f * z;
        // two tiles at a time: their products and the two chains of least
        // values overlap
        float best[2], second[2];
        int tile[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            best[c] = second[c] = __builtin_huge_valf();
            tile[c] = 0;
        }
        for (int t = 0; t < k; t += 64) {
            f32x16 d[2] = {};
            float2 a[2];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                a[c] = *reinterpret_cast<const float2*>(q + 4 * min(t + 32 * c + in, k - 1) +
                                                        2 * half);
                // targets past the group are farther than any
                if (half && t + 32 * c + in >= k) a[c].y = 1e30f;
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) d[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c].x, b0, d[c], 0, 0, 0);
#pragma unroll
            for (int c = 0; c < 2; ++c) d[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[c].y, b1, d[c], 0, 0, 0);
            const float before[2] = {best[0], best[1]};
#pragma unroll
            for (int e = 0; e < 16; ++e) {
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    // the place in the tile rides in the value's last four bits
                    const float v = __int_as_float((__float_as_int(d[c][e]) & ~15) | e);
                    second[c] = __builtin_amdgcn_fmed3f(v, best[c], second[c]);
                    best[c] = __builtin_amdgcn_fmed3f(v, best[c], lowest);  // the lesser
                }
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) tile[c] = best[c] < before[c] ? t + 32 * c : tile[c];
        }
        int args[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int e = __float_as_int(best[c]) & 15;
            args[c] = tile[c] + 8 * (e / 4) + 4 * half + e % 4;
        }
        lp_merge(best[0], second[0], args[0], best[1], second[1], args[1]);
        // the other half wave's targets of the same row
        lp_merge(best[0], second[0], args[0], __shfl_xor(best[0], 32, kWave),
                 __shfl_xor(second[0], 32, kWave), __shfl_xor(args[0], 32, kWave));
        const bool mine = half == 0 && r0 + in < k;
        const float* near = q + 4 * min(args[0], k - 1);
        double least = lp_cost(x - near[0], y - near[2], z - near[1]);
        const float m = fmaxf(aa, biggest);
        const float tol = m > 0x1p-96f && m < 0x1p96f ? 0x1p-15f * m : __builtin_huge_valf();
        // the close rows, one by one, the columns spread over the lanes
        for (unsigned long long close = __ballot(mine && !(second[0] > best[0] + tol)); close;
             close &= close - 1) {
            const int l = __ffsll((long long)close) - 1;
            const float rx = __shfl(x, l, kWave), ry = __shfl(y, l, kWave), rz = __shfl(z, l, kWave);
            double c_best = __builtin_huge_val();
            int c_col = INT_MAX;
            for (int m = lane; m < k; m += kWave) {
                const double c = lp_cost(rx - q[4 * m], ry - q[4 * m + 2], rz - q[4 * m + 1]);
                if (c < c_best) {
                    c_best = c;
                    c_col = m;
                }
            }
            wave_argmin(c_best, c_col);
            if (lane == l) {
                least = c_best;
                args[0] = c_col;
            }
        }
        if (mine) {
            finite = finite && least < __builtin_huge_val();
            u[r + 1] = least;
            col[r + 1] = args[0] + 1;
        }
    }
    return finite;
}

// Two waves a frame: the second only shares the row minima.
__global__ __launch_bounds__(kLpFrameBlock, 4) void lp_frame_kernel(LpArgs A) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int k1 = A.kmax + 1;
    double* u = reinterpret_cast<double*>(lds);
    double* v = u + k1;
    double* minv = v + k1;
    int* p = reinterpret_cast<int*>(minv + k1);
    int* way = p + k1;
    int* gat = way + k1;
    float* grx = reinterpret_cast<float*>(gat + A.kmax);  // the group's reference coordinates
    float* gry = grx + A.kmax;
    float* grz = gry + A.kmax;
    float* tx = grz + A.kmax;
    float* ty = tx + A.n_sel;
    float* tz = ty + A.n_sel;
    unsigned char* used = reinterpret_cast<unsigned char*>(tz + A.n_sel);

    const int lane = threadIdx.x & (kWave - 1);
    const bool lead = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave) == 0;
    __shared__ int s_finite;
    __shared__ float s_biggest;
    __shared__ float s_rot[9];  // R1
    __shared__ double s_tg;     // the target selection's trace
    const long long f = workgroup_index();
    if (f >= A.n_frames) return;
    float* fr = A.xyz + f * 3LL * A.n_atoms;
    const int n = A.n_sel;
    const float* rx = A.rsel;
    const float* ry = rx + n;
    const float* rz = ry + n;

    double M2[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (lead) {
        float R1[9] = {1.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f, 0.f, 1.f};
        double tg = 0.0;
        // (1) gather and centre the selection
        double s[3] = {0.0, 0.0, 0.0};
        // loads of kLpBatch atoms a lane at a time, so that their latencies overlap
        for (int a0 = lane; a0 < n; a0 += kLpBatch * kWave) {
            long long at[kLpBatch];
            float x[kLpBatch], y[kLpBatch], z[kLpBatch];
#pragma unroll
            for (int t = 0; t < kLpBatch; ++t)
                at[t] = 3LL * clamp_index(A.idx[min(a0 + t * kWave, n - 1)], A.n_atoms);
#pragma unroll
            for (int t = 0; t < kLpBatch; ++t) {
                x[t] = fr[at[t]];
                y[t] = fr[at[t] + 1];
                z[t] = fr[at[t] + 2];
            }
#pragma unroll
            for (int t = 0; t < kLpBatch; ++t) {
                const int a = a0 + t * kWave;
                if (a < n) {
                    tx[a] = x[t];
                    ty[a] = y[t];
                    tz[a] = z[t];
                    s[0] += x[t];
                    s[1] += y[t];
                    s[2] += z[t];
                }
            }
        }
        double mu[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) mu[c] = lp_sum(s[c]) / n;
        for (int a = lane; a < n; a += kWave) {
            const float x = (float)((double)tx[a] - mu[0]);
            const float y = (float)((double)ty[a] - mu[1]);
            const float z = (float)((double)tz[a] - mu[2]);
            tx[a] = x;
            ty[a] = y;
            tz[a] = z;
            tg += (double)x * x + (double)y * y + (double)z * z;
        }
        tg = lp_sum(tg);
        wave_sync();

        // (2) fit on the distinguishable atoms
        if (A.n_dis > 0) {
            const int nd = A.n_dis;
            double d[3] = {0.0, 0.0, 0.0};
            for (int k = lane; k < nd; k += kWave) {
                const int a = clamp_index(A.dis[k], n);
                d[0] += tx[a];
                d[1] += ty[a];
                d[2] += tz[a];
            }
            double dm[3];
#pragma unroll
            for (int c = 0; c < 3; ++c) dm[c] = lp_sum(d[c]) / nd;
            double M[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0}, ga = 0.0;
            const float* qx = A.rdis;
            const float* qy = qx + nd;
            const float* qz = qy + nd;
            for (int k = lane; k < nd; k += kWave) {
                const int a = clamp_index(A.dis[k], n);
                const double t[3] = {tx[a] - dm[0], ty[a] - dm[1], tz[a] - dm[2]};
                const double r[3] = {qx[k], qy[k], qz[k]};
#pragma unroll
                for (int i = 0; i < 3; ++i) {
#pragma unroll
                    for (int j = 0; j < 3; ++j) M[3 * i + j] = fma(t[i], r[j], M[3 * i + j]);
                    ga = fma(t[i], t[i], ga);
                }
            }
#pragma unroll
            for (int e = 0; e < 9; ++e) M[e] = lp_sum(M[e]);
            ga = lp_sum(ga);
            double R[9];
            qcp_solve<true>(M, 0.5 * (ga + A.traces[1]), R);
#pragma unroll
            for (int e = 0; e < 9; ++e) R1[e] = (float)R[e];
            for (int a = lane; a < n; a += kWave) {
                const float x = tx[a], y = ty[a], z = tz[a];
                tx[a] = x * R1[0] + y * R1[3] + z * R1[6];
                ty[a] = x * R1[1] + y * R1[4] + z * R1[7];
                tz[a] = x * R1[2] + y * R1[5] + z * R1[8];
            }
            wave_sync();
        }

        if (lane == 0) {
            s_tg = tg;
#pragma unroll
            for (int e = 0; e < 9; ++e) s_rot[e] = R1[e];
        }
        wave_sync();  // read by every lane below, with no group in between where all are empty
    }

    // (3) the assignment inside each group
    for (int g = 0; g < A.n_groups; ++g) {
        const int g0 = A.group_off[g];
        const int k = A.group_off[g + 1] - g0;
        if (k <= 0) continue;
        if (k > A.kmax) {  // larger than the LDS was sized for: no result
            if (lead && lane == 0) A.out[f] = __builtin_nanf("");
            return;
        }
        if (k == 1) {  // one atom keeps its label (100 such groups: 1,600 us a call, now 240)
            if (threadIdx.x == 0) {
                const int a = clamp_index(A.group_atoms[g0], n);
                const double t[3] = {tx[a], ty[a], tz[a]};
                const double r[3] = {rx[a], ry[a], rz[a]};
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) M2[3 * i + j] = fma(t[i], r[j], M2[3 * i + j]);
            }
            continue;
        }
        // The second wave's rows start at the 33rd: smaller groups are the first
        // wave's alone, without workgroup barriers (10,000 frames of 50 groups of
        // two: 827 us with them, 626 without; diffused 1,120 / 826).
        if (!lead && k <= kWave / 2) continue;
        float* q = reinterpret_cast<float*>(minv);
        int* col = reinterpret_cast<int*>(v);
        auto sync = [&] {  // of the waves that share the group
            if (k > kWave / 2)
                __syncthreads();
            else
                wave_sync();
        };
        // the group's target atoms where minv, p and way will be (16 k1 bytes,
        // after two arrays of 8 k1), the rows' columns where v will be
        if (lead) {
            float biggest = 0.0f;
            for (int b0 = lane; b0 < k; b0 += kLpBatch * kWave) {
                int at[kLpBatch];
                float x[kLpBatch], y[kLpBatch], z[kLpBatch];
#pragma unroll
                for (int t = 0; t < kLpBatch; ++t)
                    at[t] = clamp_index(A.group_atoms[g0 + min(b0 + t * kWave, k - 1)], n);
#pragma unroll
                for (int t = 0; t < kLpBatch; ++t) {
                    x[t] = rx[at[t]];
                    y[t] = ry[at[t]];
                    z[t] = rz[at[t]];
                }
#pragma unroll
                for (int t = 0; t < kLpBatch; ++t) {
                    const int j = b0 + t * kWave, a = at[t];
                    if (j < k) {
                        const float bb = fmaf(tx[a], tx[a], fmaf(ty[a], ty[a], tz[a] * tz[a]));
                        *reinterpret_cast<float4*>(q + 4 * j) = make_float4(tx[a], tz[a], ty[a], bb);
                        biggest = fmaxf(biggest, bb);
                        gat[j] = a;
                        grx[j] = x[t];
                        gry[j] = y[t];
                        grz[j] = z[t];
                    }
                }
            }
#pragma unroll
            for (int m = 1; m < kWave; m <<= 1) biggest = fmaxf(biggest, __shfl_xor(biggest, m, kWave));
            if (lane == 0) {
                s_finite = 1;
                s_biggest = biggest;
            }
        }
        sync();
        // Greedy start: every row's least cost as its dual, and the row itself
        // in that column unless a lower row is there.  Rows left over (two
        // reference atoms nearest to one target atom) are searched for; from
        // empty duals every row was (8.0 ms a call of 20,000 frames x 300
        // interchangeable atoms).
        if (!lp_row_minima(q, k, grx, gry, grz, s_biggest, u, col, lane, lead ? 0 : 32))
            s_finite = 0;
        sync();
        if (!lead) continue;
        const bool greedy = s_finite != 0;
        for (int j = lane; j <= k; j += kWave) {
            p[j] = greedy ? INT_MAX : 0;
            way[j] = j && greedy ? col[j] : 0;
            if (!greedy || j == 0) u[j] = 0.0;
        }
        wave_sync();
        for (int j = lane; j <= k; j += kWave) v[j] = 0.0;
        if (greedy)
            for (int i = 1 + lane; i <= k; i += kWave) atomicMin(&p[way[i]], i);
        wave_sync();
        unsigned free_rows = 0;  // bit s: row 1 + lane + 64 s has no column
        for (int s = 0; s * kWave < k; ++s) {
            const int i = 1 + lane + s * kWave;
            if (i <= k && !(greedy && p[way[i]] == i)) free_rows |= 1u << s;
        }
        wave_sync();
        for (int j = lane; j <= k; j += kWave) {
            if (p[j] == INT_MAX) p[j] = 0;
            way[j] = 0;
        }
        wave_sync();
        // The rows left over, kEach columns a lane at a time: one or two where the
        // group has no more, five for up to five, two beyond, where a last five
        // would be mostly repeats.  Us a call of diffused atoms with five always /
        // so: 10,000 frames of 100 atoms 5,300 / 4,000, of 32 atoms 807 / 467, one
        // frame of 100 atoms 1,020 / 780, 500 of 700 102,000 / 93,000.
        auto search = [&](auto each) {
            constexpr int kEach = decltype(each)::value;
            for (int s = 0; s * kWave < k; ++s) {
                for (unsigned long long rows = __ballot((free_rows >> s) & 1u); rows; rows &= rows - 1) {
                    const int i = s * kWave + __ffsll((long long)rows);
                    for (int j = lane; j <= k; j += kWave) {
                        minv[j] = __builtin_huge_val();
                        used[j] = 0;
                    }
                    if (lane == 0) p[0] = i;
                    wave_sync();
                    int j0 = 0;
                    // each pass marks one more column used; a free column (p = 0) is
                    // reached within i passes, so the loop ends for any costs
                    for (int pass = 0; pass <= k; ++pass) {
                        if (lane == 0) used[j0] = 1;
                        wave_sync();
                        const int i0 = p[j0];
                        const float qx = grx[i0 - 1], qy = gry[i0 - 1], qz = grz[i0 - 1];
                        const double ui = u[i0];
                        double best = __builtin_huge_val();
                        int at = INT_MAX;
                        for (int b0 = 1 + lane; b0 <= k; b0 += kEach * kWave) {
                            bool open[kEach];
                            int ta[kEach];
                            double vj[kEach], mv[kEach];
                            float dx[kEach], dy[kEach], dz[kEach];
    #pragma unroll
                            for (int t = 0; t < kEach; ++t) {
                                const int j = min(b0 + t * kWave, k);
                                open[t] = b0 + t * kWave <= k && !used[j];
                                ta[t] = gat[j - 1];
                                vj[t] = v[j];
                                mv[t] = minv[j];
                            }
    #pragma unroll
                            for (int t = 0; t < kEach; ++t) {
                                dx[t] = qx - tx[ta[t]];
                                dy[t] = qy - ty[ta[t]];
                                dz[t] = qz - tz[ta[t]];
                            }
    #pragma unroll
                            for (int t = 0; t < kEach; ++t) {
                                const int j = b0 + t * kWave;
                                const double cur = lp_cost(dx[t], dy[t], dz[t]) - ui - vj[t];
                                if (open[t]) {
                                    if (cur < mv[t]) {
                                        mv[t] = cur;
                                        minv[j] = cur;
                                        way[j] = j0;
                                    }
                                    if (mv[t] < best || at == INT_MAX) {
                                        best = mv[t];
                                        at = j;
                                    }
                                }
                            }
                        }
                        wave_argmin(best, at);
                        const double delta = best;
                        wave_sync();  // every lane has read u[i0] before it changes
                        for (int b0 = lane; b0 <= k; b0 += kEach * kWave) {
                            bool taken[kEach];
                            double was[kEach];
    #pragma unroll
                            for (int t = 0; t < kEach; ++t) taken[t] = used[min(b0 + t * kWave, k)];
    #pragma unroll
                            for (int t = 0; t < kEach; ++t) {
                                const int j = min(b0 + t * kWave, k);
                                was[t] = taken[t] ? v[j] : minv[j];
                            }
    #pragma unroll
                            for (int t = 0; t < kEach; ++t) {
                                const int j = b0 + t * kWave;
                                if (j <= k) {
                                    if (taken[t]) u[p[j]] += delta;
                                    (taken[t] ? v : minv)[j] = was[t] - delta;
                                }
                            }
                        }
                        wave_sync();
                        j0 = at;
                        if (p[j0] == 0) break;
                    }
                    if (lane == 0) {
                        int jj = j0;
                        for (int step = 0; step <= k && jj != 0; ++step) {
                            const int j1 = way[jj];
                            p[jj] = p[j1];
                            jj = j1;
                        }
                    }
                    wave_sync();
                }
            }
        };
        if (k < kWave)
            search(std::integral_constant<int, 1>{});
        else if (k < 2 * kWave || k >= kLpBatch * kWave)
            search(std::integral_constant<int, 2>{});
        else
            search(std::integral_constant<int, kLpBatch>{});
        // column j (target atom gat[j - 1]) takes row p[j] (reference atom gat[p[j] - 1])
        for (int j = 1 + lane; j <= k; j += kWave) {
            const int ta = gat[j - 1], ra = p[j] - 1;
            const double t[3] = {tx[ta], ty[ta], tz[ta]};
            const double r[3] = {grx[ra], gry[ra], grz[ra]};
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int b = 0; b < 3; ++b) M2[3 * a + b] = fma(t[a], r[b], M2[3 * a + b]);
        }
        wave_sync();  // the next group overwrites the group's arrays
    }
    if (!lead) return;

    // correlation of the relabelled selection with the reference: the
    // distinguishable atoms keep their labels
    for (int k = lane; k < A.n_dis; k += kWave) {
        const int a = clamp_index(A.dis[k], n);
        const double t[3] = {tx[a], ty[a], tz[a]};
        const double r[3] = {rx[a], ry[a], rz[a]};
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) M2[3 * i + j] = fma(t[i], r[j], M2[3 * i + j]);
    }

    // (4) QCP on the relabelled selection
#pragma unroll
    for (int e = 0; e < 9; ++e) M2[e] = lp_sum(M2[e]);
    const double rg = A.traces[0], tg = s_tg;
    double R2[9];
    double lam;
    if (A.superpose)
        lam = qcp_solve<true>(M2, 0.5 * (tg + rg), R2);
    else
        lam = qcp_solve<false>(M2, 0.5 * (tg + rg), nullptr);
    const double msd = (tg + rg - 2.0 * lam) / n;
    if (lane == 0) A.out[f] = (float)sqrt(msd > 0.0 ? msd : 0.0);
    if (!A.superpose) return;

    // superpose: every atom of the frame, centred, times R1 R2 (float, as sgemm33)
    float R3[9];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            float acc = 0.f;
#pragma unroll
            for (int q = 0; q < 3; ++q) acc += s_rot[3 * i + q] * (float)R2[3 * q + j];
            R3[3 * i + j] = acc;
        }
    double w[3] = {0.0, 0.0, 0.0};
    for (int a = lane; a < A.n_atoms; a += kWave) {
        w[0] += fr[3LL * a];
        w[1] += fr[3LL * a + 1];
        w[2] += fr[3LL * a + 2];
    }
    double wm[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) wm[c] = lp_sum(w[c]) / A.n_atoms;
    for (int a = lane; a < A.n_atoms; a += kWave) {
        const float x = (float)((double)fr[3LL * a] - wm[0]);
        const float y = (float)((double)fr[3LL * a + 1] - wm[1]);
        const float z = (float)((double)fr[3LL * a + 2] - wm[2]);
        fr[3LL * a] = x * R3[0] + y * R3[3] + z * R3[6];
        fr[3LL * a + 1] = x * R3[1] + y * R3[4] + z * R3[7];
        fr[3LL * a + 2] = x * R3[2] + y * R3[5] + z * R3[8];
    }
}

}  // namespace
}  // namespace hr

using namespace hr;

extern "C" {

size_t hr_lprmsd_workspace_bytes(int32_t n_sel, int32_t n_dis) {
    const size_t ns = n_sel > 0 ? (size_t)n_sel : 1, nd = n_dis > 0 ? (size_t)n_dis : 1;
    return align256(12 * ns) + align256(12 * nd) + align256(2 * sizeof(double));
}

int hr_lprmsd(float* xyz, int64_t n_frames, int32_t n_atoms, const float* ref_frame,
              const int32_t* atom_indices, int32_t n_sel, const int32_t* dis, int32_t n_dis,
              const int32_t* group_atoms, const int32_t* group_offsets, int32_t n_groups,
              int32_t max_group, int32_t superpose, float* out, void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms > 0 && n_sel > 0 && n_sel <= n_atoms && n_dis >= 0 &&
                   n_dis <= n_sel && n_groups >= 0 && max_group >= 0 && max_group <= n_sel,
               "invalid sizes n_frames=%lld n_atoms=%d n_sel=%d n_dis=%d n_groups=%d "
               "max_group=%d",
               (long long)n_frames, n_atoms, n_sel, n_dis, n_groups, max_group);
    HR_REQUIRE(n_frames < (1LL << 31), "too many frames (%lld)", (long long)n_frames);
    const size_t lds = lp_lds_bytes(n_sel, max_group);
    if (lds > kLpLdsMax) {
        set_error("a selection of %d atoms with a permute group of %d needs %zu bytes of LDS "
                  "per frame (at most %zu)", n_sel, max_group, lds, kLpLdsMax);
        return HR_ERR_UNSUPPORTED;
    }
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(xyz && ref_frame && atom_indices && out && workspace &&
                   (n_dis == 0 || dis) && (n_groups == 0 || (group_atoms && group_offsets)),
               "NULL pointer argument");
    hipStream_t s = (hipStream_t)stream;
    char* ws = static_cast<char*>(workspace);
    float* rsel = reinterpret_cast<float*>(ws);
    ws += align256(12 * (size_t)n_sel);
    float* rdis = reinterpret_cast<float*>(ws);
    ws += align256(12 * (size_t)(n_dis > 0 ? n_dis : 1));
    double* traces = reinterpret_cast<double*>(ws);
    hipLaunchKernelGGL(lp_ref_kernel, dim3(1), dim3(kLpBlock), 0, s, ref_frame, n_atoms, atom_indices,
                       n_sel, dis, n_dis, rsel, rdis, traces);
    int rc = launch_status("lp_ref_kernel");
    if (rc) return rc;
    LpArgs A;
    A.xyz = xyz;
    A.n_frames = n_frames;
    A.n_atoms = n_atoms;
    A.idx = atom_indices;
    A.n_sel = n_sel;
    A.dis = dis;
    A.n_dis = n_dis;
    A.group_atoms = group_atoms;
    A.group_off = group_offsets;
    A.n_groups = n_groups;
    A.kmax = max_group;
    A.rsel = rsel;
    A.rdis = rdis;
    A.traces = traces;
    A.superpose = superpose ? 1 : 0;
    A.out = out;
    // the kernel's own few words count towards the default limit of 64 KiB too
    if (lds > kLpLdsMax - 256)
        HR_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(lp_frame_kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)kLpLdsMax));
    hipLaunchKernelGGL(lp_frame_kernel, launch_grid(n_frames, kLpFrameBlock), dim3(kLpFrameBlock),
                       lds, s, A);
    return launch_status("lp_frame_kernel");
}

}  // extern "C"
