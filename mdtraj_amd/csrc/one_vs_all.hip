// One-vs-all RMSD, centering, no-superpose RMSD and superposition kernels
// (gfx950).  Layout in HBM: coordinates stay as the caller holds them
// (atom-major (F, N, 3) float32 or axis-major (F, 3, rowstride)); nothing is
// re-laid-out.  A row of 4 - 64 lanes of a wavefront owns one frame at a time
// and sweeps its selected atoms with lane-strided loads; per-frame sums are
// accumulated in FP64 in registers and reduced across the row; the QCP
// solve then runs one lane per frame (lane k finishes the k-th frame of the
// wave's current group of 64).  The reference selection and the atom indices
// are staged once per workgroup in LDS.
#include <algorithm>

#include "frames.h"

namespace hr {
namespace {

// Per-frame kernel.  One workgroup per CU holds all of the CU's waves
// (kMinWaves per SIMD).  Each wave walks its items (frame set, atom block)
// through a ring of kRing register buffers, so the loads of the next
// kRing - 1 items are in flight while one is accumulated in FP64.  A frame
// set is kWave / kRL frames, one per row of kRL lanes.  At the end of a set
// each row's sums are reduced across its lanes (DPP within 16 lanes,
// shuffles across) and parked in LDS; every 64 frames the QCP solve runs one
// lane per frame.  The workgroup owns 1/G of the frame sets: each wave takes
// a static share of the first static_pct percent of them, and the rest goes
// out in chunks of `chunk` frames by an LDS ticket, so that the waves the
// SIMD issues less often take fewer frames (process_cu).
//   kAxis   target is axis-major (F, 3, rowstride) instead of atom-major
//   kGather atom-major target with an index list
//   kStage  what the workgroup stages in LDS: kStageAll the reference
//           selection and the indices; kStageIdx the indices only (a
//           gathered selection whose reference does not fit; the reference
//           then rides the load ring); kStageNone nothing
template <Kind kKind, bool kAxis, bool kGather, int kStage, int kMinWaves, int kRL>
__global__ __launch_bounds__(CuGroup<kMinWaves>::kThreads, kMinWaves) void frames_kernel(
    const float* __restrict__ xyz, long long n_frames, long long frame_stride, int rowstride,
    const int* __restrict__ idx, int n_sel, const float* __restrict__ ref_sel,
    const double* __restrict__ ref_stats, long long self_frame, float* __restrict__ out,
    float* __restrict__ rot_out, double* __restrict__ mu_out, int static_pct, long long chunk) {
    constexpr int kNS = SumsPerFrame<kKind>::value;
    constexpr int kWaves = CuGroup<kMinWaves>::kWaves;
    constexpr int kThreads = CuGroup<kMinWaves>::kThreads;
    extern __shared__ double smem_d[];
    __shared__ unsigned s_ticket;
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    double* s_res = smem_d + wv * kWave * kNS;
    float* smem = reinterpret_cast<float*>(smem_d + kWaves * kWave * kNS);
    const float* rx = ref_sel;
    const float* ry = ref_sel + n_sel;
    const float* rz = ref_sel + 2 * n_sel;
    const int* ix = idx;
    // ref_stats == nullptr (Kind::Rmsd, kStageAll only): ref_sel is the
    // reference selection itself (n_sel atoms, xyz interleaved), and every
    // workgroup prepares it, with the prep kernel's arithmetic, into its LDS
    __shared__ double s_stats[4];
    if (threadIdx.x == 0) s_ticket = 0u;
    if constexpr (kStage != kStageNone) {
        // LDS after the result area: [reference planes (kStageAll)] [indices]
        float* s_rx = smem;
        float* s_ry = smem + n_sel;
        float* s_rz = smem + 2 * n_sel;
        int* s_idx = reinterpret_cast<int*>(kStage == kStageAll ? smem + 3 * n_sel : smem);
        if constexpr (kStage == kStageAll) {
            if (kKind == Kind::Rmsd && ref_stats == nullptr)  // uniform over the grid
                ref_prep_body(ref_sel, nullptr, n_sel, 0, s_rx, s_stats);
            else
                stage_words<kThreads>(s_rx, ref_sel, 3 * n_sel);
        }
        if constexpr (kGather) stage_words<kThreads>(s_idx, idx, n_sel);
        if constexpr (kStage == kStageAll) {
            rx = s_rx;
            ry = s_ry;
            rz = s_rz;
        }
        if constexpr (kGather) ix = s_idx;
    }
    __syncthreads();
    double rs[4] = {0.0, 0.0, 0.0, 0.0};
    if constexpr (kKind != Kind::NoSuperpose) {
        const double* st = ref_stats;
        if constexpr (kStage == kStageAll && kKind == Kind::Rmsd) {
            if (ref_stats == nullptr) st = s_stats;
        }
        rs[0] = st[0];
        rs[1] = st[1];
        rs[2] = st[2];
        rs[3] = st[3];
    }
    // whole frame sets (a set fills the wave's kWave / kRL rows): the
    // workgroup's sets b0 .. b1, the first n_static of them split evenly
    // over its waves, the rest ticketed
    constexpr int kRows = kWave / kRL;
    const long long n_sets = (n_frames + kRows - 1) / kRows;
    const long long g = blockIdx.x, n_groups = gridDim.x;
    const long long b0 = g * n_sets / n_groups, b1 = (g + 1) * n_sets / n_groups;
    const long long n_static = (b1 - b0) * static_pct / 100;
    const long long s0 = b0 + wv * n_static / kWaves, s1 = b0 + (wv + 1) * n_static / kWaves;
    process_cu<kKind, kAxis, kGather, kRL, kStage != kStageAll>(
        xyz, min(n_frames, kRows * s0), min(n_frames, kRows * s1),
        min(n_frames, kRows * (b0 + n_static)), min(n_frames, kRows * b1), chunk, &s_ticket,
        frame_stride, rowstride, ix, n_sel, rx, ry, rz, rs, self_frame, out, rot_out, mu_out, s_res,
        lane);
}

// Hands the n words at src (4-byte aligned) to put4(i, four words from i on) and
// put(i, word i) for the last ones, kLoads loads of 16 bytes a lane in flight.
// The loads are unconditional (past the end the last unit again): a load
// under a branch is waited for where the branch ends.
typedef float V4f __attribute__((ext_vector_type(4), aligned(4)));

template <int kThreads, int kLoads, typename Put4, typename Put>
__device__ __forceinline__ void copy_words(const float* __restrict__ src, int n, int tid,
                                           Put4 put4, Put put) {
    const int whole = n & ~3;
    float last = 0.0f;
    if (tid < n - whole) last = src[whole + tid];
    for (int i0 = 0; i0 < whole; i0 += 4 * kLoads * kThreads) {
        V4f v[kLoads];
#pragma unroll
        for (int t = 0; t < kLoads; ++t)
            v[t] = __builtin_nontemporal_load(reinterpret_cast<const V4f*>(
                src + min(i0 + 4 * (t * kThreads + tid), whole - 4)));
#pragma unroll
        for (int t = 0; t < kLoads; ++t) {
            const int i = i0 + 4 * (t * kThreads + tid);
            if (i < whole) put4(i, v[t]);
        }
    }
    if (tid < n - whole) put(whole + tid, last);
}

// One-vs-all over whole short frames: a lane per frame.  A wave's 64 frames
// are consecutive in memory; they come into LDS 16 bytes a lane, and each
// lane then walks its own frame there, the reference atoms being the same for
// all lanes (scalar loads).  There is nothing to reduce across lanes and no
// lane without an atom, which is what bounds rows of 4 or 8 lanes on such
// frames (vector instructions per 22-atom frame: about 37 a wave, here 17).
// Bank conflicts: lane strides of 3 n words, n a multiple of 4, would meet in
// 16 banks or fewer, so such frames are spread by a word each.
//
// Us per launch with the reference's preparation, rows of lanes against a lane
// per frame: 2,000,003 frames of 8 atoms 97 / 61; 1,000,003 of 12 57 / 34, of 16
// 61 / 43, of 22 92 / 64, of 30 98 / 87; 700,000 of 36 102 / 77; 500,000 of 40 80 /
// 67, of 45 80 / 81, of 52 83 / 91; 1,000 frames of 22 13 / 10, of 8 11 / 7.  With
// 64 frames in LDS a wave, longer frames leave the CU too few waves; hence
// kShortAtoms.  At 22 atoms HBM would allow 41 us (264 MB); the rest is the
// sums' and the fits' FP64 work, about 28 us of vector issue, and the nine
// waves a CU's LDS holds.
constexpr int kShortLoads = 9;
constexpr int kShortAtoms = 40;

// kRawRef: ref_sel is the reference itself (x, y, z interleaved) and every wave
// prepares it, with ref_prep_body's arithmetic (each of its first n_atoms
// threads has one atom), into LDS: the one launch of a small host call, where
// frames and reference are read over PCIe.
template <bool kRawRef>
__global__ __launch_bounds__(kWave, 3) void short_frames_kernel(
    const float* __restrict__ xyz, long long n_frames, int n_atoms,
    const float* __restrict__ ref_sel, const double* __restrict__ ref_stats, long long self_frame,
    float* __restrict__ out) {
    extern __shared__ __align__(16) float s_frames[];
    const int lane = threadIdx.x;
    const long long f0 = workgroup_index() * kWave;
    if (f0 >= n_frames) return;
    const int cnt = (int)min((long long)kWave, n_frames - f0);
    const int words = 3 * n_atoms, n_words = cnt * words;
    const bool spread = (n_atoms & 3) == 0;
    const float* run = xyz + f0 * words;
    __shared__ float s_ref[kRawRef ? 3 * kShortAtoms : 1];
    float ref_x = 0.0f, ref_y = 0.0f, ref_z = 0.0f;
    if (kRawRef && lane < n_atoms) {
        ref_x = ref_sel[3 * lane];
        ref_y = ref_sel[3 * lane + 1];
        ref_z = ref_sel[3 * lane + 2];
    }
    // frame of 16-byte unit u when frames are whole units: u / (words / 4)
    const unsigned magic = 0xFFFFFFFFu / (unsigned)max(words / 4, 2) + 1u;
    copy_words<kWave, kShortLoads>(run, n_words, lane, [&](int i, V4f v) {
        if (spread) {
            float* to = s_frames + i + (int)__umulhi((unsigned)i / 4, magic);
            to[0] = v.x;
            to[1] = v.y;
            to[2] = v.z;
            to[3] = v.w;
        } else {
            *reinterpret_cast<float4*>(s_frames + i) = make_float4(v.x, v.y, v.z, v.w);
        }
    }, [&](int i, float v) { s_frames[i] = v; });  // (frames of whole units end on one)
    double rs[4];
    const float* rx = ref_sel;
    if constexpr (kRawRef) {
        if (lane < n_atoms) {
            s_ref[lane] = ref_x;
            s_ref[n_atoms + lane] = ref_y;
            s_ref[2 * n_atoms + lane] = ref_z;
        }
        const double x = ref_x, y = ref_y, z = ref_z;
        rs[0] = wave_sum(x);
        rs[1] = wave_sum(y);
        rs[2] = wave_sum(z);
        rs[3] = wave_sum(fma(x, x, fma(y, y, fma(z, z, 0.0))));
        rx = s_ref;
    } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) rs[c] = ref_stats[c];
    }
    __syncthreads();
    if (lane >= cnt) return;
    const float* fr = s_frames + lane * (words + (spread ? 1 : 0));
    const float* ry = rx + n_atoms;
    const float* rz = ry + n_atoms;
    Sums s = {};
#pragma unroll 4
    for (int j = 0; j < n_atoms; ++j)
        accumulate<Kind::Rmsd>(s, fr[3 * j], fr[3 * j + 1], fr[3 * j + 2], rx[j], ry[j], rz[j]);
    const double n = (double)n_atoms;
    double M[9], ga, gb;
    centred(s, rs, n, M, ga, gb);
    const double msd = qcp_msd(M, ga, gb, n);
    const long long f = f0 + lane;
    out[f] = f == self_frame ? 0.0f : (float)sqrt(msd);
}

// In-place centering and traces, one wave per frame (two passes over the
// frame; the second usually hits in L2).  Rounding as the reference:
// double sums, float mean, float subtraction, float squares summed in double.
__global__ __launch_bounds__(kBlock) void center_kernel(float* __restrict__ xyz,
                                                        float* __restrict__ traces,
                                                        long long n_frames, int n_atoms) {
    const int lane = threadIdx.x & (kWave - 1);
    const long long wave = (long long)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave;
    const long long n_waves = (long long)gridDim.x * kWavesPerBlock;
    for (long long f = wave; f < n_frames; f += n_waves) {
        float* fr = xyz + f * 3LL * n_atoms;
        double sx = 0.0, sy = 0.0, sz = 0.0;
        for (int a = lane; a < n_atoms; a += kWave) {
            sx += (double)fr[3 * a];
            sy += (double)fr[3 * a + 1];
            sz += (double)fr[3 * a + 2];
        }
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        sz = wave_sum(sz);
        const float mx = (float)(sx / n_atoms), my = (float)(sy / n_atoms),
                    mz = (float)(sz / n_atoms);
        double tr = 0.0;
        for (int a = lane; a < n_atoms; a += kWave) {
            const float x = fr[3 * a] - mx, y = fr[3 * a + 1] - my, z = fr[3 * a + 2] - mz;
            fr[3 * a] = x;
            fr[3 * a + 1] = y;
            fr[3 * a + 2] = z;
            tr += (double)(x * x);
            tr += (double)(y * y);
            tr += (double)(z * z);
        }
        tr = wave_sum(tr);
        if (lane == 0 && traces) traces[f] = (float)tr;
    }
}

// x' = float(float(x - mu_f) R + mu_ref) of one atom, rounding as
// Trajectory.superpose does (float64 offsets applied to float32 coordinates,
// float32 rotation, core/trajectory.py:1135-1171); without translate x' = x R.
__device__ __forceinline__ void move_atom(float ax, float ay, float az, const float (&R)[9],
                                          const double (&m)[3], const double (&to)[3],
                                          int translate, float (&o)[3]) {
    const float x = translate ? (float)((double)ax - m[0]) : ax;
    const float y = translate ? (float)((double)ay - m[1]) : ay;
    const float z = translate ? (float)((double)az - m[2]) : az;
    const float tx = x * R[0] + y * R[3] + z * R[6];
    const float ty = x * R[1] + y * R[4] + z * R[7];
    const float tz = x * R[2] + y * R[5] + z * R[8];
    o[0] = translate ? (float)((double)tx + to[0]) : tx;
    o[1] = translate ? (float)((double)ty + to[1]) : ty;
    o[2] = translate ? (float)((double)tz + to[2]) : tz;
}

// Every atom of every frame moved by its frame's fit.
__global__ __launch_bounds__(kBlock) void apply_kernel(float* __restrict__ xyz, long long n_frames,
                                                       int n_atoms, const float* __restrict__ rot,
                                                       const double* __restrict__ mu,
                                                       const double* __restrict__ ref_stats,
                                                       double n_ref, int translate) {
    double to[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < 3; ++c) to[c] = translate ? ref_stats[c] / n_ref : 0.0;
    for (long long f = blockIdx.x; f < n_frames; f += gridDim.x) {
        float R[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) R[i] = rot[9 * f + i];
        double m[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < 3; ++c) m[c] = translate ? mu[3 * f + c] : 0.0;
        float* fr = xyz + f * 3LL * n_atoms;
        for (int a = threadIdx.x; a < n_atoms; a += kBlock) {
            float o[3];
            move_atom(fr[3 * a], fr[3 * a + 1], fr[3 * a + 2], R, m, to, translate, o);
            fr[3 * a] = o[0];
            fr[3 * a + 1] = o[1];
            fr[3 * a + 2] = o[2];
        }
    }
}

// Superposition in one pass over memory: a workgroup holds a run of whole
// frames in LDS (consecutive in memory), fits every one of them there, and
// writes the moved atoms back; fitting and moving in two kernels reads the
// frames twice.
//   load   16 bytes a lane, kLoads of them in flight
//   sums   a row of kRL lanes per frame, or kWavesPer waves when a run has
//          fewer frames than the workgroup has waves (their parts are added
//          below)
//   fit    one lane per frame, from the frame's sums in LDS
//   move   atom by atom to memory; whole waves per frame when frames are
//          long (the fit stays in registers), else atoms dealt out flat
// Rounding is the two kernels': the sums are FP64 in another order.
//
// Bound by HBM, a read and a write of every atom: 20,000 frames of 3,001 atoms
// (375 of them fitted), 1.44 GB, in 275-325 us by box (4.4-5.2 TB/s, the rate of
// a device copy) against 390 us for two kernels, which move 2.3 GB.  (Two
// persistent workgroups a CU, each with a second buffer filled by direct loads
// to LDS, were slower, 417 us: two frames at work on a CU instead of four.)
constexpr int kLoads = 10;
// Frames of this many atoms on keep a frame's fit in registers while whole
// waves move its atoms.
constexpr int kFlatAtoms = 192;

// Bytes before the coordinates in LDS: per frame the parts' sums, the centroid
// and the rotation.
__host__ __device__ __forceinline__ size_t superpose_head(int per_group, int parts) {
    return ((size_t)per_group * (parts * 13 * 8 + 3 * 8 + 9 * 4) + 15) / 16 * 16;
}

template <int kRL, int kWavesPer, bool kGather>
__global__ __launch_bounds__(kBlock, 4) void superpose_kernel(
    float* __restrict__ xyz, long long n_frames, int n_atoms, int per_group,
    const int* __restrict__ idx, int n_sel, const float* __restrict__ ref_sel,
    const double* __restrict__ ref_stats, int translate, float* __restrict__ rot_out,
    float* __restrict__ rmsd_out) {
    static_assert(kWavesPer == 1 || kRL == kWave, "waves share frames as whole rows");
    constexpr int kThreads = kBlock;
    constexpr int kNS = SumsPerFrame<Kind::Fit>::value;
    extern __shared__ __align__(16) unsigned char s_mem[];
    const int words = 3 * n_atoms;
    double* s_sum = reinterpret_cast<double*>(s_mem);            // per_group x kWavesPer x kNS
    double* s_mu = s_sum + (size_t)per_group * kWavesPer * kNS;     // per_group x 3
    float* s_rot = reinterpret_cast<float*>(s_mu + 3 * per_group);  // per_group x 9
    float* s_x = reinterpret_cast<float*>(s_mem + superpose_head(per_group, kWavesPer));
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const long long f0 = workgroup_index() * per_group;
    if (f0 >= n_frames) return;
    const int cnt = (int)min((long long)per_group, n_frames - f0);
    float* run = xyz + f0 * words;
    const int n_words = cnt * words;

    constexpr int kLanes = kWavesPer > 1 ? kWavesPer * kWave : kRL;
    constexpr int kRows = kThreads / kLanes;
    const int row = tid / kLanes, t = tid % kLanes;
    // kItemAtoms atoms of the selection a lane: where they are in a frame and
    // the reference's
    struct Item {
        int at[kItemAtoms];
        float x[kItemAtoms], y[kItemAtoms], z[kItemAtoms];
    } a_item, b_item;
    auto fetch = [&](int item, Item& it) {
#pragma unroll
        for (int u = 0; u < kItemAtoms; ++u) {
            const int j = min(t + (item * kItemAtoms + u) * kLanes, n_sel - 1);
            it.at[u] = 3 * (kGather ? idx[j] : j);
            it.x[u] = ref_sel[j];
            it.y[u] = ref_sel[n_sel + j];
            it.z[u] = ref_sel[2 * n_sel + j];
        }
    };
    fetch(0, a_item);

    copy_words<kThreads, kLoads>(run, n_words, tid, [&](int i, V4f v) {
        *reinterpret_cast<float4*>(s_x + i) = make_float4(v.x, v.y, v.z, v.w);
    }, [&](int i, float v) { s_x[i] = v; });
    __syncthreads();

    // the row's items in turn: frame after frame, item after item; while one is
    // accumulated the next one's indices and reference atoms are on their way
    {
        const int items = (n_sel + kItemAtoms * kLanes - 1) / (kItemAtoms * kLanes);
        int k = row, item = 0;
        Sums s = {};
        auto step = [&](Item& now, Item& next) {
            const int item_next = item + 1 < items ? item + 1 : 0;
            fetch(item_next, next);
            const float* fr = s_x + (k < cnt ? k : 0) * words;
            float bx[kItemAtoms], by[kItemAtoms], bz[kItemAtoms];
#pragma unroll
            for (int u = 0; u < kItemAtoms; ++u) {
                bx[u] = fr[now.at[u]];
                by[u] = fr[now.at[u] + 1];
                bz[u] = fr[now.at[u] + 2];
            }
#pragma unroll
            for (int u = 0; u < kItemAtoms; ++u) {
                const bool ok = t + (item * kItemAtoms + u) * kLanes < n_sel;
                accumulate<Kind::Fit>(s, valid_atom(ok, bx[u]), valid_atom(ok, by[u]),
                                      valid_atom(ok, bz[u]), now.x[u], now.y[u], now.z[u]);
            }
            if (item_next == 0) {
                row_reduce<Kind::Fit, kRL>(s);
                if (t % kRL == 0 && k < cnt)
                    store_sums<Kind::Fit>(s_sum + ((size_t)k * kWavesPer + t / kRL) * kNS, s);
                s = Sums{};
                k += kRows;
            }
            item = item_next;
        };
        const int total = (cnt + kRows - 1) / kRows * items;
        for (int i = 0; i < total; i += 2) {
            step(a_item, b_item);
            if (i + 1 < total) step(b_item, a_item);
        }
    }
    __syncthreads();

    const double n = (double)n_sel;
    if (tid < cnt) {
        Sums mine;
        load_sums<Kind::Fit>(mine, s_sum + (size_t)tid * kWavesPer * kNS);
#pragma unroll
        for (int w = 1; w < kWavesPer; ++w) {
            Sums part;
            load_sums<Kind::Fit>(part, s_sum + ((size_t)tid * kWavesPer + w) * kNS);
            mine.q += part.q;
            mine.sx += part.sx;
            mine.sy += part.sy;
            mine.sz += part.sz;
#pragma unroll
            for (int e = 0; e < 9; ++e) mine.p[e] += part.p[e];
        }
        const double rs[4] = {ref_stats[0], ref_stats[1], ref_stats[2], ref_stats[3]};
        double M[9], ga, gb, R[9];
        centred(mine, rs, n, M, ga, gb);
        const double lam = qcp_solve<true>(M, 0.5 * (ga + gb), R);
        const long long f = f0 + tid;
#pragma unroll
        for (int e = 0; e < 9; ++e) {
            s_rot[9 * tid + e] = (float)R[e];
            if (rot_out) rot_out[9 * f + e] = (float)R[e];
        }
        s_mu[3 * tid] = mine.sx / n;
        s_mu[3 * tid + 1] = mine.sy / n;
        s_mu[3 * tid + 2] = mine.sz / n;
        if (rmsd_out) {
            const double msd = (ga + gb - 2.0 * lam) / n;
            rmsd_out[f] = (float)sqrt(msd > 0.0 ? msd : 0.0);
        }
    }
    __syncthreads();

    double to[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) to[c] = translate ? ref_stats[c] / n : 0.0;
    float R[9], o[3];
    double m[3];
    auto fit_of = [&](int k) {
#pragma unroll
        for (int e = 0; e < 9; ++e) R[e] = s_rot[9 * k + e];
#pragma unroll
        for (int c = 0; c < 3; ++c) m[c] = s_mu[3 * k + c];
    };
    if (n_atoms >= kFlatAtoms) {
        constexpr int kStep = kWavesPerBlock / kWavesPer;  // frames side by side
        for (int k = wv / kWavesPer; k < cnt; k += kStep) {
            fit_of(k);
            const float* fr = s_x + k * words;
            float* dst = run + k * words;
            for (int a = wv % kWavesPer * kWave + lane; a < n_atoms; a += kWavesPer * kWave) {
                move_atom(fr[3 * a], fr[3 * a + 1], fr[3 * a + 2], R, m, to, translate, o);
                dst[3 * a] = o[0];
                dst[3 * a + 1] = o[1];
                dst[3 * a + 2] = o[2];
            }
        }
    } else {
        // frame of atom e: e / n_atoms, exact for e < 2^16 and n_atoms < 2^16
        const unsigned magic = n_atoms > 1 ? 0xFFFFFFFFu / (unsigned)n_atoms + 1u : 0u;
        for (int e = tid; e < cnt * n_atoms; e += kThreads) {
            fit_of(n_atoms > 1 ? (int)__umulhi((unsigned)e, magic) : e);
            move_atom(s_x[3 * e], s_x[3 * e + 1], s_x[3 * e + 2], R, m, to, translate, o);
            run[3 * e] = o[0];
            run[3 * e + 1] = o[1];
            run[3 * e + 2] = o[2];
        }
    }
}

template <bool kRawRef>
int launch_short(hipStream_t s, const float* xyz, long long n_frames, int n_atoms,
                 const float* ref, const double* stats, long long self_frame, float* out) {
    hipLaunchKernelGGL(short_frames_kernel<kRawRef>,
                       launch_grid((n_frames + kWave - 1) / kWave, kWave), dim3(kWave),
                       (size_t)kWave * (12 * n_atoms + 4), s, xyz, n_frames, n_atoms, ref, stats,
                       self_frame, out);
    return launch_status("short_frames_kernel");
}

struct Launch {
    size_t lds;
    int stage;  // kStageAll, kStageIdx or kStageNone
};

// Waves per SIMD of the per-frame kernel (HR_TUNE_FRAMES_WAVES_PER_SIMD).
int frames_waves_per_simd() { return tuning(HR_TUNE_FRAMES_WAVES_PER_SIMD) == 4 ? 4 : 3; }

// LDS plan of the one workgroup per CU: the result area of its waves
// always; the reference selection and the indices when they fit in the CU's
// LDS together with it, else the indices alone (gathered selections), else
// nothing.  At 3 waves/SIMD (80 KB of results) that stages selections of up
// to ~6,900 contiguous or ~5,200 gathered atoms.
template <Kind kKind>
int plan(int n_sel, bool gather, Launch* l) {
    const DeviceInfo* d = current_device();
    if (!d) return HR_ERR_HIP;
    const size_t res = result_lds_bytes<kKind>(4 * frames_waves_per_simd());
    const size_t ref = (size_t)n_sel * 3 * sizeof(float);
    const size_t ids = gather ? (size_t)n_sel * sizeof(int) : 0;
    const size_t cap = std::min(d->lds_per_block, d->lds_per_cu) - 256;  // 256: static LDS
    if (res + ref + ids <= cap) {
        l->stage = kStageAll;
        l->lds = res + ref + ids;
    } else if (gather && res + ids <= cap) {
        l->stage = kStageIdx;
        l->lds = res + ids;
    } else {
        l->stage = kStageNone;
        l->lds = res;
    }
    return HR_OK;
}

// One workgroup per CU (occupancy API: the workgroup holds all of a CU's
// waves), capped by the work: no more waves than frame sets.
template <typename Kernel>
int frames_grid(Kernel kernel, int threads, size_t lds, long long n_frames, int rows,
                int* blocks) {
    const DeviceInfo* d = current_device();
    if (!d) return HR_ERR_HIP;
    int per_cu = 0;
    HR_CHECK_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, reinterpret_cast<const void*>(kernel), threads, lds));
    if (per_cu < 1) per_cu = 1;
    long long b = (long long)per_cu * d->cu_count;
    const long long n_sets = (n_frames + rows - 1) / rows;
    const int waves = threads / kWave;
    const long long by_work = (n_sets + waves - 1) / waves;
    if (b > by_work) b = by_work;
    *blocks = (int)(b < 1 ? 1 : b);
    return HR_OK;
}

template <Kind kKind, bool kAxis, bool kGather, int kStage, int kMinWaves, int kRL>
int launch_frames_v(const Launch& l, hipStream_t s, const float* xyz, long long n_frames,
                    long long frame_stride, int rowstride, const int* idx, int n_sel,
                    const float* ref_sel, const double* ref_stats, long long self_frame,
                    float* out, float* rot_out, double* mu_out) {
    int blocks = 0, rc;
    auto k = frames_kernel<kKind, kAxis, kGather, kStage, kMinWaves, kRL>;
    constexpr int kThreads = CuGroup<kMinWaves>::kThreads;
    constexpr int kRows = kWave / kRL;
    static bool lds_attr_set = false;  // dynamic LDS beyond 64 KB needs the attribute
    if (!lds_attr_set) {
        const DeviceInfo* d = current_device();
        if (!d) return HR_ERR_HIP;
        HR_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                         hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)(std::min(d->lds_per_block, d->lds_per_cu) - 256)));
        lds_attr_set = true;
    }
    if ((rc = frames_grid(k, kThreads, l.lds, n_frames, kRows, &blocks))) return rc;
    // With at most one frame set per wave there is nothing to balance: every
    // set is assigned statically, so that no wave takes a chunk of several
    // sets in series while others idle (1,000 frames x 22 atoms: 18 us).
    const bool one_each = (n_frames + kRows - 1) / kRows <= (long long)blocks * (kThreads / kWave);
    const int pct = tuning(HR_TUNE_FRAMES_STATIC_PCT) ? tuning(HR_TUNE_FRAMES_STATIC_PCT)
                    : one_each                        ? 100
                                                      : kDefaultStaticPct;
    const long long kib = tuning(HR_TUNE_FRAMES_CHUNK_KIB) ? tuning(HR_TUNE_FRAMES_CHUNK_KIB)
                                                          : kDefaultChunkKiB;
    const long long frame_bytes = 12LL * (n_sel > 0 ? n_sel : 1);
    long long chunk = (kib * 1024 + frame_bytes - 1) / frame_bytes;
    chunk = std::max<long long>(kRows, std::min<long long>((chunk + kRows - 1) / kRows * kRows,
                                                           kWave));
    hipLaunchKernelGGL(k, dim3(blocks), dim3(kThreads), l.lds, s, xyz, n_frames, frame_stride,
                       rowstride, idx, n_sel, ref_sel, ref_stats, self_frame, out, rot_out,
                       mu_out, pct, chunk);
    return launch_status("frames_kernel");
}

// auto_row_lanes (frames.h) picks the row width; HR_TUNE_FRAMES_ROW_LANES
// overrides it.
// Register budget of the per-frame kernel: 3 waves per SIMD (no spills) or 4
// (more loads in flight, a few spilled registers); HR_TUNE_FRAMES_WAVES_PER_SIMD.
template <Kind kKind, bool kAxis, bool kGather>
int launch_frames(const Launch& l, hipStream_t s, const float* xyz, long long n_frames,
                  long long frame_stride, int rowstride, const int* idx, int n_sel,
                  const float* ref_sel, const double* ref_stats, long long self_frame, float* out,
                  float* rot_out, double* mu_out) {
    const bool four = frames_waves_per_simd() == 4;
    const int rl = tuning(HR_TUNE_FRAMES_ROW_LANES) ? tuning(HR_TUNE_FRAMES_ROW_LANES)
                                                   : auto_row_lanes(n_sel, kGather);
#define HR_FRAMES_ARGS l, s, xyz, n_frames, frame_stride, rowstride, idx, n_sel, ref_sel, \
                       ref_stats, self_frame, out, rot_out, mu_out
#define HR_FRAMES_RL(LDS, W)                                                               \
    (rl == 64   ? launch_frames_v<kKind, kAxis, kGather, LDS, W, 64>(HR_FRAMES_ARGS)       \
     : rl == 32 ? launch_frames_v<kKind, kAxis, kGather, LDS, W, 32>(HR_FRAMES_ARGS)       \
     : rl == 16 ? launch_frames_v<kKind, kAxis, kGather, LDS, W, 16>(HR_FRAMES_ARGS)       \
     : rl == 8  ? launch_frames_v<kKind, kAxis, kGather, LDS, W, 8>(HR_FRAMES_ARGS)        \
                : launch_frames_v<kKind, kAxis, kGather, LDS, W, 4>(HR_FRAMES_ARGS))
    if (l.stage == kStageAll)
        return four ? HR_FRAMES_RL(kStageAll, 4) : HR_FRAMES_RL(kStageAll, 3);
    if constexpr (kGather) {
        if (l.stage == kStageIdx)
            return four ? HR_FRAMES_RL(kStageIdx, 4) : HR_FRAMES_RL(kStageIdx, 3);
    }
    return four ? HR_FRAMES_RL(kStageNone, 4) : HR_FRAMES_RL(kStageNone, 3);
#undef HR_FRAMES_RL
#undef HR_FRAMES_ARGS
}

}  // namespace

// One launch for a small call: the per-frame kernel prepares the reference
// itself (see frames_kernel).  Returns HR_OK with *done false, launching
// nothing, when the selection does not fit the kernel's LDS whole.
int one_vs_all_fused_ref(hipStream_t s, const float* frames, long long n_frames, int n_sel,
                         const float* ref, long long self_frame, float* out, bool* done) {
    *done = false;
    if (n_sel <= kShortAtoms) {
        *done = true;
        return launch_short<true>(s, frames, n_frames, n_sel, ref, nullptr, self_frame, out);
    }
    Launch l;
    int rc = plan<Kind::Rmsd>(n_sel, false, &l);
    if (rc || l.stage != kStageAll) return rc;
    *done = true;
    return launch_frames<Kind::Rmsd, false, false>(l, s, frames, n_frames, 3LL * n_sel, 0,
                                                   nullptr, n_sel, ref, nullptr, self_frame, out,
                                                   nullptr, nullptr);
}

namespace {

// LDS of superpose_kernel for per_group frames.
size_t superpose_lds(int per_group, int parts, int n_atoms) {
    return superpose_head(per_group, parts) + 12 * (size_t)per_group * n_atoms;
}

template <int kRL, int kWavesPer, bool kGather>
int launch_superpose_v(hipStream_t s, float* xyz, long long n_frames, int n_atoms, int per_group,
                       const int* idx, int n_sel, const float* ref_sel, const double* stats,
                       int translate, float* rot_out, float* rmsd_out) {
    const long long runs = (n_frames + per_group - 1) / per_group;
    const size_t lds = superpose_lds(per_group, kWavesPer, n_atoms);
    if (lds > 64 * 1024)
        HR_CHECK_HIP(hipFuncSetAttribute(
            reinterpret_cast<const void*>(superpose_kernel<kRL, kWavesPer, kGather>),
            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((superpose_kernel<kRL, kWavesPer, kGather>), launch_grid(runs, kBlock),
                       dim3(kBlock), lds, s, xyz, n_frames, n_atoms, per_group, idx, n_sel,
                       ref_sel, stats, translate, rot_out, rmsd_out);
    return launch_status("superpose_kernel");
}

// One-pass superposition where at least two workgroups a CU fit LDS (frames of
// up to ~6,600 atoms); *done is false, and nothing is launched, where the
// two-kernel path is to be used.
//
// The frames of a run: as many bytes of frames on the way per CU as its LDS and
// four workgroups allow, whole rounds of rows (or of waves) preferred, the
// smaller run where that is the same.  Kernel us for 1.44 GB, by run: 8 atoms
// 64 frames 804, 128 557, 192 533; 22 atoms 64 411, 128 426, 151 456; 50 atoms
// 32 374, 64 330; 100 atoms 16 412, 32 313; 191 atoms 12 312, 16 293; 420 atoms
// 4 350, 7 338, 8 319; 606 atoms 4 312, 5 372, 8 369; 850 atoms 3 357, 4 307;
// 1,700 atoms 1 388, 2 311; 2,000 atoms 1 346, 2 297; 3,001 atoms 1 274, 2 275.
// (The two kernels: 8 atoms 3,303, 22 atoms 1,470, 100 atoms 575, 300 atoms 497,
// 606 atoms 455, 1,000 atoms 415, 2,000 atoms 427, 3,001 atoms 390, 4,000 atoms
// 380, 6,500 atoms 454 us, against 354 in one pass; with a single workgroup a
// CU, 8,000 atoms, one pass takes 430 us against 387.)
int superpose_one_pass(hipStream_t s, float* xyz, long long n_frames, int n_atoms, const int* idx,
                       int n_sel, const float* ref_sel, const double* stats, int translate,
                       float* rot_out, float* rmsd_out, bool* done) {
    *done = false;
    const DeviceInfo* d = current_device();
    if (!d) return HR_ERR_HIP;
    const size_t cu = std::min((size_t)160000, d->lds_per_cu);  // in whole pieces
    int group = 0, waves = 0, rl = 0;
    double best = 0.0;
    for (int g = 1; g <= kBlock; g += g < 4 ? 1 : 4) {
        const int w = g == 1 ? 4 : g == 2 ? 2 : 1;
        const size_t lds = superpose_lds(g, w, n_atoms);
        const size_t resident = std::min((size_t)4, cu / lds);
        if (resident < 2) break;
        // lanes per frame: by the selection, and no fewer than leave every row
        // of the workgroup a frame
        int lanes = n_sel < 28 ? 4 : n_sel < 112 ? 8 : n_sel < 360 ? 16 : kWave;
        while (lanes < kWave && kBlock / lanes > g) lanes *= 2;
        const int rows = kBlock / lanes;
        const double used = w > 1 ? 1.0 : (double)g / ((g + rows - 1) / rows * rows);
        const double score = (double)resident * g * used * used;
        if (score > best) {
            best = score;
            group = g;
            waves = w;
            rl = lanes;
        }
    }
    if (!group) return HR_OK;
    *done = true;
#define HR_SUP(RL, W)                                                                           \
    (idx ? launch_superpose_v<RL, W, true>(s, xyz, n_frames, n_atoms, group, idx, n_sel,        \
                                           ref_sel, stats, translate, rot_out, rmsd_out)        \
         : launch_superpose_v<RL, W, false>(s, xyz, n_frames, n_atoms, group, idx, n_sel,       \
                                            ref_sel, stats, translate, rot_out, rmsd_out))
    if (waves == 4) return HR_SUP(kWave, 4);
    if (waves == 2) return HR_SUP(kWave, 2);
    return rl == 64   ? HR_SUP(64, 1)
           : rl == 32 ? HR_SUP(32, 1)
           : rl == 16 ? HR_SUP(16, 1)
           : rl == 8  ? HR_SUP(8, 1)
                      : HR_SUP(4, 1);
#undef HR_SUP
}

int prep_ref(hipStream_t s, const float* ref, const int* ref_idx, int n_sel, int axis_rowstride,
             void* workspace, float** ref_sel, double** stats) {
    char* ws = static_cast<char*>(workspace);
    *stats = reinterpret_cast<double*>(ws);
    *ref_sel = reinterpret_cast<float*>(ws + kRefOffset);
    hipLaunchKernelGGL(ref_prep_kernel, dim3(1), dim3(kBlock), 0, s, ref, ref_idx, n_sel,
                       axis_rowstride, *ref_sel, *stats);
    return launch_status("ref_prep_kernel");
}


// Align/displace: RMS displacement of every frame's displacement set,
// rotated by its fitting rotation R_f (x R_f, about the origin), from the
// reference displacement set, in FP64; one wave per frame.  Also writes
// R_f^T, the rotation taking the reference onto frame f, as the reference's
// getMultipleAlignDisplaceRMSDs_atom_major returns it (rmsd/_rmsd.pyx:744-758
// with rot_msd_atom_major, rmsd/src/rotation_generic.h:47-102).
__global__ __launch_bounds__(kBlock) void rot_msd_kernel(const float* __restrict__ displ,
                                                         long long n_frames, int displ_stride,
                                                         int n_displ,
                                                         const float* __restrict__ displ_ref,
                                                         const float* __restrict__ rot,
                                                         float* __restrict__ out,
                                                         float* __restrict__ rot_t) {
    const int lane = threadIdx.x & (kWave - 1);
    const long long n_waves = (long long)gridDim.x * kWavesPerBlock;
    for (long long f = (long long)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; f < n_frames;
         f += n_waves) {
        double R[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) R[i] = (double)rot[9 * f + i];
        const float* fr = displ + f * 3LL * displ_stride;
        double acc = 0.0;
        for (int a = lane; a < n_displ; a += kWave) {
            const double x = fr[3 * a], y = fr[3 * a + 1], z = fr[3 * a + 2];
            const double dx = x * R[0] + y * R[3] + z * R[6] - (double)displ_ref[3 * a];
            const double dy = x * R[1] + y * R[4] + z * R[7] - (double)displ_ref[3 * a + 1];
            const double dz = x * R[2] + y * R[5] + z * R[8] - (double)displ_ref[3 * a + 2];
            acc += dx * dx + dy * dy + dz * dz;
        }
        acc = wave_sum(acc);
        if (lane == 0) out[f] = (float)sqrt(acc / n_displ);
        if (rot_t && lane < 9) rot_t[9 * f + lane] = rot[9 * f + 3 * (lane % 3) + lane / 3];
    }
}

// Centroid (FP64) of every frame's selection; one wave per frame.
__global__ __launch_bounds__(kBlock) void centroid_kernel(const float* __restrict__ xyz,
                                                          long long n_frames, int n_atoms,
                                                          const int* __restrict__ idx, int n_sel,
                                                          double* __restrict__ mu) {
    const int lane = threadIdx.x & (kWave - 1);
    const long long n_waves = (long long)gridDim.x * kWavesPerBlock;
    for (long long f = (long long)blockIdx.x * kWavesPerBlock + threadIdx.x / kWave; f < n_frames;
         f += n_waves) {
        const float* fr = xyz + f * 3LL * n_atoms;
        double sx = 0.0, sy = 0.0, sz = 0.0;
        for (int j = lane; j < n_sel; j += kWave) {
            const int a = idx ? idx[j] : j;
            sx += fr[3 * a];
            sy += fr[3 * a + 1];
            sz += fr[3 * a + 2];
        }
        sx = wave_sum(sx);
        sy = wave_sum(sy);
        sz = wave_sum(sz);
        if (lane == 0) {
            mu[3 * f] = sx / n_sel;
            mu[3 * f + 1] = sy / n_sel;
            mu[3 * f + 2] = sz / n_sel;
        }
    }
}

// RMSF, pass 1: thread = selected atom, block row = chunk of frames.  The
// displaced coordinate of frame f is (x - mu_f) R_f, with mu_f = 0 unless
// the selections are centred and R_f = I for frames already aligned.  Sums
// of d = displaced - pivot (the atom's displaced coordinate in frame 0) and
// of |d|^2 in FP64, so E|d|^2 - |E d|^2 does not cancel far from the origin.
// Bound by HBM: 480 MB (20,000 frames of 2,000 atoms, every line of a 75 %
// selection) in 99 us, 4.85 TB/s.
template <int kEach>
__global__ __launch_bounds__(kBlock) void rmsf_accum_kernel(
    const float* __restrict__ xyz, long long n_frames, int n_atoms, const int* __restrict__ idx,
    int n_sel, const float* __restrict__ rot, const double* __restrict__ mu, int n_chunks,
    double* __restrict__ partial) {
    const int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n_sel) return;
    const int a = idx ? idx[j] : j;
    const long long f0 = (long long)blockIdx.y * n_frames / n_chunks;
    const long long f1 = (long long)(blockIdx.y + 1) * n_frames / n_chunks;
    const float* p0 = xyz + 3LL * a;
    auto displaced = [&](long long f, float ax, float ay, float az, double& x, double& y,
                         double& z) {
        double px = ax, py = ay, pz = az;
        if (mu) {
            px -= mu[3 * f];
            py -= mu[3 * f + 1];
            pz -= mu[3 * f + 2];
        }
        if (rot) {
            const float* R = rot + 9 * f;
            x = px * R[0] + py * R[3] + pz * R[6];
            y = px * R[1] + py * R[4] + pz * R[7];
            z = px * R[2] + py * R[5] + pz * R[8];
        } else {
            x = px;
            y = py;
            z = pz;
        }
    };
    double qx, qy, qz;
    displaced(0, p0[0], p0[1], p0[2], qx, qy, qz);
    double sx = 0.0, sy = 0.0, sz = 0.0, ss = 0.0;
    // the loads of kEach frames are in flight together (the chunk's last frame
    // again past its end)
    const long long stride = 3LL * n_atoms;
    for (long long f = f0; f < f1; f += kEach) {
        float ax[kEach], ay[kEach], az[kEach];
#pragma unroll
        for (int t = 0; t < kEach; ++t) {
            const float* p = p0 + min(f + t, f1 - 1) * stride;
            ax[t] = p[0];
            ay[t] = p[1];
            az[t] = p[2];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < kEach; ++t) {
            double x, y, z;
            displaced(min(f + t, f1 - 1), ax[t], ay[t], az[t], x, y, z);
            if (f + t < f1) {
                x -= qx;
                y -= qy;
                z -= qz;
                sx += x;
                sy += y;
                sz += z;
                ss += x * x + y * y + z * z;
            }
        }
    }
    double* o = partial + ((size_t)blockIdx.y * n_sel + j) * 4;
    o[0] = sx;
    o[1] = sy;
    o[2] = sz;
    o[3] = ss;
}

// RMSF, pass 2: per atom, sum the chunks; sqrt(E|d|^2 - |E d|^2).  A
// workgroup takes 16 atoms, whose four sums are 64 consecutive doubles of
// every chunk, one a lane; its 16 waves take every 16th chunk each, four
// loads in flight, and meet in LDS.  (With one thread per atom walking all
// chunks, six workgroups did this in 227 us for 1,500 atoms, more than the
// two passes over 20,000 frames; now 6.6 us.)
constexpr int kFinishWaves = 16;
constexpr int kFinishAtoms = kWave / 4;

__global__ __launch_bounds__(kFinishWaves * kWave) void rmsf_finish_kernel(
    const double* __restrict__ partial, int n_chunks, int n_sel, long long n_frames,
    float* __restrict__ out) {
    __shared__ double s_sum[kFinishWaves][kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const size_t row = 4 * (size_t)n_sel;
    const size_t col = min((size_t)blockIdx.x * kWave + lane, row - 1);
    double sum = 0.0;
    constexpr int kEach = 4;
    for (int c0 = w; c0 < n_chunks; c0 += kEach * kFinishWaves) {
        double v[kEach];
#pragma unroll
        for (int t = 0; t < kEach; ++t)
            v[t] = partial[(size_t)min(c0 + t * kFinishWaves, n_chunks - 1) * row + col];
#pragma unroll
        for (int t = 0; t < kEach; ++t)
            if (c0 + t * kFinishWaves < n_chunks) sum += v[t];
    }
    s_sum[w][lane] = sum;
    __syncthreads();
    if (w) return;
#pragma unroll
    for (int i = 1; i < kFinishWaves; ++i) sum += s_sum[i][lane];
    // lanes 4 a .. 4 a + 3: the sums of d's components and of |d|^2
    const double mean = sum / (double)n_frames;
    double m2 = (lane & 3) == 3 ? 0.0 : mean * mean;
    m2 += __shfl_xor(m2, 1, kWave);
    m2 += __shfl_xor(m2, 2, kWave);
    const int j = blockIdx.x * kFinishAtoms + lane / 4;
    if ((lane & 3) == 3 && j < n_sel) {
        const double msf = mean - m2;
        out[j] = (float)sqrt(msf > 0.0 ? msf : 0.0);
    }
}

// The same for up to kFewChunks chunks (few frames or very many atoms), a
// thread per atom: 16 waves with at most one chunk each are mostly launches
// (us a call with 16 waves / a thread per atom: 3 frames of 50,000 atoms without
// a fit 13.9 / 10.2, with one 508 / 454; 10 frames of 10,000 118 / 116; 50 of
// 50,000 803 / 806.  With 20 chunks, 20 frames of 3,000 atoms: 49 / 51).
constexpr int kFewChunks = 16;

__global__ __launch_bounds__(kBlock) void rmsf_finish_few_kernel(
    const double* __restrict__ partial, int n_chunks, int n_sel, long long n_frames,
    float* __restrict__ out) {
    const int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n_sel) return;
    double s[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c = 0; c < n_chunks; ++c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += partial[((size_t)c * n_sel + j) * 4 + e];
    }
    const double n = (double)n_frames, mx = s[0] / n, my = s[1] / n, mz = s[2] / n;
    const double msf = s[3] / n - (mx * mx + my * my + mz * mz);
    out[j] = (float)sqrt(msf > 0.0 ? msf : 0.0);
}

// Frame chunks of the RMSF accumulation: about 2,048 workgroups in all (eight
// a CU, as many as are resident), at most 1,024 chunks and never more chunks
// than frames (sizes the workspace, so it depends on the problem only).
constexpr int kRmsfGroups = 2048, kRmsfMaxChunks = 1024;

int rmsf_chunks(long long n_frames, int n_sel) {
    const long long atom_blocks = (n_sel + kBlock - 1) / kBlock;
    long long c = (kRmsfGroups + atom_blocks - 1) / atom_blocks;
    if (c > kRmsfMaxChunks) c = kRmsfMaxChunks;
    if (c > n_frames) c = n_frames;
    return (int)(c < 1 ? 1 : c);
}

// Partial sums (of four doubles) to reserve for rmsf_chunks(n_frames, n_sel) *
// n_sel.  That product falls where another block of atoms takes chunks away
// (1,024 x 512 atoms, 683 x 513); with b blocks it is below n_sel (kRmsfGroups /
// b + 1) <= kRmsfGroups kBlock + n_sel, and this bound grows with both sizes, so
// that a workspace for many atoms serves fewer.
size_t rmsf_partials(long long n_frames, int n_sel) {
    const size_t chunks = (size_t)std::min(n_frames, (long long)kRmsfMaxChunks);
    return std::min(chunks * n_sel, (size_t)kRmsfGroups * kBlock + n_sel);
}

// Default chunk of hr_superpose's two kernels (MiB of coordinates);
// HR_TUNE_SUPERPOSE_CHUNK_MIB overrides it.  They serve frames too long for one
// pass and separate alignment arrays.  Us a call with chunks of 256 MiB / 1 GiB /
// all frames at once: 25,000 frames x 8,000 atoms (2.4 GB) 2,017 / 1,803 / 1,670,
// 8,000 x 25,000 3,194 / 2,097 / 1,751, 10,000 x 8,000 with an alignment array
// 1,078 / 733 / 734, 100,000 x 2,000 with one 1,543 / 1,398 / 1,365: each chunk pays
// the two kernels' ramp and drain, and the rotation gains nothing from a chunk
// that is still cached.  (1 GiB was the better by 3 % where all frames of 2,000
// atoms took this path; at the sizes that are left one chunk would be.)
constexpr int kSuperposeChunkMiB = 1024;

}  // namespace
}  // namespace hr

using namespace hr;

extern "C" {

size_t hr_rmsd_workspace_bytes(int32_t n_sel) {
    return kRefOffset + (size_t)(n_sel > 0 ? n_sel : 0) * 3 * sizeof(float);
}

int hr_center_and_trace(float* xyz, float* traces, int64_t n_frames, int32_t n_atoms,
                        void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms > 0, "invalid sizes n_frames=%lld n_atoms=%d",
               (long long)n_frames, n_atoms);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(xyz != nullptr, "xyz is NULL");
    const DeviceInfo* d = current_device();
    if (!d) return HR_ERR_HIP;
    long long waves = (long long)d->cu_count * kDefaultWavesPerCu;
    if (waves > n_frames) waves = n_frames;
    const int blocks = (int)((waves + kWavesPerBlock - 1) / kWavesPerBlock);
    hipLaunchKernelGGL(center_kernel, dim3(blocks), dim3(kBlock), 0, (hipStream_t)stream, xyz,
                       traces, (long long)n_frames, n_atoms);
    return launch_status("center_kernel");
}

int hr_rmsd_prepare_reference(const float* ref_frame, const int32_t* ref_idx, int32_t n_sel,
                              void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_sel > 0, "invalid n_sel=%d", n_sel);
    HR_REQUIRE(ref_frame && workspace, "NULL pointer argument");
    float* ref_sel;
    double* stats;
    return prep_ref((hipStream_t)stream, ref_frame, ref_idx, n_sel, 0, workspace, &ref_sel,
                    &stats);
}

int hr_rmsd_one_vs_all_prepared(const float* target, int64_t n_frames, int32_t n_atoms_total,
                                const int32_t* atom_idx, int32_t n_sel, int64_t self_frame,
                                float* out, const void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms_total > 0 && n_sel > 0,
               "invalid sizes n_frames=%lld n_atoms=%d n_sel=%d", (long long)n_frames,
               n_atoms_total, n_sel);
    HR_REQUIRE(atom_idx != nullptr || n_sel == n_atoms_total,
               "n_sel (%d) must equal n_atoms_total (%d) without atom_idx", n_sel, n_atoms_total);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(target && out && workspace, "NULL pointer argument");
    const char* ws = static_cast<const char*>(workspace);
    const double* stats = reinterpret_cast<const double*>(ws);
    const float* ref_sel = reinterpret_cast<const float*>(ws + kRefOffset);
    hipStream_t s = (hipStream_t)stream;
    if (!atom_idx && n_sel <= kShortAtoms)
        return launch_short<false>(s, target, n_frames, n_sel, ref_sel, stats, self_frame, out);
    Launch l;
    int rc = plan<Kind::Rmsd>(n_sel, atom_idx != nullptr, &l);
    if (rc) return rc;
    const long long stride = 3LL * n_atoms_total;
    if (atom_idx)
        return launch_frames<Kind::Rmsd, false, true>(l, s, target, n_frames, stride, 0, atom_idx,
                                                      n_sel, ref_sel, stats, self_frame, out,
                                                      nullptr, nullptr);
    return launch_frames<Kind::Rmsd, false, false>(l, s, target, n_frames, stride, 0, nullptr,
                                                   n_sel, ref_sel, stats, self_frame, out, nullptr,
                                                   nullptr);
}

int hr_rmsd_one_vs_all(const float* target, int64_t n_frames, int32_t n_atoms_total,
                       const int32_t* atom_idx, int32_t n_sel, const float* ref_frame,
                       const int32_t* ref_idx, int64_t self_frame, float* out, void* workspace,
                       void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms_total > 0 && n_sel > 0,
               "invalid sizes n_frames=%lld n_atoms=%d n_sel=%d", (long long)n_frames,
               n_atoms_total, n_sel);
    HR_REQUIRE(atom_idx != nullptr || n_sel == n_atoms_total,
               "n_sel (%d) must equal n_atoms_total (%d) without atom_idx", n_sel, n_atoms_total);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(target && ref_frame && out && workspace, "NULL pointer argument");
    int rc = hr_rmsd_prepare_reference(ref_frame, ref_idx, n_sel, workspace, stream);
    if (rc) return rc;
    return hr_rmsd_one_vs_all_prepared(target, n_frames, n_atoms_total, atom_idx, n_sel,
                                       self_frame, out, workspace, stream);
}

int hr_rmsd_one_vs_all_axis_major(const float* target, int64_t n_frames, int32_t n_atoms,
                                  int32_t rowstride, const float* ref_frame_axis,
                                  int32_t ref_rowstride, int64_t self_frame, float* out,
                                  void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms > 0 && rowstride >= n_atoms && ref_rowstride >= n_atoms,
               "invalid sizes n_frames=%lld n_atoms=%d rowstride=%d ref_rowstride=%d",
               (long long)n_frames, n_atoms, rowstride, ref_rowstride);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(target && ref_frame_axis && out && workspace, "NULL pointer argument");
    hipStream_t s = (hipStream_t)stream;
    float* ref_sel;
    double* stats;
    int rc = prep_ref(s, ref_frame_axis, nullptr, n_atoms, ref_rowstride, workspace, &ref_sel,
                      &stats);
    if (rc) return rc;
    Launch l;
    if ((rc = plan<Kind::Rmsd>(n_atoms, false, &l))) return rc;
    return launch_frames<Kind::Rmsd, true, false>(l, s, target, n_frames, 3LL * rowstride,
                                                  rowstride, nullptr, n_atoms, ref_sel, stats,
                                                  self_frame, out, nullptr, nullptr);
}

int hr_rmsd_nosuperpose(const float* target, int64_t n_frames, int32_t n_atoms_total,
                        const int32_t* atom_idx, int32_t n_sel, const float* ref_frame,
                        const int32_t* ref_idx, float* out, void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms_total > 0 && n_sel > 0,
               "invalid sizes n_frames=%lld n_atoms=%d n_sel=%d", (long long)n_frames,
               n_atoms_total, n_sel);
    HR_REQUIRE(atom_idx != nullptr || n_sel == n_atoms_total,
               "n_sel (%d) must equal n_atoms_total (%d) without atom_idx", n_sel, n_atoms_total);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(target && ref_frame && out && workspace, "NULL pointer argument");
    hipStream_t s = (hipStream_t)stream;
    float* ref_sel;
    double* stats;
    int rc = prep_ref(s, ref_frame, ref_idx, n_sel, 0, workspace, &ref_sel, &stats);
    if (rc) return rc;
    Launch l;
    if ((rc = plan<Kind::NoSuperpose>(n_sel, atom_idx != nullptr, &l))) return rc;
    const long long stride = 3LL * n_atoms_total;
    if (atom_idx)
        return launch_frames<Kind::NoSuperpose, false, true>(l, s, target, n_frames, stride, 0,
                                                             atom_idx, n_sel, ref_sel, stats, -1,
                                                             out, nullptr, nullptr);
    return launch_frames<Kind::NoSuperpose, false, false>(l, s, target, n_frames, stride, 0,
                                                          nullptr, n_sel, ref_sel, stats, -1, out,
                                                          nullptr, nullptr);
}

size_t hr_superpose_workspace_bytes(int64_t n_frames, int32_t n_sel) {
    const size_t nf = (size_t)(n_frames > 0 ? n_frames : 0);
    size_t b = hr_rmsd_workspace_bytes(n_sel);
    b = (b + 255) & ~(size_t)255;
    b += nf * 3 * sizeof(double);  // per-frame centroids
    b = (b + 255) & ~(size_t)255;
    b += nf * 9 * sizeof(float);  // rotations when the caller passes none
    return b;
}

int hr_superpose(float* xyz, int64_t n_frames, int32_t n_atoms, const float* align_xyz,
                 int32_t n_align_atoms, const int32_t* atom_idx, int32_t n_sel,
                 const float* ref_frame, const int32_t* ref_idx, int32_t translate,
                 float* rot_out, float* rmsd_out, void* workspace, void* stream) {
    clear_error();
    if (!align_xyz) n_align_atoms = n_atoms;
    HR_REQUIRE(n_frames >= 0 && n_atoms > 0 && n_align_atoms > 0 && n_sel > 0,
               "invalid sizes n_frames=%lld n_atoms=%d n_align_atoms=%d n_sel=%d",
               (long long)n_frames, n_atoms, n_align_atoms, n_sel);
    HR_REQUIRE(atom_idx != nullptr || n_sel == n_align_atoms,
               "n_sel (%d) must equal n_align_atoms (%d) without atom_idx", n_sel, n_align_atoms);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(xyz && ref_frame && workspace, "NULL pointer argument");
    hipStream_t s = (hipStream_t)stream;
    char* ws = static_cast<char*>(workspace);
    size_t off = (hr_rmsd_workspace_bytes(n_sel) + 255) & ~(size_t)255;
    double* mu = reinterpret_cast<double*>(ws + off);
    off += (size_t)n_frames * 3 * sizeof(double);
    off = (off + 255) & ~(size_t)255;
    float* rot = rot_out ? rot_out : reinterpret_cast<float*>(ws + off);
    float* ref_sel;
    double* stats;
    int rc = prep_ref(s, ref_frame, ref_idx, n_sel, 0, workspace, &ref_sel, &stats);
    if (rc) return rc;
    Launch l;
    if ((rc = plan<Kind::Fit>(n_sel, atom_idx != nullptr, &l))) return rc;
    if (!align_xyz) {
        bool done = false;
        rc = superpose_one_pass(s, xyz, n_frames, n_atoms, atom_idx, n_sel, ref_sel, stats,
                                (int)(translate != 0), rot_out, rmsd_out, &done);
        if (rc || done) return rc;
    }
    const float* fit = align_xyz ? align_xyz : xyz;
    const long long stride = 3LL * n_align_atoms;
    const DeviceInfo* d = current_device();
    // Fit and rotate chunk by chunk (kSuperposeChunkMiB); every frame's
    // rotation depends on that frame alone, so results equal one pass.
    const long long frame_bytes = 12LL * n_atoms;
    const int mib = tuning(HR_TUNE_SUPERPOSE_CHUNK_MIB) ? tuning(HR_TUNE_SUPERPOSE_CHUNK_MIB)
                                                        : kSuperposeChunkMiB;
    long long chunk = ((long long)mib << 20) / frame_bytes;
    if (chunk < 1) chunk = 1;
    for (long long f0 = 0; f0 < n_frames; f0 += chunk) {
        const long long nf = n_frames - f0 < chunk ? n_frames - f0 : chunk;
        float* out_f = rmsd_out ? rmsd_out + f0 : nullptr;
        if (atom_idx)
            rc = launch_frames<Kind::Fit, false, true>(l, s, fit + f0 * stride, nf, stride, 0,
                                                       atom_idx, n_sel, ref_sel, stats, -1, out_f,
                                                       rot + 9 * f0, mu + 3 * f0);
        else
            rc = launch_frames<Kind::Fit, false, false>(l, s, fit + f0 * stride, nf, stride, 0,
                                                        nullptr, n_sel, ref_sel, stats, -1, out_f,
                                                        rot + 9 * f0, mu + 3 * f0);
        if (rc) return rc;
        long long blocks = (long long)d->cu_count * 8;
        if (blocks > nf) blocks = nf;
        hipLaunchKernelGGL(apply_kernel, dim3((int)blocks), dim3(kBlock), 0, s,
                           xyz + f0 * 3LL * n_atoms, nf, n_atoms, rot + 9 * f0, mu + 3 * f0, stats,
                           (double)n_sel, (int)(translate != 0));
        if ((rc = launch_status("apply_kernel"))) return rc;
    }
    return HR_OK;
}

size_t hr_align_displace_workspace_bytes(int64_t n_frames, int32_t n_align) {
    return hr_superpose_workspace_bytes(n_frames, n_align);
}

int hr_rmsd_align_displace(const float* align, int64_t n_frames, int32_t align_stride,
                           int32_t n_align, const float* align_ref, const float* displ,
                           int32_t displ_stride, int32_t n_displ, const float* displ_ref,
                           float* rmsd_out, float* rot_out, void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_align > 0 && n_displ > 0 && align_stride >= n_align &&
                   displ_stride >= n_displ,
               "invalid sizes n_frames=%lld n_align=%d (stride %d) n_displ=%d (stride %d)",
               (long long)n_frames, n_align, align_stride, n_displ, displ_stride);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(align && align_ref && displ && displ_ref && rmsd_out && workspace,
               "NULL pointer argument");
    hipStream_t s = (hipStream_t)stream;
    char* ws = static_cast<char*>(workspace);
    size_t off = (hr_rmsd_workspace_bytes(n_align) + 255) & ~(size_t)255;
    double* mu = reinterpret_cast<double*>(ws + off);
    off += (size_t)n_frames * 3 * sizeof(double);
    off = (off + 255) & ~(size_t)255;
    float* rot = reinterpret_cast<float*>(ws + off);
    float* ref_sel;
    double* stats;
    int rc = prep_ref(s, align_ref, nullptr, n_align, 0, workspace, &ref_sel, &stats);
    if (rc) return rc;
    Launch l;
    if ((rc = plan<Kind::Fit>(n_align, false, &l))) return rc;
    rc = launch_frames<Kind::Fit, false, false>(l, s, align, n_frames, 3LL * align_stride, 0,
                                                nullptr, n_align, ref_sel, stats, -1, nullptr,
                                                rot, mu);
    if (rc) return rc;
    const DeviceInfo* d = current_device();
    long long blocks = (long long)d->cu_count * 8;
    const long long by_work = (n_frames + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks > by_work) blocks = by_work;
    hipLaunchKernelGGL(rot_msd_kernel, dim3((int)blocks), dim3(kBlock), 0, s, displ,
                       (long long)n_frames, displ_stride, n_displ, displ_ref, rot, rmsd_out,
                       rot_out);
    return launch_status("rot_msd_kernel");
}

size_t hr_rmsf_workspace_bytes(int64_t n_frames, int32_t n_sel) {
    size_t b = hr_superpose_workspace_bytes(n_frames, n_sel);
    b = (b + 255) & ~(size_t)255;
    b += rmsf_partials(n_frames > 0 ? n_frames : 1, n_sel > 0 ? n_sel : 0) * 4 * sizeof(double);
    return b;
}

int hr_rmsf(const float* xyz, int64_t n_frames, int32_t n_atoms, const int32_t* atom_idx,
            int32_t n_sel, const float* ref_frame, const int32_t* ref_idx, int32_t center,
            float* out, void* workspace, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames > 0 && n_atoms > 0 && n_sel > 0,
               "invalid sizes n_frames=%lld n_atoms=%d n_sel=%d", (long long)n_frames, n_atoms,
               n_sel);
    HR_REQUIRE(atom_idx != nullptr || n_sel == n_atoms,
               "n_sel (%d) must equal n_atoms (%d) without atom_idx", n_sel, n_atoms);
    HR_REQUIRE(xyz && out && workspace, "NULL pointer argument");
    hipStream_t s = (hipStream_t)stream;
    char* ws = static_cast<char*>(workspace);
    size_t off = (hr_rmsd_workspace_bytes(n_sel) + 255) & ~(size_t)255;
    double* mu = reinterpret_cast<double*>(ws + off);
    off += (size_t)n_frames * 3 * sizeof(double);
    off = (off + 255) & ~(size_t)255;
    float* rot = reinterpret_cast<float*>(ws + off);
    off += (size_t)n_frames * 9 * sizeof(float);
    off = (off + 255) & ~(size_t)255;
    double* partial = reinterpret_cast<double*>(ws + off);
    const DeviceInfo* d = current_device();
    if (!d) return HR_ERR_HIP;
    int rc;
    if (ref_frame) {
        float* ref_sel;
        double* stats;
        if ((rc = prep_ref(s, ref_frame, ref_idx, n_sel, 0, workspace, &ref_sel, &stats)))
            return rc;
        Launch l;
        if ((rc = plan<Kind::Fit>(n_sel, atom_idx != nullptr, &l))) return rc;
        if (atom_idx)
            rc = launch_frames<Kind::Fit, false, true>(l, s, xyz, n_frames, 3LL * n_atoms, 0,
                                                       atom_idx, n_sel, ref_sel, stats, -1,
                                                       nullptr, rot, mu);
        else
            rc = launch_frames<Kind::Fit, false, false>(l, s, xyz, n_frames, 3LL * n_atoms, 0,
                                                        nullptr, n_sel, ref_sel, stats, -1,
                                                        nullptr, rot, mu);
        if (rc) return rc;
    } else if (center) {
        long long blocks = (long long)d->cu_count * 8;
        const long long by_work = (n_frames + kWavesPerBlock - 1) / kWavesPerBlock;
        if (blocks > by_work) blocks = by_work;
        hipLaunchKernelGGL(centroid_kernel, dim3((int)blocks), dim3(kBlock), 0, s, xyz,
                           (long long)n_frames, n_atoms, atom_idx, n_sel, mu);
        if ((rc = launch_status("centroid_kernel"))) return rc;
    }
    const int n_chunks = rmsf_chunks(n_frames, n_sel);
    const int atom_blocks = (n_sel + kBlock - 1) / kBlock;
    // chunks of one frame do no more than that frame
    const auto accum = n_chunks < n_frames ? rmsf_accum_kernel<8> : rmsf_accum_kernel<1>;
    hipLaunchKernelGGL(accum, dim3(atom_blocks, n_chunks), dim3(kBlock), 0, s, xyz,
                       (long long)n_frames, n_atoms, atom_idx, n_sel, ref_frame ? rot : nullptr,
                       center ? mu : nullptr, n_chunks, partial);
    if ((rc = launch_status("rmsf_accum_kernel"))) return rc;
    const bool few = n_chunks <= kFewChunks;
    hipLaunchKernelGGL(few ? rmsf_finish_few_kernel : rmsf_finish_kernel,
                       dim3(few ? atom_blocks : (n_sel + kFinishAtoms - 1) / kFinishAtoms),
                       dim3(few ? kBlock : kFinishWaves * kWave), 0, s, partial, n_chunks, n_sel,
                       (long long)n_frames, out);
    return launch_status("rmsf_finish_kernel");
}

}  // extern "C"
