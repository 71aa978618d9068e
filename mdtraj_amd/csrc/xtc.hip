// XTC ingestion (gfx950): GROMACS-compressed trajectory bytes, resident in
// HBM, decoded into float32 (F, N, 3) coordinates in HBM, so serving pools
// and one-vs-all queries read a file without a host-side decode.
//
// Format (the reference's reader: formats/xtc/src/xdrfile_xtc.c:41-90 for
// the frame header and box, formats/xtc/src/xdrfile.c:778-1000 for the
// coordinates): big-endian 32-bit words; a frame is magic 1995, natoms,
// step, time, nine box floats, natoms again, then either 3 natoms raw
// floats (natoms <= 9) or precision, minint[3], maxint[3], smallidx, a byte
// count and that many bytes of bit stream (padded to a word).  The stream
// holds, per "large" atom, its integer coordinates less minint (one
// mixed-radix number of sizeofints(maxint - minint + 1) bits, or three
// fields when a range exceeds 2^24), a flag bit, an optional 5-bit run code
// (run length in floats, plus a -1/0/+1 change of smallidx), and the run's
// small atoms as deltas (one mixed-radix number of smallidx bits each).
//
// Frames are independent, so the host walks the headers once (hr_xtc_scan,
// the frame index) and the device decodes one frame per row of 4 to 64 lanes:
// where a group of atoms starts depends on the flags of all before it, but
// once the starts are known the groups decode side by side.  Every read is bounded by the frame's
// own bytes and every write by its atom count; a malformed frame ends with a
// non-zero status word (HR_XTC_*) instead of an out-of-range access.
#include <string.h>

#include <type_traits>

#include "common.h"

namespace hr {
namespace {

constexpr int kXtcMagic = 1995;
constexpr int kFirstIdx = 9;
// Sizes of the small-delta digits by smallidx (the format's table: the
// value at index i needs i bits for three digits).
__constant__ int kMagicInts[] = {
    0,       0,       0,       0,       0,       0,       0,       0,       0,       8,
    10,      12,      16,      20,      25,      32,      40,      50,      64,      80,
    101,     128,     161,     203,     256,     322,     406,     512,     645,     812,
    1024,    1290,    1625,    2048,    2580,    3250,    4096,    5060,    6501,    8192,
    10321,   13003,   16384,   20642,   26007,   32768,   41285,   52015,   65536,   82570,
    104031,  131072,  165140,  208063,  262144,  330280,  416127,  524287,  660561,  832255,
    1048576, 1321122, 1664510, 2097152, 2642245, 3329021, 4194304, 5284491, 6658042, 8388607,
    10568983, 13316085, 16777216};
constexpr int kLastIdx = 73;  // entries in kMagicInts
static_assert(sizeof(kMagicInts) / sizeof(kMagicInts[0]) == kLastIdx, "table size");

__host__ __device__ __forceinline__ uint32_t be32(const unsigned char* p) {
    return ((uint32_t)p[0] << 24) | ((uint32_t)p[1] << 16) | ((uint32_t)p[2] << 8) | p[3];
}

__device__ __forceinline__ uint32_t be32_word(const uint32_t* w) {
    return __builtin_bswap32(*w);
}

// Bit length of v (bits needed for 0 .. v - 1 ... v itself: the format's
// sizeofint, and sizeofints of a product).
__device__ __forceinline__ int bit_length64(uint64_t v) { return v ? 64 - __clzll(v) : 0; }

// floor(v / d) and v mod d of whole numbers held in doubles, v < 2^50 and
// d < 2^25: inv_d is 1 / d taken 2^-51 low, so that the estimate is the
// quotient or one less (the roundings are below 2^-51 together, and the
// quotient below 2^50), and v - q d is exact.
__device__ __forceinline__ double div_whole(double v, double d, double inv_d, double& rem) {
    const double q = floor(v * inv_d);
    const double r = fma(-q, d, v);
    const bool more = r >= d;
    rem = more ? r - d : r;
    return more ? q + 1.0 : q;
}
__device__ __forceinline__ double low_recip(double d) { return (1.0 / d) * (1.0 - 0x1p-51); }

// One frame belongs to a row of R lanes (64 / R frames per wave), and
// goes out in batches of up to R groups (a group: a large atom and its run of
// small ones), each batch in three steps:
//   scan   the groups' bit offsets.  Only the flag bit and the run code of a
//          group decide where the next one starts, so nothing is decoded
//          here.  A clear flag keeps the run length and smallidx, hence the
//          group's length: lane cnt + j of the row looks at the flag of the
//          j-th next group as if all before it were clear, a ballot finds the
//          first set flag, and everything up to and including that group is
//          accepted at once (water: whole batches; a chain whose run changes
//          at every group: one group a step).  The accepted group's place
//          stays in its lane's registers.
//   decode one group per lane: the mixed-radix fields, the deltas' sums, the
//          integers into the row's staging area in LDS.
//   store  the row's floats, consecutive in memory, by all its lanes.
// The frame's words come through a ring in LDS, byte-swapped on the way, with
// the next block's load in flight in registers while a batch is decoded.
// One lane per frame (the first form) decoded every field of a frame in
// series: 10,000 frames x 3,001 atoms of a chain in water took 3,254 us with
// 157 waves on the chip, 322 us here (16-lane rows; the copy rate would allow
// 96 us).  What bounds it is the scan's chain of dependent steps (about 700
// cycles a step: two LDS words, the flag, a ballot, a lane exchange) beside
// the decode's divisions; on a lone wave of 16-lane rows a batch is 3,250
// cycles of scan, 2,170 of decode, 340 of refill.  Packing a group's whole
// outcome into the exchanged word, for fewer but longer-chained instructions a
// step, measured the same or slower (326 us; 20 x 12,000 atoms 324 against
// 290 us).
template <int R>
struct XtcRow {
    static constexpr int kRows = kWave / R;   // frames per wave
    static constexpr int kRing = 16 * R;      // words in the ring, a power of two
    static constexpr int kRingRow = kRing + 4;  // and one more, the first again
    static constexpr int kBlock4 = 4 * R;     // words per block: four a lane
    static constexpr int kCap = 7 * R;        // atoms staged per batch
    static constexpr int kStage = 3 * kCap;   // integers
};
// A group is at most 96 bits of large atom, 6 of flag and run code and ten
// small atoms of 72 bits, and eleven atoms: the ring holds it with a block to
// spare, and so does the staging area.  A batch that finds too few words takes
// no group but is followed by a refill, so the batches end.
constexpr int kMaxGroupBits = 96 + 6 + 10 * 72;
static_assert((XtcRow<4>::kRing - XtcRow<4>::kBlock4) * 32 >= kMaxGroupBits + 64, "ring");
static_assert(XtcRow<4>::kCap >= 11, "staging area");

// Orders the wave's LDS accesses (the workgroup is one wave, whose LDS
// accesses complete in program order; this keeps the compiler from moving
// them).
__device__ __forceinline__ void xtc_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// n bits (1 .. 32) at bit p of a ring whose word 0 is ring word `base`.
template <int kRing>
__device__ __forceinline__ uint32_t ring_bits(const uint32_t* ring, uint32_t base, uint32_t p,
                                              int n) {
    const uint32_t w = (base + (p >> 5)) & (kRing - 1), off = p & 31;
    const uint32_t hi = ring[w], lo = ring[w + 1];  // ring[kRing] repeats ring[0]
    return ((hi << off) | ((lo >> 1) >> (31 - off))) >> (32 - n);
}

// The number whose 8-bit chunks were written least significant first, from
// its field of nbits bits read most significant bit first: the
// a = (nbits - 1) / 8 whole bytes reversed, then the last nbits - 8 a bits.
__device__ __forceinline__ uint32_t chunks_to_number(uint32_t w, int nbits) {
    const int a = (nbits - 1) >> 3, b = nbits - 8 * a;
    const uint32_t v = w & ((1u << b) - 1);
    return a ? (v << (8 * a)) | (__builtin_bswap32(w >> b) >> (32 - 8 * a)) : v;
}

// floor(v / d) and v mod d for v < 2^30 and a quotient below 2^20, d below
// 2^24: inv_d is 1 / d taken 2^-21 low, so that the estimate is the quotient
// or one less whatever the roundings (v's, the reciprocal's and the
// product's, below 2^-21 together).
__device__ __forceinline__ uint32_t div_small(uint32_t v, uint32_t d, float inv_d,
                                              uint32_t& rem) {
    const uint32_t q = (uint32_t)((float)v * inv_d);
    const uint32_t r = v - __umul24(q, d);
    rem = min(r, r - d);  // r - d wraps when r < d
    return q + (r >= d ? 1u : 0u);
}

// Three digits (x, y, z) of one mixed-radix number of nbits (<= 72) bits at
// bit p: z = V mod sz, y = (V / sz) mod sy, x = V / (sz sy) (low 32 bits).
// inv_sz, inv_sy: low_recip(sz) and low_recip(sy).
template <int kRing>
__device__ __forceinline__ void ring_ints3(const uint32_t* ring, uint32_t base, uint32_t p,
                                           int nbits, double sy, double sz, double inv_sz,
                                           double inv_sy, uint32_t (&out)[3]) {
    // whole 32-bit words are four reversed bytes
    uint32_t word[3] = {0u, 0u, 0u};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int n = nbits - 32 * k;
        if (n >= 32)
            word[k] = __builtin_bswap32(ring_bits<kRing>(ring, base, p + 32 * k, 32));
        else if (n > 0)
            word[k] = chunks_to_number(ring_bits<kRing>(ring, base, p + 32 * k, n), n);
    }
    double r, r2;
    if (nbits <= 50) {
        const double q = div_whole(fma((double)word[1], 0x1p32, (double)word[0]), sz, inv_sz, r);
        const double q2 = div_whole(q, sy, inv_sy, r2);
        // the low 32 bits of x (a stream may hold more than the ranges allow)
        out[0] = (uint32_t)(q2 - floor(q2 * 0x1p-32) * 0x1p32);
    } else {
        // long division over digits of 24 bits, most significant first
        double digit[3] = {(double)((word[1] >> 16) | (word[2] << 16)),
                           (double)((word[0] >> 24) | ((word[1] & 0xFFFFu) << 8)),
                           (double)(word[0] & 0xFFFFFFu)};
        r = r2 = 0.0;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            digit[k] = div_whole(fma(r, 0x1p24, digit[k]), sz, inv_sz, r);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            digit[k] = div_whole(fma(r2, 0x1p24, digit[k]), sy, inv_sy, r2);
        out[0] = ((uint32_t)digit[1] << 24) + (uint32_t)digit[2];
    }
    out[2] = (uint32_t)r;
    out[1] = (uint32_t)r2;
}

// Lanes of a frame's row, by the number of frames: in general the narrowest row that
// leaves the chip enough waves.  A step of the scan costs a wave the same
// whatever its rows are, so narrow rows scan more frames for it, but a frame
// alone is done sooner the wider its row (us, rows of 8 / 16 / 32 / 64 lanes):
//     20 x 12,000 atoms   1,087 / 646 / 434 / 290
//  2,000 x 3,001            340 / 226 / 149 / 126
//  4,000 x 3,001            373 / 222 / 177 / 187
// 10,000 x 3,001            412 / 322 / 364 / 398
// 16,000 x 1,000            167 / 166 / 207 / 295
// 60,000 x 43                49 / 70 / 107 / 181
// 90,000 x 600              428 / 493 / 649 / 954
// (one frame per lane, decoded in series: 3,254 us on 10,000 x 3,001).  These are
// streams of a chain in water with long runs, 0.3 groups an atom.  The water
// file that the tests read, written by the reference's encoder, has 0.93 groups
// an atom: 90,000 of its frames (600 atoms) take 789 us in rows of 8, 1,590 with
// one frame per lane.
//
// A frame of a few dozen atoms has too few groups for eight lanes, and many such
// frames leave a wave little to do (us with rows of 4 / 8 lanes, on streams whose
// flags are rarely and always set; with one frame per lane, 500,000 x 12 atoms
// took 181 and 146 us):
//  16,000 x 12 atoms    11 / 10     11 / 10
//  65,536 x 12          19 / 23     19 / 25
//  65,536 x 20          29 / 32     22 / 29
//  80,000 x 20          38 / 38     27 / 33
//  80,000 x 22          41 / 39     29 / 35
// 500,000 x 12          96 / 134    96 / 152
// 500,000 x 22         167 / 187   118 / 171
constexpr int kNarrowAtoms = 20;
constexpr long long kNarrowFrames = 65536;

inline int xtc_row_lanes(long long n_frames, int n_atoms) {
    if (n_atoms <= kNarrowAtoms && n_frames >= kNarrowFrames) return 4;
    return n_frames >= 16000 ? 8 : n_frames >= 6000 ? 16 : n_frames >= 3000 ? 32 : 64;
}

// Frames of up to kTinyAtoms atoms (stored uncompressed, as all of up to nine
// are): four lanes a frame and nothing in LDS, since the decoder's kernel, with
// its ring and eight lanes, holds too few of such short frames (us for 1 M frames
// of 1 / 2 / 3 atoms: 75 / 75 / 86 there, 29 / 34 / 40 here).  Checks and status
// words as in xtc_decode_kernel.
constexpr int kTinyAtoms = 3, kTinyLanes = 4, kTinyBlock = 256;

__global__ __launch_bounds__(kTinyBlock) void xtc_tiny_kernel(
    const unsigned char* __restrict__ data, long long n_bytes,
    const long long* __restrict__ offsets, long long n_frames, int n_atoms,
    float* __restrict__ xyz, float* __restrict__ time, int* __restrict__ step,
    float* __restrict__ box, float* __restrict__ prec, int* __restrict__ status) {
    const int l = threadIdx.x & (kTinyLanes - 1);
    const long long f =
        workgroup_index() * (kTinyBlock / kTinyLanes) + threadIdx.x / kTinyLanes;
    if (f >= n_frames) return;
    const long long beg = offsets[f], end = f + 1 < n_frames ? offsets[f + 1] : n_bytes;
    int st = HR_XTC_OK;
    if (beg < 0 || end > n_bytes || end - beg < 56 || (beg & 3)) {
        st = HR_XTC_TRUNCATED;
    } else {
        const uint32_t* pw = reinterpret_cast<const uint32_t*>(data + beg);
        const int magic = (int)be32_word(pw), natoms = (int)be32_word(pw + 1);
        const int lsize = (int)be32_word(pw + 13);
        if (l == 0) {
            step[f] = (int)be32_word(pw + 2);
            time[f] = __uint_as_float(be32_word(pw + 3));
        }
        for (int k = l; k < 9; k += kTinyLanes)
            box[9 * f + k] = __uint_as_float(be32_word(pw + 4 + k));
        if (magic != kXtcMagic) {
            st = HR_XTC_BAD_MAGIC;
        } else if (natoms != n_atoms || lsize != n_atoms) {
            st = HR_XTC_ATOMS;
        } else {
            if (l == 0) prec[f] = 0.0f;
            if (14 + 3 * n_atoms > (end - beg) / 4) {
                st = HR_XTC_TRUNCATED;
            } else {
                for (int k = l; k < 3 * n_atoms; k += kTinyLanes)
                    xyz[3 * n_atoms * f + k] = __uint_as_float(be32_word(pw + 14 + k));
            }
        }
    }
    if (l == 0) status[f] = st;
}

// offsets[f] .. offsets[f + 1] (or n_bytes) bound frame f's bytes; the host
// has checked magic and sizes when it built them.
template <int R>
__global__ __launch_bounds__(kWave, 4) void xtc_decode_kernel(
    const unsigned char* __restrict__ data, long long n_bytes,
    const long long* __restrict__ offsets, long long n_frames, int n_atoms,
    float* __restrict__ xyz, float* __restrict__ time, int* __restrict__ step,
    float* __restrict__ box, float* __restrict__ prec, int* __restrict__ status) {
    using T = XtcRow<R>;
    constexpr int kRing = T::kRing;
    __shared__ __align__(16) uint32_t s_ring[T::kRows * T::kRingRow];
    __shared__ __align__(16) int s_stage[T::kRows * T::kStage];
    __shared__ int s_magic[kLastIdx];
    const int lane = threadIdx.x, l = lane & (R - 1), row = R == kWave ? 0 : lane / R;
    // wide rows are for few frames (xtc_row_lanes), which one dimension holds
    const long long f = (R > 8 ? (long long)blockIdx.x : workgroup_index()) * T::kRows + row;
    for (int i = lane; i < kLastIdx; i += kWave) s_magic[i] = kMagicInts[i];
    xtc_wave_sync();
    uint32_t* ring = s_ring + row * T::kRingRow;
    int* stage = s_stage + row * T::kStage;

    // -- the header, by every lane of the row
    const bool exists = f < n_frames;
    const bool lead = exists && l == 0;
    const long long beg = exists ? offsets[f] : 0;
    const long long end = exists ? (f + 1 < n_frames ? offsets[f + 1] : n_bytes) : 0;
    float* out = xyz + (exists ? f : 0) * 3 * n_atoms;
    bool live = exists;  // uniform over the row from here on
    int st = HR_XTC_OK;
    if (beg < 0 || end > n_bytes || end - beg < 56 || (beg & 3)) {
        st = HR_XTC_TRUNCATED;
        live = false;
    }
    const uint32_t* pw = reinterpret_cast<const uint32_t*>(data + (live ? beg : 0));
    const long long avail_words = (end - beg) / 4;  // words of this frame
    if (live) {
        const int magic = (int)be32_word(pw), natoms = (int)be32_word(pw + 1);
        const int lsize = (int)be32_word(pw + 13);
        if (l == 0) {
            step[f] = (int)be32_word(pw + 2);
            time[f] = __uint_as_float(be32_word(pw + 3));
        }
        for (int k = l; k < 9; k += R) box[9 * f + k] = __uint_as_float(be32_word(pw + 4 + k));
        if (magic != kXtcMagic) st = HR_XTC_BAD_MAGIC;
        else if (natoms != n_atoms || lsize != n_atoms) st = HR_XTC_ATOMS;
        live = st == HR_XTC_OK;
    }
    if (n_atoms <= 9) {  // stored uncompressed
        if (live) {
            if (l == 0) prec[f] = 0.0f;
            if (14 + 3 * n_atoms > avail_words) {
                st = HR_XTC_TRUNCATED;
            } else {
                for (int k = l; k < 3 * n_atoms; k += R)
                    out[k] = __uint_as_float(be32_word(pw + 14 + k));
            }
        }
        if (lead) status[f] = st;
        return;
    }
    int32_t minint[3] = {0, 0, 0};
    uint32_t sizeint[3] = {1u, 1u, 1u};
    int smallidx = kFirstIdx, n_words = 0;
    float inv = 0.0f;
    if (live && avail_words < 23) {
        st = HR_XTC_TRUNCATED;
        live = false;
    }
    if (live) {
        const float precision = __uint_as_float(be32_word(pw + 14));
        if (l == 0) prec[f] = precision;
        inv = (float)(1.0 / (double)precision);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            minint[k] = (int32_t)be32_word(pw + 15 + k);
            sizeint[k] = be32_word(pw + 18 + k) - (uint32_t)minint[k] + 1u;
        }
        smallidx = (int)be32_word(pw + 21);
        const long long nbytes = (int)be32_word(pw + 22);
        if (nbytes < 0 || 23 + (nbytes + 3) / 4 > avail_words) {
            st = HR_XTC_TRUNCATED;
        } else if (smallidx < kFirstIdx || smallidx >= kLastIdx || !sizeint[0] || !sizeint[1] ||
                   !sizeint[2]) {  // a size of 0: maxint below minint
            st = HR_XTC_STREAM;
        }
        live = st == HR_XTC_OK;
        n_words = (int)((nbytes + 3) / 4);
    }
    if (!live) smallidx = kFirstIdx;
    if constexpr (R == 64) {  // one frame a wave: its scan runs on scalars
        smallidx = __builtin_amdgcn_readfirstlane(smallidx);
        n_words = __builtin_amdgcn_readfirstlane(n_words);
        live = __builtin_amdgcn_readfirstlane(live);
        st = __builtin_amdgcn_readfirstlane(st);
#pragma unroll
        for (int k = 0; k < 3; ++k) sizeint[k] = __builtin_amdgcn_readfirstlane(sizeint[k]);
    }
    const bool large = (sizeint[0] | sizeint[1] | sizeint[2]) > 0xFFFFFFu;
    int bitsize;  // of a large atom
    if (large) {  // three fields of up to 32 bits
        bitsize = (32 - __clz(sizeint[0])) + (32 - __clz(sizeint[1])) + (32 - __clz(sizeint[2]));
    } else {
        // bit length of the product: below 2^72, as a 64-bit product and its
        // top byte when it does not fit
        const uint64_t xy = (uint64_t)sizeint[0] * sizeint[1];     // < 2^48
        const uint64_t lo = (xy & 0xFFFFFFull) * sizeint[2];       // < 2^48
        const uint64_t hi = (xy >> 24) * sizeint[2] + (lo >> 24);  // product >> 24
        bitsize = hi ? 24 + bit_length64(hi) : bit_length64(lo);
    }
    const double size1 = (double)sizeint[1], size2 = (double)sizeint[2];
    const double inv_size1 = low_recip(size1), inv_size2 = low_recip(size2);

    // -- the ring: words base .. filled of the stream, block after block;
    // words past the stream's end read as zero and are never accepted.  The
    // loads are unconditional (a row that is done, or a word past the end,
    // reads a valid word that the ring's write drops): a load under a branch
    // is waited for where the branch ends, and here it has a whole batch's
    // time to arrive.
    if (!__any(live)) {
        if (lead) status[f] = st;
        return;
    }
    const uint32_t* w = live ? pw + 23 : reinterpret_cast<const uint32_t*>(data);
    const int last = live ? n_words - 1 : 0;  // -1 (no words) reads the header's last word
    uint32_t next[4];
    int base = 0, filled = 0;
    auto fetch = [&]() {  // four words a lane from word `filled` on
#pragma unroll
        for (int k = 0; k < 4; ++k) next[k] = w[min(filled + 4 * l + k, last)];
    };
    auto fill = [&]() {  // the block in registers to the ring, if it has room
        if (live && filled + T::kBlock4 <= base + kRing) {
            uint32_t v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v[k] = filled + 4 * l + k <= last ? __builtin_bswap32(next[k]) : 0u;
            const int at = filled & (kRing - 1);
            *reinterpret_cast<uint4*>(ring + at + 4 * l) = make_uint4(v[0], v[1], v[2], v[3]);
            if (l == 0 && at == 0) ring[kRing] = v[0];
            filled += T::kBlock4;
        }
    };
    fetch();
#pragma unroll 1
    for (int k = 0; k < kRing / T::kBlock4; ++k) {
        fill();
        fetch();
    }
    xtc_wave_sync();

    uint32_t pos = 0;  // bit of the next group, from word `base`
    int n_out = 0;
    int run3 = 0;  // small atoms of a group; a clear flag bit keeps it
    while (__any(live)) {
        const uint32_t avail = 32u * (uint32_t)(filled - base);
        const int left = n_words - base;  // words left in the stream
        const uint32_t total = 32u * (uint32_t)(left < 2 * kRing ? left : 2 * kRing);

        // -- scan.  A group is looked at only where the ring holds the longest
        // one that could start there and the staging area its eleven atoms.
        // Away from the frame's end nothing else can be wrong with it; near
        // the end (kEnd) a group is checked against the atom count and the
        // stream's bits.
        const int out0 = n_out;
        int rec_run = -1, rec_idx = kFirstIdx, rec_out = 0;  // -1: no group in this lane
        uint32_t rec_pos = 0;
        // cnt: groups taken; R once the row takes no more (nothing below then
        // changes its state)
        int cnt = live ? 0 : R;
        auto scan = [&](auto near_end) {
            constexpr bool kEnd = decltype(near_end)::value;
            const int out_lim = kEnd ? min(out0 + T::kCap - 11, n_atoms - 1) : out0 + T::kCap - 11;
            while (__any(cnt < R)) {
                const int j = l - cnt;  // what follows is unused for j < 0
                const uint32_t glen = (uint32_t)(bitsize + 1) + __umul24(run3, smallidx);
                const uint32_t p = pos + __umul24(j, glen);
                const int o = n_out + (int)__umul24(j, run3 + 1);
                const uint32_t six =
                    ring_bits<kRing>(ring, (uint32_t)base, p + (uint32_t)bitsize, 6);
                const int seen = (int)(o <= out_lim) &
                                 (int)(p + (uint32_t)(bitsize + 6) + __umul24(10, smallidx) <= avail);
                const int flag = (int)(six >> 5);
                const int code = (int)(six & 31u);
                const int g_run = flag ? (int)(__umul24(code, 171) >> 9) : run3;  // code / 3
                // what the row's lanes learn of the one that ends the step:
                // its run code, 32 with a flag to take, 64 if it is malformed
                int info = code | ((seen & flag) << 5);
                int stop = (seen ^ 1) | flag;
                if constexpr (kEnd) {
                    const uint32_t g_end = p + (uint32_t)(bitsize + (flag ? 6 : 1)) +
                                           __umul24(g_run, smallidx);
                    const int wrong =
                        seen & ((int)(o + 1 + g_run > n_atoms) | (int)(g_end > total));
                    info = wrong ? 64 : info;
                    stop |= wrong;
                }
                const unsigned long long all = __ballot((int)(j >= 0) & stop);
                int first;
                if constexpr (R == 64) {
                    first = all ? __ffsll((long long)all) - 1 : R;
                } else {
                    const uint32_t half = (lane & 32) ? (uint32_t)(all >> 32) : (uint32_t)all;
                    const uint32_t mine =
                        R == 32 ? half : (half >> (lane & 31 & ~(R - 1))) & ((1u << (R & 31)) - 1);
                    first = mine ? __ffs((int)mine) - 1 : R;
                }
                int got;
                if constexpr (R == 64)
                    got = __builtin_amdgcn_readlane(info, first & (R - 1));
                else
                    got = __shfl(info, (lane & ~(R - 1)) | (first & (R - 1)), kWave);
                const int f_info = first < R ? got : 0;
                const int with_flag = (f_info >> 5) & 1;
                const int upto = first + with_flag;
                const bool mine = j >= 0 && l < upto;
                rec_pos = mine ? p : rec_pos;
                rec_run = mine ? g_run : rec_run;
                rec_idx = mine ? smallidx : rec_idx;
                rec_out = mine ? o - out0 : rec_out;
                const int plain = first - cnt;
                const int f_run = (int)(__umul24(f_info & 31, 171) >> 9);
                pos += __umul24(plain, glen) +
                       (with_flag ? (uint32_t)(bitsize + 6) + __umul24(f_run, smallidx) : 0u);
                n_out += (int)__umul24(plain, run3 + 1) + (with_flag ? f_run + 1 : 0);
                run3 = with_flag ? f_run : run3;
                smallidx += with_flag ? (f_info & 31) - 3 * f_run - 1 : 0;
                int bad = (int)((unsigned)(smallidx - kFirstIdx) >= (unsigned)(kLastIdx - kFirstIdx));
                if constexpr (kEnd) bad |= f_info >> 6;
                st = bad ? HR_XTC_STREAM : st;
                const bool more = with_flag && !bad && (!kEnd || n_out < n_atoms);
                cnt = more ? upto : R;
            }
        };
        if (__any(live && (n_out + T::kCap >= n_atoms || total <= avail)))
            scan(std::true_type{});
        else
            scan(std::false_type{});

        // -- decode: one group a lane
        if (rec_run >= 0) {
            uint32_t big[3];
            uint32_t p = rec_pos;
            if (large) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const int n = 32 - __clz(sizeint[k]);
                    big[k] = ring_bits<kRing>(ring, (uint32_t)base, p, n);
                    p += (uint32_t)n;
                }
            } else {
                ring_ints3<kRing>(ring, (uint32_t)base, p, bitsize, size1, size2, inv_size2,
                                  inv_size1, big);
                p += (uint32_t)bitsize;
            }
            p += ring_bits<kRing>(ring, (uint32_t)base, p, 1) ? 6u : 1u;
            // the first small atom precedes the large one in the output
            // (stored swapped, for water), the others follow it
            int* to = stage + 3 * rec_out;
            int* at = to + (rec_run ? 3 : 0);
            const uint32_t size = (uint32_t)s_magic[rec_idx];
            const uint32_t half = size / 2;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                big[c] += (uint32_t)minint[c];
                at[c] = (int)big[c];
                big[c] -= half;
            }
            int skip = 6;
            if (rec_idx <= 30) {
                const float inv_size = __builtin_amdgcn_rcpf((float)size) * (1.0f - 0x1p-21f);
                // a field is read while the one before it is divided (the
                // read after the last is of whatever the ring holds there)
                uint32_t bits = ring_bits<kRing>(ring, (uint32_t)base, p, rec_idx);
                for (int k = 0; k < rec_run; ++k) {
                    const uint32_t v = chunks_to_number(bits, rec_idx);
                    p += (uint32_t)rec_idx;
                    bits = ring_bits<kRing>(ring, (uint32_t)base, p, rec_idx);
                    uint32_t r, r2;
                    const uint32_t q = div_small(v, size, inv_size, r);
                    const uint32_t q2 = div_small(q, size, inv_size, r2);
                    big[0] += q2;
                    big[1] += r2;
                    big[2] += r;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        to[c] = (int)big[c];
                        big[c] -= half;
                    }
                    to += skip;
                    skip = 3;
                }
            } else {
                const double wide = (double)size, inv_wide = low_recip(wide);
#pragma unroll 1
                for (int k = 0; k < rec_run; ++k) {
                    uint32_t d[3];
                    ring_ints3<kRing>(ring, (uint32_t)base, p, rec_idx, wide, wide, inv_wide,
                                      inv_wide, d);
                    p += (uint32_t)rec_idx;
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        big[c] += d[c];
                        to[c] = (int)big[c];
                        big[c] -= half;
                    }
                    to += skip;
                    skip = 3;
                }
            }
        }
        xtc_wave_sync();

        // -- the next block, asked for a batch ago, into the ring; the one
        // after it is asked for ahead of the stores, so that waiting for it
        // does not wait for them
        const bool write = live;
        base += (int)(pos >> 5);
        pos &= 31u;
        fill();
        fetch();
        live = live && st == HR_XTC_OK && n_out < n_atoms;

        // -- store, with the format's rounding (the integer to float, times
        // float(1 / precision)): four floats a lane, of a row that is
        // consecutive in memory
        if (write) {
            typedef float V4f __attribute__((ext_vector_type(4), aligned(4)));
            typedef __attribute__((address_space(1))) V4f GlobalV4f;
            const int n = 3 * (n_out - out0);
            auto* dst = global_out(out + 3LL * out0);
            for (int i = 4 * l; i < n; i += 4 * R) {
                const int4 c = *reinterpret_cast<const int4*>(stage + i);
                const V4f v = {__fmul_rn((float)c.x, inv), __fmul_rn((float)c.y, inv),
                               __fmul_rn((float)c.z, inv), __fmul_rn((float)c.w, inv)};
                if (i + 4 <= n) {
                    *(GlobalV4f*)(dst + i) = v;
                } else {
                    dst[i] = v.x;
                    if (i + 1 < n) dst[i + 1] = v.y;
                    if (i + 2 < n) dst[i + 2] = v.z;
                }
            }
        }
        xtc_wave_sync();
    }
    if (lead) status[f] = st;
}

}  // namespace
}  // namespace hr

using namespace hr;

extern "C" {

int hr_xtc_scan(const void* data, int64_t n_bytes, int64_t* offsets, int64_t max_frames,
                int64_t* n_frames, int32_t* n_atoms) {
    clear_error();
    HR_REQUIRE(n_frames && n_atoms, "NULL pointer argument");
    HR_REQUIRE(n_bytes >= 0 && (data || n_bytes == 0), "invalid buffer");
    HR_REQUIRE(max_frames >= 0 && (offsets || max_frames == 0), "invalid offsets buffer");
    const unsigned char* p = static_cast<const unsigned char*>(data);
    long long pos = 0, count = 0;
    int natoms = -1;
    while (pos + 4 <= n_bytes) {
        if (pos + 56 > n_bytes) {
            set_error("truncated frame header at byte %lld", pos);
            return HR_ERR_INVALID;
        }
        const int magic = (int)be32(p + pos);
        const int na = (int)be32(p + pos + 4);
        if (magic != kXtcMagic) {
            set_error("not an XTC frame at byte %lld (magic %d)", pos, magic);
            return HR_ERR_INVALID;
        }
        if (na <= 0 || (natoms >= 0 && na != natoms)) {
            set_error("frame at byte %lld holds %d atoms (first frame: %d)", pos, na, natoms);
            return HR_ERR_INVALID;
        }
        natoms = na;
        long long next;
        if (na <= 9) {
            next = pos + 56 + 12LL * na;
        } else {
            if (pos + 92 > n_bytes) {
                set_error("truncated frame at byte %lld", pos);
                return HR_ERR_INVALID;
            }
            const long long nb = (int)be32(p + pos + 88);
            if (nb < 0) {
                set_error("negative byte count in frame at byte %lld", pos);
                return HR_ERR_INVALID;
            }
            next = pos + 92 + (nb + 3) / 4 * 4;
        }
        if (next > n_bytes) {
            set_error("truncated frame at byte %lld", pos);
            return HR_ERR_INVALID;
        }
        if (count < max_frames) offsets[count] = pos;
        ++count;
        pos = next;
    }
    *n_frames = count;
    *n_atoms = natoms < 0 ? 0 : natoms;
    return HR_OK;
}

int hr_xtc_decode(const void* data, int64_t n_bytes, const int64_t* offsets, int64_t n_frames,
                  int32_t n_atoms, float* xyz, float* time, int32_t* step, float* box,
                  float* prec, int32_t* status, void* stream) {
    clear_error();
    HR_REQUIRE(n_frames >= 0 && n_atoms > 0 && n_bytes >= 0,
               "invalid sizes n_frames=%lld n_atoms=%d", (long long)n_frames, n_atoms);
    if (n_frames == 0) return HR_OK;
    HR_REQUIRE(data && offsets && xyz && time && step && box && prec && status,
               "NULL pointer argument");
    HR_REQUIRE((reinterpret_cast<uintptr_t>(data) & 3) == 0, "data must be 4-byte aligned");
    HR_REQUIRE((reinterpret_cast<uintptr_t>(xyz) & 3) == 0, "xyz must be 4-byte aligned");
    const bool tiny = n_atoms <= kTinyAtoms;
    const int r = tiny ? kTinyLanes : xtc_row_lanes(n_frames, n_atoms);
    const auto kernel = tiny      ? xtc_tiny_kernel
                        : r == 4  ? xtc_decode_kernel<4>
                        : r == 8  ? xtc_decode_kernel<8>
                        : r == 16 ? xtc_decode_kernel<16>
                        : r == 32 ? xtc_decode_kernel<32>
                                  : xtc_decode_kernel<64>;
    const int block = tiny ? kTinyBlock : kWave, frames = block / r;  // of a workgroup
    hipLaunchKernelGGL(kernel, launch_grid((n_frames + frames - 1) / frames, block), dim3(block), 0,
                       (hipStream_t)stream, static_cast<const unsigned char*>(data),
                       (long long)n_bytes, reinterpret_cast<const long long*>(offsets),
                       (long long)n_frames, n_atoms, xyz, time, step, box, prec, status);
    return launch_status("xtc_decode_kernel");
}

}  // extern "C"
