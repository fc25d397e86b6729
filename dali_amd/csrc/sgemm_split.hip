// fp32 GEMM on the bf16 matrix cores: every operand value is cut into three bf16 pieces whose sum is the value itself.
//
// Row-major view: C[M,N] = alpha * sum_s A_s[M,K_s] * B_s[K_s,N] + beta * C with A stored [M][K] or [K][M] and B stored [K][N] or [N][K].
//
// What bounds the kernels it stands in for is the fp32 matrix rate (157 TFLOP/s; a bf16 instruction does sixteen times as much per
// cycle). The cut is that of Henry, Tang and Heinecke ("Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", 2019): with h = bf16(x), m = bf16(x - h), l = x - h - m, all rounded to nearest, x = h + m + l holds exactly: 24
// significant bits in three times 8, and the exponent range of bf16 is that of fp32. Of the nine products of the pieces of a and b the six
// of weight 2^-16 and more are summed (hh, hm, mh, hl, lh, mm). m reaches 2^-8 and l 2^-17 of the value's power of two, so those left
// out, ml + lm + ll, come to at most 2^-24 |a b|: what rounding one fp32 product costs at most. Products of bf16 pieces are exact in
// fp32 and the sums are kept in fp32.
//
// Both operands are multiplied by 2^16 as they are cut and the sums by 2^-32 at the end: the smallest float, 2^-149, becomes the smallest
// bf16, so that no value is too small for its pieces (the conversion and the matrix instruction keep denormal values). Without
// that a single entry below 2^-110, as a softmax gradient has where a logit lies 76 below the largest, loses bits.
// Infinities, NaN, values from about 2^112 and sums from 2^96 on leave a scaled sum that is not finite: such a tile is redone
// with the fp32 instructions on the values as they are, whatever they come to. [256,1024].[1024,32000]: one entry in 61 below 2^-110
// 106 us as without them (246 while the last piece lost bits and such tiles were redone), a NaN in every strip of rows 244
// us, the fp32 kernels 138.
//
// A MFMA of this kind takes an accumulator that is smaller than the sum of products added to it down to a multiple of 2^-24 of that sum's
// power of two (towards minus infinity) before it rounds the result; where the accumulator is the larger one the result is rounded to
// nearest (probed with single products). Small products summed first lose their ends when hh is added. So the five small products have sums of their
// own, a 2^-8 of the result, where that does not matter; hh is summed over two slabs (32 values of k) from zero and added to
// the sums by the vector unit, as are the small ones at the end. Distance from double precision, results of [2048,2048], normal
// operands (in brackets the fp32 kernels): K = 133 0.58e-7 (2.0e-7), 512 0.86e-7 (4.1e-7), 1999 1.2e-7 (7.9e-7); [1024,1024] over 32000 2.2e-7
// (2.3e-6). Rows of one product only (a diagonal operand) 2.58e-8 in the root mean square and 9.9e-8 at worst (2.53e-8, 6.0e-8: an
// fp32 product rounded once), two and more of like size in a row already less than there; where a few of very different
// sizes make up a result (exponents spread evenly over e^-20 to e^20, K = 65) 5.3e-8 (5.1e-8). With all six in one sum a diagonal operand showed 3.3e-8 and
// 15.7e-8; with the two largest of those left out as well, 2.53e-8 and 6.0e-8, but at 131, 144 and 130 us for the three products
// below, which is the time of the fp32 kernels.
//
// A workgroup of four waves owns a 128x128 tile, a wave 64x64 of it as 2x2 accumulators of v_mfma_f32_32x32x16_bf16. Slabs of 16
// values of k come through registers (fetched one slab ahead), are cut there, once per workgroup and value, and written to
// LDS as three planes of [row][16 k] in bf16: whatever the storage order, a lane packs neighbours in k, so the transposition of
// [K][x] operands costs nothing. m and l have two stages, h a ring of four: while a slab is multiplied the next one is cut, and the second
// slab of a pair finds h of the first. One barrier per slab. 64 KiB and at most 256 registers: two workgroups share a compute unit.
//
// Measured (normal operands, steady load): [256,1024].[1024,32000] 145 -> 116 us, its gradients [1024,256].[256,32000] 130 -> 123 us and
// [256,32000].[32000,1024] 129 -> 107 us; 4096^3 943 -> 769 us, with B stored [N][K] 948 -> 757, A stored [K][M] 925 -> 770, both 946 -> 768. After
// idle time both sides are slower: 162 -> 125, 160 -> 148, 157 -> 125, 4096^3 1102 -> 995. What bounds it: the matrix instructions
// fill 0.39 (second of these) and 0.52 (third) of the cycles, cutting and adding 0.44 and 0.43, and the two hardly overlap. Measured and
// dropped: all six products in one sum, added every 32 k (735 us at 4096^3, and the loss above), hh added to the sums by the matrix
// instruction itself (710, but 1.28e-7 at K = 512 and 4.0e-7 at 32000, further off than the form before), slabs of 32 with two barriers,
// fetching two slabs ahead (spills: 1260 us), both first slabs of a tile at once (800), an order of instructions within the groups (776), no order
// between them (776 to 795), subtracting with v_dot2_f32_bf16 (slower and not exact).
//
// LDS rows are 32 bytes, two 16-byte granules of eight k. Granule g of row r lies in slot g ^ (bit 2 of r) of the row whose bit 2 is
// flipped where bit 3 of r is set: eight neighbouring rows touch eight different 16-byte columns of 128 bytes, sixteen touch sixteen of
// 256, when reading and when writing.
#include <cstdlib>
#include <type_traits>

#include "runtime.h"

namespace dali_hip {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef unsigned int uintx4 __attribute__((ext_vector_type(4)));
// loads claim element alignment only: any leading dimension, any view
typedef floatx4 floatx4u __attribute__((aligned(4)));

constexpr int kTile = 128, kSlab = 16;
constexpr int kRowBytes = kSlab * 2;
constexpr int kPlaneBytes = kTile * kSlab * 2;     // one piece of one operand
constexpr int kHighBytes = 2 * kPlaneBytes;        // h of one slab of both operands: a ring of four slabs
constexpr int kLowBytes = 4 * kPlaneBytes;         // m and l: two stages behind the ring
constexpr int kLow = 4 * kHighBytes, kLdsBytes = kLow + 2 * kLowBytes;
constexpr int kMaxTerms = 8;

// The convolutions of a channels-last image x [n, h, w, c] without padding, by their windows' positions (image, i, j) in order, position 0
// at the image's first value: neighbours `step` values apart, rows of out_w of them `row` apart, images of out_h rows `image`.
// A window's row kh is the run of `run` values from kh * line behind its position on.
struct SplitConv {
    int out_w, out_h, step, row, image, run, line;
    unsigned hw, hw_m, w_m, run_m;  // exact divisions by out_h * out_w, out_w and run
    int hw_s, w_s, run_s;
    __device__ __forceinline__ int place(int k) const {
        const int img = (int)sgemm_row_map_div((unsigned)k, hw_m, hw_s), rest = k - img * (int)hw, i = (int)sgemm_row_map_div((unsigned)rest, w_m, w_s);
        return img * image + i * row + (rest - i * out_w) * step;
    }
    // value n of a window
    __device__ __forceinline__ int within(int n) const {
        const int kh = (int)sgemm_row_map_div((unsigned)n, run_m, run_s);
        return kh * line + n - kh * run;
    }
};

// consecutive positions
struct Positions {
    int i, j, at;
    __device__ __forceinline__ void seek(const SplitConv& cv, int k) {
        const int img = (int)sgemm_row_map_div((unsigned)k, cv.hw_m, cv.hw_s), rest = k - img * (int)cv.hw;
        i = (int)sgemm_row_map_div((unsigned)rest, cv.w_m, cv.w_s);
        j = rest - i * cv.out_w;
        at = img * cv.image + i * cv.row + j * cv.step;
    }
    __device__ __forceinline__ void next(const SplitConv& cv) {
        at += cv.step;
        if (++j == cv.out_w) {
            j = 0;
            at += cv.row - cv.out_w * cv.step;
            if (++i == cv.out_h) {
                i = 0;
                at += cv.image - cv.out_h * cv.row;
            }
        }
    }
};

// What the operands are: matrices; for a convolution's result A is the image, row m the window at position m, a term per row of the
// window; for the gradient of its filters B is the image, row k the window at position k
enum Form { kPlain = 0, kWindows = 1, kFilters = 2 };

struct SplitArgs {
    const float* A[kMaxTerms];
    const float* B[kMaxTerms];
    int lda[kMaxTerms], ldb[kMaxTerms], K[kMaxTerms];
    int nseg;
    int M, N;
    float* C;
    int ldc;
    float alpha, beta;
    int tiles_m, tiles_n, shares;
    int slabs;        // of all terms together
    float* partials;  // shares > 1: [share][tile][16384], else unused
    SgemmRowMap map;
    SplitConv cv;
};

__device__ __forceinline__ float lo_part(unsigned int pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float hi_part(unsigned int pair) { return __uint_as_float(pair & 0xffff0000u); }
__device__ __forceinline__ unsigned int pack2(float a, float b) {
    const floatx2 v = {a, b};
    return __builtin_bit_cast(unsigned int, __builtin_convertvector(v, bf16x2));
}

constexpr float kScale = 0x1p16f, kScaleBack = 0x1p-32f;  // of each operand; of the sums of products

// two neighbours in k, scaled, cut into their three pieces
__device__ __forceinline__ void cut2(float a, float b, unsigned int& h, unsigned int& m, unsigned int& l) {
    a *= kScale;
    b *= kScale;
    h = pack2(a, b);
    const float a1 = a - lo_part(h), b1 = b - hi_part(h);
    m = pack2(a1, b1);
    const float a2 = a1 - lo_part(m), b2 = b1 - hi_part(m);
    l = pack2(a2, b2);
}

__device__ __forceinline__ int lds_offset(int row, int granule) {
    return (row ^ (((row >> 3) & 1) << 2)) * kRowBytes + ((granule ^ ((row >> 2) & 1)) << 4);
}

// A thread's share of one operand's slab: eight k of one row (column) of the tile, one granule of each plane.
//   KROWS (stored [x][K]): row t / 2, k from 8 (t % 2): two 16-byte loads
//   else  (stored [K][x]): column t % 128, k from 8 (t / 128): eight loads of neighbouring columns
template <bool KROWS>
struct Loader {
    int row, granule;  // within the tile
    unsigned off;      // of the first value, from the operand's first row and the slab's first k (KROWS), or from the slab's first k

    __device__ __forceinline__ void init(int tid, int x0, int x_end, int ld) {
        row = KROWS ? tid >> 1 : tid & 127;
        granule = KROWS ? tid & 1 : tid >> 7;
        set_ld(x0, x_end, ld);
    }
    // (rows past the end repeat the last one; what they sum up to is not stored)
    __device__ __forceinline__ void set_ld(int x0, int x_end, int ld) {
        const int x = min(x0 + row, x_end - 1);
        off = KROWS ? (unsigned)((x - x0) * ld + 8 * granule) : (unsigned)(8 * granule * ld + x);
    }
    // rows (columns) of windows: KROWS, from the window of the tile's first row; else from a window's first value
    __device__ __forceinline__ void set_windows(const SplitConv& cv, int x0, int x_end) {
        const int x = min(x0 + row, x_end - 1);
        off = KROWS ? (unsigned)(cv.place(x) - cv.place(x0) + 8 * granule) : (unsigned)cv.within(x);
    }
    // eight windows' values (else)
    __device__ __forceinline__ void fetch_windows(float* v, const float* p, const SplitConv& cv, Positions& at) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            v[j] = (p + at.at)[off];
            at.next(cv);
        }
    }
    __device__ __forceinline__ void fetch_windows_tail(float* v, const float* p, const SplitConv& cv, int k0, int left) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 8 * __builtin_amdgcn_readfirstlane(granule) + j;
            const float a = (p + cv.place(k0 + min(k, left - 1)))[off];
            v[j] = k < left ? a : 0.0f;
        }
    }
    // `p`: the tile's first row at the slab's first k (KROWS), the slab's first k (else)
    __device__ __forceinline__ void fetch(float* v, const float* p, int ld) const {
        if (KROWS) {
            const floatx4 a = *(const floatx4u*)(p + off), b = *(const floatx4u*)(p + off + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                v[j] = a[j];
                v[4 + j] = b[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = (p + (size_t)j * ld)[off];  // (the row in scalar registers)
        }
    }
    // the last, partly filled slab of a term: `left` values of k, the others are zero
    __device__ __forceinline__ void fetch_tail(float* v, const float* p, int ld, int left) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int k = 8 * granule + j, back = max(k - (left - 1), 0);
            const float a = p[off + (unsigned)(KROWS ? j : j * ld) - (unsigned)(KROWS ? back : back * ld)];
            v[j] = k < left ? a : 0.0f;
        }
    }
    // two of the four pairs of neighbours of `v`
    __device__ __forceinline__ static void cut_half(const float* v, int half, uintx4& h, uintx4& m, uintx4& l) {
#pragma unroll
        for (int q = 2 * half; q < 2 * half + 2; ++q) {
            unsigned int hq, mq, lq;
            cut2(v[2 * q], v[2 * q + 1], hq, mq, lq);
            h[q] = hq;
            m[q] = mq;
            l[q] = lq;
        }
    }
    // `high`, `low`: this operand's planes of the slab
    __device__ __forceinline__ void store(uintx4 h, uintx4 m, uintx4 l, char* high, char* low) const {
        const int d = lds_offset(row, granule);
        *(uintx4*)(high + d) = h;
        *(uintx4*)(low + d) = m;
        *(uintx4*)(low + d + kPlaneBytes) = l;
    }
    // as fp32, rows of 16 k and a pitch of 17 (a tile that is redone)
    __device__ __forceinline__ void store_plain(const float* v, float* lds) const {
#pragma unroll
        for (int j = 0; j < 8; ++j) lds[row * 17 + 8 * granule + j] = v[j];
    }
};

// Walks the slabs of the terms in order for the loads, which are the same instructions for every slab, so that the waits for one
// slab leave the next ones' loads in flight: a partly filled last slab is fetched sixteen values of k ending at the last (what that
// gets wrong is fetched again when it is cut), and behind the last slab of the share that one is fetched again.
template <bool TA, bool TB, int F>
struct Walk {
    Loader<!TA> a;
    Loader<TB> b;
    Positions at;  // of the slab's windows (kFilters): of this wave's eight
    const float *pa, *pb;
    int term, left, lda, ldb, todo;  // left: values of k of the term from this slab on; todo: slabs to move on to

    __device__ __forceinline__ void enter(const SplitArgs& g, int k0, int m0, int n0) {
        lda = g.lda[term];
        ldb = g.ldb[term];
        if (F != kWindows) a.set_ld(m0, g.M, lda);
        if (F != kFilters) b.set_ld(n0, g.N, ldb);
        left = g.K[term] - k0;
        k0 = min(k0, g.K[term] - kSlab);
        pa = g.A[term] + (F == kWindows ? (size_t)(g.cv.place(m0) + k0) : TA ? (size_t)k0 * lda : (size_t)m0 * lda + k0);
        pb = g.B[term] + (F == kFilters ? (size_t)0 : TB ? (size_t)n0 * ldb + k0 : (size_t)k0 * ldb);
        if (F == kFilters) at.seek(g.cv, k0 + 8 * __builtin_amdgcn_readfirstlane(b.granule));
    }
    __device__ __forceinline__ void start(const SplitArgs& g, int first_term, int k0, int count, int m0, int n0) {
        term = first_term;
        todo = count - 1;
        enter(g, k0, m0, n0);
    }
    // fetches the slab and moves on to the next
    __device__ __forceinline__ void fetch(const SplitArgs& g, float* va, float* vb, int m0, int n0) {
        a.fetch(va, pa, lda);
        Positions behind = at;
        if (F == kFilters) b.fetch_windows(vb, pb, g.cv, behind);
        else b.fetch(vb, pb, ldb);
        if (todo > 0) {
            --todo;
            left -= kSlab;
            if (left > 0) {
                const int by = min(left, kSlab);
                pa += TA ? (size_t)by * lda : (size_t)by;
                if (F != kFilters) {
                    pb += TB ? (size_t)by : (size_t)by * ldb;
                } else if (by == kSlab) {
#pragma unroll
                    for (int j = 0; j < 8; ++j) behind.next(g.cv);  // (the other half's windows)
                    at = behind;
                } else {
                    at.seek(g.cv, g.K[term] - kSlab + 8 * __builtin_amdgcn_readfirstlane(b.granule));
                }
            } else {
                ++term;
                enter(g, 0, m0, n0);
            }
        }
    }
};

// The same walk for the cutting, one to three slabs behind: tells the partly filled slabs.
template <bool TA, bool TB, int F>
struct Cutter {
    int term, left;
    __device__ __forceinline__ void start(const SplitArgs& g, int first_term, int k0) {
        term = first_term;
        left = g.K[term] - k0;
    }
    // the slab in `va`, `vb` with zeros behind the end of the term
    __device__ __forceinline__ void settle(const SplitArgs& g, const Walk<TA, TB, F>& w, float* va, float* vb, int m0, int n0) {
        if (left > 0 && left < kSlab) {
            Loader<!TA> a = w.a;
            Loader<TB> b = w.b;
            const int lda = g.lda[term], ldb = g.ldb[term], k0 = g.K[term] - left;
            if (F != kWindows) a.set_ld(m0, g.M, lda);
            if (F != kFilters) b.set_ld(n0, g.N, ldb);
            a.fetch_tail(va, g.A[term] + (F == kWindows ? (size_t)(g.cv.place(m0) + k0) : TA ? (size_t)k0 * lda : (size_t)m0 * lda + k0), lda, left);
            if (F == kFilters) b.fetch_windows_tail(vb, g.B[term], g.cv, k0, left);
            else b.fetch_tail(vb, g.B[term] + (TB ? (size_t)n0 * ldb + k0 : (size_t)k0 * ldb), ldb, left);
        }
        left -= kSlab;
        if (left <= 0 && term + 1 < g.nseg) left = g.K[++term];
    }
};

// LDS written by this wave is there and every wave has come here; loads from global memory stay in flight
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

__device__ __forceinline__ void put(const SplitArgs& g, float* d, float sum) {
    float r = g.alpha * sum;
    if (g.beta != 0.0f) r += g.beta * *d;
    *d = r;
}

__device__ __forceinline__ void store_result(const SplitArgs& g, int m, int n, float sum) {
    size_t row = (size_t)m;
    if (g.map.on) {
        const unsigned img = sgemm_row_map_div((unsigned)m, g.map.hw_m, g.map.hw_s), rest = (unsigned)m - img * g.map.hw;
        const unsigned i = sgemm_row_map_div(rest, g.map.w_m, g.map.w_s), j = rest - i * g.map.w;
        if ((int)i >= g.map.oh || (int)j >= g.map.ow) return;
        row = ((size_t)img * g.map.oh + i) * g.map.ow + j;
    }
    put(g, g.C + row * g.ldc + n, sum);
}

template <bool TA, bool TB, int F>
__global__ __launch_bounds__(256, 2) void sgemm_split_kernel(SplitArgs g) {
    __shared__ __attribute__((aligned(16))) char lds[kLdsBytes];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Every eighth workgroup runs on the same die: a die takes a run of neighbouring tiles (of one share), eight rows of tiles to
    // a band, and finds the operands its other workgroups asked for in its L2.
    const int total = g.tiles_m * g.tiles_n * g.shares;
    int id = blockIdx.x;
    const int per = total >> 3;
    if (id < per * 8) id = (id & 7) * per + (id >> 3);
    const int tiles = g.tiles_m * g.tiles_n;
    // (the quotients come out of the vector unit)
    auto uniform = [](int x) { return __builtin_amdgcn_readfirstlane(x); };
    const int share = uniform(id / tiles);
    const int tile = id - share * tiles;
    const int band = uniform(tile / (8 * g.tiles_n)), band_rows = min(8, g.tiles_m - 8 * band), in_band = tile - band * 8 * g.tiles_n;
    const int tn = uniform(in_band / band_rows), tm = 8 * band + in_band - tn * band_rows;
    const int m0 = tm * kTile, n0 = tn * kTile;
    const int s_begin = uniform(g.slabs * share / g.shares), s_end = uniform(g.slabs * (share + 1) / g.shares);

    floatx16 acc[2][2], small[2][2];  // the sums of hh; of the other products
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = small[i][j] = floatx16{};
    const int wm = 64 * (wave >> 1), wn = 64 * (wave & 1);
    Walk<TA, TB, F> w;
    w.a.init(tid, m0, g.M, 0);
    w.b.init(tid, n0, g.N, 0);
    if (F == kWindows) w.a.set_windows(g.cv, m0, g.M);
    if (F == kFilters) w.b.set_windows(g.cv, n0, g.N);
    int first_term = 0, first_k = s_begin;
    while (first_term + 1 < g.nseg && first_k >= (g.K[first_term] + kSlab - 1) / kSlab) first_k -= (g.K[first_term++] + kSlab - 1) / kSlab;
    first_k *= kSlab;
    const int count = s_end - s_begin;
    w.start(g, first_term, first_k, count, m0, n0);
    Cutter<TA, TB, F> c;
    c.start(g, first_term, first_k);
    float va[8], vb[8];
    const int ra = lds_offset(wm + (lane & 31), lane >> 5), rb = lds_offset(wn + (lane & 31), lane >> 5) + kPlaneBytes;
    // operand fragments of the wave: A and B in turn (32 rows further down the swizzle is the same)
    auto read = [&](bf16x8* a, bf16x8* b, const char* from, int b_off) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            a[i] = *(const bf16x8*)(from + ra + i * 32 * kRowBytes);
            b[i] = *(const bf16x8*)(from + rb + b_off + i * 32 * kRowBytes);
        }
    };
    auto mfma = [](bf16x8 a, bf16x8 b, floatx16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); };
    int ring = 0;  // where in the ring the pair of slabs at hand begins
    // The small products of slab `P` (its parity) of a pair, for the second also hh of both; meanwhile the next slab is cut and
    // written to LDS. Four groups, so that no more than one sum of hh is held at a time.
    auto multiply = [&](auto parity) {
        constexpr int P = decltype(parity)::value;
        const char *high = lds + ring, *low = lds + kLow + P * kLowBytes;
        bf16x8 ea[2], eb[2], pa[3][2], pb[3][2];  // h of the pair's first slab; h, m, l of this one
        read(pa[0], pb[0], high + P * kHighBytes, 0);
        read(pa[1], pb[1], low, kPlaneBytes);
        if (P == 1) read(ea, eb, high, 0);
        constexpr int PA[5] = {0, 1, 1, 0, 2}, PB[5] = {1, 0, 1, 2, 0};
        char *high_to = P == 0 ? lds + ring + kHighBytes : lds + (ring ^ (2 * kHighBytes)), *low_to = lds + kLow + (1 - P) * kLowBytes;
        uintx4 ch, cm, cl;
#pragma unroll
        for (int group = 0; group < 4; ++group) {
            const int bi = group >> 1, bj = group & 1;
            if (group == 1) read(pa[2], pb[2], low + kPlaneBytes, kPlaneBytes);
            floatx16 big;
            if (P == 1) {
                big = mfma(ea[bi], eb[bj], floatx16{});
                big = mfma(pa[0][bi], pb[0][bj], big);
            }
#pragma unroll
            for (int x = 5 * group; x < 5 * group + 5; ++x) {
                const int q = x >> 2, i = (x >> 1) & 1, j = x & 1;
                small[i][j] = mfma(pa[PA[q]][i], pb[PB[q]][j], small[i][j]);
            }
            Loader<TB>::cut_half(group < 2 ? va : vb, group & 1, ch, cm, cl);
            if (group == 1) w.a.store(ch, cm, cl, high_to, low_to);
            if (group == 3) w.b.store(ch, cm, cl, high_to + kPlaneBytes, low_to + 2 * kPlaneBytes);
            if (P == 1) acc[bi][bj] += big;
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    using Even = std::integral_constant<int, 0>;
    using Odd = std::integral_constant<int, 1>;
    w.fetch(g, va, vb, m0, n0);
    c.settle(g, w, va, vb, m0, n0);
    {
        uintx4 h, m, l;
        Loader<TB>::cut_half(va, 0, h, m, l);
        Loader<TB>::cut_half(va, 1, h, m, l);
        w.a.store(h, m, l, lds, lds + kLow);
        Loader<TB>::cut_half(vb, 0, h, m, l);
        Loader<TB>::cut_half(vb, 1, h, m, l);
        w.b.store(h, m, l, lds + kPlaneBytes, lds + kLow + 2 * kPlaneBytes);
    }
    w.fetch(g, va, vb, m0, n0);
    lds_barrier();
    // (behind the last slab it is cut once more, to where nobody reads it again)
    for (int s = 0; s < count; s += 2) {
        c.settle(g, w, va, vb, m0, n0);
        multiply(Even{});
        w.fetch(g, va, vb, m0, n0);
        lds_barrier();
        if (s + 1 < count) {
            c.settle(g, w, va, vb, m0, n0);
            multiply(Odd{});
            w.fetch(g, va, vb, m0, n0);
            lds_barrier();
        } else {
            bf16x8 a[2], b[2];
            read(a, b, lds + ring, 0);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] += mfma(a[i], b[j], floatx16{});
        }
        ring ^= 2 * kHighBytes;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] += small[i][j];

    // a sum that is not finite: this tile again with the fp32 instructions
    float probe = 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int v = 0; v < 16; ++v) probe = fmaf(acc[i][j][v], 0.0f, probe);
        }
    if (__syncthreads_or(probe != 0.0f)) {  // (0 * x is 0 for finite x and NaN else)
        float* la = (float*)lds;
        float* lb = la + kTile * 17;
        static_assert(2 * kTile * 17 * sizeof(float) <= kLdsBytes, "the fp32 slab fits the pieces' LDS");
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = floatx16{};
        w.start(g, first_term, first_k, count, m0, n0);
        c.start(g, first_term, first_k);
        w.fetch(g, va, vb, m0, n0);
        for (int r = 0; r < count; ++r) {
            c.settle(g, w, va, vb, m0, n0);
            lds_barrier();
            w.a.store_plain(va, la);
            w.b.store_plain(vb, lb);
            w.fetch(g, va, vb, m0, n0);  // (in flight while this slab is multiplied)
            lds_barrier();
            for (int k = 0; k < kSlab; k += 2) {
                float fa[2], fb[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    fa[i] = la[(wm + 32 * i + (lane & 31)) * 17 + k + (lane >> 5)];
                    fb[i] = lb[(wn + 32 * i + (lane & 31)) * 17 + k + (lane >> 5)];
                }
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] *= kScaleBack;
    }

    if (g.shares > 1) {
        floatx4* d = (floatx4*)(g.partials + ((size_t)share * tiles + tile) * (kTile * kTile)) + tid;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) d[((i * 2 + j) * 4 + q) * 256] = floatx4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        return;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn + 32 * j + (lane & 31), m = m0 + wm + 4 * (lane >> 5);
            if (n >= g.N) continue;
            float* d = g.C + (size_t)m * g.ldc + n;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int r = 32 * i + 8 * (v >> 2) + (v & 3);
                if (m + r >= g.M) continue;
                if (g.map.on) store_result(g, m + r, n, acc[i][j][v]);
                else put(g, d + (size_t)r * g.ldc, acc[i][j][v]);  // (the row's distance is the same for all lanes)
            }
        }
}

// adds the shares of a tile up in their order: a thread takes four rows of one column, sixteen workgroups a tile
__global__ __launch_bounds__(256) void sgemm_split_fold(SplitArgs g) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, tiles = g.tiles_m * g.tiles_n;
    const int tile = blockIdx.x >> 4, quad = blockIdx.x & 15;
    const floatx4* p = (const floatx4*)(g.partials + (size_t)tile * (kTile * kTile)) + quad * 256 + tid;
    const size_t pitch = (size_t)tiles * (kTile * kTile / 4);
    floatx4 sum = p[0];
    int s = 1;
    for (; s + 8 <= g.shares; s += 8) {
        floatx4 part[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) part[i] = p[(s + i) * pitch];
#pragma unroll
        for (int i = 0; i < 8; ++i) sum += part[i];
    }
    for (; s < g.shares; ++s) sum += p[s * pitch];
    const int band = tile / (8 * g.tiles_n), band_rows = min(8, g.tiles_m - 8 * band), in_band = tile - band * 8 * g.tiles_n;
    const int tm = 8 * band + in_band % band_rows, tn = in_band / band_rows;
    const int i = quad >> 3, j = (quad >> 2) & 1, q = quad & 3;
    const int n = tn * kTile + 64 * (wave & 1) + 32 * j + (lane & 31);
    const int m = tm * kTile + 64 * (wave >> 1) + 32 * i + 8 * q + 4 * (lane >> 5);
    if (n >= g.N) return;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (m + v < g.M) store_result(g, m + v, n, sum[v]);
}

// The number of shares of the inner extent, 0 where the fp32 kernels at `fp32_rate` (TFLOP/s times 10^6; over whole 64x64 tiles) are estimated to be as fast
// with what `g` describes, `beside`: and with what that form does besides, in microseconds.
int choose_shares(const SplitArgs& g, int cus, double fp32_rate, bool long_rate, double beside = 0.0) {
    const long tiles = (long)g.tiles_m * g.tiles_n;
    // Whether and in how many shares, by estimated microseconds. Workgroups that share a compute unit pass a slab each in 0.8 us, one alone in
    // 1.0; starting and ending a tile costs four slabs; adding shares up costs a launch and a read of them. The fp32 kernels by their
    // rate over whole 64x64 tiles, in TFLOP/s: 76 where several terms or a row map leave them the register-staged kernel (measured 68 to 94); 135
    // where their loads write LDS and up to four rounds of 64x64 tiles fill the chip (117 to 141); 115 over long inner extents, where they
    // cut what does not fill a round into shares (117 to 136 at 1.4 to 2.4 tiles a compute unit); 55 where operands lie off 16 bytes
    // (22 to 81 over 64 products of odd sizes, of which the split form was the faster one in all above 10 us); 112 else (70 to 145: rounds that are not full are the slow ones). Measured, us here / there, in the orders NN NT TN TT:
    //   one 128x128 tile a compute unit, refused: 2048^2 over 512 39 38 40 38 / 37 36 35 36, over 1024 69 68 69 67 / 65 65 63 64; 1024^2 over 4096
    //     63 62 63 63 / 64 61 63 61; [1883,10136] against [4486,10136] (NT) 1485 / 1411; [256,4096] over 512 24 24 24 24 / 11 11 11 11
    //   two: [2048,4096] over 256 35 34 35 35 / 37 38 36 38, over 1024 107 105 106 106 / 124 126 122 125
    //   three: [3072,4096] over 256 52 51 52 51 / 53 54 53 54, over 1024 161 160 163 160 / 185 185 180 185, over 4096 605 599 612 598 / 711 713 698 713
    //   five: [4096,5120] over 256 79 78 80 79 / 87 88 85 87, over 1024 260 254 260 256 / 310 311 301 309
    //   2.4 tiles, off 16 bytes: [573,15415] over 2683 395 397 400 396 / 581 589 910 900
    //   off 16 bytes: [1023,1025] over 1027 36 34 34 34 / 42 72 69 84, [172,60984] over 425 101 99 102 100 / 184 194 165 215, [999,1001] over 5001 81 81 78 81 / 179 146 206 251,
    //     [2001,2003] over 301 31 30 31 30 / 72 62 54 56, [4099,515] over 259 27 25 27 26 / 32 53 36 43; refused: [700,701] over 703 24 24 24 24 / 26 33 27 33
    //   shares: [256,1024] over 32000 110 108 110 110 / 131 129 132 129; [576,128] over 93312 116 114 108 110 / 118 116 119 116
    //   rows of a convolution: [100352,128] over 3 x 192 122 / 166, [3136,256] over 3 x 384 30 / 27 (refused)
    const int most = (int)(kWorkspacePartialBytes / (kTile * kTile * sizeof(float)) / tiles);
    auto estimate = [&](int sh) {
        const long per_cu = (tiles * sh + cus - 1) / cus;
        const double slabs = (double)g.slabs / sh + 4.0;
        return (per_cu < 2 ? slabs : 0.8 * (double)per_cu * slabs) + (sh > 1 ? 4.0 + 0.013 * (double)(tiles * sh) : 0.0);
    };
    int shares = 1;
    for (int sh = 2; sh <= most && sh * 8 <= g.slabs; ++sh)
        if (estimate(sh) < estimate(shares)) shares = sh;
    if (long_rate && shares == 1 && g.K[0] >= 2048) fp32_rate = 115e6;
    double flops = 0.0;
    for (int s = 0; s < g.nseg; ++s) flops += 2.0 * ((g.M + 63) / 64 * 64) * ((g.N + 63) / 64 * 64) * (double)g.K[s];
    if (estimate(shares) > 0.97 * (flops / fp32_rate + beside)) return 0;
    return (long)g.slabs * (shares + 1) < (1L << 31) ? shares : 0;
}

int launch_split(SplitArgs& g, void (*kernel)(SplitArgs)) {
    const long tiles = (long)g.tiles_m * g.tiles_n;
    g.partials = (float*)(workspace() + kWorkspaceCounterBytes);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles * g.shares)), dim3(256), 0, stream(), g);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && g.shares > 1) {
        hipLaunchKernelGGL(sgemm_split_fold, dim3((unsigned)(tiles * 16)), dim3(256), 0, stream(), g);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return fail("sgemm launch failed: %s", hipGetErrorString(e));
    return 1;
}

bool split_enabled(int cus) {
    static const int enabled = getenv("DALI_HIP_GEMM_SPLIT") ? atoi(getenv("DALI_HIP_GEMM_SPLIT")) : 1;
    return enabled && cus >= 8;
}

}  // namespace

int sgemm_split(bool ta, bool tb, int M, int N, int nseg, const int* K, const float* const* A, const int* lda, const float* const* B, const int* ldb, float alpha,
                float beta, float* C, int ldc, const SgemmRowMap& map, int cus) {
    // (A sum of two products keeps the order of summation that the fused LSTM step has. What a pair stands for is not known here: two large
    // products that have nothing to do with a cell, or two filter rows of a convolution, stay on the fp32 kernels with it.)
    if (!split_enabled(cus) || nseg < 1 || nseg > kMaxTerms || nseg == 2 || M <= 64 || N <= 64 || K[0] <= 64) return 0;
    SplitArgs g = {};
    for (int s = 0; s < nseg; ++s) {
        // offsets within a slab are 32-bit
        const size_t a_span = (ta ? (size_t)kSlab * lda[s] + M : (size_t)kTile * lda[s] + kSlab), b_span = (tb ? (size_t)kTile * ldb[s] + kSlab : (size_t)kSlab * ldb[s] + N);
        if (K[s] < kSlab || a_span >= ((size_t)1 << 30) || b_span >= ((size_t)1 << 30)) return 0;
        g.A[s] = A[s];
        g.B[s] = B[s];
        g.lda[s] = lda[s];
        g.ldb[s] = ldb[s];
        g.K[s] = K[s];
        g.slabs += (K[s] + kSlab - 1) / kSlab;
    }
    g.nseg = nseg;
    g.M = M;
    g.N = N;
    g.C = C;
    g.ldc = ldc;
    g.alpha = alpha;
    g.beta = beta;
    g.map = map;
    g.tiles_m = (M + kTile - 1) / kTile;
    g.tiles_n = (N + kTile - 1) / kTile;
    const long tiles = (long)g.tiles_m * g.tiles_n;
    if (tiles > (1L << 24)) return 0;
    bool direct = true;  // the loads of the fp32 kernels can write LDS
    for (int s = 0; s < nseg; ++s) direct = direct && lda[s] % 4 == 0 && ldb[s] % 4 == 0 && (((uintptr_t)A[s] | (uintptr_t)B[s]) & 15) == 0;
    const long tiles64 = (long)((M + 63) / 64) * ((N + 63) / 64), rounds64 = (tiles64 + cus - 1) / cus;
    const bool fills = tiles <= cus && (double)tiles64 >= 0.95 * (double)(rounds64 * cus);
    const bool staged = nseg > 2 || map.on;
    g.shares = choose_shares(g, cus, staged ? 76e6 : !direct ? 55e6 : fills ? 135e6 : 112e6, !staged && direct && !fills);
    if (g.shares == 0) return 0;
    if (!ta && !tb) return launch_split(g, sgemm_split_kernel<false, false, kPlain>);
    if (ta && !tb) return launch_split(g, sgemm_split_kernel<true, false, kPlain>);
    if (!ta && tb) return launch_split(g, sgemm_split_kernel<false, true, kPlain>);
    return launch_split(g, sgemm_split_kernel<true, true, kPlain>);
}

// What a convolution reads and how it is cut, all but the operands' addresses; false: not a case for it. (A function of the extents alone, so that it can be asked
// before operands are laid out and a result is allocated.)
static bool plan_conv_nhwc(SplitArgs& g, bool filters_gradient, int n, int h, int w, int c, int f, int fh, int fw, int stride_h, int stride_w, int cus) {
    const int oh = (h - fh) / stride_h + 1, ow = (w - fw) / stride_w + 1;
    const long positions = (long)n * oh * ow, run = (long)fw * c;
    if (!split_enabled(cus) || h < fh || w < fw || (long)n * h * w * c >= (1L << 30) || positions * f >= (1L << 30) || (long)f * fh * run >= (1L << 30)) return false;
    g = {};
    SplitConv& cv = g.cv;
    cv.out_w = ow;
    cv.out_h = oh;
    cv.step = stride_w * c;
    cv.row = stride_h * w * c;
    cv.image = h * w * c;
    cv.run = (int)run;
    cv.line = w * c;
    auto divide_by = [](unsigned d, unsigned* m, int* shift) {
        int s = 0;
        while ((1ull << s) < d) ++s;
        *m = (unsigned)(((1ull << (31 + s)) + d - 1) / d);
        *shift = s;
    };
    cv.hw = (unsigned)(oh * ow);
    divide_by(cv.hw, &cv.hw_m, &cv.hw_s);
    divide_by((unsigned)ow, &cv.w_m, &cv.w_s);
    divide_by((unsigned)run, &cv.run_m, &cv.run_s);
    if (filters_gradient) {
        g.nseg = 1;
        g.lda[0] = f;
        g.K[0] = (int)positions;
        g.M = f;
        g.N = fh * (int)run;
    } else {
        if (fh > kMaxTerms) return false;
        g.nseg = fh;
        for (int s = 0; s < fh; ++s) {
            g.ldb[s] = fh * (int)run;
            g.K[s] = (int)run;
        }
        g.M = (int)positions;
        g.N = f;
    }
    if (g.M <= 64 || g.N <= 64 || g.K[0] <= 64) return false;
    for (int s = 0; s < g.nseg; ++s) g.slabs += (g.K[s] + kSlab - 1) / kSlab;
    g.ldc = g.N;
    g.alpha = 1.0f;
    g.tiles_m = (g.M + kTile - 1) / kTile;
    g.tiles_n = (g.N + kTile - 1) / kTile;
    if ((long)g.tiles_m * g.tiles_n > (1L << 24)) return false;
    // what it stands in for: a launch that forms a patch matrix, written and read at about 4.5 TB/s, and a product (off 16 bytes at 40 to 60 TFLOP/s); at stride 1 and
    // whole vectors of channels a padded copy of the image and a sum of products
    const double product = c % 4 == 0 && f % 4 == 0 ? 112e6 : 60e6, patches = 5.0 + 8.0 * (double)positions * (fh * run) / 4.5e6;
    const bool summed = !filters_gradient && stride_h == 1 && stride_w == 1 && c % 4 == 0;
    g.shares = choose_shares(g, cus, summed ? 76e6 : product, false, summed ? 5.0 + 8.0 * n * h * w * c / 4.5e6 : patches);
    return g.shares != 0;
}

// The convolution of a channels-last image [n, h, w, c] with filters [f, fh, fw, c], without padding, and the gradient of its filters, as products whose
// one operand is the image itself, read window by window: no patch matrix is written or read, and no padded copy of the image. `result`
// as the matrix product lays it out: [n, out_h, out_w, f] (filters_gradient: [f, fh, fw, c], from `out` [n, out_h, out_w, f]). Taken where the rule above takes
// the product of that size. 1: launched; 0: not a case for it (form the patch matrix); -1: failure (message set).
// What the product alone takes is left: us, image padded or patch matrix formed first / here, [32,56,56,64] with 128 filters of 3x3 147 / 107 and gradient 169 / 112, at stride
// 2 58 / 45 and 67 / 45; [8,64,64,33], 100 of 5x5 120 / 65 and 216 / 59; [32,56,56,128], 128 of 3x3 248 / 190 and 280 / 180; [64,28,28,256], 256 of 1x1 95 / 65 and 75 / 64.
int split_conv_nhwc(bool filters_gradient, int n, int h, int w, int c, int f, int fh, int fw, int stride_h, int stride_w, const float* image, const float* other,
                    float* result, int cus) {
    SplitArgs g;
    if (!plan_conv_nhwc(g, filters_gradient, n, h, w, c, f, fh, fw, stride_h, stride_w, cus)) return 0;
    for (int s = 0; s < g.nseg; ++s) {
        g.A[s] = filters_gradient ? other : image + (size_t)s * g.cv.line;
        g.B[s] = filters_gradient ? image : other + (size_t)s * g.cv.run;
    }
    g.C = result;
    return launch_split(g, filters_gradient ? sgemm_split_kernel<true, false, kFilters> : sgemm_split_kernel<false, true, kWindows>);
}

bool split_conv_nhwc_takes(bool filters_gradient, int n, int h, int w, int c, int f, int fh, int fw, int stride_h, int stride_w, int cus) {
    SplitArgs g;
    return plan_conv_nhwc(g, filters_gradient, n, h, w, c, f, fh, fw, stride_h, stride_w, cus);
}

}  // namespace dali_hip
