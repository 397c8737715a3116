// kernels_pyramid.hip -- gfx950 kernels for the Gaussian pyramid:
//   k_blur_h / k_blur_v : one separable pass of imageproc gaussian_blur_f32 on u8
//                         (called at src/sift.rs:159,1211), optional DoG epilogue
//                         (src/sift.rs:92-124,182-204) in the vertical pass.
//   k_resize_tall/_small: image resize_exact(.., Lanczos3) (src/sift.rs:83-88), both
//                         passes in one kernel; k_resize_v/_h: the two-pass form.
//   k_luma              : colour -> grey (image 0.25.6 to_luma8, the wasm canvas rule).
//
// Exactness: every pass computes, per output pixel, acc = 0; acc = acc + p_i * w_i
// in tap order with separate multiply and add (no FMA; the file is compiled with
// -ffp-contract=off and uses __fmul_rn/__fadd_rn), then truncates to u8 -- the
// reference's arithmetic, so the levels are bit-identical to it.
#include <algorithm>

#include "edge_words.h"
#include "sift_hip.h"
#include "sift_internal.h"

namespace sh {

namespace {

constexpr int kThreads = 256;
constexpr int kHTileH = 4;    // one row per wave
constexpr int kVTileW = 256;  // 64 lanes x 4 px
constexpr int kVRows = 4;     // rows per lane in k_blur_v (a tile: 4 waves x kVRows rows)

// The job of a tile (jobs[j].tile_begin <= tile < jobs[j+1].tile_begin); every
// launch's grid is its total tile count. With more than 4 jobs the proportional
// guess tile * njobs / total is checked first: it is exact when the jobs have
// equal tile counts (a batch of equal frames), and then the lookup is two
// independent loads instead of a chain of dependent ones; otherwise, and for
// other layouts, a binary search.
template <typename Job>
__device__ __forceinline__ int find_job(const Job* __restrict__ jobs, int njobs, int tile) {
    if (njobs > 4) {
        const int g = (int)(((long long)tile * njobs) / (long long)gridDim.x);
        if (g < njobs && jobs[g].tile_begin <= tile && (g + 1 == njobs || jobs[g + 1].tile_begin > tile))
            return g;
    }
    int lo = 0, hi = njobs - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].tile_begin <= tile) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// imageproc Clamp<f32> for u8 == Rust `as u8`: truncate, saturate at 0 and 255.
// Every caller converts a sum of products of non-negative values (pixel values
// and Gaussian taps, or the luma weights), which is never negative or NaN and
// stays far below 2^32: the conversion truncates and only the upper bound needs
// a test (two instructions instead of five).
__device__ __forceinline__ unsigned u8_trunc(float x) {
    return min((unsigned)x, 255u);
}

__device__ __forceinline__ float mul_add_exact(float acc, float a, float b) {
    return __fadd_rn(acc, __fmul_rn(a, b));
}

// Sums to bytes. v_cvt_pk_u8_f32 under round toward zero equals min((unsigned)x, 255)
// for every f32 x >= 0 (checked for all of them up to 2^33) and places the byte, one
// instruction where the conversion, the bound and the packing took three. The wave's
// f32 rounding mode is switched for it and back within one asm statement: the compiler
// does not know that other arithmetic depends on the mode, and can put none between.
#define SH_TRUNCATE "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 3\n\ts_nop 1\n\t"
#define SH_ROUND_EVEN "s_setreg_imm32_b32 hwreg(HW_REG_MODE, 0, 2), 0\n\ts_nop 1"
#define SH_BYTE0(d) "v_cvt_pk_u8_f32 %" #d ", %" #d ", 0, 0\n\t"
#define SH_BYTE(d, s, k) "v_cvt_pk_u8_f32 %" #d ", %" #s ", " #k ", %" #d "\n\t"

// Word k of v: the bytes of a[4 k] .. a[4 k + 3], none of them negative.
__device__ __forceinline__ void pack_u8(const float (&a)[4], unsigned (&v)[1]) {
    float w = a[0];
    asm(SH_TRUNCATE SH_BYTE0(0) SH_BYTE(0, 1, 1) SH_BYTE(0, 2, 2) SH_BYTE(0, 3, 3) SH_ROUND_EVEN
        : "+&v"(w) : "v"(a[1]), "v"(a[2]), "v"(a[3]));
    v[0] = __float_as_uint(w);
}
__device__ __forceinline__ void pack_u8(const float (&a)[8], unsigned (&v)[2]) {
    float w0 = a[0], w1 = a[4];
    asm(SH_TRUNCATE SH_BYTE0(0) SH_BYTE0(1) SH_BYTE(0, 2, 1) SH_BYTE(1, 3, 1) SH_BYTE(0, 4, 2) SH_BYTE(1, 5, 2)
            SH_BYTE(0, 6, 3) SH_BYTE(1, 7, 3) SH_ROUND_EVEN
        : "+&v"(w0), "+&v"(w1) : "v"(a[1]), "v"(a[5]), "v"(a[2]), "v"(a[6]), "v"(a[3]), "v"(a[7]));
    v[0] = __float_as_uint(w0);
    v[1] = __float_as_uint(w1);
}
__device__ __forceinline__ void pack_u8(const float (&a)[16], unsigned (&v)[4]) {
    float w0 = a[0], w1 = a[4], w2 = a[8], w3 = a[12];
    asm(SH_TRUNCATE SH_BYTE0(0) SH_BYTE0(1) SH_BYTE0(2) SH_BYTE0(3)
            SH_BYTE(0, 4, 1) SH_BYTE(1, 5, 1) SH_BYTE(2, 6, 1) SH_BYTE(3, 7, 1)
            SH_BYTE(0, 8, 2) SH_BYTE(1, 9, 2) SH_BYTE(2, 10, 2) SH_BYTE(3, 11, 2)
            SH_BYTE(0, 12, 3) SH_BYTE(1, 13, 3) SH_BYTE(2, 14, 3) SH_BYTE(3, 15, 3) SH_ROUND_EVEN
        : "+&v"(w0), "+&v"(w1), "+&v"(w2), "+&v"(w3)
        : "v"(a[1]), "v"(a[5]), "v"(a[9]), "v"(a[13]), "v"(a[2]), "v"(a[6]), "v"(a[10]), "v"(a[14]),
          "v"(a[3]), "v"(a[7]), "v"(a[11]), "v"(a[15]));
    v[0] = __float_as_uint(w0);
    v[1] = __float_as_uint(w1);
    v[2] = __float_as_uint(w2);
    v[3] = __float_as_uint(w3);
}
// Byte 0 of v[k]: that of a[k].
__device__ __forceinline__ void each_u8(const float (&a)[2], unsigned (&v)[2]) {
    float w0 = a[0], w1 = a[1];
    asm(SH_TRUNCATE SH_BYTE0(0) SH_BYTE0(1) SH_ROUND_EVEN : "+&v"(w0), "+&v"(w1));
    v[0] = __float_as_uint(w0);
    v[1] = __float_as_uint(w1);
}
__device__ __forceinline__ void each_u8(const float (&a)[4], unsigned (&v)[4]) {
    float w0 = a[0], w1 = a[1], w2 = a[2], w3 = a[3];
    asm(SH_TRUNCATE SH_BYTE0(0) SH_BYTE0(1) SH_BYTE0(2) SH_BYTE0(3) SH_ROUND_EVEN
        : "+&v"(w0), "+&v"(w1), "+&v"(w2), "+&v"(w3));
    v[0] = __float_as_uint(w0);
    v[1] = __float_as_uint(w1);
    v[2] = __float_as_uint(w2);
    v[3] = __float_as_uint(w3);
}
// Byte 0 of v[k]: round(clamp(a[k], 0, 255)) of any sum, as a[k] + 0.5 and the
// conversion, both toward zero. The sum cannot reach an integer that the exact one does
// not, and negative sums give 0 (checked for every f32 up to 2^15).
#define SH_HALF(d) "v_add_f32 %" #d ", 0.5, %" #d "\n\t"
__device__ __forceinline__ void round_u8(const float (&a)[4], unsigned (&v)[4]) {
    float w0 = a[0], w1 = a[1], w2 = a[2], w3 = a[3];
    asm(SH_TRUNCATE SH_HALF(0) SH_HALF(1) SH_HALF(2) SH_HALF(3) SH_BYTE0(0) SH_BYTE0(1) SH_BYTE0(2) SH_BYTE0(3)
            SH_ROUND_EVEN
        : "+&v"(w0), "+&v"(w1), "+&v"(w2), "+&v"(w3));
    v[0] = __float_as_uint(w0);
    v[1] = __float_as_uint(w1);
    v[2] = __float_as_uint(w2);
    v[3] = __float_as_uint(w3);
}
__device__ __forceinline__ unsigned round_u8(float a) {
    asm(SH_TRUNCATE SH_HALF(0) SH_BYTE0(0) SH_ROUND_EVEN : "+&v"(a));
    return __float_as_uint(a);
}

__device__ __forceinline__ float q255(unsigned v) { return __fdiv_rn((float)v, 255.0f); }

// The tap tables are written by host copies before any launch and only read
// by kernels: reading them through the constant address space lets the
// wave-uniform tap loads go through scalar loads instead of vector loads.
typedef __attribute__((address_space(4))) const float ctap_t;
// Global memory (source rows): loads through it are global, not flat, loads.
typedef __attribute__((address_space(1))) const uint8_t gbyte_t;
__device__ __forceinline__ const ctap_t* as_const_taps(const float* p) {
    return (const ctap_t*)(p);
}

// ---------------------------------------------------------------------------
// Horizontal pass. Tile = (64*PX) columns x 4 rows; wave w computes row y0+w;
// lane l computes PX consecutive outputs. The row segment from the aligned word
// at or before x0-r (d = (x0-r) mod 4 elements early) is staged in LDS as f32
// with clamp-to-edge indexing (the reference's edge rule), one word of 4 pixels
// per lane and step, with pad words so that the lanes' reads, PX elements apart,
// fall in distinct banks: PX = 16 puts one pad word after every 16 elements
// (element e at e + e/16, lane stride 17 words), PX = 8 one after every 8
// (e + e/8, lane stride 9 words), PX = 2 one after every 32 (e + e/32). Either
// way a word's 4 pixels land in 4 consecutive slots.
// For PX = 8 and 16 and the tap counts of the default scale schedule (7 to 15
// taps) the taps are fully unrolled: the PX + n - 1 window inputs, elements
// base + d + k, sit at offsets hpad(d + k) from the lane's first slot (the same
// for every lane), so they are read once with immediate offsets, one code path
// per d, and every tap is a scalar register. PX = 16 gives each wave twice the
// arithmetic per staged row, against which the row's load latency is spread. Otherwise a register window of PX+4 inputs
// slides over the taps in blocks of 4; taps are zero-padded to a multiple of 4
// (p * 0 added to a non-negative sum leaves it unchanged), except that a single
// leftover tap is applied on its own, and are wave-uniform (scalar registers).
// ---------------------------------------------------------------------------
template <int PX>
__host__ __device__ __forceinline__ int hpad(int c) {
    return PX == 16 ? c + (c >> 4) : PX == 8 ? c + (c >> 3) : c + (c >> 5);
}

// NT taps over the window elements base + D + k, k < PX + NT - 1, at
// p[hpad(D + k)] (p = the slot of element base, base a multiple of PX, which is
// the padding period for PX = 8 and 16), in tap order per output; the first
// product is the first partial sum (0 + p * w0 is p * w0: p * w0 is never -0).
template <int PX, int NT, int D>
__device__ __forceinline__ void hconv_fixed(const float* __restrict__ p, const ctap_t* taps,
                                            float (&acc)[PX]) {
    constexpr int NW = PX + NT - 1;
    float win[NW];
#pragma unroll
    for (int k = 0; k < NW; k++) win[k] = p[hpad<PX>(D + k)];
    float wk[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) wk[k] = taps[k];
#pragma unroll
    for (int q = 0; q < PX; q++) acc[q] = __fmul_rn(win[q], wk[0]);
#pragma unroll
    for (int k = 1; k < NT; k++)
#pragma unroll
        for (int q = 0; q < PX; q++) acc[q] = mul_add_exact(acc[q], win[q + k], wk[k]);
}

template <int PX, int NT>
__device__ __forceinline__ void hconv_fixed_d(int d, const float* __restrict__ p,
                                              const ctap_t* taps, float (&acc)[PX]) {
    switch (d) {
        case 0: hconv_fixed<PX, NT, 0>(p, taps, acc); break;
        case 1: hconv_fixed<PX, NT, 1>(p, taps, acc); break;
        case 2: hconv_fixed<PX, NT, 2>(p, taps, acc); break;
        default: hconv_fixed<PX, NT, 3>(p, taps, acc); break;
    }
}

// Any tap count: taps in blocks of 4 (taps beyond ntaps are zero, <= ntaps_pad).
// When one tap is left over (ntaps = 4k + 1), it is applied after the blocks from
// the window registers, which then hold row[base + 4k ..], instead of a block of
// three zero taps.
template <int PX>
__device__ __forceinline__ void hconv_blocks(const float* __restrict__ row, int base,
                                             const ctap_t* taps, int ntaps, float (&acc)[PX]) {
    const bool one_left = (ntaps & 3) == 1;
    const int nb = one_left ? (ntaps & ~3) : ((ntaps + 3) & ~3);
#pragma unroll
    for (int q = 0; q < PX; q++) acc[q] = 0.0f;
    float win[PX + 4];
#pragma unroll
    for (int k = 0; k < PX; k++) win[k] = row[hpad<PX>(base + k)];
    for (int b = 0; b < nb; b += 4) {
#pragma unroll
        for (int k = 0; k < 4; k++) win[PX + k] = row[hpad<PX>(base + PX + b + k)];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float wk = taps[b + k];
#pragma unroll
            for (int q = 0; q < PX; q++) acc[q] = mul_add_exact(acc[q], win[q + k], wk);
        }
#pragma unroll
        for (int k = 0; k < PX; k++) win[k] = win[k + 4];
    }
    if (one_left) {
        const float wk = taps[nb];
#pragma unroll
        for (int q = 0; q < PX; q++) acc[q] = mul_add_exact(acc[q], win[q], wk);
    }
}

template <int PX>
__global__ __launch_bounds__(kThreads) void k_blur_h(const BlurJob* __restrict__ jobs, int njobs) {
    extern __shared__ float lds[];
    constexpr int TW = 64 * PX;
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int j = find_job(jobs, njobs, tile);
    const BlurJob& J = jobs[j];
    const int t = tile - J.tile_begin;
    const int tx = t % J.tiles_x, ty = t / J.tiles_x;
    const int x0 = tx * TW, y0 = ty * kHTileH;
    const int w = J.w, h = J.h;
    const int r = J.ntaps >> 1;
    const int npad = J.ntaps_pad;
    const int rowlen = TW + npad + 8;
    const int rowstride = hpad<PX>(rowlen + 8) + 1;

    // Wave w stages row y0+w, the words [ws, ws + 4 * nwords) with ws the aligned
    // word start at or before x0-r (clamped) as f32, and reads only that row, so
    // the waves need no work-group barrier. Aligned 4-byte words fully inside
    // [0, w) are read with one load; words at the image edges (and unaligned
    // sources) fall back to clamped bytes. The first KU words of a lane are all
    // loaded before any is written, so their loads overlap.
    const int xs = x0 - r;
    const int ws = xs & ~3;                      // first word start (may be < 0)
    const int d = xs - ws;                       // element base + k is staged element base + d + k
    const int nwords = (d + rowlen + 3) >> 2;
    const bool aligned = (((uintptr_t)J.src | (uintptr_t)J.src_pitch) & 3) == 0;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int y = y0 + wave;
    if (y >= h) return;
    gbyte_t* src = (gbyte_t*)J.src + (size_t)y * J.src_pitch;
    float* dstrow = lds + wave * rowstride;
    auto fetch = [&](int k) -> unsigned {
        const int xw = ws + 4 * k;
        if (aligned && xw >= 0 && xw + 4 <= w)
            return *(__attribute__((address_space(1))) const unsigned*)(src + xw);
        unsigned u = 0;
#pragma unroll
        for (int b = 0; b < 4; b++) u |= (unsigned)src[min(max(xw + b, 0), w - 1)] << (8 * b);
        return u;
    };
    auto put = [&](int k, unsigned u) {  // pixels 4k..4k+3: 4 consecutive slots
        float* dp = dstrow + hpad<PX>(4 * k);
        dp[0] = (float)(u & 0xff);
        dp[1] = (float)((u >> 8) & 0xff);
        dp[2] = (float)((u >> 16) & 0xff);
        dp[3] = (float)(u >> 24);
    };
    constexpr int KU = PX == 16 ? 5 : PX == 8 ? 3 : 1;  // words per lane of a row of the default kernels
    unsigned uw[KU];
#pragma unroll
    for (int i = 0; i < KU; i++)
        if (lane + 64 * i < nwords) uw[i] = fetch(lane + 64 * i);
#pragma unroll
    for (int i = 0; i < KU; i++)
        if (lane + 64 * i < nwords) put(lane + 64 * i, uw[i]);
    for (int k = lane + 64 * KU; k < nwords; k += 64) put(k, fetch(k));
    // the row's LDS writes are complete and visible to the wave before its reads
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* row = lds + wave * rowstride;
    const int base = lane * PX;
    const ctap_t* taps = as_const_taps(J.taps);
    float acc[PX];
    bool fixed = false;
    if constexpr (PX >= 8) {
        const float* p = row + hpad<PX>(base);
        fixed = true;
        switch (J.ntaps) {
            case 7: hconv_fixed_d<PX, 7>(d, p, taps, acc); break;
            case 9: hconv_fixed_d<PX, 9>(d, p, taps, acc); break;
            case 11: hconv_fixed_d<PX, 11>(d, p, taps, acc); break;
            case 13: hconv_fixed_d<PX, 13>(d, p, taps, acc); break;
            case 15: hconv_fixed_d<PX, 15>(d, p, taps, acc); break;
            default: fixed = false;
        }
    }
    if (!fixed) hconv_blocks<PX>(row, base + d, taps, J.ntaps, acc);

    const int x = x0 + base;
    if (x >= w) return;
    uint8_t* dst = J.dst + (size_t)y * J.dst_pitch + x;
    if constexpr (PX >= 8) {
        unsigned v[PX / 4];
        pack_u8(acc, v);
        if (x + PX <= w) {
            if constexpr (PX == 8) *(uint2*)dst = make_uint2(v[0], v[1]);
            else *(uint4*)dst = make_uint4(v[0], v[1], v[2], v[3]);
            return;
        }
#pragma unroll
        for (int q = 0; q < PX; q++)
            if (x + q < w) dst[q] = (uint8_t)(v[q / 4] >> (8 * (q & 3)));
    } else {
        unsigned v[PX];
        each_u8(acc, v);
#pragma unroll
        for (int q = 0; q < PX; q++)
            if (x + q < w) dst[q] = (uint8_t)v[q];
    }
}

// ---------------------------------------------------------------------------
// Vertical pass, wide octaves. Tile = 256 columns x 16 rows; lane l owns columns
// x0+4l..+3 (one u32 load per input row), wave w owns rows y0+4w..+3. For the
// tap counts of the default scale schedule (7 to 15) the taps are unrolled and
// each input row is loaded and converted once; otherwise a register window of
// 8 input rows x 4 columns slides over the taps in blocks of 4.
// Optional DoG epilogue: dog = q[G_s] - q[G_{s-1}], q[v] = v / 255.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void cvt4(unsigned v, float* o) {
    o[0] = (float)(v & 0xff);
    o[1] = (float)((v >> 8) & 0xff);
    o[2] = (float)((v >> 16) & 0xff);
    o[3] = (float)(v >> 24);
}

// v: four pixels of row y from column x, packed; kDog: with the DoG row where the job
// has one.
template <bool kDog>
__device__ __forceinline__ void store_row4(const BlurJob& J, int y, int x, unsigned v) {
    uint8_t* dst = J.dst + (size_t)y * J.dst_pitch + x;
    const int w = J.w;
    if (x + 4 <= w) {
        *(unsigned*)dst = v;
    } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (x + c < w) dst[c] = (uint8_t)(v >> (8 * c));
    }
    if (kDog && J.dog) {
        const uint8_t* prev = J.prev + (size_t)y * J.dst_pitch + x;
        float* dg = J.dog + (size_t)y * J.dog_pitch + x;
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (x + c < w) dg[c] = q255((v >> (8 * c)) & 0xff) - q255(prev[c]);
    }
}

// RV rows of four sums as packed bytes, four rows at a time.
template <int RV>
__device__ __forceinline__ void trunc_rows(const float (&acc)[RV][4], unsigned (&res)[RV]) {
#pragma unroll
    for (int q = 0; q < RV; q += 4) {
        float a[16];
        unsigned v[4];
#pragma unroll
        for (int i = 0; i < 16; i++) a[i] = acc[q + i / 4][i & 3];
        pack_u8(a, v);
#pragma unroll
        for (int i = 0; i < 4; i++) res[q + i] = v[i];
    }
}

// Any tap count: a register window of RV input rows x 4 columns slides over the
// taps in blocks of RV; the remaining taps (< RV) are applied one at a time.
template <int RV>
__device__ __forceinline__ void vconv_blocks(const uint8_t* col, int pitch, int y0, int h, int n,
                                             const ctap_t* taps, float (&acc)[RV][4]) {
#pragma unroll
    for (int q = 0; q < RV; q++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[q][c] = 0.0f;

    float lo[RV][4];
#pragma unroll
    for (int i = 0; i < RV; i++) {
        int yy = min(max(y0 + i, 0), h - 1);
        cvt4(*(const unsigned*)(col + (size_t)yy * pitch), lo[i]);
    }
    int b = 0;
    for (; b + RV <= n; b += RV) {
        float hi[RV][4];
#pragma unroll
        for (int i = 0; i < RV; i++) {
            int yy = min(max(y0 + b + RV + i, 0), h - 1);
            cvt4(*(const unsigned*)(col + (size_t)yy * pitch), hi[i]);
        }
#pragma unroll
        for (int k = 0; k < RV; k++) {
            const float wk = taps[b + k];
#pragma unroll
            for (int q = 0; q < RV; q++) {
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    const float p = (q + k < RV) ? lo[q + k][c] : hi[q + k - RV][c];
                    acc[q][c] = mul_add_exact(acc[q][c], p, wk);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < RV; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) lo[i][c] = hi[i][c];
    }
    // remaining taps (< RV): lo holds rows y0 + b .. + RV - 1
    for (; b < n; b++) {
        const float wk = taps[b];
#pragma unroll
        for (int q = 0; q < RV; q++)
#pragma unroll
            for (int c = 0; c < 4; c++) acc[q][c] = mul_add_exact(acc[q][c], lo[q][c], wk);
#pragma unroll
        for (int i = 0; i < RV - 1; i++)
#pragma unroll
            for (int c = 0; c < 4; c++) lo[i][c] = lo[i + 1][c];
        int yy = min(max(y0 + b + RV, 0), h - 1);
        cvt4(*(const unsigned*)(col + (size_t)yy * pitch), lo[RV - 1]);
    }
}

// NT taps, fully unrolled: the RV + NT - 1 input rows y0.. (clamped; y0 is
// wave-uniform, so each row is one scalar base plus the lane's column offset)
// are streamed once in increasing order, and input row i adds tap i - q to
// output row q -- per output, the taps in tap order. The first product is the
// first partial sum (p * w0 is never -0).
template <int RV, int NT>
__device__ __forceinline__ void vconv_fixed(const uint8_t* src, unsigned x, int pitch, int y0,
                                            int h, const ctap_t* taps, float (&acc)[RV][4]) {
    float wk[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) wk[k] = taps[k];
#pragma unroll
    for (int i = 0; i < RV + NT - 1; i++) {
        const int yy = min(max(y0 + i, 0), h - 1);
        gbyte_t* rowp = (gbyte_t*)src + (size_t)yy * pitch;
        float p[4];
        cvt4(*(__attribute__((address_space(1))) const unsigned*)(rowp + x), p);
#pragma unroll
        for (int q = 0; q < RV; q++) {
            const int k = i - q;
            if (k < 0 || k >= NT) continue;
#pragma unroll
            for (int c = 0; c < 4; c++)
                acc[q][c] = k == 0 ? __fmul_rn(p[c], wk[0]) : mul_add_exact(acc[q][c], p[c], wk[k]);
        }
    }
}

// RV = kVRows (4) rows per lane: tiles of 256 x 16. RV = 8 (the "v8" form, for
// the unrolled tap counts only): 256 x 32 tiles, twice the arithmetic per wave
// against the same load latency, and 8 + n - 1 input rows per 8 outputs rows.
template <int RV>
__global__ __launch_bounds__(kThreads) void k_blur_v(const BlurJob* __restrict__ jobs, int njobs) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int j = find_job(jobs, njobs, tile);
    const BlurJob& J = jobs[j];
    const int t = tile - J.tile_begin;
    const int tx = t % J.tiles_x, ty = t / J.tiles_x;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int w = J.w, h = J.h;
    const int x = tx * kVTileW + lane * 4;
    const int yb = ty * (4 * RV) + wave * RV;
    if (yb >= h || x >= w) return;
    const int r = J.ntaps >> 1;
    const int n = J.ntaps;
    const int pitch = J.src_pitch;
    const ctap_t* taps = as_const_taps(J.taps);

    float acc[RV][4];
    bool fixed = true;
    switch (n) {
        case 7: vconv_fixed<RV, 7>(J.src, x, pitch, yb - r, h, taps, acc); break;
        case 9: vconv_fixed<RV, 9>(J.src, x, pitch, yb - r, h, taps, acc); break;
        case 11: vconv_fixed<RV, 11>(J.src, x, pitch, yb - r, h, taps, acc); break;
        case 13: vconv_fixed<RV, 13>(J.src, x, pitch, yb - r, h, taps, acc); break;
        case 15: vconv_fixed<RV, 15>(J.src, x, pitch, yb - r, h, taps, acc); break;
        default: fixed = false;
    }
    if constexpr (RV == kVRows) {
        if (!fixed) vconv_blocks<RV>(J.src + x, pitch, yb - r, h, n, taps, acc);
    }
    unsigned res[RV];
    trunc_rows(acc, res);
#pragma unroll
    for (int q = 0; q < RV; q++) {
        const int y = yb + q;
        if (y >= h) break;
        store_row4<true>(J, y, x, res[q]);
    }
}

// ---------------------------------------------------------------------------
// Both passes of one blur in one kernel, for kernels of 5 to kHvMaxTaps taps. A
// work-group makes a tile of TW columns x TH rows: the horizontal pass of the
// tile's TH + 2r input rows (clamped to the image) goes to LDS as bytes, and the
// vertical pass reads them there, so the level between the passes, its write and
// its read, never leave the CU, and a level takes one launch.
// Horizontal: TW / PX lanes per row, PX outputs per lane, straight from global
// memory: a lane loads the aligned words of its PX + 2 kHalo window bytes (its
// neighbours' loads hit L1) and needs no LDS or exchange. In tiles at the left or
// right edge the word addresses are clamped and the bytes past the edge replaced
// by one v_perm per word (edge_words.h: no byte past the row's last pixel is read).
// Vertical: RV rows x 4 columns (256-column tiles) or x 1 column (64) per lane,
// each staged row read and converted once, as in k_blur_v.
// Bound: the exact multiply and add of every tap; the staged rows' 2r / TH extra
// horizontal work pays for the saved level. 64 levels of 1920 x 1080, 7 / 15 / 21
// taps: 114 / 201 / 289 us against 149 / 232 / 338 us of the best two-pass forms;
// one level of 640 x 480, 9 / 33 taps (of which about 6 us are the launch and its
// event): 6.2 / 8.4 against 12.4 us; 33 taps at 480 x 270 are the worst case met
// (48.5 against 42.7 us at 64 levels, for the tiles that do not fit the level).
// ---------------------------------------------------------------------------
template <int NT, int TW, int PX, int RV, int TH>
__device__ __forceinline__ void blur_hv_tile(const BlurJob& J, int x0, int y0, uint8_t* rows) {
    constexpr int R = NT / 2, kHalo = R <= 8 ? 8 : 16, NW = (PX + 2 * kHalo) / 4;
    constexpr int kLanes = TW / PX;               // lanes per row
    constexpr int kPassRows = kThreads / kLanes;  // rows of one pass of the work-group
    const int w = J.w, h = J.h;
    const unsigned pitch = J.src_pitch;
    const ctap_t* taps = as_const_taps(J.taps);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xl = (tid % kLanes) * PX;  // the lane's first column in the tile
    const bool inside = x0 >= kHalo && x0 + TW + kHalo <= w;
    const EdgeRow edge = edge_row(w);
    float wk[NT];
#pragma unroll
    for (int k = 0; k < NT; k++) wk[k] = taps[k];
#pragma unroll 1
    for (int r0 = 0; r0 < TH + 2 * R; r0 += kPassRows) {
        const int row = r0 + tid / kLanes;
        if (row >= TH + 2 * R) break;
        const int yy = min(max(y0 - R + row, 0), h - 1);
        gbyte_t* src = (gbyte_t*)J.src + (size_t)yy * pitch;
        const int xb = x0 + xl - kHalo;
        unsigned u[NW];
        if (inside) {
#pragma unroll
            for (int k = 0; k < NW; k++) u[k] = *(__attribute__((address_space(1))) const unsigned*)(src + xb + 4 * k);
        } else {
#pragma unroll
            for (int k = 0; k < NW; k++)
                u[k] = ((const __attribute__((address_space(1))) UnalignedWord*)(src + edge.at(xb + 4 * k)))->v;
#pragma unroll
            for (int k = 0; k < NW; k++) u[k] = __builtin_amdgcn_perm(u[k], u[k], edge.sel(xb + 4 * k));
        }
        float win[PX + NT - 1];
#pragma unroll
        for (int k = 0; k < PX + NT - 1; k++) {
            constexpr int o = kHalo - R;
            win[k] = (float)((u[(o + k) / 4] >> (8 * ((o + k) & 3))) & 0xff);
        }
        float acc[PX];
#pragma unroll
        for (int q = 0; q < PX; q++) acc[q] = __fmul_rn(win[q], wk[0]);
#pragma unroll
        for (int k = 1; k < NT; k++)
#pragma unroll
            for (int q = 0; q < PX; q++) acc[q] = mul_add_exact(acc[q], win[q + k], wk[k]);
        unsigned v[PX / 4];
        pack_u8(acc, v);
        uint8_t* to = rows + row * TW + xl;
        if constexpr (PX == 16) *(uint4*)to = make_uint4(v[0], v[1], v[2], v[3]);
        else if constexpr (PX == 8) *(uint2*)to = make_uint2(v[0], v[1]);
        else *(unsigned*)to = v[0];
    }
    __syncthreads();
    if constexpr (TW == 64) {
        static_assert(TH == RV * kThreads / 64, "one group of rows per wave");
        const int x = x0 + lane, yb = y0 + wave * RV;
        if (x >= w || yb >= h) return;
        const uint8_t* col = rows + wave * RV * TW + lane;
        float acc[RV];
#pragma unroll
        for (int i = 0; i < RV + NT - 1; i++) {
            const float p = (float)col[i * TW];
#pragma unroll
            for (int q = 0; q < RV; q++) {
                const int k = i - q;
                if (k < 0 || k >= NT) continue;
                acc[q] = k == 0 ? __fmul_rn(p, wk[0]) : mul_add_exact(acc[q], p, wk[k]);
            }
        }
        unsigned v[RV];
        each_u8(acc, v);
#pragma unroll
        for (int q = 0; q < RV; q++)
            if (yb + q < h) J.dst[(size_t)(yb + q) * J.dst_pitch + x] = (uint8_t)v[q];
        return;
    }
    const int x = x0 + 4 * lane;
    for (int g = wave; g < TH / RV; g += kThreads / 64) {
        const int yb = y0 + g * RV;
        if (yb >= h) break;
        const unsigned* col = (const unsigned*)rows + (g * RV) * (kVTileW / 4) + lane;
        float acc[RV][4];
#pragma unroll
        for (int i = 0; i < RV + NT - 1; i++) {
            float p[4];
            cvt4(col[i * (kVTileW / 4)], p);
#pragma unroll
            for (int q = 0; q < RV; q++) {
                const int k = i - q;
                if (k < 0 || k >= NT) continue;
#pragma unroll
                for (int c = 0; c < 4; c++)
                    acc[q][c] = k == 0 ? __fmul_rn(p[c], wk[0]) : mul_add_exact(acc[q][c], p[c], wk[k]);
            }
        }
        unsigned res[RV];
        trunc_rows(acc, res);
#pragma unroll
        for (int q = 0; q < RV; q++)
            if (yb + q < h && x < w) store_row4<false>(J, yb + q, x, res[q]);
    }
}

// Large launches: 256 x 64 tiles, the short and the long tap counts apart (77 and
// 85 VGPRs).
template <bool kLong>
__global__ __launch_bounds__(kThreads) void k_blur_hv(const BlurJob* __restrict__ jobs, int njobs) {
    constexpr int TW = kHvTileW, TH = kHvTileH;
    __shared__ __align__(16) uint8_t rows[(TH + (kLong ? kHvMaxTaps : kHvShortTaps) - 1) * TW];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x0 = (t % J.tiles_x) * TW, y0 = (t / J.tiles_x) * TH;
    if constexpr (!kLong) {
        switch (J.ntaps) {
            case 5: blur_hv_tile<5, TW, 16, 8, TH>(J, x0, y0, rows); break;
            case 7: blur_hv_tile<7, TW, 16, 8, TH>(J, x0, y0, rows); break;
            case 9: blur_hv_tile<9, TW, 16, 8, TH>(J, x0, y0, rows); break;
            case 11: blur_hv_tile<11, TW, 16, 8, TH>(J, x0, y0, rows); break;
            case 13: blur_hv_tile<13, TW, 16, 8, TH>(J, x0, y0, rows); break;
            default: blur_hv_tile<15, TW, 16, 8, TH>(J, x0, y0, rows); break;
        }
    } else {
        switch (J.ntaps) {
            case 17: blur_hv_tile<17, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 19: blur_hv_tile<19, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 21: blur_hv_tile<21, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 23: blur_hv_tile<23, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 25: blur_hv_tile<25, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 27: blur_hv_tile<27, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 29: blur_hv_tile<29, TW, 8, 8, TH>(J, x0, y0, rows); break;
            case 31: blur_hv_tile<31, TW, 8, 8, TH>(J, x0, y0, rows); break;
            default: blur_hv_tile<33, TW, 8, 8, TH>(J, x0, y0, rows); break;
        }
    }
}

// Small launches (single frames, small batches, deep octaves): 64 x 16 tiles of
// any of the tap counts. What counts there is the number of instructions of one
// wave (a wave alone on its SIMD issues one every 8 cycles), so a lane makes few
// outputs.
__global__ __launch_bounds__(kThreads) void k_blur_hv_small(const BlurJob* __restrict__ jobs, int njobs) {
    constexpr int TW = kHvSmallW, TH = kHvSmallH;
    __shared__ __align__(16) uint8_t rows[(TH + kHvMaxTaps - 1) * TW];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x0 = (t % J.tiles_x) * TW, y0 = (t / J.tiles_x) * TH;
    switch (J.ntaps) {
        case 5: blur_hv_tile<5, TW, 8, 4, TH>(J, x0, y0, rows); break;
        case 7: blur_hv_tile<7, TW, 8, 4, TH>(J, x0, y0, rows); break;
        case 9: blur_hv_tile<9, TW, 8, 4, TH>(J, x0, y0, rows); break;
        case 11: blur_hv_tile<11, TW, 8, 4, TH>(J, x0, y0, rows); break;
        case 13: blur_hv_tile<13, TW, 8, 4, TH>(J, x0, y0, rows); break;
        case 15: blur_hv_tile<15, TW, 8, 4, TH>(J, x0, y0, rows); break;
        case 17: blur_hv_tile<17, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 19: blur_hv_tile<19, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 21: blur_hv_tile<21, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 23: blur_hv_tile<23, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 25: blur_hv_tile<25, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 27: blur_hv_tile<27, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 29: blur_hv_tile<29, TW, 4, 4, TH>(J, x0, y0, rows); break;
        case 31: blur_hv_tile<31, TW, 4, 4, TH>(J, x0, y0, rows); break;
        default: blur_hv_tile<33, TW, 4, 4, TH>(J, x0, y0, rows); break;
    }
}

// ---------------------------------------------------------------------------
// Vertical pass, narrow octaves (and wide kernels). Tile = 64 columns x 16 rows;
// lane = column, wave w owns rows y0+4w..+3. The tile's input rows
// [y0-r, y0+16+r), clamped, are staged once in LDS as u8 (at most min(h, 16+2r)
// distinct rows, so the LDS footprint stays small even when r >> h).
// ---------------------------------------------------------------------------
constexpr int kVnTileW = 64, kVnTileH = 16;

__global__ __launch_bounds__(kThreads) void k_blur_v_narrow(const BlurJob* __restrict__ jobs,
                                                            int njobs) {
    extern __shared__ uint8_t vl[];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int j = find_job(jobs, njobs, tile);
    const BlurJob& J = jobs[j];
    const int t = tile - J.tile_begin;
    const int tx = t % J.tiles_x, ty = t / J.tiles_x;
    const int w = J.w, h = J.h;
    const int r = J.ntaps >> 1;
    const int n = J.ntaps;
    const int x0 = tx * kVnTileW, y0 = ty * kVnTileH;
    const int rlo = max(y0 - r, 0), rhi = min(y0 + kVnTileH + r, h);  // distinct rows [rlo, rhi)
    const int nrows = rhi - rlo;
    for (int i = threadIdx.x; i < nrows * kVnTileW; i += kThreads) {
        const int rr = i / kVnTileW, c = i - rr * kVnTileW;
        const int x = min(x0 + c, w - 1);
        vl[i] = J.src[(size_t)(rlo + rr) * J.src_pitch + x];
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int x = x0 + lane;
    const int yb = y0 + wave * 4;
    if (x >= w || yb >= h) return;
    const ctap_t* taps = as_const_taps(J.taps);
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    float cur[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int yy = min(max(yb + q - r, 0), h - 1);
        cur[q] = (float)vl[(yy - rlo) * kVnTileW + lane];
    }
    for (int i = 0; i < n; i++) {
        const float wk = taps[i];
#pragma unroll
        for (int q = 0; q < 4; q++) acc[q] = mul_add_exact(acc[q], cur[q], wk);
#pragma unroll
        for (int q = 0; q < 3; q++) cur[q] = cur[q + 1];
        if (i + 1 < n) {  // next input row; stays inside the staged rows
            const int yy = min(max(yb + 4 + i - r, 0), h - 1);
            cur[3] = (float)vl[(yy - rlo) * kVnTileW + lane];
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int y = yb + q;
        if (y >= h) break;
        const unsigned v = u8_trunc(acc[q]);
        J.dst[(size_t)y * J.dst_pitch + x] = (uint8_t)v;
        if (J.dog)
            J.dog[(size_t)y * J.dog_pitch + x] = q255(v) - q255(J.prev[(size_t)y * J.dst_pitch + x]);
    }
}

// ---------------------------------------------------------------------------
// Small levels (the deep octaves: a few thousand pixels, blur radii up to
// several hundred): one output per lane, so each wave's serial tap chain is as
// short as it can be and the few tiles still spread over many waves.
// Tile = 64 columns x 4 rows, wave w computes row y0+w, lane l column x0+l.
// The taps (zero-padded to a multiple of 4) sit in LDS and are read four at a
// time by all lanes at once. Every output keeps the reference's tap order and
// separate f32 multiply and add.
// ---------------------------------------------------------------------------
constexpr int kSTileW = 64, kSTileH = 4;

// Horizontal: the clamped row segments [x0-r, x0+64+n4-r) of the tile's 4 rows
// are staged as f32 (segment stride seg_stride >= 64 + n4).
__global__ __launch_bounds__(kThreads) void k_blur_h_small(const BlurJob* __restrict__ jobs,
                                                           int njobs, int seg_stride) {
    extern __shared__ float sm[];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x0 = (t % J.tiles_x) * kSTileW, y0 = (t / J.tiles_x) * kSTileH;
    const int w = J.w, h = J.h, n = J.ntaps, r = n >> 1;
    const int n4 = (n + 3) & ~3;
    float* tp = sm;
    float* seg = sm + n4;
    for (int i = threadIdx.x; i < n4; i += kThreads) tp[i] = i < n ? J.taps[i] : 0.0f;
    const int segw = kSTileW + n4;
    const float inv_segw = 1.0f / (float)segw;
    for (int i = threadIdx.x; i < kSTileH * segw; i += kThreads) {
        const int rr = (int)(((float)i + 0.5f) * inv_segw), c = i - rr * segw;
        const int y = min(y0 + rr, h - 1);
        const int x = min(max(x0 - r + c, 0), w - 1);
        seg[rr * seg_stride + c] = (float)J.src[(size_t)y * J.src_pitch + x];
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int y = y0 + wave, x = x0 + lane;
    if (y >= h || x >= w) return;
    const float* sg = seg + wave * seg_stride + lane;
    float acc = 0.0f;
#pragma unroll 2
    for (int k = 0; k < n4; k += 4) {
        const float4 t4 = *reinterpret_cast<const float4*>(tp + k);
        acc = mul_add_exact(acc, sg[k], t4.x);
        acc = mul_add_exact(acc, sg[k + 1], t4.y);
        acc = mul_add_exact(acc, sg[k + 2], t4.z);
        acc = mul_add_exact(acc, sg[k + 3], t4.w);
    }
    J.dst[(size_t)y * J.dst_pitch + x] = (uint8_t)u8_trunc(acc);
}

// acc + p * tp[k] for k in [k0, k1) in order (one input value, a run of taps):
// the taps are read 4 at a time once k is a multiple of 4 (tp is 16-byte aligned).
__device__ __forceinline__ float run_const(float acc, float p, const float* tp, int k0, int k1) {
    int k = k0;
    for (; k < k1 && (k & 3); k++) acc = mul_add_exact(acc, p, tp[k]);
#pragma unroll 2
    for (; k + 4 <= k1; k += 4) {
        const float4 t4 = *reinterpret_cast<const float4*>(tp + k);
        acc = mul_add_exact(acc, p, t4.x);
        acc = mul_add_exact(acc, p, t4.y);
        acc = mul_add_exact(acc, p, t4.z);
        acc = mul_add_exact(acc, p, t4.w);
    }
    for (; k < k1; k++) acc = mul_add_exact(acc, p, tp[k]);
    return acc;
}

// Vertical: the tile's distinct input rows [max(0, y0-r), min(h, y0+4+r)) are
// staged (at most h rows): as f32 (k_blur_v_small, up to kSmallMaxRows rows), or
// as bytes (k_blur_v_small8: 4x the rows in the same LDS, so levels of a few
// hundred rows with radii of dozens of pixels, the middle octaves, also get one
// output per lane; each tap then converts its byte). For output row y, taps
// k < r-y read row 0 and taps k >= h+r-y read row h-1 (clamp to edge): those
// runs need no loads and their bounds are the same for the whole wave.
template <typename T>
__device__ __forceinline__ void blur_v_small_tile(const BlurJob* __restrict__ jobs, int njobs,
                                                  int max_taps4, float* sm) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x0 = (t % J.tiles_x) * kSTileW, y0 = (t / J.tiles_x) * kSTileH;
    const int w = J.w, h = J.h, n = J.ntaps, r = n >> 1;
    const int n4 = (n + 3) & ~3;
    float* tp = sm;
    T* col = reinterpret_cast<T*>(sm + max_taps4);
    for (int i = threadIdx.x; i < n4; i += kThreads) tp[i] = i < n ? J.taps[i] : 0.0f;
    const int rlo = max(y0 - r, 0), rhi = min(y0 + kSTileH + r, h);
    for (int i = threadIdx.x; i < (rhi - rlo) * kSTileW; i += kThreads) {
        const int rr = i >> 6, c = i & 63;
        col[i] = (T)J.src[(size_t)(rlo + rr) * J.src_pitch + min(x0 + c, w - 1)];
    }
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int y = y0 + wave, x = x0 + lane;
    if (y >= h || x >= w) return;
    const int ka = min(max(r - y, 0), n);      // taps reading row 0
    const int kc = max(min(h + r - y, n), ka);  // taps from kc on read row h-1
    float acc = 0.0f;
    if (ka > 0) acc = run_const(acc, (float)col[(0 - rlo) * kSTileW + lane], tp, 0, ka);
    const T* cp = col + (y - r - rlo) * kSTileW + lane;
#pragma unroll 4
    for (int k = ka; k < kc; k++) acc = mul_add_exact(acc, (float)cp[k * kSTileW], tp[k]);
    if (kc < n) acc = run_const(acc, (float)col[(h - 1 - rlo) * kSTileW + lane], tp, kc, n);
    const unsigned v = u8_trunc(acc);
    J.dst[(size_t)y * J.dst_pitch + x] = (uint8_t)v;
    if (J.dog)
        J.dog[(size_t)y * J.dog_pitch + x] = q255(v) - q255(J.prev[(size_t)y * J.dst_pitch + x]);
}

__global__ __launch_bounds__(kThreads) void k_blur_v_small(const BlurJob* __restrict__ jobs,
                                                           int njobs, int max_taps4) {
    extern __shared__ __align__(16) float sm[];
    blur_v_small_tile<float>(jobs, njobs, max_taps4, sm);
}

__global__ __launch_bounds__(kThreads) void k_blur_v_small8(const BlurJob* __restrict__ jobs,
                                                            int njobs, int max_taps4) {
    extern __shared__ __align__(16) float sm8[];
    blur_v_small_tile<uint8_t>(jobs, njobs, max_taps4, sm8);
}

// ---------------------------------------------------------------------------
// Both passes of a long blur on a small level in one kernel (the deep octaves of
// single frames and small batches: a few thousand pixels, dozens to hundreds of
// taps). A work-group of 1024 threads makes a tile of kDeepW columns and up to
// kDeepH rows (the level cut evenly). Its source rows, at most the level's, and
// the replicated columns its windows need are staged as f32; the horizontal sums
// of those rows go to LDS, the rows past the image are copies of the first and the
// last, and the vertical sums read them: both are the same loop of one tap value
// for all lanes, one input, a multiply and an add, without a bound in it.
// Bound: latency (a wave alone on its SIMD issues every 8 cycles, four waves share
// 2.5), so one output per lane and narrow tiles, whose extra horizontal rows cost
// nothing while CUs are idle. Per level, with about 6 us of launch and event (two
// of them in a pair of launches): 160 x 120, 51 taps 13.0 -> 8.8 us; 80 x 60, 101 taps
// 15.6 -> 8.5; 40 x 30, 199 taps 15.4 -> 9.6; 240 x 135, 101 taps 15.5 -> 12.4. The
// host keeps the one-pass forms where the tiles fill the GPU (64 levels of
// 240 x 135, 51 taps: 53 against 37 us) or one tile is long (120 x 67, 395 taps: 22.6
// against 21.4 us).
// ---------------------------------------------------------------------------
// Sum of the taps (padded with zeros to n4, a multiple of 4) over in[k * step].
__device__ __forceinline__ float deep_sum(const float* in, int step, const float* tp, int n4) {
    float acc = 0.0f;
#pragma unroll 4
    for (int k = 0; k < n4; k += 4) {
        const float4 t4 = *reinterpret_cast<const float4*>(tp + k);
        acc = mul_add_exact(acc, in[k * step], t4.x);
        acc = mul_add_exact(acc, in[(k + 1) * step], t4.y);
        acc = mul_add_exact(acc, in[(k + 2) * step], t4.z);
        acc = mul_add_exact(acc, in[(k + 3) * step], t4.w);
    }
    return acc;
}

__global__ __launch_bounds__(kDeepThreads) void k_blur_deep(const BlurJob* __restrict__ jobs, int njobs) {
    extern __shared__ __align__(16) float dsm[];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin, tid = threadIdx.x;
    const int w = J.w, h = J.h, n = J.ntaps, r = n >> 1, n4 = (n + 3) & ~3;
    const int tiles_y = J.tiles / J.tiles_x, th = (h + tiles_y - 1) / tiles_y;
    const int x0 = (t % J.tiles_x) * kDeepW, y0 = (t / J.tiles_x) * th;
    const int rows = min(th, h - y0);
    if (rows <= 0) return;
    const int rlo = max(y0 - r, 0), nr = min(y0 + rows + r, h) - rlo;
    const int segw = kDeepW + n4, stride = deep_stride(n4);
    float* const tp = dsm;
    float* const seg = dsm + n4;             // source rows rlo.., columns x0 - r.. (clamped)
    float* const ext = seg + nr * stride;    // horizontal sums of rows y0 - r.. (clamped), kDeepW wide
    for (int i = tid; i < n4; i += kDeepThreads) tp[i] = i < n ? J.taps[i] : 0.0f;
    // up to eight bytes of a thread in flight at once: one after the other they were
    // fourteen latencies in a row (the eight launches of a 1920x1080 frame 101 -> 89 us,
    // the five of 640x480 47 -> 43). Reading a block of taps and inputs ahead of the sums
    // below, in contrast, was slower (99 us): four waves a SIMD hide those already.
    const float inv = __builtin_amdgcn_rcpf((float)segw);
    const int total = nr * segw;
    // (32-bit offsets from the first staged row: the host keeps the staged rows'
    // span within them, whatever stride the caller's frame has)
    gbyte_t* const src =
        (gbyte_t*)J.src + (size_t)rlo * J.src_pitch;
    for (int i0 = tid; i0 < total; i0 += 8 * kDeepThreads) {
        unsigned v[8];
        int at[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int i = i0 + k * kDeepThreads;
            if (i < total) {
                const int rr = (int)(((float)i + 0.5f) * inv), c = i - rr * segw;
                at[k] = rr * stride + c;
                v[k] = src[(unsigned)(rr * J.src_pitch + min(max(x0 - r + c, 0), w - 1))];
            }
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (i0 + k * kDeepThreads < total) seg[at[k]] = (float)v[k];
    }
    __syncthreads();
    const int col = tid % kDeepW, first = rlo - (y0 - r);  // row rlo's place in ext
    for (int rr = tid / kDeepW; rr < nr; rr += kDeepThreads / kDeepW)
        ext[(first + rr) * kDeepW + col] = (float)u8_trunc(deep_sum(seg + rr * stride + col, 1, tp, n4));
    __syncthreads();
    for (int i = tid; i < (rows + n4) * kDeepW; i += kDeepThreads) {  // the rows past the image's
        const int e = i / kDeepW;
        if (e < first) ext[i] = ext[first * kDeepW + col];
        else if (e >= first + nr) ext[i] = ext[(first + nr - 1) * kDeepW + col];
    }
    __syncthreads();
    for (int y = tid / kDeepW; y < rows; y += kDeepThreads / kDeepW)
        if (x0 + col < w)
            J.dst[(size_t)(y0 + y) * J.dst_pitch + x0 + col] =
                (uint8_t)u8_trunc(deep_sum(ext + y * kDeepW + col, kDeepW, tp, n4));
}

// Exact thread-per-pixel passes for kernels too wide for the LDS row tile.
__global__ __launch_bounds__(kThreads) void k_blur_h_generic(const BlurJob* __restrict__ jobs,
                                                             int njobs) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x = (t % J.tiles_x) * kThreads + threadIdx.x, y = t / J.tiles_x;
    if (x >= J.w || y >= J.h) return;
    const int r = J.ntaps >> 1;
    const uint8_t* src = J.src + (size_t)y * J.src_pitch;
    float s = 0.0f;
    for (int i = 0; i < J.ntaps; i++) {
        int xx = min(max(x + i - r, 0), J.w - 1);
        s = mul_add_exact(s, (float)src[xx], J.taps[i]);
    }
    J.dst[(size_t)y * J.dst_pitch + x] = (uint8_t)u8_trunc(s);
}

__global__ __launch_bounds__(kThreads) void k_blur_v_generic(const BlurJob* __restrict__ jobs,
                                                             int njobs) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x = (t % J.tiles_x) * kThreads + threadIdx.x, y = t / J.tiles_x;
    if (x >= J.w || y >= J.h) return;
    const int r = J.ntaps >> 1;
    float s = 0.0f;
    for (int i = 0; i < J.ntaps; i++) {
        int yy = min(max(y + i - r, 0), J.h - 1);
        s = mul_add_exact(s, (float)J.src[(size_t)yy * J.src_pitch + x], J.taps[i]);
    }
    unsigned v = u8_trunc(s);
    J.dst[(size_t)y * J.dst_pitch + x] = (uint8_t)v;
    if (J.dog)
        J.dog[(size_t)y * J.dog_pitch + x] = q255(v) - q255(J.prev[(size_t)y * J.dst_pitch + x]);
}

// Level copy (blur sigma < 1e-4, src/sift.rs:149-150) with its (zero) DoG.
__global__ __launch_bounds__(kThreads) void k_copy_level(const BlurJob* __restrict__ jobs,
                                                         int njobs) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const BlurJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int x = (t % J.tiles_x) * kThreads + threadIdx.x, y = t / J.tiles_x;
    if (x >= J.w || y >= J.h) return;
    uint8_t v = J.src[(size_t)y * J.src_pitch + x];
    J.dst[(size_t)y * J.dst_pitch + x] = v;
    if (J.dog) J.dog[(size_t)y * J.dog_pitch + x] = q255(v) - q255(v);
}

// ---------------------------------------------------------------------------
// Colour -> grey before the pyramid. RGB8 / RGBA8: DynamicImage::to_luma8 of
// image 0.25.6 (color.rs rgb_to_luma: u32 sum 2126 R + 7152 G + 722 B, divided
// by 10000 with truncation; alpha dropped), the conversion at src/sift.rs:1202.
// LUMAA8: the luma byte. RGBA8_CANVAS: src/wasm.rs:88-94, f32
// (0.299 r + 0.587 g) + 0.114 b without FMA, then `as u8` (truncate, saturate).
// A lane converts 4 consecutive pixels of one row.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned luma_srgb(unsigned r, unsigned g, unsigned b) {
    return (2126u * r + 7152u * g + 722u * b) / 10000u;
}

__device__ __forceinline__ unsigned luma_canvas(unsigned r, unsigned g, unsigned b) {
    const float l = __fadd_rn(__fadd_rn(__fmul_rn(0.299f, (float)r), __fmul_rn(0.587f, (float)g)),
                              __fmul_rn(0.114f, (float)b));
    return u8_trunc(l);
}

__global__ __launch_bounds__(kThreads) void k_luma(const LumaJob* __restrict__ jobs, int njobs) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const LumaJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int y = t / J.tiles_x;
    const int x = (t % J.tiles_x) * kLumaTileW + threadIdx.x * 4;
    if (x >= J.w || y >= J.h) return;
    const int n = min(4, J.w - x);
    const uint8_t* src = J.src + (size_t)y * J.src_pitch;
    uint8_t* dst = J.dst + (size_t)y * J.dst_pitch + x;
    unsigned l[4] = {0u, 0u, 0u, 0u};
    const int f = J.format;
    const int bpp = f == SIFT_PIXEL_RGB8 ? 3 : f == SIFT_PIXEL_LUMAA8 ? 2 : f == SIFT_PIXEL_GRAY8 ? 1 : 4;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        if (k >= n) break;
        const uint8_t* p = src + (size_t)(x + k) * bpp;
        if (bpp >= 3) {
            const unsigned r = p[0], g = p[1], b = p[2];
            l[k] = f == SIFT_PIXEL_RGBA8_CANVAS ? luma_canvas(r, g, b) : luma_srgb(r, g, b);
        } else {
            l[k] = p[0];
        }
    }
    if (n == 4 && (((uintptr_t)dst) & 3) == 0) {
        *(unsigned*)dst = l[0] | (l[1] << 8) | (l[2] << 16) | (l[3] << 24);
    } else {
        for (int k = 0; k < n; k++) dst[k] = (uint8_t)l[k];
    }
}

// ---------------------------------------------------------------------------
// Lanczos3 resize (image 0.25.6 sample::resize): vertical pass into f32 rows
// (t += p * w in window order, unrounded), then horizontal pass with
// round(clamp(t, 0, 255)). Exact reference order (separate mul and add).
// Vertical: a thread computes 4 adjacent columns of one output row (one u32
// load per tap). Horizontal: a workgroup computes 256 outputs of one row from
// the input span they need, staged in LDS.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void k_resize_v(const ResizeJob* __restrict__ jobs,
                                                       int njobs) {
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const ResizeJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int oy = t / J.tiles_x;
    const int x = ((t % J.tiles_x) * kThreads + threadIdx.x) * 4;
    if (x >= J.in_w) return;
    const int l = J.left[oy], n = J.count[oy];
    const ctap_t* wr = as_const_taps(J.weights) + (size_t)oy * J.maxtaps;  // one row for the wave
    const uint8_t* src = J.src_u8 + (size_t)l * J.src_pitch + x;
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    int i = 0;
    for (; i + 4 <= n; i += 4) {
        unsigned u[4];
#pragma unroll
        for (int k = 0; k < 4; k++) u[k] = *(const unsigned*)(src + (size_t)(i + k) * J.src_pitch);
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float wk = wr[i + k];
            float p[4];
            cvt4(u[k], p);
#pragma unroll
            for (int c = 0; c < 4; c++) s[c] = mul_add_exact(s[c], p[c], wk);
        }
    }
    for (; i < n; i++) {
        const float wk = wr[i];
        float p[4];
        cvt4(*(const unsigned*)(src + (size_t)i * J.src_pitch), p);
#pragma unroll
        for (int c = 0; c < 4; c++) s[c] = mul_add_exact(s[c], p[c], wk);
    }
    float* out = J.tmp + (size_t)oy * J.tmp_pitch + x;
    if (x + 4 <= J.in_w) {
        *(float4*)out = make_float4(s[0], s[1], s[2], s[3]);
    } else {
#pragma unroll
        for (int c = 0; c < 4; c++)
            if (x + c < J.in_w) out[c] = s[c];
    }
}

constexpr int kResizeSpan = 2 * kThreads + 64;  // input floats for 256 outputs (ratio ~2)

__global__ __launch_bounds__(kThreads) void k_resize_h(const ResizeJob* __restrict__ jobs,
                                                       int njobs) {
    __shared__ float span[kResizeRows][kResizeSpan];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const ResizeJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int y0 = (t / J.tiles_x) * kResizeRows;
    const int ox0 = (t % J.tiles_x) * kThreads;
    const int ox = ox0 + threadIdx.x;
    const int oxl = min(ox0 + kThreads, J.out_w) - 1;
    const int nrows = min(kResizeRows, J.out_h - y0);
    const int lo = J.left[ox0];
    const int hi = J.left[oxl] + J.count[oxl];  // exclusive
    const bool staged = hi - lo <= kResizeSpan;
    if (staged) {
        for (int r = 0; r < nrows; r++) {
            const float* src = J.tmp + (size_t)(y0 + r) * J.tmp_pitch;
            for (int i = threadIdx.x; i < hi - lo; i += kThreads) span[r][i] = src[lo + i];
        }
    }
    __syncthreads();
    if (ox >= J.out_w) return;
    const int l = J.left[ox], n = J.count[ox];
    const float* wr = J.weights + (size_t)ox * J.maxtaps;
    float wv[16];  // this column's weights, loaded once for all rows
    if (n <= 16) {
#pragma unroll
        for (int i = 0; i < 16; i++) wv[i] = i < n ? wr[i] : 0.0f;
    }
    for (int r = 0; r < nrows; r++) {
        const float* in = staged ? &span[r][l - lo] : J.tmp + (size_t)(y0 + r) * J.tmp_pitch + l;
        float s = 0.0f;
        if (n <= 16) {
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (i < n) s = mul_add_exact(s, in[i], wv[i]);
        } else {
            for (int i = 0; i < n; i++) s = mul_add_exact(s, in[i], wr[i]);
        }
        float c = s < 0.0f ? 0.0f : (s > 255.0f ? 255.0f : s);
        J.dst[(size_t)(y0 + r) * J.dst_pitch + ox] = (uint8_t)roundf(c);
    }
}

// ---------------------------------------------------------------------------
// Both passes of the octave step in one kernel: the vertical pass of a tile's
// rows, over the input columns its horizontal windows need, goes to LDS as f32 (the
// same t += p * w in window order as k_resize_v) and the horizontal pass reads it
// there; round_u8 makes the bytes.
// k_resize_tall: tiles of kResizeTallW x kResizeTallH outputs, four rows per wave. A
// wave's lanes hold the tile's input column quads (120 outputs need at most 64) and
// stream the rows its four windows share once, converting each texel once instead
// of once per window (the windows of an exact or nearly exact halving lie two, now
// and then three rows apart; the first and last rows, whose windows are cut, take
// each on its own). The horizontal weights go through LDS, loaded in order once per
// tile: per output and lane they were 12 loads of 64 scattered words.
// 64 levels of 1920 x 1080: 196 -> 135 us against a wave per output row without
// either (576-column tiles); 960 x 540: 58 -> 42 us; one of 3840 x 2160: 24 -> 15 us.
// ---------------------------------------------------------------------------
// NT-row windows 2 apart: output row q adds input row base + i as its tap i - 2q.
template <int NT>
__device__ __forceinline__ void resize_v_rows(gbyte_t* src, int pitch, int in_h, int base,
                                              const float (&w)[4][14], float (&s)[4][4]) {
#pragma unroll
    for (int i = 0; i < NT + 6; i++) {
        float p[4];
        cvt4(*(__attribute__((address_space(1))) const unsigned*)(src + (size_t)min(base + i, in_h - 1) * pitch), p);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = i - 2 * q;
            if (k < 0 || k >= NT) continue;
#pragma unroll
            for (int c = 0; c < 4; c++) s[q][c] = mul_add_exact(s[q][c], p[c], w[q][k]);
        }
    }
}

__global__ __launch_bounds__(kThreads) void k_resize_tall(const ResizeJob* __restrict__ jobs,
                                                          int njobs) {
    constexpr int kTaps = kResizeMaxTaps;
    __shared__ __align__(16) float vt[kThreads / 64][4][kResizeTallSpan];
    __shared__ float hw[kResizeTallW * kTaps];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const ResizeJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int ox0 = (t % J.tiles_x) * kResizeTallW, cols = min(kResizeTallW, J.out_w - ox0);
    const int y0 = (t / J.tiles_x) * kResizeTallH + wave * 4;
    const int pitch = J.src_pitch, hn = J.maxtaps;
    for (int i = threadIdx.x; i < cols * hn; i += kThreads) hw[i] = J.weights[(size_t)ox0 * hn + i];
    const int lo4 = J.left[ox0] & ~3, nq = (J.left[ox0 + cols - 1] + hn - lo4 + 3) >> 2;  // <= 64
    const int x = lo4 + 4 * lane;
    float s[4][4] = {};
    if (lane < nq && x < J.in_w && y0 < J.out_h) {
        gbyte_t* src = (gbyte_t*)J.src_u8 + x;
        const int base = J.vleft[y0];
        const int vm = J.vmaxtaps;
        int n[4], sh[4];
        bool step2 = true, taps12 = vm >= 12;  // windows 2 (or once 3) rows apart; all of 12 rows
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int oy = min(y0 + q, J.out_h - 1);
            n[q] = J.vcount[oy];
            sh[q] = J.vleft[oy] - base - 2 * q;
            step2 = step2 && sh[q] >= 0 && sh[q] + n[q] <= 14;
            taps12 = taps12 && sh[q] == 0 && n[q] <= 12;
        }
        const ctap_t* vw = as_const_taps(J.vweights);
        if (taps12) {  // the rows of weights are zero past their count
            float w[4][14];
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int k = 0; k < 12; k++) w[q][k] = vw[min(y0 + q, J.out_h - 1) * vm + k];
            resize_v_rows<12>(src, pitch, J.in_h, base, w, s);
        } else if (step2) {
            float w[4][14];
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int k = 0; k < 14; k++) {
                    const int i = k - sh[q];
                    const float v = vw[min(y0 + q, J.out_h - 1) * vm + min(max(i, 0), vm - 1)];
                    w[q][k] = i >= 0 && i < n[q] ? v : 0.0f;
                }
            resize_v_rows<14>(src, pitch, J.in_h, base, w, s);
        } else {
            for (int q = 0; q < 4; q++) {
                const int oy = min(y0 + q, J.out_h - 1);
                const int l = J.vleft[oy], n = J.vcount[oy];
                const ctap_t* vw = as_const_taps(J.vweights) + (size_t)oy * J.vmaxtaps;
                float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                for (int i = 0; i < n; i++) {
                    const float wk = vw[i];
                    float p[4];
                    cvt4(*(__attribute__((address_space(1))) const unsigned*)(src + (size_t)(l + i) * pitch), p);
#pragma unroll
                    for (int c = 0; c < 4; c++) a[c] = mul_add_exact(a[c], p[c], wk);
                }
#pragma unroll
                for (int c = 0; c < 4; c++) s[q][c] = a[c];
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) *(float4*)&vt[wave][q][4 * lane] = make_float4(s[q][0], s[q][1], s[q][2], s[q][3]);
    __syncthreads();
    // (read once: after a store the compiler would read them again, and wait for them)
    uint8_t* const dst = J.dst + (size_t)y0 * J.dst_pitch + ox0;
    const int dst_pitch = J.dst_pitch, rows = J.out_h - y0;
    for (int c0 = 0; c0 < cols; c0 += 60) {
        const int c = c0 + lane;
        if (lane >= 60 || c >= cols) continue;
        const int at = J.left[ox0 + c] - lo4;
        float wv[kTaps];
#pragma unroll
        for (int i = 0; i < kTaps; i++)
            if (i < hn) wv[i] = hw[c * hn + i];
        float h[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < kTaps; i++) {
            if (i >= hn) break;
#pragma unroll
            for (int q = 0; q < 4; q++) h[q] = mul_add_exact(h[q], vt[wave][q][at + i], wv[i]);
        }
        unsigned v[4];
        round_u8(h, v);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (q < rows) dst[(size_t)q * dst_pitch + c] = (uint8_t)v[q];
    }
}

// k_resize_small: tiles of 64 output columns x 4 rows for launches that do not fill
// the GPU, where a tile's own latency is what counts: one output row per wave, all
// its loads issued before the first product, and only its own row of LDS, so no
// barrier. One level of 640 x 480: 15.4 -> 7.4 us (of which about 6 are the launch
// and its event); 64 of 1920 x 1080 take 430 us, for the weights and texels it
// loads again for every row.
__global__ __launch_bounds__(kThreads) void k_resize_small(const ResizeJob* __restrict__ jobs,
                                                           int njobs) {
    __shared__ __align__(16) float vt[kResizeSmallH][kResizeSmallSpan];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const ResizeJob& J = jobs[find_job(jobs, njobs, tile)];
    const int t = tile - J.tile_begin;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int oy = (t / J.tiles_x) * kResizeSmallH + wave;
    if (oy >= J.out_h) return;
    const int ox0 = (t % J.tiles_x) * kResizeSmallW, ox = ox0 + lane;
    const int oxc = min(ox, J.out_w - 1), oxl = min(ox0 + kResizeSmallW, J.out_w) - 1;
    const int pitch = J.src_pitch, hn = J.maxtaps;
    const int l = J.left[oxc];
    const int lo4 = J.left[ox0] & ~3, nq = (J.left[oxl] + hn - lo4 + 3) >> 2;  // 4 nq <= kResizeSmallSpan
    const int vl = J.vleft[oy], vn = J.vcount[oy];
    const ctap_t* vw = as_const_taps(J.vweights) + (size_t)oy * J.vmaxtaps;
    const int x = lo4 + 4 * lane;
    unsigned u[kResizeMaxTaps];
    gbyte_t* src = (gbyte_t*)J.src_u8 + (size_t)vl * pitch + x;
    const bool in = lane < nq && x < J.in_w;
#pragma unroll
    for (int i = 0; i < kResizeMaxTaps; i++)
        if (i < vn && in) u[i] = *(__attribute__((address_space(1))) const unsigned*)(src + (size_t)i * pitch);
    const float* wr = J.weights + (size_t)oxc * hn;
    float wv[kResizeMaxTaps];
#pragma unroll
    for (int i = 0; i < kResizeMaxTaps; i++)
        if (i < hn) wv[i] = wr[i];
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (in) {
#pragma unroll
        for (int i = 0; i < kResizeMaxTaps; i++) {
            if (i < vn) {
                const float wk = vw[i];
                float p[4];
                cvt4(u[i], p);
#pragma unroll
                for (int c = 0; c < 4; c++) s[c] = mul_add_exact(s[c], p[c], wk);
            }
        }
    }
    if (lane < nq) *(float4*)&vt[wave][4 * lane] = make_float4(s[0], s[1], s[2], s[3]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float* row = &vt[wave][l - lo4];
    float h = 0.0f;
#pragma unroll
    for (int i = 0; i < kResizeMaxTaps; i++)
        if (i < hn) h = mul_add_exact(h, row[i], wv[i]);
    const unsigned v = round_u8(h);
    if (ox < J.out_w) J.dst[(size_t)oy * J.dst_pitch + ox] = (uint8_t)v;
}

}  // namespace

void launch_blur_h(const BlurJob* d_jobs, int njobs, int total_tiles, int max_pad, int px,
                   hipStream_t s) {
    if (total_tiles <= 0) return;
    const int rowlen = 64 * px + max_pad + 8;
    const int padded = px == 16 ? hpad<16>(rowlen + 8) : px == 8 ? hpad<8>(rowlen + 8) : hpad<2>(rowlen + 8);
    const size_t lds = (size_t)kHTileH * (padded + 1) * sizeof(float);
    if (px == 16)
        hipLaunchKernelGGL(k_blur_h<16>, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs);
    else if (px == 8)
        hipLaunchKernelGGL(k_blur_h<8>, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs);
    else
        hipLaunchKernelGGL(k_blur_h<2>, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs);
}

void launch_blur_v(const BlurJob* d_jobs, int njobs, int total_tiles, int narrow_rows,
                   hipStream_t s) {
    if (total_tiles <= 0) return;
    if (narrow_rows > 0) {
        size_t lds = (size_t)narrow_rows * kVnTileW;
        hipLaunchKernelGGL(k_blur_v_narrow, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs);
    } else {
        hipLaunchKernelGGL(k_blur_v<kVRows>, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
    }
}

void launch_blur_v8(const BlurJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_blur_v<8>, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_blur_hv(const BlurJob* d_jobs, int njobs, int total_tiles, bool longer, hipStream_t s) {
    if (total_tiles <= 0) return;
    const dim3 g(total_tiles), b(kThreads);
    if (longer) hipLaunchKernelGGL(k_blur_hv<true>, g, b, 0, s, d_jobs, njobs);
    else hipLaunchKernelGGL(k_blur_hv<false>, g, b, 0, s, d_jobs, njobs);
}

void launch_blur_hv_small(const BlurJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_blur_hv_small, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

int deep_tiles_y(int h, int ntaps) {
    const int r = ntaps / 2, least = (h + kDeepH - 1) / kDeepH;
    constexpr int pass = kDeepThreads / kDeepW;  // rows of one horizontal pass
    for (int ty = least; (h + ty - 1) / ty >= 32; ty++)
        if (std::min(h, (h + ty - 1) / ty + 2 * r) <= pass) return ty;
    return least;
}

int deep_rows(int h, int ntaps) {
    const int ty = deep_tiles_y(h, ntaps), th = (h + ty - 1) / ty;
    return std::min(h, th + 2 * (ntaps / 2));
}

size_t deep_lds_bytes(int h, int ntaps) {
    const int ty = deep_tiles_y(h, ntaps), th = (h + ty - 1) / ty;
    const size_t n4 = (size_t)((ntaps + 3) & ~3), nr = (size_t)deep_rows(h, ntaps);
    return 4 * (n4 + nr * (size_t)deep_stride((int)n4) + (th + n4) * kDeepW);
}

double deep_tile_work(int h, int ntaps) {
    const int ty = deep_tiles_y(h, ntaps), th = (h + ty - 1) / ty;
    return (double)(deep_rows(h, ntaps) + th) * kDeepW * ntaps;
}

void launch_blur_deep(const BlurJob* d_jobs, int njobs, int total_tiles, int lds, hipStream_t s) {
    if (total_tiles <= 0) return;
    // past the 64 KB a launch may ask for by default
    if (lds > 65536)
        (void)hipFuncSetAttribute((const void*)k_blur_deep, hipFuncAttributeMaxDynamicSharedMemorySize, kDeepMaxLds);
    hipLaunchKernelGGL(k_blur_deep, dim3(total_tiles), dim3(kDeepThreads), lds, s, d_jobs, njobs);
}

void launch_blur_h_small(const BlurJob* d_jobs, int njobs, int total_tiles, int max_taps4,
                         hipStream_t s) {
    if (total_tiles <= 0) return;
    const int seg_stride = kSTileW + max_taps4 + 1;
    const size_t lds = ((size_t)max_taps4 + (size_t)kSTileH * seg_stride) * sizeof(float);
    hipLaunchKernelGGL(k_blur_h_small, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs,
                       seg_stride);
}

void launch_blur_v_small(const BlurJob* d_jobs, int njobs, int total_tiles, int max_taps4,
                         int max_rows, hipStream_t s) {
    if (total_tiles <= 0) return;
    const size_t lds = ((size_t)max_taps4 + (size_t)max_rows * kSTileW) * sizeof(float);
    hipLaunchKernelGGL(k_blur_v_small, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs,
                       max_taps4);
}

void launch_blur_v_small8(const BlurJob* d_jobs, int njobs, int total_tiles, int max_taps4,
                          int max_rows, hipStream_t s) {
    if (total_tiles <= 0) return;
    const size_t lds = (size_t)max_taps4 * sizeof(float) + (size_t)max_rows * kSTileW;
    hipLaunchKernelGGL(k_blur_v_small8, dim3(total_tiles), dim3(kThreads), lds, s, d_jobs, njobs,
                       max_taps4);
}

void launch_blur_h_generic(const BlurJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_blur_h_generic, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_blur_v_generic(const BlurJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_blur_v_generic, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_copy_level(const BlurJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_copy_level, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_luma(const LumaJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_luma, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_resize_v(const ResizeJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_resize_v, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_resize_tall(const ResizeJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_resize_tall, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_resize_small(const ResizeJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_resize_small, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

void launch_resize_h(const ResizeJob* d_jobs, int njobs, int total_tiles, hipStream_t s) {
    if (total_tiles <= 0) return;
    hipLaunchKernelGGL(k_resize_h, dim3(total_tiles), dim3(kThreads), 0, s, d_jobs, njobs);
}

}  // namespace sh
