// kernels_detect.hip -- gfx950 kernels for everything after the pyramid:
//   k_extrema_tile / k_extrema  find_scale_space_extrema  src/sift.rs:510-603
//   k_scan_*      ordered compaction offsets (exclusive scan)
//   k_compact     candidate list in the reference order (octave, layer, row, column)
//   k_refine      refine_and_filter_extrema     src/sift.rs:299-474 (+ solve 478-503)
//   k_orient      assign_orientations           src/sift.rs:605-726
//   k_descriptor  compute + normalize           src/sift.rs:917-1060, 889-913
//   k_descriptor_wide  the same for windows wider than the LDS patch
//
// DoG values are never stored: every DoG sample is recomputed from the u8
// Gaussian levels as q[G_{s+1}] - q[G_s] with q[v] = v / 255 (IEEE division,
// formed without it by q255f, or read from an LDS table of it in the row-wise
// extremum and wide-window kernels), which is bit-identical to the reference's
// (G_{s+1} as f32 / 255.0) - (G_s as f32 / 255.0) (src/sift.rs:97,120).
#include <math.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "sift_internal.h"

namespace sh {

namespace {

constexpr float kPi = 3.14159274101257324219f;  // std::f32::consts::PI
constexpr float kTwoPi = 2.0f * kPi;
constexpr float kDescFix = 1048576.0f;  // 2^20: u32 fixed point of the descriptor sums, times a per-keypoint power-of-two gain
constexpr int kThreads = 256;
constexpr int kExtChunk = 1024;  // pixels of one row per chunk in k_extrema
constexpr int kScanTile = 4096;  // 256 threads x 16 elements

// Rust `f as i32`: truncation toward zero, saturating, NaN -> 0.
__device__ __forceinline__ int f2i_sat(float x) {
    if (x != x) return 0;
    if (x >= 2147483648.0f) return 2147483647;
    if (x <= -2147483648.0f) return (-2147483647 - 1);
    return (int)x;
}

// f32::rem_euclid: r = x % m; r < 0 ? r + |m| : r.
__device__ __forceinline__ float rem_euclid(float x, float m) {
    float r = fmodf(x, m);
    return r < 0.0f ? r + fabsf(m) : r;
}

__device__ __forceinline__ float pow2f(int o) { return ldexpf(1.0f, o); }
// x / 2^o, exactly the IEEE division by that power (x is 0 or far from the
// denormals), in one instruction instead of about ten
__device__ __forceinline__ float over_pow2(float x, int o) { return __builtin_amdgcn_ldexpf(x, -o); }

// Three-operand maximum / minimum of values that are never NaN. (fmaxf and fminf
// first quiet each operand the compiler cannot prove is no signalling NaN: one
// more instruction for every value read from LDS.)
__device__ __forceinline__ float max3f(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float min3f(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max2f(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float min2f(float a, float b) {
    float r;
    asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// Gradient angle in [0, 2 pi]: octant reduction a = min(|x|,|y|)/max(|x|,|y|),
// atan(a) = a * P(a^2) with P a degree-8 least-squares (Lawson-reweighted)
// fit to atan(a)/a on [0,1], evaluated with FMA (max error 1.0e-7 rad on [0,1];
// about 2e-7 rad after the quadrant corrections, comparable to a 1-2 ulp
// atan2f). Gradients here are differences of non-negative values, never -0, and
// 0 or far above 1e-30: x = y = 0 gives a = 0 without a test of its own.
__device__ __forceinline__ float grad_angle(float y, float x) {
    const float ax = fabsf(x), ay = fabsf(y);
    // selects rather than fmaxf / fminf: the operands are never NaN, and one
    // comparison serves both and the octant test below
    const bool steep = ay > ax;
    const float mx = steep ? ay : ax, mn = steep ? ax : ay;
    const float a = mn * __builtin_amdgcn_rcpf(max2f(mx, 1e-30f));
    const float s = a * a;
    float p = 0.002456706715747714f;
    p = __builtin_fmaf(p, s, -0.014401290565729141f);
    p = __builtin_fmaf(p, s, 0.0397811196744442f);
    p = __builtin_fmaf(p, s, -0.07234849780797958f);
    p = __builtin_fmaf(p, s, 0.1049894317984581f);
    p = __builtin_fmaf(p, s, -0.14161229133605957f);
    p = __builtin_fmaf(p, s, 0.19985906779766083f);
    p = __builtin_fmaf(p, s, -0.33332598209381104f);
    p = __builtin_fmaf(p, s, 0.9999998807907104f);
    float r = a * p;
    if (steep) r = 1.57079637050628662109f - r;
    if (x < 0.0f) r = 3.14159274101257324219f - r;
    return y < 0.0f ? kTwoPi - r : r;
}

// Gradient angle in descriptor bin units (pi/4 per bin, result in (-4, 4]):
// the same octant reduction, with a 5-term fit of atan(a)/a scaled by 4/pi
// (max error 1.5e-5 bin, 1.2e-5 rad; far inside the descriptor tolerance).
__device__ __forceinline__ float atan2_bins(float y, float x) {
    const float ax = fabsf(x), ay = fabsf(y);
    const float mx = fmaxf(ax, ay), mn = fminf(ax, ay);
    const float a = mn * __builtin_amdgcn_rcpf(fmaxf(mx, 1e-30f));  // 0 when x = y = 0
    const float s = a * a;
    float p = 0.026541974395513535f;
    p = __builtin_fmaf(p, s, -0.10842673480510712f);
    p = __builtin_fmaf(p, s, 0.22938744723796844f);
    p = __builtin_fmaf(p, s, -0.4205574691295624f);
    p = __builtin_fmaf(p, s, 1.2730693817138672f);
    float r = a * p;
    if (ay > ax) r = 2.0f - r;
    if (x < 0.0f) r = 4.0f - r;
    return copysignf(r, y);
}

// x / 2pi (kTwoPi) for x in [0, 36 * 2pi], as y = x * RN(1/2pi) plus one FMA
// correction: three full-rate operations in place of the IEEE division (about
// eleven). The orientation binning only takes the floor, and that equals the
// floor of the IEEE quotient for every f32 x of the range (checked
// exhaustively on the CPU, tests/c/div_two_pi_check.c); the quotient itself can
// differ in the last place, and the product alone changes the floor of 7 x.
__device__ __forceinline__ float div_two_pi(float x) {
    constexpr float rc = 1.0f / kTwoPi;
    const float y = x * rc;
    return __builtin_fmaf(__builtin_fmaf(-y, kTwoPi, x), rc, y);
}

// Bin of a gradient angle in [0, 2 pi] (36 bins; 36 stands for bin 0): (an * 36) /
// 2pi with the reference's two roundings, as gradients along the axes land exactly
// on bin edges, where the rounding decides the bin.
__device__ __forceinline__ unsigned angle_bin(float an) {
    return (unsigned)div_two_pi(an * 36.0f);
}

// x / 3 for x = 0 or x > 2^-60: one FMA correction of the product with RN(1/3).
// Equal to the IEEE division for every f32 mantissa (checked exhaustively over two
// binades; the operations scale with the exponent).
__device__ __forceinline__ float over_3(float x) {
    constexpr float rc = 1.0f / 3.0f;
    const float y = x * rc;
    return __builtin_fmaf(__builtin_fmaf(-y, 3.0f, x), rc, y);
}

// A wave-uniform f32 value moved to a scalar register (the compiler cannot prove
// that values read from LDS or computed in VALU from uniform inputs are uniform).
__device__ __forceinline__ float uniform_f(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// v / 255 in f32 without a table, for v an integer in [0, 255] held as f32:
// 1/255 split into c = RN(1/255) and cl = RN(1/255 - c), then v * c + v * cl
// with one FMA. Equal to the IEEE division v / 255.0f for every byte value
// (checked exhaustively: v / 255 lies at least 2^-33 relative from any rounding
// midpoint, and the split's error is near 2^-48); three full-rate f32
// operations with the conversion.
__device__ __forceinline__ float q255f(float v) {
    constexpr float c = 0x1.010102p-8f;
    constexpr float cl = -0x1.fdfdfep-33f;
    return __builtin_fmaf(v, c, v * cl);
}

__device__ __forceinline__ void fill_q(float* q) {
    for (int i = threadIdx.x; i < 256; i += blockDim.x) q[i] = __fdiv_rn((float)i, 255.0f);
}

template <typename T>
__device__ __forceinline__ int find_by(const T* __restrict__ a, int n, int key,
                                       int T::*field) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        int mid = (lo + hi + 1) >> 1;
        if (a[mid].*field <= key) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ unsigned long long ballot64(bool p) {
    return __ballot(p);
}

// ---------------------------------------------------------------------------
// k_extrema: one workgroup per (octave, row). For each layer s in 1..S it stages
// DoG rows y-1, y, y+1 (layers s-1, s, s+1) of a 1024-pixel chunk in LDS and
// tests each pixel against its 26 neighbours with the reference's strict rule
// (val <= n clears is_max, val >= n clears is_min). A wave ballot turns the 64
// results of 64 consecutive pixels into one bitmask word; popcounts give the
// per-(layer,row) candidate count. Rows outside the border get count 0.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void k_extrema(const OctaveDesc* __restrict__ oct, int noct,
                                                      const ImageParams* __restrict__ params,
                                                      unsigned long long* __restrict__ bits,
                                                      unsigned* __restrict__ counts) {
    __shared__ float q[256];
    __shared__ float D[3][3][kExtChunk + 2];
    __shared__ unsigned cnt;
    const int row = blockIdx.x;
    const int j = find_by(oct, noct, row, &OctaveDesc::row_begin);
    const OctaveDesc& O = oct[j];
    const ImageParams& P = params[O.img];
    const int y = row - O.row_begin;
    const int w = O.w, h = O.h, S = P.num_intervals, border = P.border;
    const bool row_ok = (y >= border) && (y < h - border);
    if (!row_ok) {
        for (int s = 1 + threadIdx.x; s <= S; s += kThreads) counts[O.slot_begin + (s - 1) * h + y] = 0;
        return;
    }
    fill_q(q);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int s = 1; s <= S; s++) {
        if (threadIdx.x == 0) cnt = 0;
        for (int cx0 = 0; cx0 < w; cx0 += kExtChunk) {
            __syncthreads();
            // stage DoG layers s-1..s+1, rows y-1..y+1, x in [cx0-1, cx0+kExtChunk+1)
            const int nstage = kExtChunk + 2;
            for (int i = threadIdx.x; i < 3 * 3 * nstage; i += kThreads) {
                const int l = i / (3 * nstage);
                const int rem = i - l * 3 * nstage;
                const int rr = rem / nstage;
                const int c = rem - rr * nstage;
                const int x = min(max(cx0 - 1 + c, 0), w - 1);
                const int yy = min(max(y - 1 + rr, 0), h - 1);
                const int lay = s - 1 + l;   // DoG layer: G_{lay+1} - G_{lay}
                const uint8_t* g0 = O.levels + (long long)lay * O.level_stride + (size_t)yy * O.pitch;
                const uint8_t* g1 = g0 + O.level_stride;
                D[l][rr][c] = q[g1[x]] - q[g0[x]];
            }
            __syncthreads();
            for (int k = 0; k < kExtChunk / kThreads; k++) {
                const int c = k * kThreads + threadIdx.x;  // wave-contiguous 64 pixels
                const int x = cx0 + c;
                bool ext = false;
                if (x >= border && x < w - border) {
                    const float v = D[1][1][c + 1];
                    bool is_max = true, is_min = true;
#pragma unroll
                    for (int l = 0; l < 3; l++) {
#pragma unroll
                        for (int rr = 0; rr < 3; rr++) {
#pragma unroll
                            for (int dx = 0; dx < 3; dx++) {
                                if (l == 1 && rr == 1 && dx == 1) continue;
                                const float nv = D[l][rr][c + dx];
                                is_max = is_max && (v > nv);
                                is_min = is_min && (v < nv);
                            }
                        }
                    }
                    ext = is_max || is_min;
                }
                const unsigned long long m = ballot64(ext);
                const int word_x = cx0 + k * kThreads + wave * 64;
                if (lane == 0 && word_x < w) {
                    bits[O.bits_begin + (long long)((s - 1) * h + y) * O.nwords + (word_x >> 6)] = m;
                    if (m) atomicAdd(&cnt, (unsigned)__popcll(m));
                }
            }
        }
        __syncthreads();
        if (threadIdx.x == 0) counts[O.slot_begin + (s - 1) * h + y] = cnt;
    }
}

// ---------------------------------------------------------------------------
// k_extrema_tile<S>: the same test on strips of 64 columns x strip_rows rows
// (16 or kExtStripRows), taken as bands of 16 rows. The S+2 DoG layers of a band plus a 1-pixel halo are
// staged in LDS as f32 (each thread holds one 8-byte word of every Gaussian level
// and writes q[G_{l+1}] - q[G_l] for its 8 pixels); the words of the next band
// are loaded into registers before the current band is tested, so their latency
// overlaps the test. In a band, lane l owns column x0+l and walks down 4 rows (one
// wave per 4 rows). Per row it reads the DoG values of every layer at x-1, x, x+1
// and forms their horizontal max / min; a rolling window of three rows gives the
// 3x3 max / min of each layer.
// The 26-neighbour maximum of layer s is then max(3x3 of s-1, 3x3 of s+1,
// row max above and below in s, left and right in s), so "v greater than every
// neighbour" is v > that maximum (likewise for the minimum) -- the reference's
// strict comparisons (src/sift.rs:571-576). The 64 results of a row form one
// bitmask word, kept by one lane of the wave until the band's words are stored
// together; the row-slot counts are integer atomics (order-independent).
//
// Bound by vector instruction issue: per 64 pixels about 20 instructions stage the
// band (with its halo) and 43 three-operand maxima and minima (half rate) test it.
// 64 x 1920x1080, 3 layers: 757 us with a store, its 64-bit address and a count per
// row and layer and with operands quieted before each maximum; 480 us so. One band
// alone: the words outside the image were gathered byte by byte, eight loads one
// after the other.
// ---------------------------------------------------------------------------
constexpr int kTileW = 64, kTileH = 16;
static_assert(kExtStripRows % kTileH == 0, "strips are whole bands");
constexpr int kExtNW = (kTileW + 16) / 8;         // 8-byte words covering [x0-8, x0+72)
constexpr int kExtItems = (kTileH + 2) * kExtNW;  // (row, word) items of a band
constexpr int kExtRW = kTileW + 8;                // staged D row: columns [x0-4, x0+68)
static_assert(kExtItems <= kThreads, "one item per thread");
typedef __attribute__((address_space(1))) const uint8_t gbyte_t;
typedef __attribute__((address_space(1))) const unsigned long long gu64_t;
typedef __attribute__((address_space(1))) const unsigned gu32_t;

// The NG level words of this thread's item of the band starting at row y0 (rows
// y0-1 .. y0+16, clamped): the aligned 8-byte word at the item's columns, or the
// nearest one of the row (rows are padded to a multiple of 64 bytes, so it lies in
// the row); columns outside [0, w) then take the value of the nearest column inside.
template <int NG>
__device__ __forceinline__ void ext_fetch(const OctaveDesc& O, int x0, int y0,
                                          unsigned long long (&u)[NG]) {
    const int i = threadIdx.x;
    if (i >= kExtItems) return;
    const int w = O.w, h = O.h;
    const int r = i / kExtNW, k = i - r * kExtNW;
    const int y = min(max(y0 - 1 + r, 0), h - 1);
    const int xw = x0 - 8 + 8 * k;
    const int xc = min(max(xw, 0), (w - 1) & ~7);
    // fits 32 bits: images are at most 65536 x 65536 (larger ones are rejected)
    const unsigned off = (unsigned)y * (unsigned)O.pitch + (unsigned)xc;
    gbyte_t* lv = (gbyte_t*)O.levels;
#pragma unroll
    for (int l = 0; l < NG; l++, lv += O.level_stride) u[l] = *(gu64_t*)(lv + off);
    if (xw < 0 || xw + 8 > w) {
        const int sh = xw < 0 ? 0 : 8 * (w - 1 - xc);  // the nearest column's byte
        const unsigned long long keep = xw == xc ? (1ull << (8 * (w - xc))) - 1ull : 0ull;
#pragma unroll
        for (int l = 0; l < NG; l++) {
            const unsigned e = ((unsigned)(u[l] >> sh) & 0xffu) * 0x01010101u;
            const unsigned long long ee = ((unsigned long long)e << 32) | e;
            u[l] = (u[l] & keep) | (ee & ~keep);
        }
    }
}

// D = q[G_{l+1}] - q[G_l] for columns [x0-4, x0+68) of the band's 18 rows (the
// test reads [x0-1, x0+65)), with q formed by q255f, equal to v / 255.0f for
// every byte value; D is the same f32 subtraction the reference makes. Column
// x0-4+j sits at D index j, so the 4-column halves of a thread's 8-byte word
// (columns x0-8+8k ..) start at 16-byte boundaries and each goes to LDS as one
// 16-byte write (the first half of word 0 and the second half of the last word
// lie outside the staged columns).
template <int NL, int NG>
__device__ __forceinline__ void ext_stage(const unsigned long long (&u)[NG],
                                          float (*D)[kTileH + 2][kExtRW]) {
    const int i = threadIdx.x;
    if (i >= kExtItems) return;
    const int r = i / kExtNW, k = i - r * kExtNW;
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        if (hh == 0 ? k == 0 : k == kExtNW - 1) continue;
        float* const dst = &D[0][r][8 * k + 4 * hh - 4];
        const unsigned w0 = (unsigned)(u[0] >> (32 * hh));
        float qlo[4];
#pragma unroll
        for (int b = 0; b < 4; b++) qlo[b] = q255f((float)((w0 >> (8 * b)) & 0xffu));
#pragma unroll
        for (int l = 0; l < NL; l++) {
            const unsigned w1 = (unsigned)(u[l + 1] >> (32 * hh));
            float qhi[4];
#pragma unroll
            for (int b = 0; b < 4; b++) qhi[b] = q255f((float)((w1 >> (8 * b)) & 0xffu));
            *reinterpret_cast<float4*>(dst + l * (kTileH + 2) * kExtRW) =
                make_float4(qhi[0] - qlo[0], qhi[1] - qlo[1], qhi[2] - qlo[2], qhi[3] - qlo[3]);
#pragma unroll
            for (int b = 0; b < 4; b++) qlo[b] = qhi[b];
        }
    }
}

// Occupancy target: the LDS bound (6 work-groups per CU for S <= 3).
template <int S>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(S <= 3 ? 6 : 3)))
void k_extrema_tile(const OctaveDesc* __restrict__ oct, int noct,
                    const ImageParams* __restrict__ params, unsigned long long* __restrict__ bits,
                    unsigned* __restrict__ counts, int strip_rows) {
    constexpr int NL = S + 2;  // DoG layers
    constexpr int NG = S + 3;  // Gaussian levels
    __shared__ __align__(16) float D[NL][kTileH + 2][kExtRW];
    const int tile = xcd_remap(blockIdx.x, gridDim.x);
    const int j = find_by(oct, noct, tile, &OctaveDesc::row_begin);
    const OctaveDesc& O = oct[j];
    const ImageParams& P = params[O.img];
    const int t = tile - O.row_begin;
    const int w = O.w, h = O.h, border = P.border;
    const int tiles_x = (w + kTileW - 1) / kTileW;
    const int x0 = (t % tiles_x) * kTileW, ys = (t / tiles_x) * strip_rows;
    const int nbands = min(strip_rows, h - ys + kTileH - 1) / kTileH;  // >= 1

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int x = x0 + lane;
    const unsigned long long cols_ok = ballot64(x >= border && x < w - border);
    unsigned long long u[NG];
    ext_fetch<NG>(O, x0, ys, u);
#pragma unroll 1
    for (int band = 0; band < nbands; band++) {
        const int y0 = ys + band * kTileH;
        if (band > 0) __syncthreads();  // the previous band's tests are done with D
        ext_stage<NL, NG>(u, D);
        if (band + 1 < nbands) ext_fetch<NG>(O, x0, y0 + kTileH, u);
        __syncthreads();

        float hmx[3][NL], hmn[3][NL], dl[3][NL], dc[3][NL], dr[3][NL];
        auto load_row = [&](int slot, int r) {
#pragma unroll
            for (int l = 0; l < NL; l++) {
                const float a = D[l][r][lane + 3];  // column x0 + lane - 1
                const float b = D[l][r][lane + 4];
                const float c = D[l][r][lane + 5];
                dl[slot][l] = a;
                dc[slot][l] = b;
                dr[slot][l] = c;
                hmx[slot][l] = max3f(a, b, c);
                hmn[slot][l] = min3f(a, b, c);
            }
        };
        const int rbase = wave * 4;  // local D row of output row y0 + wave*4 is rbase + 1
        load_row(0, rbase);
        load_row(1, rbase + 1);
        unsigned word_lo = 0, word_hi = 0;  // lane (s-1)*4 + k: the bitmask of row k, layer s
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int prv = k % 3, cur = (k + 1) % 3, nxt = (k + 2) % 3;
            load_row(nxt, rbase + k + 2);
            const int y = y0 + rbase + k;
            const unsigned long long ok = y >= border && y < h - border ? cols_ok : 0ull;
            float mx9[NL], mn9[NL];  // 3x3 maximum / minimum of each layer
#pragma unroll
            for (int l = 0; l < NL; l++) {
                mx9[l] = max3f(hmx[prv][l], hmx[cur][l], hmx[nxt][l]);
                mn9[l] = min3f(hmn[prv][l], hmn[cur][l], hmn[nxt][l]);
            }
#pragma unroll
            for (int s = 1; s <= S; s++) {
                const float mx = max3f(max3f(hmx[prv][s], hmx[nxt][s], dl[cur][s]),
                                       max2f(dr[cur][s], mx9[s - 1]), mx9[s + 1]);
                const float mn = min3f(min3f(hmn[prv][s], hmn[nxt][s], dl[cur][s]),
                                       min2f(dr[cur][s], mn9[s - 1]), mn9[s + 1]);
                const float v = dc[cur][s];
                const unsigned long long m =
                    (__builtin_amdgcn_ballot_w64(v > mx) | __builtin_amdgcn_ballot_w64(v < mn)) & ok;
                if (m) {  // wave-uniform
                    asm("v_writelane_b32 %0, %1, %2"
                        : "+v"(word_lo) : "s"((unsigned)m), "n"((s - 1) * 4 + k));
                    asm("v_writelane_b32 %0, %1, %2"
                        : "+v"(word_hi) : "s"((unsigned)(m >> 32)), "n"((s - 1) * 4 + k));
                }
            }
        }
        const int y = y0 + rbase + (lane & 3);
        if (lane < 4 * S && y < h) {
            const long long slot_local = (long long)(lane >> 2) * h + y;
            const unsigned long long m = ((unsigned long long)word_hi << 32) | word_lo;
            bits[O.bits_begin + slot_local * O.nwords + (x0 >> 6)] = m;
            if (m) atomicAdd(&counts[O.slot_begin + slot_local], (unsigned)__popcll(m));
        }
    }
}

__global__ void k_fill_u32(unsigned* __restrict__ p, int n, unsigned v) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// Exclusive scan over n uint32 (n read from device memory when n_dev != null,
// capped by n_max): three passes over 4096-element tiles.
// out has n+1 entries; out[n] = total.
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned block_excl_scan(unsigned v, unsigned* sh, unsigned& total) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        unsigned y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) sh[wave] = x;
    __syncthreads();
    unsigned wpre = 0, tot = 0;
    for (int i = 0; i < (int)(blockDim.x >> 6); i++) {
        unsigned t = sh[i];
        if (i < wave) wpre += t;
        tot += t;
    }
    __syncthreads();
    total = tot;
    return wpre + x - v;
}

__device__ __forceinline__ int scan_n(int n_static, const unsigned* n_dev) {
    if (!n_dev) return n_static;
    unsigned v = *n_dev;
    return (int)min(v, (unsigned)n_static);
}

// The 16 elements of a thread, from base on (a multiple of 16; the arrays start on
// 256-byte boundaries): four 16-byte accesses where all lie below n. As 16 guarded
// words every access of a wave touched 64 lines.
__device__ __forceinline__ void scan_load16(const unsigned* __restrict__ in, int base, int n,
                                            unsigned (&v)[16]) {
    if (base + 16 <= n) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint4 u = *reinterpret_cast<const uint4*>(in + base + 4 * i);
            v[4 * i] = u.x;
            v[4 * i + 1] = u.y;
            v[4 * i + 2] = u.z;
            v[4 * i + 3] = u.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) v[i] = (base + i < n) ? in[base + i] : 0u;
    }
}
// Writes the exclusive prefixes of v, run before them, and returns their end.
__device__ __forceinline__ unsigned scan_store16(unsigned* __restrict__ out, int base, int n,
                                                 const unsigned (&v)[16], unsigned run) {
    unsigned o[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        o[i] = run;
        run += v[i];
    }
    if (base + 16 <= n) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<uint4*>(out + base + 4 * i) = make_uint4(o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++)
            if (base + i < n) out[base + i] = o[i];
    }
    return run;
}

__global__ __launch_bounds__(kThreads) void k_scan_reduce(const unsigned* __restrict__ in, int n_max,
                                                          const unsigned* n_dev,
                                                          unsigned* __restrict__ tile_sums) {
    __shared__ unsigned sh[8];
    const int n = scan_n(n_max, n_dev);
    const int base = blockIdx.x * kScanTile;
    unsigned s = 0;
    for (int i = 0; i < kScanTile / kThreads; i++) {
        int k = base + i * kThreads + threadIdx.x;
        if (k < n) s += in[k];
    }
    unsigned tot;
    block_excl_scan(s, sh, tot);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// The candidate of every keypoint, for the descriptor's work-groups (owner may be null;
// keypoints past its size are searched for): candidate c has the keypoints [k, e), at
// most kMaxPeaks.
__device__ __forceinline__ void mark_owner(int* __restrict__ owner, int size, int c, unsigned k,
                                           unsigned e) {
    for (e = min(e, min(k + (unsigned)kMaxPeaks, (unsigned)size)); k < e; k++) owner[k] = c;
}

// Per-image keypoint ranges: summary[2+i] = koff[first candidate of image i]
// (and out_offsets[i], when given); summary[0] = total candidates (may exceed
// cap), summary[1] = total keypoints.
struct FinalizeArgs {
    const unsigned* slot_offsets;
    const int* img_slot_begin;
    int nimg;
    const unsigned* koff;
    const unsigned* total;
    int cap;
    unsigned* summary;
    unsigned* out_offsets;
};
// Image i's range (i <= nimg; 0 writes the totals too), where owned(index) says that
// the work-group has written the offset of that index.
template <typename Owned>
__device__ __forceinline__ void finalize_entry(const FinalizeArgs& F, int i, Owned owned) {
    const unsigned n = min(*F.total, (unsigned)F.cap);
    const unsigned cb = min(F.slot_offsets[F.img_slot_begin[i]], n);
    if (owned(cb)) {
        const unsigned k = F.koff[cb];
        F.summary[2 + i] = k;
        if (F.out_offsets) F.out_offsets[i] = k;
    }
    if (i == 0 && owned(n)) {
        F.summary[0] = *F.total;
        F.summary[1] = F.koff[n];
    }
}

// The second launch of a scan: every work-group adds the sums of the tiles before its
// own (the offsets' 4 M of 64 frames are 1012 tiles, four loads of a thread), which
// saves a launch between, and the keypoint offsets' scan (F.summary set) writes the
// image ranges that begin in the tile, which saves one after it (4 to 5 us each).
__global__ __launch_bounds__(kThreads) void k_scan_down(const unsigned* __restrict__ in, int n_max,
                                                        const unsigned* n_dev,
                                                        const unsigned* __restrict__ tile_sums,
                                                        unsigned* out, FinalizeArgs F,
                                                        int* __restrict__ owner) {
    __shared__ unsigned sh[8];
    const int n = scan_n(n_max, n_dev);
    const int first = blockIdx.x * kScanTile, base = first + threadIdx.x * 16;
    if (first > 0 && first >= n) return;
    unsigned v[16];
    unsigned s = 0, before = 0, prefix, tot;
    scan_load16(in, base, n, v);
    for (int i = threadIdx.x; i < (int)blockIdx.x; i += kThreads) before += tile_sums[i];
#pragma unroll
    for (int i = 0; i < 16; i++) s += v[i];
    block_excl_scan(before, sh, prefix);
    unsigned k = prefix + block_excl_scan(s, sh, tot);
    const unsigned end = scan_store16(out, base, n, v, k);
    if (base < n && base + 16 >= n) out[n] = end;
    if (n == 0 && threadIdx.x == 0) out[0] = 0;
    if (owner) {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            mark_owner(owner, n_max, base + i, k, k + v[i]);
            k += v[i];
        }
    }
    if (F.summary) {
        __threadfence_block();
        __syncthreads();  // the offsets just written are read back
        const unsigned last = min(first + kScanTile, n) - 1u;  // ~0u if n = 0
        auto owned = [&](unsigned i) {
            return (i >= (unsigned)first && i < (unsigned)n && i - (unsigned)first < (unsigned)kScanTile) ||
                   (i == (unsigned)n && last + 1u == (unsigned)n);
        };
        for (int i = threadIdx.x; i <= F.nimg; i += kThreads) finalize_entry(F, i, owned);
    }
}

// The same scan in one work-group of 1024 threads, for few elements (single
// frames, small batches): 16384-element chunks with a running carry, one
// launch instead of three. The keypoint offsets' scan (F.summary set) writes the
// per-image ranges too, which needs every offset and here is one barrier away
// instead of one launch (4 us on a single frame).
constexpr int kScanSingleThreads = 1024;
constexpr int kScanSingleMax = 1 << 16;
__global__ __launch_bounds__(kScanSingleThreads) void k_scan_single(const unsigned* __restrict__ in,
                                                                   int n_max, const unsigned* n_dev,
                                                                   unsigned* out, FinalizeArgs F,
                                                                   int* __restrict__ owner) {
    __shared__ unsigned sh[kScanSingleThreads / 64];
    const int n = scan_n(n_max, n_dev);
    unsigned carry = 0;
    for (int b = 0; b < n; b += kScanSingleThreads * 16) {
        const int base = b + threadIdx.x * 16;
        unsigned v[16];
        unsigned s = 0;
        scan_load16(in, base, n, v);
#pragma unroll
        for (int i = 0; i < 16; i++) s += v[i];
        unsigned tot;
        const unsigned ex = block_excl_scan(s, sh, tot);
        scan_store16(out, base, n, v, carry + ex);
        carry += tot;
    }
    if (threadIdx.x == 0) out[n] = carry;
    if (F.summary) {
        __threadfence_block();
        __syncthreads();  // the offsets just written are read back
        if (owner) {
            // neighbouring lanes write neighbouring words, the offsets of four candidates
            // of a lane loaded at once
            constexpr int kU = 4;
            for (int c = threadIdx.x; c < n; c += kScanSingleThreads * kU) {
                unsigned k[kU], e[kU];
#pragma unroll
                for (int j = 0; j < kU; j++) {
                    const int cj = c + j * kScanSingleThreads;
                    k[j] = cj < n ? out[cj] : 0u;
                    e[j] = cj < n ? out[cj + 1] : 0u;
                }
#pragma unroll
                for (int j = 0; j < kU; j++) mark_owner(owner, n_max, c + j * kScanSingleThreads, k[j], e[j]);
            }
        }
        for (int i = threadIdx.x; i <= F.nimg; i += kScanSingleThreads) finalize_entry(F, i, [](unsigned) { return true; });
    }
}

// ---------------------------------------------------------------------------
// k_compact: one wave per spw consecutive (octave, layer, row) slots (spw <=
// kCompactSlots: 8 for launches with many slots, 1 for single frames, whose
// few slots would otherwise leave most of the GPU idle).
// The slots' counts and offsets are read once (one lane each) and the octave is
// found once; the bitmask words of every slot with candidates (one lane per
// word, rows of at most 64 words) are loaded before any slot is written, so
// their loads overlap. For each slot the set bits are ranked with popcounts and
// a wave prefix sum and the candidates written at offsets[slot] + rank, i.e. in
// the reference's order. Rows of more than 64 words take a chunked loop.
// The work-group sums the counts of all slots before its own itself (with many
// slots, from the sums of 4096-slot tiles and the counts of its own tile) and writes
// its slots' offsets (and the total), which saves the scan's other launches: a
// single frame's few thousand counts lie in L2 (1920 x 1080: 25 KB, 13 KB per
// work-group on average), where the scan in one work-group took 5 to 10 us; with the
// tiles' sums one launch goes before where two or three did (16 frames of 640 x 480
// 36 -> 25 us).
// ---------------------------------------------------------------------------
constexpr int kCompactSlots = 8;

__device__ __forceinline__ void compact_word(unsigned long long m, int wi, int j, int y, int s,
                                             unsigned& base, int lane, Cand* __restrict__ cand,
                                             int cap) {
    const unsigned c = (unsigned)__popcll(m);
    unsigned x = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned t = __shfl_up(x, d, 64);
        if (lane >= d) x += t;
    }
    unsigned pre = base + x - c;
    const unsigned tot = __shfl(x, 63, 64);
    while (m) {
        const int b = __ffsll((long long)m) - 1;
        m &= m - 1;
        if (pre < (unsigned)cap) {
            Cand cd;
            cd.job = j;
            cd.x = wi * 64 + b;
            cd.y = y;
            cd.layer = s;
            cand[pre] = cd;
        }
        pre++;
    }
    base += tot;
}

__global__ __launch_bounds__(kThreads) void k_compact(const OctaveDesc* __restrict__ oct, int noct,
                                                      int nslots,
                                                      const unsigned long long* __restrict__ bits,
                                                      const unsigned* __restrict__ counts,
                                                      const unsigned* __restrict__ tile_sums,
                                                      unsigned* __restrict__ offsets,
                                                      Cand* __restrict__ cand, int cap, int spw) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int s0 = (blockIdx.x * (kThreads / 64) + wave) * spw;
    const int ns = min(spw, nslots - s0);
    __shared__ unsigned wsum[kThreads / 64];
    const int per = (kThreads / 64) * spw, first = blockIdx.x * per;  // slots of the work-group, <= 64
    const int tile = tile_sums ? first / kScanTile : 0;
    unsigned p = 0;
    for (int i = threadIdx.x; i < tile; i += kThreads) p += tile_sums[i];
    for (int i = tile * kScanTile + threadIdx.x * 4; i < first; i += kThreads * 4) {  // first is a multiple of 4
        const uint4 v = *reinterpret_cast<const uint4*>(counts + i);
        p += (v.x + v.y) + (v.z + v.w);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) p += __shfl_xor(p, d, 64);
    if (lane == 0) wsum[wave] = p;
    const int slot = first + lane;
    const bool mine = lane < per && slot < nslots;
    const unsigned c = mine ? counts[slot] : 0u;
    unsigned x = c;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned t = __shfl_up(x, d, 64);
        if (lane >= d) x += t;
    }
    __syncthreads();
    x += (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
    if (wave == 0 && mine) {
        offsets[slot] = x - c;
        if (slot == nslots - 1) offsets[nslots] = x;
    }
    const int at = wave * spw + lane;
    unsigned cnt_l = __shfl(c, at & 63, 64);
    const unsigned off_l = __shfl(x - c, at & 63, 64);
    if (lane >= ns) cnt_l = 0u;
    if (s0 >= nslots) return;
    const unsigned long long any = ballot64(cnt_l != 0u);
    if (any == 0ull) return;
    // each slot's octave (the slots are ordered by octave)
    int jk[kCompactSlots];
    int j = find_by(oct, noct, s0, &OctaveDesc::slot_begin);
#pragma unroll
    for (int k = 0; k < kCompactSlots; k++) {
        while (k < ns && j + 1 < noct && oct[j + 1].slot_begin <= s0 + k) j++;
        jk[k] = j;
    }
    // the bitmask words of the slots with candidates, all loads issued first
    unsigned long long m[kCompactSlots];
#pragma unroll
    for (int k = 0; k < kCompactSlots; k++) {
        m[k] = 0ull;
        if ((any >> k) & 1ull) {
            const OctaveDesc& O = oct[jk[k]];
            if (lane < O.nwords)
                m[k] = bits[O.bits_begin + (long long)(s0 + k - O.slot_begin) * O.nwords + lane];
        }
    }
#pragma unroll
    for (int k = 0; k < kCompactSlots; k++) {
        if (!((any >> k) & 1ull)) continue;
        const OctaveDesc& O = oct[jk[k]];
        const int local = s0 + k - O.slot_begin;
        const int s = local / O.h + 1, y = local - (s - 1) * O.h;
        unsigned base = __shfl(off_l, k, 64);
        compact_word(m[k], lane, jk[k], y, s, base, lane, cand, cap);
        if (O.nwords > 64) {  // rows wider than 4096 px: the remaining words by chunks
            const unsigned long long* wrow = bits + O.bits_begin + (long long)local * O.nwords;
            for (int w0 = 64; w0 < O.nwords; w0 += 64) {
                const int wi = w0 + lane;
                compact_word(wi < O.nwords ? wrow[wi] : 0ull, wi, jk[k], y, s, base, lane, cand, cap);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// k_refine: one thread per candidate; the reference's arithmetic in the same
// f32 operation order (compiled without FMA contraction).
// Bound by the gathers: a step reads 3 rows of 4 Gaussian levels, most lines of the
// pyramid in all. A word for the 3 texels of a row (12 loads a step instead of 38 of
// single bytes): 64 x 1920x1080 190 -> 156 us.
// ---------------------------------------------------------------------------
// Work-groups of one wave: the gathers of the few waves a single frame has are bound
// by a CU's requests, so they are spread over all CUs (640x480: 17.5 us with groups of
// four waves, 12.0 us; 1920x1080 19.1 and 13.4; 64 frames 157 and 151).
constexpr int kRefineThreads = 64;

// The refinement of one candidate (refine_and_filter_extrema, src/sift.rs:299-474):
// whether it is kept, and then its keypoint. kUniform: the whole wave has the same one.
template <bool kUniform>
__device__ __forceinline__ bool refine_candidate(const Cand& cd, const OctaveDesc& O,
                                                 const ImageParams& P, Keypoint& r) {
    const int nd = P.num_intervals + 2;  // DoG layers per octave
    const float scale0 = pow2f(O.octave);
    // kp.x / 2^o of the candidate ((x + 0.5) * 2^o), `as i32` (src/sift.rs:309-313)
    const float xi = (((float)cd.x + 0.5f) * scale0) / scale0;
    const float yi = (((float)cd.y + 0.5f) * scale0) / scale0;
    int cx = f2i_sat(xi), cy = f2i_sat(yi), cl = cd.layer;
    for (int step = 0; step < 5; step++) {
        if (kUniform) {
            cx = __builtin_amdgcn_readfirstlane(cx);
            cy = __builtin_amdgcn_readfirstlane(cy);
            cl = __builtin_amdgcn_readfirstlane(cl);
        }
        if (cl < 1 || cl >= nd - 1) return false;
        if (cx < 1 || cx >= O.w - 1 || cy < 1 || cy >= O.h - 1) return false;
        // the 3x3 texels around (cx, cy) of the four Gaussian levels cl - 1 .. cl + 2,
        // a row by one word (columns cx - 1 .. cx + 2: cx + 2 <= w, and a byte past
        // the last level's last row is still the arena's)
        unsigned t[4][3];
        gbyte_t* lv = (gbyte_t*)O.levels + ((long long)(cl - 1) * O.level_stride +
                                            (long long)((size_t)(cy - 1) * O.pitch + (cx - 1)));
#pragma unroll
        for (int l = 0; l < 4; l++, lv += O.level_stride)
#pragma unroll
            for (int r = 0; r < 3; r++)
                t[l][r] = ((const __attribute__((address_space(1))) UnalignedWord*)(lv + r * O.pitch))->v;
        // DoG layer cl - 1 + l at row cy - 1 + r, column cx - 1 + x
        auto dog = [&](int l, int r, int x) {
            return q255f((float)((t[l + 1][r] >> (8 * x)) & 0xffu)) -
                   q255f((float)((t[l][r] >> (8 * x)) & 0xffu));
        };
        const float pxp = dog(1, 1, 2), pxm = dog(1, 1, 0);
        const float pyp = dog(1, 2, 1), pym = dog(1, 0, 1);
        const float nxt = dog(2, 1, 1), prv = dog(0, 1, 1);
        const float dx = (pxp - pxm) / 2.0f;
        const float dy = (pyp - pym) / 2.0f;
        const float ds = (nxt - prv) / 2.0f;
        const float cv = dog(1, 1, 1);
        const float dxx = pxp + pxm - 2.0f * cv;
        const float dyy = pyp + pym - 2.0f * cv;
        const float dss = nxt + prv - 2.0f * cv;
        const float dxy = (dog(1, 2, 2) - dog(1, 2, 0) - dog(1, 0, 2) + dog(1, 0, 0)) / 4.0f;
        const float dxs = (dog(2, 1, 2) - dog(2, 1, 0) - (dog(0, 1, 2) - dog(0, 1, 0))) / 4.0f;
        const float dys = (dog(2, 2, 1) - dog(2, 0, 1) - (dog(0, 2, 1) - dog(0, 0, 1))) / 4.0f;
        // solve_linear_system (src/sift.rs:478-503), b = -g
        const float a00 = dxx, a01 = dxy, a02 = dxs, a10 = dxy, a11 = dyy, a12 = dys,
                    a20 = dxs, a21 = dys, a22 = dss;
        const float b0 = -dx, b1 = -dy, b2 = -ds;
        const float det_a = a00 * (a11 * a22 - a12 * a21) - a01 * (a10 * a22 - a12 * a20) +
                            a02 * (a10 * a21 - a11 * a20);
        if (fabsf(det_a) < 1e-10f) return false;
        const float det_x = b0 * (a11 * a22 - a12 * a21) - a01 * (b1 * a22 - a12 * b2) +
                            a02 * (b1 * a21 - a11 * b2);
        const float det_y = a00 * (b1 * a22 - a12 * b2) - b0 * (a10 * a22 - a12 * a20) +
                            a02 * (a10 * b2 - b1 * a20);
        const float det_z = a00 * (a11 * b2 - b1 * a21) - a01 * (a10 * b2 - b1 * a20) +
                            b0 * (a10 * a21 - a11 * a20);
        const float ox = det_x / det_a, oy = det_y / det_a, os = det_z / det_a;
        if (fabsf(ox) < 0.5f && fabsf(oy) < 0.5f && fabsf(os) < 0.5f) {
            const float val = cv + 0.5f * (dx * ox + dy * oy + ds * os);
            if (fabsf(val) < P.contrast_threshold) return false;
            const float tr = dxx + dyy;
            const float trace_sq = tr * tr;
            const float det = dxx * dyy - dxy * dxy;
            if (det <= 0.0f) return false;
            const float ratio = trace_sq / det;
            const float e1 = P.edge_threshold + 1.0f;
            const float thr = e1 * e1 / P.edge_threshold;
            if (ratio >= thr) return false;
            const float scale = pow2f(O.octave);
            const float fl = (float)cl + os;
            const float e = (float)O.octave + fl / (float)P.num_intervals;
            // 2.0_f32.powf(e): correctly rounded via double exp2
            const float psig = P.sigma * (float)exp2((double)e);
            r.x = ((float)cx + ox) * scale;
            r.y = ((float)cy + oy) * scale;
            r.size = psig;
            r.angle = 0.0f;
            r.response = val;
            r.octave = O.octave;
            r.layer = f2i_sat(roundf(fl));
            return true;
        } else {
            cx = f2i_sat(roundf((float)cx + ox));
            cy = f2i_sat(roundf((float)cy + oy));
            cl = f2i_sat(roundf((float)cl + os));
            if (cl < 0 || cl >= nd) return false;
        }
    }
    return false;
}

__global__ __launch_bounds__(kRefineThreads) void k_refine(const OctaveDesc* __restrict__ oct,
                                                     const ImageParams* __restrict__ params,
                                                     const Cand* __restrict__ cand,
                                                     const unsigned* __restrict__ total, int cap,
                                                     Keypoint* __restrict__ out,
                                                     int* __restrict__ valid,
                                                     float* __restrict__ cand_resp) {
    const int n = (int)min(*total, (unsigned)cap);
    for (int c = blockIdx.x * kRefineThreads + threadIdx.x; c < n; c += gridDim.x * kRefineThreads) {
        const Cand cd = cand[c];
        const OctaveDesc& O = oct[cd.job];
        if (cand_resp) {
            const uint8_t* g0 = O.levels + (long long)cd.layer * O.level_stride +
                                ((size_t)cd.y * O.pitch + cd.x);
            cand_resp[c] = q255f((float)g0[O.level_stride]) - q255f((float)g0[0]);
        }
        Keypoint r;
        const bool ok = refine_candidate<false>(cd, O, params[O.img], r);
        valid[c] = ok;
        if (ok) out[c] = r;
    }
}

// ---------------------------------------------------------------------------
// Work queue of the keypoint kernels. With a queue, a launch has as many
// work-groups as fit on the GPU at once, and each takes chunks of kChunk
// consecutive keypoints until the count is reached. Work-group b uses counter
// b % kNumXcd (the XCD the dispatcher places it on) of kNumXcd counters, zeroed
// by a fill kernel earlier on the stream; counter x's chunk c holds keypoints
// [(c * kNumXcd + x) * kChunk, + kChunk). One counter taking every item
// serialises the atomics of the whole GPU on one address (measured: 10x the
// kernel's time); eight counters and chunks make them rare. Without a queue,
// work-group b takes keypoints b, b + grid, ...
// Thread 0 takes the next chunk at the start of a chunk's last item, into the
// slot the work-group is not reading, and everyone reads it after the barrier
// that ends that item: each slot is written before a barrier, read after it,
// and not written again until every thread has read it. All threads of a
// work-group thus see the same item sequence, every item's early exits
// (`continue`) still pass the barrier that ends it, and the loop test is
// uniform.
// ---------------------------------------------------------------------------
template <int kChunk>
struct WorkQueue {
    unsigned* heads;  // kNumXcd counters; null: static grid-stride assignment
    int slot_it, left, x;

    __device__ __forceinline__ int chunk_first(int c) const { return (c * kNumXcd + x) * kChunk; }
    __device__ __forceinline__ int first(int* slots) {
        slot_it = 0;
        left = kChunk - 1;
        x = (int)(blockIdx.x % kNumXcd);
        if (!heads) return (int)blockIdx.x;
        if (threadIdx.x == 0) slots[0] = (int)atomicAdd(&heads[x], 1u);
        __syncthreads();
        return chunk_first(slots[0]);
    }
    // at the start of an item: thread 0 takes the next chunk during the last
    // item of this one
    __device__ __forceinline__ void prefetch(int* slots) {
        if (heads && left == 0 && threadIdx.x == 0)
            slots[(slot_it + 1) & 1] = (int)atomicAdd(&heads[x], 1u);
    }
    __device__ __forceinline__ int next(int* slots, int cur) {
        if (!heads) return cur + (int)gridDim.x;
        __syncthreads();
        if (left > 0) {
            left--;
            return cur + 1;
        }
        slot_it++;
        left = kChunk - 1;
        return chunk_first(slots[slot_it & 1]);
    }
};
constexpr int kOrientChunk = 8;
constexpr int kDescChunk = 2;

// Maximum over the 64 lanes of a fully active wave with DPP:
// shifts by 1, 2, 4, 8 inside each row of 16 lanes, then lane 15 of rows 0 and 2 to rows 1 and 3
// and lane 31 to rows 2 and 3; returned to every lane.
__device__ __forceinline__ unsigned wave_max_u32(unsigned x) {
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true));  // row_shr:1
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true));  // row_shr:2
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, true));  // row_shr:4
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, true));  // row_shr:8
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false)); // row_bcast:15
    x = max(x, (unsigned)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false)); // row_bcast:31
    return (unsigned)__builtin_amdgcn_readlane((int)x, 63);
}

constexpr int kOriMaxR = 16;
constexpr int kOriRows = 2 * kOriMaxR + 5;      // staged rows
constexpr int kOS = 2 * kOriMaxR + 8;           // staged row stride (bytes): 4 * ceil((3 + rows + 3) / 4)
constexpr int kOriHist = 37;                    // words of one histogram copy: 36 bins, and 36 for bin 0
static_assert(2 * kOriMaxR + 1 <= 64, "one lane per row and column of the window");
constexpr double kOriBias = 4503599627370496.0;  // 2^52

// ---------------------------------------------------------------------------
// k_orient: one wave (workgroup of 64) per refined keypoint, or (kRefine) per
// candidate, which it refines first (src/sift.rs:605-726). Each sample of the (2R+1)^2 window adds
// mag * exp(-(dx^2+dy^2)/denom) to bin floor(theta * 36 / 2pi) of a u64
// fixed-point (2^40) histogram, one of 4 copies by lane (integer adds:
// order-independent, deterministic, and as fine as the f32 contributions
// themselves). Lanes 0..35 then hold one bin each for the two [1,1,1]/3 smoothing
// passes, the max and the peak test; a ballot ranks the peaks in bin order.
//
// Windows with R <= 16 (all of the default schedule) are staged in LDS as
// bytes, every texel a sample's gradient can touch. Lane l takes the samples
// [l C, (l+1) C) in raster order, C = ceil(n / 64): lanes sit far apart in the
// window, and a lane's consecutive samples are neighbours that often share a bin,
// so they are summed in registers and added to LDS once per run. The sum is an f64
// that starts at 2^52: the samples' fixed-point values are whole numbers, so its
// low 52 bits hold the integer sum exactly (a window's total is below
// 33^2 * sqrt(2) * 2^40 < 2^51) and are added as they are; what the biases leave in
// the high 12 bits is masked off at the end.
// The loop has the same count for every lane and no test per sample: a lane's C <=
// 2R + 1 samples cross into the next row at most once, so the column table is
// written twice over and the row is a choice of two; samples off the image or past
// the window have weight 0 (they add 0 to some bin).
//
// Bound by vector instruction issue (about 100 instructions per sample step and 250
// per keypoint), with LDS two thirds busy. 64 x 1920x1080: 940 us with a table of
// v / 255 in LDS (10 LDS reads per sample, now 5), the u64 arithmetic on two words, a
// test per sample, staging by a division and IEEE divisions by 3 and by powers of
// two; 635 us so. Texels held as f32 instead of bytes (no conversion per sample):
// 777-830 us, as LDS then holds 20 work-groups per CU instead of 32 and its reads
// spread over more banks. 2 or 8 histogram copies, other row strides and an unaligned
// word for the two horizontal texels were slower too (1150 us for the last).
// ---------------------------------------------------------------------------
template <bool kRefine>
__global__ __launch_bounds__(64) void k_orient(const OctaveDesc* __restrict__ oct,
                                               const ImageParams* __restrict__ params,
                                               const Cand* __restrict__ cand,
                                               const unsigned* __restrict__ total, int cap,
                                               Keypoint* __restrict__ ref, int* __restrict__ valid,
                                               unsigned* __restrict__ npeaks,
                                               float* __restrict__ angles,
                                               unsigned* __restrict__ queue) {
    __shared__ __align__(16) unsigned long long hist[4 * kOriHist];
    __shared__ __align__(16) uint8_t pq[kOriRows * kOS];
    // per column (twice over) / row of the window: (byte offset in pq as int bits, Gaussian factor)
    __shared__ float2 ocx[2 * (2 * kOriMaxR + 1)], ocy[64];
    const int lane = threadIdx.x;
    const int n = (int)min(*total, (unsigned)cap);
    // the neighbour bins of the 36-bin circle, as ds_bpermute addresses
    const int prev4 = 4 * (lane == 0 ? 35 : lane - 1), next4 = 4 * (lane == 35 ? 0 : min(lane + 1, 63));
    __shared__ int qslot[2];
    WorkQueue<kOrientChunk> Q{queue, 0, 0, 0};
    for (int c = Q.first(qslot); c < n; c = Q.next(qslot, c)) {
        Q.prefetch(qslot);
        const Cand cd = cand[c];
        const OctaveDesc& O = oct[cd.job];
        const ImageParams& P = params[O.img];
        Keypoint kp;
        bool ok;
        if (kRefine) {
            ok = __builtin_amdgcn_readfirstlane((int)refine_candidate<true>(cd, O, P, kp)) != 0;
            if (lane == 0) {
                valid[c] = ok;
                if (ok) ref[c] = kp;
            }
            kp.x = uniform_f(kp.x);
            kp.y = uniform_f(kp.y);
            kp.size = uniform_f(kp.size);
            kp.octave = O.octave;
            kp.layer = __builtin_amdgcn_readfirstlane(kp.layer);
        } else {
            ok = valid[c] != 0;
            kp = ref[c];
        }
        if (!ok) {
            if (lane == 0) npeaks[c] = 0;
            continue;
        }
        const int S = P.num_intervals;
        const int gl = min(max(kp.layer, 0), S + 2);
        const uint8_t* g = O.levels + (long long)gl * O.level_stride;
        const int w = O.w, h = O.h, pitch = O.pitch;
        const float xo = over_pow2(kp.x, kp.octave), yo = over_pow2(kp.y, kp.octave);
        const float so = over_pow2(kp.size, kp.octave);
        if (!(so > 0.0f)) {
            if (lane == 0) npeaks[c] = 0;
            continue;
        }
        const int R = __builtin_amdgcn_readfirstlane(f2i_sat(roundf(4.5f * so)));
        const float ws = 1.5f * so;
        const float denom = 2.0f * ws * ws;
        const int side = 2 * R + 1, nsamp = side * side;
        const int iters = (nsamp + 63) >> 6;
        // weight * 2^40 = 2^(kq * (dx^2 + dy^2) + 40)
        const float kq = -1.44269504088896341f / denom;
        constexpr float lf = 40.0f;  // m = mag * weight * 2^40
        const bool lds = R <= kOriMaxR;
        const float inv_side = __builtin_amdgcn_rcpf((float)side);
        reinterpret_cast<uint4*>(hist)[lane] = make_uint4(0u, 0u, 0u, 0u);
        if (lane < 2 * kOriHist - 64)
            reinterpret_cast<uint4*>(hist)[64 + lane] = make_uint4(0u, 0u, 0u, 0u);
        if (lds) {
            // the samples' pixels (round(x_o + dx), round(y_o + dy)) and their 4-neighbours
            // lie in columns px0 .. px0 + 2R + 4 and rows py0 .. py0 + 2R + 4
            const int px0 = __builtin_amdgcn_readfirstlane((int)roundf(xo)) - R - 2;
            const int py0 = __builtin_amdgcn_readfirstlane((int)roundf(yo)) - R - 2;
            const int px0a = px0 & ~3;
            // a lane stages one 4-texel word of every kPer-th row, all loads in flight
            // at once; words and rows past the window are staged too where that saves
            // a test. Eight words of a row hold R <= 12 (2 R + 5 texels and 3 before
            // them), ten R <= 16.
            gbyte_t* const g8 = (gbyte_t*)g;
            auto stage = [&](auto words_tag, auto passes_tag) {
                constexpr int kWords = decltype(words_tag)::value, kPasses = decltype(passes_tag)::value;
                constexpr int kPer = 64 / kWords;
                const int wd = lane % kWords, row = lane / kWords;
                unsigned u[kPasses];
                if (px0a >= 0 && px0a + 4 * kWords <= pitch && py0 >= 0 && py0 + kPer * kPasses <= h) {
                    const unsigned off = __umul24(row, pitch) + 4 * wd;
                    gbyte_t* base = g8 + ((size_t)py0 * pitch + px0a);
#pragma unroll
                    for (int k = 0; k < kPasses; k++, base += kPer * pitch) u[k] = *(gu32_t*)(base + off);
                } else {
                    // words off the image are taken from its nearest word: only samples of
                    // weight 0 read them
                    const unsigned xw = min(max(px0a + 4 * wd, 0), pitch - 4);
#pragma unroll
                    for (int k = 0; k < kPasses; k++) {
                        const int yy = min(max(py0 + row + kPer * k, 0), h - 1);
                        u[k] = *(gu32_t*)(g8 + (__umul24(yy, pitch) + xw));
                    }
                }
                if (kWords > kOS / 4 && wd >= kOS / 4) return;
                uint8_t* const dst = &pq[row * kOS + 4 * wd];
#pragma unroll
                for (int k = 0; k < kPasses; k++) {
                    if (kPer * kPasses > kOriRows && row + kPer * k >= kOriRows) break;
                    *reinterpret_cast<unsigned*>(dst + kPer * kOS * k) = u[k];
                }
            };
            if (R <= 9) stage(std::integral_constant<int, 8>{}, std::integral_constant<int, 3>{});
            else if (R <= 12) stage(std::integral_constant<int, 8>{}, std::integral_constant<int, 4>{});
            else stage(std::integral_constant<int, 16>{}, std::integral_constant<int, 10>{});
            // per column and row of the window: the offset in the staged window of the
            // texel before the sample's, and the Gaussian weight's factor 2^(kq d^2 + 20)
            // of that column / row offset d (the weight of sample (dx, dy) is the product
            // of the two: one multiply per sample instead of exp2), 0 outside
            // [1, w-2] x [1, h-2]
            {
                const float d = (float)(lane - R);
                const float wf = __builtin_amdgcn_exp2f(__builtin_fmaf(kq, d * d, 0.5f * lf));
                const int xi = (int)roundf(xo + d), yi = (int)roundf(yo + d);
                const bool row_in = lane < side && yi >= 1 && yi < h - 1;
                ocy[lane] = make_float2(__int_as_float(row_in ? (yi - py0 - 1) * kOS : 0),
                                        row_in ? wf : 0.0f);
                if (lane < side) {
                    const bool col_in = xi >= 1 && xi < w - 1;
                    const float2 e = make_float2(__int_as_float(col_in ? (xi - px0a - 1) : 0),
                                                 col_in ? wf : 0.0f);
                    ocx[lane] = e;
                    ocx[lane + side] = e;
                }
            }
        }
        __syncthreads();
        unsigned long long* const hrow = hist + (lane & 3) * kOriHist;
        unsigned run_bin = 0;
        if (lds) {
            const int i0 = lane * iters;
            const int iy0 = (int)(((float)i0 + 0.5f) * inv_side);  // <= 63
            const int ix0 = i0 - iy0 * side;
            const int wrap = side - ix0;  // the first sample of the next row
            const float2 row0 = ocy[iy0], row1 = ocy[min(iy0 + 1, 63)];
            const float2* const cols = &ocx[ix0];
            double run = kOriBias;
            float gx, gy, wgt;
            auto sample = [&](int k) {
                const float2 cx = cols[k];
                const bool second = k >= wrap;
                const int off = __float_as_int(cx.x) + __float_as_int(second ? row1.x : row0.x);
                const uint8_t* const pp = pq + off;
                gx = q255f((float)pp[kOS + 2]) - q255f((float)pp[kOS]);
                gy = q255f((float)pp[2 * kOS + 1]) - q255f((float)pp[1]);
                wgt = cx.y * (second ? row1.y : row0.y);
            };
            sample(0);
            for (int k = 0; k < iters; k++) {
                const float sx = gx, sy = gy, sw = wgt;
                sample(k + 1);
                  // the next sample's reads overlap this one's arithmetic (the
                                // last one's too: ix0 + iters < 2 side, a sample of some row)
                const float m = __builtin_amdgcn_sqrtf(__builtin_fmaf(sx, sx, sy * sy)) * sw;
                const unsigned bin = angle_bin(grad_angle(sy, sx));
                if (bin != run_bin) {
                    atomicAdd(&hrow[run_bin], (unsigned long long)__double_as_longlong(run));
                    run = kOriBias;
                    run_bin = bin;
                }
                run += (double)floorf(m);
            }
            atomicAdd(&hrow[run_bin], (unsigned long long)__double_as_longlong(run));
        } else {
            const int i0 = min(lane * iters, nsamp), i1 = min(i0 + iters, nsamp);
            const int iy0 = i0 / side;
            int dy = iy0 - R, dx = i0 - iy0 * side - R;
            unsigned long long run = 0;
            for (int i = i0; i < i1; i++) {
                const int yi = f2i_sat(roundf(yo + (float)dy));
                const int xi = f2i_sat(roundf(xo + (float)dx));
                if (yi >= 1 && yi < h - 1 && xi >= 1 && xi < w - 1) {
                    const uint8_t* p = g + (size_t)yi * pitch + xi;
                    const float gx = q255f((float)p[1]) - q255f((float)p[-1]);
                    const float gy = q255f((float)p[pitch]) - q255f((float)p[-pitch]);
                    const float fdx = (float)dx, fdy = (float)dy;
                    const float wgt =
                        __builtin_amdgcn_exp2f(__builtin_fmaf(kq, __builtin_fmaf(fdx, fdx, fdy * fdy), lf));
                    const float m = __builtin_amdgcn_sqrtf(__builtin_fmaf(gx, gx, gy * gy)) * wgt;
                    const unsigned bin = angle_bin(grad_angle(gy, gx));
                    if (bin != run_bin) {
                        atomicAdd(&hrow[run_bin], run);
                        run_bin = bin;
                        run = 0;
                    }
                    run += (unsigned long long)m;
                }
                if (++dx > R) {
                    dx = -R;
                    dy++;
                }
            }
            atomicAdd(&hrow[run_bin], run);
        }
        __syncthreads();
        float hv = 0.0f;
        if (lane < 36) {
            unsigned long long sum = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) sum += hist[k * kOriHist + lane];
            if (lane == 0) {
#pragma unroll
                for (int k = 0; k < 4; k++) sum += hist[k * kOriHist + 36];
            }
            if (lds) sum &= (1ull << 52) - 1ull;
            hv = (float)((double)sum * (1.0 / 1099511627776.0));
        }
        auto from_lane = [](int lane4, float v) {
            return __int_as_float(__builtin_amdgcn_ds_bpermute(lane4, __float_as_int(v)));
        };
        for (int it = 0; it < 2; it++) {
            const float pv = from_lane(prev4, hv), nv = from_lane(next4, hv);
            if (lane < 36) hv = over_3(pv + hv + nv);
        }
        // the values are not negative: their order is that of their bits
        const float mx = __uint_as_float(wave_max_u32(__float_as_uint(hv)));
        const float thr = mx * 0.8f;
        const float pv = from_lane(prev4, hv), nv = from_lane(next4, hv);
        const bool peak = lane < 36 && hv >= thr && hv > pv && hv > nv;
        const unsigned long long m = ballot64(peak);
        if (peak) {
            const int rank = __popcll(m & ((1ull << lane) - 1ull));
            const float den = pv - 2.0f * hv + nv;
            const float off = fabsf(den) > 1e-5f ? 0.5f * (pv - nv) / den : 0.0f;
            const float step = kTwoPi / 36.0f;
            const float center = ((float)lane + 0.5f) * step;
            const float a = center + off * step;
            // rem_euclid: a itself but for the first and last bins' edges
            float fa = a;
            if (!(a >= 0.0f && a < kTwoPi)) fa = rem_euclid(a, kTwoPi);
            if (fa > kPi) fa = fa - kTwoPi;
            if (rank < kMaxPeaks) angles[(size_t)c * kMaxPeaks + rank] = fa;
        }
        if (lane == 0) npeaks[c] = min((unsigned)__popcll(m), (unsigned)kMaxPeaks);
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Descriptor helpers: clamped u8 sample, get_gauss_pixel_bilinear.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float gauss_px(const uint8_t* g, int pitch, int w, int h, int x, int y,
                                          const float* q) {
    x = min(max(x, 0), w - 1);
    y = min(max(y, 0), h - 1);
    return q[g[(size_t)y * pitch + x]];
}

// get_gauss_pixel_bilinear (src/sift.rs:238-266)
__device__ __forceinline__ float bilinear(const uint8_t* g, int pitch, int w, int h, float x,
                                          float y, const float* q) {
    const float xf = floorf(x), yf = floorf(y);
    const float xc = xf + 1.0f, yc = yf + 1.0f;
    const float dx = x - xf, dy = y - yf;
    const int x0 = f2i_sat(xf), y0 = f2i_sat(yf), x1 = f2i_sat(xc), y1 = f2i_sat(yc);
    const float q11 = gauss_px(g, pitch, w, h, x0, y0, q);
    const float q21 = gauss_px(g, pitch, w, h, x1, y0, q);
    const float q12 = gauss_px(g, pitch, w, h, x0, y1, q);
    const float q22 = gauss_px(g, pitch, w, h, x1, y1, q);
    return q11 * (1.0f - dx) * (1.0f - dy) + q21 * dx * (1.0f - dy) + q12 * (1.0f - dx) * dy +
           q22 * dx * dy;
}

// Inclusive prefix sum over the 64 lanes of a fully active wave with DPP:
// shifts by 1, 2, 4, 8 inside each row of 16 lanes (lanes without a source add
// 0), then lane 15 of rows 0 and 2 is added to rows 1 and 3, and lane 31 to
// rows 2 and 3.
__device__ __forceinline__ int wave_incl_scan(int x) {
    x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true);   // row_shr:1
    x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true);   // row_shr:2
    x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true);   // row_shr:4
    x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true);   // row_shr:8
    x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
    x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
    return x;
}

// Sum over the 64 lanes of a fully active wave (DPP scan, then lane 63),
// returned to every lane; the order of the additions is fixed.
__device__ __forceinline__ float wave_sum_dpp(float v) {
    int x = __float_as_int(v);
    x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, true)));
    x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, true)));
    x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, true)));
    x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, true)));
    x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false)));
    x = __float_as_int(__int_as_float(x) + __int_as_float(__builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false)));
    return __int_as_float(__builtin_amdgcn_readlane(x, 63));
}

// Maximum over the 64 lanes of a fully active wave, returned to every lane.
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = fmaxf(v, __shfl_xor(v, m, 64));
    return v;
}

// Per-keypoint gain of the descriptor's fixed-point scale: the largest power of
// two 2^e (0 <= e <= 40) with M * 2^e <= lim, where M bounds |gx| and |gy| of
// every sample of the window and lim is their largest possible value (255 in
// texel units, 1 in [0, 1] units). Scaled by it, a sample's contribution
// mag * weight * fix is still at most sqrt(2) * fix, so the u32 sum bound holds,
// while a low-contrast window's sums use the high bits of the words instead of
// a few units of 2^-20 (whose rounding, relative to the window's small norm,
// reached 7e-4 of L2 at 3840x2160, contrast 0.03).
// desc_fix_gain returns 2^e, desc_fix_exp e.
__device__ __forceinline__ int desc_fix_exp(float M, float lim) {
    if (!(M > 0.0f)) return 0;
    int x;
    (void)frexpf(M, &x);                  // M in [2^(x-1), 2^x)
    int e = (lim > 1.0f ? 8 : 0) - x;     // M * 2^e in [128, 256), or [0.5, 1)
    if (ldexpf(M, e) > lim) e--;
    return min(max(e, 0), 40);
}
__device__ __forceinline__ float desc_fix_gain(float M, float lim) {
    return ldexpf(1.0f, desc_fix_exp(M, lim));
}

// k_descriptor's fixed-point gain exponent for one keypoint: that of its
// patch's texel range (max - min over the waves' (max << 8) | (255 - min) words),
// the same value in every lane.
__device__ __forceinline__ int desc_range_exp(const unsigned* wrange) {
    unsigned hi = 0u, lo = 0u;
#pragma unroll
    for (int w = 0; w < kThreads / 64; w++) {
        hi = max(hi, wrange[w] >> 8);
        lo = max(lo, wrange[w] & 255u);
    }
    const int range = (int)hi - (int)(255u - lo);
    return __builtin_amdgcn_readfirstlane(desc_fix_exp((float)range, 255.0f));
}

constexpr int kDescMaxR = 31;    // LDS path for sigma_octave <= 3.65
// The instantiation for windows up to R = 28 (99.5% of the keypoints of the
// default schedule, 20400 bytes of LDS, 64 VGPRs) fits 8 work-groups per CU, the R = 31 one 6.
constexpr int kDescSmallR = 28;
// Candidate capacities up to this (single frames up to 2048 x 1536, small
// batches) take every descriptor in one launch of the R <= kDescMaxR
// instantiation.
constexpr int kDescOneLaunchCap = 131072;
// LDS sizes of the descriptor instantiation for windows up to MR.
template <int MR>
struct DescDims {
    static constexpr int GS = 2 * MR + 3;         // bilinear grid row stride (floats)
    static constexpr int PatchRows = 2 * MR + 6;  // staged patch rows
    // staged patch row stride (bytes): the aligned words of a row, up to 3 + rows + 3 bytes
    static constexpr int PS = (2 * MR + 12) / 4 * 4;
};
// One histogram cell: the even-pair table (bins 0..7 in words 0..7) and the
// odd-pair table (bin b in word 9 + b, bin 0 again in word 17); 18 words keep
// every cell, and with it every bin pair, 8-byte aligned.
constexpr int kCellWords = 18;
constexpr int kOddBase = 9;                     // word of bin 0 in the odd-pair table
constexpr int kHistWords = 36 * kCellWords;     // one copy: 6 x 6 padded cells
constexpr int kHistCopies = 2;                  // even and odd lanes scatter into separate copies
constexpr int kMaxCopySamples = 2048;           // per-copy sample bound that keeps u32 sums exact

// Trilinear scatter of one sample (src/sift.rs:1012-1049), contribution
// ((m * wx) * wy) * wa in u32 fixed point, m = weighted magnitude * fix.
// The histogram is padded to 6 x 6 spatial cells (cells -1..4 in x and y): the
// reference drops neighbours outside the 4 x 4 grid, here they land in border
// cells that are never read, so there is no clamping and the four spatial
// neighbours are constant offsets. The two angle bins (a, a+1 mod 8) of each
// spatial neighbour go in ONE 64-bit LDS add: a cell's even-pair table holds
// bins 0..7 in its words 0..7 (pairs (0,1), (2,3), ... are 8-byte aligned); its
// odd-pair table holds bin b in word 9 + b and bin 0 again in word 17, so pairs
// (1,2), (3,4), (5,6), (7,0) are aligned too. Every bin sum of a copy stays
// below 2^32 (at most kMaxCopySamples samples of at most sqrt(2) * fix + 1/2
// each), so the low word never carries into the high word.
//
// desc_bins: the bin pair address of one sample (its spatial neighbour 0), as a byte
// offset, its four spatial weights t_k and its angle fraction da; ab, the angle in
// bins, may be anywhere in (-8, 8): its integer part is taken mod 8. hbytes: the
// byte offset of the copy's cell (0, 0), as f32 (whole numbers below 2^24, exact).
// The pair of bin a lies at byte 4 a + 36 (a & 1) of its cell: one v_perm picks that
// from eight bytes.
__device__ __forceinline__ unsigned desc_bins(float hbytes, float xb, float yb, float ab, float m,
                                              float (&tt)[4], float& da) {
    const float xf = floorf(xb), yf = floorf(yb), af = floorf(ab);
    const unsigned ai = ((unsigned)(int)af) & 7u;
    const float dx = xb - xf, dy = yb - yf;
    da = ab - af;
    static_assert(kOddBase == 9 && kCellWords == 18, "the bytes below");
    const unsigned pair = __builtin_amdgcn_perm(0x40183810u, 0x30082800u, ai);  // 0, 40, 8, 48, 16, 56, 24, 64
    const unsigned cell = (unsigned)(int)__builtin_fmaf(
        yf, 6.0f * 4.0f * kCellWords, __builtin_fmaf(xf, 4.0f * kCellWords, hbytes));
    const float t0 = m * (1.0f - dx), t1 = m * dx;
    tt[0] = t0 * (1.0f - dy);
    tt[1] = t1 * (1.0f - dy);
    tt[2] = t0 * dy;
    tt[3] = t1 * dy;
    return cell + pair;
}

// Adds four pairs of fixed-point sums (a[2k], a[2k+1]) at the spatial
// neighbours of a bin pair address, each rounded as (unsigned)(a + bias):
// bias 0.5 for plain sums, 0 for sums that started at 0.5.
template <int kHalfBiased = 0>
__device__ __forceinline__ void desc_add_pairs(unsigned long long* base, const float (&a)[8]) {
    constexpr int off[4] = {0, kCellWords / 2, 6 * kCellWords / 2, 7 * kCellWords / 2};
    constexpr float bias = kHalfBiased ? 0.0f : 0.5f;
#pragma unroll
    for (int k = 0; k < 4; k++)
        atomicAdd(base + off[k], ((unsigned long long)(unsigned)(a[2 * k + 1] + bias) << 32) |
                                     (unsigned)(a[2 * k] + bias));
}

__device__ __forceinline__ void desc_scatter(unsigned* hcopy, float xb, float yb, float ab,
                                             float m) {
    float tt[4], da;
    unsigned long long* const base = reinterpret_cast<unsigned long long*>(
        reinterpret_cast<char*>(hcopy) + desc_bins(7.0f * 4.0f * kCellWords, xb, yb, ab, m, tt, da));
    const float a[8] = {tt[0] * (1.0f - da), tt[0] * da, tt[1] * (1.0f - da), tt[1] * da,
                        tt[2] * (1.0f - da), tt[2] * da, tt[3] * (1.0f - da), tt[3] * da};
    desc_add_pairs(base, a);
}

// Interval of px where c * px + d lies in (-B, B) in real arithmetic; the
// caller widens it by one sample and the per-sample window test decides.
// A coefficient too small to move c * px by 0.1% of B over the window keeps the
// whole row or none of it.
__device__ __forceinline__ void desc_row_interval(float c, float d, float B, int R, float& lo,
                                                  float& hi) {
    if (fabsf(c) * (float)(R + 1) <= 1e-3f * B) {
        const bool keep = fabsf(d) < B * 1.002f;
        lo = keep ? -1e6f : 1e6f;
        hi = keep ? 1e6f : -1e6f;
        return;
    }
    const float rc = __builtin_amdgcn_rcpf(c);  // endpoints need far less than one sample of accuracy
    const float e1 = (-B - d) * rc, e2 = (B - d) * rc;
    lo = fminf(e1, e2);
    hi = fmaxf(e1, e2);
}

// One patch row of the descriptor's bilinear grid: texels (a, a+1) of the u8
// patch at byte offset a, interpolated along x in texel units (the x half of
// get_gauss_pixel_bilinear, src/sift.rs:238-266, as one lerp). The two texels
// come from aligned words: a byte-aligned 16-bit LDS read would be an
// unaligned access.
__device__ __forceinline__ float desc_lerp(const unsigned* wp, unsigned shift, float dx) {
    const unsigned r = __builtin_amdgcn_alignbyte(wp[1], wp[0], shift);
    const float p1 = (float)(r & 255u), p2 = (float)((r >> 8) & 255u);
    return __builtin_fmaf(p2 - p1, dx, p1);
}
__device__ __forceinline__ float desc_grid_row(const unsigned* pu, int a, float dx) {
    return desc_lerp(pu + ((unsigned)a >> 2), (unsigned)a & 3u, dx);
}

// Per-keypoint geometry of compute (src/sift.rs:940-960).
struct DescGeom {
    Keypoint base;
    const uint8_t* g;
    int w, h, pitch, R, side, np;
    unsigned k0;
    float xo, yo, so, bw, denom;
};

__device__ __forceinline__ DescGeom desc_geom(int c, const OctaveDesc* __restrict__ oct,
                                              const ImageParams* __restrict__ params,
                                              const Cand* __restrict__ cand,
                                              const Keypoint* __restrict__ ref,
                                              const unsigned* __restrict__ npeaks,
                                              const unsigned* __restrict__ koff) {
    DescGeom G;
    G.np = (int)npeaks[c];
    G.base = ref[c];
    G.k0 = koff[c];
    const OctaveDesc& O = oct[cand[c].job];
    const int S = params[O.img].num_intervals;
    const int gl = min(max(G.base.layer, 0), S + 2);
    G.g = O.levels + (long long)gl * O.level_stride;
    G.w = O.w;
    G.h = O.h;
    G.pitch = O.pitch;
    G.xo = over_pow2(G.base.x, G.base.octave);
    G.yo = over_pow2(G.base.y, G.base.octave);
    G.so = over_pow2(G.base.size, G.base.octave);
    G.bw = 3.0f * G.so;
    const float win = G.bw * 4.0f;
    const float wsig = 0.5f * win;
    G.denom = 2.0f * wsig * wsig;
    G.R = G.so > 0.0f ? f2i_sat(ceilf(win * sqrtf(2.0f) * 0.5f)) : 0;
    G.side = 2 * G.R + 1;
    return G;
}

// (ix, iy) range whose x_o + (ix - R) lies in [0, w-1) and y_o + (iy - R) in
// [0, h-1) (src/sift.rs:981-987), evaluated with the reference's f32 test at
// the candidate integers.
__device__ __forceinline__ void desc_bounds(const DescGeom& G, int& bx0, int& bx1, int& by0,
                                            int& by1) {
    const float wm1 = (float)(G.w - 1), hm1 = (float)(G.h - 1);
    bx0 = 0;
    bx1 = G.side - 1;
    by0 = 0;
    by1 = G.side - 1;
    // most windows lie inside the image: their ends decide all four (the sums grow
    // with ix and iy)
    const float r = (float)G.R;
    if (G.xo - r >= 0.0f && G.xo + r < wm1 && G.yo - r >= 0.0f && G.yo + r < hm1) return;
    while (bx0 <= bx1 && G.xo + (float)(bx0 - G.R) < 0.0f) bx0++;
    while (bx1 >= bx0 && G.xo + (float)(bx1 - G.R) >= wm1) bx1--;
    while (by0 <= by1 && G.yo + (float)(by0 - G.R) < 0.0f) by0++;
    while (by1 >= by0 && G.yo + (float)(by1 - G.R) >= hm1) by1--;
}

// Wave 0: sums the histogram copies of one peak, normalises, clips at 0.2,
// renormalises (src/sift.rs:889-913) and writes the descriptor and keypoint.
// The sums are divided by the fixed-point scale `fix`, or (kDivide false)
// multiplied by its exact reciprocal inv_fix when fix is a power of two.
template <bool kDivide>
__device__ __forceinline__ void desc_finish(const unsigned* hist, float fix, double inv_fix, int l,
                                            const Keypoint& base, float angle, unsigned kidx,
                                            int kcap, Keypoint* __restrict__ kps_out,
                                            float* __restrict__ desc_out) {
    float v[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
        const int dd = 2 * l + e;  // (iy * 4 + ix) * 8 + ia
        const int a = dd & 7;
        const int cell = ((dd >> 5) + 1) * 6 + (((dd >> 3) & 3) + 1);
        unsigned long long sum = 0;
#pragma unroll
        for (int cp = 0; cp < kHistCopies; cp++) {
            const unsigned* t = hist + cp * kHistWords + cell * kCellWords;
            sum += t[a];                // even-pair table
            sum += t[kOddBase + a];     // odd-pair table
            if (a == 0) sum += t[kOddBase + 8];
        }
        v[e] = kDivide ? (float)((double)sum / (double)fix) : (float)((double)sum * inv_fix);
    }
    float v0 = v[0], v1 = v[1];
    const float nrm = sqrtf(wave_sum_dpp(v0 * v0 + v1 * v1));
    if (nrm >= 1e-8f) {
        const float inv = 1.0f / nrm;
        v0 = fminf(v0 * inv, 0.2f);
        v1 = fminf(v1 * inv, 0.2f);
        const float n2 = sqrtf(wave_sum_dpp(v0 * v0 + v1 * v1));
        if (n2 >= 1e-8f) {
            const float inv2 = 1.0f / n2;
            v0 *= inv2;
            v1 *= inv2;
        }
    }
    if (kidx < (unsigned)kcap) {
        float2* dd = (float2*)(desc_out + (size_t)kidx * 128);
        dd[l] = make_float2(v0, v1);
        if (l == 0) {
            Keypoint o = base;
            o.angle = angle;
            kps_out[kidx] = o;
        }
    }
}

// ---------------------------------------------------------------------------
// k_descriptor<MR>: one workgroup (256) per refined keypoint with R <= MR
// (sigma_octave <= 3.65), looping over its orientation peaks
// (src/sift.rs:917-1060).
// Per keypoint: the clamped u8 patch of the Gaussian level around (x_o, y_o) --
// every texel the reference's get_gauss_pixel_bilinear can touch in the
// window, with its clamp-to-edge rule -- is staged in LDS (aligned 32-bit
// copies when the patch is inside the level, clamped byte loads at the
// borders), and the bilinear samples on the shifted grid (x_o + i, y_o + j),
// |i|,|j| <= R+1, are formed once from it, in texel units (0..255): gradients
// are differences of grid values, so their angle is the same and their
// magnitude is scaled by 1/255 with the Gaussian weight. A window sample (px, py) takes its
// gradient from the four grid neighbours (the reference's bilinear(x_s +- 1, y_s)
// and bilinear(x_s, y_s +- 1)).
// Per peak, the samples of each row whose rotated bin coordinates can fall in
// (-1, 4) form one interval (the rotated window is convex); the intervals,
// widened by one sample and clipped to the in-image rectangle, are cut into at
// most 256 segments of at most `per` consecutive samples of one row, one per
// thread, so nearly every lane works on in-window samples of a single row and
// the lanes of a wave sit far apart in the window (different histogram cells). Each sample still applies the window
// test xb, yb in (-1, 4), then computes mag * exp(-(px^2+py^2)/(2 (6 sigma_o)^2))
// and atan2 and scatters trilinearly into its copy of the histogram (even and
// odd lanes use separate copies, which halves same-address collisions of the
// LDS adds; integer adds: independent of the order). The fixed-point scale is
// 2^20 times the largest power of two that keeps the patch's texel range times
// it within 255 (desc_range_exp). Wave 0 sums the copies and normalises.
// Bound by vector instruction issue: 4790 wave instructions per keypoint of
// 1920x1080 frames, 64 of which take 3850 us (4930 with 6600).
// ---------------------------------------------------------------------------
// The candidate of keypoint k: from the list of the first `size` (mark_owner), or the
// last one of the n whose offset is at most k.
__device__ __forceinline__ int desc_owner(const int* __restrict__ owner, const unsigned* __restrict__ koff,
                                          unsigned n, int size, int k) {
    if (k < size) return owner[k];
    unsigned lo = 0, hi = n - 1;
    while (lo < hi) {
        const unsigned mid = (lo + hi + 1) >> 1;
        if (koff[mid] <= (unsigned)k) lo = mid;
        else hi = mid - 1;
    }
    return (int)lo;
}

// The items of a launch of k_descriptor: every candidate with all its peaks, the
// candidates of a list, or single keypoints (a candidate's peaks apart).
enum class DescItems { kAll, kList, kPeaks };

template <int MR, DescItems kItems>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(MR <= kDescSmallR ? 8 : 6))) void k_descriptor(
    const OctaveDesc* __restrict__ oct, const ImageParams* __restrict__ params,
    const Cand* __restrict__ cand, const unsigned* __restrict__ total, int cap,
    const Keypoint* __restrict__ ref, const unsigned* __restrict__ npeaks,
    const float* __restrict__ angles, const unsigned* __restrict__ koff, int kcap,
    Keypoint* __restrict__ kps_out, float* __restrict__ desc_out,
    const unsigned* __restrict__ in_count, const int* __restrict__ in_list,
    unsigned* __restrict__ out_count, int* __restrict__ out_list, unsigned* __restrict__ queue) {
    using D = DescDims<MR>;
    constexpr int kGS = D::GS, kPatchRows = D::PatchRows, kPS = D::PS;
    static_assert(kHistCopies * kHistWords * 4 >= kPatchRows * kPS + 4, "patch shares the histograms");
    // The u8 patch (and, when they fit beside it, the grid's column and row
    // terms) are dead once the grid is built; the histograms live after that.
    constexpr int kPatchBytes = (kPatchRows * kPS + 15) / 16 * 16;
    constexpr bool kTermsInPatch = kPatchBytes + 2 * kGS * (int)sizeof(float2) <= kHistCopies * kHistWords * 4;
    __shared__ __align__(16) unsigned pu[kHistCopies * kHistWords];
    __shared__ float grid[kGS * kGS];
    __shared__ float exs[2 * MR + 1];
    __shared__ int rspan[64];  // per row: first and last column of its samples (16 bits each)
    __shared__ int rpre[65];
    __shared__ int seg_len;
    __shared__ unsigned char seg_row[kThreads];  // the row of each segment
    // per wave: (max << 8) | (255 - min) of the patch texels it staged
    __shared__ unsigned wrange[kThreads / 64];
    // whether a grid row's texel row is not the one after its predecessor's (by the wave
    // that made the rows' terms)
    __shared__ int row_skips[2];
    __shared__ float2 terms_own[kTermsInPatch ? 1 : 2 * kGS];
    __shared__ float pang[kMaxPeaks], pcos[kMaxPeaks], psin[kMaxPeaks];
    uint8_t* const patch = reinterpret_cast<uint8_t*>(pu);
    unsigned* const hist = pu;
    auto pairs = [&](unsigned byte) {
        return reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(pu) + byte);
    };
    // grid columns / rows: texel offset, fraction
    float2* const gcol = kTermsInPatch ? reinterpret_cast<float2*>(patch + kPatchBytes) : terms_own;
    float2* const grw = gcol + kGS;
    // all candidates, or the ones an instantiation for smaller windows listed
    const int n = (int)min(kItems == DescItems::kAll ? *total : *in_count,
                           (unsigned)(kItems == DescItems::kPeaks ? kcap : cap));
    __shared__ int qslot[2];
    WorkQueue<kDescChunk> Q{queue, 0, 0, 0};
    for (int idx = Q.first(qslot); idx < n; idx = Q.next(qslot, idx)) {
        Q.prefetch(qslot);
        // the thread index passes through an empty asm in every iteration, so
        // the many cheap values derived from it are formed where they are used
        // instead of being hoisted out of this loop and kept live across it
        // (spilled to scratch at 7 waves per SIMD)
        int tid = (int)threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int wave = tid >> 6, lane = tid & 63;
        const int c = kItems == DescItems::kList    ? in_list[idx]
                      : kItems == DescItems::kPeaks ? desc_owner(in_list, koff, min(*total, (unsigned)cap), cap, idx)
                                                    : idx;
        const DescGeom G = desc_geom(c, oct, params, cand, ref, npeaks, koff);
        if (G.np == 0) continue;
        const int pk0 = kItems == DescItems::kPeaks ? idx - (int)G.k0 : 0;
        const int pk1 = kItems == DescItems::kPeaks ? pk0 + 1 : G.np;
        if (G.R > MR) {  // wider windows: listed for the next instantiation
            if (threadIdx.x == 0 && pk0 == 0) out_list[atomicAdd(out_count, 1u)] = c;
            continue;
        }
        const int R = G.R, side = G.side, gside = 2 * R + 3;
        const float xo = G.xo, yo = G.yo, bw = G.bw, denom = G.denom;
        // Before the first barrier each wave also has a table of its own to make: wave 0
        // the peaks' angles, wave 1 the grid's columns, wave 2 its rows, wave 3 the
        // Gaussian factors.
        if (tid < G.np) {  // the peaks' angles and their cos / sin, once per keypoint
            const float a = angles[(size_t)c * kMaxPeaks + tid];
            pang[tid] = a;
            pcos[tid] = cosf(a);
            psin[tid] = sinf(a);
        }
        {
            const int pside = 2 * R + 6;
            const int px0 = (int)floorf(xo) - R - 2, py0 = (int)floorf(yo) - R - 2;
            const int px0a = px0 & ~3, poff = px0 - px0a;
            unsigned tmax = 0u, tmin = 255u;
            const int nw = (poff + pside + 3) >> 2;  // aligned words of a row, <= kPS / 4
            if (px0 >= 0 && py0 >= 0 && px0a + 4 * nw <= G.w && py0 + pside <= G.h) {
                // interior: the words [px0a, round_up(px0 + pside, 4)) of each row lie
                // within the image. (Ending within the row's pitch is not enough: the
                // bytes past the width are whatever the memory held, and the texel
                // range below would take them in.) 16 words of 16 rows per pass, so a
                // pass is a fixed step in memory and in LDS; the one or two words past
                // the 16th of windows with R >= 26, one row per thread.
                constexpr int kPasses = (kPatchRows + 15) / 16;
                const int row = tid >> 4, wd = tid & 15;
                gbyte_t* const rowp = (gbyte_t*)G.g + ((size_t)py0 * G.pitch + px0a);
                const unsigned off = (unsigned)row * (unsigned)G.pitch + 4u * (unsigned)wd;
                unsigned wv[kPasses], we[2] = {0u, 0u};
#pragma unroll
                for (int k = 0; k < kPasses; k++) {
                    wv[k] = 0u;  // defined on every path: nothing carried across keypoints
                    if (row + 16 * k < pside && wd < nw)
                        wv[k] = *(gu32_t*)(rowp + (off + 16u * k * (unsigned)G.pitch));
                }
                const bool more = nw > 16 && tid < pside;
                const unsigned offe = (unsigned)tid * (unsigned)G.pitch + 64u;
                if (more) {
                    we[0] = *(gu32_t*)(rowp + offe);
                    if (nw > 17) we[1] = *(gu32_t*)(rowp + (offe + 4u));
                }
                // texel range of the staged words (a few texels left and right of
                // the patch included: a wider range is still a bound)
                auto range = [&](unsigned w) {
                    const unsigned b0 = w & 255u, b1 = (w >> 8) & 255u;
                    const unsigned b2 = (w >> 16) & 255u, b3 = w >> 24;
                    tmax = max(max(tmax, max(b0, b1)), max(b2, b3));
                    tmin = min(min(tmin, min(b0, b1)), min(b2, b3));
                };
                unsigned* const pw = pu + row * (kPS / 4) + wd;
#pragma unroll
                for (int k = 0; k < kPasses; k++) {
                    if (row + 16 * k < pside && wd < nw) {
                        range(wv[k]);
                        pw[16 * k * (kPS / 4)] = wv[k];
                    }
                }
                if (more) {
                    range(we[0]);
                    pu[tid * (kPS / 4) + 16] = we[0];
                    if (nw > 17) {
                        range(we[1]);
                        pu[tid * (kPS / 4) + 17] = we[1];
                    }
                }
            } else {
                const float inv_ps = 1.0f / (float)pside;
                for (int i = tid; i < pside * pside; i += kThreads) {
                    const int v = (int)(((float)i + 0.5f) * inv_ps), u = i - v * pside;
                    const int xx = min(max(px0 + u, 0), G.w - 1), yy = min(max(py0 + v, 0), G.h - 1);
                    const unsigned t = G.g[(size_t)yy * G.pitch + xx];
                    patch[v * kPS + poff + u] = (uint8_t)t;
                    tmax = max(tmax, t);
                    tmin = min(tmin, t);
                }
            }
            // Every grid value is a convex combination of patch texels, so every
            // sample's |gx| and |gy| is at most the patch's texel range: it sets
            // the keypoint's fixed-point gain (read after the barrier below).
            tmax = wave_max_u32(tmax);
            tmin = 255u - wave_max_u32(255u - tmin);
            if (lane == 0) wrange[wave] = (tmax << 8) | (255u - tmin);
            // the grid's column and row terms: x = x_o + i (and y = y_o + j) are the
            // same f32 sums for every point of a column (row), so their texel offset
            // and fraction are formed once
            bool skips = false;
            if (tid >= 64 && tid < 64 + gside) {
                const int t = tid - 64;
                const float x = xo + (float)(t - R - 1);
                const float xf = floorf(x);
                gcol[t] = make_float2(__int_as_float(min(max((int)xf - px0, 0), pside - 2)), x - xf);
            }
            if (tid >= 128 && tid < 128 + gside) {
                const int t = tid - 128;
                const float y = yo + (float)(t - R - 1);
                const float yf = floorf(y);
                const int v0 = min(max((int)yf - py0, 0), pside - 2);
                const int first = min(max((int)floorf(yo - (float)(R + 1)) - py0, 0), pside - 2);
                skips = v0 != first + t;
                grw[t] = make_float2(__int_as_float(v0 * kPS + poff), y - yf);
            }
            if (wave >= 2) {
                const unsigned long long m = ballot64(skips);
                if (lane == 0) row_skips[wave - 2] = m != 0ull;
            }
            // Gaussian weight exp(-(px^2+py^2)/denom) as exp(-px^2/denom) * exp(-py^2/denom)
            if (tid >= 192 && tid < 192 + side) {
                const int d = tid - 192 - R;
                exs[tid - 192] = expf(-(float)(d * d) / denom);
            }
            __syncthreads();
            {
                // Thread (band, gx) walks grid column gx down one band of rows.
                // Grid row gy interpolates patch rows v0 and v0 + 1 along x
                // ("top", "bot") and then along y; the next grid row's v0 is
                // v0 + 1 except where the clamp to the patch (or the f32 sum
                // y_o + j) makes it otherwise, so its "top" is this row's "bot"
                // and each patch row is interpolated once per band. Where no row
                // skips, the walk is a fixed step of the patch: every LDS address
                // is the last one plus a constant.
                const float inv_gs = __builtin_amdgcn_rcpf((float)gside);  // quotients of small integers, + 1/2
                const int nb = (int)(((float)kThreads + 0.5f) * inv_gs);   // bands: >= 3 (gside <= 65)
                const int band = (int)(((float)tid + 0.5f) * inv_gs), gx = tid - band * gside;
                if (band < nb) {
                    const int rows = (int)(((float)(gside + nb - 1) + 0.5f) * __builtin_amdgcn_rcpf((float)nb));
                    const int gy0 = band * rows, gy1 = min(gy0 + rows, gside);
                    const float2 cxd = gcol[gx];
                    const int cxo = __float_as_int(cxd.x);
                    const float dx = cxd.y;
                    if (!(row_skips[0] | row_skips[1])) {
                        if (gy0 < gy1) {
                            const int at = __float_as_int(grw[gy0].x) + cxo;
                            const unsigned* wp = pu + ((unsigned)at >> 2);
                            const unsigned sh = (unsigned)at & 3u;
                            float top = desc_lerp(wp, sh, dx);
                            float* gp = grid + gy0 * kGS + gx;
                            const float2* rp = grw + gy0;
                            const int n = gy1 - gy0;
#pragma unroll 3
                            for (int k = 0; k < n; k++) {
                                const float bot = desc_lerp(wp + (k + 1) * (kPS / 4), sh, dx);
                                gp[k * kGS] = __builtin_fmaf(bot - top, rp[k].y, top);
                                top = bot;
                            }
                        }
                    } else {
                        float top = 0.0f;
                        // patch offset of the previous row's v0; offsets are >= 0, so
                        // the first row of the band never matches it
                        int prev = -(1 << 30);
                        for (int gy = gy0; gy < gy1; gy++) {
                            const float2 ryd = grw[gy];
                            const int ro = __float_as_int(ryd.x);
                            if (ro != prev + kPS) top = desc_grid_row(pu, ro + cxo, dx);
                            const float bot = desc_grid_row(pu, ro + kPS + cxo, dx);
                            grid[gy * kGS + gx] = __builtin_fmaf(bot - top, ryd.y, top);
                            top = bot;
                            prev = ro;
                        }
                    }
                }
            }
        }
        __syncthreads();  // patch reads done before the histograms reuse its storage
        int bx0, bx1, by0, by1;
        desc_bounds(G, bx0, bx1, by0, by1);
        const int nrows = G.so > 0.0f ? max(by1 - by0 + 1, 0) : 0;  // <= 63
        // one division per keypoint: the empty asm keeps the compiler from repeating it
        // in each place of use
        float inv_bw = 1.0f / bw;
        asm volatile("" : "+v"(inv_bw));
        for (int pk = pk0; pk < pk1; pk++) {
            const float angle = uniform_f(pang[pk]);
            for (int i = tid; i < kHistCopies * kHistWords / 4; i += kThreads)
                reinterpret_cast<uint4*>(hist)[i] = make_uint4(0u, 0u, 0u, 0u);
            const float ca = uniform_f(pcos[pk]), sa = uniform_f(psin[pk]);
            const float msa = -sa;  // -sin * px is computed as (-sin) * px, the same value
            const float abin = uniform_f(angle * (4.0f / kPi));  // the peak angle in bins
            if (tid < 64) {
                // per-row sample intervals of the rotated window, prefix-summed
                int lo = 0, cnt = 0;
                if (tid < nrows) {
                    const int cy = by0 + tid;
                    const float py = (float)(cy - R);
                    const float B = 2.5f * bw;
                    float l1, h1, l2, h2;
                    desc_row_interval(ca, sa * py, B, R, l1, h1);
                    desc_row_interval(msa, ca * py, B, R, l2, h2);
                    const float lof = fmaxf(fmaxf(l1, l2), -1e5f), hif = fminf(fminf(h1, h2), 1e5f);
                    const int a = max((int)ceilf(lof) + R - 1, bx0);
                    const int b = min((int)floorf(hif) + R + 1, bx1);
                    lo = a;
                    cnt = max(b - a + 1, 0);
                    rspan[tid] = lo | ((lo + cnt - 1) << 16);  // columns < 64, last >= lo - 1
                }
                // Each row is cut into segments of at most `per` consecutive samples,
                // one segment per thread: per is the smallest value >= T / 256 that
                // gives at most 256 segments (per <= 16: a row holds at most 63
                // samples, so per = 16 gives at most 4 * 63 segments).
                const int T = __builtin_amdgcn_readlane(wave_incl_scan(cnt), 63);
                // (quotients of integers below 80 by at most 16, + 1/2 in the dividend: a
                // product with the reciprocal, truncated, is exact)
                int per = max((T + kThreads - 1) / kThreads, 1);
                auto segments = [&]() {
                    return (int)(((float)(cnt + per - 1) + 0.5f) * __builtin_amdgcn_rcpf((float)per));
                };
                int segs = wave_incl_scan(segments());
                while (__builtin_amdgcn_readlane(segs, 63) > kThreads) {
                    per++;
                    segs = wave_incl_scan(segments());
                }
                rpre[tid + 1] = segs;  // segment prefix over the rows
                // each segment's row, one segment of every row at a time
                const int mine = segments();
                unsigned char* const sr = seg_row + (segs - mine);
                for (int k = 0; ballot64(k < mine) != 0ull; k++)
                    if (k < mine) sr[k] = (unsigned char)tid;
                // the fixed-point scale 2^(20 + fe), passed with the segment length
                const int fe = desc_range_exp(wrange);
                if (tid == 0) {
                    rpre[0] = 0;
                    seg_len = per | (fe << 16);
                }
            }
            __syncthreads();
            const int per = seg_len & 0xffff, fe = seg_len >> 16;
            const int sg = lane * 4 + wave;  // lanes of a wave take segments far apart
            if (sg < rpre[nrows]) {
                const int r0 = seg_row[sg];
                const int span = rspan[r0];
                int cx = (span & 0xffff) + (sg - rpre[r0]) * per;
                const int len = min(per, (span >> 16) - cx + 1);
                // the row's terms (src/sift.rs:967-968 at px = 0, and the row's
                // Gaussian factor), formed as the row-interval pass forms them
                const int cy = by0 + r0;
                const float py = (float)(cy - R);
                const float rz = sa * py * inv_bw, rw = ca * py * inv_bw;
                const float wyf = exs[cy] * ldexpf(kDescFix / 255.0f, fe);
                // grid point (cx, cy) of sample (cx, cy) -- the up-left neighbour -- so that
                // all four gradient neighbours sit at non-negative offsets
                const float* grow = grid + (by0 + r0) * kGS;
                // rotated bin coordinates (rx / bw, ry / bw) (src/sift.rs:967-968), advanced
                // by one sample step along the row
                const float cai = ca * inv_bw, msai = msa * inv_bw;
                // consecutive samples of a thread often share their bin pair: their
                // contributions are summed in registers, starting from 0.5 so that the
                // rounding to fixed point is a plain conversion, and added to LDS once
                // per run. The sums are defined from the start (each run resets them
                // anyway): left undefined, they were carried through the keypoint
                // loop and spilled to scratch once per keypoint.
                // A run's bin pair is held as its byte offset in the histograms. The first
                // one is a cell by lane, where the sums of no run (0.5, truncated) add
                // zero: no step has to ask whether there is a run.
                const int copy = (lane & 1) * kHistWords * 4;  // neighbouring lanes: different copies
                const float hbytes = (float)(copy + 7 * 4 * kCellWords);
                unsigned acc_base = (unsigned)(copy + (lane >> 1) % 28 * (4 * kCellWords));
                float acc[8] = {0.5f, 0.5f, 0.5f, 0.5f, 0.5f, 0.5f, 0.5f, 0.5f};
                float u = __builtin_fmaf(cai, (float)(cx - R), rz);
                float v = __builtin_fmaf(msai, (float)(cx - R), rw);
                for (int i = 0; i < len; i++, cx++, u += cai, v += msai) {
                    // window: bin coordinates u + 1.5, v + 1.5 in (-1, 4) (src/sift.rs:969-977)
                    if (!(fabsf(u) < 2.5f && fabsf(v) < 2.5f)) continue;
                    const float* gq = grow + cx;
                    const float gx = gq[kGS + 2] - gq[kGS];
                    const float gyv = gq[2 * kGS + 1] - gq[1];
                    const float mag = __builtin_amdgcn_sqrtf(__builtin_fmaf(gx, gx, gyv * gyv));
                    const float m = mag * (exs[cx] * wyf);
                    // relative angle rem_euclid(atan2 - angle, 2pi) in bins (src/sift.rs:1009):
                    // ab in (-8, 8); the bin index wraps in desc_bins (& 7 of the
                    // integer floor) and the fraction ab - floor(ab) needs no wrap
                    const float ab = atan2_bins(gyv, gx) - abin;
                    float tt[4], da;
                    const unsigned base = desc_bins(hbytes, u + 1.5f, v + 1.5f, ab, m, tt, da);
                    if (base != acc_base) {  // a new bin pair: add the finished sums
                        desc_add_pairs<1>(pairs(acc_base), acc);
                        acc_base = base;
#pragma unroll
                        for (int q8 = 0; q8 < 8; q8++) acc[q8] = 0.5f;
                    }
                    const float wa0 = 1.0f - da;
#pragma unroll
                    for (int q4 = 0; q4 < 4; q4++) {
                        acc[2 * q4] = __builtin_fmaf(tt[q4], wa0, acc[2 * q4]);
                        acc[2 * q4 + 1] = __builtin_fmaf(tt[q4], da, acc[2 * q4 + 1]);
                    }
                }
                desc_add_pairs<1>(pairs(acc_base), acc);
            }
            __syncthreads();
            if (tid < 64) {
                // the keypoint and its output slot are read again here rather than
                // kept in registers through the peak loop (the index goes through an
                // empty asm so the compiler does not reuse the first reads)
                int cr = c;
                asm volatile("" : "+v"(cr));
                desc_finish<false>(hist, 0.0f, ldexp(1.0 / (double)kDescFix, -(seg_len >> 16)), tid,
                                   ref[cr], angle,
                                   koff[cr] + (unsigned)pk, kcap, kps_out,
                            desc_out);
            }
            __syncthreads();
        }
    }
}

// ---------------------------------------------------------------------------
// k_descriptor_wide: keypoints whose window exceeds the LDS patch
// (R > 31, sigma_octave > 3.65; none with the default sigma and 3 intervals).
// The reference's f32 arithmetic per sample; 256 contiguous chunks of the (2R+1)^2
// window as in k_descriptor. The fixed-point scale drops below 2^20 when a copy
// would see more than kMaxCopySamples samples, and is raised by the gain of the
// largest |gx|, |gy| of the window's samples.
// Every sample takes four bilinear values, and the samples' points lie on one grid
// (x_o + i, y_o + j), so the values of windows up to R = kWideGridR are made once
// into LDS, from column and row tables, and a gradient is four reads instead of 16
// gathers and 12 lerps, in the pass over the gradients' maximum and in every peak.
// x_s + 1 and x_s - 1 are f32 sums of their own: where one is not the grid's
// column (past a power of two the column's fraction loses a bit the sum kept),
// the column is marked and that value formed directly. Two frames of 1023 x 767 at
// sigma 2.0 (2.4 thousand wide windows): 811 -> 233 us.
// ---------------------------------------------------------------------------
constexpr int kWideGridR = 47;
constexpr int kWideGS = 2 * kWideGridR + 3;
constexpr int kWideGroups = 2048;  // of which three fit a CU at once; each takes few windows

__global__ __launch_bounds__(kThreads) void k_descriptor_wide(
    const OctaveDesc* __restrict__ oct, const ImageParams* __restrict__ params,
    const Cand* __restrict__ cand, const unsigned* __restrict__ total, int cap,
    const Keypoint* __restrict__ ref, const unsigned* __restrict__ npeaks,
    const float* __restrict__ angles, const unsigned* __restrict__ koff, int kcap,
    Keypoint* __restrict__ kps_out, float* __restrict__ desc_out,
    const unsigned* __restrict__ wide_count, const int* __restrict__ wide_list) {
    __shared__ float q[256];
    __shared__ __align__(16) unsigned hist[kHistCopies * kHistWords];
    __shared__ float wave_gmax[kThreads / 64];
    __shared__ float grid[kWideGS * kWideGS];
    // per grid column / row: the two clamped texel positions and the fraction
    __shared__ int c0[kWideGS], c1[kWideGS], r0[kWideGS], r1[kWideGS];
    __shared__ float cd[kWideGS], rd[kWideGS];
    // sample column / row t - 1: bit 0, its -1 neighbour is not grid t - 1; bit 1, its
    // +1 neighbour is not grid t + 1
    __shared__ unsigned char cmark[kWideGS], rmark[kWideGS];
    fill_q(q);
    __syncthreads();
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    (void)total;
    (void)cap;
    const int nw = (int)*wide_count;  // keypoints k_descriptor listed
    for (int i = blockIdx.x; i < nw; i += gridDim.x) {
        const int c = wide_list[i];
        const DescGeom G = desc_geom(c, oct, params, cand, ref, npeaks, koff);
        const int R = G.R, side = G.side, nsamp = side * side, gside = side + 2;
        const float wm1 = (float)(G.w - 1), hm1 = (float)(G.h - 1);
        const int per = (nsamp + kThreads - 1) / kThreads;
        const int i0 = (lane * 4 + wave) * per;
        const int iend = min(i0 + per, nsamp);
        const bool on_grid = R <= kWideGridR;
        if (on_grid) {
            if (tid < gside || (tid >= 128 && tid < 128 + gside)) {
                const bool is_row = tid >= 128;
                const int t = is_row ? tid - 128 : tid;
                const float o = is_row ? G.yo : G.xo;
                const int last = (is_row ? G.h : G.w) - 1;
                const float x = o + (float)(t - 1 - R), xf = floorf(x);
                (is_row ? r0 : c0)[t] = min(max(f2i_sat(xf), 0), last);
                (is_row ? r1 : c1)[t] = min(max(f2i_sat(xf + 1.0f), 0), last);
                (is_row ? rd : cd)[t] = x - xf;
                (is_row ? rmark : cmark)[t] = (unsigned char)((x - 1.0f != o + (float)(t - 2 - R) ? 1 : 0) |
                                                              (x + 1.0f != o + (float)(t - R) ? 2 : 0));
            }
            __syncthreads();
            const float inv = 1.0f / (float)gside;
            for (int k = tid; k < gside * gside; k += kThreads) {
                const int gy = (int)(((float)k + 0.5f) * inv), gx = k - gy * gside;
                const float dx = cd[gx], dy = rd[gy];
                const uint8_t* const g0 = G.g + (size_t)r0[gy] * G.pitch;
                const uint8_t* const g1 = G.g + (size_t)r1[gy] * G.pitch;
                const float q11 = q[g0[c0[gx]]], q21 = q[g0[c1[gx]]];
                const float q12 = q[g1[c0[gx]]], q22 = q[g1[c1[gx]]];
                grid[gy * kWideGS + gx] = q11 * (1.0f - dx) * (1.0f - dy) + q21 * dx * (1.0f - dy) +
                                          q12 * (1.0f - dx) * dy + q22 * dx * dy;
            }
            __syncthreads();
        }
        // the gradient of sample (cx, cy) at (xs, ys)
        auto gradient = [&](int cx, int cy, float xs, float ys, float& gx, float& gy) {
            if (on_grid && (cmark[cx + 1] | rmark[cy + 1]) == 0) {
                const float* p = grid + cy * kWideGS + cx;
                gx = p[kWideGS + 2] - p[kWideGS];
                gy = p[2 * kWideGS + 1] - p[1];
            } else {
                gx = bilinear(G.g, G.pitch, G.w, G.h, xs + 1.0f, ys, q) -
                     bilinear(G.g, G.pitch, G.w, G.h, xs - 1.0f, ys, q);
                gy = bilinear(G.g, G.pitch, G.w, G.h, xs, ys + 1.0f, q) -
                     bilinear(G.g, G.pitch, G.w, G.h, xs, ys - 1.0f, q);
            }
        };
        {
            // the largest |gx|, |gy| of the in-image samples sets the keypoint's
            // fixed-point gain (written per wave, read after the first barrier of
            // the peak loop)
            float gm = 0.0f;
            int cy = i0 / side, cx = i0 - cy * side;
            for (int k = i0; k < iend && G.np > 0; k++) {
                const float xs = G.xo + (float)(cx - R), ys = G.yo + (float)(cy - R);
                if (!(xs < 0.0f || xs >= wm1 || ys < 0.0f || ys >= hm1)) {
                    float gx, gy;
                    gradient(cx, cy, xs, ys, gx, gy);
                    gm = fmaxf(gm, fmaxf(fabsf(gx), fabsf(gy)));
                }
                if (++cx == side) {
                    cx = 0;
                    cy++;
                }
            }
            gm = wave_max(gm);
            if (lane == 0) wave_gmax[wave] = gm;
        }
        for (int pk = 0; pk < G.np; pk++) {
            const float angle = angles[(size_t)c * kMaxPeaks + pk];
            for (int i = tid; i < kHistCopies * kHistWords / 4; i += kThreads)
                reinterpret_cast<uint4*>(hist)[i] = make_uint4(0u, 0u, 0u, 0u);
            __syncthreads();
            const float ca = cosf(angle), sa = sinf(angle);
            unsigned* hw = hist + (lane & 1) * kHistWords;
            const float gmax = fmaxf(fmaxf(wave_gmax[0], wave_gmax[1]), fmaxf(wave_gmax[2], wave_gmax[3]));
            const float fix = kDescFix * fminf(1.0f, (float)kMaxCopySamples / (float)(128 * per)) *
                              desc_fix_gain(gmax, 1.0f);
            int cy = i0 / side, cx = i0 - cy * side - 1;
            for (int k = i0; k < iend; k++) {
                if (++cx == side) {
                    cx = 0;
                    cy++;
                }
                const float py = (float)(cy - R), px = (float)(cx - R);
                const float rx = ca * px + sa * py;
                const float ry = -sa * px + ca * py;
                const float xb = rx / G.bw + 4.0f / 2.0f - 0.5f;
                const float yb = ry / G.bw + 4.0f / 2.0f - 0.5f;
                if (!(xb > -1.0f && xb < 4.0f && yb > -1.0f && yb < 4.0f)) continue;
                const float xs = G.xo + px, ys = G.yo + py;
                if (xs < 0.0f || xs >= wm1 || ys < 0.0f || ys >= hm1) continue;
                float gx, gy;
                gradient(cx, cy, xs, ys, gx, gy);
                const float wt = expf(-(px * px + py * py) / G.denom);
                const float mag = sqrtf(gx * gx + gy * gy);
                // rem_euclid(d, 2 pi): |d| <= 2 pi, so its remainder is d itself, or a
                // zero of its sign at the ends
                const float d = atan2f(gy, gx) - angle;
                const float m = fabsf(d) < kTwoPi ? d : copysignf(0.0f, d);
                const float ar = m < 0.0f ? m + kTwoPi : m;
                desc_scatter(hw, xb, yb, ar * 8.0f / kTwoPi, mag * wt * fix);
            }
            __syncthreads();
            if (tid < 64)
                desc_finish<true>(hist, fix, 0.0, tid, G.base, angle, G.k0 + (unsigned)pk, kcap, kps_out,
                            desc_out);
            __syncthreads();
        }
    }
}

// u8 descriptors of the WebGPU backends (src/shaders/descriptor.wgsl:256-262):
// trunc(clamp(d * 512, 0, 255)) of each value, 4 values per lane.
__device__ __forceinline__ unsigned desc_u8_of(float d) {
    return (unsigned)fminf(fmaxf(d * 512.0f, 0.0f), 255.0f);
}

__global__ __launch_bounds__(256) void k_desc_u8(const float4* __restrict__ desc,
                                                 const unsigned* __restrict__ count, int kcap,
                                                 unsigned* __restrict__ out) {
    const size_t words = (size_t)min(*count, (unsigned)kcap) * 32;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < words;
         i += (size_t)gridDim.x * blockDim.x) {
        const float4 v = desc[i];
        out[i] = desc_u8_of(v.x) | (desc_u8_of(v.y) << 8) | (desc_u8_of(v.z) << 16) |
                 (desc_u8_of(v.w) << 24);
    }
}

}  // namespace

void launch_extrema(const OctaveDesc* d_oct, int noct, int total_rows, const ImageParams* d_params,
                    unsigned long long* d_bits, unsigned* d_counts, int nslots, bool zeroed, hipStream_t s) {
    // the counters after the row-slot counts (the descriptor's lists, the work queues)
    if (!zeroed)
        hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(64), 0, s, d_counts + nslots, kCountExtra, 0u);
    if (total_rows <= 0) return;
    hipLaunchKernelGGL(k_extrema, dim3(total_rows), dim3(kThreads), 0, s, d_oct, noct, d_params,
                       d_bits, d_counts);
}

bool extrema_tile_supported(int S) { return S >= 1 && S <= 6; }

void launch_extrema_tile(int S, int strip_rows, const OctaveDesc* d_oct, int noct, int total_tiles,
                         const ImageParams* d_params, unsigned long long* d_bits, unsigned* d_counts,
                         int nslots, bool zeroed, hipStream_t s) {
    // the row-slot counts and the counters after them (the descriptor's lists, the work queues)
    if (!zeroed)
        hipLaunchKernelGGL(k_fill_u32, dim3((nslots + kCountExtra + 255) / 256), dim3(256), 0, s, d_counts,
                           nslots + kCountExtra, 0u);
    if (total_tiles <= 0) return;
    switch (S) {
#define SH_EXT(SS) \
        case SS: hipLaunchKernelGGL(k_extrema_tile<SS>, dim3(total_tiles), dim3(kThreads), 0, s, d_oct, \
                                    noct, d_params, d_bits, d_counts, strip_rows); break;
        SH_EXT(1) SH_EXT(2) SH_EXT(3) SH_EXT(4) SH_EXT(5) SH_EXT(6)
#undef SH_EXT
        default: break;
    }
}

void launch_compact(const OctaveDesc* d_oct, int noct, int nslots, const unsigned long long* d_bits,
                    const unsigned* d_counts, unsigned* d_offsets, unsigned* d_tmp, Cand* d_cand, int cap,
                    hipStream_t s) {
    if (nslots <= 0) {  // no octave: no candidates
        hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(kScanSingleThreads), 0, s, d_counts, 0, nullptr,
                           d_offsets, FinalizeArgs{}, nullptr);
        return;
    }
    // slots per wave: enough that the work-groups' reads of the counts before theirs
    // stay a few MB in all (12756 slots of 3840 x 2160: 10 MB). With the sums of tiles
    // only the counts of the group's own tile are read: 16 frames of 640 x 480 (45
    // thousand slots) take 34 / 27 / 25 / 25 us with 1 / 2 / 4 / 8 slots a wave, 8 of
    // 1280 x 720 30 / 25 / 22 / 25, 64 of 1920 x 1080 282 / 202 / 157 / 136.
    const bool tiled = nslots > kCompactScanMax;
    const int spw = nslots <= 2048                   ? 1
                    : nslots <= 4096                 ? 2
                    : nslots <= 8192                 ? 4
                    : tiled && nslots < 65536        ? 4
                                                     : kCompactSlots;
    const int per = (kThreads / 64) * spw;  // slots per work-group
    if (tiled)
        hipLaunchKernelGGL(k_scan_reduce, dim3((nslots + kScanTile - 1) / kScanTile), dim3(kThreads), 0, s,
                           d_counts, nslots, nullptr, d_tmp);
    hipLaunchKernelGGL(k_compact, dim3((nslots + per - 1) / per), dim3(kThreads), 0, s, d_oct, noct, nslots,
                       d_bits, d_counts, tiled ? d_tmp : nullptr, d_offsets, d_cand, cap, spw);
}

// The scan of the cap candidates' peak counts, of which d_total are there: d_koff has
// cap + 1 entries, d_tmp ceil(cap / 4096) + 1.
void launch_keypoint_offsets(const unsigned* d_npeaks, int cap, const unsigned* d_total, unsigned* d_koff,
                             unsigned* d_tmp, const unsigned* d_slot_offsets, const int* d_img_slot_begin,
                             int nimg, unsigned* d_summary, unsigned* d_out_offsets, int* d_owner, hipStream_t s) {
    const FinalizeArgs F{d_slot_offsets, d_img_slot_begin, nimg, d_koff, d_total, cap, d_summary, d_out_offsets};
    if (cap > kDescOneLaunchCap) d_owner = nullptr;
    if (cap <= kScanSingleMax) {
        hipLaunchKernelGGL(k_scan_single, dim3(1), dim3(kScanSingleThreads), 0, s, d_npeaks, cap, d_total,
                           d_koff, F, d_owner);
        return;
    }
    const int tiles = (cap + kScanTile - 1) / kScanTile;
    hipLaunchKernelGGL(k_scan_reduce, dim3(tiles), dim3(kThreads), 0, s, d_npeaks, cap, d_total, d_tmp);
    hipLaunchKernelGGL(k_scan_down, dim3(tiles), dim3(kThreads), 0, s, d_npeaks, cap, d_total, d_tmp, d_koff,
                       F, d_owner);
}

static int grid_for(int cap, int per_block, int max_blocks) {
    int g = (cap + per_block - 1) / per_block;
    return g < 1 ? 1 : (g > max_blocks ? max_blocks : g);
}

// Work-groups of `kernel` that fit on the current device at once (its
// occupancy times the CU count), computed once per kernel.
static int resident_groups(const void* kernel, int block) {
    static std::mutex mu;
    static std::map<const void*, int> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(kernel);
    if (it != cache.end()) return it->second;
    int per_cu = 0, cus = 0, dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, 0) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        per_cu <= 0 || cus <= 0) {
        per_cu = 4;
        cus = 256;
    }
    const int g = per_cu * cus;
    cache[kernel] = g;
    return g;
}

// The keypoint kernels take their keypoints by a static grid-stride assignment;
// SIFT_HIP_QUEUE=1 (read on every launch) gives them the device work queue
// instead (the same results; on 64 x 1920x1080 frames it was 45% slower for
// k_orient and even for k_descriptor).
static bool queue_enabled() {
    const char* e = getenv("SIFT_HIP_QUEUE");
    return e && e[0] == '1';
}

// With few candidates each orientation wave refines its own: the whole wave does one
// candidate's arithmetic, but a launch and the latency of its few waves go (k_refine and
// k_orient 640x480 24 -> 14 us, 1280x720 29 -> 21, 1920x1080 32 -> 29; 8 x 640x480, whose
// capacity is just above the limit, 45 -> 48).
bool orient_refines(int cap) { return cap <= 65536; }

void launch_refine(const OctaveDesc* d_oct, const ImageParams* d_params, const Cand* d_cand,
                   const unsigned* d_total, int cap, Keypoint* d_ref, int* d_valid,
                   float* d_cand_resp, hipStream_t s) {
    hipLaunchKernelGGL(k_refine, dim3(grid_for(cap, kRefineThreads, 8192)), dim3(kRefineThreads), 0, s, d_oct,
                       d_params, d_cand, d_total, cap, d_ref, d_valid, d_cand_resp);
}

void launch_orient(const OctaveDesc* d_oct, const ImageParams* d_params, const Cand* d_cand,
                   const unsigned* d_total, int cap, Keypoint* d_ref, int* d_valid, unsigned* d_npeaks,
                   float* d_angles, unsigned* d_queue, bool refine, hipStream_t s) {
    // work queue: as many work-groups as fit, each taking keypoints until none
    // are left; or grid-stride over the candidates with many more work-groups
    // than fit at once (each takes only a few keypoints, so the launch ends evenly).
    // Where the capacity says few candidates, half as many: the groups beyond the
    // count only start and end (640x480 17.6 us with 65536, 11.0 with 32768;
    // 1920x1080 22.5 and 19.5), while 64 frames take 648 us with 32768 and 630 with 65536.
    const int most = cap <= kDescOneLaunchCap ? 32768 : 65536;
    const bool q = queue_enabled();
    const int grid = q ? std::min(resident_groups((const void*)k_orient<false>, 64), grid_for(cap, 1, most))
                       : grid_for(cap, 1, most);
    // (d_queue: kNumXcd counters)
    if (refine)
        hipLaunchKernelGGL(k_orient<true>, dim3(grid), dim3(64), 0, s, d_oct, d_params, d_cand, d_total, cap,
                           d_ref, d_valid, d_npeaks, d_angles, q ? d_queue : nullptr);
    else
        hipLaunchKernelGGL(k_orient<false>, dim3(grid), dim3(64), 0, s, d_oct, d_params, d_cand, d_total, cap,
                           d_ref, d_valid, d_npeaks, d_angles, q ? d_queue : nullptr);
}

void launch_descriptor(const OctaveDesc* d_oct, const ImageParams* d_params, const Cand* d_cand,
                       const unsigned* d_total, int cap, const Keypoint* d_ref,
                       const unsigned* d_npeaks, const float* d_angles, const unsigned* d_koff,
                       int kcap, Keypoint* d_kps, float* d_desc, unsigned* d_wide_count,
                       int* d_wide_list, unsigned* d_mid_count, int* d_mid_list, unsigned* d_queues,
                       const unsigned* d_count, int max_radius, hipStream_t s) {
    // as k_orient: a work queue, or few keypoints per work-group. Windows up to
    // kDescSmallR run at 8 work-groups per CU and list the few others for the
    // kDescMaxR instantiation (6 per CU), which lists still wider ones for
    // k_descriptor_wide. d_queues: the two instantiations' queue counters
    // (kNumXcd each). d_count: the number of keypoints.
    const bool q = queue_enabled();
    if (cap <= kDescOneLaunchCap) {
        // few candidates (single frames, small batches): one launch of the wide
        // instantiation; the GPU is far from full, so its lower occupancy costs less
        // than the second launch's latency. It takes keypoints rather than candidates
        // (d_mid_list holds their candidates): the launch lasts as long as its
        // longest group, and a candidate's two to four peaks one after the other
        // were that (640x480: 59 us, 30 us so, and 1 us more in the offsets' scan;
        // 1920x1080: 97 and 82, 4 more), while the patch and grid that the peaks then
        // each make are work for idle CUs. Full launches keep the peaks together.
        const void* kall = (const void*)k_descriptor<kDescMaxR, DescItems::kPeaks>;
        const int most = 16384;  // 4096: 84 us at 1920x1080; 8192 to 49152: the same
        const int g = q ? std::min(resident_groups(kall, kThreads), grid_for(kcap, 1, most))
                        : grid_for(kcap, 1, most);
        hipLaunchKernelGGL((k_descriptor<kDescMaxR, DescItems::kPeaks>), dim3(g), dim3(kThreads), 0, s, d_oct,
                           d_params, d_cand, d_total, cap, d_ref, d_npeaks, d_angles, d_koff, kcap,
                           d_kps, d_desc, d_count, d_mid_list, d_wide_count, d_wide_list,
                           q ? d_queues + kNumXcd : nullptr);
        if (max_radius > kDescMaxR)
            hipLaunchKernelGGL(k_descriptor_wide, dim3(kWideGroups), dim3(kThreads), 0, s, d_oct, d_params, d_cand,
                               d_total, cap, d_ref, d_npeaks, d_angles, d_koff, kcap, d_kps, d_desc,
                               d_wide_count, d_wide_list);
        return;
    }
    const void* k28 = (const void*)k_descriptor<kDescSmallR, DescItems::kAll>;
    const void* k31 = (const void*)k_descriptor<kDescMaxR, DescItems::kList>;
    const int g28 = q ? std::min(resident_groups(k28, kThreads), grid_for(cap, 1, 49152)) : grid_for(cap, 1, 49152);
    const int g31 = q ? std::min(resident_groups(k31, kThreads), grid_for(cap, 1, 49152)) : grid_for(cap, 1, 49152);
    hipLaunchKernelGGL((k_descriptor<kDescSmallR, DescItems::kAll>), dim3(g28), dim3(kThreads), 0, s, d_oct,
                       d_params, d_cand, d_total, cap, d_ref, d_npeaks, d_angles, d_koff, kcap,
                       d_kps, d_desc, nullptr, nullptr, d_mid_count, d_mid_list, q ? d_queues : nullptr);
    if (max_radius <= kDescSmallR) return;
    hipLaunchKernelGGL((k_descriptor<kDescMaxR, DescItems::kList>), dim3(g31), dim3(kThreads), 0, s, d_oct,
                       d_params, d_cand, d_total, cap, d_ref, d_npeaks, d_angles, d_koff, kcap,
                       d_kps, d_desc, d_mid_count, d_mid_list, d_wide_count, d_wide_list,
                       q ? d_queues + kNumXcd : nullptr);
    if (max_radius > kDescMaxR)
        hipLaunchKernelGGL(k_descriptor_wide, dim3(kWideGroups), dim3(kThreads), 0, s, d_oct, d_params, d_cand,
                           d_total, cap, d_ref, d_npeaks, d_angles, d_koff, kcap, d_kps, d_desc,
                           d_wide_count, d_wide_list);
}

// A keypoint's octave sigma is sigma * 2^(l / S) with l, its refined layer, below
// S + 0.5 (the refinement keeps layers 1 .. S and offsets below 0.5), and its
// descriptor radius the ceiling of 12 sqrt(1/2) of that; 1e-4 for the roundings.
int descriptor_max_radius(float sigma, int intervals) {
    const double so = (double)sigma * exp2(1.0 + 0.5 / intervals);
    return (int)ceil(std::min(so * 6.0 * sqrt(2.0) * 1.0001, 1e9));
}

void launch_desc_u8(const float* d_desc, const unsigned* d_count, int kcap, uint8_t* d_out,
                    hipStream_t s) {
    if (kcap <= 0) return;
    const int blocks = (int)std::min<long long>(1024, ((long long)kcap * 32 + 255) / 256);
    hipLaunchKernelGGL(k_desc_u8, dim3(blocks), dim3(256), 0, s, (const float4*)d_desc, d_count, kcap,
                       (unsigned*)d_out);
}

}  // namespace sh
