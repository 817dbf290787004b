// Wide block (chunked prefill) on the matrix cores: packed-affine weights
// times up to 256 RHS, y[t][r] = sum_c (q[r,c]*s[r,g] + b[r,g]) * x[t][c],
// computed in the factored form
//     y[t][r] = sum_g ( s[r,g] * D[r,t,g] + b[r,g] * S[t,g] ),
//     D[r,t,g] = sum_{c in g} q[r,c] * x[t,c],  S[t,g] = sum_{c in g} x[t,c].
// D runs on v_mfma_f32_16x16x32_f16 with exact centred codes against x split
// into hi/lo f16 parts, accurate to 2^-22 of the value and 2^-40 of the largest
// of its RHS and 64 columns, or, in group 32, on v_mfma_f32_16x16x32_bf16 against
// the three bf16 parts of x, which are all of it; factors and scales multiply D
// in FP32 and the bias term is an FP32 matrix product of S and b
// (v_mfma_f32_16x16x4_f32 over four groups at a time).
//
// Launches: wide_prep_kernel (x images), wide_mfma_kernel and, where K is
// split across workgroups, wide_sum_kernel.
//
// wide_mfma_kernel: a workgroup of NW waves owns 16*NRT rows x 16*NCT RHS
// over one K split; wave w takes every NW-th 128-column unit (class w), all of
// the workgroup's rows and RHS: 4*NRT*NCT FP32 accumulators per lane. Each
// x fragment (1 KB) is loaded once per NRT tiles and each unpacked code is
// used for NCT RHS tiles. Codes and x go straight to registers one unit ahead;
// four consecutive lanes load 64 contiguous bytes of a code row, and the wave
// turns a tile into operand order through its own piece of LDS (loading in
// operand order, 16 rows for every 16 lanes, made the L1 look up 64 lines for
// each 512 bytes). Metadata streams through LDS, expanded to FP32, a chunk of
// four groups per class at a time. At the end the classes meet in LDS and are
// added in a fixed order.
//
// What bounds it: up to 16 RHS the codes (17408x5120, Q4, 5 RHS: 21 us with the
// prep launch, 50 MB; one wave in flight per SIMD and a prep of 5 us keep it
// from the 11 us of a copy), then issue: two products for every code (hi, lo)
// and beside 8 of them 18 vector instructions of unpacking, 16 of factors and
// scales and 8 of staging. 24 RHS 28 us, 64 RHS 49 us, 128 RHS 67 us in long
// runs, 0.68 PFLOP/s of products. A workgroup of 272 rows x 32 RHS with codes in
// operand order and without the factors and the centring took 35, 61 and 66 us;
// blocks of four, which Q8 and the other groups ran as, 145 us for 64 RHS over
// a Q8 5120x5120 (24 now).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "../../include/qmr.h"
#include "kernels.hpp"
#include "mfma_common.hpp"

namespace qmr {
namespace {

using namespace mfma;

typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

// Codes as f16, centred: less the middle of their range (8 or 128), which goes
// into the group's bias as middle * scale. Uncentred, s * D and b * S are large
// and cancel: at 5120 columns 2.4e-7 against 64 bits for Q4 and 2.6e-7 for Q8.
// A code in the low bits of 1024 (in bits 4-7 of 64) is that number plus the
// code; less the middle too it is exact, and a normal number: as subnormals of
// 2^-20 (Q4) the sums lose bits beside large columns.
constexpr float middle_of(int bits) { return bits == 4 ? 8.f : 128.f; }
// Masks and numbers stay in registers, so that one v_and_or_b32 does both.
template <int BITS>
struct CodeConsts {
    uint32_t low = BITS == 4 ? 0x000F000Fu : 0x00FF00FFu, high = 0x00F000F0u;
    uint32_t at_low = 0x64006400u, at_high = 0x54005400u;
    __device__ __forceinline__ CodeConsts() { asm("" : "+s"(low), "+s"(high), "+v"(at_low), "+v"(at_high)); }
};
template <int BITS>
__device__ __forceinline__ u4 f16_codes(const u2 &w, const CodeConsts<BITS> &c) {
    const u2 up = w >> 8;
    const _Float16 k = _Float16(1024 + middle_of(BITS)), m = _Float16(64 + 8);
    auto low = [&](uint32_t v) { return (v & c.low) | c.at_low; };
    auto high = [&](uint32_t v) { return (v & c.high) | c.at_high; };
    if constexpr (BITS == 4) {
        const h8 v = __builtin_bit_cast(h8, u4{low(w.x), high(w.x), low(up.x), high(up.x)});
        return __builtin_bit_cast(u4, v - h8{k, k, m, m, k, k, m, m});
    } else {
        return __builtin_bit_cast(u4, __builtin_bit_cast(h8, u4{low(w.x), low(up.x), low(w.y), low(up.y)}) - k);
    }
}

// Group 32: codes as bf16, centred, against x in three bf16 parts, which hold
// all 24 bits of an FP32 value over its whole range: such blocks ran on the
// vector ALU, which multiplies FP32 values, and in fewer bits a token's small
// columns would be lost beside its large ones. Error against 64 bits at 5120
// columns 1.5e-7 (Q4) and 1.4e-7 (Q8), on the vector ALU 2.5e-7 and 2.0e-7;
// with one column 1e4 times the others 1.8e-7 and 1.7e-7 (Q4 in two f16 parts
// 9e-7). The third part costs 5% at 4 RHS, 21% at 64 and 39% at 200 (9001x4160 Q4).
template <int BITS>
__device__ __forceinline__ u4 bf16_codes(const u2 &w) {
    auto pair = [](float lo, float hi) {  // exact: at most eight bits each
        return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
    };
    if constexpr (BITS == 4) {  // sixteenths
        const uint32_t even = w.x ^ 0x88888888u, odd = even >> 4;
        auto f = [](uint32_t v) { return __builtin_amdgcn_cvt_off_f32_i4(int(v)); };
        return u4{pair(f(even), f(odd)), pair(f(even >> 8), f(odd >> 8)), pair(f(even >> 16), f(odd >> 16)),
                  pair(f(even >> 24), f(odd >> 24))};
    } else {
        const uint32_t x = w.x ^ 0x80808080u, y = w.y ^ 0x80808080u;
        auto f = [](uint32_t v, int k) { return float(int8_t(v >> (8 * k))); };
        return u4{pair(f(x, 0), f(x, 1)), pair(f(x, 2), f(x, 3)), pair(f(y, 0), f(y, 1)), pair(f(y, 2), f(y, 3))};
    }
}
// Factors of a group 32 x and of its scales: code * x is at most half of x, so
// that a group's sum overflows where the sum of its x does, not before.
template <int BITS>
constexpr float kXFactor = BITS == 4 ? 1.f : 1.f / 256;
template <int BITS>
constexpr float kSFactor = BITS == 4 ? 16.f : 256.f;

template <bool G32>
__device__ __forceinline__ f4 product(const u4 &x, const u4 &codes, const f4 &c) {
    if constexpr (G32)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, x), __builtin_bit_cast(b8, codes), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, x), __builtin_bit_cast(h8, codes), c, 0, 0, 0);
}

constexpr uint32_t kUnit = 128;                 // columns per unit: four K steps of the MFMA
constexpr int kRhsBlock = 32;                   // RHS tiles come in pairs
constexpr int kFragBytes = 1024;                // one MFMA A fragment (64 lanes x 16 B)
// An image: one unit of one RHS tile. Its fragments [K step][part], then the
// column sums [quarter (group 32) or half][16] f32, then (not group 32) the
// factors [half][16] that undo the power of two of x, as the exponent byte of an
// FP32 value.
constexpr uint32_t parts_of(bool g32) { return g32 ? 3 : 2; }
constexpr uint32_t img_sums(bool g32) { return 4 * parts_of(g32) * kFragBytes; }
constexpr uint32_t img_bytes(bool g32) { return img_sums(g32) + 256; }
constexpr uint32_t kImgFactors = img_sums(false) + 128;

// A wave's piece of LDS: codes on their way to operand order, 64 bytes of each
// row (one unit of Q4 or half a unit of Q8). The 16-byte pieces of a row change
// places with every fourth row, so that neither the writes nor the reads of 16
// rows meet in a bank.
constexpr uint32_t kCodePitch = 64;
constexpr size_t code_bytes(int nrt) { return size_t(16) * nrt * kCodePitch; }
__device__ __forceinline__ uint32_t code_piece(uint32_t row16, uint32_t piece) { return (piece ^ (row16 >> 2 & 3)) * 16; }
// A chunk's metadata, two buffers: per row and class four scales, then the
// same for the biases. The pitch puts the 16 rows of a read in 16 banks (and
// with four waves and 8 row tiles it leaves room for two workgroups per CU).
constexpr int meta_pitch(int nw) { return 4 * nw + 2; }
constexpr size_t meta_bytes(int nrt, int nw) { return size_t(16) * nrt * meta_pitch(nw) * 8; }
constexpr int kRedPad = 16;  // words between row tiles of the final planes
constexpr size_t kFlagBytes = 64;  // behind the planes: a word per wave and RHS tile
constexpr size_t wide_lds_bytes(int nrt, int nct, int nw) {
    const size_t red = size_t(nw > 4 ? 4 : nw) * nrt * (nct * 256 + kRedPad) * 4;  // [plane][rt][ct][v][lane] f32
    return std::max(2 * meta_bytes(nrt, nw) + nw * code_bytes(nrt), red + kFlagBytes);
}

// Byte offsets of the contraction kernel's loads, as the per-lane vector
// offset and the wave-uniform scalar offset of a buffer load. A load outside
// its view (a row past the matrix, columns past the row, a unit past the
// split, an RHS tile past the images) gets the vector offset kOut, which by
// itself lies past every view's extent, so it reads zeros whether or not the
// range check adds the scalar offset (kOut plus any scalar offset here stays
// below 2^32); every other load has voffset + soffset + size within its view.
// The kernel takes every offset from these functions, and
// qmr_wide_address_extent walks them on the host.
struct WideAddr {
    uint32_t rows, units, tiles, row_bytes;  // units: end of the split's; tiles: RHS tiles with an image
    uint32_t ntb;                            // pairs of RHS tiles
    bool g32;
    // Lane (row16, piece) loads 16 bytes of rows row + 16 rt (row = the row
    // block's first plus row16) at byte 64 seg + 16 piece; a unit is one
    // 64-byte segment of Q4, two of Q8. Tiles from code_tiles on have no such
    // row, or the row no such bytes.
    __host__ __device__ uint32_t row_tiles(uint32_t row) const { return row < rows ? (rows - row + 15) / 16 : 0; }
    __host__ __device__ uint32_t code_tiles(uint32_t row_tiles, uint32_t u, uint32_t seg, uint32_t piece) const {
        return u < units && 64 * seg + 16 * piece < row_bytes ? row_tiles : 0;
    }
    __host__ __device__ uint32_t code_at(uint32_t row, uint32_t piece) const { return row * row_bytes + 16 * piece; }
    __host__ __device__ uint32_t code_v(uint32_t rt, uint32_t code_tiles, uint32_t code_at) const {
        return rt < code_tiles ? code_at : kOut;
    }
    __host__ __device__ uint32_t code_s(uint32_t rt, uint32_t seg) const { return rt * 16 * row_bytes + 64 * seg; }
    // Fragment f of RHS tile ct in unit u; lane l reads 16 bytes.
    __host__ __device__ uint32_t image(uint32_t u, uint32_t ct) const { return (u * 2 * ntb + ct) * img_bytes(g32); }
    __host__ __device__ uint32_t frag_v(uint32_t lane, uint32_t u, uint32_t ct) const {
        return u < units && ct < tiles ? lane * 16 : kOut;
    }
    __host__ __device__ uint32_t frag_s(uint32_t u, uint32_t ct, uint32_t f) const {
        return image(u, ct) + f * uint32_t(kFragBytes);
    }
    // Sum of RHS 16 ct + r16 over quarter `sub` of unit u (group 32) or half
    // `sub` (the other groups).
    __host__ __device__ uint32_t sum_at(uint32_t u, uint32_t sub, uint32_t ct, uint32_t r16) const {
        return u < units && ct < tiles ? image(u, ct) + img_sums(g32) + sub * 64 + r16 * 4 : kOut;
    }
    // Factors of RHS 16 ct + 4 q .. + 3 over half `sub`: four bytes.
    __host__ __device__ uint32_t factor_at(uint32_t u, uint32_t sub, uint32_t ct, uint32_t q) const {
        return u < units && ct < tiles ? image(u, ct) + kImgFactors + sub * 16 + q * 4 : kOut;
    }
};

// The scales or biases of eight consecutive groups from group g of a row on:
// 16 bytes of a window of whole words and its rest 16 bytes further. The window
// begins in the word of the first one, or as far before it as the view's end
// asks; skip() elements of it are not wanted. A view of 16-bit elements ends
// in a whole word (no buffer is shorter), whose other half is not used.
template <int META>
struct MetaWindow {
    static constexpr uint32_t kSize = META == 0 ? 4 : 2;    // bytes of an element
    static constexpr uint32_t kWords = META == 0 ? 8 : 5;
    uint32_t groups, bytes;  // of a row; of the view
    __host__ __device__ uint32_t at(uint32_t row, uint32_t g) const { return (row * groups + g) * kSize; }
    __host__ __device__ uint32_t window(uint32_t at) const {
        const uint32_t word = at & ~3u, last = bytes - 4 * kWords;
        return word < last ? word : last;
    }
    __host__ __device__ uint32_t skip(uint32_t at) const { return (at - window(at)) / kSize; }
};

// Metadata item i of thread tid: the row within the block and the groups
// 8 j.. of a chunk.
__host__ __device__ constexpr uint32_t units_per_chunk(bool g32) { return g32 ? 1 : 2; }  // four slots each
struct MetaItem {
    uint32_t row, j;
};
__host__ __device__ inline MetaItem meta_item(uint32_t tid, uint32_t i, uint32_t threads, uint32_t items_per_row) {
    const uint32_t k = tid + i * threads;  // items per row: a power of two
    return MetaItem{k >> (31 - __builtin_clz(items_per_row)), tid & (items_per_row - 1)};
}
__host__ __device__ constexpr uint32_t items_per_thread(uint32_t nrt) { return (nrt + 7) / 8; }

struct WideParams {
    const uint32_t *w;
    const void *s;
    const void *b;
    const float *x;
    float *y;              // output, or the first K split's plane
    unsigned char *img;    // [units][2 ntb] images
    uint32_t rows, cols, n;       // n = RHS count
    uint32_t group;
    uint32_t units, groups;       // 128-column units (the last may be partial) and quant groups per row
    uint32_t ntb, ncb;            // 32-RHS images, RHS blocks of the contraction
    uint32_t nrb, ns, ups;        // row blocks, K splits, units per split
    uint32_t plane;               // floats between K splits' planes (0: one split)
    uint32_t w_bytes, m_bytes, img_bytes;  // extents of the views
};

// ---- 1. Activation images: a wave per unit and RHS tile, lane (t16, c4) the
// columns 8*c4.. of the four K steps of RHS t16. ----
constexpr uint32_t kPrepWaves = 1;

// Group 32: parts are cut off, not rounded: three times eight bits are all of
// a value's, and the first does not overflow. Inf and NaN stay out of the
// fragments; NaN in place of their quarter's sum says that there are some.
template <int BITS>
__device__ __forceinline__ void put_image32(float (&xv)[4][8], unsigned char *img, uint32_t lane) {
#pragma unroll
    for (uint32_t ks = 0; ks < 4; ++ks) {
        float(&v)[8] = xv[ks];
        float bad = 0.f;  // NaN where a value is not finite
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool finite = __builtin_isfinite(v[j]);
            bad = finite ? bad : __builtin_nanf("");
            v[j] = finite ? v[j] : 0.f;
        }
        float sum = bad + (((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        if (lane < 16) reinterpret_cast<float *>(img + img_sums(true))[ks * 16 + lane] = sum;
        u4 part[3];
#pragma unroll
        for (int e2 = 0; e2 < 4; ++e2) {
            float r0 = v[2 * e2] * kXFactor<BITS>, r1 = v[2 * e2 + 1] * kXFactor<BITS>;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const uint32_t b0 = __float_as_uint(r0) & 0xFFFF0000u, b1 = __float_as_uint(r1) & 0xFFFF0000u;
                part[k][e2] = b0 >> 16 | b1;
                r0 -= __uint_as_float(b0);
                r1 -= __uint_as_float(b1);
            }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<u4 *>(img + (3 * ks + k) * kFragBytes + lane * 16) = part[k];
    }
}

// The other groups: hi and lo f16 halves under a power of two of its own for
// every RHS and 64 columns, as the block kernels have it for every group: a
// column loses bits only where another of the same 64 is 2^17 times larger.
// (One per RHS and K class asked that of an eighth of the row.)
template <int BITS>
__device__ __forceinline__ void put_image64(const float (&xv)[4][8], unsigned char *img, uint32_t lane) {
#pragma unroll
    for (uint32_t half = 0; half < 2; ++half) {
        uint32_t mb = 0;
        float sum = 0.f;
#pragma unroll
        for (uint32_t ks = 2 * half; ks < 2 * half + 2; ++ks) {
            const float(&v)[8] = xv[ks];
            sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
            for (int j = 0; j < 8; ++j) mb = max(mb, __float_as_uint(v[j]) & 0x7FFFFFFFu);
        }
        sum += __shfl_xor(sum, 16);
        sum += __shfl_xor(sum, 32);
        mb = max(mb, uint32_t(__shfl_xor(int(mb), 16)));
        mb = max(mb, uint32_t(__shfl_xor(int(mb), 32)));
        int e = 0;
        if (mb != 0u && mb < 0x7F800000u) {
            e = int(mb >> 23) - 127 - 14;  // max * 2^-e in [2^14, 2^15) for normal max
            e = e < -100 ? -100 : (e > 100 ? 100 : e);
        }
        if (lane < 16) {
            reinterpret_cast<float *>(img + img_sums(false))[half * 16 + lane] = sum;
            img[kImgFactors + half * 16 + lane] = static_cast<unsigned char>(127 + e);
        }
        const float sc = __uint_as_float(uint32_t(127 - e) << 23);
#pragma unroll
        for (uint32_t ks = 2 * half; ks < 2 * half + 2; ++ks) {
            u4 hw, lw;
#pragma unroll
            for (int e2 = 0; e2 < 4; ++e2) {
                const float v0 = xv[ks][k_of<BITS>(2 * e2)], v1 = xv[ks][k_of<BITS>(2 * e2 + 1)];
                hw[e2] = hi_pair(v0, v1, sc);
                lw[e2] = lo_pair(v0, v1, sc, hw[e2]);
            }
            *reinterpret_cast<u4 *>(img + 2 * ks * kFragBytes + lane * 16) = hw;
            *reinterpret_cast<u4 *>(img + (2 * ks + 1) * kFragBytes + lane * 16) = lw;
        }
    }
}

template <int BITS, bool G32>
__global__ __launch_bounds__(64 * kPrepWaves) void wide_prep_kernel(WideParams p, uint32_t tiles) {
    const uint32_t i = blockIdx.x * kPrepWaves + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const uint32_t u = i / tiles, ct = i % tiles;
    if (u >= p.units) return;
    const uint32_t t = ct * 16 + (lane & 15);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(p.x), 0, int(p.n * p.cols * 4u), kRsrcWord3);
    float xv[4][8];
#pragma unroll
    for (uint32_t ks = 0; ks < 4; ++ks)
        load_x8(xv[ks], xr, t, u * kUnit + 32 * ks + 8 * (lane >> 4), p.cols, t < p.n);
    unsigned char *img = p.img + (size_t(u) * 2 * p.ntb + ct) * img_bytes(G32);
    if constexpr (G32)
        put_image32<BITS>(xv, img, lane);
    else
        put_image64<BITS>(xv, img, lane);
}

// What Inf and NaN among the columns [c0, c1) of an RHS add to row r of a
// group 32 product, as the vector-ALU kernel has it: code * x times the scale,
// and the bias times x.
template <int BITS, int META>
__device__ float non_finite(const WideParams &p, uint32_t t, uint32_t c0, uint32_t c1, uint32_t r) {
    constexpr uint32_t PACK = 32 / BITS;
    float sum = 0.f;
    for (uint32_t c = c0; c < c1; ++c) {
        const float v = p.x[size_t(t) * p.cols + c];
        if (__builtin_isfinite(v)) continue;
        const uint32_t code = p.w[size_t(r) * (p.cols / PACK) + c / PACK] >> (c % PACK * BITS) & ((1u << BITS) - 1);
        const size_t g = size_t(r) * p.groups + c / 32;
        auto meta = [&](const void *m) {
            return META == 0 ? static_cast<const float *>(m)[g] : meta_f32<META>(static_cast<const uint16_t *>(m)[g]);
        };
        sum += meta(p.s) * (float(code) * v) + meta(p.b) * v;
    }
    return sum;
}

// ---- 2. The contraction. Lane (r16, q) of a wave: row r16 of every row
// tile, K chunk q of every K step; D element v of a tile is RHS 4q + v. ----
template <int BITS, int META, bool G32, int NRT, int NCT, int NW_>
__global__ __launch_bounds__(64 * NW_, 2) void wide_mfma_kernel(WideParams p) {
    constexpr uint32_t NW = NW_;
    constexpr int ROWS = 16 * NRT;
    constexpr int SEG = BITS / 4;         // 64-byte code segments per unit
    constexpr int KPS = 4 / SEG;          // K steps per segment
    constexpr int KG = G32 ? 1 : 2;       // K steps per group (or half of 128)
    constexpr int PARTS = parts_of(G32);  // of x
    constexpr int SL = 4 / KG;            // slots (groups or halves of 128) per unit
    constexpr uint32_t UPC = units_per_chunk(G32);
    constexpr int THREADS = 64 * NW_, PITCH = meta_pitch(NW_);
    constexpr int PER_T = items_per_thread(NRT);  // metadata items per thread and chunk
    constexpr int RJ = (ROWS + 63) / 64;  // waves' worth of rows
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);  // the wave's K class (uniform)
    const int lane = tid & 63;
    const int r16 = lane & 15, q = lane >> 4;
    unsigned char *turn = lds + 2 * meta_bytes(NRT, NW_) + size_t(wv) * code_bytes(NRT);
    // XCD-aware order: workgroup i runs on XCD i % 8, so the RHS blocks of one
    // row block (which read the same codes at about the same time) share an
    // XCD and its L2.
    const uint32_t xcd = blockIdx.x % 8, slot = blockIdx.x / 8;
    const uint32_t cb = slot % p.ncb, pair = (slot / p.ncb) * 8 + xcd;
    if (pair >= p.nrb * p.ns) return;
    const uint32_t rb = pair % p.nrb, split = pair / p.nrb;
    const uint32_t row0 = rb * ROWS, ct0 = cb * NCT;
    const uint32_t u0 = split * p.ups, u1 = min(u0 + p.ups, p.units);
    const WideAddr A{p.rows, u1, (p.n + 15) / 16, p.cols / (32 / BITS) * 4, p.ntb, G32};
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t *>(p.w), 0, int(p.w_bytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t ir = __builtin_amdgcn_make_buffer_rsrc(p.img, 0, int(p.img_bytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t sr = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.s), 0, int(p.m_bytes), kRsrcWord3);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.b), 0, int(p.m_bytes), kRsrcWord3);
    const f4 zero{0.f, 0.f, 0.f, 0.f};
    const CodeConsts<BITS> consts;

    // ---- codes: lane (row16, piece) loads 16 bytes of a row of every tile.
    const uint32_t row16 = uint32_t(lane) >> 2, piece = uint32_t(lane) & 3;
    const uint32_t code_at = A.code_at(row0 + row16, piece), row_tiles = A.row_tiles(row0 + row16);
    u4 raw[SEG][NRT];
    auto load_codes = [&](u4 (&dst)[NRT], uint32_t u, int sg) {
        const uint32_t seg = u * SEG + uint32_t(sg), tiles = A.code_tiles(row_tiles, u, seg, piece);
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt)
            dst[rt] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(
                                                 wr, int(A.code_v(uint32_t(rt), tiles, code_at)), int(A.code_s(uint32_t(rt), seg)), 0));
    };
    auto put_codes = [&](const u4 (&src)[NRT]) {
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt)
            *reinterpret_cast<u4 *>(turn + (rt * 16 + row16) * kCodePitch + code_piece(row16, piece)) = src[rt];
    };
    // ---- metadata of chunk c (units u0 + UPC*NW*c ..): item (row, j) = eight
    // consecutive groups of one row, shifted into place when they are used.
    const uint32_t gpu = kUnit / p.group;      // groups per unit
    const uint32_t gpc = gpu * UPC * NW;       // groups per chunk: 4 NW (group 128: 2 NW)
    const uint32_t ipr = gpc / 8;              // items per row
    const MetaWindow<META> M{p.groups, p.m_bytes};
    const uint32_t mj = meta_item(uint32_t(tid), 0, THREADS, ipr).j;
    const uint32_t g_first = gpu * u0, g_end = min(p.groups, gpu * u1);
    constexpr uint32_t WIN = MetaWindow<META>::kWords;
    struct MStage {
        u4 s0[PER_T], b0[PER_T];
        std::conditional_t<META == 0, u4, uint32_t> s1[PER_T], b1[PER_T];
    };
    auto item_row = [&](int i) { return meta_item(uint32_t(tid), uint32_t(i), THREADS, ipr).row; };
    auto item_at = [&](uint32_t rl, uint32_t c) { return M.at(row0 + rl, g_first + c * gpc + 8 * mj); };
    auto item_live = [&](uint32_t rl, uint32_t c) {
        return rl < uint32_t(ROWS) && row0 + rl < p.rows && g_first + c * gpc + 8 * mj < g_end;
    };
    auto load_meta = [&](MStage &st, uint32_t c) {
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const uint32_t rl = item_row(i);
            const uint32_t at = item_live(rl, c) ? M.window(item_at(rl, c)) : kOut;
            st.s0[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(sr, int(at), 0, 0));
            st.b0[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(br, int(at), 0, 0));
            if constexpr (META == 0) {
                st.s1[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(sr, int(at + 16u), 0, 0));
                st.b1[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(br, int(at + 16u), 0, 0));
            } else {
                st.s1[i] = __builtin_amdgcn_raw_buffer_load_b32(sr, int(at + 16u), 0, 0);
                st.b1[i] = __builtin_amdgcn_raw_buffer_load_b32(br, int(at + 16u), 0, 0);
            }
        }
    };
    // The window's elements from `skip` on (0, or 1 for a row that starts
    // inside a word; more only where the view ends, handled word by word).
    auto eight = [&](float (&out)[8], const u4 &w0, const auto &w1, uint32_t skip) {
        uint32_t w[WIN];
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = w0[k];
        if constexpr (META == 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) w[4 + k] = w1[k];
        } else {
            w[4] = w1;
        }
        const uint32_t words = META == 0 ? skip : skip >> 1;  // at most WIN - 1: the item starts inside the view
        for (uint32_t i = 0; i < WIN - 1 && i < words; ++i) {
#pragma unroll
            for (uint32_t k = 0; k + 1 < WIN; ++k) w[k] = w[k + 1];
        }
        if constexpr (META == 0) {
#pragma unroll
            for (int k = 0; k < 8; ++k) out[k] = __uint_as_float(w[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t v = __builtin_amdgcn_alignbit(w[k + 1], w[k], (skip & 1) * 16);
                out[2 * k] = meta_f32<META>(v & 0xFFFFu);
                out[2 * k + 1] = META == 1 ? __uint_as_float(v & 0xFFFF0000u) : meta_f32<META>(v >> 16);
            }
        }
    };
    auto put_meta = [&](const MStage &st, uint32_t c) {
        float *ms = reinterpret_cast<float *>(lds + (c & 1) * meta_bytes(NRT, NW_));
        float *mb = ms + ROWS * PITCH;
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const uint32_t rl = item_row(i);
            const uint32_t skip = item_live(rl, c) ? M.skip(item_at(rl, c)) : 0u;
            float sv[8], bv[8];
            eight(sv, st.s0[i], st.s1[i], skip);
            eight(bv, st.b0[i], st.b1[i], skip);
            const uint32_t g = g_first + c * gpc + 8 * mj;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) {  // past the split's groups there may be a neighbour's
                sv[k] = g + k < g_end ? sv[k] : 0.f;
                bv[k] = g + k < g_end ? __builtin_fmaf(middle_of(BITS), sv[k], bv[k]) : 0.f;
                if constexpr (G32) sv[k] *= kSFactor<BITS>;
            }
            if (rl >= uint32_t(ROWS)) continue;
            // Unit NW*i + class of the chunk: slots 4*class + 2*i + half
            // (group 32: 4*class + quarter); a group of 128 fills both halves.
            float *s_row = ms + rl * PITCH, *b_row = mb + rl * PITCH;
            if constexpr (G32) {
#pragma unroll
                for (int k = 0; k < 8; k += 2) {
                    *reinterpret_cast<f2 *>(s_row + 8 * mj + k) = f2{sv[k], sv[k + 1]};
                    *reinterpret_cast<f2 *>(b_row + 8 * mj + k) = f2{bv[k], bv[k + 1]};
                }
            } else if (p.group == 64) {
                const uint32_t ul = 4 * mj, sl = (ul % NW) * 4 + (ul / NW) * 2;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    *reinterpret_cast<f2 *>(s_row + sl + 4 * k) = f2{sv[2 * k], sv[2 * k + 1]};
                    *reinterpret_cast<f2 *>(b_row + sl + 4 * k) = f2{bv[2 * k], bv[2 * k + 1]};
                }
            } else {
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k) {
                    const uint32_t ul = 8 * mj + k, sl = (ul % NW) * 4 + (ul / NW) * 2;
                    *reinterpret_cast<f2 *>(s_row + sl) = f2{sv[k], sv[k]};
                    *reinterpret_cast<f2 *>(b_row + sl) = f2{bv[k], bv[k]};
                }
            }
        }
    };
    // ---- x
    u4 xf[4][NCT][PARTS];  // a unit's K steps; whole words: halves carried across the loop would be taken apart and put together
    auto load_x = [&](u4 (&dst)[NCT][PARTS], uint32_t u, uint32_t ks) {
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
            const int v = int(A.frag_v(uint32_t(lane), u, ct0 + uint32_t(ct)));
#pragma unroll
            for (int part = 0; part < PARTS; ++part)
                dst[ct][part] = __builtin_bit_cast(
                    u4, __builtin_amdgcn_raw_buffer_load_b128(ir, v, int(A.frag_s(u, ct0 + uint32_t(ct), PARTS * ks + uint32_t(part))), 0));
        }
    };
    // Bias A operands of chunk c: lane (t16, q) the sum of slot q.
    auto load_s = [&](float (&sop)[NCT], uint32_t c) {
        const uint32_t u = u0 + c * UPC * NW + uint32_t(wv) + (G32 ? 0u : NW * (uint32_t(q) >> 1));
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct)
            sop[ct] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                ir, int(A.sum_at(u, G32 ? uint32_t(q) : uint32_t(q) & 1, ct0 + uint32_t(ct), uint32_t(r16))), 0, 0));
    };

    // Factors of a unit's half for the lane's four RHS: exponent bytes.
    uint32_t fe[2][NCT];
    auto load_factors = [&](uint32_t (&dst)[NCT], uint32_t u, uint32_t half) {
        if constexpr (!G32)
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct)
                dst[ct] = __builtin_amdgcn_raw_buffer_load_b32(ir, int(A.factor_at(u, half, ct0 + uint32_t(ct), uint32_t(q))), 0, 0);
    };

    f4 acc[NRT][NCT];
    float sa[NCT];
    bool bad[NCT] = {};  // group 32: Inf or NaN in the columns of sa
    auto clean = [&](float (&sop)[NCT]) {
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
            const bool nan = sop[ct] != sop[ct];
            bad[ct] |= nan;
            sop[ct] = nan ? 0.f : sop[ct];
        }
    };
    {
        const uint32_t u = u0 + uint32_t(wv);
        MStage st;
        load_meta(st, 0);
#pragma unroll
        for (int sg = 0; sg < SEG; ++sg) load_codes(raw[sg], u, sg);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) load_x(xf[ks], u, uint32_t(ks));
        for (uint32_t half = 0; half < 2; ++half) load_factors(fe[half], u, half);
        load_s(sa, 0);
        __builtin_amdgcn_sched_barrier(0);  // every request before any use
        put_meta(st, 0);
    }
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc[rt][ct] = zero;
    lds_barrier();

    // Codes of K step k of the segment in the turn buffer, row tile rt, as a B operand.
    auto operand = [&](int rt, int k) {
        const unsigned char *row = turn + (rt * 16 + r16) * kCodePitch;
        const uint32_t r = uint32_t(r16), c = uint32_t(q), s = uint32_t(k);
        if constexpr (BITS == 4) return u2{*reinterpret_cast<const uint32_t *>(row + code_piece(r, s) + 4 * c), 0u};
        else return *reinterpret_cast<const u2 *>(row + code_piece(r, 2 * s + (c >> 1)) + 8 * (c & 1));
    };
    // The wave's units of the split, the last one perhaps past it (its loads
    // read zeros): the loop body has no branch, so every wait counts on the
    // loads really in flight.
    const uint32_t nu = (u1 - u0 + NW - 1) / NW;
    for (uint32_t c = 0;; ++c) {
        const float *ms = reinterpret_cast<const float *>(lds + (c & 1) * meta_bytes(NRT, NW_)) + r16 * PITCH + 4 * wv;
        const float *mb = ms + ROWS * PITCH;
        MStage st;
        float sb[NCT];
        load_meta(st, c + 1);
        load_s(sb, c + 1);
        const uint32_t n = min(UPC, nu - c * UPC);
        uint32_t h = 0;
        do {
            const uint32_t u = u0 + (c * UPC + h) * NW + uint32_t(wv), un = u + NW;
#pragma unroll
            for (int sg = 0; sg < SEG; ++sg) {
                put_codes(raw[sg]);
                load_codes(raw[sg], un, sg);
                wave_lds_sync();
#pragma unroll
                for (int k0 = 0; k0 < KPS; k0 += KG) {
                    const int ks = sg * KPS + k0, sl = ks / KG;  // the group's first K step, its slot
                    // Software-pipelined by row tile: step rt issues tile rt's
                    // products and, on the vector ALU, the epilogue of tile
                    // rt-1 and the unpacking of tile rt+1; codes and scales
                    // are read from LDS two tiles ahead.
                    u4 op[2][KG];
                    u2 w[2][KG];
                    float sv[3];
                    auto fetch = [&](int rt) {
#pragma unroll
                        for (int k = 0; k < KG; ++k) w[rt & 1][k] = operand(rt, k0 + k);
                        sv[rt % 3] = ms[rt * 16 * PITCH + SL * h + sl];
                    };
                    auto open = [&](int rt) {
#pragma unroll
                        for (int k = 0; k < KG; ++k) {
                            if constexpr (G32) op[rt & 1][k] = bf16_codes<BITS>(w[rt & 1][k]);
                            else op[rt & 1][k] = f16_codes<BITS>(w[rt & 1][k], consts);
                        }
                    };
                    f4 d[2][NCT];
                    f4 fac[NCT];
                    if constexpr (!G32)
#pragma unroll
                        for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                fac[ct][v] = __uint_as_float((v < 3 ? fe[sl & 1][ct] << (23 - 8 * v) : fe[sl & 1][ct] >> 1) & 0x7F800000u);
                    auto close = [&](int rt) {
#pragma unroll
                        for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
                            for (int v = 0; v < 4; ++v)
                                acc[rt][ct][v] = __builtin_fmaf(sv[rt % 3], G32 ? d[rt & 1][ct][v] : d[rt & 1][ct][v] * fac[ct][v],
                                                                acc[rt][ct][v]);
                    };
                    fetch(0);
                    if (NRT > 1) fetch(1);
                    open(0);
#pragma unroll
                    for (int rt = 0; rt < NRT; ++rt) {
                        __builtin_amdgcn_sched_barrier(0);
                        // All hi products before the lo ones: half the error
                        // of hi and lo in turn (2.4e-7 against 4.4e-7 at 5120
                        // columns of uncentred Q4), a quarter of lo first.
#pragma unroll
                        for (int part = 0; part < PARTS; ++part)
#pragma unroll
                            for (int k = 0; k < KG; ++k)
#pragma unroll
                                for (int ct = 0; ct < NCT; ++ct)
                                    d[rt & 1][ct] = product<G32>(xf[ks + k][ct][part], op[rt & 1][k],
                                                                 k == 0 && part == 0 ? zero : d[rt & 1][ct]);
                        if (rt + 1 < NRT) open(rt + 1);
                        if (rt > 0) close(rt - 1);
                        if (rt + 2 < NRT) fetch(rt + 2);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int k = 0; k < KG; ++k) load_x(xf[ks + k], un, uint32_t(ks + k));
                    load_factors(fe[sl & 1], un, uint32_t(sl & 1));
                    close(NRT - 1);
                }
                wave_lds_sync();
            }
            // Bias of the chunk's four slots, acc += S x b, after its first
            // unit: b * S cancels most of s * D, so in the middle the sums
            // stray half as far.
            if (h == 0) {
                if constexpr (G32) clean(sa);
#pragma unroll
                for (int rt = 0; rt < NRT; ++rt) {
                    const float bv = mb[rt * 16 * PITCH + q];
#pragma unroll
                    for (int ct = 0; ct < NCT; ++ct)
                        acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(sa[ct], bv, acc[rt][ct], 0, 0, 0);
                }
            }
        } while (++h < n);
        if ((c + 1) * UPC >= nu) break;
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) sa[ct] = sb[ct];
        put_meta(st, c + 1);
        lds_barrier();
    }

    // ---- the classes meet in LDS and are added in order. A wave stores 64
    // rows of an RHS at a time.
    lds_barrier();  // every wave is done with its piece
    float *red = reinterpret_cast<float *>(lds);
    constexpr int TILE = NCT * 256 + kRedPad;
    constexpr uint32_t PLANES = NW > 4 ? 4 : NW;
    auto place = [&](int rt, int ct, int v) -> float & {
        return red[((wv % int(PLANES)) * NRT + rt) * TILE + (ct * 4 + v) * 64 + lane];
    };
    if (wv < int(PLANES)) {
#pragma unroll
        for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
                for (int v = 0; v < 4; ++v) place(rt, ct, v) = acc[rt][ct][v];
    }
    lds_barrier();
    if constexpr (NW > PLANES) {
        if (wv >= int(PLANES)) {
#pragma unroll
            for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
                for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
                    for (int v = 0; v < 4; ++v) place(rt, ct, v) += acc[rt][ct][v];
        }
        lds_barrier();
    }
    uint32_t inf[NCT] = {};  // RHS with Inf or NaN in this split, a bit each
    if constexpr (G32) {
        uint32_t *flags = reinterpret_cast<uint32_t *>(lds + wide_lds_bytes(NRT, NCT, NW_) - kFlagBytes);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
            const uint64_t b = __ballot(bad[ct]);
            if (lane == 0) flags[wv * NCT + ct] = uint32_t(b | b >> 16 | b >> 32 | b >> 48) & 0xFFFFu;
        }
        lds_barrier();
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct)
            for (uint32_t k = 0; k < NW; ++k) inf[ct] |= flags[k * NCT + ct];
    }
    float *out = p.y + size_t(split) * p.plane;
    const uint32_t rows_here = min(uint32_t(ROWS), p.rows - row0);
    for (uint32_t i = uint32_t(wv); i < uint32_t(RJ) * 16 * NCT; i += NW) {
        const uint32_t tl = i / RJ, rl = (i % RJ) * 64 + uint32_t(lane);  // RHS 16 ct + 4 q + v of the block, row
        const uint32_t t = ct0 * 16 + tl;
        if (t >= p.n) break;  // uniform
        if (rl < rows_here) {
            const uint32_t at = (rl >> 4) * TILE + ((tl >> 4) * 4 + (tl & 3)) * 64 + ((tl >> 2) & 3) * 16 + (rl & 15);
            float sum = 0.f;
#pragma unroll
            for (uint32_t k = 0; k < PLANES; ++k) sum += red[k * NRT * TILE + at];
            if constexpr (G32)
                if ((tl < 16 ? inf[0] : inf[NCT - 1]) >> (tl % 16) & 1)
                    sum += non_finite<BITS, META>(p, t, u0 * kUnit, min(u1 * kUnit, p.cols), row0 + rl);
            out[size_t(t) * p.rows + row0 + rl] = sum;
        }
    }
}

// ---- 3. The K splits' planes, added in split order. ----
__global__ __launch_bounds__(256) void wide_sum_kernel(const float *__restrict__ planes, float *__restrict__ y,
                                                       uint32_t count, uint32_t ns) {
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < count; i += gridDim.x * 256) {
        float v = 0.f;
        for (uint32_t k = 0; k < ns; ++k) v += planes[size_t(k) * count + i];
        y[i] = v;
    }
}

template <int BITS, int META, bool G32, int NRT, int NCT, int NW>
hipError_t launch_instance(const WideParams &p, hipStream_t stream) {
    auto kernel = wide_mfma_kernel<BITS, META, G32, NRT, NCT, NW>;
    constexpr size_t lds = wide_lds_bytes(NRT, NCT, NW);
    const hipError_t e = raise_lds_limit(reinterpret_cast<const void *>(kernel), lds);
    if (e != hipSuccess) return e;
    const uint32_t grid = (p.nrb * p.ns + 7) / 8 * 8 * p.ncb;  // XCD-aware order; surplus workgroups exit
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(64 * NW), lds, stream, p);
    return hipGetLastError();
}

// The instances of a format. F16 metadata comes in blocks of up to four RHS
// only, in group 32. Those left out need more than the 256 registers of two
// waves per SIMD: 12288x4096 Q8 with 256 RHS 117 us with 8 x 2 tiles, 85 with
// 6 x 2; 5120x5120 Q8 group 32 with 24 RHS 29 us with 7 x 2, 22 with 4 x 2.
constexpr bool has_instance(int bits, int meta, bool g32, uint32_t rt, uint32_t ct) {
    return !(meta == 2 && ct > 1) && !(ct > 1 && rt >= 8 && (bits == 8 || g32)) && !(ct > 1 && rt >= 7 && bits == 8 && g32);
}

template <int BITS, int META, bool G32>
hipError_t launch_tile(const WideParams &p, const WidePlan &pl, hipStream_t stream) {
#define QMR_WIDE(RT, CT, NW)                                                                                  \
    if constexpr (has_instance(BITS, META, G32, RT, CT))                                                      \
        if (pl.rt == RT && pl.ct == CT && pl.nw == NW) return launch_instance<BITS, META, G32, RT, CT, NW>(p, stream);
    QMR_WIDE(2, 1, 8) QMR_WIDE(4, 1, 4) QMR_WIDE(4, 1, 8) QMR_WIDE(5, 1, 8) QMR_WIDE(8, 1, 8) QMR_WIDE(8, 1, 4)
    QMR_WIDE(4, 2, 4) QMR_WIDE(4, 2, 8) QMR_WIDE(5, 2, 8) QMR_WIDE(7, 2, 4) QMR_WIDE(8, 2, 4) QMR_WIDE(6, 2, 4) QMR_WIDE(6, 2, 8)
#undef QMR_WIDE
    return hipErrorNotSupported;
}

// Regions of the workspace.
struct Regions {
    size_t planes, total;
};
Regions regions(const AffineArgs &a, const WidePlan &pl) {
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t units = (a.cols + kUnit - 1) / kUnit, ntb = (a.batch + kRhsBlock - 1) / kRhsBlock;
    const bool g32 = a.group == 32;
    Regions r{};
    r.planes = up(units * 2 * ntb * img_bytes(g32));
    r.total = r.planes + (pl.ns > 1 ? size_t(pl.ns) * a.batch * a.rows * 4 : 0);
    return r;
}

// Whole rounds of a workgroup's waves per split; splits left without a unit go.
WidePlan split_units(WidePlan pl, uint32_t units) {
    pl.ups = ((units + pl.ns - 1) / pl.ns + pl.nw - 1) / pl.nw * pl.nw;
    pl.ns = (units + pl.ups - 1) / pl.ups;
    return pl;
}

}  // namespace

bool wide_mfma_supported(const AffineArgs &a) {
    if (a.bits != 4 && a.bits != 8) return false;
    if (a.group != 32 && a.group != 64 && a.group != 128) return false;
    if (a.batch < 1 || a.batch > 256 || a.residual || a.up_w) return false;
    // Codes at any 4-byte offset can be loaded, but such views run on the
    // vector ALU as blocks, in FP32, which group 32 alone keeps here.
    if (a.group != 32 && reinterpret_cast<uintptr_t>(a.w) % 16 != 0) return false;
    if (a.meta == Meta::F16 && (a.group != 32 || a.batch > 16)) return false;  // no wide block has it
    // 32-bit buffer offsets: codes reach one workgroup's rows past the
    // matrix, images one chunk of units past the row (all read as zeros).
    const uint64_t row_bytes = uint64_t(a.cols) * a.bits / 8;
    const uint64_t ntb = (a.batch + kRhsBlock - 1) / kRhsBlock;
    const uint64_t img = (uint64_t(a.cols + kUnit - 1) / kUnit + 40) * 2 * ntb * img_bytes(a.group == 32);
    const uint64_t meta = uint64_t(a.rows) * (a.cols / a.group) * (a.meta == Meta::F32 ? 4 : 2);
    return uint64_t(a.batch) * a.cols * 4 < (1ull << 31) && (uint64_t(a.rows) + 16 * 10) * row_bytes < (1ull << 31) &&
           img < (1ull << 31) && meta < (1ull << 31) && meta >= 32;
}

namespace {
struct Instance {
    uint32_t rt, ct, nw, per_cu;  // per_cu: workgroups that fit a CU (LDS, registers)
};
constexpr Instance kInstances[] = {{2, 1, 8, 1}, {4, 1, 4, 3}, {4, 1, 8, 1}, {5, 1, 8, 1}, {8, 1, 8, 1}, {8, 1, 4, 2},
                                   {4, 2, 4, 2}, {4, 2, 8, 1}, {5, 2, 8, 1}, {7, 2, 4, 2}, {8, 2, 4, 2},
                                   {6, 2, 4, 2}, {6, 2, 8, 1}};
}  // namespace

// The plan is the cheapest of the compiled instances and up to eight K splits
// under a model of what a workgroup does, fitted to the times of every plan of
// 485 products (20 shapes from 1500x2048 and 512x8192 to 24576x2560 and
// 17408x5120, 5 to 256 RHS, both code sizes, groups 32, 64 and 128): its choice
// is on average 0.8% slower than the fastest plan (1.1% on products that a fit
// to the other half has not seen), more than 13% in two only, whose images
// pass an XCD's L2 (2560x8192 group 32 with 200 RHS: 89 us, 65 in two splits).
WidePlan plan_wide(const AffineArgs &a, const DeviceLimits &lim, const WidePlan &force) {
    // Microseconds, by RHS tiles of a workgroup where there are two: a group
    // step's products per row tile, the factors of group 32 and of Q8 on them,
    // the factor of a CU with less than two waves per SIMD; a metadata chunk, a
    // workgroup, a round of them, the sum launch and its planes per million
    // floats.
    constexpr float kStep[2] = {0.089f, 0.1367f}, kG32[2] = {0.860f, 0.929f}, kQ8[2] = {1.223f, 1.047f},
                    kLone[2] = {1.942f, 1.160f}, kChunk = 0.0572f, kWork = 0.399f, kRound = 6.71f, kSum = 2.34f,
                    kPlane = 4.74f;
    const uint32_t units = (a.cols + kUnit - 1) / kUnit, nct = (a.batch + 15) / 16;
    const uint32_t steps = a.group == 32 ? 4 : 2;  // group steps per unit
    // A row block's workgroups all run on one XCD.
    constexpr uint32_t kXcds = 8;
    const uint32_t cus = std::max(uint32_t(std::max(lim.num_cus, 1)) / kXcds, 1u);
    WidePlan best;
    float best_us = 0.f;
    for (const Instance &in : kInstances) {
        if (!has_instance(int(a.bits), a.meta == Meta::F16 ? 2 : 0, a.group == 32, in.rt, in.ct)) continue;
        if ((force.rt && force.rt != in.rt) || (force.ct && force.ct != in.ct) || (force.nw && force.nw != in.nw)) continue;
        const float step = float(in.rt) * kStep[in.ct - 1] * (a.group == 32 ? kG32[in.ct - 1] : 1.f) *
                           (a.bits == 8 ? kQ8[in.ct - 1] : 1.f);
        for (const uint32_t ns : {1u, 2u, 3u, 4u, 6u, 8u}) {
            WidePlan pl;
            pl.rt = in.rt;
            pl.ct = in.ct;
            pl.nw = in.nw;
            pl.ns = force.ns ? force.ns : ns;
            pl = split_units(pl, units);
            // A split's classes all have a unit; its planes fit the scratch of
            // the encode that allocates nothing, so that both take one plan.
            if (!force.ns && ns > 1 && (units / ns < in.nw || regions(a, pl).total > QMR_STATIC_SCRATCH_BYTES)) continue;
            const uint32_t upw = pl.ups / pl.nw;
            const float work = float(in.nw) / 4.f * (float(upw * steps) * step + float((upw * steps + 3) / 4) * kChunk) + kWork;
            auto round = [&](uint32_t k) {  // k workgroups on a CU at once
                return k == 0 ? 0.f : float(k) * work * (k * in.nw < 8 ? kLone[in.ct - 1] : 1.f) + kRound;
            };
            const uint32_t wgs = ((a.rows + 16 * in.rt - 1) / (16 * in.rt) * pl.ns + kXcds - 1) / kXcds *
                                 ((nct + in.ct - 1) / in.ct);  // of the busiest XCD
            const uint32_t full = wgs / (cus * in.per_cu), rest = wgs % (cus * in.per_cu);
            float us = float(full) * round(in.per_cu) + round((rest + cus - 1) / cus);
            if (pl.ns > 1) us += kSum + float(a.batch) * float(a.rows) * float(pl.ns) * kPlane * 1e-6f;
            if (best.rt == 0 || us < best_us) best = pl, best_us = us;
        }
    }
    return best;
}

size_t wide_mfma_workspace(const AffineArgs &a, const WidePlan &pl) { return regions(a, pl).total; }
size_t wide_mfma_image_bytes(const AffineArgs &a) {
    return size_t((a.cols + kUnit - 1) / kUnit) * 2 * img_bytes(a.group == 32);
}

WideExtent wide_address_extent(const AffineArgs &a, WidePlan pl) {
    WideExtent out{};
    const bool g32 = a.group == 32;
    const uint32_t units = (a.cols + kUnit - 1) / kUnit, ntb = (a.batch + kRhsBlock - 1) / kRhsBlock;
    const uint32_t groups = a.cols / a.group, gpu = kUnit / a.group;
    const uint32_t nrb = (a.rows + 16 * pl.rt - 1) / (16 * pl.rt), ncb = ((a.batch + 15) / 16 + pl.ct - 1) / pl.ct;
    const uint32_t segs = a.bits / 4;
    pl = split_units(pl, units);
    const uint64_t meta_view = uint64_t(a.rows) * groups * (a.meta == Meta::F32 ? 4 : 2);
    out.code_extent = uint64_t(a.rows) * a.cols * a.bits / 8;
    out.image_extent = uint64_t(units) * 2 * ntb * img_bytes(g32);
    out.meta_extent = (meta_view + 3) / 4 * 4;
    auto note = [](uint64_t &mx, uint32_t v, uint32_t so, uint32_t size) {
        if (v < kOut) mx = std::max(mx, uint64_t(v) + so + size);
    };
    auto meta_loads = [&](auto window, uint32_t row0, uint32_t g_first, uint32_t g_end, uint32_t c) {
        constexpr uint32_t rest = 4 * decltype(window)::kWords - 16;
        const uint32_t threads = 64 * pl.nw, gpc = gpu * units_per_chunk(g32) * pl.nw;
        for (uint32_t tid = 0; tid < threads; ++tid)
            for (uint32_t i = 0; i < items_per_thread(pl.rt); ++i) {
                const MetaItem m = meta_item(tid, i, threads, gpc / 8);
                const uint32_t g = g_first + c * gpc + 8 * m.j, row = row0 + m.row;
                if (m.row >= 16 * pl.rt || row >= a.rows || g >= g_end) continue;
                const uint32_t at = window.at(row, g), first = window.window(at);
                note(out.meta_end, first, 0, 16);
                note(out.meta_end, first, 16, rest);
                // What is used of them: the eight groups up to the split's end.
                const uint32_t wanted = std::min(8u, g_end - g) * window.kSize;
                out.meta_short = std::max<uint64_t>(out.meta_short, first + window.skip(at) * window.kSize != at ||
                                                                        at + wanted > first + 16 + rest);
            }
    };
    for (uint32_t split = 0; split < pl.ns; ++split) {
        const uint32_t u0 = split * pl.ups, u1 = std::min(u0 + pl.ups, units);
        const WideAddr A{a.rows, u1, (a.batch + 15) / 16, a.cols / (32 / a.bits) * 4, ntb, g32};
        // Every unit, and those past the split that the prefetches reach.
        for (uint32_t u = u0; u < u1 + 2 * pl.nw; ++u) {
            for (uint32_t row0 = 0; row0 < nrb * 16 * pl.rt; row0 += 16 * pl.rt)
                for (uint32_t l = 0; l < 64; ++l)
                    for (uint32_t seg = u * segs; seg < (u + 1) * segs; ++seg) {
                        const uint32_t row = row0 + (l >> 2), tiles = A.code_tiles(A.row_tiles(row), u, seg, l & 3);
                        for (uint32_t rt = 0; rt < pl.rt; ++rt)
                            note(out.code_end, A.code_v(rt, tiles, A.code_at(row, l & 3)), A.code_s(rt, seg), 16);
                    }
            for (uint32_t ct = 0; ct < ncb * pl.ct; ++ct)
                for (uint32_t l = 0; l < 64; ++l) {
                    for (uint32_t f = 0; f < 4 * parts_of(g32); ++f)
                        note(out.image_end, A.frag_v(l, u, ct), A.frag_s(u, ct, f), 16);
                    for (uint32_t sub = 0; sub < (g32 ? 4u : 2u); ++sub)
                        note(out.image_end, A.sum_at(u, sub, ct, l & 15), 0, 4);
                    for (uint32_t sub = 0; sub < 2 && !g32; ++sub)
                        note(out.image_end, A.factor_at(u, sub, ct, l >> 4), 0, 4);
                }
        }
        const uint32_t per = units_per_chunk(g32) * pl.nw, chunks = (u1 - u0 + per - 1) / per;
        for (uint32_t c = 0; c <= chunks; ++c)
            for (uint32_t row0 = 0; row0 < nrb * 16 * pl.rt; row0 += 16 * pl.rt) {
                const uint32_t g_first = gpu * u0, g_end = std::min(groups, gpu * u1);
                if (a.meta == Meta::F32)
                    meta_loads(MetaWindow<0>{groups, uint32_t(out.meta_extent)}, row0, g_first, g_end, c);
                else
                    meta_loads(MetaWindow<1>{groups, uint32_t(out.meta_extent)}, row0, g_first, g_end, c);
            }
    }
    return out;
}

bool wide_instance(const WidePlan &pl) {
    for (const Instance &in : kInstances)
        if (in.rt == pl.rt && in.ct == pl.ct && in.nw == pl.nw) return true;
    return false;
}

hipError_t launch_wide_mfma(const AffineArgs &a, const WidePlan &pl, unsigned char *workspace, hipStream_t stream) {
    const Regions r = regions(a, pl);
    WideParams p;
    p.w = a.w;
    p.s = a.s;
    p.b = a.b;
    p.x = a.x;
    p.img = workspace;
    float *planes = reinterpret_cast<float *>(workspace + r.planes);
    p.y = pl.ns > 1 ? planes : a.y;
    p.plane = pl.ns > 1 ? a.batch * a.rows : 0;
    p.rows = a.rows;
    p.cols = a.cols;
    p.n = a.batch;
    p.group = a.group;
    p.units = (a.cols + kUnit - 1) / kUnit;
    p.groups = a.cols / a.group;
    p.ntb = (a.batch + kRhsBlock - 1) / kRhsBlock;
    p.ncb = ((a.batch + 15) / 16 + pl.ct - 1) / pl.ct;
    p.nrb = (a.rows + 16 * pl.rt - 1) / (16 * pl.rt);
    p.ns = pl.ns;
    p.ups = pl.ups;
    p.w_bytes = uint32_t(uint64_t(a.rows) * a.cols * a.bits / 8);
    p.m_bytes = uint32_t((uint64_t(a.rows) * p.groups * (a.meta == Meta::F32 ? 4 : 2) + 3) / 4 * 4);
    const bool g32 = a.group == 32;
    p.img_bytes = uint32_t(size_t(p.units) * 2 * p.ntb * img_bytes(g32));
    const uint32_t tiles = (a.batch + 15) / 16;
    const auto prep = a.bits == 4 ? (g32 ? wide_prep_kernel<4, true> : wide_prep_kernel<4, false>)
                                  : (g32 ? wide_prep_kernel<8, true> : wide_prep_kernel<8, false>);
    hipLaunchKernelGGL(prep, dim3((p.units * tiles + kPrepWaves - 1) / kPrepWaves), dim3(64 * kPrepWaves), 0, stream, p, tiles);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    auto launch = [&](auto bits) {
        constexpr int B = decltype(bits)::value;
        if (a.meta == Meta::F32) return g32 ? launch_tile<B, 0, true>(p, pl, stream) : launch_tile<B, 0, false>(p, pl, stream);
        if (a.meta == Meta::BF16) return g32 ? launch_tile<B, 1, true>(p, pl, stream) : launch_tile<B, 1, false>(p, pl, stream);
        return launch_tile<B, 2, true>(p, pl, stream);
    };
    e = a.bits == 4 ? launch(std::integral_constant<int, 4>{}) : launch(std::integral_constant<int, 8>{});
    if (e != hipSuccess || pl.ns == 1) return e;
    const uint32_t count = a.batch * a.rows;
    hipLaunchKernelGGL(wide_sum_kernel, dim3(std::min((count + 255) / 256, 2048u)), dim3(256), 0, stream, planes, a.y,
                       count, pl.ns);
    return hipGetLastError();
}

}  // namespace qmr
